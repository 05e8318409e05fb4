// The BF16 reduced leapfrog with the operators on the CU as far as they fit; of
// few columns and many modes, on several CUs.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rom_device.hpp"
#include "rom_internal.hpp"
#include "shaw_common.hpp"

namespace shaw {
namespace {

typedef float flt2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

typedef unsigned u2 __attribute__((ext_vector_type(2)));

// the split of writeSplitRows with the hardware's conversion (round to nearest
// even, as f32ToBf16; a NaN becomes a quiet NaN)
__device__ __forceinline__ void splitRowsHw(const double (&q)[4], u2& h, u2& l) {
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const flt2 x = {(float)q[2 * p], (float)q[2 * p + 1]};
    const unsigned hb = __builtin_bit_cast(unsigned, __builtin_convertvector(x, bf16x2));
    h[p] = hb;
    const flt2 hf = {__uint_as_float(hb << 16), __uint_as_float(hb & 0xffff0000u)};
    l[p] = __builtin_bit_cast(unsigned, __builtin_convertvector(x - hf, bf16x2));
  }
}

__device__ __forceinline__ void writeSplitRowsHw(int4v* S, int loOff, int rt, int lane, const double (&q)[4]) {
  u2 h, l;
  splitRowsHw(q, h, l);
  const int item = (4 * (rt / 2) + lane / 16) * kTileCols + lane % 16;
  reinterpret_cast<u2*>(S + item)[rt % 2] = h;
  reinterpret_cast<u2*>(S + loOff + item)[rt % 2] = l;
}

// One workgroup advances 16 column slots as k_rom_steps_bf / k_rom_steps_bfm
// do (same splits, products and FP64 updates in the same order, so every value
// is theirs); here both operators, 2 KG row tiles by KG groups, are loaded into
// registers and LDS once per launch. Those kernels re-read both operators from
// L2 every step, and a CU's share of the L2 (about 90 GB/s measured, 64 B a
// clock at most) set their time. Bound now by the chain of a half-step (split
// -> LDS -> barrier -> products -> FP64 update), by MFMA from K = 192, and at
// K = 256 by the groups that still stream. Per step at 1024 columns, before ->
// now: BF16x3 K = 64 2.19 -> 0.54 us, 128 2.21 -> 0.90, 192 5.52 -> 1.57, 256
// 5.56 -> 2.62; BF16x4 2.56 -> 0.60, 2.57 -> 1.00, 7.20 -> 2.25, 7.25 -> 4.46.
// Waves: 2 KG row tiles in one or two per wave, at most 256 VGPRs, so that no
// operand passes through an AGPR; four waves of twice the tiles copy every
// operand out of AGPRs before its product (K = 192 BF16x3 1.98 against 2.40).
//
// SPLIT > 1: that many workgroups share a tile of 16 columns, each with 1 /
// SPLIT of the row tiles (one per wave), so that the operators fit the CUs that
// few columns would leave idle. After a half-step each wave writes its rows'
// split to a.xbuf and the workgroup reads the whole of it back from there. Bound
// by that exchange (1.4 us; more as the workgroups fill the chip) and the chain
// of 2 KG or more products; one workgroup a tile is bound by streaming the
// operators. Per step, one (of 4096 columns, all CUs streaming) -> several:
// BF16x4 K = 384 16.2 us -> 4.2 at 16 columns, 4.4 at 384, 4.6 at 640, 7.9 at
// 1280; K = 512 26.6 -> 4.8 at 16, 7.4 at 512, 12.7 at 1024; BF16x3 K = 384 9.6
// -> 4.3 at 640, 5.0 at 1280; K = 512 17.8 -> 9.0 at 512, 11.8 at 1024. (Flags that say the
// rows are there, read before them, are two more trips to memory: K = 384 5.8 us
// at 16 columns, 8.2 at 384.)
template <int PARTS, int KG, int WAVES, int RR, int LL, int DR, bool MACRO, int SPLIT>
__global__ void __launch_bounds__(WAVES * 64) k_rom_resident(RomArgs a) {
  constexpr int K = 32 * KG, TILES = 2 * KG, OWN = TILES / SPLIT, TPW = OWN / WAVES;
  static_assert(TILES % (SPLIT * WAVES) == 0, "whole row tiles per wave");
  using P = Place<KG, RR, LL, DR>;
  constexpr int S = P::S, NR = S < DR ? S : DR;  // ring slots in use
  using Item = typename Prec<PARTS>::Item;
  using Acc = typename Prec<PARTS>::Acc;
  extern __shared__ double sm[];
  int4v* Sv = reinterpret_cast<int4v*>(sm);
  int4v* Ss = Sv + 4 * K;
  constexpr int lo = 2 * K;
  int4v* Al = Ss + 4 * K;  // [operator][own tile][LL][part][lane]
  // the workgroups of a tile are eight apart: on one XCD, in whose L2 they share
  // what still streams of the operators, where workgroups go round the eight
  const int tile = SPLIT == 1 ? (int)blockIdx.x : (int)(blockIdx.x / (8 * SPLIT) * 8 + blockIdx.x % 8);
  const int part = SPLIT == 1 ? 0 : (int)(blockIdx.x / 8 % SPLIT);
  if (SPLIT > 1 && tile >= (int)a.tiles) return;
  if (SPLIT == 1 && a.repeat && !repeats(a, blockIdx.x)) return;
  const int slot0 = tile * kTileCols;
  const int tid = threadIdx.x, lane = tid % 64, col = lane % 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  int rt[TPW];  // this wave's row tiles, the same of both operators
#pragma unroll
  for (int t = 0; t < TPW; ++t) rt[t] = part * OWN + wave + t * WAVES;
  const uint64_t colQ = (uint64_t)(slot0 + col) * K;
  double qv[TPW][4], qs[TPW][4], bv[TPW][4];
#pragma unroll
  for (int t = 0; t < TPW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      bv[t][r] = a.b[colQ + rt[t] * 16 + rowBf16(lane, r)];
      qv[t][r] = a.qv[colQ + rt[t] * 16 + rowBf16(lane, r)];
      qs[t][r] = a.qs[colQ + rt[t] * 16 + rowBf16(lane, r)];
    }
  if constexpr (SPLIT == 1) {
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      writeSplitRowsHw(Sv, lo, rt[t], lane, qv[t]);
      writeSplitRowsHw(Ss, lo, rt[t], lane, qs[t]);
    }
  } else {
#pragma nounroll
    for (int x = wave; x < TILES; x += WAVES) {
      double v[4], s[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = a.qv[colQ + x * 16 + rowBf16(lane, r)];
        s[r] = a.qs[colQ + x * 16 + rowBf16(lane, r)];
      }
      writeSplitRowsHw(Sv, lo, x, lane, v);
      writeSplitRowsHw(Ss, lo, x, lane, s);
    }
  }
  const uint32_t s0 = (uint32_t)a.stepCol[slot0 + col];
  const uint32_t hz = (uint32_t)a.horizon[slot0 + col];
  const uint32_t ev = (uint32_t)a.every[slot0 + col];
  const double* fcol = a.ftab + (uint64_t)(slot0 + col) * a.maxSteps;
  uint32_t span = hz > s0 ? hz - s0 : 0;  // steps to the tile's last horizon
#pragma unroll
  for (int off = 32; off >= 1; off /= 2) {
    const uint32_t o = (uint32_t)__shfl_xor((int)span, off);
    span = o > span ? o : span;
  }
  uint32_t steps = (uint64_t)span > a.nsteps ? (uint32_t)a.nsteps : span;
  uint32_t mk = 0, mk2 = 0;  // mk one-steps, mk2 macro steps, then one-steps to the end
  if constexpr (MACRO) launchPlan(a, s0, hz, ev, a.quiet[slot0 + col], span, steps, mk, mk2);
  steps = (uint32_t)__builtin_amdgcn_readfirstlane((int)steps);

  // Item of group g of row tile t (of this wave) of an operator: a scalar base
  // and a lane offset. The bases are opaque where their loads belong (inside
  // the step loop for the streamed groups): the loads are loop invariants
  // that the compiler would otherwise keep in registers it does not have.
  const uint32_t laneOff = (uint32_t)lane * sizeof(Item);
  auto at = [&](const char* op, int t, int g) -> const Item& {
    return *reinterpret_cast<const Item*>(op + ((size_t)rt[t] * KG + g) * 64 * sizeof(Item) + laneOff);
  };
  auto opaque = [](const void* x) {
    const char* y = static_cast<const char*>(x);
    asm volatile("" : "+s"(y));
    return y;
  };
  const char* A[2];
  Item res[2][TPW][RR > 0 ? RR : 1], ring[NR > 0 ? NR : 1][TPW];
  Acc acc[TPW];
  // acc = (operator op) X; the ring holds the first NR streamed groups of op on
  // entry and of the other operator at the end
  auto products = [&](auto opc, const int4v* X) {
    constexpr int op = decltype(opc)::value;
#pragma unroll
    for (int t = 0; t < TPW; ++t) acc[t] = Acc{0, 0, 0, 0};
    // the state's operands are read two groups ahead
    const int4v* Xl = X + (lane / 16) * kTileCols + col;
    int4v xb[3][2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      xb[g][0] = Xl[4 * g * kTileCols];
      xb[g][1] = Xl[lo + 4 * g * kTileCols];
    }
#pragma unroll
    for (int g = 0; g < KG; ++g) {
      if (g + 2 < KG) {
        xb[(g + 2) % 3][0] = Xl[4 * (g + 2) * kTileCols];
        xb[(g + 2) % 3][1] = Xl[lo + 4 * (g + 2) * kTileCols];
      }
      __builtin_amdgcn_sched_barrier(0);
      const int4v xh = xb[g % 3][0], xl = xb[g % 3][1];
      const bool str = P::streamed(g);
      const int n = P::index(g);
      Item it[TPW];
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        if (str) {
          it[t] = ring[n % (NR > 0 ? NR : 1)][t];
        } else if (n < LL) {
#pragma unroll
          for (int p = 0; p < PARTS; ++p) it[t].p[p] = Al[(((op * OWN + wave + t * WAVES) * LL + n) * PARTS + p) * 64 + lane];
        } else {
          it[t] = res[op][t][n >= LL ? n - LL : 0];
        }
      }
      // the row tiles take turns, so that consecutive MFMAs are independent
#pragma unroll
      for (int t = 0; t < TPW; ++t) acc[t] = mfmaBf16x32(it[t].p[0], xh, acc[t]);
#pragma unroll
      for (int t = 0; t < TPW; ++t) acc[t] = mfmaBf16x32(it[t].p[0], xl, acc[t]);
#pragma unroll
      for (int t = 0; t < TPW; ++t) acc[t] = mfmaBf16x32(it[t].p[1], xh, acc[t]);
      if constexpr (PARTS == 3)
#pragma unroll
        for (int t = 0; t < TPW; ++t) acc[t] = mfmaBf16x32(it[t].p[2], xh, acc[t]);
      if (str) {
#pragma unroll
        for (int t = 0; t < TPW; ++t)
          ring[n % (NR > 0 ? NR : 1)][t] =
              n + NR < S ? at(A[op], t, P::group(n + NR < S ? n + NR : 0))
                         : at(A[1 - op], t, P::group(n % (NR > 0 ? NR : 1)));
        __builtin_amdgcn_sched_barrier(0);  // the refill leaves here, not at the end of the products
      }
    }
  };
  // fills the registers, LDS and ring (every wave reads back only what it wrote)
  auto loadOperators = [&] {
    A[0] = opaque(a.av);
    A[1] = opaque(a.as);
#pragma unroll
    for (int op = 0; op < 2; ++op)
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int g = 0; g < KG; ++g) {
          const int n = P::index(g);
          if (P::streamed(g)) {
            if (op == 0 && n < NR) ring[n < NR ? n : 0][t] = at(A[0], t, g);
          } else if (n < LL) {
            const Item it = at(A[op], t, g);
#pragma unroll
            for (int p = 0; p < PARTS; ++p) Al[(((op * OWN + wave + t * WAVES) * LL + n) * PARTS + p) * 64 + lane] = it.p[p];
          } else {
            res[op][t][n >= LL ? n - LL : 0] = at(A[op], t, g);
          }
        }
  };
  // SPLIT > 1: an exchange moves a split (or both) from the tile's waves to all
  // its workgroups
  uint64_t* const xbuf = a.xbuf + (uint64_t)tile * kXbufs * 2 * 8 * K;  // [buffer][dof][8 K]
  int cur = 0, old = kXbufs - 1;  // buffers of this exchange and the one before
  // the group did not meet; the exchange before moved both dofs; a word never came
  bool missed = false, both = false, lost = a.noWords != 0;
  // place of this lane's rows of tile t among the words of a buffer's dof
  auto word = [&](int t) { return 2 * ((4 * (rt[t] / 2) + lane / 16) * kTileCols + col) + rt[t] % 2; };
  auto publish = [&](int dof, double (&q)[TPW][4]) {
    uint64_t* x = xbuf + (cur * 2 + dof) * 8 * K;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      u2 hl[2];
      splitRowsHw(q[t], hl[0], hl[1]);
#pragma unroll
      for (int p = 0; p < 2; ++p)
        putWord(x + p * 2 * lo + word(t), __builtin_bit_cast(uint64_t, hl[p]));
    }
  };
  auto empty = [&](int buf, int dof) {
    uint64_t* x = xbuf + (buf * 2 + dof) * 8 * K;
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int p = 0; p < 2; ++p) put(x + p * 2 * lo + word(t), kEmpty);
  };
  auto collect = [&](int dof, int4v* S) {
    static_assert(8 * K % (64 * WAVES) == 0, "whole rounds");
    collectWords<8 * K / (64 * WAVES), 64 * WAVES>(xbuf + (cur * 2 + dof) * 8 * K + tid, reinterpret_cast<uint64_t*>(S) + tid,
                                                   lost);
  };
  auto turn = [&] {
    old = cur;
    cur = cur + 1 == kXbufs ? 0 : cur + 1;
  };
  if (SPLIT > 1 && steps) {
    for (int x = 0; x < kXbufs; ++x) {
      empty(x, 0);
      empty(x, 1);
    }
    // not met: nothing is changed, a repeating launch runs the tile. (Eight waves
    // without macro steps skip all steps instead of returning here, which spills
    // two more registers: BF16x4 K = 384, 1024 columns 6.5 us a step against 7.0;
    // the others are faster so: K = 512, 512 columns 6.0 against 6.7)
    if (!joinGroup(a, tile, SPLIT * WAVES, lane)) {
      if constexpr (WAVES < 8 || MACRO) return;
      missed = true;
      steps = mk2 = 0;
    }
  }
  // the new split of a dof to every wave that reads it
  auto share = [&](int dof, double (&q)[TPW][4], int4v* S) {
    if constexpr (SPLIT == 1) {
#pragma unroll
      for (int t = 0; t < TPW; ++t) writeSplitRowsHw(S, lo, rt[t], lane, q[t]);
    } else {
      written();
      publish(dof, q);
      collect(dof, S);
    }
    __syncthreads();
    if constexpr (SPLIT > 1) {
      empty(old, 1 - dof);
      if (both) empty(old, dof);
      both = false;
      turn();
    }
  };
  constexpr int RW = SPLIT * WAVES;  // waves that take the receivers' row tiles
#pragma nounroll
  for (int seg = 0; seg < (MACRO ? 2 : 1); ++seg) {
    const uint32_t from = seg == 0 ? 0u : mk + a.macro * mk2;
    const uint32_t to = seg == 0 ? (mk2 ? mk : steps) : (mk2 ? steps : 0u);
    if (from < to) {
      loadOperators();
      __syncthreads();  // both splits are in LDS
      const uint32_t sf = s0 + from;
      // forcing of four steps at a time, step j of them in lanes 16 j .. 16 j + 15
      // (one column each), the next four loaded during these: a step does not
      // wait for memory
      auto forcing = [&](uint32_t s) { return s + lane / 16 < hz ? fcol[s + lane / 16] : 0.0; };
      double f4 = forcing(sf), f4next = f4;
      uint32_t phase = ev ? (sf + 1) % ev : 0;
      uint32_t nextIdx = ev ? (sf + 1) / ev : 0;
      for (uint32_t it = from; it < to; ++it) {
        A[0] = opaque(a.av);
        A[1] = opaque(a.as);
        const uint32_t s = s0 + it;
        const bool act = s < hz;
        const uint32_t j = (it - from) % 4;
        if (j == 0) {
          f4 = f4next;
          f4next = forcing(s + 4);
        }
        const double fdt = __shfl(f4, (int)(16 * j) + col) * a.dt;  // (0 past the horizon)
        const bool smp = act && ev > 0 && phase == 0;
        const bool anySample = (__ballot(smp) & 0xffffull) != 0;
        // velocity: q_v += dt Ar_v q_s ; q_v += (f dt) b
        products(std::integral_constant<int, 0>{}, Ss);
        // (selects, kept from becoming branches: the tiles' updates are one
        // block of independent chains)
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const double y = qv[t][r] + a.dt * (double)acc[t][r];
            double z = y + fdt * bv[t][r];
            asm("" : "+v"(z));
            qv[t][r] = act ? z : qv[t][r];
          }
        share(0, qv, Sv);
        // stress: q_s += dt Ar_s q_v
        products(std::integral_constant<int, 1>{}, Sv);
        if (anySample) receivers<PARTS, 1, RW, 2>(a, Sv, lo, part * WAVES + wave, lane, smp, nextIdx - 1, slot0);
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            double z = qs[t][r] + a.dt * (double)acc[t][r];
            asm("" : "+v"(z));
            qs[t][r] = act ? z : qs[t][r];
          }
        share(1, qs, Ss);
        if (ev && act) {
          phase = phase + 1 == ev ? 0 : phase + 1;
          if (phase == 0) ++nextIdx;
        }
      }
    }
    if constexpr (MACRO) {
      if (seg == 0 && mk2) {
        // macro steps: the blocks of G stream from L2 through a two-deep
        // ring, which starts on the next block while one ends. At 256 modes groups
        // that are all padding are left out: unequal dofs pad alike (256 and 128
        // modes, 1024 columns: BF16x3 8.1 -> 6.3 us a macro step, BF16x4 11.4 ->
        // 9.1; kernels of the dofs' own sizes take 6.6 and 9.1). In a loop, which
        // costs equal dofs 2 %; smaller and shared ones are faster without
        const bool act = s0 + mk < hz;
        Item mring[2][TPW];
        auto stream = [&](auto zero, const char* G, uint32_t groups, const char* next, const int4v* X) {
          if constexpr (decltype(zero)::value)
#pragma unroll
            for (int t = 0; t < TPW; ++t) acc[t] = Acc{0, 0, 0, 0};
          if (KG == 8 && groups < KG) {
#pragma nounroll
            for (uint32_t g = 0; g < groups; g += 2) {
              const char* src = g + 2 < groups ? G + (size_t)(g + 2) * 64 * sizeof(Item) : next;
#pragma unroll
              for (int q = 0; q < 2; ++q) {
                groupProducts<PARTS, TPW>(mring[q], (int)g + q, X, lo, lane, acc);
#pragma unroll
                for (int t = 0; t < TPW; ++t) mring[q][t] = at(src, t, q);
                __builtin_amdgcn_sched_barrier(0);
              }
            }
            return;
          }
#pragma unroll
          for (int g = 0; g < KG; ++g) {
            groupProducts<PARTS, TPW>(mring[g % 2], g, X, lo, lane, acc);
#pragma unroll
            for (int t = 0; t < TPW; ++t) mring[g % 2][t] = g + 2 < KG ? at(G, t, g + 2) : at(next, t, g + 2 - KG);
            __builtin_amdgcn_sched_barrier(0);
          }
        };
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int t = 0; t < TPW; ++t) mring[g][t] = at(opaque(a.gvv), t, g);
        __syncthreads();  // both splits are in LDS
        for (uint32_t it = 0; it < mk2; ++it) {
          const char *gvv = opaque(a.gvv), *gvs = opaque(a.gvs), *gsv = opaque(a.gsv), *gss = opaque(a.gss);
          stream(std::true_type{}, gvv, a.groupsV, gvs, Sv);
          stream(std::false_type{}, gvs, a.groupsS, gsv, Ss);
          if (act)
#pragma unroll
            for (int t = 0; t < TPW; ++t)
#pragma unroll
              for (int r = 0; r < 4; ++r) qv[t][r] = qv[t][r] + a.dt * (double)acc[t][r];
          stream(std::true_type{}, gsv, a.groupsV, gss, Sv);
          stream(std::false_type{}, gss, a.groupsS, gvv, Ss);
          if (act)
#pragma unroll
            for (int t = 0; t < TPW; ++t)
#pragma unroll
              for (int r = 0; r < 4; ++r) qs[t][r] = qs[t][r] + a.dt * (double)acc[t][r];
          if constexpr (SPLIT == 1) {
            __syncthreads();  // every read of the old splits done
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
              writeSplitRowsHw(Sv, lo, rt[t], lane, qv[t]);
              writeSplitRowsHw(Ss, lo, rt[t], lane, qs[t]);
            }
          } else {
            written();
            publish(0, qv);
            publish(1, qs);
            __syncthreads();  // every read of the old splits done
            collect(0, Sv);
            collect(1, Ss);
          }
          __syncthreads();  // the new splits complete
          if constexpr (SPLIT > 1) {
            empty(old, 0);
            empty(old, 1);
            both = true;
            turn();
          }
          // the macro step's last step is sampled when it ends at a multiple of the period
          const uint64_t sn = (uint64_t)s0 + mk + (uint64_t)(it + 1) * a.macro;
          const bool smp = act && ev > 0 && sn % ev == 0;
          if ((__ballot(smp) & 0xffffull) != 0)
            receivers<PARTS, 1, RW, 2>(a, Sv, lo, part * WAVES + wave, lane, smp, smp ? (uint32_t)(sn / ev - 1) : 0u, slot0);
        }
        __syncthreads();  // the next one-steps write the split the receivers read
      }
    }
  }
#pragma unroll
  for (int t = 0; t < TPW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      a.qv[colQ + rt[t] * 16 + rowBf16(lane, r)] = qv[t][r];
      a.qs[colQ + rt[t] * 16 + rowBf16(lane, r)] = qs[t][r];
    }
  if (SPLIT > 1 && missed) return;  // (the states are as they were read)
  if constexpr (SPLIT > 1) reportLost(lost, lane);
  // (no workgroup of the tile is still to read its counters or states: a tile
  // with steps has had an exchange, one without writes what it read)
  if (part == 0 && tid < kTileCols) {
    // a.nsteps steps, or fewer when every column reached its horizon (the
    // same counts), or more under a time budget
    const uint64_t h = a.horizon[slot0 + tid];
    const uint64_t st = a.stepCol[slot0 + tid], s = st + (MACRO ? (uint64_t)steps : a.nsteps);
    a.stepCol[slot0 + tid] = s < h ? s : (st < h ? h : st);
  }
}

template <int PARTS, int KG, int WAVES, int RR, int LL, int DR, int SPLIT = 1>
bool launchKG(RomArgs a, uint32_t tiles, hipStream_t stream) {
  constexpr size_t lds = (8 * 32 * KG + (size_t)2 * (2 * KG / SPLIT) * LL * PARTS * 64) * 16;
  static_assert(lds <= 160 * 1024, "LDS of one CU");
  auto go = [&](auto kernel) {
    SHAW_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    if constexpr (SPLIT == 1) {
      hipLaunchKernelGGL(kernel, dim3(tiles), dim3(WAVES * 64), lds, stream, a);
      return true;
    } else {
      return launchCooperative((const void*)kernel, (tiles + 7) / 8 * 8 * SPLIT, WAVES * 64, lds, a, stream);
    }
  };
  return a.macro ? go(k_rom_resident<PARTS, KG, WAVES, RR, LL, DR, true, SPLIT>)
                 : go(k_rom_resident<PARTS, KG, WAVES, RR, LL, DR, false, SPLIT>);
}

}  // namespace

bool launchCooperative(const void* kernel, unsigned groups, unsigned threads, size_t lds, const RomArgs& a, hipStream_t stream) {
  RomArgs copy = a;
  void* args[] = {&copy};
  const hipError_t e = hipLaunchCooperativeKernel(kernel, dim3(groups), dim3(threads), args, (unsigned)lds, stream);
  if (e == hipErrorCooperativeLaunchTooLarge) (void)hipGetLastError();
  else SHAW_HIP(e);
  return e == hipSuccess;
}

// BF16, the workgroups of a tile of 16 columns (1: one): four row tiles each, or
// eight, while the chip holds all workgroups at once, one to a CU. Not up to 256
// modes: BF16x4 4.5 us a step in one workgroup, 4.2 in four, which a cooperative
// launch of a few steps takes back; BF16x3 2.7, two exchanges 2.8. FP64, those of
// one set of four columns or, above 256 modes, of two, four row tiles each.
uint32_t residentSplit(int parts, uint32_t modes, uint64_t tiles, int cus, uint32_t& sets) {
  sets = 1;
  const uint32_t most = modes / 64;
  auto fits = [&](uint64_t groups, uint32_t split) { return (groups + 7) / 8 * 8 * split <= (uint64_t)cus; };
  if (parts == 0) {
    if (modes < 256) return 1;
    if (fits(4 * tiles, most)) return most;
    if (modes == 256 || !fits(2 * tiles, most)) return 1;
    sets = 2;
    return most;
  }
  if (modes < 384) return 1;
  for (const uint32_t split : {most, most / 2})
    if (fits(tiles, split)) return split;
  return 1;
}
// A cooperative launch and its first meeting cost about what three unshared steps
// do (1280 columns of K = 384 BF16x3, launches in a row: 4 steps 59 us against 57,
// 2 steps 48 against 37), about what nine do at 256 modes FP64 (4 steps 41 us
// against 34, 16 steps 87 against 110). Unshared steps of dofs so unequal that the
// square pad costs more than it saves are dearer (64 columns, FP64 512 and 64
// modes: 28.9 us each and a shared launch of one 41; 384: 14.9 and 39 of two; 256:
// 6.2 and 43 of four; BF16x4 512 and 64: 21 and 43 of two, but with half as many
// workgroups a tile on a fuller chip 27 and 76).
uint64_t shareFrom(int parts, uint64_t kv, uint64_t ks, uint32_t modes, uint32_t split) {
  const uint64_t lo = kv < ks ? kv : ks, hi = kv < ks ? ks : kv;
  if (parts) return split == modes / 64 && (hi + 127) / 128 > (lo + 127) / 128 + 1 ? 2 : 4;
  if (lo <= 64) return hi <= 256 ? 5 : hi <= 384 ? 2 : 1;
  return hi <= 256 ? 10 : 4;
}
uint64_t residentExchange(uint32_t modes, uint64_t tiles) { return tiles * kXbufs * 2 * 8 * modes; }

// FP64, padded dofs lo <= hi: up to how many rounds of workgroups of four columns
// (64 tiles of 16 columns each, all CUs) the square product in k_rom_f64 is
// faster than k_rom_steps, which computes the dofs as they are, 16 columns a
// workgroup. A round against k_rom_steps, us: hi = 128: 1.6 against 3.7 (lo = 64);
// 192: 3.8 against 5.0 (64), 8.4 (128); 256: 7.1 against 6.0 (64), 10.2 (128),
// 14.1 (192); 384 18 against 14.6 (64), 26.6 (128), 35.1 (320), of 320 modes 13.2
// (64), 26.6 (192), 32.4 (320), and two rounds 35.4 against 38.2 (384 both); 512
// 34 against 23.1 (64), 42.3 (128), of 448 modes 21.1 (64), 38.6 (128). Equal dofs
// of up to 256 modes pad alike either way: romF64Fits chooses for each launch.
static uint64_t squareRounds(uint32_t lo, uint32_t hi) {
  if (lo == hi && hi <= 256) return ~0ull;
  if (hi == 128) return 2;
  if (lo == 64) return hi == 192 ? 1 : 0;
  return hi == 192 || (lo == 384 && hi == 384) ? 2 : 1;
}

uint32_t residentModes(int parts, uint64_t kv, uint64_t ks, uint64_t cols, int cus) {
  const uint64_t k = kv > ks ? kv : ks, tiles = (cols + kTileCols - 1) / kTileCols;
  const uint32_t modes = k <= 256 ? (uint32_t)((k + 63) / 64 * 64) : k <= 384 ? 384 : 512;
  uint32_t sets;
  const bool shared = residentSplit(parts, modes, tiles, cus, sets) > 1;
  const uint32_t lo = (uint32_t)(((kv < ks ? kv : ks) + 63) / 64 * 64), hi = (uint32_t)((k + 63) / 64 * 64);
  // BF16 above 256 modes: one workgroup a tile streams nearly all of the
  // operators, and a square pad of unequal dofs would add to it; shared tiles of
  // 512 modes nearly fill the chip from 57 on (BF16x3 960 columns 11.5 us a step,
  // of dofs of 512 and 128 modes 11.4 in one workgroup a tile; 896 columns 10.3)
  if (parts == 2 && modes == 512 && lo <= 128 && tiles > 56) return 0;
  if (parts) return k <= 256 || shared || (kv + 127) / 128 == (ks + 127) / 128 ? modes : 0;
  return shared || (tiles + 63) / 64 <= squareRounds(lo, hi) ? modes : 0;
}

bool launchRomResident(int parts, const RomArgs& a, uint32_t split, hipStream_t stream) {
  const int kg = (int)a.Kvp / 32;
  const uint32_t grid = a.tiles;
  auto shared = [&] {
    if (parts == 2) {
      if (kg == 12) return split == 6 ? launchKG<2, 12, 4, 8, 4, 1, 6>(a, grid, stream) : launchKG<2, 12, 8, 9, 3, 1, 3>(a, grid, stream);
      return split == 8 ? launchKG<2, 16, 4, 10, 6, 1, 8>(a, grid, stream) : launchKG<2, 16, 8, 9, 3, 1, 4>(a, grid, stream);
    }
    if (kg == 12) return split == 6 ? launchKG<3, 12, 4, 8, 4, 1, 6>(a, grid, stream) : launchKG<3, 12, 8, 6, 2, 1, 3>(a, grid, stream);
    return split == 8 ? launchKG<3, 16, 4, 12, 4, 1, 8>(a, grid, stream) : launchKG<3, 16, 8, 6, 2, 1, 4>(a, grid, stream);
  };
  if (split > 1 && shared()) return true;
  if (parts == 2) {
    switch (kg) {
      case 2: launchKG<2, 2, 4, 2, 0, 1>(a, grid, stream); break;
      case 4: launchKG<2, 4, 8, 4, 0, 1>(a, grid, stream); break;
      case 6: launchKG<2, 6, 12, 5, 1, 1>(a, grid, stream); break;
      case 8: launchKG<2, 8, 8, 3, 2, 1>(a, grid, stream); break;
      case 12: launchKG<2, 12, 8, 1, 1, 1>(a, grid, stream); break;
      default: launchKG<2, 16, 8, 0, 0, 1>(a, grid, stream); break;
    }
  } else {
    switch (kg) {
      case 2: launchKG<3, 2, 4, 2, 0, 1>(a, grid, stream); break;
      case 4: launchKG<3, 4, 8, 4, 0, 1>(a, grid, stream); break;
      case 6: launchKG<3, 6, 12, 2, 1, 1>(a, grid, stream); break;
      case 8: launchKG<3, 8, 8, 2, 1, 1>(a, grid, stream); break;
      case 12: launchKG<3, 12, 8, 0, 0, 2>(a, grid, stream); break;
      default: launchKG<3, 16, 8, 0, 0, 1>(a, grid, stream); break;
    }
  }
  return false;
}

}  // namespace shaw
