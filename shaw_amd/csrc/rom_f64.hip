// The FP64 reduced leapfrog in workgroups of four column slots, the operators
// on the CU as far as they fit.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rom_device.hpp"
#include "rom_internal.hpp"
#include "shaw_common.hpp"

namespace shaw {
namespace {

constexpr int kCols = 4;  // column slots per workgroup

// v_mfma_f64_4x4x4_4b_f64: four 4 x 4 blocks, K = 4. With A as the
// 16 x 16 x 4 form holds it (lane l: A[l % 16][l / 16]) and the same four columns
// of B in every block (lane l: B[l / 16][l % 4]) the blocks are the four row
// quarters of one row tile: D: lane l holds D[4 * (l / 4 % 4) + l / 16][l % 4].
// Both forms add a product's terms in k order with one rounding each, so a
// column's values do not depend on the form (tests/test_gpu_rom_f64.py).
__device__ __forceinline__ double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// Both operators are G row tiles by G k-groups (16 modes each). Per row tile RR
// groups sit in registers, LL in LDS, the rest stream from L2 through a ring of
// DR groups, spread evenly among the resident ones (as in rom_resident.hip).
//
// k_rom_steps gives a workgroup 16 columns, so 1024 columns are 64 workgroups
// on 256 CUs, and a CU's FP64 MFMA rate sets the step (K = 256: 13.7 us of
// products, 18 us measured). The 4 x 4 x 4 form has the same rate at a quarter
// of the columns: four times the workgroups, each a quarter of the time, and
// the operators re-read from L2 only where they do not fit the CU. Bound by
// the chain of a half-step at K = 64, by MFMA and the state's LDS reads to 192,
// by the streamed groups from 256 on (a CU reads 126 GB/s when all stream).
// Per step at 1024 columns, k_rom_steps -> k_rom_f64: K = 64 2.44 -> 0.66 us,
// 128 5.90 -> 1.59, 192 11.1 -> 3.7, 256 17.9 -> 7.7, 384 38.0 -> 18.3, 512
// 65.6 -> 34.5. (Waves and places are the fastest of those tried: at K = 256
// one row tile a wave 8.8 us, four 8.3, a ring of four 8.0.)
template <int G, int WAVES, int RR, int LL, int DR>
__global__ void __launch_bounds__(WAVES * 64) k_rom_f64(RomArgs a) {
  constexpr int K = 16 * G, TPW = G / WAVES;
  static_assert(G % WAVES == 0, "whole row tiles per wave");
  using P = Place<G, RR, LL, DR>;
  constexpr int S = P::S, NR = S < DR ? S : DR;
  constexpr int RS = NR > 0 ? NR : 1;
  extern __shared__ double sm[];
  double* Xv = sm;           // [K][4] q_v
  double* Xs = Xv + K * kCols;
  dbl4* Al = reinterpret_cast<dbl4*>(Xs + K * kCols);  // [operator][tile][LL][lane]
  if (a.repeat && !repeats(a, blockIdx.x)) return;
  const int slot0 = blockIdx.x * kCols;
  const int tid = threadIdx.x, lane = tid % 64, col = lane % kCols;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const uint32_t s0 = (uint32_t)a.stepCol[slot0 + col];
  const uint32_t hz = (uint32_t)a.horizon[slot0 + col];
  const uint32_t ev = (uint32_t)a.every[slot0 + col];
  uint32_t steps = hz > s0 ? hz - s0 : 0;  // to the last horizon of the workgroup
#pragma unroll
  for (int off = 2; off >= 1; off /= 2) {
    const uint32_t o = (uint32_t)__shfl_xor((int)steps, off);
    steps = o > steps ? o : steps;
  }
  if ((uint64_t)steps > a.nsteps) steps = (uint32_t)a.nsteps;
  steps = (uint32_t)__builtin_amdgcn_readfirstlane((int)steps);
  if (steps == 0) return;  // no active column: states and counters stay

  const int row = 4 * (lane / 4 % 4) + lane / 16;  // of this lane in a row tile
  int rt[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) rt[t] = wave + t * WAVES;
  const uint64_t colQ = (uint64_t)(slot0 + col) * K;
  double qv[TPW], qs[TPW], bv[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const int m = rt[t] * 16 + row;
    qv[t] = a.qv[colQ + m];
    qs[t] = a.qs[colQ + m];
    bv[t] = a.b[colQ + m];
    Xv[m * kCols + col] = qv[t];
    Xs[m * kCols + col] = qs[t];
  }
  // item of group g of row tile t of an operator: a scalar base, opaque where
  // its loads belong, and a lane offset (see rom_resident.hip)
  const uint32_t laneOff = (uint32_t)lane * sizeof(dbl4);
  auto at = [&](const char* op, int t, int g) -> const dbl4& {
    return *reinterpret_cast<const dbl4*>(op + ((size_t)rt[t] * G + g) * 64 * sizeof(dbl4) + laneOff);
  };
  auto opaque = [](const void* x) {
    const char* y = static_cast<const char*>(x);
    asm volatile("" : "+s"(y));
    return y;
  };
  const char* A[2] = {opaque(a.av), opaque(a.as)};
  dbl4 res[2][TPW][RR > 0 ? RR : 1], ring[RS][TPW];
#pragma unroll
  for (int op = 0; op < 2; ++op)
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int n = P::index(g);
        if (P::streamed(g)) {
          if (op == 0 && n < NR) ring[n < NR ? n : 0][t] = at(A[0], t, g);
        } else if (n < LL) {
          Al[((op * G + rt[t]) * LL + n) * 64 + lane] = at(A[op], t, g);
        } else {
          res[op][t][n >= LL ? n - LL : 0] = at(A[op], t, g);
        }
      }
  double acc[TPW];
  const int xOff = (lane / 16) * kCols + col;
  // acc = (operator op) X; the ring holds the first streamed groups of op on
  // entry and of the other operator at the end
  auto products = [&](auto opc, const double* X) {
    constexpr int op = decltype(opc)::value;
    const double* Xl = X + xOff;
#pragma unroll
    for (int t = 0; t < TPW; ++t) acc[t] = 0.0;
    double xb[2][4];  // the state's operands, read one group ahead
#pragma unroll
    for (int s = 0; s < 4; ++s) xb[0][s] = Xl[4 * s * kCols];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g + 1 < G)
#pragma unroll
        for (int s = 0; s < 4; ++s) xb[(g + 1) % 2][s] = Xl[(16 * (g + 1) + 4 * s) * kCols];
      const bool str = P::streamed(g);
      const int n = P::index(g);
      dbl4 it[TPW];
#pragma unroll
      for (int t = 0; t < TPW; ++t)
        it[t] = str ? ring[n % RS][t]
                    : (n < LL ? Al[((op * G + rt[t]) * LL + (n < LL ? n : 0)) * 64 + lane] : res[op][t][n >= LL ? n - LL : 0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < TPW; ++t) acc[t] = mfma4(it[t][s], xb[g % 2][s], acc[t]);
      if (str)
#pragma unroll
        for (int t = 0; t < TPW; ++t)
          ring[n % RS][t] = n + NR < S ? at(A[op], t, P::group(n + NR < S ? n + NR : 0)) : at(A[1 - op], t, P::group(n % RS));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const double* fcol = a.ftab + (uint64_t)(slot0 + col) * a.maxSteps;
  // forcing of four steps at a time, step j of them in lanes 16 j .. 16 j + 15,
  // the next four loaded during these
  auto forcing = [&](uint32_t s) { return s + lane / 16 < hz ? fcol[s + lane / 16] : 0.0; };
  double f4 = forcing(s0), f4next = f4;
  uint32_t phase = ev ? (s0 + 1) % ev : 0;    // (s + 1) mod every
  uint32_t nextIdx = ev ? (s0 + 1) / ev : 0;  // index of the next sample
  __syncthreads();  // the states are in LDS
  for (uint32_t it = 0; it < steps; ++it) {
    A[0] = opaque(a.av);
    A[1] = opaque(a.as);
    const uint32_t s = s0 + it;
    const bool act = s < hz;
    const uint32_t j = it % 4;
    if (j == 0) {
      f4 = f4next;
      f4next = forcing(s + 4);
    }
    const double fdt = __shfl(f4, (int)(16 * j) + col) * a.dt;  // (0 past the horizon)
    const bool smp = act && ev > 0 && phase == 0;
    const bool anySample = (__ballot(smp) & 0xfull) != 0;
    // velocity: q_v += dt Ar_v q_s ; q_v += (f dt) b
    products(std::integral_constant<int, 0>{}, Xs);
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const double y = qv[t] + a.dt * acc[t];
      double z = y + fdt * bv[t];
      asm("" : "+v"(z));
      qv[t] = act ? z : qv[t];
      Xv[(rt[t] * 16 + row) * kCols + col] = qv[t];
    }
    __syncthreads();
    // stress: q_s += dt Ar_s q_v
    products(std::integral_constant<int, 1>{}, Xv);
    if (anySample)
      for (int rc = wave; rc < (int)a.Rp / 16; rc += WAVES) {  // receivers: C q_v
        const dbl4* C = reinterpret_cast<const dbl4*>(a.c) + (size_t)rc * G * 64 + lane;
        double y = 0.0;
#pragma unroll 2  // (sample steps are rare: few registers)
        for (int g = 0; g < G; ++g) {
          const dbl4 ci = C[g * 64];
#pragma unroll
          for (int q = 0; q < 4; ++q) y = mfma4(ci[q], Xv[(16 * g + 4 * q) * kCols + xOff], y);
        }
        const uint32_t m = rc * 16 + row;
        if (smp && m < a.R)  // per slot LayoutLeft [R x Tcap]
          a.seis[(uint64_t)(slot0 + col) * a.R * a.Tcap + (uint64_t)a.R * (nextIdx - 1) + m] = y;
      }
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      double z = qs[t] + a.dt * acc[t];
      asm("" : "+v"(z));
      qs[t] = act ? z : qs[t];
      Xs[(rt[t] * 16 + row) * kCols + col] = qs[t];
    }
    __syncthreads();
    if (ev && act) {
      phase = phase + 1 == ev ? 0 : phase + 1;
      if (phase == 0) ++nextIdx;
    }
  }
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    a.qv[colQ + rt[t] * 16 + row] = qv[t];
    a.qs[colQ + rt[t] * 16 + row] = qs[t];
  }
  if (tid < kCols) {
    const uint64_t h = a.horizon[slot0 + tid];
    const uint64_t st = a.stepCol[slot0 + tid], s = st + a.nsteps;
    a.stepCol[slot0 + tid] = s < h ? s : (st < h ? h : st);
  }
}

// The same with SETS sets of four columns shared by SPLIT workgroups, each with 1 /
// SPLIT of the row tiles, so that the operators of few columns fit the CUs that
// those would leave idle and are read once for all sets. After a half-step each
// wave writes its rows to a.xbuf and its workgroup reads all rows back from
// there. Bound by that exchange (1.4 us) and the chain of 4 G products. Per step,
// k_rom_f64 -> this: K = 256 6.3 us -> 4.0 at 16 columns, 4.2 at 256; 384 15.4 ->
// 5.1 at 160, 8.3 at 320; 512 30.1 -> 7.6 at 128, 10.4 at 256. (Two sets of 256
// modes, half the row tiles each, 1024 columns: 9.2 us against 8.0; two sets by
// turns, one's exchange behind the other's products, 10.0.) A kernel of its own: as
// an instantiation of this body k_rom_f64 lost 3 to 8 % at K = 64.
template <int G, int WAVES, int RR, int LL, int DR, int SPLIT, int SETS>
__global__ void __launch_bounds__(WAVES * 64) k_rom_f64_shared(RomArgs a) {
  constexpr int K = 16 * G, OWN = G / SPLIT, TPW = OWN / WAVES;
  static_assert(G % (SPLIT * WAVES) == 0, "whole row tiles per wave");
  using P = Place<G, RR, LL, DR>;
  constexpr int S = P::S, NR = S < DR ? S : DR;
  constexpr int RS = NR > 0 ? NR : 1;
  extern __shared__ double sm[];
  dbl4* Al = reinterpret_cast<dbl4*>(sm + SETS * 2 * K * kCols);  // [operator][own tile][LL][lane]
  auto X = [&](int u, int dof) { return sm + (u * 2 + dof) * K * kCols; };  // [K][4] q_v or q_s of set u
  const int group = (int)(blockIdx.x / (8 * SPLIT) * 8 + blockIdx.x % 8), part = (int)(blockIdx.x / 8 % SPLIT);
  if (group >= (int)a.tiles * (kTileCols / (kCols * SETS))) return;
  const int slot0 = group * kCols * SETS;
  const int tid = threadIdx.x, lane = tid % 64, col = lane % kCols;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  uint32_t s0[SETS], hz[SETS], ev[SETS];
  uint32_t steps = 0;  // to the last horizon of the workgroup
#pragma unroll
  for (int u = 0; u < SETS; ++u) {
    const int slot = slot0 + u * kCols + col;
    s0[u] = (uint32_t)a.stepCol[slot];
    hz[u] = (uint32_t)a.horizon[slot];
    ev[u] = (uint32_t)a.every[slot];
    const uint32_t o = hz[u] > s0[u] ? hz[u] - s0[u] : 0;
    steps = o > steps ? o : steps;
  }
#pragma unroll
  for (int off = 2; off >= 1; off /= 2) {
    const uint32_t o = (uint32_t)__shfl_xor((int)steps, off);
    steps = o > steps ? o : steps;
  }
  if ((uint64_t)steps > a.nsteps) steps = (uint32_t)a.nsteps;
  steps = (uint32_t)__builtin_amdgcn_readfirstlane((int)steps);
  if (steps == 0) return;  // no active column: states and counters stay

  const int row = 4 * (lane / 4 % 4) + lane / 16;  // of this lane in a row tile
  int rt[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) rt[t] = part * OWN + wave + t * WAVES;
  double q[SETS][2][TPW], bv[SETS][TPW];  // q: [set][q_v, q_s]
#pragma unroll
  for (int u = 0; u < SETS; ++u) {
    const uint64_t colQ = (uint64_t)(slot0 + u * kCols + col) * K;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int m = rt[t] * 16 + row;
      q[u][0][t] = a.qv[colQ + m];
      q[u][1][t] = a.qs[colQ + m];
      bv[u][t] = a.b[colQ + m];
    }
#pragma nounroll
    for (int x = wave; x < G; x += WAVES) {
      const int m = x * 16 + row;
      X(u, 0)[m * kCols + col] = a.qv[colQ + m];
      X(u, 1)[m * kCols + col] = a.qs[colQ + m];
    }
  }
  // item of group g of row tile t of an operator: a scalar base, opaque where
  // its loads belong, and a lane offset (see rom_resident.hip)
  const uint32_t laneOff = (uint32_t)lane * sizeof(dbl4);
  auto at = [&](const char* op, int t, int g) -> const dbl4& {
    return *reinterpret_cast<const dbl4*>(op + ((size_t)rt[t] * G + g) * 64 * sizeof(dbl4) + laneOff);
  };
  auto opaque = [](const void* x) {
    const char* y = static_cast<const char*>(x);
    asm volatile("" : "+s"(y));
    return y;
  };
  const char* A[2] = {opaque(a.av), opaque(a.as)};
  dbl4 res[2][TPW][RR > 0 ? RR : 1], ring[RS][TPW];
#pragma unroll
  for (int op = 0; op < 2; ++op)
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int n = P::index(g);
        if (P::streamed(g)) {
          if (op == 0 && n < NR) ring[n < NR ? n : 0][t] = at(A[0], t, g);
        } else if (n < LL) {
          Al[((op * OWN + wave + t * WAVES) * LL + n) * 64 + lane] = at(A[op], t, g);
        } else {
          res[op][t][n >= LL ? n - LL : 0] = at(A[op], t, g);
        }
      }
  double acc[SETS][TPW];
  const int xOff = (lane / 16) * kCols + col;
  // acc[u] = (operator op) X(u, 1 - op); the ring holds the first streamed
  // groups of op on entry and of the other operator at the end
  auto products = [&](auto opc) {
    constexpr int op = decltype(opc)::value;
    double xb[2][SETS][4];  // the states' operands, read one group ahead
#pragma unroll
    for (int u = 0; u < SETS; ++u) {
#pragma unroll
      for (int t = 0; t < TPW; ++t) acc[u][t] = 0.0;
#pragma unroll
      for (int s = 0; s < 4; ++s) xb[0][u][s] = X(u, 1 - op)[xOff + 4 * s * kCols];
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g + 1 < G)
#pragma unroll
        for (int u = 0; u < SETS; ++u)
#pragma unroll
          for (int s = 0; s < 4; ++s) xb[(g + 1) % 2][u][s] = X(u, 1 - op)[xOff + (16 * (g + 1) + 4 * s) * kCols];
      const bool str = P::streamed(g);
      const int n = P::index(g);
      dbl4 it[TPW];
#pragma unroll
      for (int t = 0; t < TPW; ++t)
        it[t] = str ? ring[n % RS][t]
                    : (n < LL ? Al[((op * OWN + wave + t * WAVES) * LL + (n < LL ? n : 0)) * 64 + lane]
                              : res[op][t][n >= LL ? n - LL : 0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
          for (int u = 0; u < SETS; ++u) acc[u][t] = mfma4(it[t][s], xb[g % 2][u][s], acc[u][t]);
      if (str)
#pragma unroll
        for (int t = 0; t < TPW; ++t)
          ring[n % RS][t] = n + NR < S ? at(A[op], t, P::group(n + NR < S ? n + NR : 0)) : at(A[1 - op], t, P::group(n % RS));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // forcing of four steps at a time, step j of them in lanes 16 j .. 16 j + 15,
  // the next four loaded during these
  auto forcing = [&](int u, uint32_t s) {
    return s + lane / 16 < hz[u] ? a.ftab[(uint64_t)(slot0 + u * kCols + col) * a.maxSteps + s + lane / 16] : 0.0;
  };
  double f4[SETS], f4next[SETS];
  uint32_t phase[SETS], nextIdx[SETS];  // (s + 1) mod every; index of the next sample
#pragma unroll
  for (int u = 0; u < SETS; ++u) {
    f4[u] = forcing(u, s0[u]);
    asm volatile("" : "+v"(f4[u]));  // waits here, not in every step
    f4next[u] = 0.0;
    phase[u] = ev[u] ? (s0[u] + 1) % ev[u] : 0;
    nextIdx[u] = ev[u] ? (s0[u] + 1) / ev[u] : 0;
  }
  constexpr int RW = SPLIT * WAVES;  // waves that take the receivers' row tiles
  // exchanges of set u: half-steps 0 (q_v), 1 (q_s), 2, ... of the launch
  uint64_t* const xbuf = a.xbuf + (uint64_t)group * SETS * kXbufs * K * kCols;  // [set][buffer][K][4]
  int cur = 0, old = kXbufs - 1;  // buffers of this half-step and the one before
  bool lost = a.noWords != 0;
  auto buffer = [&](int u, int x) { return xbuf + (u * kXbufs + x) * K * kCols; };
  auto empty = [&](int u, int x) {
#pragma unroll
    for (int t = 0; t < TPW; ++t) put(buffer(u, x) + (rt[t] * 16 + row) * kCols + col, kEmpty);
  };
#pragma unroll
  for (int u = 0; u < SETS; ++u)
    for (int x = 0; x < kXbufs; ++x) empty(u, x);
  if (!joinGroup(a, group, RW, lane)) return;  // nothing is changed: a repeating launch runs the columns
  // the new rows of q_v or q_s to all that read them
  auto share = [&](auto dofc) {
    constexpr int dof = decltype(dofc)::value;
    written();
#pragma unroll
    for (int u = 0; u < SETS; ++u)
#pragma unroll
      for (int t = 0; t < TPW; ++t)
        putWord(buffer(u, cur) + (rt[t] * 16 + row) * kCols + col, __builtin_bit_cast(uint64_t, q[u][dof][t]));
    static_assert(K * kCols % (64 * WAVES) == 0, "whole rounds");
#pragma unroll
    for (int u = 0; u < SETS; ++u)
      collectWords<K * kCols / (64 * WAVES), 64 * WAVES>(buffer(u, cur) + tid, reinterpret_cast<uint64_t*>(X(u, dof)) + tid, lost);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < SETS; ++u) empty(u, old);
    old = cur;
    cur = cur + 1 == kXbufs ? 0 : cur + 1;
  };
  __syncthreads();  // the states are in LDS
  for (uint32_t it = 0; it < steps; ++it) {
    A[0] = opaque(a.av);
    A[1] = opaque(a.as);
    const uint32_t j = it % 4;
    double fdt[SETS];
    bool smp[SETS], anySample = false;
#pragma unroll
    for (int u = 0; u < SETS; ++u) {
      const uint32_t s = s0[u] + it;
      if (j == 0) {
        asm volatile("");
        f4next[u] = forcing(u, s + 4);
      }
      fdt[u] = __shfl(f4[u], (int)(16 * j) + col) * a.dt;  // (0 past the horizon)
      smp[u] = s < hz[u] && ev[u] > 0 && phase[u] == 0;
      anySample = anySample || (__ballot(smp[u]) & 0xfull) != 0;
    }
    // velocity: q_v += dt Ar_v q_s ; q_v += (f dt) b
    products(std::integral_constant<int, 0>{});
#pragma unroll
    for (int u = 0; u < SETS; ++u)
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        const double y = q[u][0][t] + a.dt * acc[u][t];
        double z = y + fdt[u] * bv[u][t];
        asm("" : "+v"(z));
        q[u][0][t] = s0[u] + it < hz[u] ? z : q[u][0][t];
      }
    share(std::integral_constant<int, 0>{});
    // stress: q_s += dt Ar_s q_v
    products(std::integral_constant<int, 1>{});
    if (anySample)
      for (int rc = part * WAVES + wave; rc < (int)a.Rp / 16; rc += RW) {  // receivers: C q_v
        const dbl4* C = reinterpret_cast<const dbl4*>(a.c) + (size_t)rc * G * 64 + lane;
#pragma unroll
        for (int u = 0; u < SETS; ++u) {
          double y = 0.0;
#pragma unroll 2  // (sample steps are rare: few registers)
          for (int g = 0; g < G; ++g) {
            const dbl4 ci = C[g * 64];
#pragma unroll
            for (int k = 0; k < 4; ++k) y = mfma4(ci[k], X(u, 0)[(16 * g + 4 * k) * kCols + xOff], y);
          }
          const uint32_t m = rc * 16 + row;
          if (smp[u] && m < a.R)  // per slot LayoutLeft [R x Tcap]
            a.seis[(uint64_t)(slot0 + u * kCols + col) * a.R * a.Tcap + (uint64_t)a.R * (nextIdx[u] - 1) + m] = y;
        }
      }
#pragma unroll
    for (int u = 0; u < SETS; ++u)
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        double z = q[u][1][t] + a.dt * acc[u][t];
        asm("" : "+v"(z));
        q[u][1][t] = s0[u] + it < hz[u] ? z : q[u][1][t];
      }
    share(std::integral_constant<int, 1>{});
    if (j == 3)  // (the copy waits for the load, so it comes late and as a branch)
#pragma unroll
      for (int u = 0; u < SETS; ++u) {
        asm volatile("" : "+v"(f4next[u]));
        f4[u] = f4next[u];
      }
#pragma unroll
    for (int u = 0; u < SETS; ++u)
      if (ev[u] && s0[u] + it < hz[u]) {
        phase[u] = phase[u] + 1 == ev[u] ? 0 : phase[u] + 1;
        if (phase[u] == 0) ++nextIdx[u];
      }
  }
#pragma unroll
  for (int u = 0; u < SETS; ++u)
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const uint64_t at0 = (uint64_t)(slot0 + u * kCols + col) * K + rt[t] * 16 + row;
      a.qv[at0] = q[u][0][t];
      a.qs[at0] = q[u][1][t];
    }
  reportLost(lost, lane);
  // (all workgroups of the columns have read the counters: they have met)
  if (part == 0 && tid < kCols * SETS) {
    const uint64_t h = a.horizon[slot0 + tid];
    const uint64_t st = a.stepCol[slot0 + tid], s = st + a.nsteps;
    a.stepCol[slot0 + tid] = s < h ? s : (st < h ? h : st);
  }
}

template <int G, int WAVES, int RR, int LL, int DR>
void launchF64(const RomArgs& a, uint64_t cols, hipStream_t stream) {
  constexpr size_t lds = (size_t)2 * 16 * G * kCols * 8 + (size_t)2 * G * LL * 64 * 32;
  static_assert(lds <= 160 * 1024, "LDS of one CU");
  const auto kernel = k_rom_f64<G, WAVES, RR, LL, DR>;
  SHAW_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kernel, dim3((unsigned)(cols / kCols)), dim3(WAVES * 64), lds, stream, a);
}

template <int G, int WAVES, int RR, int LL, int DR, int SPLIT, int SETS>
bool launchF64Shared(const RomArgs& a, hipStream_t stream) {
  constexpr size_t lds = (size_t)SETS * 2 * 16 * G * kCols * 8 + (size_t)2 * (G / SPLIT) * LL * 64 * 32;
  static_assert(lds <= 160 * 1024, "LDS of one CU");
  const auto kernel = k_rom_f64_shared<G, WAVES, RR, LL, DR, SPLIT, SETS>;
  SHAW_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const unsigned groups = a.tiles * (kTileCols / (kCols * SETS));
  return launchCooperative((const void*)kernel, (groups + 7) / 8 * 8 * SPLIT, WAVES * 64, lds, a, stream);
}

}  // namespace

// Four columns a workgroup while the CUs they fill pay for re-reading the
// operators: at K = 64, resident, always (4096 columns 1.9 us against 2.6, 32768
// 14.0 against 17.0); at 128 up to 448 active tiles of 16 columns, 1.6 us a round of
// 64 (4096 columns 6.9 us against 7.1, 7168 11.7 against 12.2, 8192 13.2 against 12.7);
// above, one round of workgroups per 64 tiles (K = 256: 7.7 us a round) against
// k_rom_steps' 18 us for up to 256 of them: two rounds.
bool romF64Fits(uint32_t modes, uint64_t activeTiles) {
  return modes <= 64 || activeTiles <= (modes <= 128 ? 448 : 128);
}

void launchRomF64(const RomArgs& a, hipStream_t stream) {
  const uint64_t cols = (uint64_t)a.tiles * kTileCols;
  switch (a.Kvp / 64) {
    case 1: launchF64<4, 4, 4, 0, 1>(a, cols, stream); break;
    case 2: launchF64<8, 8, 8, 0, 1>(a, cols, stream); break;
    case 3: launchF64<12, 4, 8, 3, 1>(a, cols, stream); break;
    case 4: launchF64<16, 8, 4, 2, 2>(a, cols, stream); break;
    case 6: launchF64<24, 8, 2, 1, 1>(a, cols, stream); break;
    default: launchF64<32, 8, 0, 1, 2>(a, cols, stream); break;
  }
}

bool launchRomF64Shared(const RomArgs& a, uint32_t sets, hipStream_t stream) {
  switch (a.Kvp / 64) {
    case 4: return launchF64Shared<16, 4, 8, 4, 1, 4, 1>(a, stream);
    case 6: return sets == 1 ? launchF64Shared<24, 4, 16, 7, 1, 6, 1>(a, stream) : launchF64Shared<24, 4, 16, 6, 1, 6, 2>(a, stream);
    default: return sets == 1 ? launchF64Shared<32, 4, 14, 7, 2, 8, 1>(a, stream) : launchF64Shared<32, 4, 14, 6, 2, 8, 2>(a, stream);
  }
}

}  // namespace shaw
