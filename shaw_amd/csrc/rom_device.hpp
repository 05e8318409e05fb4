// Device code shared by the reduced-leapfrog kernels (rom.hip,
// rom_resident.hip): kernel arguments, MFMA wrappers, bf16 splits, operator
// products through a register ring, receivers and the macro-step plan.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

namespace shaw {

// ------------------------------------------------------------ reduced leapfrog
// Operators are packed for the MFMA A operand in lane items, laid out
// [rowTile][group][lane] so that one wave reads contiguous memory per group:
//   FP64:   32-byte items; group g of row tile t covers k-steps 4g..4g+3 of
//           16 x 16 x 4; lane l holds A[16t + l%16][16g + 4s + l/16], s < 4.
//   BF16x3 / BF16x4: 2 / 3 parts of 16 bytes (hi, lo, residual bf16 parts);
//           group g covers k = 32g .. 32g + 31, one 16 x 16 x 32 product per
//           part; part p of lane l holds that part of
//           A[16t + l%16][32g + 16s + 4(l/16) + e] at position 4s + e,
//           s < 2, e < 4 (the state's split uses the same k order).
// Padded sizes are multiples of kRing groups (64 for FP64, 128 for BF16), of
// two groups (64) for engines of up to 256 modes whose operators stay on the CU.
struct RomArgs {
  const void* av;       // Ar_v: rows Kvp, k-dim Ksp
  const void* as;       // Ar_s: rows Ksp, k-dim Kvp
  const void* c;        // C:    rows Rp,  k-dim Kvp
  double* qv;           // [slot][Kvp]
  double* qs;           // [slot][Ksp]
  const double* b;      // [slot][Kvp]
  const double* ftab;   // [slot][maxSteps]
  uint64_t* stepCol;    // [slot]
  const uint64_t* horizon;
  const uint64_t* every;
  double* seis;         // [slot][R][Tcap]
  uint32_t Kvp, Ksp, Rp, R;
  uint64_t maxSteps, Tcap, nsteps;
  double dt;
  // macro steps (BF16 kernels): the blocks of G = (F^m - I) / dt, F the
  // one-step matrix of [q_v; q_s]: G_vv [Kvp x Kvp], G_vs [Kvp x Ksp], G_sv,
  // G_ss, packed as the operators; m = 0 turns them off
  const void *gvv, *gvs, *gsv, *gss;
  uint32_t groupsV, groupsS;  // the dofs' k-groups of 32 modes that are not all padding, even
  const uint32_t* quiet;  // [slot] first step from which the column's forcing is negligible
  uint32_t macro;
  // time budget (macro steps on): 0, nsteps steps for every tile; w > 0, the
  // time of nsteps one-steps for every tile, a macro step costing w of them,
  // so tiles taking macro steps advance further (stepCol holds how far)
  uint32_t budget;
  // tiles of 16 columns; and where several workgroups share columns (SPLIT > 1):
  // exchange buffers, the groups' meeting words (joinGroup), the launch's number,
  // from 1, how often a wave looks in vain for the others, whether it does not wait
  // for their words at all (a test), and host memory: [0] the last launch in which
  // a group did not meet, [1] the last in which a word of an exchange never came
  uint32_t tiles;
  uint64_t* xbuf;
  uint64_t* meet;
  uint64_t launch;
  uint32_t meetTries, noWords;
  uint64_t* gaveUp;
  // sets > 0: a launch that repeats `launch` for the groups that did not meet in
  // it, of that many workgroups of an unshared launch each; the others return
  uint32_t repeat;
};

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));
typedef short shrt4 __attribute__((ext_vector_type(4)));
typedef short shrt16 __attribute__((ext_vector_type(16)));

constexpr int kTileCols = 16;  // column slots per workgroup
constexpr int kWaves = 8;      // waves per ROM workgroup (16 at 9..16 row tiles)

// ------------------------------------------------------------ exchange
// Workgroups that share a tile of columns exchange states through memory, in
// device scope, 64 bits at a time. (They have met first: joinGroup.) A reader
// takes each word from memory until it is not kEmpty (four bf16 NaNs, a double's
// NaN), so nothing is waited for but the data. Exchanges of a tile take turns on
// three buffers. After exchange e every wave has read e - 1, and its writer
// empties it; that is out (written) before the writer's words of e + 1, and so
// before anyone who has them looks there for exchange e + 2. (A fourth buffer,
// which leaves the emptying another exchange, measured the same within 2 %.)
constexpr uint64_t kEmpty = ~0ull;
constexpr int kXbufs = 3;
constexpr int kMeetStride = 16;  // words from one group's meeting word to the next: a cache line each
constexpr uint32_t kMaxTries = 1u << 24;  // looks of a bounded wait, each a read of memory (about 10 s)
__device__ __forceinline__ void put(uint64_t* x, uint64_t v) {
  __hip_atomic_store(x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get(const uint64_t* x) {
  return __hip_atomic_load(x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void putWord(uint64_t* x, uint64_t v) { put(x, v == kEmpty ? kEmpty >> 1 : v); }
__device__ __forceinline__ void written() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// d[i * STRIDE] = x[i * STRIDE], i < N, once all are there. (The workgroups have
// met, so all run and every word comes. Should one not, lost is set, the wave
// goes on with what it has and reportLost tells the host.)
template <int N, int STRIDE>
__device__ __forceinline__ void collectWords(const uint64_t* x, uint64_t* d, bool& lost) {
  uint64_t v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = kEmpty;
  for (uint32_t tries = 0;; ++tries) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (v[i] == kEmpty) v[i] = get(x + i * STRIDE);
    bool missing = false;
#pragma unroll
    for (int i = 0; i < N; ++i) missing |= v[i] == kEmpty;
    if (lost || __ballot(missing) == 0) break;
    lost = tries > kMaxTries;
  }
#pragma unroll
  for (int i = 0; i < N; ++i) d[i * STRIDE] = v[i];
}
__device__ __forceinline__ void tellHost(uint64_t* word, uint64_t v) {
  __hip_atomic_store(word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// (The arguments are read again from the kernel's argument block: kept in registers
// from the start they displaced others of the step loop.)
__device__ __forceinline__ void reportLost(bool lost, int lane) {
  if (!lost) return;
  typedef const __attribute__((address_space(4))) RomArgs* Args;
  Args a = (Args)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  if (lane == 0) tellHost(a->gaveUp + 1, a->launch);
}
// A group's meeting word: launch number, kNotMet, waves that came. All `waves`
// waves of a group meet in a launch or none of them does: a wave that looked in
// vain too often puts kNotMet in by a compare-exchange against a count that is not
// full, which fails once the last wave has come, and a wave that finds kNotMet
// gives up too. (A cooperative launch makes sure of the room on an empty chip only:
// a long launch of another stream can keep part of a group waiting for a CU.) What
// the wave wrote before is out when the others have met it.
constexpr uint64_t kNotMet = 1u << 15;
__device__ __forceinline__ bool joinGroup(const RomArgs& a, uint32_t group, uint32_t waves, int lane) {
  written();
  bool met = false;
  if (lane == 0) {
    uint64_t* const word = a.meet + (uint64_t)group * kMeetStride;
    (void)__hip_atomic_fetch_max(word, a.launch << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint64_t v = __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    for (uint32_t tries = 0;; ++tries) {
      if (v & kNotMet) break;
      met = (v & (kNotMet - 1)) == waves;
      if (met) break;
      if (tries < a.meetTries) {
        v = get(word);
      } else if (__hip_atomic_compare_exchange_strong(word, &v, v | kNotMet, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT)) {
        tellHost(a.gaveUp, a.launch);
        break;
      }  // (else v is the word as it was: a wave has come or given up meanwhile, at most `waves` times)
    }
  }
  asm volatile("" ::: "memory");
  return __builtin_amdgcn_readfirstlane((int)met) != 0;
}
// whether an unshared workgroup of a repeating launch has anything to do
__device__ __forceinline__ bool repeats(const RomArgs& a, uint32_t workgroup) {
  const uint64_t v = a.meet[(uint64_t)(workgroup / a.repeat) * kMeetStride];
  return (v >> 16) == a.launch && (v & kNotMet) != 0;
}

// ------------------------------------------------------------ bf16 helpers
__host__ __device__ inline unsigned short f32ToBf16(float x) {
  // round to nearest even
  unsigned int u;
  std::memcpy(&u, &x, 4);
  if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)(u >> 16);  // inf/nan
  const unsigned int lsb = (u >> 16) & 1u;
  u += 0x7fffu + lsb;
  return (unsigned short)(u >> 16);
}
__host__ __device__ inline float bf16ToF32(unsigned short h) {
  const unsigned int u = (unsigned int)h << 16;
  float x;
  std::memcpy(&x, &u, 4);
  return x;
}

// ------------------------------------------------------------ MFMA lane layouts
// v_mfma_f64_16x16x4f64 (one 16x16 output block, K = 4):
//   A: lane l holds A[l % 16][l / 16];  B: lane l holds B[l / 16][l % 16]
//   D: lane l, register r holds D[l / 16 + 4 * r][l % 16]
// v_mfma_f32_16x16x16bf16_1k:
//   A: lane l holds A[l % 16][4 * (l / 16) + e], e = 0..3
//   B: lane l holds B[4 * (l / 16) + e][l % 16]
//   D: lane l, register r holds D[4 * (l / 16) + r][l % 16]
// v_mfma_f32_16x16x32_bf16 (gfx950; twice the bf16 products per instruction
// of the 16x16x16 form):
//   A: lane l holds A[l % 16][8 * (l / 16) + e], e = 0..7
//   B: lane l holds B[8 * (l / 16) + e][l % 16]
//   D: as 16x16x16
// The ROM kernels rely only on A's value e of lane group l / 16 meeting B's
// value e of the same lane group, and on D's layout.
// These are checked on the device by shaw_debug_mfma (tests/test_gpu_rom.py).
typedef int int4v __attribute__((ext_vector_type(4)));
typedef short shrt8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ inline dbl4 mfmaF64(double a, double b, dbl4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ inline flt4 mfmaBf16(shrt4 a, shrt4 b, flt4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }
__device__ inline flt4 mfmaBf16x32(int4v a, int4v b, flt4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// result row of register r in lane l
__device__ inline int rowF64(int lane, int r) { return lane / 16 + 4 * r; }
__device__ inline int rowBf16(int lane, int r) { return 4 * (lane / 16) + r; }

// A tile's macro plan for a budget of B steps: k one-steps first (until every
// active column is at a multiple of m and quiet), then k2 macro steps (every
// column still active then at least m k2 steps from its horizon, within B).
// k2 = 0 when the tile cannot take any: active columns at different
// residues mod m, or sampled at a period that is not a multiple of m. Lanes
// hold column lane % 16 (each column 4 times); every wave computes the same.
__device__ __forceinline__ void macroPlan(uint32_t m, uint32_t s, uint32_t hz, uint32_t ev, uint32_t quiet, uint64_t B,
                                          uint64_t& k, uint64_t& k2) {
  const bool act = s < hz;
  int bad = act && ((ev != 0 && ev % m != 0) || quiet == 0xffffffffu);
  const uint32_t r = s % m;
  uint32_t rmin = act ? r : 0xffffffffu, rmax = act ? r : 0u;
  uint32_t kq = act && quiet > s ? quiet - s : 0u;
#pragma unroll
  for (int off = 32; off >= 1; off /= 2) {
    const uint32_t a = (uint32_t)__shfl_xor((int)rmin, off), b = (uint32_t)__shfl_xor((int)rmax, off);
    const uint32_t c = (uint32_t)__shfl_xor((int)kq, off);
    rmin = a < rmin ? a : rmin;
    rmax = b > rmax ? b : rmax;
    kq = c > kq ? c : kq;
    bad |= __shfl_xor(bad, off);
  }
  k = B;
  k2 = 0;
  if (rmin > rmax || bad || rmin != rmax) return;  // no active column, or no common macro point
  const uint64_t k0 = (uint64_t)kq + (m - (rmin + kq % m) % m) % m;
  uint64_t lim = ~0ull;  // macro steps the columns still active at k0 allow
  if (act && (uint64_t)hz > (uint64_t)s + k0) lim = ((uint64_t)hz - s - k0) / m;
#pragma unroll
  for (int off = 32; off >= 1; off /= 2) {
    const uint64_t o = (uint64_t)__shfl_xor((long long)lim, off);
    lim = o < lim ? o : lim;
  }
  if (lim == ~0ull || k0 > B) return;
  const uint64_t n = (B - k0) / m < lim ? (B - k0) / m : lim;
  if (n == 0) return;
  k = k0;
  k2 = n;
}

// A tile's launch under macro steps: steps in all (at most span, the steps to
// its last horizon), of which mk one-steps, mk2 macro steps, then one-steps to
// the end; the same in every lane.
__device__ __forceinline__ void launchPlan(const RomArgs& a, uint32_t s0, uint32_t hz, uint32_t ev, uint32_t quiet,
                                           uint32_t span, uint32_t& steps, uint32_t& mkOut, uint32_t& mk2Out) {
  uint64_t mk = 0, mk2 = 0;
  if (a.macro && a.budget) {
    // the time of T one-steps: mk one-steps, mk2 macro steps of a.budget
    // one-steps' time each, one-steps for the rest (horizons below 2^31)
    const uint64_t T = a.nsteps < (1ull << 31) ? a.nsteps : (1ull << 31);
    macroPlan(a.macro, s0, hz, ev, quiet, T * a.macro, mk, mk2);
    const uint64_t planned = mk2;  // what the horizons allow
    if (mk2) {
      const uint64_t cap = mk < T ? (T - mk) / a.budget : 0;
      mk2 = mk2 < cap ? mk2 : cap;
    }
    if (mk2) {
      // the time left goes to one-steps; unless a column nears its horizon,
      // whole multiples of m only, so the tile ends aligned for the next launch
      uint64_t rest = T - mk - a.budget * mk2;
      if (mk2 < planned) rest -= rest % a.macro;
      const uint64_t end = mk + (uint64_t)a.macro * mk2 + rest;
      steps = end < (uint64_t)span ? (uint32_t)end : span;
    }
  } else if (a.macro) {
    macroPlan(a.macro, s0, hz, ev, quiet, a.nsteps, mk, mk2);
  }
  // the plan is the same in every lane: keep it in scalar registers
  steps = (uint32_t)__builtin_amdgcn_readfirstlane((int)steps);
  mkOut = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)mk);
  mk2Out = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)mk2);
}

// Where a step reads the operators' k-groups from: RR groups of every row tile
// sit in registers, LL in LDS, the other KG - RR - LL stream from L2 through a
// ring of DR groups. The streamed groups are spread evenly, so the products of
// the resident ones hide each refill.
template <int KG, int RR, int LL, int DR>
struct Place {
  static constexpr int S = KG - RR - LL;
  static constexpr int group(int s) { return s * KG / (S > 0 ? S : 1); }  // the s-th streamed group
  static constexpr bool streamed(int g) {
    for (int q = 0; q < S; ++q)
      if (group(q) == g) return true;
    return false;
  }
  // index of group g among those of its kind (streamed, or not: LDS first)
  static constexpr int index(int g) {
    int n = 0;
    for (int q = 0; q < g; ++q) n += streamed(q) == streamed(g);
    return n;
  }
};

constexpr int kRing = 4;  // operator groups kept in flight per row tile

// PARTS = 0: FP64 operators; 2: bf16 hi + lo (BF16x3); 3: bf16 hi + lo +
// residual (BF16x4). Ring items: a dbl4 (FP64) or PARTS 16-byte parts, part p
// holding that part's 8 bf16 values of group g (32 B or 48 B).
template <int PARTS>
struct BfItem {
  int4v p[PARTS];
};
template <int PARTS>
struct Prec {
  using Item = BfItem<PARTS>;
  using Acc = flt4;
};
template <>
struct Prec<0> {
  using Item = dbl4;
  using Acc = dbl4;
};

// B operand of k-step group g. FP64: X is the state [K][16] in LDS. BF16:
// X is the state's bf16 split (writeSplitRows): hi parts, then lo parts, each
// [K/32][4][16] items of 8 bf16 values in the operator's k order, so a
// lane's operand of a group is one 16-byte read.
template <int PARTS, int TPW>
__device__ __forceinline__ void groupProducts(const typename Prec<PARTS>::Item (&ag)[TPW], int g, const void* X,
                                              int loOff, int lane, typename Prec<PARTS>::Acc (&acc)[TPW]) {
  if constexpr (PARTS == 0) {
    const double* Xd = static_cast<const double*>(X);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const double xb = Xd[((4 * g + s) * 4 + lane / 16) * kTileCols + lane % 16];
#pragma unroll
      for (int t = 0; t < TPW; ++t) acc[t] = mfmaF64(ag[t][s], xb, acc[t]);
    }
  } else {
    const int4v* Xh = static_cast<const int4v*>(X);
    const int item = (4 * g + lane / 16) * kTileCols + lane % 16;
    const int4v xh = Xh[item], xl = Xh[loOff + item];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      acc[t] = mfmaBf16x32(ag[t].p[0], xh, acc[t]);
      acc[t] = mfmaBf16x32(ag[t].p[0], xl, acc[t]);
      acc[t] = mfmaBf16x32(ag[t].p[1], xh, acc[t]);
      if constexpr (PARTS == 3) acc[t] = mfmaBf16x32(ag[t].p[2], xh, acc[t]);
    }
  }
}

// operator groups kept in flight per row tile: kRing, or 2 where the ring
// of all the wave's tiles would not fit the registers (register-resident
// states: beside one tile of 8 waves)
template <int PARTS, int TPW, int WAVES, bool RESIDENT>
constexpr int ringDepth() {
  return RESIDENT ? (TPW == 1 && WAVES <= 8 ? kRing : 2) : (PARTS * TPW > 9 ? 2 : kRing);
}

// issue the loads of groups 0 .. D-1 of the wave's row tiles
template <int PARTS, int TPW, int D>
__device__ __forceinline__ void preloadRing(const void* __restrict__ Araw, int kGroups, const int (&rt)[TPW], int lane,
                                            typename Prec<PARTS>::Item (&ring)[D][TPW]) {
  using Item = typename Prec<PARTS>::Item;
  const Item* A = reinterpret_cast<const Item*>(Araw);
#pragma unroll
  for (int d = 0; d < D; ++d) {
#pragma unroll
    for (int t = 0; t < TPW; ++t) ring[d][t] = A[((size_t)rt[t] * kGroups + d) * 64 + lane];
    __builtin_amdgcn_sched_barrier(0);  // issue order = consumption order
  }
}

// acc[t] = (row tile rt[t] of A) X over all kGroups groups; the ring holds
// groups 0 .. D-1 on entry (preloadRing) and is refilled D groups ahead
// (ZERO = false: add to acc instead, for a product of two operator blocks)
template <int PARTS, int TPW, int D, bool ZERO = true>
__device__ __forceinline__ void consumeRing(const void* __restrict__ Araw, int kGroups, const int (&rt)[TPW],
                                            const void* X, int loOff, int lane,
                                            typename Prec<PARTS>::Item (&ring)[D][TPW],
                                            typename Prec<PARTS>::Acc (&acc)[TPW]) {
  using Item = typename Prec<PARTS>::Item;
  const Item* A = reinterpret_cast<const Item*>(Araw);
  const Item* row[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    if constexpr (ZERO) acc[t] = typename Prec<PARTS>::Acc{0, 0, 0, 0};
    row[t] = A + (size_t)rt[t] * kGroups * 64 + lane;
  }
  int g0 = 0;
  for (; g0 + D < kGroups; g0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      groupProducts<PARTS, TPW>(ring[d], g0 + d, X, loOff, lane, acc);
#pragma unroll
      for (int t = 0; t < TPW; ++t) ring[d][t] = row[t][(g0 + d + D) * 64];
      // keep this group's refill here: the scheduler would otherwise sink all
      // refills of the round to its end, shortening the prefetch distance
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) groupProducts<PARTS, TPW>(ring[d], g0 + d, X, loOff, lane, acc);
}

template <int PARTS, int TPW, int D = ringDepth<PARTS, TPW, kWaves, false>()>
__device__ __forceinline__ void tileProducts(const void* __restrict__ Araw, int kGroups, const int (&rt)[TPW],
                                             const void* X, int loOff, int lane, typename Prec<PARTS>::Acc (&acc)[TPW]) {
  typename Prec<PARTS>::Item ring[D][TPW];
  preloadRing<PARTS, TPW, D>(Araw, kGroups, rt, lane, ring);
  consumeRing<PARTS, TPW, D>(Araw, kGroups, rt, X, loOff, lane, ring, acc);
}

__device__ __forceinline__ int accRow(int parts, int lane, int r) { return parts ? rowBf16(lane, r) : rowF64(lane, r); }

template <int PARTS, int TPW, int WAVES, int D = ringDepth<PARTS, TPW, kWaves, false>()>
__device__ __forceinline__ void receivers(const RomArgs& a, const void* Xv, int loOff, int wave, int lane, bool sample,
                                          uint32_t sampleIdx, int slot0) {
  const int rowTiles = a.Rp / 16, kGroups = PARTS ? a.Kvp / 32 : a.Kvp / 16;
  for (int rt0 = wave; rt0 < rowTiles; rt0 += WAVES * TPW) {
    int rt[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) rt[t] = rt0 + t * WAVES < rowTiles ? rt0 + t * WAVES : rt0;
    typename Prec<PARTS>::Acc acc[TPW];
    tileProducts<PARTS, TPW, D>(a.c, kGroups, rt, Xv, loOff, lane, acc);
    const int col = lane % 16;
#pragma unroll
    for (int t = 0; t < TPW; ++t)
      if (rt0 + t * WAVES < rowTiles && sample)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = rt[t] * 16 + accRow(PARTS, lane, r);
          // per slot LayoutLeft [R x Tcap]
          if (row < (int)a.R)
            a.seis[(uint64_t)(slot0 + col) * a.R * a.Tcap + (uint64_t)a.R * sampleIdx + row] = (double)acc[t][r];
        }
  }
}

// the bf16 split of the 4 state rows a lane holds after the products of row
// tile rt (rows 16 rt + 4 (lane / 16) + r, column lane % 16): x = float(q),
// hi = bf16(x), lo = bf16(x - hi), both rounded to nearest even. Item
// (4 g + q') * 16 + c of the split holds, at position 4 s + e, k = 32 g +
// 16 s + 4 q' + e of column c (the operator's k order, see the packing
// above); here g = rt / 2, s = rt % 2, q' = lane / 16, e = r
__device__ __forceinline__ void writeSplitRows(int4v* S, int loOff, int rt, int lane, const double (&q)[4]) {
  shrt4 h, l;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float x = (float)q[r];
    const unsigned short hb = f32ToBf16(x);
    h[r] = (short)hb;
    l[r] = (short)f32ToBf16(x - bf16ToF32(hb));
  }
  const int item = (4 * (rt / 2) + lane / 16) * kTileCols + lane % 16;
  *(reinterpret_cast<shrt4*>(S + item) + rt % 2) = h;
  *(reinterpret_cast<shrt4*>(S + loOff + item) + rt % 2) = l;
}

}  // namespace
}  // namespace shaw
