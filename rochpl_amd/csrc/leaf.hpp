// Register-resident cooperative leaf of the panel factorisation
// (HPL_pdpanrlT, src/pfact/HPL_pdpanrlT_device.cpp:23-468): one launch per
// leaf of <= 32 columns.  Instantiated in k_leaf*.hip for each (register
// type T, storage type S) pair: FP64 for the HPL solve, FP32 for the panels
// of the mixed-precision factorisations.
//
// Every workgroup keeps its slice of the leaf (NT threads, RPT rows of 32
// columns each) in registers for the whole leaf.  A row never moves: each carries
// a label, the row it stands for at the moment, and an interchange swaps two
// labels.  At the end every row is stored where its label says.  Per column:
//   1. each workgroup finds its candidate max |a|, ties to the lower label
//      (DPP lane exchanges within a wave, then the waves through LDS);
//   2. the wave holding the candidate row stores it into the workgroup's
//      slot, every 32-bit half of a value in an 8-byte word whose other half
//      is the column's sequence number, so that a word is complete as soon
//      as its number is seen: no release, no acquire, no separate flag;
//   3. the waves read all slots, polling the words themselves, into LDS;
//      after one workgroup barrier every wave picks the pivot row;
//   4. labels are swapped, the rows left are divided by the pivot, and the
//      next column is updated;
//   5. the other columns are updated, the pivot row's values broadcast within
//      the FMA (DPP), while the next column's candidates are under way (see
//      leaf_publish).  The pivot row is finished: workgroup 0 keeps it in LDS
//      for the end.
// Slots are double-buffered by column parity, so a workgroup that runs ahead
// never overwrites a slot another workgroup still reads.  A grid of one
// workgroup passes the row through LDS only.  The reference instead parks
// its leaf on a pinned host flag once per column and lets a host thread run
// HPL_pdmxswp (:94-117,455-463).
//
// One column's code is looped over, with static register indices: the tile's
// first 8 positions rotate by one per column, all 32 by 8 after 8 columns.
// With all 32 columns instantiated the leaf was bound by instruction fetch
// (300 KB of code, each instruction run once).
//
// Every wait is bounded: after kSpinLimit polls a workgroup raises *err and
// all workgroups leave the kernel, so a grid that is not co-resident cannot
// hang the device.
#pragma once

#include <climits>
#include <type_traits>

#include "hplx_internal.hpp"
#include "lds_stream.hpp"

namespace hplx {
namespace leaf {

constexpr uint32_t kSpinLimit = 1u << 22;
constexpr int      kTurn      = 8;  // columns per turn of the column loop
// slot layout (8-byte words, sequence number in the upper half): [0..63] the
// candidate row's 32-bit halves (FP32: [0..31] its values), [64..67] its
// header: key (upper, lower half), label, the row it was loaded from, the
// row's factor in the update it still lacks (lower, upper half)
constexpr int kSlotHead = 64, kHeadWords = 6;
static_assert(kSlotHead + kHeadWords <= kSlotStride, "slot too small");
// Up to kNear workgroups every candidate row is read along with its header
// (one memory round trip); with more the headers come first and then only
// the pivot row.
constexpr int kNear = 32;
// Time until the first poll of the slots (x 64 cycles): what the candidates
// take to be seen.  A poll that comes too early costs a whole round trip: 4096
// / 9001 / 32000 rows, us with 0, 3, 6, 9, 12: 95.7 / 99.7 / 115.5, 89.4 / 95.1
// / 112.8, 89.3 / 91.8 / 110.9, 91.9 / 92.0 / 110.8, 94.2 / 95.9 / 111.3.
constexpr int kFirstPoll = 7;

struct LeafArgs {
  void*    P;          // panel top-left (panel row 0), storage type S
  int      lda;
  int      m;          // panel rows
  int      JB;         // panel width (row interchanges span it)
  int      c0;         // first leaf column (panel relative)
  int      w;          // leaf width, <= 32
  int*     ipiv;       // panel-relative pivots (+ row_offset) written here
  int      row_offset;
  int*     info;       // first exact zero pivot, 1-based global column
  int      info_base;  // global column of panel column 0
  double*  slots;      // 2 x (kMaxGrid+1) x kSlotStride 8-byte words
  uint32_t seq_base;   // unique per launch; column j publishes seq_base+j+1
  int*     err;
  int      grid;       // workgroups taking part: 0 .. grid-1 (<= gridDim.x)
};

// Shared-memory scratch of the leaf kernel.
template <typename T>
struct LeafShared {
  alignas(16) T cand[kNear][kLeafMax];    // the workgroups' candidate rows
  alignas(16) T row[2][kLeafMax];         // this workgroup's, by column parity
  alignas(16) T fin[kLeafMax][kLeafMax];  // workgroup 0: the finished top rows
  // the pivot row, by column parity, as the tile is arranged for its column and
  // for the next
  alignas(16) T ucur[2][2][kLeafMax];
  alignas(16) T nl[2];                    // this workgroup's candidate's factor
  alignas(16) uint32_t head[kNear][8];    // the candidates' headers
  alignas(16) uint32_t wave[2][16][4];    // the waves' candidates, as headers
  int      sel[2];  // the pivot's label and the row it was loaded from
  uint32_t sel_nl[2];  // and its factor's halves
  int ok;
};

// (a, b, c, d) = (b, c, d, a) in place.  In assembly because the compiler,
// given the moves, keeps a second copy of the tile and spills it.
__device__ inline void rotate4(double& a, double& b, double& c, double& d) {
  double t;
  asm volatile(
      "v_mov_b64 %4, %0\n\tv_mov_b64 %0, %1\n\tv_mov_b64 %1, %2\n\t"
      "v_mov_b64 %2, %3\n\tv_mov_b64 %3, %4"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "=&v"(t));
}
__device__ inline void rotate4(float& a, float& b, float& c, float& d) {
  float t;
  asm volatile(
      "v_mov_b32 %4, %0\n\tv_mov_b32 %0, %1\n\tv_mov_b32 %1, %2\n\t"
      "v_mov_b32 %2, %3\n\tv_mov_b32 %3, %4"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "=&v"(t));
}

// (a, ..., h) = (b, ..., h, a) in place.
__device__ inline void rotate8(double& a, double& b, double& c, double& d, double& e, double& f, double& g,
                               double& h) {
  double t;
  asm volatile(
      "v_mov_b64 %8, %0\n\tv_mov_b64 %0, %1\n\tv_mov_b64 %1, %2\n\t"
      "v_mov_b64 %2, %3\n\tv_mov_b64 %3, %4\n\tv_mov_b64 %4, %5\n\t"
      "v_mov_b64 %5, %6\n\tv_mov_b64 %6, %7\n\tv_mov_b64 %7, %8"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f), "+v"(g), "+v"(h),
        "=&v"(t));
}
__device__ inline void rotate8(float& a, float& b, float& c, float& d, float& e, float& f, float& g,
                               float& h) {
  float t;
  asm volatile(
      "v_mov_b32 %8, %0\n\tv_mov_b32 %0, %1\n\tv_mov_b32 %1, %2\n\t"
      "v_mov_b32 %2, %3\n\tv_mov_b32 %3, %4\n\tv_mov_b32 %4, %5\n\t"
      "v_mov_b32 %5, %6\n\tv_mov_b32 %6, %7\n\tv_mov_b32 %7, %8"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f), "+v"(g), "+v"(h),
        "=&v"(t));
}

template <typename T, typename S>
__device__ inline T load_s(const S* p) {
  return static_cast<T>(*p);
}

template <typename T, typename S>
__device__ inline void store_s(S* p, T v) {
  *p = static_cast<S>(v);
}

__device__ inline int readlane(int x, int l) {
  return __builtin_amdgcn_readlane(x, l);
}
__device__ inline uint32_t readlane(uint32_t x, int l) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x), l));
}
__device__ inline double readlane(double x, int l) {
  return __hiloint2double(readlane(__double2hiint(x), l),
                          readlane(__double2loint(x), l));
}
__device__ inline float readlane(float x, int l) {
  return __int_as_float(readlane(__float_as_int(x), l));
}

// The order of the candidates is that of their keys, (upper, lower) half as
// unsigned numbers, then of their labels, the smaller first.  A row's key is
// the bit pattern of |a|, the upper half raised by kKeyBase; 0: no row; 1: a
// NaN in the top row (taken if the column has no number at all, other NaNs
// never).
constexpr uint32_t kKeyBase = 2, kKeyTopNan = 1;

__device__ inline uint32_t hi_bits(double x) {
  return static_cast<uint32_t>(__double2hiint(x));
}
__device__ inline uint32_t lo_bits(double x) {
  return static_cast<uint32_t>(__double2loint(x));
}
__device__ inline uint32_t hi_bits(float x) { return __float_as_uint(x); }
__device__ inline uint32_t lo_bits(float) { return 0; }
__device__ inline double from_halves(uint32_t lo, uint32_t hi, double) {
  return __hiloint2double(static_cast<int>(hi), static_cast<int>(lo));
}
__device__ inline float from_halves(uint32_t lo, uint32_t, float) {
  return __uint_as_float(lo);
}
template <typename T>
constexpr uint32_t kInfBits = sizeof(T) == 8 ? 0x7ff00000u : 0x7f800000u;

template <int CTRL, int ROW_MASK>
__device__ inline uint32_t max_dpp(uint32_t k) {
  const uint32_t o = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
      0, static_cast<int>(k), CTRL, ROW_MASK, 0xF, false));
  return o > k ? o : k;
}

// Maximum over each row of 16 lanes, in each of them.
__device__ inline uint32_t row_max(uint32_t k) {
  k = max_dpp<0xB1, 0xF>(k);      // quad_perm [1,0,3,2]
  k = max_dpp<0x4E, 0xF>(k);      // quad_perm [2,3,0,1]
  k = max_dpp<0x141, 0xF>(k);     // row_half_mirror
  return max_dpp<0x140, 0xF>(k);  // row_mirror
}

// Maximum over the wave: within a row of 16 lanes by quad permutes and
// mirrors, across rows by broadcasts of lane 15 (into rows 1 and 3) and lane
// 31 (into rows 2 and 3).
__device__ inline uint32_t wave_max(uint32_t k) {
  k = row_max(k);
  k = max_dpp<0x142, 0xA>(k);  // row_bcast:15
  k = max_dpp<0x143, 0xC>(k);  // row_bcast:31
  return readlane(k, 63);
}

// Of the lanes in `mask` (not empty; equal upper halves) the first one in the
// candidates' order, nearly always the only one; of empty candidates (upper
// half 0) any.
__device__ inline int first_of(unsigned long long mask, uint32_t hi,
                               uint32_t lo, int lab) {
  int best = __builtin_ctzll(mask);
  mask &= mask - 1;
  if(mask && hi) {
    uint32_t bo = readlane(lo, best);
    int      bl = readlane(lab, best);
    for(; mask; mask &= mask - 1) {
      const int      l = __builtin_ctzll(mask), x = readlane(lab, l);
      const uint32_t o = readlane(lo, l);
      if(o > bo || (o == bo && x < bl)) {
        bo   = o;
        bl   = x;
        best = l;
      }
    }
  }
  return best;
}

__device__ inline unsigned long long ld_word(const unsigned long long* p) {
  return __hip_atomic_load(const_cast<unsigned long long*>(p), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_word(unsigned long long* p, uint32_t seq, uint32_t x) {
  __hip_atomic_store(p, (static_cast<unsigned long long>(seq) << 32) | x,
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Word of a candidate row that a lane carries.
template <typename T>
__device__ inline int word_of(int lane) {
  return sizeof(T) == 8 ? lane : lane & (kLeafMax - 1);
}

// Word of a header that a lane carries.
__device__ inline int head_word(int lane) {
  return (lane & 7) < kHeadWords ? lane & 7 : 0;
}

// A wait's poll failed: true when the grid has to stop.
__device__ inline bool give_up(uint32_t& spins, int* err) {
  ++spins;
  if((spins & 255u) == 0 &&
     __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    return true;
  if(spins > kSpinLimit) {
    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  }
  __builtin_amdgcn_s_sleep(1);
  return false;
}

// Every workgroup's candidate of sequence `seq` into sh.cand / sh.head: wave
// w of NW takes slots w, w + NW, ..., up to four.  (Two polls under way at a
// time are no faster: the barrier that follows waits for both.)  False on
// timeout or error.
template <typename T, int NW>
__device__ __forceinline__ bool gather_all(const LeafArgs& a,
                                           const unsigned long long* slots,
                                           uint32_t seq, LeafShared<T>& sh) {
  constexpr int kBatch = kNear / NW;
  constexpr int kRowWords = kLeafMax * sizeof(T) / 4;
  const int     lane = threadIdx.x & 63;
  const int     wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t*     cand = reinterpret_cast<uint32_t*>(&sh.cand[0][0]);
  uint32_t      spins = 0;
  unsigned      pending = 0;
#pragma unroll
  for(int k = 0; k < kBatch; ++k)
    if(wave + k * NW < a.grid) pending |= 1u << k;
  if(!pending) return true;
  struct Poll {
    unsigned long long rw[kBatch], hw[kBatch];
  };
  const unsigned long long* row = slots + wave * kSlotStride + word_of<T>(lane);
  const unsigned long long* head = slots + wave * kSlotStride + kSlotHead + head_word(lane);
  auto issue = [&](Poll& p) {
#pragma unroll
    for(int k = 0; k < kBatch; ++k)
      if(pending & (1u << k)) {
        p.rw[k] = ld_word(row + k * NW * kSlotStride);
        p.hw[k] = ld_word(head + k * NW * kSlotStride);
      }
  };
  auto check = [&](const Poll& p) {
#pragma unroll
    for(int k = 0; k < kBatch; ++k)
      if(pending & (1u << k)) {
        const bool in = static_cast<uint32_t>(p.rw[k] >> 32) == seq &&
                        static_cast<uint32_t>(p.hw[k] >> 32) == seq;
        if(__all(in)) {
          const int g = wave + k * NW;
          cand[g * kRowWords + word_of<T>(lane)] = static_cast<uint32_t>(p.rw[k]);
          if(lane < kHeadWords) sh.head[g][lane] = static_cast<uint32_t>(p.hw[k]);
          pending &= ~(1u << k);
        }
      }
  };
  __builtin_amdgcn_s_sleep(kFirstPoll);
  for(;;) {
    Poll p;
    issue(p);
    check(p);
    if(!pending) return true;
    if(give_up(spins, a.err)) return false;
  }
}

// The same for many workgroups, on one wave: lane l waits for the headers of
// slots l, l + 64, ..., the wave picks the pivot and waits for its row
// (sh.cand[0]; sh.sel its label and own row).
template <typename T>
__device__ __forceinline__ bool gather_pivot(const LeafArgs& a,
                                             const unsigned long long* slots,
                                             uint32_t seq, LeafShared<T>& sh) {
  const int lane = threadIdx.x & 63;
  uint32_t  kh = 0, kl = 0, spins = 0;
  int       gl = INT_MAX, go = 0, gg = 0;
  for(int g0 = 0; g0 < a.grid; g0 += 128) {
    unsigned long long h[2][4];
    bool               wait[2] = {g0 + lane < a.grid, g0 + 64 + lane < a.grid};
    while(__any(wait[0] || wait[1])) {
#pragma unroll
      for(int k = 0; k < 2; ++k)
        if(wait[k]) {
          const unsigned long long* s =
              slots + (g0 + 64 * k + lane) * kSlotStride + kSlotHead;
#pragma unroll
          for(int i = 0; i < 4; ++i) h[k][i] = ld_word(s + i);
        }
      bool late = false;
#pragma unroll
      for(int k = 0; k < 2; ++k)
        if(wait[k]) {
          bool in = true;
#pragma unroll
          for(int i = 0; i < 4; ++i)
            in = in && static_cast<uint32_t>(h[k][i] >> 32) == seq;
          wait[k] = !in;
          late    = late || !in;
          if(in) {
            const uint32_t hi = static_cast<uint32_t>(h[k][0]);
            const uint32_t lo = static_cast<uint32_t>(h[k][1]);
            const int      l  = static_cast<int>(h[k][2]);
            if(hi > kh || (hi == kh && (lo > kl || (lo == kl && l < gl)))) {
              kh = hi;
              kl = lo;
              gl = l;
              go = static_cast<int>(h[k][3]);
              gg = g0 + 64 * k + lane;
            }
          }
        }
      if(__any(late) && give_up(spins, a.err)) return false;
    }
  }
  const uint32_t top = wave_max(kh);
  const int      w   = first_of(__ballot(kh == top), top, kl, gl);
  const int      g   = readlane(gg, w);
  const int      lb = readlane(gl, w), org = readlane(go, w);
  if(lane == 0) {
    sh.sel[0] = lb;
    sh.sel[1] = org;
  }
  const unsigned long long* s = slots + g * kSlotStride;
  for(;;) {
    const unsigned long long x = ld_word(s + word_of<T>(lane));
    const unsigned long long y = ld_word(s + kSlotHead + 4 + (lane & 1));
    if(__all(static_cast<uint32_t>(x >> 32) == seq && static_cast<uint32_t>(y >> 32) == seq)) {
      reinterpret_cast<uint32_t*>(&sh.cand[0][0])[word_of<T>(lane)] =
          static_cast<uint32_t>(x);
      if(lane < 2) sh.sel_nl[lane] = static_cast<uint32_t>(y);
      return true;
    }
    if(give_up(spins, a.err)) return false;
  }
}

// v[POS + i][Q0 + q] += u[POS + i] * nl[Q0 + q] for i = 0 .. 7, q < 1 or 3,
// u[N] the value that lane N mod 16 of each row of 16 lanes holds.  In assembly for
// the DPP form of the FMA, which the compiler does not form; the wait states
// cover a VALU write of u just before.  Every lane of the wave has to be
// active.
template <int POS, int Q0>
__device__ __forceinline__ void fma_group1(double (&v)[kLeafMax][1], double u,
                                           const double (&nl)[1]) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %8, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %8, %9 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %8, %9 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %8, %9 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %4, %8, %9 row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %5, %8, %9 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %6, %8, %9 row_newbcast:%16 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %7, %8, %9 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
      : "+v"(v[POS + 0][Q0 + 0]), "+v"(v[POS + 1][Q0 + 0]), "+v"(v[POS + 2][Q0 + 0]), "+v"(v[POS + 3][Q0 + 0]), "+v"(v[POS + 4][Q0 + 0]), "+v"(v[POS + 5][Q0 + 0]), "+v"(v[POS + 6][Q0 + 0]), "+v"(v[POS + 7][Q0 + 0])
      : "v"(u), "v"(nl[Q0 + 0]), "n"((POS + 0) & 15), "n"((POS + 1) & 15), "n"((POS + 2) & 15), "n"((POS + 3) & 15), "n"((POS + 4) & 15), "n"((POS + 5) & 15), "n"((POS + 6) & 15), "n"((POS + 7) & 15));
}
template <int POS, int Q0>
__device__ __forceinline__ void fma_group1(float (&v)[kLeafMax][1], float u,
                                           const float (&nl)[1]) {
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %8, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %8, %9 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %8, %9 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %8, %9 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %4, %8, %9 row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %5, %8, %9 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %6, %8, %9 row_newbcast:%16 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %7, %8, %9 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
      : "+v"(v[POS + 0][Q0 + 0]), "+v"(v[POS + 1][Q0 + 0]), "+v"(v[POS + 2][Q0 + 0]), "+v"(v[POS + 3][Q0 + 0]), "+v"(v[POS + 4][Q0 + 0]), "+v"(v[POS + 5][Q0 + 0]), "+v"(v[POS + 6][Q0 + 0]), "+v"(v[POS + 7][Q0 + 0])
      : "v"(u), "v"(nl[Q0 + 0]), "n"((POS + 0) & 15), "n"((POS + 1) & 15), "n"((POS + 2) & 15), "n"((POS + 3) & 15), "n"((POS + 4) & 15), "n"((POS + 5) & 15), "n"((POS + 6) & 15), "n"((POS + 7) & 15));
}
template <int POS, int Q0>
__device__ __forceinline__ void fma_group3(double (&v)[kLeafMax][3], double u,
                                           const double (&nl)[3]) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %24, %25 row_newbcast:%28 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %24, %26 row_newbcast:%28 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %24, %27 row_newbcast:%28 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %24, %25 row_newbcast:%29 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %4, %24, %26 row_newbcast:%29 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %5, %24, %27 row_newbcast:%29 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %6, %24, %25 row_newbcast:%30 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %7, %24, %26 row_newbcast:%30 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %8, %24, %27 row_newbcast:%30 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %9, %24, %25 row_newbcast:%31 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %10, %24, %26 row_newbcast:%31 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %11, %24, %27 row_newbcast:%31 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %12, %24, %25 row_newbcast:%32 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %13, %24, %26 row_newbcast:%32 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %14, %24, %27 row_newbcast:%32 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %15, %24, %25 row_newbcast:%33 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %16, %24, %26 row_newbcast:%33 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %17, %24, %27 row_newbcast:%33 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %18, %24, %25 row_newbcast:%34 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %19, %24, %26 row_newbcast:%34 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %20, %24, %27 row_newbcast:%34 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %21, %24, %25 row_newbcast:%35 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %22, %24, %26 row_newbcast:%35 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %23, %24, %27 row_newbcast:%35 row_mask:0xf bank_mask:0xf\n\t"
      : "+v"(v[POS + 0][Q0 + 0]), "+v"(v[POS + 0][Q0 + 1]), "+v"(v[POS + 0][Q0 + 2]), "+v"(v[POS + 1][Q0 + 0]), "+v"(v[POS + 1][Q0 + 1]), "+v"(v[POS + 1][Q0 + 2]), "+v"(v[POS + 2][Q0 + 0]), "+v"(v[POS + 2][Q0 + 1]), "+v"(v[POS + 2][Q0 + 2]), "+v"(v[POS + 3][Q0 + 0]), "+v"(v[POS + 3][Q0 + 1]), "+v"(v[POS + 3][Q0 + 2]), "+v"(v[POS + 4][Q0 + 0]), "+v"(v[POS + 4][Q0 + 1]), "+v"(v[POS + 4][Q0 + 2]), "+v"(v[POS + 5][Q0 + 0]), "+v"(v[POS + 5][Q0 + 1]), "+v"(v[POS + 5][Q0 + 2]), "+v"(v[POS + 6][Q0 + 0]), "+v"(v[POS + 6][Q0 + 1]), "+v"(v[POS + 6][Q0 + 2]), "+v"(v[POS + 7][Q0 + 0]), "+v"(v[POS + 7][Q0 + 1]), "+v"(v[POS + 7][Q0 + 2])
      : "v"(u), "v"(nl[Q0 + 0]), "v"(nl[Q0 + 1]), "v"(nl[Q0 + 2]), "n"((POS + 0) & 15), "n"((POS + 1) & 15), "n"((POS + 2) & 15), "n"((POS + 3) & 15), "n"((POS + 4) & 15), "n"((POS + 5) & 15), "n"((POS + 6) & 15), "n"((POS + 7) & 15));
}
template <int POS, int Q0>
__device__ __forceinline__ void fma_group3(float (&v)[kLeafMax][3], float u,
                                           const float (&nl)[3]) {
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %24, %25 row_newbcast:%28 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %24, %26 row_newbcast:%28 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %24, %27 row_newbcast:%28 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %24, %25 row_newbcast:%29 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %4, %24, %26 row_newbcast:%29 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %5, %24, %27 row_newbcast:%29 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %6, %24, %25 row_newbcast:%30 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %7, %24, %26 row_newbcast:%30 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %8, %24, %27 row_newbcast:%30 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %9, %24, %25 row_newbcast:%31 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %10, %24, %26 row_newbcast:%31 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %11, %24, %27 row_newbcast:%31 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %12, %24, %25 row_newbcast:%32 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %13, %24, %26 row_newbcast:%32 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %14, %24, %27 row_newbcast:%32 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %15, %24, %25 row_newbcast:%33 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %16, %24, %26 row_newbcast:%33 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %17, %24, %27 row_newbcast:%33 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %18, %24, %25 row_newbcast:%34 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %19, %24, %26 row_newbcast:%34 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %20, %24, %27 row_newbcast:%34 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %21, %24, %25 row_newbcast:%35 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %22, %24, %26 row_newbcast:%35 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %23, %24, %27 row_newbcast:%35 row_mask:0xf bank_mask:0xf\n\t"
      : "+v"(v[POS + 0][Q0 + 0]), "+v"(v[POS + 0][Q0 + 1]), "+v"(v[POS + 0][Q0 + 2]), "+v"(v[POS + 1][Q0 + 0]), "+v"(v[POS + 1][Q0 + 1]), "+v"(v[POS + 1][Q0 + 2]), "+v"(v[POS + 2][Q0 + 0]), "+v"(v[POS + 2][Q0 + 1]), "+v"(v[POS + 2][Q0 + 2]), "+v"(v[POS + 3][Q0 + 0]), "+v"(v[POS + 3][Q0 + 1]), "+v"(v[POS + 3][Q0 + 2]), "+v"(v[POS + 4][Q0 + 0]), "+v"(v[POS + 4][Q0 + 1]), "+v"(v[POS + 4][Q0 + 2]), "+v"(v[POS + 5][Q0 + 0]), "+v"(v[POS + 5][Q0 + 1]), "+v"(v[POS + 5][Q0 + 2]), "+v"(v[POS + 6][Q0 + 0]), "+v"(v[POS + 6][Q0 + 1]), "+v"(v[POS + 6][Q0 + 2]), "+v"(v[POS + 7][Q0 + 0]), "+v"(v[POS + 7][Q0 + 1]), "+v"(v[POS + 7][Q0 + 2])
      : "v"(u), "v"(nl[Q0 + 0]), "v"(nl[Q0 + 1]), "v"(nl[Q0 + 2]), "n"((POS + 0) & 15), "n"((POS + 1) & 15), "n"((POS + 2) & 15), "n"((POS + 3) & 15), "n"((POS + 4) & 15), "n"((POS + 5) & 15), "n"((POS + 6) & 15), "n"((POS + 7) & 15));
}
// The same for positions 1 .. 7 of the turn's 8 (u[N] for position N) at
// step j: positions from 8 - j on hold finished columns and are left alone.
template <int Q0>
__device__ __forceinline__ void fma_turn1(double (&v)[kLeafMax][1], double u,
                                          const double (&nl)[1], int j) {
  asm("s_nop 1\n\t"
      "s_cmp_gt_u32 %9, 6\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %0, %7, %8 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 5\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %1, %7, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 4\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %2, %7, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 3\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %3, %7, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 2\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %4, %7, %8 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 1\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %5, %7, %8 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 0\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %6, %7, %8 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      ".Lleaf%=:"
      : "+v"(v[1][Q0 + 0]), "+v"(v[2][Q0 + 0]), "+v"(v[3][Q0 + 0]), "+v"(v[4][Q0 + 0]), "+v"(v[5][Q0 + 0]), "+v"(v[6][Q0 + 0]), "+v"(v[7][Q0 + 0])
      : "v"(u), "v"(nl[Q0 + 0]), "s"(j)
      : "scc");
}
template <int Q0>
__device__ __forceinline__ void fma_turn1(float (&v)[kLeafMax][1], float u,
                                          const float (&nl)[1], int j) {
  asm("s_nop 1\n\t"
      "s_cmp_gt_u32 %9, 6\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %0, %7, %8 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 5\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %1, %7, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 4\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %2, %7, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 3\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %3, %7, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 2\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %4, %7, %8 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 1\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %5, %7, %8 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %9, 0\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %6, %7, %8 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      ".Lleaf%=:"
      : "+v"(v[1][Q0 + 0]), "+v"(v[2][Q0 + 0]), "+v"(v[3][Q0 + 0]), "+v"(v[4][Q0 + 0]), "+v"(v[5][Q0 + 0]), "+v"(v[6][Q0 + 0]), "+v"(v[7][Q0 + 0])
      : "v"(u), "v"(nl[Q0 + 0]), "s"(j)
      : "scc");
}
template <int Q0>
__device__ __forceinline__ void fma_turn3(double (&v)[kLeafMax][3], double u,
                                          const double (&nl)[3], int j) {
  asm("s_nop 1\n\t"
      "s_cmp_gt_u32 %25, 6\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %0, %21, %22 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %21, %23 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %21, %24 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 5\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %3, %21, %22 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %4, %21, %23 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %5, %21, %24 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 4\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %6, %21, %22 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %7, %21, %23 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %8, %21, %24 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 3\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %9, %21, %22 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %10, %21, %23 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %11, %21, %24 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 2\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %12, %21, %22 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %13, %21, %23 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %14, %21, %24 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 1\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %15, %21, %22 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %16, %21, %23 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %17, %21, %24 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 0\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f64_dpp %18, %21, %22 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %19, %21, %23 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %20, %21, %24 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      ".Lleaf%=:"
      : "+v"(v[1][Q0 + 0]), "+v"(v[1][Q0 + 1]), "+v"(v[1][Q0 + 2]), "+v"(v[2][Q0 + 0]), "+v"(v[2][Q0 + 1]), "+v"(v[2][Q0 + 2]), "+v"(v[3][Q0 + 0]), "+v"(v[3][Q0 + 1]), "+v"(v[3][Q0 + 2]), "+v"(v[4][Q0 + 0]), "+v"(v[4][Q0 + 1]), "+v"(v[4][Q0 + 2]), "+v"(v[5][Q0 + 0]), "+v"(v[5][Q0 + 1]), "+v"(v[5][Q0 + 2]), "+v"(v[6][Q0 + 0]), "+v"(v[6][Q0 + 1]), "+v"(v[6][Q0 + 2]), "+v"(v[7][Q0 + 0]), "+v"(v[7][Q0 + 1]), "+v"(v[7][Q0 + 2])
      : "v"(u), "v"(nl[Q0 + 0]), "v"(nl[Q0 + 1]), "v"(nl[Q0 + 2]), "s"(j)
      : "scc");
}
template <int Q0>
__device__ __forceinline__ void fma_turn3(float (&v)[kLeafMax][3], float u,
                                          const float (&nl)[3], int j) {
  asm("s_nop 1\n\t"
      "s_cmp_gt_u32 %25, 6\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %0, %21, %22 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %21, %23 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %21, %24 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 5\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %3, %21, %22 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %4, %21, %23 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %5, %21, %24 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 4\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %6, %21, %22 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %7, %21, %23 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %8, %21, %24 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 3\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %9, %21, %22 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %10, %21, %23 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %11, %21, %24 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 2\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %12, %21, %22 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %13, %21, %23 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %14, %21, %24 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 1\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %15, %21, %22 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %16, %21, %23 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %17, %21, %24 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "s_cmp_gt_u32 %25, 0\n\ts_cbranch_scc1 .Lleaf%=\n\t"
      "v_fmac_f32_dpp %18, %21, %22 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %19, %21, %23 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %20, %21, %24 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      ".Lleaf%=:"
      : "+v"(v[1][Q0 + 0]), "+v"(v[1][Q0 + 1]), "+v"(v[1][Q0 + 2]), "+v"(v[2][Q0 + 0]), "+v"(v[2][Q0 + 1]), "+v"(v[2][Q0 + 2]), "+v"(v[3][Q0 + 0]), "+v"(v[3][Q0 + 1]), "+v"(v[3][Q0 + 2]), "+v"(v[4][Q0 + 0]), "+v"(v[4][Q0 + 1]), "+v"(v[4][Q0 + 2]), "+v"(v[5][Q0 + 0]), "+v"(v[5][Q0 + 1]), "+v"(v[5][Q0 + 2]), "+v"(v[6][Q0 + 0]), "+v"(v[6][Q0 + 1]), "+v"(v[6][Q0 + 2]), "+v"(v[7][Q0 + 0]), "+v"(v[7][Q0 + 1]), "+v"(v[7][Q0 + 2])
      : "v"(u), "v"(nl[Q0 + 0]), "v"(nl[Q0 + 1]), "v"(nl[Q0 + 2]), "s"(j)
      : "scc");
}

struct LeafMoves {
  int piv, dst, src;
};

// A column is two halves.  leaf_publish finds the pivot candidate of column jj
// (its values x, the column already updated) and sends it; leaf_receive waits
// for the pivot row, scales the column, and forms the next column's values.
// Between the two, while the exchange is under way, the rank-1 update of the
// column before is applied to the tile (leaf_update) -- so a candidate's row is
// sent without that update and with the row's factor in it, and whoever
// receives it applies it, with the same FMA.  A workgroup by itself (SINGLE)
// has nothing to wait for and updates its tile first.
//
// Tile positions (every register of the tile is addressed statically): column
// jb0 + j, jb0 a multiple of 8, is in position 0; positions [0, 8 - j) hold the
// columns from there on and [8 - j, 8) the j columns finished in this turn;
// [8, act) hold the unfinished columns of the next turns.  leaf_update leaves
// the tile arranged for the next column.
//
// lab: the labels of the thread's rows, -1 for a row that is finished or
// outside the panel, whose registers may then hold anything.  nl: minus the rows'
// factors in the last update.  dst: lane i >= 32 the label of the row loaded
// from row c0 + i - 32 (-1 once it is a pivot row); src: lane i < 32 the row
// that the pivot row of column i was loaded from; piv: lane i < 32 its label
// then.
template <typename T, int NT, int RPT, bool SINGLE>
__device__ __forceinline__ void leaf_publish(const LeafArgs& a,
                                             const T (&v)[kLeafMax][RPT],
                                             const T (&x)[RPT], const T (&nl)[RPT],
                                             const int (&lab)[RPT],
                                             LeafShared<T>& sh, int jj) {
  constexpr int NW   = NT / 64;
  const int     t    = threadIdx.x;
  const int     lane = t & 63;
  const int     wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int     b    = blockIdx.x;
  const int     par  = jj & 1;
  const int     gc   = a.c0 + jj;  // current top row == current column
  // ---- step 1: candidate max |a(r, gc)| over the labels left, first by the
  // upper halves alone
  uint32_t k[RPT], top = 0;
#pragma unroll
  for(int q = 0; q < RPT; ++q) {
    k[q] = lab[q] >= 0 ? hi_bits(x[q]) & 0x7fffffffu : 0u;
    top  = k[q] > top ? k[q] : top;
  }
  top = wave_max(top);
  uint32_t kl = 0;
  int      kb = INT_MAX, kq = 0, hits = 0;
  unsigned long long at = 0;
#pragma unroll
  for(int q = RPT - 1; q >= 0; --q) {
    const bool               is = k[q] == top;
    const unsigned long long w  = __ballot(is);
    hits += __builtin_popcountll(w);
    at |= w;
    kl = is ? lo_bits(x[q]) : kl;
    kb = is ? lab[q] : kb;
    kq = is ? q : kq;
  }
  int owner;
  top += kKeyBase;
  if(hits == 1 && top < kInfBits<T> + kKeyBase) {
    owner = __builtin_ctzll(at);
  } else {
    // ties, an infinity, a NaN, a zero column or no row: the exact order
    uint32_t kh = 0;
    kl          = 0;
    kb          = INT_MAX;
    kq          = 0;
#pragma unroll
    for(int q = 0; q < RPT; ++q) {
      const T    y   = x[q];
      const bool nan = !(y == y);
      uint32_t   h   = (hi_bits(y) & 0x7fffffffu) + kKeyBase, l = lo_bits(y);
      if(nan) {
        h = lab[q] == gc ? kKeyTopNan : 0;
        l = 0;
      }
      if(lab[q] >= 0 && h > 0 &&
         (h > kh || (h == kh && (l > kl || (l == kl && lab[q] < kb))))) {
        kh = h;
        kl = l;
        kb = lab[q];
        kq = q;
      }
    }
    top   = wave_max(kh);
    owner = first_of(__ballot(kh == top), top, kl, kb);
  }
  const uint32_t wlo = readlane(kl, owner);
  const int      wlb = readlane(kb, owner);
  kq                 = readlane(kq, owner);
  if(lane == 0) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<u4*>(sh.wave[par][wave]) =
        u4{top, wlo, static_cast<uint32_t>(wlb), 0u};
  }
  __syncthreads();
  // sh.wave of this parity is written again two barriers on
  const uint32_t ch = sh.wave[par][lane & (NW - 1)][0];
  const uint32_t cl = sh.wave[par][lane & (NW - 1)][1];
  const int      cb = static_cast<int>(sh.wave[par][lane & (NW - 1)][2]);
  top               = readlane(row_max(ch), 0);
  const int ww = first_of(__ballot(ch == top) & ((1u << NW) - 1), top, cl, cb);
  const int lb = readlane(cb, ww);
  // the row that workgroup candidate was loaded from
  const int CH  = NT * RPT;
  int       org = a.c0 + b * CH + kq * NT + wave * 64 + owner;
  // ---- the candidate row, by its wave
  if(wave == ww && lb != INT_MAX && lane == owner) {
    // as the tile will be arranged for this column
    const bool turn  = (jj & (kTurn - 1)) == 0;
    T* const   first = sh.row[par] + (turn ? kLeafMax - kTurn : 0);
    T* const   rest  = sh.row[par] - (turn ? kTurn : 0);
#pragma unroll
    for(int q = 0; q < RPT; ++q)
      if(kq == q) {
        if constexpr(SINGLE) {
#pragma unroll
          for(int c = 0; c < kLeafMax; ++c) sh.row[par][c] = v[c][q];
        } else {
#pragma unroll
          for(int c = 0; c < kTurn; ++c) first[(c - 1) & (kTurn - 1)] = v[c][q];
#pragma unroll
          for(int c = kTurn; c < kLeafMax; ++c) rest[c] = v[c][q];
          sh.nl[par] = nl[q];
        }
        // keeps the cases apart: merged, they would index the tile by kq
        asm volatile("; row %0" : : "n"(q));
      }
    if constexpr(SINGLE) {
      sh.sel[0] = lb;
      sh.sel[1] = org;
    }
  }
  if constexpr(SINGLE) return;
  // A workgroup without rows left publishes an empty candidate (key 0, label
  // INT_MAX).
  if(wave == ww) {
    const uint32_t      seq  = a.seq_base + jj + 1;
    unsigned long long* mine = reinterpret_cast<unsigned long long*>(a.slots) +
                               (static_cast<size_t>(par) * (kMaxGrid + 1) + b) * kSlotStride;
    // the wave's lanes see its own LDS stores in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint32_t* half = reinterpret_cast<const uint32_t*>(sh.row[par]);
    const uint32_t* fact = reinterpret_cast<const uint32_t*>(&sh.nl[par]);
    st_word(mine + word_of<T>(lane), seq, half[word_of<T>(lane)]);
    if(lane < kHeadWords)
      st_word(mine + kSlotHead + lane, seq,
              lane == 0   ? top
              : lane == 1 ? wlo
              : lane == 2 ? static_cast<uint32_t>(lb)
              : lane == 3 ? static_cast<uint32_t>(org)
                          : fact[sizeof(T) == 8 ? lane - 4 : 0]);
  }
}

// False if the grid has to stop.
template <typename T, int NT, int RPT, bool SINGLE>
__device__ __forceinline__ bool leaf_receive(const LeafArgs& a, T (&v)[kLeafMax][RPT],
                                             T (&x)[RPT], T (&nl)[RPT], int (&lab)[RPT],
                                             LeafShared<T>& sh, LeafMoves& mv, int& zero,
                                             int jj) {
  constexpr int NW   = NT / 64;
  const int     t    = threadIdx.x;
  const int     lane = t & 63;
  const int     wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int     b    = blockIdx.x;
  const int     jb0 = jj & ~(kTurn - 1), j = jj & (kTurn - 1), par = j & 1;
  const int     gc = a.c0 + jj;
  int       p, po;  // the pivot's label, the row it was loaded from
  uint32_t  nlo = 0, nhi = 0;
  const T*  urow;
  if constexpr(SINGLE) {
    __syncthreads();
    p    = sh.sel[0];
    po   = sh.sel[1];
    urow = sh.row[par];
  } else {
    const uint32_t            seq = a.seq_base + jj + 1;
    const unsigned long long* slots =
        reinterpret_cast<const unsigned long long*>(a.slots) +
        static_cast<size_t>(par) * (kMaxGrid + 1) * kSlotStride;
    const bool near = a.grid <= kNear;
    if(near ? !gather_all<T, NW>(a, slots, seq, sh)
            : wave == 0 && !gather_pivot<T>(a, slots, seq, sh))
      sh.ok = 0;
    __syncthreads();
    if(!sh.ok) return false;
    if(near) {  // every wave picks the pivot itself
      uint32_t gh = 0, go = 0;
      int      gl = INT_MAX;
      if(lane < a.grid) {
        gh = sh.head[lane][0];
        go = sh.head[lane][1];
        gl = static_cast<int>(sh.head[lane][2]);
      }
      const uint32_t top = wave_max(gh);
      const int g = first_of(__ballot(gh == top) & ((1ull << a.grid) - 1), top, go, gl);
      p           = readlane(gl, g);
      po          = static_cast<int>(sh.head[g][3]);
      nlo         = sh.head[g][4];
      nhi         = sh.head[g][5];
      urow        = sh.cand[g];
    } else {
      p    = sh.sel[0];
      po   = sh.sel[1];
      nlo  = sh.sel_nl[0];
      nhi  = sh.sel_nl[1];
      urow = sh.cand[0];
    }
  }
  p  = __builtin_amdgcn_readfirstlane(p);
  po = __builtin_amdgcn_readfirstlane(po);
  // the pivot row's positions c and 16 + c
  const int c  = lane & 15;
  T         u0 = urow[c], u1 = urow[16 + c];
  if constexpr(!SINGLE) {
    // with the update it lacks: that of the column before, which is not
    // finished in positions [0, 8 - j) of this turn and [8, act)
    const int act = (a.w + kTurn - 1) / kTurn * kTurn - jb0;
    const T   pnl = from_halves(nlo, nhi, T(0));
    const T   c0 = sh.ucur[par ^ 1][1][c], c1 = sh.ucur[par ^ 1][1][16 + c];
    if(jj > 0) {
      u0 = c < kTurn - j || (c >= kTurn && c < act) ? fma(c0, pnl, u0) : u0;
      u1 = 16 + c < act ? fma(c1, pnl, u1) : u1;
    }
    // for later, each copy by a wave of its own; read after the next column's
    // barriers
    if(lane < 16) {
      if(wave == 2) {
        sh.ucur[par][0][c]      = u0;
        sh.ucur[par][0][16 + c] = u1;
      }
      if(wave == 3) {
        const bool turn = j == kTurn - 1;
        sh.ucur[par][1][c < kTurn ? ((c - 1) & (kTurn - 1)) + (turn ? kLeafMax - kTurn : 0)
                                  : c - (turn ? kTurn : 0)] = u0;
        sh.ucur[par][1][16 + c - (turn ? kTurn : 0)]        = u1;
      }
    }
  }
  if(b == 0 && wave == 1 && lane < 16) {
    sh.fin[jj][c < kTurn ? jb0 + ((c + j) & (kTurn - 1)) : (c + jb0) & (kLeafMax - 1)] = u0;
    sh.fin[jj][(c + 16 + jb0) & (kLeafMax - 1)] = u1;
  }
  const T piv = readlane(u0, 0);
  if(piv == T(0) && zero < 0) zero = jj;
  // interchange rows gc and p (the pivot row is finished), scale
  mv.piv = lane == jj ? p : mv.piv;
  mv.src = lane == jj ? po : mv.src;
  mv.dst = mv.dst == p ? -1 : mv.dst == gc ? p : mv.dst;
#pragma unroll
  for(int q = 0; q < RPT; ++q) {
    lab[q] = lab[q] == p ? -1 : lab[q] == gc ? p : lab[q];
    if(piv != T(0)) v[0][q] = v[0][q] / piv;
    nl[q] = -v[0][q];
  }
  if constexpr(!SINGLE) {  // the next column, updated
    const T un = readlane(u0, j < kTurn - 1 ? 1 : kTurn);
#pragma unroll
    for(int q = 0; q < RPT; ++q)
      x[q] = fma(un, nl[q], j < kTurn - 1 ? v[1][q] : v[kTurn][q]);
  }
  // sh.cand / sh.row are rewritten only after later barriers, which every
  // wave reaches after its reads here
  return true;
}

// The turn's positions 0 .. 7 rotated by one.
template <typename T, int RPT>
__device__ __forceinline__ void rotate_turn(T (&v)[kLeafMax][RPT]) {
#pragma unroll
  for(int q = 0; q < RPT; ++q)
    rotate8(v[0][q], v[1][q], v[2][q], v[3][q], v[4][q],
            v[5][q], v[6][q], v[7][q]);
}

// The next turn's columns come to the front, the finished ones go to the end.
template <typename T, int RPT>
__device__ __forceinline__ void rotate_turns(T (&v)[kLeafMax][RPT]) {
#pragma unroll
  for(int i = 0; i < kTurn; ++i)
#pragma unroll
    for(int q = 0; q < RPT; ++q)
      rotate4(v[i][q], v[i + 8][q], v[i + 16][q], v[i + 24][q]);
}

// The rank-1 update of column jj (none before column 0), and the arrangement
// for the next column.
template <typename T, int RPT, bool SINGLE>
__device__ __forceinline__ void leaf_update(T (&v)[kLeafMax][RPT], const T (&nl)[RPT],
                                            const LeafShared<T>& sh, int w, int jj) {
  // the pivot row's positions 0..15 / 16..31, in every 16 lanes
  const int lane = threadIdx.x & 15;
  const T*  u    = SINGLE ? sh.row[jj & 1] : sh.ucur[jj & 1][0];
  const T   u0 = u[lane], u1 = u[16 + lane];
  const int j   = __builtin_amdgcn_readfirstlane(jj & (kTurn - 1));
  const int act = (w + kTurn - 1) / kTurn * kTurn - (jj & ~(kTurn - 1));
  if(jj >= 0) {
    if constexpr(RPT == 1) {
      fma_turn1<0>(v, u0, nl, j);
      if(act > 8) fma_group1<8, 0>(v, u0, nl);
      if(act > 16) fma_group1<16, 0>(v, u1, nl);
      if(act > 24) fma_group1<24, 0>(v, u1, nl);
    } else {
      fma_turn3<0>(v, u0, nl, j);
      if(act > 8) fma_group3<8, 0>(v, u0, nl);
      if(act > 16) fma_group3<16, 0>(v, u1, nl);
      if(act > 24) fma_group3<24, 0>(v, u1, nl);
    }
  }
  rotate_turn(v);
  if(j == kTurn - 1) rotate_turns(v);
}

// One leaf on workgroups 0 .. a.grid-1 of NT threads, RPT rows each: the
// body of leaf_kernel, also run by the persistent panel kernel
// (k_panel_kernel.hip) once per leaf.  Workgroups whose rows all lie at or
// below a.m take part in every exchange with an empty candidate.
template <typename T, typename S, int NT, int RPT, bool SINGLE>
__device__ __forceinline__ void leaf_run(const LeafArgs& a, LeafShared<T>& sh) {
  constexpr int NW   = NT / 64;
  constexpr int CH   = NT * RPT;  // rows per workgroup
  const int     t    = threadIdx.x;
  const int     lane = t & 63;
  const int     wave = t >> 6;
  const int     b    = blockIdx.x;
  const int     G    = a.grid;
  S*            P    = static_cast<S*>(a.P);

  int          lab[RPT];  // the row each slot stands for; -1: none
  T            v[kLeafMax][RPT];
#pragma unroll
  for(int q = 0; q < RPT; ++q) {
    const int row = a.c0 + b * CH + q * NT + t;
    lab[q]        = row < a.m ? row : -1;
  }
  // arranged as if the column before the first had ended a turn
#pragma unroll
  for(int c = 0; c < kLeafMax; ++c) {
    const S*  col = P + static_cast<size_t>(a.c0 + c) * a.lda;
    const int p   = (c + kTurn) & (kLeafMax - 1);
    const int pos = p < kTurn ? (p + 1) & (kTurn - 1) : p;
#pragma unroll
    for(int q = 0; q < RPT; ++q)
      v[pos][q] = (c < a.w && lab[q] >= 0)
                       ? load_s<T, S>(col + static_cast<unsigned>(lab[q]))
                       : T(0);
  }
  if(t == 0) sh.ok = 1;
  // every row has been read before any candidate of it is published, and so
  // before any workgroup stores a row
  wait_vm<0>();

  LeafMoves mv;
  mv.piv   = 0;
  mv.src   = a.c0 + (lane & (kLeafMax - 1));
  mv.dst   = lane < kLeafMax ? -2 : mv.src;
  int zero = -1;  // the first column with a zero pivot
  T   x[RPT], nl[RPT];
#pragma unroll
  for(int q = 0; q < RPT; ++q) {
    x[q]  = v[kTurn][q];  // column 0
    nl[q] = T(0);
  }
#pragma unroll 1
  for(int jj = 0; jj < a.w; ++jj) {
    if constexpr(SINGLE) {
      leaf_update<T, RPT, true>(v, nl, sh, a.w, jj - 1);
      leaf_publish<T, NT, RPT, true>(a, v, v[0], nl, lab, sh, jj);
      leaf_receive<T, NT, RPT, true>(a, v, x, nl, lab, sh, mv, zero, jj);
    } else {
      leaf_publish<T, NT, RPT, false>(a, v, x, nl, lab, sh, jj);
      leaf_update<T, RPT, false>(v, nl, sh, a.w, jj - 1);
      if(!leaf_receive<T, NT, RPT, false>(a, v, x, nl, lab, sh, mv, zero, jj)) return;
    }
  }
  // the last turn to its end
#pragma unroll 1
  for(int j = (a.w - 1) & (kTurn - 1); j < kTurn; ++j) rotate_turn(v);
  rotate_turns(v);
  const int jb0 = (a.w + kTurn - 1) & ~(kTurn - 1);

  // ---- write the leaf back: the rows below where their labels say, the
  // finished top rows by workgroup 0
#pragma unroll
  for(int c = 0; c < kLeafMax; ++c) {
    const int cc = (c + jb0) & (kLeafMax - 1);  // the column position c holds
    if(cc < a.w) {
      S* col = P + static_cast<size_t>(a.c0 + cc) * a.lda;
#pragma unroll
      for(int q = 0; q < RPT; ++q)
        if(lab[q] >= 0)
          store_s<T, S>(col + static_cast<unsigned>(lab[q]), v[c][q]);
    }
  }
  if(b == 0) {
    __syncthreads();  // sh.fin
    const int r = t & (kLeafMax - 1);
    if(r < a.w)
      for(int c = t / kLeafMax; c < a.w; c += NT / kLeafMax)
        store_s<T, S>(P + a.c0 + r + static_cast<size_t>(a.c0 + c) * a.lda,
                      sh.fin[r][c]);
    if(t < a.w) a.ipiv[a.c0 + t] = mv.piv + a.row_offset;
    if(t == 0 && zero >= 0 && *a.info == 0)
      *a.info = a.info_base + a.c0 + zero + 1;
  }

  // ---- apply the leaf's moves to the other panel columns
  const int others = a.JB - a.w;
  const int dst    = lane < kLeafMax ? a.c0 + lane : mv.dst;
  if(dst >= 0 && dst != mv.src) {
    // a wave takes columns idx, idx + stride, ...; each column's sources are
    // all loaded (one instruction) before any of its destinations is stored,
    // and kBatch columns are in flight at once
    constexpr int kBatch = 8;
    const int     stride = G * NW;
    for(int idx0 = b * NW + wave; idx0 < others; idx0 += kBatch * stride) {
      S x[kBatch];
#pragma unroll
      for(int u = 0; u < kBatch; ++u) {
        const int idx = idx0 + u * stride;
        const int c   = idx < a.c0 ? idx : idx + a.w;
        if(idx < others) x[u] = P[mv.src + static_cast<size_t>(c) * a.lda];
      }
#pragma unroll
      for(int u = 0; u < kBatch; ++u) {
        const int idx = idx0 + u * stride;
        const int c   = idx < a.c0 ? idx : idx + a.w;
        if(idx < others) P[dst + static_cast<size_t>(c) * a.lda] = x[u];
      }
    }
  }
}

// Bound by latency: per column one workgroup-wide and one grid-wide exchange
// and the issue of about 150 (one row per thread) or 290 instructions, of which
// the update's and the arrangement's run beside the exchange; HBM traffic is
// one read and one write of the leaf.  Time of a 32-column leaf of m rows, us,
// FP64 (FP32): with the leaf unrolled / with the update before the exchange /
// now:
//   m = 500 131 (128) / 45 (39) / 43 (41), 1500 160 (158) / 68 (60) / 65 (56),
//   4000 222 (216) / 99 (87) / 90 (84), 16000 246 (239) / 112 (102) / 100 (91),
//   65000 276 (270) / 135 (126) / 134 (115),
//   131072 318 (320) / 154 (148) / 151 (127).
template <typename T, typename S, int NT, int RPT, bool SINGLE>
__global__ __launch_bounds__(NT) void leaf_kernel(LeafArgs a) {
  __shared__ LeafShared<T> sh;
  if(__hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    return;
  leaf_run<T, S, NT, RPT, SINGLE>(a, sh);
}

}  // namespace leaf

// Kernel entry of the FP64 or FP32 leaf with rpt (1 or kLeafRPT) rows per
// thread, for one workgroup (single) or several (defined in k_leaf*.hip).
template <typename T>
const void* leaf_kernel_ptr(int rpt, bool single);

}  // namespace hplx
