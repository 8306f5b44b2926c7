// RMSNorm of x[rows, cols] over cols for bf16 (dtype 1) and fp16 (dtype 2) rows, behind the reference's C-ABI `launch`
// (rmsnorm/kernel.cu:132-139) plus a weighted entry `rmsnorm_launch_weighted`.
//
// Per row (rmsnorm/kernel.cu:1-8, rmsnorm/candidate.py:3-4):
//   sum  = sum of x^2                                   (each square is exact in fp32 for a 2-byte format)
//   inv  = T(rsqrt(float(sum) / cols + eps))            (fp32 mean and eps, rsqrt rounded to x's dtype)
//   y    = T(x * inv)                                   (one round to nearest even; the product is exact in fp32)
//   y    = T(w * y)                                     (weighted entry only: torch's `w * y` on dtype tensors)
// The fused residual entry (`rmsnorm_add_launch`) first forms h = T(x + residual), writes it to residual_out and
// normalizes h as above: torch's `h = x + residual; y = rmsnorm(h)` on dtype tensors, one pass over memory.
// The squares are summed in fp64, which makes the sum exact to far below fp32 resolution, so float(sum) is the
// correctly rounded fp32 sum and does not depend on the summation order; rsqrt is evaluated in fp64 and rounded to
// fp32 (the correctly rounded fp32 rsqrt). The reference's fp32 sum and rsqrtf are within an fp32 ulp or two of these
// values; the result differs from it only where that ulp moves inv across a rounding boundary of the dtype. A NaN in a
// row makes the row NaN and a sum beyond the fp32 range makes inv 0, as in the reference.
//
// Rows whose length is a multiple of 8 with 16-byte aligned x, y (and w) run the row kernel: a group of WAVES waves
// holds one row in registers as NV 16-byte vectors per lane, reduces the sum over the group (DPP within a wave, LDS
// slots across waves) and writes y from the registers; each lane holds the weight vectors of its columns once for all
// rows. Workgroups are persistent and load their next row while they reduce and store the current one. Rows of any
// other length from 8 columns up, or otherwise aligned, run the same kernel with element-aligned vectors (Form kAny);
// aligned rows of at most 32 vectors share waves, four at a time, when there are many of them (rmsnorm_short). What is
// left (rows of fewer than 8 columns, or longer than 16 waves hold) takes a generic kernel (one workgroup per row,
// scalar accesses, two passes).
#include <climits>
#include <cmath>
#include <type_traits>

#include "host.hpp"
#include "rowwise.hpp"

using namespace rw;

namespace {

constexpr int kMaxNv = 8;
constexpr int kMaxWaves = 16;

template <int NV>
struct Regs {
  u32x4 v[NV];
};

// How rows lie under a group's vectors: kFull, as many aligned vectors as the group holds; kPart, fewer; kAny, rows of
// any length (at least a vector) at any element alignment: the row's last vector is moved back to end with the row, its
// first elements being another lane's (the same bits, and the same results when they are stored twice).
enum Form { kPart = 0, kFull = 1, kAny = 2 };

// The lane's place in its rows. Lane t of the group's G holds vectors t, t + G, ..., clamped into the row.
template <int FORM, int G>
struct Place {
  static constexpr int V = 8;
  long long nvec;
  int cols, t;
  int wave0;  // the wave's first lane in the group: wave-uniform
  // whether vector k holds elements of the row in some lane of the wave, and (kAny) whole vectors of them in every lane
  __device__ __forceinline__ bool used(int k) const { return FORM == kFull || (long long)k * G + wave0 < nvec; }
  __device__ __forceinline__ bool whole(int k) const { return (k * G + wave0 + kWave) * V <= cols; }
  __device__ __forceinline__ int start(int k) const { return (k * G + t) * V; }  // vector k's first element
  __device__ __forceinline__ bool in(int k) const {
    return FORM == kFull || (FORM == kAny ? start(k) < cols : (long long)k * G + t < nvec);
  }
  __device__ __forceinline__ uint32_t any_at(int k) const { return (uint32_t)least(start(k), cols - V) * 2u; }  // bytes
  // the first elements of vector k that are another lane's
  __device__ __forceinline__ int skip(int k) const { return start(k) - least(start(k), cols - V); }

  template <bool NTL>
  __device__ __forceinline__ u32x4 load(const void* base, long long row, int k) const {
    if constexpr (FORM == kAny) {
      return load16_at<NTL>(static_cast<const char*>(base) + row * cols * 2, any_at(k));
    } else {
      long long i = (long long)k * G + t;
      if constexpr (FORM == kPart) i = i < nvec ? i : nvec - 1;
      return load16<NTL>(base, row * nvec + i);
    }
  }
  template <bool NTS>
  __device__ __forceinline__ void store(void* base, long long row, int k, const u32x4& v) const {
    if constexpr (FORM == kAny) store16_at<NTS>(static_cast<char*>(base) + row * cols * 2, any_at(k), v);
    else store16<NTS>(base, row * nvec + (long long)k * G + t, v);
  }
};

template <int FORM, int G, int NV, bool NTL>
__device__ __forceinline__ void load_vectors(Regs<NV>& r, const void* base, long long row, const Place<FORM, G>& at) {
#pragma unroll
  for (int k = 0; k < NV; ++k) r.v[k] = at.template load<NTL>(base, row, k);
}

// inv from the exact sum of squares: fp32 mean and eps as the reference, rsqrt correctly rounded to fp32, then to T.
template <typename T>
__device__ __forceinline__ float row_inv(double sum, int cols, float eps) {
  const float mean = (float)sum / (float)cols;
  const float v = mean + eps;
  const float inv32 = (float)(1.0 / sqrt((double)v));
  return round_to<T>(inv32);
}

// Keeps a product apart from its rounding to fp16 (fused into one mixed-precision multiply-add with +0, a product of -0
// comes out as +0).
template <typename T>
__device__ __forceinline__ void apart(float& v) {
  if constexpr (std::is_same<T, F16>::value) asm volatile("" : "+v"(v));
}

// Whether vectors past the row's end for the whole wave are passed over: 16384 x 5120 bf16 64.2 -> 62.3 us, with a
// residual 1% slower; 64 x 640, whose lanes hold two vectors, 2.28 -> 2.37.
template <int FORM, int NV, bool RES> constexpr bool kSkips = FORM == kAny || (FORM == kPart && !RES && NV >= 4);

template <typename T, int WAVES, int NV, int FORM, bool HAS_W, bool RES, bool NTS>
__device__ __forceinline__ void norm_row(const Regs<NV>& r, const Regs<NV>& w, void* y, void* res_out, long long row,
                                         const Place<FORM, WAVES * kWave>& at, float eps, bool active, double* slots,
                                         int wave, int first) {
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    if (kSkips<FORM, NV, RES> && !at.used(k)) continue;
    float f[T::V];
    unpack<T>(r.v[k], f);
    if (FORM == kAny && !at.whole(k)) {
      const int skip = at.skip(k);
#pragma unroll
      for (int i = 0; i < T::V; ++i) acc += i >= skip ? (double)(f[i] * f[i]) : 0.0;
    } else {
      const bool ok = FORM == kAny || at.in(k);
#pragma unroll
      for (int i = 0; i < T::V; ++i) acc += ok ? (double)(f[i] * f[i]) : 0.0;
    }
  }
  acc = group_reduce<WAVES>(acc, OpSum{}, slots, wave, first);
  const float inv = row_inv<T>(acc, at.cols, eps);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    if (active && at.in(k)) {
      // (kAny: h is stored only here, behind the reduction, which every wave reaches with its vectors loaded: in place,
      // a vector moved back at the row's end reads elements that another wave writes)
      if constexpr (RES && FORM == kAny) at.template store<NTS>(res_out, row, k, r.v[k]);
      float f[T::V];
      unpack<T>(r.v[k], f);
#pragma unroll
      for (int e = 0; e < T::V; ++e) {
        f[e] = f[e] * inv;
        apart<T>(f[e]);
      }
      if constexpr (HAS_W) {
        float g[T::V];
        unpack<T>(w.v[k], g);
#pragma unroll
        for (int e = 0; e < T::V; ++e) {
          f[e] = g[e] * round_to<T>(f[e]);
          apart<T>(f[e]);
        }
      }
      at.template store<NTS>(y, row, k, pack<T>(f));
    }
  }
}

// Fused residual: r becomes h = T(x + residual), which is written to res_out (the lane's own vectors: res_out may be
// residual, and y may be x; kAny rows are written by norm_row).
template <typename T, int FORM, int G, int NV, bool NTS>
__device__ __forceinline__ void add_residual(Regs<NV>& r, const Regs<NV>& res, void* res_out, long long row,
                                             const Place<FORM, G>& at, bool active) {
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    if (FORM == kAny && !at.used(k)) continue;
    float a[T::V], b[T::V];
    unpack<T>(r.v[k], a);
    unpack<T>(res.v[k], b);
#pragma unroll
    for (int e = 0; e < T::V; ++e) a[e] = a[e] + b[e];
    r.v[k] = pack<T>(a);
    if (FORM != kAny && active && at.in(k)) at.template store<NTS>(res_out, row, k, r.v[k]);
  }
}

// Row kernel. A block is max(WAVES, 4) waves; GROUPS = block waves / WAVES groups walk their own rows with a uniform
// trip count (a group past the last row loads an in-bounds row and stores nothing). Two LDS slot arrays alternate
// between consecutive rows, so a slot is never rewritten before the barrier of the next reduction.
// With RES the group also loads the residual rows, forms h = T(x + residual) and writes it to res_out before the
// normalisation (x and y, and residual and res_out, may be the same buffers: a lane reads its vectors before it
// writes them).
template <typename T, int WAVES, int NV, int FORM, bool HAS_W, bool RES, bool NTL, bool NTS>
__global__ void __launch_bounds__((WAVES < 4 ? 4 : WAVES) * 64)
    rmsnorm_rows(const void* x, const void* res, const void* __restrict__ w, void* y, void* res_out, long long rows,
                 long long nvec, int cols, float eps) {
  constexpr int BW = WAVES < 4 ? 4 : WAVES;
  constexpr int GROUPS = BW / WAVES;
  constexpr int G = WAVES * kWave;
  __shared__ double slots[2][BW];
  const int wave = kSkips<FORM, NV, RES> ? __builtin_amdgcn_readfirstlane(wave_id()) : wave_id();
  const int first = (wave / WAVES) * WAVES;
  const Place<FORM, G> at{nvec, cols, (int)threadIdx.x - first * kWave, (wave - first) * kWave};
  const long long step = (long long)gridDim.x * GROUPS;
  long long base = (long long)blockIdx.x * GROUPS;
  if (base >= rows) return;
  const long long last = rows - 1;
  Regs<NV> wr;
  if constexpr (HAS_W) load_vectors<FORM, G, NV, false>(wr, w, 0, at);
  long long ra = base + wave / WAVES;
  Regs<NV> a, b;
  Regs<RES ? NV : 1> ea, eb;  // residual rows
  load_vectors<FORM, G, NV, NTL>(a, x, ra < rows ? ra : last, at);
  if constexpr (RES) load_vectors<FORM, G, NV, NTL>(ea, res, ra < rows ? ra : last, at);
  while (true) {
    const long long rb = ra + step;
    load_vectors<FORM, G, NV, NTL>(b, x, rb < rows ? rb : last, at);
    if constexpr (RES) {
      load_vectors<FORM, G, NV, NTL>(eb, res, rb < rows ? rb : last, at);
      add_residual<T, FORM, G, NV, NTS>(a, ea, res_out, ra, at, ra < rows);
    }
    norm_row<T, WAVES, NV, FORM, HAS_W, RES, NTS>(a, wr, y, res_out, ra, at, eps, ra < rows, slots[0], wave, first);
    base += step;
    if (base >= rows) break;
    ra = rb;
    const long long rc = ra + step;
    load_vectors<FORM, G, NV, NTL>(a, x, rc < rows ? rc : last, at);
    if constexpr (RES) {
      load_vectors<FORM, G, NV, NTL>(ea, res, rc < rows ? rc : last, at);
      add_residual<T, FORM, G, NV, NTS>(b, eb, res_out, ra, at, ra < rows);
    }
    norm_row<T, WAVES, NV, FORM, HAS_W, RES, NTS>(b, wr, y, res_out, ra, at, eps, ra < rows, slots[1], wave, first);
    base += step;
    if (base >= rows) break;
    ra = rc;
  }
}

// Short rows (at most 32 vectors: the norm of each query or key head): 16 lanes hold a row, NV vectors per lane, and a
// wave takes kShortSets sets of four rows at once, so that every lane holds data, and the row factor's chain (fp64
// square root and divisions, about 100 instructions) runs once per wave for all sixteen rows: the reduction over a
// row's lanes first trades the four sets within each quad of lanes (two steps that halve the values a lane holds),
// which leaves set q's sum in the lanes with lane % 4 == q, and every lane reads its sets' factors back from its quad.
// Waves are persistent and load their next sixteen rows while they work on these; no LDS and no barrier. Bound by
// memory at 128 columns, by instruction issue below.
// 163840 x 128 bf16 with a weight: 62.9 us as a wave per row with 16 of 64 lanes holding data, 16 us here.
constexpr int kShortLanes = 16, kShortSets = 4;
constexpr int kShortRows = kShortSets * (kWave / kShortLanes);  // a wave's rows per step
constexpr int kDppRor4 = 0x124, kDppRor8 = 0x128;               // row_ror: rotation within a 16-lane row

// The sum over each 16-lane row of every set's value, for the set lane % 4.
__device__ __forceinline__ double short_sums(const double (&a)[kShortSets], int lane) {
  static_assert(kShortSets == 4, "two trading steps");
  const bool odd = lane & 1, upper = lane & 2;
  const double e = (odd ? a[1] : a[0]) + dpp<kDppXor1>(odd ? a[0] : a[1]);
  const double f = (odd ? a[3] : a[2]) + dpp<kDppXor1>(odd ? a[2] : a[3]);
  double s = (upper ? f : e) + dpp<kDppXor2>(upper ? e : f);
  s += dpp<kDppRor4>(s);
  return s + dpp<kDppRor8>(s);
}

template <typename T, int NV, bool HAS_W>
__global__ void __launch_bounds__(256)
    rmsnorm_short(const void* x, const void* __restrict__ w, void* y, long long rows, int nvec, int cols, float eps) {
  const int lane = lane_id(), l = lane & (kShortLanes - 1), sub = lane / kShortLanes;
  const int per_block = (int)blockDim.x / kWave;
  const long long wave = (long long)blockIdx.x * per_block + __builtin_amdgcn_readfirstlane(wave_id());
  const long long step = (long long)gridDim.x * per_block * kShortRows;
  u32x4 wr[HAS_W ? NV : 1];
  if constexpr (HAS_W) {
#pragma unroll
    for (int k = 0; k < NV; ++k) wr[k] = load16<false>(w, least(k * kShortLanes + l, nvec - 1));
  }
  struct Step {
    u32x4 v[kShortSets][NV];
  };
  // vector k of the lane's row of set u, of the sixteen rows from `first` on; a row past the last and a vector past the
  // row's end are clamped (and not stored)
  auto at = [&](long long first, int u, int k) __attribute__((always_inline)) {
    const long long left = rows - 1 - first;
    const int r = u * (kWave / kShortLanes) + sub;
    return (uint32_t)((left < r ? (int)left : r) * nvec + least(k * kShortLanes + l, nvec - 1));
  };
  auto load = [&](Step& s, long long first) __attribute__((always_inline)) {
    if (first >= rows) first = rows - 1;
#pragma unroll
    for (int u = 0; u < kShortSets; ++u)
#pragma unroll
      for (int k = 0; k < NV; ++k)
        s.v[u][k] = load16<true>(static_cast<const char*>(x) + first * nvec * 16, at(first, u, k));
  };
  auto work = [&](const Step& s, long long first) __attribute__((always_inline)) {
    double acc[kShortSets];
#pragma unroll
    for (int u = 0; u < kShortSets; ++u) {
      acc[u] = 0.0;
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        float f[T::V];
        unpack<T>(s.v[u][k], f);
        double a = 0.0;
#pragma unroll
        for (int i = 0; i < T::V; ++i) a += (double)(f[i] * f[i]);
        acc[u] += k * kShortLanes + l < nvec ? a : 0.0;
      }
    }
    const float mine = row_inv<T>(short_sums(acc, lane), cols, eps);  // the factor of set lane % 4
    const float inv[kShortSets] = {dpp<0x00>(mine), dpp<0x55>(mine), dpp<0xAA>(mine), dpp<0xFF>(mine)};
#pragma unroll
    for (int u = 0; u < kShortSets; ++u) {
      const bool in = first + u * (kWave / kShortLanes) + sub < rows;
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        if (!in || k * kShortLanes + l >= nvec) continue;
        float f[T::V];
        unpack<T>(s.v[u][k], f);
#pragma unroll
        for (int e = 0; e < T::V; ++e) {
          f[e] = f[e] * inv[u];
          apart<T>(f[e]);
        }
        if constexpr (HAS_W) {
          float g[T::V];
          unpack<T>(wr[k], g);
#pragma unroll
          for (int e = 0; e < T::V; ++e) {
            f[e] = g[e] * round_to<T>(f[e]);
            apart<T>(f[e]);
          }
        }
        store16<true>(static_cast<char*>(y) + first * nvec * 16, at(first, u, k), pack<T>(f));
      }
    }
  };
  long long first = wave * kShortRows;
  if (first >= rows) return;
  Step a, b;
  load(a, first);
  while (true) {
    load(b, first + step);
    work(a, first);
    first += step;
    if (first >= rows) break;
    load(a, first + step);
    work(b, first);
    first += step;
    if (first >= rows) break;
  }
}

// Generic kernel: any row length and alignment, one 256-thread block per row (grid-strided), two scalar passes.
// With RES, pass 1 writes h = T(x + residual) to res_out and pass 2 reads h back (the thread's own elements).
template <typename T, bool HAS_W, bool RES>
__global__ void __launch_bounds__(256)
    rmsnorm_generic(const void* x, const void* res, const void* __restrict__ w, void* y, void* res_out,
                    long long rows, int cols, float eps) {
  __shared__ double slots[2][4];
  const int wave = wave_id();
  int parity = 0;
  const void* src = RES ? (const void*)res_out : x;
  for (long long row = blockIdx.x; row < rows; row += gridDim.x, parity ^= 1) {
    const long long o = row * (long long)cols;
    double acc = 0.0;
    for (int j = threadIdx.x; j < cols; j += 256) {
      float f = load_elem<T>(x, o + j);
      if constexpr (RES) {
        f = round_to<T>(f + load_elem<T>(res, o + j));
        store_elem<T>(res_out, o + j, f);
      }
      acc += (double)(f * f);
    }
    acc = group_reduce<4>(acc, OpSum{}, slots[parity], wave, 0);
    const float inv = row_inv<T>(acc, cols, eps);
    for (int j = threadIdx.x; j < cols; j += 256) {
      float v = load_elem<T>(src, o + j) * inv;
      apart<T>(v);
      if constexpr (HAS_W) {
        v = load_elem<T>(w, j) * round_to<T>(v);
        apart<T>(v);
      }
      store_elem<T>(y, o + j, v);
    }
  }
}

// ---- host side ------------------------------------------------------------------------------------------------------

// Tuning slots (0 = automatic): waves per row, vectors per lane, resident blocks per CU, forced generic kernel (1),
// non-temporal loads (1 on, 2 off), the short rows' kernel for every row it can hold (1) or none (2).
enum { kTuneWaves = 0, kTuneNv = 1, kTuneBlocksPerCu = 2, kTuneGeneric = 3, kTuneNtLoads = 4, kTuneShort = 5 };

int pow2_at_least(long long v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

template <typename Kernel>
int blocks_per_cu(Kernel k, int threads) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, threads, 0) != hipSuccess || n <= 0) {
    (void)hipGetLastError();
    n = 1;
  }
  return n;
}

struct Args {
  const void* x;
  const void* w;
  void* y;
  const void* res;
  void* res_out;
  long long rows;
  long long nvec;
  int cols;
  float eps;
  hipStream_t stream;
  bool any;  // rows of any length and alignment
};

template <typename T, int WAVES, int NV, int FORM, bool HAS_W, bool RES, bool NTL>
int launch_k(const Args& a) {
  constexpr int BW = WAVES < 4 ? 4 : WAVES;
  constexpr int GROUPS = BW / WAVES;
  auto kern = rmsnorm_rows<T, WAVES, NV, FORM, HAS_W, RES, NTL, true>;
  static int occ = 0;
  if (occ <= 0) occ = blocks_per_cu(kern, BW * kWave);
  // about 8 resident waves per CU by default (more waves only contend for the memory queues; measured on MI355X); 32
  // for rows of at most 96 vectors, whose waves hold too little in flight (65536 rows bf16: 264 columns 28.4 -> 20.5
  // us, 512 columns 31.0 -> 24.4, 640 columns 38.1 -> 31.9, but 1024 columns 44.9 -> 47.0)
  int per_cu = rw_host::tune_get(kTuneBlocksPerCu);
  if (per_cu <= 0 && WAVES == 1 && a.nvec <= 96) per_cu = 8;
  if (per_cu <= 0) per_cu = 8 / BW > 1 ? 8 / BW : 1;
  if (per_cu > occ) per_cu = occ;
  const long long need = (a.rows + GROUPS - 1) / GROUPS;
  long long grid = (long long)rw_host::device_cus() * per_cu;
  if (grid > need) grid = need;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(BW * kWave), 0, a.stream, a.x, a.res, a.w, a.y, a.res_out, a.rows,
                     a.nvec, a.cols, a.eps);
  return (int)hipGetLastError();
}

template <typename T, int WAVES, int NV, bool HAS_W, bool RES, bool NTL>
int launch_nv(const Args& a) {
  if constexpr (NTL)  // (the tuning slot that switches it off is for aligned rows)
    if (a.any) return launch_k<T, WAVES, NV, kAny, HAS_W, RES, true>(a);
  if (a.nvec == (long long)WAVES * kWave * NV) return launch_k<T, WAVES, NV, kFull, HAS_W, RES, NTL>(a);
  return launch_k<T, WAVES, NV, kPart, HAS_W, RES, NTL>(a);
}

template <typename T, int WAVES, bool HAS_W, bool RES, bool NTL>
int launch_w(int nv, const Args& a) {
  switch (nv) {
    case 1: return launch_nv<T, WAVES, 1, HAS_W, RES, NTL>(a);
    case 2: return launch_nv<T, WAVES, 2, HAS_W, RES, NTL>(a);
    case 4: return launch_nv<T, WAVES, 4, HAS_W, RES, NTL>(a);
    case 8: return launch_nv<T, WAVES, 8, HAS_W, RES, NTL>(a);
    default: return rw_host::kInvalid;
  }
}

template <typename T, bool HAS_W, bool RES, bool NTL>
int launch_rows(int waves, int nv, const Args& a) {
  switch (waves) {
    case 1: return launch_w<T, 1, HAS_W, RES, NTL>(nv, a);
    case 2: return launch_w<T, 2, HAS_W, RES, NTL>(nv, a);
    case 4: return launch_w<T, 4, HAS_W, RES, NTL>(nv, a);
    case 8: return launch_w<T, 8, HAS_W, RES, NTL>(nv, a);
    case 16: return launch_w<T, 16, HAS_W, RES, NTL>(nv, a);
    default: return rw_host::kInvalid;
  }
}

template <typename T, int NV, bool HAS_W>
int launch_short(const Args& a) {
  auto kern = rmsnorm_short<T, NV, HAS_W>;
  const long long cus = rw_host::device_cus();
  const long long waves = (a.rows + kShortRows - 1) / kShortRows;
  int per_cu = rw_host::tune_get(kTuneBlocksPerCu);
  if (per_cu <= 0) per_cu = 6;  // 24 waves per CU (163840 x 128 bf16: 8 waves 17.0 us, 16 17.4, 24 15.8, 32 16.4)
  // one wave per block until every CU has four: few rows then spread over the GPU
  const int per_block = waves >= 4 * cus ? 4 : 1;
  long long grid = (waves + per_block - 1) / per_block;
  if (grid > cus * per_cu * 4 / per_block) grid = cus * per_cu * 4 / per_block;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(per_block * kWave), 0, a.stream, a.x, a.w, a.y, a.rows,
                     (int)a.nvec, a.cols, a.eps);
  return (int)hipGetLastError();
}

// Whether rows of at most 32 vectors share waves: sixteen of them take longer than the row kernel's one, which few rows
// do not make up for. Kernel times in us, a wave per row / shared: 128 columns bf16 64 rows 2.1 / 2.5, 2048 2.5 / 2.7,
// 3000 2.7 / 2.7, 8192 4.1 / 3.1; 256 columns 64 rows 2.1 / 3.2, 6000 3.7 / 4.0, 8192 4.3 / 4.1, 32768 11.2 / 7.2.
bool takes_short(long long rows, long long nvec) {
  const int want = rw_host::tune_get(kTuneShort);
  if (want > 0) return want == 1;
  return rows >= (nvec <= kShortLanes ? 12LL : 28LL) * rw_host::device_cus();
}

template <typename T, bool HAS_W, bool RES = false>
int launch_typed(const void* x, const void* w, void* y, long long rows, int cols, float eps, hipStream_t stream,
                 const void* res = nullptr, void* res_out = nullptr) {
  const bool vec = cols % T::V == 0 && rw_host::aligned16(x) && rw_host::aligned16(y) &&
                   (!HAS_W || rw_host::aligned16(w)) &&
                   (!RES || (rw_host::aligned16(res) && rw_host::aligned16(res_out)));
  const long long nvec = ((long long)cols + T::V - 1) / T::V;
  auto even = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 1u) == 0; };
  const bool any = !vec && cols >= T::V && even(x) && even(y) && even(w) && even(res) && even(res_out);
  if ((vec || any) && rw_host::tune_get(kTuneGeneric) != 1 && nvec <= (long long)kMaxWaves * kWave * kMaxNv) {
    // One wave per row up to 4 vectors per lane (2048 two-byte columns), then more waves at 4 vectors per lane (and 8
    // per lane once 16 waves are not enough).
    auto auto_waves = [&] {
      const int w = pow2_at_least((nvec + (long long)kWave * 4 - 1) / ((long long)kWave * 4));
      return w > kMaxWaves ? kMaxWaves : w;
    };
    auto auto_nv = [&](int w) { return pow2_at_least((nvec + (long long)w * kWave - 1) / ((long long)w * kWave)); };
    int waves = rw_host::tune_get(kTuneWaves), nv = rw_host::tune_get(kTuneNv);
    if constexpr (!RES) {
      if (vec && nvec <= 2 * kShortLanes && waves <= 0 && nv <= 0 && takes_short(rows, nvec)) {
        // 65536 x 256 bf16 28.0 -> 14.4 us, 65536 x 8 23.7 -> 4.6
        const Args a{x, w, y, res, res_out, rows, nvec, cols, eps, stream, any};
        return nvec <= kShortLanes ? launch_short<T, 1, HAS_W>(a) : launch_short<T, 2, HAS_W>(a);
      }
    }
    if (waves <= 0) waves = auto_waves();
    if (nv <= 0) nv = auto_nv(waves);
    // a tuned shape the row kernel does not have (launch_rows below) is ignored: the automatic choice runs
    const bool shape = (waves == 1 || waves == 2 || waves == 4 || waves == 8 || waves == 16) &&
                       (nv == 1 || nv == 2 || nv == 4 || nv == 8);
    if (!shape) {
      waves = auto_waves();
      nv = auto_nv(waves);
    }
    if ((long long)waves * kWave * nv >= nvec) {
      const Args a{x, w, y, res, res_out, rows, nvec, cols, eps, stream, any};
      // non-temporal loads unless switched off (2): x is read once
      return any || rw_host::tune_get(kTuneNtLoads) != 2 ? launch_rows<T, HAS_W, RES, true>(waves, nv, a)
                                                  : launch_rows<T, HAS_W, RES, false>(waves, nv, a);
    }
  }
  long long grid = (long long)rw_host::device_cus() * 8;
  if (grid > rows) grid = rows;
  hipLaunchKernelGGL((rmsnorm_generic<T, HAS_W, RES>), dim3((unsigned)grid), dim3(256), 0, stream, x, res, w, y,
                     res_out, rows, cols, eps);
  return (int)hipGetLastError();
}

// The reference's argument checks (rmsnorm/kernel.cu:134-135). `threads` is its CUDA block size: validated the same
// way and otherwise unused, since the row grouping is chosen from the row length.
int validate(long long rows, int cols, int threads) {
  if (rows > 2147483647LL || cols <= 0 || threads < 32 || threads > 1024 || threads % 32) return rw_host::kInvalid;
  return rw_host::kOk;
}

}  // namespace

// rmsnorm/kernel.cu:132 `launch`: dtype 1 = bf16, 2 = fp16; y = x * inv with no weight. rows <= 0 is a no-op.
extern "C" int launch(const void* x, void* y, long long rows, int cols, int dtype, float eps, int threads,
                      hipStream_t stream) {
  if (rows <= 0) return rw_host::kOk;
  if (validate(rows, cols, threads)) return rw_host::kInvalid;
  if (dtype == 1) return launch_typed<BF16, false>(x, nullptr, y, rows, cols, eps, stream);
  if (dtype == 2) return launch_typed<F16, false>(x, nullptr, y, rows, cols, eps, stream);
  return rw_host::kInvalid;
}

// Weighted RMSNorm (no counterpart in the reference, which has no weight): y = T(w * T(x * inv)) with w[cols] in x's
// dtype; w == nullptr gives `launch`'s result. Same argument checks and return codes as `launch`.
extern "C" int rmsnorm_launch_weighted(const void* x, const void* weight, void* y, long long rows, int cols, int dtype,
                                       float eps, int threads, hipStream_t stream) {
  if (!weight) return launch(x, y, rows, cols, dtype, eps, threads, stream);
  if (rows <= 0) return rw_host::kOk;
  if (validate(rows, cols, threads)) return rw_host::kInvalid;
  if (dtype == 1) return launch_typed<BF16, true>(x, weight, y, rows, cols, eps, stream);
  if (dtype == 2) return launch_typed<F16, true>(x, weight, y, rows, cols, eps, stream);
  return rw_host::kInvalid;
}

// Fused residual add + RMSNorm (no counterpart in the reference; the step before an inference layer's norm):
// h = T(x + residual) is written to residual_out, then y = RMSNorm(h) (times weight when weight != nullptr), in one
// pass: x and residual read once, residual_out and y written once. residual_out may be residual and y may be x (in
// place). Same argument checks and return codes as `launch`; residual and residual_out must not be null.
extern "C" int rmsnorm_add_launch(const void* x, const void* residual, const void* weight, void* y, void* residual_out,
                                  long long rows, int cols, int dtype, float eps, int threads, hipStream_t stream) {
  if (rows <= 0) return rw_host::kOk;
  if (validate(rows, cols, threads) || !residual || !residual_out) return rw_host::kInvalid;
  if (dtype == 1)
    return weight ? launch_typed<BF16, true, true>(x, weight, y, rows, cols, eps, stream, residual, residual_out)
                  : launch_typed<BF16, false, true>(x, nullptr, y, rows, cols, eps, stream, residual, residual_out);
  if (dtype == 2)
    return weight ? launch_typed<F16, true, true>(x, weight, y, rows, cols, eps, stream, residual, residual_out)
                  : launch_typed<F16, false, true>(x, nullptr, y, rows, cols, eps, stream, residual, residual_out);
  return rw_host::kInvalid;
}

extern "C" int rmsnorm_tune(int slot, int value) { return rw_host::tune_set(slot, value); }
