// Row-wise softmax over the last dim of x[rows, cols] for fp32 (dtype 0) and bf16 (dtype 1) rows, every value
// accumulated in fp32 and each output rounded once (round to nearest even for bf16), behind the reference's C-ABI
// `launch` (softmax/kernel.cu:520-527, softmax/seed.cu:68-81).
//
// Tiers, chosen by row length in 16-byte vectors (4 fp32 or 8 bf16 elements). The first two have an instantiation for
// rows whose length is a multiple of the vector width and whose x and y are 16-byte aligned, and one for any other rows
// of at least one vector (AnyRow):
//  - many short rows (at most 64 vectors): four rows side by side in a wave; see softmax_short.
//  - row tier (rows up to 16 waves x 64 lanes x 8 vectors = 32768 fp32 / 65536 bf16 columns): a group of WAVES waves
//    holds one row in registers, NV 16-byte vectors per lane. A max and a sum of exp(x - max) are reduced over the
//    group (DPP inside each wave, one LDS slot per wave across waves) and y = exp(x - max) / sum is written from the
//    registers: one HBM read and one write per element. Workgroups are persistent: each walks the rows with a stride
//    of the grid and loads its next row while it reduces and stores the current one.
//  - co-resident tier (longer rows, up to 64 chunks of 16384 elements): one pass over x for any number of rows; see
//    softmax_coop.
//  - stream tier (longer rows still, aligned): one workgroup per row, two passes, no workspace; see softmax_stream.
//  - generic tier (what is left: rows shorter than a vector, and unaligned rows beyond the co-resident tier or, in
//    place, beyond the row tier): one workgroup per row, three scalar passes (max, sum, write).
// The library allocates no device memory: the co-resident tier exchanges its chunk pairs through a static device
// table whose entries carry a per-launch tag, so nothing has to be cleared between launches; launches recorded into a
// HIP graph take fresh tags at every replay (see softmax_coop).
// Aligned rows of the row tier and the stream tier multiply by the fp32 reciprocal of the row sum (the reference
// divides, softmax/kernel.cu:240; the two differ by at most 1.5 ulp in fp32 and are within the 1e-5 relative tolerance
// of the fp64 oracle); rows of other lengths and alignments, short fp32 rows and the fp32 chunks held as x take the
// quotient (quotient below), the generic tier the division.
#include <climits>
#include <cmath>
#include <mutex>

#include "host.hpp"
#include "rowwise.hpp"

using namespace rw;

namespace {

constexpr int kMaxNv = 8;       // 16-byte vectors a lane holds per row (32 fp32 / 64 bf16 values)
constexpr int kMaxWaves = 16;   // waves that share a row in the row tier (1024 threads)

template <int NV>
struct Regs {
  u32x4 v[NV];
};

// Lane t of a group of G lanes holds vectors t, t + G, ..., t + (NV - 1) G of the row: each load instruction of the
// group covers G * 16 contiguous bytes. Without FULL the index is clamped into the row (the duplicate is ignored), so
// the loads are issued unconditionally and the wait for them is not merged with a branch.
template <int G, int NV, bool FULL, bool NTL>
__device__ __forceinline__ void load_vectors(Regs<NV>& r, const void* base, long long first, long long count, int t) {
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    long long i = (long long)k * G + t;
    if constexpr (!FULL) i = i < count ? i : count - 1;
    r.v[k] = load16<NTL>(base, first + i);
  }
}

// exp(x - m) for the held vectors; returns the lane's sum over its valid elements (sequential order).
template <typename T, int G, int NV, bool FULL>
__device__ __forceinline__ float exp_and_sum(float (&f)[NV][T::V], float m, long long count, int t) {
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const bool ok = FULL || (long long)k * G + t < count;
#pragma unroll
    for (int i = 0; i < T::V; ++i) {
      f[k][i] = exp_to<T>(f[k][i] - m);
      s += ok ? f[k][i] : 0.0f;
    }
  }
  return s;
}

template <typename T, int G, int NV, bool FULL>
__device__ __forceinline__ float lane_max(const Regs<NV>& r, float (&f)[NV][T::V], long long count, int t) {
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    unpack<T>(r.v[k], f[k]);
    const bool ok = FULL || (long long)k * G + t < count;
#pragma unroll
    for (int i = 0; i < T::V; ++i) m = ok ? fmaxf(m, f[k][i]) : m;
  }
  return m;
}

// y = f * (1 / s): one division per row and a product per element (within 1.5 ulp of f / s; an element-wise fp32
// division is a multi-instruction sequence that made these kernels compute-bound).
template <typename T, int G, int NV, bool FULL, bool NTS>
__device__ __forceinline__ void scale_store(float (&f)[NV][T::V], float s, void* base, long long first,
                                            long long count, int t, bool active) {
  const float inv = 1.0f / s;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const long long i = (long long)k * G + t;
    if (active && (FULL || i < count)) {
#pragma unroll
      for (int e = 0; e < T::V; ++e) f[k][e] = f[k][e] * inv;
      store16<NTS>(base, first + i, pack<T>(f[k]));
    }
  }
}

// The sum of a vector's elements from the first `skip` on, in pairs.
template <typename T>
__device__ __forceinline__ float sum_vector(const float (&f)[T::V], int skip) {
  float a[T::V];
#pragma unroll
  for (int i = 0; i < T::V; ++i) a[i] = i >= skip ? f[i] : 0.0f;
#pragma unroll
  for (int d = 1; d < T::V; d *= 2)
#pragma unroll
    for (int i = 0; i < T::V; i += 2 * d) a[i] += a[i + d];
  return a[0];
}

// e / s within a correctly rounded division's last bit, from inv = 1 / s: the product, corrected by its remainder (one
// Newton step of the quotient).
__device__ __forceinline__ float quotient(float e, float s, float inv) {
  const float q = e * inv;
  return __builtin_fmaf(__builtin_fmaf(-q, s, e), inv, q);
}

template <typename T, int WAVES, int NV, bool FULL, bool NTS>
__device__ __forceinline__ void softmax_row(const Regs<NV>& r, void* y, long long row, long long nvec, int t,
                                            bool active, float* slots0, float* slots1, int wave, int first) {
  constexpr int G = WAVES * kWave;
  float f[NV][T::V];
  float m = lane_max<T, G, NV, FULL>(r, f, nvec, t);
  m = group_reduce<WAVES>(m, OpMax{}, slots0, wave, first);
  float s = exp_and_sum<T, G, NV, FULL>(f, m, nvec, t);
  s = group_reduce<WAVES>(s, OpSum{}, slots1, wave, first);
  scale_store<T, G, NV, FULL, NTS>(f, s, y, row * nvec, nvec, t, active);
}

// Row tier. A block is max(WAVES, 4) waves; GROUPS = block waves / WAVES groups each walk their own rows. The loop
// trip count is uniform over the block (a group past the last row loads an in-bounds row and stores nothing), so the
// LDS barriers of a multi-wave group are reached by every wave.
template <typename T, int WAVES, int NV, bool FULL, bool NTL, bool NTS>
__global__ void __launch_bounds__((WAVES < 4 ? 4 : WAVES) * 64)
    softmax_rows(const void* __restrict__ x, void* __restrict__ y, long long rows, long long nvec) {
  constexpr int BW = WAVES < 4 ? 4 : WAVES;
  constexpr int GROUPS = BW / WAVES;
  constexpr int G = WAVES * kWave;
  __shared__ float slots[2][BW];
  const int wave = wave_id();
  const int first = (wave / WAVES) * WAVES;
  const int t = (int)threadIdx.x - first * kWave;
  const long long step = (long long)gridDim.x * GROUPS;
  long long base = (long long)blockIdx.x * GROUPS;
  if (base >= rows) return;
  const long long last = rows - 1;
  long long ra = base + wave / WAVES;
  Regs<NV> a, b;
  load_vectors<G, NV, FULL, NTL>(a, x, (ra < rows ? ra : last) * nvec, nvec, t);
  while (true) {
    const long long rb = ra + step;
    load_vectors<G, NV, FULL, NTL>(b, x, (rb < rows ? rb : last) * nvec, nvec, t);
    softmax_row<T, WAVES, NV, FULL, NTS>(a, y, ra, nvec, t, ra < rows, slots[0], slots[1], wave, first);
    base += step;
    if (base >= rows) break;
    ra = rb;
    const long long rc = ra + step;
    load_vectors<G, NV, FULL, NTL>(a, x, (rc < rows ? rc : last) * nvec, nvec, t);
    softmax_row<T, WAVES, NV, FULL, NTS>(b, y, ra, nvec, t, ra < rows, slots[0], slots[1], wave, first);
    base += step;
    if (base >= rows) break;
    ra = rc;
  }
}

// Row tier for rows of any length from one vector up and any element alignment: the lanes' vectors start at the row's
// first element, wherever it lies, and a vector that would pass the row's end is moved back to end with it. Its first
// elements are then another lane's of the same workgroup (the same bits, from the same maximum and sum: the same
// results when they are stored twice), so the maximum takes every loaded element and the sum leaves out the first
// `skip` of the vector; only the wave that holds the row's end looks at that, and vectors that lie past the end for a
// whole wave are not worked on. 8192 x 3001 bf16: 62.1 us through the scalar kernel's three passes of 2-byte accesses,
// 18.3 us here (17.0 with exp_narrow and the reciprocal, which round 1.3e-4 of the distinct values of a row otherwise
// than the fp64 softmax; the scalar kernel's expf and division 0.45e-4, as here).
template <typename T, int WAVES, int NV>
struct AnyRow {
  static constexpr int G = WAVES * kWave, V = T::V;
  int cols, t;
  int first;  // the wave's first lane in the group: wave-uniform

  __device__ __forceinline__ int start(int k) const { return (k * G + t) * V; }
  __device__ __forceinline__ int offset(int k) const { return least(start(k), cols - V); }
  __device__ __forceinline__ bool used(int k) const { return (k * G + first) * V < cols; }          // by some lane
  __device__ __forceinline__ bool whole(int k) const { return (k * G + first + kWave) * V <= cols; }  // in every lane

  __device__ __forceinline__ void load(Regs<NV>& r, const void* x, long long row) const {
    const char* base = static_cast<const char*>(x) + row * cols * T::bytes;
#pragma unroll
    for (int k = 0; k < NV; ++k) r.v[k] = load16_at<false>(base, (uint32_t)(offset(k) * T::bytes));
  }

  __device__ __forceinline__ void softmax(const Regs<NV>& r, void* y, long long row, bool active, float* slots0,
                                          float* slots1, int wave, int first_wave) const {
    float f[NV][V];
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      unpack<T>(r.v[k], f[k]);
#pragma unroll
      for (int i = 0; i < V; ++i) m = fmaxf(m, f[k][i]);
    }
    m = group_reduce<WAVES>(m, OpMax{}, slots0, wave, first_wave);
    float s[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      s[k] = 0.0f;
      if (!used(k)) continue;
#pragma unroll
      for (int i = 0; i < V; ++i) f[k][i] = exp_nonpositive(f[k][i] - m);
      s[k] = whole(k) ? sum_vector<T>(f[k], 0) : sum_vector<T>(f[k], start(k) - offset(k));
    }
    // in pairs, as within a vector and over the waves: the error of a long chain of additions is kept out (unaligned
    // fp32 rows of 10000, 2-norm of the error: 8.5e-8 in the scalar kernel, 9.6e-8 with the waves one after another)
#pragma unroll
    for (int d = 1; d < NV; d *= 2)
#pragma unroll
      for (int k = 0; k < NV; k += 2 * d) s[k] += s[k + d];
    const float sum = group_sum_pairs<WAVES>(s[0], slots1, wave, first_wave);
    const float inv = 1.0f / sum;
    char* base = static_cast<char*>(y) + row * cols * T::bytes;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (!active || start(k) >= cols) continue;
#pragma unroll
      for (int i = 0; i < V; ++i) f[k][i] = quotient(f[k][i], sum, inv);
      store16_at<true>(base, (uint32_t)(offset(k) * T::bytes), pack<T>(f[k]));
    }
  }
};

template <typename T, int WAVES, int NV>
__global__ void __launch_bounds__((WAVES < 4 ? 4 : WAVES) * 64)
    softmax_rows_any(const void* __restrict__ x, void* __restrict__ y, long long rows, int cols) {
  constexpr int BW = WAVES < 4 ? 4 : WAVES;
  constexpr int GROUPS = BW / WAVES;
  __shared__ float slots[2][BW];
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int first = (wave / WAVES) * WAVES;
  const AnyRow<T, WAVES, NV> a{cols, (int)threadIdx.x - first * kWave, (wave - first) * kWave};
  const long long step = (long long)gridDim.x * GROUPS;
  long long base = (long long)blockIdx.x * GROUPS;
  if (base >= rows) return;
  const long long last = rows - 1;
  long long ra = base + wave / WAVES;
  Regs<NV> p, q;
  a.load(p, x, ra < rows ? ra : last);
  while (true) {
    const long long rb = ra + step;
    a.load(q, x, rb < rows ? rb : last);
    a.softmax(p, y, ra, ra < rows, slots[0], slots[1], wave, first);
    base += step;
    if (base >= rows) break;
    ra = rb;
    const long long rc = ra + step;
    a.load(p, x, rc < rows ? rc : last);
    a.softmax(q, y, ra, ra < rows, slots[0], slots[1], wave, first);
    base += step;
    if (base >= rows) break;
    ra = rc;
  }
}

// Short rows (at most 64 vectors: attention over a short context, a router's experts), of any length from one vector up
// and any element alignment: 16 lanes hold a row, NV vectors per lane (placed as AnyRow's), four rows side by side in a
// wave, and a wave takes SETS times four rows per step, so that lanes hold data and several loads are in flight where a
// wave per row would have one, mostly empty. The reductions stay inside a 16-lane DPP row; no LDS and no barrier. Waves
// are persistent and load their next rows while they work on these.
// 65536 rows, us as a wave per row / here: fp32 8 columns 20.3 / 4.7, 64 21.8 / 6.4, 128 22.0 / 10.9, 256 22.9 / 20.2;
// bf16 64 23.6 / 5.4, 131 22.2 / 10.1 (54 in the scalar kernel), 512 23.5 / 21.5.
// FINE: the exponential and the quotient within an fp32 ulp (fp32 rows, and bf16 rows that would otherwise take the
// scalar kernel); without it exp_narrow and the reciprocal, as in the row tier (65536 x 64 bf16 5.4 us, FINE 6.7).
constexpr int kShortLanes = 16;

template <typename Op>
__device__ __forceinline__ float short_reduce(float v, Op op) {
  v = op(v, dpp<kDppXor1>(v));
  v = op(v, dpp<kDppXor2>(v));
  v = op(v, dpp<kDppHalfMirror>(v));
  return op(v, dpp<kDppMirror>(v));
}

template <typename T, int NV, bool FINE>
__global__ void __launch_bounds__(256)
    softmax_short(const void* __restrict__ x, void* __restrict__ y, long long rows, int cols) {
  constexpr int V = T::V, SIDE = kWave / kShortLanes, SETS = NV == 1 ? 4 : 2;
  constexpr int ROWS = SETS * SIDE;  // a wave's rows per step
  const int lane = lane_id(), l = lane & (kShortLanes - 1), sub = lane / kShortLanes;
  const int per_block = (int)blockDim.x / kWave;
  const long long step = (long long)gridDim.x * per_block * ROWS;
  struct Step {
    u32x4 v[SETS][NV];
  };
  auto start = [&](int k) { return (k * kShortLanes + l) * V; };
  // the byte of vector k of the lane's row of set u, from the wave's first row on; a row past the last is the last
  auto at = [&](long long first, int u, int k) __attribute__((always_inline)) {
    const long long left = rows - 1 - first;
    const int r = u * SIDE + sub;
    return (uint32_t)(((left < r ? (int)left : r) * cols + least(start(k), cols - V)) * T::bytes);
  };
  auto load = [&](Step& s, long long first) __attribute__((always_inline)) {
    if (first >= rows) first = rows - 1;
    const char* base = static_cast<const char*>(x) + first * cols * T::bytes;
#pragma unroll
    for (int u = 0; u < SETS; ++u)
#pragma unroll
      for (int k = 0; k < NV; ++k) s.v[u][k] = load16_at<false>(base, at(first, u, k));
  };
  auto work = [&](const Step& s, long long first) __attribute__((always_inline)) {
    char* base = static_cast<char*>(y) + first * cols * T::bytes;
#pragma unroll
    for (int u = 0; u < SETS; ++u) {
      float f[NV][V];
      float m = -INFINITY;
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        unpack<T>(s.v[u][k], f[k]);
#pragma unroll
        for (int i = 0; i < V; ++i) m = fmaxf(m, f[k][i]);
      }
      m = short_reduce(m, OpMax{});
      float p[NV];
#pragma unroll
      for (int k = 0; k < NV; ++k) {
#pragma unroll
        for (int i = 0; i < V; ++i) f[k][i] = FINE ? exp_nonpositive(f[k][i] - m) : exp_narrow(f[k][i] - m);
        p[k] = sum_vector<T>(f[k], start(k) - least(start(k), cols - V));
      }
#pragma unroll
      for (int d = 1; d < NV; d *= 2)
#pragma unroll
        for (int k = 0; k < NV; k += 2 * d) p[k] += p[k + d];
      const float sum = short_reduce(p[0], OpSum{});
      const float inv = 1.0f / sum;
      const bool in = first + u * SIDE + sub < rows;
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        if (!in || start(k) >= cols) continue;
#pragma unroll
        for (int i = 0; i < V; ++i) f[k][i] = FINE ? quotient(f[k][i], sum, inv) : f[k][i] * inv;
        store16_at<true>(base, at(first, u, k), pack<T>(f[k]));
      }
    }
  };
  long long first = ((long long)blockIdx.x * per_block + __builtin_amdgcn_readfirstlane(wave_id())) * ROWS;
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

// Stream tier (aligned rows too long for the co-resident tier, or when it is declined): one workgroup of WAVES waves
// per row, persistent over rows, two passes and no workspace. Pass 1 keeps each lane's online (max, sum of exp(x -
// max)) over its vectors, U of them in flight per lane, merged over the workgroup (M = max m, S = sum s * exp(m - M));
// pass 2 reads the row again and writes exp(x - M) * (1 / S): 2R + 1W, the second read mostly from the caches.
template <typename T, int WAVES, bool NTS>
__global__ void __launch_bounds__(WAVES * 64)
    softmax_stream(const void* __restrict__ x, void* __restrict__ y, long long rows, long long nvec) {
  constexpr int G = WAVES * kWave;
  constexpr int U = 4;
  __shared__ float slots[2][WAVES];
  const int t = (int)threadIdx.x;
  for (long long row = blockIdx.x; row < rows; row += gridDim.x) {
    const long long base = row * nvec;
    float m = -INFINITY, s = 0.0f;
    for (long long i0 = 0; i0 < nvec; i0 += (long long)G * U) {
      u32x4 r[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const long long i = i0 + (long long)u * G + t;
        r[u] = load16<false>(x, base + (i < nvec ? i : nvec - 1));  // clamped: issued unconditionally
      }
      float f[U][T::V];
      float cm = -INFINITY;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        unpack<T>(r[u], f[u]);
        const bool ok = i0 + (long long)u * G + t < nvec;
#pragma unroll
        for (int e = 0; e < T::V; ++e) cm = ok ? fmaxf(cm, f[u][e]) : cm;
      }
      if (cm > m) {  // rescale the running sum to the new maximum (-inf elements never raise it)
        s = s * expf(m - cm);
        m = cm;
      }
      // while there is no maximum, elements are taken from 0: -inf adds nothing, a NaN makes the sum NaN
      const float from = m == -INFINITY ? 0.0f : m;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool ok = i0 + (long long)u * G + t < nvec;
#pragma unroll
        for (int e = 0; e < T::V; ++e) s += ok ? exp_to<T>(f[u][e] - from) : 0.0f;
      }
    }
    const float M = group_reduce<WAVES>(m, OpMax{}, slots[0], wave_id(), 0);
    const float S =
        group_reduce<WAVES>(s * expf(m - (M == -INFINITY ? 0.0f : M)), OpSum{}, slots[1], wave_id(), 0);
    const float inv = 1.0f / S;  // an all -inf row: M = -inf, S = 0, and every output NaN (as the fp64 reference)
    for (long long i = t; i < nvec; i += G) {
      float f[T::V];
      unpack<T>(load16<false>(x, base + i), f);
#pragma unroll
      for (int e = 0; e < T::V; ++e) f[e] = exp_to<T>(f[e] - M) * inv;
      store16<NTS>(y, base + i, pack<T>(f));
    }
    __syncthreads();  // the slots are written again by the next row's reductions
  }
}

// Co-resident tier: long rows in chunks of WAVES x 64 x NV vectors, one workgroup per chunk, every workgroup of a
// launch resident at once (the grid never exceeds the GPU's resident slots of this kernel): x is read once (1R + 1W).
// The grid is `groups` row groups of `chunks` workgroups; group g handles rows g, g + groups, ..., one row per
// iteration, so any number of rows keeps one pass over x. Per iteration, each workgroup holds its chunk in registers,
// as x or as e = exp(x - m) in fp32 (HOLD below), reduces it to its online-softmax pair (m, s = sum of e), and
// publishes the pair into its slot of the device-scope pair table; wave 0 polls the group's slots until every chunk's
// pair of this row is there, merges them in a fixed order (the online-softmax merge, the same lanes and order in every
// workgroup of the row, so all agree bit for bit; softmax/kernel.cu:121-152 is the reference's form of it), and the
// chunk is written as exp(x - M) / S or as e * (exp(m - M) / S), the latter within 3 fp32 ulp of the once-rounded value
// before the output's rounding.
//
// The pair table needs no clearing: each pair is two 64-bit words, (tag << 32 | m bits) and (tag << 32 | s bits),
// stored with device-coherent stores, and a word counts only when its tag is this launch's tag for the iteration.
// Every launch gets a fresh range of tags; tag 0, the table's load-time contents, is never handed out. An eager launch
// takes its range from the host, in [1, 2^31). A launch recorded into a HIP graph cannot: its kernel arguments are
// replayed as they were captured, and every replay would wait for the tags the previous replay left in the table. It
// takes its range on the device instead, at every replay, from a cell of its own that a one-wave kernel node just
// before it fills from a device counter (softmax_coop_cell), in [2^31, 2^32); so no two launches, eager or replayed,
// share a tag. The table is double-buffered by iteration parity: a chunk writes its slot of parity p again two
// iterations later, by which time every workgroup of its group has published the iteration in between, and so has
// read parity p. A launch on another stream that uses the same slots at the same time can only make a wait fail (its
// tags differ), never pass.
//
// The wait is bounded by time: after wait_ticks of the 100 MHz s_memrealtime clock with pairs still missing (other
// kernels holding CUs, so that the row's workgroups are not all resident) the workgroup takes the missing pairs from x
// itself, by the operations of their own workgroups in their order, so the outputs are the same bits either way; only
// the time suffers, by about two reads of each missing chunk per waiting workgroup. In place (aligned rows longer than
// the row tier holds) a chunk is written only after its pair was published and read back, so that a workgroup that took
// it from x while it was written finds the pair there afterwards, unless another launch has taken the slot since.
constexpr int kCoopMaxChunks = 64;   // a row's chunks: one slot each, polled by one lane each of one wave
constexpr int kCoopSlots = 4096;     // pair slots per parity: the most workgroups one launch may have
constexpr int kCoopCells = 4096;     // captured launches per device with a tag cell of their own
constexpr unsigned kDeviceTags = 0x80000000u;  // the top bit marks the tags handed out on the device
__device__ __align__(256) unsigned long long g_coop_pairs[2][kCoopSlots][2];
__device__ unsigned g_coop_cells[kCoopCells];     // each captured launch's first tag, refreshed at every replay
__device__ unsigned long long g_coop_device_next;  // tags handed out on the device so far

// The tag of iteration it of a launch whose first tag is tag0: host tags never reach the top bit (the host restarts
// its range before they would), device tags keep it and wrap within the top half.
__device__ __forceinline__ unsigned coop_tag(unsigned tag0, int it) {
  return (((tag0 & ~kDeviceTags) + (unsigned)it) & ~kDeviceTags) | (tag0 & kDeviceTags);
}

// Clears the pair table (before a launch whose tags restart after the tag counter wrapped).
__device__ __forceinline__ void coop_clear_table(unsigned first, unsigned stride) {
  unsigned long long* p = &g_coop_pairs[0][0][0];
  for (unsigned i = first; i < 2u * kCoopSlots * 2u; i += stride)
    __hip_atomic_store(p + i, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The kernel node ahead of a captured co-resident launch: takes `iters` fresh device tags and leaves the first in the
// launch's cell. When the range reaches the end of the device half of the tag space the table is cleared first, as the
// host does for its half, so that a pair left from the previous round of the counter can never match (another
// stream's launch using the table meanwhile can only see its wait fail).
__global__ void __launch_bounds__(256) softmax_coop_cell(int cell, unsigned iters) {
  __shared__ unsigned long long old;
  if (threadIdx.x == 0)
    old = __hip_atomic_fetch_add(&g_coop_device_next, (unsigned long long)iters, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const unsigned long long lo = old & ~(unsigned long long)kDeviceTags;
  if (lo + iters > (unsigned long long)kDeviceTags) coop_clear_table(threadIdx.x, 256);
  if (threadIdx.x == 0)
    __hip_atomic_store(&g_coop_cells[cell], kDeviceTags | (unsigned)lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// LOOP: some row group has more than one row (groups < rows); without it every workgroup takes one row, and the
// kernel is compiled without the loop (which costs registers: fewer resident workgroups).
// ANY: rows of any length (nvec vectors, the last one partial) and element alignment. The row's last vector is moved
// back to end with the row (AnyRow), its first `skip` elements being another lane's.
// FINE: the exponential within an fp32 ulp, for fp32 rows, for bf16 rows that the scalar kernel would take and for
// those that an eager launch takes from the row tier and holds as e; other bf16 rows take exp_narrow. (Share of a bf16
// row's distinct values that are rounded otherwise than the fp64 softmax's: 512 x 40000 aligned 1.27e-4 in the row
// tier, here 1.40e-4 with exp_narrow and 0.59e-4 FINE; unaligned 0.59e-4 in the scalar kernel and here.)
// HOLD: the chunk is held as e = exp(x - m) and written as e * (exp(m - M) / S); otherwise it is held as x, and the
// exponential is taken again from M. Holding e saves an exponential per element, which long chunks of many rows feel
// (1024 x 50000 fp32 77 us against 84, bf16 44 against 50), and costs fp32 rows accuracy where the chunk is short (mean
// relative error of 16 x 128256 fp32: 1.47e-7 in four times longer chunks, 1.57e-7 as e, 1.03e-7 from x). So short
// chunks and unaligned fp32 rows are held as x.
// The waves per SIMD asked of the compiler are those it reaches by itself without the code behind a wait that ended,
// which would otherwise cost the loop's bf16 forms one of four (256 x 262144 52.0 us, 54.5 with three).
template <typename T, int WAVES, int NV, bool NTL, bool NTS, bool LOOP, bool ANY, bool FINE>
__global__ void __launch_bounds__(WAVES * 64, NV * T::V == 64 ? 4 : ANY ? 7 : 8)
    softmax_coop(const void* __restrict__ x, void* __restrict__ y, long long rows, long long nvec, long long cols,
                 int chunks, int groups, int slot0, unsigned tag0, int cell, unsigned wait_ticks) {
  constexpr int G = WAVES * kWave;
  // a captured launch (cell >= 0) reads its first tag from its cell, filled by the kernel node just before it
  if (cell >= 0) tag0 = __hip_atomic_load(&g_coop_cells[cell], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  constexpr long long CH = (long long)G * NV;
  static_assert(kCoopMaxChunks == kWave, "a lane of wave 0 for each chunk's pair");
  __shared__ float slots[2][WAVES];
  __shared__ float ms[2];
  __shared__ unsigned long long missing;       // the chunks whose pairs had not come when the wait ended
  __shared__ float pairs[kCoopMaxChunks][2];  // the row's pairs then
  const int c = (int)(blockIdx.x % (unsigned)chunks), group = (int)(blockIdx.x / (unsigned)chunks);
  // a chunk's place in the row: its first vector (< 2^31: at most kCoopMaxChunks chunks of CH vectors), its vectors,
  // and (ANY) the elements from its first to the row's end, at least one
  struct Part {
    int first, count, reach;
  };
  auto part = [&](int q) __attribute__((always_inline)) {
    const int first = q * (int)CH;
    return Part{first, nvec - first < CH ? (int)(nvec - first) : (int)CH, (int)(cols - (long long)first * T::V)};
  };
  const Part own = part(c);
  const int t0 = (int)threadIdx.x;
  const int wave0 = __builtin_amdgcn_readfirstlane(t0 & ~(kWave - 1));
  const int iters = (int)((rows - group + groups - 1) / groups);
  constexpr bool PREFETCH = LOOP && T::V == 8;
  constexpr bool HOLD = NV == 64 / T::V && !(ANY && T::bytes == 4);
  auto exp_of = [](float d) __attribute__((always_inline)) { return FINE ? exp_nonpositive(d) : exp_narrow(d); };
  Regs<NV> next;  // PREFETCH: the next row's raw chunk, loaded during the wait
  // ANY: elements of the row from V before the chunk's first on; a vector past the row's last whole start is moved back
  // to it
  auto offset = [&](const Part& p, int k, int t) __attribute__((always_inline)) {
    return (uint32_t)((least((k * G + t) * T::V, p.reach - T::V) + T::V) * T::bytes);
  };
  auto chunk_base = [&](const Part& p, long long row) __attribute__((always_inline)) {
    return (row * cols + ((long long)p.first - 1) * T::V) * T::bytes;
  };
  auto load_chunk = [&](Regs<NV>& r, const Part& p, long long row, int t) __attribute__((always_inline)) {
    if constexpr (ANY) {
      const char* base = static_cast<const char*>(x) + chunk_base(p, row);
#pragma unroll
      for (int k = 0; k < NV; ++k) r.v[k] = load16_at<NTL>(base, offset(p, k, t));
    } else {
      load_vectors<G, NV, false, NTL>(r, x, row * nvec + p.first, p.count, t);
    }
  };
  // the maximum of m and vector k's elements; its elements' exponentials from `from` and their sum
  auto max_with = [&](const Part& p, const u32x4& v, int k, int t, float m) __attribute__((always_inline)) {
    float f[T::V];
    unpack<T>(v, f);
    const bool ok = k * G + t < p.count;
#pragma unroll
    for (int i = 0; i < T::V; ++i) m = ok ? fmaxf(m, f[i]) : m;
    return m;
  };
  auto exps = [&](const Part& p, const u32x4& v, int k, int t, float from, float (&f)[T::V])
                  __attribute__((always_inline)) {
    unpack<T>(v, f);
    const bool ok = k * G + t < p.count;
#pragma unroll
    for (int i = 0; i < T::V; ++i) {
      f[i] = exp_of(f[i] - from);
      if (!ANY) f[i] = ok ? f[i] : 0.0f;
    }
    int skip = 0;  // ANY: the first elements of the vector, another lane's
    if (ANY && (k * G + wave0 + kWave) * T::V > p.reach) {
      const int start = (k * G + t) * T::V;
      skip = start - least(start, p.reach - T::V);
    }
    return sum_vector<T>(f, skip);
  };
  if constexpr (PREFETCH) load_chunk(next, own, group, t0);
  for (int it = 0; it < iters; ++it) {
    const long long row = group + (long long)it * groups;
    // the lane's offsets are formed anew each iteration (hoisted out of the loop they would hold NV 64-bit offsets in
    // registers for its whole length)
    int t = t0;
    if constexpr (LOOP) asm volatile("" : "+v"(t));
    const unsigned long long tag = (unsigned long long)coop_tag(tag0, it) << 32;
    unsigned long long(*table)[2] = g_coop_pairs[it & 1] + slot0 + group * chunks;
    Regs<NV> r;
    if constexpr (PREFETCH) r = next;
    else load_chunk(r, own, row, t);
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < NV; ++k) m = max_with(own, r.v[k], k, t, m);
    m = group_reduce<WAVES>(m, OpMax{}, slots[0], wave_id(), 0);
    // a chunk of only -inf and NaN has m = -inf (fmaxf takes the other operand of a NaN): its elements are taken from 0
    // instead, -inf to 0 and NaN to NaN, so that a NaN reaches s, the row's S, and through it every output of the row
    float e[NV][T::V];
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) s += exps(own, r.v[k], k, t, m == -INFINITY ? 0.0f : m, e[k]);
    s = group_reduce<WAVES>(s, OpSum{}, slots[1], wave_id(), 0);
    // the next row's loads go out before the wait and the stores (bf16; for fp32 the two chunks together would halve
    // the resident workgroups)
    if constexpr (PREFETCH)
      if (it + 1 < iters) load_chunk(next, own, row + groups, t);
    if (t == 0) {  // an all -inf chunk publishes (-inf, 0), which adds nothing to the merge; with a NaN, (-inf, NaN)
      __hip_atomic_store(&table[c][0], tag | __float_as_uint(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&table[c][1], tag | __float_as_uint(s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // a chunk's pair by the lane of its number in wave 0, for those of the launch's iteration; whether it has come
    auto look = [&](unsigned long long& wm, unsigned long long& ws) __attribute__((always_inline)) {
      if ((wm >> 32) != (tag >> 32))
        wm = __hip_atomic_load(&table[lane_id()][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((ws >> 32) != (tag >> 32))
        ws = __hip_atomic_load(&table[lane_id()][1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return (wm >> 32) == (tag >> 32) && (ws >> 32) == (tag >> 32);
    };
    auto merge = [&](float pm, float ps) __attribute__((always_inline)) {
      const float M = wave_max(pm);
      const float S = wave_sum(ps * expf(pm - (M == -INFINITY ? 0.0f : M)));  // (-inf, s): 0, or NaN where s is
      if (lane_id() == 0) {
        ms[0] = M;
        ms[1] = S;
      }
    };
    if (wave_id() == 0) {
      const bool mine = lane_id() < chunks;
      unsigned long long wm = 0, ws = 0;
      const unsigned long long start = __builtin_amdgcn_s_memrealtime();
      unsigned long long left;
      while ((left = __ballot(mine && !look(wm, ws))) != 0) {
        // (the clock is a scalar read, so the decision is the wave's; readfirstlane states it)
        if (__builtin_amdgcn_readfirstlane((int)(__builtin_amdgcn_s_memrealtime() - start > wait_ticks))) break;
        __builtin_amdgcn_s_sleep(1);
      }
      const float pm = mine ? __uint_as_float((unsigned)wm) : -INFINITY;
      const float ps = mine ? __uint_as_float((unsigned)ws) : 0.0f;
      if (left == 0) {
        merge(pm, ps);
      } else {
        pairs[lane_id()][0] = pm;
        pairs[lane_id()][1] = ps;
      }
      if (lane_id() == 0) missing = left;
    }
    __syncthreads();
    if (__builtin_expect(missing != 0, 0)) {
      // the missing pairs from x, by the operations and in the order of the chunks' own workgroups (the offsets formed
      // anew, vector by vector: kept from above, or several loads in flight, they would cost the kernel its registers)
      int u = t;
      asm volatile("" : "+v"(u));
      const unsigned long long out = missing;
      for (unsigned long long left = out; left; left &= left - 1) {
        const int q = __builtin_ctzll(left);
        const Part p = part(q);
        auto load = [&](int k) __attribute__((always_inline)) {
          if constexpr (ANY) return load16_at<false>(static_cast<const char*>(x) + chunk_base(p, row), offset(p, k, u));
          else return load16<false>(x, row * nvec + p.first + least(k * G + u, p.count - 1));
        };
        float qm = -INFINITY, qs = 0.0f;
#pragma unroll 1
        for (int k = 0; k < NV; ++k) qm = max_with(p, load(k), k, u, qm);
        qm = group_reduce<WAVES>(qm, OpMax{}, slots[0], wave_id(), 0);
#pragma unroll 1
        for (int k = 0; k < NV; ++k) {
          float f[T::V];
          qs += exps(p, load(k), k, u, qm == -INFINITY ? 0.0f : qm, f);
        }
        qs = group_reduce<WAVES>(qs, OpSum{}, slots[1], wave_id(), 0);
        if (threadIdx.x == 0) {
          pairs[q][0] = qm;
          pairs[q][1] = qs;
        }
      }
      if (wave_id() == 0) {
        wave_lds_sync();  // lane 0's pairs before the other lanes' reads
        float pm = pairs[lane_id()][0], ps = pairs[lane_id()][1];
        unsigned long long wm = 0, ws = 0;
        // (a pair that has come meanwhile is taken: in place, its workgroup may have written its chunk since)
        if ((out >> lane_id() & 1) && look(wm, ws)) {
          pm = __uint_as_float((unsigned)wm);
          ps = __uint_as_float((unsigned)ws);
        }
        merge(pm, ps);
      }
      __syncthreads();
      if constexpr (!HOLD) load_chunk(r, own, row, u);  // (not kept in registers meanwhile)
    }
    const float M = ms[0], S = ms[1];
    // HOLD: an all -inf chunk (e = 0) gives 0, or NaN when the whole row is -inf (S = 0) or S is NaN
    const float scale = HOLD ? (m == -INFINITY ? 0.0f : expf(m - M)) / S : 1.0f / S;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int i = k * G + t;
      if (i < own.count) {
        float f[T::V];
        if constexpr (!HOLD) unpack<T>(r.v[k], f);
#pragma unroll
        for (int j = 0; j < T::V; ++j) {
          if constexpr (HOLD) f[j] = e[k][j] * scale;
          else if constexpr (FINE) f[j] = quotient(exp_of(f[j] - M), S, scale);
          else f[j] = exp_of(f[j] - M) * scale;
        }
        if constexpr (ANY) {
          if (k == 0 && own.reach < T::V) {
            // a last chunk of less than a vector (lane 0 alone): the first elements are the chunk before's, which may
            // round them otherwise
            const long long end = row * cols + cols;
#pragma unroll
            for (int j = 0; j < T::V; ++j)
              if (j >= T::V - own.reach) store_elem<T>(y, end - T::V + j, f[j]);
            continue;
          }
          store16_at<NTS>(static_cast<char*>(y) + chunk_base(own, row), offset(own, k, t), pack<T>(f));
        }
        else store16<NTS>(y, row * nvec + own.first + i, pack<T>(f));
      }
    }
    if constexpr (!LOOP) break;
    __syncthreads();  // ms, missing and the reduction slots are written again by the next row
  }
}

// Clears the pair table (before an eager launch whose tags restart after the host's tag counter wrapped).
__global__ void __launch_bounds__(256) softmax_coop_clear() {
  coop_clear_table(blockIdx.x * 256 + threadIdx.x, gridDim.x * 256);
}

// Generic tier: any row length and alignment; one 256-thread block per row (grid-strided), three scalar passes.
template <typename T>
__global__ void __launch_bounds__(256)
    softmax_generic(const void* __restrict__ x, void* __restrict__ y, long long rows, long long cols) {
  __shared__ float slots[2][4];
  const int wave = wave_id();
  for (long long row = blockIdx.x; row < rows; row += gridDim.x) {
    const long long o = row * cols;
    float m = -INFINITY;
    for (long long j = threadIdx.x; j < cols; j += 256) m = fmaxf(m, load_elem<T>(x, o + j));
    m = group_reduce<4>(m, OpMax{}, slots[0], wave, 0);
    float s = 0.0f;
    for (long long j = threadIdx.x; j < cols; j += 256) s += expf(load_elem<T>(x, o + j) - m);
    s = group_reduce<4>(s, OpSum{}, slots[1], wave, 0);
    for (long long j = threadIdx.x; j < cols; j += 256) store_elem<T>(y, o + j, expf(load_elem<T>(x, o + j) - m) / s);
    __syncthreads();  // slots are rewritten by the next row's reductions
  }
}

// ---- host side ------------------------------------------------------------------------------------------------------

// Tuning slots (0 = automatic), for sweeps and tests: row-tier waves per row, row-tier vectors per lane, row-tier
// resident blocks per CU, stream-tier waves, co-resident row groups (fewer forces more rows per workgroup), preferred
// tier (1 row, 2 stream, 3 generic, 4 co-resident; a tier that cannot take the rows is passed over for the automatic
// choice), non-temporal loads (1 on, 2 off), the co-resident tier's wait budget in 100 MHz ticks (tests force its
// fallback with 1), the co-resident tier's vectors per lane (the longest chunks', half or a quarter of it), the short
// rows' kernel for every row it can hold (1) or none (2).
enum { kTuneWaves = 0, kTuneNv = 1, kTuneBlocksPerCu = 2, kTuneStreamWaves = 3, kTuneCoopGroups = 4, kTuneTier = 5,
       kTuneNtLoads = 6, kTuneWaitTicks = 7, kTuneCoopNv = 8, kTuneShort = 9 };
constexpr unsigned kCoopWaitTicks = 10000;  // 100 us: tens of times a row's arrival skew, a few launch lengths

bool aligned_to(const void* p, int bytes) { return (reinterpret_cast<uintptr_t>(p) & (uintptr_t)(bytes - 1)) == 0; }

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

template <typename T, int WAVES, int NV, bool FULL, bool NTL>
int launch_rows_k(const void* x, void* y, long long rows, long long nvec, hipStream_t stream) {
  constexpr int BW = WAVES < 4 ? 4 : WAVES;
  constexpr int GROUPS = BW / WAVES;
  auto kern = softmax_rows<T, WAVES, NV, FULL, NTL, true>;
  static int occ = 0;  // resident blocks per CU of this instantiation (idempotent cache)
  if (occ <= 0) occ = blocks_per_cu(kern, BW * kWave);
  // about 8 resident waves per CU by default: with two register sets per wave that keeps enough loads in flight,
  // and more waves only contend (measured on MI355X); rows of 8 waves take 16 (two blocks): [4096, 4096] fp32 as 8
  // waves x 2 vectors 24.61 -> 24.37 us (means of six fresh allocations each), [2048, 8192] as 8 waves x 4 vectors
  // 25.69 -> 25.12 us (interleaved runs on one box)
  int per_cu = rw_host::tune_get(kTuneBlocksPerCu);
  if (per_cu <= 0) per_cu = WAVES == 8 ? 2 : (8 / BW > 1 ? 8 / BW : 1);
  if (per_cu > occ) per_cu = occ;
  const long long need = (rows + GROUPS - 1) / GROUPS;
  long long grid = (long long)rw_host::device_cus() * per_cu;
  if (grid > need) grid = need;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(BW * kWave), 0, stream, x, y, rows, nvec);
  return (int)hipGetLastError();
}

template <typename T, int WAVES, int NV, bool NTL>
int launch_rows_nv(const void* x, void* y, long long rows, long long nvec, hipStream_t stream) {
  if (nvec == (long long)WAVES * kWave * NV) return launch_rows_k<T, WAVES, NV, true, NTL>(x, y, rows, nvec, stream);
  return launch_rows_k<T, WAVES, NV, false, NTL>(x, y, rows, nvec, stream);
}

template <typename T, int WAVES, bool NTL>
int launch_rows_w(int nv, const void* x, void* y, long long rows, long long nvec, hipStream_t stream) {
  switch (nv) {
    case 1: return launch_rows_nv<T, WAVES, 1, NTL>(x, y, rows, nvec, stream);
    case 2: return launch_rows_nv<T, WAVES, 2, NTL>(x, y, rows, nvec, stream);
    case 4: return launch_rows_nv<T, WAVES, 4, NTL>(x, y, rows, nvec, stream);
    case 8: return launch_rows_nv<T, WAVES, 8, NTL>(x, y, rows, nvec, stream);
    case 16:  // (through the tuning slots: one or two waves holding a row of up to 8192 fp32 / 16384 bf16 elements)
      if constexpr (WAVES <= 2) return launch_rows_nv<T, WAVES, 16, NTL>(x, y, rows, nvec, stream);
      else return rw_host::kInvalid;
    default: return rw_host::kInvalid;
  }
}

template <typename T, bool NTL>
int launch_rows(int waves, int nv, const void* x, void* y, long long rows, long long nvec, hipStream_t stream) {
  switch (waves) {
    case 1: return launch_rows_w<T, 1, NTL>(nv, x, y, rows, nvec, stream);
    case 2: return launch_rows_w<T, 2, NTL>(nv, x, y, rows, nvec, stream);
    case 4: return launch_rows_w<T, 4, NTL>(nv, x, y, rows, nvec, stream);
    case 8: return launch_rows_w<T, 8, NTL>(nv, x, y, rows, nvec, stream);
    case 16: return launch_rows_w<T, 16, NTL>(nv, x, y, rows, nvec, stream);
    default: return rw_host::kInvalid;
  }
}

// Rows of any length and element alignment (softmax_rows_any).
template <typename T, int WAVES, int NV>
int launch_any_k(const void* x, void* y, long long rows, int cols, hipStream_t stream) {
  constexpr int BW = WAVES < 4 ? 4 : WAVES;
  constexpr int GROUPS = BW / WAVES;
  auto kern = softmax_rows_any<T, WAVES, NV>;
  static int occ = 0;  // resident blocks per CU of this instantiation (idempotent cache)
  if (occ <= 0) occ = blocks_per_cu(kern, BW * kWave);
  int per_cu = rw_host::tune_get(kTuneBlocksPerCu);
  // fp32 rows of four vectors a lane and more: the resident waves of launch_rows_k; otherwise about 24 waves per CU,
  // whose loads are fewer or whose rows take more work per byte (8192 x 3001 fp32 as 4 waves x 4 vectors: 33.5 us with
  // two blocks per CU, 34.3 with four; bf16 as 2 waves x 4 vectors: 19.9 with two, 18.6 with three, 18.2 with six)
  if (per_cu <= 0) {
    const int resident = T::bytes == 4 && NV >= 4 ? (WAVES == 8 ? 16 : 8) : 24;
    per_cu = resident / BW > 1 ? resident / BW : 1;
  }
  if (per_cu > occ) per_cu = occ;
  const long long need = (rows + GROUPS - 1) / GROUPS;
  long long grid = (long long)rw_host::device_cus() * per_cu;
  if (grid > need) grid = need;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(BW * kWave), 0, stream, x, y, rows, cols);
  return (int)hipGetLastError();
}

template <typename T, int WAVES>
int launch_any_w(int nv, const void* x, void* y, long long rows, int cols, hipStream_t stream) {
  switch (nv) {
    case 1: return launch_any_k<T, WAVES, 1>(x, y, rows, cols, stream);
    case 2: return launch_any_k<T, WAVES, 2>(x, y, rows, cols, stream);
    case 4: return launch_any_k<T, WAVES, 4>(x, y, rows, cols, stream);
    default: return launch_any_k<T, WAVES, 8>(x, y, rows, cols, stream);
  }
}

template <typename T>
int launch_any(int waves, int nv, const void* x, void* y, long long rows, int cols, hipStream_t stream) {
  switch (waves) {
    case 1: return launch_any_w<T, 1>(nv, x, y, rows, cols, stream);
    case 2: return launch_any_w<T, 2>(nv, x, y, rows, cols, stream);
    case 4: return launch_any_w<T, 4>(nv, x, y, rows, cols, stream);
    case 8: return launch_any_w<T, 8>(nv, x, y, rows, cols, stream);
    default: return launch_any_w<T, 16>(nv, x, y, rows, cols, stream);
  }
}

template <typename T, int NV, bool FINE>
int launch_short_nv(const void* x, void* y, long long rows, int cols, hipStream_t stream) {
  constexpr int ROWS = (NV == 1 ? 4 : 2) * (kWave / kShortLanes);
  const long long cus = rw_host::device_cus(), waves = (rows + ROWS - 1) / ROWS;
  int per_cu = rw_host::tune_get(kTuneBlocksPerCu);
  if (per_cu <= 0) per_cu = 6;
  // one wave per block until every CU has four: few rows then spread over the GPU
  const int per_block = waves >= 4 * cus ? 4 : 1;
  long long grid = (waves + per_block - 1) / per_block;
  if (grid > cus * per_cu * 4 / per_block) grid = cus * per_cu * 4 / per_block;
  hipLaunchKernelGGL((softmax_short<T, NV, FINE>), dim3((unsigned)grid), dim3(per_block * kWave), 0, stream, x, y, rows,
                     cols);
  return (int)hipGetLastError();
}

template <typename T, bool FINE>
int launch_short(const void* x, void* y, long long rows, long long cols, hipStream_t stream) {
  const long long nvec = (cols + T::V - 1) / T::V;
  if (nvec <= kShortLanes) return launch_short_nv<T, 1, FINE>(x, y, rows, (int)cols, stream);
  if (nvec <= 2 * kShortLanes) return launch_short_nv<T, 2, FINE>(x, y, rows, (int)cols, stream);
  return launch_short_nv<T, 4, FINE>(x, y, rows, (int)cols, stream);
}

template <typename T, int WAVES>
int launch_stream_w(const void* x, void* y, long long rows, long long nvec, hipStream_t stream) {
  long long grid = (long long)rw_host::device_cus() * (16 / WAVES > 1 ? 16 / WAVES : 1);
  if (grid > rows) grid = rows;
  hipLaunchKernelGGL((softmax_stream<T, WAVES, true>), dim3((unsigned)grid), dim3(WAVES * kWave), 0, stream, x, y,
                     rows, nvec);
  return (int)hipGetLastError();
}

template <typename T>
int launch_stream(const void* x, void* y, long long rows, long long nvec, hipStream_t stream) {
  switch (rw_host::tune_get(kTuneStreamWaves)) {
    case 4: return launch_stream_w<T, 4>(x, y, rows, nvec, stream);
    case 8: return launch_stream_w<T, 8>(x, y, rows, nvec, stream);
    default: return launch_stream_w<T, 16>(x, y, rows, nvec, stream);
  }
}

// The co-resident tier's tags of eager launches: per device, the next unused one of the host's half of the tag space,
// [1, 2^31) (0 is never handed out: it is the pair table's contents at load). A launch takes one per iteration; when
// the range would pass 2^31 - 1, the table is cleared on the launch's stream and the tags start again at 1.
unsigned coop_tags(int dev, unsigned n, hipStream_t stream, int* err) {
  static std::mutex mu;
  static unsigned next[64];
  std::lock_guard<std::mutex> lock(mu);
  unsigned& nx = next[dev & 63];
  *err = rw_host::kOk;
  if (nx == 0 || (unsigned long long)nx + n > (unsigned long long)kDeviceTags) {
    hipLaunchKernelGGL(softmax_coop_clear, dim3(16), dim3(256), 0, stream);
    *err = (int)hipGetLastError();
    nx = 1;
  }
  const unsigned t = nx;
  nx += n;
  return t;
}

// The first of a launch's n pair slots: launches take the table's slots in turn, so that launches that overlap on other
// streams seldom meet in a slot (where their waits would fail).
int coop_slots(int dev, int n) {
  static std::mutex mu;
  static int next[64];
  std::lock_guard<std::mutex> lock(mu);
  int& nx = next[dev & 63];
  const int first = nx + n <= kCoopSlots ? nx : 0;
  nx = first + n;
  return first;
}

// A captured launch's tag cell: per device, cells are handed out once each, in capture order, and never reused (a
// graph may be replayed at any time). Returns -1 when the device's cells are used up; such a launch takes the stream
// tier, which keeps no state between launches.
int coop_cell(int dev) {
  static std::mutex mu;
  static int next[64];
  std::lock_guard<std::mutex> lock(mu);
  int& nx = next[dev & 63];
  if (nx >= kCoopCells) return -1;
  return nx++;
}

// Whether work issued to `stream` is being recorded into a graph (an error reads as not capturing: the launch then
// fails or runs as an eager one would).
bool capturing(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return status != hipStreamCaptureStatusNone;
}

struct CoopLaunch {
  const void* x;
  void* y;
  long long rows, nvec, cols;
  hipStream_t stream;
};
constexpr int kCoopWaves = 4;

// The vectors per lane of a launch of one row per workgroup: the longest chunks (64 elements per lane), half or a
// quarter of them.
//  - bf16: shorter as long as no CU gets more workgroups. us by workgroups: 24 x 70000 120 5.6, 216 5.3, 432 5.9; 48 x
//    70000 240 6.1, 432 6.3, 864 7.5; 24 x 128256 192 5.6, 384 6.2, 768 6.9; 1 x 262144 16 5.5, 32 5.0, 64 4.6; 96 x
//    33000 288 7.8, 480 7.0, 864 7.5.
//  - fp32, whose long chunks fill the registers: half as long up to four workgroups of the long ones per CU (200 x 50000
//    800 17.0, 1400 13.6; 24 x 262144 384 11.6, 768 10.8; 96 x 128256 768 17.5, 1536 16.7), and a quarter while those
//    are under four per CU and, beyond one per CU, at most 16 per row (200 x 20000 600 9.4, 1000 7.8; 1 x 262144 32 5.7,
//    64 4.9; but 16 x 128256 256 6.3, 512 6.6; 24 x 70000 216 5.8, 432 6.2; 24 x 262144 1536 13.5; 16 x 262144 512 9.0,
//    1024 10.3).
template <typename T>
int coop_nv(long long rows, long long nvec) {
  constexpr int NV = 64 / T::V;
  const long long cus = rw_host::device_cus();
  auto chunks = [&](int n) { return (nvec + kCoopWaves * kWave * n - 1) / (kCoopWaves * kWave * n); };
  auto grid = [&](int n) { return rows * chunks(n); };
  int nv = NV;
  if constexpr (T::bytes == 4) {
    if (grid(NV) >= 4 * cus) return NV;
    return grid(NV / 4) < 4 * cus && (grid(NV / 4) <= cus || chunks(NV / 4) <= 16) ? NV / 4 : NV / 2;
  }
  while (nv > NV / 4 && (grid(nv / 2) + cus - 1) / cus == (grid(nv) + cus - 1) / cus) nv /= 2;
  return nv;
}

// The launch of a co-resident kernel over `groups` row groups of `chunks` workgroups.
template <typename Kernel>
int launch_coop_k(Kernel kern, const CoopLaunch& a, long long chunks, long long groups) {
  const long long iters = (a.rows + groups - 1) / groups;
  if (iters > 0x40000000LL) return 1;
  int dev = 0, err = (int)hipGetDevice(&dev);
  if (err != rw_host::kOk) return err;
  unsigned tag0 = 0;
  int cell = -1;
  if (capturing(a.stream)) {
    // recorded into a graph: the tags are taken on the device at every replay, by a kernel node ahead of the launch
    cell = coop_cell(dev);
    if (cell < 0) return 1;
    hipLaunchKernelGGL(softmax_coop_cell, dim3(1), dim3(256), 0, a.stream, cell, (unsigned)iters);
    err = (int)hipGetLastError();
  } else {
    tag0 = coop_tags(dev, (unsigned)iters, a.stream, &err);
  }
  if (err != rw_host::kOk) return err;
  const int budget = rw_host::tune_get(kTuneWaitTicks);
  const unsigned ticks = budget > 0 ? (unsigned)budget : kCoopWaitTicks;
  const int slot0 = coop_slots(dev, (int)(groups * chunks));
  hipLaunchKernelGGL(kern, dim3((unsigned)(groups * chunks)), dim3(kCoopWaves * kWave), 0, a.stream, a.x, a.y, a.rows,
                     a.nvec, a.cols, (int)chunks, (int)groups, slot0, tag0, cell, ticks);
  return (int)hipGetLastError();
}

// One row per workgroup: chunks of 4 waves x 64 lanes x NV vectors, when every row's chunks fit on the GPU at once.
// Returns 1, launching nothing, when they do not (or a row has more than kCoopMaxChunks of them).
template <typename T, int NV, bool NTL, bool ANY, bool FINE>
int launch_coop_one(const CoopLaunch& a) {
  // (aligned bf16 chunks held as x round as the row tier does: not FINE)
  auto one = softmax_coop<T, kCoopWaves, NV, NTL, true, false, ANY, FINE && (ANY || T::bytes == 4 || NV == 64 / T::V)>;
  static int occ = 0;  // resident blocks per CU (idempotent cache)
  if (occ <= 0) occ = blocks_per_cu(one, kCoopWaves * kWave);
  constexpr long long CH = (long long)kCoopWaves * kWave * NV;
  const long long chunks = (a.nvec + CH - 1) / CH;
  long long slots = (long long)rw_host::device_cus() * occ;
  if (slots > kCoopSlots) slots = kCoopSlots;
  if (chunks > kCoopMaxChunks || a.rows * chunks > slots) return 1;
  return launch_coop_k(one, a, chunks, a.rows);
}

// Co-resident tier: chunks of 4 waves x 64 lanes x 64 elements (16 fp32 or 8 bf16 vectors per lane), at most
// kCoopMaxChunks per row; shorter chunks (half or a quarter as long) when the rows are so few that those still leave
// the GPU lightly filled (coop_nv); row groups walking several rows (an instantiation of its own: the loop costs
// registers) when the rows' chunks do not fit on the GPU at once. Returns 1, launching nothing, when one row's chunks
// do not fit.
template <typename T, bool NTL, bool ANY, bool FINE>
int launch_coop(const CoopLaunch& a, int most_iters = INT_MAX) {
  constexpr int NV = 64 / T::V;
  constexpr long long CH = (long long)kCoopWaves * kWave * NV;
  const int want = rw_host::tune_get(kTuneCoopGroups);
  const long long cus = rw_host::device_cus();
  if (want <= 0 || want >= a.rows) {
    int nv = rw_host::tune_get(kTuneCoopNv);
    if (nv != NV && nv != NV / 2 && nv != NV / 4) nv = coop_nv<T>(a.rows, a.nvec);
    int rc = 1;  // a shape whose chunks are too many for the GPU or for a row takes the next longer chunks
    if (nv == NV / 4) rc = launch_coop_one<T, NV / 4, NTL, ANY, FINE>(a);
    if (rc == 1 && nv <= NV / 2) rc = launch_coop_one<T, NV / 2, NTL, ANY, FINE>(a);
    if (rc == 1) rc = launch_coop_one<T, NV, NTL, ANY, FINE>(a);
    if (rc != 1) return rc;
  }
  auto loop = softmax_coop<T, kCoopWaves, NV, NTL, true, true, ANY, FINE>;
  static int occ = 0;  // resident blocks per CU (idempotent cache)
  if (occ <= 0) occ = blocks_per_cu(loop, kCoopWaves * kWave);
  const long long chunks = (a.nvec + CH - 1) / CH;
  long long slots = cus * occ;
  if (slots > kCoopSlots) slots = kCoopSlots;
  if (chunks > kCoopMaxChunks || chunks > slots) return 1;
  long long groups = slots / chunks;
  if (want > 0 && want < groups) groups = want;
  if (groups > a.rows) groups = a.rows;
  if ((a.rows + groups - 1) / groups > most_iters) return 1;
  return launch_coop_k(loop, a, chunks, groups);
}

template <typename T>
int launch_generic(const void* x, void* y, long long rows, long long cols, hipStream_t stream) {
  long long grid = (long long)rw_host::device_cus() * 8;
  if (grid > rows) grid = rows;
  hipLaunchKernelGGL(softmax_generic<T>, dim3((unsigned)grid), dim3(256), 0, stream, x, y, rows, cols);
  return (int)hipGetLastError();
}

// Whether the tuning slots ask for a row-tier shape that the kernels have.
bool row_shape_tuned() {
  const int w = rw_host::tune_get(kTuneWaves), n = rw_host::tune_get(kTuneNv);
  auto pow2_to = [](int v, int most) { return v >= 0 && v <= most && (v & (v - 1)) == 0; };
  return (w || n) && pow2_to(w, kMaxWaves) && pow2_to(n, 16) && !(n == 16 && (w == 0 || w > 2));
}

// Rows that the row tier could hold but the co-resident tier takes faster: rows of more than 4096 vectors, which in the
// row tier are 16 waves x 8 vectors, with registers spilled unless the row fills them (bf16: 600 x 40000 33.5 -> 22.1
// us, 1024 x 50000 55.2 -> 49.3, 3000 x 64000 177 -> 145; full rows of 65536 as long as a workgroup has at most three,
// 400 rows 21.9 -> 19.3, 600 rows 30.5 -> 27.4, but 1024 rows 50.1 -> 52.3; fp32 when every row's chunks are resident
// at once: 256 x 32768 15.0 -> 12.2, 512 x 20000 19.0 -> 15.8, but 2048 x 32768 97 -> 103 in row groups), and rows of
// more than 2048 vectors when they are too few to
// fill the GPU with one workgroup each (1 x 10000 fp32 4.5 -> 3.7, 16 x 32768 bf16 4.8 -> 4.0; 128 x 16384 fp32 6.0
// either way). A launch that is being captured stays in the row tier, which needs no second node and no tag cell, and
// so does one in place (its callers look), where a timed-out wait's second read of the row would meet outputs.
template <typename T>
bool coop_instead_of_rows(long long rows, long long nvec, hipStream_t stream) {
  if (rw_host::tune_get(kTuneTier) != 0 || row_shape_tuned()) return false;
  return (nvec > 4096 || (nvec > 2048 && rows <= 32)) && !capturing(stream);
}

// Whether rows of at most 64 vectors share waves: eight or sixteen of them take longer than the row tier's one, which
// few rows do not make up for. Kernel times in us, a wave per row / shared: 128 columns fp32 64 rows 2.0 / 2.4, 2048
// 2.2 / 2.5, 4096 2.9 / 2.6, 16384 6.6 / 3.6; 64 columns bf16 64 rows 2.0 / 2.8, 4096 3.0 / 2.9; more than 32 vectors:
// bf16 4096 x 257 3.6 / 4.8, 8000 x 257 4.6 / 5.3, 65536 x 257 22.4 / 20.0; fp32 4096 x 200 3.1 / 3.6, 65536 x 256 22.9
// / 20.2.
bool takes_short(long long rows, long long nvec) {
  const int want = rw_host::tune_get(kTuneShort);
  if (want > 0) return want == 1;
  return rows >= (nvec <= 2 * kShortLanes ? 16LL : 32LL) * rw_host::device_cus();
}

template <typename T>
int launch_typed(const void* x, void* y, long long rows, long long cols, hipStream_t stream) {
  const bool vec = cols % T::V == 0 && rw_host::aligned16(x) && rw_host::aligned16(y);
  const int tier = rw_host::tune_get(kTuneTier);
  const bool any = cols >= T::V && aligned_to(x, T::bytes) && aligned_to(y, T::bytes);
  if (tier == 3 || !(vec || any)) return launch_generic<T>(x, y, rows, cols, stream);
  const long long nvec = (cols + T::V - 1) / T::V;
  if (any && nvec <= 4 * kShortLanes && tier == 0 && !row_shape_tuned() && takes_short(rows, nvec))
    return vec ? launch_short<T, T::bytes == 4>(x, y, rows, cols, stream)
               : launch_short<T, true>(x, y, rows, cols, stream);
  if (!vec) {
    const CoopLaunch coop{x, y, rows, nvec, cols, stream};
    if (nvec > (long long)kMaxWaves * kWave * kMaxNv || tier == 4) {
      // (in place, a workgroup whose wait timed out would read a row that others have begun to overwrite)
      const int rc = x != y ? launch_coop<T, false, true, true>(coop) : 1;
      return rc != 1 ? rc : launch_generic<T>(x, y, rows, cols, stream);
    }
    if (x != y && coop_instead_of_rows<T>(rows, nvec, stream)) {
      const int rc = launch_coop<T, false, true, true>(coop, T::bytes == 4 ? 1 : INT_MAX);
      if (rc != 1) return rc;
    }
    int waves = rw_host::tune_get(kTuneWaves), nv = rw_host::tune_get(kTuneNv);
    auto pow2_to = [](int v, int most) { return v >= 1 && v <= most && (v & (v - 1)) == 0; };
    if (!pow2_to(waves, kMaxWaves)) {
      waves = pow2_at_least(((nvec + 3) / 4 + kWave - 1) / kWave);
      // (fp32 rows for 16 waves of 4 vectors: 8 waves of 8 when there are rows for two such blocks per CU, 1024 x 16383
      // 24.1 -> 22.0 us; bf16 600 x 32001 23.4 us as 16 x 4, 24.2 as 8 x 8)
      if (T::bytes == 4 && waves == kMaxWaves && rows >= 2LL * rw_host::device_cus()) waves = kMaxWaves / 2;
      waves = waves > kMaxWaves ? kMaxWaves : waves;
    }
    const int need = pow2_at_least((nvec + (long long)waves * kWave - 1) / ((long long)waves * kWave));
    if (!pow2_to(nv, kMaxNv) || nv < need) nv = need;
    if (nv > kMaxNv) return launch_generic<T>(x, y, rows, cols, stream);
    return launch_any<T>(waves, nv, x, y, rows, (int)cols, stream);
  }
  if (tier == 2) return launch_stream<T>(x, y, rows, nvec, stream);
  const CoopLaunch coop{x, y, rows, nvec, cols, stream};
  if (x != y && nvec <= (long long)kMaxWaves * kWave * kMaxNv && coop_instead_of_rows<T>(rows, nvec, stream)) {
    const int iters = T::bytes == 4 ? 1 : nvec == (long long)kMaxWaves * kWave * kMaxNv ? 3 : INT_MAX;
    const int rc = launch_coop<T, false, false, true>(coop, iters);
    if (rc != 1) return rc;
  }
  const bool ntl = rw_host::tune_get(kTuneNtLoads) == 1;
  if (tier != 4 && nvec <= (long long)kMaxWaves * kWave * kMaxNv) {
    // Row tier: 4 vectors per lane as long as 16 waves suffice, then up to 8; except that rows of 513 to 1024
    // vectors take 8 waves of 2 vectors rather than 4 waves of 4 (more waves with fewer loads each; [4096, 4096]
    // fp32 24.61 -> 24.37 us measured).
    auto auto_waves = [&] {
      const long long lanes = (nvec + 3) / 4;
      const int w = pow2_at_least((lanes + kWave - 1) / kWave);
      return w == 4 ? 8 : w > kMaxWaves ? kMaxWaves : w;
    };
    auto auto_nv = [&](int w) { return pow2_at_least((nvec + (long long)w * kWave - 1) / ((long long)w * kWave)); };
    int waves = rw_host::tune_get(kTuneWaves), nv = rw_host::tune_get(kTuneNv);
    if (waves <= 0) waves = auto_waves();
    if (nv <= 0) nv = auto_nv(waves);
    // a tuned shape the row kernel does not have (launch_rows below) is ignored: the automatic choice runs
    const bool shape = (waves == 1 || waves == 2 || waves == 4 || waves == 8 || waves == 16) &&
                       (nv == 1 || nv == 2 || nv == 4 || nv == 8 || (nv == 16 && waves <= 2));
    if (!shape) {
      waves = auto_waves();
      nv = auto_nv(waves);
    }
    if ((long long)waves * kWave * nv >= nvec) {
      return ntl ? launch_rows<T, true>(waves, nv, x, y, rows, nvec, stream)
                 : launch_rows<T, false>(waves, nv, x, y, rows, nvec, stream);
    }
  }
  constexpr bool kFine = T::bytes == 4;
  const int rc = ntl ? launch_coop<T, true, false, kFine>(coop) : launch_coop<T, false, false, kFine>(coop);
  if (rc != 1) return rc;
  return launch_stream<T>(x, y, rows, nvec, stream);
}

}  // namespace

// softmax/kernel.cu:520 `launch`: dtype 0 = fp32, 1 = bf16. `threads` and `aux` are the reference's block-size hints
// for its CUDA tiers; they are accepted and not used (as softmax/seed.cu:70-71 does): the tier and shape are chosen
// from the row length. rows <= 0 or cols <= 0 is a successful no-op.
extern "C" int launch(const void* x, void* y, long long rows, long long cols, int dtype, int threads, int aux,
                      hipStream_t stream) {
  (void)threads;
  (void)aux;
  if (rows <= 0 || cols <= 0) return rw_host::kOk;
  if (dtype == 0) return launch_typed<F32>(x, y, rows, cols, stream);
  if (dtype == 1) return launch_typed<BF16>(x, y, rows, cols, stream);
  return rw_host::kInvalid;
}

// Tuning override for parameter sweeps (see the slot list above); 0 restores the automatic choice.
extern "C" int softmax_tune(int slot, int value) { return rw_host::tune_set(slot, value); }
