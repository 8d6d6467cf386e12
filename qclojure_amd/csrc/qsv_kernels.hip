// qsv_kernels.hip — state initialisation, conversions, FP64 reductions
// (norm, overlaps, one-qubit expectations), sampling and measurement of libqsv.
//
// State layout: 2^n amplitudes, interleaved (re, im); c128 = double2 (16 B),
// c64 = float2 (8 B). Reference qubit q is index bit b = n-1-q.
#include "qsv_internal.h"

#include <algorithm>

namespace qsv {

template <typename R> struct VT;
template <> struct VT<double> { using T = double2; };
template <> struct VT<float> { using T = float2; };

template <typename R>
__global__ __launch_bounds__(kBlock) void k_fill_basis(typename VT<R>::T* __restrict__ psi, uint64_t S, uint64_t idx)
{
  using T = typename VT<R>::T;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < S; i += stride) {
    T v;
    v.x = (i == idx) ? R(1) : R(0);
    v.y = R(0);
    psi[i] = v;
  }
}

// Plain streaming copy (non-temporal), 4 amplitudes per thread.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_copy(const typename VT<R>::T* __restrict__ src,
                                                 typename VT<R>::T* __restrict__ dst, uint64_t S)
{
  typedef R V __attribute__((ext_vector_type(2)));
  const V* s = reinterpret_cast<const V*>(src);
  V* d = reinterpret_cast<V*>(dst);
  const uint64_t base = (uint64_t)blockIdx.x * (kBlock * 4) + threadIdx.x;
  V v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint64_t i = base + (uint64_t)k * kBlock;
    if (i < S) v[k] = __builtin_nontemporal_load(s + i);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint64_t i = base + (uint64_t)k * kBlock;
    if (i < S) __builtin_nontemporal_store(v[k], d + i);
  }
}

// One pass over two states of any precisions: partials of Re/Im <a|b>,
// sum |a|^2, sum |b|^2 (FP64) and max |a_i - b_i|.
template <typename RA, typename RB>
__global__ __launch_bounds__(kBlock) void k_compare(const typename VT<RA>::T* __restrict__ a,
                                                    const typename VT<RB>::T* __restrict__ b, uint64_t S,
                                                    double* __restrict__ partials)
{
  __shared__ double sh[kBlock / 64];
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  double re = 0.0, im = 0.0, na = 0.0, nb = 0.0, mx = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < S; i += stride) {
    const double ax = a[i].x, ay = a[i].y, bx = b[i].x, by = b[i].y;
    re += ax * bx + ay * by;
    im += ax * by - ay * bx;
    na += ax * ax + ay * ay;
    nb += bx * bx + by * by;
    const double dx = ax - bx, dy = ay - by;
    mx = fmax(mx, sqrt(dx * dx + dy * dy));
  }
  double vals[4] = {re, im, na, nb};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    double v = vals[q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) partials[(uint64_t)q * kReduceBlocks + blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
    __syncthreads();
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_down(mx, off, 64));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0)
    partials[4ull * kReduceBlocks + blockIdx.x] = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
}

__global__ __launch_bounds__(kBlock) void k_final_max(const double* __restrict__ partials, double* __restrict__ out)
{
  __shared__ double sh[kBlock / 64];
  double m = 0.0;
  for (int i = threadIdx.x; i < kReduceBlocks; i += kBlock) m = fmax(m, partials[i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_down(m, off, 64));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) *out = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_scale(typename VT<R>::T* __restrict__ psi, uint64_t S, R f)
{
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < S; i += stride) {
    auto v = psi[i];
    v.x *= f;
    v.y *= f;
    psi[i] = v;
  }
}

// normalize-state with the norm^2 already on the device (norm2[0]): divide by
// the norm when it exceeds 1e-12, else leave the amplitudes.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_scale_by_norm(typename VT<R>::T* __restrict__ psi, uint64_t S,
                                                          const double* __restrict__ norm2)
{
  const double nrm = sqrt(norm2[0]);
  if (!(nrm > 1e-12)) return;
  const R f = (R)(1.0 / nrm);
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < S; i += stride) {
    auto v = psi[i];
    v.x *= f;
    v.y *= f;
    psi[i] = v;
  }
}

__global__ __launch_bounds__(kBlock) void k_f64_to_c64(const double2* __restrict__ src, float2* __restrict__ dst,
                                                        uint64_t count)
{
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < count; i += stride) {
    const double2 v = src[i];
    dst[i] = make_float2((float)v.x, (float)v.y);
  }
}

__global__ __launch_bounds__(kBlock) void k_c64_to_f64(const float2* __restrict__ src, double2* __restrict__ dst,
                                                        uint64_t count)
{
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < count; i += stride) {
    const float2 v = src[i];
    dst[i] = make_double2((double)v.x, (double)v.y);
  }
}

// ---------------------------------------------------------------------------
// FP64 reductions: fixed grid of kReduceBlocks blocks writes per-block
// partials, then one block per value sums them in a fixed order (the result
// is deterministic run to run).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// Sum over the block; the result is valid in thread 0.
__device__ __forceinline__ double block_sum(double v, double* sh)
{
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < kBlock / 64; ++i) r += sh[i];
  }
  __syncthreads();
  return r;
}

// partials[v * kReduceBlocks + b] -> out[v]
__global__ __launch_bounds__(kBlock) void k_final_sum(const double* __restrict__ partials, double* __restrict__ out)
{
  __shared__ double sh[kBlock / 64];
  const double* p = partials + (uint64_t)blockIdx.x * kReduceBlocks;
  double acc = 0.0;
  for (int i = threadIdx.x; i < kReduceBlocks; i += kBlock) acc += p[i];
  const double r = block_sum(acc, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = r;
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_norm2(const typename VT<R>::T* __restrict__ psi, uint64_t S,
                                                   double* __restrict__ partials)
{
  __shared__ double sh[kBlock / 64];
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  double acc0 = 0.0, acc1 = 0.0;
  uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  for (; i + stride < S; i += 2 * stride) {
    const auto a = psi[i];
    const auto b = psi[i + stride];
    acc0 += (double)a.x * a.x + (double)a.y * a.y;
    acc1 += (double)b.x * b.x + (double)b.y * b.y;
  }
  if (i < S) {
    const auto a = psi[i];
    acc0 += (double)a.x * a.x + (double)a.y * a.y;
  }
  const double r = block_sum(acc0 + acc1, sh);
  if (threadIdx.x == 0) partials[blockIdx.x] = r;
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_inner(const typename VT<R>::T* __restrict__ a,
                                                   const typename VT<R>::T* __restrict__ b, uint64_t S,
                                                   double* __restrict__ partials)
{
  __shared__ double sh[kBlock / 64];
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  double re = 0.0, im = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < S; i += stride) {
    const auto x = a[i];
    const auto y = b[i];
    // conj(x) * y
    re += (double)x.x * y.x + (double)x.y * y.y;
    im += (double)x.x * y.y - (double)x.y * y.x;
  }
  const double r0 = block_sum(re, sh);
  const double r1 = block_sum(im, sh);
  if (threadIdx.x == 0) {
    partials[blockIdx.x] = r0;
    partials[kReduceBlocks + blockIdx.x] = r1;
  }
}

// <psi| O on bit tbit |psi>
template <typename R>
__global__ __launch_bounds__(kBlock) void k_expect1q(const typename VT<R>::T* __restrict__ psi, uint64_t half,
                                                      uint64_t tbit, Mat2<double> M, double* __restrict__ partials)
{
  __shared__ double sh[kBlock / 64];
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  const uint64_t lo = tbit - 1;
  double re = 0.0, im = 0.0;
  for (uint64_t p = (uint64_t)blockIdx.x * kBlock + threadIdx.x; p < half; p += stride) {
    const uint64_t i0 = ((p & ~lo) << 1) | (p & lo);
    const auto A = psi[i0];
    const auto B = psi[i0 | tbit];
    const double a0r = A.x, a0i = A.y, a1r = B.x, a1i = B.y;
    const double y0r = M.m[0] * a0r - M.m[1] * a0i + M.m[2] * a1r - M.m[3] * a1i;
    const double y0i = M.m[0] * a0i + M.m[1] * a0r + M.m[2] * a1i + M.m[3] * a1r;
    const double y1r = M.m[4] * a0r - M.m[5] * a0i + M.m[6] * a1r - M.m[7] * a1i;
    const double y1i = M.m[4] * a0i + M.m[5] * a0r + M.m[6] * a1i + M.m[7] * a1r;
    re += a0r * y0r + a0i * y0i + a1r * y1r + a1i * y1i;
    im += a0r * y0i - a0i * y0r + a1r * y1i - a1i * y1r;
  }
  const double r0 = block_sum(re, sh);
  const double r1 = block_sum(im, sh);
  if (threadIdx.x == 0) {
    partials[blockIdx.x] = r0;
    partials[kReduceBlocks + blockIdx.x] = r1;
  }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_probs(const typename VT<R>::T* __restrict__ psi, uint64_t offset,
                                                   uint64_t count, double* __restrict__ out)
{
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < count; k += stride) {
    const auto a = psi[offset + k];
    out[k] = (double)a.x * a.x + (double)a.y * a.y;
  }
}

// ---------------------------------------------------------------------------
// Shot sampling (measure-state, inverse CDF): chunk sums, inclusive scan of
// chunk sums, then one wave per shot: a search over chunks and a wave scan
// inside the chunk. Bound by the one read of the state (chunk sums 350 us for
// 2 GiB); 1000 shots take 7 to 10 us, a chain of loads per shot (15 to 20 us
// with binary searches and 64 amplitudes a step).
// ---------------------------------------------------------------------------
template <typename R>
__global__ __launch_bounds__(kBlock) void k_chunk_sums(const typename VT<R>::T* __restrict__ psi, int chunk_log,
                                                        double* __restrict__ sums)
{
  __shared__ double sh[kBlock / 64];
  const uint64_t c0 = (uint64_t)blockIdx.x << chunk_log, len = 1ull << chunk_log;
  double acc = 0.0;
  for (uint64_t k = threadIdx.x; k < len; k += kBlock) {
    const auto a = psi[c0 + k];
    acc += (double)a.x * a.x + (double)a.y * a.y;
  }
  const double r = block_sum(acc, sh);
  if (threadIdx.x == 0) sums[blockIdx.x] = r;
}

// The prefix over chunk sums is kept in groups of 1024 chunks: entry c of group
// g holds the sum of the group's chunks up to c, except the group's last entry,
// which holds the sum of everything up to it. A state of 2^20 amplitudes or
// fewer is one group and its entries are the plain inclusive prefix. Groups are
// scanned by one workgroup each (k_scan_groups), their totals by one more
// (k_scan_totals); the serial walk of one workgroup over all chunk sums that
// these replace took 347 us on 27 qubits (2^17 sums), as long as reading the
// 2 GiB state; they take 5 us each.
constexpr int kGroupLog = 10;

__device__ __forceinline__ double wave_scan(double v, int lane)
{
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double t = __shfl_up(v, off, 64);
    if (lane >= off) v += t;
  }
  return v;
}

__global__ __launch_bounds__(kBlock) void k_scan_groups(double* __restrict__ v, uint64_t n)
{
  __shared__ double tot[kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t b = ((uint64_t)blockIdx.x << kGroupLog) + 4 * threadIdx.x;
  double x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = b + k < n ? v[b + k] : 0.0;
#pragma unroll
  for (int k = 1; k < 4; ++k) x[k] += x[k - 1];
  const double inc = wave_scan(x[3], lane);
  if (lane == 63) tot[w] = inc;
  __syncthreads();
  double off = 0.0;
  for (int k = 0; k < w; ++k) off += tot[k];
  const double before = __shfl_up(inc, 1, 64);
  if (lane) off += before;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (b + k < n) v[b + k] = off + x[k];
}

// Running totals of the groups, in place at each group's last entry.
__global__ __launch_bounds__(1024) void k_scan_totals(double* __restrict__ v, uint64_t groups)
{
  __shared__ double tot[1024];
  auto at = [&](uint64_t g) -> double& { return v[(g << kGroupLog) + (1u << kGroupLog) - 1]; };
  const uint64_t seg = (groups + 1023) / 1024;
  const uint64_t b = threadIdx.x * seg, e = (b + seg < groups) ? b + seg : groups;
  double run = 0.0;
  for (uint64_t k = b; k < e; ++k) run += at(k);
  tot[threadIdx.x] = run;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const double t = (threadIdx.x >= (unsigned)off) ? tot[threadIdx.x - off] : 0.0;
    __syncthreads();
    tot[threadIdx.x] += t;
    __syncthreads();
  }
  run = threadIdx.x ? tot[threadIdx.x - 1] : 0.0;
  for (uint64_t k = b; k < e; ++k) {
    run += at(k);
    at(k) = run;
  }
}

__device__ __forceinline__ double uniform01(uint64_t seed, uint64_t k)
{
  uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// The first k in [0, n) with !(val(k) < r), n if there is none: the wave probes
// 64 places at a time (a binary search is a chain of 10 to 17 dependent loads).
template <typename F>
__device__ __forceinline__ uint64_t wave_search(uint64_t n, double r, int lane, F&& val)
{
  uint64_t lo = 0, len = n;
  while (len) {
    const uint64_t step = (len + 63) >> 6;
    const uint64_t first = (uint64_t)lane * step, last = first + step < len ? first + step : len;
    const uint64_t hit = __ballot(first < len && !(val(lo + last - 1) < r));
    if (!hit) return n;
    const uint64_t at = (uint64_t)(__ffsll((unsigned long long)hit) - 1) * step;
    if (step == 1) return lo + at;
    lo += at;
    len = at + step < len ? step : len - at;
  }
  return n;
}

// The same by a binary search: the same value in every lane, one load a step.
template <typename F>
__device__ __forceinline__ uint64_t binary_search(uint64_t n, double r, F&& val)
{
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (val(mid) < r) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// One wave per shot. Few shots are a chain of loads each: the search probes 64
// places at a time, the shot's chunk is read in one round of loads, sixteen
// neighbouring amplitudes a lane, and scanned over the wave once, and the lane
// that holds the outcome walks its own sixteen. MANY of them are bound by what
// they read: one load a step of the search, and the chunk 64 neighbouring
// amplitudes at a time up to the outcome.
template <typename R, bool MANY>
__global__ __launch_bounds__(kBlock) void k_sample(const typename VT<R>::T* __restrict__ psi, uint64_t S,
                                                    int chunk_log, const double* __restrict__ prefix,
                                                    uint64_t nchunks, uint64_t shots, uint64_t seed,
                                                    uint64_t* __restrict__ out)
{
  const int lane = threadIdx.x & 63;
  const uint64_t shot = (uint64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (shot >= shots) return;
  constexpr uint64_t G = 1ull << kGroupLog;
  const double total = prefix[nchunks - 1];
  const double r = uniform01(seed, shot) * total;
  // first chunk whose inclusive prefix is >= r: its group, then the chunk in it
  uint64_t g = 0;
  const uint64_t ng = nchunks > G ? nchunks / G : 1;
  auto search = [&](uint64_t n, auto&& val) {
    if constexpr (MANY) return binary_search(n, r, val);
    else return wave_search(n, r, lane, val);
  };
  if (ng > 1) g = search(ng, [&](uint64_t k) { return prefix[k * G + G - 1]; });
  const double off = g && g < ng ? prefix[g * G - 1] : 0.0;
  uint64_t c = nchunks;
  if (g < ng) {
    const uint64_t len = nchunks < G ? nchunks : G;
    c = g * G + search(len, [&](uint64_t k) {
      const double v = prefix[g * G + k];
      return ng > 1 && k == G - 1 ? v : off + v;
    });
  }
  if (c >= nchunks) {
    if (lane == 0) out[shot] = S - 1;
    return;
  }
  const double run = (c & (G - 1)) ? off + prefix[c - 1] : off;
  const uint32_t len = 1u << chunk_log, per = len < 64 ? 1u : len >> 6;
  const uint64_t c0 = c << chunk_log;
  if constexpr (MANY) {
    double sum = run;
    for (uint32_t piece = 0; piece < len; piece += 64) {
      double w = 0.0;
      if (piece + lane < len) {
        const auto a = psi[c0 + piece + lane];
        w = (double)a.x * a.x + (double)a.y * a.y;
      }
      w = wave_scan(w, lane);
      const uint64_t hit = __ballot(sum + w >= r && piece + lane < len);
      if (hit) {
        if (lane == 0) out[shot] = c0 + piece + (uint64_t)(__ffsll((unsigned long long)hit) - 1);
        return;
      }
      sum += __shfl(w, 63, 64);
    }
    if (lane == 0) out[shot] = c0 + len - 1;
    return;
  }
  double v[1 << (kSampleChunkLog - 6)], sum = 0.0;
#pragma unroll
  for (uint32_t j = 0; j < (1u << (kSampleChunkLog - 6)); ++j) {
    v[j] = 0.0;
    if (j < per && lane * per + j < len) {
      const auto a = psi[c0 + lane * per + j];
      v[j] = (double)a.x * a.x + (double)a.y * a.y;
    }
  }
#pragma unroll
  for (uint32_t j = 0; j < (1u << (kSampleChunkLog - 6)); ++j) sum += v[j];
  const double inc = wave_scan(sum, lane);
  double cum = __shfl_up(inc, 1, 64);
  cum = run + (lane ? cum : 0.0);
  const uint64_t hit = __ballot(run + inc >= r && lane * per < len);
  if (!hit) {
    if (lane == 0) out[shot] = c0 + len - 1;
    return;
  }
  if (lane != __ffsll((unsigned long long)hit) - 1) return;
  uint32_t pick = per - 1;
  bool found = false;
#pragma unroll
  for (uint32_t j = 0; j < (1u << (kSampleChunkLog - 6)); ++j) {
    cum += v[j];
    if (!found && j < per && cum >= r) {
      pick = j;
      found = true;
    }
  }
  out[shot] = c0 + lane * per + pick;
}

// ---------------------------------------------------------------------------
// Partial measurement.
// ---------------------------------------------------------------------------
struct PosArgs {
  int32_t m;
  int32_t pos[24];
};

__device__ __forceinline__ uint64_t gather_bits(uint64_t i, const PosArgs& p)
{
  uint64_t o = 0;
  for (int j = 0; j < p.m; ++j) o |= ((i >> p.pos[j]) & 1ull) << j;
  return o;
}

// All that k_outcome_hist_lds is told, in one cache line: arguments come from host
// memory (one bit of 13 qubits 40.6 -> 40.1 us a call against 240 bytes of them).
template <typename T>
struct HistArgs {
  const T* psi;
  double* hist;
  uint64_t S, walk, mask;
  uint8_t pos[12], m, pad[3];   // 63 from m on: no chain of loads, none set
  uint64_t out;                 // four bits each: outcome bits of the walked measured bits, lowest first
  __device__ __forceinline__ uint32_t gather(uint64_t i) const
  {
    uint32_t o = 0;
#pragma unroll
    for (int j = 0; j < 12; ++j) o |= (uint32_t)((i >> pos[j]) & 1ull) << j;
    return o;
  }
  __device__ __forceinline__ uint32_t outer(int q) const { return 1u << ((out >> (4 * q)) & 15u); }
};
static_assert(sizeof(HistArgs<double>) == 64);

// Weights of the outcomes of m <= 12 measured bits. Thread t of a block takes the
// amplitudes whose low bits are t; it walks the subsets of `walk`, index bits
// above those, with the measured ones outermost and eight loads in flight, so a
// sum stays in a register while the outcome does. It is then summed over the
// lanes with the same outcome and added to the block's LDS histogram. One LDS
// atomic per amplitude before, up to 64 lanes on one address: the three measured
// bits of 24 qubits, complex128, 102 us; now 49 us, the time of the read. RUNS: at
// least eight amplitudes of an outcome in a row. A launch fetches its code cold,
// so that case has a kernel of its own, half as long: in one body with the other
// a call took 1 us more at 13 qubits and 3 more at 24.
template <typename R, bool RUNS>
__global__ __launch_bounds__(kBlock) void k_outcome_hist_lds(const HistArgs<typename VT<R>::T> p)
{
  using T = typename VT<R>::T;
  const T* __restrict__ psi = p.psi;
  double* __restrict__ hist = p.hist;
  const uint64_t S = p.S, walk = p.walk, mask = p.mask;
  extern __shared__ double h[];
  constexpr uint32_t kFly = 8;
  const int no = 1 << p.m;
  for (int k = threadIdx.x; k < no; k += kBlock) h[k] = 0.0;
  __syncthreads();
  const uint32_t t = threadIdx.x, lane = t & 63u;
  uint64_t first = (uint64_t)blockIdx.x * kBlock;
  for (uint64_t r = walk; r; r &= r - 1) {   // the block's number in the bits that are not walked
    const uint64_t below = (r & (0 - r)) - 1;
    first = ((first & ~below) << 1) | (first & below);
  }
  const bool in = first + t < S;   // (a state of less than a block)
  uint64_t outer = walk & mask, inner = walk & ~mask;
  const int run_log = __popcll(inner);
  const uint32_t total = 1u << __popcll(walk), runs = 1u << run_log;
  const uint32_t same = ~(uint32_t)mask & 63u;   // lane bits the outcome does not see
  // An outcome is that of the first amplitude and of the walk's place: E outcomes in
  // a row differ in the lowest measured bits of the walk.
  const uint32_t mine = p.gather(first) | p.gather(t);
  uint64_t d[3];   // the walk's first three bits: the eight loads in flight
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    uint64_t& from = inner ? inner : outer;
    d[j] = from & (0 - from);
    from &= ~d[j];
  }
  uint64_t o = 0, k = 0;   // the rest of it: subsets of the outer and, within, of the inner bits
  auto off = [&](uint32_t f) { return (f & 1 ? d[0] : 0) + (f & 2 ? d[1] : 0) + (f & 4 ? d[2] : 0); };
  const uint32_t each = RUNS ? runs : kFly;   // amplitudes a round
  for (uint32_t l = 0; l < total; l += each) {
    double w[kFly];
    uint32_t E = 1;
    if constexpr (RUNS) {   // one outcome
      double acc = 0.0;
      do {
        const T* at = psi + (first + o + k);
        T v[kFly];
#pragma unroll
        for (uint32_t f = 0; f < kFly; ++f) v[f] = (at + off(f))[t];
#pragma unroll
        for (uint32_t f = 0; f < kFly; ++f) w[f] = (double)v[f].x * v[f].x + (double)v[f].y * v[f].y;
        acc += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
        k = (k - inner) & inner;
      } while (k);
      w[0] = acc;
    } else {
      const T* at = psi + (first + o);
      T v[kFly];
      if (total >= kFly) {
#pragma unroll
        for (uint32_t f = 0; f < kFly; ++f) v[f] = (at + off(f))[t];
      } else {
#pragma unroll
        for (uint32_t f = 0; f < kFly; ++f) {
          v[f].x = v[f].y = R(0);
          if (f < total && in) v[f] = (at + off(f))[t];
        }
      }
#pragma unroll
      for (uint32_t f = 0; f < kFly; ++f) w[f] = (double)v[f].x * v[f].x + (double)v[f].y * v[f].y;
      if (runs == 4) {
        w[0] = (w[0] + w[1]) + (w[2] + w[3]);
        w[1] = (w[4] + w[5]) + (w[6] + w[7]);
      } else if (runs == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = w[2 * e] + w[2 * e + 1];
      }
      E = (total < kFly ? total : kFly) / runs;
    }
    o = (o - outer) & outer;
    // Sums over the lanes with the same outcomes: of E outcomes each lane keeps one
    // half and hands the other to its partner, and the last one is summed as usual:
    // eight outcomes take 10 exchanges and one atomic instead of 48 and eight.
    uint32_t to = mine, idle = 0;
    int q = 0;
    for (uint32_t c = l >> run_log; c; c >>= 1, ++q) to |= c & 1 ? p.outer(q) : 0;
    for (uint32_t left = same; left; left &= left - 1) {
      const uint32_t bit = left & (0 - left);
      const bool up = lane & bit;
      if (RUNS || E == 1) {
        w[0] += __shfl_xor(w[0], bit, 64);
        idle |= bit;
      } else if (E == 8) {
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = (up ? w[e + 4] : w[e]) + __shfl_xor(up ? w[e] : w[e + 4], bit, 64);
        to |= up ? p.outer(2) : 0;
        E = 4;
      } else if (E == 4) {
#pragma unroll
        for (int e = 0; e < 2; ++e) w[e] = (up ? w[e + 2] : w[e]) + __shfl_xor(up ? w[e] : w[e + 2], bit, 64);
        to |= up ? p.outer(1) : 0;
        E = 2;
      } else {
        w[0] = (up ? w[1] : w[0]) + __shfl_xor(up ? w[0] : w[1], bit, 64);
        to |= up ? p.outer(0) : 0;
        E = 1;
      }
    }
    if (!(lane & idle) && in) {
#pragma unroll
      for (uint32_t e = 0; e < (RUNS ? 1 : kFly); ++e)
        if (e < E)
          atomicAdd(&h[to | (e & 1 ? p.outer(0) : 0) | (e & 2 ? p.outer(1) : 0) | (e & 4 ? p.outer(2) : 0)], w[e]);
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < no; k += kBlock)
    if (h[k] != 0.0) atomicAdd(&hist[k], h[k]);
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_outcome_hist_global(const typename VT<R>::T* __restrict__ psi,
                                                                 uint64_t S, PosArgs p, double* __restrict__ hist)
{
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < S; i += stride) {
    const auto a = psi[i];
    const double v = (double)a.x * a.x + (double)a.y * a.y;
    if (v != 0.0) atomicAdd(&hist[gather_bits(i, p)], v);
  }
}

__global__ __launch_bounds__(kBlock) void k_zero_f64(double* __restrict__ v, uint64_t n)
{
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) v[i] = 0.0;
}

// Scales the amplitudes whose measured bits (mask) read `want`; the others are
// set to zero unread. Three measured bits of 24 qubits, complex128: 65 us with
// every amplitude read, now 37 us.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_collapse(typename VT<R>::T* __restrict__ psi, uint64_t S, uint64_t mask,
                                                      uint64_t want, R scale)
{
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < S; i += stride) {
    typename VT<R>::T a;
    a.x = a.y = R(0);
    if ((i & mask) == want) {
      a = psi[i];
      a.x *= scale;
      a.y *= scale;
    }
    psi[i] = a;
  }
}

// ---------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------
static inline unsigned stream_grid(uint64_t S)
{
  uint64_t g = (S + kBlock - 1) / kBlock;
  const uint64_t cap = 256ull * 64;  // 64 workgroups per CU on 256 CUs
  return (unsigned)(g < 1 ? 1 : (g > cap ? cap : g));
}

void launch_fill_basis(int prec, void* psi, uint64_t S, uint64_t idx, hipStream_t st)
{
  const unsigned g = stream_grid(S);
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_fill_basis<double>), dim3(g), dim3(kBlock), 0, st, (double2*)psi, S, idx);
  else
    hipLaunchKernelGGL((k_fill_basis<float>), dim3(g), dim3(kBlock), 0, st, (float2*)psi, S, idx);
}

void launch_copy(int prec, const void* src, void* dst, uint64_t S, hipStream_t st)
{
  const unsigned g = (unsigned)((S + kBlock * 4 - 1) / (kBlock * 4));
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_copy<double>), dim3(g), dim3(kBlock), 0, st, (const double2*)src, (double2*)dst, S);
  else
    hipLaunchKernelGGL((k_copy<float>), dim3(g), dim3(kBlock), 0, st, (const float2*)src, (float2*)dst, S);
}

void launch_compare(int pa, const void* a, int pb, const void* b, uint64_t S, double* partials, double* out,
                    hipStream_t st)
{
  const dim3 g(kReduceBlocks), blk(kBlock);
  if (pa == QSV_C128 && pb == QSV_C128)
    hipLaunchKernelGGL((k_compare<double, double>), g, blk, 0, st, (const double2*)a, (const double2*)b, S, partials);
  else if (pa == QSV_C128)
    hipLaunchKernelGGL((k_compare<double, float>), g, blk, 0, st, (const double2*)a, (const float2*)b, S, partials);
  else if (pb == QSV_C128)
    hipLaunchKernelGGL((k_compare<float, double>), g, blk, 0, st, (const float2*)a, (const double2*)b, S, partials);
  else
    hipLaunchKernelGGL((k_compare<float, float>), g, blk, 0, st, (const float2*)a, (const float2*)b, S, partials);
  hipLaunchKernelGGL(k_final_sum, dim3(4), blk, 0, st, partials, out);
  hipLaunchKernelGGL(k_final_max, dim3(1), blk, 0, st, partials + 4ull * kReduceBlocks, out + 4);
}

void launch_scale(int prec, void* psi, uint64_t S, double f, hipStream_t st)
{
  const unsigned g = stream_grid(S);
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_scale<double>), dim3(g), dim3(kBlock), 0, st, (double2*)psi, S, f);
  else
    hipLaunchKernelGGL((k_scale<float>), dim3(g), dim3(kBlock), 0, st, (float2*)psi, S, (float)f);
}

void launch_renorm(int prec, void* psi, uint64_t S, double* partials, double* out, hipStream_t st)
{
  launch_norm2(prec, psi, S, partials, out, st);
  const unsigned g = stream_grid(S);
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_scale_by_norm<double>), dim3(g), dim3(kBlock), 0, st, (double2*)psi, S, out);
  else
    hipLaunchKernelGGL((k_scale_by_norm<float>), dim3(g), dim3(kBlock), 0, st, (float2*)psi, S, out);
}

void launch_f64_to_c64(const double* src, void* dst, uint64_t count, hipStream_t st)
{
  hipLaunchKernelGGL(k_f64_to_c64, dim3(stream_grid(count)), dim3(kBlock), 0, st, (const double2*)src, (float2*)dst,
                     count);
}

void launch_c64_to_f64(const void* src, double* dst, uint64_t count, hipStream_t st)
{
  hipLaunchKernelGGL(k_c64_to_f64, dim3(stream_grid(count)), dim3(kBlock), 0, st, (const float2*)src, (double2*)dst,
                     count);
}

void launch_norm2(int prec, const void* psi, uint64_t S, double* partials, double* out, hipStream_t st)
{
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_norm2<double>), dim3(kReduceBlocks), dim3(kBlock), 0, st, (const double2*)psi, S, partials);
  else
    hipLaunchKernelGGL((k_norm2<float>), dim3(kReduceBlocks), dim3(kBlock), 0, st, (const float2*)psi, S, partials);
  hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(kBlock), 0, st, partials, out);
}

void launch_inner(int prec, const void* a, const void* b, uint64_t S, double* partials, double* out, hipStream_t st)
{
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_inner<double>), dim3(kReduceBlocks), dim3(kBlock), 0, st, (const double2*)a,
                       (const double2*)b, S, partials);
  else
    hipLaunchKernelGGL((k_inner<float>), dim3(kReduceBlocks), dim3(kBlock), 0, st, (const float2*)a,
                       (const float2*)b, S, partials);
  hipLaunchKernelGGL(k_final_sum, dim3(2), dim3(kBlock), 0, st, partials, out);
}

void launch_expect1q(int prec, const void* psi, uint64_t S, uint64_t tbit, const double m[8], double* partials,
                     double* out, hipStream_t st)
{
  Mat2<double> M;
  for (int k = 0; k < 8; ++k) M.m[k] = m[k];
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_expect1q<double>), dim3(kReduceBlocks), dim3(kBlock), 0, st, (const double2*)psi, S / 2,
                       tbit, M, partials);
  else
    hipLaunchKernelGGL((k_expect1q<float>), dim3(kReduceBlocks), dim3(kBlock), 0, st, (const float2*)psi, S / 2,
                       tbit, M, partials);
  hipLaunchKernelGGL(k_final_sum, dim3(2), dim3(kBlock), 0, st, partials, out);
}

void launch_probs(int prec, const void* psi, uint64_t offset, uint64_t count, double* out, hipStream_t st)
{
  const unsigned g = stream_grid(count);
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_probs<double>), dim3(g), dim3(kBlock), 0, st, (const double2*)psi, offset, count, out);
  else
    hipLaunchKernelGGL((k_probs<float>), dim3(g), dim3(kBlock), 0, st, (const float2*)psi, offset, count, out);
}

void launch_sample(int prec, const void* psi, uint64_t S, double* chunk_prefix, uint64_t shots, uint64_t seed,
                   uint64_t* out, hipStream_t st)
{
  int n = 0;
  while ((1ull << n) < S) ++n;
  const int chunk_log = n < kSampleChunkLog ? n : kSampleChunkLog;
  const uint64_t nchunks = S >> chunk_log;
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_chunk_sums<double>), dim3((unsigned)nchunks), dim3(kBlock), 0, st, (const double2*)psi,
                       chunk_log, chunk_prefix);
  else
    hipLaunchKernelGGL((k_chunk_sums<float>), dim3((unsigned)nchunks), dim3(kBlock), 0, st, (const float2*)psi,
                       chunk_log, chunk_prefix);
  const uint64_t groups = (nchunks + (1ull << kGroupLog) - 1) >> kGroupLog;
  hipLaunchKernelGGL(k_scan_groups, dim3((unsigned)groups), dim3(kBlock), 0, st, chunk_prefix, nchunks);
  if (groups > 1) hipLaunchKernelGGL(k_scan_totals, dim3(1), dim3(1024), 0, st, chunk_prefix, groups);
  if (shots == 0) return;
  const unsigned g = (unsigned)((shots + (kBlock / 64) - 1) / (kBlock / 64));
  // The two ways meet at about 2000 shots (calls of 1000, 2000, 4000 and 65536 shots
  // from 18 qubits, few / many: 34.5 / 38.5, 39.6 / 38.7, 49.5 / 42.4, 303 / 144 us).
  const bool many = shots > 2048;
  auto run = [&](auto kernel, auto* amps) {
    hipLaunchKernelGGL(kernel, dim3(g), dim3(kBlock), 0, st, amps, S, chunk_log, chunk_prefix, nchunks, shots, seed,
                       out);
  };
  if (prec == QSV_C128) {
    if (many) run(k_sample<double, true>, (const double2*)psi);
    else run(k_sample<double, false>, (const double2*)psi);
  } else {
    if (many) run(k_sample<float, true>, (const float2*)psi);
    else run(k_sample<float, false>, (const float2*)psi);
  }
}

void launch_outcome_hist(int prec, const void* psi, uint64_t S, int m, const int* pos, double* hist, hipStream_t st)
{
  PosArgs p{};
  p.m = m;
  for (int j = 0; j < m; ++j) p.pos[j] = pos[j];
  const uint64_t no = 1ull << m;
  hipLaunchKernelGGL(k_zero_f64, dim3(stream_grid(no)), dim3(kBlock), 0, st, hist, no);
  if (m <= 12) {
    uint64_t mask = 0;
    for (int j = 0; j < m; ++j) mask |= 1ull << pos[j];
    // At most 512 blocks, 1024 where the read dominates: each adds its outcomes to
    // the same few global sums (one measured bit of 20 qubits: 51 us a call with 256
    // blocks, 56 with 512, 63 with 1024; of 22 qubits 73 with 512, 77 with 1024). 16
    // amplitudes a thread, 8 below 2^20 (one round of loads). A thread walks bits
    // that are not measured as long as there are any, so its sums are few (the nine
    // middle qubits of 22: 98 us when it walked the next bits above its own, 63 now;
    // one LDS atomic an amplitude 78). The highest of them up to 64 MiB, where blocks
    // side by side then read side by side (one bit of 20 qubits 46 / 52 us, six of 22
    // 61 / 67); the lowest above (six of 24: 129 / 119) and with 12 measured bits,
    // whose blocks then meet fewer outcomes (of 16 qubits 59 / 47).
    const int n = 63 - __builtin_clzll(S), block = 8;
    int walked = 0;
    uint64_t walk = 0;
    if (n > block) {
      const uint64_t above = (S - 1) & ~(uint64_t)(kBlock - 1);
      const uint64_t from[2] = {above & ~mask, above & mask};
      const bool high = m < 12 && S * (prec == QSV_C128 ? 16 : 8) <= 64ull << 20;
      walked = std::max(n - block - (n >= 23 ? 10 : 9), std::min(n >= 20 ? 4 : 3, __builtin_popcountll(from[0])));
      int left = walked;
      for (uint64_t r : from)
        for (; r && left; --left) {
          const uint64_t bit = high ? 1ull << (63 - __builtin_clzll(r)) : r & (0 - r);
          walk |= bit;
          r &= ~bit;
        }
    }
    const unsigned g = n > block ? (unsigned)(S >> (block + walked)) : 1u;
    auto run = [&](auto kernel, auto* amps) {
      HistArgs<std::remove_const_t<std::remove_pointer_t<decltype(amps)>>> a{amps, hist, S, walk, mask};
      a.m = (uint8_t)m;
      for (int j = 0; j < 12; ++j) a.pos[j] = (uint8_t)(j < m ? pos[j] : 63);
      int q = 0;
      for (uint64_t r = walk & mask; r; r &= r - 1, ++q)
        for (int j = 0; j < m; ++j)
          if ((r & (0 - r)) == 1ull << pos[j]) a.out |= (uint64_t)j << (4 * q);
      hipLaunchKernelGGL(kernel, dim3(g), dim3(kBlock), no * sizeof(double), st, a);
    };
    const bool runs = __builtin_popcountll(walk & ~mask) >= 3;   // eight amplitudes of one outcome and more
    if (prec == QSV_C128) {
      if (runs) run(k_outcome_hist_lds<double, true>, (const double2*)psi);
      else run(k_outcome_hist_lds<double, false>, (const double2*)psi);
    } else {
      if (runs) run(k_outcome_hist_lds<float, true>, (const float2*)psi);
      else run(k_outcome_hist_lds<float, false>, (const float2*)psi);
    }
  } else {
    if (prec == QSV_C128)
      hipLaunchKernelGGL((k_outcome_hist_global<double>), dim3(stream_grid(S)), dim3(kBlock), 0, st,
                         (const double2*)psi, S, p, hist);
    else
      hipLaunchKernelGGL((k_outcome_hist_global<float>), dim3(stream_grid(S)), dim3(kBlock), 0, st,
                         (const float2*)psi, S, p, hist);
  }
}

void launch_collapse(int prec, void* psi, uint64_t S, int m, const int* pos, uint64_t sel, double scale,
                     hipStream_t st)
{
  uint64_t mask = 0, want = 0;
  for (int j = 0; j < m; ++j) {
    mask |= 1ull << pos[j];
    want |= ((sel >> j) & 1ull) << pos[j];
  }
  const unsigned g = stream_grid(S);
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_collapse<double>), dim3(g), dim3(kBlock), 0, st, (double2*)psi, S, mask, want, scale);
  else
    hipLaunchKernelGGL((k_collapse<float>), dim3(g), dim3(kBlock), 0, st, (float2*)psi, S, mask, want, (float)scale);
}

}  // namespace qsv
