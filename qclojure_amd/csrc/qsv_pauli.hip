// qsv_pauli.hip — Pauli-string expectations, many strings per state read.
//
// <P> of a string with X part x and sign part s (Y counts in both) is, up to
// (-i)^#Y, the sum over i of (-1)^popc(i & s) conj(a_i) a_{i ^ x}. The terms of
// i and i ^ x are conjugates up to the sign (-1)^#Y, so half the pairs and one
// real component (Re for an even #Y, Im for an odd one) give the value.
//
// k_pauli_tile (large states): a workgroup holds a tile of 2^12 amplitudes
// (12 index bits, the low ones among them for whole cache lines) and serves
// every string of the sweep from it:
//   * Z strings: a Walsh-Hadamard transform of the tile's probabilities (three
//     radix-16 rounds, 12 additions an amplitude, FP64) leaves in W[m] the sum
//     of (-1)^popc(l & m) p_l; each string is then one LDS read by one thread;
//   * strings whose X part lies in the tile bits: pairs are read from LDS, two
//     strings that share the X part per read, and eight sums are reduced over
//     the wave together (10 lane exchanges instead of 48).
// The state is read once per sweep whatever the number of strings, so the
// sweep is bound by HBM for Z strings and by LDS reads (16 B an amplitude and
// X part) otherwise. The kernel before this one kept eight strings in
// registers, paid a popcount and a select per string and amplitude and re-read
// partners from memory. One MI355X, complex128: 27 <Z> of 27 qubits, 4 launches
// of 1308 us before, one of 396 us (5.4 TB/s) now; the 97 strings of a 25-qubit
// Heisenberg chain 13 launches of 481 us before, 3 sweeps of 216 us now.
//
// k_energy_tile (batches): <H> of a Z-string Hamiltonian on each of many states,
// a tile's strings summed with their coefficients as soon as its transform is
// done. Bound by the read of the states. Popcount, select and addition per
// string and amplitude, as before: six groups of MaxCut states of 15 to 20
// qubits, complex64, 819 us; now 153 us.
//
// k_pauli_direct (small states, and X parts wider than a tile): one grid row
// per string over the pairs of that string alone.
#include "qsv_internal.h"

namespace qsv {

namespace {

template <typename R> struct QV;
template <> struct QV<double> { typedef double T __attribute__((ext_vector_type(2))); };
template <> struct QV<float> { typedef float T __attribute__((ext_vector_type(2))); };

constexpr int kTB = 12;
constexpr uint32_t kTile = 1u << kTB;

// XOR-linear bank swizzle of a tile-local index: it rewrites the low four
// bits, so accesses that step by 16 or 256 elements spread over the banks.
__device__ __forceinline__ uint32_t pswz(uint32_t l) { return l ^ (((l >> 4) ^ (l >> 8)) & 15u); }

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

__device__ __forceinline__ void wht16(double (&p)[16])
{
#pragma unroll
  for (int h = 1; h < 16; h <<= 1)
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (!(k & h)) {
        const double a = p[k], b = p[k | h];
        p[k] = a + b;
        p[k | h] = a - b;
      }
}

__device__ __forceinline__ double sign_of(uint64_t bits) { return (__popcll(bits) & 1) ? -1.0 : 1.0; }

}  // namespace

// Persistent workgroups over the tiles; partials[item * gridDim.x + block].
// Items: the nz Z strings, then two per X unit. X: the sweep has X units (its
// tile is kept in LDS as complex numbers; without it only the FP64 plane of
// the transform is).
template <typename R, bool X>
__global__ __launch_bounds__(kBlock) void k_pauli_tile(const typename QV<R>::T* __restrict__ psi, uint64_t ntiles,
                                                       PauliSweep sw, double* __restrict__ partials)
{
  using T = typename QV<R>::T;
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr uint32_t kBuf = X && sizeof(T) == 16 ? kTile * 16 : kTile * 8;
  double* W = reinterpret_cast<double*>(smem);
  T* tile = reinterpret_cast<T*>(smem);
  double* acc = reinterpret_cast<double*>(smem + kBuf);   // [4 waves][2 * kPauliUnits]
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
  // this thread's part of the load addresses (local bits 0..7 = thread bits)
  uint64_t gt = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) gt |= ((t >> j) & 1u) ? (1ull << sw.pos[j]) : 0ull;
  uint64_t gs[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) gs[j] = 1ull << sw.pos[8 + j];
  auto base_of = [&](uint64_t b) {
#pragma unroll
    for (int i = 0; i < kTB; ++i) {
      const int p = sw.pos[i];
      const uint64_t lo = b & ((1ull << p) - 1ull);
      b = ((b ^ lo) << 1) | lo;
    }
    return b;
  };
  T v[16];
  auto load = [&](uint64_t base) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const uint64_t g = base | gt | ((k & 1) ? gs[0] : 0ull) | ((k & 2) ? gs[1] : 0ull) | ((k & 4) ? gs[2] : 0ull) |
                         ((k & 8) ? gs[3] : 0ull);
      v[k] = psi[g];
    }
  };
  const bool has_z = t < (uint32_t)sw.nz;
  const uint64_t zs = has_z ? sw.zmask[t] : 0ull;
  uint32_t zl = 0;   // the string's tile-local bits
#pragma unroll
  for (int i = 0; i < kTB; ++i) zl |= (uint32_t)((zs >> sw.pos[i]) & 1ull) << i;
  double zacc = 0.0;
  if constexpr (X)
    for (uint32_t e = t; e < 4u * 2u * kPauliUnits; e += kBlock) acc[e] = 0.0;

  uint64_t tl = blockIdx.x;
  uint64_t base = base_of(tl);
  if (tl < ntiles) load(base);
  for (; tl < ntiles; tl += gridDim.x) {
    const uint64_t next = tl + gridDim.x;
    const uint64_t nbase = base_of(next);
    __syncthreads();   // the previous tile's LDS is no longer read
    if (sw.nz) {
      double p[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) p[k] = (double)v[k].x * v[k].x + (double)v[k].y * v[k].y;
      if (!X && next < ntiles) load(nbase);   // in flight during the transform
      wht16(p);   // local bits 8..11
#pragma unroll
      for (int k = 0; k < 16; ++k) W[pswz(t | (uint32_t)k << 8)] = p[k];
      __syncthreads();
      const uint32_t m = (t & 15u) | (t >> 4) << 8;
#pragma unroll
      for (int k = 0; k < 16; ++k) p[k] = W[pswz(m | (uint32_t)k << 4)];
      wht16(p);   // local bits 4..7
#pragma unroll
      for (int k = 0; k < 16; ++k) W[pswz(m | (uint32_t)k << 4)] = p[k];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 16; ++k) p[k] = W[pswz(t << 4 | (uint32_t)k)];
      wht16(p);   // local bits 0..3
#pragma unroll
      for (int k = 0; k < 16; ++k) W[pswz(t << 4 | (uint32_t)k)] = p[k];
      __syncthreads();
      if (has_z) zacc += sign_of(base & zs) * W[pswz(zl)];
      if constexpr (X) __syncthreads();   // W and the complex tile share the LDS
    }
    if constexpr (X) {
#pragma unroll
      for (int k = 0; k < 16; ++k) tile[pswz(t | (uint32_t)k << 8)] = v[k];
      __syncthreads();
      if (next < ntiles) load(nbase);   // in flight while the strings are summed
      for (int u0 = 0; u0 < sw.nu; u0 += 4) {
        double s8[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const PauliUnit& u = sw.u[u0 + q];   // padded to a multiple of four with zero weights
          const uint32_t x = u.x, b = u.top;   // top: index of x's highest bit
          auto ins = [&](uint32_t j) { return ((j >> b) << (b + 1)) | (j & ((1u << b) - 1u)); };
          const uint32_t it = ins(t);
          const uint32_t at = pswz(it), xs = pswz(x);
          double v0 = 0.0, v1 = 0.0;
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const uint32_t ik = ins((uint32_t)k << 8);
            const uint32_t a0 = at ^ pswz(ik);
            const T a = tile[a0], c = tile[a0 ^ xs];
            const double ar = a.x, ai = a.y, br = c.x, bi = c.y;
            const double re = ar * br + ai * bi, im = ar * bi - ai * br;
            const double c0 = u.im0 ? im : re, c1 = u.im1 ? im : re;
            v0 += ((__popc(ik & u.s0) & 1) ? -1.0 : 1.0) * c0;
            v1 += ((__popc(ik & u.s1) & 1) ? -1.0 : 1.0) * c1;
          }
          // signs of the thread's own bits and of the tile
          const uint64_t h0 = base & u.g0, h1 = base & u.g1;
          s8[2 * q] = ((__popc(it & u.s0) + __popcll(h0)) & 1) ? -v0 : v0;
          s8[2 * q + 1] = ((__popc(it & u.s1) + __popcll(h1)) & 1) ? -v1 : v1;
        }
        // eight sums over 64 lanes: after three halving exchanges lane L holds
        // its eighth of sum L >> 3
#pragma unroll
        for (int h = 4, m = 32; h >= 1; h >>= 1, m >>= 1)
#pragma unroll
          for (int j = 0; j < h; ++j) {
            const bool up = (lane & (uint32_t)m) != 0;
            const double keep = up ? s8[j + h] : s8[j], send = up ? s8[j] : s8[j + h];
            s8[j] = keep + __shfl_xor(send, m, 64);
          }
        double r = s8[0];
#pragma unroll
        for (int m = 4; m >= 1; m >>= 1) r += __shfl_xor(r, m, 64);
        if ((lane & 7u) == 0) acc[w * 2 * kPauliUnits + 2 * u0 + (lane >> 3)] += r;
      }
    }
    base = nbase;
  }
  const uint64_t nb = gridDim.x;
  if (has_z) partials[(uint64_t)t * nb + blockIdx.x] = zacc;
  if constexpr (X) {
    __syncthreads();
    for (uint32_t e = t; e < 2u * (uint32_t)sw.nu; e += kBlock)
      partials[((uint64_t)sw.nz + e) * nb + blockIdx.x] =
          (acc[e] + acc[2 * kPauliUnits + e]) + (acc[4 * kPauliUnits + e] + acc[6 * kPauliUnits + e]);
  }
}

// One string per grid row: partials[row * gridDim.x + block] (straight into
// the result when the row has one block).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_pauli_direct(const typename QV<R>::T* __restrict__ psi, uint64_t S,
                                                         PauliRows rows, double* __restrict__ partials)
{
  __shared__ double sh[kBlock / 64];
  const uint64_t x = rows.x[blockIdx.y], s = rows.s[blockIdx.y];
  const bool im = (rows.im >> blockIdx.y) & 1ull;
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  uint64_t j = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  double acc = 0.0;
  if (x == 0) {
    for (; j < S; j += stride) {
      const auto a = psi[j];
      acc += sign_of(j & s) * ((double)a.x * a.x + (double)a.y * a.y);
    }
  } else {
    const uint64_t lo = (1ull << (63 - __clzll(x))) - 1ull;
    for (; j < S / 2; j += stride) {
      const uint64_t i = ((j & ~lo) << 1) | (j & lo);
      const auto a = psi[i];
      const auto b = psi[i ^ x];
      const double ar = a.x, ai = a.y, br = b.x, bi = b.y;
      acc += sign_of(i & s) * (im ? ar * bi - ai * br : ar * br + ai * bi);
    }
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partials[(uint64_t)blockIdx.y * gridDim.x + blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// out[item] = fixed-order sum of the item's nb partials.
__global__ __launch_bounds__(kBlock) void k_pauli_final(const double* __restrict__ partials, uint32_t nb,
                                                        double* __restrict__ out)
{
  __shared__ double sh[kBlock / 64];
  const double* p = partials + (uint64_t)blockIdx.x * nb;
  double acc = 0.0;
  for (uint32_t i = threadIdx.x; i < nb; i += kBlock) acc += p[i];
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

namespace {

template <typename R, bool X>
hipError_t sweep_launch(const void* psi, uint64_t S, const PauliSweep& sw, double* partials, double* out,
                        hipStream_t st)
{
  constexpr size_t kBuf = X && sizeof(R) == 8 ? kTile * 16 : kTile * 8;
  constexpr size_t kLds = kBuf + (X ? sizeof(double) * 4 * 2 * kPauliUnits : 0);
  const uint64_t ntiles = S >> kTB;
  // resident workgroups: two per CU with a complex128 tile (67 KiB of the
  // 160), four without X units
  const uint64_t cap = X ? kPauliXBlocks : kReduceBlocks;
  const unsigned grid = (unsigned)(ntiles < cap ? ntiles : cap);
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pauli_tile<R, X>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_pauli_tile<R, X>), dim3(grid), dim3(kBlock), kLds, st, (const typename QV<R>::T*)psi, ntiles,
                     sw, partials);
  hipLaunchKernelGGL(k_pauli_final, dim3((unsigned)(sw.nz + 2 * sw.nu)), dim3(kBlock), 0, st, (const double*)partials,
                     grid, out);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_pauli_sweep(int prec, const void* psi, uint64_t S, const PauliSweep& sw, double* partials,
                              double* out, hipStream_t st)
{
  if (prec == QSV_C128)
    return sw.nu ? sweep_launch<double, true>(psi, S, sw, partials, out, st)
                 : sweep_launch<double, false>(psi, S, sw, partials, out, st);
  return sw.nu ? sweep_launch<float, true>(psi, S, sw, partials, out, st)
               : sweep_launch<float, false>(psi, S, sw, partials, out, st);
}

hipError_t launch_pauli_rows(int prec, const void* psi, uint64_t S, const PauliRows& rows, int n, double* partials,
                             double* out, hipStream_t st)
{
  // 2048 amplitudes per workgroup, at most the partials' room per string
  const uint64_t want = (S + 2047) / 2048, cap = kReduceBlocks;
  const unsigned nb = (unsigned)(want < cap ? want : cap);
  double* dst = nb == 1 ? out : partials;
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_pauli_direct<double>), dim3(nb, n), dim3(kBlock), 0, st, (const QV<double>::T*)psi, S, rows,
                       dst);
  else
    hipLaunchKernelGGL((k_pauli_direct<float>), dim3(nb, n), dim3(kBlock), 0, st, (const QV<float>::T*)psi, S, rows,
                       dst);
  if (nb > 1)
    hipLaunchKernelGGL(k_pauli_final, dim3(n), dim3(kBlock), 0, st, (const double*)partials, nb, out);
  return hipGetLastError();
}

// Block (x, y) sums its share of state y, whose strings are tz[t0..t1) (trange:
// per state), into partials[y * gridDim.x + x]. S is a multiple of the tile.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_energy_tile(const typename QV<R>::T* __restrict__ states, uint64_t S,
                                                        const uint64_t* __restrict__ tz,
                                                        const double* __restrict__ tc,
                                                        const uint64_t* __restrict__ trange, uint64_t t0, uint64_t t1,
                                                        double* __restrict__ partials)
{
  __shared__ double W[kTile];
  __shared__ double red[4];
  const uint32_t t = threadIdx.x;
  const uint64_t y = blockIdx.y;
  const auto* psi = states + y * S;
  if (trange) {
    t0 = trange[2 * y];
    t1 = trange[2 * y + 1];
  }
  double acc = 0.0;
  for (uint64_t base = (uint64_t)blockIdx.x << kTB; base < S; base += (uint64_t)gridDim.x << kTB) {
    double p[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const auto v = psi[base + t + ((uint32_t)k << 8)];
      p[k] = (double)v.x * v.x + (double)v.y * v.y;
    }
    wht16(p);   // bits 8..11
    __syncthreads();   // the previous tile's transform is no longer read
#pragma unroll
    for (int k = 0; k < 16; ++k) W[pswz(t | (uint32_t)k << 8)] = p[k];
    __syncthreads();
    const uint32_t m = (t & 15u) | (t >> 4) << 8;
#pragma unroll
    for (int k = 0; k < 16; ++k) p[k] = W[pswz(m | (uint32_t)k << 4)];
    wht16(p);   // bits 4..7
#pragma unroll
    for (int k = 0; k < 16; ++k) W[pswz(m | (uint32_t)k << 4)] = p[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) p[k] = W[pswz(t << 4 | (uint32_t)k)];
    wht16(p);   // bits 0..3
#pragma unroll
    for (int k = 0; k < 16; ++k) W[pswz(t << 4 | (uint32_t)k)] = p[k];
    __syncthreads();
    for (uint64_t k = t0 + t; k < t1; k += kBlock) {
      const uint64_t z = tz[k];
      acc += sign_of(base & z) * tc[k] * W[pswz((uint32_t)z & (kTile - 1u))];
    }
  }
  acc = wave_sum(acc);
  if ((t & 63u) == 0) red[t >> 6] = acc;
  __syncthreads();
  if (t == 0) partials[y * gridDim.x + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// out[dest[y]] = fixed-order sum of the nb partials of state y (out[y] without dest).
__global__ __launch_bounds__(64) void k_sum_group(const double* __restrict__ partials, uint32_t nb,
                                                  const uint64_t* __restrict__ dest, double* __restrict__ out)
{
  const uint64_t y = blockIdx.x;
  double acc = 0.0;
  for (uint32_t k = threadIdx.x; k < nb; k += 64) acc += partials[y * nb + k];
  acc = wave_sum(acc);
  if (threadIdx.x == 0) out[dest ? dest[y] : y] = acc;
}

static void energy_launch(int prec, const void* states, uint64_t S, unsigned count, const uint64_t* tz,
                          const double* tc, const uint64_t* trange, uint64_t nterms, double* partials, unsigned blocks,
                          const uint64_t* dest, double* out, hipStream_t st)
{
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_energy_tile<double>), dim3(blocks, count), dim3(kBlock), 0, st,
                       (const QV<double>::T*)states, S, tz, tc, trange, (uint64_t)0, nterms, partials);
  else
    hipLaunchKernelGGL((k_energy_tile<float>), dim3(blocks, count), dim3(kBlock), 0, st, (const QV<float>::T*)states,
                       S, tz, tc, trange, (uint64_t)0, nterms, partials);
  hipLaunchKernelGGL(k_sum_group, dim3(count), dim3(64), 0, st, partials, blocks, dest, out);
}

void launch_zexpect_group(int prec, const void* base, uint64_t S, unsigned count, const uint64_t* tz,
                          const double* tc, const uint64_t* trange, double* partials, unsigned blocks_per_state,
                          const uint64_t* dest, double* out, hipStream_t st)
{
  if (count) energy_launch(prec, base, S, count, tz, tc, trange, 0, partials, blocks_per_state, dest, out, st);
}

void launch_zexpect(int prec, const void* psi, uint64_t S, const uint64_t* tz, const double* tc, uint64_t nterms,
                    double* partials, double* out, hipStream_t st)
{
  const uint64_t tiles = S >> kTB;
  energy_launch(prec, psi, S, 1, tz, tc, nullptr, nterms, partials,
                (unsigned)(tiles < (uint64_t)kReduceBlocks ? tiles : kReduceBlocks), nullptr, out, st);
}

}  // namespace qsv
