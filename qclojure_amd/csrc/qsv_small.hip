// qsv_small.hip — small circuits: a whole register, a whole program, one workgroup.
//
// A register of n <= 13 (complex128) or 14 (complex64) qubits is one tile of the
// fused passes' micro-op programs: 2^(n - 4) threads hold 16 amplitudes each in
// FP64 registers, layout changes go through LDS, and the program runs from first
// op to last without touching memory for amplitudes. At the end the workgroup
// stores the state, or reduces a Z-string Hamiltonian, or both.
//
// One wave holds up to 10 qubits and needs no barrier at all. The kernel this
// replaces kept the state in LDS and swept it once per gate with a barrier
// after each; a state of fewer than 12 qubits of its own took one launch per
// gate. Bound by the chain of ops (their fetches are hidden by a read of the
// program up front and a fetch one op ahead). Kernel time, before and now: 280
// batched QAOA instances of 8 to 14 qubits 1206 -> 535 us (four size classes),
// 1000 noisy trajectories of 11 qubits 320 -> 85 us, the small requests of a
// served burst 1780 -> 590 us, a 5-qubit program 25 launches -> one of 12 us.
#include "qsv_ops.h"

namespace qsv {

namespace {

// Threads that hold amplitudes of their own.
__device__ __forceinline__ uint32_t live_threads(int n) { return n > 4 ? 1u << (n - 4) : 1u; }

template <int NT, typename T>
__device__ __forceinline__ void load_slots(const T* __restrict__ psi, uint64_t ga, const uint64_t* cols, uint64_t S,
                                           Slots<double>& x)
{
  each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
    constexpr int k = decltype(kk)::value;
    const uint64_t sl = global_slot<k>(cols);
    const bool in = sl < S;
    const T v = psi[in ? ga ^ sl : 0];
    x.re[k] = in ? (double)v.x : 0.0;
    x.im[k] = in ? (double)v.y : 0.0;
  });
}
template <typename R, int NT, typename T>
__device__ __forceinline__ void store_slots(T* __restrict__ psi, uint64_t ga, const uint64_t* cols, uint64_t S,
                                            const Slots<double>& x)
{
  each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
    constexpr int k = decltype(kk)::value;
    const uint64_t sl = global_slot<k>(cols);
    if (sl < S) {
      T v;
      v.x = (R)x.re[k];
      v.y = (R)x.im[k];
      psi[ga ^ sl] = v;
    }
  });
}

// <H> = sum_x |a_x|^2 sum_t c_t (-1)^popc(x & z_t) of the tile in registers. The
// 16 probabilities of a thread become their 16 signed sums (a Walsh-Hadamard
// transform over the slot bits), kept in LDS; a string then costs one LDS read
// and a sign.
template <int NT>
__device__ __forceinline__ double z_energy(const Slots<double>& x, const uint64_t* cols, uint32_t xt, uint32_t live,
                                           char* smem, const uint64_t* __restrict__ tz, const double* __restrict__ tc,
                                           uint64_t t0, uint64_t t1)
{
  const uint32_t t = threadIdx.x, lane = t & 63u, nthr = 1u << NT;
  double* W = reinterpret_cast<double*>(smem);
  double p[16];
  each<0, 16>([&](auto kk) __attribute__((always_inline)) {
    constexpr int k = decltype(kk)::value;
    p[k] = t < live ? x.re[k] * x.re[k] + x.im[k] * x.im[k] : 0.0;
  });
  each<0, 4>([&](auto hh) __attribute__((always_inline)) {
    constexpr int h = 1 << decltype(hh)::value;
    each<0, 16>([&](auto kk) __attribute__((always_inline)) {
      constexpr int k = decltype(kk)::value;
      if constexpr (!(k & h)) {
        const double a = p[k], b = p[k | h];
        p[k] = a + b;
        p[k | h] = a - b;
      }
    });
  });
  __syncthreads();   // the last relayout's LDS is no longer read
  each<0, 16>([&](auto kk) __attribute__((always_inline)) {
    constexpr int k = decltype(kk)::value;
    W[k * nthr + t] = p[k];
  });
  uint32_t r[4];
  each<0, 4>([&](auto ii) __attribute__((always_inline)) { r[decltype(ii)::value] = (uint32_t)cols[kColT + decltype(ii)::value]; });
  double acc = 0.0;
  for (uint64_t b = t0; b < t1; b += 64) {
    const uint64_t at = b + lane;
    const uint32_t zl = at < t1 ? (uint32_t)tz[at] : 0u;
    const double cl = at < t1 ? tc[at] : 0.0;
    const int cnt = (int)(t1 - b < 64 ? t1 - b : 64);
    for (int j = 0; j < cnt; ++j) {
      const uint32_t z = (uint32_t)__builtin_amdgcn_readlane((int)zl, j);
      const int clo = __builtin_amdgcn_readlane(__double2loint(cl), j);
      const int chi = __builtin_amdgcn_readlane(__double2hiint(cl), j);
      const uint32_t m = (__popc(z & r[0]) & 1) | (__popc(z & r[1]) & 1) << 1 | (__popc(z & r[2]) & 1) << 2 |
                         (__popc(z & r[3]) & 1) << 3;
      acc += __hiloint2double(chi ^ (int)(__popc(xt & z) << 31), clo) * W[m * nthr + t];
    }
  }
  // fixed-order sum over the waves that hold amplitudes
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  __syncthreads();
  if (lane == 0) W[t >> 6] = acc;
  __syncthreads();
  double e = 0.0;
  for (uint32_t w = 0; w < (live + 63) / 64; ++w) e += W[w];
  return e;
}

}  // namespace

template <int NT, bool KRAUS>
__global__ __launch_bounds__(1 << NT, 4) void k_small(const char* __restrict__ progs,
                                                      const SmallInst* __restrict__ insts, SmallInst one, int prec,
                                                      void* __restrict__ states, const uint64_t* __restrict__ tz,
                                                      const double* __restrict__ tc, double* __restrict__ energies,
                                                      const KrausOp* __restrict__ kraus, uint64_t seed, uint64_t traj0)
{
  typedef double D2 __attribute__((ext_vector_type(2)));
  typedef float F2 __attribute__((ext_vector_type(2)));
  extern __shared__ __align__(16) char smem[];
  // trajectories all run `one`, their states back to back
  SmallInst in;
  if constexpr (KRAUS) in = one;
  else in = insts[blockIdx.x];
  const uint64_t S = 1ull << in.n;
  if constexpr (KRAUS) in.io += (uint64_t)blockIdx.x * S;
  const uint32_t t = threadIdx.x, live = live_threads(in.n);
  // whole waves without amplitudes leave (a barrier does not wait for them);
  // lanes without any repeat those of their wave's first ones
  const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
  if (first && first >= live) return;
  const char* prog = progs + in.prog;
  const PHead& h = *reinterpret_cast<const PHead*>(prog);
  touch(prog, h.bytes);
  Slots<double> x;
  {
    const uint64_t ga = global_part<NT>(t, h.gload);
    if (h.renorm & FP_INIT_ZERO) {
      each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        x.re[k] = (ga ^ global_slot<k>(h.gload)) == 0 ? 1.0 : 0.0;
        x.im[k] = 0.0;
      });
    } else {
      // registers of fewer than 4 qubits (one thread) leave slots empty
      if (prec == QSV_C128) load_slots<NT>(static_cast<const D2*>(states) + in.io, ga, h.gload, S, x);
      else load_slots<NT>(static_cast<const F2*>(states) + in.io, ga, h.gload, S, x);
    }
  }
  if constexpr (KRAUS) {
    const KrausRun kr{kraus, seed, traj0 + blockIdx.x, live};
    run_ops<double, NT, true>(prog, smem, 0, x, &kr);
  } else {
    run_ops<double, NT, false>(prog, smem, 0, x);
  }
  if (h.store_wait) {   // every wave's loads are done before any store
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  const uint64_t ga = global_part<NT>(t, h.gstore);
  if (in.io != ~0ull && t < live) {
    if (prec == QSV_C128) store_slots<double, NT>(static_cast<D2*>(states) + in.io, ga, h.gstore, S, x);
    else store_slots<float, NT>(static_cast<F2*>(states) + in.io, ga, h.gstore, S, x);
  }
  if (in.dest != ~0ull) {
    const double e = z_energy<NT>(x, h.gstore, (uint32_t)ga, live, smem, tz, tc, in.t0, in.t1);
    if (t == 0) energies[in.dest] = e;
  }
}

// 64, 256, 512 or 1024 threads: registers of up to 10, 12, 13 and 14 qubits.
int small_class(int n) { return n <= 10 ? 6 : n <= 12 ? 8 : n - 4; }

namespace {

template <int NT, bool KRAUS>
hipError_t launch_class(const SmallRun& r, unsigned count, hipStream_t st)
{
  constexpr size_t lds = (8u << (NT + 4)) + 16 * sizeof(double);
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_small<NT, KRAUS>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_small<NT, KRAUS>), dim3(count), dim3(1 << NT), lds, st, r.progs, r.insts, r.one, r.prec,
                     r.states, r.tz, r.tc, r.energies, r.kraus, r.seed, r.traj0);
  return hipGetLastError();
}

template <bool KRAUS>
hipError_t launch_any(const SmallRun& r, int cls, unsigned count, hipStream_t st)
{
  switch (cls) {
  case 6: return launch_class<6, KRAUS>(r, count, st);
  case 8: return launch_class<8, KRAUS>(r, count, st);
  case 9: return launch_class<9, KRAUS>(r, count, st);
  default: return launch_class<10, KRAUS>(r, count, st);
  }
}

}  // namespace

hipError_t launch_small(const SmallRun& r, int cls, unsigned count, hipStream_t st)
{
  if (count == 0) return hipSuccess;
  return r.kraus ? launch_any<true>(r, cls, count, st) : launch_any<false>(r, cls, count, st);
}

}  // namespace qsv
