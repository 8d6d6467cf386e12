// qsv_batch.hip — shots of many small states stored back to back.
#include "qsv_internal.h"

namespace qsv {

template <typename R> struct BV;
template <> struct BV<double> { typedef double T __attribute__((ext_vector_type(2))); };
template <> struct BV<float> { typedef float T __attribute__((ext_vector_type(2))); };

// Shots for many small states in an arena: one workgroup per state. Chunk
// sums (FP64) and their inclusive scan live in LDS; each shot is a binary
// search over chunks and a scan inside its chunk (inverse CDF, as measure-state).

__device__ __forceinline__ double uni01(uint64_t seed, uint64_t k)
{
  uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

template <typename R>
__global__ __launch_bounds__(256) void k_batch_sample(const typename BV<R>::T* __restrict__ arena,
                                                      const SampleJob* __restrict__ jobs,
                                                      uint64_t* __restrict__ outcomes,
                                                      double* __restrict__ norms)
{
  __shared__ double cum[256];
  const SampleJob jb = jobs[blockIdx.x];
  const auto* psi = arena + jb.state_offset;
  const uint64_t S = 1ull << jb.n;
  const uint32_t nch = S < 256 ? (uint32_t)S : 256u;
  const uint64_t C = S / nch;
  const uint32_t tid = threadIdx.x;
  double v = 0.0;
  if (tid < nch)
    for (uint64_t k = 0; k < C; ++k) {
      const auto a = psi[(uint64_t)tid * C + k];
      v += (double)a.x * a.x + (double)a.y * a.y;
    }
  cum[tid] = v;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const double t = (tid >= (uint32_t)off) ? cum[tid - off] : 0.0;
    __syncthreads();
    cum[tid] += t;
    __syncthreads();
  }
  const double total = cum[nch - 1];
  if (norms && tid == 0) norms[blockIdx.x] = total;
  for (uint64_t s = tid; s < jb.shots; s += 256) {
    const double r = uni01(jb.seed, s) * total;
    uint32_t lo = 0, hi = nch;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (cum[mid] < r) lo = mid + 1; else hi = mid;
    }
    uint64_t out = S - 1;
    if (lo < nch) {
      double run = lo ? cum[lo - 1] : 0.0;
      out = (uint64_t)lo * C + C - 1;
      for (uint64_t k = 0; k < C; ++k) {
        const auto a = psi[(uint64_t)lo * C + k];
        run += (double)a.x * a.x + (double)a.y * a.y;
        if (run >= r) { out = (uint64_t)lo * C + k; break; }
      }
    }
    outcomes[jb.out_offset + s] = out;
  }
}

void launch_batch_sample(int prec, const void* arena, const void* jobs, unsigned njobs, uint64_t* outcomes,
                         double* norms, hipStream_t st)
{
  if (njobs == 0) return;
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_batch_sample<double>), dim3(njobs), dim3(256), 0, st, (const BV<double>::T*)arena,
                       (const SampleJob*)jobs, outcomes, norms);
  else
    hipLaunchKernelGGL((k_batch_sample<float>), dim3(njobs), dim3(256), 0, st, (const BV<float>::T*)arena,
                       (const SampleJob*)jobs, outcomes, norms);
}

}  // namespace qsv
