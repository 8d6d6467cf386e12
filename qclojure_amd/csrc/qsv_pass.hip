// qsv_pass.hip — fused tiled passes: the micro-op programs of qsv_compile.hip.
//
// A pass owns TB = 12 tile bits of the index. Each workgroup of 256 threads
// loads one tile of 2^12 amplitudes (16 per thread, in registers), runs the
// pass's micro-ops and stores the tile back, so the state crosses HBM once per
// pass however many gates the pass holds.
//
// The layout of a tile in registers is linear over GF(2): thread t, slot k
// holds the local index XOR_j t_j c_j XOR XOR_i k_i r_i. A micro-op names the
// register bit of its target, the slot mask of its register-bit controls and
// the thread-id mask of its thread-bit controls: the kernel decodes nothing and
// takes only uniform branches; a lane whose controls are not set applies the
// identity through its coefficients.
//
// Changing the layout is one LDS round trip (PO_RELAYOUT). When the wave-id
// bits of the thread index name the same tile bits before and after, every wave
// keeps its own amplitudes and the round trip needs no workgroup barrier; the
// host marks those. A wave only ever reads the addresses of the layout it
// enters and writes those of the layout it leaves, so one barrier per exchanged
// plane is enough. FP64 tiles cross LDS one plane (real, then imaginary) at a
// time, so a workgroup needs 32 KiB of LDS.
//
// Arithmetic type A: FP64 for complex128 and for complex64 states whose passes
// are asked for in FP64 (held in FP64 registers, rounded at the store); FP32
// for other complex64 passes, which also report per-tile norms and apply the
// previous pass's renormalisation scale at load (TileNorm in qsv_internal.h).
// What bounds it: the tile's access pattern (loads and stores alone stream at
// 5.3 TB/s) with the gates' instructions partly on top; on few tiles the chain
// of ops, whose fetch from memory is hidden behind the op before. Against the
// interpreter that ran every gate as an op and kept two copies of the tile
// (three waves per SIMD), per launch: dense 27-qubit complex128 layers 1257 ->
// 885 us, 19-qubit ones 47 -> 23 us, 540 gates on one 12-qubit tile 524 -> 122 us.
#include "qsv_ops.h"

namespace qsv {

namespace {

constexpr int kThreads = 256;
// A launch of few tiles is a chain of ops whose fetches miss every cache (the
// program was just written): its workgroups read the program into L2 first.
// 540 gates on one tile 146 -> 122 us, 19-qubit passes (128 tiles) 23.5 -> 22.9;
// with thousands of tiles most find it there anyway.
constexpr uint32_t kTouchTiles = 512;

// Is some amplitude of the workgroup's tile not zero? A register that has just
// been set to |0..0> is nothing but zeros outside a few tiles until each of its
// qubits has met a gate, three passes or so later. A pass is linear: such a tile
// needs neither its ops nor a store. Two barriers and 64 ORs (32 in FP32) a thread
// for the others (a dense 27-qubit pass 943 us without, 948 with). The first of
// seven passes over 27 qubits 943 -> 460 us at most and, unread where the earlier
// passes cannot have put anything (FP_REACH), the second 35 and the third 95; a
// 26-qubit complex64 ansatz 508 -> 105 and 46 us.
template <typename A>
__device__ __forceinline__ bool any_nonzero(const Slots<A>& x, uint32_t* flags)
{
  uint32_t hi = 0, lo = 0;   // bits with and without a sign
  each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
    constexpr int k = decltype(kk)::value;
    if constexpr (sizeof(A) == 8) {
      hi |= (uint32_t)__double2hiint(x.re[k]) | (uint32_t)__double2hiint(x.im[k]);
      lo |= (uint32_t)__double2loint(x.re[k]) | (uint32_t)__double2loint(x.im[k]);
    } else {
      hi |= __float_as_uint(x.re[k]) | __float_as_uint(x.im[k]);
    }
  });
  const uint32_t t = threadIdx.x;
  const bool mine = __any((hi << 1) | lo);
  if ((t & 63u) == 0) flags[t >> 6] = mine;
  __syncthreads();
  const uint32_t any = flags[0] | flags[1] | flags[2] | flags[3];
  __syncthreads();   // the tile's LDS overlays the flags
  return __builtin_amdgcn_readfirstlane((int)any) != 0;
}

}  // namespace

// One tile of one pass per workgroup. GROUP: many states of S amplitudes back
// to back; instance blockIdx.y runs the program at byte offset offs[y] of
// `progs` (negative: no pass this round); group passes do not renormalise.
template <typename R, typename A, bool GROUP>
__global__ __launch_bounds__(kThreads, sizeof(A) == 4 ? 5 : 4) void k_pass(typename PV<R>::T* __restrict__ psi,
                                                                           const char* __restrict__ progs,
                                                                           TileNorm nb, uint64_t S,
                                                                           const int64_t* __restrict__ offs)
{
  using T = typename PV<R>::T;
  constexpr int TB = kPassTileBits, NT = TB - 4;
  // the tile's LDS; also the per-wave partial sums of the norm reductions
  __shared__ __align__(16) char smem[8u << TB];
  double* red = reinterpret_cast<double*>(smem);
  const char* prog = progs;
  if constexpr (GROUP) {
    const int64_t off = offs[blockIdx.y];
    if (off < 0) return;
    psi += (uint64_t)blockIdx.y * S;
    prog += off;
  }
  // The dispatcher hands consecutive workgroups to the 8 XCDs in turn: map
  // them so that each XCD streams one contiguous eighth of the tiles (its own
  // L2 and translation caches then see neighbouring addresses)
  const uint32_t g = gridDim.x, b = blockIdx.x;
  const uint32_t tile = (g & 7u) ? b : (b & 7u) * (g >> 3) + (b >> 3);
  const uint32_t t = threadIdx.x;
  const PHead& h = *reinterpret_cast<const PHead*>(prog);

  // tile base: zeros inserted at the tile's global bits (ascending)
  uint64_t base = tile;
#pragma unroll
  for (int i = 0; i < TB; ++i) {
    const int p = h.sorted_pos[i];
    const uint64_t lo = base & ((1ull << p) - 1ull);
    base = ((base ^ lo) << 1) | lo;
  }

  Slots<A> x;
  const int rn = h.renorm;
  uint64_t tmask = 0;
  // a scale that is not finite would turn zeros into NaN
  const bool keep = (rn & FP_KEEP_ZERO) && !(sizeof(A) == 4 && (rn & FP_RENORM_APPLY) && !(nb.ctl[1] < 1e30));
  if constexpr (!GROUP) {
    // A tile that no nonzero amplitude of the earlier passes can lie in is not
    // even read: its base has a bit set, or clear, that none of those has. The
    // launch's own tiles extend `reach` meanwhile, but one that passed this test
    // adds nothing but the tile's bits, which the test leaves out: every wave of a
    // workgroup decides alike.
    if (rn & FP_REACH) {
#pragma unroll
      for (int i = 0; i < TB; ++i) tmask |= 1ull << h.sorted_pos[i];
      if (rn & FP_REACH_USE) {
        const uint64_t set = __hip_atomic_load(nb.reach, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t clear = __hip_atomic_load(nb.reach + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t bits = (((uint64_t)gridDim.x << TB) - 1ull) & ~tmask;
        if (keep && (((base & ~set) | (~base & ~clear)) & bits)) {
          if constexpr (sizeof(A) == 4) {
            if (t == 0 && (rn & FP_RENORM_OUT)) nb.part_out[tile] = 0.0;
          }
          return;
        }
      }
    }
  }
  {
    const uint64_t ga = base ^ global_part<NT>(t, h.gload);
    if (rn & FP_INIT_ZERO) {
      // |0..0>: amplitude 1 at global index 0, nothing read
      each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        x.re[k] = (ga ^ global_slot<k>(h.gload)) == 0 ? (A)1 : (A)0;
        x.im[k] = (A)0;
      });
    } else {
      each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        const T v = __builtin_nontemporal_load(psi + (ga ^ global_slot<k>(h.gload)));
        x.re[k] = (A)v.x;
        x.im[k] = (A)v.y;
      });
    }
  }
  if (gridDim.x <= kTouchTiles) touch(prog, h.bytes);
  if (rn & FP_INIT_ZERO) {
    if (base != 0 && keep) {
      const uint64_t ga = base ^ global_part<NT>(t, h.gload);
      each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        T v;
        v.x = v.y = R(0);
        __builtin_nontemporal_store(v, psi + (ga ^ global_slot<k>(h.gload)));
      });
      return;
    }
  } else if (rn & FP_KEEP_ZERO) {
    if (!any_nonzero(x, reinterpret_cast<uint32_t*>(smem)) && keep) {
      if constexpr (sizeof(A) == 4) {
        if (t == 0 && (rn & FP_RENORM_IN)) nb.part_in[tile] = 0.0;
        if (t == 0 && (rn & FP_RENORM_OUT)) nb.part_out[tile] = 0.0;
      }
      return;
    }
    if constexpr (!GROUP) {
      if ((rn & FP_REACH) && t == 0) {
        const uint64_t set = base | tmask, clear = ~base;   // both, for the tile's own bits
        if (set & ~__hip_atomic_load(nb.reach, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(nb.reach, set);
        if (clear & ~__hip_atomic_load(nb.reach + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
          atomicOr(nb.reach + 1, clear);
      }
    }
  }
  if constexpr (sizeof(A) == 4) {
    if (rn & FP_RENORM_APPLY) {
      const A sc = (A)nb.ctl[1];
      each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        x.re[k] *= sc;
        x.im[k] *= sc;
      });
    }
    if (rn & FP_RENORM_IN) {
      const double v = block_sum(norm2_slots(x), red);
      if (t == 0) nb.part_in[tile] = v;
      __syncthreads();
    }
  }

  run_ops<A, NT>(prog, smem, base, x);
  if (h.store_wait) {   // every wave's loads are done before any store
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

  {
    uint64_t ga = base ^ global_part<NT>(t, h.gstore);
    const PShift* sh = reinterpret_cast<const PShift*>(prog + h.shift_off);
    for (int j = 0; j < h.nshift; ++j) ga ^= (base >> sh[j].bit) & 1u ? sh[j].g : 0ull;
    each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
      constexpr int k = decltype(kk)::value;
      T v;
      v.x = (R)x.re[k];
      v.y = (R)x.im[k];
      __builtin_nontemporal_store(v, psi + (ga ^ global_slot<k>(h.gstore)));
    });
  }
  if constexpr (sizeof(A) == 4) {
    if (rn & FP_RENORM_OUT) {
      __syncthreads();   // red[] overlays the tile's LDS
      const double v = block_sum(norm2_slots(x), red);
      if (t == 0) nb.part_out[tile] = v;
    }
  }
}

// |0..0> in every state of a group.
template <typename R>
__global__ __launch_bounds__(256) void k_fill_group(typename PV<R>::T* __restrict__ base, uint64_t total, uint64_t S)
{
  using T = typename PV<R>::T;
  for (uint64_t j = (uint64_t)blockIdx.x * 256 + threadIdx.x; j < total; j += (uint64_t)gridDim.x * 256) {
    T v;
    v.x = (j & (S - 1)) == 0 ? R(1) : R(0);
    v.y = R(0);
    base[j] = v;
  }
}

// One workgroup: fixed-order sums of the per-tile norms, then the scale the
// next pass applies at load.
__global__ __launch_bounds__(1024) void k_norm_ctl(const double* __restrict__ part_in,
                                                   const double* __restrict__ part_out, uint64_t ntiles, int first,
                                                   double* __restrict__ ctl)
{
  __shared__ double sa[1024], sb[1024];
  const uint32_t t = threadIdx.x;
  double a = 0.0, b = 0.0;
  for (uint64_t i = t; i < ntiles; i += 1024) {
    if (first) a += part_in[i];
    b += part_out[i];
  }
  sa[t] = a;
  sb[t] = b;
  __syncthreads();
  for (uint32_t w = 512; w > 0; w >>= 1) {
    if (t < w) {
      sa[t] += sa[t + w];
      sb[t] += sb[t + w];
    }
    __syncthreads();
  }
  if (t == 0) {
    const double target = first ? sa[0] : ctl[0];
    ctl[0] = target;
    ctl[1] = (target > 0.0 && sb[0] > 0.0) ? sqrt(target / sb[0]) : 1.0;
  }
}

void launch_pass(int prec, bool f32, void* psi, const char* dprog, uint64_t ntiles, const TileNorm& nb,
                 hipStream_t st)
{
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_pass<double, double, false>), dim3((unsigned)ntiles), dim3(kThreads), 0, st,
                       (PV<double>::T*)psi, dprog, nb, 0, (const int64_t*)nullptr);
  else if (f32)
    hipLaunchKernelGGL((k_pass<float, float, false>), dim3((unsigned)ntiles), dim3(kThreads), 0, st,
                       (PV<float>::T*)psi, dprog, nb, 0, (const int64_t*)nullptr);
  else
    hipLaunchKernelGGL((k_pass<float, double, false>), dim3((unsigned)ntiles), dim3(kThreads), 0, st,
                       (PV<float>::T*)psi, dprog, nb, 0, (const int64_t*)nullptr);
}

void launch_pass_group(int prec, void* base, uint64_t S, unsigned count, const char* progs, const int64_t* offs,
                       hipStream_t st)
{
  // complex64 groups compute in FP64: no per-instance renormalisation needed
  const TileNorm none{nullptr, nullptr, nullptr, nullptr};
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_pass<double, double, true>), dim3((unsigned)(S >> kPassTileBits), count), dim3(kThreads),
                       0, st, (PV<double>::T*)base, progs, none, S, offs);
  else
    hipLaunchKernelGGL((k_pass<float, double, true>), dim3((unsigned)(S >> kPassTileBits), count), dim3(kThreads),
                       0, st, (PV<float>::T*)base, progs, none, S, offs);
}

void launch_fill_group(int prec, void* base, uint64_t S, uint64_t count, hipStream_t st)
{
  const uint64_t total = S * count;
  const uint64_t want = (total + 255) / 256;
  const unsigned grid = (unsigned)(want < 65536 ? want : 65536);
  if (prec == QSV_C128)
    hipLaunchKernelGGL((k_fill_group<double>), dim3(grid), dim3(256), 0, st, (PV<double>::T*)base, total, S);
  else
    hipLaunchKernelGGL((k_fill_group<float>), dim3(grid), dim3(256), 0, st, (PV<float>::T*)base, total, S);
}

void launch_norm_ctl(const TileNorm& nb, uint64_t ntiles, bool first, hipStream_t st)
{
  hipLaunchKernelGGL(k_norm_ctl, dim3(1), dim3(1024), 0, st, nb.part_in, nb.part_out, ntiles, first ? 1 : 0, nb.ctl);
}

}  // namespace qsv
