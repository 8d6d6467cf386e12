// qsv_ops.h — device code that runs the micro-op programs of qsv_compile.hip on a
// tile held by one workgroup; included by the tiled passes (qsv_pass.hip) and
// the whole-register kernel of small circuits (qsv_small.hip).
#pragma once
#include "qsv_internal.h"

namespace qsv {

namespace {

template <typename R> struct PV;
template <> struct PV<double> { typedef double T __attribute__((ext_vector_type(2))); };
template <> struct PV<float> { typedef float T __attribute__((ext_vector_type(2))); };

constexpr int kSlots = 16;

__device__ __forceinline__ double mad(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float mad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <int V> using Int = std::integral_constant<int, V>;

// f(k) for k = K .. N-1 with k a compile-time constant: slots must only ever
// be indexed by constants, or they leave registers.
template <int K, int N, typename F>
__device__ __forceinline__ void each(F&& f)
{
  if constexpr (K < N) {
    f(std::integral_constant<int, K>{});
    each<K + 1, N>(f);
  }
}

// One op's fields and coefficients in scalar registers, fetched one op ahead.
template <typename A> struct OpRegs {
  int32_t code;
  uint32_t tmask, kc, aux;
  int32_t cnt, flag;
  uint64_t gm;
  uint32_t w[16];   // the union: coefficients or packed columns
  __device__ __forceinline__ A m(int i) const
  {
    if constexpr (sizeof(A) == 8) return __hiloint2double((int)w[2 * i + 1], (int)w[2 * i]);
    else return __uint_as_float(w[i]);
  }
  __device__ __forceinline__ uint32_t col(int i) const { return (w[i >> 1] >> (16 * (i & 1))) & 0xffffu; }
};
template <typename A>
__device__ __forceinline__ void fetch(OpRegs<A>& o, const POp* p)
{
  o.code = p->code;
  o.tmask = p->tmask;
  o.kc = p->kc;
  o.aux = p->aux;
  o.cnt = p->cnt;
  o.flag = p->flag;
  o.gm = p->gm;
  const uint32_t* w = reinterpret_cast<const uint32_t*>(p->m);
#pragma unroll
  for (int i = 0; i < 16; ++i) o.w[i] = w[i];
}

// Fixed-order sum of v over the workgroup (valid in thread 0); red[] must
// hold one double per wave.
__device__ __forceinline__ double block_sum(double v, double* red)
{
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const uint32_t t = threadIdx.x;
  if ((t & 63u) == 0) red[t >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (t == 0)
    for (uint32_t w = 0; w < (blockDim.x >> 6); ++w) s += red[w];
  return s;
}

// Workgroup-scope LDS ordering, or wave-scope when only the wave's own
// addresses are involved.
__device__ __forceinline__ void lds_sync(bool wave_local)
{
  if (wave_local) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// A thread's 16 slots: A re[16], im[16], indexed by constants only.
template <typename A>
struct Slots {
  A re[kSlots], im[kSlots];
};

// A uniform value as a per-lane one: conditions on it become selects. As uniform
// branches around every slot they would cost the tile a second set of registers.
__device__ __forceinline__ uint32_t per_lane(uint32_t v)
{
  uint32_t r;
  asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(v));
  return r;
}

// A real 2x2 applied to (a, b) in place: one temporary, no moves.
template <typename A>
__device__ __forceinline__ void real2(A m0, A m1, A m2, A m3, A& a, A& b)
{
  const A t = m2 * a;
  a = m0 * a;
  a = mad(m1, b, a);
  b = mad(m3, b, t);
}

// (re, im) *= (dr, di) in place.
template <typename A>
__device__ __forceinline__ void cmul(A dr, A di, A& re, A& im)
{
  const A t = di * re;
  re = dr * re;
  re = mad(-di, im, re);
  im = mad(dr, im, t);
}

// A general 2x2 applied to (a, b) in place, in the order that lets each value
// be overwritten as soon as its last use is done.
template <typename A>
__device__ __forceinline__ void general2(const A (&m)[8], A& ar, A& ai, A& br, A& bi)
{
  const A xr = mad(-m[5], ai, m[4] * ar), xi = mad(m[5], ar, m[4] * ai);
  const A u = m[1] * ar;
  ar = m[0] * ar;
  ar = mad(-m[1], ai, ar);
  ai = mad(m[0], ai, u);
  ar = mad(m[2], br, ar);
  ar = mad(-m[3], bi, ar);
  ai = mad(m[2], bi, ai);
  ai = mad(m[3], br, ai);
  const A w = mad(m[7], br, xi);
  br = mad(m[6], br, xr);
  br = mad(-m[7], bi, br);
  bi = mad(m[6], bi, w);
  __builtin_amdgcn_sched_barrier(0);   // one pair at a time: the scheduler would keep the temporaries of all eight
}

// XOR of the columns of t's set bits; cols(j) for j < NT.
template <int NT, typename F>
__device__ __forceinline__ uint32_t thread_part(uint32_t t, F&& cols)
{
  uint32_t b = 0;
  each<0, NT>([&](auto jj) __attribute__((always_inline)) {
    constexpr int j = decltype(jj)::value;
    b ^= (uint32_t)((int32_t)(t << (31 - j)) >> 31) & cols(j);
  });
  return b;
}

// XOR of the slot columns of k's set bits: uniform, by scalar instructions.
template <int K, typename F>
__device__ __forceinline__ uint32_t slot_part(F&& cols)
{
  uint32_t b = 0;
  if constexpr (K & 1) b ^= cols(0);
  if constexpr (K & 2) b ^= cols(1);
  if constexpr (K & 4) b ^= cols(2);
  if constexpr (K & 8) b ^= cols(3);
  return b;
}

template <typename A>
__device__ __forceinline__ double norm2_slots(const Slots<A>& x)
{
  double s = 0.0;
  each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
    constexpr int k = decltype(kk)::value;
    const double re = x.re[k], im = x.im[k];
    s += re * re + im * im;
  });
  return s;
}

// What PO_KRAUS ops need: the operators of all sites, and which trajectory this
// workgroup runs on how many threads.
struct KrausRun {
  const KrausOp* table;
  uint64_t seed, traj;
  uint32_t live;
};
// The counter-based uniform of qsv_uniform.
__device__ __forceinline__ double site_uniform(uint64_t seed, uint64_t k)
{
  uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// Runs the ops of a program on a workgroup's tile of 2^(NT + 4) amplitudes.
// smem: 8 bytes per amplitude, and 8 per wave where there are PO_KRAUS ops.
// base: the tile's base index (its bits outside the tile).
// kr: the trajectory a program with PO_KRAUS ops runs (null otherwise).
template <typename A, int NT, bool KRAUS = false>
__device__ __forceinline__ void run_ops(const char* __restrict__ prog, char* smem, uint64_t base, Slots<A>& x,
                                        const KrausRun* kr = nullptr)
{
  constexpr bool SPLIT = sizeof(A) == 8;
  typedef A P2 __attribute__((ext_vector_type(2)));
  const uint32_t t = threadIdx.x;
  const PHead& h = *reinterpret_cast<const PHead*>(prog);
  const POp* ops = reinterpret_cast<const POp*>(prog + sizeof(PHead));
  const int nops = h.nops;
  auto at = [&](uint32_t e) __attribute__((always_inline)) -> A* { return reinterpret_cast<A*>(smem + e); };
  auto at2 = [&](uint32_t e) __attribute__((always_inline)) -> P2* { return reinterpret_cast<P2*>(smem + e); };
  uint32_t lb = 0;   // byte offset of this thread's part in the layout of the last relayout
  OpRegs<A> nx;
  fetch(nx, ops);   // (there is at least the unread one)
  // no fetch is pending when the loop starts: the wait for the next op then
  // stands at the end of the loop, behind the current op's work
  asm volatile("" ::"s"(nx.code), "s"(nx.cnt), "s"(nx.w[0]), "s"(nx.w[15]));
  for (int i = 0; i < nops; ++i) {
    const OpRegs<A> op = nx;
    fetch(nx, ops + i + 1);   // the program ends with one unread op
    if (op.gm & ~base) continue;   // a control outside the tile is not set
    const int code = op.code;
    // One flat dispatch whose cases share no code: a case that is merged with
    // another in part makes the compiler keep a second copy of the tile.
    auto dense = [&](auto rbc, auto dmc) __attribute__((always_inline)) {
      constexpr int rb = decltype(rbc)::value, dm = decltype(dmc)::value, d = 1 << rb;
      asm volatile("; dense %0 %1" ::"i"(rb), "i"(dm));
      const bool act = (t & op.tmask) == op.tmask;
      if constexpr (dm == PM_EXCHANGE) {
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          if constexpr (!(k & d)) {
            const A ar = x.re[k], ai = x.im[k], br = x.re[k | d], bi = x.im[k | d];
            x.re[k] = act ? br : ar;
            x.im[k] = act ? bi : ai;
            x.re[k | d] = act ? ar : br;
            x.im[k | d] = act ? ai : bi;
          }
        });
      } else if constexpr (dm == PM_REAL) {
        const A m0 = act ? op.m(0) : (A)1, m1 = act ? op.m(2) : (A)0;
        const A m2 = act ? op.m(4) : (A)0, m3 = act ? op.m(6) : (A)1;
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          if constexpr (!(k & d)) {
            real2(m0, m1, m2, m3, x.re[k], x.re[k | d]);
            real2(m0, m1, m2, m3, x.im[k], x.im[k | d]);
          }
        });
      } else if constexpr (dm == PM_RX) {
        // real diagonal, imaginary off-diagonal i m3, i m5: a real 2x2 on
        // (a.re, b.im) and one of the other signs on (a.im, b.re)
        const A m0 = act ? op.m(0) : (A)1, m3 = act ? op.m(3) : (A)0;
        const A m5 = act ? op.m(5) : (A)0, m6 = act ? op.m(6) : (A)1;
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          if constexpr (!(k & d)) {
            real2(m0, -m3, m5, m6, x.re[k], x.im[k | d]);
            real2(m0, m3, -m5, m6, x.im[k], x.re[k | d]);
          }
        });
      } else {
        const uint32_t kc = per_lane(op.kc);
        A m[8];
        each<0, 8>([&](auto ii) __attribute__((always_inline)) {
          constexpr int e = decltype(ii)::value;
          m[e] = act ? op.m(e) : (A)(e == 0 || e == 6 ? 1 : 0);
        });
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          if constexpr (!(k & d)) {
            if constexpr (dm == PM_GENERAL) {
              general2(m, x.re[k], x.im[k], x.re[k | d], x.im[k | d]);
            } else {   // PO_DENSE_K: only the pairs whose slot controls are set
              A ar = x.re[k], ai = x.im[k], br = x.re[k | d], bi = x.im[k | d];
              general2(m, ar, ai, br, bi);
              const bool in = ((uint32_t)k & kc) == kc;
              x.re[k] = in ? ar : x.re[k];
              x.im[k] = in ? ai : x.im[k];
              x.re[k | d] = in ? br : x.re[k | d];
              x.im[k | d] = in ? bi : x.im[k | d];
            }
          }
        });
      }
      asm volatile("; end %0 %1" ::"i"(rb), "i"(dm));
    };
    // diagonal on a register bit of an FP32 pass: one factor per lane for the
    // clear bit, one for the set bit
    auto phase2 = [&](auto rbc) __attribute__((always_inline)) {
      if constexpr (!SPLIT) {
        constexpr int rb = decltype(rbc)::value;
        A gr = op.m(0), gi = op.m(1), fr = op.m(6), fi = op.m(7);
        const PTerm* tm = reinterpret_cast<const PTerm*>(prog + op.aux);
        for (int j = 0; j < op.cnt; ++j) {
          const PTerm& q = tm[j];
          const bool on = (t & q.tmask) == q.tmask && !(q.gmask & ~base);
          cmul(on ? q.f[0] : (A)1, on ? q.f[1] : (A)0, fr, fi);
          cmul(on ? q.f[2] : (A)1, on ? q.f[3] : (A)0, gr, gi);
        }
        asm volatile("; phase2 %0" ::"i"(rb));
        const uint32_t kc = per_lane(op.kc);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          const bool in = ((uint32_t)k & kc) == kc;
          cmul(in ? ((k >> rb) & 1 ? fr : gr) : (A)1, in ? ((k >> rb) & 1 ? fi : gi) : (A)0, x.re[k], x.im[k]);
        });
        asm volatile("; end %0" ::"i"(rb));
      }
    };
    // noise operator of site kc: the first of its cnt operators whose running
    // weight exceeds the trajectory's uniform (the last one otherwise), then,
    // where flagged, the division by the norm when that exceeds 1e-12
    auto kraus = [&](auto rbc) __attribute__((always_inline)) {
      constexpr int rb = decltype(rbc)::value, d = 1 << rb;
      asm volatile("; kraus %0" ::"i"(rb));
      const double u = site_uniform(kr->seed, kr->traj * QSV_TRAJ_SLOTS + op.kc);
      const KrausOp* tab = kr->table + op.aux;
      double acc = 0.0;
      int j = 0;
      for (; j < op.cnt - 1; ++j) {
        acc += tab[j].w;
        if (u < acc) break;
      }
      A m[8];
      each<0, 8>([&](auto ii) __attribute__((always_inline)) {
        constexpr int e = decltype(ii)::value;
        m[e] = (A)tab[j].m[e];
      });
      each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        if constexpr (!(k & d)) general2(m, x.re[k], x.im[k], x.re[k | d], x.im[k | d]);
      });
      if (op.flag) {
        double v = t < kr->live ? norm2_slots(x) : 0.0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if constexpr (NT > 6) {
          double* red = reinterpret_cast<double*>(smem + (8u << (NT + 4)));
          if ((t & 63u) == 0) red[t >> 6] = v;
          __syncthreads();
          v = 0.0;
          for (uint32_t w = 0; w < (kr->live + 63) / 64; ++w) v += red[w];   // one order in every thread
          __syncthreads();
        }
        const double nrm = sqrt(v);
        const A f = (A)(nrm > 1e-12 ? 1.0 / nrm : 1.0);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          x.re[k] *= f;
          x.im[k] *= f;
        });
      }
      asm volatile("; end kraus %0" ::"i"(rb));
    };
#define QSV_DENSE(RB)                                                                            \
  case PO_DENSE + 4 * RB + PM_GENERAL: dense(Int<RB>{}, Int<PM_GENERAL>{}); break;               \
  case PO_DENSE + 4 * RB + PM_REAL: dense(Int<RB>{}, Int<PM_REAL>{}); break;                     \
  case PO_DENSE + 4 * RB + PM_RX: dense(Int<RB>{}, Int<PM_RX>{}); break;                         \
  case PO_DENSE + 4 * RB + PM_EXCHANGE: dense(Int<RB>{}, Int<PM_EXCHANGE>{}); break;             \
  case PO_DENSE_K + RB: dense(Int<RB>{}, Int<4>{}); break
    switch (code) {
    QSV_DENSE(0);
    QSV_DENSE(1);
    QSV_DENSE(2);
    QSV_DENSE(3);
#undef QSV_DENSE
    case PO_PHASE: {
      // one factor per lane: the uniform part times the terms of the lane's set bits
      A fr = op.m(0), fi = op.m(1);
      const PTerm* tm = reinterpret_cast<const PTerm*>(prog + op.aux);
      for (int j = 0; j < op.cnt; ++j) {
        const PTerm& q = tm[j];
        const bool on = (t & q.tmask) == q.tmask && !(q.gmask & ~base);
        if constexpr (SPLIT) {
          cmul(on ? (A)q.d[0] : (A)1, on ? (A)q.d[1] : (A)0, fr, fi);
        } else {
          const bool set = (t & q.tbit) == q.tbit && !(q.gbit & ~base);
          const A qr = set ? q.f[0] : q.f[2], qi = set ? q.f[1] : q.f[3];
          cmul(on ? qr : (A)1, on ? qi : (A)0, fr, fi);
        }
      }
      auto all_with = [&](auto mask) __attribute__((always_inline)) {
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          if constexpr ((k & decltype(mask)::value) == decltype(mask)::value) cmul(fr, fi, x.re[k], x.im[k]);
        });
      };
      const uint32_t kc = op.kc;
      if (kc == 0) all_with(std::integral_constant<int, 0>{});
      else if (kc == 1) all_with(std::integral_constant<int, 1>{});
      else if (kc == 2) all_with(std::integral_constant<int, 2>{});
      else if (kc == 4) all_with(std::integral_constant<int, 4>{});
      else if (kc == 8) all_with(std::integral_constant<int, 8>{});
      else {
        const uint32_t kv = per_lane(kc);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          const bool in = ((uint32_t)k & kv) == kv;
          cmul(in ? fr : (A)1, in ? fi : (A)0, x.re[k], x.im[k]);
        });
      }
      break;
    }
#define QSV_PHASE2(RB)                                                                           \
  case PO_PHASE2 + RB: phase2(Int<RB>{}); break
    QSV_PHASE2(0);
    QSV_PHASE2(1);
    QSV_PHASE2(2);
    QSV_PHASE2(3);
#undef QSV_PHASE2
    case PO_RELAYOUT: {
      const bool local = (op.flag & PR_LOCAL) != 0;
      if (op.flag & PR_WAIT) __syncthreads();
      uint32_t fb = (op.flag & PR_SAME)
                        ? lb
                        : thread_part<NT>(t, [&](int j) __attribute__((always_inline)) { return op.col(j); }) << 3;
      const PShift* sh = reinterpret_cast<const PShift*>(prog + op.aux);
      for (int j = 0; j < op.cnt; ++j) fb ^= (base >> sh[j].bit) & 1u ? sh[j].col << 3 : 0u;
      lb = thread_part<NT>(t, [&](int j) __attribute__((always_inline)) { return op.col(kCols + j); }) << 3;
      auto from = [&](auto kk) __attribute__((always_inline)) {
        return slot_part<decltype(kk)::value>(
            [&](int j) __attribute__((always_inline)) { return op.col(kColT + j) << 3; });
      };
      auto to = [&](auto kk) __attribute__((always_inline)) {
        return slot_part<decltype(kk)::value>(
            [&](int j) __attribute__((always_inline)) { return op.col(kCols + kColT + j) << 3; });
      };
      if constexpr (SPLIT) {
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) { *at(fb ^ from(kk)) = x.re[decltype(kk)::value]; });
        lds_sync(local);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) { x.re[decltype(kk)::value] = *at(lb ^ to(kk)); });
        lds_sync(local);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) { *at(fb ^ from(kk)) = x.im[decltype(kk)::value]; });
        lds_sync(local);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) { x.im[decltype(kk)::value] = *at(lb ^ to(kk)); });
      } else {
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          P2 v;
          v.x = x.re[k];
          v.y = x.im[k];
          *at2(fb ^ from(kk)) = v;
        });
        lds_sync(local);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          const P2 v = *at2(lb ^ to(kk));
          x.re[k] = v.x;
          x.im[k] = v.y;
        });
      }
      // nothing may move above the reads of this wave's next writes
      lds_sync(true);
      break;
    }
    case PO_BLOCKADE: {
      // phase where exactly one blockade bit is set: thread part popcount(t &
      // aux), register part popcount(k & kc)
      const uint32_t pt = __popc(t & op.aux);
      const A pr = op.m(0), pi = op.m(1);
      each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        const bool on = pt + (uint32_t)__builtin_popcount((uint32_t)k & op.kc) == 1u;
        cmul(on ? pr : (A)1, on ? pi : (A)0, x.re[k], x.im[k]);
      });
      break;
    }
    case PO_SWAP: {
      // exchange local bits a = kc, b = aux (times the phase) where the local
      // control bits tmask are set: every thread writes its slots to permuted
      // LDS addresses and reads its own back
      __syncthreads();
      const uint32_t tl = thread_part<NT>(t, [&](int j) __attribute__((always_inline)) { return op.col(j); });
      const POp& full = ops[i];
      const A pr = (A)full.sc[0], pi = (A)full.sc[1];
      const uint32_t ba = 1u << op.kc, bb = 1u << op.aux, tmk = op.tmask;
      auto swz = [](uint32_t l) { return l ^ (((l >> 4) ^ (l >> 8)) & 15u); };   // its own inverse
      auto own = [&](auto kk) __attribute__((always_inline)) {
        return tl ^ slot_part<decltype(kk)::value>(
                        [&](int j) __attribute__((always_inline)) { return op.col(kColT + j); });
      };
      auto moves = [&](uint32_t e) __attribute__((always_inline)) -> bool {
        const uint32_t l = swz(e);
        return ((l & tmk) == tmk) && (((l & ba) != 0) != ((l & bb) != 0));
      };
      const uint32_t dsw = swz(ba ^ bb);
      each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        const bool mv = moves(own(kk));
        cmul(mv ? pr : (A)1, mv ? pi : (A)0, x.re[k], x.im[k]);
      });
      each<0, 2>([&](auto cc) __attribute__((always_inline)) {
        constexpr int c = decltype(cc)::value;
        if constexpr (SPLIT || c == 0) {
          each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
            constexpr int k = decltype(kk)::value;
            const uint32_t e = own(kk), to = (e ^ (moves(e) ? dsw : 0u)) << 3;
            if constexpr (SPLIT) {
              *at(to) = c ? x.im[k] : x.re[k];
            } else {
              P2 v;
              v.x = x.re[k];
              v.y = x.im[k];
              *at2(to) = v;
            }
          });
          __syncthreads();
          each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
            constexpr int k = decltype(kk)::value;
            const uint32_t e = own(kk) << 3;
            if constexpr (SPLIT) {
              (c ? x.im[k] : x.re[k]) = *at(e);
            } else {
              const P2 v = *at2(e);
              x.re[k] = v.x;
              x.im[k] = v.y;
            }
          });
          __syncthreads();
        }
      });
      break;
    }
    case PO_KRAUS + 0: if constexpr (KRAUS) kraus(Int<0>{}); break;
    case PO_KRAUS + 1: if constexpr (KRAUS) kraus(Int<1>{}); break;
    case PO_KRAUS + 2: if constexpr (KRAUS) kraus(Int<2>{}); break;
    case PO_KRAUS + 3: if constexpr (KRAUS) kraus(Int<3>{}); break;
    default: {
      // PO_BLOCK (FP32 arithmetic): Y = U X for the wave's 16 x 64 matrix X
      // (row = slot, column = lane) on the matrix cores, as four column blocks
      // of 16 lanes, 12 v_mfma_f32_16x16x4f32 each (three real products per
      // complex one). X crosses LDS at the addresses of the stage's layout, the
      // wave's own, so the round trip is wave-local. The offsets are XOR-linear
      // in the thread and slot bits: lane 16 cb + jc's slot s sits at
      // (wave part ^ jc part ^ cb part) ^ ls[s].
      if constexpr (!SPLIT) {
        typedef float f4 __attribute__((ext_vector_type(4)));
        const uint32_t l = t & 63u, kr = l >> 4, jc = l & 15u;
        const float2* tab = reinterpret_cast<const float2*>(prog + op.aux);
        float ur[4], ui[4], us[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const float2 u = tab[kk * 64 + l];
          ur[kk] = u.x;
          ui[kk] = u.y;
          us[kk] = u.x + u.y;
        }
        auto tcol = [&](int j) __attribute__((always_inline)) { return op.col(j) << 3; };
        auto scol = [&](int j) __attribute__((always_inline)) { return op.col(kColT + j) << 3; };
        const uint32_t fb = thread_part<NT>(t, tcol);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          P2 v;
          v.x = x.re[k];
          v.y = x.im[k];
          *at2(fb ^ slot_part<k>(scol)) = v;
        });
        lds_sync(true);
        const uint32_t pj = thread_part<NT>((t & ~63u) | jc, tcol);
        const uint32_t rin = (kr & 1u ? scol(0) : 0u) ^ (kr & 2u ? scol(1) : 0u);    // B rows 4 kk + kr
        const uint32_t rout = (kr & 1u ? scol(2) : 0u) ^ (kr & 2u ? scol(3) : 0u);   // C rows 4 kr + e
        each<0, 4>([&](auto cbc) __attribute__((always_inline)) {
          constexpr int cb = decltype(cbc)::value;
          const uint32_t pb = pj ^ (cb & 1 ? tcol(4) : 0u) ^ (cb & 2 ? tcol(5) : 0u);
          float br[4], bi[4];
          each<0, 4>([&](auto kc) __attribute__((always_inline)) {
            constexpr int kk = decltype(kc)::value;
            const P2 v = *at2(pb ^ rin ^ slot_part<4 * kk>(scol));
            br[kk] = v.x;
            bi[kk] = v.y;
          });
          // three real products (Gauss): P1 = Ur Xr, P2 = Ui Xi,
          // P3 = (Ur + Ui)(Xr + Xi); Y = (P1 - P2) + i (P3 - P1 - P2)
          f4 p1 = {0.f, 0.f, 0.f, 0.f}, p2 = {0.f, 0.f, 0.f, 0.f}, p3 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) {
            p1 = __builtin_amdgcn_mfma_f32_16x16x4f32(ur[kk], br[kk], p1, 0, 0, 0);
            p2 = __builtin_amdgcn_mfma_f32_16x16x4f32(ui[kk], bi[kk], p2, 0, 0, 0);
            p3 = __builtin_amdgcn_mfma_f32_16x16x4f32(us[kk], br[kk] + bi[kk], p3, 0, 0, 0);
          }
          // element e of lane l is row 4 (l / 16) + e, column l % 16 of the block
          each<0, 4>([&](auto ec) __attribute__((always_inline)) {
            constexpr int e = decltype(ec)::value;
            P2 v;
            v.x = p1[e] - p2[e];
            v.y = p3[e] - p1[e] - p2[e];
            *at2(pb ^ rout ^ slot_part<e>(scol)) = v;
          });
        });
        lds_sync(true);
        each<0, kSlots>([&](auto kk) __attribute__((always_inline)) {
          constexpr int k = decltype(kk)::value;
          const P2 v = *at2(fb ^ slot_part<k>(scol));
          x.re[k] = v.x;
          x.im[k] = v.y;
        });
        lds_sync(true);
      }
      break;
    }
    }
  }
}

// Reads one word of every cache line of a program, all lines at once: the op
// fetches that follow one another then find them in the L2 cache, not in HBM.
__device__ __forceinline__ void touch(const char* prog, int bytes)
{
  uint32_t acc = 0;
  for (int o = threadIdx.x * 128; o < bytes; o += blockDim.x * 128)
    acc ^= *reinterpret_cast<const uint32_t*>(prog + o);
  asm volatile("" ::"v"(acc));
}

// Global element offsets of this thread's part for the columns c[0..NT).
template <int NT>
__device__ __forceinline__ uint64_t global_part(uint32_t t, const uint64_t* c)
{
  uint64_t g = 0;
  each<0, NT>([&](auto jj) __attribute__((always_inline)) {
    constexpr int j = decltype(jj)::value;
    g ^= ((t >> j) & 1u) ? c[j] : 0ull;
  });
  return g;
}
template <int K>
__device__ __forceinline__ uint64_t global_slot(const uint64_t* c)
{
  uint64_t g = 0;
  if constexpr (K & 1) g ^= c[kColT + 0];
  if constexpr (K & 2) g ^= c[kColT + 1];
  if constexpr (K & 4) g ^= c[kColT + 2];
  if constexpr (K & 8) g ^= c[kColT + 3];
  return g;
}

}  // namespace

}  // namespace qsv
