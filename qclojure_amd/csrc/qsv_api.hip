// qsv_api.hip — the C ABI of libqsv (include/qsv.h).
//
// Decodes qsv_op records exactly as the reference dispatcher
// apply-gate-to-state does (src/org/soulspace/qclojure/domain/circuit.clj:933-1072)
// and turns each into one streaming kernel on the state's own HIP stream.
#include <algorithm>
#include <array>
#include <cstddef>
#include <map>
#include <atomic>
#include <chrono>
#include <complex>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <initializer_list>
#include <mutex>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include <sys/prctl.h>

#include "qsv_internal.h"

using namespace qsv;

namespace {
thread_local std::string g_err;
std::mutex g_mu;
bool g_init = false;
int g_device = 0;

int fail(int code, const std::string& msg)
{
  g_err = msg;
  return code;
}

#define HIPCHK(x)                                                                          \
  do {                                                                                     \
    hipError_t e_ = (x);                                                                   \
    if (e_ != hipSuccess) return fail(QSV_E_DEVICE, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

struct Pending {
  int cls;
  hipEvent_t a, b;
  double bytes;
};

void pool_release();
void batch_cache_release();
}  // namespace

struct qsv_state {
  int n = 0;
  int prec = QSV_C128;
  int device = 0;
  uint64_t S = 0;
  void* amps = nullptr;
  hipStream_t stream = nullptr;
  // Calls that only read a state may come from several threads at once; what
  // they share is scratch memory, held by one of them at a time from its first
  // launch to the wait for its results.
  mutable std::mutex scratch_mu;
  double* partials = nullptr;   // kPartials doubles
  double* dout = nullptr;       // kReduceOut doubles of reduction results
  double* prefix = nullptr;     // sampling chunk prefix (lazy)
  double* hist = nullptr;       // measurement histogram (lazy)
  uint64_t hist_cap = 0;
  bool timing = false;
  std::vector<Pending> pending;
  std::vector<hipEvent_t> evpool;
  qsv_kernel_stat stats[QSV_KCLASS_COUNT] = {};
  // fused-pass descriptor ring (pinned host staging + device copy per slot)
  struct PassSlot {
    char* host = nullptr;
    char* dev = nullptr;
    size_t cap = 0;   // bytes
    hipEvent_t event = nullptr;
  };
  static constexpr int kRing = 4;
  PassSlot ring[kRing];
  int ring_next = 0;
  PassSlot* ring_pending = nullptr;
  uint64_t passes_launched = 0;
  int tile_low = -1;            // tile low-run width forced by the tuner (-1: none)
  int reach_left = 0;           // passes that may still track where amplitudes can be
  double* norm_buf = nullptr;   // complex64 FP32 passes: per-tile norms (2 x ntiles) + control (2)
  uint64_t* shot_dev = nullptr;   // qsv_sample's outcomes (lazy, at most kShotsKept)
  uint64_t shot_cap = 0;
  uint64_t* samp_dev = nullptr;   // serving: reusable shot buffers (grow only)
  uint64_t* samp_host = nullptr;  // pinned
  uint64_t samp_cap = 0;
  double* norm_host = nullptr;    // serving: pinned FP64 sum |a|^2 read back after sampling
  uint64_t bytes_per_amp() const { return prec == QSV_C128 ? 16 : 8; }
};

// Scratch of qsv_sample_noalloc: the FP64 chunk prefix of the sampler (one
// partial sum per 2^kSampleChunkLog amplitudes, for states of up to
// QSV_NOALLOC_MAX_QUBITS qubits) followed by the device copy of the outcomes
// (up to QSV_NOALLOC_MAX_SHOTS). Every GPU the library runs on holds its own
// copy until the process ends; host code reaches it only through the address
// hipGetSymbolAddress returns for the current device (g_scratch_ptr).
constexpr uint64_t kNoAllocPrefixBytes = (1ull << (QSV_NOALLOC_MAX_QUBITS - kSampleChunkLog)) * sizeof(double);
constexpr uint64_t kNoAllocShotBytes = QSV_NOALLOC_MAX_SHOTS * sizeof(uint64_t);
static __device__ __align__(256) unsigned char scratch[kNoAllocPrefixBytes + kNoAllocShotBytes];

namespace {

constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices] = {};

// Resolves this device's copy of `scratch`; the device must be current.
// Caller holds g_mu.
int resolve_scratch_locked(int device)
{
  if (device < 0 || device >= kMaxDevices) return fail(QSV_E_INVALID, "device index beyond the scratch table");
  if (g_scratch_ptr[device]) return QSV_OK;
  void* p = nullptr;
  HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p) return fail(QSV_E_DEVICE, "hipGetSymbolAddress returned a null scratch address");
  g_scratch_ptr[device] = p;
  return QSV_OK;
}

int ensure_init()
{
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_init) return QSV_OK;
  int count = 0;
  HIPCHK(hipGetDeviceCount(&count));
  if (count <= 0) return fail(QSV_E_DEVICE, "no HIP device visible");
  HIPCHK(hipSetDevice(g_device));
  int rc = resolve_scratch_locked(g_device);
  if (rc) return rc;
  g_init = true;
  return QSV_OK;
}

hipEvent_t take_event(qsv_state* s)
{
  if (!s->evpool.empty()) {
    hipEvent_t e = s->evpool.back();
    s->evpool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}

int flush_timing(qsv_state* s)
{
  if (s->pending.empty()) return QSV_OK;
  HIPCHK(hipEventSynchronize(s->pending.back().b));
  for (auto& p : s->pending) {
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, p.a, p.b));
    s->stats[p.cls].launches += 1;
    s->stats[p.cls].total_ms += ms;
    s->stats[p.cls].bytes += p.bytes;
    s->evpool.push_back(p.a);
    s->evpool.push_back(p.b);
  }
  s->pending.clear();
  return QSV_OK;
}

template <class F>
int timed(qsv_state* s, int cls, double bytes, F&& launch)
{
  if (!s->timing) {
    launch();
    return QSV_OK;
  }
  hipEvent_t a = take_event(s), b = take_event(s);
  if (!a || !b) return fail(QSV_E_DEVICE, "hipEventCreate failed");
  HIPCHK(hipEventRecord(a, s->stream));
  launch();
  HIPCHK(hipEventRecord(b, s->stream));
  s->pending.push_back({cls, a, b, bytes});
  if (s->pending.size() >= 2048) return flush_timing(s);
  return QSV_OK;
}

InsArgs make_ins(uint64_t S, std::vector<int> bits, uint64_t orMask)
{
  std::sort(bits.begin(), bits.end());
  InsArgs a{};
  a.nins = (int)bits.size();
  for (size_t k = 0; k < bits.size(); ++k) a.ins[k] = bits[k];
  a.count = S >> bits.size();
  a.orMask = orMask;
  return a;
}

void gate_matrix(int kind, double angle, double out[8])
{
  // gate.clj:38-283, row-major (re, im).
  double m[8] = {1, 0, 0, 0, 0, 0, 1, 0};
  const double s2 = 1.0 / std::sqrt(2.0);
  switch (kind) {
  case QSV_OP_X: m[0] = 0; m[2] = 1; m[4] = 1; m[6] = 0; break;
  case QSV_OP_Y: m[0] = 0; m[3] = -1; m[5] = 1; m[6] = 0; break;
  case QSV_OP_Z: m[6] = -1; break;
  case QSV_OP_H: m[0] = s2; m[2] = s2; m[4] = s2; m[6] = -s2; break;
  case QSV_OP_S: m[6] = 0; m[7] = 1; break;
  case QSV_OP_SDG: m[6] = 0; m[7] = -1; break;
  case QSV_OP_T: m[6] = std::cos(M_PI / 4); m[7] = std::sin(M_PI / 4); break;
  case QSV_OP_TDG: m[6] = std::cos(M_PI / -4); m[7] = std::sin(M_PI / -4); break;
  case QSV_OP_PHASE: m[6] = std::cos(angle); m[7] = std::sin(angle); break;
  case QSV_OP_RX: {
    const double c = std::cos(angle / 2), s = std::sin(angle / 2);
    m[0] = c; m[3] = -s; m[5] = -s; m[6] = c; break;
  }
  case QSV_OP_RY: {
    const double c = std::cos(angle / 2), s = std::sin(angle / 2);
    m[0] = c; m[2] = -s; m[4] = s; m[6] = c; break;
  }
  case QSV_OP_RZ:
    m[0] = std::cos(angle / -2); m[1] = std::sin(angle / -2);
    m[6] = std::cos(angle / 2); m[7] = std::sin(angle / 2); break;
  default: break;
  }
  std::memcpy(out, m, sizeof(m));
}

inline bool is_diag(const double m[8]) { return m[2] == 0 && m[3] == 0 && m[4] == 0 && m[5] == 0; }
inline bool is_one(double re, double im) { return re == 1.0 && im == 0.0; }

// Bits below this stay inside the wavefront (their 2^thr-amplitude runs are
// shorter than a 128 B line); bits at or above it are enumerated by insertion.
inline int low_bit_threshold(const qsv_state* s) { return s->prec == QSV_C128 ? 3 : 4; }

// Control bits of a gate, held inline: decoding and folding hundreds of
// thousands of gates per batched call allocate nothing per gate. No gate
// kind has more than two controls.
struct CtlBits {
  static constexpr int kMax = 4;
  int n = 0;
  int c[kMax] = {0, 0, 0, 0};
  CtlBits() = default;
  CtlBits(std::initializer_list<int> l)
  {
    if (l.size() > (size_t)kMax) {   // an internal invariant: never silently drop a control
      std::fprintf(stderr, "qsv: a gate with %zu controls (at most %d)\n", l.size(), kMax);
      std::abort();
    }
    for (int x : l) c[n++] = x;
  }
  const int* begin() const { return c; }
  const int* end() const { return c + n; }
  size_t size() const { return (size_t)n; }
  bool empty() const { return n == 0; }
  bool operator==(const CtlBits& o) const
  {
    if (n != o.n) return false;
    for (int i = 0; i < n; ++i)
      if (c[i] != o.c[i]) return false;
    return true;
  }
};

// 2x2 `m` applied to target bit tb where all control bits are set (no controls
// for a plain 1-qubit gate). Diagonal matrices take the phase kernel, which
// touches only the |1> half of the target when m00 == 1.
// Algorithmic bytes: each touched amplitude is read once and written once.
int apply_ctl_bits(qsv_state* s, const CtlBits& cbits, int tb, const double m[8])
{
  const uint64_t B = s->bytes_per_amp();
  const int thr = low_bit_threshold(s);
  std::vector<int> ins;
  uint64_t hor = 0, lpred = 0;
  for (int c : cbits) {
    if (c >= thr) { ins.push_back(c); hor |= 1ull << c; }
    else lpred |= 1ull << c;
  }
  double touched = (double)(s->S >> cbits.size());
  GateArgs g{};
  if (is_diag(m)) {
    const double d0[2] = {m[0], m[1]}, d1[2] = {m[6], m[7]};
    if (is_one(m[0], m[1])) {
      touched /= 2;
      if (tb >= thr) { ins.push_back(tb); hor |= 1ull << tb; }
      else lpred |= 1ull << tb;
    }
    g.ins = make_ins(s->S, ins, hor);
    g.lo_pred = lpred;
    g.tbit = 1ull << tb;
    return timed(s, QSV_KCLASS_DIAG, 2.0 * touched * B,
                 [&] { launch_phase(s->prec, s->amps, g, d0, d1, s->stream); });
  }
  if (tb >= thr) { ins.push_back(tb); g.tbit = 1ull << tb; }
  else g.lo_t = 1ull << tb;
  g.ins = make_ins(s->S, ins, hor);
  g.lo_pred = lpred;
  return timed(s, QSV_KCLASS_PAIR, 2.0 * touched * B,
               [&] { launch_gate1(s->prec, s->amps, g, m, s->stream); });
}

// Exchange of index bits b1, b2 (times ph) where all control bits are set.
int apply_swap_bits(qsv_state* s, const CtlBits& cbits, int b1, int b2, const double ph[2])
{
  const uint64_t B = s->bytes_per_amp();
  const int thr = low_bit_threshold(s);
  std::vector<int> ins;
  uint64_t hor = 0, lpred = 0;
  for (int c : cbits) {
    if (c >= thr) { ins.push_back(c); hor |= 1ull << c; }
    else lpred |= 1ull << c;
  }
  SwapArgs a{};
  if (b1 < thr && b2 >= thr) std::swap(b1, b2);
  if (b1 >= thr && b2 >= thr) {
    ins.push_back(b1);
    ins.push_back(b2);
    a.hA = 1ull << b1;
    a.hB = 1ull << b2;
  } else if (b1 >= thr) {
    ins.push_back(b1);
    a.hA = 1ull << b1;
    a.lB = 1ull << b2;
  } else {
    a.lA = 1ull << b1;
    a.lB = 1ull << b2;
  }
  a.ins = make_ins(s->S, ins, hor);
  a.lo_pred = lpred;
  const double touched = (double)(s->S >> (cbits.size() + 1));
  return timed(s, QSV_KCLASS_PERM, 2.0 * touched * B,
               [&] { launch_swap2(s->prec, s->amps, a, ph, s->stream); });
}

// The reference's apply-controlled-gate applies the transpose of g
// (gate.clj:461-486): new[i0] = g00 a0 + g10 a1, new[i1] = g01 a0 + g11 a1.
void transpose2(const double g[8], double t[8])
{
  t[0] = g[0]; t[1] = g[1];
  t[2] = g[4]; t[3] = g[5];
  t[4] = g[2]; t[5] = g[3];
  t[6] = g[6]; t[7] = g[7];
}

// A program's first passes keep track of where nonzero amplitudes can be, so
// that the tiles elsewhere are not read (six layers of 27 qubits from |0..0>:
// 6.13 -> 4.94 ms). States below 256 MiB are read from the memory-side cache. A
// dense state only pays for it (24 qubits, complex128: 15 us of the first pass's
// 100), so a state has kReachTotal such passes from when it was last set, copied
// or measured, and a program of a single pass, which no pass follows, has none.
constexpr int kReachPasses = 4, kReachTotal = 2 * kReachPasses;
constexpr double kReachBytes = 256.0 * (1 << 20);
constexpr size_t kReachHead = 256;   // room for TileNorm::reach before the programs of a launch

int measure_impl(qsv_state* s, uint64_t mask, double u, uint64_t* outcome, double* probs_out)
{
  const int n = s->n;
  if (mask == 0 || (n < 64 && (mask >> n) != 0)) return fail(QSV_E_INVALID, "measure: qubit set empty or out of range");
  std::vector<int> pos;
  for (int q = 0; q < n; ++q)
    if ((mask >> q) & 1ull) pos.push_back(n - 1 - q);
  const int m = (int)pos.size();
  if (m > 20) return fail(QSV_E_UNSUPPORTED, "measure: more than 20 measured qubits");
  const uint64_t no = 1ull << m;
  if (s->hist_cap < no) {
    if (s->hist) hipFree(s->hist);
    s->hist = nullptr;
    HIPCHK(hipMalloc(&s->hist, no * sizeof(double)));
    s->hist_cap = no;
  }
  int rc = timed(s, QSV_KCLASS_OTHER, (double)s->S * s->bytes_per_amp(),
                 [&] { launch_outcome_hist(s->prec, s->amps, s->S, m, pos.data(), s->hist, s->stream); });
  if (rc) return rc;
  std::vector<double> pr(no);
  HIPCHK(hipMemcpyAsync(pr.data(), s->hist, no * sizeof(double), hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  // selection as measure-specific-qubits (state.clj:962-971)
  double total = 0.0;
  for (uint64_t o = 0; o < no; ++o) total += pr[o];
  const double r = u * total;
  double cum = 0.0;
  uint64_t sel = 0;
  for (uint64_t o = 0; o < no; ++o) {
    cum += pr[o];
    if (cum < r) sel = o + 1; else break;
  }
  if (sel > no - 1) sel = no - 1;
  const double p = pr[sel];
  const double f = p > 0 ? 1.0 / std::sqrt(p) : 1.0;
  rc = timed(s, QSV_KCLASS_OTHER, 2.0 * s->S * s->bytes_per_amp(),
             [&] { launch_collapse(s->prec, s->amps, s->S, m, pos.data(), sel, f, s->stream); });
  if (rc) return rc;
  s->reach_left = kReachTotal;
  if (outcome) *outcome = sel;
  if (probs_out) std::memcpy(probs_out, pr.data(), no * sizeof(double));
  return QSV_OK;
}

bool qok(int q, int n) { return q >= 0 && q < n; }

// A decoded gate in global index-bit coordinates (bit b = n-1-q).
enum { BG_MEASURE = 10 };
// Records that act on the whole state and never enter a fused pass.
inline bool runs_alone(int kind) { return kind == BG_MEASURE || kind == FG_RENORM; }

struct BGate {
  int kind = FG_DENSE;     // FG_DENSE, FG_PHASE, FG_SWAP, FG_BLOCKADE or BG_MEASURE
  CtlBits cbits;           // control bits (all must be 1)
  int a = -1, b = -1;      // target bit / swap bits
  uint64_t bmask = 0;      // blockade index bits; measured qubit mask for BG_MEASURE
  bool phase_only = false;
  double m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  double u = 0.0;          // BG_MEASURE uniform
};

uint64_t gate_bits(const BGate& g)
{
  uint64_t v = 0;
  for (int c : g.cbits) v |= 1ull << c;
  if (g.a >= 0) v |= 1ull << g.a;
  if (g.b >= 0) v |= 1ull << g.b;
  if (g.kind == FG_BLOCKADE) v |= g.bmask;
  return v;
}

void emit_ctl(std::vector<BGate>& out, CtlBits cbits, int tb, const double m[8])
{
  BGate g;
  g.cbits = cbits;
  g.a = tb;
  std::memcpy(g.m, m, sizeof(g.m));
  if (is_diag(m)) {
    g.kind = FG_PHASE;
    g.phase_only = is_one(m[0], m[1]);
  }
  out.push_back(std::move(g));
}

void emit_swap(std::vector<BGate>& out, CtlBits cbits, int b1, int b2, double pr, double pi)
{
  BGate g;
  g.kind = FG_SWAP;
  g.cbits = cbits;
  g.a = b1;
  g.b = b2;
  g.m[0] = pr;
  g.m[1] = pi;
  out.push_back(std::move(g));
}

// apply-gate-to-state (circuit.clj:933-1072) for one op: validate and emit
// its gates. Controlled gates carry the transpose of the target matrix, as the
// reference's apply-controlled-gate applies it (gate.clj:461-486).
int decode_op(int n, const qsv_op& op, uint32_t flags, uint64_t seed, uint64_t* measure_k, std::vector<BGate>& out)
{
  const int k = op.kind;
  double m[8], t[8];
  auto bit = [n](int q) { return n - 1 - q; };
  switch (k) {
  case QSV_OP_X: case QSV_OP_Y: case QSV_OP_Z: case QSV_OP_H: case QSV_OP_S: case QSV_OP_SDG:
  case QSV_OP_T: case QSV_OP_TDG: case QSV_OP_RX: case QSV_OP_RY: case QSV_OP_RZ: case QSV_OP_PHASE:
    if (!qok(op.q[0], n)) return fail(QSV_E_INVALID, "target qubit out of range");
    gate_matrix(k, op.angle, m);
    emit_ctl(out, {}, bit(op.q[0]), m);
    return QSV_OK;
  case QSV_OP_U:
    if (!qok(op.q[0], n)) return fail(QSV_E_INVALID, "target qubit out of range");
    emit_ctl(out, {}, bit(op.q[0]), op.m);
    return QSV_OK;
  case QSV_OP_CNOT: case QSV_OP_CZ: case QSV_OP_CY: case QSV_OP_RYDBERG_CZ:
  case QSV_OP_CRX: case QSV_OP_CRY: case QSV_OP_CRZ: {
    const int c = op.q[0], tq = op.q[1];
    if (!qok(c, n) || !qok(tq, n) || c == tq) return fail(QSV_E_INVALID, "control/target invalid");
    const int gk = (k == QSV_OP_CNOT) ? QSV_OP_X
                 : (k == QSV_OP_CZ || k == QSV_OP_RYDBERG_CZ) ? QSV_OP_Z
                 : (k == QSV_OP_CY) ? QSV_OP_Y
                 : (k == QSV_OP_CRX) ? QSV_OP_RX
                 : (k == QSV_OP_CRY) ? QSV_OP_RY : QSV_OP_RZ;
    gate_matrix(gk, op.angle, m);
    transpose2(m, t);
    emit_ctl(out, {bit(c)}, bit(tq), t);
    return QSV_OK;
  }
  case QSV_OP_CU: {
    const int c = op.q[0], tq = op.q[1];
    if (!qok(c, n) || !qok(tq, n) || c == tq) return fail(QSV_E_INVALID, "control/target invalid");
    emit_ctl(out, {bit(c)}, bit(tq), op.m);
    return QSV_OK;
  }
  case QSV_OP_SWAP: case QSV_OP_ISWAP: {
    const int q1 = op.q[0], q2 = op.q[1];
    if (!qok(q1, n) || !qok(q2, n) || q1 == q2) return fail(QSV_E_INVALID, "swap qubits invalid");
    // the reference shifts by the qubit numbers themselves (gate.clj:768-778, 823-833)
    const bool msb = (flags & QSV_FLAG_MSB_SWAP) != 0;
    const int b1 = msb ? bit(q1) : q1, b2 = msb ? bit(q2) : q2;
    if (k == QSV_OP_ISWAP) emit_swap(out, {}, b1, b2, 0.0, 1.0);
    else emit_swap(out, {}, b1, b2, 1.0, 0.0);
    return QSV_OK;
  }
  case QSV_OP_TOFFOLI: {
    const int a = op.q[0], b = op.q[1], c = op.q[2];
    if (!qok(a, n) || !qok(b, n) || !qok(c, n) || a == b || a == c || b == c)
      return fail(QSV_E_INVALID, "toffoli qubits invalid");
    gate_matrix(QSV_OP_X, 0, m);
    emit_ctl(out, {bit(a), bit(b)}, bit(c), m);
    return QSV_OK;
  }
  case QSV_OP_FREDKIN: {
    const int a = op.q[0], b = op.q[1], c = op.q[2];
    if (!qok(a, n) || !qok(b, n) || !qok(c, n) || a == b || a == c || b == c)
      return fail(QSV_E_INVALID, "fredkin qubits invalid");
    emit_swap(out, {bit(a)}, bit(b), bit(c), 1.0, 0.0);
    return QSV_OK;
  }
  case QSV_OP_RYDBERG_CPHASE: {
    const int c = op.q[0], tq = op.q[1];
    if (!qok(c, n) || !qok(tq, n) || c == tq) return fail(QSV_E_INVALID, "control/target invalid");
    const double dm[8] = {1, 0, 0, 0, 0, 0, std::cos(op.angle), std::sin(op.angle)};
    emit_ctl(out, {bit(c)}, bit(tq), dm);
    return QSV_OK;
  }
  case QSV_OP_RYDBERG_BLOCKADE: {
    if (op.mask == 0 || (n < 64 && (op.mask >> n) != 0)) return fail(QSV_E_INVALID, "blockade qubit set invalid");
    BGate g;
    g.kind = FG_BLOCKADE;
    for (int q = 0; q < n; ++q)
      if ((op.mask >> q) & 1ull) g.bmask |= 1ull << bit(q);
    g.m[0] = std::cos(op.angle);
    g.m[1] = std::sin(op.angle);
    out.push_back(std::move(g));
    return QSV_OK;
  }
  case QSV_OP_GLOBAL_RX: case QSV_OP_GLOBAL_RY: case QSV_OP_GLOBAL_RZ: case QSV_OP_GLOBAL_H:
  case QSV_OP_GLOBAL_X: case QSV_OP_GLOBAL_Y: case QSV_OP_GLOBAL_Z: {
    // global-*-gate (gate.clj:1098-1253): the gate on qubits 0..n-1 in turn
    int gk;
    double ang = op.angle;
    switch (k) {
    case QSV_OP_GLOBAL_RX: gk = QSV_OP_RX; break;
    case QSV_OP_GLOBAL_RY: gk = QSV_OP_RY; break;
    case QSV_OP_GLOBAL_RZ: gk = QSV_OP_RZ; break;
    case QSV_OP_GLOBAL_H: gk = QSV_OP_H; break;
    case QSV_OP_GLOBAL_X: gk = QSV_OP_RX; ang = M_PI; break;
    case QSV_OP_GLOBAL_Y: gk = QSV_OP_RY; ang = M_PI; break;
    default: gk = QSV_OP_RZ; ang = M_PI; break;
    }
    gate_matrix(gk, ang, m);
    for (int q = 0; q < n; ++q) emit_ctl(out, {}, bit(q), m);
    return QSV_OK;
  }
  case QSV_OP_MEASURE: {
    if (op.mask == 0 || (n < 64 && (op.mask >> n) != 0)) return fail(QSV_E_INVALID, "measure: qubit set empty or out of range");
    BGate g;
    g.kind = BG_MEASURE;
    g.bmask = op.mask;
    g.u = qsv_uniform(seed, (*measure_k)++);
    out.push_back(std::move(g));
    return QSV_OK;
  }
  default:
    return fail(QSV_E_UNSUPPORTED, "Unknown gate type (kind " + std::to_string(k) + ")");
  }
}

int run_direct(qsv_state* s, const BGate& g)
{
  switch (g.kind) {
  case FG_DENSE:
  case FG_PHASE:
    return apply_ctl_bits(s, g.cbits, g.a, g.m);
  case FG_SWAP:
    return apply_swap_bits(s, g.cbits, g.a, g.b, g.m);
  case FG_BLOCKADE:
    return timed(s, QSV_KCLASS_DIAG, 2.0 * s->S * s->bytes_per_amp(),
                 [&] { launch_blockade(s->prec, s->amps, s->S, g.bmask, g.m, s->stream); });
  case FG_RENORM:
    return timed(s, QSV_KCLASS_OTHER, 3.0 * s->S * s->bytes_per_amp(),
                 [&] { launch_renorm(s->prec, s->amps, s->S, s->partials, s->dout, s->stream); });
  default:
    return measure_impl(s, g.bmask, g.u, nullptr, nullptr);
  }
}

// ---- fused passes --------------------------------------------------------
// Pass descriptors travel through a small ring of pinned host + device
// buffers; a slot is reused only after the event recorded behind its last
// pass has completed.
int pass_block_cost()
{
  const char* e = std::getenv("QSV_PASS_BLOCKS");   // read per launch: a test may lower it
  return e ? std::max(0, std::atoi(e)) : 650;
}

int upload_passes(qsv_state* s, const std::vector<char>& progs, const char** dev)
{
  auto& slot = s->ring[s->ring_next];
  s->ring_next = (s->ring_next + 1) % qsv_state::kRing;
  if (slot.event) HIPCHK(hipEventSynchronize(slot.event));
  const size_t need = progs.size();
  if (slot.cap < need) {
    // (passes of later slots may use the reach words that a slot starts with)
    HIPCHK(hipStreamSynchronize(s->stream));
    if (slot.host) HIPCHK(hipHostFree(slot.host));
    if (slot.dev) HIPCHK(hipFree(slot.dev));
    slot.host = nullptr;
    slot.dev = nullptr;
    slot.cap = 0;
    const size_t cap = std::max<size_t>(need + need / 2, 256 << 10);
    HIPCHK(hipHostMalloc((void**)&slot.host, cap, hipHostMallocDefault));
    HIPCHK(hipMalloc((void**)&slot.dev, cap));
    slot.cap = cap;
  }
  if (!slot.event) HIPCHK(hipEventCreateWithFlags(&slot.event, hipEventDisableTiming));
  std::memcpy(slot.host, progs.data(), need);
  HIPCHK(hipMemcpyAsync(slot.dev, slot.host, need, hipMemcpyHostToDevice, s->stream));
  *dev = slot.dev;
  s->ring_pending = &slot;
  return QSV_OK;
}

// The passes of one program on their way to the device: compiled one by one,
// launched a few at a time.
struct PassRun {
  bool f32 = false;
  int block_cost = 0;                      // FP32 passes: register-bit runs of that cost become PO_BLOCK ops
  std::complex<double> scalar{1.0, 0.0};   // the factors common to the whole state
  int reach = 0;                           // passes that tracked reach; kReachPasses: no more
  unsigned long long* reach_at = nullptr;  // in the buffer of the first launch (the ring reuses it after
                                           // four; tracked passes are in the first three)
  // compiled and not launched yet
  std::vector<char> progs;
  std::vector<size_t> at;
  std::vector<int> renorm;                 // FP_RENORM_* of each
  bool reach_head = false;                 // they start with room for TileNorm::reach
};

// |index> in s.
void fill_basis(qsv_state* s, uint64_t index)
{
  launch_fill_basis(s->prec, s->amps, s->S, index, s->stream);
  s->reach_left = kReachTotal;
}

// Compiles the next pass of a run. The last one applies the factors common to the
// whole state; `only`: it is the first one too.
void add_pass(qsv_state* s, PassRun& run, const FPass& p, bool last, bool only)
{
  if ((double)s->S * s->bytes_per_amp() < kReachBytes || only) run.reach = kReachPasses;
  if (run.reach == 0 && s->reach_left > 0) {
    run.progs.resize(kReachHead, 0);
    run.reach_head = true;
  }
  run.at.push_back(compile_pass(p, run.f32, run.block_cost, run.scalar, last, run.progs));
  run.renorm.push_back(p.renorm);
  PHead h;
  std::memcpy(&h, run.progs.data() + run.at.back(), sizeof(h));
  if (run.reach < kReachPasses && s->reach_left > 0 && (h.renorm & FP_KEEP_ZERO)) {
    h.renorm |= FP_REACH | (run.reach++ ? FP_REACH_USE : 0);
    --s->reach_left;
    std::memcpy(run.progs.data() + run.at.back(), &h, sizeof(h));
  } else {
    run.reach = kReachPasses;   // a pass that does not track it ends it
  }
}

int launch_passes(qsv_state* s, PassRun& run)
{
  if (run.at.empty()) return QSV_OK;
  const uint64_t ntiles = s->S >> kPassTileBits;
  TileNorm nb{nullptr, nullptr, nullptr, nullptr};
  if (run.f32) {
    if (!s->norm_buf) HIPCHK(hipMalloc((void**)&s->norm_buf, (2 * ntiles + 2) * sizeof(double)));
    nb = TileNorm{s->norm_buf, s->norm_buf + ntiles, s->norm_buf + 2 * ntiles, nullptr};
  }
  const char* dev = nullptr;
  int rc = upload_passes(s, run.progs, &dev);
  if (rc) return rc;
  if (run.reach_head) run.reach_at = reinterpret_cast<unsigned long long*>(const_cast<char*>(dev));
  nb.reach = run.reach_at;
  for (size_t i = 0; i < run.at.size(); ++i) {
    const char* p = dev + run.at[i];
    rc = timed(s, QSV_KCLASS_BLOCK, 2.0 * s->S * s->bytes_per_amp(),
               [&] { launch_pass(s->prec, run.f32, s->amps, p, ntiles, nb, s->stream); });
    if (rc) return rc;
    if (run.renorm[i] & FP_RENORM_OUT) {
      const bool first = (run.renorm[i] & FP_RENORM_IN) != 0;
      rc = timed(s, QSV_KCLASS_OTHER, (first ? 2.0 : 1.0) * ntiles * sizeof(double),
                 [&] { launch_norm_ctl(nb, ntiles, first, s->stream); });
      if (rc) return rc;
    }
  }
  HIPCHK(hipEventRecord(s->ring_pending->event, s->stream));
  s->passes_launched += run.at.size();
  run.progs.clear();
  run.at.clear();
  run.renorm.clear();
  run.reach_head = false;
  return QSV_OK;
}

// Index bits 0..L-1 are always tile bits, so a wave's loads are runs of 2^L
// amplitudes. Longer runs stream better but leave fewer tile bits for gates.
// Order of precedence: the tuner's per-state override while it measures,
// QSV_TILE_LOWBITS, the tuned width of this precision, then 4 (the shortest
// 30-qubit layers for both precisions in a sweep of 3..8).
std::atomic<int> g_tuned_low[2] = {{-1}, {-1}};

int tile_low_bits(const qsv_state* s)
{
  static const int env = [] {
    const char* v = std::getenv("QSV_TILE_LOWBITS");
    return v ? std::atoi(v) : -1;
  }();
  const int TB = kPassTileBits;
  const int tuned = g_tuned_low[s->prec == QSV_C128 ? 0 : 1].load();
  int L = s->tile_low >= 0 ? s->tile_low : env >= 0 ? env : tuned >= 0 ? tuned : 4;
  return std::max(low_bit_threshold(s), std::min(L, TB - 2));
}

// Which arithmetic a dense 2x2 (row-major, interleaved re/im) needs.
int dense_structure(const double m[8])
{
  if (m[0] == 0 && m[1] == 0 && m[6] == 0 && m[7] == 0 && m[2] == 1 && m[3] == 0 && m[4] == 1 && m[5] == 0)
    return DM_EXCHANGE;
  if (m[1] == 0 && m[3] == 0 && m[5] == 0 && m[7] == 0) return DM_REAL;
  if (m[1] == 0 && m[7] == 0 && m[2] == 0 && m[4] == 0) return DM_RX;
  return DM_GENERAL;
}

// A gate on tile-local bits (loc: local bit of each global bit, -1 outside the
// tile, where only controls and phases may lie).
void local_gate(const BGate& g, const int loc[64], FGate& fg)
{
  fg = FGate{};
  fg.kind = g.kind;
  fg.a = g.a >= 0 ? loc[g.a] : -1;
  fg.b = g.b >= 0 ? loc[g.b] : -1;
  if (g.kind == FG_PHASE && fg.a < 0) fg.gt = 1ull << g.a;
  for (int c : g.cbits) {
    if (loc[c] >= 0) fg.cmask |= 1u << loc[c];
    else fg.gmask |= 1ull << c;
  }
  if (g.kind == FG_BLOCKADE)
    for (uint64_t m = g.bmask; m; m &= m - 1) fg.bmask |= 1u << loc[__builtin_ctzll(m)];
  fg.sub = g.kind == FG_DENSE ? dense_structure(g.m) : (g.phase_only ? 1 : 0);
  std::memcpy(fg.m, g.m, sizeof(fg.m));
}

// Build one pass from the chosen gates (program order) and the tile bit set.
void build_pass(const qsv_state* s, const std::vector<BGate>& gs, const std::vector<size_t>& chosen, uint64_t set,
                FPass& p)
{
  const int TB = kPassTileBits;
  const int L = std::min(tile_low_bits(s), TB - 4);
  p.tb = TB;
  p.low = L;
  uint64_t tile = set;
  for (int b = 0; __builtin_popcountll(tile) < TB; ++b) tile |= 1ull << b;
  // Local bit order: the low run first (coalesced lanes), then the other tile
  // bits, and at local bits TB-2, TB-1 the two that the fewest dense gates
  // target. Register masks avoid those two where they can, so the wave-id
  // bits of the thread index (the top two non-register bits) stay on them
  // and most layout changes are wave-local.
  int ntarget[64] = {};
  for (size_t i = 0; i < chosen.size(); ++i) {
    const BGate& g = gs[chosen[i]];
    if (g.kind == FG_DENSE && g.a >= 0 && !(g.cbits.size() == 1 && dense_structure(g.m) == DM_EXCHANGE)) ntarget[g.a]++;
  }
  int w1 = -1, w2 = -1;   // the two least-targeted non-low tile bits
  for (int b = s->n - 1; b >= L; --b) {
    if (!((tile >> b) & 1ull)) continue;
    if (w1 < 0 || ntarget[b] < ntarget[w1]) { w2 = w1; w1 = b; }
    else if (w2 < 0 || ntarget[b] < ntarget[w2]) w2 = b;
  }
  int loc[64];
  for (int b = 0; b < 64; ++b) loc[b] = -1;
  int nl = 0;
  for (int b = 0; b < L; ++b) { p.pos[nl] = b; loc[b] = nl++; }
  for (int b = L; b < s->n; ++b)
    if (((tile >> b) & 1ull) && b != w1 && b != w2) { p.pos[nl] = b; loc[b] = nl++; }
  for (int b : {std::min(w1, w2), std::max(w1, w2)})
    if (b >= 0) { p.pos[nl] = b; loc[b] = nl++; }
  int ns = 0;
  for (int b = 0; b < s->n; ++b)
    if ((tile >> b) & 1ull) p.sorted_pos[ns++] = b;
  p.gates.resize(chosen.size());
  for (size_t i = 0; i < chosen.size(); ++i) local_gate(gs[chosen[i]], loc, p.gates[i]);
}

// The last pass of a run of passes needs no scale for a successor.
void end_run(FPass& last)
{
  int& rn = last.renorm;
  rn &= ~FP_RENORM_OUT;
  if (!(rn & FP_RENORM_APPLY)) rn = 0;
}

// Planning passes. A pass costs one trip of the state through HBM however many
// gates it holds, so fewer passes is what counts: only bits that a gate moves
// amplitudes along have to be tile bits, and gates whose shared bits are
// diagonal in both pass each other. Against taking every bit of a gate into the
// tile and blocking on any shared bit, six random layers of 27 qubits take 7
// passes instead of 9 (9.35 -> 8.0 ms in all), a two-layer MaxCut ansatz of 26
// qubits 5 instead of 8 (2.95 -> 2.57 ms), and the 512 circuits of a batch of
// such ansatzes 29 group launches instead of 55.
// What a gate asks of a pass: the bits that must be tile bits, the bits it acts
// on non-diagonally (x) and diagonally (z). Two gates commute where every bit
// they share is diagonal in both.
struct GateBits {
  uint64_t need, x, z;
};
GateBits pass_bits(const BGate& g)
{
  GateBits b{0, 0, 0};
  for (int c : g.cbits) b.z |= 1ull << c;
  if (g.kind == FG_DENSE) {
    b.need = b.x = 1ull << g.a;
  } else if (g.kind == FG_SWAP) {
    b.x = (1ull << g.a) | (1ull << g.b);
    b.need = b.x | b.z;
  } else if (g.kind == FG_BLOCKADE) {
    b.need = g.bmask;
    b.z |= g.bmask;
  } else if (g.kind == FG_PHASE) {
    b.z |= 1ull << g.a;
    // a first entry that cannot be divided out: the gate runs as a dense one
    if (!g.phase_only && !is_phase(g.m[0], g.m[1])) b.need = 1ull << g.a;
  }
  return b;
}
// The bits of the gates a pass leaves out so far.
struct Blocked {
  uint64_t x = 0, z = 0;
  bool passes(const GateBits& g) const { return !(g.x & (x | z)) && !(g.z & x); }
  void add(const GateBits& g)
  {
    x |= g.x;
    z |= g.z;
  }
};

// Greedy fusion of gs (program order) into passes. emit(pass) receives each
// pass, barrier(i) each gate that must run alone (a measurement, or a gate
// wider than a tile); both return a status. With f32, every pass gets the
// renormalisation flags of its position in its run of passes.
// The passes fuse_walk chose for a program: per pass, its gates (indices into
// the program) and its tile bit set. build_pass on the same gates and set
// rebuilds the pass, whatever the gates' matrices.
using PassShape = std::vector<std::pair<std::vector<uint32_t>, uint64_t>>;

template <class Emit, class Barrier>
int fuse_walk(const qsv_state* s, const std::vector<BGate>& gs, bool f32, Emit&& emit, Barrier&& barrier,
              PassShape* record = nullptr)
{
  const int TB = kPassTileBits;
  const int L = tile_low_bits(s);
  const uint64_t lowmask = (1ull << L) - 1ull;
  const uint64_t all = (s->n >= 64) ? ~0ull : ((1ull << s->n) - 1ull);
  const int max_gates = f32 ? kMaxPassGatesF32 : kMaxPassGates;
  const size_t N = gs.size();
  std::vector<char> done(N, 0);
  std::vector<GateBits> gbits(N);
  for (size_t i = 0; i < N; ++i) gbits[i] = pass_bits(gs[i]);
  std::vector<size_t> chosen;
  std::vector<GateBits> wbits;   // the window's gates, contiguous
  constexpr size_t kWindow = 1024, kCandidates = 64;
  // Gates with a target that a pass with tile bits `set` could take, in program
  // order, from the window: a gate whose needed bits are all in the set and that commutes with
  // every gate left out before it. The scan ends where every bit is blocked or
  // two layers' worth of gates in a row were left out. A gate left out only
  // because of its needed bits is where a larger set would part from this one:
  // `at` receives the scan's state there, one entry per set of missing bits
  // (the others cannot let any further gate in by themselves).
  struct Scan {
    Blocked out;
    size_t k = 0;
    int cnt = 0;
    uint64_t add = 0;
  };
  const size_t kMisses = 2 * (size_t)s->n + 8;
  auto absorbed = [&](Scan sc, uint64_t set, std::vector<Scan>* at) -> int {
    size_t misses = 0;
    for (; sc.k < wbits.size(); ++sc.k) {
      const GateBits& gb = wbits[sc.k];
      const bool free = sc.out.passes(gb);
      const uint64_t add = gb.need & ~set;
      if (free && !add) {
        misses = 0;
        if (gb.need && ++sc.cnt >= max_gates) break;
        continue;
      }
      if (at && free && at->size() < kCandidates) {
        bool seen = false;
        for (const Scan& c : *at) seen |= c.add == add;
        if (!seen) {
          at->push_back(sc);
          at->back().add = add;
        }
      }
      sc.out.add(gb);
      if ((sc.out.x & all) == all || ++misses > kMisses) break;
    }
    return sc.cnt;
  };
  std::vector<Scan> cands;
  size_t first = 0;
  bool run_first = true;   // the next pass starts a run (renormalisation target)
  int rc;
  while (true) {
    while (first < N && done[first]) ++first;
    if (first >= N) break;
    const BGate& g0 = gs[first];
    if (runs_alone(g0.kind) || __builtin_popcountll(gbits[first].need | lowmask) > TB) {
      if ((rc = barrier(first))) return rc;
      done[first] = 1;
      run_first = true;
      continue;
    }
    // Tile bits: the low run and the first gate's bits, then, while there is
    // room, the missing bits of one gate of the window at a time, choosing the
    // addition that lets the most further gates into the pass per added bit
    // (this pairs the partners of two-qubit gates instead of taking bits in
    // program order).
    uint64_t set = lowmask | gbits[first].need;
    if (s->n <= TB) {
      set = all;
    } else {
      wbits.clear();
      for (size_t i = first; i < N && wbits.size() < kWindow; ++i) {
        if (done[i]) continue;
        if (runs_alone(gs[i].kind)) break;
        wbits.push_back(gbits[i]);
      }
    }
    while (__builtin_popcountll(set) < TB) {
      cands.clear();
      const int base = absorbed(Scan{}, set, &cands);
      uint64_t best = 0;
      double best_score = 0.0;
      for (const Scan& c : cands) {
        if (__builtin_popcountll(set | c.add) > TB) continue;
        const double score = double(absorbed(c, set | c.add, nullptr) - base) / __builtin_popcountll(c.add);
        if (score > best_score) {
          best_score = score;
          best = c.add;
        }
      }
      if (!best) break;
      set |= best;
    }
    Blocked out;
    chosen.clear();
    size_t scanned = 0;
    for (size_t i = first; i < N && scanned < 4096; ++i) {
      if (done[i]) continue;
      ++scanned;
      if (runs_alone(gs[i].kind)) break;
      const GateBits& gb = gbits[i];
      if (out.passes(gb)) {
        const uint64_t nu = set | gb.need;
        if (__builtin_popcountll(nu) <= TB && chosen.size() < (size_t)max_gates) {
          set = nu;
          chosen.push_back(i);
          continue;
        }
      }
      out.add(gb);
      if ((out.x & all) == all) break;
    }
    FPass p;
    build_pass(s, gs, chosen, set, p);
    for (size_t i : chosen) done[i] = 1;
    if (record) record->emplace_back(std::vector<uint32_t>(chosen.begin(), chosen.end()), set);
    p.renorm = f32 ? (FP_RENORM_OUT | (run_first ? FP_RENORM_IN : FP_RENORM_APPLY)) : 0;
    run_first = false;
    if ((rc = emit(std::move(p)))) return rc;
  }
  return QSV_OK;
}

// ---- gate folding on the host (fused and batched paths) -------------------
// 2x2 complex products, row-major (re, im) pairs: c = a b.
void mul2(const double a[8], const double b[8], double c[8])
{
  for (int r = 0; r < 2; ++r)
    for (int col = 0; col < 2; ++col) {
      double re = 0, im = 0;
      for (int k = 0; k < 2; ++k) {
        const double ar = a[2 * (2 * r + k)], ai = a[2 * (2 * r + k) + 1];
        const double br = b[2 * (2 * k + col)], bi = b[2 * (2 * k + col) + 1];
        re += ar * br - ai * bi;
        im += ar * bi + ai * br;
      }
      c[2 * (2 * r + col)] = re;
      c[2 * (2 * r + col) + 1] = im;
    }
}

// a b == b a exactly (diagonal pairs; X with an X-axis rotation; ...).
bool commutes_exactly(const double a[8], const double b[8])
{
  double ab[8], ba[8];
  mul2(a, b, ab);
  mul2(b, a, ba);
  for (int k = 0; k < 8; ++k)
    if (!(ab[k] == ba[k])) return false;
  return true;
}

bool is_exchange(const double m[8])
{
  return m[0] == 0 && m[1] == 0 && m[2] == 1 && m[3] == 0 && m[4] == 1 && m[5] == 0 && m[6] == 0 && m[7] == 0;
}

void set_1q(BGate& g, const double m[8])
{
  std::memcpy(g.m, m, sizeof(g.m));
  g.kind = is_diag(m) ? FG_PHASE : FG_DENSE;
  g.phase_only = g.kind == FG_PHASE && is_one(m[0], m[1]);
}

bool is_1q(const BGate& g) { return (g.kind == FG_DENSE || g.kind == FG_PHASE) && g.cbits.empty(); }

// Does the one-qubit matrix m on bit b commute with gate x (which touches b)?
bool commutes_on_bit(const BGate& x, int b, const double m[8])
{
  if (x.kind == FG_DENSE || x.kind == FG_PHASE) {
    for (int c : x.cbits)
      if (c == b) return is_diag(m);   // b is a control: only diagonals commute with its projectors
    return commutes_exactly(m, x.m);   // b is the target
  }
  if (x.kind == FG_BLOCKADE) return is_diag(m);
  return false;
}

// Rewrite a decoded program into an equivalent one with fewer gates, exactly
// in the mathematics (floating-point rounding aside):
//  * CNOT(c,t) D CNOT(c,t) with D = diag(d0, d1) a one-qubit gate on t is the
//    diagonal |c,t> -> d_{t xor c} |c,t>: D on t, then diag(d1/d0, d0/d1) on t
//    controlled by c (two phase gates instead of two exchanges and a phase);
//  * a one-qubit gate is multiplied into the previous one-qubit gate on its
//    bit when every gate in between that touches the bit commutes with it.
// Measurements and renormalisations stay where they are and stop folding.
std::vector<BGate> fold_gates(const std::vector<BGate>& in)
{
  std::vector<BGate> out;
  out.reserve(in.size());
  // per bit: index in out of its pending one-qubit gate (-1: none), and the
  // gates touching the bit after that one (reused across calls)
  int last[64];
  std::fill(last, last + 64, -1);
  thread_local std::vector<int> since[64];
  auto reset = [&]() {
    std::fill(last, last + 64, -1);
    for (auto& v : since) v.clear();
  };
  reset();
  auto take = [&](const BGate& g) {
    if (runs_alone(g.kind)) {
      out.push_back(g);
      reset();
      return;
    }
    if (is_1q(g)) {
      const int b = g.a;
      if (last[b] >= 0) {
        bool ok = true;
        for (int j : since[b])
          if (!commutes_on_bit(out[j], b, g.m)) { ok = false; break; }
        if (ok) {
          double r[8];
          mul2(g.m, out[last[b]].m, r);
          set_1q(out[last[b]], r);
          return;
        }
      }
      out.push_back(g);
      last[b] = (int)out.size() - 1;
      since[b].clear();
      return;
    }
    out.push_back(g);
    const int idx = (int)out.size() - 1;
    uint64_t bits = gate_bits(g);
    while (bits) {
      const int b = __builtin_ctzll(bits);
      bits &= bits - 1;
      if (last[b] >= 0) since[b].push_back(idx);
    }
  };
  for (size_t i = 0; i < in.size(); ++i) {
    if (i + 2 < in.size()) {
      const BGate &x = in[i], &d = in[i + 1], &y = in[i + 2];
      const bool cnot = x.kind == FG_DENSE && x.cbits.size() == 1 && is_exchange(x.m);
      if (cnot && y.kind == FG_DENSE && y.cbits == x.cbits && y.a == x.a && is_exchange(y.m) && is_1q(d) &&
          d.a == x.a && is_diag(d.m)) {
        const double d0r = d.m[0], d0i = d.m[1], d1r = d.m[6], d1i = d.m[7];
        const double n0 = d0r * d0r + d0i * d0i, n1 = d1r * d1r + d1i * d1i;
        if (n0 > 0 && n1 > 0) {
          BGate p = d;
          set_1q(p, d.m);
          BGate c;
          c.kind = FG_PHASE;
          c.cbits = x.cbits;
          c.a = x.a;
          // d1 / d0 and d0 / d1
          c.m[0] = (d1r * d0r + d1i * d0i) / n0;
          c.m[1] = (d1i * d0r - d1r * d0i) / n0;
          c.m[6] = (d0r * d1r + d0i * d1i) / n1;
          c.m[7] = (d0i * d1r - d0r * d1i) / n1;
          c.phase_only = is_one(c.m[0], c.m[1]);
          take(p);
          take(c);
          i += 2;
          continue;
        }
      }
    }
    take(in[i]);
  }
  return out;
}

constexpr size_t kKeepGates = 1 << 13;   // a thread's working memory, kept from program to program

// A whole-register program (qsv_small.hip) of gates [g0, g1), none of which
// runs alone, appended to `out`; zero: it starts from |0..0>.
size_t compile_small(int n, const BGate* g0, const BGate* g1, bool zero, std::vector<char>& out)
{
  thread_local FPass p;   // (for the memory of its gates)
  p.tb = std::max(n, 4);
  p.renorm = zero ? FP_INIT_ZERO : 0;
  int loc[64];
  for (int b = 0; b < 64; ++b) loc[b] = b;
  for (int b = 0; b < 16; ++b) p.pos[b] = p.sorted_pos[b] = b;
  const size_t count = (size_t)(g1 - g0);
  if (p.gates.capacity() > std::max(count, kKeepGates)) std::vector<FGate>().swap(p.gates);
  p.gates.resize(count);
  for (size_t i = 0; i < count; ++i) local_gate(g0[i], loc, p.gates[i]);
  std::complex<double> scalar(1.0, 0.0);
  return compile_pass(p, false, 0, scalar, true, out);
}

// Fused programs of states smaller than a pass's tile: one launch per run of
// gates between those that run alone (per gate, a launch each: a 5-qubit
// program of 32 gates took 110 us).
int run_small(qsv_state* s, const std::vector<BGate>& gs)
{
  constexpr size_t kMaxGates = 1 << 14;   // bounds a program
  // So few gates cost less as launches of their own: copying a program up and
  // waiting for the copy takes as long as three of them. A call of one to four
  // gates and a wait, launches / program: 13.5 / 19, 16.5 / 19.5, 19 / 20, 21 /
  // 20.5 us; among others 5.5 / 11, 8.5 / 11, 11.3 / 11.4, 14 / 12 us.
  constexpr size_t kFewGates = 3;
  for (size_t i = 0; i < gs.size();) {
    size_t j = i;
    while (j < gs.size() && j - i < kMaxGates && !runs_alone(gs[j].kind)) ++j;
    if (j - i <= kFewGates) {
      const size_t end = std::max(j, i + 1);   // those, or the one that runs alone
      for (; i < end; ++i)
        if (const int rc = run_direct(s, gs[i])) return rc;
      continue;
    }
    std::vector<char> buf(256, 0);   // the instance, then its program
    SmallInst in{};
    in.n = s->n;
    in.prog = compile_small(s->n, &gs[i], &gs[i] + (j - i), false, buf);
    in.dest = ~0ull;
    std::memcpy(buf.data(), &in, sizeof(in));
    const char* dev = nullptr;
    int rc = upload_passes(s, buf, &dev);
    if (rc) return rc;
    SmallRun r{};
    r.prec = s->prec;
    r.progs = dev;
    r.insts = reinterpret_cast<const SmallInst*>(dev);
    r.states = s->amps;
    hipError_t e = hipSuccess;
    rc = timed(s, QSV_KCLASS_BLOCK, 2.0 * s->S * s->bytes_per_amp(),
               [&] { e = launch_small(r, small_class(s->n), 1, s->stream); });
    if (rc) return rc;
    HIPCHK(e);
    HIPCHK(hipEventRecord(s->ring_pending->event, s->stream));
    i = j;
  }
  return QSV_OK;
}

// flags: QSV_FLAG_FP64_PASSES keeps complex64 pass arithmetic in FP64; by
// default it is FP32, renormalised pass by pass (15 % faster per 30-qubit
// layer: no conversions, same register budget), and its register-bit runs
// become matrix-core blocks unless QSV_FLAG_VALU_PASSES. The gates are
// folded first.
int run_fused(qsv_state* s, const std::vector<BGate>& gs_in, uint32_t flags)
{
  const std::vector<BGate> gs = fold_gates(gs_in);
  if (s->n < kPassTileBits) return run_small(s, gs);
  const bool f32 = s->prec == QSV_C64 && !(flags & QSV_FLAG_FP64_PASSES);
  const bool blocks = !(flags & QSV_FLAG_VALU_PASSES);
  // Passes are launched while later ones are still planned and compiled: one, then
  // two, four and so on, so that the device starts early and the uploads stay few.
  // The newest pass waits until it is known whether it ends its run. Six layers of
  // 27 qubits 6.33 -> 6.13 ms, a two-layer 26-qubit ansatz 1.74 -> 1.64 ms, ten
  // layers of 19 qubits 311 -> 303 us. A register of one tile gains nothing from
  // splitting its only pass: 12 qubits 272 us whole, 303 us in pieces of 64 gates.
  size_t chunk = 1;
  PassRun run;
  run.f32 = f32;
  run.block_cost = f32 && blocks ? pass_block_cost() : 0;
  FPass newest;
  bool waiting = false, first = true;   // newest is not compiled yet; it starts its run
  auto end = [&]() {
    if (!waiting) return (int)QSV_OK;
    waiting = false;
    end_run(newest);
    add_pass(s, run, newest, true, first && run.at.empty());
    first = true;
    return launch_passes(s, run);
  };
  const int rc = fuse_walk(
      s, gs, f32,
      [&](FPass&& p) {
        if (waiting) {
          add_pass(s, run, newest, false, false);
          first = false;
        }
        newest = std::move(p);
        waiting = true;
        if (run.at.size() < chunk) return (int)QSV_OK;
        chunk = std::min<size_t>(2 * chunk, 512);
        return launch_passes(s, run);
      },
      [&](size_t i) {
        const int r = end();
        run.reach = kReachPasses;
        return r ? r : run_direct(s, gs[i]);
      });
  return rc ? rc : end();
}

// ---- Pauli-string expectations ------------------------------------------------
// Registers of at least this many qubits take the tiled sweeps; in smaller ones
// a few tiles leave most CUs idle and the state sits in the caches, so one grid
// row per string is faster. Whole calls, rows / tiles, complex128: n Z strings
// 30.5 / 30.3 us at 18 qubits, 33.0 / 29.8 at 19, 39 / 30 at 20; the 4n - 3
// strings of a Heisenberg chain 44 / 59 us at 18, 53 / 58 at 19, 82 / 62 at 20
// (complex64 within 15 % of these).
// A string by itself is a row: nothing shares its sweep, whose staging then
// only adds (a sweep / a row, one X-type string: 32 / 27 us at 20 qubits,
// 44 / 36 at 22, 80 / 64 at 24, 830 / 774 at 28; one Z string 29 / 27, 38 / 36,
// 67 / 63, 810 / 795). One Z string over complex64 is the exception, bound by the
// row's instructions: 51 / 49 us at 24 qubits, 71 / 72 at 25, 124 / 173 at 26.
constexpr int kPauliTileZ = 19, kPauliTileX = 20, kPauliLoneZ32 = 25;

// out[t] = Re((-i)^ny (sum_i (-1)^popc(i & sm) conj(a_i) a_(i ^ xm))) for every
// string t. Strings are taken 256 at a time: their launches follow one another
// and their results come back in one copy.
int pauli_sums(const qsv_state* s, const std::vector<uint64_t>& xm, const std::vector<uint64_t>& sm,
               const std::vector<int>& ny, double* out)
{
  constexpr size_t kChunk = 256;
  const int TB = 12, L = low_bit_threshold(s);
  const uint64_t low = (1ull << L) - 1ull;
  const uint64_t n_terms = xm.size();
  std::vector<double> res(kReduceOut);
  for (uint64_t t0 = 0; t0 < n_terms; t0 += kChunk) {
    const uint64_t t1 = std::min<uint64_t>(n_terms, t0 + kChunk);
    std::vector<std::pair<int, uint64_t>> slot_of;   // result slot -> string
    int slots = 0;
    std::vector<uint64_t> zs, xs, rows;   // strings by the kernel that takes them
    for (uint64_t t = t0; t < t1; ++t) {
      const bool lone = t1 - t0 == 1 && (xm[t] || s->prec == QSV_C128 || s->n < kPauliLoneZ32);
      if (lone || s->n < (xm[t] ? kPauliTileX : kPauliTileZ) || __builtin_popcountll(xm[t] | low) > TB) rows.push_back(t);
      else (xm[t] ? xs : zs).push_back(t);
    }
    // strings with the same X part next to each other, X parts by their highest bit
    std::stable_sort(xs.begin(), xs.end(), [&](uint64_t a, uint64_t b) { return xm[a] < xm[b]; });
    struct Pair { uint64_t a, b; bool two; };
    std::vector<Pair> pending;
    for (size_t k = 0; k < xs.size(); ++k) {
      const bool two = k + 1 < xs.size() && xm[xs[k + 1]] == xm[xs[k]];
      pending.push_back({xs[k], two ? xs[k + 1] : xs[k], two});
      k += two ? 1 : 0;
    }
    size_t zi = 0;
    while (zi < zs.size() || !pending.empty()) {
      PauliSweep sw{};
      uint64_t set = low;
      std::vector<Pair> take, left;
      for (const Pair& p : pending) {
        if (take.size() < (size_t)kPauliUnits && __builtin_popcountll(set | xm[p.a]) <= TB) {
          set |= xm[p.a];
          take.push_back(p);
        } else {
          left.push_back(p);
        }
      }
      pending.swap(left);
      for (int b = 0; __builtin_popcountll(set) < TB; ++b) set |= 1ull << b;
      for (int b = 0, k = 0; b < s->n; ++b)
        if ((set >> b) & 1ull) sw.pos[k++] = b;
      auto local = [&](uint64_t m) {
        uint32_t l = 0;
        for (int k = 0; k < TB; ++k) l |= (uint32_t)((m >> sw.pos[k]) & 1ull) << k;
        return l;
      };
      while (zi < zs.size() && sw.nz < kPauliZ) {
        slot_of.emplace_back(slots + sw.nz, zs[zi]);
        sw.zmask[sw.nz++] = sm[zs[zi++]];
      }
      for (size_t k = 0; k < take.size(); ++k) {
        const uint64_t a = take[k].a, b = take[k].b;
        PauliUnit& u = sw.u[k];
        u.x = local(xm[a]);
        u.top = 31 - __builtin_clz(u.x);
        u.s0 = local(sm[a]);
        u.s1 = local(sm[b]);
        u.g0 = sm[a] & ~set;
        u.g1 = sm[b] & ~set;
        u.im0 = ny[a] & 1;
        u.im1 = ny[b] & 1;
        slot_of.emplace_back(slots + sw.nz + 2 * (int)k, a);
        if (take[k].two) slot_of.emplace_back(slots + sw.nz + 2 * (int)k + 1, b);
      }
      // whole groups of four units (the padding repeats the last one, unread)
      sw.nu = ((int)take.size() + 3) & ~3;
      for (int k = (int)take.size(); k < sw.nu; ++k) sw.u[k] = sw.u[take.size() - 1];
      HIPCHK(launch_pauli_sweep(s->prec, s->amps, s->S, sw, s->partials, s->dout + slots, s->stream));
      slots += sw.nz + 2 * sw.nu;
    }
    for (size_t r0 = 0; r0 < rows.size(); r0 += kPauliRows) {
      PauliRows pr{};
      const int nr = (int)std::min<size_t>(kPauliRows, rows.size() - r0);
      for (int r = 0; r < nr; ++r) {
        const uint64_t t = rows[r0 + r];
        pr.x[r] = xm[t];
        pr.s[r] = sm[t];
        pr.im |= (uint64_t)(ny[t] & 1) << r;
        slot_of.emplace_back(slots + r, t);
      }
      HIPCHK(launch_pauli_rows(s->prec, s->amps, s->S, pr, nr, s->partials, s->dout + slots, s->stream));
      slots += nr;
    }
    HIPCHK(hipMemcpyAsync(res.data(), s->dout, sizeof(double) * slots, hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    for (const auto& st : slot_of) {
      // half the pairs: twice the sum; (-i)^ny i^(ny & 1) is -1 for ny = 2, 3 mod 4
      const double f = xm[st.second] ? 2.0 : 1.0;
      out[st.second] = ((ny[st.second] & 2) ? -f : f) * res[st.first];
    }
  }
  return QSV_OK;
}

// Pass shapes of grouped batch programs, by program structure: an optimiser
// loop resubmits the same circuits with new angles, and the fuser's choices
// depend only on which bits each gate touches, whether a diagonal one needs its
// target in the tile (its first entry is no phase), and the tile width, so a
// structure seen before skips the fuser's search. Keyed by the exact
// structure (hash plus full comparison); cleared when it grows past a bound.
struct ShapeEntry {
  std::vector<uint64_t> key;
  PassShape shape;
};
std::mutex g_shape_mu;
std::unordered_map<uint64_t, std::vector<ShapeEntry>> g_shapes;
size_t g_shape_count = 0;
constexpr size_t kMaxShapes = 16384;

std::vector<uint64_t> structure_key(int n, int prec, int L, const std::vector<BGate>& gs)
{
  std::vector<uint64_t> k;
  k.reserve(3 + 3 * gs.size());
  k.push_back((uint64_t)n | ((uint64_t)prec << 8) | ((uint64_t)L << 16));
  for (const BGate& g : gs) {
    k.push_back((uint64_t)(uint32_t)g.kind | ((uint64_t)(uint32_t)(g.a + 1) << 16) |
                ((uint64_t)(uint32_t)(g.b + 1) << 32) | ((uint64_t)g.cbits.size() << 48) |
                // a diagonal gate whose entries make its target a tile bit
                ((uint64_t)(g.kind == FG_PHASE && pass_bits(g).need) << 56));
    uint64_t c = 0;
    for (int x : g.cbits) c = (c << 8) | (uint64_t)(x + 1);
    k.push_back(c);
    k.push_back(g.bmask);
  }
  return k;
}

uint64_t key_hash(const std::vector<uint64_t>& k)
{
  uint64_t h = 1469598103934665603ull;
  for (uint64_t v : k) {
    h ^= v;
    h *= 1099511628211ull;
    h ^= h >> 29;
  }
  return h;
}

// Passes of one instance of a grouped batch (FP64 arithmetic, no
// renormalisation), appended to `bytes` truncated after the last gate; false
// if the program needs a gate run alone.
bool plan_group_passes(int n, int prec, const std::vector<BGate>& gs, std::vector<char>& bytes,
                       std::vector<int64_t>& offsets)
{
  qsv_state view;   // planning only: no device memory behind it
  view.n = n;
  view.prec = prec;
  view.S = 1ull << n;
  std::vector<FPass> passes;
  std::vector<uint64_t> key = structure_key(n, prec, tile_low_bits(&view), gs);
  const uint64_t h = key_hash(key);
  PassShape shape;
  bool hit = false;
  {
    std::lock_guard<std::mutex> lk(g_shape_mu);
    auto it = g_shapes.find(h);
    if (it != g_shapes.end())
      for (const ShapeEntry& e : it->second)
        if (e.key == key) {
          shape = e.shape;
          hit = true;
          break;
        }
  }
  if (hit) {
    std::vector<size_t> chosen;
    for (const auto& ps : shape) {
      chosen.assign(ps.first.begin(), ps.first.end());
      passes.emplace_back();
      build_pass(&view, gs, chosen, ps.second, passes.back());
    }
  }
  bool ok = true;
  if (!hit)
    fuse_walk(
        &view, gs, false,
        [&](FPass&& p) {
          passes.push_back(std::move(p));
          return QSV_OK;
        },
        [&](size_t) {
          ok = false;
          return QSV_E_UNSUPPORTED;
        },
        &shape);
  if (!hit && ok) {
    std::lock_guard<std::mutex> lk(g_shape_mu);
    if (g_shape_count >= kMaxShapes) {
      g_shapes.clear();
      g_shape_count = 0;
    }
    g_shapes[h].push_back(ShapeEntry{std::move(key), std::move(shape)});
    ++g_shape_count;
  }
  // the instance's first pass writes |0..0> itself
  std::complex<double> scalar(1.0, 0.0);
  for (size_t i = 0; ok && i < passes.size(); ++i) {
    if (i == 0) passes[i].renorm |= FP_INIT_ZERO;
    offsets.push_back((int64_t)compile_pass(passes[i], false, 0, scalar, i + 1 == passes.size(), bytes));
  }
  return ok;
}

int check_state(const qsv_state* s)
{
  if (!s || !s->amps) return fail(QSV_E_INVALID, "null or destroyed state");
  HIPCHK(hipSetDevice(s->device));
  return QSV_OK;
}

constexpr uint64_t kXferChunk = 1ull << 24;  // amplitudes per staged transfer
constexpr uint64_t kShotsKept = 1ull << 16;  // outcomes of qsv_sample that a state keeps room for

}  // namespace

namespace qsv {
int api_fail(int code, const char* msg) { return fail(code, msg); }
int api_ensure_init() { return ensure_init(); }
int api_state_raw(const ::qsv_state* s, void** amps, hipStream_t* st, int* n, int* prec)
{
  if (!s) return fail(QSV_E_INVALID, "null state");
  *amps = s->amps;
  *st = s->stream;
  *n = s->n;
  *prec = s->prec;
  return QSV_OK;
}
}  // namespace qsv

extern "C" {

int qsv_init(int device)
{
  std::lock_guard<std::mutex> lk(g_mu);
  int count = 0;
  HIPCHK(hipGetDeviceCount(&count));
  if (device < 0 || device >= count) return fail(QSV_E_INVALID, "device index out of range");
  HIPCHK(hipSetDevice(device));
  int rc = resolve_scratch_locked(device);
  if (rc) return rc;
  g_device = device;
  g_init = true;
  return QSV_OK;
}

int qsv_shutdown(void)
{
  pool_release();
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_init) hipDeviceSynchronize();
  g_init = false;
  return QSV_OK;
}

int qsv_device_query(qsv_device_info* out)
{
  if (!out) return fail(QSV_E_INVALID, "null output");
  int rc = ensure_init();
  if (rc) return rc;
  hipDeviceProp_t p;
  HIPCHK(hipGetDeviceProperties(&p, g_device));
  std::memset(out, 0, sizeof(*out));
  std::snprintf(out->name, sizeof(out->name), "%s", p.name);
  std::snprintf(out->arch, sizeof(out->arch), "%s", p.gcnArchName);
  out->compute_units = p.multiProcessorCount;
  out->wavefront_size = p.warpSize;
  size_t fr = 0, tot = 0;
  HIPCHK(hipMemGetInfo(&fr, &tot));
  out->hbm_bytes = tot;
  out->hbm_free_bytes = fr;
  return QSV_OK;
}

const char* qsv_last_error(void) { return g_err.c_str(); }

const char* qsv_version(void) { return "qsv 0.1.0 (gfx950)"; }

double qsv_uniform(uint64_t seed, uint64_t k)
{
  uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

int qsv_state_create(int num_qubits, int precision, qsv_state** out)
{
  if (!out) return fail(QSV_E_INVALID, "null output");
  *out = nullptr;
  if (num_qubits < 1 || num_qubits > 36) return fail(QSV_E_INVALID, "num_qubits must be in [1, 36]");
  if (precision != QSV_C128 && precision != QSV_C64) return fail(QSV_E_INVALID, "unknown precision");
  int rc = ensure_init();
  if (rc) return rc;
  auto* s = new qsv_state();
  s->n = num_qubits;
  s->prec = precision;
  s->device = g_device;
  s->S = 1ull << num_qubits;
  auto cleanup = [&](int code, const std::string& msg) {
    if (s->amps) hipFree(s->amps);
    if (s->partials) hipFree(s->partials);
    if (s->dout) hipFree(s->dout);
    if (s->stream) hipStreamDestroy(s->stream);
    delete s;
    return fail(code, msg);
  };
  if (hipSetDevice(s->device) != hipSuccess) return cleanup(QSV_E_DEVICE, "hipSetDevice failed");
  if (hipMalloc(&s->amps, s->S * s->bytes_per_amp()) != hipSuccess)
    return cleanup(QSV_E_NOMEM, "hipMalloc of state vector failed (" + std::to_string(s->S * s->bytes_per_amp()) + " B)");
  if (hipMalloc(&s->partials, sizeof(double) * kPartials) != hipSuccess)
    return cleanup(QSV_E_NOMEM, "hipMalloc of reduction scratch failed");
  if (hipMalloc(&s->dout, sizeof(double) * kReduceOut) != hipSuccess)
    return cleanup(QSV_E_NOMEM, "hipMalloc of reduction output failed");
  if (hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess)
    return cleanup(QSV_E_DEVICE, "hipStreamCreate failed");
  fill_basis(s, 0);
  if (hipStreamSynchronize(s->stream) != hipSuccess) return cleanup(QSV_E_DEVICE, "initialising |0..0> failed");
  *out = s;
  return QSV_OK;
}

int qsv_state_destroy(qsv_state* s)
{
  if (!s) return QSV_OK;
  hipSetDevice(s->device);
  if (s->stream) hipStreamSynchronize(s->stream);
  for (auto& p : s->pending) {
    hipEventDestroy(p.a);
    hipEventDestroy(p.b);
  }
  for (auto e : s->evpool) hipEventDestroy(e);
  for (auto& slot : s->ring) {
    if (slot.host) hipHostFree(slot.host);
    if (slot.dev) hipFree(slot.dev);
    if (slot.event) hipEventDestroy(slot.event);
  }
  if (s->amps) hipFree(s->amps);
  if (s->partials) hipFree(s->partials);
  if (s->dout) hipFree(s->dout);
  if (s->prefix) hipFree(s->prefix);
  if (s->hist) hipFree(s->hist);
  if (s->norm_buf) hipFree(s->norm_buf);
  if (s->shot_dev) hipFree(s->shot_dev);
  if (s->samp_dev) hipFree(s->samp_dev);
  if (s->samp_host) hipHostFree(s->samp_host);
  if (s->stream) hipStreamDestroy(s->stream);
  delete s;
  return QSV_OK;
}

int qsv_state_num_qubits(const qsv_state* s) { return s ? s->n : QSV_E_INVALID; }
int qsv_state_precision(const qsv_state* s) { return s ? s->prec : QSV_E_INVALID; }

int qsv_state_init_basis(qsv_state* s, uint64_t index)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (index >= s->S) return fail(QSV_E_INVALID, "basis index out of range");
  fill_basis(s, index);
  HIPCHK(hipGetLastError());
  return QSV_OK;
}

int qsv_state_upload(qsv_state* s, const double* amps, uint64_t offset, uint64_t count)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (!amps || offset > s->S || count > s->S - offset) return fail(QSV_E_INVALID, "upload range invalid");
  s->reach_left = kReachTotal;
  if (s->prec == QSV_C128) {
    HIPCHK(hipMemcpyAsync((char*)s->amps + offset * 16, amps, count * 16, hipMemcpyHostToDevice, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    return QSV_OK;
  }
  double* stage = nullptr;
  const uint64_t chunk = std::min<uint64_t>(count, kXferChunk);
  HIPCHK(hipMalloc(&stage, chunk * 16));
  for (uint64_t done = 0; done < count; done += chunk) {
    const uint64_t c = std::min(chunk, count - done);
    hipError_t e = hipMemcpyAsync(stage, amps + 2 * done, c * 16, hipMemcpyHostToDevice, s->stream);
    if (e == hipSuccess) launch_f64_to_c64(stage, (char*)s->amps + (offset + done) * 8, c, s->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
    if (e != hipSuccess) {
      hipFree(stage);
      return fail(QSV_E_DEVICE, std::string("upload: ") + hipGetErrorString(e));
    }
  }
  hipFree(stage);
  return QSV_OK;
}

int qsv_state_download(const qsv_state* s, double* amps, uint64_t offset, uint64_t count)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (!amps || offset > s->S || count > s->S - offset) return fail(QSV_E_INVALID, "download range invalid");
  if (s->prec == QSV_C128) {
    HIPCHK(hipMemcpyAsync(amps, (const char*)s->amps + offset * 16, count * 16, hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    return QSV_OK;
  }
  double* stage = nullptr;
  const uint64_t chunk = std::min<uint64_t>(count, kXferChunk);
  HIPCHK(hipMalloc(&stage, chunk * 16));
  for (uint64_t done = 0; done < count; done += chunk) {
    const uint64_t c = std::min(chunk, count - done);
    launch_c64_to_f64((const char*)s->amps + (offset + done) * 8, stage, c, s->stream);
    hipError_t e = hipMemcpyAsync(amps + 2 * done, stage, c * 16, hipMemcpyDeviceToHost, s->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
    if (e != hipSuccess) {
      hipFree(stage);
      return fail(QSV_E_DEVICE, std::string("download: ") + hipGetErrorString(e));
    }
  }
  hipFree(stage);
  return QSV_OK;
}

int qsv_state_copy(qsv_state* dst, const qsv_state* src)
{
  int rc = check_state(dst);
  if (rc) return rc;
  rc = check_state(src);
  if (rc) return rc;
  if (dst->n != src->n || dst->prec != src->prec) return fail(QSV_E_INVALID, "copy: shape or precision mismatch");
  HIPCHK(hipStreamSynchronize(src->stream));
  launch_copy(src->prec, src->amps, dst->amps, src->S, dst->stream);
  dst->reach_left = kReachTotal;
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(dst->stream));
  return QSV_OK;
}

int qsv_state_compare(const qsv_state* a, const qsv_state* b, double out[5])
{
  int rc = check_state(a);
  if (rc) return rc;
  rc = check_state(b);
  if (rc) return rc;
  if (!out) return fail(QSV_E_INVALID, "null output");
  if (a->n != b->n) return fail(QSV_E_INVALID, "compare: qubit counts differ");
  HIPCHK(hipStreamSynchronize(b->stream));
  std::lock_guard<std::mutex> lk(a->scratch_mu);
  launch_compare(a->prec, a->amps, b->prec, b->amps, a->S, a->partials, a->dout, a->stream);
  HIPCHK(hipMemcpyAsync(out, a->dout, sizeof(double) * 5, hipMemcpyDeviceToHost, a->stream));
  HIPCHK(hipStreamSynchronize(a->stream));
  return QSV_OK;
}

int qsv_state_sync(qsv_state* s)
{
  int rc = check_state(s);
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(s->stream));
  return QSV_OK;
}

int qsv_apply_program(qsv_state* s, const qsv_op* ops, uint64_t n_ops, uint32_t flags, uint64_t seed)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (n_ops && !ops) return fail(QSV_E_INVALID, "null ops");
  // decode and validate the whole program before launching anything
  std::vector<BGate> gates;
  gates.reserve(n_ops);
  uint64_t mk = 0;
  for (uint64_t i = 0; i < n_ops; ++i) {
    rc = decode_op(s->n, ops[i], flags, seed, &mk, gates);
    if (rc) {
      g_err = "op " + std::to_string(i) + ": " + g_err;
      return rc;
    }
  }
  if (flags & QSV_FLAG_FUSE) {
    rc = run_fused(s, gates, flags);
  } else {
    rc = QSV_OK;
    for (const auto& g : gates)
      if ((rc = run_direct(s, g))) break;
  }
  if (rc) return rc;
  HIPCHK(hipGetLastError());
  return QSV_OK;
}

int qsv_norm2(const qsv_state* s, double* out)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (!out) return fail(QSV_E_INVALID, "null output");
  std::lock_guard<std::mutex> lk(s->scratch_mu);
  launch_norm2(s->prec, s->amps, s->S, s->partials, s->dout, s->stream);
  HIPCHK(hipMemcpyAsync(out, s->dout, sizeof(double), hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  return QSV_OK;
}

int qsv_normalize(qsv_state* s)
{
  double n2 = 0;
  int rc = qsv_norm2(s, &n2);
  if (rc) return rc;
  const double norm = std::sqrt(n2);
  // normalize-state: divide only if norm > tolerance (state.clj:545-549)
  if (norm > 0 && norm > 1e-12) launch_scale(s->prec, s->amps, s->S, 1.0 / norm, s->stream);
  HIPCHK(hipGetLastError());
  return QSV_OK;
}

int qsv_probabilities(const qsv_state* s, uint64_t offset, uint64_t count, double* out)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (!out || offset > s->S || count > s->S - offset) return fail(QSV_E_INVALID, "probability range invalid");
  if (count == 0) return QSV_OK;
  double* buf = nullptr;
  const uint64_t chunk = std::min<uint64_t>(count, kXferChunk);
  HIPCHK(hipMalloc(&buf, chunk * sizeof(double)));
  for (uint64_t done = 0; done < count; done += chunk) {
    const uint64_t c = std::min(chunk, count - done);
    launch_probs(s->prec, s->amps, offset + done, c, buf, s->stream);
    hipError_t e = hipMemcpyAsync(out + done, buf, c * sizeof(double), hipMemcpyDeviceToHost, s->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
    if (e != hipSuccess) {
      hipFree(buf);
      return fail(QSV_E_DEVICE, std::string("probabilities: ") + hipGetErrorString(e));
    }
  }
  hipFree(buf);
  return QSV_OK;
}

int qsv_sample(const qsv_state* cs, uint64_t shots, uint64_t seed, uint64_t* outcomes)
{
  int rc = check_state(cs);
  if (rc) return rc;
  if (shots && !outcomes) return fail(QSV_E_INVALID, "null outcomes");
  std::lock_guard<std::mutex> lk(cs->scratch_mu);
  auto* s = const_cast<qsv_state*>(cs);
  if (!s->prefix) {
    const uint64_t nch = std::max<uint64_t>(1, s->S >> kSampleChunkLog);
    HIPCHK(hipMalloc(&s->prefix, nch * sizeof(double)));
  }
  // outcomes: up to kShotsKept in a device buffer that the state keeps (a
  // hipMalloc and the device-wide wait of a hipFree per call otherwise)
  uint64_t* dout = nullptr;
  const bool keep = shots <= kShotsKept;
  if (keep) {
    if (shots > s->shot_cap) {
      if (s->shot_dev) HIPCHK(hipFree(s->shot_dev));
      s->shot_dev = nullptr;
      s->shot_cap = 0;
      const uint64_t cap = std::max<uint64_t>(shots, 1024);
      HIPCHK(hipMalloc((void**)&s->shot_dev, cap * sizeof(uint64_t)));
      s->shot_cap = cap;
    }
    dout = s->shot_dev;
  } else {
    HIPCHK(hipMalloc(&dout, shots * sizeof(uint64_t)));
  }
  launch_sample(s->prec, s->amps, s->S, s->prefix, shots, seed, dout, s->stream);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && shots)
    e = hipMemcpyAsync(outcomes, dout, shots * sizeof(uint64_t), hipMemcpyDeviceToHost, s->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
  if (!keep) hipFree(dout);
  if (e != hipSuccess) return fail(QSV_E_DEVICE, std::string("sample: ") + hipGetErrorString(e));
  return QSV_OK;
}

int qsv_sample_noalloc(const qsv_state* s, uint64_t shots, uint64_t seed, uint64_t* outcomes)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (shots && !outcomes) return fail(QSV_E_INVALID, "null outcomes");
  if (s->n > QSV_NOALLOC_MAX_QUBITS)
    return fail(QSV_E_INVALID, "qsv_sample_noalloc: " + std::to_string(s->n) + " qubits exceed the scratch limit of " +
                                   std::to_string(QSV_NOALLOC_MAX_QUBITS));
  if (shots > QSV_NOALLOC_MAX_SHOTS)
    return fail(QSV_E_INVALID, "qsv_sample_noalloc: " + std::to_string(shots) + " shots exceed the scratch limit of " +
                                   std::to_string(QSV_NOALLOC_MAX_SHOTS));
  void* base = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    rc = resolve_scratch_locked(s->device);  // s->device is current (check_state)
    base = g_scratch_ptr[s->device];
  }
  if (rc) return rc;
  // the sampler overwrites every chunk sum and every outcome it reads back,
  // so nothing in the scratch needs clearing between calls
  double* prefix = static_cast<double*>(base);
  uint64_t* dout = reinterpret_cast<uint64_t*>(static_cast<unsigned char*>(base) + kNoAllocPrefixBytes);
  launch_sample(s->prec, s->amps, s->S, prefix, shots, seed, dout, s->stream);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && shots)
    e = hipMemcpyAsync(outcomes, dout, shots * sizeof(uint64_t), hipMemcpyDeviceToHost, s->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
  if (e != hipSuccess) return fail(QSV_E_DEVICE, std::string("sample_noalloc: ") + hipGetErrorString(e));
  return QSV_OK;
}

int qsv_measure_qubits(qsv_state* s, uint64_t mask, double u, uint64_t* outcome, double* probs)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (!(u >= 0.0 && u < 1.0)) return fail(QSV_E_INVALID, "uniform must lie in [0, 1)");
  rc = measure_impl(s, mask, u, outcome, probs);
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(s->stream));
  return QSV_OK;
}

int qsv_expect_pauli(const qsv_state* s, const char* strings, uint64_t n_terms, double* out)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (n_terms && (!strings || !out)) return fail(QSV_E_INVALID, "null argument");
  const int n = s->n;
  std::vector<uint64_t> xm(n_terms), sm(n_terms);
  std::vector<int> ny(n_terms);
  for (uint64_t t = 0; t < n_terms; ++t) {
    const char* p = strings + t * (uint64_t)n;
    uint64_t x = 0, sg = 0;
    int y = 0;
    for (int q = 0; q < n; ++q) {
      const uint64_t b = 1ull << (n - 1 - q);
      switch (p[q]) {
      case 'I': break;
      case 'X': x |= b; break;
      case 'Y': x |= b; sg |= b; ++y; break;
      case 'Z': sg |= b; break;
      default: return fail(QSV_E_INVALID, "pauli string holds a character outside IXYZ");
      }
    }
    xm[t] = x; sm[t] = sg; ny[t] = y;
  }
  std::lock_guard<std::mutex> lk(s->scratch_mu);
  return pauli_sums(s, xm, sm, ny, out);
}

int qsv_expect_1q(const qsv_state* s, int qubit, const double m[8], double out[2])
{
  int rc = check_state(s);
  if (rc) return rc;
  if (!m || !out) return fail(QSV_E_INVALID, "null argument");
  if (!qok(qubit, s->n)) return fail(QSV_E_INVALID, "qubit out of range");
  std::lock_guard<std::mutex> lk(s->scratch_mu);
  launch_expect1q(s->prec, s->amps, s->S, 1ull << (s->n - 1 - qubit), m, s->partials, s->dout, s->stream);
  HIPCHK(hipMemcpyAsync(out, s->dout, sizeof(double) * 2, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  return QSV_OK;
}

int qsv_inner(const qsv_state* a, const qsv_state* b, double out[2])
{
  int rc = check_state(a);
  if (rc) return rc;
  rc = check_state(b);
  if (rc) return rc;
  if (!out) return fail(QSV_E_INVALID, "null output");
  if (a->n != b->n || a->prec != b->prec) return fail(QSV_E_INVALID, "inner: shape or precision mismatch");
  HIPCHK(hipStreamSynchronize(b->stream));
  std::lock_guard<std::mutex> lk(a->scratch_mu);
  launch_inner(a->prec, a->amps, b->amps, a->S, a->partials, a->dout, a->stream);
  HIPCHK(hipMemcpyAsync(out, a->dout, sizeof(double) * 2, hipMemcpyDeviceToHost, a->stream));
  HIPCHK(hipStreamSynchronize(a->stream));
  return QSV_OK;
}

}  // extern "C"

namespace {

// Pooled device states for batched circuits too large for one workgroup's
// registers, keyed by (num_qubits, precision); reused across batches.
std::mutex g_pool_mu;
std::vector<qsv_state*> g_pool[2][40];
constexpr int kPoolPerSize = 8;

int pool_get(int n, int prec, int slot, qsv_state** out)
{
  std::lock_guard<std::mutex> lk(g_pool_mu);
  auto& v = g_pool[prec][n];
  while ((int)v.size() <= slot) {
    qsv_state* s = nullptr;
    int rc = qsv_state_create(n, prec, &s);
    if (rc) return rc;
    v.push_back(s);
  }
  *out = v[slot];
  return QSV_OK;
}

// Arena of grouped batch states (grow only; used under the batch mutex).
constexpr uint64_t kGroupArenaBytes = 8ull << 30;
void* g_group_arena = nullptr;
uint64_t g_group_cap = 0;

int grow_group_arena(uint64_t bytes)
{
  if (bytes <= g_group_cap) return QSV_OK;
  if (g_group_arena) HIPCHK(hipFree(g_group_arena));
  g_group_arena = nullptr;
  g_group_cap = 0;
  HIPCHK(hipMalloc(&g_group_arena, bytes));
  g_group_cap = bytes;
  return QSV_OK;
}

void pool_release()
{
  std::lock_guard<std::mutex> lk(g_pool_mu);
  for (auto& per_prec : g_pool)
    for (auto& v : per_prec) {
      for (qsv_state* s : v) qsv_state_destroy(s);
      v.clear();
    }
  if (g_group_arena) hipFree(g_group_arena);
  g_group_arena = nullptr;
  g_group_cap = 0;
  batch_cache_release();
}

template <class T>
int dev_upload(const std::vector<T>& v, T** d, hipStream_t st)
{
  *d = nullptr;
  if (v.empty()) return QSV_OK;
  HIPCHK(hipMalloc((void**)d, v.size() * sizeof(T)));
  HIPCHK(hipMemcpyAsync(*d, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, st));
  return QSV_OK;
}

// Buffers and streams of qsv_batch_expect_z, kept from call to call (grow
// only; used under the batch mutex, and only while the call's streams are
// idle at its start): allocating and freeing them per call took a sizeable
// part of a 4096-instance call.
struct GrowBuf {
  void* p = nullptr;
  size_t cap = 0;
  bool pinned = false;
};
// One instantiated launch sequence of the grouped passes, found again by the
// launch parameters it was captured with.
struct GroupGraph {
  std::vector<uint64_t> key;
  hipGraphExec_t exec = nullptr;
  uint64_t used = 0;
};
struct BatchCache {
  hipStream_t st = nullptr, gst = nullptr;
  GrowBuf recs_h{nullptr, 0, true};   // pinned staging of the small circuits' programs
  GrowBuf bytes_h{nullptr, 0, true};  // pinned staging of the grouped pass programs
  GrowBuf recs, insts, tz, tc, energy, bytes, offs, meta, part;
  std::vector<GroupGraph> graphs;   // at most kGroupGraphs, least recently used replaced
  uint64_t tick = 0;
};
constexpr size_t kGroupGraphs = 4;
BatchCache g_batch;

// One chunk of a grouped batch: c states of S amplitudes back to back in the
// arena, `rounds` pass launches, then one energy reduction.
struct GroupChunk {
  uint64_t S = 0, c = 0, rounds = 0;
  uint64_t table_at = 0;   // first entry of the chunk's rounds x c program offsets
  uint64_t meta_at = 0;    // first entry of its term ranges and destinations
  uint64_t bps = 1;        // reduction blocks per state
  uint32_t fill = 0;       // some instance has no pass: fill the arena first
};
// Device buffers that every launch of a grouped batch reads or writes.
struct GroupLaunch {
  int prec = 0;
  void* arena = nullptr;
  const char* progs = nullptr;
  const int64_t* table = nullptr;
  const uint64_t* meta = nullptr;
  double* part = nullptr;
  const uint64_t* tz = nullptr;
  const double* tc = nullptr;
  double* energy = nullptr;
};

void issue_group_launches(const GroupLaunch& g, const std::vector<GroupChunk>& chunks, hipStream_t st)
{
  for (const GroupChunk& ch : chunks) {
    if (ch.fill) launch_fill_group(g.prec, g.arena, ch.S, ch.c, st);
    for (uint64_t r = 0; r < ch.rounds; ++r)
      launch_pass_group(g.prec, g.arena, ch.S, (unsigned)ch.c, g.progs, g.table + ch.table_at + r * ch.c, st);
    launch_zexpect_group(g.prec, g.arena, ch.S, (unsigned)ch.c, g.tz, g.tc, g.meta + ch.meta_at, g.part,
                         (unsigned)ch.bps, g.meta + ch.meta_at + 2 * ch.c, g.energy, st);
  }
}

// Runs the launch sequence of a grouped batch on st. By default the sequence
// is captured once into a HIP graph (kernel nodes only) and replayed whenever
// a later call has the same launches and buffers: an optimiser loop that only
// changes angles resubmits the whole batch as one graph launch, its programs
// rewritten in place. QSV_BATCH_GRAPH=0 issues the kernels one by one.
int run_group_launches(const GroupLaunch& g, const std::vector<GroupChunk>& chunks, hipStream_t st)
{
  const char* env = std::getenv("QSV_BATCH_GRAPH");
  if (env && env[0] == '0') {
    issue_group_launches(g, chunks, st);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? QSV_OK : fail(QSV_E_DEVICE, std::string("batch: launch failed: ") + hipGetErrorString(e));
  }
  std::vector<uint64_t> key = {(uint64_t)g.prec,          (uint64_t)(uintptr_t)g.arena, (uint64_t)(uintptr_t)g.progs,
                               (uint64_t)(uintptr_t)g.table, (uint64_t)(uintptr_t)g.meta,  (uint64_t)(uintptr_t)g.part,
                               (uint64_t)(uintptr_t)g.tz,    (uint64_t)(uintptr_t)g.tc,    (uint64_t)(uintptr_t)g.energy};
  for (const GroupChunk& ch : chunks)
    key.insert(key.end(), {ch.S, ch.c, ch.rounds, ch.table_at, ch.meta_at, ch.bps, (uint64_t)ch.fill});
  GroupGraph* hit = nullptr;
  for (GroupGraph& gg : g_batch.graphs)
    if (gg.exec && gg.key == key) hit = &gg;
  if (!hit) {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    if (hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) != hipSuccess)
      return fail(QSV_E_DEVICE, "batch: stream capture failed to start");
    issue_group_launches(g, chunks, st);
    const hipError_t le = hipGetLastError();
    const hipError_t ce = hipStreamEndCapture(st, &graph);
    hipError_t ie = hipSuccess;
    if (le == hipSuccess && ce == hipSuccess) ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    if (graph) hipGraphDestroy(graph);
    if (le != hipSuccess || ce != hipSuccess || ie != hipSuccess) {
      if (exec) hipGraphExecDestroy(exec);
      const hipError_t e = le != hipSuccess ? le : ce != hipSuccess ? ce : ie;
      return fail(QSV_E_DEVICE, std::string("batch: graph capture failed: ") + hipGetErrorString(e));
    }
    if (g_batch.graphs.size() < kGroupGraphs) {
      g_batch.graphs.emplace_back();
      hit = &g_batch.graphs.back();
    } else {
      hit = &g_batch.graphs[0];
      for (GroupGraph& gg : g_batch.graphs)
        if (gg.used < hit->used) hit = &gg;
      // the stream is idle at a call's start: the old graph has finished
      if (hit->exec) hipGraphExecDestroy(hit->exec);
    }
    hit->key = std::move(key);
    hit->exec = exec;
  }
  hit->used = ++g_batch.tick;
  if (hipGraphLaunch(hit->exec, st) != hipSuccess) return fail(QSV_E_DEVICE, "batch: graph launch failed");
  return QSV_OK;
}

int grow(GrowBuf& b, size_t bytes)
{
  bytes = std::max<size_t>(bytes, 256);
  if (bytes <= b.cap) return QSV_OK;
  if (b.p) HIPCHK(b.pinned ? hipHostFree(b.p) : hipFree(b.p));
  b.p = nullptr;
  b.cap = 0;
  if (b.pinned) HIPCHK(hipHostMalloc(&b.p, bytes, hipHostMallocDefault));
  else HIPCHK(hipMalloc(&b.p, bytes));
  b.cap = bytes;
  return QSV_OK;
}

// Copies n elements to a grow-only device buffer on stream st.
template <class T>
int upload(GrowBuf& b, const T* src, size_t n, hipStream_t st)
{
  int rc = grow(b, n * sizeof(T));
  if (rc) return rc;
  if (n) HIPCHK(hipMemcpyAsync(b.p, src, n * sizeof(T), hipMemcpyHostToDevice, st));
  return QSV_OK;
}

void batch_cache_release()
{
  for (GroupGraph& gg : g_batch.graphs)
    if (gg.exec) hipGraphExecDestroy(gg.exec);
  g_batch.graphs.clear();
  {
    std::lock_guard<std::mutex> lk(g_shape_mu);
    g_shapes.clear();
    g_shape_count = 0;
  }
  for (GrowBuf* b : {&g_batch.recs_h, &g_batch.bytes_h, &g_batch.recs, &g_batch.insts, &g_batch.tz, &g_batch.tc,
                     &g_batch.energy, &g_batch.bytes, &g_batch.offs, &g_batch.meta, &g_batch.part}) {
    if (b->p) (void)(b->pinned ? hipHostFree(b->p) : hipFree(b->p));
    b->p = nullptr;
    b->cap = 0;
  }
  if (g_batch.st) hipStreamDestroy(g_batch.st);
  if (g_batch.gst) hipStreamDestroy(g_batch.gst);
  g_batch.st = g_batch.gst = nullptr;
}

}  // namespace

extern "C" {

int qsv_batch_expect_z(const qsv_batch_desc* d, double* energies)
{
  if (!d || !energies) return fail(QSV_E_INVALID, "null argument");
  if (d->precision != QSV_C128 && d->precision != QSV_C64) return fail(QSV_E_INVALID, "unknown precision");
  const uint64_t N = d->n_instances;
  if (N == 0) return QSV_OK;
  // the pooled states are shared: batches on one process run one at a time
  static std::mutex batch_mu;
  std::lock_guard<std::mutex> batch_lock(batch_mu);
  if (!d->num_qubits || !d->op_offsets || !d->term_offsets || (d->op_offsets[N] && !d->ops) ||
      (d->term_offsets[N] && (!d->term_zmask || !d->term_coeff)))
    return fail(QSV_E_INVALID, "batch descriptor has null arrays");
  // instance i reads ops [op_offsets[i], op_offsets[i+1]) and terms
  // [term_offsets[i], term_offsets[i+1]): both must be non-decreasing
  for (uint64_t i = 0; i < N; ++i)
    if (d->op_offsets[i] > d->op_offsets[i + 1] || d->term_offsets[i] > d->term_offsets[i + 1])
      return fail(QSV_E_INVALID, "instance " + std::to_string(i) + ": offsets must be non-decreasing");
  int rc = ensure_init();
  if (rc) return rc;
  HIPCHK(hipSetDevice(g_device));
  const int prec = d->precision;
  const int small_n = prec == QSV_C128 ? kSmallC128 : kSmallC64;
  const size_t B = prec == QSV_C128 ? 16 : 8;

  const uint64_t T0 = d->term_offsets[0];
  const uint64_t n_terms = d->term_offsets[N] - T0;
  std::vector<SmallInst> insts(N);
  std::vector<uint64_t> tz(n_terms);
  std::vector<double> tc(n_terms);
  std::vector<uint64_t> big_idx;
  std::vector<uint64_t> small_idx;
  for (uint64_t i = 0; i < N; ++i) {
    const int n = d->num_qubits[i];
    if (n < 1 || n > 34) return fail(QSV_E_INVALID, "instance " + std::to_string(i) + ": num_qubits out of range");
  }
  // Decode every instance, convert its Z terms, and plan and compile the passes
  // of the large ones; the small ones' programs follow when the device is busy
  // with those (small ones first left it idle for the larger half of the
  // planning: 512 MaxCut instances of 8 to 20 qubits 5.87 -> 4.98 ms), or at once
  // where there are no large ones: starting the host threads a second time costs
  // as much as compiling a hundred small circuits. Both phases are independent
  // per instance and run on a pool of host threads (at most 16); errors are
  // reported for the first failing instance in order, decode errors before term
  // errors, as a sequential pass would.
  std::vector<std::vector<BGate>> decoded(N);
  struct Plan {
    std::vector<char> bytes;
    std::vector<int64_t> offs;
    bool ok = false;
  };
  std::vector<int> dec_rc(N, 0);
  std::vector<std::string> dec_err(N);
  std::vector<char> term_bad(N, 0);
  std::vector<std::vector<char>> small_prog(N);
  std::vector<Plan> plans(N);
  bool any_large = false;
  for (uint64_t i = 0; i < N; ++i) any_large |= d->num_qubits[i] > small_n;
  const unsigned hw = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
  const unsigned nt = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(hw, N / 8 + 1));
  auto parallel_over = [&](uint64_t count, auto&& body) {
    std::atomic<uint64_t> next{0};
    auto worker = [&]() {
      for (uint64_t i; (i = next.fetch_add(1)) < count;) body(i);
    };
    std::vector<std::thread> pool;
    for (unsigned t = 1; t < nt; ++t) pool.emplace_back(worker);
    worker();
    for (auto& t : pool) t.join();
  };
  // A small circuit's program goes straight to the pinned staging memory that
  // earlier calls left (the stream is idle, nothing reads it), each at the next
  // free offset; where that memory is too short, the programs are gathered
  // again once it has grown.
  std::atomic<uint64_t> staged{0};   // programs are multiples of 256 bytes
  auto compile_one = [&](uint64_t i) {
    decoded[i] = fold_gates(decoded[i]);
    std::vector<char>& prog = small_prog[i];
    compile_small(d->num_qubits[i], decoded[i].data(), decoded[i].data() + decoded[i].size(), true, prog);
    const uint64_t at = staged.fetch_add(prog.size());
    insts[i].prog = at;
    if (at + prog.size() <= g_batch.recs_h.cap)
      std::memcpy(static_cast<char*>(g_batch.recs_h.p) + at, prog.data(), prog.size());
  };
  parallel_over(N, [&](uint64_t i) {
    const int n = d->num_qubits[i];
    uint64_t mk = 0;
    decoded[i].reserve(d->op_offsets[i + 1] - d->op_offsets[i] + 8);   // about one gate per op
    for (uint64_t k = d->op_offsets[i]; k < d->op_offsets[i + 1]; ++k) {
      if (d->ops[k].kind == QSV_OP_MEASURE) {
        dec_rc[i] = QSV_E_UNSUPPORTED;
        dec_err[i] = "instance " + std::to_string(i) + ": measurements are not batched";
        break;
      }
      const int r = decode_op(n, d->ops[k], 0, 0, &mk, decoded[i]);
      if (r) {
        dec_rc[i] = r;
        dec_err[i] = "instance " + std::to_string(i) + ", op " + std::to_string(k - d->op_offsets[i]) + ": " + g_err;
        break;
      }
    }
    // Z masks with bit q = Z on qubit q, to basis-index bits (qubit q = bit n-1-q)
    for (uint64_t k = d->term_offsets[i]; k < d->term_offsets[i + 1]; ++k) {
      const uint64_t qm = d->term_zmask[k];
      if (n < 64 && (qm >> n)) term_bad[i] = 1;
      uint64_t bm = 0;
      for (int q = 0; q < n; ++q)
        if ((qm >> q) & 1ull) bm |= 1ull << (n - 1 - q);
      tz[k - T0] = bm;
      tc[k - T0] = d->term_coeff[k];
    }
    if (dec_rc[i] || (n <= small_n && any_large)) return;
    if (n <= small_n) {
      compile_one(i);
      return;
    }
    decoded[i] = fold_gates(decoded[i]);
    plans[i].ok = plan_group_passes(n, prec, decoded[i], plans[i].bytes, plans[i].offs);
  });
  for (uint64_t i = 0; i < N; ++i)
    if (dec_rc[i]) return fail(dec_rc[i], dec_err[i]);
  for (uint64_t i = 0; i < N; ++i)
    if (term_bad[i]) return fail(QSV_E_INVALID, "instance " + std::to_string(i) + ": Z term on a missing qubit");
  for (uint64_t i = 0; i < N; ++i) {
    const int n = d->num_qubits[i];
    SmallInst& in = insts[i];
    in.n = n;
    in.t0 = d->term_offsets[i] - T0;
    in.t1 = d->term_offsets[i + 1] - T0;
    in.io = ~0ull;
    in.dest = i;
    (n <= small_n ? small_idx : big_idx).push_back(i);
  }

  if (!g_batch.st && hipStreamCreateWithFlags(&g_batch.st, hipStreamNonBlocking) != hipSuccess)
    return fail(QSV_E_DEVICE, "batch: stream creation failed");
  hipStream_t st = g_batch.st;
  hipEvent_t uploaded = nullptr;
  auto cleanup = [&]() {
    hipStreamSynchronize(st);
    if (uploaded) hipEventDestroy(uploaded);
    uploaded = nullptr;
  };
  if ((rc = upload(g_batch.tz, tz.data(), tz.size(), st)) || (rc = upload(g_batch.tc, tc.data(), tc.size(), st)) ||
      (rc = grow(g_batch.energy, N * sizeof(double)))) {
    cleanup();
    return rc;
  }
  uint64_t* const d_tz = static_cast<uint64_t*>(g_batch.tz.p);
  double* const d_tc = static_cast<double*>(g_batch.tc.p);
  double* const d_energy = static_cast<double*>(g_batch.energy.p);
  // the pooled states' streams read the uploaded terms: order them after the copies
  if (hipEventCreateWithFlags(&uploaded, hipEventDisableTiming) != hipSuccess ||
      hipEventRecord(uploaded, st) != hipSuccess) {
    cleanup();
    return fail(QSV_E_DEVICE, "batch: event creation failed");
  }
  // The small circuits: compile them if that is still to do, copy the programs
  // up, one launch per size class, largest circuits first, so the long workgroups
  // start early.
  std::vector<SmallInst> small;   // read by its copy until the stream is waited for
  auto run_small_circuits = [&]() -> int {
    if (any_large) parallel_over(small_idx.size(), [&](uint64_t k) { compile_one(small_idx[k]); });
    const uint64_t bytes = staged.load();
    if (bytes > g_batch.recs_h.cap) {
      const int rc = grow(g_batch.recs_h, bytes + bytes / 2);
      if (rc) return rc;
      for (uint64_t i : small_idx)
        std::memcpy(static_cast<char*>(g_batch.recs_h.p) + insts[i].prog, small_prog[i].data(), small_prog[i].size());
    }
    int rc = QSV_OK;
    char* const recs = static_cast<char*>(g_batch.recs_h.p);
    std::stable_sort(small_idx.begin(), small_idx.end(),
                     [&](uint64_t a, uint64_t b) { return insts[a].n > insts[b].n; });
    for (uint64_t i : small_idx) small.push_back(insts[i]);
    if ((rc = upload(g_batch.recs, recs, bytes, st)) || (rc = upload(g_batch.insts, small.data(), small.size(), st)))
      return rc;
    for (size_t k = 0; k < small.size();) {
      const int cls = small_class(small[k].n);
      size_t e = k;
      while (e < small.size() && small_class(small[e].n) == cls) ++e;
      SmallRun r{};
      r.prec = prec;
      r.progs = static_cast<const char*>(g_batch.recs.p);
      r.insts = static_cast<const SmallInst*>(g_batch.insts.p) + k;
      r.tz = d_tz;
      r.tc = d_tc;
      r.energies = d_energy;
      const hipError_t le = launch_small(r, cls, (unsigned)(e - k), st);
      if (le != hipSuccess)
        return fail(QSV_E_DEVICE, std::string("batch: small circuits: ") + hipGetErrorString(le));
      k = e;
    }
    return QSV_OK;
  };
  // circuits too large for one workgroup, grouped by qubit count: all instances of a
  // group sit back to back in one arena and advance one pass round per launch
  // (k_pass group mode, FP64 arithmetic); a program that needs a gate run
  // alone takes a pooled state of its own instead.
  std::vector<qsv_state*> used;
  std::vector<size_t> singles;
  bool small_done = false;
  {
    std::map<int, std::vector<size_t>, std::greater<int>> by_n;   // n (largest first) -> positions in big_idx
    for (size_t k = 0; k < big_idx.size(); ++k) by_n[insts[big_idx[k]].n].push_back(k);
    // Plan every chunk first. The descriptors of all chunks go up in one copy
    // each, so the launches of the whole batch follow one another with no host
    // wait, and the sequence can be replayed as one graph.
    std::vector<GroupChunk> chunks;
    std::vector<std::pair<const Plan*, uint64_t>> copies;   // program bytes and where they go
    uint64_t n_bytes = 0;
    std::vector<int64_t> table;
    std::vector<uint64_t> meta;   // per chunk: term ranges (2c), then destinations (c)
    uint64_t arena_need = 0;
    size_t part_need = 0;
    for (auto& kv : by_n) {
      const int n = kv.first;
      const uint64_t S = 1ull << n;
      const uint64_t per_chunk = std::max<uint64_t>(1, std::min<uint64_t>(65535, kGroupArenaBytes / (S * B)));
      std::vector<size_t>& members = kv.second;
      for (size_t c0 = 0; c0 < members.size(); c0 += per_chunk) {
        std::vector<std::vector<int64_t>> offs_of;
        std::vector<size_t> chunk;
        for (size_t m = c0; m < members.size() && m < c0 + per_chunk; ++m) {
          Plan& pl = plans[big_idx[members[m]]];
          if (pl.ok) {
            // per-instance descriptors are 256-byte multiples: appending keeps them aligned
            const int64_t base = (int64_t)n_bytes;
            copies.emplace_back(&pl, n_bytes);
            n_bytes += pl.bytes.size();
            std::vector<int64_t> offs(pl.offs);
            for (int64_t& o : offs) o += base;
            chunk.push_back(members[m]);
            offs_of.push_back(std::move(offs));
          } else {
            singles.push_back(members[m]);
          }
        }
        if (chunk.empty()) continue;
        GroupChunk ch{};
        ch.S = S;
        ch.c = chunk.size();
        for (const auto& o : offs_of) {
          ch.rounds = std::max<uint64_t>(ch.rounds, o.size());
          // every instance's first pass starts from |0..0>; an instance with
          // no pass at all needs the arena filled
          ch.fill |= o.empty() ? 1u : 0u;
        }
        ch.table_at = table.size();
        table.resize(table.size() + std::max<uint64_t>(1, ch.rounds * ch.c), -1);
        for (uint64_t y = 0; y < ch.c; ++y)
          for (size_t r = 0; r < offs_of[y].size(); ++r) table[ch.table_at + r * ch.c + y] = offs_of[y][r];
        ch.meta_at = meta.size();
        meta.resize(meta.size() + 3 * ch.c);
        for (uint64_t y = 0; y < ch.c; ++y) {
          const uint64_t i = big_idx[chunk[y]];
          meta[ch.meta_at + 2 * y] = insts[i].t0;
          meta[ch.meta_at + 2 * y + 1] = insts[i].t1;
          meta[ch.meta_at + 2 * ch.c + y] = i;
        }
        ch.bps = std::max<uint64_t>(1, std::min<uint64_t>(64, S / 4096));
        arena_need = std::max(arena_need, ch.c * S * B);
        part_need = std::max<size_t>(part_need, (size_t)(ch.c * ch.bps));
        chunks.push_back(ch);
      }
    }
    if (!chunks.empty()) {
      hipStream_t gst = nullptr;
      if ((!g_batch.gst && hipStreamCreateWithFlags(&g_batch.gst, hipStreamNonBlocking) != hipSuccess) ||
          hipStreamWaitEvent(gst = g_batch.gst, uploaded, 0) != hipSuccess) {
        cleanup();
        return fail(QSV_E_DEVICE, "batch: group stream setup failed");
      }
      // the group stream is idle here (the previous call ended with a wait on
      // it): growing and rewriting its buffers is safe
      // the programs are gathered into pinned staging memory on the host
      // threads, then copied up in one transfer
      if ((rc = grow(g_batch.bytes_h, n_bytes))) {
        cleanup();
        return rc;
      }
      char* const staged = static_cast<char*>(g_batch.bytes_h.p);
      parallel_over(copies.size(), [&](uint64_t k) {
        const std::vector<char>& b = copies[k].first->bytes;
        std::memcpy(staged + copies[k].second, b.data(), b.size());
      });
      if ((rc = grow_group_arena(arena_need)) || (rc = grow(g_batch.part, part_need * sizeof(double))) ||
          (rc = upload(g_batch.bytes, staged, n_bytes, gst)) ||
          (rc = upload(g_batch.offs, table.data(), table.size(), gst)) ||
          (rc = upload(g_batch.meta, meta.data(), meta.size(), gst))) {
        hipStreamSynchronize(gst);
        cleanup();
        return rc;
      }
      GroupLaunch gl{};
      gl.prec = prec;
      gl.arena = g_group_arena;
      gl.progs = static_cast<const char*>(g_batch.bytes.p);
      gl.table = static_cast<const int64_t*>(g_batch.offs.p);
      gl.meta = static_cast<const uint64_t*>(g_batch.meta.p);
      gl.part = static_cast<double*>(g_batch.part.p);
      gl.tz = d_tz;
      gl.tc = d_tc;
      gl.energy = d_energy;
      rc = run_group_launches(gl, chunks, gst);
      if (!rc) rc = run_small_circuits();
      small_done = true;
      hipError_t ge = hipStreamSynchronize(gst);
      if (rc) {
        cleanup();
        return rc;
      }
      if (ge != hipSuccess) {
        cleanup();
        return fail(QSV_E_DEVICE, std::string("batch: grouped passes failed: ") + hipGetErrorString(ge));
      }
    }
  }
  if (!small_done && (rc = run_small_circuits())) {
    cleanup();
    return rc;
  }
  // programs that need a gate run alone: fused passes on pooled states,
  // spread over the pool's streams so that several run at once
  int slot_rr[2][40] = {};
  for (size_t k : singles) {
    const uint64_t i = big_idx[k];
    const int n = insts[i].n;
    qsv_state* s = nullptr;
    const int slot = slot_rr[prec][n]++ % kPoolPerSize;
    if ((rc = pool_get(n, prec, slot, &s))) {
      cleanup();
      return rc;
    }
    if (hipStreamWaitEvent(s->stream, uploaded, 0) != hipSuccess) {
      cleanup();
      return fail(QSV_E_DEVICE, "batch: stream wait failed");
    }
    fill_basis(s, 0);
    if ((rc = run_fused(s, decoded[i], 0))) {
      cleanup();
      return rc;
    }
    launch_zexpect(prec, s->amps, s->S, d_tz + insts[i].t0, d_tc + insts[i].t0, insts[i].t1 - insts[i].t0,
                   s->partials, d_energy + i, s->stream);
    used.push_back(s);
  }
  hipError_t e = hipGetLastError();
  for (qsv_state* s : used)
    if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(energies, d_energy, N * sizeof(double), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  cleanup();
  if (e != hipSuccess) return fail(QSV_E_DEVICE, std::string("batch: ") + hipGetErrorString(e));
  return QSV_OK;
}

}  // extern "C"

namespace {

double norm2_entries(const double m[8])
{
  double s = 0.0;
  for (int e = 0; e < 8; ++e) s += m[e] * m[e];
  return s;
}
void singular_values(const double m[8], double* least, double* most)
{
  const double re = m[0] * m[6] - m[1] * m[7] - m[2] * m[4] + m[3] * m[5];
  const double im = m[0] * m[7] + m[1] * m[6] - m[2] * m[5] - m[3] * m[4];
  const double det = std::hypot(re, im), t = norm2_entries(m);
  *most = std::sqrt(0.5 * (t + std::sqrt(std::max(0.0, t * t - 4.0 * det * det))));
  *least = *most > 0.0 ? det / *most : 0.0;
}
double least_singular(const double m[8])
{
  double least, most;
  singular_values(m, &least, &most);
  return least;
}
// Are the rows of m orthogonal and of equal length, to `tol` of that length squared?
bool unitary_multiple(const double m[8], double tol)
{
  const double r0 = m[0] * m[0] + m[1] * m[1] + m[2] * m[2] + m[3] * m[3];
  const double r1 = m[4] * m[4] + m[5] * m[5] + m[6] * m[6] + m[7] * m[7];
  const double re = m[0] * m[4] + m[1] * m[5] + m[2] * m[6] + m[3] * m[7];
  const double im = m[1] * m[4] - m[0] * m[5] + m[3] * m[6] - m[2] * m[7];
  return r0 > 1e-200 && std::abs(r0 - r1) <= tol * r0 && std::abs(re) <= tol * r0 && std::abs(im) <= tol * r0;
}

}  // namespace

extern "C" {

int qsv_noisy_trajectories(int num_qubits, int precision, const qsv_op* ops, uint64_t n_ops,
                           const qsv_kraus_site* sites, uint64_t n_sites, uint64_t n_traj, uint64_t seed,
                           uint64_t* outcomes, uint64_t n_keep, double* final_states)
{
  const int n = num_qubits;
  if (n < 1 || n > 34) return fail(QSV_E_INVALID, "num_qubits out of range");
  if (precision != QSV_C128 && precision != QSV_C64) return fail(QSV_E_INVALID, "unknown precision");
  if ((n_ops && !ops) || (n_sites && !sites) || (n_traj && !outcomes) || (n_keep && !final_states))
    return fail(QSV_E_INVALID, "null argument");
  if (n_keep > n_traj) return fail(QSV_E_INVALID, "n_keep exceeds n_traj");
  if (n_sites >= QSV_TRAJ_SLOTS) return fail(QSV_E_INVALID, "too many noise sites");
  if (n_traj == 0) return QSV_OK;
  int rc = ensure_init();
  if (rc) return rc;
  HIPCHK(hipSetDevice(g_device));
  // clean gates of each op, in order
  std::vector<BGate> clean;
  std::vector<size_t> op_end(n_ops);
  uint64_t mk = 0;
  for (uint64_t i = 0; i < n_ops; ++i) {
    if (ops[i].kind == QSV_OP_MEASURE)
      return fail(QSV_E_UNSUPPORTED, "op " + std::to_string(i) + ": mid-circuit measurements are not supported in trajectories");
    rc = decode_op(n, ops[i], 0, 0, &mk, clean);
    if (rc) {
      g_err = "op " + std::to_string(i) + ": " + g_err;
      return rc;
    }
    op_end[i] = clean.size();
  }
  // each site's operators, scaled (the reference renormalises after applying
  // one, so any positive multiple gives the same state): to 1 where they are a
  // multiple of a unitary, which then keeps the norm, otherwise to
  // max |k_ij| = 1; and their selection weights max |k_ij|^2 (channel.clj:203-212)
  std::vector<std::vector<std::array<double, 8>>> kops(n_sites);
  std::vector<std::vector<double>> kw(n_sites);
  for (uint64_t k = 0; k < n_sites; ++k) {
    const qsv_kraus_site& st = sites[k];
    if (st.after_op >= n_ops) return fail(QSV_E_INVALID, "site " + std::to_string(k) + ": after_op out of range");
    if (k && st.after_op < sites[k - 1].after_op) return fail(QSV_E_INVALID, "sites must be ordered by after_op");
    if (st.qubit < 0 || st.qubit >= n) return fail(QSV_E_INVALID, "site " + std::to_string(k) + ": qubit out of range");
    if (st.n_kraus < 1 || st.n_kraus > QSV_MAX_KRAUS)
      return fail(QSV_E_INVALID, "site " + std::to_string(k) + ": n_kraus must be 1.." + std::to_string(QSV_MAX_KRAUS));
    for (int j = 0; j < st.n_kraus; ++j) {
      double mx = 0.0;
      for (int e = 0; e < 4; ++e) mx = std::max(mx, st.m[j][2 * e] * st.m[j][2 * e] + st.m[j][2 * e + 1] * st.m[j][2 * e + 1]);
      if (!(mx > 0.0) || !std::isfinite(mx))
        return fail(QSV_E_INVALID, "site " + std::to_string(k) + ": Kraus operator " + std::to_string(j) + " is zero or not finite");
      std::array<double, 8> a;
      const bool unitary = unitary_multiple(st.m[j], 1e-14);
      const double sc = 1.0 / std::sqrt(unitary ? 0.5 * norm2_entries(st.m[j]) : mx);
      for (int e = 0; e < 8; ++e) a[e] = st.m[j][e] * sc;
      kops[k].push_back(a);
      kw[k].push_back(mx);
    }
  }
  auto choose = [&](uint64_t k, double u) -> int {
    const int nk = (int)kw[k].size();
    if (nk == 1) return 0;
    double acc = 0.0;
    for (int j = 0; j < nk; ++j) {
      acc += kw[k][j];
      if (u < acc || j >= nk - 1) return j;
    }
    return nk - 1;
  };
  // one trajectory's gate list: clean gates of op i, then its sites' operators.
  // A chosen operator scaled to max |k_ij| = 1 shrinks the norm, at most by its
  // smaller singular value. A renormalisation is a barrier of two state passes
  // here, so one follows every 16th site, and further ones keep the norm that the
  // operators since the last may have left above kLeastNorm: far from the 1e-12
  // below which a renormalisation leaves a state alone. An operator that could
  // take it below by itself (a projector) has one on either side.
  constexpr double kLeastNorm = 1e-8;
  std::vector<std::vector<double>> shrink(n_sites);
  for (uint64_t k = 0; k < n_sites; ++k)
    for (const auto& a : kops[k]) shrink[k].push_back(std::min(1.0, least_singular(a.data())));
  std::vector<double> clean_shrink(clean.size(), 1.0);
  for (size_t g = 0; g < clean.size(); ++g)
    if (clean[g].kind == FG_DENSE || clean[g].kind == FG_PHASE)
      clean_shrink[g] = std::min(1.0, least_singular(clean[g].m));
  auto trajectory_gates = [&](uint64_t t, std::vector<BGate>& out) {
    out.clear();
    size_t g = 0, k = 0;
    double least = 1.0;   // the norm is at least this
    auto renorm = [&]() {
      BGate r;
      r.kind = FG_RENORM;
      out.push_back(std::move(r));
      least = 1.0;
    };
    auto before = [&](double s) {
      if (!(least * s >= kLeastNorm) && least < 0.5) renorm();
      least *= s;
    };
    for (uint64_t i = 0; i < n_ops; ++i) {
      for (; g < op_end[i]; ++g) {
        before(clean_shrink[g]);
        out.push_back(clean[g]);
      }
      for (; k < n_sites && sites[k].after_op == i; ++k) {
        const int j = choose(k, qsv_uniform(seed, t * QSV_TRAJ_SLOTS + k));
        before(shrink[k][j]);
        emit_ctl(out, {}, n - 1 - sites[k].qubit, kops[k][j].data());
        if (least < kLeastNorm || (k + 1) % 16 == 0) renorm();
      }
    }
  };
  // the measurement of trajectory t draws qsv_uniform(seed, t * SLOTS + SLOTS - 1),
  // which is the sampler's shot 0 of seed_m below
  auto measure_seed = [&](uint64_t t) -> uint64_t {
    return seed + (t * QSV_TRAJ_SLOTS + QSV_TRAJ_SLOTS - 1) * 0x9E3779B97F4A7C15ull;
  };
  const size_t B = precision == QSV_C128 ? 16 : 8;
  const uint64_t S = 1ull << n;
  const int small_n = precision == QSV_C128 ? kSmallC128 : kSmallC64;
  std::vector<double> host_state;
  auto keep_state = [&](const void* dev_amps, int prec, uint64_t t, hipStream_t st) -> int {
    // copy one final state to the caller as normalised interleaved FP64
    host_state.resize(2 * S);
    double* dst = final_states + t * 2 * S;
    if (prec == QSV_C128) {
      HIPCHK(hipMemcpyAsync(dst, dev_amps, S * 16, hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
    } else {
      std::vector<float> f(2 * S);
      HIPCHK(hipMemcpyAsync(f.data(), dev_amps, S * 8, hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      for (uint64_t e = 0; e < 2 * S; ++e) dst[e] = f[e];
    }
    double nrm = 0.0;
    for (uint64_t e = 0; e < 2 * S; ++e) nrm += dst[e] * dst[e];
    if (nrm > 0.0) {
      const double inv = 1.0 / std::sqrt(nrm);
      for (uint64_t e = 0; e < 2 * S; ++e) dst[e] *= inv;
    }
    return QSV_OK;
  };
  std::vector<BGate> gs;
  if (n <= small_n) {
    // one workgroup per trajectory, all running one program: its noise sites
    // draw their uniform and choose their operator on the device. Final states
    // go to an arena (chunks bound it to 1 GiB), one shot each.
    // A renormalisation follows a site where the operators since the last one may
    // have taken the norm out of range (the compiler counts: sites of different
    // qubits run in no particular order), or every site where a gate of the program
    // does not keep the norm itself.
    bool unitary = true;
    for (const BGate& g : clean)
      if (g.kind == FG_DENSE || g.kind == FG_PHASE)
        unitary &= unitary_multiple(g.m, 1e-12) && std::abs(0.5 * norm2_entries(g.m) - 1.0) <= 1e-12;
    std::vector<KrausOp> table;
    FPass p;
    p.tb = std::max(n, 4);
    p.renorm = FP_INIT_ZERO;
    int loc[64];
    for (int b = 0; b < 64; ++b) loc[b] = b;
    for (int b = 0; b < 16; ++b) p.pos[b] = p.sorted_pos[b] = b;
    size_t g = 0, k = 0;
    for (uint64_t i = 0; i < n_ops; ++i) {
      for (; g < op_end[i]; ++g) {
        p.gates.emplace_back();
        local_gate(clean[g], loc, p.gates.back());
      }
      for (; k < n_sites && sites[k].after_op == i; ++k) {
        FGate f{};
        f.kind = FG_KRAUS;
        f.a = n - 1 - sites[k].qubit;
        f.b = (int32_t)k;
        f.cmask = (uint32_t)table.size();
        f.bmask = unitary ? 0u : 1u;
        f.m[0] = 1.0;   // the norm's least and most factor over the operators that a uniform below 1 reaches
        f.m[1] = 1.0;
        double acc = 0.0;
        for (int j = 0; j < sites[k].n_kraus && acc < 1.0; ++j) {
          KrausOp o;
          o.w = kw[k][j];
          acc += o.w;
          std::memcpy(o.m, kops[k][j].data(), sizeof(o.m));
          table.push_back(o);
          ++f.sub;
          double least, most;
          singular_values(o.m, &least, &most);
          f.m[0] = std::min(f.m[0], least);
          f.m[1] = std::max(f.m[1], most);
        }
        p.gates.push_back(f);
      }
    }
    if (table.empty()) table.push_back(KrausOp{});
    std::vector<char> prog;
    std::complex<double> scalar(1.0, 0.0);
    compile_pass(p, false, 0, scalar, true, prog);
    const uint64_t chunk = std::max<uint64_t>(1, std::min<uint64_t>(n_traj, (1ull << 30) / (S * B)));
    hipStream_t st = nullptr;
    HIPCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    void* arena = nullptr;
    char* d_prog = nullptr;
    KrausOp* d_table = nullptr;
    SampleJob* d_jobs = nullptr;
    uint64_t* d_out = nullptr;
    auto cleanup = [&]() {
      hipStreamSynchronize(st);
      hipFree(arena);
      hipFree(d_prog);
      hipFree(d_table);
      hipFree(d_jobs);
      hipFree(d_out);
      hipStreamDestroy(st);
    };
    if (hipMalloc(&arena, chunk * S * B) != hipSuccess ||
        hipMalloc((void**)&d_out, chunk * sizeof(uint64_t)) != hipSuccess ||
        hipMalloc((void**)&d_jobs, chunk * sizeof(SampleJob)) != hipSuccess) {
      cleanup();
      return fail(QSV_E_NOMEM, "trajectories: arena allocation failed");
    }
    if ((rc = dev_upload(prog, &d_prog, st)) || (rc = dev_upload(table, &d_table, st))) {
      cleanup();
      return rc;
    }
    std::vector<SampleJob> jobs(chunk);
    for (uint64_t t0 = 0; t0 < n_traj; t0 += chunk) {
      const uint64_t c = std::min(chunk, n_traj - t0);
      for (uint64_t i = 0; i < c; ++i) jobs[i] = SampleJob{i * S, i, 1, measure_seed(t0 + i), n, 0};
      SmallRun r{};
      r.prec = precision;
      r.progs = d_prog;
      r.one.n = n;
      r.one.dest = ~0ull;
      r.states = arena;
      r.kraus = d_table;
      r.seed = seed;
      r.traj0 = t0;
      hipError_t e = launch_small(r, small_class(n), (unsigned)c, st);
      if (e == hipSuccess) e = hipMemcpyAsync(d_jobs, jobs.data(), c * sizeof(SampleJob), hipMemcpyHostToDevice, st);
      if (e == hipSuccess) {
        launch_batch_sample(precision, arena, d_jobs, (unsigned)c, d_out, nullptr, st);
        e = hipGetLastError();
      }
      if (e == hipSuccess) e = hipMemcpyAsync(outcomes + t0, d_out, c * sizeof(uint64_t), hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipStreamSynchronize(st);
      if (e != hipSuccess) {
        cleanup();
        return fail(QSV_E_DEVICE, std::string("trajectories: ") + hipGetErrorString(e));
      }
      for (uint64_t i = 0; i < c && t0 + i < n_keep; ++i) {
        if ((rc = keep_state((const char*)arena + i * S * B, precision, t0 + i, st))) {
          cleanup();
          return rc;
        }
      }
    }
    cleanup();
    return QSV_OK;
  }
  // larger states: one state of this call's own, trajectory after
  // trajectory, fused passes
  qsv_state* s = nullptr;
  if ((rc = qsv_state_create(n, precision, &s))) return rc;
  uint64_t* d_out = nullptr;
  if (hipMalloc((void**)&d_out, sizeof(uint64_t)) != hipSuccess ||
      hipMalloc(&s->prefix, std::max<uint64_t>(1, s->S >> kSampleChunkLog) * sizeof(double)) != hipSuccess) {
    hipFree(d_out);
    qsv_state_destroy(s);
    return fail(QSV_E_NOMEM, "trajectories: allocation failed");
  }
  for (uint64_t t = 0; t < n_traj && !rc; ++t) {
    trajectory_gates(t, gs);
    fill_basis(s, 0);
    if ((rc = run_fused(s, gs, 0))) break;
    launch_sample(s->prec, s->amps, s->S, s->prefix, 1, measure_seed(t), d_out, s->stream);
    if (hipMemcpyAsync(outcomes + t, d_out, sizeof(uint64_t), hipMemcpyDeviceToHost, s->stream) != hipSuccess ||
        hipStreamSynchronize(s->stream) != hipSuccess) {
      rc = fail(QSV_E_DEVICE, "trajectories: launch failed");
      break;
    }
    if (t < n_keep) rc = keep_state(s->amps, s->prec, t, s->stream);
  }
  hipFree(d_out);
  const int drc = qsv_state_destroy(s);
  return rc ? rc : drc;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Serving: a native request loop with admission by state bytes and
// continuous batching (see include/qsv.h).
// ---------------------------------------------------------------------------
namespace {

using Clock = std::chrono::steady_clock;

struct SrvReq {
  uint64_t id = 0;
  int n = 0;
  std::vector<BGate> gates;
  std::vector<char> prog;   // small requests: the compiled program
  bool raw = false;         // ... still to be compiled by the scheduler
  uint64_t shots = 0, seed = 0;
  Clock::time_point t_submit, t_admit, t_done;
  int status = QSV_REQ_QUEUED;
  std::string err;
  std::vector<uint64_t> outcomes;
  double norm2 = NAN;       // FP64 sum |a|^2 of the final state, from the sampler
  uint64_t bytes = 0;
  bool small = false;
  bool cancel = false;      // cancelled while admitted: finishes as QSV_REQ_CANCELLED
  // in flight (large requests)
  qsv_state* st = nullptr;
  uint64_t* d_out = nullptr;
  uint64_t* h_out = nullptr;
  hipEvent_t ev = nullptr;
};

// Reusable device/host buffers for one batched launch of small requests.
struct SmallSlot {
  void* arena = nullptr;       size_t arena_cap = 0;     // final states, back to back
  char* progs = nullptr;       size_t progs_cap = 0;
  SmallInst* insts = nullptr;  size_t insts_cap = 0;
  SampleJob* jobs = nullptr;   size_t jobs_cap = 0;
  uint64_t* d_out = nullptr;   size_t out_cap = 0;
  uint64_t* h_out = nullptr;   size_t hout_cap = 0;
  double* d_norm = nullptr;    size_t norm_cap = 0;      // FP64 sum |a|^2 per request
  double* h_norm = nullptr;    size_t hnorm_cap = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev = nullptr;
  bool busy = false;
  std::vector<SrvReq*> reqs;
  std::vector<uint64_t> out_offsets;
};

template <class T>
int grow_dev(T** p, size_t* cap, size_t need)
{
  if (*cap >= need) return QSV_OK;
  if (*p) HIPCHK(hipFree(*p));
  *p = nullptr;
  const size_t c = std::max(need, (*cap) * 2);
  HIPCHK(hipMalloc((void**)p, c * sizeof(T)));
  *cap = c;
  return QSV_OK;
}

int grow_arena(void** p, size_t* cap, size_t need)
{
  if (*cap >= need) return QSV_OK;
  if (*p) HIPCHK(hipFree(*p));
  *p = nullptr;
  const size_t c = std::max(need, (*cap) * 2);
  HIPCHK(hipMalloc(p, c));
  *cap = c;
  return QSV_OK;
}

}  // namespace

struct qsv_server {
  qsv_server_config cfg{};
  uint64_t budget = 0, in_use = 0;
  int small_n = 14;   // the largest register of one workgroup
  std::mutex mu;
  std::condition_variable cv_work, cv_done;
  std::deque<SrvReq*> queue;
  std::vector<SrvReq*> pending_small, pending_large, running_large;
  std::unordered_map<uint64_t, SrvReq*> reqs;
  uint64_t next_id = 1;
  bool stop = false;
  std::thread th;
  // Small requests are folded and compiled by whichever thread is free: a
  // submitter leaves that to the scheduler while fewer than kRawMost wait for it,
  // and does it itself otherwise. All by submitters, bursts of 64 and 128 tiny
  // requests took 1.13 and 2.64 ms instead of 0.82 and 1.88 gate by gate; all by
  // the scheduler, large requests would wait for them.
  static constexpr int kRawMost = 4;
  std::atomic<int> raw{0};
  // Finished requests' states are kept for reuse (a hipFree waits for the
  // whole device, which would stall every request in flight) up to
  // budget / 5 bytes; beyond that they are freed.
  std::vector<qsv_state*> free_states[40];
  uint64_t cached_bytes = 0;
  static constexpr int kSlots = 4;
  SmallSlot slots[kSlots];
  qsv_server_stats stats{};
  std::string fatal;

  int inflight() const
  {
    int k = (int)running_large.size() + (int)pending_large.size() + (int)pending_small.size();
    for (const auto& s : slots)
      if (s.busy) k += (int)s.reqs.size();
    return k;
  }
};

namespace {

uint64_t state_bytes(const qsv_state* s) { return s->S * s->bytes_per_amp(); }

// Only the scheduler thread touches free_states and cached_bytes.
int take_state(qsv_server* sv, int n, qsv_state** out)
{
  auto& fl = sv->free_states[n];
  if (!fl.empty()) {
    *out = fl.back();
    fl.pop_back();
    sv->cached_bytes -= state_bytes(*out);
    return QSV_OK;
  }
  return qsv_state_create(n, sv->cfg.precision, out);
}

void give_state(qsv_server* sv, qsv_state* s)
{
  const uint64_t b = state_bytes(s);
  if (sv->cached_bytes + b <= sv->budget / 5) {
    sv->free_states[s->n].push_back(s);
    sv->cached_bytes += b;
  } else {
    qsv_state_destroy(s);
  }
}

void finish(qsv_server* sv, SrvReq* r, int status, const std::string& err)
{
  // called with sv->mu held, for an admitted request
  if (r->cancel && status == QSV_REQ_COMPLETED) {
    status = QSV_REQ_CANCELLED;
    r->outcomes.clear();
  }
  r->status = status;
  r->err = err;
  r->t_done = Clock::now();
  sv->in_use -= r->bytes;
  if (status == QSV_REQ_COMPLETED) sv->stats.completed++;
  else if (status == QSV_REQ_CANCELLED) sv->stats.cancelled++;
  else sv->stats.failed++;
}

// Outcome of polling a completion event: hipErrorNotReady means the work is
// still in flight; any status other than that and hipSuccess is a device
// error, which fails the request instead of leaving it running for ever.
enum { POLL_DONE, POLL_PENDING, POLL_FAILED };
int poll_event(hipEvent_t ev, std::string* err)
{
  const hipError_t e = hipEventQuery(ev);
  if (e == hipSuccess) return POLL_DONE;
  if (e == hipErrorNotReady) return POLL_PENDING;
  *err = std::string("device error while the request ran: ") + hipGetErrorString(e);
  return POLL_FAILED;
}

// A small request's whole-register program (large requests are folded by the
// fused runner, or run gate by gate without FUSE).
void prepare_small(qsv_server* sv, SrvReq* r)
{
  if (sv->cfg.flags & QSV_FLAG_FUSE) r->gates = fold_gates(r->gates);
  compile_small(r->n, r->gates.data(), r->gates.data() + r->gates.size(), true, r->prog);
  std::vector<BGate>().swap(r->gates);
}

// Launch every pending small request as one batched launch on a free slot.
int launch_small(qsv_server* sv, std::vector<SrvReq*>& batch)
{
  SmallSlot* slot = nullptr;
  for (auto& s : sv->slots)
    if (!s.busy) { slot = &s; break; }
  if (!slot) return 1;  // all slots in flight; retry later
  const int prec = sv->cfg.precision;
  const size_t B = prec == QSV_C128 ? 16 : 8;
  std::vector<char> progs;
  size_t prog_bytes = 0;
  for (SrvReq* r : batch) {
    if (r->raw) {
      prepare_small(sv, r);
      r->raw = false;
      --sv->raw;
    }
    prog_bytes += r->prog.size();
  }
  progs.reserve(prog_bytes);
  std::vector<SmallInst> insts(batch.size());
  std::vector<SampleJob> jobs(batch.size());
  slot->out_offsets.assign(batch.size(), 0);
  uint64_t arena_amps = 0, nout = 0;
  for (size_t k = 0; k < batch.size(); ++k) {
    SrvReq* r = batch[k];
    SmallInst& in = insts[k];
    in.n = r->n;
    in.prog = progs.size();   // programs are multiples of 256 bytes
    progs.insert(progs.end(), r->prog.begin(), r->prog.end());
    in.io = arena_amps;
    in.dest = ~0ull;
    jobs[k] = SampleJob{arena_amps, nout, r->shots, r->seed, r->n, 0};
    slot->out_offsets[k] = nout;
    arena_amps += 1ull << r->n;
    nout += r->shots;
  }
  std::stable_sort(insts.begin(), insts.end(), [](const SmallInst& a, const SmallInst& b) { return a.n > b.n; });
  int rc;
  if ((rc = grow_arena(&slot->arena, &slot->arena_cap, std::max<uint64_t>(arena_amps, 1) * B))) return rc;
  if ((rc = grow_dev(&slot->progs, &slot->progs_cap, std::max<size_t>(progs.size(), 1)))) return rc;
  if ((rc = grow_dev(&slot->insts, &slot->insts_cap, insts.size()))) return rc;
  if ((rc = grow_dev(&slot->jobs, &slot->jobs_cap, jobs.size()))) return rc;
  if ((rc = grow_dev(&slot->d_out, &slot->out_cap, std::max<uint64_t>(nout, 1)))) return rc;
  if ((rc = grow_dev(&slot->d_norm, &slot->norm_cap, jobs.size()))) return rc;
  if (slot->hnorm_cap < jobs.size()) {
    if (slot->h_norm) HIPCHK(hipHostFree(slot->h_norm));
    slot->h_norm = nullptr;
    const size_t c = std::max<size_t>(jobs.size(), slot->hnorm_cap * 2);
    HIPCHK(hipHostMalloc((void**)&slot->h_norm, c * sizeof(double), hipHostMallocDefault));
    slot->hnorm_cap = c;
  }
  if (slot->hout_cap < nout) {
    if (slot->h_out) HIPCHK(hipHostFree(slot->h_out));
    slot->h_out = nullptr;
    const size_t c = std::max<size_t>(nout, slot->hout_cap * 2);
    HIPCHK(hipHostMalloc((void**)&slot->h_out, c * sizeof(uint64_t), hipHostMallocDefault));
    slot->hout_cap = c;
  }
  if (!slot->stream) HIPCHK(hipStreamCreateWithFlags(&slot->stream, hipStreamNonBlocking));
  if (!slot->ev) HIPCHK(hipEventCreateWithFlags(&slot->ev, hipEventDisableTiming));
  HIPCHK(hipMemcpyAsync(slot->progs, progs.data(), progs.size(), hipMemcpyHostToDevice, slot->stream));
  HIPCHK(hipMemcpyAsync(slot->insts, insts.data(), insts.size() * sizeof(SmallInst), hipMemcpyHostToDevice, slot->stream));
  HIPCHK(hipMemcpyAsync(slot->jobs, jobs.data(), jobs.size() * sizeof(SampleJob), hipMemcpyHostToDevice, slot->stream));
  for (size_t k = 0; k < insts.size();) {
    const int cls = small_class(insts[k].n);
    size_t e = k;
    while (e < insts.size() && small_class(insts[e].n) == cls) ++e;
    SmallRun run{};
    run.prec = prec;
    run.progs = slot->progs;
    run.insts = slot->insts + k;
    run.states = slot->arena;
    HIPCHK(launch_small(run, cls, (unsigned)(e - k), slot->stream));
    k = e;
  }
  launch_batch_sample(prec, slot->arena, slot->jobs, (unsigned)jobs.size(), slot->d_out, slot->d_norm, slot->stream);
  if (nout)
    HIPCHK(hipMemcpyAsync(slot->h_out, slot->d_out, nout * sizeof(uint64_t), hipMemcpyDeviceToHost, slot->stream));
  HIPCHK(hipMemcpyAsync(slot->h_norm, slot->d_norm, jobs.size() * sizeof(double), hipMemcpyDeviceToHost, slot->stream));
  HIPCHK(hipEventRecord(slot->ev, slot->stream));
  HIPCHK(hipGetLastError());
  slot->reqs = batch;
  slot->busy = true;
  sv->stats.small_batches++;
  sv->stats.small_batched_requests += batch.size();
  return QSV_OK;
}

int launch_large(qsv_server* sv, SrvReq* r)
{
  int rc = take_state(sv, r->n, &r->st);
  if (rc) return rc;
  qsv_state* s = r->st;
  fill_basis(s, 0);
  if (sv->cfg.flags & QSV_FLAG_FUSE) rc = run_fused(s, r->gates, sv->cfg.flags);
  else {
    for (const auto& g : r->gates)
      if ((rc = run_direct(s, g))) break;
  }
  if (rc) return rc;
  if (!s->prefix) HIPCHK(hipMalloc(&s->prefix, std::max<uint64_t>(1, s->S >> kSampleChunkLog) * sizeof(double)));
  if (r->shots > s->samp_cap) {
    // grow the state's shot buffers (the state is idle: it was just taken)
    if (s->samp_dev) HIPCHK(hipFree(s->samp_dev));
    if (s->samp_host) HIPCHK(hipHostFree(s->samp_host));
    s->samp_dev = nullptr;
    s->samp_host = nullptr;
    s->samp_cap = 0;
    const uint64_t cap = std::max<uint64_t>(r->shots, 1024);
    HIPCHK(hipMalloc((void**)&s->samp_dev, cap * sizeof(uint64_t)));
    HIPCHK(hipHostMalloc((void**)&s->samp_host, cap * sizeof(uint64_t), hipHostMallocDefault));
    s->samp_cap = cap;
  }
  if (!s->norm_host) HIPCHK(hipHostMalloc((void**)&s->norm_host, sizeof(double), hipHostMallocDefault));
  r->d_out = s->samp_dev;
  r->h_out = s->samp_host;
  launch_sample(s->prec, s->amps, s->S, s->prefix, r->shots, r->seed, r->d_out, s->stream);
  if (r->shots)
    HIPCHK(hipMemcpyAsync(r->h_out, r->d_out, r->shots * sizeof(uint64_t), hipMemcpyDeviceToHost, s->stream));
  // the last inclusive chunk sum is the state's FP64 sum |a|^2
  const uint64_t nch = std::max<uint64_t>(1, s->S >> std::min<int>(s->n, kSampleChunkLog));
  HIPCHK(hipMemcpyAsync(s->norm_host, s->prefix + (nch - 1), sizeof(double), hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipEventCreateWithFlags(&r->ev, hipEventDisableTiming));
  HIPCHK(hipEventRecord(r->ev, s->stream));
  HIPCHK(hipGetLastError());
  return QSV_OK;
}

void release_large(qsv_server* sv, SrvReq* r, bool device_error = false)
{
  // the shot buffers belong to the state, which goes back to the cache
  // (not after a device error: then it is freed)
  if (r->ev) hipEventDestroy(r->ev);
  r->ev = nullptr;
  r->d_out = nullptr;
  r->h_out = nullptr;
  if (r->st) {
    if (device_error) qsv_state_destroy(r->st);
    else give_state(sv, r->st);
  }
  r->st = nullptr;
}

void server_loop(qsv_server* sv)
{
  hipSetDevice(g_device);
  // the waits below are of 50 us: the default slack of another 50 us would
  // double them (a burst of four tiny requests 204 -> 146 us)
  prctl(PR_SET_TIMERSLACK, 1000UL, 0UL, 0UL, 0UL);
  std::unique_lock<std::mutex> lk(sv->mu);
  while (true) {
    bool progressed = false;
    // 1. admission: arrival order, while the states fit the budget
    const int cap = sv->cfg.max_inflight > 0 ? sv->cfg.max_inflight : 32;
    while (!sv->queue.empty()) {
      SrvReq* r = sv->queue.front();
      // (cancelled requests leave the queue in qsv_server_cancel)
      if (sv->in_use + r->bytes > sv->budget && sv->in_use > 0) break;
      if (sv->inflight() >= cap) break;
      sv->queue.pop_front();
      sv->in_use += r->bytes;
      r->t_admit = Clock::now();
      r->status = QSV_REQ_RUNNING;
      (r->small ? sv->pending_small : sv->pending_large).push_back(r);
      progressed = true;
    }
    // 2. launches (outside the lock: submitters keep queueing meanwhile)
    std::vector<SrvReq*> smalls, larges;
    if (!sv->pending_small.empty()) {
      bool free_slot = false;
      for (auto& s : sv->slots) free_slot |= !s.busy;
      if (free_slot) smalls.swap(sv->pending_small);
    }
    larges.swap(sv->pending_large);
    if (!smalls.empty() || !larges.empty()) {
      lk.unlock();
      std::vector<std::pair<SrvReq*, std::string>> failed;
      if (!smalls.empty()) {
        const int rc = launch_small(sv, smalls);
        if (rc) for (SrvReq* r : smalls) failed.push_back({r, "batched launch failed: " + g_err});
      }
      std::vector<SrvReq*> started;
      for (SrvReq* r : larges) {
        const int rc = launch_large(sv, r);
        if (rc) failed.push_back({r, g_err});
        else started.push_back(r);
      }
      lk.lock();
      for (SrvReq* r : started) sv->running_large.push_back(r);
      for (auto& f : failed) {
        release_large(sv, f.first);
        finish(sv, f.first, QSV_REQ_FAILED, f.second);
      }
      if (!failed.empty()) sv->cv_done.notify_all();
      progressed = true;
    }
    // 3. completions (a device error fails the request and frees what it held)
    bool done_any = false;
    std::string perr;
    for (size_t k = 0; k < sv->running_large.size();) {
      SrvReq* r = sv->running_large[k];
      const int pr = poll_event(r->ev, &perr);
      if (pr != POLL_PENDING) {
        if (pr == POLL_DONE) {
          r->outcomes.assign(r->h_out, r->h_out + r->shots);
          r->norm2 = *r->st->norm_host;
        }
        release_large(sv, r, pr == POLL_FAILED);
        finish(sv, r, pr == POLL_DONE ? QSV_REQ_COMPLETED : QSV_REQ_FAILED, pr == POLL_DONE ? "" : perr);
        sv->running_large[k] = sv->running_large.back();
        sv->running_large.pop_back();
        done_any = true;
      } else {
        ++k;
      }
    }
    for (auto& slot : sv->slots) {
      if (!slot.busy) continue;
      const int pr = poll_event(slot.ev, &perr);
      if (pr == POLL_PENDING) continue;
      for (size_t k = 0; k < slot.reqs.size(); ++k) {
        SrvReq* r = slot.reqs[k];
        if (pr == POLL_DONE) {
          r->outcomes.assign(slot.h_out + slot.out_offsets[k], slot.h_out + slot.out_offsets[k] + r->shots);
          r->norm2 = slot.h_norm[k];
          finish(sv, r, QSV_REQ_COMPLETED, "");
        } else {
          finish(sv, r, QSV_REQ_FAILED, perr);
        }
      }
      slot.reqs.clear();
      slot.busy = false;
      done_any = true;
    }
    if (done_any) {
      sv->cv_done.notify_all();
      progressed = true;
    }
    const bool busy = !sv->running_large.empty() ||
                      std::any_of(std::begin(sv->slots), std::end(sv->slots), [](const SmallSlot& s) { return s.busy; });
    if (sv->stop && sv->queue.empty() && !busy && sv->pending_small.empty() && sv->pending_large.empty()) break;
    if (!progressed) {
      if (busy) sv->cv_work.wait_for(lk, std::chrono::microseconds(50));
      else sv->cv_work.wait_for(lk, std::chrono::milliseconds(5));
    }
  }
}

void fill_info(const SrvReq* r, qsv_request_info* info)
{
  if (!info) return;
  std::memset(info, 0, sizeof(*info));
  info->status = r->status;
  info->num_qubits = r->n;
  info->shots = r->shots;
  auto ms = [](Clock::time_point a, Clock::time_point b) {
    return std::chrono::duration<double, std::milli>(b - a).count();
  };
  if (r->status != QSV_REQ_QUEUED) info->queue_ms = ms(r->t_submit, r->t_admit);
  if (r->status >= QSV_REQ_COMPLETED) info->latency_ms = ms(r->t_submit, r->t_done);
  std::snprintf(info->error, sizeof(info->error), "%s", r->err.c_str());
  info->norm2 = r->status == QSV_REQ_COMPLETED ? r->norm2 : NAN;
}

}  // namespace

extern "C" {

int qsv_server_create(const qsv_server_config* cfg, qsv_server** out)
{
  if (!cfg || !out) return fail(QSV_E_INVALID, "null argument");
  if (cfg->precision != QSV_C64 && cfg->precision != QSV_C128) return fail(QSV_E_INVALID, "unknown precision");
  int rc = ensure_init();
  if (rc) return rc;
  HIPCHK(hipSetDevice(g_device));
  auto* sv = new qsv_server();
  sv->cfg = *cfg;
  sv->small_n = cfg->precision == QSV_C128 ? kSmallC128 : kSmallC64;
  size_t fr = 0, tot = 0;
  if (hipMemGetInfo(&fr, &tot) != hipSuccess) {
    delete sv;
    return fail(QSV_E_DEVICE, "hipMemGetInfo failed");
  }
  sv->budget = cfg->hbm_budget_bytes ? cfg->hbm_budget_bytes : (uint64_t)(0.8 * (double)fr);
  sv->stats.hbm_budget_bytes = sv->budget;
  sv->th = std::thread(server_loop, sv);
  *out = sv;
  return QSV_OK;
}

int qsv_server_submit(qsv_server* sv, int num_qubits, const qsv_op* ops, uint64_t n_ops, uint64_t shots,
                      uint64_t seed, uint64_t* request_id)
{
  if (!sv || !request_id || (n_ops && !ops)) return fail(QSV_E_INVALID, "null argument");
  if (num_qubits < 1 || num_qubits > 34) return fail(QSV_E_INVALID, "num_qubits must be in [1, 34]");
  auto* r = new SrvReq();
  r->t_submit = Clock::now();
  r->n = num_qubits;
  r->shots = shots;
  r->seed = seed;
  uint64_t mk = 0;
  r->gates.reserve(n_ops + 8);   // about one gate per op
  for (uint64_t i = 0; i < n_ops; ++i) {
    if (ops[i].kind == QSV_OP_MEASURE) {
      delete r;
      return fail(QSV_E_UNSUPPORTED, "op " + std::to_string(i) + ": mid-circuit measurement is not served");
    }
    const int rc = decode_op(num_qubits, ops[i], sv->cfg.flags, seed, &mk, r->gates);
    if (rc) {
      delete r;
      g_err = "op " + std::to_string(i) + ": " + g_err;
      return rc;
    }
  }
  const uint64_t B = sv->cfg.precision == QSV_C128 ? 16 : 8;
  r->bytes = (1ull << num_qubits) * B;
  r->small = sv->cfg.batch_small && num_qubits <= sv->small_n;
  if (r->bytes > sv->budget) {
    delete r;
    return fail(QSV_E_NOMEM, "request state exceeds the HBM budget");
  }
  if (r->small) {
    if (sv->raw < qsv_server::kRawMost) {
      r->raw = true;
      ++sv->raw;
    } else {
      prepare_small(sv, r);
    }
  }
  {
    std::lock_guard<std::mutex> lk(sv->mu);
    r->id = sv->next_id++;
    sv->reqs[r->id] = r;
    sv->queue.push_back(r);
    sv->stats.submitted++;
    sv->stats.max_queue_depth = std::max<uint64_t>(sv->stats.max_queue_depth, sv->queue.size());
    *request_id = r->id;
  }
  sv->cv_work.notify_one();
  return QSV_OK;
}

int qsv_server_status(qsv_server* sv, uint64_t request_id, qsv_request_info* info)
{
  if (!sv) return fail(QSV_E_INVALID, "null server");
  std::lock_guard<std::mutex> lk(sv->mu);
  auto it = sv->reqs.find(request_id);
  if (it == sv->reqs.end()) return fail(QSV_E_NOTFOUND, "unknown request id");
  fill_info(it->second, info);
  return QSV_OK;
}

int qsv_server_wait(qsv_server* sv, uint64_t request_id, double timeout_s, qsv_request_info* info,
                    uint64_t* outcomes)
{
  if (!sv) return fail(QSV_E_INVALID, "null server");
  std::unique_lock<std::mutex> lk(sv->mu);
  auto it = sv->reqs.find(request_id);
  if (it == sv->reqs.end()) return fail(QSV_E_NOTFOUND, "unknown request id");
  SrvReq* r = it->second;
  const auto deadline = Clock::now() + std::chrono::duration<double>(timeout_s);
  while (r->status < QSV_REQ_COMPLETED) {
    if (sv->cv_done.wait_until(lk, deadline) == std::cv_status::timeout && r->status < QSV_REQ_COMPLETED) {
      fill_info(r, info);
      return fail(QSV_E_STATE, "request not complete before the timeout");
    }
  }
  fill_info(r, info);
  if (outcomes && r->status == QSV_REQ_COMPLETED) std::memcpy(outcomes, r->outcomes.data(), r->shots * sizeof(uint64_t));
  sv->reqs.erase(it);
  delete r;
  return QSV_OK;
}

int qsv_server_cancel(qsv_server* sv, uint64_t request_id, int* outcome)
{
  if (!sv || !outcome) return fail(QSV_E_INVALID, "null argument");
  {
    std::lock_guard<std::mutex> lk(sv->mu);
    auto it = sv->reqs.find(request_id);
    if (it == sv->reqs.end()) return fail(QSV_E_NOTFOUND, "unknown request id");
    SrvReq* r = it->second;
    if (r->status >= QSV_REQ_COMPLETED) {
      *outcome = QSV_CANCEL_CANNOT;
      return QSV_OK;
    }
    *outcome = QSV_CANCEL_DONE;
    if (r->status == QSV_REQ_QUEUED) {
      // never admitted: it holds no device memory and leaves the queue now
      auto q = std::find(sv->queue.begin(), sv->queue.end(), r);
      if (q != sv->queue.end()) sv->queue.erase(q);
      if (r->raw) --sv->raw;
      r->raw = false;
      r->t_admit = r->t_done = Clock::now();
      r->status = QSV_REQ_CANCELLED;
      sv->stats.cancelled++;
    } else {
      // admitted: its launches are on the device; it finishes as cancelled
      r->cancel = true;
      return QSV_OK;
    }
  }
  sv->cv_done.notify_all();
  return QSV_OK;
}

int qsv_server_stats_read(qsv_server* sv, qsv_server_stats* out)
{
  if (!sv || !out) return fail(QSV_E_INVALID, "null argument");
  std::lock_guard<std::mutex> lk(sv->mu);
  *out = sv->stats;
  out->queued_now = sv->queue.size();
  out->inflight_now = (uint64_t)sv->inflight();
  out->hbm_in_use_bytes = sv->in_use;
  out->hbm_budget_bytes = sv->budget;
  return QSV_OK;
}

int qsv_server_destroy(qsv_server* sv)
{
  if (!sv) return QSV_OK;
  {
    std::lock_guard<std::mutex> lk(sv->mu);
    sv->stop = true;
  }
  sv->cv_work.notify_all();
  if (sv->th.joinable()) sv->th.join();
  for (auto& kv : sv->reqs) delete kv.second;
  for (auto& fl : sv->free_states)
    for (qsv_state* s : fl) qsv_state_destroy(s);
  for (auto& s : sv->slots) {
    if (s.stream) hipStreamSynchronize(s.stream);
    hipFree(s.arena);
    hipFree(s.progs);
    hipFree(s.insts);
    hipFree(s.jobs);
    hipFree(s.d_out);
    if (s.h_out) hipHostFree(s.h_out);
    if (s.ev) hipEventDestroy(s.ev);
    if (s.stream) hipStreamDestroy(s.stream);
  }
  delete sv;
  return QSV_OK;
}

int qsv_timing_enable(qsv_state* s, int enable)
{
  int rc = check_state(s);
  if (rc) return rc;
  if (!enable) {
    rc = flush_timing(s);
    if (rc) return rc;
  }
  s->timing = enable != 0;
  return QSV_OK;
}

int qsv_timing_read(qsv_state* s, qsv_kernel_stat out[QSV_KCLASS_COUNT], int reset)
{
  int rc = check_state(s);
  if (rc) return rc;
  rc = flush_timing(s);
  if (rc) return rc;
  if (out) std::memcpy(out, s->stats, sizeof(s->stats));
  if (reset) std::memset(s->stats, 0, sizeof(s->stats));
  return QSV_OK;
}

int qsv_tune_fused(int precision, int num_qubits, qsv_tune_result* out)
{
  if (!out) return fail(QSV_E_INVALID, "null output");
  if (precision != QSV_C128 && precision != QSV_C64) return fail(QSV_E_INVALID, "unknown precision");
  const int n = num_qubits ? num_qubits : 26;
  if (n < 16 || n > 30) return fail(QSV_E_INVALID, "tuning state must have 16..30 qubits");
  std::memset(out, 0, sizeof(*out));
  qsv_state* s = nullptr;
  int rc = qsv_state_create(n, precision, &s);
  if (rc) return rc;
  // the timed program: kTuneLayers layers of one gate per bit drawn from H,
  // RX, RY and RZ (the random-layer workloads' mix), then CNOTs on a fixed
  // pseudo-random matching per layer
  constexpr int kTuneLayers = 8;
  std::vector<BGate> layer;
  const double xm[8] = {0, 0, 1, 0, 1, 0, 0, 0};
  const int kinds[4] = {QSV_OP_H, QSV_OP_RX, QSV_OP_RY, QSV_OP_RZ};
  std::vector<int> perm(n);
  uint64_t x = 0x2545F4914F6CDD1Dull;
  auto next = [&x]() {
    x ^= x << 13; x ^= x >> 7; x ^= x << 17;
    return x;
  };
  for (int l = 0; l < kTuneLayers; ++l) {
    for (int b = 0; b < n; ++b) {
      const uint64_t r = next();
      double gm[8];
      gate_matrix(kinds[r & 3], 0.1 + 6.0 * (double)((r >> 8) & 1023) / 1024.0, gm);
      emit_ctl(layer, {}, b, gm);
    }
    for (int b = 0; b < n; ++b) perm[b] = b;
    for (int b = n - 1; b > 0; --b) std::swap(perm[b], perm[(int)(next() % (uint64_t)(b + 1))]);
    for (int k = 0; k + 1 < n; k += 2) emit_ctl(layer, {perm[k]}, perm[k + 1], xm);
  }
  // each candidate's time: the device time of its kernels (per-launch events),
  // not the host's fusion and compilation before them
  const int TB = kPassTileBits;
  const int lo = low_bit_threshold(s), hi = std::min(TB - 4, lo + QSV_TUNE_MAX - 1);
  double best = 1e300;
  int bestL = 4;
  s->timing = true;
  for (int L = lo; L <= hi && !rc; ++L) {
    s->tile_low = L;
    double t = 1e300;
    for (int rep = 0; rep < 3 && !rc; ++rep) {   // the first run is a warm-up
      std::memset(s->stats, 0, sizeof(s->stats));
      if ((rc = run_fused(s, layer, 0)) || (rc = flush_timing(s))) break;
      double ms = 0.0;
      for (const auto& st : s->stats) ms += st.total_ms;
      if (rep) t = std::min(t, ms / kTuneLayers);
    }
    if (rc) break;
    out->candidate[out->n_candidates] = L;
    out->ms[out->n_candidates++] = t;
    best = std::min(best, t);
  }
  // the narrowest width within 1 % of the fastest: a narrower run leaves more
  // tile bits for gates, which longer programs turn into fewer passes
  for (int i = out->n_candidates - 1; i >= 0; --i)
    if (out->ms[i] <= 1.01 * best) bestL = out->candidate[i];
  const int drc = qsv_state_destroy(s);
  if (rc) return rc;
  if (drc) return drc;
  out->low_bits = bestL;
  g_tuned_low[precision == QSV_C128 ? 0 : 1].store(bestL);
  return QSV_OK;
}

}  // extern "C"
