// qsv_compile.hip — fused passes compiled into the micro-op programs of k_pass
// (host code).
//
// Only dense 2x2s need their target among the four register bits of the layout
// they run in. The rest costs little or nothing:
//   * CNOTs and swaps permute the tile's indices linearly over GF(2), and so
//     does a layout: they are applied to the columns of the current layout and
//     take effect in the addresses of the next round trip through LDS (or of
//     the store). On 30-qubit random layers they were 40 % of a pass's ops, 105
//     vector instructions each on complex128.
//   * Diagonal gates become factors of the amplitudes whose bits are all set,
//     kept with their bit mask and multiplied together until a dense gate, a
//     CNOT target or the end of the pass needs them applied: thread bits cost
//     one complex product per lane and factor, not one per amplitude. Factors
//     common to the whole state are collected over a run of passes.
//   * Bits outside the tile are constants in it: controls and phases on them
//     are conditions on the tile's base, a CNOT controlled by one is a shift of
//     the tile's indices, so only dense targets and swapped bits have to be
//     tile bits at all.
// A unitary without structure stays one op of four complex products a pair. Taken
// apart into diagonal * real * diagonal it needs half of them, but three ops and
// rounded phases that are alike for every amplitude: 60 layers of such gates on 10
// qubits were off by 5.5e-15 instead of 1.8e-15, and 12-qubit random layers took
// 240 us instead of 219 (only dense layers of nothing else on states in HBM gained:
// 24 qubits 936 us instead of 970).
// Gates are taken from per-bit queues: everything that can run in the current
// layout runs, then the next layout takes the register bits of the dense gates
// that wait.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "qsv_internal.h"

namespace qsv {

namespace {

using C = std::complex<double>;

inline uint32_t pass_swz(uint32_t l) { return l ^ (((l >> 4) ^ (l >> 8)) & 15u); }

// A PO_BLOCK costs a wave 48 v_mfma_f32_16x16x4f32 (three real 16 x 16 x 16
// products per column block of 16 lanes: 0.66 ms per 2^30 amplitudes at the
// FP32 matrix peak) plus an LDS round trip, whatever it absorbs, so it pays
// only for long runs of expensive ops: vector instructions per wave of each
// register-bit op in an FP32 pass.
int reg_op_cost(const POp& op)
{
  if (op.code < PO_DENSE_K) {
    const int dm = op.code & 3;
    return dm == PM_GENERAL ? 147 : dm == PM_EXCHANGE ? 40 : 83;
  }
  if (op.code < PO_PHASE) return 147;
  if (op.code < PO_BLOCKADE) return op.code == PO_PHASE && op.kc ? 60 : 101;
  return 101;   // PO_BLOCKADE
}

// Slot bits an op of a stage reads or writes; `reg_only`: it has no
// thread-bit part, so it is the same 16 x 16 map on every thread's slots.
uint32_t op_slot_bits(const POp& op, bool* reg_only)
{
  if (op.code < PO_DENSE_K) {
    *reg_only = op.tmask == 0 && op.gm == 0;
    return 1u << (op.code >> 2);
  }
  if (op.code < PO_PHASE) {
    *reg_only = op.tmask == 0 && op.gm == 0;
    return (1u << (op.code - PO_DENSE_K)) | op.kc;
  }
  *reg_only = op.code < PO_BLOCKADE ? op.cnt == 0 : op.code == PO_BLOCKADE && op.aux == 0;
  return op.kc | (op.code > PO_PHASE && op.code < PO_BLOCKADE ? 1u << (op.code - PO_PHASE2) : 0u);
}

// v = (map of a register-bit op) v on one thread's 16 slots, as k_pass applies it.
void apply_reg_op(const POp& op, C v[16])
{
  const uint32_t kc = op.kc;
  if (op.code < PO_PHASE) {
    const int rb = op.code < PO_DENSE_K ? op.code >> 2 : op.code - PO_DENSE_K;
    const int d = 1 << rb;
    const C m00(op.m[0], op.m[1]), m01(op.m[2], op.m[3]), m10(op.m[4], op.m[5]), m11(op.m[6], op.m[7]);
    for (int k = 0; k < 16; ++k) {
      if ((k & d) || ((uint32_t)k & kc) != kc) continue;
      const C a = v[k], b = v[k | d];
      v[k] = m00 * a + m01 * b;
      v[k | d] = m10 * a + m11 * b;
    }
  } else if (op.code == PO_PHASE) {
    for (int k = 0; k < 16; ++k)
      if (((uint32_t)k & kc) == kc) v[k] *= C(op.m[0], op.m[1]);
  } else if (op.code < PO_BLOCKADE) {
    const int rb = op.code - PO_PHASE2;
    for (int k = 0; k < 16; ++k)
      if (((uint32_t)k & kc) == kc) v[k] *= (k >> rb) & 1 ? C(op.m[6], op.m[7]) : C(op.m[0], op.m[1]);
  } else {   // PO_BLOCKADE without a thread part
    for (int k = 0; k < 16; ++k)
      if (__builtin_popcount((uint32_t)k & kc) == 1) v[k] *= C(op.m[0], op.m[1]);
  }
}

// Diagonal factors not applied yet: where the tile bits `mask` and the bits
// `gmask` outside it are set, `on` and `off` by the value of tile bit t or
// outside bit gt (neither: `on`)
struct Factor {
  uint32_t mask;
  uint64_t gmask;
  int t;
  uint64_t gt;
  C on, off;
  uint32_t bits() const { return mask | (t >= 0 ? 1u << t : 0u); }
};
struct Keyed {
  int key;
  Factor f;
};
struct GateInfo {
  uint32_t bits;   // tile bits it acts on
  int8_t cls;      // PHASE, LINEAR or OTHER
  int8_t waits;    // its bits' queues that it is not the front of
};

// A thread's working memory, kept from pass to pass (up to kKeepOps ops): a
// program of a hundred gates spends as long in malloc as on its gates otherwise.
struct Scratch {
  static constexpr size_t kKeepOps = 1 << 14;
  std::vector<POp> ops;
  std::vector<PTerm> terms;
  std::vector<PShift> shifts;
  std::vector<float> blk;
  std::vector<Factor> pend;
  std::vector<Keyed> now;
  std::vector<GateInfo> info;
  std::vector<int> queue;
  void clear()
  {
    if (ops.capacity() > kKeepOps || queue.capacity() > 4 * kKeepOps) *this = Scratch{};
    ops.clear();
    terms.clear();
    shifts.clear();
    blk.clear();
    pend.clear();
  }
};

struct Compiler {
  // wave-index bits as functionals of the logical index, and the global bits
  // whose value in the tile's base flips them
  struct Waves {
    uint32_t r[4] = {};
    uint64_t o[4] = {};
  };
  const FPass& p;
  const bool f32;
  const int block_cost;
  const int TB, NT;        // tile bits, thread bits
  const uint32_t FULL;
  Scratch& mem;
  std::vector<POp>& ops = mem.ops;
  std::vector<PTerm>& terms = mem.terms;
  std::vector<PShift>& shifts = mem.shifts;
  std::vector<float>& blk = mem.blk;
  int nblk = 0;
  size_t stage0 = 0;       // first op of the current stage
  uint16_t stage_col[kCols] = {};
  Waves stage_wr;

  // current layout: logical index columns of thread bits and slots, and the
  // clean layout they started from
  uint32_t ct[kColT] = {}, cr[4] = {};
  uint32_t reg = 0;
  Waves wr;
  // shifts of the layout: global bit outside the tile -> local index
  std::vector<std::pair<int, uint32_t>> co;
  uint32_t row_dirty = 0;  // bits whose value is not one physical bit's
  uint32_t col_dirty = 0;  // bits whose flip is not one physical bit's
  uint16_t last_to[kCols] = {};
  bool have_last = false;
  Waves own;               // after the last LDS round trip
  bool have_own = false;
  Waves load_wr;
  size_t last_site = SIZE_MAX;       // the last PO_KRAUS op,
  double least = 1.0, most = 1.0;    // and the range of the norm since the last renormalisation
  bool synced = false;     // every wave's tile has crossed a workgroup barrier

  std::vector<Factor>& pend = mem.pend;
  std::vector<Keyed>& now = mem.now;   // flush's own
  C& scalar;

  Compiler(const FPass& p_, bool f32_, int bc, C& sc, Scratch& m)
      : p(p_), f32(f32_), block_cost(bc), TB(p_.tb), NT(p_.tb - 4), FULL((1u << p_.tb) - 1u), mem(m), scalar(sc)
  {
  }

  uint32_t rank_in(uint32_t mask, int b) const { return __builtin_popcount(mask & ((1u << b) - 1u)); }
  uint32_t slot_mask(uint32_t local) const
  {
    uint32_t m = 0;
    for (uint32_t l = local & reg; l; l &= l - 1) m |= 1u << rank_in(reg, __builtin_ctz(l));
    return m;
  }
  uint32_t tid_mask(uint32_t local) const
  {
    const uint32_t nonreg = FULL & ~reg;
    uint32_t m = 0;
    for (uint32_t l = local & nonreg; l; l &= l - 1) m |= 1u << rank_in(nonreg, __builtin_ctz(l));
    return m;
  }
  POp& emit(int code)
  {
    ops.emplace_back();   // zeros
    POp& op = ops.back();
    op.code = code;
    return op;
  }

  void set_clean(uint32_t r)
  {
    reg = r;
    row_dirty = col_dirty = 0;
    int j = 0, i = 0;
    for (int b = 0; b < TB; ++b) {
      if ((r >> b) & 1u) cr[i++] = 1u << b;
      else ct[j++] = 1u << b;
    }
    wr = Waves{};
    for (int k = 0; k + 6 < NT; ++k) wr.r[k] = ct[6 + k];
    co.clear();
  }
  void lds_columns(uint16_t col[kCols]) const
  {
    std::memset(col, 0, kCols * sizeof(uint16_t));
    for (int j = 0; j < NT; ++j) col[j] = (uint16_t)pass_swz(ct[j]);
    for (int i = 0; i < 4; ++i) col[kColT + i] = (uint16_t)pass_swz(cr[i]);
  }
  void begin_stage()
  {
    stage0 = ops.size();
    lds_columns(stage_col);
    stage_wr = wr;
  }
  bool same_waves(const Waves& a, const Waves& b) const
  {
    for (int k = 0; k + 6 < NT; ++k)
      if (a.r[k] != b.r[k] || a.o[k] != b.o[k]) return false;
    return true;
  }
  void relayout(uint32_t r)
  {
    if (block_cost > 0) form_blocks();
    POp& op = emit(PO_RELAYOUT);
    lds_columns(op.col);
    const Waves from = wr;
    if (have_last && co.empty() && !std::memcmp(last_to, op.col, sizeof(last_to))) op.flag |= PR_SAME;
    op.aux = (uint32_t)shifts.size();   // index now, byte offset when the program is laid out
    for (const auto& c : co)
      if (c.second) shifts.push_back(PShift{(uint32_t)c.first, pass_swz(c.second), 0});
    op.cnt = (int32_t)(shifts.size() - op.aux);
    if (have_own && !same_waves(own, from)) op.flag |= PR_WAIT;
    set_clean(r);
    lds_columns(op.col + kCols);
    std::memcpy(last_to, op.col + kCols, sizeof(last_to));
    have_last = true;
    if (same_waves(from, wr)) op.flag |= PR_LOCAL;
    else synced = true;
    own = wr;
    have_own = true;
    begin_stage();
  }

  // ---- diagonal factors -----------------------------------------------------
  void add_term(uint32_t mask, uint64_t gmask, C f)
  {
    if (f == C(1.0, 0.0)) return;
    if (mask == 0 && gmask == 0) {
      scalar *= f;
      return;
    }
    add_two(mask, gmask, -1, 0, f, f);
  }
  void add_two(uint32_t mask, uint64_t gmask, int t, uint64_t gt, C on, C off)
  {
    for (auto& f : pend)
      if (f.mask == mask && f.gmask == gmask && f.t == t && f.gt == gt) {
        f.on *= on;
        f.off *= off;
        return;
      }
    pend.push_back(Factor{mask, gmask, t, gt, on, off});
  }
  // Can every pending factor with one of the bits `touch` be applied here?
  bool can_flush(uint32_t touch) const
  {
    for (const auto& f : pend)
      if ((f.bits() & touch) && (f.bits() & row_dirty)) return false;
    return true;
  }
  // Applies the pending factors with one of the bits `touch`, one op per set of
  // slot bits; `with`: a factor of every amplitude joins the group without slot bits.
  void flush(uint32_t touch, C with = C(1.0, 0.0), bool all = false)
  {
    bool any = all || with != C(1.0, 0.0);
    for (size_t i = 0; i < pend.size() && !any; ++i) any = (pend[i].bits() & touch) != 0;
    if (!any) return;
    // the factors to apply, each with its group: slot mask and, for a target on
    // a slot, its register bit
    now.clear();
    size_t w = 0;
    if (with != C(1.0, 0.0)) now.push_back({0, Factor{0, 0, -1, 0, with, with}});
    for (size_t i = 0; i < pend.size(); ++i) {
      if (!all && !(pend[i].bits() & touch)) {
        if (w != i) pend[w] = pend[i];
        ++w;
        continue;
      }
      const Factor& f = pend[i];
      const bool on_slot = f.t >= 0 && ((reg >> f.t) & 1u);
      now.push_back({(int)slot_mask(f.mask) | (on_slot ? (int)(rank_in(reg, f.t) + 1) << 4 : 0), f});
    }
    pend.resize(w);
    for (size_t i = 0; i < now.size(); ++i) {
      const int key = now[i].key;
      if (key < 0) continue;
      const uint32_t kc = (uint32_t)key & 15u;
      const int rb = (key >> 4) - 1;
      C on(1.0, 0.0), off(1.0, 0.0);
      const size_t first_term = terms.size();
      for (size_t j = i; j < now.size(); ++j) {
        if (now[j].key != key) continue;
        now[j].key = -1;
        const Factor& f = now[j].f;
        const uint32_t tm = tid_mask(f.mask), tb = f.t >= 0 && rb < 0 ? tid_mask(1u << f.t) : 0u;
        if (!tm && !tb && !f.gmask && !f.gt) {
          on *= f.on;
          off *= f.off;
          continue;
        }
        PTerm q;
        std::memset(&q, 0, sizeof(q));
        q.tmask = tm;
        q.tbit = tb;
        q.gmask = f.gmask;
        q.gbit = f.gt;
        if (f32) {
          q.f[0] = (float)f.on.real();
          q.f[1] = (float)f.on.imag();
          q.f[2] = (float)f.off.real();
          q.f[3] = (float)f.off.imag();
        } else {
          q.d[0] = f.on.real();
          q.d[1] = f.on.imag();
        }
        terms.push_back(q);
      }
      const int cnt = (int)(terms.size() - first_term);
      if (!cnt && on == C(1.0, 0.0) && (rb < 0 || off == on)) continue;
      POp& op = emit(rb < 0 ? PO_PHASE : PO_PHASE2 + rb);
      const C lead = rb < 0 ? on : off;
      op.kc = kc;
      op.m[0] = lead.real();
      op.m[1] = lead.imag();
      op.m[6] = on.real();
      op.m[7] = on.imag();
      op.aux = (uint32_t)first_term;   // index now, byte offset when the program is laid out
      op.cnt = cnt;
    }
  }

  // ---- matrix-core blocks -----------------------------------------------------
  // Fold the register-bit ops of the stage just ended into dense 16 x 16
  // blocks. Scanning in order, an op without a thread-bit part joins the open
  // block if its slot bits miss those of every op set aside since the block
  // opened; an op with a thread-bit part is set aside and runs after the block
  // (ops on disjoint bits commute). A block whose ops cost the vector units
  // less than block_cost keeps its ops in program order.
  void form_blocks()
  {
    const std::vector<POp> src(ops.begin() + stage0, ops.end());
    ops.resize(stage0);
    std::vector<int> in, aside;
    uint32_t aside_bits = 0;
    int cost = 0;
    auto close = [&]() {
      if (cost >= block_cost && nblk < kMaxPassBlocks) {
        C U[16][16];
        for (int col = 0; col < 16; ++col) {
          C v[16];
          for (int k = 0; k < 16; ++k) v[k] = k == col ? 1.0 : 0.0;
          for (int i : in) apply_reg_op(src[i], v);
          for (int k = 0; k < 16; ++k) U[k][col] = v[k];
        }
        for (int kk = 0; kk < 4; ++kk)
          for (int l = 0; l < 64; ++l) {
            const C u = U[l & 15][4 * kk + (l >> 4)];
            blk.push_back((float)u.real());
            blk.push_back((float)u.imag());
          }
        POp& b = emit(PO_BLOCK);
        b.aux = (uint32_t)nblk++;   // index now, byte offset when the program is laid out
        std::memcpy(b.col, stage_col, sizeof(stage_col));
        own = stage_wr;
        have_own = true;
        for (int i : aside) ops.push_back(src[i]);
      } else {
        std::vector<int> all(in);
        all.insert(all.end(), aside.begin(), aside.end());
        std::sort(all.begin(), all.end());
        for (int i : all) ops.push_back(src[i]);
      }
      in.clear();
      aside.clear();
      aside_bits = 0;
      cost = 0;
    };
    for (int i = 0; i < (int)src.size(); ++i) {
      if (src[i].code == PO_SWAP) {
        close();
        ops.push_back(src[i]);
        continue;
      }
      bool reg_only = false;
      const uint32_t sb = op_slot_bits(src[i], &reg_only);
      if (reg_only) {
        if (sb & aside_bits) close();
        in.push_back(i);
        cost += reg_op_cost(src[i]);
      } else {
        aside.push_back(i);
        aside_bits |= sb;
      }
    }
    close();
  }

  // ---- gates --------------------------------------------------------------------
  // a phase, which can be divided out and applied later without moving the norm
  static bool usable(C d) { return is_phase(d.real(), d.imag()); }
  static C over(C a, C b) { return a * std::conj(b) / std::norm(b); }
  static uint32_t gate_bits(const FGate& g)
  {
    if (g.kind == FG_KRAUS) return 1u << g.a;
    uint32_t m = g.cmask | (g.kind == FG_BLOCKADE ? g.bmask : 0u);
    if (g.a >= 0) m |= 1u << g.a;
    if (g.b >= 0) m |= 1u << g.b;
    return m;
  }
  // CNOTs and plain (phased) swaps
  static bool is_linear(const FGate& g)
  {
    if (g.kind == FG_DENSE)
      return g.sub == DM_EXCHANGE && __builtin_popcount(g.cmask) + __builtin_popcountll(g.gmask) == 1;
    return g.kind == FG_SWAP && g.cmask == 0 && g.gmask == 0 && usable(C(g.m[0], g.m[1]));
  }
  // A diagonal gate as factors on bit masks (its first entry is 1 or a phase).
  void take_phase(const FGate& g)
  {
    const C d0(g.m[0], g.m[1]), d1(g.m[6], g.m[7]);
    const uint32_t t = g.a >= 0 ? 1u << g.a : 0u;
    if (g.sub) {   // d0 == 1
      add_term(g.cmask | t, g.gmask | g.gt, d1);
      return;
    }
    // FP32 passes keep both entries: rounded alike (a Z rotation's are
    // conjugates) they leave the weights of the two halves as they are, where
    // one rounded factor on one half moves them against each other
    if (f32) {
      add_two(g.cmask, g.gmask, g.a, g.gt, d1, d0);
      return;
    }
    add_term(g.cmask, g.gmask, d0);
    add_term(g.cmask | t, g.gmask | g.gt, over(d1, d0));
  }

  bool run_linear(const FGate& g)
  {
    if (g.kind == FG_SWAP) {
      const int a = g.a, b = g.b;
      auto sw = [&](uint32_t m) {
        const uint32_t x = ((m >> a) ^ (m >> b)) & 1u;
        return m ^ (x << a) ^ (x << b);
      };
      for (auto& f : pend) {
        f.mask = sw(f.mask);
        if (f.t == a || f.t == b) f.t = a + b - f.t;
      }
      for (int j = 0; j < NT; ++j) ct[j] = sw(ct[j]);
      for (auto& c : cr) c = sw(c);
      for (auto& w : wr.r) w = sw(w);
      for (auto& c : co) c.second = sw(c.second);
      const uint32_t ab = (1u << a) | (1u << b);
      row_dirty |= ab;
      col_dirty |= ab;
      const C ph(g.m[0], g.m[1]);
      if (ph != C(1.0, 0.0)) {
        add_term(1u << a, 0, ph);
        add_term(1u << b, 0, ph);
        add_term(ab, 0, 1.0 / (ph * ph));
      }
      return true;
    }
    const uint32_t t = 1u << g.a, c = g.cmask;
    if (!can_flush(t)) return false;
    flush(t);
    if (g.gmask) {   // the control outside the tile: a shift
      const int b = __builtin_ctzll(g.gmask);
      bool found = false;
      for (auto& x : co)
        if (x.first == b) {
          x.second ^= t;
          found = true;
        }
      if (!found) co.emplace_back(b, t);
      for (int k = 0; k < 4; ++k)
        if (wr.r[k] & t) wr.o[k] ^= g.gmask;
      row_dirty |= t;
      return true;
    }
    for (int j = 0; j < NT; ++j)
      if (ct[j] & c) ct[j] ^= t;
    for (auto& x : cr)
      if (x & c) x ^= t;
    for (auto& x : co)
      if (x.second & c) x.second ^= t;
    for (auto& w : wr.r)
      if (w & t) w ^= c;
    row_dirty |= t;
    col_dirty |= t | c;
    return true;
  }

  // Runs a gate that is neither diagonal nor linear if the layout allows it.
  bool run_gate(const FGate& g)
  {
    if (g.kind == FG_BLOCKADE) {
      if (g.bmask & row_dirty) return false;
      POp& op = emit(PO_BLOCKADE);
      op.kc = slot_mask(g.bmask);
      op.aux = tid_mask(g.bmask);
      op.m[0] = g.m[0];
      op.m[1] = g.m[1];
      return true;
    }
    if (g.kind == FG_SWAP) {
      if (row_dirty | col_dirty) return false;
      const uint32_t ab = (1u << g.a) | (1u << g.b);
      flush(ab);
      POp& op = emit(PO_SWAP);
      op.kc = (uint32_t)g.a;
      op.aux = (uint32_t)g.b;
      op.tmask = g.cmask;
      op.sc[0] = g.m[0];
      op.sc[1] = g.m[1];
      lds_columns(op.col);
      own = wr;
      have_own = true;
      synced = true;
      return true;
    }
    const uint32_t t = 1u << g.a;
    if (!(reg & t) || ((row_dirty | col_dirty) & t) || !can_flush(t)) return false;
    const int rb = (int)rank_in(reg, g.a);
    if (g.kind == FG_KRAUS) {
      flush(t);
      // A renormalisation after the site before this one, or after this one, where
      // the norm could otherwise be out of range; far from the 1e-12 below which a
      // renormalisation leaves a state alone. An operator that could take the norm
      // there by itself (a projector) has one on either side.
      constexpr double kLeastNorm = 1e-8, kMostNorm = 1e8;
      if (last_site != SIZE_MAX && ((!(least * g.m[0] >= kLeastNorm) && least < 0.5) || !(most * g.m[1] <= kMostNorm))) {
        ops[last_site].flag = 1;
        least = most = 1.0;
      }
      POp& op = emit(PO_KRAUS + rb);
      op.kc = (uint32_t)g.b;
      op.aux = g.cmask;
      op.cnt = g.sub;
      least *= g.m[0];
      most *= g.m[1];
      op.flag = g.bmask || !(least >= kLeastNorm) ? 1 : 0;
      if (op.flag) least = most = 1.0;
      last_site = ops.size() - 1;
      return true;
    }
    if (g.cmask & row_dirty) return false;
    const int sub = g.kind == FG_DENSE ? g.sub : DM_GENERAL;
    flush(t);
    const uint32_t kc = slot_mask(g.cmask);
    POp& op = emit(kc ? PO_DENSE_K + rb : PO_DENSE + 4 * rb + sub);
    op.kc = kc;
    op.tmask = tid_mask(g.cmask);
    op.gm = g.gmask;
    std::memcpy(op.m, g.m, sizeof(g.m));
    if (g.kind == FG_PHASE) op.m[2] = op.m[3] = op.m[4] = op.m[5] = 0.0;
    return true;
  }

  // Fill a register mask to four bits: bits above the low run, highest first
  // (consecutive layouts then tend to share them) without the two that name
  // the wave, then those two, then low bits.
  uint32_t fill(uint32_t r) const
  {
    const int L = p.low;
    for (int b = TB - 3; b >= L && __builtin_popcount(r) < 4; --b) r |= 1u << b;
    for (int b = TB - 1; b >= std::max(0, TB - 2) && __builtin_popcount(r) < 4; --b) r |= 1u << b;
    for (int b = 0; b < TB && __builtin_popcount(r) < 4; ++b) r |= 1u << b;
    return r;
  }
  bool coalesced() const
  {
    for (int j = 0; j < p.low; ++j)
      if (ct[j] >> p.low) return false;
    return true;
  }
  void global_columns(uint64_t out[kCols]) const
  {
    auto g = [&](uint32_t l) {
      uint64_t v = 0;
      for (; l; l &= l - 1) v |= 1ull << p.pos[__builtin_ctz(l)];
      return v;
    };
    for (int j = 0; j < kColT; ++j) out[j] = j < NT ? g(ct[j]) : 0;
    for (int i = 0; i < 4; ++i) out[kColT + i] = g(cr[i]);
  }

  void run(PHead& h, bool last)
  {
    const int N = (int)p.gates.size();
    // Per-bit queues of the gates in program order. A gate is ready when it is
    // the front of all its bits' queues; `ready` holds, per class of gates, the
    // lowest bits of the ready ones.
    enum { PHASE, LINEAR, OTHER };
    std::vector<GateInfo>& info = mem.info;
    info.resize(N);
    uint32_t ready[3] = {};
    int left = N;
    ops.reserve(2 * N + 16);
    size_t head[16] = {}, end[16] = {};   // of the queues, back to back in `queue`
    auto at_front = [&](int i) {
      GateInfo& f = info[i];
      if (--f.waits == 0) ready[f.cls] |= f.bits & -f.bits;
    };
    for (int i = 0; i < N; ++i) {
      const FGate& g = p.gates[i];
      GateInfo& f = info[i];
      f.bits = gate_bits(g);
      f.cls = (int8_t)(g.kind == FG_PHASE && (g.sub || usable(C(g.m[0], g.m[1]))) ? PHASE
                       : is_linear(g)                                             ? LINEAR
                                                                                  : OTHER);
      if (!f.bits) {   // a phase on bits outside the tile: one factor per tile
        take_phase(g);
        --left;
        continue;
      }
      f.waits = (int8_t)__builtin_popcount(f.bits);
      for (uint32_t m = f.bits; m; m &= m - 1) ++end[__builtin_ctz(m)];
    }
    size_t total = 0;
    for (int b = 0; b < TB; ++b) {
      head[b] = total;
      total += end[b];
      end[b] = head[b];
    }
    std::vector<int>& queue = mem.queue;
    queue.resize(total);
    for (int i = 0; i < N; ++i)
      for (uint32_t m = info[i].bits; m; m &= m - 1) queue[end[__builtin_ctz(m)]++] = i;
    for (int b = 0; b < TB; ++b)
      if (head[b] < end[b]) at_front(queue[head[b]]);
    auto consume = [&](int i) {
      const GateInfo& f = info[i];
      --left;
      ready[f.cls] &= ~(f.bits & -f.bits);
      for (uint32_t m = f.bits; m; m &= m - 1) {
        const int b = __builtin_ctz(m);
        if (++head[b] < end[b]) at_front(queue[head[b]]);
      }
    };
    auto ready_gate = [&](uint32_t m) { return queue[head[__builtin_ctz(m)]]; };
    // the next layout: the targets of waiting dense gates. `first`: the load
    // layout, whose lanes must cover the low run; later ones take low bits as
    // soon as they are wanted, so that the last layout can store.
    auto next_regs = [&](bool first) {
      int want[16], n = 0;   // gates, those on low bits before the others
      for (uint32_t m = ready[OTHER]; m; m &= m - 1) {
        const int i = ready_gate(m);
        const FGate& g = p.gates[i];
        if (g.kind == FG_SWAP || g.kind == FG_BLOCKADE || (first && g.a < p.low)) continue;
        want[n++] = g.a < p.low ? i - N : i;
      }
      std::sort(want, want + n);
      uint32_t r = 0;
      for (int k = 0; k < n && k < 4; ++k) r |= 1u << p.gates[want[k] < 0 ? want[k] + N : want[k]].a;
      return r;
    };
    // gates that wait for nothing: diagonal ones leave the queues at once
    auto drain_phases = [&]() {
      const bool any = ready[PHASE] != 0;
      while (ready[PHASE]) {
        const int i = ready_gate(ready[PHASE]);
        take_phase(p.gates[i]);
        consume(i);
      }
      return any;
    };
    drain_phases();
    set_clean(fill(next_regs(true)));
    if (!coalesced()) set_clean(fill(0));
    global_columns(h.gload);
    load_wr = wr;
    begin_stage();
    while (left) {
      bool any = true, moved = false;
      while (any) {   // everything this layout can run
        any = drain_phases();
        for (uint32_t m = ready[OTHER]; m; m &= m - 1) {
          const int i = ready_gate(m);
          if (!run_gate(p.gates[i])) continue;
          consume(i);
          any = true;
        }
        moved |= any;
      }
      for (uint32_t m = ready[LINEAR]; m; m &= m - 1) {
        const int i = ready_gate(m);
        if (!run_linear(p.gates[i])) continue;
        consume(i);
        moved = true;
      }
      if (moved || !left) continue;
      relayout(fill(next_regs(false)));
    }
    C g(1.0, 0.0);
    if (last) {
      g = scalar;
      scalar = C(1.0, 0.0);
    }
    if (!can_flush(FULL)) relayout(fill(0));
    flush(FULL, g, true);
    if (!coalesced()) relayout(fill(0));
    else if (block_cost > 0) form_blocks();
    global_columns(h.gstore);
    h.shift_off = (int32_t)shifts.size();   // index now, byte offset when the program is laid out
    for (const auto& c : co)
      if (c.second) {
        uint64_t v = 0;
        for (uint32_t l = c.second; l; l &= l - 1) v |= 1ull << p.pos[__builtin_ctz(l)];
        shifts.push_back(PShift{(uint32_t)c.first, 0, v});
      }
    h.nshift = (int32_t)shifts.size() - h.shift_off;
    // the tile is updated in place: a wave may overwrite amplitudes that another
    // one has not loaded yet when the layouts name the waves differently
    h.store_wait = !synced && !same_waves(load_wr, wr) ? 1 : 0;
  }
};

}  // namespace

size_t compile_pass(const FPass& p, bool f32, int block_cost, std::complex<double>& scalar, bool last,
                    std::vector<char>& out)
{
  PHead h;
  std::memset(&h, 0, sizeof(h));
  // entries of magnitude at most 1 keep every product of a pass finite, in FP32 too
  bool tame = std::abs(scalar.real()) <= 1.001 && std::abs(scalar.imag()) <= 1.001;
  for (const FGate& g : p.gates)
    for (double m : g.m) tame &= std::abs(m) <= 1.001;
  h.renorm = p.renorm | (tame ? FP_KEEP_ZERO : 0);
  std::memcpy(h.sorted_pos, p.sorted_pos, sizeof(h.sorted_pos));
  thread_local Scratch mem;
  mem.clear();
  Compiler c(p, f32, block_cost, scalar, mem);
  c.run(h, last);
  h.nops = (int32_t)c.ops.size();
  const size_t terms_at = (sizeof(PHead) + (c.ops.size() + 1) * sizeof(POp) + 31) & ~(size_t)31;
  const size_t shifts_at = terms_at + c.terms.size() * sizeof(PTerm);
  const size_t blk_at = shifts_at + c.shifts.size() * sizeof(PShift);
  h.shift_off = (int32_t)(shifts_at + h.shift_off * sizeof(PShift));
  for (POp& op : c.ops) {
    if (op.code >= PO_PHASE && op.code < PO_BLOCKADE) op.aux = (uint32_t)(terms_at + op.aux * sizeof(PTerm));
    else if (op.code == PO_RELAYOUT) op.aux = (uint32_t)(shifts_at + op.aux * sizeof(PShift));
    else if (op.code == PO_BLOCK) op.aux = (uint32_t)(blk_at + op.aux * kBlockTable);
    if (f32 && (op.code <= PO_BLOCKADE)) {
      float f[8];
      for (int k = 0; k < 8; ++k) f[k] = (float)op.m[k];
      std::memset(op.m, 0, sizeof(op.m));
      std::memcpy(op.f, f, sizeof(f));
    }
  }
  const size_t bytes = (blk_at + c.blk.size() * sizeof(float) + 255) & ~(size_t)255;
  h.bytes = (int32_t)bytes;
  const size_t at = (out.size() + 255) & ~(size_t)255;
  out.resize(at + bytes, 0);
  char* d = out.data() + at;
  std::memcpy(d, &h, sizeof(h));
  if (!c.ops.empty()) std::memcpy(d + sizeof(PHead), c.ops.data(), c.ops.size() * sizeof(POp));
  if (!c.terms.empty()) std::memcpy(d + terms_at, c.terms.data(), c.terms.size() * sizeof(PTerm));
  if (!c.shifts.empty()) std::memcpy(d + shifts_at, c.shifts.data(), c.shifts.size() * sizeof(PShift));
  if (!c.blk.empty()) std::memcpy(d + blk_at, c.blk.data(), c.blk.size() * sizeof(float));
  return at;
}

}  // namespace qsv
