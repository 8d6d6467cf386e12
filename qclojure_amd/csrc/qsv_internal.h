// qsv_internal.h — shared between the kernel file and the C-ABI file.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <complex>
#include <string>
#include <vector>
#include "../../include/qsv.h"

struct qsv_state;

namespace qsv {

constexpr int kBlock = 256;          // threads per workgroup (4 waves of 64)
constexpr int kReduceBlocks = 1024;  // fixed grid for FP64 reductions
constexpr int kPartials = 128 * kReduceBlocks;   // doubles of reduction scratch per state
constexpr int kReduceOut = 4096;     // doubles of reduction results per state
constexpr int kSampleChunkLog = 10;  // amplitudes per chunk in the sampling prefix

// Zero-bit insertion plan: enumerate `count` indices j and map each to the
// full index by inserting zeros at the ascending bit positions ins[0..nins)
// and OR-ing `orMask` (bits forced to one, e.g. controls).
struct InsArgs {
  uint64_t count;
  uint64_t orMask;
  int32_t nins;
  int32_t ins[5];
};

template <typename R>
struct Mat2 {
  R m[8];  // row-major 2x2, (re, im) interleaved
};

template <typename R>
struct Cplx {
  R re, im;
};

// A per-gate launch: high bits are inserted (ins), low bits (< threshold) are
// lane bits: lo_pred must all be set for the gate to act, lo_t is a low
// target. tbit is a high target (pair kernel) or the target whose value picks
// d0/d1 (phase kernel).
struct GateArgs {
  InsArgs ins;
  uint64_t lo_pred;
  uint64_t tbit;
  uint64_t lo_t;
};

// Two-bit exchange: hA/hB are high bits (0 when low), lA/lB low bits.
// Exactly one high bit is always passed as hA with the low one as lB.
struct SwapArgs {
  InsArgs ins;
  uint64_t lo_pred;
  uint64_t hA, hB;
  uint64_t lA, lB;
};

// ---- launchers ---------------------------------------------------------------
// All take a raw device pointer to the amplitude array (interleaved complex128
// or complex64, passed as void*) and launch on `st`.
// qsv_gates.hip
void launch_gate1(int prec, void* psi, const GateArgs& g, const double m[8], hipStream_t st);
void launch_phase(int prec, void* psi, const GateArgs& g, const double d0[2], const double d1[2], hipStream_t st);
void launch_swap2(int prec, void* psi, const SwapArgs& s, const double ph[2], hipStream_t st);
void launch_blockade(int prec, void* psi, uint64_t S, uint64_t bmask, const double ph[2], hipStream_t st);
// qsv_kernels.hip
void launch_fill_basis(int prec, void* psi, uint64_t S, uint64_t idx, hipStream_t st);
void launch_scale(int prec, void* psi, uint64_t S, double f, hipStream_t st);
// normalize-state without a host round trip: FP64 norm into out[0], then
// the scale by 1/norm when the norm exceeds 1e-12 (partials: kReduceBlocks doubles)
void launch_renorm(int prec, void* psi, uint64_t S, double* partials, double* out, hipStream_t st);
void launch_copy(int prec, const void* src, void* dst, uint64_t S, hipStream_t st);
// out[0..4] = Re <a|b>, Im <a|b>, sum |a|^2, sum |b|^2, max |a_i - b_i|;
// partials holds 5 * kReduceBlocks doubles.
void launch_compare(int pa, const void* a, int pb, const void* b, uint64_t S, double* partials, double* out,
                    hipStream_t st);
void launch_f64_to_c64(const double* src, void* dst, uint64_t count, hipStream_t st);
void launch_c64_to_f64(const void* src, double* dst, uint64_t count, hipStream_t st);

// FP64 reductions. `partials` holds kReduceBlocks * nterms * 2 doubles; the
// final values land in out[0..nterms*2) (re, im) on the device.
void launch_norm2(int prec, const void* psi, uint64_t S, double* partials, double* out, hipStream_t st);
void launch_inner(int prec, const void* a, const void* b, uint64_t S, double* partials, double* out,
                  hipStream_t st);
void launch_expect1q(int prec, const void* psi, uint64_t S, uint64_t tbit, const double m[8], double* partials,
                     double* out, hipStream_t st);
// Pauli-string sums (qsv_pauli.hip). One sweep over tiles of 12 index bits
// `pos` (ascending): nz Z strings (basis-index masks) and nu units, a multiple
// of four, of two strings each that share the X part x (tile-local, top = its
// highest bit). A string's sign part is split into tile-local bits s and the
// bits outside the tile g; im picks Im instead of Re. Results: out[0..nz) the
// Z sums, out[nz + 2 u + j] the sum over half the pairs of string j of unit u.
constexpr int kPauliZ = 128;
constexpr int kPauliUnits = 48;
constexpr int kPauliXBlocks = 512;
struct PauliUnit {
  uint32_t x, top;
  uint32_t s0, s1;
  uint64_t g0, g1;
  int32_t im0, im1;
};
struct PauliSweep {
  int32_t nz, nu;
  int32_t pos[12];
  uint64_t zmask[kPauliZ];
  PauliUnit u[kPauliUnits];
};
hipError_t launch_pauli_sweep(int prec, const void* psi, uint64_t S, const PauliSweep& sw, double* partials,
                              double* out, hipStream_t st);
// n <= kPauliRows strings, each over the state on its own: x == 0 the whole
// sum, else half the pairs (bit r of im: Im instead of Re of string r).
constexpr int kPauliRows = 64;
struct PauliRows {
  uint64_t x[kPauliRows], s[kPauliRows];
  uint64_t im;
};
hipError_t launch_pauli_rows(int prec, const void* psi, uint64_t S, const PauliRows& rows, int n, double* partials,
                             double* out, hipStream_t st);
void launch_probs(int prec, const void* psi, uint64_t offset, uint64_t count, double* out, hipStream_t st);

// Sampling: chunk sums -> inclusive prefix -> one wave per shot.
void launch_sample(int prec, const void* psi, uint64_t S, double* chunk_prefix, uint64_t shots, uint64_t seed,
                   uint64_t* out, hipStream_t st);

// Measurement of a qubit subset: outcome histogram (bits gathered at positions
// pos[0..m)), then collapse.
void launch_outcome_hist(int prec, const void* psi, uint64_t S, int m, const int* pos, double* hist,
                         hipStream_t st);
void launch_collapse(int prec, void* psi, uint64_t S, int m, const int* pos, uint64_t sel, double scale,
                     hipStream_t st);

// ---- fused tiled passes: planning (qsv_api.hip) ------------------------------
// Gates per pass. FP32 passes are renormalised between passes, which bounds
// the norm drift a pass may gather.
constexpr int kMaxPassGates = 1024, kMaxPassGatesF32 = 96;

// FG_RENORM: divide the state by its FP64 norm when that exceeds 1e-12, as
// normalize-state does after a Kraus operator (in trajectories above one
// workgroup; a barrier between fused passes, never inside one).
// FG_KRAUS: a noise site of a trajectory program (an operator chosen on the
// device); only in FGate lists.
enum { FG_DENSE = 0, FG_PHASE = 1, FG_SWAP = 2, FG_BLOCKADE = 3, FG_RENORM = 4, FG_KRAUS = 5 };
// Is re + i im a phase, up to rounding? Such a first entry of a diagonal gate
// can be divided out.
inline bool is_phase(double re, double im)
{
  const double d = re * re + im * im - 1.0;
  return d < 2e-9 && d > -2e-9;
}
// Structure of a dense 2x2, which decides the arithmetic it needs per pair:
// general (16 real multiply-adds), real entries (8), real diagonal with
// imaginary off-diagonal, as RX (8), or the exchange [[0,1],[1,0]] (none).
enum { DM_GENERAL = 0, DM_REAL = 1, DM_RX = 2, DM_EXCHANGE = 3 };

// A gate in tile-local bit coordinates. FG_KRAUS: target a, site b, operators
// cmask .. cmask + sub - 1 of the table, which change the norm by a factor between
// m[0] <= 1 and m[1] >= 1; bmask: renormalise afterwards in any case.
struct FGate {
  int32_t kind;        // FG_*
  int32_t a, b;        // dense/phase target a; swap bits a, b
  uint32_t cmask;      // local control bits (all must be 1)
  uint32_t bmask;      // blockade bits
  uint64_t gmask;      // control bits outside the tile (global; all must be 1)
  uint64_t gt;         // FG_PHASE with its target outside the tile (a < 0): the global target bit
  int32_t sub;         // FG_PHASE: 1 when d0 == 1; FG_DENSE: DM_* structure of m
  double m[8];         // dense: row-major 2x2; phase: d0 = m[0..1], d1 = m[6..7]; swap/blockade: phase m[0..1]
};

// Complex64 passes compute in FP32 by default. The rounded 2x2 matrices are
// unitary only to ~1e-7, so the norm would drift by that much per gate; it is
// removed pass by pass instead: a pass sums |amplitude|^2 per tile in FP64
// (FP_RENORM_OUT, and FP_RENORM_IN for the input of the first pass of a run),
// a one-workgroup kernel turns the sums into scale = sqrt(target / norm^2),
// and the next pass multiplies its loads by it (FP_RENORM_APPLY).
enum { FP_RENORM_APPLY = 1, FP_RENORM_IN = 2, FP_RENORM_OUT = 4 };
// Pass program flags beside them. FP_INIT_ZERO: the pass starts from |0..0>
// instead of loading the state (the first pass round of a grouped batch).
// FP_KEEP_ZERO (set by the compiler): every coefficient is finite, so a tile of
// zeros stays one.
// FP_REACH: the pass extends `reach` (below); FP_REACH_USE: and skips the tiles
// outside it.
enum { FP_INIT_ZERO = 8, FP_KEEP_ZERO = 16, FP_REACH = 32, FP_REACH_USE = 64 };

struct TileNorm {
  double* part_in;    // per-tile input norm^2 (first pass of a run)
  double* part_out;   // per-tile output norm^2
  double* ctl;        // [0] target norm^2, [1] scale for the next pass
  // index bits that are set [0] and clear [1] in some amplitude that may be
  // nonzero, from the passes so far
  unsigned long long* reach;
};

// The gates of one pass in program order, on tile-local bits.
struct FPass {
  int32_t tb = 12;                  // tile bits
  int32_t low = 0;                  // the low run: local bits 0..low-1 are global bits 0..low-1
  int32_t renorm = 0;               // FP_RENORM_* bits
  int32_t pos[16] = {};             // global index bit of tile-local bit i
  int32_t sorted_pos[16] = {};      // the same bits in ascending order
  std::vector<FGate> gates;
};

// ---- fused passes as micro-op programs (qsv_compile.hip, qsv_pass.hip) -------
// A pass compiled against the layouts it runs in: every op names the register
// bit, slot mask and thread-id mask it acts on.
constexpr int kPassTileBits = 12;
// Dense structures share the DM_* numbering.
enum { PM_GENERAL = DM_GENERAL, PM_REAL = DM_REAL, PM_RX = DM_RX, PM_EXCHANGE = DM_EXCHANGE };
enum {
  PO_DENSE = 0,       // + 4 * register bit + structure (PM_*): 0..15, no slot controls
  PO_DENSE_K = 16,    // + register bit: any 2x2 on the slot pairs whose bits kc are set, 16..19
  PO_PHASE = 20,      // one factor per lane on the slots whose bits kc are set (0, one or more)
  PO_PHASE2 = 21,     // + register bit, 21..24: one factor per lane for that bit set, one for it clear, on the slots kc
  PO_BLOCKADE = 25,   // phase where exactly one of the bits aux (thread) / kc (slot) is set
  PO_RELAYOUT = 26,   // layout col[0..13] -> layout col[14..27]; flag: PR_*
  PO_SWAP = 27,       // exchange local bits kc and aux where the local bits tmask are set (layout col[0..13])
  PO_KRAUS = 29,      // + register bit, 29..32: one of cnt noise operators from aux of site kc; flag: renormalise
  PO_BLOCK = 28,      // dense 16x16 on the four register bits (FP32 passes only): table at byte offset aux
};
// PO_RELAYOUT: the round trip stays inside each wave; the old layout is the one
// the previous relayout ended in; the workgroup must wait before writing.
enum { PR_LOCAL = 1, PR_SAME = 2, PR_WAIT = 4 };
// A register layout is a linear map over GF(2): thread t, slot k holds the
// tile-local index XOR_j t_j c_j XOR XOR_i k_i r_i. col[] lists the LDS element
// indices of the columns (the bank swizzle is linear too): c_0..c_9, r_0..r_3.
constexpr int kColT = 10, kCols = 14;
struct POp {
  int32_t code;
  uint32_t tmask;     // thread-id bits that must be set (thread-bit controls)
  uint32_t kc;        // slot bits that must be set (register-bit controls)
  uint32_t aux;       // PO_PHASE, PO_PHASE2, PO_RELAYOUT: byte offset of the terms or shifts
  int32_t cnt;        // ... and their number
  int32_t flag;
  uint64_t gm;        // global bits outside the tile that must be set, else the op is skipped
  double sc[2];       // PO_SWAP: the exchanged amplitudes' phase
  union {
    double m[8];      // row-major 2x2; PO_PHASE, PO_BLOCKADE: a factor in m[0..1]; PO_PHASE2: clear m[0..1], set m[6..7]
    float f[8];       // the same rounded, in the programs of FP32 passes
    uint16_t col[32]; // PO_RELAYOUT, PO_SWAP and PO_BLOCK (float programs keep no m there)
  };
};
static_assert(sizeof(POp) == 112, "ops are read in aligned dwords");
// A factor of PO_PHASE or PO_PHASE2 on the lanes with all bits of tmask set, in
// tiles with all bits of gmask set. In FP32 programs it has two values: PO_PHASE
// takes `on` where the thread bits tbit and the tile bits gbit are set and `off`
// otherwise (both 0: always `on`), PO_PHASE2 `on` for the set and `off` for the
// clear register bit.
struct PTerm {
  uint32_t tmask, tbit;
  uint64_t gmask, gbit;
  union {
    double d[2];      // FP64 programs
    float f[4];       // FP32 programs: on, off
  };
};
static_assert(sizeof(PTerm) == 40, "terms are 40 bytes");
// The indices of a tile whose base has global bit `bit` set are shifted (XOR):
// by LDS element `col` where a relayout leaves the layout, by global offset `g`
// at the store. CNOTs whose control lies outside the tile leave these.
struct PShift {
  uint32_t bit, col;
  uint64_t g;
};
// PO_BLOCK tables per pass: 4 steps x 64 lanes of (re, im) FP32, lane l of
// step kk holding U[l % 16][4 kk + l / 16] (the A operand of
// v_mfma_f32_16x16x4f32), U indexed by slot.
constexpr int kMaxPassBlocks = 8;
constexpr size_t kBlockTable = 4 * 64 * 2 * sizeof(float);
struct PHead {
  int32_t nops;
  int32_t renorm;                   // FP_RENORM_* bits
  int32_t bytes;                    // of the whole program
  int32_t store_wait;               // waves store where others load, with no barrier between: wait first
  int32_t nshift, shift_off;        // shifts of the store
  int32_t sorted_pos[16];           // the tile's global bits in ascending order
  uint64_t gload[kCols], gstore[kCols];   // global index columns of the load and store layouts
};
// In memory: the header, the ops and one unread op (the kernel fetches an op
// ahead), the terms, the shifts, the block tables.
// A program appended to `out` (at a multiple of 256 bytes); returns its offset.
// f32: an FP32 pass; block_cost > 0: runs of register-bit ops that cost the
// vector units at least that become PO_BLOCK ops. `scalar` collects factors
// common to the whole state: multiplied into it, applied (and reset) by this
// pass when `last`.
size_t compile_pass(const FPass& p, bool f32, int block_cost, std::complex<double>& scalar, bool last,
                    std::vector<char>& out);
// f32: complex64 arithmetic in FP32 (ignored for complex128, always FP64)
void launch_pass(int prec, bool f32, void* psi, const char* dprog, uint64_t ntiles, const TileNorm& nb,
                 hipStream_t st);
// A group of `count` states of S amplitudes (S >= one tile) back to back: one
// pass round (offs[y] = byte offset of instance y's program in `progs`, or -1).
void launch_pass_group(int prec, void* base, uint64_t S, unsigned count, const char* progs, const int64_t* offs,
                       hipStream_t st);

// The scale the next pass of a complex64 FP32 run applies (from the per-tile norms).
void launch_norm_ctl(const TileNorm& nb, uint64_t ntiles, bool first, hipStream_t st);
void launch_fill_group(int prec, void* base, uint64_t S, uint64_t count, hipStream_t st);

// ---- small circuits: a whole register per workgroup (qsv_small.hip) ------------
// Registers of up to kSmallC128 / kSmallC64 qubits run a whole program in one
// workgroup of 2^(n - 4) threads, FP64 arithmetic, 2^n * 8 B of LDS.
constexpr int kSmallC128 = 13, kSmallC64 = 14;
struct SmallInst {
  int32_t n;
  int32_t pad;
  uint64_t prog;         // byte offset of the program
  uint64_t io;           // amplitude offset of the state, ~0: none (it starts at |0..0> and is not stored)
  uint64_t t0, t1;       // Z terms [t0, t1)
  uint64_t dest;         // energies[dest], ~0: none
};
struct KrausOp {
  double w;              // selection weight
  double m[8];
};
struct SmallRun {
  int32_t prec;
  const char* progs;
  const SmallInst* insts;   // one per workgroup
  SmallInst one;            // with PO_KRAUS ops: every workgroup's, states back to back from one.io
  void* states;
  const uint64_t* tz;
  const double* tc;
  double* energies;
  const KrausOp* kraus;     // null: no PO_KRAUS ops; trajectory traj0 + workgroup otherwise
  uint64_t seed, traj0;
};
// Launches of one size class: registers of the class of `n` qubits.
int small_class(int n);
hipError_t launch_small(const SmallRun& r, int cls, unsigned count, hipStream_t st);
// <H> = sum_k c_k <Z-string_k> of one state of S >= 2^12 amplitudes into out[0];
// partials holds kReduceBlocks doubles.
void launch_zexpect(int prec, const void* psi, uint64_t S, const uint64_t* tz, const double* tc, uint64_t nterms,
                    double* partials, double* out, hipStream_t st);
// The same of `count` states of S amplitudes back to back: trange[2y..2y+1]
// = term range of state y, partials >= count * blocks_per_state doubles,
// out[dest[y]] = <H> of state y.
void launch_zexpect_group(int prec, const void* base, uint64_t S, unsigned count, const uint64_t* tz,
                          const double* tc, const uint64_t* trange, double* partials, unsigned blocks_per_state,
                          const uint64_t* dest, double* out, hipStream_t st);

// Shots for many small states stored back to back in an arena; norms
// (optional) receives each state's FP64 sum of |a|^2.
struct SampleJob {
  uint64_t state_offset;   // amplitude offset in the arena
  uint64_t out_offset;     // outcome offset
  uint64_t shots;
  uint64_t seed;
  int32_t n;
  int32_t pad;
};
void launch_batch_sample(int prec, const void* arena, const void* jobs, unsigned njobs, uint64_t* outcomes,
                         double* norms, hipStream_t st);
// Shared with the linear-algebra module (qsv_la.hip): set the calling
// thread's error message and return `code`; make sure the runtime is
// initialised; reach a state's amplitude buffer and stream.
int api_fail(int code, const char* msg);
int api_ensure_init();
int api_state_raw(const struct ::qsv_state* s, void** amps, hipStream_t* st, int* n, int* prec);

}  // namespace qsv
