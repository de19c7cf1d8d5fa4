// Host-side structures and kernel launchers shared by the HIP translation
// units of libmugpu.so.  Nothing here is part of the public C-ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "fft_core.hpp"
#include "mugpu.h"

namespace mugpu {

// ---- error handling --------------------------------------------------------
void set_error(const char* fmt, ...);
int hip_fail(hipError_t e, const char* what, const char* file, int line);
#define MUGPU_HIP(call)                                                   \
  do {                                                                    \
    hipError_t e_ = (call);                                               \
    if (e_ != hipSuccess) return ::mugpu::hip_fail(e_, #call, __FILE__, __LINE__); \
  } while (0)
#define MUGPU_TRY(call)          \
  do {                           \
    int rc_ = (call);            \
    if (rc_ != MUGPU_OK) return rc_; \
  } while (0)

// Device allocation of the library's own buffers (cells, tangents, plans,
// work vectors): a failed hipMalloc has its sticky error cleared (the next
// launch check would report it otherwise), the field cache is handed back to
// the device after the library stream's work, and the allocation is retried
// once.  On failure *p is nullptr and MUGPU_EMEMORY is returned with `what`
// in the message.
int dev_alloc(void** p, size_t bytes, const char* what);
template <typename T>
inline int dev_alloc(T** p, size_t bytes, const char* what) {
  return dev_alloc(reinterpret_cast<void**>(p), bytes, what);
}

// Squared stopping threshold of one inner FP32 CG solve of the mixed-precision
// refinement, for the inner system A d = r64 / |r64| whose start residual has
// squared norm rdr: the inner solve stops at inner_tol relative or, when that
// is more than the outer tolerance still asks for, once |r64| times its
// relative residual is half the outer threshold (tol2 = tol^2 |b|^2, rr =
// |r64|^2).  FP32 CG converges evenly to about 1e-4 relative and slows beyond
// it, so the first inner solve stops at inner_tol; the last one of a solve at
// a tolerance above inner_tol^2 stops as soon as the outer test will pass.
inline double inner_threshold2(double inner_tol, double tol2, double rr, double rdr) {
  const double need2 = 0.25 * tol2 / rr;
  const double rel2 = inner_tol * inner_tol;
  return (need2 > rel2 ? need2 : rel2) * rdr;
}

hipStream_t stream();
// route the library's launches to another stream (nullptr: the library
// stream); used by the serving loop, which drives two streams from one thread
void set_current_stream(hipStream_t s);
// while a stream is captured into a graph, the per-launch event timing is off
void set_capturing(bool on);
int max_lds_per_block();
// per-launch event timing of one kernel class (MUGPU_K_*), off by default
void timing_begin(int kclass);
void timing_end(int kclass);
// position in the timing record, and dropping the launches recorded since a
// position (launches that returned at once; not counted anywhere)
int64_t timing_mark();
void timing_void(int64_t from);

// ---- tangent representations of the directional-stiffness product --------
// FULL: the reference's stored K, nc*nc entries per voxel, entry r + nc*c is
//       K(r, c) (src/common/T4_map_proxy.hh:83-105)
// ISO : (lambda, mu) per voxel; dP = lambda tr(dF) I + mu (dF + dF^T), the
//       contraction with C = lambda Itrac + 2 mu Isymm
// HEP : dim^3 per voxel, M(i,m,n) at i + d m + d^2 n, for the j-independent
//       Kirchhoff->PK1 tangent K(i,m,j,n) = M(i,m,n)
//       (src/materials/materials_toolbox.hh:394-406)
// SYM : the upper triangle r <= c of a major-symmetric K (finite-strain
//       hyperelastic laws and the consistent elasto-plastic tangent),
//       nc (nc + 1) / 2 entries, row by row
// LEF : FP64 finite-strain cells of linear elastic laws (LE1-4; eigenstrains
//       symmetric, else S is not): F, the PK2 stress S (Voigt order) and (lambda, mu), from which dP = dF S +
//       F (C : sym(F^T dF)) is formed; dim^2 + dim (dim + 1) / 2 + 2 numbers, 17
//       in 3D where the matrix has 45
// HCT : FP64 3D cells of HyperElastoPlastic1 with the consistent tangent alone:
//       the 26 numbers of hct_product (op_stages.hpp)
// A CG iteration reads the tangent once per voxel, so its size counts (256^3
// HCT: r2c pass 2.57 -> 2.04 ms; 175x147x99 LEF: 340 -> 261 us).
//
// Storage is voxel-blocked: blocks of kTanBlock consecutive voxels, entry
// major inside a block, so that lanes on consecutive voxels read one
// contiguous run per entry (coalesced) while a voxel's entries stay in one
// block.
enum TangentKind { TAN_FULL = 0, TAN_ISO = 1, TAN_HEP = 2, TAN_SYM = 3, TAN_LEF = 4, TAN_HCT = 5 };
constexpr int kHct = 26;
constexpr int kTanBlock = 64;
__host__ __device__ inline int tangent_stride(int kind, int dim) {
  const int nc = dim * dim;
  if (kind == TAN_LEF) return nc + dim * (dim + 1) / 2 + 2;
  if (kind == TAN_HCT) return kHct;
  return kind == TAN_FULL ? nc * nc
                          : kind == TAN_ISO ? 2 : kind == TAN_HEP ? dim * dim * dim : nc * (nc + 1) / 2;
}
// number of values allocated for a tangent over npix voxels
inline int64_t tangent_values(int kind, int dim, int64_t npix) {
  return (npix + kTanBlock - 1) / kTanBlock * kTanBlock * tangent_stride(kind, dim);
}
// offset of entry q of voxel v for a stride of S entries per voxel
__host__ __device__ inline int64_t tan_off(int64_t v, int q, int S) {
  return (v / kTanBlock) * ((int64_t)S * kTanBlock) + (int64_t)q * kTanBlock + (v % kTanBlock);
}
// packed index of K(r, c), r <= c, in the SYM representation of an n x n matrix
__host__ __device__ constexpr int sym_index(int r, int c, int n) {
  return r * n - r * (r - 1) / 2 + (c - r);
}

// device scalar block used by the CG kernels
// SC_TOL2: squared stopping threshold of a batched inner CG
// SC_XALPHA: alpha of a pending x update (kept apart from SC_ALPHA, which
// the next solve on the cell overwrites)
// SC_RDR1: with SC_RDR, the r . r of alternate iterations of a chunk whose
// scalars are folded into the passes (ScalarFold)
enum Scalar { SC_RDR = 0, SC_PAP, SC_ALPHA, SC_NEWRDR, SC_BETA, SC_TMP0, SC_TMP1, SC_TOL2,
              SC_XALPHA, SC_RDR1, SC_COUNT };

// Scalars of an FP64 CG iteration without kernels of their own, for grids whose
// passes have at most kFoldMax workgroups: every workgroup of the c2r pass sums
// the first pass's partials of p . K p itself (alpha), and every workgroup of
// the next r2c pass the c2r pass's partials of r . r (beta and the loop test);
// workgroup 0 stores what the host and the later kernels read.  A pass that
// waits for a chunk's previous kernel anyway then costs a few hundred ns more
// instead of a launch of 4 to 5 us; with more partials than kFoldMax the
// redundant reads cost more than that, and k_finalize runs.  All of them sum in
// one order (fold_sum), so any mixture gives the same bits.
struct ScalarFold {
  double* pk = nullptr;  // partials of p . K p (r2c writes, c2r sums); null: not folded
  const double* rr = nullptr;  // r2c: partials of r . r to sum; null: beta is in the scalar block
  int nrr = 0;                 // their number
  int npk = 0;                 // c2r: number of p . K p partials
  int iter = 0;                // iterations of the chunk already run
  int* ctl = nullptr;          // CTL_* words (r2c with rr)
  double* scal = nullptr;
  double* aring = nullptr;     // OpSpec::aring
};
constexpr int kFoldMax = 1024;
// directions of a chunk of CG iterations kept before they are added to x
// (ring_flush); alpha of iteration i in aring[i % kRing]
constexpr int kRing = 8;

// ---- passes of run-time length (fft_gen.hpp) -------------------------------
constexpr int kGenMaxPass = 12;
constexpr int kGenQ = 4;          // output pairs of a prime radix formed at once
constexpr int kGenTB = 2;         // such tasks held per thread
constexpr int kGenMaxNT = 512;    // threads per workgroup
constexpr int kGenThreads = 256;  // aimed at, where the passes can use them
constexpr int kGenVals = 18;      // complex values of a line held per thread
constexpr size_t kGenMaxLds = 150 * 1024;
constexpr size_t kGenLds = 40 * 1024;  // four workgroups per CU
// radices with a compiled butterfly, and how many of them a thread holds
__host__ __device__ constexpr bool gen_compiled(int R) {
  return R <= 5 || R == 7 || R == 8 || R == 9 || R == 11 || R == 13 || R == 17;
}
__host__ __device__ constexpr int gen_held(int R) { return R >= 16 ? 1 : 16 / R; }
struct GenPass {
  int R, NS, nb, step;  // radix, span before it, n / R, n / (NS R)
  unsigned magic;       // j / NS = (j magic) >> 32
};
struct GenAxis {
  int n, np, cls;  // cls 1: a radix above 9
  GenPass ps[kGenMaxPass];
};
// shape of a workgroup: `mult` row pairs or k-points, L lines, P threads per
// line; NT = 0: the axis does not fit
struct GenShape {
  int mult = 0, L = 0, P = 0, NT = 0, NT_bwd = 0;
  size_t lds = 0, lds_bwd = 0;  // _bwd: of the c2r pass
};
bool gen_radices(int n, GenAxis& ax);
// (nc components per point, nl lines per row or k-point)
GenShape gen_last_shape(const GenAxis& ax, int nc, int nl, int64_t rows);
GenShape gen_axis0_shape(const GenAxis& ax, int nl, int64_t plane);
GenShape gen_strided_shape(const GenAxis& ax, int64_t inner, int64_t outer);

// Workgroups are dispatched to the 8 XCDs round robin (workgroup b runs on
// XCD b mod 8), each XCD with its own L2.  Tiles next to each other in HBM
// share cache lines at their edges, so the tile of workgroup b is chosen to
// give every XCD one contiguous range of tiles: neighbours then meet in the
// same L2.
constexpr int kXcds = 8;
__device__ __forceinline__ int64_t xcd_tile(int64_t b, int64_t total) {
  const int64_t q = total / kXcds, r = total - q * kXcds;
  const int64_t x = b % kXcds, local = b / kXcds;
  return x * q + (x < r ? x : r) + local;
}

// ---- FFT plan -----------------------------------------------------------------
struct FftPlan {
  int dim = 0, nc = 0, prec = MUGPU_FP64;
  int res[3] = {1, 1, 1}, hres[3] = {1, 1, 1};
  int64_t N = 0, kpts = 0;
  AxisPlan ax[3];
  void* tw64[3] = {nullptr, nullptr, nullptr};  // double2 tables W_n^m
  void* tw32[3] = {nullptr, nullptr, nullptr};  // float2 tables
  // z-pass: rows per workgroup; strided passes: lines per workgroup
  int zrb = 1;
  int yW = 1;
  int xW = 1;      // plain axis-0 pass
  int xWk = 1;     // fused axis-0 projection pass: k-points per workgroup
  int xNT = 256;   // threads of the fused pass
  void* partials = nullptr;  // double per z-pass workgroup
  int64_t wg_r2c = 0, wg_c2r = 0;  // workgroups of the latest FP64 last-axis launches (their partials)
  int64_t nzblocks = 0;      // z-pass workgroups, the largest of nzb
  int64_t nzb[2] = {0, 0};   // c2r workgroups (p.Ap partials) per precision (0 FP64, 1 FP32)
  bool fastax[3] = {false, false, false};  // compile-time-length passes (fft_fast.hip)
  // run-time-length passes per axis (genax: the axis has them)
  GenAxis gen[3];
  bool genax[3] = {false, false, false};
  GenShape gen_last[2], gen_axis0[2], gen_str[3][2];  // one line per component; packed
  // packed symmetric lines (op_stages.hpp) of FP64 small-strain operators: every
  // axis has a pass that takes them (can_pack), whether the plan's own operators
  // use them too or only the CG iterations (general, plan_init), and whether
  // the run in hand does (packed)
  bool general = true, can_pack = false, packed = false;
  int lines() const { return packed ? dim * (dim + 1) / 2 : nc; }
  // variant of each compile-time-length pass (bit 0: 8 values per thread
  // instead of 16 or 12; bit 1: half the rows or k-points per workgroup, for
  // the last-axis and first-axis projection passes), per precision (0 FP64,
  // 1 FP32), per pass and per form: 0 one line per component, 1 the same with an
  // isotropic tangent (r2c pass), 2 packed lines (FP64 last-axis and projection
  // passes), whose tiles are two thirds as wide (first axis at 256^3: the variant best for
  // nine lines takes 687 us on six, the best one 415; at 128^3 52.6 and 43.7)
  unsigned char fvar[2][5][3] = {};
  ScalarFold fold;  // of the run in hand (operator_impl)
  bool fold_ok = false;  // no last-axis pass of this plan has more than kFoldMax workgroups
  // while set: every pass kernel returns at once when active[0] == 0 (CG
  // iterations launched ahead of the host's stopping test)
  const int* active = nullptr;
};
// passes with variants
enum FastVariantPass { FV_R2C = 0, FV_STRIDED1 = 1, FV_AXIS0 = 2, FV_C2R = 3, FV_STRIDED0 = 4, FV_COUNT = 5 };
// variant of a pass for an axis length, dimension, precision and tangent
// class, from the tuned table (fft_tuned.inc)
int fast_variant(int pass, int n, int dim, int prec, int form);
// make fast_variant return `variant` for a pass and precision wherever that
// variant exists (-1: the tuned table again); plans read it when created
void force_variant(int pass, int prec, int variant);
// whether a pass variant exists (and differs from variant 0's tile) for
// this length, dimension and precision
bool fast_variant_valid(int pass, int n, int dim, int prec, int variant);

// general: passes of run-time length where they fit, packed symmetric lines in
// every operator.  Cells of the FP32-refined solve and the served ones have not
// been moved to them (their FP32 loop keeps the plain schedule on nine
// components), so they give the bits they always gave.  Nothing in their
// accuracy asks for it: x carries the FP32 rounding of the inner solves, 1.5e-6
// relative, far above a last-bit change of any pass
int plan_init(FftPlan& p, int dim, const int* res, int nc, int prec, bool general = true);
void plan_free(FftPlan& p);

// projection parameters handed to the fused axis-0 kernel
struct ProjParams {
  int kind = -1;  // MUGPU_PROJ_*; -1 none
  int allow_even = 0;
  double L[3] = {1, 1, 1};
  double norm = 1.0;
};

// input stage of the last-axis r2c pass
// IN_TAN_PUPDATE_X: kernel form of IN_TAN_PUPDATE that also applies x +=
// alpha p_old (chosen by the launcher when OpSpec::xvec is set)
// IN_TAN_S: kernel form of IN_TAN and IN_TAN_PUPDATE for packed symmetric CG
// vectors (OpSpec::sym)
enum InMode { IN_PLAIN = 0, IN_TAN = 1, IN_TAN_PUPDATE = 2, IN_TAN_PUPDATE_X = 3, IN_TAN_S = 4 };
// output stage of the last-axis c2r pass
// OUT_RUPD: r += alpha A p with the partials of r . r, for solves whose alpha is
// known before the inverse transform (OpSpec::fin_alpha)
// OUT_RUPD_S: kernel form of OUT_RUPD for packed symmetric CG vectors
enum OutMode { OUT_PLAIN = 0, OUT_DOT = 1, OUT_RUPD = 2, OUT_RUPD_S = 3 };
// forms of a pass over packed symmetric CG vectors
enum SymFlags {
  SYM_SRC_FULL = 1,  // p and r come from fields of dim^2 components
  SYM_UPDATE = 2,    // p = -r + beta p (else p is taken as it is)
  SYM_OUT_FULL = 4   // r goes to a field of dim^2 components
};

struct OpSpec {
  int in_mode = IN_PLAIN;
  const void* in = nullptr;      // real field (plan precision)
  const void* rvec = nullptr;    // CG residual for IN_TAN_PUPDATE
  void* pout = nullptr;          // updated p for IN_TAN_PUPDATE
  // IN_TAN_PUPDATE with compile-time-length last axis only: x += alpha p_old
  // on the way in (alpha = scal[SC_ALPHA], the previous iteration's), so
  // that the CG update need not read p again
  void* xvec = nullptr;
  const double* scal = nullptr;  // device scalars (SC_BETA)
  int tan_kind = TAN_FULL;
  const void* tangent = nullptr; // plan precision
  int out_mode = OUT_PLAIN;
  void* out = nullptr;           // real field (plan precision); OUT_RUPD: r
  const void* dotv = nullptr;    // vector dotted with the output for OUT_DOT
  // FP64, IN_TAN*: alpha = r . r / (p . K p) is formed in fin_alpha (the scalar
  // block) right after the first pass, from that pass's partials of p . K p.
  // It equals r . r / (p . G K p) for p in the range of G, the orthogonal
  // projector, so OUT_RUPD can use it and A p need not be stored
  double* fin_alpha = nullptr;
  void* ap_out = nullptr;        // OUT_RUPD: also store A p here (optional)
  // with fin_alpha: workgroups of the latest c2r pass and the buffer for the
  // partials of p . K p, where the scalars may be folded into the passes
  double* fold_pk = nullptr;
  int fold_iter = 0;             // iterations of the chunk already run; > 0: beta is folded too
  // packed runs with an early alpha: pout holds the packed components of p
  // (always written), in and rvec (the r that is read) too unless
  // SYM_SRC_FULL, out (the r that is written) unless SYM_OUT_FULL
  bool sym = false;
  int sym_flags = 0;
  double* aring = nullptr;       // also store alpha in aring[iteration % kRing]
};

// full operator: r2c (with input stage) -> [axis passes] -> projection ->
// [inverse axis passes] -> c2r (with output stage); spectrum is workspace
int run_operator(FftPlan& p, int prec, const OpSpec& op, const ProjParams& pj,
                 void* spectrum);
// engine transforms (no projection)
int run_r2c(FftPlan& p, int prec, const void* in, void* spectrum);
int run_c2r(FftPlan& p, int prec, void* spectrum, void* out);

struct BatchSlot;
// passes for axis lengths 16, 32, 48, 64, 96, 128, 256, 512 (fft_fast.hip)
bool fast_size(int n);
// rows per workgroup of the last-axis passes in a variant
int fast_rows_per_block(int n, int dim, int variant);
int fast_r2c(FftPlan& p, int prec, const OpSpec& op, void* spec);
int fast_c2r(FftPlan& p, int prec, const OpSpec& op, void* spec);
int fast_strided(FftPlan& p, int prec, int ax, void* spec, int sign);
int fast_axis0_project(FftPlan& p, int prec, const ProjParams& pj, void* spec);
// passes along axes of run-time length (fft_gen_last.hip, fft_gen_axis.hip)
int gen_r2c(FftPlan& p, int prec, const OpSpec& op, void* spec);
int gen_c2r(FftPlan& p, int prec, const OpSpec& op, void* spec);
int gen_strided(FftPlan& p, int prec, int ax, void* spec, int sign);
int gen_axis0_project(FftPlan& p, int prec, const ProjParams& pj, void* spec);
// the HBM pattern of the first-axis pass alone (n rows of plane k-points of nc
// complex components, tiles of kp k-points), in place (fft_fast.hip)
int line_pattern(void* data, int prec, int n, int64_t plane, int nc, int kp);
// batched FP32 operator G:(K:p) with the p update and the p . Ap partials,
// one RVE per slot (fft_fast.hip)
int fast_batch_operator(FftPlan& p, const BatchSlot* d_slots, int nslots);
// batched k_finalize (alpha or beta + stopping test) and x, r update (cg.hip)
int batch_finalize(const BatchSlot* d_slots, int nslots, int64_t count, int mode);
int batch_cg_update(const BatchSlot* d_slots, int nslots, int64_t n);

// ---- batched inner CG (serving) -------------------------------------------
// One RVE of a batch of equal-resolution RVEs whose FP32 inner CG iterations
// run in the same launches (slot = blockIdx.z).  ctl[0] active flag, ctl[1]
// iterations done, ctl[2] iteration limit; a finished slot is skipped by
// every later launch, so a solve stops exactly where it would stop alone.
struct BatchSlot {
  const float* tan;
  float* x;
  float* r;
  float* p;
  float* Ap;
  float2* spec;
  double* scal;   // SC_* block of this RVE
  double* zpart;  // per-workgroup partials of the c2r pass (p . Ap)
  double* upart;  // per-workgroup partials of the update (r . r)
  int* ctl;
  int tan_kind;
  int kind;        // projection (MUGPU_PROJ_*)
  int allow_even;
  double L[3];
  double norm;
};
enum BatchCtl { CTL_ACTIVE = 0, CTL_ITER = 1, CTL_MAXIT = 2, CTL_COUNT = 4 };

// one inner CG iteration for the slots [0, nslots) of a batch (FP32 operator,
// FP64 scalars); slots must share the plan's resolution
int batch_cg_iteration(FftPlan& p, const BatchSlot* d_slots, int nslots);

// ---- reductions and vector kernels (cg.hip) --------------------------------
int dot_device(int prec, const void* a, const void* b, int64_t n, double* d_partials,
               double* d_scal, int slot);
// ctl (optional, CTL_* words): skip when ctl[CTL_ACTIVE] == 0; FIN_BETA then
// also applies SolverCG's loop test (ctl[CTL_ITER] + 1 < ctl[CTL_MAXIT] and
// r.r > scal[SC_TOL2]) and clears CTL_ACTIVE when it fails
// aring (FIN_ALPHA): OpSpec::aring
int finalize(const double* d_partials, int64_t count, double* d_scal, int mode,
             int* ctl = nullptr, double* aring = nullptr);
// ctl = {active, 0 iterations, maxit}, scal[SC_TOL2] = tol2 (on the stream)
int set_ctl(int* ctl, int maxit, double* d_scal, double tol2);
enum FinalizeMode { FIN_ALPHA = 0, FIN_BETA = 1, FIN_STORE_TMP0 = 2, FIN_STORE_TMP1 = 3,
                    FIN_STORE_RDR = 4 };
// x == nullptr: x is updated elsewhere (OpSpec::xvec of the next r2c)
int cg_update(int prec, void* x, void* r, const void* p, const void* Ap, const double* d_scal,
              int64_t n, double* d_partials, int* ctl = nullptr);
// x += alpha p with alpha = scal[slot] (the update left over when the CG
// x update rides on the next iteration's r2c)
int axpy_alpha(int prec, void* x, const void* p, const double* d_scal, int64_t n,
               int slot = SC_ALPHA);
// scal[to] = scal[from] on the device
int scal_copy(double* d_scal, int from, int to);
// beta after the last iteration of a folded chunk (ctl != null: where the chunk
// still ran; `iters` iterations of it were queued) or after a single step
int fold_beta(const double* rr, int count, double* d_scal, int* ctl, int iters);
// x += sum alpha_i p_i over the iterations [base, base + len) of a chunk that were
// run, then, after the last one run, p and (sym) r in their full fields
struct RingFlush {
  const double* p[kRing];  // directions, packed symmetric with `sym`
  const double* before;    // direction of iteration base - 1, null for base = 0
  double* x;
  double* p_out;
  double* r_out;
  const double* rs;      // sym: packed r, copied to r_out if the last iteration has not run
  const double* scal;
  const double* aring;
  const int* ctl;        // CTL_* words, null: every iteration was run
  int64_t n;             // values of x
  int base, len, total;  // total: iterations of the chunk
};
int ring_flush(const RingFlush& a, int dim, bool sym);
// start of an FP64 solve: x = 0, r = -b, p = b; b.b into scal[SC_RDR] and
// scal[SC_TMP0], |b - g|^2 into scal[SC_TMP1]
int cg_start_vectors(const double* b, const double* g, double* x, double* r, double* p, int64_t n,
                     double* d_partials, double* d_scal);
int axpby(int prec, double a, const void* x, double b, void* y, int64_t n);
int convert(int from_prec, const void* src, int to_prec, void* dst, int64_t n, double scale);
// x64 += scale d32; with p32: scale (d32 + scal[SC_ALPHA] p32)
int add_scaled_convert(void* x64, const void* d32, double scale, int64_t n,
                       const void* p32 = nullptr, const double* d_scal = nullptr);
// inner-solve start of the mixed CG: r32 = -s r64, p32 = -r32, x32 = 0,
// r32.r32 finalized into scal (mode as for finalize)
int mixed_start(const double* r64, double s, float* r32, float* p32, float* x32, int64_t n,
                double* d_partials, double* d_scal, int mode);
// r = b - r (r holds A x on entry), r.r finalized into scal
int residual_dot(const double* b, double* r, int64_t n, double* d_partials, double* d_scal,
                 int mode);
int fill_uniform(double* F, const double* h_val, int nc, int64_t npix, int add);
constexpr int kRedBlocks = 4096;  // capacity of the partial-sum buffers
constexpr int kRedGrid = 1024;    // default workgroup cap of the grid-stride kernels

// ---- materials (materials.hip) ----------------------------------------------
struct MaterialDev {
  int family = 0;
  double young = 0, poisson = 0, lambda = 0, mu = 0, bulk = 0, tau_y0 = 0, H = 0;
  std::vector<int64_t> h_pix;
  std::vector<double> h_params;  // per pixel
  int ppn = 0;
  std::vector<double> h_C;       // MUGPU_LEG: C_ijkl at (i + d j) + d^2 (k + d l)
  double* d_C = nullptr;
  bool major_sym = true;         // MUGPU_LEG: C_ijkl == C_klij; MUGPU_LE2: symmetric eigenstrains
  int* d_pix = nullptr;
  double* d_params = nullptr;
  double* Fp[2] = {nullptr, nullptr};
  double* be[2] = {nullptr, nullptr};
  double* ep[2] = {nullptr, nullptr};
  int cur = 0;
  int64_t n_pixels = -1;  // pixel count when h_pix is not kept on the host
};

int eval_material(const MaterialDev& m, int dim, int form, const double* F, double* P,
                  int tan_kind, double* tangent, int need_tangent);

// serving: the material stage of several requests of one resolution in one
// launch (one request per blockIdx.y): small-strain per-voxel isotropic
// elasticity (MaterialLinearElastic4 over all pixels), writing the stress P,
// the right-hand side -P, the TAN_ISO tangent and its FP32 copy, bit for bit
// what eval_material and convert write
struct ServeMatSlot {
  const double* F;
  const double* params;  // (lambda, mu) per voxel
  double* P;
  double* rhs;
  double* tan64;
  float* tan32;
};
constexpr int kServeMatSlots = 64;  // requests per launch (passed by value)
int serve_material_batch(int dim, const ServeMatSlot* slots, int nslots, int64_t n);

}  // namespace mugpu
