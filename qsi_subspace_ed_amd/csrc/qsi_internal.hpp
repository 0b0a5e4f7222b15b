// Internal objects behind the C ABI handles.
#pragma once

#include <atomic>
#include <vector>

#include "qsi_common.hpp"

namespace qsi {

// Largest basis dimension: ranks are uint32, and a kernel with one thread per
// row (rounded up to whole 256-thread workgroups) must stay below the 2^32
// work-items a dispatch can hold.
constexpr int64_t kMaxDim = (int64_t{1} << 32) - 512;

// Off-diagonal term in pull form.  For a row state s the term contributes
//   c * sgn * (-1)^popcount(~s & Z) * x[rank(s ^ X)]
// when (s & m) == v.  With s' = s ^ X the pre-image, this is the reference's
// precondition (s' & down) == 0 && (s' & up) == up rewritten on s:
//   m = up | down,  v = up ^ (X & m).
struct OffTerm {
  uint64_t m[2];
  uint64_t v[2];
  uint64_t X[2];
  uint64_t Z[2];
  double c;     // coefficient (single-vector apply)
  double sgn;   // +-1 operator sign
  int32_t slot; // coefficient slot for block applies (-1: use c)
  int32_t cls;  // coefficient class (block applies), -1 when classes are off
};

// Off-diagonal terms of one coefficient class share their per-column
// coefficient in a block apply: slot `slot` of the column (or `c` when the
// apply has no per-column coefficients or slot < 0).  Block applies keep the
// classes' coefficients in LDS instead of loading each term's.
struct CoefClass {
  double c;
  int32_t slot;
  int32_t pad;
};
constexpr int kMaxCoefClasses = 8;

// Diagonal term.  kind 0: c * sgn * (-1)^popcount(~s & Z) when (s & m) == v
// (a Z string times up/down projectors, m = up | down, v = up), else 0;
// kind 1: c * sgn * (2 popcount(s & Z) - popcount(Z))  (a sum of single-site
// Z terms that share one coefficient and slot, merged on the host).
struct DiagTerm {
  uint64_t m[2];
  uint64_t v[2];
  uint64_t Z[2];
  double c;
  double sgn;
  int32_t kind;
  int32_t slot;
};

// What a wavefront needs of an off-diagonal term as one scalar load: projector
// mask and value, the reversed flip's value v ^ (X & m), c * sgn.
template <int NW>
struct alignas(32 * NW) TermRec {
  uint64_t m[NW];
  uint64_t v[NW];
  uint64_t u[NW];
  double c;
};
static_assert(sizeof(TermRec<1>) == 32 && sizeof(TermRec<2>) == 64, "4 or 8 words");

// The off-diagonal terms field by field, n entries each (a multiple of 64, the
// tail zero), so a wavefront's lanes read one field of 64 terms with one
// coalesced load (projector mask, value and flip mask per word; the flip mask's
// bucket key with the term's class, sign and whether it has a Z string in the
// upper half), and then as TermRec records.
struct TermPlanes {
  static constexpr int kCount = 7;
  static constexpr uint32_t kNegative = 256, kHasZ = 512;  // class in bits 0-7
  const uint64_t* p;
  int n;
  __host__ __device__ const uint64_t* m(int w) const { return p + (3 * w) * n; }
  __host__ __device__ const uint64_t* v(int w) const { return p + (3 * w + 1) * n; }
  __host__ __device__ const uint64_t* X(int w) const { return p + (3 * w + 2) * n; }
  __host__ __device__ const uint64_t* key() const { return p + 6 * n; }
  __host__ __device__ const uint64_t* rec() const { return p + kCount * n; }
};

}  // namespace qsi

struct qsi_basis_s {
  int64_t dim = 0;
  int n_spins = 0;
  int nw = 1;
  int kbits = 0;
  int n_seg = 0;  // bucket key fields (see BasisView)
  uint8_t seg_lo[qsi::kKeySegs] = {};
  uint8_t seg_w[qsi::kKeySegs] = {};
  int device = 0;
  uint64_t* d_states = nullptr;  // dim * nw words
  uint32_t* d_table = nullptr;   // 2^kbits + 1
  ulonglong2* d_hash = nullptr;  // hash index (null if not built)
  uint32_t* d_slots = nullptr;   // slot index, 2 * dim entries (null if not built)
  uint32_t* d_lowkeys = nullptr; // low keys, dim entries (null if not built)
  int n_low = 0;                 // low-key runs (see BasisView)
  uint8_t low_lo[qsi::kLowSegs] = {};
  uint8_t low_w[qsi::kLowSegs] = {};
  uint64_t infmask[2] = {0, 0};  // informative positions (bit p: spin p)
  int hbits = 0;
  std::atomic<int> refs{1};

  qsi::HashView hview() const {
    qsi::HashView h;
    h.slots = d_hash;
    h.mask = (hbits > 0) ? ((uint64_t{1} << hbits) - 1) : 0;
    h.hbits = hbits;
    return h;
  }

  qsi::BasisView view() const {
    qsi::BasisView v;
    v.states = d_states;
    v.table = d_table;
    v.slots = d_slots;
    v.lowkeys = d_lowkeys;
    v.dim = dim;
    v.kbits = kbits;
    v.n_spins = n_spins;
    v.n_seg = n_seg;
    for (int q = 0; q < qsi::kKeySegs; ++q) {
      v.seg_lo[q] = seg_lo[q];
      v.seg_w[q] = seg_w[q];
    }
    v.n_low = n_low;
    for (int q = 0; q < qsi::kLowSegs; ++q) {
      v.low_lo[q] = low_lo[q];
      v.low_w[q] = low_w[q];
    }
    return v;
  }
};

struct qsi_op_s {
  qsi_basis_s* basis = nullptr;
  int n_off = 0;
  int n_diag = 0;
  int n_slots = 0;
  bool has_z = false;  // any off-diagonal term with a Z string
  int variant = 0;     // apply kernel: one of the QSI_APPLY_* values
  qsi::OffTerm* d_off = nullptr;
  qsi::DiagTerm* d_diag = nullptr;
  uint64_t* d_planes = nullptr;  // TermPlanes data (in the allocation of d_off)
  int n_plane = 0;
  bool ordered = false;          // every off-diagonal term's X lies under its m
  bool paired = false;           // every off-diagonal term's reverse flip is a term's too
  bool symmetric = false;        // ... with the same coefficient, slot, sign and Z string
  // sampled on large bases: of the pairs of 128 rows and a term that connect, the
  // share with a target outside the basis
  float miss_share = 0.0f;
  std::vector<qsi::OffTerm> h_off;
  std::vector<qsi::DiagTerm> h_diag;
  int n_cls = 0;  // coefficient classes (0: more than kMaxCoefClasses)
  qsi::CoefClass* d_cls = nullptr;
  std::vector<qsi::CoefClass> h_cls;
  // cached connectivity (qsi_op_cache_connectivity): CSR over the rows (64-bit
  // offsets: a 96-spin operator has 3.3e10 nonzeros), the
  // rank of each connected state (0xFFFFFFFF if absent) and its coefficient
  // class | negative-sign bit << 7, off-diagonal terms in term order
  uint64_t* d_rowptr = nullptr;
  uint32_t* d_cj = nullptr;
  uint8_t* d_cm = nullptr;
  int64_t conn_nnz = -1;  // -1: not cached (connected terms; absent ones included)
  int conn_pad = 1;       // rows padded to multiples of conn_pad entries (1 or 4)
  int blk_cfg = 1;        // block-apply configuration (qsi_op_autotune)
  int cached_pipe = 8;    // gathers in flight per lane of the cached apply (4-32)
  // how the low-key kernels confirm a candidate (qsi_op_verify_lowkeys):
  // 0 compare its state; 1 compare its low key (no connected state outside
  // the basis shares a bucket key and low key with a basis state); 2 no
  // compare (every connected state is in the basis).  A property of the terms
  // and the basis, both fixed, so it holds for any build of the keys.
  int lowkeys_check = 0;

  qsi::TermPlanes planes() const { return {d_planes, n_plane}; }
};

namespace qsi {

void basis_retain(qsi_basis_s* b);
void basis_release(qsi_basis_s* b);
// takes ownership of d_states (dim x nw words, device)
int basis_adopt_device(uint64_t* d_states, int64_t dim, int n_spins, int bucket_bits,
                       qsi_basis_s** out);

// Launch helpers shared by the solvers (all stream ordered).
// y = yscale * y_in + H x  (y_in may be null or alias y); if dot_out is
// non-null, *dot_out (device) = sum_i x[i] * y[i] after the update.
int launch_apply(const qsi_op_s* op, const double* x, double* y,
                 const double* y_in, double yscale, double* dot_partials,
                 double* dot_out, hipStream_t s);
// as launch_apply, with the y_in scale multiplied by yscale_dev[0] (device)
int launch_apply_dev(const qsi_op_s* op, const double* x, double* y,
                     const double* y_in, double yscale,
                     const double* yscale_dev, double* dot_partials,
                     double* dot_out, hipStream_t s);
// as launch_apply_dev, with x read as xs_dev[0] * x and y_in as
// ys_dev[0] * y_in (either may be null: scale 1).  The products are the
// values a separate scaling pass would have stored, so the result has the
// same bits as applying to the scaled vectors.  Scales need dot_partials
// (only the dot-product kernel instances read them).
int launch_apply_scaled(const qsi_op_s* op, const double* x, double* y,
                        const double* y_in, double yscale, const double* yscale_dev,
                        const double* xs_dev, const double* ys_dev, double* dot_partials,
                        double* dot_out, hipStream_t s);
int64_t apply_num_blocks(const qsi_op_s* op);
// AUTO takes the wavefront-per-row kernel, which no other variant names
bool auto_takes_rows(const qsi_op_s* op);

// streaming vector kernels; partial buffers need max_vec_partials() doubles
// (gs_partials() for launch_gs_step)
int max_vec_partials();
int gs_partials(bool plain);
int launch_dot(const double* a, const double* b, int64_t n, double* partials,
               double* out, hipStream_t s);
int launch_axpy(double alpha, const double* x, double* y, int64_t n,
                hipStream_t s, const double* xs_dev = nullptr);
int launch_scal(double alpha, double* x, int64_t n, hipStream_t s);
// u -= alpha_dev[0] v; nrm_out[0] = ||u||, nrm_out[1] = 1/||u||; v is read as
// vs_dev[0] * v when vs_dev is given
int launch_axpy_norm(const double* alpha_dev, const double* v, double* u,
                     int64_t n, double* partials, double* nrm_out,
                     hipStream_t s, const double* vs_dev = nullptr);
// Classical Gram-Schmidt of w against V[:, 0:m] (column-major, ld ldv) in two
// passes and, when they leave |V^T w| > 1e-12 |w|, a third: hcol[0..m) receives
// the projections (the third pass's correction included), beta[0] = |w| at the
// end, beta[1] = 1 / beta[0] (0 if w vanishes), and w is scaled by beta[1].
// partials: gs_partials() doubles.  All on the device (no host
// synchronisation).  plain: the sums in kernels of their own, for operators that
// are not symmetric (their results at the restart limit depend on every rounding).
int launch_gs_step(const double* V, int64_t ldv, int m, double* w, int64_t n, double* partials,
                   double* hcol, double* beta, bool plain, hipStream_t s);
// out[j] = V[:, j] . w for j < m; partials: gs_partials(true) doubles
int launch_multidot(const double* V, int64_t ldv, int m, const double* w, int64_t n,
                    double* partials, double* out, hipStream_t s);

// Rayleigh-Ritz of n_jobs thick-restart Lanczos matrices of order m <= kRitzMax,
// one workgroup each.  Workgroup b takes job[b], whose kept[b] first vectors
// are Ritz vectors of the values theta[job * theta_stride + i] and whose column
// j >= kept[b] of projections starts at cols[job * job_stride + j * ldc].  It
// writes the ascending eigenvalues to theta (of the job) and out_theta
// (out_stride apart by workgroup), the eigenvectors to Y + job * y_stride
// (column-major m x m) and their last components to out_last.
constexpr int kRitzMax = 48;
struct RitzArgs {
  const double* cols;
  int64_t job_stride;
  int ldc;
  int m;
  double* theta;
  int64_t theta_stride;
  double* Y;
  int64_t y_stride;
  double* out_theta;
  double* out_last;
  int64_t out_stride;
  uint8_t job[64], kept[64];
};
int launch_ritz(const RitzArgs& a, int n_jobs, hipStream_t s);

// out[:, 0:k] = V[:, 0:m] Y  (Y m x k column-major, device)
int launch_combine(const double* V, int64_t ldv, int m, const double* Y, int k,
                   double* out, int64_t ldo, int64_t n, hipStream_t s);
int launch_randn(double* v, int64_t n, uint64_t seed, hipStream_t s);
int launch_copy_scaled(const double* s_dev, const double* y, double* x,
                       int64_t n, hipStream_t s);
// y += c * s_dev[0] * x
int launch_axpy_dev(const double* s_dev, double c, const double* x, double* y,
                    int64_t n, hipStream_t s);

// Psi[:, b] += c[b] * v for b < nb (c on the device; Psi column-major); v is
// read as vs_dev[0] * v when vs_dev is given
int launch_accum_cols(const double* v, double* Psi, int64_t ld, int nb, const double* c,
                      int64_t n, hipStream_t s, const double* vs_dev = nullptr);

// One of several operators applied together (device pointers of a qsi_op_s).
struct EachOp {
  const OffTerm* off;
  const DiagTerm* dg;
  int n_off;
  int n_diag;
  int col;  // first output column (k_observe)
};
// Y[:, l * n_vec + v] = O_l psi[:, v] (ops: n_ops records on the device; psi and
// Y column-major): one launch for many operators of a few terms each.
int launch_apply_each(const qsi_basis_s* basis, const EachOp* ops, int n_ops, const double* psi,
                      int64_t ld, int n_vec, double* Y, int64_t ldy, hipStream_t s);
// out[b * pa + a] = A[:, a] . B[:, b] over n rows (column-major); partials holds
// gram_partials() doubles, with same = (A is B).
size_t gram_partials(int pa, int pb, bool same, int64_t n);
int launch_gram(const double* A, int64_t lda, int pa, const double* B, int64_t ldb, int pb,
                int64_t n, double* partials, double* out, hipStream_t s);

// Expectations (same = 0: columns O_l psi_v against psi) or correlations (same
// = 1: against each other) of operators of a few terms without storing the
// columns: wavefront w of a workgroup forms the columns of list w.
struct ObserveArgs {
  const OffTerm* off;  // list by list, slot = the operator's first column
  const EachOp* diag;  // operators with diagonal terms, list by list
  const int* cols;     // columns, list by list
  int off_begin[5], diag_begin[5], col_begin[5];
  int P, n_vec, same, tiles;
};
bool observe_fits(const qsi_basis_s* basis, int P, int n_vec, bool gram);
int observe_blocks(int64_t n);
int observe_tiles(int P, bool gram);
// out[b * P + a] as launch_gram; partials: observe_blocks() * observe_tiles() * 256
int launch_observe(const qsi_basis_s* basis, const ObserveArgs& q, const double* psi, int64_t ld,
                   double* partials, double* out, hipStream_t s);

// The 3-term Lanczos coefficient run behind qsi_lanczos_coeffs on
// caller-provided device buffers: v (D, the start vector, normalised here;
// clobbered), u (D), partials (lanczos_coeffs_partials(op) doubles), ab
// (3 M doubles), scal (2 doubles).  Allocates nothing; synchronises.
int64_t lanczos_coeffs_partials(const qsi_op_s* op);
int lanczos_coeffs_run(const qsi_op_s* op, double* v, double* u, double* partials, double* ab,
                       double* scal, int M, double* h_alpha, double* h_beta, int* n_steps,
                       hipStream_t s);

}  // namespace qsi
