// Block Lanczos recurrences for many start vectors on several operators in
// one launch per kernel — the batched FTLM path.
//
// R start vectors per sector (operator + basis) run the reference's 3-term
// recurrence (components/linalg_routines/src/lanczos.cpp:111-146, without the
// convergence checks) side by side, M steps, no reorthogonalisation, which is
// what FTLM needs: the (alpha, beta) coefficients of every sample.  Sectors of
// different basis size share each launch: their rows are cut into tiles
// and one persistent grid of wavefronts walks the concatenated tile list, so
// each basis state's flip tests and rank lookups serve all R columns.
//
// Per step (three rotating D x R blocks holding v_{j-1}, v_j unnormalised,
// A = w_{j-1}, B = w_j with v = scale * column, and C):
//   k_blk_apply      C = H B, per-workgroup partials of <B_c, C_c>
//   k_blk_finalize   alpha[s][c] = scale_B^2 <B_c, C_c>
//   k_blk_update     C = scale_B (C - alpha B) - beta scale_A A, partials of |C_c|^2,
//                    history index += 1
//   k_blk_finalize   beta[s][c] = |C_c|, scale_C = 1/beta (0 when beta underflows);
//                    then (A, B, C) <- (B, C, A)
// No pass rewrites a block to normalise it.  The four launches of a step are
// captured once per rotation phase as a HIP graph and replayed.
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "qsi_blockk.hpp"
#include "qsi_hostla.hpp"

namespace qsi {
namespace {

__device__ __forceinline__ int find_sector(const BlkArgs& a, int64_t tile) {
  int s = 0;
  for (int k = 1; k < a.n_sec; ++k)
    if (tile >= a.sec[k].tile_begin) s = k;
  return s;
}

// Sum of v over the lanes that share this lane's column (lanes c, c+G, ...).
__device__ __forceinline__ double sum_over_groups(double v, int G) {
  for (int o = G; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

constexpr int kBlkVecBlocks = 2048;  // workgroups of a vector pass
// A tile is one wavefront's work.  With 64 rows each, a 48-spin sector (87 546
// rows) is 1368 wavefronts on 1024 SIMDs, each waiting for one gather after the
// other, so smaller bases are cut finer: down to the rows of one pass and no
// further than kTileRowsMin, until there are kBlkFill* tiles.  48 spins, cached:
// 16 columns 47 -> 24 us, 64 columns 169 -> 76 us; at 2.76 M rows the tiles stay
// whole.  The searching kernel finds the entries with one lane per row, so short
// tiles leave its lanes idle: 64 columns 195 us whole, 138 us cut for 4096 tiles,
// and a two-sector recurrence of 16 columns (131 us a step) takes 187 us when
// cut for 16384.
constexpr int kTileRowsMin = 8;
constexpr int64_t kBlkFillSearch = 4096, kBlkFillCached = 32768;
constexpr int kBlkCap = 1024;        // LDS flip entries per wavefront and round
constexpr int kBlkSuper = 256;       // off-diagonal terms per round (4 masks)
constexpr int kBlkBatch = 4;         // lookups in flight per lane (phase A)

__device__ __forceinline__ void blk_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Factor of a diagonal term on state s, without its coefficient.
template <int NW>
__device__ __forceinline__ double diag_factor(const DiagTerm& d, const State<NW>& s) {
  if (d.kind == 0) return diag_ok<NW>(d, s) ? d.sgn * (1 - 2 * parity_notz<NW>(s, d.Z)) : 0.0;
  int nz = __popcll(d.Z[0]);
  if constexpr (NW == 2) nz += __popcll(d.Z[1]);
  return d.sgn * static_cast<double>(2 * popc_and<NW>(s, d.Z) - nz);
}

// CPL neighbouring columns of one row of X or of the coefficient table (8-byte
// aligned; two columns are one 16-byte load).
template <int CPL>
struct ColVec {
  double v[CPL];
};
template <int CPL>
__device__ __forceinline__ ColVec<CPL> load_cols(const double* p) {
  ColVec<CPL> r;
  __builtin_memcpy(&r, p, sizeof(r));
  return r;
}

// A wavefront's place in a row-major block: G lanes per row, CPL neighbouring
// columns each (R >= CPL).  The last columns, where CPL does not divide R, are
// computed by a lane that also reads the columns before them and leaves those
// alone, so every load stays inside its row.
template <int CPL>
struct ColLane {
  int grp;    // row within the pass
  int col;    // first column it reads
  int skip;   // leading columns that another lane writes
  int rpp;    // rows per pass
  bool ok;    // it has a column and a row
  __device__ __forceinline__ ColLane(int lane, int G, int R) {
    grp = lane / G;
    rpp = 64 / G;
    const int c = CPL * (lane % G);
    ok = c < R && grp < rpp;
    col = CPL == 1 ? (ok ? c : 0) : max(0, min(c, R - CPL));
    skip = CPL == 1 ? 0 : (ok ? c - col : 0);
  }
};

// out[c] = the workgroup's sum of column c's v: over the row groups by
// butterfly (G a power of two), over the wavefronts in order through LDS.
// Every thread of the workgroup calls it.
template <int CPL>
__device__ __forceinline__ void store_partials(double (&red)[kBlkWaves][64], const ColLane<CPL>& q,
                                               int G, int R, const ColVec<CPL>& v,
                                               double* __restrict__ out) {
#pragma unroll
  for (int u = 0; u < CPL; ++u) {
    const double t = sum_over_groups(v.v[u], G);
    if (q.grp == 0 && q.ok && u >= q.skip) red[threadIdx.x >> 6][q.col + u] = t;
  }
  __syncthreads();
  if (static_cast<int>(threadIdx.x) < R) {
    double t = red[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kBlkWaves; ++w) t += red[w][threadIdx.x];
    out[threadIdx.x] = t;
  }
  __syncthreads();
}

// coef[k][c] = column c's coefficient of class k, by the whole workgroup.
__device__ __forceinline__ void load_coefs(double (&coef)[kMaxCoefClasses][64], const BlkSector& S,
                                           int R) {
  for (int e = threadIdx.x; e < S.n_cls * R; e += kBlkThreads) {
    const CoefClass& K = S.cls[e / R];
    coef[e / R][e % R] = (S.coeffs && K.slot >= 0) ? S.coeffs[K.slot * R + e % R] : K.c;
  }
}

// Y[:, c] = H_c X[:, c] (or Y += H_c X) for R columns of row-major blocks,
// and (partials != null) per-workgroup, per-sector partials of
// <X[:, c], Y[:, c]>.
//
// Each wavefront takes a tile of up to 64 rows in two phases per round:
//   A  one lane per row finds the row's connected terms, looks up the
//      pre-image ranks BATCH at a time and writes (rank, term or class, sign)
//      entries to LDS in term order; the lookup keys are the row's bucket key
//      and state XOR the flip's, staged in LDS;
//   B  G lanes per row, CPL columns each, walk the row's entries and read X's
//      row as one coalesced segment per connected state, kPipe entries in
//      flight.
// A round covers up to kBlkSuper terms and as many rows as fit kBlkCap LDS
// entries (a whole tile on the lattices up to 72 spins: half as many entries
// cut most tiles in two, and a round's phase A runs half empty); partial sums
// of rows cut by a round boundary go through Y.  The classes' column
// coefficients are read from LDS, one copy per workgroup: the tiles of a
// workgroup's wavefronts are neighbours, and sectors start at multiples of
// kBlkWaves tiles, so all its wavefronts are in one sector at a time.
// Contributions are added in term order, then the diagonal terms in order, so
// column c's result depends only on X[:, c] and its coefficients.
//
// Bound: phase A is the lookups of a single-vector apply (one column: 366 us
// at 64 spins, 2.76 M rows, where that apply takes 266), phase B the gather of
// X's rows through the L2 misses.  64 spins, 1 / 7 / 16 / 64 columns, one
// (g, B) each: 0.37 / 0.64 / 0.98 / 3.1 ms; 2.00 ms for seven columns when the
// flip tests' term loads were vector loads (they alone took 300 us), a round
// held 512 entries, a lane had one column and chose its coefficient in
// registers.  Four wavefronts per SIMD: with five, the LDS of one workgroup
// more does not fit and a persistent grid leaves a second wave of workgroups;
// six at 768 entries a round takes 0.75 ms for seven columns.
template <int NW, int BATCH, int CPL>
__global__ __launch_bounds__(kBlkThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_blk_apply(
    BlkArgs a, const double* __restrict__ X, double* __restrict__ Y,
    double* __restrict__ partials) {
  constexpr int kPipe = 6;
  // entry: rank (kNoRank if absent); class, or term - round base without
  // classes (bits 0-7), total sign negative (bit 8)
  __shared__ uint32_t lds_rank[kBlkWaves][kBlkCap];
  __shared__ uint16_t lds_meta[kBlkWaves][kBlkCap];
  __shared__ double coef[kMaxCoefClasses][64];
  // flip masks, and bucket keys with class and sign, of the sector's first
  // kBlkSuper terms (later ones are read from the planes)
  __shared__ uint64_t flip[NW][kBlkSuper];
  __shared__ uint64_t tkey[kBlkSuper];
  const int lane = threadIdx.x & 63;
  // wave-uniform values kept in scalar registers
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t* ent = lds_rank[wv];
  uint16_t* met = lds_meta[wv];
  __shared__ double red[kBlkWaves][64];
  const int G = a.G, R = a.R;
  const ColLane<CPL> q(lane, G, R);
  const int grp = q.grp, col = q.col, skip = q.skip, rpp = q.rpp;
  const bool col_ok = q.ok;
  const int64_t n_waves = static_cast<int64_t>(gridDim.x) * kBlkWaves;
  // tiles are visited in increasing order, so sectors come in order: one
  // running dot product, flushed when the workgroup's sector changes
  ColVec<CPL> dot{};
  int flushed = 0;  // sectors [0, flushed) have their partial written
  auto flush_to = [&](int upto, int cur) {
    for (; partials && flushed < upto; ++flushed)
      store_partials(red, q, G, R, flushed == cur ? dot : ColVec<CPL>{},
                     partials + (static_cast<int64_t>(flushed) * gridDim.x + blockIdx.x) * R);
  };
  int cur = -1;
  for (int64_t tb0 = static_cast<int64_t>(blockIdx.x) * kBlkWaves; tb0 < a.n_tiles;
       tb0 += n_waves) {
    const int s = __builtin_amdgcn_readfirstlane(find_sector(a, tb0));  // the workgroup's
    const BlkSector& S = a.sec[s];
    // the rows' states are on their way while the sector's terms are staged
    const int64_t t = tb0 + wv;
    const int64_t r_begin = (t - S.tile_begin) * a.tile_rows;
    const int n_rows = static_cast<int>(min<int64_t>(a.tile_rows, S.b.dim - r_begin));
    const bool live = t < a.n_tiles && n_rows > 0;  // not a padding tile
    const bool row_ok = live && lane < n_rows;
    const State<NW> st = load_state_cached<NW>(S.b.states, row_ok ? r_begin + lane : 0);
    if (s != cur) {
      flush_to(s, cur);
      cur = s;
      dot = ColVec<CPL>{};
      __syncthreads();  // no wavefront still reads the last sector's
      load_coefs(coef, S, R);
      for (int e = threadIdx.x; e < min(S.n_off, kBlkSuper); e += kBlkThreads) {
#pragma unroll
        for (int w = 0; w < NW; ++w) flip[w][e] = S.tp.X(w)[e];
        tkey[e] = S.tp.key()[e];
      }
      __syncthreads();
    }
    if (!live) continue;
    const uint32_t ks = bucket_key<NW>(S.b, st);
    const int n_sc = max(1, (S.n_off + kBlkSuper - 1) / kBlkSuper);
    for (int sc = 0; sc < n_sc; ++sc) {
      const int tb = sc * kBlkSuper;
      const int tn = min(kBlkSuper, S.n_off - tb);
      // connected terms of this lane's row: term tb + 64 q + u at bit 63 - u
      uint64_t conn[4];
      int cnt = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int qn = min(64, tn - q * 64);
        conn[q] = qn > 0 ? connect_mask<NW>(S.off + tb + q * 64, qn, st) : 0;
        if (!row_ok) conn[q] = 0;
        cnt += __popcll(conn[q]);
      }
      int incl = cnt;
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      const int excl = incl - cnt;
      for (int ra = 0; ra < 64;) {
        const int base = __shfl(excl, ra, 64);
        const uint64_t fits = __ballot(lane >= ra && incl - base <= kBlkCap);
        const int rb = ra + __popcll(fits);  // >= ra + 1: cnt <= kBlkSuper <= kBlkCap
        // phase A: this lane's connected terms, in term order
        if (lane >= ra && lane < rb && cnt > 0) {
          int pos = excl - base;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            uint64_t m = conn[q];
            while (m) {
              State<NW> key[BATCH];
              uint32_t bk[BATCH], cs[BATCH];
              bool act[BATCH];
              int tl[BATCH];
              uint32_t rk[BATCH];
#pragma unroll
              for (int g = 0; g < BATCH; ++g) {
                act[g] = m != 0;
                const int z = act[g] ? __builtin_clzll(m) : 0;
                tl[g] = q * 64 + z;
                m &= ~(uint64_t{1} << 63 >> z);
#pragma unroll
                for (int w = 0; w < NW; ++w)
                  key[g].w[w] = st.w[w] ^ (sc == 0 ? flip[w][tl[g]] : S.tp.X(w)[tb + tl[g]]);
                const uint64_t k = sc == 0 ? tkey[tl[g]] : S.tp.key()[tb + tl[g]];
                bk[g] = ks ^ static_cast<uint32_t>(k);
                cs[g] = static_cast<uint32_t>(k >> 32);
              }
              lookup_batch_at<NW, BATCH>(S.b, key, bk, act, rk);
#pragma unroll
              for (int g = 0; g < BATCH; ++g) {
                if (act[g]) {
                  bool ng = cs[g] & TermPlanes::kNegative;
                  if (cs[g] & TermPlanes::kHasZ)
                    ng ^= parity_notz<NW>(st, S.off[tb + tl[g]].Z) != 0;
                  ent[pos] = rk[g];
                  met[pos] = static_cast<uint16_t>((S.n_cls > 0 ? cs[g] & 255 : tl[g]) |
                                                   (ng ? 256 : 0));
                  ++pos;
                }
              }
            }
          }
        }
        blk_wave_sync();
        // phase B: G lanes per row
        const int n_pass = (rb - ra + rpp - 1) / rpp;
        for (int p = 0; p < n_pass; ++p) {
          const int r = ra + p * rpp + grp;
          const int rs = min(r, 63);
          const int e0 = __shfl(excl, rs, 64) - base;
          const int e1 = __shfl(incl, rs, 64) - base;
          if (r < rb && r < n_rows && col_ok) {
            const int64_t row = S.row_off + r_begin + r;
            double* yp[CPL];
            ColVec<CPL> acc;
#pragma unroll
            for (int u = 0; u < CPL; ++u) {
              yp[u] = Y + (a.y_colmajor ? (col + u) * a.ldy + row : row * a.ldy + col + u);
              acc.v[u] = (sc > 0 || a.accumulate) && u >= skip ? *yp[u] : 0.0;
            }
            for (int e = e0; e < e1; e += kPipe) {
              uint32_t J[kPipe];
              uint32_t mt[kPipe];
              ColVec<CPL> xj[kPipe];
#pragma unroll
              for (int u = 0; u < kPipe; ++u) {
                J[u] = e + u < e1 ? ent[e + u] : kNoRank;
                mt[u] = e + u < e1 ? met[e + u] : 0u;
              }
#pragma unroll
              for (int u = 0; u < kPipe; ++u)
                xj[u] = J[u] != kNoRank
                            ? load_cols<CPL>(X + (S.row_off + static_cast<int64_t>(J[u])) * a.ldx + col)
                            : ColVec<CPL>{};
              auto add = [&](int u, const ColVec<CPL>& c) {
#pragma unroll
                for (int v = 0; v < CPL; ++v)
                  if (fabs(xj[u].v[v]) > kApplyTol)
                    acc.v[v] += (mt[u] & 256 ? -c.v[v] : c.v[v]) * xj[u].v[v];
              };
              auto own = [&](int u) {  // the coefficient of the entry's own term
                const OffTerm& T = S.off[tb + static_cast<int>(mt[u] & 255)];
                ColVec<CPL> c;
#pragma unroll
                for (int v = 0; v < CPL; ++v)
                  c.v[v] = (S.coeffs && T.slot >= 0) ? S.coeffs[T.slot * R + col + v] : T.c;
                return c;
              };
              auto classed = [&](int u) { return load_cols<CPL>(&coef[mt[u] & 255][col]); };
              if constexpr (CPL > 1) {
#pragma unroll
                for (int u = 0; u < kPipe; ++u)
                  if (J[u] != kNoRank) add(u, S.n_cls > 0 ? classed(u) : own(u));
              } else if (S.n_cls > 0) {
#pragma unroll
                for (int u = 0; u < kPipe; ++u)
                  if (J[u] != kNoRank) add(u, classed(u));
              } else {
                // all of them before the first is used (12.8 -> 11.7 us for one
                // column of 4096 rows; two columns per lane cost registers that
                // the coefficient classes miss: 642 -> 652 us for seven)
                ColVec<CPL> c[kPipe];
#pragma unroll
                for (int u = 0; u < kPipe; ++u) c[u] = own(u);
#pragma unroll
                for (int u = 0; u < kPipe; ++u)
                  if (J[u] != kNoRank) add(u, c[u]);
              }
            }
            if (sc == n_sc - 1) {
              const State<NW> sr = load_state_cached<NW>(S.b.states, r_begin + r);
              const ColVec<CPL> xi = load_cols<CPL>(X + row * a.ldx + col);
              for (int k = 0; k < S.n_diag; ++k) {
                const DiagTerm d = const_load(S.dg + k);
                const double f = diag_factor<NW>(d, sr);
#pragma unroll
                for (int v = 0; v < CPL; ++v) {
                  const double c =
                      (S.coeffs && d.slot >= 0) ? S.coeffs[d.slot * R + col + v] : d.c;
                  acc.v[v] += c * xi.v[v] * f;
                }
              }
#pragma unroll
              for (int v = 0; v < CPL; ++v) dot.v[v] += xi.v[v] * acc.v[v];
            }
#pragma unroll
            for (int v = 0; v < CPL; ++v)
              if (v >= skip) *yp[v] = acc.v[v];
          }
        }
        blk_wave_sync();
        ra = rb;
      }
    }
  }
  flush_to(a.n_sec, cur);
}

// ---- cached connectivity ---------------------------------------------------
// Rows' connected states are fixed by the basis and the term list, so an
// operator applied many times (a solve engine, an FTLM run) can keep them:
// per row, in term order, the rank J (kNoRank if absent) and one byte
// (coefficient class | negative total sign << 7).  A block apply is then a
// pure gather: no flip tests, no searches.

// counts[i] = number of connected off-diagonal terms of row i, rounded up to
// a multiple of `pad` (1 or 4: rows padded to whole groups of four entries).
template <int NW>
__global__ __launch_bounds__(256) void k_cc_count(BasisView b, const OffTerm* __restrict__ off,
                                                  int n_off, int pad,
                                                  uint64_t* __restrict__ counts) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= b.dim) return;
  const State<NW> st = load_state_cached<NW>(b.states, i);
  uint64_t n = 0;
  for (int t = 0; t < n_off; ++t) n += term_ok<NW>(off[t], st) ? 1u : 0u;
  counts[i] = (n + pad - 1) / pad * pad;
}

// Entries of row i at rowptr[i]...: ranks looked up kBlkBatch at a time.
template <int NW>
__global__ __launch_bounds__(256) void k_cc_fill(BasisView b, const OffTerm* __restrict__ off,
                                                 int n_off, const uint64_t* __restrict__ rowptr,
                                                 uint32_t* __restrict__ cj,
                                                 uint8_t* __restrict__ cm) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= b.dim) return;
  const State<NW> st = load_state_cached<NW>(b.states, i);
  uint64_t pos = rowptr[i];
  for (int t0 = 0; t0 < n_off; t0 += 64) {
    const int tn = min(64, n_off - t0);
    uint64_t m = 0;
    for (int u = 0; u < tn; ++u)
      m |= static_cast<uint64_t>(term_ok<NW>(off[t0 + u], st)) << u;
    while (m) {
      State<NW> key[kBlkBatch];
      bool act[kBlkBatch];
      int tt[kBlkBatch];
      uint32_t rk[kBlkBatch];
#pragma unroll
      for (int g = 0; g < kBlkBatch; ++g) {
        act[g] = m != 0;
        tt[g] = t0 + (act[g] ? __builtin_ctzll(m) : 0);
        m &= m - 1;
        key[g] = xor_state<NW>(st, off[tt[g]].X);
      }
      lookup_batch<NW, kBlkBatch>(b, key, act, rk);
#pragma unroll
      for (int g = 0; g < kBlkBatch; ++g) {
        if (act[g]) {
          const OffTerm& T = off[tt[g]];
          const bool ng = (T.sgn < 0.0) != static_cast<bool>(parity_notz<NW>(st, T.Z));
          cj[pos] = rk[g];
          cm[pos] = static_cast<uint8_t>((T.cls & 0x7F) | (ng ? 0x80 : 0));
          ++pos;
        }
      }
    }
  }
  // padding entries (padded layout): absent, so every apply skips them
  for (const uint64_t end = rowptr[i + 1]; pos < end; ++pos) {
    cj[pos] = kNoRank;
    cm[pos] = 0;
  }
}

// PIPE entries of a row's cached connectivity from entry e (a multiple of 4):
// columns four at a time with one 16-byte load, class bytes with one 4-byte
// load (the arrays are allocated in whole groups); entries outside the row
// [e0, e1) read as absent.
template <int PIPE>
__device__ __forceinline__ void load_entries(const BlkSector& S, uint64_t e, uint64_t e0,
                                             uint64_t e1, uint32_t (&J)[PIPE],
                                             uint8_t (&mt)[PIPE]) {
  static_assert(PIPE % 4 == 0, "groups of four");
#pragma unroll
  for (int u = 0; u < PIPE; u += 4) {
    const uint64_t g = e + u;
    const bool in = g < e1;
    const uint4 j4 = in ? reinterpret_cast<const uint4*>(S.cj)[g >> 2]
                       : make_uint4(kNoRank, kNoRank, kNoRank, kNoRank);
    const uint32_t m4 = in ? reinterpret_cast<const uint32_t*>(S.cm)[g >> 2] : 0u;
    const uint32_t jv[4] = {j4.x, j4.y, j4.z, j4.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool mine = g + k >= e0 && g + k < e1;
      J[u + k] = mine ? jv[k] : kNoRank;
      mt[u + k] = static_cast<uint8_t>(m4 >> (8 * k));
    }
  }
}

// The block apply over cached connectivity: same arithmetic, order and
// results as k_blk_apply.  G lanes per row, CPL columns each (blk_cpl), PIPE entries'
// gathers in flight.  G may be any width up to 64 when no partials are asked
// for (a wavefront then serves floor(64 / G) rows per pass); with partials it
// must be a power of two (the per-column sums cross row groups by butterfly).
// The class's coefficients come from LDS: one read of CPL columns instead of a
// choice among eight registers per column and entry (2.76 M rows of 64 spins, 16
// columns in pairs 0.87 -> 0.68 ms, 64 columns 3.4 -> 2.7 ms; then bound by the
// gathers' L2 misses, 15.5 GB of X's rows at 5.7 TB/s).  One column per lane keeps
// the choice, where an LDS read per entry serves one product (64 spins, 3 / 8 / 16
// columns: 270 / 486 / 920 us, from LDS 309 / 572 / 1008).
template <int NW, int PIPE, int CPL>
__global__ __launch_bounds__(kBlkThreads) void k_blk_capply(
    BlkArgs a, const double* __restrict__ X, double* __restrict__ Y,
    double* __restrict__ partials) {
  __shared__ double coef[kMaxCoefClasses][64];
  __shared__ double red[kBlkWaves][64];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.G, R = a.R;
  const ColLane<CPL> q(lane, G, R);
  const int col = q.col;
  const int64_t n_waves = static_cast<int64_t>(gridDim.x) * kBlkWaves;
  ColVec<CPL> dot{};
  int flushed = 0;
  auto flush_to = [&](int upto, int cur) {
    for (; partials && flushed < upto; ++flushed)
      store_partials(red, q, G, R, flushed == cur ? dot : ColVec<CPL>{},
                     partials + (static_cast<int64_t>(flushed) * gridDim.x + blockIdx.x) * R);
  };
  int cur = -1;
  double cc[kMaxCoefClasses];  // this lane's column (CPL == 1)
  for (int64_t tb0 = static_cast<int64_t>(blockIdx.x) * kBlkWaves; tb0 < a.n_tiles;
       tb0 += n_waves) {
    const int s = __builtin_amdgcn_readfirstlane(find_sector(a, tb0));  // the workgroup's
    const BlkSector& S = a.sec[s];
    if (s != cur) {
      flush_to(s, cur);
      cur = s;
      dot = ColVec<CPL>{};
      __syncthreads();  // no wavefront still reads the last sector's
      load_coefs(coef, S, R);
      __syncthreads();
      if constexpr (CPL == 1) {
#pragma unroll
        for (int c = 0; c < kMaxCoefClasses; ++c) cc[c] = c < S.n_cls ? coef[c][q.col] : 0.0;
      }
    }
    const int64_t t = tb0 + wv;
    const int64_t r_begin = (t - S.tile_begin) * a.tile_rows;
    const int n_rows = static_cast<int>(min<int64_t>(a.tile_rows, S.b.dim - r_begin));
    if (t >= a.n_tiles || n_rows <= 0 || !q.ok) continue;  // padding tiles
    for (int r = q.grp; r < n_rows; r += q.rpp) {
      const int64_t i = r_begin + r;
      const int64_t row = S.row_off + i;
      double* yp[CPL];
      ColVec<CPL> acc;
#pragma unroll
      for (int u = 0; u < CPL; ++u) {
        yp[u] = Y + (a.y_colmajor ? (col + u) * a.ldy + row : row * a.ldy + col + u);
        acc.v[u] = a.accumulate && u >= q.skip ? *yp[u] : 0.0;
      }
      const uint64_t e0 = S.rowptr[i], e1 = S.rowptr[i + 1];
      for (uint64_t e = e0 & ~uint64_t{3}; e < e1; e += PIPE) {
        uint32_t J[PIPE];
        uint8_t mt[PIPE];
        ColVec<CPL> xj[PIPE];
        load_entries<PIPE>(S, e, e0, e1, J, mt);
#pragma unroll
        for (int u = 0; u < PIPE; ++u)
          xj[u] = J[u] != kNoRank
                      ? load_cols<CPL>(X + (S.row_off + static_cast<int64_t>(J[u])) * a.ldx + col)
                      : ColVec<CPL>{};
#pragma unroll
        for (int u = 0; u < PIPE; ++u) {
          if (J[u] == kNoRank) continue;
          ColVec<CPL> c;
          if constexpr (CPL == 1) {
            c.v[0] = cc[0];
#pragma unroll
            for (int z = 1; z < kMaxCoefClasses; ++z)
              if ((mt[u] & 0x7F) == z) c.v[0] = cc[z];
          } else {
            c = load_cols<CPL>(&coef[mt[u] & 0x7F][col]);
          }
#pragma unroll
          for (int v = 0; v < CPL; ++v)
            if (fabs(xj[u].v[v]) > kApplyTol)
              acc.v[v] += (mt[u] & 0x80 ? -c.v[v] : c.v[v]) * xj[u].v[v];
        }
      }
      const State<NW> sr = load_state_cached<NW>(S.b.states, i);
      const ColVec<CPL> xi = load_cols<CPL>(X + row * a.ldx + col);
      for (int k = 0; k < S.n_diag; ++k) {
        const DiagTerm d = const_load(S.dg + k);
        const double f = diag_factor<NW>(d, sr);
#pragma unroll
        for (int v = 0; v < CPL; ++v) {
          const double c = (S.coeffs && d.slot >= 0) ? S.coeffs[d.slot * R + col + v] : d.c;
          acc.v[v] += c * xi.v[v] * f;
        }
      }
#pragma unroll
      for (int v = 0; v < CPL; ++v) {
        dot.v[v] += xi.v[v] * acc.v[v];
        if (v >= q.skip) *yp[v] = acc.v[v];
      }
    }
  }
  flush_to(a.n_sec, cur);
}

// C = fb C - alpha fb B - beta fa A per column (fb, fa: the scales sB, sA of
// the unnormalised blocks B and A, 1 when null; beta, A skipped when A is
// null); |C_c|^2 partials per workgroup and sector.  Advances step (if given).
__global__ __launch_bounds__(kBlkThreads) void k_blk_update(
    BlkArgs a, const double* __restrict__ A, const double* B,
    double* C, const double* __restrict__ alpha,
    const double* __restrict__ beta, double* __restrict__ partials,
    const double* __restrict__ sA, const double* __restrict__ sB, int* __restrict__ step) {
  __shared__ double red[kBlkWaves][64];
  const int G = a.G, R = a.R;
  const ColLane<1> q(threadIdx.x & 63, G, R);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n_waves = static_cast<int64_t>(gridDim.x) * kBlkWaves;
  ColVec<1> nrm{};
  int flushed = 0;
  auto flush_to = [&](int upto, int cur) {
    for (; flushed < upto; ++flushed)
      store_partials(red, q, G, R, flushed == cur ? nrm : ColVec<1>{},
                     partials + (static_cast<int64_t>(flushed) * gridDim.x + blockIdx.x) * R);
  };
  int cur = -1;
  for (int64_t tb0 = static_cast<int64_t>(blockIdx.x) * kBlkWaves; tb0 < a.n_tiles;
       tb0 += n_waves) {
    const int s = __builtin_amdgcn_readfirstlane(find_sector(a, tb0));  // the workgroup's
    const BlkSector& S = a.sec[s];
    if (s != cur) {
      flush_to(s, cur);
      cur = s;
      nrm = ColVec<1>{};
    }
    const int64_t t = tb0 + wv;
    if (t >= a.n_tiles || !q.ok) continue;
    const int64_t r_begin = (t - S.tile_begin) * a.tile_rows;
    const int n_rows = static_cast<int>(min<int64_t>(a.tile_rows, S.b.dim - r_begin));
    // the tile's elements, as uniform bases and 32-bit offsets
    const int64_t base = (S.row_off + r_begin) * R;
    double* Ct = C + base;
    const double* Bt = B + base;
    const double* At = A ? A + base : nullptr;
    const double al = alpha ? alpha[s * R + q.col] : 0.0;
    const double be = A ? beta[s * R + q.col] : 0.0;
    // the blocks hold unnormalised vectors: v_B = fb B, v_A = fa A, and C
    // holds H B, so H v_B = fb C
    const double fb = sB ? sB[s * R + q.col] : 1.0;
    const double fa = sA ? sA[s * R + q.col] : 1.0;
    const double alb = al * fb, bea = be * fa;
    // eight rows per round: their loads are issued together; the norm is
    // still accumulated row by row in order
    constexpr int kU = 8;
    for (int i0 = q.grp; i0 < n_rows; i0 += kU * q.rpp) {
      double cv[kU], bv[kU], av[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int i = i0 + u * q.rpp;
        const uint32_t gi = i * R + q.col;
        const bool in = i < n_rows;
        cv[u] = in ? Ct[gi] : 0.0;
        bv[u] = in ? Bt[gi] : 0.0;
        av[u] = in && A ? At[gi] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int i = i0 + u * q.rpp;
        if (i >= n_rows) continue;
        const uint32_t gi = i * R + q.col;
        double w = fb * cv[u] - alb * bv[u];
        if (A) w -= bea * av[u];
        if (fb == 0.0) w = 0.0;  // a column whose beta underflowed stays zero
        Ct[gi] = w;
        nrm.v[0] += w * w;
      }
    }
  }
  flush_to(a.n_sec, cur);
  if (step && blockIdx.x == 0 && threadIdx.x == 0) step[0] += 1;
}

// Fixed-order sums of the workgroups' partials, kFinCols columns of one sector
// per workgroup (grid: ceil(R / kFinCols) x sectors): neighbouring threads read
// neighbouring columns, and a workgroup's loads are in flight together (1024
// partials of two sectors and 64 columns: 5.8 us, 10 us with a workgroup per
// column and a partial per wavefront).
// mode 0 (alpha): out[s*R+c] = sum, times sq[s*R+c]^2 when sq is given.  mode 1
// (beta): out[s*R+c] = sqrt(sum), out2[s*R+c] = 1/beta or 0.  hist (optional) receives the value at
// hist[(s*R + c)*M + step[0] - back].
constexpr int kFinCols = 8;
constexpr int kFinThreads = 1024;
__global__ __launch_bounds__(kFinThreads) void k_blk_finalize(
    const double* __restrict__ partials, int n_blocks, int R, int mode,
    double* __restrict__ out, double* __restrict__ out2, double* __restrict__ hist,
    const int* __restrict__ step, int back, int M, const double* __restrict__ sq) {
  constexpr int kRows = kFinThreads / kFinCols;
  __shared__ double red[kRows][kFinCols];
  const int s = blockIdx.y;
  const int u = threadIdx.x % kFinCols, g = threadIdx.x / kFinCols;
  const int c = blockIdx.x * kFinCols + u;
  double v = 0.0;
  if (c < R) {
    const double* p = partials + static_cast<int64_t>(s) * n_blocks * R + c;
#pragma unroll 8
    for (int w = g; w < n_blocks; w += kRows) v += p[static_cast<int64_t>(w) * R];
  }
  red[g][u] = v;
  for (int h = kRows / 2; h > 0; h >>= 1) {
    __syncthreads();
    if (g < h) red[g][u] += red[g + h][u];
  }
  if (g == 0 && c < R) {
    const int sc = s * R + c;
    double r = red[0][u];
    if (mode == 0 && sq) r = r * sq[sc] * sq[sc];
    if (mode == 1) {
      r = sqrt(r);
      out2[sc] = r > 1e-300 ? 1.0 / r : 0.0;
    }
    out[sc] = r;
    if (hist) hist[static_cast<int64_t>(sc) * M + step[0] - back] = r;
  }
}

// C *= 1/beta per (sector, column).
__global__ __launch_bounds__(kBlkThreads) void k_blk_scale(
    BlkArgs a, double* __restrict__ C, const double* __restrict__ invb) {
  const int lane = threadIdx.x & 63;
  const int G = a.G, R = a.R;
  const int grp = lane / G, col = lane % G;
  const bool col_ok = col < R;
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * kBlkWaves + (threadIdx.x >> 6);
  const int64_t n_waves = static_cast<int64_t>(gridDim.x) * kBlkWaves;
  const int rows_per_pass = 64 / G;
  for (int64_t t = wave; t < a.n_tiles; t += n_waves) {
    const int s = find_sector(a, t);
    const BlkSector& S = a.sec[s];
    const int64_t r_begin = (t - S.tile_begin) * a.tile_rows;
    const int64_t r_end = min<int64_t>(r_begin + a.tile_rows, S.b.dim);
    if (!col_ok) continue;
    const double f = invb[s * R + col];
    constexpr int kU = 8;
    for (int64_t i0 = r_begin + grp; i0 < r_end; i0 += kU * rows_per_pass) {
      double cv[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int64_t i = i0 + u * rows_per_pass;
        cv[u] = i < r_end ? C[(S.row_off + i) * R + col] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int64_t i = i0 + u * rows_per_pass;
        if (i < r_end) C[(S.row_off + i) * R + col] = cv[u] * f;
      }
    }
  }
}

struct DevMem {
  std::vector<void*> ptrs;
  ~DevMem() {
    for (void* p : ptrs) (void)hipFree(p);
  }
  template <typename T>
  hipError_t alloc(T** p, size_t n) {
    void* q = nullptr;
    hipError_t e = hipMalloc(&q, std::max<size_t>(n * sizeof(T), 8));
    if (e == hipSuccess) {
      ptrs.push_back(q);
      *p = static_cast<T*>(q);
    }
    return e;
  }
};

}  // namespace

namespace {

using BlkKernel = void (*)(BlkArgs, const double*, double*, double*);

// Block-apply kernel of a configuration: cached kernels by gathers in flight
// (4, 8, 16; half as many of four columns), searching kernels by lookups in
// flight (6 or 4 by the state's words; 2); cpl columns per lane (blk_cpl).
template <int CPL>
BlkKernel cached_kernel(int nw, int k) {
  constexpr int P8 = CPL == 4 ? 4 : 8, P16 = CPL == 4 ? 8 : 16;
  if (nw == 1)
    return k == 0 ? k_blk_capply<1, 4, CPL>
                  : (k == 2 ? k_blk_capply<1, P16, CPL> : k_blk_capply<1, P8, CPL>);
  return k == 0 ? k_blk_capply<2, 4, CPL>
                : (k == 2 ? k_blk_capply<2, P16, CPL> : k_blk_capply<2, P8, CPL>);
}
template <int CPL>
BlkKernel search_kernel(int nw, int k) {
  if (nw == 1) return k == 2 ? k_blk_apply<1, 2, CPL> : k_blk_apply<1, 6, CPL>;
  return k == 2 ? k_blk_apply<2, 2, CPL> : k_blk_apply<2, 4, CPL>;
}
BlkKernel blk_kernel(int nw, bool cached, int cfg, int cpl) {
  const int k = blk_cfg_kernel(cfg);
  if (!cached) return cpl == 1 ? search_kernel<1>(nw, k) : search_kernel<2>(nw, k);
  return cpl == 1   ? cached_kernel<1>(nw, k)
         : cpl == 2 ? cached_kernel<2>(nw, k)
                    : cached_kernel<4>(nw, k);
}

}  // namespace

int blk_cpl(const BlkArgs& a) {
  const bool cached = blk_cached(a);
  if (a.R < 2 || (cached && !blk_cfg_pairs(a.cfg))) return 1;
  // Four columns per lane halve the instructions per entry and column, and
  // with them the wavefronts that share a row: worth it from 12 columns on,
  // where enough passes of 64 lanes are left to fill the chip (64 columns of
  // 2.76 M, 87 546 rows: 2.75 -> 2.55 ms, 77 -> 68 us; but 16 columns of 87 546
  // rows 24 -> 30 us, 8 columns of 2.76 M 410 -> 421 us).
  int64_t rows = 0;
  for (int s = 0; s < a.n_sec; ++s) rows += a.sec[s].b.dim;
  return cached && a.R >= 12 && rows * a.R >= int64_t{1} << 22 ? 4 : 2;
}

void blk_set_tiles(BlkArgs& a) {
  int64_t rows = 0;
  for (int s = 0; s < a.n_sec; ++s) rows += a.sec[s].b.dim;
  // rows of one pass of a wavefront, at most
  const int pass = a.R >= 2 ? std::min(64, 128 / a.G) : 64 / a.G;
  a.tile_rows = kTileRows;
  const int64_t fill = blk_cached(a) ? kBlkFillCached : kBlkFillSearch;
  while (a.tile_rows > std::max(pass, kTileRowsMin) && rows < fill * a.tile_rows) a.tile_rows /= 2;
  int64_t tiles = 0;
  for (int s = 0; s < a.n_sec; ++s) {
    a.sec[s].tile_begin = tiles;
    // whole workgroups of tiles (the last ones may be empty)
    const int64_t wg = static_cast<int64_t>(a.tile_rows) * kBlkWaves;
    tiles += (a.sec[s].b.dim + wg - 1) / wg * kBlkWaves;
  }
  a.n_tiles = tiles;
}

int blk_apply_blocks(const BlkArgs& a, int nw) {
  const bool cached = blk_cached(a);
  const int cpl = blk_cpl(a), cfg = a.cfg;
  // resident blocks per CU of each kernel: [cached][nw - 1][kernel][columns per lane];
  // atomics, as host threads may launch concurrently (they store equal
  // values).  The CU count is a function-local static, whose initialisation
  // is thread-safe, so no thread can see an occupancy without it.
  static std::atomic<int> per_cu[2][2][3][5];
  static const int n_cu = [] {
    int dev = 0, cu = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cu <= 0)
      cu = 256;
    return cu;
  }();
  std::atomic<int>& occ = per_cu[cached ? 1 : 0][nw - 1][blk_cfg_kernel(cfg)][cpl];
  int o_cu = occ.load(std::memory_order_relaxed);
  if (o_cu == 0) {
    int o = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &o, blk_kernel(nw, cached, cfg, cpl), kBlkThreads, 0);
    o_cu = (e == hipSuccess && o > 0) ? o : 4;
    occ.store(o_cu, std::memory_order_relaxed);
  }
  int64_t resident = static_cast<int64_t>(o_cu) * n_cu;
  if (blk_cfg_half(cfg)) resident = std::max<int64_t>(1, resident / 2);
  const int64_t need = (a.n_tiles + kBlkWaves - 1) / kBlkWaves;
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(need, resident)));
}

int launch_blk_apply(const BlkArgs& a, int nw, int n_blocks, const double* X, double* Y,
                     double* partials, hipStream_t s) {
  const bool cached = blk_cached(a);
  const int cpl = blk_cpl(a);
  BlkArgs b = a;
  // lanes per row: as many as hold the columns; a power of two in the
  // searching kernels and where partials cross row groups by butterfly
  const int w = (a.R + cpl - 1) / cpl;
  b.G = 1;
  while (b.G < w) b.G <<= 1;
  if (cached && !partials) b.G = w;
  hipLaunchKernelGGL(blk_kernel(nw, cached, a.cfg, cpl), dim3(n_blocks), dim3(kBlkThreads), 0,
                     s, b, X, Y, partials);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int op_cache_connectivity(qsi_op_s* op, bool enable, bool allow_pad) {
  auto release = [&]() {
    if (op->d_rowptr) (void)hipFree(op->d_rowptr);
    if (op->d_cj) (void)hipFree(op->d_cj);
    if (op->d_cm) (void)hipFree(op->d_cm);
    op->d_rowptr = nullptr;
    op->d_cj = nullptr;
    op->d_cm = nullptr;
    op->conn_nnz = -1;
  };
  if (!enable) {
    if (op->conn_nnz >= 0) QSI_CHECK_HIP(hipDeviceSynchronize());
    release();
    if (op->variant == QSI_APPLY_CACHED) op->variant = QSI_APPLY_AUTO;
    return QSI_OK;
  }
  if (op->conn_nnz >= 0) return QSI_OK;
  QSI_REQUIRE(op->n_cls > 0 || op->n_off == 0,
              "qsi_op_cache_connectivity: more than 8 coefficient classes");
  const int64_t D = op->basis->dim;
  const auto view = op->basis->view();
  const uint32_t grid = static_cast<uint32_t>((D + 255) / 256);
  void* tmp = nullptr;
  size_t tmp_bytes = 0;
  hipError_t e = hipMalloc(&op->d_rowptr, static_cast<size_t>(D + 1) * sizeof(uint64_t));
  // row offsets: counts (rounded up to multiples of pad), then an in-place
  // exclusive scan of the D + 1 values (the last count is 0); returns the total
  auto offsets = [&](int pad, uint64_t* total) -> hipError_t {
    hipError_t r = hipMemset(op->d_rowptr, 0, static_cast<size_t>(D + 1) * sizeof(uint64_t));
    if (r == hipSuccess && D > 0) {
      if (op->basis->nw == 1)
        hipLaunchKernelGGL(k_cc_count<1>, dim3(grid), dim3(256), 0, 0, view, op->d_off, op->n_off,
                           pad, op->d_rowptr);
      else
        hipLaunchKernelGGL(k_cc_count<2>, dim3(grid), dim3(256), 0, 0, view, op->d_off, op->n_off,
                           pad, op->d_rowptr);
      r = hipGetLastError();
    }
    if (r == hipSuccess && !tmp) {
      r = hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, op->d_rowptr, op->d_rowptr, D + 1);
      if (r == hipSuccess) r = hipMalloc(&tmp, std::max<size_t>(tmp_bytes, 1));
    }
    if (r == hipSuccess)
      r = hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, op->d_rowptr, op->d_rowptr, D + 1);
    if (r == hipSuccess)
      r = hipMemcpy(total, op->d_rowptr + D, sizeof(uint64_t), hipMemcpyDeviceToHost);
    return r;
  };
  uint64_t nnz = 0, slots = 0;
  if (e == hipSuccess) e = offsets(1, &nnz);
  // Rows padded to whole groups of four entries let the cached apply read
  // every group with one aligned load (about 15 % faster at 64 spins); the
  // padding (at most 3 entries, 15 bytes, per row) is spent only when the
  // padded arrays leave a quarter of the free memory (at least 1 GiB) unused.
  if (e == hipSuccess) {
    size_t free_b = 0, total_b = 0;
    const size_t padded = (nnz + 3 * static_cast<size_t>(D)) * 5;
    if (allow_pad && hipMemGetInfo(&free_b, &total_b) == hipSuccess &&
        free_b > padded + std::max<size_t>(free_b / 4, size_t{1} << 30)) {
      e = offsets(4, &slots);
      op->conn_pad = 4;
    } else {
      slots = nnz;
      op->conn_pad = 1;
    }
  }
  if (tmp) (void)hipFree(tmp);
  // rounded up to whole 16-byte groups of columns (the cached apply reads the
  // columns four at a time from 16-byte aligned addresses, and the class
  // bytes four at a time)
  const size_t cap = std::max<size_t>((slots + 3) & ~uint64_t{3}, 4);
  if (e == hipSuccess) e = hipMalloc(&op->d_cj, cap * sizeof(uint32_t));
  if (e == hipSuccess) e = hipMalloc(&op->d_cm, cap);
  if (e == hipSuccess && D > 0) {
    if (op->basis->nw == 1)
      hipLaunchKernelGGL(k_cc_fill<1>, dim3(grid), dim3(256), 0, 0, view, op->d_off, op->n_off,
                         op->d_rowptr, op->d_cj, op->d_cm);
    else
      hipLaunchKernelGGL(k_cc_fill<2>, dim3(grid), dim3(256), 0, 0, view, op->d_off, op->n_off,
                         op->d_rowptr, op->d_cj, op->d_cm);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    release();
    set_error(std::string("qsi_op_cache_connectivity: ") + hipGetErrorString(e));
    return e == hipErrorOutOfMemory ? QSI_E_NOMEM : QSI_E_HIP;
  }
  op->conn_nnz = nnz;
  return QSI_OK;
}

}  // namespace qsi

using namespace qsi;

namespace {

// Block-apply arguments over the sectors' operators (rows concatenated in
// sector order), R columns with row stride R; *rows = total rows.
BlkArgs sector_args(const qsi_op_t* ops, int n_sectors, int R, const double* const* d_coeffs,
                    int64_t* rows_out) {
  BlkArgs args{};
  args.n_sec = n_sectors;
  args.R = R;
  int G = 64;
  while (G / 2 >= R && G > 1) G >>= 1;
  args.G = G;
  args.ldx = args.ldy = R;
  args.accumulate = 0;
  args.y_colmajor = 0;
  int64_t rows = 0;
  for (int s = 0; s < n_sectors; ++s) {
    const qsi_op_s* op = ops[s];
    BlkSector& S = args.sec[s];
    S.b = op->basis->view();
    S.off = op->d_off;
    S.tp = op->planes();
    S.dg = op->d_diag;
    S.cls = op->d_cls;
    S.n_cls = op->n_cls;
    S.rowptr = op->d_rowptr;
    S.cj = op->d_cj;
    S.cm = op->d_cm;
    S.n_off = op->n_off;
    S.n_diag = op->n_diag;
    S.coeffs = d_coeffs ? d_coeffs[s] : nullptr;
    S.row_off = rows;
    rows += op->basis->dim;
  }
  blk_set_tiles(args);
  args.cfg = ops[0]->blk_cfg;
  *rows_out = rows;
  return args;
}

}  // namespace

extern "C" int qsi_lanczos_block(const qsi_op_t* ops, int n_sectors, int R,
                                 const double* const* d_V0,
                                 const double* const* d_coeffs, int M,
                                 double* h_alpha, double* h_beta, int use_graph,
                                 double* elapsed_ms) {
  QSI_REQUIRE(ops && d_V0 && h_alpha && h_beta, "qsi_lanczos_block: null argument");
  QSI_REQUIRE(n_sectors >= 1 && n_sectors <= kMaxSectors,
              "qsi_lanczos_block: n_sectors must be in [1, 8]");
  QSI_REQUIRE(R >= 1 && R <= 64, "qsi_lanczos_block: R must be in [1, 64]");
  QSI_REQUIRE(M >= 1, "qsi_lanczos_block: M must be >= 1");
  const int nw = ops[0]->basis->nw;
  for (int s = 0; s < n_sectors; ++s) {
    QSI_REQUIRE(ops[s] != nullptr && ops[s]->basis->dim > 0, "qsi_lanczos_block: empty sector");
    QSI_REQUIRE(ops[s]->basis->nw == nw, "qsi_lanczos_block: sectors mix <=64 and >64 spins");
    QSI_REQUIRE(d_V0[s] != nullptr, "qsi_lanczos_block: null start block");
    QSI_REQUIRE(!d_coeffs || !d_coeffs[s] || ops[s]->n_slots > 0,
                "qsi_lanczos_block: coefficients given for an operator without slots");
  }
  int64_t rows = 0;
  BlkArgs args = sector_args(ops, n_sectors, R, d_coeffs, &rows);
  // persistent grids: enough wavefronts to fill the chip, never more than tiles
  const int n_blocks = blk_apply_blocks(args, nw);
  const int n_vec = static_cast<int>(std::min<int64_t>(args.n_tiles / kBlkWaves, kBlkVecBlocks));
  const size_t blk = static_cast<size_t>(rows) * R;
  DevMem mem;
  double *A = nullptr, *B = nullptr, *C = nullptr, *part = nullptr;
  double *alpha = nullptr, *beta = nullptr, *invb = nullptr, *ha = nullptr, *hb = nullptr;
  int* step = nullptr;
  const int SR = n_sectors * R;
  QSI_CHECK_HIP(mem.alloc(&A, blk));
  QSI_CHECK_HIP(mem.alloc(&B, blk));
  QSI_CHECK_HIP(mem.alloc(&C, blk));
  QSI_CHECK_HIP(mem.alloc(&part, static_cast<size_t>(SR) * std::max(n_blocks, n_vec)));
  QSI_CHECK_HIP(mem.alloc(&alpha, SR));
  QSI_CHECK_HIP(mem.alloc(&beta, SR));
  QSI_CHECK_HIP(mem.alloc(&invb, SR));
  QSI_CHECK_HIP(mem.alloc(&ha, static_cast<size_t>(SR) * M));
  QSI_CHECK_HIP(mem.alloc(&hb, static_cast<size_t>(SR) * M));
  QSI_CHECK_HIP(mem.alloc(&step, 1));
  hipStream_t st = nullptr;
  QSI_CHECK_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  struct StreamGuard {
    hipStream_t s;
    ~StreamGuard() { (void)hipStreamDestroy(s); }
  } sg{st};
  for (int s = 0; s < n_sectors; ++s) {
    QSI_CHECK_HIP(hipMemcpyAsync(B + args.sec[s].row_off * R, d_V0[s],
                                 static_cast<size_t>(ops[s]->basis->dim) * R * sizeof(double),
                                 hipMemcpyDeviceToDevice, st));
  }
  QSI_CHECK_HIP(hipMemsetAsync(A, 0, blk * sizeof(double), st));
  QSI_CHECK_HIP(hipMemsetAsync(beta, 0, SR * sizeof(double), st));
  QSI_CHECK_HIP(hipMemsetAsync(step, 0, sizeof(int), st));
  // normalise the start columns: B = B / |B_c|
  const dim3 fin((R + kFinCols - 1) / kFinCols, n_sectors);
  hipLaunchKernelGGL(k_blk_update, dim3(n_vec), dim3(kBlkThreads), 0, st, args,
                     static_cast<const double*>(nullptr), B, B, static_cast<const double*>(nullptr),
                     static_cast<const double*>(nullptr), part, static_cast<const double*>(nullptr),
                     static_cast<const double*>(nullptr), static_cast<int*>(nullptr));
  QSI_CHECK_LAUNCH();
  // (C = B - 0*B: the kernel writes back B unchanged and produces |B_c|^2)
  hipLaunchKernelGGL(k_blk_finalize, fin, dim3(kFinThreads), 0, st, part, n_vec, R, 1,
                     beta, invb, static_cast<double*>(nullptr), static_cast<const int*>(nullptr), 0,
                     M, static_cast<const double*>(nullptr));
  QSI_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_blk_scale, dim3(n_vec), dim3(kBlkThreads), 0, st, args, B, invb);
  QSI_CHECK_LAUNCH();
  QSI_CHECK_HIP(hipMemsetAsync(beta, 0, SR * sizeof(double), st));

  // The blocks hold the Lanczos vectors unnormalised, each column with its
  // scale (v = scale * column) in scl[k] beside bufs[k]: the step applies H to
  // the unnormalised B, folds B's scale into alpha and the update, and the
  // new column's scale is 1/beta — no pass rewrites a block to normalise it.
  // B starts normalised (scale 1); A is zero.
  double* bufs[3] = {A, B, C};
  double* scl[3] = {nullptr, nullptr, nullptr};
  for (int k = 0; k < 3; ++k) {
    QSI_CHECK_HIP(mem.alloc(&scl[k], SR));
    std::vector<double> ones(static_cast<size_t>(SR), 1.0);
    QSI_CHECK_HIP(hipMemcpyAsync(scl[k], ones.data(), SR * sizeof(double),
                                 hipMemcpyHostToDevice, st));
    QSI_CHECK_HIP(hipStreamSynchronize(st));
  }
  auto enqueue_step = [&](int p) -> int {
    double* a = bufs[p % 3];
    double* b = bufs[(p + 1) % 3];
    double* c = bufs[(p + 2) % 3];
    const double* sa = scl[p % 3];
    const double* sb = scl[(p + 1) % 3];
    double* sc = scl[(p + 2) % 3];
    const int rc = launch_blk_apply(args, nw, n_blocks, b, c, part, st);
    if (rc != QSI_OK) return rc;
    hipLaunchKernelGGL(k_blk_finalize, fin, dim3(kFinThreads), 0, st, part, n_blocks, R, 0,
                       alpha, static_cast<double*>(nullptr), ha, step, 0, M, sb);
    QSI_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_blk_update, dim3(n_vec), dim3(kBlkThreads), 0, st, args, a, b, c,
                       alpha, beta, part, sa, sb, step);
    QSI_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_blk_finalize, fin, dim3(kFinThreads), 0, st, part, n_vec, R, 1,
                       beta, sc, hb, step, 1, M, static_cast<const double*>(nullptr));
    QSI_CHECK_LAUNCH();
    return QSI_OK;
  };

  hipEvent_t e0, e1;
  QSI_CHECK_HIP(hipEventCreate(&e0));
  QSI_CHECK_HIP(hipEventCreate(&e1));
  struct EvGuard {
    hipEvent_t a, b;
    ~EvGuard() {
      (void)hipEventDestroy(a);
      (void)hipEventDestroy(b);
    }
  } eg{e0, e1};
  if (use_graph) {
    // one graph per rotation phase p: (A, B, C) = (bufs[p], bufs[p+1], bufs[p+2])
    hipGraphExec_t exec[3] = {nullptr, nullptr, nullptr};
    struct ExecGuard {
      hipGraphExec_t* e;
      ~ExecGuard() {
        for (int k = 0; k < 3; ++k)
          if (e[k]) (void)hipGraphExecDestroy(e[k]);
      }
    } xg{exec};
    for (int p = 0; p < 3 && p < M; ++p) {
      hipGraph_t g = nullptr;
      QSI_CHECK_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      const int rc = enqueue_step(p);
      hipGraph_t g2 = nullptr;
      const hipError_t ec = hipStreamEndCapture(st, &g2);
      g = g2;
      if (rc != QSI_OK) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
      }
      QSI_CHECK_HIP(ec);
      const hipError_t ei = hipGraphInstantiate(&exec[p], g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      QSI_CHECK_HIP(ei);
    }
    QSI_CHECK_HIP(hipEventRecord(e0, st));
    for (int j = 0; j < M; ++j) QSI_CHECK_HIP(hipGraphLaunch(exec[j % 3], st));
    QSI_CHECK_HIP(hipEventRecord(e1, st));
    QSI_CHECK_HIP(hipStreamSynchronize(st));
  } else {
    QSI_CHECK_HIP(hipEventRecord(e0, st));
    for (int j = 0; j < M; ++j) {
      const int p = j % 3;
      const int rc = enqueue_step(p);
      if (rc != QSI_OK) return rc;
    }
    QSI_CHECK_HIP(hipEventRecord(e1, st));
    QSI_CHECK_HIP(hipStreamSynchronize(st));
  }
  if (elapsed_ms) {
    float ms = 0.f;
    QSI_CHECK_HIP(hipEventElapsedTime(&ms, e0, e1));
    *elapsed_ms = ms;
  }
  QSI_CHECK_HIP(hipMemcpy(h_alpha, ha, static_cast<size_t>(SR) * M * sizeof(double),
                          hipMemcpyDeviceToHost));
  QSI_CHECK_HIP(hipMemcpy(h_beta, hb, static_cast<size_t>(SR) * M * sizeof(double),
                          hipMemcpyDeviceToHost));
  return QSI_OK;
}

// Eigenvalues and first eigenvector components of one Lanczos tridiagonal
// (Gauss quadrature nodes and weights for FTLM).
namespace {

// Average milliseconds per call of f(), timed with events on stream s: after
// one warm-up call, `reps` calls, repeated with more calls when those took
// under 5 ms.
template <typename F>
int time_ms(F&& f, int reps, hipStream_t s, double* ms) {
  hipEvent_t e0, e1;
  QSI_CHECK_HIP(hipEventCreate(&e0));
  QSI_CHECK_HIP(hipEventCreate(&e1));
  int rc = f();
  for (int pass = 0; pass < 2 && rc == QSI_OK; ++pass) {
    (void)hipEventRecord(e0, s);
    for (int r = 0; r < reps && rc == QSI_OK; ++r) rc = f();
    (void)hipEventRecord(e1, s);
    (void)hipEventSynchronize(e1);
    float t = 0.f;
    (void)hipEventElapsedTime(&t, e0, e1);
    *ms = t / reps;
    if (pass == 0) {
      const int want = *ms > 0.0 ? std::min(200, static_cast<int>(5.0 / *ms) + 1) : reps;
      if (want <= reps) break;
      reps = want;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

// Times every block-apply configuration (kernel x grid) of `a` on X, Y
// (rows x R) and returns the fastest.
int tune_block(BlkArgs a, int nw, int reps, const double* X, double* Y, int* pick,
               double* pick_ms) {

  const bool cached = blk_cached(a);
  const std::vector<int> kernels = cached ? std::vector<int>{0, 1, 2} : std::vector<int>{1, 2};
  const int n_pairs = cached && a.R >= 2 ? 2 : 1;
  *pick = -1;
  for (int k : kernels) {
    for (int cf = 0; cf < 2 * n_pairs; ++cf) {
      const int half = cf & 1, pairs = cf >> 1;
      a.cfg = k | (half << 2) | (pairs << 3);
      const int nb = blk_apply_blocks(a, nw);
      double ms = 0.0;
      const int rc = time_ms([&]() { return launch_blk_apply(a, nw, nb, X, Y, nullptr, nullptr); },
                             reps, nullptr, &ms);
      if (rc != QSI_OK) return rc;
      if (*pick < 0 || ms < *pick_ms) {
        *pick = a.cfg;
        *pick_ms = ms;
      }
    }
  }
  return QSI_OK;
}

}  // namespace

extern "C" int qsi_block_autotune(const qsi_op_t* ops, int n_sectors, int R, int reps, int* best,
                                  double* best_ms) {
  QSI_REQUIRE(ops != nullptr, "qsi_block_autotune: null argument");
  QSI_REQUIRE(n_sectors >= 1 && n_sectors <= kMaxSectors,
              "qsi_block_autotune: n_sectors must be in [1, 8]");
  QSI_REQUIRE(R >= 1 && R <= 64, "qsi_block_autotune: R must be in [1, 64]");
  const int nw = ops[0]->basis->nw;
  for (int s = 0; s < n_sectors; ++s) {
    QSI_REQUIRE(ops[s] != nullptr && ops[s]->basis->dim > 0, "qsi_block_autotune: empty sector");
    QSI_REQUIRE(ops[s]->basis->nw == nw, "qsi_block_autotune: sectors mix <=64 and >64 spins");
  }
  reps = std::max(1, reps);
  // each configuration runs a few steps of the block Lanczos recurrence
  // itself (the apply between the recurrence's vector kernels behaves
  // differently from back-to-back applies), from Gaussian start blocks
  constexpr int kSteps = 8;
  DevMem mem;
  std::vector<const double*> v0(n_sectors, nullptr), cp(n_sectors, nullptr);
  for (int s = 0; s < n_sectors; ++s) {
    double* v = nullptr;
    const int64_t n = ops[s]->basis->dim * R;
    QSI_CHECK_HIP(mem.alloc(&v, static_cast<size_t>(n)));
    int rc = launch_randn(v, n, 12345 + s, nullptr);
    if (rc != QSI_OK) return rc;
    v0[s] = v;
    if (ops[s]->n_slots > 0) {
      double* c = nullptr;
      QSI_CHECK_HIP(mem.alloc(&c, static_cast<size_t>(ops[s]->n_slots) * R));
      rc = launch_randn(c, static_cast<int64_t>(ops[s]->n_slots) * R, 7 + s, nullptr);
      if (rc != QSI_OK) return rc;
      cp[s] = c;
    }
  }
  QSI_CHECK_HIP(hipDeviceSynchronize());
  std::vector<double> ha(static_cast<size_t>(n_sectors) * R * kSteps),
      hb(static_cast<size_t>(n_sectors) * R * kSteps);
  std::vector<int> saved(n_sectors);
  for (int s = 0; s < n_sectors; ++s) saved[s] = ops[s]->blk_cfg;
  int64_t rows = 0;
  const bool cached = blk_cached(sector_args(ops, n_sectors, R, cp.data(), &rows));
  const std::vector<int> kernels = cached ? std::vector<int>{0, 1, 2} : std::vector<int>{1, 2};
  const int n_pairs = cached && R >= 2 ? 2 : 1;
  int pick = -1;
  double pick_ms = 0.0;
  for (int k : kernels) {
    for (int cf = 0; cf < 2 * n_pairs; ++cf) {
      const int half = cf & 1, pairs = cf >> 1;
      const int cfg = k | (half << 2) | (pairs << 3);
      for (int s = 0; s < n_sectors; ++s) ops[s]->blk_cfg = cfg;
      double ms = 0.0;
      for (int r = 0; r <= reps; ++r) {  // the first run warms up
        double t = 0.0;
        const int rc = qsi_lanczos_block(ops, n_sectors, R, v0.data(), cp.data(), kSteps,
                                         ha.data(), hb.data(), 0, &t);
        if (rc != QSI_OK) {
          for (int q = 0; q < n_sectors; ++q) ops[q]->blk_cfg = saved[q];
          return rc;
        }
        if (r > 0) ms += t / kSteps;
      }
      ms /= reps;
      if (pick < 0 || ms < pick_ms) {
        pick = cfg;
        pick_ms = ms;
      }
    }
  }
  for (int s = 0; s < n_sectors; ++s) ops[s]->blk_cfg = pick;
  if (best) *best = pick;
  if (best_ms) *best_ms = pick_ms;
  return QSI_OK;
}

extern "C" int qsi_op_autotune(qsi_op_t op, int R, int reps, double* d_x, double* d_y,
                               int* best, double* best_ms) {
  QSI_REQUIRE(op != nullptr, "qsi_op_autotune: null operator");
  QSI_REQUIRE(R >= 0 && R <= 64, "qsi_op_autotune: R must be in [0, 64]");
  reps = std::max(1, reps);
  const int64_t D = op->basis->dim;
  if (D == 0) return QSI_OK;
  const size_t n = static_cast<size_t>(D) * std::max(R, 1);
  DevMem mem;
  if (!d_x) {
    QSI_CHECK_HIP(mem.alloc(&d_x, n));
    // Gaussian input: every term's |x_J| is above the apply tolerance
    const int rc = launch_randn(d_x, static_cast<int64_t>(n), 12345, nullptr);
    if (rc != QSI_OK) return rc;
  }
  if (!d_y) QSI_CHECK_HIP(mem.alloc(&d_y, n));
  double* coeffs = nullptr;
  if (R > 0 && op->n_slots > 0) {
    QSI_CHECK_HIP(mem.alloc(&coeffs, static_cast<size_t>(op->n_slots) * R));
    const int rc = launch_randn(coeffs, static_cast<int64_t>(op->n_slots) * R, 7, nullptr);
    if (rc != QSI_OK) return rc;
  }
  QSI_CHECK_HIP(hipDeviceSynchronize());
  int pick = -1;
  double pick_ms = 0.0;
  if (R == 0) {
    std::vector<int> cand = {QSI_APPLY_LANE, QSI_APPLY_LANE2, QSI_APPLY_LANE4, QSI_APPLY_LANE8,
                             QSI_APPLY_WINDOW};
    // a kernel that only AUTO takes (2970 states: 7.3 us where the best of the
    // others takes 12.4)
    if (auto_takes_rows(op)) cand.push_back(QSI_APPLY_AUTO);
    if (op->basis->d_hash) {
      cand.push_back(QSI_APPLY_HASH);
      cand.push_back(QSI_APPLY_HASH4);
    }
    if (op->basis->d_slots) {
      cand.push_back(QSI_APPLY_SLOT2);
      cand.push_back(QSI_APPLY_SLOT3);
      cand.push_back(QSI_APPLY_SLOT4);
    }
    if (op->basis->d_lowkeys) {
      cand.push_back(QSI_APPLY_LOW2);
      cand.push_back(QSI_APPLY_LOW4);
      cand.push_back(QSI_APPLY_LOW8);
    }
    // the cached kernel once per gather depth (4, 8, 16, 32)
    std::vector<int> pipes(cand.size(), 8);
    if (op->conn_nnz >= 0) {
      for (int p : {4, 8, 16, 32}) {
        cand.push_back(QSI_APPLY_CACHED);
        pipes.push_back(p);
      }
    }
    const int saved = op->variant, saved_pipe = op->cached_pipe;
    int pick_pipe = saved_pipe;
    for (size_t k = 0; k < cand.size(); ++k) {
      op->variant = cand[k];
      op->cached_pipe = pipes[k];
      double ms = 0.0;
      const int rc = time_ms(
          [&]() { return launch_apply(op, d_x, d_y, nullptr, 0.0, nullptr, nullptr, nullptr); },
          reps, nullptr, &ms);
      if (rc != QSI_OK) {
        op->variant = saved;
        op->cached_pipe = saved_pipe;
        return rc;
      }
      if (pick < 0 || ms < pick_ms) {
        pick = cand[k];
        pick_pipe = pipes[k];
        pick_ms = ms;
      }
    }
    op->variant = pick;
    op->cached_pipe = pick_pipe;
  } else {
    const double* cp[1] = {coeffs};
    int64_t rows = 0;
    BlkArgs a = sector_args(&op, 1, R, cp, &rows);
    const int rc = tune_block(a, op->basis->nw, reps, d_x, d_y, &pick, &pick_ms);
    if (rc != QSI_OK) return rc;
    op->blk_cfg = pick;
  }
  if (best) *best = pick;
  if (best_ms) *best_ms = pick_ms;
  return QSI_OK;
}

extern "C" int qsi_op_cache_connectivity(qsi_op_t op, int enable, int64_t* nnz) {
  QSI_REQUIRE(op != nullptr, "qsi_op_cache_connectivity: null operator");
  QSI_REQUIRE(enable >= 0 && enable <= 2, "qsi_op_cache_connectivity: enable must be 0, 1 or 2");
  const int rc = op_cache_connectivity(op, enable != 0, enable == 1);
  if (nnz) *nnz = op->conn_nnz;
  return rc;
}

extern "C" int qsi_op_connectivity_padding(qsi_op_t op) {
  return op && op->conn_nnz >= 0 ? op->conn_pad : -1;
}

extern "C" int qsi_tridiag_eig(const double* d, const double* e, int n,
                               double* evals, double* first_row) {
  QSI_REQUIRE(d && evals && n >= 1 && (n == 1 || e), "qsi_tridiag_eig: bad arguments");
  std::vector<double> dv(d, d + n), ev(e ? e : d, e ? e + std::max(n - 1, 0) : d), w, fr;
  if (!hostla::tridiag_eig(dv, ev, w, nullptr, first_row ? &fr : nullptr)) {
    set_error("qsi_tridiag_eig: no convergence");
    return QSI_E_NOCONV;
  }
  std::copy(w.begin(), w.end(), evals);
  if (first_row) std::copy(fr.begin(), fr.end(), first_row);
  return QSI_OK;
}

extern "C" int qsi_tridiag_quadrature(const double* d, int64_t ldd, const double* e, int64_t lde,
                                      const int* n, int R, double* nodes, double* weights) {
  QSI_REQUIRE(d && e && n && nodes && weights && R >= 0, "qsi_tridiag_quadrature: bad arguments");
  double work = 0.0;
  for (int r = 0; r < R; ++r) {
    QSI_REQUIRE(n[r] >= 1 && n[r] <= ldd && n[r] - 1 <= lde,
                "qsi_tridiag_quadrature: bad sample length");
    work += static_cast<double>(n[r]) * n[r];
  }
  // samples are taken from a counter, so threads that start late or not at
  // all only leave more to the others
  std::atomic<int> next{0}, rc{QSI_OK};
  auto run = [&]() {
    try {
      std::vector<double> dv, ev, w, fr;
      for (int r; (r = next.fetch_add(1)) < R;) {
        dv.assign(d + r * ldd, d + r * ldd + n[r]);
        ev.assign(e + r * lde, e + r * lde + n[r] - 1);
        if (!hostla::tridiag_eig(dv, ev, w, nullptr, &fr)) {
          rc.store(QSI_E_NOCONV);
          continue;
        }
        for (int k = 0; k < n[r]; ++k) {
          nodes[r * ldd + k] = w[k];
          weights[r * ldd + k] = fr[k] * fr[k];
        }
      }
    } catch (const std::bad_alloc&) {
      rc.store(QSI_E_NOMEM);
    }
  };
  // one sample costs about 50 ns per n^2, starting a thread about 20 us: 0.4 ms
  // of work per thread; no more of them than the process may run on (ranks that
  // share a node are confined to their cores)
  cpu_set_t set;
  const int cores = sched_getaffinity(0, sizeof(set), &set) == 0
                        ? std::max(1, CPU_COUNT(&set))
                        : static_cast<int>(std::max(1u, std::thread::hardware_concurrency()));
  const int nt = std::min({16, cores, R, 1 + static_cast<int>(std::min(work / 8192.0, 64.0))});
  std::vector<std::thread> pool;
  try {
    for (int t = 1; t < nt; ++t) pool.emplace_back(run);
  } catch (const std::exception&) {
    // no more threads: this one does their share
  }
  run();
  for (auto& t : pool) t.join();
  if (rc.load() == QSI_E_NOCONV) set_error("qsi_tridiag_quadrature: no convergence");
  if (rc.load() == QSI_E_NOMEM) set_error("qsi_tridiag_quadrature: host allocation failed");
  return rc.load();
}
