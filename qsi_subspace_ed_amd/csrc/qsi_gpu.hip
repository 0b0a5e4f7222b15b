// Device side of the qsi library: device basis + top-bit bucket table,
// matrix-free pull apply (single vector and block), connectivity
// materialiser and streaming FP64 vector kernels.  gfx950 only.
//
// Reference behaviour being replaced (file:line in the reference tree):
//   ZBasisInterp::find_bounds / search   components/operator/src/operator.cpp:38-86
//   SymbolicPMROperator::applyState      components/operator/include/operator.hpp:232-254
//   LazyOpSum::evaluate_add_off_diag_omp components/operator/src/operator_matrix.cpp:28-60
//   LazyOpSum::evaluate_add_diagonal     components/operator/src/operator_matrix.cpp:65-82
//   LazyOpSum::toSparseMatrix            components/operator/include/operator_matrix.hpp:79-105
//
// The reference pushes: for each term and each column j it finds
// J = rank(O s_j) and atomically adds c*sign*x_j to y_J.  Here every output
// row i pulls instead: for each term whose precondition holds on the
// pre-image s_i ^ X, it gathers x at rank(s_i ^ X).  Both compute
// y_i = sum_j H_ij x_j for the same H (no symmetry is assumed), but the pull
// form writes each y_i exactly once, so it needs no atomics and its sum order
// is fixed (term order, then diagonal terms) — results are deterministic.

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "qsi_blockk.hpp"
#include "qsi_device.hpp"
#include "qsi_internal.hpp"
#include "qsi_reduce.hpp"

namespace qsi {

constexpr int kApplyBlock = 256;
constexpr double kSparseTol = 1e-14;  // toSparseMatrix default tol

// ============================================================================
// Basis: bucket table
// ============================================================================

// First rank whose bucket key is >= k (a bisection over the basis).
template <int NW>
__device__ __forceinline__ uint32_t table_entry(const BasisView& b, int64_t k) {
  int64_t lo = 0, n = b.dim;
  while (n > 0) {
    const int64_t half = n >> 1;
    const State<NW> s = load_state_cached<NW>(b.states, lo + half);
    if (static_cast<int64_t>(bucket_key<NW>(b, s)) < k) {
      lo = lo + half + 1;
      n = n - half - 1;
    } else {
      n = half;
    }
  }
  return static_cast<uint32_t>(lo);
}

// table[k] = first rank whose bucket key is >= k, for k in [0, 2^K].
// Grid-stride: a dispatch holds fewer than 2^32 work-items, and a 32-bit key
// has 2^32 + 1 entries.
template <int NW>
__global__ void k_build_table(BasisView b, int64_t nkeys, uint32_t* __restrict__ table) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; k <= nkeys;
       k += stride)
    table[k] = table_entry<NW>(b, k);
}

// mask[p / 64] bit p % 64 = 1 if some neighbouring pair of the sorted basis
// first differs at bit p.  Grid-stride; one global OR per word per block.
template <int NW>
__global__ __launch_bounds__(256) void k_diff_bits(const uint64_t* __restrict__ states,
                                                   int64_t dim,
                                                   unsigned long long* __restrict__ mask) {
  __shared__ unsigned long long sm[2];
  if (threadIdx.x < 2) sm[threadIdx.x] = 0;
  __syncthreads();
  unsigned long long m0 = 0, m1 = 0;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i + 1 < dim;
       i += stride) {
    const State<NW> a = load_state_cached<NW>(states, i);
    const State<NW> c = load_state_cached<NW>(states, i + 1);
    if constexpr (NW == 2) {
      const uint64_t hi = a.w[1] ^ c.w[1];
      if (hi) {
        m1 |= 1ull << (63 - __clzll(hi));
        continue;
      }
    }
    const uint64_t lo = a.w[0] ^ c.w[0];
    if (lo) m0 |= 1ull << (63 - __clzll(lo));
  }
  if (m0) atomicOr(&sm[0], m0);
  if (m1) atomicOr(&sm[1], m1);
  __syncthreads();
  if (threadIdx.x < 2 && sm[threadIdx.x]) atomicOr(&mask[threadIdx.x], sm[threadIdx.x]);
}

// Insert every basis state into the hash index (slots pre-filled with ones).
// A thread claims a free slot by a compare-and-swap on its rank word and then
// writes the state; keys are unique, so no insertion compares keys.
template <int NW>
__global__ void k_build_hash(const uint64_t* __restrict__ states, int64_t dim,
                             ulonglong2* __restrict__ slots, uint64_t mask,
                             int hbits) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= dim) return;
  const State<NW> s = load_state_cached<NW>(states, i);
  uint64_t p = hash_home<NW>(s, hbits);
  for (;;) {
    unsigned long long* rank_word =
        (NW == 1) ? reinterpret_cast<unsigned long long*>(&slots[p].y)
                  : reinterpret_cast<unsigned long long*>(&slots[2 * p + 1].x);
    const unsigned long long old =
        atomicCAS(rank_word, static_cast<unsigned long long>(kHashEmpty),
                  static_cast<unsigned long long>(i));
    if (old == kHashEmpty) {
      if constexpr (NW == 1) {
        slots[p].x = s.w[0];
      } else {
        slots[2 * p].x = s.w[0];
        slots[2 * p].y = s.w[1];
      }
      return;
    }
    p = (p + 1) & mask;
  }
}

// Place every basis state in its bucket's slot region (slots pre-filled with
// kSlotEmpty): linear probing from the state's home, a slot claimed by a
// compare-and-swap.  A bucket above kSlotMaxBucket states sets *too_big and
// places nothing.
// For every row and connecting term of an operator: whether the target's
// low-key lookup ends on a candidate with the target's bucket key and low key
// but another state (a target outside the basis that differs from a basis
// state only at positions fixed in the basis: *bad |= 1), and whether any
// target is outside the basis (*bad |= 2) (qsi_op_verify_lowkeys).
template <int NW>
__global__ void k_verify_lowkeys(BasisView b, const OffTerm* __restrict__ off, int n_off,
                                 unsigned int* __restrict__ bad) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= b.dim) return;
  const State<NW> s = load_state_cached<NW>(b.states, i);
  bool clash = false, absent = false;
  for (int t = 0; t < n_off; ++t) {
    if (!term_ok<NW>(off[t], s)) continue;
    const State<NW> key = xor_state<NW>(s, off[t].X);
    uint32_t lo, n;
    bucket_bounds(b.table, bucket_key<NW>(b, key), lo, n);
    if (n == 0) {
      absent = true;
      continue;
    }
    const uint32_t r = low_key<NW>(b, key);
    while (n > 1) {
      const uint32_t half = n >> 1;
      lo = b.lowkeys[lo + half] <= r ? lo + half : lo;
      n -= half;
    }
    if (b.lowkeys[lo] != r) absent = true;
    else if (!st_eq<NW>(load_state_cached<NW>(b.states, lo), key)) clash = true;
  }
  if (clash || absent) atomicOr(bad, (clash ? 1u : 0u) | (absent ? 2u : 0u));
}

// cnt[0] += (tile, term) pairs that connect, of gridDim.x tiles of 128 rows spread
// evenly over the basis; cnt[1] += those with a target that is not in the basis.
// One tile per workgroup, its wavefronts taking every fourth term.
template <int NW>
__global__ __launch_bounds__(256) void k_sample_closed(BasisView b,
                                                       const OffTerm* __restrict__ off, int n_off,
                                                       unsigned int* __restrict__ cnt) {
  const int lane = threadIdx.x % kWave;
  const int64_t r0 = b.dim / 128 / gridDim.x * blockIdx.x * 128 + lane;
  const State<NW> s0 = load_state_cached<NW>(b.states, r0);
  const State<NW> s1 = load_state_cached<NW>(b.states, r0 + 64);
  unsigned int conn = 0, missing = 0;
  for (int t = threadIdx.x / kWave; t < n_off; t += 4) {
    const OffTerm& T = off[t];
    const bool c0 = term_ok<NW>(T, s0), c1 = term_ok<NW>(T, s1);
    if (!__any(c0 || c1)) continue;
    const bool miss = (c0 && basis_lookup<NW>(b, xor_state<NW>(s0, T.X)) < 0) ||
                      (c1 && basis_lookup<NW>(b, xor_state<NW>(s1, T.X)) < 0);
    ++conn;
    missing += __any(miss) ? 1u : 0u;
  }
  if (lane == 0) {
    atomicAdd(cnt, conn);
    atomicAdd(cnt + 1, missing);
  }
}

// lowkeys[i] = low key of state i (qsi_basis_build_lowkeys)
template <int NW>
__global__ void k_build_lowkeys(BasisView b, uint32_t* __restrict__ lowkeys) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= b.dim) return;
  lowkeys[i] = low_key<NW>(b, load_state_cached<NW>(b.states, i));
}

template <int NW>
__global__ void k_build_slots(BasisView b, uint32_t* __restrict__ slots,
                              unsigned int* __restrict__ too_big) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= b.dim) return;
  const State<NW> s = load_state_cached<NW>(b.states, i);
  uint32_t lo, n;
  bucket_bounds(b.table, bucket_key<NW>(b, s), lo, n);
  if (n > kSlotMaxBucket) {
    atomicOr(too_big, 1u);
    return;
  }
  const uint64_t h = slot_hash<NW>(s);
  const uint32_t m = 2 * n;
  const uint32_t e = (slot_fp(h) << 16) | static_cast<uint32_t>(i - lo);
  uint32_t* reg = slots + 2 * static_cast<uint64_t>(lo);
  uint32_t p = slot_home(h, m);
  while (atomicCAS(reg + p, kSlotEmpty, e) != kSlotEmpty) p = p + 1 == m ? 0 : p + 1;
}

template <int NW>
__global__ void k_search(BasisView b, const uint64_t* __restrict__ q, int64_t n,
                         int64_t* __restrict__ rank) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  State<NW> s;
  // queries always come as [lo, hi] pairs
  s.w[0] = q[2 * i];
  if constexpr (NW == 2) s.w[1] = q[2 * i + 1];
  bool ok = true;
  if constexpr (NW == 1) ok = (q[2 * i + 1] == 0);
  rank[i] = !ok ? -1 : b.slots ? slot_lookup<NW>(b, s) : basis_lookup<NW>(b, s);
}

// ============================================================================
// Apply: one lane per output row
// ============================================================================

// Flip masks and signed coefficients of the first kLdsTerms off-diagonal
// terms, staged in LDS by every workgroup: lookups re-form their connected
// state and take their coefficient from here instead of gathering each
// lane's term from global memory.
constexpr int kLdsTerms = 256;
template <int NW>
struct TermsLds {
  uint64_t X[NW][kLdsTerms];
  double c[kLdsTerms];  // c * sgn
};

template <int NW>
__device__ __forceinline__ bool stage_terms(TermsLds<NW>& tl, const OffTerm* __restrict__ off,
                                            int n_off) {
  const bool lds = n_off <= kLdsTerms;
  if (lds) {
    for (int t = threadIdx.x; t < n_off; t += blockDim.x) {
#pragma unroll
      for (int w = 0; w < NW; ++w) tl.X[w][t] = off[t].X[w];
      tl.c[t] = off[t].c * off[t].sgn;
    }
  }
  __syncthreads();
  return lds;
}

template <int NW>
__device__ __forceinline__ State<NW> term_target(const TermsLds<NW>& tl, bool lds,
                                                 const OffTerm* __restrict__ off,
                                                 const State<NW>& s, int t) {
  State<NW> r;
#pragma unroll
  for (int w = 0; w < NW; ++w) r.w[w] = s.w[w] ^ (lds ? tl.X[w][t] : off[t].X[w]);
  return r;
}

// Terms as the lane and low-key kernels stage them in LDS, kLdsTerms at a
// time: flip masks, signed coefficients, and each flip mask's bucket key and
// low key.  Both keys select bits of a state, so they commute with a flip:
// key(s ^ X) = key(s) ^ key(X).  A lookup forms its keys from the row's own
// keys with an XOR instead of gathering them bit field by bit field from
// the connected state.
template <int NW>
struct LowTermsLds {
  uint64_t X[NW][kLdsTerms];
  double c[kLdsTerms];   // c * sgn
  uint2 key[kLdsTerms];  // bucket key, low key (0 without low keys) of X
};

// Stages terms [0, n) of `off` (n <= kLdsTerms).  Every thread of the
// workgroup calls it; `reuse` (uniform) first waits until every thread is
// done with the previous chunk.
template <int NW>
__device__ __forceinline__ void stage_low_terms(LowTermsLds<NW>& tl, const BasisView& b,
                                                const OffTerm* __restrict__ off, int n,
                                                bool reuse) {
  if (reuse) __syncthreads();
  for (int t = threadIdx.x; t < n; t += blockDim.x) {
    State<NW> X;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      X.w[w] = off[t].X[w];
      tl.X[w][t] = X.w[w];
    }
    tl.c[t] = off[t].c * off[t].sgn;
    tl.key[t] = make_uint2(bucket_key<NW>(b, X), b.lowkeys ? low_key<NW>(b, X) : 0u);
  }
  __syncthreads();
}

template <int NW>
__device__ __forceinline__ State<NW> staged_target(const LowTermsLds<NW>& tl,
                                                   const State<NW>& s, uint32_t t) {
  State<NW> r;
#pragma unroll
  for (int w = 0; w < NW; ++w) r.w[w] = s.w[w] ^ tl.X[w][t];
  return r;
}

// v of one lane, in all.
__device__ __forceinline__ double read_lane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// y[i] = yscale * y_in[i] + sum_t H_{i,t} x[...] + d(s_i) x[i]
// If DOT, partials[block] = sum over the block's rows of x[i] * y[i].
// Lane variant: every lane walks its own row's connected states and runs a
// full table lookup for each.  G lookups go through the bucket table, the
// bisection and the x gather together, and every stage issues the loads of
// all G (those of unfinished lookups) before it uses any, so a lane keeps G
// loads in flight; contributions are still added in term order.  An empty
// asm statement that reads each loaded value after the last load of the
// stage keeps the compiler from moving a use next to its load, which would
// make every load wait for the one before.
template <int NW, bool HAS_Z, bool DOT, int G>
__global__ __launch_bounds__(kApplyBlock)
__attribute__((amdgpu_waves_per_eu(G >= 8 ? 3 : G >= 4 ? 5 : 8))) void k_apply_lane(
    BasisView b, const OffTerm* __restrict__ off, int n_off,
    const DiagTerm* __restrict__ dg, int n_diag, const double* __restrict__ x,
    double* y, const double* y_in, double yscale,
    const double* __restrict__ yscale_dev, double* __restrict__ partials,
    const double* __restrict__ xs_dev, const double* __restrict__ ys_dev) {
  const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
  if (yscale_dev) yscale *= yscale_dev[0];
  // x and y_in are read as xs * x and ys * y_in.  Only the dot-product
  // instances (the Lanczos step) take scales; elsewhere they are the
  // constant 1 and the multiplies fold away.
  const double xs = (DOT && xs_dev) ? xs_dev[0] : 1.0;
  const double ys = (DOT && ys_dev) ? ys_dev[0] : 1.0;
  __shared__ LowTermsLds<NW> tl;
  const int64_t i = static_cast<int64_t>(blk) * kApplyBlock + threadIdx.x;
  const bool live = i < b.dim;
  State<NW> s = {};
  double xi = 0.0, acc = 0.0, prod = 0.0;
  uint32_t ks = 0;
  if (live) {
    s = load_state_cached<NW>(b.states, i);
    xi = x[i] * xs;
    acc = y_in ? yscale * (y_in[i] * ys) : 0.0;
    ks = bucket_key<NW>(b, s);
  }
  for (int c0 = 0; c0 < n_off; c0 += kLdsTerms) {
    const int cn = min(kLdsTerms, n_off - c0);
    stage_low_terms<NW>(tl, b, off + c0, cn, c0 > 0);
    if (!live) continue;
    for (int t0 = 0; t0 < cn; t0 += 64) {
      const int tn = min(64, cn - t0);
      // which terms connect this row (term t0 + t at bit 63 - t)
      uint64_t mask = connect_mask<NW>(off + c0 + t0, tn, s);
      while (mask) {
        uint32_t tt[G], lo[G], n[G];
        bool act[G];
        uint2 p[G];
        // bucket bounds of all G lookups (each connected state is re-formed
        // from the row and the staged flip mask where it is compared)
#pragma unroll
        for (int g = 0; g < G; ++g) {
          act[g] = mask != 0;
          const uint32_t z = act[g] ? static_cast<uint32_t>(__builtin_clzll(mask)) : 0u;
          tt[g] = t0 + z;
          mask &= ~(uint64_t{1} << 63 >> z);
          p[g] = make_uint2(0u, 0u);
          if (act[g]) __builtin_memcpy(&p[g], b.table + (ks ^ tl.key[tt[g]].x), sizeof(uint2));
        }
#pragma unroll
        for (int g = 0; g < G; ++g) asm volatile("" : "+v"(p[g].x), "+v"(p[g].y));
        bool more = false;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          lo[g] = p[g].x;
          n[g] = act[g] ? p[g].y - p[g].x : 0u;
          more |= n[g] > 1;
        }
        // interleaved bisection down to one candidate per key: the G probes,
        // then the G updates (a finished lookup has half = 0: no change)
        while (more) {
          State<NW> m[G];
#pragma unroll
          for (int g = 0; g < G; ++g) {
            m[g] = State<NW>{};
            if (n[g] > 1) m[g] = load_state_cached<NW>(b.states, lo[g] + (n[g] >> 1));
          }
          // every probe of the group is used only after all were issued
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int w = 0; w < NW; ++w) asm volatile("" : "+v"(m[g].w[w]));
          more = false;
#pragma unroll
          for (int g = 0; g < G; ++g) {
            const uint32_t half = n[g] >> 1;
            lo[g] = st_le<NW>(m[g], staged_target<NW>(tl, s, tt[g])) ? lo[g] + half : lo[g];
            n[g] -= half;
            more |= n[g] > 1;
          }
        }
        // the candidate's state and x are loaded together (lo < dim whenever
        // the bucket is not empty); x counts only if the state matches
        double xj[G], c[G];
        State<NW> f[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          xj[g] = 0.0;
          c[g] = tl.c[tt[g]];
          if (n[g] == 1) {
            f[g] = load_state_cached<NW>(b.states, lo[g]);
            xj[g] = x[lo[g]];
          }
        }
        // the scale is applied where the values are consumed, after every
        // gather of the group has been issued
#pragma unroll
        for (int g = 0; g < G; ++g) xj[g] *= xs;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if (n[g] == 1 && st_eq<NW>(f[g], staged_target<NW>(tl, s, tt[g])) &&
              fabs(xj[g]) > kApplyTol) {
            double cg = c[g];
            if constexpr (HAS_Z) {
              if (parity_notz<NW>(s, off[c0 + tt[g]].Z)) cg = -cg;
            }
            acc += cg * xj[g];
          }
        }
      }
    }
  }
  if (live) {
    acc = diag_accumulate<NW>(acc, xi, s, dg, n_diag);
    y[i] = acc;
    if constexpr (DOT) prod = xi * acc;
  }
  if constexpr (DOT) {
    const double bs = block_sum<kApplyBlock>(prod);
    if (threadIdx.x == 0) partials[blk] = bs;
  }
}

// Row variant, for bases that leave the lane variant with a wavefront or two on
// each compute unit: one wavefront per row, one term per lane.  All of a row's
// lookups go through the table, the bisection and the gather at once, so the
// kernel is one chain of dependent loads where a lane that walks its row's
// terms four at a time waits for that chain two to eight times.  The
// contributions are then added by every lane alike, in term order and with the
// lane variant's multiply-adds, so y is bit-identical.
template <int NW, bool HAS_Z>
__global__ __launch_bounds__(kApplyBlock) void k_apply_row(
    BasisView b, const OffTerm* __restrict__ off, int n_off,
    const DiagTerm* __restrict__ dg, int n_diag, const double* __restrict__ x,
    double* y, const double* y_in, double yscale, const double* __restrict__ yscale_dev) {
  const int lane = threadIdx.x % kWave;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * (kApplyBlock / kWave) +
                    __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (i >= b.dim) return;
  if (yscale_dev) yscale *= yscale_dev[0];
  const State<NW> s = load_state_cached<NW>(b.states, i);
  const double xi = x[i];
  double acc = y_in ? yscale * y_in[i] : 0.0;
  for (int t0 = 0; t0 < n_off; t0 += kWave) {
    const bool in = t0 + lane < n_off;
    const OffTerm& T = off[in ? t0 + lane : 0];
    bool hit = in && term_ok<NW>(T, s);
    const State<NW> key = xor_state<NW>(s, T.X);
    double c = T.c * T.sgn;
    if constexpr (HAS_Z) {
      if (parity_notz<NW>(s, T.Z)) c = -c;
    }
    uint32_t lo = 0, n = 0;
    if (hit) {
      uint2 p;
      __builtin_memcpy(&p, b.table + bucket_key<NW>(b, key), sizeof(uint2));
      lo = p.x;
      n = p.y - p.x;
    }
    while (n > 1) {
      const uint32_t half = n >> 1;
      if (st_le<NW>(load_state_cached<NW>(b.states, lo + half), key)) lo += half;
      n -= half;
    }
    double xj = 0.0;
    if (n == 1) {
      const State<NW> f = load_state_cached<NW>(b.states, lo);
      xj = x[lo];
      if (!st_eq<NW>(f, key)) xj = 0.0;
    }
    for (uint64_t mask = __ballot(fabs(xj) > kApplyTol); mask; mask &= mask - 1) {
      const int l = __builtin_ctzll(mask);
      const double cl = read_lane(c, l), xl = read_lane(xj, l);
      acc += cl * xl;
    }
  }
  acc = diag_accumulate<NW>(acc, xi, s, dg, n_diag);
  if (lane == 0) y[i] = acc;
}

// Low-key variant (QSI_APPLY_LOW*): as the lane variant, but the bisection
// of a bucket probes the 4-byte low keys (qsi_basis_build_lowkeys) instead of
// whole states — four times as many candidates per cache line, and the state
// array is touched once per lookup at most, for the candidate.  The
// candidate is the last state of the bucket whose low key is <= the
// target's, the same state the lane variant's bisection ends on, so y is
// bit-identical.  A lookup keeps only its term, bucket start, bucket size and
// (below eight lookups per lane) its low key.  Every stage issues the loads of
// all G lookups (those not yet finished) before it uses any, as in the lane
// variant, so a lane keeps G loads in flight through the table, each
// bisection step and the gathers.
//
// CHECK says how a candidate is confirmed.  kLowCmpState: its state is
// loaded and compared.  kLowCmpKey (qsi_op_verify_lowkeys found that a target
// whose bucket key and low key match a basis state is that state): its low
// key is compared, and the state array is not read.  kLowTrusted (the pass
// also found every connected state in the basis): the candidate is the
// target, with no compare.
constexpr int kLowCmpState = 0, kLowCmpKey = 1, kLowTrusted = 2;
template <int NW, bool HAS_Z, bool DOT, int G, int CHECK>
__global__ __launch_bounds__(kApplyBlock)
__attribute__((amdgpu_waves_per_eu(
    G >= 8 ? ((CHECK == 2 || (CHECK == 1 && NW == 1)) && !HAS_Z ? 8 : 5) : HAS_Z ? 6 : 8)))
void k_apply_low(
    BasisView b, const OffTerm* __restrict__ off, int n_off,
    const DiagTerm* __restrict__ dg, int n_diag, const double* __restrict__ x,
    double* y, const double* y_in, double yscale,
    const double* __restrict__ yscale_dev, double* __restrict__ partials,
    const double* __restrict__ xs_dev, const double* __restrict__ ys_dev) {
  const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
  if (yscale_dev) yscale *= yscale_dev[0];
  // scales as in k_apply_lane (dot-product instances only)
  const double xs = (DOT && xs_dev) ? xs_dev[0] : 1.0;
  const double ys = (DOT && ys_dev) ? ys_dev[0] : 1.0;
  __shared__ LowTermsLds<NW> tl;
  const int64_t i = static_cast<int64_t>(blk) * kApplyBlock + threadIdx.x;
  const bool live = i < b.dim;
  State<NW> s = {};
  double xi = 0.0, acc = 0.0, prod = 0.0;
  uint32_t ks = 0, ls = 0;
  if (live) {
    s = load_state_cached<NW>(b.states, i);
    xi = x[i] * xs;
    acc = y_in ? yscale * (y_in[i] * ys) : 0.0;
    ks = bucket_key<NW>(b, s);
    ls = low_key<NW>(b, s);
  }
  for (int c0 = 0; c0 < n_off; c0 += kLdsTerms) {
    const int cn = min(kLdsTerms, n_off - c0);
    stage_low_terms<NW>(tl, b, off + c0, cn, c0 > 0);
    if (!live) continue;
    for (int t0 = 0; t0 < cn; t0 += 64) {
      const int tn = min(64, cn - t0);
      uint64_t mask = connect_mask<NW>(off + c0 + t0, tn, s);
      while (mask) {
        // per lookup: term, bucket start, bucket size (0: nothing to find),
        // and below eight lookups the target's low key (with eight it is
        // re-formed from the staged keys where it is compared, which keeps
        // the kernel within the registers of eight waves per SIMD); bucket
        // bounds of all G lookups loaded first
        uint32_t tt[G], lo[G], n[G];
        constexpr bool kKeepLow = G < 8;
        uint32_t r[kKeepLow ? G : 1];
        auto target_low = [&](int g) -> uint32_t {
          if constexpr (kKeepLow) return r[g];
          else return ls ^ tl.key[tt[g]].y;
        };
        bool act[G];
        uint2 p[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          act[g] = mask != 0;
          const uint32_t z = act[g] ? static_cast<uint32_t>(__builtin_clzll(mask)) : 0u;
          tt[g] = t0 + z;
          mask &= ~(uint64_t{1} << 63 >> z);
          const uint2 kx = tl.key[tt[g]];
          if constexpr (kKeepLow) r[g] = ls ^ kx.y;
          p[g] = make_uint2(0u, 0u);
          if (act[g]) __builtin_memcpy(&p[g], b.table + (ks ^ kx.x), sizeof(uint2));
        }
#pragma unroll
        for (int g = 0; g < G; ++g) asm volatile("" : "+v"(p[g].x), "+v"(p[g].y));
        bool more = false;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          lo[g] = p[g].x;
          n[g] = act[g] ? p[g].y - p[g].x : 0u;
          more |= n[g] > 1;
        }
        // interleaved bisection on the low keys down to one candidate: the G
        // probes, then the G updates (a finished lookup has half = 0: no
        // change)
        while (more) {
          uint32_t m[G];
#pragma unroll
          for (int g = 0; g < G; ++g) {
            m[g] = 0;
            if (n[g] > 1) m[g] = b.lowkeys[lo[g] + (n[g] >> 1)];
          }
          // every probe of the group is used only after all were issued
#pragma unroll
          for (int g = 0; g < G; ++g) asm volatile("" : "+v"(m[g]));
          more = false;
#pragma unroll
          for (int g = 0; g < G; ++g) {
            const uint32_t half = n[g] >> 1;
            lo[g] = m[g] <= target_low(g) ? lo[g] + half : lo[g];
            n[g] -= half;
            more |= n[g] > 1;
          }
        }
        // candidates in chunks of up to four: every candidate state and x of
        // a chunk first, then its compares and sums (in term order)
        constexpr int CH = G % 4 == 0 ? 4 : G % 3 == 0 ? 3 : G % 2 == 0 ? 2 : 1;
        static_assert(G % CH == 0, "candidate chunks must tile the lookups");
#pragma unroll
        for (int g0 = 0; g0 < G; g0 += CH) {
          State<NW> f[CH];
          uint32_t fk[CH];
          double xj[CH], c[CH];
#pragma unroll
          for (int u = 0; u < CH; ++u) {
            xj[u] = 0.0;
            c[u] = tl.c[tt[g0 + u]];
            if (n[g0 + u] == 1) {
              if constexpr (CHECK == kLowCmpKey) fk[u] = b.lowkeys[lo[g0 + u]];
              if constexpr (CHECK == kLowCmpState) f[u] = load_state_cached<NW>(b.states, lo[g0 + u]);
              xj[u] = x[lo[g0 + u]];
            }
          }
#pragma unroll
          for (int u = 0; u < CH; ++u) xj[u] *= xs;
#pragma unroll
          for (int u = 0; u < CH; ++u) {
            if (n[g0 + u] == 1 && fabs(xj[u]) > kApplyTol) {
              const int t = static_cast<int>(tt[g0 + u]);
              bool hit = true;
              if constexpr (CHECK == kLowCmpKey) hit = fk[u] == target_low(g0 + u);
              if constexpr (CHECK == kLowCmpState) {
                hit = st_eq<NW>(f[u], staged_target<NW>(tl, s, tt[g0 + u]));
              }
              if (hit) {
                double cu = c[u];
                if constexpr (HAS_Z) {
                  if (parity_notz<NW>(s, off[c0 + t].Z)) cu = -cu;
                }
                acc += cu * xj[u];
              }
            }
          }
        }
      }
    }
  }
  if (live) {
    acc = diag_accumulate<NW>(acc, xi, s, dg, n_diag);
    y[i] = acc;
    if constexpr (DOT) prod = xi * acc;
  }
  if constexpr (DOT) {
    const double bs = block_sum<kApplyBlock>(prod);
    if (threadIdx.x == 0) partials[blk] = bs;
  }
}

// Slot variant: as the lane variant, with each connected state found through
// the slot index under its bucket (bucket bounds, then slots from the
// state's home until an empty slot or a fingerprint match, whose state and x
// are loaded together) instead of a bisection of the bucket.  G lookups per
// lane are carried through the stages together; contributions are added in
// term order, so y is bit-identical to the other variants.  A lookup keeps
// only its bucket start, size and fingerprint, probe position, candidate
// rank and term (the connected state is re-formed from the row and the
// term's flip mask where needed), so four lookups fit the register budget of
// seven waves per SIMD.
template <int NW, bool HAS_Z, bool DOT, int G>
__global__ __launch_bounds__(kApplyBlock) void k_apply_slot(
    BasisView b, const OffTerm* __restrict__ off, int n_off,
    const DiagTerm* __restrict__ dg, int n_diag, const double* __restrict__ x,
    double* y, const double* y_in, double yscale,
    const double* __restrict__ yscale_dev, double* __restrict__ partials,
    const double* __restrict__ xs_dev, const double* __restrict__ ys_dev) {
  const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
  if (yscale_dev) yscale *= yscale_dev[0];
  // x and y_in are read as xs * x and ys * y_in.  Only the dot-product
  // instances (the Lanczos step) take scales; elsewhere they are the
  // constant 1 and the multiplies fold away.
  const double xs = (DOT && xs_dev) ? xs_dev[0] : 1.0;
  const double ys = (DOT && ys_dev) ? ys_dev[0] : 1.0;
  __shared__ TermsLds<NW> tl;
  const bool lds = stage_terms<NW>(tl, off, n_off);
  const int64_t i = static_cast<int64_t>(blk) * kApplyBlock + threadIdx.x;
  double prod = 0.0;
  if (i < b.dim) {
    const State<NW> s = load_state_cached<NW>(b.states, i);
    const double xi = x[i] * xs;
    double acc = y_in ? yscale * (y_in[i] * ys) : 0.0;
    for (int t0 = 0; t0 < n_off; t0 += 64) {
      const int tn = min(64, n_off - t0);
      uint64_t mask = 0;
      for (int t = 0; t < tn; ++t) {
        mask |= static_cast<uint64_t>(term_ok<NW>(off[t0 + t], s)) << t;
      }
      while (mask) {
        // per lookup: stage (bits 8-9: 0 absent, 1 probing, 2 candidate,
        // 3 found) | term offset in the chunk (bits 0-7); bucket start;
        // bucket size << 16 | fingerprint; probe position; candidate rank
        uint32_t tg[G], lo[G], nf[G], p[G], J[G];
        double xj[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const bool act = mask != 0;
          const uint32_t tt = act ? __builtin_ctzll(mask) : 0;
          mask &= mask - 1;
          tg[g] = tt;
          lo[g] = 0;
          nf[g] = 0;
          p[g] = 0;
          J[g] = 0;
          xj[g] = 0.0;
          if (act) {
            const State<NW> key = term_target<NW>(tl, lds, off, s, t0 + tt);
            uint32_t n;
            bucket_bounds(b.table, bucket_key<NW>(b, key), lo[g], n);
            const uint64_t h = slot_hash<NW>(key);
            nf[g] = (n << 16) | slot_fp(h);
            p[g] = slot_home(h, 2 * n);
            tg[g] |= (n ? 1u : 0u) << 8;
          }
        }
        bool more = true;
        while (more) {
          more = false;
          uint32_t e[G];
#pragma unroll
          for (int g = 0; g < G; ++g) {
            e[g] = (tg[g] >> 8) == 1 ? b.slots[2 * static_cast<uint64_t>(lo[g]) + p[g]]
                                     : kSlotEmpty;
          }
#pragma unroll
          for (int g = 0; g < G; ++g) {
            if ((tg[g] >> 8) == 1) {
              if (e[g] == kSlotEmpty) {
                tg[g] &= 0xFFu;
              } else if ((e[g] >> 16) == (nf[g] & 0xFFFFu)) {
                J[g] = lo[g] + (e[g] & 0xFFFFu);
                tg[g] = (tg[g] & 0xFFu) | (2u << 8);
              } else {
                p[g] = p[g] + 1 == 2 * (nf[g] >> 16) ? 0 : p[g] + 1;
                more = true;
              }
            }
          }
          State<NW> f[G];
#pragma unroll
          for (int g = 0; g < G; ++g) {
            if ((tg[g] >> 8) == 2) {
              f[g] = load_state_cached<NW>(b.states, J[g]);
              xj[g] = x[J[g]];
            }
          }
#pragma unroll
          for (int g = 0; g < G; ++g) {
            if ((tg[g] >> 8) == 2) {
              const State<NW> key = term_target<NW>(tl, lds, off, s, t0 + (tg[g] & 0xFFu));
              if (st_eq<NW>(f[g], key)) {
                tg[g] = (tg[g] & 0xFFu) | (3u << 8);
              } else {
                tg[g] = (tg[g] & 0xFFu) | (1u << 8);
                p[g] = p[g] + 1 == 2 * (nf[g] >> 16) ? 0 : p[g] + 1;
                more = true;
              }
            }
          }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) xj[g] *= xs;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if ((tg[g] >> 8) == 3 && fabs(xj[g]) > kApplyTol) {
            const int t = t0 + (tg[g] & 0xFFu);
            double c = lds ? tl.c[t] : off[t].c * off[t].sgn;
            if constexpr (HAS_Z) {
              if (parity_notz<NW>(s, off[t].Z)) c = -c;
            }
            acc += c * xj[g];
          }
        }
      }
    }
    acc = diag_accumulate<NW>(acc, xi, s, dg, n_diag);
    y[i] = acc;
    if constexpr (DOT) prod = xi * acc;
  }
  if constexpr (DOT) {
    const double bs = block_sum<kApplyBlock>(prod);
    if (threadIdx.x == 0) partials[blk] = bs;
  }
}

// Cached variant: the row's connected ranks come from the operator's cached
// connectivity (qsi_op_cache_connectivity), so an apply is a gather with no
// flip tests or searches.  Same terms, order and arithmetic as the lane
// variant, so y is bit-identical.
//
// ALIGNED: the rows are padded to whole groups of four (conn_pad 4), so every
// group the loop loads belongs to the row and no entry needs masking.
template <int NW, bool DOT, int PIPE, bool ALIGNED>
__global__ __launch_bounds__(kApplyBlock) void k_apply_cached(
    BasisView b, const CoefClass* __restrict__ cls, int n_cls,
    const uint64_t* __restrict__ rowptr, const uint32_t* __restrict__ cj,
    const uint8_t* __restrict__ cm, const DiagTerm* __restrict__ dg, int n_diag,
    const double* __restrict__ x, double* y, const double* y_in, double yscale,
    const double* __restrict__ yscale_dev, double* __restrict__ partials,
    const double* __restrict__ xs_dev, const double* __restrict__ ys_dev) {
  const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
  if (yscale_dev) yscale *= yscale_dev[0];
  // x and y_in are read as xs * x and ys * y_in.  Only the dot-product
  // instances (the Lanczos step) take scales; elsewhere they are the
  // constant 1 and the multiplies fold away.
  const double xs = (DOT && xs_dev) ? xs_dev[0] : 1.0;
  const double ys = (DOT && ys_dev) ? ys_dev[0] : 1.0;
  double cc[kMaxCoefClasses];
#pragma unroll
  for (int k = 0; k < kMaxCoefClasses; ++k) cc[k] = k < n_cls ? cls[k].c : 0.0;
  const int64_t i = static_cast<int64_t>(blk) * kApplyBlock + threadIdx.x;
  double prod = 0.0;
  if (i < b.dim) {
    const double xi = x[i] * xs;
    double acc = y_in ? yscale * (y_in[i] * ys) : 0.0;
    // the row's state (for the diagonal) is loaded before the gathers so its
    // latency overlaps theirs
    const State<NW> si = load_state_cached<NW>(b.states, i);
    const uint64_t e0 = rowptr[i], e1 = rowptr[i + 1];
    // columns and class bytes come four at a time from 16- and 4-byte aligned
    // groups (the arrays are allocated in whole groups); without padding,
    // entries of the neighbouring rows in the first and last group are masked
    // off
    for (uint64_t e = ALIGNED ? e0 : (e0 & ~uint64_t{3}); e < e1; e += PIPE) {
      uint32_t J[PIPE];
      uint8_t mt[PIPE];
      double xj[PIPE];
#pragma unroll
      for (int u = 0; u < PIPE; u += 4) {
        const uint64_t g = e + u;
        const bool in = g < e1;
        const uint4 j4 = in ? reinterpret_cast<const uint4*>(cj)[g >> 2]
                           : make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu);
        const uint32_t m4 = in ? reinterpret_cast<const uint32_t*>(cm)[g >> 2] : 0u;
        const uint32_t jv[4] = {j4.x, j4.y, j4.z, j4.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool mine = ALIGNED || (g + k >= e0 && g + k < e1);
          J[u + k] = mine ? jv[k] : 0xFFFFFFFFu;
          mt[u + k] = static_cast<uint8_t>(m4 >> (8 * k));
        }
      }
#pragma unroll
      for (int u = 0; u < PIPE; ++u) xj[u] = J[u] != 0xFFFFFFFFu ? x[J[u]] : 0.0;
      // the scale is applied after every gather of the group has been issued
#pragma unroll
      for (int u = 0; u < PIPE; ++u) xj[u] *= xs;
#pragma unroll
      for (int u = 0; u < PIPE; ++u) {
        if (J[u] != 0xFFFFFFFFu && fabs(xj[u]) > kApplyTol) {
          const int k = mt[u] & 0x7F;
          double c = cc[0];
#pragma unroll
          for (int q = 1; q < kMaxCoefClasses; ++q)
            if (k == q) c = cc[q];
          if (mt[u] & 0x80) c = -c;
          acc += c * xj[u];
        }
      }
    }
    if (n_diag > 0) acc = diag_accumulate<NW>(acc, xi, si, dg, n_diag);
    y[i] = acc;
    if constexpr (DOT) prod = xi * acc;
  }
  if constexpr (DOT) {
    const double bs = block_sum<kApplyBlock>(prod);
    if (threadIdx.x == 0) partials[blk] = bs;
  }
}

// Hash variant (default when the basis has a hash index): as the lane
// variant, but each connected state is found with one probe of the hash index
// (one 16-byte slot, ~1.2 probes on average) instead of a bucket bisection.
template <int NW, bool HAS_Z, bool DOT, int G>
__global__ __launch_bounds__(kApplyBlock) void k_apply_hash(
    BasisView b, HashView hv, const OffTerm* __restrict__ off, int n_off,
    const DiagTerm* __restrict__ dg, int n_diag, const double* __restrict__ x,
    double* y, const double* y_in, double yscale,
    const double* __restrict__ yscale_dev, double* __restrict__ partials,
    const double* __restrict__ xs_dev, const double* __restrict__ ys_dev) {
  const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
  if (yscale_dev) yscale *= yscale_dev[0];
  // x and y_in are read as xs * x and ys * y_in.  Only the dot-product
  // instances (the Lanczos step) take scales; elsewhere they are the
  // constant 1 and the multiplies fold away.
  const double xs = (DOT && xs_dev) ? xs_dev[0] : 1.0;
  const double ys = (DOT && ys_dev) ? ys_dev[0] : 1.0;
  const int64_t i = static_cast<int64_t>(blk) * kApplyBlock + threadIdx.x;
  double prod = 0.0;
  if (i < b.dim) {
    const State<NW> s = load_state_cached<NW>(b.states, i);
    const double xi = x[i] * xs;
    double acc = y_in ? yscale * (y_in[i] * ys) : 0.0;
    for (int t0 = 0; t0 < n_off; t0 += 64) {
      const int tn = min(64, n_off - t0);
      uint64_t mask = 0;
      for (int t = 0; t < tn; ++t) {
        mask |= static_cast<uint64_t>(term_ok<NW>(off[t0 + t], s)) << t;
      }
      while (mask) {
        int tt[G];
        bool live[G];
        State<NW> key[G];
        uint64_t pos[G];
        int64_t J[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          live[g] = mask != 0;
          tt[g] = live[g] ? t0 + __builtin_ctzll(mask) : t0;
          mask &= mask - 1;
          key[g] = xor_state<NW>(s, off[tt[g]].X);
          pos[g] = hash_home<NW>(key[g], hv.hbits);
          J[g] = -1;
        }
        // interleaved probing
        bool more = true;
        while (more) {
          more = false;
#pragma unroll
          for (int g = 0; g < G; ++g) {
            if (live[g]) {
              uint64_t rk, k0, k1 = 0;
              if constexpr (NW == 1) {
                const ulonglong2 e = hv.slots[pos[g]];
                k0 = e.x;
                rk = e.y;
              } else {
                const ulonglong2 e = hv.slots[2 * pos[g]];
                const ulonglong2 r = hv.slots[2 * pos[g] + 1];
                k0 = e.x;
                k1 = e.y;
                rk = r.x;
              }
              bool eq = (k0 == key[g].w[0]);
              if constexpr (NW == 2) eq = eq && (k1 == key[g].w[1]);
              if (rk == kHashEmpty) {
                live[g] = false;
              } else if (eq) {
                J[g] = static_cast<int64_t>(rk);
                live[g] = false;
              } else {
                pos[g] = (pos[g] + 1) & hv.mask;
                more = true;
              }
            }
          }
        }
        double xj[G];
#pragma unroll
        for (int g = 0; g < G; ++g) xj[g] = (J[g] >= 0) ? x[J[g]] : 0.0;
#pragma unroll
        for (int g = 0; g < G; ++g) xj[g] *= xs;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if (J[g] >= 0 && fabs(xj[g]) > kApplyTol) {
            const OffTerm& T = off[tt[g]];
            double c = T.c * T.sgn;
            if constexpr (HAS_Z) {
              if (parity_notz<NW>(s, T.Z)) c = -c;
            }
            acc += c * xj[g];
          }
        }
      }
    }
    acc = diag_accumulate<NW>(acc, xi, s, dg, n_diag);
    y[i] = acc;
    if constexpr (DOT) prod = xi * acc;
  }
  if constexpr (DOT) {
    const double bs = block_sum<kApplyBlock>(prod);
    if (threadIdx.x == 0) partials[blk] = bs;
  }
}

// ----------------------------------------------------------------------------
// Window variant.  A wavefront owns 128 consecutive rows, two per lane (lane l
// holds rows l and 64 + l).  For one term, the rows it connects share the
// term's projector bits, so their targets s ^ X increase with the row, and
// every basis state between the first and the last target that the reversed
// flip connects (its projector bits are v ^ X) is the target of one of those
// rows: the p-th connected row's target is the p-th such state.  So a
// wavefront looks up two ranks per term (first and last target) instead of one
// per row and term, reads the basis states and x between them with coalesced
// loads (a window: 128 ranks, two per lane), and matches rows to states by
// counting bits of lane masks, with no search and no key compare.  On the
// 64-spin ice basis 128 rows connect through 39 of the 128 terms, 36 rows each,
// and a term's targets span 80 ranks at the median (a quarter span more than
// one window).  Per batch of up to 64 terms that the bits shared by all 128
// rows do not rule out:
//   1. one compare per term and 64 rows gives the row masks, kept in lane q
//      for the q-th term;
//   2. lane q looks up the ranks of its first and last target (both
//      bisections in flight together) and lists its windows in LDS;
//   3. the windows are taken in order with P of them in flight; a window's
//      matching lanes write x to LDS compacted, the term's rows read it back
//      by their own index, and add it in term order.
// A target may be missing from the basis, or a state in the range may have no
// partner row (a sector the terms do not close).  CHECK also passes the
// matched states through LDS and compares them with the rows' targets; a term
// with a mismatch (also one that flips a spin its projector leaves open, whose
// targets do not keep the rows' order), an end that is not found or a range
// beyond kWinMax windows is done by per-row lookups.  Without CHECK (every
// connected state is in the basis, every flip's reverse is a term too, every
// flipped spin under the projector) only the last can be.
// What bounds it on two-word states is the L2's misses: states and x of a window
// are 24 bytes a rank, a third of them matched, and the rows in flight on an XCD
// reach more ranks than its L2 holds (96 spins: 1.98 TB per apply at 7.0 TB/s, 39 %
// hits; 72 spins 8.4 GB at 7 TB/s).  At 64 spins no unit is at its limit (0.80 GB at
// 4.4 TB/s, texture units busy 70 and 88 %, VALU issue 69 %).  Wider tiles,
// fewer or more windows in flight and fewer wavefronts measured no better.
// Against four lookups in flight per row (LANE4, no low keys): 64 spins 266 ->
// 200 us, 72 spins 2.09 -> 1.47 ms, 80 spins 17.6 -> 10.1 ms, 96 spins 543 -> 301 ms.
// Contributions are added in term order, then the diagonal, and the dot
// product's partials are those of 256 rows, exactly as in the lane variant, so
// y and the partials are bit-identical.
// ----------------------------------------------------------------------------

constexpr int kWavesPerBlock = kApplyBlock / 64;
// windows in flight per wavefront, and wavefronts per SIMD
// (7 wavefronts of 4 windows measured best at 64 spins: 8 x 2 188, 6 x 4 200, 4 x 8
// 220 us)
template <int NW, bool CHECK>
constexpr int kWinItems = NW == 1 ? 4 : 2;
template <int NW, bool CHECK>
constexpr int kWinWaves = NW == 1 ? 7 : 5;
// AUTO takes the window kernel from this many states and (against kernels that
// compare) terms on; against LOW8 on two-word states only from the second
constexpr int64_t kWinMinDim = int64_t{1} << 21;
constexpr int64_t kWinMinDimLow2 = int64_t{1} << 28;
constexpr int kWinMinTerms = 32;
// and the row kernel up to this many states, for few terms up to the second number
constexpr int64_t kRowMaxDim = int64_t{1} << 14;
constexpr int64_t kRowMaxDimFew = int64_t{1} << 12;
constexpr int kRowMinTerms = 16;
constexpr int kWinRows = 128;  // rows of a wavefront, and ranks of a window
constexpr int kWinMax = 8;     // windows of one term (a wider range: per-row lookups)
// Windows of a term whose first and last target have ranks la and lz in a basis of
// dim states; 0 (per-row lookups) if they are too many, pass the end of the
// arrays, or the targets do not keep the rows' order.  With la <= lz < dim <=
// 2^32 - 512 the end of the last one does not pass 2^32.
__host__ __device__ constexpr uint32_t win_count(uint32_t la, uint32_t lz, uint32_t dim) {
  const uint32_t n = (lz - la) / kWinRows + 1;
  return la <= lz && n <= kWinMax && la + n * kWinRows <= dim ? n : 0;
}
static_assert(win_count(0, 127, 128) == 1 && win_count(1, 127, 128) == 0 &&
              win_count(0, 128, 256) == 2 && win_count(0, 1024, 4096) == 0 &&
              win_count(5, 4, 4096) == 0);
// a last target far before the first one wraps to a short range there
static_assert(win_count(0xFFFFFDFEu, 0, 0xFFFFFE00u) == 0 &&
              win_count(0xFFFFFDFFu, 1, 0xFFFFFE00u) == 0);
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t readlane32(uint32_t v, int lane) {
  return __builtin_amdgcn_readlane(v, lane);
}

// v with lane `lane`'s value replaced by val (val and lane wave-uniform); the
// compiler intrinsic, which has no builtin of its own.
extern "C" __device__ int qsi_amdgcn_writelane(int val, int lane, int v) __asm(
    "llvm.amdgcn.writelane.i32");

__device__ __forceinline__ uint32_t writelane32(uint32_t val, int lane, uint32_t v) {
  return static_cast<uint32_t>(
      qsi_amdgcn_writelane(static_cast<int>(val), lane, static_cast<int>(v)));
}

__device__ __forceinline__ uint64_t first_lane64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

// OR of v over the wavefront (row shifts and row broadcasts, result uniform).
__device__ __forceinline__ uint32_t wave_or32(uint32_t v) {
  v |= __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v |= __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v |= __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v |= __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v |= __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v |= __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return readlane32(v, 63);
}

__device__ __forceinline__ uint64_t wave_or64(uint64_t v) {
  const uint32_t lo = wave_or32(static_cast<uint32_t>(v));
  const uint32_t hi = wave_or32(static_cast<uint32_t>(v >> 32));
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

// Set bits of m below this lane, plus base.
__device__ __forceinline__ uint32_t lanes_below(uint64_t m, uint32_t base) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), base));
}

// Inclusive sum of v over the wavefront's lanes.
__device__ __forceinline__ uint32_t wave_scan_add(uint32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}

// Elements 2 lane and 2 lane + 1 from a wave-uniform address, read in 16-byte
// pieces (8-byte aligned).  The empty asm keeps the address in scalar registers
// (the load adds the lane's offset); otherwise the compiler adds in the vector
// unit.
template <typename T>
__device__ __forceinline__ void load_window(const void* p, int lane, T (&v)[2]) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(8)));
  typedef const __attribute__((address_space(1))) char* gptr;
  gptr g = (gptr)p;
  asm("" : "+s"(g));
  constexpr uint32_t kBytes = 2 * sizeof(T);
  u32x4 piece[kBytes / 16];
#pragma unroll
  for (uint32_t k = 0; k < kBytes / 16; ++k)
    piece[k] = *(const __attribute__((address_space(1))) u32x4*)(
        g + static_cast<uint32_t>(lane) * kBytes + 16 * k);
  __builtin_memcpy(&v[0], &piece[0], kBytes);
}

// Lanes whose state the term connects, and whose state its reverse connects.
template <int NW>
__device__ __forceinline__ uint64_t rec_lanes(const State<NW>& s, const TermRec<NW>& A) {
  uint64_t b = ~uint64_t{0};
#pragma unroll
  for (int w = 0; w < NW; ++w) b &= __builtin_amdgcn_ballot_w64((s.w[w] & A.m[w]) == A.v[w]);
  return b;
}
template <int NW>
__device__ __forceinline__ uint64_t rec_hits(const State<NW>& s, const TermRec<NW>& A) {
  uint64_t b = ~uint64_t{0};
#pragma unroll
  for (int w = 0; w < NW; ++w) b &= __builtin_amdgcn_ballot_w64((s.w[w] & A.m[w]) == A.u[w]);
  return b;
}

// The listed terms (term t_k in lane k, nq of them; also in LDS at list[k].x, as
// a lane may not read a register of one that has finished) by per-row lookups, G in
// flight per lane, as the lane variant's rounds: acc gains this lane's row's
// contributions.  What a batch takes when most of its terms lead out of the
// basis.
template <int NW, bool HAS_Z>
__device__ __forceinline__ void win_batch_by_rows(
    const BasisView& b, const OffTerm* __restrict__ off, const TermPlanes& tp,
    const TermRec<NW>* __restrict__ tr, int t, const uint2* list, int nq,
    const double* __restrict__ x, double xs, const State<NW>& s, uint32_t ks, bool row_ok, double& acc) {
  constexpr int G = NW == 1 ? 4 : 2;
  uint32_t word[2] = {0, 0};
  for (int k = 0; k < 64; ++k) {
    uint64_t m = 0;
    if (k < nq) m = rec_lanes<NW>(s, tr[readlane32(t, k)]);
    word[k >> 5] = shift_in_lane(word[k >> 5], m);
  }
  uint64_t mask = row_ok ? static_cast<uint64_t>(word[0]) << 32 | word[1] : 0;
  while (mask) {
    int tt[G];
    uint32_t lo[G], n[G];
    State<NW> key[G];
    uint2 p[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const bool act = mask != 0;
      const int z = act ? __builtin_clzll(mask) : 0;
      mask &= ~(uint64_t{1} << 63 >> z);
      tt[g] = static_cast<int>(list[z].x);
      p[g] = make_uint2(0u, 0u);
#pragma unroll
      for (int w = 0; w < NW; ++w) key[g].w[w] = s.w[w] ^ tp.X(w)[tt[g]];
      if (act)
        __builtin_memcpy(&p[g], b.table + (ks ^ static_cast<uint32_t>(tp.key()[tt[g]])),
                         sizeof(uint2));
    }
#pragma unroll
    for (int g = 0; g < G; ++g) asm volatile("" : "+v"(p[g].x), "+v"(p[g].y));
    bool more = false;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      lo[g] = p[g].x;
      n[g] = p[g].y - p[g].x;
      more |= n[g] > 1;
    }
    while (more) {
      State<NW> m[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        m[g] = State<NW>{};
        if (n[g] > 1) m[g] = load_state_cached<NW>(b.states, lo[g] + (n[g] >> 1));
      }
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int w = 0; w < NW; ++w) asm volatile("" : "+v"(m[g].w[w]));
      more = false;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const uint32_t half = n[g] >> 1;
        lo[g] = st_le<NW>(m[g], key[g]) ? lo[g] + half : lo[g];
        n[g] -= half;
        more |= n[g] > 1;
      }
    }
    double xj[G];
    State<NW> f[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      xj[g] = 0.0;
      if (n[g] == 1) {
        f[g] = load_state_cached<NW>(b.states, lo[g]);
        xj[g] = x[lo[g]];
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      xj[g] *= xs;
      if (n[g] == 1 && st_eq<NW>(f[g], key[g]) && fabs(xj[g]) > kApplyTol) {
        double cg = tr[tt[g]].c;
        if constexpr (HAS_Z) {
          if (parity_notz<NW>(s, off[tt[g]].Z)) cg = -cg;
        }
        acc += cg * xj[g];
      }
    }
  }
}

template <int NW, bool HAS_Z, bool DOT, bool CHECK>
__global__ __launch_bounds__(kApplyBlock)
__attribute__((amdgpu_waves_per_eu(kWinWaves<NW, CHECK>))) void k_apply_win(
    BasisView b, const OffTerm* __restrict__ off, int n_off, TermPlanes tp,
    const TermRec<NW>* __restrict__ tr, const DiagTerm* __restrict__ dg, int n_diag, const double* __restrict__ x,
    double* y, const double* y_in, double yscale,
    const double* __restrict__ yscale_dev, double* __restrict__ partials,
    const double* __restrict__ xs_dev, const double* __restrict__ ys_dev) {
  constexpr int P = kWinItems<NW, CHECK>;
  constexpr int R = 2;  // rows of a lane, and ranks of a lane's window share
  // the 64 listed windows are whole groups of P: a group past lane 63 would wrap
  static_assert(64 % P == 0, "P divides the windows listed at a time");
  // a term's matched x (and states), compacted: fewer than 128 before its last
  // window, and at most 128 more from that one
  constexpr int kEx = 2 * kWinRows;
  __shared__ double ex[kWavesPerBlock][kEx];
  __shared__ State<NW> exs[CHECK ? kWavesPerBlock : 1][CHECK ? kEx : 1];
  __shared__ int list[kWavesPerBlock][128];    // terms not ruled out
  __shared__ uint2 item[kWavesPerBlock][64];   // windows: first rank, flags
  // flags of a window: first / last window of its term, term for per-row
  // lookups; the last lane to read in bits 3-8; the term from bit 9 on
  constexpr uint32_t kFirst = 1u, kLast = 2u, kSlow = 4u;
  constexpr int kLane = 3, kTerm = 9;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
  if (yscale_dev) yscale *= yscale_dev[0];
  // x and y_in are read as xs * x and ys * y_in.  Only the dot-product
  // instances (the Lanczos step) take scales; elsewhere they are the
  // constant 1 and the multiplies fold away.
  const double xs = (DOT && xs_dev) ? xs_dev[0] : 1.0;
  const double ys = (DOT && ys_dev) ? ys_dev[0] : 1.0;
  const int64_t r0 = (static_cast<int64_t>(blk) * kWavesPerBlock + wid) * kWinRows;
  double prod[R] = {0.0, 0.0};
  if (r0 < b.dim) {  // wave-uniform
    State<NW> s[R];
    double acc[R];
    uint32_t ks[R];
    uint64_t rows[R];  // lanes with a row
    uint64_t same[NW], s0[NW];  // the bits all rows share; the first row
#pragma unroll
    for (int q = 0; q < R; ++q) {
      // lanes past the end hold the first row's state and connect to nothing
      const int64_t i = r0 + 64 * q + lane;
      const int64_t left = b.dim - (r0 + 64 * q);
      rows[q] = left >= 64 ? ~uint64_t{0} : left > 0 ? ~uint64_t{0} >> (64 - left) : 0;
      s[q] = load_state_cached<NW>(b.states, i < b.dim ? i : r0);
      acc[q] = 0.0;
      if (y_in && i < b.dim) acc[q] = yscale * (y_in[i] * ys);
      ks[q] = bucket_key<NW>(b, s[q]);
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      s0[w] = first_lane64(s[0].w[w]);
      same[w] = ~wave_or64((s[0].w[w] ^ s0[w]) | (s[1].w[w] ^ s0[w]));
    }
    const uint32_t dim32 = static_cast<uint32_t>(b.dim);
    const uint32_t top = dim32 - kWinRows;  // the basis has at least kWinRows states
    int n_list = 0;
    for (int t0 = 0; t0 < n_off || n_list > 0; t0 += 64) {
      if (t0 < n_off) {
        // terms that the shared bits do not rule out (the planes are padded
        // to whole chunks)
        const int t = t0 + lane;
        bool alive = t < n_off;
#pragma unroll
        for (int w = 0; w < NW; ++w)
          alive = alive && ((s0[w] ^ tp.v(w)[t]) & tp.m(w)[t] & same[w]) == 0;
        const uint64_t live = __builtin_amdgcn_ballot_w64(alive);
        const uint32_t at = lanes_below(live, n_list);
        if (alive) list[wid][at] = t;
        n_list += __popcll(live);
        if (n_list < 64 && t0 + 64 < n_off) continue;
        wave_sync();
      }
      if (n_list == 0) break;
      const int nq = min(n_list, 64);
      // lanes past the list hold the record that connects nothing
      const int t = lane < nq ? list[wid][lane] : n_off;
      n_list -= nq;
      if (n_list > 0) {  // the rest moves to the front
        const int t2 = list[wid][64 + lane];
        wave_sync();
        list[wid][lane] = t2;
      }
      wave_sync();
      // 1. row masks of the q-th term in lane q
      uint32_t mlo[R] = {0, 0}, mhi[R] = {0, 0};
      for (int k0 = 0; k0 < nq; k0 += 4) {
        TermRec<NW> A[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) A[u] = tr[readlane32(t, k0 + u)];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
          for (int q = 0; q < R; ++q) {
            const uint64_t mk = rec_lanes<NW>(s[q], A[u]) & rows[q];
            mlo[q] = writelane32(static_cast<uint32_t>(mk), k0 + u, mlo[q]);
            mhi[q] = writelane32(static_cast<uint32_t>(mk >> 32), k0 + u, mhi[q]);
          }
        }
      }
      // 2. ranks of the first and the last connected row's targets
      const bool a_hi = (mlo[0] | mhi[0]) == 0, z_hi = (mlo[1] | mhi[1]) != 0;
      const uint64_t ma = a_hi ? static_cast<uint64_t>(mhi[1]) << 32 | mlo[1]
                               : static_cast<uint64_t>(mhi[0]) << 32 | mlo[0];
      const uint64_t mz = z_hi ? static_cast<uint64_t>(mhi[1]) << 32 | mlo[1]
                               : static_cast<uint64_t>(mhi[0]) << 32 | mlo[0];
      const bool has = ma != 0;
      const int ra = has ? __builtin_ctzll(ma) : 0, rz = has ? 63 - __builtin_clzll(mz) : 0;
      State<NW> ka, kz;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const uint64_t X = tp.X(w)[t];
        const uint64_t a0 = __shfl(s[0].w[w], ra, 64), a1 = __shfl(s[1].w[w], ra, 64);
        const uint64_t z0 = __shfl(s[0].w[w], rz, 64), z1 = __shfl(s[1].w[w], rz, 64);
        ka.w[w] = (a_hi ? a1 : a0) ^ X;
        kz.w[w] = (z_hi ? z1 : z0) ^ X;
      }
      const uint32_t kx = static_cast<uint32_t>(tp.key()[t]);
      const uint32_t ba0 = __shfl(ks[0], ra, 64), ba1 = __shfl(ks[1], ra, 64);
      const uint32_t bz0 = __shfl(ks[0], rz, 64), bz1 = __shfl(ks[1], rz, 64);
      uint2 pa = make_uint2(0u, 0u), pz = make_uint2(0u, 0u);
      if (has) {
        __builtin_memcpy(&pa, b.table + ((a_hi ? ba1 : ba0) ^ kx), sizeof(uint2));
        __builtin_memcpy(&pz, b.table + ((z_hi ? bz1 : bz0) ^ kx), sizeof(uint2));
      }
      asm volatile("" : "+v"(pa.x), "+v"(pa.y), "+v"(pz.x), "+v"(pz.y));
      uint32_t la = pa.x, na = pa.y - pa.x, lz = pz.x, nz = pz.y - pz.x;
      while (na > 1 || nz > 1) {
        State<NW> fa{}, fz{};
        if (na > 1) fa = load_state_cached<NW>(b.states, la + (na >> 1));
        if (nz > 1) fz = load_state_cached<NW>(b.states, lz + (nz >> 1));
#pragma unroll
        for (int w = 0; w < NW; ++w) asm volatile("" : "+v"(fa.w[w]), "+v"(fz.w[w]));
        const uint32_t ha = na >> 1, hz = nz >> 1;
        la = st_le<NW>(fa, ka) ? la + ha : la;
        lz = st_le<NW>(fz, kz) ? lz + hz : lz;
        na -= ha;
        nz -= hz;
      }
      bool good = has;
      if constexpr (CHECK) {
        good = na == 1 && nz == 1;
        if (good) {
          const State<NW> fa = load_state_cached<NW>(b.states, la);
          const State<NW> fz = load_state_cached<NW>(b.states, lz);
          good = st_eq<NW>(fa, ka) && st_eq<NW>(fz, kz);
        }
      }
      uint32_t n_win = win_count(la, lz, dim32);
      good = good && n_win != 0;
      if constexpr (CHECK) {
        const int bad = __popcll(__builtin_amdgcn_ballot_w64(has && !good));
        if (2 * bad > __popcll(__builtin_amdgcn_ballot_w64(has))) {
          item[wid][lane] = make_uint2(static_cast<uint32_t>(t), 0u);
          wave_sync();
#pragma unroll
          for (int q = 0; q < R; ++q)
            win_batch_by_rows<NW, HAS_Z>(b, off, tp, tr, t, item[wid], nq, x, xs, s[q], ks[q],
                                         __builtin_amdgcn_inverse_ballot_w64(rows[q]), acc[q]);
          wave_sync();
          continue;
        }
      }
      n_win = good ? n_win : has ? 1u : 0u;
      const uint32_t end = wave_scan_add(n_win);
      const int n_items = static_cast<int>(readlane32(end, 63));
      // contribution of term tt to this lane's row q
      auto add = [&](int q, uint32_t tt, double c, double xj) {
        if constexpr (HAS_Z) {
          if (parity_notz<NW>(s[q], off[tt].Z)) c = -c;
          if (fabs(xj) > kApplyTol) acc[q] += c * xj;
        } else {
          // under a branch: as a select it costs two more vector instructions
          if (fabs(xj) > kApplyTol)
            asm volatile("v_fma_f64 %0, %1, %2, %0" : "+v"(acc[q]) : "v"(xj), "s"(c));
        }
      };
      // 3. the windows, 64 listed at a time (all of this loop's control is
      //    wave-uniform)
      uint32_t base = 0;  // matches in the current term's windows so far
      for (int i0 = 0; i0 < n_items; i0 += 64) {
        for (uint32_t w = 0; w < n_win; ++w) {
          const uint32_t id = end - n_win + w - i0;
          if (id < 64) {
            item[wid][id] = make_uint2(
                min(la + w * kWinRows, top),  // below top unless the term is slow
                static_cast<uint32_t>(t) << kTerm | (w == 0 ? kFirst : 0u) |
                    (w + 1 == n_win ? kLast : 0u) | (good ? 0u : kSlow) |
                    (min(lz - la - w * kWinRows, kWinRows - 1u) >> 1) << kLane);
          }
        }
        wave_sync();
        const int n = min(n_items - i0, 64);
        // entries past the end hold the term that matches nothing
        const uint2 it = lane < n ? item[wid][lane]
                                  : make_uint2(0u, static_cast<uint32_t>(n_off) << kTerm);
        wave_sync();
        State<NW> ws[P][R];
        double wx[P][R];
        auto issue = [&](int p, int id) {
          // no load is under a condition: it could not be counted, only waited
          // for with all others.  Lanes past the last target read its line again
          // and match after every row's state.
          const uint32_t from = readlane32(it.x, id & 63);
          const int wl = min(lane, static_cast<int>(readlane32(it.y, id & 63) >> kLane & 63));
          load_window<State<NW>>(b.states + static_cast<int64_t>(from) * NW, wl, ws[p]);
          load_window<double>(x + from, wl, wx[p]);
          // the order of the windows' loads is what their waits count
          __builtin_amdgcn_sched_barrier(0);
        };
        // a term by per-row lookups
        auto by_rows = [&](int tt, const TermRec<NW>& A) {
#pragma unroll 1
          for (int q = 0; q < R; ++q) {
            const State<NW> sq = q == 0 ? s[0] : s[1];
            if (__builtin_amdgcn_inverse_ballot_w64(rec_lanes<NW>(sq, A) & (q == 0 ? rows[0] : rows[1]))) {
              const State<NW> want = xor_state<NW>(sq, off[tt].X);
              const int64_t r = basis_lookup<NW>(b, want);
              const double xj = r >= 0 ? x[r] * xs : 0.0;
              if (r >= 0 && q == 0) add(0, tt, A.c, xj);
              if (r >= 0 && q == 1) add(1, tt, A.c, xj);
            }
          }
        };
#pragma unroll
        for (int p = 0; p < P; ++p) issue(p, p);
        for (int id0 = 0; id0 < n; id0 += P) {
#pragma unroll
          for (int p = 0; p < P; ++p) {
            const uint32_t f = readlane32(it.y, id0 + p);
            const int tt = static_cast<int>(f >> kTerm);
            const TermRec<NW> A = tr[tt];
            if (f & kSlow) {
              by_rows(tt, A);
            } else {
              if (f & kFirst) base = 0;
              uint64_t hit[R];
#pragma unroll
              for (int q = 0; q < R; ++q) hit[q] = rec_hits<NW>(ws[p][q], A);  // ranks 2 l + q
              uint32_t at = lanes_below(hit[1], lanes_below(hit[0], base));
              if (__builtin_amdgcn_inverse_ballot_w64(hit[0])) {
                ex[wid][at] = wx[p][0];
                if constexpr (CHECK) exs[wid][at] = ws[p][0];
                ++at;
              }
              if (__builtin_amdgcn_inverse_ballot_w64(hit[1])) {
                ex[wid][at] = wx[p][1];
                if constexpr (CHECK) exs[wid][at] = ws[p][1];
              }
              if (!(f & kLast)) {
                base += static_cast<uint32_t>(__popcll(hit[0]) + __popcll(hit[1]));
                if constexpr (CHECK) {
                  // no row reads past entry 127: more matches than that
                  // (without a partner row each) only need to stay inside
                  base = base < kWinRows ? base : kWinRows;
                }
              } else {
                wave_sync();
                uint64_t msk[R];
                double xj[R];
                uint64_t bad = 0;
#pragma unroll
                for (int q = 0; q < R; ++q) {
                  msk[q] = rec_lanes<NW>(s[q], A) & rows[q];
                  const uint32_t from = lanes_below(msk[q], q == 0 ? 0u : __popcll(msk[0]));
                  xj[q] = ex[wid][from];
                  if constexpr (CHECK) {
                    const State<NW> fs = exs[wid][from];
                    const State<NW> want = xor_state<NW>(s[q], off[tt].X);
                    bad |= msk[q] & ~__builtin_amdgcn_ballot_w64(st_eq<NW>(fs, want));
                  }
                }
                if (CHECK && bad != 0) {
                  by_rows(tt, A);
                } else {
#pragma unroll
                  for (int q = 0; q < R; ++q)
                    if (__builtin_amdgcn_inverse_ballot_w64(msk[q])) add(q, tt, A.c, xj[q] * xs);
                }
                wave_sync();
              }
            }
            issue(p, id0 + p + P);
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int64_t i = r0 + 64 * q + lane;
      if (i < b.dim) {
        const double xi = x[i] * xs;
        acc[q] = diag_accumulate<NW>(acc[q], xi, s[q], dg, n_diag);
        y[i] = acc[q];
        if constexpr (DOT) prod[q] = xi * acc[q];
      }
    }
  }
  if constexpr (DOT) {
    // one partial per 256 rows, summed as block_sum does
    __shared__ double red[kWavesPerBlock * R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double v = wave_sum(prod[q]);
      if (lane == 0) red[wid * R + q] = v;
    }
    __syncthreads();
    constexpr int kPer = kApplyBlock / 64;  // 64-row sums of one partial
    const int64_t pb = static_cast<int64_t>(blk) * R + threadIdx.x;
    if (threadIdx.x < R && pb * kApplyBlock < b.dim) {
      double v = 0.0;
#pragma unroll
      for (int w = 0; w < kPer; ++w) v += red[threadIdx.x * kPer + w];
      partials[pb] = v;
    }
  }
}


// ============================================================================
// Connectivity (row-major triplets of the off-diagonal part + diagonal)
// ============================================================================

template <int NW>
__global__ void k_conn(BasisView b, const OffTerm* __restrict__ off, int n_off,
                       const DiagTerm* __restrict__ dg, int n_diag,
                       const int64_t* __restrict__ offsets,
                       int64_t* __restrict__ counts, int64_t* __restrict__ rows,
                       int64_t* __restrict__ cols, double* __restrict__ vals,
                       double* __restrict__ diag) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= b.dim) return;
  const State<NW> s = load_state_cached<NW>(b.states, i);
  int64_t pos = offsets ? offsets[i] : 0;
  int64_t cnt = 0;
  for (int t = 0; t < n_off; ++t) {
    const OffTerm& T = off[t];
    if (!term_ok<NW>(T, s)) continue;
    const int64_t J = basis_lookup<NW>(b, xor_state<NW>(s, T.X));
    if (J < 0) continue;
    double c = T.c * T.sgn;
    if (parity_notz<NW>(s, T.Z)) c = -c;
    if (!(fabs(c) > kSparseTol)) continue;
    if (offsets) {
      rows[pos] = i;
      cols[pos] = J;
      vals[pos] = c;
      ++pos;
    }
    ++cnt;
  }
  if (counts) counts[i] = cnt;
  if (diag) diag[i] = diag_accumulate<NW>(0.0, 1.0, s, dg, n_diag);
}

// ============================================================================
// Streaming FP64 vector kernels
// ============================================================================

constexpr int kVecBlock = 256;

inline int vec_blocks(int64_t n) {
  int64_t nb = (n + kVecBlock * 4 - 1) / (kVecBlock * 4);
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(nb, 8192)));
}

// Workgroups of the projection passes that leave their sums to a kernel of
// their own: about 16 rows per thread, but at least 1024 workgroups while there
// are 4 rows per thread to give them.
inline int proj_blocks(int64_t n) {
  const int64_t want = (n + kVecBlock * 16 - 1) / (kVecBlock * 16);
  return static_cast<int>(std::min<int64_t>(vec_blocks(n), std::max<int64_t>(want, 1024)));
}

// The grid-stride dot, axpy-norm and device-scalar scale kernels take
// kVecUnroll of a thread's elements per round, all loads first, and
// accumulate in element order (the sums are the ones a one-element loop
// gives).
constexpr int kVecUnroll = 8;

__global__ __launch_bounds__(kVecBlock) void k_dot_partial(
    const double* __restrict__ a, const double* __restrict__ b, int64_t n,
    double* __restrict__ partials) {
  double v = 0.0;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kVecBlock;
  int64_t i = static_cast<int64_t>(blockIdx.x) * kVecBlock + threadIdx.x;
  for (; i + (kVecUnroll - 1) * stride < n; i += kVecUnroll * stride) {
    double av[kVecUnroll], bv[kVecUnroll];
#pragma unroll
    for (int k = 0; k < kVecUnroll; ++k) {
      av[k] = a[i + k * stride];
      bv[k] = b[i + k * stride];
    }
#pragma unroll
    for (int k = 0; k < kVecUnroll; ++k) v += av[k] * bv[k];
  }
  for (; i < n; i += stride) v += a[i] * b[i];
  v = block_sum<kVecBlock>(v);
  if (threadIdx.x == 0) partials[blockIdx.x] = v;
}

__global__ __launch_bounds__(kVecBlock) void k_axpy(double alpha,
                                                    const double* __restrict__ x,
                                                    double* __restrict__ y,
                                                    int64_t n,
                                                    const double* __restrict__ xs_dev) {
  const double xs = xs_dev ? xs_dev[0] : 1.0;  // x is read as xs * x
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kVecBlock + threadIdx.x;
       i < n; i += static_cast<int64_t>(gridDim.x) * kVecBlock)
    y[i] += alpha * (x[i] * xs);
}

__global__ __launch_bounds__(kVecBlock) void k_scal(double alpha,
                                                    double* __restrict__ x,
                                                    int64_t n) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kVecBlock + threadIdx.x;
       i < n; i += static_cast<int64_t>(gridDim.x) * kVecBlock)
    x[i] *= alpha;
}

// u -= (*alpha) v, partials[b] = sum u^2 over the workgroup's share
__global__ __launch_bounds__(kVecBlock) void k_axpy_dev_norm(
    const double* __restrict__ alpha, const double* __restrict__ v,
    double* __restrict__ u, int64_t n, double* __restrict__ partials,
    const double* __restrict__ vs_dev) {
  const double a = alpha[0];
  const double vs = vs_dev ? vs_dev[0] : 1.0;  // v is read as vs * v
  double acc = 0.0;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kVecBlock;
  int64_t i = static_cast<int64_t>(blockIdx.x) * kVecBlock + threadIdx.x;
  for (; i + (kVecUnroll - 1) * stride < n; i += kVecUnroll * stride) {
    double uv[kVecUnroll], vv[kVecUnroll];
#pragma unroll
    for (int k = 0; k < kVecUnroll; ++k) {
      uv[k] = u[i + k * stride];
      vv[k] = v[i + k * stride] * vs;
    }
#pragma unroll
    for (int k = 0; k < kVecUnroll; ++k) {
      const double w = uv[k] - a * vv[k];
      u[i + k * stride] = w;
      acc += w * w;
    }
  }
  for (; i < n; i += stride) {
    const double w = u[i] - a * (v[i] * vs);
    u[i] = w;
    acc += w * w;
  }
  acc = block_sum<kVecBlock>(acc);
  if (threadIdx.x == 0) partials[blockIdx.x] = acc;
}

// ---- tall-skinny kernels for full reorthogonalisation ----------------------
// V is column-major with leading dimension ldv (column j at V + j*ldv).

constexpr int kMaxCols = 64;

// Gram-Schmidt step of w against V[:, 0:m] in three kernels.  Each one that
// needs a sum over all rows adds up the partials of the kernel before it by
// itself: with at most kGsBlocks workgroups that is a few loads per lane from
// the L2, where kernels of their own for the sums and for the tail's scalars
// cost three launches of 3-4 us per step.  87 546 rows, ten columns on average:
// 35 -> 14 us of kernels per step in 3 launches instead of 6; at 2.76 M rows
// the reads of V bound passes 1 and 2 (42 and 48 us, 5.4 TB/s), and 256
// workgroups of 512 threads keep enough of them in flight.
// partials[j * gridDim.x + workgroup] is column j's.
// SUMS = false (operators that are not symmetric, whose results depend on every
// rounding): the sums are k_finalize_cols's, over more workgroups.
constexpr int kGsBlocks = kSumBlocks;

// Pass 1: partials of V[:, 0:m]^T w, 16 columns at a time.
template <int T>
__global__ __launch_bounds__(T) void k_gs_dots(
    const double* __restrict__ V, int64_t ldv, int m, const double* __restrict__ w,
    int64_t n, double* __restrict__ partials) {
  __shared__ double red[T / kWave][16];
  const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  for (int j0 = 0; j0 < m; j0 += 16) {
    const int jn = min(16, m - j0);
    double acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.0;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * T + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * T) {
      // every load of the row first, then unpredicated updates (absent
      // columns load as 0 and leave their unused sums unchanged), so a lane
      // keeps all its column loads in flight
      const double wi = w[i];
      double v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = j < jn ? V[(j0 + j) * ldv + i] : 0.0;
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[j] += v[j] * wi;
    }
    const double t = wave_sum_many<16>(acc, lane);
    if (lane % 4 == 0) red[wid][lane / 4] = t;
    __syncthreads();
    if (threadIdx.x < jn) {
      double r = 0.0;
#pragma unroll
      for (int k = 0; k < T / kWave; ++k) r += red[k][threadIdx.x];
      partials[static_cast<int64_t>(j0 + threadIdx.x) * gridDim.x + blockIdx.x] = r;
    }
    __syncthreads();
  }
}

// out[j] = sum_b partials[j * nb + b], one workgroup per column j, fixed order
__global__ __launch_bounds__(256) void k_finalize_cols(const double* __restrict__ partials,
                                                       int nb, double* __restrict__ out) {
  const double* p = partials + static_cast<int64_t>(blockIdx.x) * nb;
  double v = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) v += p[b];
  v = block_sum<256>(v);
  if (threadIdx.x == 0) out[blockIdx.x] = v;
}

// Pass 2: h = pass 1's sums (written to hcol by one workgroup; part1 itself
// without SUMS), w -= V[:, 0:m] h, and from the same read of V the partials of V[:, 0:m]^T w_new (columns
// 0..m-1) and of w_new . w_new (column m), m <= MAXC.
template <int T, int MAXC, bool SUMS>
__global__ __launch_bounds__(T) void k_gs_sub_dots(
    const double* __restrict__ V, int64_t ldv, int m, const double* __restrict__ part1,
    double* __restrict__ hcol, double* __restrict__ w, int64_t n,
    double* __restrict__ partials) {
  __shared__ double hs[MAXC];
  __shared__ double red[T / kWave][MAXC + 1];
  const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  if (threadIdx.x < MAXC) hs[threadIdx.x] = !SUMS && threadIdx.x < m ? part1[threadIdx.x] : 0.0;
  __syncthreads();
  if constexpr (SUMS) {
    sum_partials<T>(part1, gridDim.x, m, hs);
    if (blockIdx.x == 0 && threadIdx.x < m) hcol[threadIdx.x] = hs[threadIdx.x];
  }
  double acc[MAXC], nrm = 0.0;
#pragma unroll
  for (int j = 0; j < MAXC; ++j) acc[j] = 0.0;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * T + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * T) {
    // every load of the row first (absent columns load as 0, and their h is
    // 0, so the sum and the dots are unchanged), then the sums in column
    // order, so a lane keeps all its column loads in flight
    double vr[MAXC];
#pragma unroll
    for (int j = 0; j < MAXC; ++j) vr[j] = j < m ? V[j * ldv + i] : 0.0;
    const double wo = w[i];
    double sum = 0.0;
#pragma unroll
    for (int j = 0; j < MAXC; ++j) sum += vr[j] * hs[j];
    const double wn = wo - sum;
    w[i] = wn;
#pragma unroll
    for (int j = 0; j < MAXC; ++j) acc[j] += vr[j] * wn;
    nrm += wn * wn;
  }
  nrm = wave_sum(nrm);
  const double t = wave_sum_many<MAXC>(acc, lane);
  if (lane % (kWave / MAXC) == 0) red[wid][lane / (kWave / MAXC)] = t;
  if (lane == 0) red[wid][MAXC] = nrm;
  __syncthreads();
  for (int j = threadIdx.x; j <= m; j += T) {
    const int src = j == m ? MAXC : j;
    double r = 0.0;
#pragma unroll
    for (int k = 0; k < T / kWave; ++k) r += red[k][src];
    partials[static_cast<int64_t>(j) * gridDim.x + blockIdx.x] = r;
  }
}

// The tail of the step: g[0..m) = V^T w and g[m] = w . w from pass 2's
// partials (part2 itself without SUMS).  A third pass w -= V g is needed when |V^T w| > 1e-12 |w|; its
// correction is added to the projected column hcol[0..m) and the norm follows
// it.  Then w *= 1 / |w|, and one workgroup writes beta[0] = |w|, beta[1] =
// 1 / |w| (0 for a vanishing w).
template <int T, bool SUMS>
__global__ __launch_bounds__(T) void k_gs_tail(
    const double* __restrict__ V, int64_t ldv, int m, const double* __restrict__ part2,
    double* __restrict__ hcol, double* __restrict__ w, int64_t n, double* __restrict__ beta) {
  __shared__ double g[kMaxCols + 1];
  if constexpr (SUMS) {
    sum_partials<T>(part2, gridDim.x, m + 1, g);
  } else {
    if (threadIdx.x <= m) g[threadIdx.x] = part2[threadIdx.x];
    __syncthreads();
  }
  double g2 = 0.0;
  for (int j = 0; j < m; ++j) g2 += g[j] * g[j];
  const double q = g[m];
  const bool need = q > 0.0 && g2 > 1e-24 * q;
  const double b2 = need ? q - g2 : q;
  const double b = b2 > 0.0 ? sqrt(b2) : 0.0;
  const double a = b > 0.0 ? 1.0 / b : 0.0;
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) {
      beta[0] = b;
      beta[1] = a;
    }
    if (need && threadIdx.x < m) hcol[threadIdx.x] += g[threadIdx.x];
  }
  const int64_t stride = static_cast<int64_t>(gridDim.x) * T;
  int64_t i = static_cast<int64_t>(blockIdx.x) * T + threadIdx.x;
  if (!need) {
    for (; i + (kVecUnroll - 1) * stride < n; i += kVecUnroll * stride) {
      double xv[kVecUnroll];
#pragma unroll
      for (int k = 0; k < kVecUnroll; ++k) xv[k] = w[i + k * stride];
#pragma unroll
      for (int k = 0; k < kVecUnroll; ++k) w[i + k * stride] = xv[k] * a;
    }
    for (; i < n; i += stride) w[i] *= a;
    return;
  }
  for (; i < n; i += stride) {
    double acc = 0.0;
    for (int j = 0; j < m; ++j) acc += V[j * ldv + i] * g[j];
    w[i] = (w[i] - acc) * a;
  }
}

// ---- Rayleigh-Ritz of the thick-restart solvers -----------------------------
// One workgroup per projected matrix (RitzArgs): all eigenpairs by Jacobi
// rotations, matrix and vectors in LDS.  A sweep is N - 1 rounds of N / 2
// rotations on disjoint index pairs (round robin), where a cyclic sweep is
// N (N - 1) / 2 rotations one after the other.  A round is a chain of latencies
// (LDS, the angle, two barriers).  The vectors of a thick restart are kept for
// good and never normalised again, so c must round to either side alike: from
// the hardware's reciprocal root with a single Newton step it came out 2^-53 too
// large for every tangent of 1e-8 to 1e-5, and kept vectors grew by 2e-14 a restart
// (square norm, order 40; eigenvalues with them), where host rotations leave them
// within 1e-15 on average.  Blocks
// on and above the diagonal are computed and mirrored: a matrix that rounding
// makes unsymmetric keeps that difference in every rotation and never gets
// diagonal.  Orders 8, 16, 24, 32, 48: 33, 80, 150, 218, 662 us; one matrix of order
// 15 takes 95 us on a host core, of order 20 to 24 about 300, while the device
// idles.
constexpr int kRitzThreads = 256;
__global__ __launch_bounds__(kRitzThreads) void k_ritz(RitzArgs a) {
  constexpr int LD = kRitzMax + 1;
  __shared__ double A[kRitzMax * LD];
  __shared__ double U[kRitzMax * LD];
  __shared__ double2 rot[kRitzMax / 2];
  __shared__ double red[2][kRitzThreads / kWave];
  const int t = threadIdx.x, lane = t % kWave, wid = t / kWave;
  const int m = a.m, N = (m + 1) & ~1, H = N / 2;
  // thread (x0, y): pairs or rows x0, x0 + xs, ... and pair y of each round
  const int lp = 32 - __builtin_clz(static_cast<unsigned>(max(H - 1, 1)));
  const int y = t & ((1 << lp) - 1), x0 = t >> lp, xs = kRitzThreads >> lp;
  const int job = a.job[blockIdx.x], k = a.kept[blockIdx.x];
  const double* cols = a.cols + job * a.job_stride;
  double* theta = a.theta + job * a.theta_stride;
  // the kept Ritz values, their couplings to the first new vector, and the
  // projections onto the new vectors (the rest is rounding noise)
  for (int e = t; e < N * N; e += kRitzThreads) {
    const int i = min(e / N, e % N), j = max(e / N, e % N);
    double v = 0.0;
    if (j < k) v = i == j ? theta[j] : 0.0;
    else if (j < m && (i >= k || j == k)) v = cols[j * a.ldc + i];
    A[(e / N) * LD + e % N] = v;
    U[(e / N) * LD + e % N] = e / N == e % N ? 1.0 : 0.0;
  }
  __syncthreads();
  bool bad = false;  // a NaN in the matrix
  for (int sweep = 0; sweep < 64; ++sweep) {
    double off = 0.0, tot = 0.0;
    for (int x = x0; x < N && y < H; x += xs) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int z = 2 * y + h;
        const double v = A[x * LD + z] * A[x * LD + z];
        tot += v;
        if (x != z) off += v;
      }
    }
    off = wave_sum(off);
    tot = wave_sum(tot);
    if (lane == 0) {
      red[0][wid] = off;
      red[1][wid] = tot;
    }
    __syncthreads();
    off = tot = 0.0;
#pragma unroll
    for (int w = 0; w < kRitzThreads / kWave; ++w) {
      off += red[0][w];
      tot += red[1][w];
    }
    // the same in every thread
    bad = tot != tot;
    if (bad || off == 0.0 || off <= 1e-32 * tot) break;
    for (int r = 0; r < N - 1; ++r) {
      // pair u of the round: the last index stays, the others go around
      auto pair = [&](int u, int& p, int& q) {
        p = r + u;
        p = p >= N - 1 ? p - (N - 1) : p;
        q = r - u;
        q = u == 0 ? N - 1 : (q < 0 ? q + N - 1 : q);
      };
      if (t < H) {
        int p, q;
        pair(t, p, q);
        // tt = tan of the smaller angle that annihilates A[p][q]
        const double b = 2.0 * A[p * LD + q], d = A[q * LD + q] - A[p * LD + p];
        double2 cs = make_double2(1.0, 0.0);
        if (b != 0.0) {
          const double h2 = fma(d, d, b * b);
          const double h = h2 > 1e-290 && h2 < 1e290 ? sqrt(h2) : hypot(d, b);
          const double tt = (d < 0.0 ? -b : b) / (fabs(d) + h);
          // c = (1 + tt^2)^-1/2: the hardware's reciprocal root, a Newton step of
          // third order, and one with the rounding errors of 1 + tt^2 and of z g put
          // back
          const double z = fma(tt, tt, 1.0), zl = fma(tt, tt, 1.0 - z);
          double g = __builtin_amdgcn_rsq(z);
          const double e = fma(-z * g, g, 1.0);
          g = fma(g * e, fma(0.375, e, 0.5), g);
          const double zg = z * g, zgl = fma(z, g, -zg);
          const double er = fma(-zg, g, 1.0) - fma(zl * g, g, zgl * g);
          cs.x = fma(0.5 * g, er, g);
          cs.y = tt * cs.x;
        }
        rot[t] = cs;
      }
      __syncthreads();
      if (y < H) {
        int u, v;
        pair(y, u, v);
        const double2 C = rot[y];
        for (int x = x0; x <= y; x += xs) {
          int p, q;
          pair(x, p, q);
          const double2 R = rot[x];
          const double pu = A[p * LD + u], pv = A[p * LD + v];
          const double qu = A[q * LD + u], qv = A[q * LD + v];
          const double pu1 = C.x * pu - C.y * pv, pv1 = C.y * pu + C.x * pv;
          const double qu1 = C.x * qu - C.y * qv, qv1 = C.y * qu + C.x * qv;
          const double a00 = R.x * pu1 - R.y * qu1, a10 = R.y * pu1 + R.x * qu1;
          const double a01 = R.x * pv1 - R.y * qv1, a11 = R.y * pv1 + R.x * qv1;
          A[p * LD + u] = A[u * LD + p] = a00;
          A[p * LD + v] = A[v * LD + p] = a01;
          A[q * LD + v] = A[v * LD + q] = a11;
          if (x != y) A[q * LD + u] = A[u * LD + q] = a10;
        }
        for (int x = x0; x < m; x += xs) {
          const double iu = U[x * LD + u], iv = U[x * LD + v];
          U[x * LD + u] = C.x * iu - C.y * iv;
          U[x * LD + v] = C.y * iu + C.x * iv;
        }
      }
      __syncthreads();
    }
  }
  // ascending order, NaN behind every number, ties by index: every index has a
  // rank of its own, so every output is written.  A matrix with a NaN has no
  // eigenpairs: all its outputs are NaN (a request's values stand where an
  // earlier one's stood)
  double* Y = a.Y + job * a.y_stride;
  for (int e = t; e < m * m; e += kRitzThreads) {
    const int j = e / m, i = e % m;
    const double d = A[j * LD + j];
    int rank = 0;
    for (int u = 0; u < m; ++u) {
      const double du = A[u * LD + u];
      rank += (d != d ? du == du : du < d) || ((du == d || (d != d && du != du)) && u < j) ? 1 : 0;
    }
    const double nan = __builtin_nan("");
    const double w = bad ? nan : U[i * LD + j], th = bad ? nan : d;
    Y[rank * m + i] = w;
    if (i == 0) {
      theta[rank] = th;
      a.out_theta[blockIdx.x * a.out_stride + rank] = th;
    }
    if (i == m - 1) a.out_last[blockIdx.x * a.out_stride + rank] = w;
  }
}

// out[:, c] = V[:, 0:m] Y[:, c] for c < k (Y column-major m x k, on device);
// output columns in chunks of 8 so V is read ceil(k/8) times.
__global__ __launch_bounds__(kVecBlock) void k_combine(
    const double* __restrict__ V, int64_t ldv, int m, const double* __restrict__ Y,
    int k, double* __restrict__ out, int64_t ldo, int64_t n) {
  __shared__ double ys[kMaxCols * kMaxCols];
  for (int t = threadIdx.x; t < m * k; t += kVecBlock) ys[t] = Y[t];
  __syncthreads();
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kVecBlock + threadIdx.x;
       i < n; i += static_cast<int64_t>(gridDim.x) * kVecBlock) {
    for (int c0 = 0; c0 < k; c0 += 8) {
      double acc[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) acc[c] = 0.0;
      // eight columns' loads in flight (one at a time: 181 us for 20 columns of
      // 2.76 M rows onto 7, where the bytes take about 120)
      for (int j0 = 0; j0 < m; j0 += 8) {
        double vj[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) vj[j] = j0 + j < m ? V[(j0 + j) * ldv + i] : 0.0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (j0 + j >= m) break;
#pragma unroll
          for (int c = 0; c < 8; ++c)
            if (c0 + c < k) acc[c] += vj[j] * ys[(c0 + c) * m + j0 + j];
        }
      }
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (c0 + c < k) out[(c0 + c) * ldo + i] = acc[c];
    }
  }
}

// x[i] = s_dev[0] * y[i]
__global__ __launch_bounds__(kVecBlock) void k_copy_scaled(
    const double* __restrict__ s, const double* __restrict__ y,
    double* __restrict__ x, int64_t n) {
  const double a = s[0];
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kVecBlock + threadIdx.x;
       i < n; i += static_cast<int64_t>(gridDim.x) * kVecBlock)
    x[i] = a * y[i];
}

// y += s_dev[0] * c * x
__global__ __launch_bounds__(kVecBlock) void k_axpy_dev(
    const double* __restrict__ s, double c, const double* __restrict__ x,
    double* __restrict__ y, int64_t n) {
  const double a = c * s[0];
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kVecBlock + threadIdx.x;
       i < n; i += static_cast<int64_t>(gridDim.x) * kVecBlock)
    y[i] += a * x[i];
}

// Psi[:, b] += c[b] * v for b < nb (Psi column-major, leading dimension ld):
// one read of v feeds every column.  v is read as vs * v.
__global__ __launch_bounds__(kVecBlock) void k_accum_cols(
    const double* __restrict__ v, double* __restrict__ Psi, int64_t ld, int nb,
    const double* __restrict__ c, int64_t n, const double* __restrict__ vs_dev) {
  const double vs = vs_dev ? vs_dev[0] : 1.0;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kVecBlock + threadIdx.x;
       i < n; i += static_cast<int64_t>(gridDim.x) * kVecBlock) {
    const double vi = v[i] * vs;
    for (int b = 0; b < nb; ++b) Psi[b * ld + i] += c[b] * vi;
  }
}

// ============================================================================
// Many small operators on a few vectors, and inner products of many columns
// ============================================================================

// Y[:, l * n_vec + v] = O_l psi_v for the operators l of this workgroup's
// chunk (blockIdx.y).  One lane per row: the row's state is read once for all
// operators, and a term's rank is looked up once for all vectors (kEachVecs of
// them per round).  Per output the sum runs in term order, then the diagonal,
// as in the apply kernels, so the columns have the same bits.
constexpr int kEachVecs = 4;
constexpr int kEachOps = 8;  // operators of one workgroup

template <int NW>
__global__ __launch_bounds__(kApplyBlock) void k_apply_each(
    BasisView b, const EachOp* __restrict__ ops, int n_ops, const double* __restrict__ psi,
    int64_t ld, int n_vec, double* __restrict__ Y, int64_t ldy) {
  const int64_t i = static_cast<int64_t>(xcd_remap(blockIdx.x, gridDim.x)) * kApplyBlock +
                    threadIdx.x;
  if (i >= b.dim) return;
  const State<NW> s = load_state_cached<NW>(b.states, i);
  const int l1 = min(n_ops, static_cast<int>(blockIdx.y + 1) * kEachOps);
  for (int l = blockIdx.y * kEachOps; l < l1; ++l) {
    const EachOp O = ops[l];
    for (int v0 = 0; v0 < n_vec; v0 += kEachVecs) {
      const double* x = psi + v0 * ld;
      double acc[kEachVecs] = {};
      for (int t = 0; t < O.n_off; ++t) {
        const OffTerm& T = O.off[t];
        if (!term_ok<NW>(T, s)) continue;
        const int64_t J = basis_lookup<NW>(b, xor_state<NW>(s, T.X));
        if (J < 0) continue;
        double c = T.c * T.sgn;
        if (parity_notz<NW>(s, T.Z)) c = -c;
#pragma unroll
        for (int v = 0; v < kEachVecs; ++v) {
          if (v0 + v < n_vec) {
            const double xj = x[v * ld + J];
            if (fabs(xj) > kApplyTol) acc[v] += c * xj;
          }
        }
      }
#pragma unroll
      for (int v = 0; v < kEachVecs; ++v) {
        if (v0 + v < n_vec) {
          if (O.n_diag > 0)
            acc[v] = diag_accumulate<NW>(acc[v], x[v * ld + i], s, O.dg, O.n_diag);
          Y[static_cast<int64_t>(l * n_vec + v0 + v) * ldy + i] = acc[v];
        }
      }
    }
  }
}

// Inner products of the columns of A (pa) and B (pb) over n rows, on the FP64
// matrix cores.  blockIdx.y is a pair of 64-column blocks (of the upper triangle
// when A and B are the same matrix), blockIdx.x a slab of rows.  A wavefront
// takes 16 rows at a time: lane l reads four consecutive rows 4 (l / 16) of
// column l % 16 (a whole 128-byte line per column), and the four rows feed four
// 16x16x4 products per pair of 16-column blocks; which rows share a product does
// not matter to the sum.  The four wavefronts' 64 x 64 sums meet in LDS in a fixed
// order, and part[(slab, pair)] holds the slab's result.  Reading the columns
// once per pair of blocks instead of once per 16 columns and output column is
// what it is for.
constexpr int kGramCols = 64;
typedef double f64x4 __attribute__((ext_vector_type(4)));

// The column blocks (ba, bb) of a pair: row by row of the upper triangle (same)
// or of all nbb columns of blocks.
__device__ __forceinline__ void gram_pair(int64_t pair, int nbb, int same, int* ba, int* bb) {
  if (same) {
    int a = 0;
    while (pair >= nbb - a) pair -= nbb - a++;
    *ba = a;
    *bb = a + static_cast<int>(pair);
  } else {
    *ba = static_cast<int>(pair / nbb);
    *bb = static_cast<int>(pair % nbb);
  }
}

__global__ __launch_bounds__(256) void k_gram(const double* __restrict__ A, int64_t lda, int pa,
                                              const double* __restrict__ B, int64_t ldb, int pb,
                                              int64_t n, int64_t slab, int same, int64_t pairs,
                                              double* __restrict__ part) {
  __shared__ double sum[kGramCols * kGramCols];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t pair = static_cast<int64_t>(blockIdx.z) * gridDim.y + blockIdx.y;
  if (pair >= pairs) return;
  int ba, bb;
  gram_pair(pair, (pb + kGramCols - 1) / kGramCols, same, &ba, &bb);
  const int a0 = ba * kGramCols, b0 = bb * kGramCols;
  const int ta = min(4, (pa - a0 + 15) / 16), tb = min(4, (pb - b0 + 15) / 16);
  const int c = lane & 15, k = lane >> 4;
  f64x4 acc[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[u][v] = f64x4{0.0, 0.0, 0.0, 0.0};
  const int64_t r_end = min<int64_t>(n, (blockIdx.x + 1) * slab);
  for (int64_t r = blockIdx.x * slab + wid * 16; r < r_end; r += 64) {
    double fa[4][4], fb[4][4];
    // columns past the last repeat it (their sums are not stored); rows past
    // the end count as zero
    auto load = [&](const double* M, int64_t ld, int col, double (&f)[4]) {
      const double* p = M + static_cast<int64_t>(col) * ld + r + 4 * k;
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = r + 4 * k + j < r_end ? p[j] : 0.0;
    };
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (u < ta) load(A, lda, min(a0 + 16 * u + c, pa - 1), fa[u]);
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (v < tb) load(B, ldb, min(b0 + 16 * v + c, pb - 1), fb[v]);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (u < ta && v < tb) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[u][j], fb[v][j], acc[u][v], 0, 0, 0);
        }
  }
  // lane l holds rows l / 16 + 4 q and column l % 16 of each 16 x 16 product
  for (int w = 0; w < 4; ++w) {
    if (wid == w) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            double& o = sum[(16 * u + k + 4 * q) * kGramCols + 16 * v + c];
            o = w == 0 ? acc[u][v][q] : o + acc[u][v][q];
          }
    }
    __syncthreads();
  }
  double* out = part + (blockIdx.x * pairs + pair) * (kGramCols * kGramCols);
  for (int t = threadIdx.x; t < kGramCols * kGramCols; t += 256) out[t] = sum[t];
}

// out[b * pa + a] = the slabs' sums of (a, b) (and its mirror image when the two
// matrices are the same) for T-column blocks: a workgroup sums 32 neighbouring
// entries, eight groups of slabs side by side (every eighth slab each), which
// are added in a fixed order.
template <int T>
__global__ __launch_bounds__(256) void k_gram_sum(const double* __restrict__ part, int n_slab,
                                                  int pa, int pb, int same, int64_t pairs,
                                                  double* __restrict__ out) {
  __shared__ double red[8][32];
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 32 + (threadIdx.x & 31);
  const int g = threadIdx.x >> 5;
  double v = 0.0;
  for (int s = g; s < n_slab; s += 8) v += part[s * pairs * (T * T) + e];
  red[g][threadIdx.x & 31] = v;
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int k = 1; k < 8; ++k) v += red[k][threadIdx.x];
  int ba, bb;
  gram_pair(e / (T * T), (pb + T - 1) / T, same, &ba, &bb);
  const int k = static_cast<int>(e % (T * T));
  const int a = ba * T + k / T, b = bb * T + k % T;
  if (a >= pa || b >= pb) return;
  out[static_cast<int64_t>(b) * pa + a] = v;
  if (same && ba != bb) out[static_cast<int64_t>(a) * pa + b] = v;
}

// The same inner products for operators of a few terms each, without the
// columns O_l psi_v ever going to memory: a workgroup takes 64 rows at a time,
// forms those rows of every column in LDS (lane = row, wavefront w the
// operators of list w; four lookups in flight per lane; sums in term order,
// then the diagonal), and multiplies them on the matrix cores, each wavefront
// with the 16 x 16 products w, w + 4, ... of its own.  part[(workgroup, product)]
// holds the workgroup's sums.  With stored columns the products read every
// column once per output column and 64-column block: 48 operators on two 48-spin
// vectors took 6.9 ms for expectations and correlations, 96 launches of 4 us and
// 98 of 28 us each; this way 0.37 ms, 2 x 63 us of it in this kernel, bound by the
// latency of the lookups, and 2 x 12 us in the sums.  Columns [0, P) are the operators', and for
// expectations (same = 0) n_vec columns of psi follow at the next multiple of 16.
constexpr int kObsCols = 128;  // most columns of the operators
constexpr int kObsVecs = 16;   // most columns of psi for expectations
constexpr int kObsTiles = kObsCols / 16 * (kObsCols / 16 + 1) / 2;
constexpr int kObsLd = 66;     // LDS rows of a column: 64 and two that spread the banks

template <int NW>
__global__ __launch_bounds__(256) void k_observe(BasisView b, ObserveArgs q,
                                                 const double* __restrict__ psi, int64_t ld,
                                                 double* __restrict__ part) {
  extern __shared__ double col[];  // [column][kObsLd]
  constexpr int G = 4;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nb = (q.P + 15) / 16;
  const int n_cols = 16 * nb + (q.same ? 0 : 16);
  const int c = lane & 15, k = lane >> 4;
  // this wavefront's products
  constexpr int kMine = kObsTiles / 4;
  int tu[kMine], tv[kMine], mine = 0;
  for (int t = wid; t < q.tiles; t += 4) {
    int u = t, v = nb;  // expectations: block u against psi's
    if (q.same) gram_pair(t, nb, 1, &u, &v);
#pragma unroll
    for (int m = 0; m < kMine; ++m)
      if (m == mine) {
        tu[m] = u;
        tv[m] = v;
      }
    ++mine;
  }
  f64x4 acc[kMine];
#pragma unroll
  for (int m = 0; m < kMine; ++m) acc[m] = f64x4{0.0, 0.0, 0.0, 0.0};
  // columns that no operator writes stay zero
  for (int e = threadIdx.x; e < n_cols * kObsLd; e += 256) col[e] = 0.0;
  __syncthreads();
  const int64_t chunks = (b.dim + 63) / 64;
  for (int64_t ch = blockIdx.x; ch < chunks; ch += gridDim.x) {
    const int64_t i = ch * 64 + lane;
    const bool row_ok = i < b.dim;
    const State<NW> s = load_state_cached<NW>(b.states, row_ok ? i : ch * 64);
    for (int e = q.col_begin[wid]; e < q.col_begin[wid + 1]; ++e) col[q.cols[e] * kObsLd + lane] = 0.0;
    if (!q.same && wid == 0)
      for (int v = 0; v < q.n_vec; ++v)
        col[(16 * nb + v) * kObsLd + lane] = row_ok ? psi[v * ld + i] : 0.0;
    const int t1 = q.off_begin[wid + 1];
    for (int t0 = q.off_begin[wid]; t0 < t1; t0 += 64) {
      uint64_t mask = connect_mask<NW>(q.off + t0, min(64, t1 - t0), s);
      if (!row_ok) mask = 0;
      while (mask) {
        int tt[G];
        bool act[G];
        State<NW> key[G];
        uint32_t rk[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          act[g] = mask != 0;
          const int z = act[g] ? __builtin_clzll(mask) : 0;
          tt[g] = t0 + z;
          mask &= ~(uint64_t{1} << 63 >> z);
          key[g] = xor_state<NW>(s, q.off[tt[g]].X);
        }
        lookup_batch<NW, G>(b, key, act, rk);
        for (int v = 0; v < q.n_vec; ++v) {
          double xj[G];
#pragma unroll
          for (int g = 0; g < G; ++g) xj[g] = rk[g] != kNoRank ? psi[v * ld + rk[g]] : 0.0;
#pragma unroll
          for (int g = 0; g < G; ++g) {
            if (rk[g] != kNoRank && fabs(xj[g]) > kApplyTol) {
              const OffTerm& T = q.off[tt[g]];
              double cg = T.c * T.sgn;
              if (parity_notz<NW>(s, T.Z)) cg = -cg;
              col[(T.slot + v) * kObsLd + lane] += cg * xj[g];
            }
          }
        }
      }
    }
    for (int d = q.diag_begin[wid]; d < q.diag_begin[wid + 1]; ++d) {
      const EachOp& O = q.diag[d];
      if (row_ok)
        for (int v = 0; v < q.n_vec; ++v) {
          double& y = col[(O.col + v) * kObsLd + lane];
          y = diag_accumulate<NW>(y, psi[v * ld + i], s, O.dg, O.n_diag);
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kMine; ++m) {
      if (m < mine) {
        const double* A = col + (16 * tu[m] + c) * kObsLd + k;
        const double* B = col + (16 * tv[m] + c) * kObsLd + k;
#pragma unroll
        for (int j = 0; j < 16; ++j)
          acc[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[4 * j], B[4 * j], acc[m], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  double* out = part + static_cast<int64_t>(blockIdx.x) * q.tiles * 256;
#pragma unroll
  for (int m = 0; m < kMine; ++m)
    if (m < mine)
#pragma unroll
      for (int e = 0; e < 4; ++e) out[(wid + 4 * m) * 256 + (k + 4 * e) * 16 + c] = acc[m][e];
}

// ============================================================================
// Host helpers
// ============================================================================

namespace {
thread_local std::string g_err;
}

void set_error(const std::string& msg) { g_err = msg; }
const char* get_error() { return g_err.c_str(); }

void basis_retain(qsi_basis_s* b) { b->refs.fetch_add(1); }
void basis_release(qsi_basis_s* b) {
  if (b->refs.fetch_sub(1) == 1) {
    if (b->d_states) (void)hipFree(b->d_states);
    if (b->d_table) (void)hipFree(b->d_table);
    if (b->d_hash) (void)hipFree(b->d_hash);
    if (b->d_slots) (void)hipFree(b->d_slots);
    if (b->d_lowkeys) (void)hipFree(b->d_lowkeys);
    delete b;
  }
}

int64_t apply_num_blocks(const qsi_op_s* op) {
  return (op->basis->dim + kApplyBlock - 1) / kApplyBlock;
}

template <int NW, bool DOT, bool ALIGNED>
static void launch_cached_t(const qsi_op_s* op, dim3 grid, dim3 block, const BasisView& v,
                            const double* x, double* y, const double* y_in, double yscale,
                            const double* yscale_dev, double* partials, const double* xs_dev,
                            const double* ys_dev, hipStream_t s) {
  auto k = op->cached_pipe == 32 ? k_apply_cached<NW, DOT, 32, ALIGNED>
         : op->cached_pipe == 4  ? k_apply_cached<NW, DOT, 4, ALIGNED>
         : op->cached_pipe == 16 ? k_apply_cached<NW, DOT, 16, ALIGNED>
                                 : k_apply_cached<NW, DOT, 8, ALIGNED>;
  hipLaunchKernelGGL(k, grid, block, 0, s, v, op->d_cls, op->n_cls, op->d_rowptr, op->d_cj,
                     op->d_cm, op->d_diag, op->n_diag, x, y, y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
}

bool auto_takes_rows(const qsi_op_s* op) {
  return op->conn_nnz < 0 &&
         op->basis->dim <= (op->n_off < kRowMinTerms ? kRowMaxDimFew : kRowMaxDim);
}

template <int NW, bool HAS_Z, bool DOT>
static void launch_apply_t(const qsi_op_s* op, const double* x, double* y,
                           const double* y_in, double yscale,
                           const double* yscale_dev, double* partials,
                           const double* xs_dev, const double* ys_dev, hipStream_t s) {
  const int64_t nb = apply_num_blocks(op);
  const dim3 grid(static_cast<uint32_t>(nb)), block(kApplyBlock);
  // the window kernel's workgroups take two blocks of rows
  const dim3 wgrid(static_cast<uint32_t>((nb + 1) / 2));
  const auto v = op->basis->view();
  int variant = op->variant;
  // AUTO: the cached connectivity when it exists.  Else, on bases of a few
  // thousand states, a wavefront per row (call to call, a call's host side being
  // 7.8 us, row / LANE4 / LOW8 in us: 2970 states 7.8 / 12.4 / 11.9, 13122 states
  // 9.1 / 14.5 / 14.7, 87546 states 54 / 20 / 19), but not for the dot-product
  // instances, whose partials are sums over 256 rows, nor on more than 4096 states
  // for few terms, which a lane does in a round or two (13122 states, 1 / 4 / 8 / 16
  // / 32 terms, row / LANE4: 4.5 / 3.3, 4.8 / 3.7, 5.1 / 4.2, 5.5 / 5.4, 5.8 / 7.9).
  // Else, without low keys whose
  // candidates need no compare, the window kernel on bases large enough to fill
  // the chip with its 128-row wavefronts (WINDOW / LANE4 / LOW4 in us: 32 spins
  // 35 / 12 / 13, 293394 states 33 / 25 / 25, 1062882 states 55 / 52 / 53, 64 spins 200 /
  // 266 / 273, 72 spins 1467 / 2089 / 1831; 80 spins 10.1 / 17.6 / 14.3 and 96 spins
  // 301 / 543 ms), if few of the sampled (tile, term) pairs have a target outside
  // the basis: such a term is done again by per-row lookups.  By the share of such
  // pairs, WINDOW / LANE4 / LOW4 unverified / LOW4 after mode 1: 60 spins at 0 171 /
  // 224 / 218 / - us, 2 % 201 / 221 / 214 / 202, 5 % 238 / 224 / 215 / 202; 64 spins, one
  // pair, 1 % 356 / 522 / - / 449; 64 spins, 4 % 254 / 271 / - / 235, 11 % 312 / 269 / - / 233,
  // 30 % 428 / 268 / - / 231; 72 spins, one pair, 1 % 2.92 / 4.20 / 3.57 / 2.82 ms, 2 %
  // 3.27 / 4.21 / 3.57 / 2.82, 5 % 3.93 / 4.21 / 3.57 / 2.82; 64 spins, two pairs, 32 %
  // 115 / 91 ms.  So up to 1/32, with key compares (mode 1) up to 1/64 and one-word
  // states only; and from 32 terms on (1 / 8 / 16 / 32 / 64 of them, WINDOW / LANE4 in
  // us: 64 spins 27 / 19, 39 / 30, 49 / 38, 66 / 68, 111 / 132; 72 spins 134 / 130, 241 /
  // 231, 310 / 296, 434 / 488, 703 / 943).  With low keys that need no compare LOW8, except where WINDOW
  // without its compare is the faster: one-word states on large bases (WINDOW /
  // LOW8: 293394 states 33 / 21, 64 spins 181 / 190, 60 spins 166 / 191 us) and bases so
  // large that the 31-bit bucket key leaves long bisections (72 spins 1.21 / 1.18,
  // 80 spins 9.47 / 9.38, 96 spins 278 / 292 ms).
  if (variant == QSI_APPLY_AUTO) {
    const int64_t dim = op->basis->dim;
    if constexpr (!DOT) {
      if (auto_takes_rows(op)) {
        const int64_t rb = kApplyBlock / kWave;
        hipLaunchKernelGGL((k_apply_row<NW, HAS_Z>), dim3(static_cast<uint32_t>((dim + rb - 1) / rb)),
                           block, 0, s, v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in,
                           yscale, yscale_dev);
        return;
      }
    }
    const int check = op->basis->d_lowkeys ? op->lowkeys_check : kLowCmpState;
    const bool trusted = check == kLowTrusted;
    bool window = dim >= kWinMinDim && op->ordered;
    if (trusted) window = window && op->paired && (NW == 1 || dim >= kWinMinDimLow2);
    else if (op->n_off < kWinMinTerms) window = false;
    else if (check == kLowCmpKey) window = window && NW == 1 && op->miss_share <= 1.0f / 64;
    else window = window && op->miss_share <= 1.0f / 32;
    variant = op->conn_nnz >= 0        ? QSI_APPLY_CACHED
              : window                 ? QSI_APPLY_WINDOW
              : trusted                ? QSI_APPLY_LOW8
              : op->basis->d_lowkeys   ? QSI_APPLY_LOW4
                                       : QSI_APPLY_LANE4;
  }
  // a slot or low-key variant chosen while the basis had that index, which
  // has been dropped since, falls back to the lane kernel (LANE4 for SLOT4,
  // LANE2 for SLOT2 and SLOT3; the same depth for LOW*)
  if (!op->basis->d_slots && variant >= QSI_APPLY_SLOT2 && variant <= QSI_APPLY_SLOT3)
    variant = variant == QSI_APPLY_SLOT4 ? QSI_APPLY_LANE4 : QSI_APPLY_LANE2;
  if (!op->basis->d_lowkeys && variant >= QSI_APPLY_LOW2 && variant <= QSI_APPLY_LOW8)
    variant = variant == QSI_APPLY_LOW2 ? QSI_APPLY_LANE2
            : variant == QSI_APPLY_LOW4 ? QSI_APPLY_LANE4 : QSI_APPLY_LANE8;
  switch (variant) {
    case QSI_APPLY_CACHED:
      // gathers in flight per lane: op->cached_pipe (4, 8, 16 or 32; autotuned)
      if (op->conn_pad == 4)
        launch_cached_t<NW, DOT, true>(op, grid, block, v, x, y, y_in, yscale, yscale_dev,
                                       partials, xs_dev, ys_dev, s);
      else
        launch_cached_t<NW, DOT, false>(op, grid, block, v, x, y, y_in, yscale, yscale_dev,
                                        partials, xs_dev, ys_dev, s);
      break;
    case QSI_APPLY_LANE:
      hipLaunchKernelGGL((k_apply_lane<NW, HAS_Z, DOT, 1>), grid, block, 0, s, v,
                         op->d_off, op->n_off, op->d_diag, op->n_diag, x, y,
                         y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_LANE2:
      hipLaunchKernelGGL((k_apply_lane<NW, HAS_Z, DOT, 2>), grid, block, 0, s, v,
                         op->d_off, op->n_off, op->d_diag, op->n_diag, x, y,
                         y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_WINDOW:
      // a window holds kWinRows states.  No compare of matched states when
      // every connected state is in the basis, every flip's reverse is a term
      // of the operator too, and targets keep the rows' order
      if (op->basis->dim < kWinRows)
        hipLaunchKernelGGL((k_apply_lane<NW, HAS_Z, DOT, 4>), grid, block, 0, s, v,
                           op->d_off, op->n_off, op->d_diag, op->n_diag, x, y,
                           y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      else if (op->lowkeys_check == kLowTrusted && op->paired && op->ordered)
        hipLaunchKernelGGL((k_apply_win<NW, HAS_Z, DOT, false>), wgrid, block, 0, s, v,
                           op->d_off, op->n_off, op->planes(),
                           reinterpret_cast<const TermRec<NW>*>(op->planes().rec()), op->d_diag, op->n_diag, x, y,
                           y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      else
        hipLaunchKernelGGL((k_apply_win<NW, HAS_Z, DOT, true>), wgrid, block, 0, s, v,
                           op->d_off, op->n_off, op->planes(),
                           reinterpret_cast<const TermRec<NW>*>(op->planes().rec()), op->d_diag, op->n_diag, x, y,
                           y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_LANE8:
      hipLaunchKernelGGL((k_apply_lane<NW, HAS_Z, DOT, 8>), grid, block, 0, s, v,
                         op->d_off, op->n_off, op->d_diag, op->n_diag, x, y,
                         y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_HASH:
      hipLaunchKernelGGL((k_apply_hash<NW, HAS_Z, DOT, 1>), grid, block, 0, s, v,
                         op->basis->hview(), op->d_off, op->n_off, op->d_diag,
                         op->n_diag, x, y, y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_HASH4:
      hipLaunchKernelGGL((k_apply_hash<NW, HAS_Z, DOT, 4>), grid, block, 0, s, v,
                         op->basis->hview(), op->d_off, op->n_off, op->d_diag,
                         op->n_diag, x, y, y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_SLOT2:
      hipLaunchKernelGGL((k_apply_slot<NW, HAS_Z, DOT, 2>), grid, block, 0, s, v,
                         op->d_off, op->n_off, op->d_diag, op->n_diag, x, y,
                         y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_SLOT4:
      hipLaunchKernelGGL((k_apply_slot<NW, HAS_Z, DOT, 4>), grid, block, 0, s, v,
                         op->d_off, op->n_off, op->d_diag, op->n_diag, x, y,
                         y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_SLOT3:
      hipLaunchKernelGGL((k_apply_slot<NW, HAS_Z, DOT, 3>), grid, block, 0, s, v,
                         op->d_off, op->n_off, op->d_diag, op->n_diag, x, y,
                         y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_LOW2:
      if (op->lowkeys_check == kLowTrusted)
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 2, kLowTrusted>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      else if (op->lowkeys_check == kLowCmpKey)
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 2, kLowCmpKey>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      else
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 2, kLowCmpState>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_LOW4:
      if (op->lowkeys_check == kLowTrusted)
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 4, kLowTrusted>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      else if (op->lowkeys_check == kLowCmpKey)
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 4, kLowCmpKey>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      else
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 4, kLowCmpState>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      break;
    case QSI_APPLY_LOW8:
      if (op->lowkeys_check == kLowTrusted)
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 8, kLowTrusted>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      else if (op->lowkeys_check == kLowCmpKey)
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 8, kLowCmpKey>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      else
        hipLaunchKernelGGL((k_apply_low<NW, HAS_Z, DOT, 8, kLowCmpState>), grid, block, 0, s,
                           v, op->d_off, op->n_off, op->d_diag, op->n_diag, x, y, y_in, yscale,
                           yscale_dev, partials, xs_dev, ys_dev);
      break;
    default:  // QSI_APPLY_LANE4
      hipLaunchKernelGGL((k_apply_lane<NW, HAS_Z, DOT, 4>), grid, block, 0, s, v,
                         op->d_off, op->n_off, op->d_diag, op->n_diag, x, y,
                         y_in, yscale, yscale_dev, partials, xs_dev, ys_dev);
  }

}

int launch_apply(const qsi_op_s* op, const double* x, double* y,
                 const double* y_in, double yscale, double* dot_partials,
                 double* dot_out, hipStream_t s) {
  return launch_apply_dev(op, x, y, y_in, yscale, nullptr, dot_partials,
                          dot_out, s);
}

int launch_apply_dev(const qsi_op_s* op, const double* x, double* y,
                     const double* y_in, double yscale,
                     const double* yscale_dev, double* dot_partials,
                     double* dot_out, hipStream_t s) {
  return launch_apply_scaled(op, x, y, y_in, yscale, yscale_dev, nullptr, nullptr, dot_partials,
                             dot_out, s);
}

// Sums n per-workgroup partials into out (mode as in k_finalize_sum) in a
// fixed order.  Arrays longer than 8 chunks are first reduced chunk by chunk
// in place (k_sum_chunks), so a single workgroup never streams millions of
// partials; the partials are clobbered.
static void launch_finalize(double* partials, int64_t n, double* out, int mode,
                            hipStream_t s) {
  constexpr int64_t kChunk = 4096;
  if (n > 8 * kChunk) {
    const int64_t g = (n + kChunk - 1) / kChunk;
    hipLaunchKernelGGL(k_sum_chunks<256>, dim3(static_cast<uint32_t>(g)), dim3(256), 0, s,
                       partials, n, kChunk);
    hipLaunchKernelGGL(k_finalize_sum<256>, dim3(1), dim3(256), 0, s, partials, g, out, mode,
                       kChunk);
  } else {
    hipLaunchKernelGGL(k_finalize_sum<256>, dim3(1), dim3(256), 0, s, partials, n, out, mode,
                       int64_t{1});
  }
}

int launch_apply_scaled(const qsi_op_s* op, const double* x, double* y,
                        const double* y_in, double yscale, const double* yscale_dev,
                        const double* xs_dev, const double* ys_dev, double* dot_partials,
                        double* dot_out, hipStream_t s) {
  const bool dot = dot_partials != nullptr;
  // the kernels honour the scales only in their dot-product instances
  QSI_REQUIRE(dot || (xs_dev == nullptr && ys_dev == nullptr),
              "launch_apply_scaled: scales need the dot product");
  const int nw = op->basis->nw;
  const bool hz = op->has_z;
#define QSI_LAUNCH(NW_, HZ_, D_) \
  launch_apply_t<NW_, HZ_, D_>(op, x, y, y_in, yscale, yscale_dev, dot_partials, xs_dev, \
                               ys_dev, s)
  if (nw == 1) {
    if (hz) { if (dot) QSI_LAUNCH(1, true, true); else QSI_LAUNCH(1, true, false); }
    else    { if (dot) QSI_LAUNCH(1, false, true); else QSI_LAUNCH(1, false, false); }
  } else {
    if (hz) { if (dot) QSI_LAUNCH(2, true, true); else QSI_LAUNCH(2, true, false); }
    else    { if (dot) QSI_LAUNCH(2, false, true); else QSI_LAUNCH(2, false, false); }
  }
#undef QSI_LAUNCH
  QSI_CHECK_LAUNCH();
  if (dot) {
    launch_finalize(dot_partials, apply_num_blocks(op), dot_out, 0, s);
    QSI_CHECK_LAUNCH();
  }
  return QSI_OK;
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// Gaussian entries from a counter-based generator: Box-Muller on two
// splitmix64 (Steele, Lea & Flood 2014) uniforms per entry, so v[i] depends
// on (seed, i) only, whatever the launch shape.
__global__ void k_randn(double* __restrict__ v, int64_t n, uint64_t seed) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t a = splitmix64(seed ^ splitmix64(2 * static_cast<uint64_t>(i)));
  const uint64_t b = splitmix64(seed ^ splitmix64(2 * static_cast<uint64_t>(i) + 1));
  const double u1 = (static_cast<double>(a >> 11) + 0.5) * 0x1.0p-53;
  const double u2 = (static_cast<double>(b >> 11) + 0.5) * 0x1.0p-53;
  v[i] = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}

int launch_randn(double* v, int64_t n, uint64_t seed, hipStream_t s) {
  if (n <= 0) return QSI_OK;
  hipLaunchKernelGGL(k_randn, dim3(static_cast<uint32_t>((n + 255) / 256)), dim3(256), 0, s, v,
                     n, seed);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_dot(const double* a, const double* b, int64_t n, double* partials,
               double* out, hipStream_t s) {
  const int nb = vec_blocks(n);
  hipLaunchKernelGGL(k_dot_partial, dim3(nb), dim3(kVecBlock), 0, s, a, b, n,
                     partials);
  QSI_CHECK_LAUNCH();
  launch_finalize(partials, nb, out, 0, s);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_axpy(double alpha, const double* x, double* y, int64_t n,
                hipStream_t s, const double* xs_dev) {
  hipLaunchKernelGGL(k_axpy, dim3(vec_blocks(n)), dim3(kVecBlock), 0, s, alpha,
                     x, y, n, xs_dev);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_scal(double alpha, double* x, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_scal, dim3(vec_blocks(n)), dim3(kVecBlock), 0, s, alpha,
                     x, n);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

// u -= alpha_dev * v; nrm_out[0] = ||u||, nrm_out[1] = 1/||u||
int launch_axpy_norm(const double* alpha_dev, const double* v, double* u,
                     int64_t n, double* partials, double* nrm_out,
                     hipStream_t s, const double* vs_dev) {
  const int nb = vec_blocks(n);
  hipLaunchKernelGGL(k_axpy_dev_norm, dim3(nb), dim3(kVecBlock), 0, s,
                     alpha_dev, v, u, n, partials, vs_dev);
  QSI_CHECK_LAUNCH();
  launch_finalize(partials, nb, nrm_out, 1, s);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int max_vec_partials() { return 8192; }
constexpr int kPlainPartials = 1 << 17;
int gs_partials(bool plain) {
  return plain ? kPlainPartials + kMaxCols + 1 : kGsBlocks * (2 * kMaxCols + 1);
}

namespace {
// Pass 2 of 16, 32 or 64 columns at most.
template <int T, bool SUMS>
void launch_gs_sub_dots(int nb, const double* V, int64_t ldv, int m, const double* part1,
                        double* hcol, double* w, int64_t n, double* part2, hipStream_t s) {
  if (m <= 16)
    hipLaunchKernelGGL((k_gs_sub_dots<T, 16, SUMS>), dim3(nb), dim3(T), 0, s, V, ldv, m, part1,
                       hcol, w, n, part2);
  else if (m <= 32)
    hipLaunchKernelGGL((k_gs_sub_dots<T, 32, SUMS>), dim3(nb), dim3(T), 0, s, V, ldv, m, part1,
                       hcol, w, n, part2);
  else if constexpr (T <= kVecBlock)
    hipLaunchKernelGGL((k_gs_sub_dots<T, 64, SUMS>), dim3(nb), dim3(T), 0, s, V, ldv, m, part1,
                       hcol, w, n, part2);
}

template <int T>
void launch_gs(const double* V, int64_t ldv, int m, double* w, int64_t n, double* partials,
               double* hcol, double* beta, hipStream_t s) {
  double* part2 = partials + static_cast<int64_t>(kGsBlocks) * kMaxCols;
  const int nb = static_cast<int>(std::min<int64_t>((n + T - 1) / T, kGsBlocks));
  hipLaunchKernelGGL(k_gs_dots<T>, dim3(nb), dim3(T), 0, s, V, ldv, m, w, n, partials);
  launch_gs_sub_dots<T, true>(nb, V, ldv, m, partials, hcol, w, n, part2, s);
  hipLaunchKernelGGL((k_gs_tail<T, true>), dim3(nb), dim3(T), 0, s, V, ldv, m, part2, hcol, w, n,
                     beta);
}
}  // namespace

int launch_gs_step(const double* V, int64_t ldv, int m, double* w, int64_t n, double* partials,
                   double* hcol, double* beta, bool plain, hipStream_t s) {
  if (m <= 0 || m > kMaxCols) {
    set_error("launch_gs_step: column count out of range");
    return QSI_E_INVALID;
  }
  if (plain) {
    double* g = partials + kPlainPartials;
    const int nb = std::max(1, std::min(proj_blocks(n), kPlainPartials / (m + 1)));
    hipLaunchKernelGGL(k_gs_dots<kVecBlock>, dim3(nb), dim3(kVecBlock), 0, s, V, ldv, m, w, n,
                       partials);
    hipLaunchKernelGGL(k_finalize_cols, dim3(m), dim3(256), 0, s, partials, nb, hcol);
    launch_gs_sub_dots<kVecBlock, false>(nb, V, ldv, m, hcol, nullptr, w, n, partials, s);
    hipLaunchKernelGGL(k_finalize_cols, dim3(m + 1), dim3(256), 0, s, partials, nb, g);
    hipLaunchKernelGGL((k_gs_tail<kVecBlock, false>), dim3(vec_blocks(n)), dim3(kVecBlock), 0, s,
                       V, ldv, m, g, hcol, w, n, beta);
  } else if (m <= 32) {
    launch_gs<512>(V, ldv, m, w, n, partials, hcol, beta, s);
  } else {
    launch_gs<kVecBlock>(V, ldv, m, w, n, partials, hcol, beta, s);
  }
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_multidot(const double* V, int64_t ldv, int m, const double* w, int64_t n,
                    double* partials, double* out, hipStream_t s) {
  for (int j0 = 0; j0 < m; j0 += kMaxCols) {
    const int jn = std::min(kMaxCols, m - j0);
    const int nb = std::max(1, std::min(proj_blocks(n), kPlainPartials / jn));
    hipLaunchKernelGGL(k_gs_dots<kVecBlock>, dim3(nb), dim3(kVecBlock), 0, s, V + j0 * ldv, ldv,
                       jn, w, n, partials);
    QSI_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_finalize_cols, dim3(jn), dim3(256), 0, s, partials, nb, out + j0);
    QSI_CHECK_LAUNCH();
  }
  return QSI_OK;
}

int launch_ritz(const RitzArgs& a, int n_jobs, hipStream_t s) {
  if (n_jobs < 1 || n_jobs > kMaxCols || a.m < 1 || a.m > kRitzMax) {
    set_error("launch_ritz: size out of range");
    return QSI_E_INVALID;
  }
  hipLaunchKernelGGL(k_ritz, dim3(n_jobs), dim3(kRitzThreads), 0, s, a);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_combine(const double* V, int64_t ldv, int m, const double* Y, int k,
                   double* out, int64_t ldo, int64_t n, hipStream_t s) {
  if (m > kMaxCols || k > kMaxCols) {
    set_error("launch_combine: too many columns");
    return QSI_E_INVALID;
  }
  hipLaunchKernelGGL(k_combine, dim3(vec_blocks(n)), dim3(kVecBlock), 0, s, V,
                     ldv, m, Y, k, out, ldo, n);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_copy_scaled(const double* s_dev, const double* y, double* x,
                       int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_copy_scaled, dim3(vec_blocks(n)), dim3(kVecBlock), 0, s,
                     s_dev, y, x, n);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_axpy_dev(const double* s_dev, double c, const double* x, double* y,
                    int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_axpy_dev, dim3(vec_blocks(n)), dim3(kVecBlock), 0, s,
                     s_dev, c, x, y, n);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_accum_cols(const double* v, double* Psi, int64_t ld, int nb, const double* c,
                      int64_t n, hipStream_t s, const double* vs_dev) {
  hipLaunchKernelGGL(k_accum_cols, dim3(vec_blocks(n)), dim3(kVecBlock), 0, s, v, Psi, ld, nb,
                     c, n, vs_dev);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int launch_apply_each(const qsi_basis_s* basis, const EachOp* ops, int n_ops, const double* psi,
                      int64_t ld, int n_vec, double* Y, int64_t ldy, hipStream_t s) {
  const dim3 grid(static_cast<uint32_t>((basis->dim + kApplyBlock - 1) / kApplyBlock),
                  static_cast<uint32_t>((n_ops + kEachOps - 1) / kEachOps));
  if (basis->nw == 1)
    hipLaunchKernelGGL(k_apply_each<1>, grid, dim3(kApplyBlock), 0, s, basis->view(), ops, n_ops,
                       psi, ld, n_vec, Y, ldy);
  else
    hipLaunchKernelGGL(k_apply_each<2>, grid, dim3(kApplyBlock), 0, s, basis->view(), ops, n_ops,
                       psi, ld, n_vec, Y, ldy);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

namespace {
int64_t gram_pairs(int pa, int pb, bool same) {
  const int64_t na = (pa + kGramCols - 1) / kGramCols, nb = (pb + kGramCols - 1) / kGramCols;
  return same ? na * (na + 1) / 2 : na * nb;
}
// Rows of a slab: 1024 workgroups over all pairs, at least 256 rows each; 352 on
// smaller bases, where allocating more partial sums than 11 MB takes longer than
// it gives (24 long operators on 3 vectors of 48 spins: 2.03 -> 1.69 ms).
int64_t gram_slab(int pa, int pb, bool same, int64_t n) {
  const int64_t groups = n > 1 << 20 ? 1024 : 352;
  const int64_t want = std::max<int64_t>(1, groups / gram_pairs(pa, pb, same));
  return std::max<int64_t>(256, ((n + want - 1) / want + 63) / 64 * 64);
}
}  // namespace

size_t gram_partials(int pa, int pb, bool same, int64_t n) {
  const int64_t slab = gram_slab(pa, pb, same, n);
  return static_cast<size_t>((n + slab - 1) / slab * gram_pairs(pa, pb, same)) * kGramCols *
         kGramCols;
}

int launch_gram(const double* A, int64_t lda, int pa, const double* B, int64_t ldb, int pb,
                int64_t n, double* partials, double* out, hipStream_t s) {
  const bool same = A == B && pa == pb && lda == ldb;
  const int64_t pairs = gram_pairs(pa, pb, same), slab = gram_slab(pa, pb, same, n);
  const int64_t n_slab = (n + slab - 1) / slab;
  const uint32_t py = static_cast<uint32_t>(std::min<int64_t>(pairs, 65535));
  const uint32_t pz = static_cast<uint32_t>((pairs + py - 1) / py);
  hipLaunchKernelGGL(k_gram, dim3(static_cast<uint32_t>(n_slab), py, pz), dim3(256), 0, s, A, lda,
                     pa, B, ldb, pb, n, slab, same ? 1 : 0, pairs, partials);
  QSI_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_gram_sum<kGramCols>,
                     dim3(static_cast<uint32_t>(pairs * (kGramCols * kGramCols / 32))), dim3(256),
                     0, s, partials, static_cast<int>(n_slab), pa, pb, same ? 1 : 0, pairs, out);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

bool observe_fits(const qsi_basis_s* basis, int P, int n_vec, bool gram) {
  // From three columns on.  Its wavefronts wait for one lookup after the other,
  // and with fewer operators than wavefronts most of them wait for the rest:
  // expectations of one ring, this pass / an apply and a multi-dot: 48 spins 71 / 46
  // us, 64 spins 217 / 101, 72 spins 1598 / 510; four rings on 48 spins 72 / 91.  On
  // large bases of two-word states the lookups take longer: 72 spins, 16 columns
  // 3.3 / 2.9 ms, 32 columns 4.3 / 6.5; correlations of 8 columns 2.77 / 2.72, of 16
  // 3.5 / 7.4.
  const int few = basis->nw == 2 && basis->dim >= int64_t{1} << 22 ? (gram ? 8 : 16) : 2;
  return P > few && P <= kObsCols && (gram || n_vec <= kObsVecs);
}

int observe_blocks(int64_t n) {
  // one workgroup per CU while the partial sums they leave would be most of the
  // traffic (and while their buffer, 11 MB for 96 columns, stays cheap to
  // allocate: a 22 MB one costs 0.3 ms a call), three on large bases
  return static_cast<int>(std::min<int64_t>((n + 63) / 64, n > (1 << 20) ? 768 : 256));
}

int observe_tiles(int P, bool gram) {
  const int nb = (P + 15) / 16;
  return gram ? nb * (nb + 1) / 2 : nb;
}

int launch_observe(const qsi_basis_s* basis, const ObserveArgs& q, const double* psi, int64_t ld,
                   double* partials, double* out, hipStream_t s) {
  const int nb = (q.P + 15) / 16, blocks = observe_blocks(basis->dim);
  const size_t lds = static_cast<size_t>(16 * nb + (q.same ? 0 : 16)) * kObsLd * sizeof(double);
  auto kern = basis->nw == 1 ? k_observe<1> : k_observe<2>;
  // the attribute is the process's: every call sets the most that any call needs,
  // or a thread with fewer columns could lower it under another's launch
  QSI_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (kObsCols + 16) * kObsLd * static_cast<int>(sizeof(double))));
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), lds, s, basis->view(), q, psi, ld, partials);
  QSI_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_gram_sum<16>, dim3(q.tiles * 8), dim3(256), 0, s, partials, blocks, q.P,
                     q.same ? q.P : q.n_vec, q.same, static_cast<int64_t>(q.tiles), out);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

}  // namespace qsi

// ============================================================================
// C ABI: library, basis, operator, apply, connectivity, vector ops
// ============================================================================

using namespace qsi;

extern "C" {

const char* qsi_last_error(void) { return get_error(); }

const char* qsi_version(void) { return "qsi-gpu 0.1 gfx950"; }

int qsi_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

// K = ceil(log2 D) + 7, at most 31 (an 8 GiB table) and at most n_spins.
// Ice-rule bases fill buckets very unevenly, so the table is kept wide: on
// the 64-spin Q=0 basis the 29-bit key leaves a lookup-weighted mean bucket
// of ~3.4 states (the apply 5 % faster than with 27 bits); on the 96-spin
// basis the 31-bit cap still leaves ~115 (the low-key apply 3 % faster than
// with 30 bits, one bisection step fewer).
static int auto_bucket_bits(int64_t dim, int n_spins) {
  int lg = 0;
  while ((int64_t{1} << lg) < dim) ++lg;
  int k = lg + 7;
  k = std::min(k, 31);
  k = std::min(k, n_spins);
  return std::max(k, 1);
}


// Chooses the bucket key fields from the basis's informative bit positions
// (k_diff_bits) and builds the bucket table.  K = bucket_bits, or automatic;
// at most the informative positions (a smaller K then splits the basis into
// single states) and at most kKeySegs fields.  Synchronises.
static hipError_t basis_build_index(qsi_basis_s* b, int bucket_bits) {
  int K = bucket_bits ? bucket_bits : auto_bucket_bits(b->dim, b->n_spins);
  unsigned long long hmask[2] = {0, 0};
  hipError_t e = hipSuccess;
  if (b->dim >= 2) {
    unsigned long long* dmask = nullptr;
    e = hipMalloc(&dmask, 2 * sizeof(unsigned long long));
    if (e != hipSuccess) return e;
    e = hipMemset(dmask, 0, 2 * sizeof(unsigned long long));
    const int64_t want = (b->dim + 255) / 256;
    const uint32_t grid = static_cast<uint32_t>(std::min<int64_t>(want, 8192));
    if (e == hipSuccess) {
      if (b->nw == 1)
        hipLaunchKernelGGL(k_diff_bits<1>, dim3(grid), dim3(256), 0, 0, b->d_states, b->dim, dmask);
      else
        hipLaunchKernelGGL(k_diff_bits<2>, dim3(grid), dim3(256), 0, 0, b->d_states, b->dim, dmask);
      e = hipGetLastError();
    }
    if (e == hipSuccess)
      e = hipMemcpy(hmask, dmask, sizeof(hmask), hipMemcpyDeviceToHost);
    (void)hipFree(dmask);
    if (e != hipSuccess) return e;
  }
  b->infmask[0] = hmask[0];
  b->infmask[1] = hmask[1];
  // informative positions from the top; a run starts a new field, and once
  // kKeySegs fields exist the last one is extended down over the gap (the
  // fixed positions it then covers do not break the ordering)
  b->n_seg = 0;
  int taken = 0;  // key width so far
  for (int p = b->n_spins - 1; p >= 0 && taken < K; --p) {
    if (!((hmask[p >> 6] >> (p & 63)) & 1ull)) continue;
    const int q = b->n_seg - 1;
    if (q >= 0 && b->seg_lo[q] == p + 1) {
      b->seg_lo[q] = static_cast<uint8_t>(p);
      b->seg_w[q] += 1;
      taken += 1;
    } else if (b->n_seg < kKeySegs) {
      b->seg_lo[b->n_seg] = static_cast<uint8_t>(p);
      b->seg_w[b->n_seg] = 1;
      ++b->n_seg;
      taken += 1;
    } else {
      const int grow = b->seg_lo[q] - p;
      if (taken + grow > K) break;
      b->seg_lo[q] = static_cast<uint8_t>(p);
      b->seg_w[q] += grow;
      taken += grow;
    }
  }
  if (taken == 0) {  // no informative position (dim < 2): the top K bits
    K = std::min(K, b->n_spins);
    b->n_seg = 1;
    b->seg_lo[0] = static_cast<uint8_t>(b->n_spins - K);
    b->seg_w[0] = static_cast<uint8_t>(K);
    taken = K;
  }
  b->kbits = taken;
  const size_t nkeys = size_t{1} << b->kbits;
  e = hipMalloc(&b->d_table, (nkeys + 1) * sizeof(uint32_t));
  if (e != hipSuccess) return e;
  const uint32_t grid = static_cast<uint32_t>(std::min<size_t>((nkeys + 1 + 255) / 256, 1u << 20));
  const int64_t nk = static_cast<int64_t>(nkeys);
  if (b->nw == 1)
    hipLaunchKernelGGL(k_build_table<1>, dim3(grid), dim3(256), 0, 0, b->view(), nk, b->d_table);
  else
    hipLaunchKernelGGL(k_build_table<2>, dim3(grid), dim3(256), 0, 0, b->view(), nk, b->d_table);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipDeviceSynchronize();
  return e;
}

int qsi_basis_create_ex(const uint64_t* h_lohi, int64_t dim, int n_spins,
                        int bucket_bits, int with_hash, qsi_basis_t* out) {
  QSI_REQUIRE(out != nullptr, "qsi_basis_create: out is null");
  *out = nullptr;
  QSI_REQUIRE(h_lohi != nullptr || dim == 0, "qsi_basis_create: states are null");
  QSI_REQUIRE(dim >= 0 && dim <= kMaxDim,
              "qsi_basis_create: dim must be in [0, 2^32 - 512]");
  QSI_REQUIRE(n_spins >= 1 && n_spins <= 128,
              "qsi_basis_create: n_spins must be in [1, 128]");
  QSI_REQUIRE(bucket_bits >= 0 && bucket_bits <= 32 && bucket_bits <= n_spins,
              "qsi_basis_create: bucket_bits must be in [0, min(32, n_spins)]");
  const int nw = n_spins <= 64 ? 1 : 2;
  // validate: in range and strictly increasing
  for (int64_t i = 0; i < dim; ++i) {
    const uint64_t lo = h_lohi[2 * i], hi = h_lohi[2 * i + 1];
    bool in_range;
    if (n_spins <= 64) in_range = hi == 0 && (n_spins == 64 || (lo >> n_spins) == 0);
    else in_range = (n_spins == 128) || (hi >> (n_spins - 64)) == 0;
    if (!in_range) {
      set_error("qsi_basis_create: state " + std::to_string(i) +
                " has bits at or above n_spins");
      return QSI_E_INVALID;
    }
    if (i > 0) {
      const uint64_t plo = h_lohi[2 * i - 2], phi = h_lohi[2 * i - 1];
      if (!(phi < hi || (phi == hi && plo < lo))) {
        set_error("qsi_basis_create: states are not strictly increasing at row " +
                  std::to_string(i));
        return QSI_E_INVALID;
      }
    }
  }
  auto* b = new (std::nothrow) qsi_basis_s();
  if (!b) {
    set_error("qsi_basis_create: host allocation failed");
    return QSI_E_NOMEM;
  }
  b->dim = dim;
  b->n_spins = n_spins;
  b->nw = nw;
  (void)hipGetDevice(&b->device);
  const size_t words = static_cast<size_t>(std::max<int64_t>(dim, 1)) * nw;
  auto fail = [&](hipError_t e, const char* what) {
    set_error(std::string("qsi_basis_create: ") + what + ": " + hipGetErrorString(e));
    basis_release(b);
    return e == hipErrorOutOfMemory ? QSI_E_NOMEM : QSI_E_HIP;
  };
  hipError_t e = hipMalloc(&b->d_states, words * sizeof(uint64_t));
  if (e != hipSuccess) return fail(e, "hipMalloc(states)");
  if (dim > 0) {
    if (nw == 2) {
      e = hipMemcpy(b->d_states, h_lohi, words * sizeof(uint64_t),
                    hipMemcpyHostToDevice);
    } else {
      std::vector<uint64_t> lo(static_cast<size_t>(dim));
      for (int64_t i = 0; i < dim; ++i) lo[i] = h_lohi[2 * i];
      e = hipMemcpy(b->d_states, lo.data(), words * sizeof(uint64_t),
                    hipMemcpyHostToDevice);
    }
    if (e != hipSuccess) return fail(e, "hipMemcpy(states)");
  } else {
    e = hipMemset(b->d_states, 0, words * sizeof(uint64_t));
    if (e != hipSuccess) return fail(e, "hipMemset(states)");
  }
  e = basis_build_index(b, bucket_bits);
  if (e != hipSuccess) return fail(e, "bucket table");
  if (with_hash && dim > 0) {
    int hb = 1;
    while ((int64_t{1} << hb) < 2 * dim) ++hb;  // load factor <= 1/2
    const size_t slots = size_t{1} << hb;
    const size_t bytes = slots * sizeof(ulonglong2) * nw;
    e = hipMalloc(&b->d_hash, bytes);
    if (e != hipSuccess) return fail(e, "hipMalloc(hash)");
    e = hipMemset(b->d_hash, 0xFF, bytes);
    if (e != hipSuccess) return fail(e, "hipMemset(hash)");
    b->hbits = hb;
    const uint32_t g2 = static_cast<uint32_t>((dim + 255) / 256);
    const uint64_t mask = slots - 1;
    if (nw == 1)
      hipLaunchKernelGGL(k_build_hash<1>, dim3(g2), dim3(256), 0, 0, b->d_states,
                         dim, b->d_hash, mask, hb);
    else
      hipLaunchKernelGGL(k_build_hash<2>, dim3(g2), dim3(256), 0, 0, b->d_states,
                         dim, b->d_hash, mask, hb);
    e = hipGetLastError();
    if (e != hipSuccess) return fail(e, "k_build_hash launch");
    e = hipDeviceSynchronize();
    if (e != hipSuccess) return fail(e, "k_build_hash");
  }
  *out = b;
  return QSI_OK;
}

int qsi_basis_create(const uint64_t* h_lohi, int64_t dim, int n_spins,
                     int bucket_bits, qsi_basis_t* out) {
  return qsi_basis_create_ex(h_lohi, dim, n_spins, bucket_bits, 0, out);
}

int qsi_basis_has_hash(qsi_basis_t b) { return b && b->d_hash ? 1 : 0; }

int qsi_basis_build_slots(qsi_basis_t b, int enable) {
  QSI_REQUIRE(b != nullptr, "qsi_basis_build_slots: null basis");
  QSI_REQUIRE(enable == 0 || enable == 1, "qsi_basis_build_slots: enable must be 0 or 1");
  if (!enable || b->d_slots) {
    if (!enable && b->d_slots) {
      QSI_CHECK_HIP(hipDeviceSynchronize());  // no apply may still read it
      QSI_CHECK_HIP(hipFree(b->d_slots));
      b->d_slots = nullptr;
    }
    return QSI_OK;
  }
  if (b->dim == 0) return QSI_OK;
  const size_t n = 2 * static_cast<size_t>(b->dim);
  uint32_t* slots = nullptr;
  unsigned int* flag = nullptr;
  hipError_t e = hipMalloc(&slots, n * sizeof(uint32_t));
  if (e != hipSuccess) {
    set_error(std::string("qsi_basis_build_slots: hipMalloc: ") + hipGetErrorString(e));
    return e == hipErrorOutOfMemory ? QSI_E_NOMEM : QSI_E_HIP;
  }
  e = hipMalloc(&flag, sizeof(unsigned int));
  if (e == hipSuccess) e = hipMemset(flag, 0, sizeof(unsigned int));
  if (e == hipSuccess) e = hipMemset(slots, 0xFF, n * sizeof(uint32_t));
  if (e == hipSuccess) {
    qsi::BasisView v = b->view();
    const uint32_t grid = static_cast<uint32_t>((b->dim + 255) / 256);
    if (b->nw == 1)
      hipLaunchKernelGGL(qsi::k_build_slots<1>, dim3(grid), dim3(256), 0, 0, v, slots, flag);
    else
      hipLaunchKernelGGL(qsi::k_build_slots<2>, dim3(grid), dim3(256), 0, 0, v, slots, flag);
    e = hipGetLastError();
  }
  unsigned int too_big = 0;
  if (e == hipSuccess) e = hipMemcpy(&too_big, flag, sizeof(too_big), hipMemcpyDeviceToHost);
  if (flag) (void)hipFree(flag);
  if (e != hipSuccess || too_big) {
    (void)hipFree(slots);
    if (e != hipSuccess) {
      set_error(std::string("qsi_basis_build_slots: ") + hipGetErrorString(e));
      return QSI_E_HIP;
    }
    set_error("qsi_basis_build_slots: a bucket holds more than 65535 states "
              "(a wider bucket key is needed)");
    return QSI_E_INVALID;
  }
  b->d_slots = slots;
  return QSI_OK;
}

int qsi_basis_has_slots(qsi_basis_t b) { return b && b->d_slots ? 1 : 0; }

int qsi_basis_build_lowkeys(qsi_basis_t b, int enable) {
  QSI_REQUIRE(b != nullptr, "qsi_basis_build_lowkeys: null basis");
  QSI_REQUIRE(enable == 0 || enable == 1, "qsi_basis_build_lowkeys: enable must be 0 or 1");
  if (!enable || b->d_lowkeys) {
    if (!enable && b->d_lowkeys) {
      QSI_CHECK_HIP(hipDeviceSynchronize());  // no apply may still read it
      QSI_CHECK_HIP(hipFree(b->d_lowkeys));
      b->d_lowkeys = nullptr;
    }
    return QSI_OK;
  }
  if (b->dim == 0) return QSI_OK;
  // the informative positions below the key's lowest bit, as runs from the top
  int key_lo = b->n_spins;
  for (int q = 0; q < b->n_seg; ++q) key_lo = std::min<int>(key_lo, b->seg_lo[q]);
  int n_low = 0, bits = 0;
  uint8_t lo[qsi::kLowSegs] = {}, w[qsi::kLowSegs] = {};
  for (int p = key_lo - 1; p >= 0; --p) {
    if (!((b->infmask[p >> 6] >> (p & 63)) & 1ull)) continue;
    ++bits;
    if (n_low > 0 && lo[n_low - 1] == p + 1) {
      lo[n_low - 1] = static_cast<uint8_t>(p);
      w[n_low - 1] += 1;
    } else {
      if (n_low == qsi::kLowSegs) { n_low = qsi::kLowSegs + 1; break; }
      lo[n_low] = static_cast<uint8_t>(p);
      w[n_low] = 1;
      ++n_low;
    }
  }
  QSI_REQUIRE(bits <= qsi::kLowBits && n_low <= qsi::kLowSegs,
              "qsi_basis_build_lowkeys: more than 32 informative positions lie below the "
              "bucket key (a wider key is needed)");
  uint32_t* keys = nullptr;
  hipError_t e = hipMalloc(&keys, static_cast<size_t>(b->dim) * sizeof(uint32_t));
  if (e != hipSuccess) {
    set_error(std::string("qsi_basis_build_lowkeys: hipMalloc: ") + hipGetErrorString(e));
    return e == hipErrorOutOfMemory ? QSI_E_NOMEM : QSI_E_HIP;
  }
  b->n_low = n_low;
  for (int q = 0; q < qsi::kLowSegs; ++q) {
    b->low_lo[q] = lo[q];
    b->low_w[q] = w[q];
  }
  const qsi::BasisView v = b->view();
  const uint32_t grid = static_cast<uint32_t>((b->dim + 255) / 256);
  if (b->nw == 1)
    hipLaunchKernelGGL(qsi::k_build_lowkeys<1>, dim3(grid), dim3(256), 0, 0, v, keys);
  else
    hipLaunchKernelGGL(qsi::k_build_lowkeys<2>, dim3(grid), dim3(256), 0, 0, v, keys);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    (void)hipFree(keys);
    set_error(std::string("qsi_basis_build_lowkeys: ") + hipGetErrorString(e));
    return QSI_E_HIP;
  }
  b->d_lowkeys = keys;
  return QSI_OK;
}

int qsi_basis_has_lowkeys(qsi_basis_t b) { return b && b->d_lowkeys ? 1 : 0; }

}  // extern "C"

namespace qsi {
namespace {

// flag[0] = 1 when some state has bits at or above n_spins, 2 when the
// states are not strictly increasing (any offender's code; plain stores).
template <int NW>
__global__ void k_check_sorted(const uint64_t* __restrict__ st, int64_t dim, int n_spins,
                               int* __restrict__ flag) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= dim) return;
  const State<NW> s = load_state_cached<NW>(st, i);
  bool bad_range;
  if constexpr (NW == 1) bad_range = n_spins < 64 && (s.w[0] >> n_spins) != 0;
  else bad_range = n_spins < 128 && (s.w[1] >> (n_spins - 64)) != 0;
  bool bad_order = false;
  if (i > 0) bad_order = !st_lt<NW>(load_state_cached<NW>(st, i - 1), s);
  if (bad_range || bad_order) flag[0] = bad_range ? 1 : 2;
}

}  // namespace

// A basis over device states the caller hands over (dim x nw words, freed by
// the basis): validates them on the device and builds the bucket table.
int basis_adopt_device(uint64_t* d_states, int64_t dim, int n_spins, int bucket_bits,
                       qsi_basis_s** out) {
  *out = nullptr;
  if (dim > kMaxDim) {
    (void)hipFree(d_states);
    set_error("qsi_basis: more than 2^32 - 512 states");
    return QSI_E_INVALID;
  }
  auto* b = new (std::nothrow) qsi_basis_s();
  if (!b) {
    (void)hipFree(d_states);
    set_error("qsi_basis: host allocation failed");
    return QSI_E_NOMEM;
  }
  b->dim = dim;
  b->n_spins = n_spins;
  b->nw = n_spins <= 64 ? 1 : 2;
  (void)hipGetDevice(&b->device);
  b->d_states = d_states;
  auto fail = [&](hipError_t e, const char* what) {
    set_error(std::string("qsi_basis: ") + what + ": " + hipGetErrorString(e));
    basis_release(b);
    return e == hipErrorOutOfMemory ? QSI_E_NOMEM : QSI_E_HIP;
  };
  int* flag = nullptr;
  hipError_t e = hipMalloc(&flag, sizeof(int));
  if (e == hipSuccess) e = hipMemset(flag, 0, sizeof(int));
  if (e != hipSuccess) return fail(e, "validation buffer");
  if (dim > 0) {
    const uint32_t g = static_cast<uint32_t>((dim + 255) / 256);
    if (b->nw == 1)
      hipLaunchKernelGGL(k_check_sorted<1>, dim3(g), dim3(256), 0, 0, d_states, dim, n_spins, flag);
    else
      hipLaunchKernelGGL(k_check_sorted<2>, dim3(g), dim3(256), 0, 0, d_states, dim, n_spins, flag);
  }
  int hflag = 0;
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpy(&hflag, flag, sizeof(int), hipMemcpyDeviceToHost);
  (void)hipFree(flag);
  if (e != hipSuccess) return fail(e, "validation");
  if (hflag) {
    set_error(hflag & 1 ? "qsi_basis: a state has bits at or above n_spins"
                        : "qsi_basis: states are not strictly increasing");
    basis_release(b);
    return QSI_E_INVALID;
  }
  e = basis_build_index(b, bucket_bits);
  if (e != hipSuccess) return fail(e, "bucket table");
  *out = b;
  return QSI_OK;
}

}  // namespace qsi

extern "C" {

int qsi_basis_download(qsi_basis_t b, uint64_t* h_lohi) {
  QSI_REQUIRE(b != nullptr && (h_lohi || b->dim == 0), "qsi_basis_download: null argument");
  if (b->dim == 0) return QSI_OK;
  if (b->nw == 2) {
    QSI_CHECK_HIP(hipMemcpy(h_lohi, b->d_states, static_cast<size_t>(b->dim) * 16,
                            hipMemcpyDeviceToHost));
  } else {
    std::vector<uint64_t> lo(static_cast<size_t>(b->dim));
    QSI_CHECK_HIP(hipMemcpy(lo.data(), b->d_states, lo.size() * 8, hipMemcpyDeviceToHost));
    for (int64_t i = 0; i < b->dim; ++i) {
      h_lohi[2 * i] = lo[i];
      h_lohi[2 * i + 1] = 0;
    }
  }
  return QSI_OK;
}

int qsi_basis_destroy(qsi_basis_t b) {
  if (b) basis_release(b);
  return QSI_OK;
}

int64_t qsi_basis_dim(qsi_basis_t b) { return b ? b->dim : -1; }
int qsi_basis_n_spins(qsi_basis_t b) { return b ? b->n_spins : -1; }
int qsi_basis_bucket_bits(qsi_basis_t b) { return b ? b->kbits : -1; }

int qsi_basis_key_fields(qsi_basis_t b, int* n_fields, int* lo, int* width) {
  QSI_REQUIRE(b && n_fields && lo && width, "qsi_basis_key_fields: null argument");
  *n_fields = b->n_seg;
  for (int q = 0; q < kKeySegs; ++q) {
    lo[q] = q < b->n_seg ? b->seg_lo[q] : 0;
    width[q] = q < b->n_seg ? b->seg_w[q] : 0;
  }
  return QSI_OK;
}

int qsi_basis_search(qsi_basis_t b, const uint64_t* d_lohi, int64_t n,
                     int64_t* d_rank, qsi_stream_t stream) {
  QSI_REQUIRE(b != nullptr, "qsi_basis_search: null basis");
  QSI_REQUIRE(n >= 0, "qsi_basis_search: n < 0");
  if (n == 0) return QSI_OK;
  QSI_REQUIRE(d_lohi && d_rank, "qsi_basis_search: null pointer");
  const uint32_t grid = static_cast<uint32_t>((n + 255) / 256);
  auto s = static_cast<hipStream_t>(stream);
  if (b->nw == 1)
    hipLaunchKernelGGL(k_search<1>, dim3(grid), dim3(256), 0, s, b->view(),
                       d_lohi, n, d_rank);
  else
    hipLaunchKernelGGL(k_search<2>, dim3(grid), dim3(256), 0, s, b->view(),
                       d_lohi, n, d_rank);
  QSI_CHECK_LAUNCH();
  return QSI_OK;
}

int qsi_op_create(qsi_basis_t b, const qsi_term_t* terms, int n_terms,
                  int n_slots, qsi_op_t* out) {
  QSI_REQUIRE(out != nullptr, "qsi_op_create: out is null");
  *out = nullptr;
  QSI_REQUIRE(b != nullptr, "qsi_op_create: null basis");
  QSI_REQUIRE(n_terms >= 0 && (terms != nullptr || n_terms == 0),
              "qsi_op_create: bad terms");
  QSI_REQUIRE(n_slots >= 0, "qsi_op_create: n_slots < 0");
  const int nw = b->nw;
  auto* op = new (std::nothrow) qsi_op_s();
  if (!op) {
    set_error("qsi_op_create: host allocation failed");
    return QSI_E_NOMEM;
  }
  // merged single-site Z terms: coefficient -> mask (kept in first-seen order)
  std::vector<DiagTerm> fields;
  for (int t = 0; t < n_terms; ++t) {
    const qsi_term_t& T = terms[t];
    const uint64_t bad_hi = (nw == 1) ? (T.X[1] | T.Z[1] | T.up[1] | T.down[1]) : 0;
    if (bad_hi) {
      delete op;
      set_error("qsi_op_create: term " + std::to_string(t) +
                " acts on spins >= 64 but the basis has <= 64 spins");
      return QSI_E_INVALID;
    }
    if (T.slot >= 0 && T.slot >= n_slots) {
      delete op;
      set_error("qsi_op_create: term slot out of range");
      return QSI_E_INVALID;
    }
    // a term whose sign is 0 or whose up/down masks overlap is identically 0
    if (T.sign == 0 || (T.up[0] & T.down[0]) || (T.up[1] & T.down[1])) continue;
    if ((T.X[0] | T.X[1]) == 0) {
      // diagonal: a Z string, possibly times up/down projectors (a ring
      // that visits a spin twice reduces to one)
      const bool proj = (T.up[0] | T.up[1] | T.down[0] | T.down[1]) != 0;
      const int nz = __builtin_popcountll(T.Z[0]) + __builtin_popcountll(T.Z[1]);
      if (nz == 1 && !proj) {
        // single-site Z: c * sign * Z_i.  Unslotted terms merge on equal
        // c * sign; slotted ones on equal (slot, c, sign), so that slot
        // coefficients (which replace c) apply to the whole group.
        const bool slotted = T.slot >= 0;
        const double ce = slotted ? T.coeff : T.coeff * T.sign;
        const double sg = slotted ? static_cast<double>(T.sign) : 1.0;
        bool merged = false;
        for (auto& f : fields) {
          if (f.slot == T.slot && f.c == ce && f.sgn == sg) {
            f.Z[0] |= T.Z[0];
            f.Z[1] |= T.Z[1];
            merged = true;
            break;
          }
        }
        if (!merged) {
          DiagTerm d{};
          d.Z[0] = T.Z[0];
          d.Z[1] = T.Z[1];
          d.c = ce;
          d.sgn = sg;
          d.kind = 1;
          d.slot = T.slot;
          fields.push_back(d);
        }
        continue;
      }
      DiagTerm d{};
      for (int w = 0; w < 2; ++w) {
        d.m[w] = T.up[w] | T.down[w];
        d.v[w] = T.up[w];
      }
      d.Z[0] = T.Z[0];
      d.Z[1] = T.Z[1];
      d.c = T.coeff;
      d.sgn = static_cast<double>(T.sign);
      d.kind = 0;
      d.slot = T.slot;
      op->h_diag.push_back(d);
    } else {
      OffTerm o{};
      for (int w = 0; w < 2; ++w) {
        o.m[w] = T.up[w] | T.down[w];
        o.v[w] = T.up[w] ^ (T.X[w] & o.m[w]);
        o.X[w] = T.X[w];
        o.Z[w] = T.Z[w];
      }
      o.c = T.coeff;
      o.sgn = static_cast<double>(T.sign);
      o.slot = T.slot;
      if (o.Z[0] | o.Z[1]) op->has_z = true;
      op->h_off.push_back(o);
    }
  }
  for (auto& f : fields) op->h_diag.push_back(f);
  // coefficient classes: (slot, c) pairs of the off-diagonal terms
  bool cls_ok = true;
  for (auto& o : op->h_off) {
    int k = 0;
    while (k < static_cast<int>(op->h_cls.size()) &&
           !(op->h_cls[k].slot == o.slot && op->h_cls[k].c == o.c))
      ++k;
    if (k == static_cast<int>(op->h_cls.size())) {
      if (k == kMaxCoefClasses) {
        cls_ok = false;
        break;
      }
      op->h_cls.push_back(CoefClass{o.c, o.slot, 0});
    }
    o.cls = k;
  }
  if (!cls_ok) {
    op->h_cls.clear();
    for (auto& o : op->h_off) o.cls = -1;
  }
  op->n_cls = static_cast<int>(op->h_cls.size());
  op->n_off = static_cast<int>(op->h_off.size());
  op->n_diag = static_cast<int>(op->h_diag.size());
  op->n_slots = n_slots;
  // ordered: every flipped spin is under the term's projector, so targets keep the
  // rows' order.  paired: every term's reverse (the same flip from the flipped
  // projector values) is a term too.  symmetric: with the same coefficient, slot, Z
  // string and sign, the terms being the reversed terms.  A Z on a spin that the
  // projector fixes is a sign; a Z on a flipped one changes the reverse's sign.
  {
    using Key = std::array<uint64_t, 10>;  // X, m, v; Z, coefficient, slot and sign
    auto key = [](const OffTerm& o, bool rev) {
      Key k{};
      int odd = o.sgn < 0.0 ? 1 : 0;
      for (int w = 0; w < 2; ++w) {
        const uint64_t z = o.Z[w] & ~o.m[w];
        odd += __builtin_popcountll(o.Z[w] & o.m[w] & ~o.v[w]);
        if (rev) odd += __builtin_popcountll(z & o.X[w]);
        k[w] = o.X[w];
        k[2 + w] = o.m[w];
        k[4 + w] = rev ? o.v[w] ^ (o.X[w] & o.m[w]) : o.v[w];
        k[6 + w] = z;
      }
      std::memcpy(&k[8], &o.c, sizeof(double));
      k[9] = static_cast<uint64_t>(static_cast<int64_t>(o.slot)) << 1 | (odd & 1);
      return k;
    };
    std::vector<Key> have;
    have.reserve(op->h_off.size());
    for (auto& o : op->h_off) have.push_back(key(o, false));
    std::sort(have.begin(), have.end());
    const bool once = std::adjacent_find(have.begin(), have.end()) == have.end();
    std::vector<Key> rev;
    op->ordered = op->paired = op->symmetric = true;
    for (auto& o : op->h_off) {
      op->ordered = op->ordered && ((o.X[0] & ~o.m[0]) | (o.X[1] & ~o.m[1])) == 0;
      if (!op->paired) continue;
      Key k = key(o, true), flip{};
      std::copy(k.begin(), k.begin() + 6, flip.begin());
      const auto at = std::lower_bound(have.begin(), have.end(), flip);
      op->paired = at != have.end() && std::equal(flip.begin(), flip.begin() + 6, at->begin());
      // terms listed once: as many different reverses, so each a term is enough
      op->symmetric = op->symmetric && op->paired &&
                      (!once || std::binary_search(at, have.end(), k));
      if (!once) rev.push_back(k);
    }
    if (!once && op->symmetric) {
      std::sort(rev.begin(), rev.end());
      op->symmetric = have == rev;
    }
  }
  // the terms field by field and as TermRec records, behind the full records
  // and padded to whole chunks of 64
  op->n_plane = op->n_off / 64 * 64 + 64;
  const size_t off_bytes = (std::max<size_t>(1, op->h_off.size()) * sizeof(OffTerm) + 63) / 64 * 64;
  std::vector<uint64_t> planes(static_cast<size_t>(op->n_plane) *
                                   (TermPlanes::kCount + sizeof(TermRec<2>) / sizeof(uint64_t)),
                               0);
  for (int t = 0; t < op->n_off; ++t) {
    const OffTerm& o = op->h_off[t];
    const double cs = o.c * o.sgn;
    uint64_t cw;
    std::memcpy(&cw, &cs, sizeof(cw));
    const uint32_t info = (o.cls >= 0 ? static_cast<uint32_t>(o.cls) : 0u) |
                          (o.sgn < 0.0 ? TermPlanes::kNegative : 0u) |
                          ((o.Z[0] | o.Z[1]) ? TermPlanes::kHasZ : 0u);
    const uint64_t bk = static_cast<uint64_t>(info) << 32 |
                        (nw == 1 ? bucket_key<1>(b->view(), State<1>{{o.X[0]}})
                                 : bucket_key<2>(b->view(), State<2>{{o.X[0], o.X[1]}}));
    const uint64_t field[TermPlanes::kCount] = {o.m[0], o.v[0], o.X[0], o.m[1],
                                                o.v[1], o.X[1], bk};
    for (int q = 0; q < TermPlanes::kCount; ++q)
      planes[static_cast<size_t>(q) * op->n_plane + t] = field[q];
    uint64_t* rec = planes.data() + static_cast<size_t>(TermPlanes::kCount) * op->n_plane +
                    static_cast<size_t>(t) * (nw == 1 ? sizeof(TermRec<1>) : sizeof(TermRec<2>)) /
                        sizeof(uint64_t);
    for (int w = 0; w < nw; ++w) {
      rec[w] = o.m[w];
      rec[nw + w] = o.v[w];
      rec[2 * nw + w] = o.v[w] ^ (o.X[w] & o.m[w]);
    }
    rec[3 * nw] = cw;
  }
  // record n_off connects nothing and has no match
  {
    uint64_t* rec = planes.data() + static_cast<size_t>(TermPlanes::kCount) * op->n_plane +
                    static_cast<size_t>(op->n_off) * (nw == 1 ? sizeof(TermRec<1>) : sizeof(TermRec<2>)) /
                        sizeof(uint64_t);
    rec[nw] = rec[2 * nw] = 1;
  }
  hipError_t e = hipMalloc(&op->d_off, off_bytes + planes.size() * sizeof(uint64_t));
  if (e == hipSuccess) {
    op->d_planes = reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(op->d_off) + off_bytes);
  }
  if (e == hipSuccess && !planes.empty())
    e = hipMemcpy(op->d_planes, planes.data(), planes.size() * sizeof(uint64_t),
                  hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMalloc(&op->d_diag, std::max<size_t>(1, op->h_diag.size()) * sizeof(DiagTerm));
  if (e == hipSuccess && op->n_off)
    e = hipMemcpy(op->d_off, op->h_off.data(), op->h_off.size() * sizeof(OffTerm),
                  hipMemcpyHostToDevice);
  if (e == hipSuccess && op->n_diag)
    e = hipMemcpy(op->d_diag, op->h_diag.data(), op->h_diag.size() * sizeof(DiagTerm),
                  hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMalloc(&op->d_cls, kMaxCoefClasses * sizeof(CoefClass));
  if (e == hipSuccess && op->n_cls)
    e = hipMemcpy(op->d_cls, op->h_cls.data(), op->h_cls.size() * sizeof(CoefClass),
                  hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    if (op->d_off) (void)hipFree(op->d_off);
    if (op->d_diag) (void)hipFree(op->d_diag);
    if (op->d_cls) (void)hipFree(op->d_cls);
    delete op;
    set_error(std::string("qsi_op_create: ") + hipGetErrorString(e));
    return e == hipErrorOutOfMemory ? QSI_E_NOMEM : QSI_E_HIP;
  }
  if (b->dim >= kWinMinDim && op->n_off > 0) {
    // how many of the window kernel's (tile, term) pairs have a target outside the
    // basis, by 64 tiles: AUTO's choice between kernels of equal results
    unsigned int* cnt = nullptr;
    unsigned int h[2] = {0, 0};
    e = hipMalloc(&cnt, sizeof(h));
    if (e == hipSuccess) e = hipMemset(cnt, 0, sizeof(h));
    if (e == hipSuccess) {
      if (nw == 1)
        hipLaunchKernelGGL(k_sample_closed<1>, dim3(64), dim3(256), 0, 0, b->view(), op->d_off,
                           op->n_off, cnt);
      else
        hipLaunchKernelGGL(k_sample_closed<2>, dim3(64), dim3(256), 0, 0, b->view(), op->d_off,
                           op->n_off, cnt);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(h, cnt, sizeof(h), hipMemcpyDeviceToHost);
    if (cnt) (void)hipFree(cnt);
    if (e != hipSuccess) {
      (void)hipFree(op->d_off);
      (void)hipFree(op->d_diag);
      (void)hipFree(op->d_cls);
      delete op;
      set_error(std::string("qsi_op_create: ") + hipGetErrorString(e));
      return QSI_E_HIP;
    }
    op->miss_share = h[0] ? static_cast<float>(h[1]) / static_cast<float>(h[0]) : 0.0f;
  }
  basis_retain(b);
  op->basis = b;
  *out = op;
  return QSI_OK;
}

int qsi_op_destroy(qsi_op_t op) {
  if (!op) return QSI_OK;
  if (op->d_off) (void)hipFree(op->d_off);
  if (op->d_diag) (void)hipFree(op->d_diag);
  if (op->d_cls) (void)hipFree(op->d_cls);
  if (op->d_rowptr) (void)hipFree(op->d_rowptr);
  if (op->d_cj) (void)hipFree(op->d_cj);
  if (op->d_cm) (void)hipFree(op->d_cm);
  if (op->basis) basis_release(op->basis);
  delete op;
  return QSI_OK;
}

int64_t qsi_op_dim(qsi_op_t op) { return op ? op->basis->dim : -1; }

int qsi_op_set_variant(qsi_op_t op, int variant) {
  QSI_REQUIRE(op != nullptr, "qsi_op_set_variant: null operator");
  QSI_REQUIRE(variant >= QSI_APPLY_AUTO && variant <= QSI_APPLY_LOW8,
              "qsi_op_set_variant: unknown variant");
  QSI_REQUIRE(op->basis->d_slots || variant < QSI_APPLY_SLOT2 || variant > QSI_APPLY_SLOT3,
              "qsi_op_set_variant: the basis has no slot index (qsi_basis_build_slots)");
  QSI_REQUIRE(op->basis->d_lowkeys || variant < QSI_APPLY_LOW2,
              "qsi_op_set_variant: the basis has no low keys (qsi_basis_build_lowkeys)");
  QSI_REQUIRE(variant != QSI_APPLY_CACHED || op->conn_nnz >= 0,
              "qsi_op_set_variant: no cached connectivity (qsi_op_cache_connectivity)");
  QSI_REQUIRE(op->basis->d_hash || (variant != QSI_APPLY_HASH && variant != QSI_APPLY_HASH4),
              "qsi_op_set_variant: the basis has no hash index");
  op->variant = variant;
  return QSI_OK;
}

int qsi_op_verify_lowkeys(qsi_op_t op, int* mode) {
  QSI_REQUIRE(op != nullptr, "qsi_op_verify_lowkeys: null operator");
  QSI_REQUIRE(op->basis->d_lowkeys != nullptr,
              "qsi_op_verify_lowkeys: the basis has no low keys (qsi_basis_build_lowkeys)");
  op->lowkeys_check = qsi::kLowCmpState;
  unsigned int* bad = nullptr;
  unsigned int h_bad = 0;
  QSI_CHECK_HIP(hipMalloc(&bad, sizeof(unsigned int)));
  hipError_t e = hipMemset(bad, 0, sizeof(unsigned int));
  if (e == hipSuccess && op->basis->dim > 0 && op->n_off > 0) {
    const qsi::BasisView v = op->basis->view();
    const uint32_t grid = static_cast<uint32_t>((op->basis->dim + 255) / 256);
    if (op->basis->nw == 1)
      hipLaunchKernelGGL(qsi::k_verify_lowkeys<1>, dim3(grid), dim3(256), 0, 0, v, op->d_off,
                         op->n_off, bad);
    else
      hipLaunchKernelGGL(qsi::k_verify_lowkeys<2>, dim3(grid), dim3(256), 0, 0, v, op->d_off,
                         op->n_off, bad);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(&h_bad, bad, sizeof(h_bad), hipMemcpyDeviceToHost);
  (void)hipFree(bad);
  if (e != hipSuccess) {
    set_error(std::string("qsi_op_verify_lowkeys: ") + hipGetErrorString(e));
    return QSI_E_HIP;
  }
  op->lowkeys_check = (h_bad & 1u) ? qsi::kLowCmpState
                    : (h_bad & 2u) ? qsi::kLowCmpKey
                                   : qsi::kLowTrusted;
  if (mode) *mode = op->lowkeys_check;
  return QSI_OK;
}

int qsi_op_get_variant(qsi_op_t op) { return op ? op->variant : -1; }

int qsi_op_set_cached_pipe(qsi_op_t op, int pipe) {
  QSI_REQUIRE(op != nullptr, "qsi_op_set_cached_pipe: null operator");
  QSI_REQUIRE(pipe == 4 || pipe == 8 || pipe == 16 || pipe == 32,
              "qsi_op_set_cached_pipe: pipe must be 4, 8, 16 or 32");
  op->cached_pipe = pipe;
  return QSI_OK;
}

int qsi_op_get_cached_pipe(qsi_op_t op) { return op ? op->cached_pipe : -1; }

int qsi_op_set_block_cfg(qsi_op_t op, int cfg) {
  QSI_REQUIRE(op != nullptr, "qsi_op_set_block_cfg: null operator");
  QSI_REQUIRE(cfg >= 0 && cfg <= 15 && blk_cfg_kernel(cfg) <= 2,
              "qsi_op_set_block_cfg: cfg must be kernel 0-2, plus 4 for a half grid, "
              "plus 8 for column pairs");
  op->blk_cfg = cfg;
  return QSI_OK;
}

int qsi_op_get_block_cfg(qsi_op_t op) { return op ? op->blk_cfg : -1; }
int qsi_op_n_offdiag(qsi_op_t op) { return op ? op->n_off : -1; }
int qsi_op_n_diag(qsi_op_t op) { return op ? op->n_diag : -1; }

int qsi_op_apply(qsi_op_t op, const double* d_x, double* d_y, int accumulate,
                 qsi_stream_t stream) {
  QSI_REQUIRE(op != nullptr, "qsi_op_apply: null operator");
  if (op->basis->dim == 0) return QSI_OK;
  QSI_REQUIRE(d_x && d_y, "qsi_op_apply: null vector");
  QSI_REQUIRE(d_x != d_y, "qsi_op_apply: x and y must not alias");
  return launch_apply(op, d_x, d_y, accumulate ? d_y : nullptr, 1.0, nullptr,
                      nullptr, static_cast<hipStream_t>(stream));
}

int qsi_op_apply_host(qsi_op_t op, const double* h_x, double* h_y,
                      int accumulate) {
  QSI_REQUIRE(op != nullptr, "qsi_op_apply_host: null operator");
  const int64_t D = op->basis->dim;
  if (D == 0) return QSI_OK;
  QSI_REQUIRE(h_x && h_y, "qsi_op_apply_host: null vector");
  double *dx = nullptr, *dy = nullptr;
  const size_t bytes = static_cast<size_t>(D) * sizeof(double);
  QSI_CHECK_HIP(hipMalloc(&dx, bytes));
  hipError_t e = hipMalloc(&dy, bytes);
  if (e == hipSuccess) e = hipMemcpy(dx, h_x, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess && accumulate) e = hipMemcpy(dy, h_y, bytes, hipMemcpyHostToDevice);
  int rc = QSI_OK;
  if (e == hipSuccess) {
    rc = launch_apply(op, dx, dy, accumulate ? dy : nullptr, 1.0, nullptr,
                      nullptr, nullptr);
    if (rc == QSI_OK) e = hipMemcpy(h_y, dy, bytes, hipMemcpyDeviceToHost);
  }
  (void)hipFree(dx);
  if (dy) (void)hipFree(dy);
  if (e != hipSuccess) {
    set_error(std::string("qsi_op_apply_host: ") + hipGetErrorString(e));
    return QSI_E_HIP;
  }
  return rc;
}

int qsi_op_apply_block(qsi_op_t op, const double* d_X, int64_t ldx, double* d_Y,
                       int64_t ldy, int R, const double* d_coeffs,
                       int accumulate, qsi_stream_t stream) {
  QSI_REQUIRE(op != nullptr, "qsi_op_apply_block: null operator");
  QSI_REQUIRE(R >= 1 && R <= 64, "qsi_op_apply_block: R must be in [1, 64]");
  QSI_REQUIRE(ldx >= R && ldy >= R, "qsi_op_apply_block: ld < R");
  QSI_REQUIRE(d_coeffs == nullptr || op->n_slots > 0,
              "qsi_op_apply_block: coefficients given but the operator has no slots");
  if (op->basis->dim == 0) return QSI_OK;
  QSI_REQUIRE(d_X && d_Y, "qsi_op_apply_block: null matrix");
  QSI_REQUIRE(d_X != d_Y, "qsi_op_apply_block: X and Y must not alias");
  BlkArgs a{};
  a.n_sec = 1;
  a.R = R;
  int G = 64;
  while (G / 2 >= R && G > 1) G >>= 1;
  a.G = G;
  a.ldx = ldx;
  a.ldy = ldy;
  a.accumulate = accumulate ? 1 : 0;
  a.y_colmajor = 0;
  a.sec[0].b = op->basis->view();
  a.sec[0].off = op->d_off;
  a.sec[0].tp = op->planes();
  a.sec[0].dg = op->d_diag;
  a.sec[0].cls = op->d_cls;
  a.sec[0].n_cls = op->n_cls;
  a.sec[0].coeffs = d_coeffs;
  a.sec[0].n_off = op->n_off;
  a.sec[0].n_diag = op->n_diag;
  a.sec[0].rowptr = op->d_rowptr;
  a.sec[0].cj = op->d_cj;
  a.sec[0].cm = op->d_cm;
  blk_set_tiles(a);
  a.cfg = op->blk_cfg;
  const int nb = blk_apply_blocks(a, op->basis->nw);
  return launch_blk_apply(a, op->basis->nw, nb, d_X, d_Y, nullptr,
                          static_cast<hipStream_t>(stream));
}

int qsi_op_connectivity(qsi_op_t op, int64_t* nnz, int64_t* d_rows,
                        int64_t* d_cols, double* d_vals, double* d_diag) {
  QSI_REQUIRE(op != nullptr && nnz != nullptr, "qsi_op_connectivity: null argument");
  const int64_t D = op->basis->dim;
  if (D == 0) {
    *nnz = 0;
    return QSI_OK;
  }
  int64_t *counts = nullptr, *offsets = nullptr;
  void* tmp = nullptr;
  size_t tmp_bytes = 0;
  const uint32_t grid = static_cast<uint32_t>((D + 255) / 256);
  auto cleanup = [&]() {
    if (counts) (void)hipFree(counts);
    if (offsets) (void)hipFree(offsets);
    if (tmp) (void)hipFree(tmp);
  };
  hipError_t e = hipMalloc(&counts, static_cast<size_t>(D + 1) * sizeof(int64_t));
  if (e == hipSuccess) e = hipMalloc(&offsets, static_cast<size_t>(D + 1) * sizeof(int64_t));
  if (e == hipSuccess) e = hipMemset(counts, 0, static_cast<size_t>(D + 1) * sizeof(int64_t));
  if (e != hipSuccess) {
    cleanup();
    set_error(std::string("qsi_op_connectivity: ") + hipGetErrorString(e));
    return QSI_E_HIP;
  }
  auto view = op->basis->view();
  if (op->basis->nw == 1)
    hipLaunchKernelGGL(k_conn<1>, dim3(grid), dim3(256), 0, 0, view, op->d_off,
                       op->n_off, op->d_diag, op->n_diag, nullptr, counts,
                       nullptr, nullptr, nullptr, d_rows ? d_diag : nullptr);
  else
    hipLaunchKernelGGL(k_conn<2>, dim3(grid), dim3(256), 0, 0, view, op->d_off,
                       op->n_off, op->d_diag, op->n_diag, nullptr, counts,
                       nullptr, nullptr, nullptr, d_rows ? d_diag : nullptr);
  e = hipGetLastError();
  if (e == hipSuccess)
    e = hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, counts, offsets, D + 1);
  if (e == hipSuccess) e = hipMalloc(&tmp, std::max<size_t>(tmp_bytes, 1));
  if (e == hipSuccess)
    e = hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, counts, offsets, D + 1);
  int64_t total = 0;
  if (e == hipSuccess)
    e = hipMemcpy(&total, offsets + D, sizeof(int64_t), hipMemcpyDeviceToHost);
  if (e != hipSuccess) {
    cleanup();
    set_error(std::string("qsi_op_connectivity: ") + hipGetErrorString(e));
    return QSI_E_HIP;
  }
  if (d_rows == nullptr) {
    *nnz = total;
    cleanup();
    return QSI_OK;
  }
  if (*nnz < total || !d_cols || !d_vals || !d_diag) {
    cleanup();
    set_error("qsi_op_connectivity: output arrays too small or null");
    return QSI_E_INVALID;
  }
  if (op->basis->nw == 1)
    hipLaunchKernelGGL(k_conn<1>, dim3(grid), dim3(256), 0, 0, view, op->d_off,
                       op->n_off, op->d_diag, op->n_diag, offsets, nullptr,
                       d_rows, d_cols, d_vals, d_diag);
  else
    hipLaunchKernelGGL(k_conn<2>, dim3(grid), dim3(256), 0, 0, view, op->d_off,
                       op->n_off, op->d_diag, op->n_diag, offsets, nullptr,
                       d_rows, d_cols, d_vals, d_diag);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipDeviceSynchronize();
  cleanup();
  if (e != hipSuccess) {
    set_error(std::string("qsi_op_connectivity: ") + hipGetErrorString(e));
    return QSI_E_HIP;
  }
  *nnz = total;
  return QSI_OK;
}

int qsi_vec_dot(const double* d_a, const double* d_b, int64_t n, double* h_out,
                qsi_stream_t stream) {
  QSI_REQUIRE(h_out != nullptr, "qsi_vec_dot: null output");
  if (n <= 0) {
    *h_out = 0.0;
    return QSI_OK;
  }
  QSI_REQUIRE(d_a && d_b, "qsi_vec_dot: null vector");
  auto s = static_cast<hipStream_t>(stream);
  double* buf = nullptr;
  QSI_CHECK_HIP(hipMalloc(&buf, (max_vec_partials() + 2) * sizeof(double)));
  int rc = launch_dot(d_a, d_b, n, buf + 2, buf, s);
  hipError_t e = hipSuccess;
  if (rc == QSI_OK) e = hipMemcpyAsync(h_out, buf, sizeof(double), hipMemcpyDeviceToHost, s);
  if (rc == QSI_OK && e == hipSuccess) e = hipStreamSynchronize(s);
  (void)hipFree(buf);
  if (e != hipSuccess) {
    set_error(std::string("qsi_vec_dot: ") + hipGetErrorString(e));
    return QSI_E_HIP;
  }
  return rc;
}

int qsi_vec_axpy(double alpha, const double* d_x, double* d_y, int64_t n,
                 qsi_stream_t stream) {
  if (n <= 0) return QSI_OK;
  QSI_REQUIRE(d_x && d_y, "qsi_vec_axpy: null vector");
  return launch_axpy(alpha, d_x, d_y, n, static_cast<hipStream_t>(stream));
}

int qsi_vec_scal(double alpha, double* d_x, int64_t n, qsi_stream_t stream) {
  if (n <= 0) return QSI_OK;
  QSI_REQUIRE(d_x, "qsi_vec_scal: null vector");
  return launch_scal(alpha, d_x, n, static_cast<hipStream_t>(stream));
}

int qsi_vec_randn(double* d_x, int64_t n, uint64_t seed, qsi_stream_t stream) {
  if (n <= 0) return QSI_OK;
  QSI_REQUIRE(d_x, "qsi_vec_randn: null vector");
  return launch_randn(d_x, n, seed, static_cast<hipStream_t>(stream));
}

}  // extern "C"
