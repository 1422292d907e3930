// Fused multi-input, multi-output LTI state space of order M <= 4 with up to
// four inputs and four outputs per step, in one pass (philtorch/lti/ssm.py:
// 386-589: state_space with a 3D input (batch, time, features), B an M x F
// matrix, C a P x M matrix, D a P x F matrix, each per row or shared; the
// glue of lti/ssm.py:467-471, 493-506 and _ssm_C_D :513-589 folded into the
// scan):
//     h[0] = zi,  y[t] = C h[t] + D x[t],  h[t+1] = A h[t] + B x[t],  zf = h[T]
// x is [rows, T, F] and y [rows, T, P], both with the features innermost.
// Per step F inputs and P outputs move; the reference route writes and reads
// B x, the state sequence, its shifted copy, C h and D x.
//
// The decomposition and the look-back are the LTI state space's
// (phs_ss.hpp): a lane folds its K steps of B x[t] from a zero state in
// compute precision, the data waves scan these vectors against a table of
// A^(K 2^i) in LDS (every map's matrix part is a known power of A, so a level
// is M^2 work on a vector, not M^3 on a map), a look-back wave resolves the
// tile's entry state over vector status words, and pass 2 re-runs the steps
// from each lane's entry state, writing C h + D x.  The input width F is a
// template parameter of the LTI kernel (a lane reads its K steps' inputs,
// consecutive elements of the row, straight into registers), the output
// width P an argument: outputs leave through P planes in LDS, so that the
// stores cover the span's contiguous block.  The time-varying kernel
// (lpv_mimo_kernel) stages its inputs through such planes too.  The
// reversed mode (REV) runs the model backwards in time: the gradients w.r.t.
// x and zi are that mode on the adjoint model (A^T, input matrix C^T, output
// matrix B^T, feedthrough D^T).  The coefficient gradients reduce against the
// state before every step, which the LTI kernel's HS mode writes beside the
// outputs or alone, and the time-varying kernel gives where P + M fit its
// planes, else as its output with C = I and no D.
#pragma once

#include "phs_lpvss.hpp"

namespace phs {

// Largest F and P of a call (the register arrays of the model and of a
// lane's per-step inputs and outputs are this wide).
constexpr int kMimoMaxIO = 4;

template <class Alg>
struct MimoArgs {
  using E = typename Alg::elem;
  const E *A;  // [rows, M, M] row-major; time-varying (lpv_mimo_kernel): [rows, T, M, M]
  int64_t A_stride;  // elements between rows (0 = shared)
  int A_trans;       // time-varying: read each step's matrix transposed (the adjoint model's A[t]^T)
  const E *Bm;  // [rows, M, F]
  int64_t b_stride;
  const E *Cm;  // [rows, P, M]
  int64_t c_stride;
  const E *Dm;  // [rows, P, F]; nullptr: no feedthrough
  int64_t d_stride;
  int F, P;
  unsigned p_magic18;  // ceil(2^18 / P) (mimo_split)
  uint64_t f_magic, p_magic;  // ceil(2^32 / F), ceil(2^32 / P): e / F = (e * f_magic) >> 32 for small e
  // the state before every step [B, T, M] as well (nullable;
  // lpv_mimo_kernel: P + M <= kMimoMaxIO planes), m_magic = ceil(2^32 / M)
  E *hs;
  uint64_t m_magic;
  const E *zi;  // [B, M]; nullptr: zeros
  const E *x;   // [B, T, F]
  E *y;         // [B, T, P]
  E *zf;        // [B, M]; nullable (the state after the last step scanned)
  int64_t B, T_len, tiles_per_row;
  uint64_t b_magic;  // tile id -> row by multiply and shift (row_split)
  unsigned b_shift;
  unsigned long long *claims;
  unsigned tiles, per_stripe, spin_limit;
  unsigned agg_only;  // testing: tiles after a row's first publish no inclusive state
  uint64_t *status;
};

// 3 data waves and a look-back wave; a lane owns K consecutive steps (64
// bytes of one feature), whose inputs it holds in registers from the load to
// pass 2, a wave 64 K steps.  Outputs (P planes) and, in the states mode,
// groups of kHsGroup states leave through the wave's part of dynamic LDS; a
// lane's steps lie kPitch = K + 1 elements apart there, so that the lanes'
// writes of one step fall in distinct banks.
//
// What bounds it: vector instructions and a tile's latency, not bytes.  At
// order 4, 2 in and 2 out, 16 x 480000 fp32, with inputs staged through LDS
// planes, every width padded to four and 8 steps a lane it issued 233 vector
// instructions a step and took 103 us; with the exact input width, its
// model in scalar registers and 16 steps a lane 58 (2.1 TB/s).  8 steps a
// lane take 76, 7 data waves 76; 3 in and 3 out 115 -> 74 (8 steps: 85);
// order 2, 1 in and 1 out 56 -> 31; order 4 fp64 (16 x 240000) 115 -> 60.
//
// Half as many steps a lane where 64 bytes of every feature are too many:
// order 4 with 4 inputs in fp32 always (4 out: with 16 steps a lane it
// spilled 46 to 66 VGPRs and took 125 us for 107, 16 x 24001 27.1 for 21.3),
// and in fp64 with 3 or 4 inputs in the SHORT form, for launches whose tiles
// would not fill the chip (kMimoShortTiles).
template <class Alg, int F, bool SHORT = false>
struct MimoShape {
  using E = typename Alg::elem;
  static constexpr int M = int(sizeof(typename Alg::s_state) / sizeof(E));
  static constexpr bool kHasShort = sizeof(E) == 8 && M == 4 && F >= 3;
  static_assert(kHasShort || !SHORT, "no short form");
  static constexpr int kWaves = 3;
  static constexpr int kThreads = 64 * (kWaves + 1);
  static constexpr int K = (SHORT || (sizeof(E) == 4 && M == 4 && F == 4) ? 32 : 64) / int(sizeof(E));
  static constexpr int kSpan = 64 * K;
  static constexpr int kTile = kWaves * kSpan;
  static constexpr int kPitch = K + 1;
  static constexpr int kPlane = 64 * kPitch;
  // states mode: a lane's group of states, at most 64 bytes of whole vectors
  static constexpr int kHsFit = (M == 3 ? 4 : 16 / M) * 4 / int(sizeof(E));
  static constexpr int kHsGroup = kHsFit < K ? kHsFit : K;
  static constexpr int kHsVecs = kHsGroup * int(sizeof(typename Alg::s_state)) / 16;
  static constexpr int kMinWaves = sizeof(E) == 4 ? 3 : 2;
  // dynamic LDS of a launch with P output planes
  static size_t lds_bytes(int P, bool hs) {
    return size_t(kWaves) * (align16(size_t(P) * kPlane * sizeof(E)) + (hs ? 64 * 16 * size_t(kHsVecs) : 0));
  }
  static constexpr __host__ __device__ size_t align16(size_t n) { return (n + 15) / 16 * 16; }
};

// Fewer tiles than this take the SHORT form: two workgroups of the long one
// fit a CU.  Order 4 fp64, 4 in and 4 out, forward (us), long / short: 16 x
// 3000 24.8 / 18.1, 16 x 24001 (256 long tiles) 28.1 / 23.6, 16 x 131072
// (1376) 76.0 / 78.0, 1024 x 4096 (3072) 129 / 139; 3 in and 4 out 21.4 /
// 17.4, 23.8 / 21.6, 63.7 / 72.6, 108 / 132.
constexpr int64_t kMimoShortTiles = 512;

// The span's element e of a [T, P] row block: step e / P, output e % P, for
// e < 64 K P <= 4096 (24-bit multiplies; magic = ceil(2^18 / P)).
__device__ __forceinline__ void mimo_split(unsigned e, unsigned P, unsigned magic, unsigned &s, unsigned &p) {
  s = __umul24(e, magic) >> 18;
  p = e - __umul24(s, P);
}

// The model of row b in two halves, each loaded where it is first needed
// (a half that lives across the wave scan holds registers the scan's maps
// want): the input side, A and the columns of B as state vectors; the output
// side, the rows of C as state vectors and D by element.  Zero past F and P,
// so that every step runs the same arithmetic whatever the widths.
template <class Alg>
struct MimoIn {
  typename Alg::s_coef A;
  typename Alg::s_state b[kMimoMaxIO];
};
template <class Alg>
struct MimoOut {
  using E = typename Alg::elem;
  typename Alg::s_state c[kMimoMaxIO];
  E d[kMimoMaxIO][kMimoMaxIO];
};

template <class Alg>
__device__ __forceinline__ MimoIn<Alg> mimo_in(const MimoArgs<Alg> &a, int64_t row) {
  using E = typename Alg::elem;
  using V = SsView<Alg>;
  constexpr int M = V::M;
  MimoIn<Alg> m;
  m.A = V::load_mat(a.A + row * a.A_stride);
  const E *bp = a.Bm + row * a.b_stride;
#pragma unroll
  for (int j = 0; j < kMimoMaxIO; ++j) {
    union {
      typename Alg::s_state s;
      E e[M];
    } u;
#pragma unroll
    for (int i = 0; i < M; ++i) u.e[i] = j < a.F ? bp[i * a.F + j] : E(0);
    m.b[j] = u.s;
  }
  return m;
}

template <class Alg>
__device__ __forceinline__ MimoOut<Alg> mimo_out(const MimoArgs<Alg> &a, int64_t row) {
  using E = typename Alg::elem;
  using V = SsView<Alg>;
  constexpr int M = V::M;
  MimoOut<Alg> m;
  const E *cp = a.Cm + row * a.c_stride;
  const E *dp = a.Dm ? a.Dm + row * a.d_stride : nullptr;
#pragma unroll
  for (int j = 0; j < kMimoMaxIO; ++j) {
    union {
      typename Alg::s_state s;
      E e[M];
    } u;
#pragma unroll
    for (int i = 0; i < M; ++i) u.e[i] = j < a.P ? cp[j * M + i] : E(0);
    m.c[j] = u.s;
#pragma unroll
    for (int f = 0; f < kMimoMaxIO; ++f) m.d[j][f] = (dp && j < a.P && f < a.F) ? dp[j * a.F + f] : E(0);
  }
  return m;
}

// B u for one step's inputs u (zero past F)
template <class Alg>
__device__ __forceinline__ typename Alg::s_state mimo_bx(const MimoIn<Alg> &m, const typename Alg::elem (&u)[kMimoMaxIO]) {
  using E = typename Alg::elem;
  constexpr int M = SsView<Alg>::M;
  union {
    typename Alg::s_state s;
    E e[M];
  } o, ub;
#pragma unroll
  for (int i = 0; i < M; ++i) o.e[i] = E(0);
#pragma unroll
  for (int f = 0; f < kMimoMaxIO; ++f) {
    ub.s = m.b[f];
#pragma unroll
    for (int i = 0; i < M; ++i) o.e[i] = fma(ub.e[i], u[f], o.e[i]);
  }
  return o.s;
}

// The elements [lo, hi) of a block of `len` elements starting at element
// `base` of a row of `lim` elements that lie inside the row (clamped to
// [0, len]; lo >= hi when none do).  One bounds test per element serves
// every span: a separate unchecked path for whole spans made the compiler
// keep both paths' loads live (2.9 KB of scratch per lane).
__device__ __forceinline__ void mimo_block_range(int64_t base, int64_t lim, int len, int &lo, int &hi) {
  const int64_t l = base < 0 ? -base : 0, h = lim - base;
  lo = int(l < len ? l : len);
  hi = int(h < 0 ? 0 : (h < len ? h : len));
}

// Stages a wave's span of one [T, W] row block into W LDS planes: plane j
// holds feature j of the span's 64 K steps in scan order (forward: scan
// position s0 + s is time s0 + s; REV: time T-1-s0-s).  Steps outside the
// row read 0.  The global side is the span's contiguous block of 64 K W
// elements, lane-strided (element e = i 64 + lane is step e / W, feature
// e % W of the block).
template <class Alg, bool REV, class Sh>
__device__ __forceinline__ void mimo_stage_in(const typename Alg::elem *row, int64_t s0, int64_t T, int W,
                                              uint64_t w_magic, typename Alg::elem *lds, int lane) {
  using E = typename Alg::elem;
  constexpr int S = Sh::kSpan, K = Sh::K, kMax = K * kMimoMaxIO;
  // the block starts at element `base` of the row (negative or past the row
  // for the spans that leave it); its elements [lo, hi) lie inside the row
  const int64_t base = (REV ? T - s0 - S : s0) * W;
  const int n = K * W;  // elements per lane
  int lo, hi;
  mimo_block_range(base, T * W, S * W, lo, hi);
  E v[kMax];
#pragma unroll
  for (int i = 0; i < kMax; ++i) {
    const int e = i * 64 + lane;
    v[i] = E(0);
    if (i < n && e >= lo && e < hi) v[i] = row[base + e];
  }
#pragma unroll
  for (int i = 0; i < kMax; ++i) {
    if (i < n) {
      const unsigned e = unsigned(i * 64 + lane);
      const unsigned s = unsigned((uint64_t(e) * w_magic) >> 32);
      const unsigned j = e - s * unsigned(W);
      lds[j * Sh::kPlane + (REV ? S - 1 - int(s) : int(s))] = v[i];
    }
  }
}

// The inverse of mimo_stage_in for a wave's outputs: W planes out to the
// span's block of the [T, W] row; steps outside the row are not written.
template <class Alg, bool REV, class Sh>
__device__ __forceinline__ void mimo_stage_out(typename Alg::elem *row, int64_t s0, int64_t T, int W,
                                               uint64_t w_magic, const typename Alg::elem *lds, int lane) {
  using E = typename Alg::elem;
  constexpr int S = Sh::kSpan, K = Sh::K, kMax = K * kMimoMaxIO;
  const int64_t base = (REV ? T - s0 - S : s0) * W;
  const int n = K * W;
  int lo, hi;
  mimo_block_range(base, T * W, S * W, lo, hi);
  E v[kMax];
#pragma unroll
  for (int i = 0; i < kMax; ++i) {
    if (i < n) {
      const unsigned e = unsigned(i * 64 + lane);
      const unsigned s = unsigned((uint64_t(e) * w_magic) >> 32);
      const unsigned j = e - s * unsigned(W);
      v[i] = lds[j * Sh::kPlane + (REV ? S - 1 - int(s) : int(s))];
    }
  }
#pragma unroll
  for (int i = 0; i < kMax; ++i) {
    const int e = i * 64 + lane;
    if (i < n && e >= lo && e < hi) row[base + e] = v[i];
  }
}

// Time of scan position s in a row of T steps.
template <bool REV>
__device__ __forceinline__ int64_t mimo_time(int64_t s, int64_t T) {
  return REV ? T - 1 - s : s;
}

// One step's F features of a row.
template <typename E, int F>
struct IoVec {
  E e[F];
};

// The row's model at input width F, wave-uniform: fp32 entries in scalar
// registers (one scalar operand an FMA), fp64 ones as the compiler places
// them (the matrices alone would fill the scalar registers).
template <class Alg, int F>
struct MimoModel {
  using E = typename Alg::elem;
  static constexpr int M = SsView<Alg>::M;
  E A[M][M], b[M][F], c[kMimoMaxIO][M], d[kMimoMaxIO][F];
};
template <typename E>
__device__ __forceinline__ E mimo_uniform(E v) {
  if constexpr (sizeof(E) == 4)
    return read_lane(v, 0);
  else
    return v;
}
template <class Alg, int F>
__device__ __forceinline__ void mimo_model(const MimoArgs<Alg> &a, int64_t row, MimoModel<Alg, F> &m) {
  using E = typename Alg::elem;
  constexpr int M = SsView<Alg>::M;
  const E *pA = a.A + row * a.A_stride, *pb = a.Bm + row * a.b_stride, *pc = a.Cm + row * a.c_stride;
  const E *pd = a.Dm ? a.Dm + row * a.d_stride : pA;
  // every read before any use; past P (or without D) an in-bounds stand-in, not used
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) m.A[i][j] = pA[i * M + j];
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int f = 0; f < F; ++f) m.b[i][f] = pb[i * F + f];
#pragma unroll
  for (int p = 0; p < kMimoMaxIO; ++p) {
    const int pp = p < a.P ? p : 0;
#pragma unroll
    for (int i = 0; i < M; ++i) m.c[p][i] = pc[pp * M + i];
#pragma unroll
    for (int f = 0; f < F; ++f) m.d[p][f] = pd[a.Dm ? pp * F + f : 0];
  }
}
template <class Alg, int F>
__device__ __forceinline__ void mimo_model_uniform(MimoModel<Alg, F> &m) {
  constexpr int M = SsView<Alg>::M;
#pragma unroll
  for (int i = 0; i < M; ++i) {
#pragma unroll
    for (int j = 0; j < M; ++j) m.A[i][j] = mimo_uniform(m.A[i][j]);
#pragma unroll
    for (int f = 0; f < F; ++f) m.b[i][f] = mimo_uniform(m.b[i][f]);
  }
#pragma unroll
  for (int p = 0; p < kMimoMaxIO; ++p) {
#pragma unroll
    for (int i = 0; i < M; ++i) m.c[p][i] = mimo_uniform(m.c[p][i]);
#pragma unroll
    for (int f = 0; f < F; ++f) m.d[p][f] = mimo_uniform(m.d[p][f]);
  }
}

// o = B u in storage precision
template <class Alg, int F>
__device__ __forceinline__ void mimo_bu(const MimoModel<Alg, F> &m, const IoVec<typename Alg::elem, F> &u,
                                        typename Alg::elem (&o)[SsView<Alg>::M]) {
#pragma unroll
  for (int i = 0; i < SsView<Alg>::M; ++i) {
    o[i] = m.b[i][0] * u.e[0];
#pragma unroll
    for (int f = 1; f < F; ++f) o[i] = fma(m.b[i][f], u.e[f], o[i]);
  }
}

// A lane's K steps from a zero state, sum_k A^(K-1-k) B x[k], in compute
// precision (the vector part of its map; the matrix part is A^K).  Folding
// in storage precision let float32 rounding in the lane maps of a model
// with a large transient gain reach 3e-4 of the output's range, ten times a
// sequential float32 loop's error; from an exact entry state, pass 2's K
// float32 steps add only a few ulps.  mid: the same over the first K/2 steps
// (fp32: pass 2 takes the state at the lane's middle from it, exact to
// compute precision, so its float32 steps run K/2 at a time: 16 in a row
// took the order-4 outputs from 9e-8 to 1.5e-7 of their norm).
template <class Alg, int F, int K>
__device__ __forceinline__ typename Alg::state mimo_lane_fold(const MimoModel<Alg, F> &m,
                                                              const IoVec<typename Alg::elem, F> (&X)[K],
                                                              typename Alg::state *mid = nullptr) {
  using C = typename Alg::ct;
  using E = typename Alg::elem;
  constexpr int M = SsView<Alg>::M;
  C A[M][M], v[M];
  E o[M];
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) A[i][j] = up(m.A[i][j]);
  mimo_bu<Alg, F>(m, X[0], o);
#pragma unroll
  for (int i = 0; i < M; ++i) v[i] = up(o[i]);
#pragma unroll
  for (int k = 1; k < K; ++k) {
    if (mid && k == K / 2) {
      union {
        typename Alg::state s;
        C e[M];
      } um;
#pragma unroll
      for (int i = 0; i < M; ++i) um.e[i] = v[i];
      *mid = um.s;
    }
    C n[M];
    mimo_bu<Alg, F>(m, X[k], o);
#pragma unroll
    for (int i = 0; i < M; ++i) {
      n[i] = up(o[i]);
#pragma unroll
      for (int j = M - 1; j >= 0; --j) n[i] = mad(A[i][j], v[j], n[i]);
    }
#pragma unroll
    for (int i = 0; i < M; ++i) v[i] = n[i];
  }
  union {
    typename Alg::state s;
    C e[M];
  } u;
#pragma unroll
  for (int i = 0; i < M; ++i) u.e[i] = v[i];
  return u.s;
}

// State entering tile position `span` of a row, folded from the inputs (the
// look-back's bounded-wait fallback; out of line, cold): 64 K steps at a
// time, st <- A^(64 K) st + the chunk's total.
template <class Alg, int F, bool REV, bool SHORT>
__device__ __noinline__ typename Alg::state mimo_prefix_fallback(const MimoArgs<Alg> *ap, int64_t b, int64_t span,
                                                                int lane, typename Alg::state st,
                                                                const SsPowers<Alg> *tab) {
  const MimoArgs<Alg> &a = *ap;
  using X = IoVec<typename Alg::elem, F>;
  constexpr int K = MimoShape<Alg, F, SHORT>::K;
  MimoModel<Alg, F> m;
  mimo_model<Alg, F>(a, b, m);
  const X *xrow = reinterpret_cast<const X *>(a.x) + b * a.T_len;
  for (int64_t off = 0; off < span; off += 64 * K) {
    ss_reload_tables();
    X xs[K];
    ss_load<REV, X, K>(xrow, off + int64_t(lane) * K, a.T_len, xs);
    typename Alg::state v[1] = {mimo_lane_fold<Alg, F, K>(m, xs)};
    ss_lane_scan<Alg, 1, false>(v, lane, tab->pw);
    st = Alg::affine(tab->pw[6], st, read_lane(v[0], 63));
  }
  return st;
}

// HS: also the state before every step into a.hs (with P = 0 the states
// alone): 16 x 480000 fp32, order 4, 2 in 2 out, 76 us with the outputs and 62
// without, where a second pass with C the identity took 95.
template <class Alg, int F, bool REV, bool HS, bool SHORT>
__global__ __launch_bounds__((MimoShape<Alg, F, SHORT>::kThreads),
                             (MimoShape<Alg, F, SHORT>::kMinWaves)) void mimo_ss_kernel(MimoArgs<Alg> a) {
  using E = typename Alg::elem;
  using S = typename Alg::state;
  using SS = typename Alg::s_state;
  using V = SsView<Alg>;
  using Sh = MimoShape<Alg, F, SHORT>;
  using St = SsStatus<Alg>;
  using X = IoVec<E, F>;
  constexpr int K = Sh::K, kWaves = Sh::kWaves, kP = Sh::kPlane, M = V::M;

  __shared__ S s_wagg[kWaves];  // wave aggregates (matrix part A^(64 K))
  __shared__ S s_wpre[kWaves];  // exclusive wave prefixes (matrix part A^(64 K w))
  __shared__ S s_in;
  __shared__ unsigned s_id, s_tag;
  __shared__ uint64_t s_look[St::kLookWords];
  __shared__ SsPowers<Alg> s_tab;
  constexpr bool kMid = sizeof(E) == 4;  // (fp64 steps are in compute precision)
  __shared__ typename Alg::coef s_half;  // A^(K/2)
  extern __shared__ __align__(16) unsigned char mimo_dyn[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the tile is the workgroup's index; the look-back wave claims for the
  // call's tag (claim_tag), so the data waves' loads do not wait for it
  const int64_t id = blockIdx.x;
  if (id >= a.tiles) {  // padding of the last stripe round: counted, then gone
    if (tid == 0) claim_tile(a.claims, a.per_stripe, s_id, s_tag);
    return;
  }
  unsigned tag = 0;
  int64_t q, b;  // tile position along the row, row
  split_tile(id, a.B, a.b_magic, a.b_shift, q, b);
  const int64_t T = a.T_len;

  if (w == kWaves) {
    // ================= look-back wave: power tables, then the look-back
    ss_build_powers<Alg, K, 1, kWaves>(reinterpret_cast<const typename Alg::s_coef *>(a.A + b * a.A_stride), &s_tab,
                                       lane, kMid ? &s_half : nullptr);
    __syncthreads();  // power tables
    tag = claim_tag(a.claims, a.per_stripe, lane);
    uint64_t *row_status = a.status + b * a.tiles_per_row * St::kStride;
    const S virt = a.zi ? Alg::load_s(V::load_vec(a.zi + b * M)) : Alg::szero();
    S yin = virt;
    __syncthreads();  // wave aggregates are in s_wagg
    // exclusive wave prefixes and the tile aggregate (every lane, uniformly)
    S tagg = Alg::szero();
#pragma unroll
    for (int j = 0; j < kWaves; ++j) {
      if (lane == 0) s_wpre[j] = tagg;
      tagg = Alg::affine(s_tab.pw[7], tagg, s_wagg[j]);
    }
    if (q > 0) {
      if (lane == 0) publish(row_status + q * St::kStride + St::kVecWords, tagg, tag);
      if (!ss_lookback<Alg>(row_status, virt, lane, tag, a.spin_limit, s_look, &s_tab, q, yin))
        yin = mimo_prefix_fallback<Alg, F, REV, SHORT>(kernel_args<MimoArgs<Alg>>(), b, q * Sh::kTile, lane, virt, &s_tab);
    }
    if (q + 1 < a.tiles_per_row && lane == 0 && !(a.agg_only && q > 0))
      publish(row_status + q * St::kStride, Alg::affine(s_tab.gp[0], yin, tagg), tag);
    if (lane == 0) s_in = yin;
    __syncthreads();  // entry state is in s_in
    return;
  }

  // ================= data waves
  const size_t plane_bytes = Sh::align16(size_t(a.P) * kP * sizeof(E));
  unsigned char *dyn = mimo_dyn + w * (plane_bytes + (HS ? 64 * 16 * Sh::kHsVecs : 0));
  E *yout = reinterpret_cast<E *>(dyn);
  const int64_t s0 = q * Sh::kTile + int64_t(w) * Sh::kSpan;  // the wave's first scan position
  const int64_t l0 = s0 + int64_t(lane) * K;                  // the lane's
  MimoModel<Alg, F> m;
  mimo_model<Alg, F>(a, b, m);
  X u[K];
  ss_load<REV, X, K>(reinterpret_cast<const X *>(a.x) + b * T, l0, T, u);
  mimo_model_uniform<Alg, F>(m);

  // ---- pass 1: the lane's K steps of B x[t] folded from a zero state, then
  // the wave's vector scan.  Steps past the row's end carry a zero input and
  // only touch the aggregate of its last tile, which nobody reads.
  S mid = Alg::szero();
  S v[1] = {mimo_lane_fold<Alg, F, K>(m, u, kMid ? &mid : nullptr)};
  __syncthreads();  // power tables
  ss_lane_scan<Alg, 1, false>(v, lane, s_tab.pw);
  const S prev = shfl_from(v[0], lane - 1);
  S ent[1] = {lane > 0 ? prev : Alg::szero()};
  if (lane == 63) s_wagg[w] = v[0];
  __syncthreads();  // wave aggregates are in s_wagg
  __syncthreads();  // entry state is in s_in
  // the wave's entry state A^(64 K w) s_in + its exclusive prefix; a lane
  // enters at A^(K lane) of that plus its own exclusive prefix
  {
    S st = s_in;
    for (int j = 0; j < w; ++j) st = Alg::affine(s_tab.pw[6], st, Alg::szero());
    st = Alg::sadd(st, s_wpre[w]);
    S sv[1] = {st};
    ss_pow_apply<Alg, 6, 1>(s_tab.pw, lane, sv);
    ent[0] = Alg::sadd(sv[0], ent[0]);
  }
  union {
    SS s;
    E e[M];
  } h;
  h.s = Alg::store_s(ent[0]);
  SS hmid = h.s;  // the state before step K/2
  if constexpr (kMid) hmid = Alg::store_s(Alg::affine(s_half, ent[0], mid));

  // ---- pass 2: y = C h + D x, then the step
  const bool has_d = a.Dm != nullptr;
  const bool ends = a.zf && s0 < T && T <= s0 + Sh::kSpan;  // the row's last step lies in the span
  const int k_end = ends ? int(T - 1 - s0) - lane * K : -1;
  constexpr int G = HS ? Sh::kHsGroup : K;
  static_assert(K % G == 0, "whole groups");
  SS *hrow = HS ? reinterpret_cast<SS *>(a.hs) + b * T : nullptr;
#pragma unroll
  for (int g0 = 0; g0 < K; g0 += G) {
    SS Hg[HS ? G : 1];
#pragma unroll
    for (int k2 = 0; k2 < G; ++k2) {
      const int k = g0 + k2;
      if (kMid && k == K / 2) h.s = hmid;
      if constexpr (HS) Hg[k2] = h.s;
#pragma unroll
      for (int p = 0; p < kMimoMaxIO; ++p) {
        if (p < a.P) {
          E o = m.c[p][0] * h.e[0];
#pragma unroll
          for (int i = 1; i < M; ++i) o = fma(m.c[p][i], h.e[i], o);
          if (has_d) {
#pragma unroll
            for (int f = 0; f < F; ++f) o = fma(m.d[p][f], u[k].e[f], o);
          }
          yout[p * kP + lane * Sh::kPitch + k] = o;
        }
      }
      E n[M];
      mimo_bu<Alg, F>(m, u[k], n);
#pragma unroll
      for (int i = 0; i < M; ++i)
#pragma unroll
        for (int j = M - 1; j >= 0; --j) n[i] = fma(m.A[i][j], h.e[j], n[i]);
#pragma unroll
      for (int i = 0; i < M; ++i) h.e[i] = n[i];
      if (ends && k == k_end) {
#pragma unroll
        for (int i = 0; i < M; ++i) a.zf[b * M + i] = h.e[i];
      }
    }
    if constexpr (HS) {
      // a lane's group of states is at most 64 bytes: its vectors go out
      // through LDS so that a store instruction covers whole pieces
      constexpr int NV = Sh::kHsVecs;
      uint4 *wb = reinterpret_cast<uint4 *>(dyn + plane_bytes);
      const int64_t span_lo = REV ? T - s0 - Sh::kSpan : s0;
      if constexpr (NV > 1 && (NV & (NV - 1)) == 0) {
        if (span_lo >= 0 && span_lo + Sh::kSpan <= T) {
          ss_lds_put<NV, REV, G>(wb, lane, 0, Hg);
          wave_sync();
#pragma unroll
          for (int j = 0; j < NV; ++j) {
            const int c = j * 64 + lane, L = c / NV, vv = c % NV;
            const int64_t lo = REV ? T - s0 - int64_t(L) * K - g0 - G : s0 + int64_t(L) * K + g0;
            reinterpret_cast<RowVec *>(hrow + lo)[vv] = row_vec(wb[L * NV + (vv ^ lds_swizzle<NV>(L))]);
          }
          wave_sync();
          continue;
        }
      }
      ss_store<REV, SS, G>(hrow, l0 + g0, T, Hg);
    }
  }
  wave_sync();  // the span's outputs are in the planes
  {
    // the span's block of the [T, P] row, four consecutive elements a lane
    const int P = a.P;
    E *yrow = a.y + b * T * P;
    const int64_t base = (REV ? T - s0 - Sh::kSpan : s0) * P;
    int lo, hi;
    mimo_block_range(base, T * P, Sh::kSpan * P, lo, hi);
    constexpr int kV = 16 / int(sizeof(E));
    struct alignas(16) Out {
      E e[kV];
    };
    for (int i = 0; i < K * P / kV; ++i) {
      const int e0 = (i * 64 + lane) * kV;
      Out o;
#pragma unroll
      for (int c = 0; c < kV; ++c) {
        unsigned s, p;
        mimo_split(unsigned(e0 + c), unsigned(P), a.p_magic18, s, p);
        const int ss = REV ? Sh::kSpan - 1 - int(s) : int(s);
        o.e[c] = yout[p * kP + ss + ss / K];
      }
      if (e0 >= lo && e0 + kV <= hi) {
        uint4 t;
        __builtin_memcpy(&t, &o, 16);
        *reinterpret_cast<RowVec *>(yrow + base + e0) = row_vec(t);
      } else {
#pragma unroll
        for (int c = 0; c < kV; ++c)
          if (e0 + c >= lo && e0 + c < hi) yrow[base + e0 + c] = o.e[c];
      }
    }
  }
}

// ---------------------------------------------------------------- time-varying A
// The LPV (parameter-varying) model with several inputs and outputs
// (philtorch/lpv/ssm.py:337-581 with a 3D x or matrix-valued B, C, D that
// are constant in time):
//     h[0] = zi,  y[t] = C h[t] + D x[t],  h[t+1] = A[t] h[t] + B x[t],  zf = h[T]
// A is [rows, T, M, M]; B, C, D and the staging of x and y are the LTI
// kernel's.  Every step has its own matrix, so the scan is the generic
// time-varying one (phs_scan.hpp), as in lpv_ss_kernel: a lane folds its K
// steps (A[t], B x[t]) into a map, wave scans of maps chain the lanes, and
// the look-back resolves map status words.  K is 32 bytes of state-order-2
// coefficients' worth (fp32 8, fp64 4 steps; orders 3-4 half that: a lane
// holds its K matrices).
template <class Alg>
struct LpvMimoShape {
  using E = typename Alg::elem;
  static constexpr int kM = SsView<Alg>::M;
  static constexpr int kWaves = 3;
  static constexpr int kThreads = 64 * (kWaves + 1);
  static constexpr int K = (kM <= 2 ? 32 : 16) / int(sizeof(E));
  static constexpr int kSpan = 64 * K;
  static constexpr int kTile = kWaves * kSpan;
  static constexpr int kPlane = kSpan + 16 / int(sizeof(E));
  static constexpr int kWaveElems = kMimoMaxIO * kPlane;
  // waves per SIMD of the launch bounds: orders 1-2 fit 168 VGPRs (3 waves,
  // three workgroups per CU), orders 3-4 take 256 (2)
  static constexpr int kMinWaves = kM <= 2 ? 3 : 2;
};

// A lane's K matrices A[t] in scan order from scan position s0 (past the
// row: zero), transposed where the adjoint reads them so.
template <class Alg, bool REV, int K>
__device__ __forceinline__ void lpv_mimo_load_A(const MimoArgs<Alg> &a, int64_t b, int64_t s0,
                                                typename Alg::s_coef (&Ak)[K]) {
  using SC = typename Alg::s_coef;
  const SC *row = reinterpret_cast<const SC *>(a.A + b * a.A_stride);
  lpv_load<REV, SC, K>(row, s0, a.T_len, Ak, Alg::s_czero());
  if (a.A_trans) {
#pragma unroll
    for (int k = 0; k < K; ++k) Ak[k] = Alg::s_adjoint(Ak[k]);  // real: the transpose
  }
}

// State entering tile position `span` of a row, folded from the inputs (the
// look-back's bounded-wait fallback; out of line, cold).
template <class Alg, bool REV>
__device__ __noinline__ typename Alg::state lpv_mimo_prefix_fallback(const MimoArgs<Alg> *ap, int64_t b,
                                                                    int64_t span, int lane,
                                                                    typename Alg::state virt) {
  const MimoArgs<Alg> &a = *ap;
  using E = typename Alg::elem;
  using SC = typename Alg::s_coef;
  using SS = typename Alg::s_state;
  using M = Map<Alg>;
  constexpr int K = LpvMimoShape<Alg>::K;
  auto op = [](const M &p, const M &q) { return compose<Alg>(p, q); };
  const MimoIn<Alg> mdl = mimo_in<Alg>(a, b);  // (its A is not read)
  const E *xrow = a.x + b * a.T_len * a.F;
  const SC dummy = Alg::s_czero();
  M acc = map_identity<Alg>();
  for (int64_t off = 0; off < span; off += 64 * K) {
    const int64_t c0 = off + int64_t(lane) * K;
    SC Ak[K];
    lpv_mimo_load_A<Alg, REV, K>(a, b, c0, Ak);
    SS xs[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t s = c0 + k;
      E u[kMimoMaxIO];
#pragma unroll
      for (int f = 0; f < kMimoMaxIO; ++f) {
        u[f] = E(0);
        if (f < a.F && s < a.T_len) u[f] = xrow[mimo_time<REV>(s, a.T_len) * a.F + f];
      }
      xs[k] = mimo_bx<Alg>(mdl, u);
    }
    M m = lane_map<Alg, true, false, K>(Ak, xs, dummy);
    m = wave_scan_incl(m, lane, op);
    acc = compose<Alg>(acc, read_lane(m, 63));
  }
  return apply<Alg>(acc, virt);
}

// HS: also the state before every step into a.hs (a separate instance, so
// the plain forward carries none of it).
template <class Alg, bool REV, bool HS = false>
__global__ __launch_bounds__(LpvMimoShape<Alg>::kThreads, LpvMimoShape<Alg>::kMinWaves) void lpv_mimo_kernel(
    MimoArgs<Alg> a) {
  using E = typename Alg::elem;
  using S = typename Alg::state;
  using SC = typename Alg::s_coef;
  using SS = typename Alg::s_state;
  using M = Map<Alg>;
  using V = SsView<Alg>;
  using Sh = LpvMimoShape<Alg>;
  using St = StatusShape<Alg>;
  constexpr int K = Sh::K, kWaves = Sh::kWaves, kP = Sh::kPlane;

  __shared__ M s_wagg[kWaves];
  __shared__ M s_wpre[kWaves];
  __shared__ S s_in;
  __shared__ unsigned s_id, s_tag;
  __shared__ uint64_t s_look[St::kLookWords];
  __shared__ E s_io[kWaves * Sh::kWaveElems];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t id = blockIdx.x;
  if (id >= a.tiles) {  // padding of the last stripe round: counted, then gone
    if (tid == 0) claim_tile(a.claims, a.per_stripe, s_id, s_tag);
    return;
  }
  unsigned tag = 0;
  int64_t q, b;  // tile position along the row, row
  split_tile(id, a.B, a.b_magic, a.b_shift, q, b);
  const int64_t T = a.T_len;
  auto op = [](const M &p, const M &q2) { return compose<Alg>(p, q2); };

  if (w == kWaves) {
    // ================= look-back wave
    tag = claim_tag(a.claims, a.per_stripe, lane);
    uint64_t *row_status = a.status + b * a.tiles_per_row * St::kStride;
    const S virt = a.zi ? Alg::load_s(V::load_vec(a.zi + b * V::M)) : Alg::szero();
    __syncthreads();  // wave aggregates are in s_wagg
    M v = lane < kWaves ? s_wagg[lane] : map_identity<Alg>();
    v = wave_scan_incl(v, lane, op);
    const M wex = wave_shift_up(v, lane, map_identity<Alg>());
    if (lane < kWaves) s_wpre[lane] = wex;
    const M tagg = read_lane(v, kWaves - 1);
    S yin = virt;
    if (q > 0) {
      if (lane == 0) publish(row_status + q * St::kStride + St::kIncWords, tagg, tag);
      Lookback<Alg> lb = lookback_start<Alg>(q);
      if (!lookback<Alg>(row_status, virt, lane, tag, a.spin_limit, s_look, lb, yin))
        yin = lpv_mimo_prefix_fallback<Alg, REV>(kernel_args<MimoArgs<Alg>>(), b, q * Sh::kTile, lane, virt);
    }
    if (q + 1 < a.tiles_per_row && lane == 0 && !(a.agg_only && q > 0))
      publish(row_status + q * St::kStride, apply<Alg>(tagg, yin), tag);
    if (lane == 0) s_in = yin;
    __syncthreads();  // entry state is in s_in
    return;
  }

  // ================= data waves
  E *io = s_io + w * Sh::kWaveElems;  // F input planes, then P output planes
  const int64_t s0 = q * Sh::kTile + int64_t(w) * Sh::kSpan;  // the wave's first scan position
  mimo_stage_in<Alg, REV, Sh>(a.x + b * T * a.F, s0, T, a.F, a.f_magic, io, lane);
  SC Ak[K];
  lpv_mimo_load_A<Alg, REV, K>(a, b, s0 + int64_t(lane) * K, Ak);
  const MimoIn<Alg> mi = mimo_in<Alg>(a, b);  // (its A is not read)
  wave_sync();  // the span's inputs are in the planes

  auto inputs = [&](int k, E (&u)[kMimoMaxIO]) {
#pragma unroll
    for (int f = 0; f < kMimoMaxIO; ++f) u[f] = f < a.F ? io[f * kP + lane * K + k] : E(0);
  };

  // ---- pass 1: the lane map of (A[t], B x[t]) over its K steps, the wave
  // scan.  Steps past the row's end carry a zero matrix and input and only
  // touch the aggregate of its last tile, which nobody reads.
  SS X[K];  // B x[t], kept for pass 2
#pragma unroll
  for (int k = 0; k < K; ++k) {
    E u[kMimoMaxIO];
    inputs(k, u);
    X[k] = mimo_bx<Alg>(mi, u);
  }
  const SC dummy = Alg::s_czero();
  M m = lane_map<Alg, true, false, K>(Ak, X, dummy);
  m = wave_scan_incl(m, lane, op);
  const M ex = wave_shift_up(m, lane, map_identity<Alg>());
  if (lane == 63) s_wagg[w] = m;
  __syncthreads();  // wave aggregates are in s_wagg
  __syncthreads();  // entry state is in s_in
  SS h = Alg::store_s(apply<Alg>(ex, apply<Alg>(s_wpre[w], s_in)));

  // ---- pass 2: y = C h + D x, then the step
  const MimoOut<Alg> mo = mimo_out<Alg>(a, b);
  const int64_t l0 = s0 + int64_t(lane) * K;
  const bool has_d = a.Dm != nullptr;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    E u[kMimoMaxIO];
    if (has_d) inputs(k, u);
#pragma unroll
    for (int p = 0; p < kMimoMaxIO; ++p) {
      if (p < a.P) {
        E o = V::dot(mo.c[p], h);
        if (has_d) {
#pragma unroll
          for (int f = 0; f < kMimoMaxIO; ++f) o = fma(mo.d[p][f], u[f], o);
        }
        io[p * kP + lane * K + k] = o;
      }
    }
    if constexpr (HS) {  // the state before the step into planes P.., the lane's own (already read) slots
      union {
        SS s;
        E e[V::M];
      } hu;
      hu.s = h;
#pragma unroll
      for (int i = 0; i < V::M; ++i) io[(a.P + i) * kP + lane * K + k] = hu.e[i];
    }
    h = Alg::s_affine(Ak[k], h, X[k]);
    if (a.zf && l0 + k == T - 1) {
      union {
        SS s;
        E e[V::M];
      } zu;
      zu.s = h;
#pragma unroll
      for (int i = 0; i < V::M; ++i) a.zf[b * V::M + i] = zu.e[i];
    }
  }
  wave_sync();  // the span's outputs are in the planes
  mimo_stage_out<Alg, REV, Sh>(a.y + b * T * a.P, s0, T, a.P, a.p_magic, io, lane);
  if constexpr (HS) mimo_stage_out<Alg, REV, Sh>(a.hs + b * T * V::M, s0, T, V::M, a.m_magic, io + a.P * kP, lane);
}

}  // namespace phs
