// Batched F3R: many independent systems (and right-hand sides) solved in
// lockstep, every launch covering all of them.
//
// Each segment (one system with one right-hand side) occupies a contiguous
// row range of one block-diagonal matrix, padded to a whole number of
// 2048-row tiles, so a workgroup never straddles two segments.  The SpMVs are
// the single solver's SELL kernels on the concatenated matrices (fp64, fp32,
// fp16 values; the SDAINV factors likewise).  Every reduction is per
// segment: each block writes its partial sums, and one block per segment
// adds its blocks' partials in a fixed order and does that segment's
// Hessenberg / Givens / Richardson-weight work.  Each outer step of all
// segments is replayed from one HIP graph, after which the host reads one
// array of residual norms for all segments.  A segment that has
// converged stops counting steps and keeps its solution; its vectors may run
// on with the others, and the breakdown guards below (a zero norm, a zero
// rotation, a zero pivot) keep them finite.
//
// The nest is the HALF build's: fp64 FGMRES(m1) with restarts > fp32
// FGMRES(m2) on fp32 values > fp32-basis FGMRES(m3) on fp16 values >
// adaptive Richardson(m4, c) in fp16 with SDAINV (work/src/f3r-gpu.cpp:
// 210-266), each segment with its own probes' weights.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <limits>
#include <map>
#include <numeric>

#include "common.hpp"
#include "device.hpp"
#include "internal.hpp"
#include "quad.hpp"
#include "sell_kernel.hpp"

namespace f3r {
namespace {

// ---------------------------------------------------- device helpers ---
template <class T> __device__ void givens_guarded(T *H, T *cs, T *sn, T *e, int j, bool e0_one) {
  for (int i = 0; i < j; ++i) {
    T t = H[i], h1 = H[i + 1];
    H[i] = fma_<T>(cs[i], t, sn[i] * h1);
    H[i + 1] = fma_<T>(-sn[i], t, cs[i] * h1);
  }
  T t = (T)sqrt(fma_<T>(H[j], H[j], H[j + 1] * H[j + 1]));
  if (t > (T)0) {
    cs[j] = H[j] / t;
    sn[j] = H[j + 1] / t;
  } else {  // a zero column (a segment that has run dry): identity rotation
    cs[j] = 1;
    sn[j] = 0;
  }
  H[j] = t;
  H[j + 1] = 0;
  T ej = (j == 0 && e0_one) ? (T)1 : e[j];
  e[j + 1] = -sn[j] * ej;
  e[j] = cs[j] * ej;
}

template <class T> __device__ void hess_solve_guarded(const T *H, int ldh, const T *e, T *y, int j) {
  for (int i = j - 1; i >= 0; --i) {
    T t = e[i];
    for (int q = j - 1; q > i; --q) t = fma_<T>(-H[q * ldh + i], y[q], t);
    const T d = H[i * ldh + i];
    y[i] = d != (T)0 ? t / d : (T)0;
  }
}

// Per-segment Richardson state (work/src/f3r-gpu.cpp:224-260)
struct RichSeg {
  double sum[16];
  double ome[16];
  double alpha[16];
  int nprobe;
};

__global__ void k_b_rich_reset(int nseg, RichSeg *st) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  for (int k = 0; k < 16; ++k) {
    st[s].sum[k] = 1.0;
    st[s].ome[k] = 1.0;
    st[s].alpha[k] = 0.0;
  }
  st[s].nprobe = 0;
}

// ----------------------------------------------------------- kernels ---
// Block b covers the tile of rows [b * kTile, (b + 1) * kTile), all in
// segment bseg[b]; thread t takes rows b * kTile + t + q * kBlock, q < kRows
// (coalesced).  Segments are padded to whole tiles, so the grid is exactly
// the row count / kTile.
constexpr int kRows = 8;
constexpr int64_t kTile = (int64_t)kBlock * kRows;

__device__ __forceinline__ int64_t tile_row(int q) { return (int64_t)blockIdx.x * kTile + threadIdx.x + (int64_t)q * kBlock; }
// the same tile as kRows / 4 groups of 4 consecutive rows per thread (one
// 8- or 16-byte access per vector and group; segments and vectors start on
// tile boundaries, so every group is aligned)
constexpr int kQuads = kRows / 4;
__device__ __forceinline__ int64_t tile_quad(int q, int b) {
  return (int64_t)b * kTile + ((int64_t)threadIdx.x + (int64_t)q * kBlock) * 4;
}
__device__ __forceinline__ int64_t tile_quad(int q) { return tile_quad(q, (int)blockIdx.x); }

// block partial sums of <w, V_k> for the NV columns of blockIdx.y (k < ncols):
// partial[k * gridDim.x + block]
// Basis columns: column 0 at V0, column k >= 1 at V + k * ld, its values
// scaled by csc[k * nsegs + seg] when csc is given (a column left
// unnormalised in memory; the fp32 product is what a normalised copy holds)
template <class S> __device__ __forceinline__ const S *bcol(const S *V0, const S *V, int64_t ld, int k) {
  return k == 0 ? V0 : V + (int64_t)k * ld;
}
template <class A> __device__ __forceinline__ A bscale(const A *csc, int nsegs, int k, int seg) {
  return csc && k > 0 ? csc[(int64_t)k * nsegs + seg] : (A)1;
}

template <class S, class A, int NV>
__global__ __launch_bounds__(kBlock) void k_b_mdot(const S *__restrict__ w, const S *__restrict__ V0,
                                                   const S *__restrict__ V, int64_t ld, int ncols,
                                                   const A *__restrict__ csc, int nsegs,
                                                   const int32_t *__restrict__ bseg, A *__restrict__ partial) {
  __shared__ A lds[NV * kWavesPerBlock];
  const int k0 = blockIdx.y * NV;
  const int seg = bseg[blockIdx.x];
  A sk[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) sk[k] = k0 + k < ncols ? bscale(csc, nsegs, k0 + k, seg) : (A)1;
  A v[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = (A)0;
  for (int q = 0; q < kQuads; ++q) {
    const int64_t i = tile_quad(q);
    const V4<S> wq = ld4(w + i);
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (k0 + k < ncols) {
        const V4<S> vq = ld4(bcol(V0, V, ld, k0 + k) + i);
#pragma unroll
        for (int c = 0; c < 4; ++c) v[k] = fma_<A>((A)to_acc(wq.v[c]), (A)to_acc(vq.v[c]) * sk[k], v[k]);
      }
  }
  block_sum<A, NV>(v, lds);
  if (threadIdx.x == 0)
    for (int k = 0; k < NV && k0 + k < ncols; ++k) partial[(int64_t)(k0 + k) * gridDim.x + blockIdx.x] = v[k];
}

// H[seg * hs + k] = the partials of segment seg's blocks, added in block
// order; grid (segments, columns)
template <class A>
__global__ __launch_bounds__(kBlock) void k_b_dots_finish(const A *__restrict__ partial, int G,
                                                          const int32_t *__restrict__ sb0,
                                                          const int32_t *__restrict__ snb, A *H, int64_t hs) {
  __shared__ A lds[kWavesPerBlock];
  const int seg = blockIdx.x, k = blockIdx.y;
  const int32_t b0 = sb0[seg], nb = snb[seg];
  A v[1] = {(A)0};
  for (int32_t b = threadIdx.x; b < nb; b += kBlock) v[0] += partial[(int64_t)k * G + b0 + b];
  block_sum<A, 1>(v, lds);
  if (threadIdx.x == 0) H[(int64_t)seg * hs + k] = v[0];
}

// w = S(w - V h) with h of the block's segment (MULMV order); block partial
// of ||w||^2 of the stored w.  With dpart (the segments' block partials of the
// dots) each block adds its segment's up itself, and a segment's first block
// stores them in H: a launch less (4.6 us at 5.93 M rows) for nb x ncols loads
// that run beside the first rows'.
template <class S, class A>
__global__ __launch_bounds__(kBlock) void k_b_update(S *__restrict__ w, const S *__restrict__ V0,
                                                     const S *__restrict__ V, int64_t ld, int ncols,
                                                     const A *__restrict__ csc, int nsegs, A *H, int64_t hs,
                                                     const int32_t *__restrict__ bseg, A *__restrict__ partial,
                                                     const A *__restrict__ dpart, const int32_t *__restrict__ sb0,
                                                     const int32_t *__restrict__ snb) {
  __shared__ A h[128], sk[128];
  __shared__ A lds[kWavesPerBlock];
  const int seg = bseg[blockIdx.x];
  if (dpart) {
    const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int32_t b0 = sb0[seg], nb = snb[seg];
    for (int k = wave; k < ncols; k += kWavesPerBlock) {
      A a = (A)0;
      for (int32_t b = lane; b < nb; b += kWave) a += dpart[(int64_t)k * gridDim.x + b0 + b];
      a = wave_sum(a);
      if (lane == 0) {
        h[k] = a;
        if ((int)blockIdx.x == b0) H[(int64_t)seg * hs + k] = a;
      }
    }
  }
  for (int k = threadIdx.x; k < ncols; k += kBlock) {
    if (!dpart) h[k] = H[(int64_t)seg * hs + k];
    sk[k] = bscale(csc, nsegs, k, seg);
  }
  __syncthreads();
  A v[1] = {(A)0};
  for (int q = 0; q < kQuads; ++q) {
    const int64_t i = tile_quad(q);
    const V4<S> v0 = ld4(V0 + i);
    V4<S> wq = ld4(w + i);
    A r[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) r[c] = ((A)to_acc(v0.v[c]) * sk[0]) * h[0];
    for (int k = 1; k < ncols; ++k) {
      const V4<S> vk = ld4(V + (int64_t)k * ld + i);
#pragma unroll
      for (int c = 0; c < 4; ++c) r[c] = fma_<A>((A)to_acc(vk.v[c]) * sk[k], h[k], r[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      wq.v[c] = cvt<S>((A)to_acc(wq.v[c]) - r[c]);
      const A wf = (A)to_acc(wq.v[c]);
      v[0] = fma_<A>(wf, wf, v[0]);
    }
    st4(w + i, wq);
  }
  block_sum<A, 1>(v, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = v[0];
}

// block partial of ||v||^2 (the outer level's residual norm)
template <class A>
__global__ __launch_bounds__(kBlock) void k_b_norm2(const A *__restrict__ v, A *__restrict__ partial) {
  __shared__ A lds[kWavesPerBlock];
  A s[1] = {(A)0};
  for (int q = 0; q < kRows; ++q) {
    const A x = v[tile_row(q)];
    s[0] = fma_<A>(x, x, s[0]);
  }
  block_sum<A, 1>(s, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// Right-hand sides and initial guesses into the tiles of all segments (zero
// in the padding), and the block sums of ||b||^2.  bp[seg], xp[seg]: the
// callers' vectors; rows[seg] of them.  One launch; a copy per vector and a
// dot per segment, each waited for, took 3 ms of 16 for 64 segments.
__global__ __launch_bounds__(kBlock) void k_b_take(const double *const *bp, const double *const *xp,
                                                   const int32_t *__restrict__ rows, const int32_t *__restrict__ bseg,
                                                   const int32_t *__restrict__ sb0, double *__restrict__ b,
                                                   double *__restrict__ x, double *__restrict__ partial) {
  __shared__ double lds[kWavesPerBlock];
  const int seg = bseg[blockIdx.x];
  const int64_t r0 = (int64_t)sb0[seg] * kTile;
  const int32_t n = rows[seg];
  const double *bs = bp[seg], *xs = xp[seg];
  double s[1] = {0.0};
  double bv[kRows], xv[kRows];
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int64_t k = tile_row(q) - r0;
    bv[q] = k < n ? bs[k] : 0.0;
    xv[q] = k < n ? xs[k] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int64_t i = tile_row(q);
    b[i] = bv[q];
    x[i] = xv[q];
    s[0] = fma_<double>(bv[q], bv[q], s[0]);
  }
  block_sum<double, 1>(s, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}
// the solutions back into the callers' vectors
__global__ __launch_bounds__(kBlock) void k_b_give(const double *__restrict__ x, double *const *xp,
                                                   const int32_t *__restrict__ rows, const int32_t *__restrict__ bseg,
                                                   const int32_t *__restrict__ sb0) {
  const int seg = bseg[blockIdx.x];
  const int64_t r0 = (int64_t)sb0[seg] * kTile;
  const int32_t n = rows[seg];
  double *xs = xp[seg];
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int64_t i = tile_row(q), k = i - r0;
    if (k < n) xs[k] = x[i];
  }
}

// One block per segment: ||w|| from its blocks' partials, then H(j+1, j),
// 1/||w|| (0 for a zero vector), the guarded Givens step and |e_{j+1}|.
// H, e, cs, sn point at segment 0's column j / arrays; strides per segment.
template <class A>
__global__ __launch_bounds__(kBlock) void k_b_norm_finish(const A *__restrict__ partial, const int32_t *__restrict__ sb0,
                                                          const int32_t *__restrict__ snb, A *H, int64_t hs, A *cs,
                                                          A *sn, int64_t ms, A *e, int64_t es, int j, int e0_one,
                                                          A *inv, double *status) {
  __shared__ A lds[kWavesPerBlock];
  const int seg = blockIdx.x;
  const int32_t b0 = sb0[seg], nb = snb[seg];
  A v[1] = {(A)0};
  for (int32_t b = threadIdx.x; b < nb; b += kBlock) v[0] += partial[b0 + b];
  block_sum<A, 1>(v, lds);
  if (threadIdx.x == 0) {
    A *Hc = H + (int64_t)seg * hs;
    const A nv = (A)sqrt(v[0]);
    Hc[j + 1] = nv;
    inv[seg] = nv > (A)0 ? (A)1 / nv : (A)0;
    if (cs) {
      A *ee = e + (int64_t)seg * es;
      givens_guarded<A>(Hc, cs + (int64_t)seg * ms, sn + (int64_t)seg * ms, ee, j, e0_one != 0);
      if (status) status[seg] = fabs((double)ee[j + 1]);
    } else if (status) {
      status[seg] = (double)nv;  // the residual norm itself (start of a cycle)
    }
  }
}

// v *= inv[segment of the tile]
template <class S, class A>
__global__ __launch_bounds__(kBlock) void k_b_vscale(S *__restrict__ v, const A *__restrict__ inv,
                                                     const int32_t *__restrict__ bseg) {
  const A a = inv[bseg[blockIdx.x]];
  for (int q = 0; q < kQuads; ++q) {
    const int64_t i = tile_quad(q);
    V4<S> x = ld4(v + i);
#pragma unroll
    for (int c = 0; c < 4; ++c) x.v[c] = cvt<S>((A)to_acc(x.v[c]) * a);
    st4(v + i, x);
  }
}

// out = TO(Z y) (accumulate: out += Z y) with y solved from the block's
// segment's j x j triangle; j = jseg[segment] or jall (jseg null)
template <class S, class A, class TO>
__global__ __launch_bounds__(kBlock) void k_b_combine(const S *__restrict__ Z, int64_t ld, const A *H, int64_t hs,
                                                      int ldh, const A *e, int64_t es, const int32_t *jseg, int jall,
                                                      const int32_t *__restrict__ bseg, TO *__restrict__ out,
                                                      int accumulate, const float *__restrict__ zsc) {
  __shared__ A y[128];
  const int seg = bseg[blockIdx.x];
  const int j = jseg ? jseg[seg] : jall;
  if (j == 0) {
    if (!accumulate)
      for (int q = 0; q < kRows; ++q) out[tile_row(q)] = cvt<TO>((A)0);
    return;
  }
  if (threadIdx.x == 0) hess_solve_guarded<A>(H + (int64_t)seg * hs, ldh, e + (int64_t)seg * es, y, j);
  __syncthreads();
  // zsc: Z holds z * s (fp16 storage, s a power of two): z = Z * zsc exactly
  const A zs = zsc ? (A)zsc[seg] : (A)1;
  for (int q = 0; q < kQuads; ++q) {
    const int64_t i = tile_quad(q);
    const V4<S> z0 = ld4(Z + i);
    A r[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) r[c] = ((A)to_acc(z0.v[c]) * zs) * y[0];
    for (int k = 1; k < j; ++k) {
      const V4<S> zk = ld4(Z + (int64_t)k * ld + i);
#pragma unroll
      for (int c = 0; c < 4; ++c) r[c] = fma_<A>((A)to_acc(zk.v[c]) * zs, y[k], r[c]);
    }
    V4<TO> o;
    if (accumulate) {
      o = ld4(out + i);
#pragma unroll
      for (int c = 0; c < 4; ++c) o.v[c] = cvt<TO>((A)to_acc(o.v[c]) + r[c]);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) o.v[c] = cvt<TO>(r[c]);
    }
    st4(out + i, o);
  }
}

template <class SI, class SO>
__global__ __launch_bounds__(kBlock) void k_b_cast(const SI *__restrict__ in, SO *__restrict__ out) {
  for (int q = 0; q < kRows; ++q) {
    const int64_t i = tile_row(q);
    out[i] = cvt<SO>(to_acc(in[i]));
  }
}

// out = SO(in * f[segment]) (conversions into and out of the fp16 level)
template <class SI, class SO>
__global__ __launch_bounds__(kBlock) void k_b_entry(const SI *__restrict__ in, SO *__restrict__ out,
                                                    const float *__restrict__ f, const int32_t *__restrict__ bseg) {
  const float a = f[bseg[blockIdx.x]];
  for (int q = 0; q < kRows; ++q) {
    const int64_t i = tile_row(q);
    out[i] = cvt<SO>(to_acc(in[i]) * a);
  }
}

// block partials of <t, t> and <t, r> (Richardson probe): partial[q * G + b]
__global__ __launch_bounds__(kBlock) void k_b_probe_dots(const half_t *__restrict__ t, const half_t *__restrict__ r,
                                                         float *__restrict__ partial) {
  __shared__ float lds[2 * kWavesPerBlock];
  float v[2] = {0.f, 0.f};
  for (int q = 0; q < kRows; ++q) {
    const int64_t i = tile_row(q);
    const float ti = to_acc(t[i]);
    v[0] = fma_<float>(ti, ti, v[0]);
    v[1] = fma_<float>(ti, to_acc(r[i]), v[1]);
  }
  block_sum<float, 2>(v, lds);
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = v[0];
    partial[(int64_t)gridDim.x + blockIdx.x] = v[1];
  }
}

// one block per segment: alpha_k = <t, r> / <t, t>, then the running mean of
// the weights (probe count den = probes + 1: the initial weight 1 counts)
__global__ __launch_bounds__(kBlock) void k_b_probe_finish(const float *__restrict__ partial, int G,
                                                           const int32_t *__restrict__ sb0,
                                                           const int32_t *__restrict__ snb, RichSeg *st, int k) {
  __shared__ float lds[2 * kWavesPerBlock];
  const int seg = blockIdx.x;
  const int32_t b0 = sb0[seg], nb = snb[seg];
  float v[2] = {0.f, 0.f};
  for (int32_t b = threadIdx.x; b < nb; b += kBlock) {
    v[0] += partial[b0 + b];
    v[1] += partial[(int64_t)G + b0 + b];
  }
  block_sum<float, 2>(v, lds);
  if (threadIdx.x == 0) {
    RichSeg &s = st[seg];
    const float al = v[0] > 0.f ? v[1] / v[0] : 0.f;
    if (k == 0) s.nprobe += 1;
    const float den = (float)(s.nprobe + 1);
    const float sm = (float)s.sum[k] + al;
    s.sum[k] = sm;
    s.ome[k] = sm / den;
    s.alpha[k] = al;
  }
}

// ho = fp16(ho * w) (step 0) or ho2 = fp16(w * t2 + ho) (step k), w the
// segment's weight (alpha on a probe call, else the running mean)
__global__ __launch_bounds__(kBlock) void k_b_l4_scale(half_t *__restrict__ ho, const RichSeg *__restrict__ st,
                                                       int probe, const int32_t *__restrict__ bseg) {
  const RichSeg &s = st[bseg[blockIdx.x]];
  const float w = (float)(probe ? s.alpha[0] : s.ome[0]);
  for (int q = 0; q < kRows; ++q) {
    const int64_t i = tile_row(q);
    ho[i] = cvt<half_t>(to_acc(ho[i]) * w);
  }
}
__global__ __launch_bounds__(kBlock) void k_b_l4_update(const half_t *__restrict__ t2, const half_t *__restrict__ ho,
                                                        half_t *__restrict__ ho2, const RichSeg *__restrict__ st, int k,
                                                        int probe, const int32_t *__restrict__ bseg) {
  const RichSeg &s = st[bseg[blockIdx.x]];
  const float w = (float)(probe ? s.alpha[k] : s.ome[k]);
  for (int q = 0; q < kRows; ++q) {
    const int64_t i = tile_row(q);
    ho2[i] = cvt<half_t>(fma_<float>(w, to_acc(t2[i]), to_acc(ho[i])));
  }
}

// SpMV of a block-diagonal matrix stored once per system, applied to the NR
// copies (right-hand sides) of each system's vectors: copy c of the rows of
// chunk s lies at vector row = matrix row + shift[s] + c * stride[s].  One
// lane takes a matrix row and keeps NR sums, so each value and column index
// is read once for all copies; every sum runs in slot order, as in k_sell.
// Epilogue: y = acc (b null) or y = b - acc, at the vector rows.
// Offset chunks gather x through a buffer resource over x's nx elements: the
// per-lane byte offset is the row's, the chunk offset and the copy's stride
// ride in the scalar offset (no per-lane address arithmetic per gather).
template <class V, class X, class ACC, int K, int NR, class Y>
__device__ __forceinline__ void sell_mr_row(const SellArgs &a, int r, const V *__restrict__ val,
                                            const X *__restrict__ x, int64_t nx, const int32_t *__restrict__ cshift,
                                            const int32_t *__restrict__ cstride, Y *__restrict__ y,
                                            const Y *__restrict__ b, const int32_t *__restrict__ cseg,
                                            const float *__restrict__ ysc) {
  typedef const __attribute__((address_space(4))) int32_t *const_i32;
  const int s = r >> a.log2C;
  const int j = r - (s << a.log2C);
  const int C = 1 << a.log2C;
  const int rem = a.n - (s << a.log2C);
  const int tc = rem < C ? rem : C;
  const int su = __builtin_amdgcn_readfirstlane(s);  // C >= 64: one chunk per wavefront
  const int cw = a.cwidth[su];
  const int groups = chunk_groups(cw);
  const int32_t shift = cshift[su], stride = cstride[su];
  int64_t pos = (int64_t)a.cptr[su] + (int64_t)j * K;
  const int64_t step = (int64_t)tc * K;
  ACC acc[NR];
#pragma unroll
  for (int c = 0; c < NR; ++c) acc[c] = 0;
  const int64_t vr = (int64_t)r + shift;
  const int32_t start = a.iptr ? a.iptr[su] : 0;
  if (a.iptr && start < 0) {
    const const_i32 off = (const_i32)(a.coff + (-start - 1));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)((uintptr_t)x - (uintptr_t)a.off_bias * sizeof(X)), (short)0,
        (int)((nx + a.off_bias) * (int64_t)sizeof(X)), kBufferWord3);
    const int vo = (int)(vr * (int64_t)sizeof(X));
    const int bias = a.off_bias, cst = stride * (int)sizeof(X);
#pragma unroll 2
    for (int g = 0; g < groups; ++g, pos += step) {
      const Pack<V, K> pv = load_pack<V, K>(val + pos);
      X xv[K][NR];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int so = (off[g * K + k] + bias) * (int)sizeof(X);
#pragma unroll
        for (int c = 0; c < NR; ++c) xv[k][c] = buffer_gather<X>(rs, vo, so + c * cst);
      }
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int c = 0; c < NR; ++c) acc[c] = fma_<ACC>((ACC)to_acc(pv.v[k]), (ACC)to_acc(xv[k][c]), acc[c]);
    }
    if constexpr (K >= 2) {
      if (cw & kHalfTail) {  // the half group (K / 2 slots per row, rows consecutive)
        constexpr int H = K / 2;
        const Pack<V, H> pv = load_pack<V, H>(val + ((int64_t)a.cptr[su] + (int64_t)groups * step + (int64_t)j * H));
        X xv[H][NR];
#pragma unroll
        for (int k = 0; k < H; ++k) {
          const int so = (off[groups * K + k] + bias) * (int)sizeof(X);
#pragma unroll
          for (int c = 0; c < NR; ++c) xv[k][c] = buffer_gather<X>(rs, vo, so + c * cst);
        }
#pragma unroll
        for (int k = 0; k < H; ++k)
#pragma unroll
          for (int c = 0; c < NR; ++c) acc[c] = fma_<ACC>((ACC)to_acc(pv.v[k]), (ACC)to_acc(xv[k][c]), acc[c]);
      }
    }
  } else {
    const int32_t *__restrict__ ip = a.idx + (a.iptr ? (int64_t)start : (int64_t)a.cptr[su]) + (int64_t)j * K;
    for (int g = 0; g < groups; ++g, pos += step, ip += step) {
      const Pack<V, K> pv = load_pack<V, K>(val + pos);
      const Pack<int32_t, K> pi = load_pack<int32_t, K>(ip);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int64_t col = (int64_t)pi.v[k] + shift;
#pragma unroll
        for (int c = 0; c < NR; ++c)
          acc[c] = fma_<ACC>((ACC)to_acc(pv.v[k]), (ACC)to_acc(x[col + (int64_t)c * stride]), acc[c]);
      }
    }
  }
  // ysc: x held z * s (fp16 storage, s a power of two per segment), so
  // y = sum * (1/s) is the sum over z exactly
#pragma unroll
  for (int c = 0; c < NR; ++c) {
    const int64_t o = vr + (int64_t)c * stride;
    const ACC sum = ysc ? acc[c] * (ACC)ysc[cseg[su] + c] : acc[c];
    y[o] = b ? cvt<Y>((ACC)to_acc(b[o]) - sum) : cvt<Y>(sum);
  }
}

template <class V, class X, class ACC, int K, int NR, class Y>
__global__ __launch_bounds__(kBlock) void k_sell_mr(SellArgs a, const V *__restrict__ val, const X *__restrict__ x,
                                                    int64_t nx, const int32_t *__restrict__ cshift,
                                                    const int32_t *__restrict__ cstride, Y *__restrict__ y,
                                                    const Y *__restrict__ b, const int32_t *__restrict__ cseg,
                                                    const float *__restrict__ ysc) {
  for (int r = xcd_block() * kBlock + threadIdx.x; r < a.n; r += gridDim.x * kBlock)
    sell_mr_row<V, X, ACC, K, NR, Y>(a, r, val, x, nx, cshift, cstride, y, b, cseg, ysc);
}

// The same product by value codes (quad.hpp), where every system has few
// distinct values: a lane takes four matrix rows of NR copies, so codes are
// decoded once for all copies and x is read in windows.  The gathers and their
// latency, not the bytes, were the plain product's cost (0.32 of the memory
// rate for 4 copies; 5.93 M rows in fp16: now 17 us, and with the other steps'
// products a solve 14.1 -> 11.1 ms).
template <class V, class X, class ACC, int K, int NR, class Y>
__global__ __launch_bounds__(kBlock) void k_quad_mr(SellArgs a, QuadArgs qa, const V *__restrict__ val,
                                                    const X *__restrict__ x, int64_t nx,
                                                    const int32_t *__restrict__ cshift,
                                                    const int32_t *__restrict__ cstride, Y *__restrict__ y,
                                                    const Y *__restrict__ b, const int32_t *__restrict__ cseg,
                                                    const float *__restrict__ ysc) {
  __shared__ QuadPair<V> lut[256];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if ((int)blockIdx.x < qa.nfb) {  // blocks that are not coded: a chunk per wave
    const int c = (int)blockIdx.x * kWavesPerBlock + wave;
    if (c < qa.nfc) {
      const int r = qa.fchunk[c] * 64 + lane;
      if (r < a.n) sell_mr_row<V, X, ACC, K, NR, Y>(a, r, val, x, nx, cshift, cstride, y, b, cseg, ysc);
    }
    return;
  }
  const int blk = quad_block<V>(a, qa, lut);
  if ((int64_t)blk * kQuadBlock >= a.n) return;
  const int4 e = qa.blk[blk];
  const int tab = __builtin_amdgcn_readfirstlane(e.x), unit = __builtin_amdgcn_readfirstlane(e.y);
  if (tab < 0) return;
  // the block's rows lie in one tile: one shift and stride (its first chunk's)
  const int su = blk * (kQuadBlock / 64);
  const int32_t shift = cshift[su], stride = cstride[su], seg = cseg[su];
  const int64_t vr = (int64_t)blk * kQuadBlock + 4 * lane + shift;
  V4<Y> bv[NR];
  if (b)
#pragma unroll
    for (int c = 0; c < NR; ++c) bv[c] = ld4(b + vr + (int64_t)c * stride);
  ACC acc[NR][4];
  quad_rows<NR, V, X, ACC>(qa, tab, unit, lut, quad_rsrc<X>(x, nx, qa.bias), (int)(vr * (int64_t)sizeof(X)),
                           stride * (int)sizeof(X), acc);
#pragma unroll
  for (int c = 0; c < NR; ++c) {
    const ACC sc = ysc ? (ACC)ysc[seg + c] : (ACC)1;
    V4<Y> o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const ACC sum = ysc ? acc[c][q] * sc : acc[c][q];
      o.v[q] = b ? cvt<Y>((ACC)to_acc(bv[c].v[q]) - sum) : cvt<Y>(sum);
    }
    st4(y + vr + (int64_t)c * stride, o);
  }
}

// The multi-copy SpMV with K threads per row (int32-index layout): lane k of
// a matrix row sums slot k of each of the row's groups for all NR copies,
// then the K lanes add their sums by shuffles (the sums are reassociated).
template <class V, class X, class ACC, int K, int NR, class Y>
__global__ __launch_bounds__(kBlock) void k_sell_mr_lanes(SellArgs a, const V *__restrict__ val,
                                                          const X *__restrict__ x, const int32_t *__restrict__ cshift,
                                                          const int32_t *__restrict__ cstride, Y *__restrict__ y,
                                                          const Y *__restrict__ b, const int32_t *__restrict__ cseg,
                                                          const float *__restrict__ ysc) {
  static_assert(K >= 2 && kWave % K == 0, "K lanes of a row lie in one wavefront");
  constexpr int kRowsPerBlock = kBlock / K;
  const int k = threadIdx.x % K;
  for (int r0 = xcd_block() * kRowsPerBlock; r0 < a.n; r0 += gridDim.x * kRowsPerBlock) {
    const int r = r0 + threadIdx.x / K;
    ACC acc[NR];
#pragma unroll
    for (int c = 0; c < NR; ++c) acc[c] = 0;
    int s = 0;
    int64_t vr = 0, stride = 0;
    if (r < a.n) {
      s = r >> a.log2C;
      const int j = r - (s << a.log2C);
      const int C = 1 << a.log2C;
      const int rem = a.n - (s << a.log2C);
      const int tc = rem < C ? rem : C;
      const int groups = chunk_groups(a.cwidth[s]);
      const int64_t shift = cshift[s];
      stride = cstride[s];
      vr = (int64_t)r + shift;
      int64_t pos = (int64_t)a.cptr[s] + (int64_t)j * K + k;
      const int64_t step = (int64_t)tc * K;
      for (int g = 0; g < groups; ++g, pos += step) {
        const ACC v = (ACC)to_acc(val[pos]);
        const int64_t col = (int64_t)a.idx[pos] + shift;
#pragma unroll
        for (int c = 0; c < NR; ++c) acc[c] = fma_<ACC>(v, (ACC)to_acc(x[col + (int64_t)c * stride]), acc[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < NR; ++c)
#pragma unroll
      for (int off = K / 2; off > 0; off >>= 1) acc[c] += __shfl_xor(acc[c], off, kWave);
    if (r < a.n && k == 0) {
#pragma unroll
      for (int c = 0; c < NR; ++c) {
        const int64_t o = vr + (int64_t)c * stride;
        const ACC sum = ysc ? acc[c] * (ACC)ysc[cseg[s] + c] : acc[c];
        y[o] = b ? cvt<Y>((ACC)to_acc(b[o]) - sum) : cvt<Y>(sum);
      }
    }
  }
}

// An SDAINV factor split by row kind: a row whose only entry is its diagonal
// is an elementwise product (dval), any other row is a CSR row summed in
// column order with fp32 accumulation, as the SELL SpMV sums it; dval holds
// an fp16 NaN for those rows.  M = Z W^T x is k_b_m where all rows are short,
// else two launches:
//   k_b_mw: t = W^T x for every row (tile blocks: diagonal rows; row blocks:
//           the CSR rows), and y = Z t for the rows where Z is diagonal;
//   k_b_mz: y = Z t for the CSR rows of Z.  They read t of other rows: t of
//           a diagonal row of W is recomputed from x, t of a CSR row of W
//           is read back (k_b_mw stores t for those rows only).
// Each row's products are those of applying W^T, then Z, one at a time.
struct Factor16 {
  DevPtr dval, rows, rseg, rptr, col, val;  // rseg: segment of each CSR row
  int32_t nr = 0;
};
// dval is indexed by vector row + dsh[segment]: the right-hand sides of one
// system share one copy of its diagonals when they share its factors

__device__ __forceinline__ bool is_nan16(half_t v) {
  return (__builtin_bit_cast(uint16_t, v) & 0x7fffu) > 0x7c00u;
}

// input x_i of M: fp16 x, or the level-4 entry fp16(in * scale[seg]) computed
// here (and stored into hin by the tile blocks)
struct MIn {
  const half_t *x;
  const float *in;
  const float *sc;
  half_t *hin;
  const float *inv;  // `in` is an unnormalised basis column: in * inv[seg] (null: 1)
  __device__ __forceinline__ float iv(int seg) const { return inv ? inv[seg] : 1.f; }
  __device__ __forceinline__ half_t get(int64_t i, int seg) const {
    return in ? cvt<half_t>((to_acc(in[i]) * iv(seg)) * sc[seg]) : x[i];
  }
};

// what becomes of y_i = (M x)_i: 0 stored; 1 scaled by the segment's ome_0
// and stored; 2 the Richardson update fp16(fma(ome_k, y_i, ho_i)) stored;
// 3 that update converted out of the fp16 level, out_i = fp32(.) * iscale
struct MOut {
  int mode;
  half_t *y;
  const RichSeg *rs;
  int k;
  const half_t *ho;
  float *out;
  const float *iscale;
  // the segment's weight (modes 1-3)
  __device__ __forceinline__ float weight(int seg) const {
    return mode == 0 ? 0.f : (float)rs[seg].ome[mode == 1 ? 0 : k];
  }
  // hov = ho[i] (modes 2, 3), w = weight(seg)
  __device__ __forceinline__ void put(int64_t i, int seg, half_t v, half_t hov, float w) const {
    if (mode == 0) {
      y[i] = v;
    } else if (mode == 1) {
      y[i] = cvt<half_t>(to_acc(v) * w);
    } else {
      const half_t h = cvt<half_t>(fma_<float>(w, to_acc(v), to_acc(hov)));
      if (mode == 2)
        y[i] = h;
      else
        out[i] = cvt<float>(to_acc(h) * iscale[seg]);
    }
  }
  __device__ __forceinline__ void put(int64_t i, int seg, half_t v) const {
    put(i, seg, v, mode >= 2 ? ho[i] : (half_t)0, weight(seg));
  }
  // four consecutive rows (i aligned to 4): the same values as put() per row
  __device__ __forceinline__ void put4(int64_t i, int seg, const V4<half_t> &v, const V4<half_t> &hov,
                                       float w) const {
    if (mode <= 2) {
      V4<half_t> r;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        r.v[c] = mode == 0   ? v.v[c]
                 : mode == 1 ? cvt<half_t>(to_acc(v.v[c]) * w)
                             : cvt<half_t>(fma_<float>(w, to_acc(v.v[c]), to_acc(hov.v[c])));
      st4(y + i, r);
    } else {
      const float is = iscale[seg];
      V4<float> r;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        r.v[c] = cvt<float>(to_acc(cvt<half_t>(fma_<float>(w, to_acc(v.v[c]), to_acc(hov.v[c])))) * is);
      st4(out + i, r);
    }
  }
};

struct FacArgs {
  const half_t *__restrict__ d;
  const int32_t *__restrict__ rows;
  const int32_t *__restrict__ rseg;
  const int32_t *__restrict__ rptr;
  const int32_t *__restrict__ col;
  const half_t *__restrict__ val;
  int32_t nr;
};

// the rows of tile block b that are diagonal in both factors
__device__ __forceinline__ void b_m_tile(int b, const MIn &xin, const half_t *__restrict__ wd,
                                         const half_t *__restrict__ zd, const int64_t *__restrict__ dsh,
                                         const int32_t *__restrict__ bseg, const MOut &o) {
  // every load of the thread's rows first, then the stores (a branch
  // between a row's loads would keep one row's loads in flight at a time)
  const int seg = bseg[b];
  const float w = o.weight(seg);
  const float sc = xin.in ? xin.sc[seg] : 0.f, iv = xin.iv(seg);
  const int64_t sh = dsh[seg];
  V4<half_t> xi[kQuads], dw[kQuads], dz[kQuads], hov[kQuads];
#pragma unroll
  for (int q = 0; q < kQuads; ++q) {
    const int64_t i = tile_quad(q, b);
    if (xin.in) {
      const V4<float> f = ld4(xin.in + i);
#pragma unroll
      for (int c = 0; c < 4; ++c) xi[q].v[c] = cvt<half_t>((f.v[c] * iv) * sc);
    } else {
      xi[q] = ld4(xin.x + i);
    }
    dw[q] = ld4(wd + i + sh);
    dz[q] = ld4(zd + i + sh);
    if (o.mode >= 2) hov[q] = ld4(o.ho + i);
  }
#pragma unroll
  for (int q = 0; q < kQuads; ++q) {
    const int64_t i = tile_quad(q, b);
    if (xin.in) st4(xin.hin + i, xi[q]);
    bool plain = true;  // all four rows diagonal in W and Z
    V4<half_t> yv;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      plain = plain && !is_nan16(dw[q].v[c]) && !is_nan16(dz[q].v[c]);
      const half_t ti = cvt<half_t>(to_acc(dw[q].v[c]) * to_acc(xi[q].v[c]));
      yv.v[c] = cvt<half_t>(to_acc(dz[q].v[c]) * to_acc(ti));
    }
    if (plain) {
      o.put4(i, seg, yv, o.mode >= 2 ? hov[q] : yv, w);
      continue;
    }
    // a CSR row of W or Z is not a tile block's
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (!is_nan16(dw[q].v[c]) && !is_nan16(dz[q].v[c])) o.put(i + c, seg, yv.v[c], hov[q].v[c], w);
  }
}

// A row that is not diagonal in W or Z, both of at most kMRow entries a row:
// y_i = sum_g z_g fp16(sum_u w_gu x_c(gu)), g over Z's row i and u over W's
// row of Z's column g (one entry where that row is diagonal; one g where Z's
// row i is).  Slot u of group g of row r is at wc / wv[(g * nr + r) * kMRow +
// u], column -1 where there is none; meta: {vector row of the first copy, its
// segment, the copies' stride, groups}.
constexpr int kMRow = 4;
struct MRows {
  const int4 *__restrict__ meta;
  const int4 *__restrict__ wc;
  const half_t *__restrict__ wv, *__restrict__ z;
  int32_t nr;
};

// y = M x in one launch, where the rows of W and Z have at most kMRow entries:
// blocks below GR take rows of `R`, one thread for the NR copies of a row, and
// work t = W^T x of their columns out again; the rest are tile blocks.  The
// second launch for Z's rows and the indexes read once per copy were a third
// of M's time; the row blocks come first, so that their chain of three loads
// runs beside the tile blocks' streaming, which is what bounds M then.
// 5.93 M rows, 4 copies, 9% of the rows not diagonal: 30.3 -> 17.8 us.
template <int NR, bool IN>
__global__ __launch_bounds__(kBlock) void k_b_m(MIn xin, MRows R, int GR, const half_t *__restrict__ wd,
                                                const half_t *__restrict__ zd, const int64_t *__restrict__ dsh,
                                                const int32_t *__restrict__ bseg, MOut o) {
  if ((int)blockIdx.x >= GR) {
    b_m_tile((int)blockIdx.x - GR, xin, wd, zd, dsh, bseg, o);
    return;
  }
  const int32_t r = (int32_t)blockIdx.x * kBlock + threadIdx.x;
  if (r >= R.nr) return;
  const int4 m = R.meta[r];
  int4 wc[kMRow];
  V4<half_t> wv[kMRow];
#pragma unroll
  for (int g = 0; g < kMRow; ++g) {
    wc[g] = R.wc[(int64_t)g * R.nr + r];
    wv[g] = ld4(R.wv + ((int64_t)g * R.nr + r) * kMRow);
  }
  const V4<half_t> z = ld4(R.z + (int64_t)r * kMRow);
  float iv[NR], sc[NR], acc[NR];
#pragma unroll
  for (int c = 0; c < NR; ++c) {
    iv[c] = IN ? xin.iv(m.y + c) : 1.f;
    sc[c] = IN ? xin.sc[m.y + c] : 1.f;
    acc[c] = 0.f;
  }
#pragma unroll
  for (int g = 0; g < kMRow; ++g) {
    if (g >= m.w) break;
    const int32_t col[kMRow] = {wc[g].x, wc[g].y, wc[g].z, wc[g].w};
    typename std::conditional<IN, float, half_t>::type xv[kMRow][NR];
#pragma unroll
    for (int u = 0; u < kMRow; ++u)
#pragma unroll
      for (int c = 0; c < NR; ++c) {
        const int64_t q = (int64_t)(col[u] < 0 ? m.x : col[u]) + (int64_t)c * m.z;
        if constexpr (IN)
          xv[u][c] = xin.in[q];
        else
          xv[u][c] = xin.x[q];
      }
#pragma unroll
    for (int c = 0; c < NR; ++c) {
      float t = 0.f;
#pragma unroll
      for (int u = 0; u < kMRow; ++u) {
        half_t xu;
        if constexpr (IN)
          xu = cvt<half_t>((xv[u][c] * iv[c]) * sc[c]);
        else
          xu = xv[u][c];
        if (col[u] >= 0) t = fma_<float>(to_acc(wv[g].v[u]), to_acc(xu), t);
      }
      acc[c] = fma_<float>(to_acc(z.v[g]), to_acc(cvt<half_t>(t)), acc[c]);
    }
  }
#pragma unroll
  for (int c = 0; c < NR; ++c) o.put((int64_t)m.x + (int64_t)c * m.z, m.y + c, cvt<half_t>(acc[c]));
}

__global__ __launch_bounds__(kBlock) void k_b_mw(MIn xin, FacArgs W, const half_t *__restrict__ zd,
                                                 const int64_t *__restrict__ dsh, half_t *__restrict__ t, int G,
                                                 const int32_t *__restrict__ bseg, MOut o) {
  if ((int)blockIdx.x < G) {
    b_m_tile((int)blockIdx.x, xin, W.d, zd, dsh, bseg, o);
    return;
  }
  const int32_t r = (int32_t)(blockIdx.x - G) * kBlock + threadIdx.x;
  if (r >= W.nr) return;
  const int64_t i = W.rows[r];
  const int seg = W.rseg[r];
  float acc = 0.f;
  for (int32_t k = W.rptr[r]; k < W.rptr[r + 1]; ++k)
    acc = fma_<float>(to_acc(W.val[k]), to_acc(xin.get(W.col[k], seg)), acc);
  const half_t ti = cvt<half_t>(acc);
  t[i] = ti;
  const half_t dz = zd[i + dsh[seg]];
  if (!is_nan16(dz)) o.put(i, seg, cvt<half_t>(to_acc(dz) * to_acc(ti)));
}

__global__ __launch_bounds__(kBlock) void k_b_mz(FacArgs Z, MIn xin, const half_t *__restrict__ wd,
                                                 const int64_t *__restrict__ dsh, const half_t *__restrict__ t,
                                                 MOut o) {
  const int32_t r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= Z.nr) return;
  const int seg = Z.rseg[r];
  const int64_t sh = dsh[seg];
  float acc = 0.f;
  for (int32_t k = Z.rptr[r]; k < Z.rptr[r + 1]; ++k) {
    const int32_t c = Z.col[k];
    const half_t dw = wd[c + sh];
    const half_t tc = is_nan16(dw) ? t[c] : cvt<half_t>(to_acc(dw) * to_acc(xin.get(c, seg)));
    acc = fma_<float>(to_acc(Z.val[k]), to_acc(tc), acc);
  }
  o.put(Z.rows[r], seg, cvt<half_t>(acc));
}

// ----------------------------------------------------------- solver ---
template <class T> struct BLevel {
  int m = 0;
  DevPtr V, Z, H, cs, sn, e, inv;  // V, Z column-major (ld = N); per segment H, cs, sn, e, inv
  DevPtr csc;  // per column and segment 1/||w|| of columns left unnormalised (level 3)
  T *Vc(int64_t N, int k) const { return V->as<T>() + (int64_t)k * N; }
  T *Zc(int64_t N, int k) const { return Z->as<T>() + (int64_t)k * N; }
  int64_t hs() const { return (int64_t)(m + 1) * m; }
};

HostCSR concat(const std::vector<const HostCSR *> &parts, const std::vector<int64_t> &off, int64_t N) {
  HostCSR R;
  int64_t nnz = 0;
  for (const HostCSR *p : parts) nnz += p->nnz();
  F3R_CHECK(N < INT32_MAX && nnz < INT32_MAX, F3R_ERR_RANGE, "batch: more than 2^31 rows or nonzeros in all");
  R.n = R.ncols = (int32_t)N;
  R.rptr.assign(N + 1, 0);
  R.idx.resize(nnz);
  R.val.resize(nnz);
  int64_t q = 0;
  for (size_t s = 0; s < parts.size(); ++s) {
    const HostCSR &A = *parts[s];
    const int32_t o = (int32_t)off[s];
    for (int32_t i = 0; i < A.n; ++i) {
      for (int32_t k = A.rptr[i]; k < A.rptr[i + 1]; ++k, ++q) {
        R.idx[q] = A.idx[k] + o;
        R.val[q] = A.val[k];
      }
      R.rptr[o + i + 1] = (int32_t)q;
    }
    for (int64_t r = o + A.n; r < off[s + 1]; ++r) R.rptr[r + 1] = (int32_t)q;  // padding rows: empty
  }
  return R;
}

}  // namespace

struct BatchSolver {
  std::shared_ptr<Context> ctx;
  f3r_params p{};
  int nseg = 0;
  int64_t N = 0;
  int G = 0;  // tiles of kTile rows
  int32_t snb_max = 0;  // tiles of the largest segment
  // up to this many tiles (262 K rows) and 16 columns a block adds the dots of
  // its segment up itself: two loads a lane and column at most
  static constexpr int32_t kDirectBlocks = 128;
  std::vector<int64_t> off;
  std::vector<int32_t> nrow;
  DevPtr bseg, sb0, snb, scale, iscale;
  std::shared_ptr<SellShared> sh, sh16;
  std::shared_ptr<QuadSet> quad;  // NR > 1: value codes, a table per system (null: too many values)
  DevPtr A64, A32, A16;
  // NR > 1: each system's matrix is stored once for its NR right-hand sides
  // (chunk -> vector-row shift and copy stride, per layout)
  int NR = 1;
  // flags bit 4: the SpMVs with K threads per row (int32-index layouts)
  bool lanes = false;
  DevPtr csh, cst, csh16, cst16;
  Factor16 W, Z;
  // the rows that are not diagonal, where k_b_m takes them (mr_nr < 0: k_b_mw and k_b_mz do)
  DevPtr mr_meta, mr_wc, mr_wv, mr_z;
  int32_t mr_nr = -1;
  int mr_copies = 1;
  DevPtr dsh;  // per segment: vector row -> row of the factor diagonals
  DevPtr cseg;  // NR > 1: per chunk, the segment of its first copy
  // level 3's Z as the fp16 Richardson output h (Z = h / s exactly, s the
  // segment's power-of-two range scale): NR > 1 and every s a power of two
  bool zh = false;
  DevPtr Zh3;
  half_t *zh3(int k) const { return Zh3->as<half_t>() + (int64_t)k * N; }
  DevPtr partial, rich, rows;  // rows: per segment, without the padding
  DevPtr b_int, x_int;
  // per-segment host values that the kernels read and write in pinned host
  // memory (no copy commands): status, the residual norms; jseg, the steps of
  // a cycle; bp / xp, the callers' vectors of a solve
  void *pin = nullptr;
  double *status = nullptr;
  int32_t *jseg = nullptr;
  const double **bp = nullptr;
  double **xp = nullptr;
  // outer level (fp64)
  BLevel<double> L1;
  BLevel<float> L2, L3;
  DevPtr hin, hout, hout2, hr, tmp, tt, t2;
  int64_t cnt = 0, calls = 0;
  std::map<uint64_t, hipGraphExec_t> graphs;  // level-2 body per probe pattern
  // a whole outer step per (probe pattern, step index j)
  std::map<std::pair<uint64_t, int>, hipGraphExec_t> step_graphs;
  static constexpr size_t kMaxStepGraphs = 64;
  std::vector<hipGraph_t> graph_src;

  BatchSolver() = default;
  BatchSolver(const BatchSolver &) = delete;
  BatchSolver &operator=(const BatchSolver &) = delete;
  ~BatchSolver() {
    for (auto &g : graphs) (void)hipGraphExecDestroy(g.second);
    for (auto &g : step_graphs) (void)hipGraphExecDestroy(g.second);
    for (auto &g : graph_src) (void)hipGraphDestroy(g);
    if (pin) (void)hipHostFree(pin);
  }
  // the pinned values (device addresses equal to the host's)
  void alloc_pinned() {
    const size_t n = (size_t)nseg;
    F3R_HIP(hipHostMalloc(&pin, n * (8 + 8 + 8 + 4), hipHostMallocDefault));
    void *dev = nullptr;
    F3R_HIP(hipHostGetDevicePointer(&dev, pin, 0));
    F3R_CHECK(dev == pin, F3R_ERR_HIP, "batch: pinned memory without a unified address");
    status = static_cast<double *>(pin);
    xp = reinterpret_cast<double **>(status + n);
    bp = const_cast<const double **>(xp + n);
    jseg = reinterpret_cast<int32_t *>(xp + 2 * n);
  }

  hipStream_t st() const { return ctx->stream; }
  int32_t *bs() const { return bseg->as<int32_t>(); }

  // y = A x (b null) or y = b - A x over all segments, A the fp64/fp32 copy
  // (layout sh) or the fp16 one (sh16)
  template <class V, class X, class Y, class ACC>
  // ysc (NR > 1 only): per-segment factor on the sums (x stored scaled)
  void spmv(const V *val, bool half_layout, const X *x, Y *y, const Y *b, const float *ysc = nullptr) {
    const SellShared &L = half_layout ? *sh16 : *sh;
    SellArgs a = sell_args(L, false);
    if (NR == 1) {
      F3R_CHECK(ysc == nullptr, F3R_ERR_STATE, "batch: scaled SpMV needs shared matrices");
      a.lanes = lanes ? L.K : 1;  // K threads per row
      if (b)
        launch_sell<V, X, ACC>(L.K, a, val, x, EpiResid<Y, Y, ACC>{y, b, nullptr}, st());
      else
        launch_sell<V, X, ACC>(L.K, a, val, x, EpiStore<Y, ACC>{y, nullptr}, st());
      return;
    }
    const int32_t *shf = (half_layout ? csh16 : csh)->as<int32_t>(), *str = (half_layout ? cst16 : cst)->as<int32_t>();
    const dim3 g((a.n + kBlock - 1) / kBlock);
    auto go = [&](auto kt, auto nt) {
      constexpr int K = decltype(kt)::value, R = decltype(nt)::value;
      if constexpr (K >= 2) {
        if (lanes) {  // K threads per matrix row
          const dim3 gl((unsigned)(((int64_t)a.n * K + kBlock - 1) / kBlock));
          hipLaunchKernelGGL((k_sell_mr_lanes<V, X, ACC, K, R, Y>), gl, dim3(kBlock), 0, st(), a, val, x, shf, str,
                             y, b, (const int32_t *)cseg->as<int32_t>(), ysc);
          return;
        }
      }
      if (quad) {
        const QuadArgs qa = quad->template args<V>();
        hipLaunchKernelGGL((k_quad_mr<V, X, ACC, K, R, Y>), dim3(quad_blocks(a, qa)), dim3(kBlock), 0, st(), a, qa,
                           val, x, (int64_t)N, shf, str, y, b, (const int32_t *)cseg->as<int32_t>(), ysc);
        return;
      }
      hipLaunchKernelGGL((k_sell_mr<V, X, ACC, K, R, Y>), g, dim3(kBlock), 0, st(), a, val, x, (int64_t)N, shf, str, y,
                         b, (const int32_t *)cseg->as<int32_t>(), ysc);
    };
    auto byk = [&](auto nt) {
      switch (L.K) {
        case 1: go(std::integral_constant<int, 1>(), nt); break;
        case 2: go(std::integral_constant<int, 2>(), nt); break;
        case 4: go(std::integral_constant<int, 4>(), nt); break;
        default: go(std::integral_constant<int, 8>(), nt); break;
      }
    };
    if (NR == 2)
      byk(std::integral_constant<int, 2>());
    else
      byk(std::integral_constant<int, 4>());
  }

  template <class T> void alloc_level(BLevel<T> &L, int m) {
    L.m = m;
    // vectors end in 64 bytes of padding: a product's windows of x reach past the last row
    L.V = dev_alloc(sizeof(T) * N * (m + 1) + 64);
    L.Z = dev_alloc(sizeof(T) * N * m + 64);
    L.H = dev_alloc(sizeof(T) * nseg * L.hs());
    L.cs = dev_alloc(sizeof(T) * nseg * m);
    L.sn = dev_alloc(sizeof(T) * nseg * m);
    L.e = dev_alloc(sizeof(T) * nseg * (m + 1));
    L.inv = dev_alloc(sizeof(T) * nseg);
    L.csc = dev_alloc(sizeof(T) * nseg * (m + 1));
  }

  // one Arnoldi step j of level L (w = V_{j+1} already holds A z_j).  V0:
  // column 0 (the level's input, not copied).  lazy: V_{j+1} stays
  // unnormalised, its 1/||w|| per segment goes to csc column j + 1 and every
  // reader applies it (no scaling pass)
  template <class T> void arnoldi(BLevel<T> &L, int j, int e0_one, double *stat, const T *V0, bool lazy) {
    const int ncols = j + 1;
    T *H = L.H->template as<T>();
    T *part = partial->as<T>();
    const T *csc = lazy ? L.csc->template as<T>() : nullptr;
    const T *Vb = L.Vc(N, 0);
    if (ncols <= 4)
      hipLaunchKernelGGL((k_b_mdot<T, T, 4>), dim3(G, 1), dim3(kBlock), 0, st(), (const T *)L.Vc(N, j + 1), V0, Vb,
                         N, ncols, csc, nseg, (const int32_t *)bs(), part);
    else if (ncols <= 8)
      hipLaunchKernelGGL((k_b_mdot<T, T, 8>), dim3(G, 1), dim3(kBlock), 0, st(), (const T *)L.Vc(N, j + 1), V0, Vb,
                         N, ncols, csc, nseg, (const int32_t *)bs(), part);
    else
      hipLaunchKernelGGL((k_b_mdot<T, T, 16>), dim3(G, (ncols + 15) / 16), dim3(kBlock), 0, st(),
                         (const T *)L.Vc(N, j + 1), V0, Vb, N, ncols, csc, nseg, (const int32_t *)bs(), part);
    // small segments' dots are added up by their readers
    const bool direct = snb_max <= kDirectBlocks && ncols <= 16;
    if (!direct)
      hipLaunchKernelGGL(k_b_dots_finish<T>, dim3(nseg, ncols), dim3(kBlock), 0, st(), (const T *)part, G,
                         (const int32_t *)sb0->as<int32_t>(), (const int32_t *)snb->as<int32_t>(),
                         H + (int64_t)j * (L.m + 1), L.hs());
    T *npart = part + (int64_t)ncols * G;  // the dots' sums are still read
    hipLaunchKernelGGL((k_b_update<T, T>), dim3(G), dim3(kBlock), 0, st(), L.Vc(N, j + 1), V0, Vb, N, ncols, csc,
                       nseg, H + (int64_t)j * (L.m + 1), L.hs(), (const int32_t *)bs(), npart,
                       (const T *)(direct ? part : nullptr), (const int32_t *)sb0->as<int32_t>(),
                       (const int32_t *)snb->as<int32_t>());
    hipLaunchKernelGGL(k_b_norm_finish<T>, dim3(nseg), dim3(kBlock), 0, st(), (const T *)npart,
                       (const int32_t *)sb0->as<int32_t>(), (const int32_t *)snb->as<int32_t>(),
                       H + (int64_t)j * (L.m + 1), L.hs(), L.cs->template as<T>(), L.sn->template as<T>(),
                       (int64_t)L.m, L.e->template as<T>(), (int64_t)(L.m + 1), j, e0_one,
                       lazy ? L.csc->template as<T>() + (int64_t)(j + 1) * nseg : L.inv->template as<T>(), stat);
    if (lazy) return;
    hipLaunchKernelGGL((k_b_vscale<T, T>), dim3(G), dim3(kBlock), 0, st(), L.Vc(N, j + 1),
                       (const T *)L.inv->template as<T>(), (const int32_t *)bs());
  }

  static FacArgs fac(const Factor16 &F) {
    return {F.dval->as<half_t>(), F.rows->as<int32_t>(), F.rseg->as<int32_t>(), F.rptr->as<int32_t>(),
            F.col->as<int32_t>(), F.val->as<half_t>(), F.nr};
  }
  // y = M x with M = Z W^T (ainv.hpp:110-114): W^T first, then Z; x given
  // by `xin`, y consumed by `o`
  void precond(const MIn &xin, const MOut &o) {
    if (mr_nr >= 0) {
      const MRows R{mr_meta->as<int4>(), mr_wc->as<int4>(), mr_wv->as<half_t>(), mr_z->as<half_t>(), mr_nr};
      const int gr = (mr_nr + kBlock - 1) / kBlock;
      auto go = [&](auto nt) {
        constexpr int NC = decltype(nt)::value;
        hipLaunchKernelGGL((xin.in ? k_b_m<NC, true> : k_b_m<NC, false>), dim3(G + gr), dim3(kBlock), 0, st(), xin, R,
                           gr, (const half_t *)W.dval->as<half_t>(), (const half_t *)Z.dval->as<half_t>(),
                           (const int64_t *)dsh->as<int64_t>(), (const int32_t *)bs(), o);
      };
      if (mr_copies == 4)
        go(std::integral_constant<int, 4>());
      else if (mr_copies == 2)
        go(std::integral_constant<int, 2>());
      else
        go(std::integral_constant<int, 1>());
      return;
    }
    half_t *t = tmp->as<half_t>();
    const int gw = (W.nr + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(k_b_mw, dim3(G + gw), dim3(kBlock), 0, st(), xin, fac(W), (const half_t *)Z.dval->as<half_t>(),
                       (const int64_t *)dsh->as<int64_t>(), t, G, (const int32_t *)bs(), o);
    if (Z.nr > 0) {
      // k_b_mz reads x as k_b_mw does (in the entry call: fp16(in * s) from
      // the fp32 input)
      hipLaunchKernelGGL(k_b_mz, dim3((Z.nr + kBlock - 1) / kBlock), dim3(kBlock), 0, st(), fac(Z), xin,
                         (const half_t *)W.dval->as<half_t>(), (const int64_t *)dsh->as<int64_t>(), (const half_t *)t,
                         o);
    }
  }
  void precond(const half_t *in, half_t *out) {
    precond(MIn{in, nullptr, nullptr, nullptr, nullptr}, MOut{0, out, nullptr, 0, nullptr, nullptr, nullptr});
  }

  void probe(const half_t *x, const half_t *r, int k) {
    half_t *t = tt->as<half_t>();
    spmv<half_t, half_t, half_t, float>(A16->as<half_t>(), true, x, t, nullptr);
    float *part = partial->as<float>();
    hipLaunchKernelGGL(k_b_probe_dots, dim3(G), dim3(kBlock), 0, st(), (const half_t *)t, r, part);
    hipLaunchKernelGGL(k_b_probe_finish, dim3(nseg), dim3(kBlock), 0, st(), (const float *)part, G,
                       (const int32_t *)sb0->as<int32_t>(), (const int32_t *)snb->as<int32_t>(),
                       rich->as<RichSeg>(), k);
  }

  // adaptive Richardson in fp16 (work/src/f3r-gpu.cpp:229-260), per segment
  // in_inv: per-segment 1/||w|| of an unnormalised input column (null: 1)
  // hz: the fp16 result h itself instead of out = h / s
  void level4(const float *in, const float *in_inv, float *out, half_t *hz = nullptr) {
    ++cnt;
    ++calls;
    const bool pr = (cnt % p.c) == 0;
    half_t *hi = hin->as<half_t>(), *ho = hout->as<half_t>(), *ho2 = hout2->as<half_t>();
    half_t *hr_ = hr->as<half_t>(), *tw = t2->as<half_t>();
    RichSeg *rs = rich->as<RichSeg>();
    // entry hin = fp16(in * s) fused into the first application of M; off
    // probe calls the weighting by ome_0 is fused too
    const float *isc = iscale->as<float>();
    precond(MIn{nullptr, in, scale->as<float>(), hi, in_inv},
            MOut{pr ? 0 : 1, ho, rs, 0, nullptr, nullptr, nullptr});
    if (pr) {
      probe(ho, hi, 0);
      hipLaunchKernelGGL(k_b_l4_scale, dim3(G), dim3(kBlock), 0, st(), ho, (const RichSeg *)rs, 1,
                         (const int32_t *)bs());
    }
    bool done = false;  // the last step already wrote the result
    for (int k = 1; k < p.m4; ++k) {
      const bool last = k == p.m4 - 1;
      half_t *hn = last && hz ? hz : ho2;  // the step's fp16 result
      spmv<half_t, half_t, half_t, float>(A16->as<half_t>(), true, (const half_t *)ho, hr_, (const half_t *)hi);
      if (pr) {
        precond(hr_, tw);
        probe(tw, hr_, k);
        hipLaunchKernelGGL(k_b_l4_update, dim3(G), dim3(kBlock), 0, st(), (const half_t *)tw, (const half_t *)ho,
                           hn, (const RichSeg *)rs, k, 1, (const int32_t *)bs());
        done = last && hz;
      } else {
        // the weighted update (and on the last step the way out of the
        // fp16 level, unless hz takes h itself) fused into M
        precond(MIn{hr_, nullptr, nullptr, nullptr, nullptr},
                MOut{last && !hz ? 3 : 2, hn, rs, k, (const half_t *)ho, out, isc});
        done = last;
      }
      std::swap(ho, ho2);
    }
    if (done) return;
    if (hz)
      hipLaunchKernelGGL((k_b_cast<half_t, half_t>), dim3(G), dim3(kBlock), 0, st(), (const half_t *)ho, hz);
    else
      hipLaunchKernelGGL((k_b_entry<half_t, float>), dim3(G), dim3(kBlock), 0, st(), (const half_t *)ho, out, isc,
                         (const int32_t *)bs());
  }

  // FGMRES(m3) on the fp16 values, fp32 basis, normalize = false
  // (V_0 is the level-2 column itself; the other columns stay unnormalised)
  void level3(const float *in, float *out) {
    BLevel<float> &L = L3;
    const float *isc = iscale->as<float>();
    for (int j = 0; j < L.m; ++j) {
      const float *vin = j == 0 ? in : L.Vc(N, j);
      const float *vinv = j == 0 ? nullptr : L.csc->as<float>() + (int64_t)j * nseg;
      if (zh) {
        level4(vin, vinv, nullptr, zh3(j));
        spmv<half_t, half_t, float, float>(A16->as<half_t>(), true, (const half_t *)zh3(j), L.Vc(N, j + 1), nullptr,
                                           isc);
      } else {
        level4(vin, vinv, L.Zc(N, j));
        spmv<half_t, float, float, float>(A16->as<half_t>(), true, (const float *)L.Zc(N, j), L.Vc(N, j + 1),
                                          nullptr);
      }
      arnoldi(L, j, 1, nullptr, in, true);
    }
    if (zh)
      hipLaunchKernelGGL((k_b_combine<half_t, float, float>), dim3(G), dim3(kBlock), 0, st(), (const half_t *)zh3(0),
                         N, (const float *)L.H->as<float>(), L.hs(), L.m + 1, (const float *)L.e->as<float>(),
                         (int64_t)(L.m + 1), (const int32_t *)nullptr, L.m, (const int32_t *)bs(), out, 0, isc);
    else
      hipLaunchKernelGGL((k_b_combine<float, float, float>), dim3(G), dim3(kBlock), 0, st(), (const float *)L.Zc(N, 0),
                         N, (const float *)L.H->as<float>(), L.hs(), L.m + 1, (const float *)L.e->as<float>(),
                         (int64_t)(L.m + 1), (const int32_t *)nullptr, L.m, (const int32_t *)bs(), out, 0,
                         (const float *)nullptr);
  }

  // the level-2 Arnoldi loop: every buffer it touches is the solver's own, so
  // the same launches serve every call with the same probe positions
  void level2_body() {
    BLevel<float> &L = L2;
    for (int j = 0; j < L.m; ++j) {
      level3(L.Vc(N, j), L.Zc(N, j));
      spmv<float, float, float, float>(A32->as<float>(), false, (const float *)L.Zc(N, j), L.Vc(N, j + 1), nullptr);
      arnoldi(L, j, 1, nullptr, (const float *)L.Vc(N, 0), false);
    }
  }

  // probe positions of the next level-2 body as a bit mask (bit q: the q-th
  // level-4 call probes); UINT64_MAX when not representable
  uint64_t next_pattern() const {
    const int64_t calls_per = (int64_t)p.m2 * p.m3;
    if (calls_per > 63) return UINT64_MAX;
    uint64_t mask = 0;
    for (int64_t q = 0; q < calls_per; ++q)
      if (((cnt + q + 1) % p.c) == 0) mask |= 1ULL << q;
    return mask | (1ULL << 63);
  }

  // FGMRES(m2) on the fp32 values, fp32 basis, normalize = false.  With
  // use_graph the body is captured once per probe pattern (at most 33) and
  // replayed: it holds no host synchronisation, memset or host copy, and the
  // Richardson weights and probe results stay in device memory between calls
  // body_graph false: the body is launched eagerly (inside a capture of the
  // whole outer step)
  void level2(const double *in, double *out, bool body_graph) {
    BLevel<float> &L = L2;
    hipLaunchKernelGGL((k_b_cast<double, float>), dim3(G), dim3(kBlock), 0, st(), in, L.Vc(N, 0));
    const uint64_t key = p.use_graph && body_graph ? next_pattern() : UINT64_MAX;
    if (key == UINT64_MAX || (graphs.size() > 32 && graphs.find(key) == graphs.end())) {
      level2_body();
    } else {
      auto it = graphs.find(key);
      if (it == graphs.end()) {
        const int64_t cnt0 = cnt, calls0 = calls;
        hipGraph_t gr;
        F3R_HIP(hipStreamBeginCapture(st(), hipStreamCaptureModeThreadLocal));
        try {
          level2_body();
        } catch (...) {
          (void)hipStreamEndCapture(st(), &gr);
          throw;
        }
        F3R_HIP(hipStreamEndCapture(st(), &gr));
        hipGraphExec_t ex;
        const hipError_t e = hipGraphInstantiate(&ex, gr, nullptr, nullptr, 0);
        if (e != hipSuccess) (void)hipGraphDestroy(gr);
        F3R_HIP(e);
        graph_src.push_back(gr);
        it = graphs.emplace(key, ex).first;
        cnt = cnt0;  // the capture only recorded the calls
        calls = calls0;
      }
      F3R_HIP(hipGraphLaunch(it->second, st()));
      cnt += (int64_t)p.m2 * p.m3;
      calls += (int64_t)p.m2 * p.m3;
    }
    hipLaunchKernelGGL((k_b_combine<float, float, double>), dim3(G), dim3(kBlock), 0, st(),
                       (const float *)L.Zc(N, 0), N, (const float *)L.H->as<float>(), L.hs(), L.m + 1,
                       (const float *)L.e->as<float>(), (int64_t)(L.m + 1), (const int32_t *)nullptr, L.m,
                       (const int32_t *)bs(), out, 0, (const float *)nullptr);
  }

  // outer Arnoldi step j of every segment: level 2 on V_j into Z_j, the fp64
  // SpMV into V_{j+1} and the outer Gram-Schmidt / Givens step, whose |e_{j+1}|
  // per segment lands in `status`.  With use_graph the whole step is
  // captured once per (probe pattern, j) and replayed as one graph launch
  // (beyond kMaxStepGraphs of them, only the level-2 bodies are replayed).
  void outer_step(int j) {
    BLevel<double> &L = L1;
    double *V = L.V->as<double>();
    auto body = [&](bool body_graph) {
      level2(V + (int64_t)j * N, L.Zc(N, j), body_graph);
      spmv<double, double, double, double>(A64->as<double>(), false, (const double *)L.Zc(N, j),
                                           V + (int64_t)(j + 1) * N, nullptr);
      arnoldi(L, j, 0, status, (const double *)L.Vc(N, 0), false);
    };
    const uint64_t pat = p.use_graph ? next_pattern() : UINT64_MAX;
    const auto key = std::make_pair(pat, j);
    auto it = step_graphs.find(key);
    if (pat == UINT64_MAX || (it == step_graphs.end() && step_graphs.size() >= kMaxStepGraphs)) {
      body(true);
      return;
    }
    if (it == step_graphs.end()) {
      const int64_t cnt0 = cnt, calls0 = calls;
      hipGraph_t gr;
      F3R_HIP(hipStreamBeginCapture(st(), hipStreamCaptureModeThreadLocal));
      try {
        body(false);
      } catch (...) {
        (void)hipStreamEndCapture(st(), &gr);
        throw;
      }
      F3R_HIP(hipStreamEndCapture(st(), &gr));
      hipGraphExec_t ex;
      const hipError_t e = hipGraphInstantiate(&ex, gr, nullptr, nullptr, 0);
      if (e != hipSuccess) (void)hipGraphDestroy(gr);
      F3R_HIP(e);
      graph_src.push_back(gr);
      it = step_graphs.emplace(key, ex).first;
      cnt = cnt0;  // the capture only recorded the calls
      calls = calls0;
    }
    F3R_HIP(hipGraphLaunch(it->second, st()));
    cnt += (int64_t)p.m2 * p.m3;
    calls += (int64_t)p.m2 * p.m3;
  }

  std::vector<double> read_status() {
    F3R_HIP(hipStreamSynchronize(st()));
    return std::vector<double>(status, status + nseg);
  }

  // Restarted<double>(FGMRES<double>(A, L2, {m1, true}), {restart}) per segment
  // |e| / ||b|| against eps; a zero right-hand side is met only by a zero residual
  static double rel(double e, double nb) { return nb > 0 ? e / nb : (e == 0 ? 0.0 : HUGE_VAL); }

  void solve(const std::vector<double> &nrm_b, std::vector<f3r_result> &res) {
    BLevel<double> &L = L1;
    const int m1 = L.m;
    double *V = L.V->as<double>(), *Hd = L.H->as<double>();
    std::vector<char> solved(nseg, 0);
    std::vector<int32_t> iters(nseg, 0), cycles(nseg, 0);
    std::vector<double> last(nseg, 0.0);
    cnt = p.c;
    calls = 0;
    hipLaunchKernelGGL(k_b_rich_reset, dim3((nseg + 63) / 64), dim3(64), 0, st(), nseg, rich->as<RichSeg>());
    for (int cyc = 0; cyc < p.restart; ++cyc) {
      std::vector<char> active(nseg, 0);
      for (int s = 0; s < nseg; ++s) active[s] = !solved[s];
      // r = b - A x, e_0 = ||r||, V_0 = r / ||r||
      spmv<double, double, double, double>(A64->as<double>(), false, (const double *)x_int->as<double>(), V,
                                           (const double *)b_int->as<double>());
      hipLaunchKernelGGL(k_b_norm2<double>, dim3(G), dim3(kBlock), 0, st(), (const double *)V, partial->as<double>());
      // no rotation (j = -1): e_0 = ||r|| is written where H(j + 1) would go
      hipLaunchKernelGGL(k_b_norm_finish<double>, dim3(nseg), dim3(kBlock), 0, st(),
                         (const double *)partial->as<double>(), (const int32_t *)sb0->as<int32_t>(),
                         (const int32_t *)snb->as<int32_t>(), L.e->as<double>(), (int64_t)(m1 + 1),
                         (double *)nullptr, (double *)nullptr, (int64_t)0, (double *)nullptr, (int64_t)0, -1, 0,
                         L.inv->as<double>(), status);
      hipLaunchKernelGGL((k_b_vscale<double, double>), dim3(G), dim3(kBlock), 0, st(), V,
                         (const double *)L.inv->as<double>(), (const int32_t *)bs());
      std::vector<double> e = read_status();
      std::vector<int32_t> jdone(nseg, 0);
      bool any = false;
      for (int s = 0; s < nseg; ++s) {
        if (!active[s]) continue;
        last[s] = e[s];
        ++cycles[s];
        if (rel(e[s], nrm_b[s]) < p.eps) {
          solved[s] = 1;
          active[s] = 0;
        } else {
          any = true;
        }
      }
      if (!any) break;
      int j = 0;
      for (; j < m1; ++j) {
        outer_step(j);
        std::vector<double> st_h = read_status();
        bool left = false;
        for (int s = 0; s < nseg; ++s) {
          if (!active[s]) continue;
          ++iters[s];
          jdone[s] = j + 1;
          last[s] = st_h[s];
          if (rel(st_h[s], nrm_b[s]) < p.eps) {
            solved[s] = 1;
            active[s] = 0;
          } else {
            left = true;
          }
        }
        if (!left) break;
      }
      // x += Z y(j_s) for every segment that stepped in this cycle
      std::copy(jdone.begin(), jdone.end(), jseg);
      hipLaunchKernelGGL((k_b_combine<double, double, double>), dim3(G), dim3(kBlock), 0, st(),
                         (const double *)L.Zc(N, 0), N, (const double *)Hd, L.hs(), m1 + 1,
                         (const double *)L.e->as<double>(), (int64_t)(m1 + 1), (const int32_t *)jseg,
                         0, (const int32_t *)bs(), x_int->as<double>(), 1, (const float *)nullptr);
      F3R_HIP(hipStreamSynchronize(st()));  // jseg is written again by the next cycle
    }
    F3R_HIP(hipGetLastError());
    res.resize(nseg);
    for (int s = 0; s < nseg; ++s) {
      res[s] = f3r_result{};
      res[s].is_solved = solved[s];
      res[s].res_iter = iters[s];
      res[s].res_nrm2 = last[s];
      res[s].nrm_b = nrm_b[s];
      res[s].precond_calls = calls;
      res[s].outer_cycles = cycles[s];
    }
  }
};

BatchSolver *batch_create(std::shared_ptr<Context> ctx, const std::vector<std::shared_ptr<Mat>> &A,
                          const std::vector<std::shared_ptr<Prec>> &P, const f3r_params &p) {
  F3R_CHECK(!A.empty() && A.size() == P.size(), F3R_ERR_ARG, "batch: one matrix and one preconditioner per segment");
  F3R_CHECK(p.m1 >= 1 && p.m1 <= 120 && p.m2 >= 1 && p.m2 <= 16 && p.m3 >= 1 && p.m3 <= 16 && p.m4 >= 1 &&
                p.m4 <= 16 && p.c >= 1 && p.restart >= 1,
            F3R_ERR_ARG, "batch: m1 in [1, 120], m2, m3, m4 in [1, 16], c, restart >= 1");
  // the lockstep nest is the adaptive-weight HALF F3R nest only
  F3R_CHECK(p.variant == 0 && p.static_weight == 0.0 && p.depth == 0, F3R_ERR_ARG,
            "batch: only the HALF F3R nest with adaptive weights (variant 0, static_weight 0, depth 0)");
  // k_sell_mr reads a chunk's header once per wavefront (C >= 64) and a tile
  // holds whole chunks (C <= kTile); K selects a built kernel
  F3R_CHECK(p.C == 0 || (p.C >= 64 && p.C <= kTile && (p.C & (p.C - 1)) == 0), F3R_ERR_ARG,
            "batch: C must be a power of two in [64, 2048] (0 = 64)");
  F3R_CHECK(p.K == 0 || p.K == 1 || p.K == 2 || p.K == 4 || p.K == 8, F3R_ERR_ARG,
            "batch: K must be 1, 2, 4 or 8 (0 = 4)");
  F3R_CHECK(!(p.flags & 16) || (p.index == 0 && p.K != 1), F3R_ERR_ARG,
            "batch: K threads per row (flags bit 4) need the int32-index layout (index 0) and K >= 2");
  auto B = std::make_unique<BatchSolver>();
  B->ctx = ctx;
  B->p = p;
  B->lanes = (p.flags & 16) != 0;
  B->nseg = (int)A.size();
  const int nseg = B->nseg;
  B->off.assign(nseg + 1, 0);
  B->nrow.resize(nseg);
  std::vector<const HostCSR *> pa(nseg), pw(nseg), pz(nseg);
  std::vector<float> sc(nseg), isc(nseg);
  for (int s = 0; s < nseg; ++s) {
    F3R_CHECK(A[s] && A[s]->host && A[s]->format == 0, F3R_ERR_ARG, "batch: CSR matrices");
    const HostCSR &h = *A[s]->host;
    F3R_CHECK(h.n > 0 && h.n == h.ncols, F3R_ERR_ARG, "batch: square non-empty matrices");
    F3R_CHECK(P[s] && P[s]->kind == 0 && P[s]->host.f[0].n == h.n, F3R_ERR_ARG,
              "batch: an SDAINV preconditioner of each segment's matrix");
    B->nrow[s] = h.n;
    B->off[s + 1] = B->off[s] + (h.n + kTile - 1) / kTile * kTile;
    pa[s] = &h;
    pw[s] = &P[s]->host.f[1];
    pz[s] = &P[s]->host.f[0];
    const double rs = p.range_scale > 0 ? p.range_scale
                                        : std::ldexp(1.0, (int)std::floor(std::log2(std::max(1.0, std::sqrt((double)h.n) / 4.0))));
    sc[s] = (float)rs;
    isc[s] = (float)(1.0 / rs);
  }
  const int64_t N = B->off[nseg];
  F3R_CHECK(N / kTile < INT32_MAX, F3R_ERR_RANGE, "batch: too many rows");
  B->N = N;
  B->G = (int)(N / kTile);
  Context *c = ctx.get();
  // block -> segment, segment -> first block and block count
  std::vector<int32_t> bseg(B->G), sb0(nseg), snb(nseg);
  for (int s = 0; s < nseg; ++s) {
    sb0[s] = (int32_t)(B->off[s] / kTile);
    snb[s] = (int32_t)((B->off[s + 1] - B->off[s]) / kTile);
    for (int32_t b = 0; b < snb[s]; ++b) bseg[sb0[s] + b] = s;
    B->snb_max = std::max(B->snb_max, snb[s]);
  }
  auto up32 = [&](const std::vector<int32_t> &v) {
    DevPtr d = dev_alloc(sizeof(int32_t) * std::max<size_t>(1, v.size()));
    F3R_HIP(hipMemcpyAsync(d->p, v.data(), sizeof(int32_t) * v.size(), hipMemcpyHostToDevice, c->stream));
    return d;
  };
  auto upf = [&](const std::vector<float> &v) {
    DevPtr d = dev_alloc(sizeof(float) * std::max<size_t>(1, v.size()));
    F3R_HIP(hipMemcpyAsync(d->p, v.data(), sizeof(float) * v.size(), hipMemcpyHostToDevice, c->stream));
    return d;
  };
  B->bseg = up32(bseg);
  B->sb0 = up32(sb0);
  B->snb = up32(snb);
  B->scale = upf(sc);
  B->iscale = upf(isc);
  F3R_HIP(hipStreamSynchronize(c->stream));
  // the block-diagonal matrices; one row order (sigma = 1) keeps segments contiguous
  const int C = p.C > 0 ? p.C : 64;
  const int K = p.K > 0 ? p.K : 4;
  const bool offsets = p.index != 0;
  // consecutive segments of one matrix (a system's right-hand sides): when
  // every system has the same count NR in {2, 4}, its matrix is laid out
  // once and the SpMVs serve the NR copies together
  {
    std::vector<int> runs;
    for (int s = 0; s < nseg;) {
      int e = s + 1;
      while (e < nseg && A[e].get() == A[s].get()) ++e;
      runs.push_back(e - s);
      s = e;
    }
    const int r0 = runs[0];
    bool same = r0 == 2 || r0 == 4;
    for (int r : runs) same = same && r == r0;
    B->NR = same ? r0 : 1;
  }
  const int NR = B->NR;
  std::vector<const HostCSR *> msys;  // one part per stored matrix
  std::vector<int64_t> moff(1, 0);     // matrix row offsets (whole tiles)
  for (int s = 0; s < nseg; s += NR) {
    msys.push_back(pa[s]);
    moff.push_back(moff.back() + (B->off[s + 1] - B->off[s]));
  }
  const int64_t NM = moff.back();
  // chunk (of C rows) -> shift from matrix row to vector row, copy stride
  auto chunk_tables = [&](DevPtr &dsh, DevPtr &dst) {
    const int64_t nch = (NM + C - 1) / C;
    std::vector<int32_t> sh_(std::max<int64_t>(1, nch)), st_(std::max<int64_t>(1, nch)), sg_(std::max<int64_t>(1, nch));
    for (size_t m = 0; m < msys.size(); ++m) {
      const int64_t seg0 = (int64_t)m * NR;
      for (int64_t ch = moff[m] / C; ch < moff[m + 1] / C; ++ch) {
        sh_[ch] = (int32_t)(B->off[seg0] - moff[m]);
        st_[ch] = (int32_t)(B->off[seg0 + 1] - B->off[seg0]);
        sg_[ch] = (int32_t)seg0;
      }
    }
    dsh = up32(sh_);
    dst = up32(st_);
    B->cseg = up32(sg_);
    F3R_HIP(hipStreamSynchronize(c->stream));  // the host tables are released here
  };
  if (NR > 1) {
    chunk_tables(B->csh, B->cst);
    B->csh16 = B->csh;  // both layouts have chunks of C rows in one order
    B->cst16 = B->cst;
  }
  {
    HostCSR big = NR > 1 ? concat(msys, moff, NM) : concat(pa, B->off, N);
    const std::vector<int64_t> &parts = NR > 1 ? moff : B->off;
    // fp16 copy: K = 8 once rows average 12 entries (a 27-point row then
    // takes 4 slot groups instead of 7; a 7-point row takes 1 either way)
    const int K16 = p.K > 0 ? p.K : (big.nnz() >= (int64_t)12 * big.n ? 8 : 4);
    HostSell hs = build_sell(big, C, 1, K, nullptr, false, offsets, &parts);
    B->sh = upload_sell_shared(c, hs, false);
    B->A64 = upload_sell_values(c, hs, F3R_F64);
    B->A32 = upload_sell_values(c, hs, F3R_F32);
    if (K16 == K) {
      B->sh16 = B->sh;
      B->A16 = upload_sell_values(c, hs, F3R_F16);
    } else {
      HostSell h16 = build_sell(big, C, 1, K16, nullptr, false, offsets, &parts);
      B->sh16 = upload_sell_shared(c, h16, false);
      B->A16 = upload_sell_values(c, h16, F3R_F16);
    }
    if (NR > 1 && !B->lanes) B->quad = build_quads(c, *B->sh, B->A64->as<double>(), moff);
    // k_sell_mr gathers x (fp64 at most) of offset chunks through a buffer
    // resource whose size and byte offsets are 32-bit
    const int64_t bias = std::max(B->sh->off_bias, B->sh16->off_bias);
    F3R_CHECK(NR == 1 || (N + bias) * (int64_t)sizeof(double) < ((int64_t)1 << 31), F3R_ERR_RANGE,
              "batch: the padded rows of all segments exceed the 2^28 a multi-copy SpMV can address");
  }
  // the SDAINV factors: diagonal-only rows as a vector, the rest as CSR rows
  // a system's right-hand sides share its diagonals when they share its
  // preconditioner
  bool share_d = NR > 1;
  for (int s = 0; s < nseg && share_d; ++s) share_d = P[s].get() == P[s - s % NR].get();
  std::vector<int64_t> dshift(nseg, 0);
  if (share_d)
    for (int s = 0; s < nseg; ++s) dshift[s] = moff[s / NR] - B->off[s];
  const HostCSR Wm = concat(pw, B->off, N), Zm = concat(pz, B->off, N);
  auto plain = [](const HostCSR &M, int32_t i) { return M.rptr[i + 1] - M.rptr[i] == 1 && M.idx[M.rptr[i]] == i; };
  auto csr_row = [&](const HostCSR &M, int32_t i) { return M.rptr[i + 1] > M.rptr[i] && !plain(M, i); };
  // k_b_m works t of a Z row's columns out again for each row: that is up to
  // kMRow^2 gathers a row where the two launches have 2 kMRow, so it is for
  // short rows (a 7-point matrix's factors have at most 4 entries a row).
  // Solves of 7-point systems only, every row with 2 to 4 entries: 8 of 48^3
  // rows by 4 right-hand sides 19.8 -> 9.1 ms, by one 6.7 -> 5.6 ms
  bool one = true;
  for (int32_t i = 0; i < (int32_t)N && one; ++i)
    one = Wm.rptr[i + 1] - Wm.rptr[i] <= kMRow && Zm.rptr[i + 1] - Zm.rptr[i] <= kMRow;
  auto factor = [&](const HostCSR &M) {
    std::vector<double> d(N, 0.0);
    std::vector<int32_t> rows, rp(1, 0), cl;
    std::vector<double> vl;
    for (int32_t i = 0; i < M.n; ++i) {
      const int32_t b = M.rptr[i], e = M.rptr[i + 1];
      if (plain(M, i)) {
        d[i] = M.val[b];
      } else if (e > b) {
        d[i] = std::numeric_limits<double>::quiet_NaN();  // marks a CSR row
        if (one) continue;
        rows.push_back(i);
        for (int32_t k = b; k < e; ++k) {
          cl.push_back(M.idx[k]);
          vl.push_back(M.val[k]);
        }
        rp.push_back((int32_t)cl.size());
      }
    }
    std::vector<int32_t> rseg(rows.size());
    for (size_t q = 0; q < rows.size(); ++q)
      rseg[q] = (int32_t)(std::upper_bound(B->off.begin(), B->off.end(), (int64_t)rows[q]) - B->off.begin() - 1);
    if (share_d) {  // segment s's diagonals at matrix rows: those of its first copy
      std::vector<double> ds(NM, 0.0);
      for (int s = 0; s < nseg; s += NR)
        std::copy(d.begin() + B->off[s], d.begin() + B->off[s + 1], ds.begin() + moff[s / NR]);
      d.swap(ds);
    }
    Factor16 F;
    F.dval = upload_values(c, d, F3R_F16);
    F.nr = (int32_t)rows.size();
    F.rows = up32(rows);
    F.rseg = up32(rseg);
    F.rptr = up32(rp);
    F.col = up32(cl);
    F.val = upload_values(c, vl, F3R_F16);
    F3R_HIP(hipStreamSynchronize(c->stream));  // the host arrays above are released here
    return F;
  };
  {
    DevPtr d = dev_alloc(sizeof(int64_t) * std::max(1, nseg));
    F3R_HIP(hipMemcpyAsync(d->p, dshift.data(), sizeof(int64_t) * nseg, hipMemcpyHostToDevice, c->stream));
    F3R_HIP(hipStreamSynchronize(c->stream));
    B->dsh = d;
  }
  B->W = factor(Wm);
  B->Z = factor(Zm);
  if (one) {
    B->mr_copies = share_d ? NR : 1;
    std::vector<int32_t> rows;
    for (int s = 0; s < nseg; s += B->mr_copies)
      for (int64_t i = B->off[s]; i < B->off[s + 1]; ++i)
        if (csr_row(Wm, (int32_t)i) || csr_row(Zm, (int32_t)i)) rows.push_back((int32_t)i);
    const size_t nr = rows.size(), ns = std::max<size_t>(1, nr);
    std::vector<int32_t> meta(4 * ns, 0), wc(ns * kMRow * kMRow, -1);
    std::vector<double> wv(ns * kMRow * kMRow, 0.0), zv(ns * kMRow, 0.0);
    int s = 0;
    for (size_t q = 0; q < nr; ++q) {
      const int32_t i = rows[q];
      while (i >= B->off[s + 1]) ++s;
      const int32_t zb = Zm.rptr[i], ng = Zm.rptr[i + 1] - zb;
      meta[4 * q] = i;
      meta[4 * q + 1] = s;
      meta[4 * q + 2] = (int32_t)(B->off[s + 1] - B->off[s]);
      meta[4 * q + 3] = ng;
      for (int32_t g = 0; g < ng; ++g) {
        zv[q * kMRow + g] = Zm.val[zb + g];
        const int32_t k = Zm.idx[zb + g], wb = Wm.rptr[k], nw = Wm.rptr[k + 1] - wb;
        const size_t at = ((size_t)g * nr + q) * kMRow;
        for (int32_t u = 0; u < nw; ++u) {
          wc[at + u] = Wm.idx[wb + u];
          wv[at + u] = Wm.val[wb + u];
        }
        if (nw == 0) wc[at] = k;  // an empty row: 0 * x
      }
    }
    B->mr_meta = up32(meta);
    B->mr_wc = up32(wc);
    B->mr_wv = upload_values(c, wv, F3R_F16);
    B->mr_z = upload_values(c, zv, F3R_F16);
    B->mr_nr = (int32_t)nr;
    F3R_HIP(hipStreamSynchronize(c->stream));  // the host arrays above are released here
  }
  F3R_HIP(hipStreamSynchronize(c->stream));
  // work space
  B->alloc_level(B->L1, p.m1);
  B->alloc_level(B->L2, p.m2);
  B->alloc_level(B->L3, p.m3);
  {
    bool pow2 = true;
    for (float v : sc) {
      int e = 0;
      pow2 = pow2 && std::frexp(v, &e) == 0.5f;
    }
    B->zh = NR > 1 && pow2;
    if (B->zh) B->Zh3 = dev_alloc(sizeof(half_t) * N * p.m3 + 64);
  }
  auto hv = [&]() { return dev_alloc(sizeof(half_t) * N + 64); };
  B->hin = hv();
  B->hout = hv();
  B->hout2 = hv();
  B->hr = hv();
  B->tmp = hv();
  B->tt = hv();
  B->t2 = hv();
  B->b_int = dev_alloc(sizeof(double) * N);
  B->x_int = dev_alloc(sizeof(double) * N + 64);
  B->partial = dev_alloc(sizeof(double) * (int64_t)B->G * (p.m1 + 1 + 16));
  B->rows = up32(B->nrow);
  B->alloc_pinned();
  B->rich = dev_alloc(sizeof(RichSeg) * nseg);
  F3R_HIP(hipStreamSynchronize(c->stream));
  return B.release();
}

}  // namespace f3r

// ================================================================ C ABI ===
using namespace f3r;

struct f3r_batch_s {
  BatchSolver *b;
};

extern "C" {

int f3r_batch_create(f3r_ctx ctx, int32_t nseg, const f3r_mat *A, const f3r_prec *P, const f3r_params *params,
                     f3r_batch *out) {
  F3R_API_BEGIN
  F3R_CHECK(ctx && A && P && params && out && nseg > 0, F3R_ERR_ARG, "batch_create: null argument");
  *out = nullptr;
  auto c = ctx_of(ctx);
  std::vector<std::shared_ptr<Mat>> am(nseg);
  std::vector<std::shared_ptr<Prec>> pp(nseg);
  for (int s = 0; s < nseg; ++s) {
    F3R_CHECK(A[s] && P[s], F3R_ERR_ARG, "batch_create: null matrix or preconditioner");
    am[s] = mat_of(A[s]);
    pp[s] = prec_of(P[s]);
  }
  BatchSolver *b = batch_create(c, am, pp, *params);
  *out = new f3r_batch_s{b};
  F3R_API_END
}

int f3r_batch_solve(f3r_batch B, const f3r_vec *b, f3r_vec *x, f3r_result *res) {
  F3R_API_BEGIN
  F3R_CHECK(B && b && x && res, F3R_ERR_ARG, "batch_solve: null argument");
  BatchSolver *S = B->b;
  hipStream_t st = S->ctx->stream;
  const int nseg = S->nseg;
  std::vector<double> nrm_b(nseg);
  // kernels reach the callers' vectors on this GPU; those on another are copied
  bool here = true;
  for (int s = 0; s < nseg; ++s) {
    Vec *bv = vec_of(b[s]), *xv = vec_of(x[s]);
    F3R_CHECK(bv && xv && bv->dtype == F3R_F64 && xv->dtype == F3R_F64 && bv->n == S->nrow[s] && xv->n == S->nrow[s],
              F3R_ERR_ARG, "batch_solve: b and x of each segment: fp64 vectors of its matrix size");
    here = here && bv->ctx->device == S->ctx->device && xv->ctx->device == S->ctx->device;
  }
  F3R_HIP(hipStreamSynchronize(st));  // the last solve's reads of the pinned pointers
  for (int s = 0; s < nseg; ++s) {
    S->bp[s] = static_cast<const double *>(vec_of(b[s])->ptr());
    S->xp[s] = static_cast<double *>(vec_of(x[s])->ptr());
  }
  const int32_t *rows = S->rows->as<int32_t>(), *bseg = S->bs(), *sb0 = S->sb0->as<int32_t>();
  if (here) {
    hipLaunchKernelGGL(k_b_take, dim3(S->G), dim3(kBlock), 0, st, S->bp, (const double *const *)S->xp, rows, bseg, sb0,
                       S->b_int->as<double>(), S->x_int->as<double>(), S->partial->as<double>());
  } else {
    F3R_HIP(hipMemsetAsync(S->b_int->p, 0, sizeof(double) * S->N, st));
    F3R_HIP(hipMemsetAsync(S->x_int->p, 0, sizeof(double) * S->N, st));
    for (int s = 0; s < nseg; ++s) {
      const size_t bytes = sizeof(double) * S->nrow[s];
      F3R_HIP(hipMemcpyAsync(S->b_int->as<double>() + S->off[s], S->bp[s], bytes, hipMemcpyDeviceToDevice, st));
      F3R_HIP(hipMemcpyAsync(S->x_int->as<double>() + S->off[s], S->xp[s], bytes, hipMemcpyDeviceToDevice, st));
    }
    hipLaunchKernelGGL(k_b_norm2<double>, dim3(S->G), dim3(kBlock), 0, st, (const double *)S->b_int->as<double>(),
                       S->partial->as<double>());
  }
  // no rotation (j = -1), no Hessenberg column: the norm itself
  hipLaunchKernelGGL(k_b_norm_finish<double>, dim3(nseg), dim3(kBlock), 0, st, (const double *)S->partial->as<double>(),
                     sb0, (const int32_t *)S->snb->as<int32_t>(), S->L1.e->as<double>(), (int64_t)(S->L1.m + 1),
                     (double *)nullptr, (double *)nullptr, (int64_t)0, (double *)nullptr, (int64_t)0, -1, 0,
                     S->L1.inv->as<double>(), S->status);
  F3R_HIP(hipGetLastError());
  nrm_b = S->read_status();
  const auto t0 = std::chrono::steady_clock::now();
  std::vector<f3r_result> r;
  S->solve(nrm_b, r);
  F3R_HIP(hipStreamSynchronize(st));
  const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (here)
    hipLaunchKernelGGL(k_b_give, dim3(S->G), dim3(kBlock), 0, st, (const double *)S->x_int->as<double>(), S->xp, rows,
                       bseg, sb0);
  else
    for (int s = 0; s < nseg; ++s)
      F3R_HIP(hipMemcpyAsync(S->xp[s], S->x_int->as<double>() + S->off[s], sizeof(double) * S->nrow[s],
                             hipMemcpyDeviceToDevice, st));
  F3R_HIP(hipGetLastError());
  for (int s = 0; s < nseg; ++s) {
    r[s].solve_s = secs;
    res[s] = r[s];
  }
  F3R_HIP(hipStreamSynchronize(st));
  F3R_API_END
}

int f3r_batch_info(f3r_batch B, int64_t *rows, int32_t *segments) {
  F3R_API_BEGIN
  F3R_CHECK(B && rows && segments, F3R_ERR_ARG, "batch_info: null argument");
  *rows = B->b->N;
  *segments = B->b->nseg;
  F3R_API_END
}

int f3r_batch_destroy(f3r_batch B) {
  F3R_API_BEGIN
  if (B) {
    (void)hipStreamSynchronize(B->b->ctx->stream);
    delete B->b;
    delete B;
  }
  F3R_API_END
}

}  // extern "C"
