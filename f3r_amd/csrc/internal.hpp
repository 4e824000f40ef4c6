// Declarations shared between the translation units of libf3r_amd.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "sell_kernel.hpp"

namespace f3r {

// Innermost preconditioner: SDAINV (M = Z D^-1 W^T as two SELL SpMVs, or two
// diagonal scalings when both factors are diagonal) or ILU(0) (level-scheduled
// triangular solves).  Values in `dtype`, sums in fp32 for fp16 / fp32 data.
struct Prec {
  std::shared_ptr<Context> ctx;
  int kind = 0;  // 0 SDAINV, 1 ILU(0)
  int dtype = F3R_F16;
  double tol = 0.1, acc = 1.0;
  int32_t n = 0;
  int where = 0;  // factors built: 0 host, 1 device, 2 device asked, host ran
  HostFactors host;
  DevPtr tmp;
  // SDAINV
  std::shared_ptr<Mat> W, Z;  // W holds W^T (rows w_i), Z holds Z D^-1
  bool diag = false;
  DevPtr dw, dz;              // diagonals when `diag`
  DevPtr dwz;                 // fp16 only: (dw[i], dz[i]) interleaved, one 4-byte load per row
  // at most 4 diagonals in each factor: band form (kBand values a row, W's
  // then Z's)
  DevPtr bwz;
  int32_t bow[4] = {}, boz[4] = {};
  // ILU(0)
  std::vector<int32_t> l_lptr, u_lptr;  // level pointers into *_rows
  DevPtr l_rows, u_rows, l_rptr, l_idx, l_val, u_rptr, u_idx, u_val, u_dinv;
  // block-Jacobi split with at least kBjBlockKernel blocks: rows grouped by
  // block, one workgroup per block (bj_groups of them)
  int32_t bj_blocks = 0, bj_groups = 0;
  DevPtr lb_rows, lb_ptr, lb_start, ub_rows, ub_ptr, ub_start;
  // fused L+U solve with the block's vector in LDS (bj_R entries per record;
  // 0: not used), on bj_waves wavefronts: the record streams and, per block,
  // its first segment and its records
  int32_t bj_R = 0, bj_waves = 1;
  size_t bj_lds = 0;
  DevPtr bj_rec, bj_blk;
  // its kernels take the entry themselves (no vector for its result needed)
  bool has_fused_entry() const { return kind == 0 || bj_R != 0; }
};
// LDS the fused block-Jacobi kernel may take for a block's vector
constexpr size_t kBjLdsBytes = 64 * 1024;
// fewer diagonal blocks than this: one launch per level instead (a block
// per workgroup would leave most of the GPU idle)
constexpr int32_t kBjBlockKernel = 32;

// One application of M inside the innermost level, with the element-wise work
// around it: the entry from the basis vector above (normalised in passing and
// converted to the storage type S) and the weighted update of the Richardson
// iterate.  Every kind of M does these in its own kernels, so a call costs no
// launch (2.4 to 4.9 us each at 64^3 to 96^3) beyond M's own.
// S: storage and type of M; F: type of the basis vector (F = S outside the
// HALF build, where nothing is scaled or converted).
template <class S, class F> struct MIo {
  // input: `in`, or the entry from `raw`
  const S *in = nullptr;
  const F *raw = nullptr;
  // block sums of ||raw||^2 left by the Arnoldi step that made it (null: raw
  // is normalised); every block adds them up itself, the first one also
  // writes the norm to its place in the Hessenberg column
  const F *npart = nullptr;
  int nparts = 0;
  F *hnorm = nullptr;
  F *vout = nullptr;       // the normalised vector (with npart; not raw: rows gather raw meanwhile)
  F s = 1;                 // hin = S(raw * inv * s)
  S *hin = nullptr;        // null with S = F: the normalised vector is M's input
  // output: x = M in; out = x, S(x * w) with `w`, or S(fma(w, x, add)) with
  // `add` too; outf (instead of out): the last, in F and unscaled
  S *out = nullptr;
  const double *w = nullptr;
  const S *add = nullptr;
  F *outf = nullptr;
  F inv_s = 1;
  S *scratch = nullptr;  // a vector of S for kinds of M without fused kernels (with add)
};
template <class S, class F> void prec_apply_io(Prec *P, const MIo<S, F> &io, hipStream_t st);
// the entry alone: h = S(raw * inv * s) where h is not null, and vout
template <class S, class F>
void prec_entry(const MIo<S, F> &io, int64_t n, S *h, int num_cu, hipStream_t st);

// the entry of one element (constructed by every thread of a block: the
// block adds up the norm's partial sums; WIDE: a block of more than kBlock threads)
template <class S, class F> struct MEntry {
  F iv, s;
  bool has_inv;
  template <class WIDE = std::false_type>
  __device__ explicit MEntry(const MIo<S, F> &io, WIDE = WIDE()) : iv(1), s(io.s), has_inv(io.npart != nullptr) {
    if (!has_inv) return;
    const F nv = sqrt(parts_sum<F, WIDE::value>(io.npart, io.nparts));
    if (blockIdx.x == 0 && threadIdx.x == 0) *io.hnorm = nv;
    iv = (F)1 / nv;
  }
  __device__ __forceinline__ F norm(F v) const { return has_inv ? v * iv : v; }
  __device__ __forceinline__ S store(F v) const {  // v normalised
    if constexpr (std::is_same<S, F>::value) return v; else return cvt<S>(v * s);
  }
  __device__ __forceinline__ auto operator()(F v) const { return to_acc(store(norm(v))); }
};
// the output of one element
template <class S, class F> struct MExit {
  using A = typename Acc<S>::type;
  S *out;
  const S *add;
  F *outf;
  A w;
  F inv_s;
  bool weighted;
  __device__ explicit MExit(const MIo<S, F> &io)
      : out(io.out), add(io.add), outf(io.outf), w(io.w ? (A)*io.w : (A)1), inv_s(io.inv_s), weighted(io.w != nullptr) {}
  __device__ __forceinline__ S pre(int64_t r) const { return add ? add[r] : S(0); }
  __device__ __forceinline__ S value(S x, S ad) const {
    if (!weighted) return x;
    return add ? cvt<S>(fma_<A>(w, to_acc(x), to_acc(ad))) : cvt<S>(to_acc(x) * w);
  }
  __device__ __forceinline__ void put(int64_t r, S x, S ad) const {
    const S h = value(x, ad);
    if (outf) outf[r] = (F)to_acc(h) * inv_s;
    else out[r] = h;
  }
};
// a row's diagonal factors (w, z): one 32-bit word in fp16
template <class S> struct DiagWZ {
  const S *w = nullptr, *z = nullptr;
  struct V {
    S w, z;
  };
  __device__ __forceinline__ V at(int64_t r) const { return {w[r], z[r]}; }
};
template <> struct DiagWZ<half_t> {
  const uint32_t *wz = nullptr;
  struct V {
    half_t w, z;
  };
  static __device__ __forceinline__ V unpack(uint32_t v) {
    return {__builtin_bit_cast(half_t, (uint16_t)(v & 0xffffu)), __builtin_bit_cast(half_t, (uint16_t)(v >> 16))};
  }
  __device__ __forceinline__ V at(int64_t r) const { return unpack(wz[r]); }
};
template <class S> inline DiagWZ<S> diag_wz(const Prec &P) {
  if constexpr (std::is_same<S, half_t>::value) return {P.dwz->template as<uint32_t>()};
  else return {P.dw->template as<S>(), P.dz->template as<S>()};
}
// z (w x) of a row, each product rounded to S
template <class S> __device__ __forceinline__ S diag_apply(const typename DiagWZ<S>::V &d, S x) {
  using A = typename Acc<S>::type;
  const S t = cvt<S>(fma_<A>(to_acc(d.w), to_acc(x), (A)0));
  return cvt<S>(fma_<A>(to_acc(d.z), to_acc(t), (A)0));
}

std::shared_ptr<Context> ctx_create(int device);
// The context's landing slot for one fp64 result of a kernel: arm_scalar
// before the launch gives the address the kernel stores to (one 8-byte
// system-scope store), wait_scalar returns the value.
double *arm_scalar(Context *c);
double wait_scalar(Context *c);
SellArgs sell_args(const SellShared &sh, bool with_perm);
DevPtr upload_values(Context *ctx, const std::vector<double> &v, int dtype);
HostCSR permute_csr(const HostCSR &M, const std::vector<int32_t> &perm);
void prec_build_device(Prec *P, const std::vector<int32_t> *perm, int32_t C, int32_t K, bool offsets = true);
void prec_apply_raw(Prec *P, const void *in, void *out, hipStream_t st);
void vec_copy(Vec *s, Vec *d);
// dot product of two device arrays (fp16 data summed in fp32), host result
double dot_raw(Context *c, int da, const void *a, int db, const void *b, int64_t n);

#define F3R_API_BEGIN try {
#define F3R_API_END                                   \
  }                                                   \
  catch (const f3r::Error &e) {                       \
    f3r::set_error(e.msg);                            \
    return e.status;                                  \
  }                                                   \
  catch (const std::bad_alloc &) {                    \
    f3r::set_error("host allocation failed");         \
    return F3R_ERR_ALLOC;                             \
  }                                                   \
  catch (const std::exception &e) {                   \
    f3r::set_error(e.what());                         \
    return F3R_ERR_ARG;                               \
  }                                                   \
  return F3R_OK;

}  // namespace f3r

struct f3r_ctx_s;
struct f3r_vec_s;
struct f3r_mat_s;
struct f3r_prec_s;
namespace f3r {
std::shared_ptr<Context> ctx_of(f3r_ctx c);
Vec *vec_of(f3r_vec v);
std::shared_ptr<Mat> mat_of(f3r_mat m);
std::shared_ptr<Prec> prec_of(f3r_prec p);
f3r_prec wrap_prec(std::shared_ptr<Prec> p);  // new handle owning a reference
f3r_vec wrap_vec(const Vec &v);                // new handle of a vector (view)
void release_vec(f3r_vec v);
// device build of a SELL-C-sigma layout from a device CSR (build.hip), the
// columns renumbered into the sorted order when `renumber`; false (nothing
// built) when a chunk or a sigma window is too long for the on-chip sorts
bool build_sell_device(Context *c, const HostCSR &A, const int32_t *d_rptr, const int32_t *d_col,
                       const double *d_val, int32_t C, int32_t sigma, int32_t K, bool offsets, bool renumber,
                       std::shared_ptr<SellShared> &sh, DevPtr &sval);
// device factorisations (factor.hip), bit-identical to sdainv_host /
// ilu0_host; false (F untouched) when a row outgrows the device capacity
bool sdainv_device(Context *c, const HostCSR &A, const int32_t *d_rptr, const int32_t *d_col, const double *d_val,
                   double tol, double acc, HostFactors &F);
bool ilu0_device(Context *c, const HostCSR &A, const int32_t *d_rptr, const int32_t *d_col, const double *d_val,
                 int32_t blocks, double acc, HostFactors &F);
// fp64 slot values on the device -> dtype (correctly rounded)
DevPtr cast_values_device(Context *c, const DevPtr &v64, int64_t n, int dtype);
}  // namespace f3r
