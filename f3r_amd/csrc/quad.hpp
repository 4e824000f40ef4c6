// SpMV of matrices with few distinct values (constant-coefficient stencils,
// and those with a handful of boundary variants): a row's values are 4-bit
// codes into a table of at most 16 numbers, and a lane sums four consecutive
// rows.
//
// What bounds the plain chunk-offset SpMV (sell_kernel.hpp) at 128^3, 27
// points, fp16 is the value stream (56 B a row, 21 to 26 us a launch) and
// behind it the x gathers (27 two-byte gathers a row, 11 us of the address
// unit).  Codes take 16 B a row for every precision together.  Four rows of a
// lane read x in windows: the columns u, u + 1, u + 2 of a stencil line and
// rows r .. r + 3 are six consecutive elements, one or two vector loads in
// place of twelve gathers.  Codes are decoded two at a time through a table of
// all 256 pairs in LDS.  The sums run in slot order with the same products:
// the bits of the plain SpMV.
//
// Measured at 128^3, 27 points (us a launch, plain -> coded): fp16 with the
// level-3 dots 25.9 -> 14.4, fp16 Richardson step 23.4 -> 12.0, fp32 51 -> 18,
// fp64 97 -> 18.
#pragma once

#include <utility>

#include "sell_kernel.hpp"

namespace f3r {

constexpr int kQuadBlock = 256;  // rows of one wavefront
constexpr int kQuadRuns = 32;    // runs (and slots) of a block at most
// the runs of consecutive column offsets of a block's rows: run i covers the
// offsets u[i] .. u[i] + m[i] - 1, m <= 3, ascending
struct QuadTab {
  int32_t nruns, words, kind, nslots;
  int32_t u[kQuadRuns], m[kQuadRuns];
};
// shapes with unrolled sums: 27 points (nine runs of three) and 7 points
// (1, 1, 3, 1, 1); kind 0 loops over its runs
constexpr int kQuad27 = 1, kQuad7 = 2;

template <class V> struct QuadPair {
  V v[2];
};
struct QuadArgs {
  // per 256-row block: table (-1: not coded), first 16-byte unit of its codes,
  // value table (one per system of a batch; the blocks of a workgroup share it)
  const int4 *__restrict__ blk;
  const u32x4 *__restrict__ codes;   // unit w * 64 + l of a block: code word w of the rows of lane l
  const QuadTab *__restrict__ tabs;
  const void *__restrict__ lut;      // 256 pairs of V per value table
  const int32_t *__restrict__ fchunk;  // 64-row chunks of the blocks that are not coded
  int32_t nfb, nfc;                  // workgroups that take them (four each), and their number
  int32_t bias;                      // > -(smallest offset), even
};

// six (or N) consecutive elements of x from index r0 + u, r0 the lane's first row
template <class X, int N> struct QuadWindow {
  X v[N];
  template <class L> static __device__ __forceinline__ L load(__amdgpu_buffer_rsrc_t rs, int vo, int so) {
    if constexpr (sizeof(L) == 16) return __builtin_bit_cast(L, __builtin_amdgcn_raw_buffer_load_b128(rs, vo, so, 0));
    else return __builtin_bit_cast(L, __builtin_amdgcn_raw_buffer_load_b64(rs, vo, so, 0));
  }
  __device__ __forceinline__ QuadWindow(__amdgpu_buffer_rsrc_t rs, int vo, int u, int bias, int cs) {
    constexpr int kBytes = N * (int)sizeof(X);
    if constexpr (sizeof(X) == 2) {
      // dword-aligned loads: one element more when u is odd, dropped by a
      // funnel shift (the parity is the wave's: r0 is a multiple of four)
      const int odd = u & 1;
      const u32x4 d = load<u32x4>(rs, vo, (u - odd + bias) * 2 + cs);
      const unsigned sh = odd ? 16u : 0u;
      uint32_t w[3] = {__builtin_amdgcn_alignbit(d[1], d[0], sh), __builtin_amdgcn_alignbit(d[2], d[1], sh),
                       __builtin_amdgcn_alignbit(d[3], d[2], sh)};
      static_assert(N <= 6, "eight halves are loaded");
      __builtin_memcpy(v, w, kBytes);
    } else {
      const int so = (u + bias) * (int)sizeof(X) + cs;
#pragma unroll
      for (int b = 0; b + 16 <= kBytes; b += 16) {
        const u32x4 d = load<u32x4>(rs, vo, so + b);
        __builtin_memcpy(reinterpret_cast<char *>(v) + b, &d, 16);
      }
      if constexpr (kBytes % 16 == 8) {
        const u32x2 d = load<u32x2>(rs, vo, so + kBytes - 8);
        __builtin_memcpy(reinterpret_cast<char *>(v) + kBytes - 8, &d, 8);
      }
      static_assert(kBytes % 8 == 0, "whole loads");
    }
  }
};

// the windows of one run in NR copies of the vector, `cs` bytes apart
template <class X, int N, int NR> struct QuadWindows {
  QuadWindow<X, N> w[NR];
  template <int... C>
  __device__ __forceinline__ QuadWindows(__amdgpu_buffer_rsrc_t rs, int vo, int u, int bias, int cs,
                                         std::integer_sequence<int, C...>)
      : w{QuadWindow<X, N>(rs, vo, u, bias, C * cs)...} {}
  __device__ __forceinline__ QuadWindows(__amdgpu_buffer_rsrc_t rs, int vo, int u, int bias, int cs)
      : QuadWindows(rs, vo, u, bias, cs, std::make_integer_sequence<int, NR>()) {}
};

// acc[c][q] += the run's M slots (codes of slots T .. T + M - 1 of each row)
template <int T, int M, class X, class ACC, int N, int NR, class Pair>
__device__ __forceinline__ void quad_run(const QuadWindows<X, N, NR> &w, const Pair &pair, ACC (&acc)[NR][4]) {
#pragma unroll
  for (int j = 0; j < M; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const ACC v = (ACC)to_acc(pair(q, T + j));
#pragma unroll
      for (int c = 0; c < NR; ++c) acc[c][q] = fma_<ACC>(v, (ACC)to_acc(w.w[c].v[q + j]), acc[c][q]);
    }
}

// sums of rows r0 .. r0 + 3 of a coded block, for NR copies of x whose rows
// lie cs bytes apart; rs: a buffer resource over x - bias, vo: the byte offset
// of row r0
template <int NR, class V, class X, class ACC>
__device__ __forceinline__ void quad_rows(const QuadArgs &qa, int tab, int unit, const QuadPair<V> *lut,
                                          __amdgpu_buffer_rsrc_t rs, int vo, int cs, ACC (&acc)[NR][4]) {
  typedef const __attribute__((address_space(4))) QuadTab *const_tab;
  const const_tab tb = (const_tab)(qa.tabs + tab);
  const int lane = threadIdx.x & (kWave - 1);
  const u32x4 *__restrict__ cp = qa.codes + unit + lane;
  const int bias = qa.bias;
#pragma unroll
  for (int c = 0; c < NR; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[c][q] = 0;
  using W6 = QuadWindows<X, 6, NR>;
  using W4 = QuadWindows<X, 4, NR>;
  if (tb->kind == kQuad27) {
    u32x4 c[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) c[w] = cp[w * kWave];
    auto pair = [&](int q, int t) { return lut[(c[t / 8][q] >> (8 * (t / 2 % 4))) & 255u].v[t & 1]; };
    // three lines of a plane at a time: their windows in flight together
    auto plane = [&](auto pt) {
      constexpr int P = decltype(pt)::value;
      const W6 w0(rs, vo, tb->u[3 * P], bias, cs), w1(rs, vo, tb->u[3 * P + 1], bias, cs),
          w2(rs, vo, tb->u[3 * P + 2], bias, cs);
      quad_run<9 * P, 3>(w0, pair, acc);
      quad_run<9 * P + 3, 3>(w1, pair, acc);
      quad_run<9 * P + 6, 3>(w2, pair, acc);
    };
    plane(std::integral_constant<int, 0>());
    plane(std::integral_constant<int, 1>());
    plane(std::integral_constant<int, 2>());
  } else if (tb->kind == kQuad7) {
    const u32x4 c = cp[0];
    auto pair = [&](int q, int t) { return lut[(c[q] >> (8 * (t / 2))) & 255u].v[t & 1]; };
    const W4 w0(rs, vo, tb->u[0], bias, cs), w1(rs, vo, tb->u[1], bias, cs), w3(rs, vo, tb->u[3], bias, cs),
        w4(rs, vo, tb->u[4], bias, cs);
    const W6 w2(rs, vo, tb->u[2], bias, cs);
    quad_run<0, 1>(w0, pair, acc);
    quad_run<1, 1>(w1, pair, acc);
    quad_run<2, 3>(w2, pair, acc);
    quad_run<5, 1>(w3, pair, acc);
    quad_run<6, 1>(w4, pair, acc);
  } else {
    int t = 0;
    u32x4 c = cp[0];
    for (int i = 0; i < tb->nruns; ++i) {
      const W6 w(rs, vo, tb->u[i], bias, cs);
      const int m = tb->m[i];
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (j < m) {
          if ((t & 7) == 0) c = cp[(t >> 3) * kWave];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const ACC v = (ACC)to_acc(lut[(c[q] >> (4 * (t & 7))) & 15u].v[0]);
#pragma unroll
            for (int k = 0; k < NR; ++k) acc[k][q] = fma_<ACC>(v, (ACC)to_acc(w.w[k].v[q + j]), acc[k][q]);
          }
          ++t;
        }
    }
  }
}
// nx elements of x behind a fictitious x - bias, and the padding behind them
template <class X>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t quad_rsrc(const X *x, int64_t nx, int bias) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)((uintptr_t)x - (uintptr_t)bias * sizeof(X)), (short)0,
                                           (int)((nx + bias) * (int64_t)sizeof(X)) + 64, kBufferWord3);
}
// the 256-row block of this wave, and its workgroup's value table into LDS
template <class V>
__device__ __forceinline__ int quad_block(const SellArgs &a, const QuadArgs &qa, QuadPair<V> *lut) {
  static_assert(kBlock == 256, "a thread per pair of the table");
  // XCD k takes the k-th contiguous eighth of the rows (xcd_block)
  const int g = (int)gridDim.x - qa.nfb, b0 = (int)blockIdx.x - qa.nfb;
  const int b = g % kXcds ? b0 : b0 % kXcds * (g / kXcds) + b0 / kXcds;
  lut[threadIdx.x] = static_cast<const QuadPair<V> *>(qa.lut)[qa.blk[b * kWavesPerBlock].z * 256 + threadIdx.x];
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(b * kWavesPerBlock + (int)threadIdx.x / kWave);
}

// An epilogue (sell_kernel.hpp) may also provide, for four consecutive rows of
// a lane, Pre4, pre4(r0) and row4(r0, acc, pre, state) with vector accesses,
// and the host's vec4(), true when its pointers allow them (aligned to 4
// elements).
template <class Epi, class = void> struct HasRow4 : std::false_type {};
template <class Epi> struct HasRow4<Epi, std::void_t<typename Epi::Pre4>> : std::true_type {};

template <class V, class X, class ACC, int K, class Epi>
__global__ __launch_bounds__(kBlock) void k_quad(SellArgs a, QuadArgs qa, const V *__restrict__ val,
                                                 const X *__restrict__ x, Epi epi, int vec) {
  __shared__ QuadPair<V> lut[256];
  typename Epi::State st{};
  const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if ((int)blockIdx.x < qa.nfb) {
    // rows of the blocks that are not coded: a chunk per wave, a row per lane
    const int c = (int)blockIdx.x * kWavesPerBlock + wave;
    if (c < qa.nfc) {
      const int r = qa.fchunk[c] * 64 + lane;
      if (r < a.n) {
        const typename Epi::Pre p = epi.pre(r);
        epi.row(r, sell_row<V, X, ACC, K>(a, val, x, r), p, st);
      }
    }
  } else {
    const int blk = quad_block<V>(a, qa, lut);
    if ((int64_t)blk * kQuadBlock < a.n) {
      const int4 e = qa.blk[blk];
      const int tab = __builtin_amdgcn_readfirstlane(e.x), unit = __builtin_amdgcn_readfirstlane(e.y);
      if (tab >= 0) {
        const int r0 = blk * kQuadBlock + 4 * lane;
        const __amdgpu_buffer_rsrc_t rs = quad_rsrc<X>(x, a.n, qa.bias);
        // lanes past the last row read where the last row's lane does
        const int vo = (r0 < a.n ? r0 : (a.n - 1) & ~3) * (int)sizeof(X);
        ACC acc[1][4];
        bool done = false;
        if constexpr (HasRow4<Epi>::value) {
          if (vec && (blk + 1) * kQuadBlock <= a.n) {
            const typename Epi::Pre4 p = epi.pre4(r0);
            quad_rows<1, V, X, ACC>(qa, tab, unit, lut, rs, vo, 0, acc);
            epi.row4(r0, acc[0], p, st);
            done = true;
          }
        }
        if (!done) {
          quad_rows<1, V, X, ACC>(qa, tab, unit, lut, rs, vo, 0, acc);
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (r0 + q < a.n) epi.row(r0 + q, acc[0][q], epi.pre(r0 + q), st);
        }
      }
    }
  }
  epi.finish(st);
}

// workgroups of k_quad
inline int quad_blocks(const SellArgs &a, const QuadArgs &qa) {
  return qa.nfb + (int)(((int64_t)a.n + kBlock * 4 - 1) / (kBlock * 4));
}

template <int K, class V, class X, class ACC, class Epi>
inline void launch_quad(const SellArgs &a, const QuadArgs &qa, const V *val, const X *x, Epi epi, hipStream_t st) {
  int vec = 0;
  if constexpr (HasRow4<Epi>::value) vec = epi.vec4() ? 1 : 0;
  hipLaunchKernelGGL((k_quad<V, X, ACC, K, Epi>), dim3(quad_blocks(a, qa)), dim3(kBlock), 0, st, a, qa, val, x, epi,
                     vec);
}

// the codes of a matrix on the device, shared by its precisions
struct QuadSet {
  DevPtr blk, codes, tabs, fchunk, lut64, lut32, lut16;
  int32_t nfb = 0, nfc = 0, bias = 0;
  // what one product reads of the matrix: codes, and the value slots and
  // column indices of the chunks that are not coded
  int64_t code_bytes = 0, plain_slots = 0, plain_idx = 0;
  double algo_bytes(int32_t n, int sv, int sx, int sy) const {
    return (double)code_bytes + (double)plain_slots * sv + 4.0 * (double)plain_idx + (double)n * (sx + sy);
  }
  template <class V> QuadArgs args() const {
    const DevPtr &l = sizeof(V) == 8 ? lut64 : sizeof(V) == 4 ? lut32 : lut16;
    return {blk->as<int4>(), codes->as<u32x4>(), tabs->as<QuadTab>(), l->p, fchunk->as<int32_t>(), nfb, nfc, bias};
  }
};
// Fewer rows than this leave k_quad's waves (256 rows each) too few for the
// GPU's 1024 SIMDs to hide their latency.
constexpr int32_t kQuadMinRows = 1 << 17;
// null when the matrix has more than 16 distinct values (0 among them), its
// chunks are not 64 rows of offset form, or it has too few rows.  systems: the
// first rows of the diagonal blocks with value tables of their own (multiples
// of 1024; empty: one table), the last entry the end
std::shared_ptr<QuadSet> build_quads(Context *c, const SellShared &sh, const double *val64,
                                     const std::vector<int64_t> &systems = {});

}  // namespace f3r
