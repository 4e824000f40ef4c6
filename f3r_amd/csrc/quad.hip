// Builds the 4-bit value codes of quad.hpp from a chunk-offset SELL layout on
// the device:
//   1. the distinct fp64 values of all slots, at most 16 (a first pass over a
//      sample, so that a matrix of varying coefficients is turned down in a
//      few microseconds)
//   2. host: per 256 rows (four chunks) the union of their column offsets,
//      split into runs of consecutive offsets; equal unions share a table
//   3. each row's codes, in the order of its block's table
#include <algorithm>
#include <cstring>
#include <map>

#include "common.hpp"
#include "internal.hpp"
#include "quad.hpp"

namespace f3r {
namespace {

constexpr unsigned long long kEmpty = 0x7ff8f3f3f3f3f3f4ULL;  // a NaN: no matrix value that is coded
struct Dict {
  unsigned long long v[16];
  int overflow;
};

__global__ void k_dict_init(Dict *dicts) {
  Dict *d = dicts + blockIdx.x;
  if (threadIdx.x < 16) d->v[threadIdx.x] = threadIdx.x == 0 ? 0ull : kEmpty;
  if (threadIdx.x == 0) d->overflow = 0;
}
// about `samples` evenly spaced values (0: all) of each system's slots into
// its dictionary; system g: slots sptr[g] .. sptr[g + 1] - 1
__global__ __launch_bounds__(256) void k_dict(const int32_t *__restrict__ sptr, int samples,
                                              const double *__restrict__ vals, Dict *dicts) {
  Dict *d = dicts + blockIdx.y;
  const double *__restrict__ val = vals + sptr[blockIdx.y];
  const int64_t n = sptr[blockIdx.y + 1] - sptr[blockIdx.y];
  const int64_t stride = samples > 0 && n > samples ? n / samples : 1;
  __shared__ unsigned long long seen[16];
  if (threadIdx.x < 16) seen[threadIdx.x] = __hip_atomic_load(&d->v[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  for (int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) * stride; i < n;
       i += (int64_t)gridDim.x * blockDim.x * stride) {
    const double f = val[i];
    const unsigned long long u = __double_as_longlong(f);
    bool found = false;
    for (int k = 0; k < 16; ++k) found = found || seen[k] == u;
    if (found) continue;
    if (__hip_atomic_load(&d->overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    if (f != f) {  // no NaN
      __hip_atomic_store(&d->overflow, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    int k = 0;
    for (; k < 16; ++k) {
      const unsigned long long old = atomicCAS(&d->v[k], kEmpty, u);
      if (old == kEmpty || old == u) break;
    }
    if (k == 16) {
      __hip_atomic_store(&d->overflow, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    seen[k] = u;  // the same value from every thread of the block
  }
}

// one row per thread: codes of the slots of its block's table.  map[(table *
// 4 + chunk of the block) * kQuadRuns + t]: the chunk's slot of table slot t
__global__ __launch_bounds__(256) void k_quad_codes(int32_t n, int32_t K, const int32_t *__restrict__ cptr,
                                                    const int32_t *__restrict__ cwidth, const double *__restrict__ val,
                                                    const int4 *__restrict__ blk, const QuadTab *__restrict__ tabs,
                                                    const int8_t *__restrict__ map, const Dict *__restrict__ dicts,
                                                    uint32_t *__restrict__ codes) {
  __shared__ unsigned long long dv[16];
  const int b = blockIdx.x, r = b * kQuadBlock + threadIdx.x, j = threadIdx.x;
  const int4 e = blk[b];
  if (threadIdx.x < 16) dv[threadIdx.x] = dicts[e.z].v[threadIdx.x];
  __syncthreads();
  if (e.x < 0) return;
  const QuadTab &tb = tabs[e.x];
  const int s = r / 64, tc = n - s * 64 < 64 ? n - s * 64 : 64;
  const int8_t *mp = map + ((int64_t)e.x * 4 + (s & 3)) * kQuadRuns;
  for (int w = 0; w < tb.words; ++w) {
    uint32_t word = 0;
    for (int t = 8 * w; t < 8 * w + 8 && t < tb.nslots; ++t) {
      const int cs = r < n ? mp[t] : -1;
      if (cs < 0) continue;
      const unsigned long long u =
          __double_as_longlong(val[chunk_slot_pos(cptr[s], cwidth[s], tc, r - s * 64, cs, K)]);
      uint32_t code = 0;
      for (int k = 1; k < 16; ++k) code = dv[k] == u ? (uint32_t)k : code;
      word |= code << (4 * (t & 7));
    }
    codes[((int64_t)e.y + w * 64 + j / 4) * 4 + j % 4] = word;
  }
}

template <class V> __global__ void k_quad_lut(const Dict *__restrict__ dicts, QuadPair<V> *__restrict__ luts) {
  const Dict *d = dicts + blockIdx.x;
  QuadPair<V> *lut = luts + 256 * blockIdx.x;
  const int i = threadIdx.x;
  auto at = [&](int k) {
    const unsigned long long u = d->v[k];
    return u == kEmpty ? V(0) : cvt<V>(__longlong_as_double((long long)u));
  };
  lut[i].v[0] = at(i & 15);
  lut[i].v[1] = at(i >> 4);
}

DevPtr upload(Context *c, const void *p, size_t bytes) {
  DevPtr d = dev_alloc(std::max<size_t>(bytes, 16));
  if (bytes) F3R_HIP(hipMemcpyAsync(d->p, p, bytes, hipMemcpyHostToDevice, c->stream));
  return d;
}

}  // namespace

std::shared_ptr<QuadSet> build_quads(Context *c, const SellShared &sh, const double *val64,
                                     const std::vector<int64_t> &systems) {
  if (sh.n < kQuadMinRows || sh.C != 64 || !sh.iptr || sh.lanes != 1 || sh.n >= (1 << 27)) return nullptr;
  hipStream_t st = c->stream;
  const int32_t nch = sh.nchunks, nb = (sh.n + kQuadBlock - 1) / kQuadBlock;
  std::vector<int64_t> sys = systems;
  if (sys.empty()) sys = {0, sh.n};
  const int ng = (int)sys.size() - 1;
  std::vector<int32_t> cptr(nch + 1), sptr;
  F3R_HIP(hipMemcpyAsync(cptr.data(), sh.cptr->p, 4 * ((size_t)nch + 1), hipMemcpyDeviceToHost, st));
  F3R_HIP(hipStreamSynchronize(st));
  for (int64_t r : sys) sptr.push_back(cptr[(r + 63) / 64]);
  DevPtr dsptr = upload(c, sptr.data(), 4 * sptr.size());
  DevPtr dict = dev_alloc(sizeof(Dict) * ng);
  Dict *dd = dict->as<Dict>();
  const int32_t *sp = dsptr->as<int32_t>();
  hipLaunchKernelGGL(k_dict_init, dim3(ng), dim3(64), 0, st, dd);
  hipLaunchKernelGGL(k_dict, dim3(1, ng), dim3(256), 0, st, sp, 1024, val64, dd);
  hipLaunchKernelGGL(k_dict, dim3(std::max(1, 2048 / ng), ng), dim3(256), 0, st, sp, 0, val64, dd);
  F3R_HIP(hipGetLastError());
  std::vector<Dict> hd(ng);
  F3R_HIP(hipMemcpyAsync(hd.data(), dd, sizeof(Dict) * ng, hipMemcpyDeviceToHost, st));
  F3R_HIP(hipStreamSynchronize(st));
  int64_t coded = 0;
  for (int g = 0; g < ng; ++g) coded += hd[g].overflow ? 0 : sys[g + 1] - sys[g];
  if (coded * 16 < (int64_t)sh.n * 15) return nullptr;
  std::vector<int32_t> iptr(nch), cw(nch), coff(sh.coff->bytes / 4);
  F3R_HIP(hipMemcpyAsync(iptr.data(), sh.iptr->p, 4 * (size_t)nch, hipMemcpyDeviceToHost, st));
  F3R_HIP(hipMemcpyAsync(cw.data(), sh.cwidth->p, 4 * (size_t)nch, hipMemcpyDeviceToHost, st));
  F3R_HIP(hipMemcpyAsync(coff.data(), sh.coff->p, 4 * coff.size(), hipMemcpyDeviceToHost, st));
  F3R_HIP(hipStreamSynchronize(st));
  // whole workgroups: the last one's waves read their blocks' entries too
  std::vector<int4> blk((nb + kWavesPerBlock - 1) / kWavesPerBlock * kWavesPerBlock, int4{-1, 0, 0, 0});
  int g = 0;
  std::vector<QuadTab> tabs;
  std::vector<int8_t> map;
  std::vector<int32_t> fchunk;
  std::map<std::vector<int32_t>, int> known;  // table starts of a block's chunks -> table
  int32_t umin = 0;
  int64_t units = 0;
  std::vector<int32_t> key, last;
  int last_tab = -1;
  for (int32_t b = 0; b < nb; ++b) {
    const int32_t s0 = b * 4, s1 = std::min(nch, s0 + 4);
    while (sys[g + 1] <= (int64_t)b * kQuadBlock) ++g;
    blk[b].z = g;
    bool ok = !hd[g].overflow;
    key.clear();
    for (int32_t s = s0; s < s1; ++s) {
      const bool none = chunk_slots(cw[s], sh.K) == 0;  // rows without entries (a batch's padding)
      ok = ok && (none || iptr[s] < 0);
      key.push_back(none ? 0 : iptr[s]);
      key.push_back(cw[s]);
    }
    int tab = -1;
    if (ok && key == last) {
      tab = last_tab;
    } else if (ok) {
      auto it = known.find(key);
      if (it != known.end()) {
        tab = it->second;
      } else {
        // a chunk's table ascends up to its padding (offset 0, value 0)
        std::vector<std::vector<int32_t>> us;
        std::vector<int32_t> all;
        for (int32_t s = s0; s < s1; ++s) {
          const int32_t w = chunk_slots(cw[s], sh.K);
          const int32_t *o = coff.data() + (w ? -iptr[s] - 1 : 0);
          int32_t t = w ? 1 : 0;
          while (t < w && o[t] > o[t - 1]) ++t;
          us.emplace_back(o, o + t);
          all.insert(all.end(), us.back().begin(), us.back().end());
        }
        std::sort(all.begin(), all.end());
        all.erase(std::unique(all.begin(), all.end()), all.end());
        if ((int)all.size() <= kQuadRuns) {
          QuadTab q{};
          q.nslots = (int32_t)all.size();
          const int32_t words = (q.nslots + 7) / 8;
          q.words = words == 3 ? 4 : std::max(1, words);
          for (size_t t = 0; t < all.size(); ++t) {
            if (q.nruns > 0 && q.m[q.nruns - 1] < 3 && q.u[q.nruns - 1] + q.m[q.nruns - 1] == all[t]) {
              ++q.m[q.nruns - 1];
            } else {
              q.u[q.nruns] = all[t];
              q.m[q.nruns++] = 1;
            }
          }
          auto runs = [&](std::vector<int32_t> m) { return std::equal(m.begin(), m.end(), q.m); };
          if (q.nruns == 9 && runs(std::vector<int32_t>(9, 3))) q.kind = kQuad27;
          if (q.nruns == 5 && runs({1, 1, 3, 1, 1})) q.kind = kQuad7;
          tab = (int)tabs.size();
          tabs.push_back(q);
          for (int k = 0; k < 4; ++k)
            for (int t = 0; t < kQuadRuns; ++t) {
              int8_t slot = -1;
              if (k < (int)us.size() && t < q.nslots) {
                auto f = std::lower_bound(us[k].begin(), us[k].end(), all[t]);
                if (f != us[k].end() && *f == all[t]) slot = (int8_t)(f - us[k].begin());
              }
              map.push_back(slot);
            }
        }
        known[key] = tab;
      }
    }
    if (ok) {
      last = key;
      last_tab = tab;
    }
    // every row of the block reads every offset of the table, within its system
    if (tab >= 0) {
      const QuadTab &q = tabs[tab];
      const int64_t r0 = (int64_t)b * kQuadBlock, r1 = std::min<int64_t>(sh.n, r0 + kQuadBlock);
      const int32_t lo = q.u[0], hi = q.nruns ? q.u[q.nruns - 1] + q.m[q.nruns - 1] - 1 : 0;
      if (r0 + lo < sys[g] || r1 - 1 + hi >= sys[g + 1]) tab = -1;
      else umin = std::min(umin, lo);
    }
    if (tab >= 0) {
      blk[b] = int4{tab, (int32_t)units, g, 0};
      units += (int64_t)tabs[tab].words * 64;
    } else {
      for (int32_t s = s0; s < s1; ++s) fchunk.push_back(s);
    }
  }
  // worth it when nearly all rows are coded
  if ((int64_t)fchunk.size() * 16 > nch) return nullptr;
  auto q = std::make_shared<QuadSet>();
  q->bias = (-umin + 1 + 7) / 8 * 8;
  q->nfc = (int32_t)fchunk.size();
  q->nfb = ((q->nfc + kWavesPerBlock - 1) / kWavesPerBlock + kXcds - 1) / kXcds * kXcds;  // the rest keep their XCDs
  q->code_bytes = units * (int64_t)sizeof(u32x4);
  for (int32_t s : fchunk) {
    q->plain_slots += cptr[s + 1] - cptr[s];
    if (iptr[s] >= 0) q->plain_idx += cptr[s + 1] - cptr[s];
  }
  q->blk = upload(c, blk.data(), sizeof(int4) * blk.size());
  q->tabs = upload(c, tabs.data(), sizeof(QuadTab) * tabs.size());
  q->fchunk = upload(c, fchunk.data(), 4 * fchunk.size());
  DevPtr dmap = upload(c, map.data(), map.size());
  q->codes = dev_alloc(sizeof(u32x4) * std::max<int64_t>(units, 1));
  hipLaunchKernelGGL(k_quad_codes, dim3(nb), dim3(kQuadBlock), 0, st, sh.n, sh.K, sh.cptr->as<int32_t>(),
                     sh.cwidth->as<int32_t>(), val64, q->blk->as<int4>(), q->tabs->as<QuadTab>(),
                     (const int8_t *)dmap->as<int8_t>(), (const Dict *)dd, q->codes->as<uint32_t>());
  q->lut64 = dev_alloc(256 * sizeof(QuadPair<double>) * ng);
  q->lut32 = dev_alloc(256 * sizeof(QuadPair<float>) * ng);
  q->lut16 = dev_alloc(256 * sizeof(QuadPair<half_t>) * ng);
  hipLaunchKernelGGL(k_quad_lut<double>, dim3(ng), dim3(256), 0, st, (const Dict *)dd, q->lut64->as<QuadPair<double>>());
  hipLaunchKernelGGL(k_quad_lut<float>, dim3(ng), dim3(256), 0, st, (const Dict *)dd, q->lut32->as<QuadPair<float>>());
  hipLaunchKernelGGL(k_quad_lut<half_t>, dim3(ng), dim3(256), 0, st, (const Dict *)dd, q->lut16->as<QuadPair<half_t>>());
  F3R_HIP(hipGetLastError());
  F3R_HIP(hipStreamSynchronize(st));  // the host tables are released here
  return q;
}

}  // namespace f3r
