// QuadDecomposition::decompose (QuadDecomposition.cpp:311-445) for meshes
// that live in HBM.  Its data-parallel half runs on the device:
//   - the half-edges (QuadDecomposition.cpp:355-365): one key (from, to) per
//     triangle edge, radix-sorted stably over its significant bits with the
//     insertion number 3t + k as the value, so each directed edge's list is
//     contiguous and in the order the reference appends to it;
//   - per half-edge, the start of its reverse edge's list (a binary search);
//   - the candidate graph (:366-384): the reference links triangle t, edge by
//     edge, with the triangles already listed on the reverse edge (those
//     inserted up to t's last edge) that pass the 0.5-unit plane test
//     (:326-343, with the host CPU's RSQRTPS from its table and DPPS's
//     summation order).  A link enters both triangles' lists, so t's list
//     holds first its own links and then those that later triangles make with
//     it, by their insertion numbers: exactly the entries of its three reverse
//     lists from there on, merged.  One thread per triangle gathers its list in
//     that order (a count pass, a scan, a fill pass), so nothing is sorted;
//   - the quads (:392-441), once the matching is known: one thread per
//     triangle, positions from a scan of which triangles write.
// The matching itself (:28-309) is a sequential augmenting-path search with
// blossom shrinking; it runs on the host (rz_quad.cpp) over the adjacency
// lists copied back, and the partners are copied to the device.
//
// Bound by the host: 1.3 ms of matching for the city mesh's 807 k list
// entries, then the copies (pinned, so 57 GB/s) and the key sort.  Emitting the
// links in order and sorting them by (triangle, place) took a second 64-bit
// radix sort and its buffers; with it, and with every buffer allocated per
// call, rz_prepare_mesh_device took 12.3 ms for that mesh, and takes 3.2 ms.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <cstdint>
#include <new>
#include <vector>

#include "rasterizer_amd.h"
#include "rz_kernels.h"
#include "rz_quad.h"
#include "rz_scratch.h"
#include "rz_x86.h"

namespace rzd {

namespace {

constexpr uint32_t kQdBlock = 256;
uint32_t qd_grid(size_t n) { return uint32_t((n + kQdBlock - 1) / kQdBlock); }

struct QdParams {
  const uint32_t* idx;  // 3 per triangle
  const float4* vertices;
  uint32_t nTri, nHalf;
  uint32_t bits;         // of a vertex number: key = from << bits | to
  const uint64_t* keys;  // sorted half-edge keys
  const uint32_t* seqs;  // their insertion numbers
  const uint32_t* revFirst;  // per insertion number: first entry of the reverse edge's list
  const uint32_t* rsq;       // 8192-entry RSQRTPS table
  uint32_t* degree;          // count pass: entries of each triangle's list
  const uint32_t* start;     // fill pass: its first entry
  int* adj;                  // fill pass: the lists
  uint32_t* bad;
};

__device__ __forceinline__ uint64_t edge_key(uint32_t from, uint32_t to, uint32_t bits) {
  return (uint64_t(from) << bits) | to;
}
__device__ __forceinline__ uint32_t next3(uint32_t k) { return k == 2u ? 0u : k + 1u; }
__device__ __forceinline__ uint32_t prev3(uint32_t k) { return k == 0u ? 2u : k - 1u; }

// Both triangles (v0, v1, v2) and (v2, v3, v0) keep v1 - v3 within 0.5 of
// their planes (QuadDecomposition.cpp:326-343): normals from cross products
// scaled by RSQRTPS of their squared length, distances as DPPS; a NaN
// distance does not exceed the bound (COMISS compares false).
__device__ bool mergeable(float4 v0, float4 v1, float4 v2, float4 v3, const uint32_t* __restrict__ rsq) {
  const V3 n0 = approx_normalize(cross3(sub3(v1, v0), sub3(v2, v0)), rsq);
  const V3 n2 = approx_normalize(cross3(sub3(v3, v2), sub3(v0, v2)), rsq);
  const V3 d = sub3(v1, v3);
  const float a = __builtin_fabsf(dp3(n0, d)), b = __builtin_fabsf(dp3(n2, d));
  return !(a > 0.5f || b > 0.5f);
}

// Half-edge h = 3t + k runs from i[k] to i[(k + 1) % 3].  Every index is
// the origin of one half-edge, so this is where indices are checked.
__global__ void __launch_bounds__(kQdBlock) qd_half_edges_kernel(const uint32_t* __restrict__ idx, uint32_t nTri,
                                                                 uint32_t nVertices, uint32_t bits,
                                                                 uint64_t* __restrict__ keys,
                                                                 uint32_t* __restrict__ seqs, uint32_t* __restrict__ bad) {
  const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= 3u * nTri) return;
  const uint32_t t = h / 3u, k = h - 3u * t;
  const uint32_t a = idx[h], b = idx[3u * t + next3(k)];
  if (a >= nVertices) atomicOr(bad, 1u);
  keys[h] = edge_key(a, b, bits);
  seqs[h] = h;
}

__global__ void __launch_bounds__(kQdBlock) qd_reverse_kernel(const uint64_t* __restrict__ keys,
                                                              const uint32_t* __restrict__ seqs, uint32_t nHalf,
                                                              uint32_t bits, uint32_t* __restrict__ revFirst) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nHalf) return;
  const uint64_t key = keys[p];
  const uint64_t rev = ((key & ((uint64_t(1) << bits) - 1u)) << bits) | (key >> bits);
  uint32_t lo = 0, hi = nHalf;  // first entry >= rev
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (keys[mid] < rev) lo = mid + 1u;
    else hi = mid;
  }
  revFirst[seqs[p]] = lo;
}

// Triangle t's adjacency list (QuadDecomposition.cpp:366-384): its own links,
// edge by edge, each with the reverse list's entries inserted up to t's last
// edge (t itself included, which enters twice), in list order; then the links
// of later triangles with t, by their half-edges' insertion numbers, which is
// the order of the rest of t's three reverse lists merged.  A later triangle's
// plane test runs over its own edge, as when the reference reaches it.
template <bool FILL>
__global__ void __launch_bounds__(kQdBlock) qd_adjacency_kernel(QdParams p) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= p.nTri) return;
  const uint32_t* i = p.idx + 3u * size_t(t);
  const uint32_t v[3] = {i[0], i[1], i[2]};
  const float4 x[3] = {p.vertices[v[0]], p.vertices[v[1]], p.vertices[v[2]]};
  uint32_t n = 0;
  int* out = FILL ? p.adj + p.start[t] : nullptr;
  auto push = [&](uint32_t nb) {
    if (FILL) out[n] = int(nb);
    ++n;
  };
  uint64_t rev[3];
  uint32_t at[3];
#pragma unroll
  for (uint32_t k = 0; k < 3; ++k) {
    rev[k] = edge_key(v[next3(k)], v[k], p.bits);
    uint32_t j = p.revFirst[3u * t + k];
    for (; j < p.nHalf && p.keys[j] == rev[k]; ++j) {
      const uint32_t s = p.seqs[j];
      if (s > 3u * t + 2u) break;  // listed after t
      const uint32_t nb = s / 3u;
      const uint32_t apex = p.idx[3u * size_t(nb) + prev3(s - 3u * nb)];
      if (!mergeable(x[k], p.vertices[apex], x[next3(k)], x[prev3(k)], p.rsq)) continue;
      push(nb);
      if (nb == t) push(nb);
    }
    at[k] = j;
  }
  // The next entry of each list, or none, in registers: an edge that thousands
  // of triangles share makes this the longest chain (3,000 triangles on one edge
  // in both directions: rz_quad_decompose_device 4.5 ms with the three entries
  // loaded again in each step, 3.3 ms so).
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  uint32_t head[3];
  auto load_head = [&](uint32_t k) {
    head[k] = at[k] < p.nHalf && p.keys[at[k]] == rev[k] ? p.seqs[at[k]] : kNone;
  };
#pragma unroll
  for (uint32_t k = 0; k < 3; ++k) load_head(k);
  while (true) {
    const uint32_t s = min(head[0], min(head[1], head[2]));
    if (s == kNone) break;
    const uint32_t from = s == head[0] ? 0u : s == head[1] ? 1u : 2u;
#pragma unroll
    for (uint32_t k = 0; k < 3; ++k)
      if (k == from) {
        ++at[k];
        load_head(k);
        const uint32_t nb = s / 3u, kk = s - 3u * nb;
        const uint32_t* o = p.idx + 3u * size_t(nb);
        // The later triangle's edge runs from v[next3(k)] to v[k].
        if (mergeable(x[next3(k)], x[prev3(k)], x[k], p.vertices[o[prev3(kk)]], p.rsq)) push(nb);
      }
  }
  if (!FILL) p.degree[t] = n;
}

// Which triangles write a quad: a single one (its degenerate quad) and the
// lower triangle of a matched pair; one matched to itself writes nothing.
__global__ void __launch_bounds__(kQdBlock) qd_writers_kernel(const int* __restrict__ mate, uint32_t nTri,
                                                              uint32_t* __restrict__ writes) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > nTri) return;
  if (t == nTri) {
    writes[t] = 0u;  // the scan's total
    return;
  }
  const int nb = mate[t];
  writes[t] = (nb == -1 || uint32_t(nb) > t) ? 1u : 0u;
}

// The quads in triangle order (QuadDecomposition.cpp:392-441): a single
// triangle becomes (i0, i2, i1, i0); a matched pair is written from the
// lower triangle's first edge whose reverse list holds the partner, as
// (i[k], i[k+2], i[k+1], the partner's apex on that edge).
__global__ void __launch_bounds__(kQdBlock) qd_emit_kernel(QdParams p, const int* __restrict__ mate,
                                                           const uint32_t* __restrict__ pos, uint32_t* __restrict__ out) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= p.nTri) return;
  const int nb = mate[t];
  if (!(nb == -1 || uint32_t(nb) > t)) return;
  const uint32_t* i = p.idx + 3u * size_t(t);
  uint32_t* o = out + 4u * size_t(pos[t]);
  if (nb == -1) {
    o[0] = i[0];
    o[1] = i[2];
    o[2] = i[1];
    o[3] = i[0];
    return;
  }
  for (uint32_t k = 0; k < 3u; ++k) {
    const uint64_t rev = edge_key(i[next3(k)], i[k], p.bits);
    for (uint32_t j = p.revFirst[3u * t + k]; j < p.nHalf && p.keys[j] == rev; ++j) {
      const uint32_t s = p.seqs[j];
      if (s / 3u != uint32_t(nb)) continue;
      o[0] = i[k];
      o[1] = i[prev3(k)];
      o[2] = i[next3(k)];
      o[3] = p.idx[s - s % 3u + prev3(s % 3u)];
      return;
    }
  }
  atomicOr(p.bad, 2u);  // a matched pair shares no edge: not reachable from the links
}

__global__ void __launch_bounds__(kQdBlock) qd_gather_kernel(const float4* __restrict__ vertices,
                                                             const uint32_t* __restrict__ quadIdx, uint32_t nWords,
                                                             float4* __restrict__ out) {
  const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w < nWords) out[w] = vertices[quadIdx[w]];
}

// List lengths add up without wrapping, so that too many links are refused.
struct SatPlus {
  __host__ __device__ uint32_t operator()(uint32_t a, uint32_t b) const { return a + b < a ? 0xFFFFFFFFu : a + b; }
};

}  // namespace

#define QD_HIP(call)                                \
  do {                                              \
    if ((call) != hipSuccess) return RZ_ERR_DEVICE; \
  } while (0)

hipError_t launch_quad_gather(const float* vertices, const uint32_t* quadIdx, uint32_t nWords, float* out,
                              hipStream_t stream) {
  if (nWords == 0) return hipSuccess;
  qd_gather_kernel<<<qd_grid(nWords), kQdBlock, 0, stream>>>(reinterpret_cast<const float4*>(vertices), quadIdx,
                                                             nWords, reinterpret_cast<float4*>(out));
  return hipGetLastError();
}

int quad_decompose_run(hipStream_t stream, Scratch& scratch, uint32_t nTri, const uint32_t* d_idx,
                       const float* d_vertices, uint32_t nVertices, const uint32_t* d_rsqrt, uint32_t* d_out,
                       uint32_t* nOut) {
  *nOut = 0;
  if (nTri == 0) return RZ_OK;
  if (nTri > 0x7FFFFFFFu / 3u) return RZ_ERR_TOO_LARGE;
  const uint32_t nHalf = 3u * nTri;
  uint32_t bits = 1;
  while (bits < 32 && (uint64_t(1) << bits) < nVertices) ++bits;
  size_t sortBytes = 0, scanBytes = 0;
  QD_HIP(rocprim::radix_sort_pairs(nullptr, sortBytes, static_cast<uint64_t*>(nullptr), static_cast<uint64_t*>(nullptr),
                                   static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr), nHalf, 0u,
                                   2u * bits, stream));
  QD_HIP(rocprim::exclusive_scan(nullptr, scanBytes, static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr),
                                 0u, size_t(nTri) + 1, SatPlus(), stream));
  Scratch::Frame frame(scratch);
  uint64_t* keys = scratch.take<uint64_t>(nHalf);
  uint64_t* sortedKeys = scratch.take<uint64_t>(nHalf);
  uint32_t* seqs = scratch.take<uint32_t>(nHalf);
  uint32_t* sortedSeqs = scratch.take<uint32_t>(nHalf);
  uint32_t* revFirst = scratch.take<uint32_t>(nHalf);
  uint32_t* degree = scratch.take<uint32_t>(size_t(nTri) + 1);  // then: which triangles write a quad
  uint32_t* start = scratch.take<uint32_t>(size_t(nTri) + 1);   // then: the quads' positions
  int* mates = scratch.take<int>(nTri);
  uint32_t* words = scratch.take<uint32_t>(1);
  unsigned char* temp = scratch.take<unsigned char>(std::max(sortBytes, scanBytes));
  if (!keys || !sortedKeys || !seqs || !sortedSeqs || !revFirst || !degree || !start || !mates || !words || !temp)
    return RZ_ERR_OUT_OF_MEMORY;
  QD_HIP(hipMemsetAsync(words, 0, 4, stream));

  // Half-edges, sorted by (key, insertion number).
  qd_half_edges_kernel<<<qd_grid(nHalf), kQdBlock, 0, stream>>>(d_idx, nTri, nVertices, bits, keys, seqs, words);
  QD_HIP(hipGetLastError());
  uint32_t bad = 0;
  QD_HIP(hipMemcpyAsync(&bad, words, 4, hipMemcpyDeviceToHost, stream));
  QD_HIP(hipStreamSynchronize(stream));
  if (bad) return RZ_ERR_INVALID_ARGUMENT;
  size_t bytes = sortBytes;
  QD_HIP(rocprim::radix_sort_pairs(temp, bytes, keys, sortedKeys, seqs, sortedSeqs, nHalf, 0u, 2u * bits, stream));
  qd_reverse_kernel<<<qd_grid(nHalf), kQdBlock, 0, stream>>>(sortedKeys, sortedSeqs, nHalf, bits, revFirst);
  QD_HIP(hipGetLastError());

  // Adjacency lists: count, scan, fill.
  QdParams P{};
  P.idx = d_idx;
  P.vertices = reinterpret_cast<const float4*>(d_vertices);
  P.nTri = nTri;
  P.nHalf = nHalf;
  P.bits = bits;
  P.keys = sortedKeys;
  P.seqs = sortedSeqs;
  P.revFirst = revFirst;
  P.rsq = d_rsqrt;
  P.degree = degree;
  P.start = start;
  P.bad = words;
  QD_HIP(hipMemsetAsync(degree + nTri, 0, 4, stream));
  qd_adjacency_kernel<false><<<qd_grid(nTri), kQdBlock, 0, stream>>>(P);
  QD_HIP(hipGetLastError());
  bytes = scanBytes;
  QD_HIP(rocprim::exclusive_scan(temp, bytes, degree, start, 0u, size_t(nTri) + 1, SatPlus(), stream));
  uint32_t nAdj = 0;
  QD_HIP(hipMemcpyAsync(&nAdj, start + nTri, 4, hipMemcpyDeviceToHost, stream));
  QD_HIP(hipStreamSynchronize(stream));
  if (nAdj > 0x7FFFFFFFu) return RZ_ERR_TOO_LARGE;
  P.adj = scratch.take<int>(nAdj);
  if (!P.adj) return RZ_ERR_OUT_OF_MEMORY;
  qd_adjacency_kernel<true><<<qd_grid(nTri), kQdBlock, 0, stream>>>(P);
  QD_HIP(hipGetLastError());

  // The matching, on the host: the lists come and the partners go through
  // pinned memory where it can be had.
  const size_t hostWords = size_t(nTri) + 1 + nAdj + nTri;
  try {
    std::vector<uint32_t> pageable;
    uint32_t* h = static_cast<uint32_t*>(scratch.host(hostWords * 4));
    if (!h) {
      pageable.resize(hostWords);
      h = pageable.data();
    }
    int* adj = reinterpret_cast<int*>(h + size_t(nTri) + 1);
    int* mate = adj + nAdj;
    QD_HIP(hipMemcpyAsync(h, start, (size_t(nTri) + 1) * 4, hipMemcpyDeviceToHost, stream));
    if (nAdj) QD_HIP(hipMemcpyAsync(adj, P.adj, size_t(nAdj) * 4, hipMemcpyDeviceToHost, stream));
    QD_HIP(hipStreamSynchronize(stream));
    rzq::match(nTri, h, adj, mate);
    QD_HIP(hipMemcpyAsync(mates, mate, size_t(nTri) * 4, hipMemcpyHostToDevice, stream));
    if (!pageable.empty()) QD_HIP(hipStreamSynchronize(stream));
  } catch (const std::bad_alloc&) {
    return RZ_ERR_OUT_OF_MEMORY;
  }

  // The quads.
  qd_writers_kernel<<<qd_grid(size_t(nTri) + 1), kQdBlock, 0, stream>>>(mates, nTri, degree);
  QD_HIP(hipGetLastError());
  bytes = scanBytes;
  QD_HIP(rocprim::exclusive_scan(temp, bytes, degree, start, 0u, size_t(nTri) + 1, SatPlus(), stream));
  qd_emit_kernel<<<qd_grid(nTri), kQdBlock, 0, stream>>>(P, mates, start, d_out);
  QD_HIP(hipGetLastError());
  uint32_t quads = 0;
  QD_HIP(hipMemcpyAsync(&quads, start + nTri, 4, hipMemcpyDeviceToHost, stream));
  QD_HIP(hipMemcpyAsync(&bad, words, 4, hipMemcpyDeviceToHost, stream));
  QD_HIP(hipStreamSynchronize(stream));
  if (bad) return RZ_ERR_DEVICE;
  *nOut = 4u * quads;
  return RZ_OK;
}

}  // namespace rzd
