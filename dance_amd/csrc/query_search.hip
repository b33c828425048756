// Host side of the query search (dance_search / dance_search_resident in
// include/dance_hip.h): uploads what is not resident, launches k_query with
// the candidate-list width for L, and returns the k best ids and distances.
// Used by the recall measurement and by callers that want GPU search over a
// built graph (reference counterpart: DiskANN search_memory_index, filtered
// start points integrations/dance-diskann-78256bba.patch:20583-20600).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "../../include/dance_hip.h"
#include "host_common.h"
#include "query_kernels.h"

namespace dance {
namespace {

using namespace qs;

std::mutex g_qmu;
DanceSearchStats g_qstats{};

constexpr size_t kCtrBytes = 3 * 8;           // distances, expansions, capped queries
constexpr size_t kSendBytes = 512ull << 10;  // least bytes of an input copy that is followed by another
constexpr uint32_t kMaxL = 1024;  // 16 slots per lane
constexpr uint64_t kGathersPerL = 24;  // rows a query gathers per list entry
// Widest rows and lists that have a kernel for packed rows.
constexpr int kPackedCpl = 4, kPackedPs = 2;
int pick_ps(uint32_t L) { return L <= 64 ? 1 : L <= 128 ? 2 : L <= 256 ? 4 : L <= 512 ? 8 : 16; }

struct SearchIn {
  const void* data;  // device rows (resident) or host rows
  bool data_on_device;
  int dtype;
  uint32_t N, dim;
  const uint32_t* graph;  // device (resident) or host
  const uint32_t* degree;
  bool graph_on_device;
  uint32_t R;
  const uint32_t* starts;
  uint32_t nstarts;
  const uint32_t* start_off;  // host, nq + 1 entries (nullptr: 1 shared or nq starts)
  const void* queries;  // host
  uint32_t nq, k, L;
  const uint32_t* label_offsets;  // host, optional
  const uint32_t* labels;
  const uint32_t* query_labels;
  uint32_t* ids_out;  // host
  float* d_out;
};

int run_search(const SearchIn& in) {
  if (!in.data || !in.graph || !in.degree || !in.starts || !in.queries || !in.ids_out || !in.d_out) {
    std::fprintf(stderr, "[dance_search] null input pointer.\n");
    return -1;
  }
  if (in.N == 0 || in.dim == 0 || in.R == 0 || in.nq == 0 || in.k == 0 || in.k > kMaxK || in.L < in.k ||
      in.L > kMaxL || (!in.start_off && in.nstarts != 1 && in.nstarts != in.nq)) {
    std::fprintf(stderr, "[dance_search] invalid parameters N=%u dim=%u R=%u nq=%u k=%u L=%u nstarts=%u\n", in.N,
                 in.dim, in.R, in.nq, in.k, in.L, in.nstarts);
    return -1;
  }
  if (in.start_off) {
    bool ok = in.start_off[0] == 0;
    for (uint32_t q = 0; ok && q < in.nq; ++q) ok = in.start_off[q] <= in.start_off[q + 1];
    if (!ok) {
      std::fprintf(stderr, "[dance_search] start_offsets must start at 0 and not decrease\n");
      return -1;
    }
  }
  const bool filt = in.label_offsets || in.labels || in.query_labels;
  if (filt && !(in.label_offsets && in.labels && in.query_labels)) {
    std::fprintf(stderr, "[dance_search] label filter needs offsets, labels and query labels\n");
    return -1;
  }
  if (in.dtype != DANCE_F32 && in.dtype != DANCE_U8 && in.dtype != DANCE_F16) {
    std::fprintf(stderr, "[dance_search] unsupported dtype %d\n", in.dtype);
    return -1;
  }
  std::lock_guard<std::mutex> lk(g_qmu);
  g_qstats = DanceSearchStats{};
  const size_t row_bytes = (size_t)in.dim * elem_bytes(in.dtype);
  // The call's small inputs and its results lie in one block, in copy order:
  // starts, their offsets, query labels, queries, counters, ids, distances.
  const size_t b_starts = arena_bytes((size_t)in.nstarts * 4);
  const size_t b_off = in.start_off ? arena_bytes((size_t)(in.nq + 1) * 4) : 0;
  const size_t b_qlab = filt ? arena_bytes((size_t)in.nq * 4) : 0;
  const size_t b_q = arena_bytes(row_bytes * in.nq);
  const size_t b_in = b_starts + b_off + b_qlab + b_q + arena_bytes(kCtrBytes);
  const size_t b_res = arena_bytes((size_t)in.nq * in.k * 4);
  const uint32_t ntotal = filt ? in.label_offsets[in.N] : 0u;
  CallLease lease;  // opened below, when what it holds is known
  Rows base, qr;
  const size_t stride = row_layout(base, in.dtype, in.N, in.dim);
  // Rows that fill the kernels' chunk group are read as they are. Others are
  // copied into padded rows, or read packed when the call gathers fewer rows
  // than that copy would touch: a query gathers about kGathersPerL rows per
  // list entry. Measured with the copy and packed (kernel / call): 16 queries of
  // L 50 over 200k x 100 fp32 0.25 / 0.86 and 0.24 / 0.43 ms, of L 100 over 500k x
  // 200 uint8 0.66 / 1.35 and 0.74 / 0.99 ms; 10k of L 100 over 500k x 100 fp32
  // 2.57 / 3.53 and 3.54 / 3.95 ms (packed rows straddle one cache line more, and
  // their last chunk takes more instructions).
  // (Uploaded rows start at an allocation, which is aligned.)
  const bool whole =
      stride == row_bytes && (!in.data_on_device || (reinterpret_cast<uintptr_t>(in.data) & 15u) == 0);
  const int ps = pick_ps(in.L);
  const bool in_place = !whole && pick_cpl(base.rs.nch) <= kPackedCpl && ps <= kPackedPs &&
                        (uint64_t)in.nq * in.L * kGathersPerL < in.N;
  // The lease holds what this call allocates and no more: 16 queries over 200k
  // resident rows lease 2 MiB, 10k queries of 96 dimensions 8 MiB.
  size_t need = b_in + 2 * b_res;
  if (stride != row_bytes) need += arena_bytes(stride * in.nq);
  if (!in.data_on_device) need += arena_bytes(row_bytes * in.N);
  if (!whole && !in_place) need += arena_bytes(stride * in.N);
  if (!in.graph_on_device) need += arena_bytes((size_t)in.N * in.R * 4) + arena_bytes((size_t)in.N * 4);
  if (filt) need += arena_bytes((size_t)(in.N + 1) * 4) + arena_bytes((size_t)std::max(1u, ntotal) * 4);
  DCHECK(lease.open(need));
  const hipStream_t s = lease.stream();
  const void* packed = in.data;  // the base rows in device memory, as the caller packed them
  DevBuf up;
  if (!in.data_on_device) {
    DCHECK(up.alloc(row_bytes * in.N));
    DCHECK(copy_pageable(up.p, in.data, row_bytes * in.N, hipMemcpyHostToDevice));
    packed = up.p;
  }
  if (whole)
    base.rs.rows = static_cast<const uint4*>(packed);
  else if (!in_place)
    DCHECK(setup_rows(base, packed, true, in.dtype, in.dtype, in.N, in.dim, s));
  const int cpl = pick_cpl(base.rs.nch);
  if (cpl < 0) {
    std::fprintf(stderr, "[dance_search] dim=%u is beyond the supported row width\n", in.dim);
    return -1;
  }
  DevBuf blk, g, dg, off, lab;
  DCHECK(blk.alloc(b_in + 2 * b_res));
  char* const d_in = blk.as<char>();
  char* const d_ctr = d_in + b_in - arena_bytes(kCtrBytes);
  // Pinned halves of the lease: inputs, results. A copy from or to pageable
  // memory moves 8 GB/s and takes 10 us or more; inputs are sent while the rest
  // is still written. With the leased memory and stream: 16 queries of L 50 over
  // 200k x 96 0.40 -> 0.25 ms (kernel 0.22), 10k of L 100 over 1M x 96 2.85 ->
  // 2.69 ms (kernel 2.42), 1k filtered over 100k 0.87 -> 0.66 ms (kernel 0.50).
  // Without pinned memory the copies are plain ones.
  char* const pin = lease.host();
  if (pin && b_in <= kCallHostBytes / 2) {
    size_t sent = 0, at = 0;
    auto put = [&](const void* src, size_t bytes, size_t room) -> int {
      for (size_t o = 0; o < bytes; o += kSendBytes) {  // the first pieces travel while the next are written
        const size_t n = std::min(kSendBytes, bytes - o);
        std::memcpy(pin + at + o, static_cast<const char*>(src) + o, n);
        if (at + o + n - sent >= kSendBytes) {
          DHIP(hipMemcpyAsync(d_in + sent, pin + sent, at + o + n - sent, hipMemcpyHostToDevice, s));
          sent = at + o + n;
        }
      }
      at += room;
      return 0;
    };
    DCHECK(put(in.starts, (size_t)in.nstarts * 4, b_starts));
    if (in.start_off) DCHECK(put(in.start_off, (size_t)(in.nq + 1) * 4, b_off));
    if (filt) DCHECK(put(in.query_labels, (size_t)in.nq * 4, b_qlab));
    DCHECK(put(in.queries, row_bytes * in.nq, b_q));
    std::memset(pin + at, 0, kCtrBytes);
    DHIP(hipMemcpyAsync(d_in + sent, pin + sent, at + kCtrBytes - sent, hipMemcpyHostToDevice, s));
  } else {
    if (in.nstarts) DHIP(hipMemcpyAsync(d_in, in.starts, (size_t)in.nstarts * 4, hipMemcpyHostToDevice, s));
    if (in.start_off)
      DHIP(hipMemcpyAsync(d_in + b_starts, in.start_off, (size_t)(in.nq + 1) * 4, hipMemcpyHostToDevice, s));
    if (filt)
      DHIP(hipMemcpyAsync(d_in + b_starts + b_off, in.query_labels, (size_t)in.nq * 4, hipMemcpyHostToDevice, s));
    DCHECK(copy_pageable(d_in + b_starts + b_off + b_qlab, in.queries, row_bytes * in.nq, hipMemcpyHostToDevice));
    DHIP(hipMemsetAsync(d_ctr, 0, kCtrBytes, s));
  }
  DCHECK(setup_rows(qr, d_in + b_starts + b_off + b_qlab, true, in.dtype, in.dtype, in.nq, in.dim, s));
  const uint32_t* dgraph = in.graph;
  const uint32_t* ddeg = in.degree;
  if (!in.graph_on_device) {
    DCHECK(g.alloc((size_t)in.N * in.R * 4));
    DCHECK(dg.alloc((size_t)in.N * 4));
    DHIP(hipMemcpyAsync(g.p, in.graph, (size_t)in.N * in.R * 4, hipMemcpyHostToDevice, s));
    DHIP(hipMemcpyAsync(dg.p, in.degree, (size_t)in.N * 4, hipMemcpyHostToDevice, s));
    dgraph = g.as<uint32_t>();
    ddeg = dg.as<uint32_t>();
  }
  if (filt) {
    DCHECK(off.alloc((size_t)(in.N + 1) * 4));
    DCHECK(lab.alloc((size_t)std::max(1u, ntotal) * 4));
    DHIP(hipMemcpyAsync(off.p, in.label_offsets, (size_t)(in.N + 1) * 4, hipMemcpyHostToDevice, s));
    if (ntotal) DHIP(hipMemcpyAsync(lab.p, in.labels, (size_t)ntotal * 4, hipMemcpyHostToDevice, s));
  }
  char* const d_ids = d_in + b_in;
  char* const d_dist = d_ids + b_res;
  QArgs a{in.N, in.R, dgraph, ddeg, reinterpret_cast<const uint32_t*>(d_in), in.nstarts,
          in.start_off ? reinterpret_cast<const uint32_t*>(d_in + b_starts) : nullptr, in.nq, in.k, in.L,
          16u * in.L + 1024u, filt ? off.as<uint32_t>() : nullptr, filt ? lab.as<uint32_t>() : nullptr,
          filt ? reinterpret_cast<const uint32_t*>(d_in + b_starts + b_off) : nullptr,
          reinterpret_cast<uint32_t*>(d_ids), reinterpret_cast<float*>(d_dist),
          reinterpret_cast<unsigned long long*>(d_ctr), static_cast<const uint8_t*>(packed), (uint32_t)row_bytes};
  DHIP(hipEventRecord(lease.set.e0, s));
  const uint32_t grid = (in.nq + kWaves - 1) / kWaves;
  const size_t lds = (size_t)kWaves * kLds * 4;
  DCHECK(with_dt_cpl(base.kind(), cpl, [&](auto dt, auto c) {
    constexpr int DT = decltype(dt)::value, CPL = decltype(c)::value;
    auto go = [&](auto p) {
      constexpr int PS = decltype(p)::value;
      if constexpr (CPL <= kPackedCpl && PS <= kPackedPs) {
        if (in_place) {
          hipLaunchKernelGGL((k_query<DT, CPL, PS, true>), dim3(grid), dim3(kBlock), lds, s, base.rs, qr.rs, a);
          return;
        }
      }
      hipLaunchKernelGGL((k_query<DT, CPL, PS, false>), dim3(grid), dim3(kBlock), lds, s, base.rs, qr.rs, a);
    };
    if (ps == 1)
      go(IC<1>{});
    else if (ps == 2)
      go(IC<2>{});
    else if (ps == 4)
      go(IC<4>{});
    else if (ps == 8)
      go(IC<8>{});
    else
      go(IC<16>{});
    DHIP(hipGetLastError());
    return 0;
  }));
  DHIP(hipEventRecord(lease.set.e1, s));
  unsigned long long c3[kCtrBytes / 8];
  const size_t res_bytes = (size_t)in.nq * in.k * 4;
  const size_t b_out = arena_bytes(kCtrBytes) + 2 * b_res;
  if (pin && b_out <= kCallHostBytes / 2) {
    char* const out = pin + kCallHostBytes / 2;
    DHIP(hipMemcpyAsync(out, d_ctr, b_out, hipMemcpyDeviceToHost, s));
    DHIP(hipStreamSynchronize(s));
    std::memcpy(c3, out, sizeof(c3));
    std::memcpy(in.ids_out, out + (d_ids - d_ctr), res_bytes);
    std::memcpy(in.d_out, out + (d_dist - d_ctr), res_bytes);
  } else {
    DHIP(hipMemcpyAsync(in.ids_out, d_ids, res_bytes, hipMemcpyDeviceToHost, s));
    DHIP(hipMemcpyAsync(in.d_out, d_dist, res_bytes, hipMemcpyDeviceToHost, s));
    DHIP(hipMemcpyAsync(c3, d_ctr, sizeof(c3), hipMemcpyDeviceToHost, s));
    DHIP(hipStreamSynchronize(s));
  }
  lease.done();
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, lease.set.e0, lease.set.e1);
  g_qstats.kernel_ms = ms;
  g_qstats.distances = c3[0];
  g_qstats.expansions = c3[1];
  g_qstats.capped_queries = c3[2];
  return 0;
}

}  // namespace
}  // namespace dance

using namespace dance;

extern "C" {

int dance_release_memory(void) {
  dance::CallPool::get().release();
  dance::release_stages();
  return 0;
}

int dance_search(const void* h_data, int dtype, uint32_t num_points, uint32_t dim, const uint32_t* h_graph,
                 const uint32_t* h_degree, uint32_t R, const uint32_t* starts, uint32_t num_starts,
                 const void* h_queries, uint32_t num_queries, uint32_t k, uint32_t L,
                 const uint32_t* point_label_offsets, const uint32_t* point_labels, const uint32_t* query_labels,
                 uint32_t* ids_out, float* dists_out) {
  return run_search(SearchIn{h_data, false, dtype, num_points, dim, h_graph, h_degree, false, R, starts, num_starts,
                             nullptr, h_queries, num_queries, k, L, point_label_offsets, point_labels, query_labels,
                             ids_out, dists_out});
}

int dance_search_resident(const void* d_data, int dtype, uint32_t num_points, uint32_t dim, const uint32_t* d_graph,
                          const uint32_t* d_degree, uint32_t R, const uint32_t* starts, uint32_t num_starts,
                          const void* h_queries, uint32_t num_queries, uint32_t k, uint32_t L,
                          const uint32_t* point_label_offsets, const uint32_t* point_labels,
                          const uint32_t* query_labels, uint32_t* ids_out, float* dists_out) {
  return run_search(SearchIn{d_data, true, dtype, num_points, dim, d_graph, d_degree, true, R, starts, num_starts,
                             nullptr, h_queries, num_queries, k, L, point_label_offsets, point_labels, query_labels,
                             ids_out, dists_out});
}

int dance_search_multistart(const void* h_data, int dtype, uint32_t num_points, uint32_t dim,
                            const uint32_t* h_graph, const uint32_t* h_degree, uint32_t R,
                            const uint32_t* start_offsets, const uint32_t* starts, const void* h_queries,
                            uint32_t num_queries, uint32_t k, uint32_t L, const uint32_t* point_label_offsets,
                            const uint32_t* point_labels, const uint32_t* query_labels, uint32_t* ids_out,
                            float* dists_out) {
  if (!start_offsets) return -1;
  return run_search(SearchIn{h_data, false, dtype, num_points, dim, h_graph, h_degree, false, R,
                             starts, num_queries ? start_offsets[num_queries] : 0u, start_offsets, h_queries,
                             num_queries, k, L, point_label_offsets, point_labels, query_labels, ids_out,
                             dists_out});
}

int dance_search_multistart_resident(const void* d_data, int dtype, uint32_t num_points, uint32_t dim,
                                     const uint32_t* d_graph, const uint32_t* d_degree, uint32_t R,
                                     const uint32_t* start_offsets, const uint32_t* starts, const void* h_queries,
                                     uint32_t num_queries, uint32_t k, uint32_t L,
                                     const uint32_t* point_label_offsets, const uint32_t* point_labels,
                                     const uint32_t* query_labels, uint32_t* ids_out, float* dists_out) {
  if (!start_offsets) return -1;
  return run_search(SearchIn{d_data, true, dtype, num_points, dim, d_graph, d_degree, true, R,
                             starts, num_queries ? start_offsets[num_queries] : 0u, start_offsets, h_queries,
                             num_queries, k, L, point_label_offsets, point_labels, query_labels, ids_out,
                             dists_out});
}

void dance_get_last_search_stats(DanceSearchStats* stats) {
  if (!stats) return;
  std::lock_guard<std::mutex> lk(g_qmu);
  *stats = g_qstats;
}

}  // extern "C"
