// Locality schedule shared by the standard and the filtered builds: each
// vertex's nearest of K pivot rows (one octet per vertex, eight vertices per
// wave). Vertices sorted by cell make the waves in flight work on
// neighbouring vertices, whose searches, candidate rows and reverse sources
// overlap in L2 and the MALL. The schedule only changes the order in which
// independent vertices are processed, never a result.
#pragma once

#include "wave.h"

namespace dance {

constexpr uint32_t kCellsBlock = 256;  // 4 waves, 32 vertices per workgroup

inline uint32_t cells_grid(uint32_t N) { return (N + 31u) / 32u; }

// Sort key of a vertex from its nearest pivots b1, b2, b3 (nearest first).
// levels = 3 orders the vertices of a cell (b1) by their second and third
// nearest pivots, i.e. by the neighbouring cells they face, so the vertices
// in flight together are closer than in vertex-id order; levels = 1 keys by
// the cell alone. Three levels need K^3 <= 2^32 (K <= 1625).
constexpr uint32_t kCellLevelsMaxK = 1625;
__host__ __device__ inline uint32_t cell_levels(uint32_t K, uint32_t levels) {
  return (levels >= 3 && K <= kCellLevelsMaxK) ? 3u : 1u;
}
__device__ __forceinline__ uint32_t cell_key(uint32_t b1, uint32_t b2, uint32_t b3, uint32_t K, uint32_t levels) {
  return levels == 3u ? (b1 * K + b2) * K + b3 : b1;
}
// Keeps the three smallest (d, k) in order, first on ties.
struct Nearest3 {
  float d1 = FLT_MAX, d2 = FLT_MAX, d3 = FLT_MAX;
  uint32_t k1 = 0, k2 = 0, k3 = 0;
  __device__ __forceinline__ void add(float d, uint32_t k) {
    if (d < d1) {
      d3 = d2;
      k3 = k2;
      d2 = d1;
      k2 = k1;
      d1 = d;
      k1 = k;
    } else if (d < d2) {
      d3 = d2;
      k3 = k2;
      d2 = d;
      k2 = k;
    } else if (d < d3) {
      d3 = d;
      k3 = k;
    }
  }
};

// Cells for N rows: the default count, but at least kMinCellRows rows a cell (a
// finer order costs more pivots than its locality saves: 10k-row builds, 50
// of them, 111.6 ms with 64 cells, 117.1 with 1024; 100k rows 71.1 ms with 64
// or 256, 71.8 with 1024; at 300k 1024 is the best) and no schedule below
// kMinCells cells (2k rows: 1.19 ms without, 1.21 with 64, 1.32 with 1024).
constexpr uint32_t kMinCellRows = 256, kMinCells = 16;
inline uint32_t cells_for(uint32_t N, uint32_t most) {
  const uint32_t k = N / kMinCellRows;
  return k < kMinCells ? 0u : (k < most ? k : most);
}

// Pivot k of K is row floor(k N / K) (evenly spaced).
static __global__ void k_pivots(uint32_t N, uint32_t K, uint32_t* __restrict__ piv) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < K) piv[k] = (uint32_t)(((uint64_t)k * N) / K);
}

// cell[v] = the sort key of row v's nearest pivots (first on ties; levels
// from cell_levels), vid[v] = v.
template <int DT, int CPL>
__global__ __launch_bounds__(kCellsBlock) void k_cells(RowSet rs, uint32_t N, const uint32_t* __restrict__ pivots,
                                                       uint32_t K, uint32_t levels, uint32_t* __restrict__ cell,
                                                       uint32_t* __restrict__ vid) {
  const uint32_t lane = lane_id(), grp = lane >> 3, sub = lane & 7u;
  const uint32_t w = blockIdx.x * (kCellsBlock / 64u) + wave_index();
  const uint32_t v = w * 8u + grp;
  if (w * 8u >= N) return;
  const bool act = v < N;
  uint4 xv[CPL];
  load_row<CPL>(rs, act ? v : 0u, act, sub, xv);
  Nearest3 nb;
  for (uint32_t k = 0; k < K; ++k) {
    uint4 pv[CPL];
    load_row<CPL>(rs, pivots[k], true, sub, pv);
    nb.add(octet_finish<DT, CPL>(rs, sub, xv, pv), k);
  }
  if (act && sub == 0) {
    cell[v] = cell_key(nb.k1, nb.k2, nb.k3, K, levels);
    vid[v] = v;
  }
}

// a = s^2 sum(q^2) of a code row from its header {s, r, lo, hi} (lo is a - r^2 up
// to the bound's slack); 0 for rows without codes, whose r is infinite.
__device__ __forceinline__ float code_norm(const uint4& h) {
  const float r = __uint_as_float(h.y), lo = __uint_as_float(h.z);
  return r < __builtin_inff() ? __builtin_fmaf(r, r, lo) : 0.0f;
}

// Nearest pivots on the matrix cores, for code rows (U8 = false, 128 bytes) and
// uint8 rows of STEPS x 32 bytes (U8 = true): one wave per 32 vertices, int8
// MFMA tiles of 32 pivots (rows) x 32 vertices (columns) over the row's bytes
// (code chunks 1-7, or the uint8 bytes shifted by -128). The vertices'
// fragments stay in registers up to 8 steps and are read again per tile
// beyond. Bound by the pivot rows read from L2 (every wave reads them all).
// uint8 rows of 192 bytes at N = 250k, K = 1024 took 7.7 ms with one octet per
// vertex and pivot (k_cells), the 10k-row builds of the stitched case 0.77 ms
// each. Lane l holds, for vertex
// l % 32, pivots 8 (v >> 2) + (v & 3) + 4 (l >> 5) of each tile (v < 16), in
// ascending order, keeps its own three nearest (first on ties), and the two
// halves of a vertex merge by (distance, pivot) at the end. The distances
// are k_cells_q's exactly (the same fp32 expression on the same integer dot
// for code rows; the integer squared distance for uint8 rows, which
// k_cells_q's fp32 expression also yields below 2^24), so the cells are too.
template <bool U8, int STEPS>
__global__ __launch_bounds__(256) void k_cells_mfma(const uint4* __restrict__ rows, uint32_t stride16, uint32_t N,
                                                    const uint32_t* __restrict__ pivots, uint32_t K,
                                                    uint32_t levels, uint32_t* __restrict__ cell,
                                                    uint32_t* __restrict__ vid) {
  __shared__ int pn_i[4][32];    // uint8 rows: |pivot'|^2
  __shared__ float pn_f[4][32];  // code rows: a and s of the pivot
  __shared__ float ps_f[4][32];
  const uint32_t w = wave_index(), lane = lane_id(), jl = lane & 31u, half = lane >> 5;
  const uint32_t v0 = (blockIdx.x * 4u + w) * 32u;
  if (v0 >= N) return;  // the whole wave; no block-wide barrier follows
  const uint32_t v = v0 + jl;
  const bool act = v < N;
  constexpr bool kHold = STEPS <= 8;
  // 16 bytes of row `id` for K-step s: chunk 2 s + half of the uint8 row, or
  // chunk 1 + 2 s + half of the code row (its last would be past the row: 0)
  auto frag = [&](uint32_t id, bool ok, uint32_t step) -> v4i_t {
    const uint32_t c = (U8 ? 0u : 1u) + 2u * step + half;
    if (!ok || c >= 2u * STEPS) return v4i_t{0, 0, 0, 0};
    const uint4 q = rows[(size_t)id * stride16 + c];
    if constexpr (U8)
      return v4i_t{(int)(q.x ^ 0x80808080u), (int)(q.y ^ 0x80808080u), (int)(q.z ^ 0x80808080u),
                   (int)(q.w ^ 0x80808080u)};
    else
      return v4i_t{(int)q.x, (int)q.y, (int)q.z, (int)q.w};
  };
  v4i_t B[kHold ? STEPS : 1];
  if constexpr (kHold) {
#pragma unroll
    for (uint32_t st = 0; st < STEPS; ++st) B[st] = frag(v, act, st);
  }
  int xn = 0;
  float xa = 0.0f, xs = 1.0f;
  if constexpr (U8) {
    int part = 0;
#pragma unroll
    for (uint32_t st = 0; st < STEPS; ++st) part = i8_sq4(kHold ? B[kHold ? st : 0] : frag(v, act, st), part);
    xn = part + __shfl_xor(part, 32);
  } else if (act) {
    const uint4 h = rows[(size_t)v * stride16];
    xs = __uint_as_float(h.x);
    xa = code_norm(h);
  }
  Nearest3 nb;
  for (uint32_t t0 = 0; t0 < K; t0 += 32) {
    const uint32_t pi = t0 + jl;
    const bool pok = pi < K;
    const uint32_t pid = pok ? pivots[pi] : 0u;
    int part = 0;  // uint8 rows: sum of squares of this lane's share of the pivot
    v16i_t acc = {};
#pragma unroll
    for (uint32_t st = 0; st < STEPS; ++st) {
      const v4i_t A = frag(pid, pok, st);
      if constexpr (U8) part = i8_sq4(A, part);
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, kHold ? B[kHold ? st : 0] : frag(v, act, st), acc, 0, 0, 0);
    }
    wave_sync();  // the previous tile's reads of the pivot terms are done
    if constexpr (U8) {
      part += __shfl_xor(part, 32);
      if (lane < 32u) pn_i[w][jl] = part;
    } else {
      if (lane < 32u && pok) {
        const uint4 h = rows[(size_t)pid * stride16];
        pn_f[w][jl] = code_norm(h);
        ps_f[w][jl] = __uint_as_float(h.x);
      }
    }
    wave_sync();
    static_for<0, 16>([&](auto vc) {
      constexpr uint32_t vv = decltype(vc)::value, ir0 = 8u * (vv >> 2) + (vv & 3u);
      const uint32_t ir = ir0 + 4u * half, k = t0 + ir;
      if (k < K) {
        float d;
        if constexpr (U8)
          d = u8_gram_dist(xn, pn_i[w][ir], acc[vv]);
        else
          d = xa + pn_f[w][ir] - 2.0f * xs * ps_f[w][ir] * (float)acc[vv];
        nb.add(d, k);
      }
    });
  }
  // merge the upper half's three into the lower half's, by (distance, pivot)
  const float e1 = __shfl_xor(nb.d1, 32), e2 = __shfl_xor(nb.d2, 32), e3 = __shfl_xor(nb.d3, 32);
  const uint32_t f1 = (uint32_t)__shfl_xor((int)nb.k1, 32), f2 = (uint32_t)__shfl_xor((int)nb.k2, 32),
                 f3 = (uint32_t)__shfl_xor((int)nb.k3, 32);
  if (half == 0u && act) {
    // two sorted lists of three, popped from the front by selects
    float a1 = nb.d1, a2 = nb.d2, a3 = nb.d3, b1 = e1, b2 = e2, b3 = e3;
    uint32_t ka1 = nb.k1, ka2 = nb.k2, ka3 = nb.k3, kb1 = f1, kb2 = f2, kb3 = f3;
    uint32_t out[3];
#pragma unroll
    for (int o = 0; o < 3; ++o) {
      const bool ta = a1 < b1 || (a1 == b1 && ka1 < kb1);
      out[o] = ta ? ka1 : kb1;
      a1 = ta ? a2 : a1;
      ka1 = ta ? ka2 : ka1;
      a2 = ta ? a3 : a2;
      ka2 = ta ? ka3 : ka2;
      b1 = ta ? b1 : b2;
      kb1 = ta ? kb1 : kb2;
      b2 = ta ? b2 : b3;
      kb2 = ta ? kb2 : kb3;
    }
    cell[v] = cell_key(out[0], out[1], out[2], K, levels);
    vid[v] = v;
  }
}

}  // namespace dance
