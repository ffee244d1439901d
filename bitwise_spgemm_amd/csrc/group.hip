// group.hip — row grouping by bitmask (first-fit disjoint groups per tile of
// tile_rows rows x one 32-column word), spilled-row CSR, un-grouping.
//
// A workgroup of one or four waves (tiles spread over every CU, no two placement
// chains share a CU's scalar unit) owns one tile: the waves load its words, the first
// walks its rows 64 at a time (lane l <-> row j0 + l) and places them, the waves
// store the results.  Per chunk one vector pass finds the lanes that fit some
// group; the first of them joins, and again from the rows after it, so that the
// serial chain is one step per row that joins.  The result equals the serial
// ascending-row first fit exactly.
#include "bws_internal.hpp"

namespace bws {
namespace {

constexpr int kBlock = 256;
constexpr int kGroupPF = 32;  // 64-row chunks whose words a grouping wave loads at once

__global__ void k_zero_i64(int64_t* p) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0;
}

// A tile's group masks.  GC > 0: the group count is GC, known at compile
// time, and the masks sit in scalar registers, so the placement loop tests
// them and adds to them without moving them between lanes and scalars.
// GC == 0 (any count up to 32): lane g < G of one vector register holds mask
// g, read back with v_readlane.
template <int GC>
struct GroupMasks {
  uint32_t m[GC];
  __device__ GroupMasks() {
#pragma unroll
    for (int g = 0; g < GC; ++g) m[g] = 0u;
  }
  __device__ uint32_t get(int g) const {  // g wave-uniform
    uint32_t v = 0u;
#pragma unroll
    for (int i = 0; i < GC; ++i)
      if (i == g) v = m[i];
    return v;
  }
  // first group that word w fits (GC if none)
  __device__ int fit(uint32_t w, int) const {
    int f = GC;
#pragma unroll
    for (int g = GC - 1; g >= 0; --g)
      if ((m[g] & w) == 0u) f = g;
    return f;
  }
  // gj, mj wave-uniform; gj >= GC adds nothing
  __device__ void add(int gj, uint32_t mj, int) {
#pragma unroll
    for (int g = 0; g < GC; ++g) m[g] |= g == gj ? mj : 0u;
  }
  __device__ uint32_t lane_value(int lane) const {
    uint32_t v = 0u;
#pragma unroll
    for (int g = 0; g < GC; ++g)
      if (lane == g) v = m[g];
    return v;
  }
};

template <>
struct GroupMasks<0> {
  uint32_t v = 0u;
  __device__ uint32_t get(int g) const {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, g);
  }
  __device__ int fit(uint32_t w, int G) const {
    int f = G;
    for (int g = 0; g < G; ++g)
      if (f == G && (get(g) & w) == 0u) f = g;
    return f;
  }
  __device__ void add(int gj, uint32_t mj, int lane) {  // gj >= G adds nothing
    if (lane == gj) v |= mj;
  }
  __device__ uint32_t lane_value(int) const { return v; }
};

template <bool HAS_VALUES, int GC, int NW>
__global__ void __launch_bounds__(64 * NW)
k_group_rows(const uint32_t* __restrict__ W, int64_t rows, int64_t cols, int64_t wpr,
             int64_t ldw,
             const int64_t* __restrict__ row_ptr, const float* __restrict__ values, int T, int G,
             int64_t tiles, int32_t* __restrict__ group_id, uint32_t* __restrict__ group_mask,
             float* __restrict__ group_vals, int32_t* __restrict__ member_row,
             int32_t* __restrict__ spill_cnt, int32_t* __restrict__ spill_nnz,
             int32_t* __restrict__ spill_table, int32_t* __restrict__ spill_rev,
             unsigned long long* __restrict__ grouped_nnz, int64_t per_xcd) {
  // All NW waves load words and store results, the first alone places rows (that
  // is sequential, and what bounds the kernel).
  __shared__ uint32_t s_word[kGroupPF * 64];   // the words of a group of chunks
  __shared__ uint8_t s_gid[kGroupPF * 64];     // group of the rows that joined one
  __shared__ uint64_t s_joined[kGroupPF];      // which rows of a chunk those are
  __shared__ int32_t s_base[kGroupPF + 1];     // spilled rows before a chunk
  __shared__ int32_t s_nnz[NW];
  const int lane = lane_id();
  const int wave = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // XCD-contiguous tile ranges: the tiles of neighbouring words of the same
  // rows share an XCD, so the 128-byte lines of group_id they fill together
  // are merged in one L2 before they are written
  for (int64_t b = blockIdx.x; b < 8 * per_xcd; b += gridDim.x) {
    const int64_t t = (b & 7) * per_xcd + (b >> 3);
    if (t >= tiles) continue;
    const int64_t rt = t / wpr, w = t - rt * wpr;
    const int64_t row0 = rt * T;
    const int64_t rem = rows - row0;
    const int nrows = rem < T ? (int)rem : T;
    GroupMasks<GC> gms;
    // 0/1 masks with a compile-time group count: lane i < 32 holds the member
    // row of bit i of each group, written once per tile
    constexpr bool kRegMembers = !HAS_VALUES && GC > 0;
    constexpr bool kRefit = NW > 1 && (GC == 1 || GC == 2);
    int32_t mem[GC > 0 ? GC : 1];
#pragma unroll
    for (int g = 0; g < (GC > 0 ? GC : 1); ++g) mem[g] = -1;
    int32_t cnt = 0;       // spilled rows so far (the first wave's; wave-uniform)
    int32_t snnz_lane = 0;
    // one chunk of 64 rows, in row order (the first-fit order).  The lanes that
    // fit some group are the candidates; the first of them joins its group (its
    // word read with v_readlane), and the candidates are taken anew from the
    // later rows.  The group masks only grow, so a row passed over would not
    // have fitted in its turn: this is the serial ascending-row first fit
    // exactly, in as many steps as rows join.  With more than two groups, where
    // testing all rows again costs more than passing over some, and in short
    // tiles, where most candidates join, it steps through the chunk's candidates.
    auto chunk = [&](int j0, uint32_t m, int u) {
      int32_t gid = 0;
      const uint64_t nz = __ballot(m != 0u);
      uint64_t cand = __ballot(m != 0u && gms.fit(m, G) < G);
      uint64_t joined = 0;
      while (cand) {
        const int jl = (int)__builtin_ctzll(cand);
        const uint32_t mj = (uint32_t)__builtin_amdgcn_readlane((int)m, jl);
        const int gj = gms.fit(mj, G);
        const bool ok = gj < G;
        joined |= (uint64_t)ok << jl;
        gid = lane == jl && ok ? gj : gid;
        gms.add(gj, mj, lane);
        if constexpr (kRegMembers) {
          const bool mine = (mj & wbit(lane & 31)) != 0u;
#pragma unroll
          for (int g = 0; g < (GC > 0 ? GC : 1); ++g) mem[g] = mine && g == gj ? j0 + jl : mem[g];
        } else if (ok) {
          int64_t vbase = 0;
          if (HAS_VALUES) {
            const int64_t r = row0 + j0 + jl;
            int64_t part = 0;
            for (int64_t x = lane; x < w; x += 64) part += __popc(W[r * ldw + x]);  // full words
            vbase = row_ptr[r] + wave_sum(part);
          }
          if (lane < 32 && (mj & wbit(lane))) {
            const int64_t idx = (t * G + gj) * 32 + lane;
            if (member_row) member_row[idx] = j0 + jl;
            group_vals[idx] = HAS_VALUES ? values[vbase + rank_before(mj, lane)] : 1.0f;
          }
        }
        if constexpr (kRefit) cand = __ballot(m != 0u && gms.fit(m, G) < G) & ~((2ull << jl) - 1ull);
        else cand &= cand - 1ull;
      }
      const uint64_t spillers = nz & ~joined;
      if constexpr (NW > 1) {
        if (joined) s_gid[u * 64 + lane] = (uint8_t)gid;
        if (lane == 0) {
          s_joined[u] = joined;
          s_base[u] = cnt;
        }
      } else {  // the row's result in place of its word: (slot + 1) << 8 | (group + 1)
        int32_t slot = -1;
        if ((spillers >> lane) & 1ull) {
          slot = cnt + __popcll(spillers & ((1ull << lane) - 1ull));
          gid = -1;
          snnz_lane += __popc(m);
        }
        s_word[u * 64 + lane] = ((uint32_t)(slot + 1) << 8) | (uint32_t)(gid + 1);
      }
      cnt += __popcll(spillers);
    };
    const uint32_t vb = valid_bits(w, cols);
    // a single wave meets its own lanes' LDS words alone and needs no barrier
    auto sync = [] {
      if constexpr (NW > 1) __syncthreads();
    };
    for (int b0 = 0; b0 < nrows; b0 += 64 * kGroupPF) {
      const int nch = min(kGroupPF, (nrows - b0 + 63) / 64);
      // a wave's chunks are wave, wave + NW, ..: their words are all loaded before
      // the first is placed, four chunks at a time under a wave-uniform test,
      // unconditional within it (rows past the tile read its last row and are
      // zeroed)
      if (b0) sync();  // the words before have been read
      constexpr int kPer = kGroupPF / NW;
      uint32_t mm[kPer];
#pragma unroll
      for (int q = 0; q < kPer; q += 4) {
        if (NW * q < nch) {
#pragma unroll
          for (int x = q; x < q + 4; ++x) {
            const int j = b0 + 64 * (NW * x + wave) + lane;
            mm[x] = W[(row0 + (j < nrows ? j : nrows - 1)) * ldw + w];
          }
        }
      }
#pragma unroll
      for (int q = 0; q < kPer; q += 4) {
        if (NW * q < nch) {
#pragma unroll
          for (int x = q; x < q + 4; ++x) {
            const int u = NW * x + wave;
            s_word[u * 64 + lane] = b0 + 64 * u + lane < nrows ? mm[x] & vb : 0u;
          }
        }
      }
      sync();
      if (wave == 0) {
        uint32_t next = s_word[lane];
#pragma unroll 1
        for (int u = 0; u < nch; ++u) {
          // (a chunk ahead, except with many groups: 3% slower there)
          const uint32_t m = GC > 0 ? next : s_word[u * 64 + lane];
          if (GC > 0) next = s_word[(u + 1 < nch ? u + 1 : u) * 64 + lane];
          chunk(b0 + 64 * u, m, u);
        }
        if (NW > 1 && lane == 0) s_base[kGroupPF] = cnt;
      }
      sync();
#pragma unroll(NW > 1 ? 2 : 1)
      for (int u = wave; u < nch; u += NW) {
        const int j = b0 + 64 * u + lane;
        const uint32_t m = s_word[u * 64 + lane];
        int32_t gid, slot;
        if constexpr (NW > 1) {
          const bool joined = (s_joined[u] >> lane) & 1ull;
          const bool spill = m != 0u && !joined;
          const uint64_t spillers = __ballot(spill);
          slot = spill ? s_base[u] + __popcll(spillers & ((1ull << lane) - 1ull)) : -1;
          gid = joined ? (int32_t)s_gid[u * 64 + lane] : spill ? -1 : 0;
          if (spill) snnz_lane += __popc(m);
        } else {
          slot = (int32_t)(m >> 8) - 1;
          gid = (int32_t)(m & 0xffu) - 1;
        }
        if (j < nrows) {
          group_id[(row0 + j) * ldw + w] = gid;
          if (spill_rev) spill_rev[t * T + j] = slot;
          if (spill_table && slot >= 0) spill_table[t * T + slot] = j;
        }
      }
    }
    int32_t snnz = wave_sum(snnz_lane);  // of this wave's chunks
    if constexpr (NW > 1) {
      cnt = __builtin_amdgcn_readfirstlane(s_base[kGroupPF]);
      if (lane == 0) s_nnz[wave] = snnz;
      __syncthreads();
    }
    if (spill_rev)
      for (int j = nrows + threadIdx.x; j < T; j += 64 * NW) spill_rev[t * T + j] = -1;
    if (spill_table)
      for (int s = cnt + threadIdx.x; s < T; s += 64 * NW) spill_table[t * T + s] = 0;
    if (wave != 0) continue;
    if constexpr (kRegMembers) {
#pragma unroll
      for (int g = 0; g < (GC > 0 ? GC : 1); ++g) {
        if (lane < 32) {
          const bool set = (gms.get(g) & wbit(lane)) != 0u;
          const int64_t idx = (t * G + g) * 32 + lane;
          group_vals[idx] = set ? 1.0f : 0.0f;
          if (member_row) member_row[idx] = set ? mem[g] : -1;
        }
      }
    } else {
      for (int g = 0; g < G; ++g) {
        const uint32_t gmg = gms.get(g);
        if (lane < 32 && !(gmg & wbit(lane))) {
          const int64_t idx = (t * G + g) * 32 + lane;
          group_vals[idx] = 0.0f;
          if (member_row) member_row[idx] = -1;
        }
      }
    }
    const uint32_t gm_lane = gms.lane_value(lane);
    if (lane < G) group_mask[t * G + lane] = gm_lane;
    if constexpr (NW > 1) {
      snnz = 0;
#pragma unroll
      for (int x = 0; x < NW; ++x) snnz += s_nnz[x];
    }
    const int32_t tile_nnz = wave_sum(lane < G ? __popc(gm_lane) : 0);
    if (lane == 0) {
      spill_cnt[t] = cnt;
      spill_nnz[t] = snnz;
      if (grouped_nnz) atomicAdd(grouped_nnz, (unsigned long long)tile_nnz);
    }
  }
}

template <bool HAS_VALUES>
__global__ void __launch_bounds__(kBlock)
k_group_spilled_csr(const uint32_t* __restrict__ W, int64_t cols, int64_t wpr, int64_t ldw,
                    const int64_t* __restrict__ row_ptr, const float* __restrict__ values,
                    const int32_t* __restrict__ woff, int T, int64_t tiles,
                    const int32_t* __restrict__ spill_cnt, const int32_t* __restrict__ spill_table,
                    const int32_t* __restrict__ row_off, const int32_t* __restrict__ nnz_off,
                    int32_t* __restrict__ row_end, int32_t* __restrict__ col,
                    float* __restrict__ val) {
  const int lane = lane_id();
  for (int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); t < tiles;
       t += (int64_t)gridDim.x * 4) {
    const int64_t rt = t / wpr, w = t - rt * wpr;
    const int cnt = spill_cnt[t];
    const int32_t roff = row_off[t], noff = nnz_off[t];
    int32_t carry = 0;
    for (int s0 = 0; s0 < cnt; s0 += 64) {
      const int s = s0 + lane;
      const bool valid = s < cnt;
      const int64_t r = rt * T + (valid ? spill_table[t * T + s] : 0);
      uint32_t m = valid ? (W[r * ldw + w] & valid_bits(w, cols)) : 0u;
      const int32_t p = __popc(m);
      const int32_t incl = wave_incl_scan(p);
      int32_t e = noff + carry + incl - p;
      if (valid) row_end[roff + s] = carry + incl;
      int64_t vb = HAS_VALUES && valid ? row_ptr[r] + woff[r * wpr + w] : 0;
      while (m) {
        const int i = __clz(m);
        m &= ~wbit(i);
        col[e] = i;
        val[e] = HAS_VALUES ? values[vb++] : 1.0f;
        ++e;
      }
      carry += __builtin_amdgcn_readlane(incl, 63);
    }
  }
}

template <bool GATHER>
__global__ void __launch_bounds__(kBlock)
k_group_scatter(const uint32_t* __restrict__ W, int64_t rows, int64_t cols, int64_t wpr,
                int64_t ldw,
                const int32_t* __restrict__ group_id, float* __restrict__ group_vals, int T,
                int G, float* __restrict__ D, int64_t ld) {
  const int64_t n = rows * wpr;
  for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * kBlock) {
    const int64_t r = e / wpr, w = e - r * wpr;
    const int32_t g = group_id[r * ldw + w];
    if (g < 0) continue;
    const int64_t t = (r / T) * wpr + w;
    uint32_t m = W[r * ldw + w] & valid_bits(w, cols);
    while (m) {
      const int i = __clz(m);
      m &= ~wbit(i);
      float* gv = &group_vals[(t * G + g) * 32 + i];
      float* d = &D[r * ld + 32 * w + i];
      if (GATHER) *gv = *d;
      else *d = *gv;
    }
  }
}

inline int grid_for(int64_t items, int64_t per_block) {
  int64_t g = ceil_div(items, per_block);
  if (g < 1) g = 1;
  if (g > 65536) g = 65536;
  return (int)g;
}

}  // namespace
}  // namespace bws

using namespace bws;

extern "C" {

int64_t bws_group_tiles(int64_t rows, int64_t cols, int32_t tile_rows) {
  if (rows < 0 || cols < 0 || tile_rows < 1) return -1;
  return ceil_div(rows, tile_rows) * words_for(cols);
}

bws_status bws_group_rows(const bws_bitmap* A, int32_t tile_rows, int32_t max_groups,
                          const bws_groups* out, bws_stream stream) {
  BWS_TRY(check_bitmap(A, false));
  if (tile_rows < 1 || tile_rows > 65536 || max_groups < 1 || max_groups > 32 || !out)
    return BWS_EINVAL;
  const int64_t tiles = bws_group_tiles(A->rows, A->cols, tile_rows);
  if (tiles > 0 && (!out->group_id || !out->group_mask || !out->group_vals || !out->spill_cnt ||
                    !out->spill_nnz))
    return BWS_EINVAL;
  if (out->grouped_nnz) {
    hipLaunchKernelGGL(k_zero_i64, dim3(1), dim3(64), 0, stream, out->grouped_nnz);
  }
  if (tiles == 0) return launch_check();
  const int64_t wpr = words_for(A->cols);
  auto* gn = reinterpret_cast<unsigned long long*>(out->grouped_nnz);
  const int64_t per_xcd = ceil_div(tiles, 8);
  // a multiple of 8 (each workgroup keeps to one XCD's range), at most 65536
  const int grid = (int)(8 * per_xcd < 65536 ? 8 * per_xcd : 65536);
#define BWS_GROUP_W(HV, GC, NW)                                                             \
  hipLaunchKernelGGL((k_group_rows<HV, GC, NW>), dim3(grid), dim3(64 * NW), 0, stream,            \
                     A->words, A->rows, A->cols, wpr, A->ldw, A->row_ptr, A->values,            \
                     (int)tile_rows, (int)max_groups, tiles, out->group_id, out->group_mask,     \
                     out->group_vals, out->member_row, out->spill_cnt, out->spill_nnz,          \
                     out->spill_table, out->spill_rev, gn, per_xcd)
#define BWS_GROUP(HV, GC)                      \
  do {                                         \
    if (wide) BWS_GROUP_W(HV, GC, 4);          \
    else BWS_GROUP_W(HV, GC, 1);               \
  } while (0)
#define BWS_GROUP_G(HV)              \
  switch (max_groups) {              \
    case 1: BWS_GROUP(HV, 1); break; \
    case 2: BWS_GROUP(HV, 2); break; \
    case 3: BWS_GROUP(HV, 3); break; \
    case 4: BWS_GROUP(HV, 4); break; \
    default: BWS_GROUP_W(HV, 0, 1);  \
  }
  // Four waves where the tiles are long and few enough that the waiting ones take
  // nobody's place (us, one wave | four): 4096², 2048-row tiles, 2 groups 26.0 | 22.8,
  // 512 rows 28.1 | 25.9; 8192², 2048 rows (1024 tiles) 46.4 | 36.2, 1024 rows, 4
  // groups (2048 tiles) 57.4 | 62.0; 4096², 256 rows 38.1 | 39.1.
  const bool wide = tile_rows >= 512 && tiles <= 1024;
  if (A->values) {
    BWS_GROUP_G(true);
  } else {
    BWS_GROUP_G(false);
  }
#undef BWS_GROUP_G
#undef BWS_GROUP
#undef BWS_GROUP_W
  return launch_check();
}

size_t bws_group_spilled_workspace_size(int64_t rows, int64_t cols, int32_t tile_rows) {
  if (rows < 0 || cols < 0 || tile_rows < 1) return 0;
  const int64_t tiles = bws_group_tiles(rows, cols, tile_rows);
  Carve c(nullptr);
  c.take<int32_t>((size_t)(rows * words_for(cols)));
  c.take<char>(scan_workspace_bytes(tiles));
  return c.used + 256;
}

bws_status bws_group_spilled_csr(const bws_bitmap* A, int32_t tile_rows,
                                 const int32_t* spill_cnt, const int32_t* spill_nnz,
                                 const int32_t* spill_table, int32_t* spill_row_off,
                                 int32_t* spill_nnz_off, int32_t* row_end, int32_t* col,
                                 float* val, void* workspace, size_t workspace_bytes,
                                 bws_stream stream) {
  BWS_TRY(check_bitmap(A, false));
  if (tile_rows < 1 || tile_rows > 65536) return BWS_EINVAL;
  const int64_t tiles = bws_group_tiles(A->rows, A->cols, tile_rows);
  if (!spill_row_off || !spill_nnz_off) return BWS_EINVAL;
  if (tiles > 0 && (!spill_cnt || !spill_nnz || !spill_table || !row_end || !col || !val))
    return BWS_EINVAL;
  if (!ws_ok(workspace, workspace_bytes,
               bws_group_spilled_workspace_size(A->rows, A->cols, tile_rows)))
    return BWS_EWORKSPACE;
  const int64_t wpr = words_for(A->cols);
  Carve c(workspace);
  int32_t* woff = c.take<int32_t>((size_t)(A->rows * wpr));
  void* scan_ws = c.take<char>(scan_workspace_bytes(tiles));
  BWS_TRY(launch_exclusive_scan_i32(spill_cnt, tiles, spill_row_off, scan_ws, stream));
  BWS_TRY(launch_exclusive_scan_i32(spill_nnz, tiles, spill_nnz_off, scan_ws, stream));
  if (tiles == 0) return BWS_OK;
  if (A->values) {
    BWS_TRY(launch_word_offsets(A->words, A->rows, A->cols, A->ldw, woff, stream));
    hipLaunchKernelGGL(k_group_spilled_csr<true>, dim3(grid_for(tiles, 4)), dim3(kBlock), 0,
                       stream, A->words, A->cols, wpr, A->ldw, A->row_ptr, A->values, woff,
                       (int)tile_rows, tiles, spill_cnt, spill_table, spill_row_off,
                       spill_nnz_off, row_end, col, val);
  } else {
    hipLaunchKernelGGL(k_group_spilled_csr<false>, dim3(grid_for(tiles, 4)), dim3(kBlock), 0,
                       stream, A->words, A->cols, wpr, A->ldw, A->row_ptr, A->values, woff,
                       (int)tile_rows, tiles, spill_cnt, spill_table, spill_row_off,
                       spill_nnz_off, row_end, col, val);
  }
  return launch_check();
}

bws_status bws_group_scatter(const uint32_t* W, int64_t rows, int64_t cols, int64_t ldw,
                             const int32_t* group_id, const float* group_vals,
                             int32_t tile_rows, int32_t max_groups, float* D, int64_t ld,
                             bws_stream stream) {
  if (!dims_ok(rows, cols) || !ldw_ok(cols, ldw) || !ld_ok(cols, ld)) return BWS_EINVAL;
  if (tile_rows < 1 || tile_rows > 65536 || max_groups < 1 || max_groups > 32) return BWS_EINVAL;
  if (rows == 0 || cols == 0) return BWS_OK;
  if (!W || !group_id || !group_vals || !D) return BWS_EINVAL;
  const int64_t wpr = words_for(cols);
  hipLaunchKernelGGL(k_group_scatter<false>, dim3(grid_for(rows * wpr, kBlock)), dim3(kBlock), 0,
                     stream, W, rows, cols, wpr, ldw, group_id, const_cast<float*>(group_vals),
                     (int)tile_rows, (int)max_groups, D, ld);
  return launch_check();
}

bws_status bws_group_gather(const float* D, int64_t ld, const uint32_t* W, int64_t rows,
                            int64_t cols, int64_t ldw, const int32_t* group_id,
                            int32_t tile_rows, int32_t max_groups, float* group_vals,
                            bws_stream stream) {
  if (!dims_ok(rows, cols) || !ldw_ok(cols, ldw) || !ld_ok(cols, ld)) return BWS_EINVAL;
  if (tile_rows < 1 || tile_rows > 65536 || max_groups < 1 || max_groups > 32) return BWS_EINVAL;
  if (rows == 0 || cols == 0) return BWS_OK;
  if (!W || !group_id || !group_vals || !D) return BWS_EINVAL;
  const int64_t wpr = words_for(cols);
  hipLaunchKernelGGL(k_group_scatter<true>, dim3(grid_for(rows * wpr, kBlock)), dim3(kBlock), 0,
                     stream, W, rows, cols, wpr, ldw, group_id, group_vals, (int)tile_rows,
                     (int)max_groups, const_cast<float*>(D), ld);
  return launch_check();
}

}  // extern "C"
