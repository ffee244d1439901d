// spmm_direct.hip — FP32 product of a 0/1 bitmap on the matrix cores in one
// launch without a workspace, for outputs too small to fill the chip with the
// vector-add kernels' tiles (gfx950, v_mfma_f32_16x16x32_bf16, split3.hpp).
//
// Workgroup: DW waves and one 128 x 32 tile of C.  Each wave computes the whole
// tile over every DW-th 32-row K step, so no two waves share a B value: a wave
// loads its B values straight from global memory in MFMA fragment order, splits
// them in registers and multiplies, without a barrier in the loop.  The rows'
// bitmap words go through LDS once per 4096 K columns: read from global memory
// step by step they were four times B's traffic, a cache line per row for 4 bytes
// of it.  The partial tiles are added through LDS at the end.
//
// What bounds it is the vector unit: an MFMA leaves room for about two vector
// operations (7.0, 7.2, 7.4, 8.8, 10.6 ns per MFMA and SIMD with 0 to 4), and a
// step is 48 MFMAs, 120 operations of splitting (7.5 per value of B) and 80 of
// building A's operands (10 per row tile).  A tile of R x C MFMA tiles takes
// 60 C + 10 R of them for 12 R C MFMAs: with R C = 16 (the accumulators) 8 x 2 is
// the least.  64 x 64 tiles (4 x 4, 280 operations) measured 3001 x 2053 x 516
// 32.5 us against 26.2, 2048 x 2048 x 1024 31.5 against 25.8, 500 x 2000 x 300
// 19.0 against 14.7.  Taking the upper halves off with dot products
// (v_dot2_f32_bf16, exact, 20% fewer operations) was slower: they do not run
// beside the MFMAs.
//
// Columns: lane (j = l % 16, q = l / 16) loads the two columns 2j, 2j + 1 of each
// of its K rows 8q .. 8q+7 with one 8-byte load, and MFMA tile b takes column
// 2j + b of them as its index j.  Its outputs then hold columns 8q + 2e + b in
// accumulator e: a lane's accumulators of a row are eight neighbouring columns.
#include "split3.hpp"

#include <type_traits>

namespace bws {
namespace {

constexpr int kDM = 128, kDN = 32;            // tile rows and columns
constexpr int kDA = kDM / 16, kDB = kDN / 16;  // MFMA tiles down and across
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2_u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

// hi, mid and lo of column c of eight K rows, and the smallest 2|b| - 1 seen
// (unsigned, so that zero is the largest).
__device__ __forceinline__ void split8(const f32x2_u (&v)[8], int c, uint4& hi, uint4& mid,
                                       uint4& lo, uint32_t& least) {
  uint32_t h[8], m[8], l[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t u = __float_as_uint(v[e][c]);
    h[e] = u & 0xFFFF0000u;
    const float r = v[e][c] - __uint_as_float(h[e]);  // exact
    m[e] = __float_as_uint(r) & 0xFFFF0000u;
    l[e] = __float_as_uint(r - __uint_as_float(m[e]));  // exact, 8 bits
    least = min(least, 2u * u - 1u);
  }
  // the upper halves of two values in one word
  auto up = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); };
  hi = make_uint4(up(h[0], h[1]), up(h[2], h[3]), up(h[4], h[5]), up(h[6], h[7]));
  mid = make_uint4(up(m[0], m[1]), up(m[2], m[3]), up(m[4], m[5]), up(m[6], m[7]));
  lo = make_uint4(up(l[0], l[1]), up(l[2], l[3]), up(l[4], l[5]), up(l[6], l[7]));
}

// x is not to be trusted: not finite, or below kSmallOut where some b was tiny.
__device__ __forceinline__ bool not_exact(float x, bool any_tiny) {
  const float m = fabsf(x);
  return !(m < __builtin_inff()) || (any_tiny && m < kSmallOut);
}

// A wave's outputs once more as FP32 sums over the set bits, ascending k, as the
// vector-add kernels form them: sums[x][i] of row row0 + 16x + j, column n0 + 8q + i.
// 128 rows of B at a time go through the LDS that held the partial tiles of these
// rows, which no other wave reads (16 KiB in DW pieces, part_bytes apart; 16-byte
// units swizzled by the row); a lane walks its row's bits, four in flight.  The waves
// do it by themselves: a barrier at the kernel's end, good or bad outputs, kept the
// next workgroup off the CU (703 x 3181 x 3984, 750 tiles, 61 us then 66).  Bound by
// LDS reads, a row of B per set bit.  Us for ordinary B, for B with an Inf in every
// column and for the vector-add kernel on that B (output by output it was 305, 885 and
// 735 at the first, second and fourth):
//   1024 x 1024 x 1024, 10% of A   12.5   54  41     (50%  12.4  112   94)
//   2048 x 1024 x 2048,  5%        30    116  36     (50%  31    336   96)
//   4095 x 2000 x 2047, 10%       115    577 253
//   256 x 512 x 192,     5%         8.8   25  18
// Loading the next 128 rows ahead of the sums gave nothing (55 and 113 at the first).
template <int DW>
__device__ __forceinline__ void vector_sums(const uint32_t* __restrict__ W, int64_t M, int64_t K,
                                            int64_t ldw, const float* __restrict__ B, int64_t ldb,
                                            int64_t N, int64_t row0, int64_t n0, uint8_t* own,
                                            uint32_t part_bytes, float (&sums)[kDA / DW][8]) {
  constexpr int NX = kDA / DW;
  constexpr uint32_t kPieceRows = 16 * NX;
  static_assert(kPieceRows * DW == 128 && kDN * 4 == 128, "four bitmap words, 128 bytes a row");
  const int lane = threadIdx.x & 63;
  const int j = lane & 15, q = lane >> 4;
  const int64_t nks = ceil_div(K, 32);
  auto at = [&](uint32_t k, uint32_t unit) {
    return reinterpret_cast<f32x4*>(own + (k / kPieceRows) * part_bytes + (k % kPieceRows) * 128u +
                                    ((unit ^ (k & 7u)) << 4));
  };
#pragma unroll
  for (int x = 0; x < NX; ++x)
#pragma unroll
    for (int i = 0; i < 8; ++i) sums[x][i] = 0.0f;
  for (int64_t w0 = 0; w0 < nks; w0 += 4) {
    f32x4 v[16];
    uint32_t wd[NX][4];
    const int64_t c = n0 + 4 * (lane & 7);
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int64_t k = 32 * w0 + 8 * u + (lane >> 3);
      const float* p = B + (k < K ? k : K - 1) * ldb;
      if (c + 4 <= N) {
        v[u] = *reinterpret_cast<const f32x4_u*>(p + c);
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) v[u][t] = p[c + t < N ? c + t : N - 1];
      }
    }
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int64_t row = row0 + 16 * x + j;
      const uint32_t* wp = W + (row < M ? row : M - 1) * ldw + w0;
#pragma unroll
      for (int t = 0; t < 4; ++t) wd[x][t] = w0 + t < nks ? wp[t] & valid_bits(w0 + t, K) : 0u;
    }
    asm volatile("" ::: "memory");  // (a wave's LDS accesses stay in order)
#pragma unroll
    for (int u = 0; u < 16; ++u) *at(8 * u + (lane >> 3), lane & 7) = v[u];
    asm volatile("" ::: "memory");
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
      for (int t = 0; t < 4; t += 2) {
        uint64_t m = ((uint64_t)wd[x][t] << 32) | wd[x][t + 1];
        while (m) {
          f32x4 b[4][2];
          bool on[4];
          uint32_t k = 0;
#pragma unroll
          for (int e = 0; e < 4; ++e) {  // past the last bit: its row again, not added
            on[e] = m != 0ull;
            if (on[e]) {
              const int z = __clzll((long long)m);
              m &= ~(1ull << (63 - z));
              k = 32u * t + (uint32_t)z;
            }
            b[e][0] = *at(k, 2 * q);
            b[e][1] = *at(k, 2 * q + 1);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (on[e]) {
#pragma unroll
              for (int i = 0; i < 8; ++i) sums[x][i] += b[e][i >> 2][i & 3];
            }
        }
      }
    asm volatile("" ::: "memory");
  }
}

template <int DW>
__global__ void __launch_bounds__(DW * 64, 2)
k_spmm_direct(const uint32_t* __restrict__ W, int64_t M, int64_t K, int64_t ldw,
              const float* __restrict__ B, int64_t ldb, int64_t N, float* __restrict__ C,
              int64_t ldc, float alpha, float beta, int64_t row_blocks, int64_t col_blocks,
              int64_t per_xcd, int vec) {
  constexpr int kDW = 32 * DW;  // bitmap words of a row in LDS at once,
  __shared__ f32x4 part[DW][kDA * kDB][64];  // in the room of the partial tiles
  static_assert(kDW * kDM * 4 == sizeof(part), "");
  __shared__ uint32_t tiny[DW];
  uint32_t(*const words)[kDM] = reinterpret_cast<uint32_t(*)[kDM]>(&part[0][0][0]);
  const int64_t tile = xcd_tile(blockIdx.x, per_xcd);
  if (tile >= row_blocks * col_blocks) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t cb = tile / row_blocks, rb = tile - cb * row_blocks;
  const int64_t m0 = rb * kDM, n0 = cb * kDN;
  const int j = lane & 15, q = lane >> 4;
  const int nks = (int)ceil_div(K, 32);

  // words c kDW .. of the tile's rows into LDS, word by word (rows past M read row
  // M - 1 and are never stored; bits past K are zero)
  auto load_words = [&](int c) {
    const int nw = nks - c * kDW < kDW ? nks - c * kDW : kDW;
    const int units = (nw + 3) / 4 * kDM;
#pragma unroll 4
    for (int i = threadIdx.x; i < units; i += DW * 64) {
      const int r = i % kDM, w = i / kDM * 4;
      const int64_t row = m0 + r < M ? m0 + r : M - 1;
      const uint32_t* p = W + row * ldw + c * kDW + w;
      u32x4_u v;
      if (w + 4 < nw) {
        v = *reinterpret_cast<const u32x4_u*>(p);
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          v[t] = w + t < nw ? p[t] & valid_bits((int64_t)c * kDW + w + t, K) : 0u;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) words[w + t][r] = v[t];
    }
  };
  const int64_t lcol = n0 + 2 * j;
  const int64_t lclamp = lcol + 2 <= N ? lcol : (N >= 2 ? N - 2 : 0);
  const bool shift = lcol != lclamp;
  const uint32_t loff = (uint32_t)((8 * q * ldb + lclamp) * 4);
  const bool partial_pair = N % 2 != 0 && n0 + kDN > N;
  const int nfull = N >= 2 ? (int)(K / 32) : 0;  // a narrower B takes the tail path throughout
  struct Raw {
    f32x2_u v[8];
  };
  // a full step (32 rows below K): one code path of 8 loads, so that the wait
  // for a step's loads is not a wait for the next one's; past the last step the
  // last one is loaded again
  auto load = [&](int s, Raw& r) {
    s = s < nfull ? s : nfull - 1;
    const float* p = B + (int64_t)s * 32 * ldb;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      r.v[e] = *reinterpret_cast<const f32x2_u*>(reinterpret_cast<const char*>(p + e * ldb) + loff);
  };
  // any step: rows past K read row K - 1 and meet zero bits, columns past N
  // read column N - 1 and are not stored
  auto load_tail = [&](int s, Raw& r) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int64_t k = 32 * (int64_t)s + 8 * q + e;
      const float* p = B + (k < K ? k : K - 1) * ldb;
#pragma unroll
      for (int c = 0; c < 2; ++c) r.v[e][c] = p[lcol + c < N ? lcol + c : N - 1];
    }
  };

  // the sums of hi and of mid and lo apart: the chain of the larger ones is
  // a third as long, and the roundings of the smaller ones do not count
  f32x4 acc[kDA][kDB], low[kDA][kDB];
#pragma unroll
  for (int a = 0; a < kDA; ++a)
#pragma unroll
    for (int b = 0; b < kDB; ++b) acc[a][b] = low[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t least = 0xFFFFFFFFu;

  auto multiply = [&](int s, Raw& r, auto fresh, auto next) {
    if (fresh.value && partial_pair && shift) {  // column N - 1, loaded from N - 2 on
#pragma unroll
      for (int e = 0; e < 8; ++e) r.v[e][0] = r.v[e][1];
    }
    uint4 hi[kDB], mid[kDB], lo[kDB];
#pragma unroll
    for (int b = 0; b < kDB; ++b) split8(r.v, b, hi[b], mid[b], lo[b], least);
    uint32_t w[kDA];
#pragma unroll
    for (int a = 0; a < kDA; ++a) w[a] = words[s % kDW][16 * a + j];
    // the next step's loads, into r's registers, run beside all of this step's
    // MFMAs; the wave in its MFMAs goes first, the other one of its SIMD splits
    // (28.5 us without the priority where 26.7 with it)
    __builtin_amdgcn_sched_barrier(0);
    next();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int a0 = 0; a0 < kDA; a0 += 2) {
      const uint4 af[2] = {a_frag01(w[a0], q), a_frag01(w[a0 + 1], q)};
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < kDB; ++b) acc[a0 + a][b] = mfma<1>(hi[b], af[a], acc[a0 + a][b]);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < kDB; ++b) low[a0 + a][b] = mfma<1>(lo[b], af[a], low[a0 + a][b]);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < kDB; ++b) low[a0 + a][b] = mfma<1>(mid[b], af[a], low[a0 + a][b]);
#pragma unroll
      for (int i = 0; i < 6 * kDB; ++i) {  // the next row tiles' operands between them
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two VALU
      }
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  };
  Raw r0;
  int s = wave;
  if (s < nfull) load(s, r0);
  for (int c = 0; c * kDW < nks; ++c) {
    if (c) __syncthreads();
    load_words(c);
    __syncthreads();
    const int full = nfull < (c + 1) * kDW ? nfull : (c + 1) * kDW;
    for (; s < full; s += DW) multiply(s, r0, std::true_type{}, [&] { load(s + DW, r0); });
    const int end = nks < (c + 1) * kDW ? nks : (c + 1) * kDW;
    for (; s < end; s += DW) {
      load_tail(s, r0);
      multiply(s, r0, std::false_type{}, [] {});
    }
  }
#pragma unroll
  for (int a = 0; a < kDA; ++a)
#pragma unroll
    for (int b = 0; b < kDB; ++b) acc[a][b] += low[a][b];

  // partial tiles: every wave's through LDS, then each wave adds and stores its
  // share of the row tiles (waves w and w + DW / 2 first, then those in order)
  __syncthreads();  // the words have been read
#pragma unroll
  for (int i = 0; i < kDA * kDB; ++i) part[wave][i][lane] = acc[i / kDB][i % kDB];
  const bool some_tiny = __ballot(least < 2u * kTinyBits - 1u) != 0ull;
  if (lane == 0) tiny[wave] = some_tiny ? 1u : 0u;
  __syncthreads();
  uint32_t any_tiny = 0u;
#pragma unroll
  for (int w = 0; w < DW; ++w) any_tiny |= tiny[w];

  // row tile a, accumulator e of tile b of lane (j, q): row 16a + j, column
  // 8q + 2e + b.  Outputs that are not to be trusted wait (a bit each in bad).
  constexpr int NX = kDA / DW;
  uint32_t bad[NX], any_bad = 0u;
#pragma unroll
  for (int x = 0; x < NX; ++x) {
    const int a = wave * NX + x;
    const int64_t row = m0 + 16 * a + j;
    f32x4 sum[kDB];
    bad[x] = 0u;
#pragma unroll
    for (int b = 0; b < kDB; ++b) {
      const int i = a * kDB + b;
      sum[b] = part[0][i][lane] + part[DW / 2][i][lane];
#pragma unroll
      for (int w = 1; w < DW / 2; ++w) sum[b] += part[w][i][lane] + part[w + DW / 2][i][lane];
    }
    if (row >= M) continue;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t col = n0 + 8 * q + 4 * h;
      if (col >= N) continue;
      f32x4 v = {sum[0][2 * h], sum[1][2 * h], sum[0][2 * h + 1], sum[1][2 * h + 1]};
      uint32_t wait = 0u;
#pragma unroll
      for (int b = 0; b < 4; ++b)
        if (not_exact(v[b], any_tiny != 0u) && col + b < N) wait |= 1u << b;
      bad[x] |= wait << (4 * h);
      v *= alpha;
      float* c = C + row * ldc + col;
      if (vec && col + 3 < N && wait == 0u) {
        if (beta != 0.0f) {
          const f32x4 o = *reinterpret_cast<const f32x4*>(c);
#pragma unroll
          for (int b = 0; b < 4; ++b) v[b] = fmaf(beta, o[b], v[b]);
        }
        *reinterpret_cast<f32x4*>(c) = v;
      } else {
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if (col + b < N && !((wait >> b) & 1u))
            c[b] = beta != 0.0f ? fmaf(beta, c[b], v[b]) : v[b];
      }
    }
    any_bad |= bad[x];
  }
  if (__ballot(any_bad != 0u) == 0ull) return;  // (of this wave)
  float again[NX][8];
  vector_sums<DW>(W, M, K, ldw, B, ldb, N, m0 + 16 * NX * wave, n0,
                  reinterpret_cast<uint8_t*>(&part[0][wave * NX * kDB][0]), sizeof(part[0]), again);
#pragma unroll
  for (int x = 0; x < NX; ++x) {
    float* c = C + (m0 + 16 * (wave * NX + x) + j) * ldc + n0 + 8 * q;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if ((bad[x] >> i) & 1u) {
        const float v = alpha * again[x][i];
        c[i] = beta != 0.0f ? fmaf(beta, c[i], v) : v;
      }
  }
}

}  // namespace

// max_tiles: of 64 x 64 (the callers' measure of an output).
bool spmm_direct_ok(const bws_bitmap* A, int64_t ldb, int64_t N, int64_t max_tiles) {
  const int64_t rows = ceil_div(A->rows, 64), cols = ceil_div(N, 64);
  return rows <= max_tiles && cols <= max_tiles && rows * cols <= max_tiles &&
         A->cols < ((int64_t)1 << 31) && ldb < (1 << 24);  // 32-bit steps and offsets
}

bws_status launch_spmm_direct(const bws_bitmap* A, const float* B, int64_t ldb, int64_t N,
                              float* C, int64_t ldc, float alpha, float beta, hipStream_t s) {
  const int64_t row_blocks = ceil_div(A->rows, kDM), col_blocks = ceil_div(N, kDN);
  const int64_t tiles = row_blocks * col_blocks, per_xcd = ceil_div(tiles, 8);
  const int vec = ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
  auto launch = [&](auto kernel, int waves) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * per_xcd)), dim3(64 * waves), 0, s, A->words,
                       A->rows, A->cols, A->ldw, B, ldb, N, C, ldc, alpha, beta, row_blocks,
                       col_blocks, per_xcd, vec);
  };
  // as many waves a workgroup as fill the chip once (two per SIMD): with tiles of
  // 128 x 32, us with 8 | 4 | 2 waves: 1024³ (256 tiles) 10.2 | 11.8 | 19.5, 3001 x
  // 2053 x 516 (408) 29.3 | 26.2 | 45.7, 2048 x 1024 x 2048 (1024) 36.7 | 29.9 | 28.0;
  // two are slower in long products (4095³: 425 | 364 | 393)
  const int waves = tiles <= 256 ? 8 : tiles <= 512 || tiles > 1024 || A->cols > 1024 ? 4 : 2;
  if (waves == 8) launch(k_spmm_direct<8>, 8);
  else if (waves == 4) launch(k_spmm_direct<4>, 4);
  else launch(k_spmm_direct<2>, 2);
  return launch_check();
}

}  // namespace bws
