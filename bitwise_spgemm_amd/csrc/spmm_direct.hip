// spmm_direct.hip — FP32 product of a 0/1 bitmap on the matrix cores in one
// launch without a workspace, for outputs too small to fill the chip with the
// vector-add kernels' tiles (gfx950, v_mfma_f32_16x16x32_bf16, split3.hpp).
//
// Workgroup: DW waves and one 64 x 64 tile of C.  Each wave computes the whole
// tile over every DW-th 32-row K step, so no two waves share a B value: a wave
// loads its B values straight from global memory in MFMA fragment order, splits
// them in registers and multiplies, without LDS or a barrier in the loop.  The
// partial tiles are added through LDS at the end, in the order of the waves.
//
// Columns: lane (j = l % 16, q = l / 16) loads the four columns 4j .. 4j+3 of
// each of its K rows 8q .. 8q+7 with one 16-byte load, and MFMA tile b takes
// column 4j + b of them as its index j.  Its outputs then hold columns
// 16q + 4e + b in accumulator e: the four tiles' accumulators e of a lane are
// four neighbouring columns.
#include "split3.hpp"

namespace bws {
namespace {

constexpr int kDT = 64;        // tile rows and columns
constexpr int kDA = kDT / 16;  // MFMA tiles each way
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

// hi, mid and lo of column c of eight K rows, and the smallest 2|b| - 1 seen
// (unsigned, so that zero is the largest).
__device__ __forceinline__ void split8(const f32x4 (&v)[8], int c, uint4& hi, uint4& mid,
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

template <int DW>
__global__ void __launch_bounds__(DW * 64, 2)
k_spmm_direct(const uint32_t* __restrict__ W, int64_t M, int64_t K, int64_t ldw,
              const float* __restrict__ B, int64_t ldb, int64_t N, float* __restrict__ C,
              int64_t ldc, float alpha, float beta, int64_t row_blocks, int64_t col_blocks,
              int64_t per_xcd, int vec) {
  __shared__ f32x4 part[DW / 2][kDA * kDA][64];
  __shared__ uint32_t tiny;
  const int64_t tile = xcd_tile(blockIdx.x, per_xcd);
  if (tile >= row_blocks * col_blocks) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t cb = tile / row_blocks, rb = tile - cb * row_blocks;
  const int64_t m0 = rb * kDT, n0 = cb * kDT;
  const int j = lane & 15, q = lane >> 4;
  const int nks = (int)ceil_div(K, 32);
  if (threadIdx.x == 0) tiny = 0u;

  // the rows' bitmap words (rows past M read row M - 1, never stored)
  uint32_t arow[kDA];
#pragma unroll
  for (int a = 0; a < kDA; ++a) {
    const int64_t row = m0 + 16 * a + j;
    arow[a] = (uint32_t)((row < M ? row : M - 1) * ldw);
  }
  const int64_t lcol = n0 + 4 * j;
  const int64_t lclamp = lcol + 4 <= N ? lcol : (N >= 4 ? N - 4 : 0);
  const int shift = (int)(lcol - lclamp < 4 ? lcol - lclamp : 0);
  const uint32_t loff = (uint32_t)((8 * q * ldb + lclamp) * 4);
  const bool partial_quad = N % 4 != 0 && n0 + kDT > N;
  const int nfull = N >= 4 ? (int)(K / 32) : 0;  // a narrower B takes the tail path throughout
  struct Raw {
    f32x4 v[8];
    uint32_t w[kDA];
  };
  // a full step (32 rows below K): one code path of 12 loads, so that the wait
  // for a step's loads is not a wait for the next one's; past the last step the
  // last one is loaded again
  auto load = [&](int s, Raw& r) {
    s = s < nfull ? s : nfull - 1;
#pragma unroll
    for (int a = 0; a < kDA; ++a) r.w[a] = W[arow[a] + (uint32_t)s];
    const float* p = B + (int64_t)s * 32 * ldb;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      r.v[e] = *reinterpret_cast<const f32x4_u*>(reinterpret_cast<const char*>(p + e * ldb) + loff);
  };
  // any step: rows past K read row K - 1 and meet zero bits, columns past N
  // read column N - 1 and are not stored
  auto load_tail = [&](int s, Raw& r) {
#pragma unroll
    for (int a = 0; a < kDA; ++a) r.w[a] = W[arow[a] + (uint32_t)s];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int64_t k = 32 * (int64_t)s + 8 * q + e;
      const float* p = B + (k < K ? k : K - 1) * ldb;
#pragma unroll
      for (int c = 0; c < 4; ++c) r.v[e][c] = p[lcol + c < N ? lcol + c : N - 1];
    }
  };

  // the sums of hi and of mid and lo apart: the chain of the larger ones is
  // a third as long, and the roundings of the smaller ones do not count
  f32x4 acc[kDA][kDA], low[kDA][kDA];
#pragma unroll
  for (int a = 0; a < kDA; ++a)
#pragma unroll
    for (int b = 0; b < kDA; ++b) acc[a][b] = low[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t least = 0xFFFFFFFFu;

  auto multiply = [&](int s, Raw& r, bool fresh, auto next) {
    const uint32_t vb = valid_bits(s, K);
    uint4 af[kDA];
#pragma unroll
    for (int a = 0; a < kDA; ++a) af[a] = a_frag01(__brev(r.w[a] & vb), q);
    if (fresh && partial_quad) {  // the quad that holds column N - 1, loaded from N - 4 on
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        f32x4 v = r.v[e];
        if (shift == 1) v = f32x4{v[1], v[2], v[3], v[3]};
        if (shift == 2) v = f32x4{v[2], v[3], v[3], v[3]};
        if (shift == 3) v = f32x4{v[3], v[3], v[3], v[3]};
        r.v[e] = v;
      }
    }
#pragma unroll
    for (int b = 0; b < kDA; ++b) {
      uint4 hi, mid, lo;
      split8(r.v, b, hi, mid, lo, least);
      if (b == kDA - 1) next();  // r's registers are free
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < kDA; ++a) acc[a][b] = mfma<1>(hi, af[a], acc[a][b]);
#pragma unroll
      for (int a = 0; a < kDA; ++a) low[a][b] = mfma<1>(lo, af[a], low[a][b]);
#pragma unroll
      for (int a = 0; a < kDA; ++a) low[a][b] = mfma<1>(mid, af[a], low[a][b]);
    }
  };
  Raw r0;
  int s = wave;
  if (s < nfull) {
    load(s, r0);
    for (; s < nfull; s += DW) multiply(s, r0, true, [&] { load(s + DW, r0); });
  }
  for (; s < nks; s += DW) {
    load_tail(s, r0);
    multiply(s, r0, false, [] {});
  }
#pragma unroll
  for (int a = 0; a < kDA; ++a)
#pragma unroll
    for (int b = 0; b < kDA; ++b) acc[a][b] += low[a][b];

  // partial tiles: the upper half of the waves through LDS into the lower half,
  // then those
  __syncthreads();
  if (least < 2u * kTinyBits - 1u) tiny = 1u;
  if (wave >= DW / 2) {
#pragma unroll
    for (int i = 0; i < kDA * kDA; ++i) part[wave - DW / 2][i][lane] = acc[i / kDA][i % kDA];
  }
  __syncthreads();
  if (wave < DW / 2) {
#pragma unroll
    for (int i = 0; i < kDA * kDA; ++i) {
      acc[i / kDA][i % kDA] += part[wave][i][lane];
      part[wave][i][lane] = acc[i / kDA][i % kDA];
    }
  }
  __syncthreads();
  const bool any_tiny = tiny != 0u;

  // row tile a, accumulator e of lane (j, q): row 16a + j, columns 16q + 4e .. +3;
  // wave w stores the quads (a, e) with 4a + e in [w PER, (w + 1) PER)
  constexpr int PER = kDA * 4 / DW;
#pragma unroll
  for (int x = 0; x < PER; ++x) {
    const int i = wave * PER + x, a = i >> 2, e = i & 3;
    const int64_t row = m0 + 16 * a + j, col = n0 + 16 * q + 4 * e;
    if (row >= M || col >= N) continue;
    f32x4 v;
#pragma unroll
    for (int b = 0; b < kDA; ++b) {
      const float* p = reinterpret_cast<const float*>(&part[0][a * kDA + b][lane]) + e;
      float t = p[0];
#pragma unroll
      for (int w = 1; w < DW / 2; ++w) t += p[w * (kDA * kDA * 64 * 4)];
      v[b] = t;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if ((out_of_range(v[b]) || (any_tiny && v[b] == 0.0f)) && col + b < N)
        v[b] = row_sum(W + row * ldw, K, B + col + b, ldb);
    v *= alpha;
    float* c = C + row * ldc + col;
    if (vec && col + 3 < N) {
      if (beta != 0.0f) {
        const f32x4 o = *reinterpret_cast<const f32x4*>(c);
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = fmaf(beta, o[b], v[b]);
      }
      *reinterpret_cast<f32x4*>(c) = v;
    } else {
#pragma unroll
      for (int b = 0; b < 4; ++b)
        if (col + b < N) c[b] = beta != 0.0f ? fmaf(beta, c[b], v[b]) : v[b];
    }
  }
}

}  // namespace

// bws_spmm: outputs of up to kDirectTiles = 512 tiles (2^21 elements): within them the product takes
// 0.4 to 0.95 of the vector-add kernels' time at 1% density and less above
// (those walk K at one workgroup's pace whatever the mask holds): 1024³ 14 us
// against 26 (1%) to 92 (50%), 4096 x 1024 x 512 23 against 26 to 93, 4096² x 512
// 58 against 91 to 358.  Beyond, at 2048³, it is 63 against 52 (1%), 62 (5%), 77
// (10%).
bool spmm_direct_ok(const bws_bitmap* A, int64_t ldb, int64_t N, int64_t max_tiles) {
  const int64_t rows = ceil_div(A->rows, kDT), cols = ceil_div(N, kDT);
  return rows <= max_tiles && cols <= max_tiles && rows * cols <= max_tiles &&
         A->cols < ((int64_t)1 << 31) &&                            // 32-bit steps,
         A->rows * A->ldw < ((int64_t)1 << 32) && ldb < (1 << 24);  // and offsets
}

bws_status launch_spmm_direct(const bws_bitmap* A, const float* B, int64_t ldb, int64_t N,
                              float* C, int64_t ldc, float alpha, float beta, hipStream_t s) {
  const int64_t row_blocks = ceil_div(A->rows, kDT), col_blocks = ceil_div(N, kDT);
  const int64_t tiles = row_blocks * col_blocks, per_xcd = ceil_div(tiles, 8);
  const int vec = ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
  const dim3 grid((unsigned)(8 * per_xcd));
  // eight waves where the tiles leave CUs idle (128 tiles, K = 4096: 31.5 us
  // against 35.1), four where workgroups share CUs (512 tiles: 58 against 61)
  if (tiles <= 192)
    hipLaunchKernelGGL(k_spmm_direct<8>, grid, dim3(512), 0, s, A->words, A->rows, A->cols, A->ldw,
                       B, ldb, N, C, ldc, alpha, beta, row_blocks, col_blocks, per_xcd, vec);
  else
    hipLaunchKernelGGL(k_spmm_direct<4>, grid, dim3(256), 0, s, A->words, A->rows, A->cols, A->ldw,
                       B, ldb, N, C, ldc, alpha, beta, row_blocks, col_blocks, per_xcd, vec);
  return launch_check();
}

}  // namespace bws
