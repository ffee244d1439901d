// spmm_direct16.hip — 16-bit and split-BF16 product of a 0/1 bitmap for small
// outputs with a long K (split BF16: any K), in one launch without a workspace (gfx950, v_mfma_f32_16x16x32).
//
// The staged tiles of spmm_mfma.hip walk all of K in every workgroup, a barrier
// and an LDS round trip per stage: with few tiles that chain is the time and
// the chip is idle.  Here K is shared out: eight waves and one tile of C, each
// wave the whole tile over every eighth 32-row K step, B straight from global
// memory in MFMA fragment order (packed, and rounded if it is FP32, in
// registers), without LDS for B or a barrier in the loop.  The bitmap words go
// through LDS, the partial tiles are added through it at the end.  Any width and
// alignment of B's rows is taken as it is.
//
// Tiles of 64 x 64 while they leave CUs idle; with more of them every 64 rows
// reading all of B is what takes the time (12 TB/s out of L2 at 1999 x 3100 x
// 1000), so there they are 128 x 64.  us, staged | 64 x 64 | 128 x 64, FP16:
//   500 x 2000 x 300    14.6 | 10.0 | 13.4     1024 x 2048 x 1024  13.0 | 10.3 | 14.0
//   1024 x 4096 x 512   20.1 | 13.6 | 19.8     1999 x 3100 x 1000  25.0 | 27.6 | 19.1
//   1024 x 1024 x 1024   7.9 |  8.3 | 10.9     4096 x 4096 x 512   29.6 | 27.9 | 21.5
// Loading two to four steps ahead, which there are registers for, was slower.
//
// Columns: lane (j = l % 16, q = l / 16) loads the four columns 4j .. 4j+3 of
// each of its K rows 8q .. 8q+7 with one load, and MFMA tile b takes column
// 4j + b of them as its index j.  Its outputs then hold columns 16q + 4e + b in
// accumulator e: the four tiles' accumulators e of a lane are neighbours.
#include "mfma4_tile.hpp"

#include <type_traits>

namespace bws {
namespace {

constexpr int DW = 8;                // waves
constexpr int kEN = 64;              // tile columns
constexpr int kEB = kEN / 16;        // MFMA tiles across
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t u16x4_u __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(4)));

// PREC 1 = BF16, 2 = FP16, 3 = BF16X2 (b = hi + lo, two products); F32: B is FP32 and rounded or split; kEA: MFMA tiles down (4 or 8).
template <int PREC, bool F32, int kEA>
__global__ void __launch_bounds__(DW * 64, 2)
k_spmm_direct16(const uint32_t* __restrict__ W, int64_t M, int64_t K, int64_t ldw,
                const void* __restrict__ Bv, int64_t ldb, int64_t N, float* __restrict__ C,
                int64_t ldc, float alpha, float beta, int64_t row_blocks, int64_t col_blocks,
                int64_t per_xcd, int vec) {
  using Elem = std::conditional_t<F32, float, uint16_t>;
  using Vec = std::conditional_t<F32, f32x4_u, u16x4_u>;
  constexpr int kEM = kEA * 16;            // tile rows
  constexpr int kDW = 256 * DW / kEA;      // bitmap words of a row in LDS at once,
  __shared__ f32x4 part[DW][4 * kEB][64];  // in the room of the partial tiles
  static_assert(kDW * kEM * 4 == sizeof(part), "");
  uint32_t(*const words)[kEM] = reinterpret_cast<uint32_t(*)[kEM]>(&part[0][0][0]);
  const int64_t tile = xcd_tile(blockIdx.x, per_xcd);
  if (tile >= row_blocks * col_blocks) return;
  const Elem* __restrict__ B = static_cast<const Elem*>(Bv);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t cb = tile / row_blocks, rb = tile - cb * row_blocks;
  const int64_t m0 = rb * kEM, n0 = cb * kEN;
  const int j = lane & 15, q = lane >> 4;
  const int nks = (int)ceil_div(K, 32);

  // words c kDW .. of the tile's rows into LDS, word by word (rows past M read row
  // M - 1 and are never stored; bits past K are zero), bit reversed for a_frag_bits
  auto load_words = [&](int c) {
    const int nw = nks - c * kDW < kDW ? nks - c * kDW : kDW;
    const int units = (nw + 3) / 4 * kEM;
#pragma unroll 4
    for (int i = threadIdx.x; i < units; i += DW * 64) {
      const int r = i % kEM, w = i / kEM * 4;
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
      for (int t = 0; t < 4; ++t) words[w + t][r] = __brev(v[t]);
    }
  };
  const int64_t lcol = n0 + 4 * j;
  const int64_t lclamp = lcol + 4 <= N ? lcol : (N >= 4 ? N - 4 : 0);
  const int shift = (int)(lcol - lclamp < 4 ? lcol - lclamp : 0);
  const uint32_t loff = (uint32_t)((8 * q * ldb + lclamp) * sizeof(Elem));
  const bool partial_quad = N % 4 != 0 && n0 + kEN > N;
  const int nfull = N >= 4 ? (int)(K / 32) : 0;  // a narrower B takes the tail path throughout
  struct Raw {
    Vec v[8];
  };
  // a full step (32 rows below K): one code path of 8 loads, so that the wait for
  // a step's loads is not a wait for the next one's; past the last step the last
  // one is loaded again
  auto load = [&](int s, Raw& r) {
    s = s < nfull ? s : nfull - 1;
    const Elem* p = B + (int64_t)s * 32 * ldb;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      r.v[e] = *reinterpret_cast<const Vec*>(reinterpret_cast<const char*>(p + e * ldb) + loff);
  };
  // any step: rows past K read row K - 1 and meet zero bits, columns past N
  // read column N - 1 and are not stored
  auto load_tail = [&](int s, Raw& r) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int64_t k = 32 * (int64_t)s + 8 * q + e;
      const Elem* p = B + (k < K ? k : K - 1) * ldb;
#pragma unroll
      for (int c = 0; c < 4; ++c) r.v[e][c] = p[lcol + c < N ? lcol + c : N - 1];
    }
  };

  // BF16X2: the sums of lo apart, so that its products do not lengthen the chain
  // of the large ones (the matrix unit does not round its sums to nearest)
  constexpr int NP = PREC == 3 ? 2 : 1;
  f32x4 acc[kEA][kEB], low[PREC == 3 ? kEA : 1][kEB];
#pragma unroll
  for (int a = 0; a < kEA; ++a)
#pragma unroll
    for (int b = 0; b < kEB; ++b) {
      acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (PREC == 3) low[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  auto multiply = [&](int s, Raw& r, auto fresh, auto next) {
    if (fresh.value && partial_quad) {  // the quad that holds column N - 1, loaded from N - 4 on
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        Vec v = r.v[e];
        if (shift == 1) v = Vec{v[1], v[2], v[3], v[3]};
        if (shift == 2) v = Vec{v[2], v[3], v[3], v[3]};
        if (shift == 3) v = Vec{v[3], v[3], v[3], v[3]};
        r.v[e] = v;
      }
    }
    uint4 bf[NP][kEB];
#pragma unroll
    for (int b = 0; b < kEB; ++b) {
      uint32_t d[4], l[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        if constexpr (F32) {
          const float x0 = r.v[2 * p][b], x1 = r.v[2 * p + 1][b];
          d[p] = PREC == 2 ? f32_to_f16_rne(x0) | f32_to_f16_rne(x1) << 16
                           : f32_to_bf16_rne(x0) | f32_to_bf16_rne(x1) << 16;
          if constexpr (PREC == 3)
            l[p] = f32_to_bf16_rne(x0 - __uint_as_float(d[p] << 16)) |
                   f32_to_bf16_rne(x1 - __uint_as_float(d[p] & 0xFFFF0000u)) << 16;
        } else {
          d[p] = (uint32_t)r.v[2 * p][b] | (uint32_t)r.v[2 * p + 1][b] << 16;
        }
      }
      bf[0][b] = make_uint4(d[0], d[1], d[2], d[3]);
      if constexpr (PREC == 3) bf[NP - 1][b] = make_uint4(l[0], l[1], l[2], l[3]);
    }
    uint32_t w[kEA];
#pragma unroll
    for (int a = 0; a < kEA; ++a) w[a] = words[s % kDW][16 * a + j];
    // the next step's loads, into r's registers, run beside all of this step's
    // MFMAs; the wave in its MFMAs goes first, the others of its SIMD pack
    __builtin_amdgcn_sched_barrier(0);
    next();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int a = 0; a < kEA; ++a) {
      const uint4 af = a_frag_bits<PREC>(w[a], q);
#pragma unroll
      for (int b = 0; b < kEB; ++b) acc[a][b] = mfma<PREC>(bf[0][b], af, acc[a][b]);
      if constexpr (PREC == 3) {
#pragma unroll
        for (int b = 0; b < kEB; ++b) low[a][b] = mfma<PREC>(bf[NP - 1][b], af, low[a][b]);
      }
#pragma unroll
      for (int b = 0; b < NP * kEB; ++b) {  // the next row tile's operand between them
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // three VALU
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

  // partial tiles: every wave's through LDS, 64 rows at a time, then a pair of waves
  // adds and stores a row tile, each two of the four accumulators e.  BF16X2 adds
  // the waves' hi sums and their lo sums apart and meets them in one rounding, as
  // the product in two passes does: with lo added to each wave's hi sum before,
  // K = 16384 at 50% with B in [1, 1.125) was 6.2e-8 of its norm off, 4.8e-8 there.
  constexpr int PER = 2;
  const int a = wave / 2, e0 = wave % 2 * PER;
  typedef float part_t __attribute__((ext_vector_type(PER)));
#pragma unroll
  for (int h = 0; h < kEA / 4; ++h) {
    const int64_t row = m0 + 64 * h + 16 * a + j;
    part_t sum[kEB];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      __syncthreads();  // the words, or what was there before, have been read
#pragma unroll
      for (int i = 0; i < 4 * kEB; ++i) {
        if (p == 0) part[wave][i][lane] = acc[4 * h + i / kEB][i % kEB];
        else part[wave][i][lane] = low[4 * h + i / kEB][i % kEB];
      }
      __syncthreads();
#pragma unroll
      for (int b = 0; b < kEB; ++b) {
        auto at = [&](int w) {
          return *reinterpret_cast<const part_t*>(
              reinterpret_cast<const float*>(&part[w][a * kEB + b][lane]) + e0);
        };
        part_t x = at(0);
#pragma unroll
        for (int w = 1; w < DW; ++w) x += at(w);
        sum[b] = p == 0 ? x : sum[b] + x;
      }
    }
    if (row >= M) continue;
#pragma unroll
    for (int y = 0; y < PER; ++y) {
      const int64_t col = n0 + 16 * q + 4 * (e0 + y);
      if (col >= N) continue;
      f32x4 v;
#pragma unroll
      for (int b = 0; b < kEB; ++b) v[b] = alpha * sum[b][y];
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
}

template <int PREC, bool F32>
bws_status launch_direct16(const bws_bitmap* A, const void* B, int64_t ldb, int64_t N, float* C,
                           int64_t ldc, float alpha, float beta, hipStream_t s) {
  const int64_t tiles64 = ceil_div(A->rows, 64) * ceil_div(N, 64);
  const int64_t rows = PREC == 3 || tiles64 <= 256 ? 64 : 128;  // (256 accumulators a lane)
  const int64_t row_blocks = ceil_div(A->rows, rows), col_blocks = ceil_div(N, kEN);
  const int64_t per_xcd = ceil_div(row_blocks * col_blocks, 8);
  const int vec = ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * per_xcd)), dim3(64 * DW), 0, s, A->words,
                       A->rows, A->cols, A->ldw, B, ldb, N, C, ldc, alpha, beta, row_blocks,
                       col_blocks, per_xcd, vec);
  };
  if constexpr (PREC != 3) {
    if (rows == 128) {
      launch(k_spmm_direct16<PREC, F32, 8>);
      return launch_check();
    }
  }
  launch(k_spmm_direct16<PREC, F32, 4>);
  return launch_check();
}

}  // namespace

// Outputs of up to 256 tiles of 64 x 64 with K of at least 1280 and of up to 512
// with 2048 (figures above): the staged tiles' time is K's, this kernel has about
// 6 and 9 us besides.  BF16X2 of up to 512: the other side is a pass that splits B
// and two products; us, that | this: 200 x 16 x 100 10.4 | 6.6, 500 x 1000 x 300 19.8 |
// 11.5, 1999 x 3100 x 1000 60.6 | 42.1; at 1024 tiles, 2048 x 256 x 2048, 23.0 | 28.2.
// Where N is no multiple of 8 a short K goes to the kernel that splits B in
// registers, one launch too: 1359 x 32 x 1351 (484 tiles) 12.5 | 22.2, K 128 17.3 |
// 23.0, K 256 27.0 | 24.5; 32000 x 128 x 60 (500) 12.7 | 15.6, K 256 17.0 | 17.0;
// 1000 x 32 x 1001 (256) 11.9 | 12.7, K 64 13.2 | 12.7, 1000 x 32 x 1004 12.0 | 8.7.
bool spmm_direct16_ok(const bws_bitmap* A, int32_t precision, int64_t ldb, int64_t N) {
  const int64_t rows = ceil_div(A->rows, 64), cols = ceil_div(N, 64);
  const int64_t most = precision == BWS_PREC_BF16X2
                           ? (N % 8 == 0 || A->cols >= 256      ? 512
                              : N % 4 == 0 || A->cols >= 64 ? 256
                                                            : 128)
                       : A->cols < 1280 ? 0
                       : A->cols < 2048 ? 256
                                        : 512;
  return rows <= most && cols <= most && rows * cols <= most &&
         A->cols < ((int64_t)1 << 31) && ldb < (1 << 24);  // 32-bit steps and offsets
}

bws_status launch_spmm_direct16(const bws_bitmap* A, const void* B, int32_t b_dtype,
                                int32_t precision, int64_t ldb, int64_t N, float* C, int64_t ldc,
                                float alpha, float beta, hipStream_t s) {
  const bool f32 = b_dtype == BWS_DTYPE_F32;
  if (precision == BWS_PREC_BF16X2)
    return launch_direct16<3, true>(A, B, ldb, N, C, ldc, alpha, beta, s);
  if (precision == BWS_PREC_FP16)
    return f32 ? launch_direct16<2, true>(A, B, ldb, N, C, ldc, alpha, beta, s)
               : launch_direct16<2, false>(A, B, ldb, N, C, ldc, alpha, beta, s);
  return f32 ? launch_direct16<1, true>(A, B, ldb, N, C, ldc, alpha, beta, s)
             : launch_direct16<1, false>(A, B, ldb, N, C, ldc, alpha, beta, s);
}

}  // namespace bws
