// spmm_planes.hip — the FP32 product of a 0/1 bitmap for outputs that fill the
// chip with 256 x 256 tiles: the streamed vector-add kernel (stream_tile.hpp)
// for sparse masks, the matrix cores for dense ones (gfx950,
// v_mfma_f32_16x16x32_bf16, B split exactly into three BF16 planes,
// split3.hpp), chosen on the device by the mask's density.
//
// The matrix form costs three dense BF16 products whatever the mask holds (4096³:
// 338 to 349 us with the 22 us of the split, 1.27 PFLOP/s of BF16 in the product);
// the vector-add kernel takes one LDS read and four adds per bit and lane (207 us
// at 5%, 318 at 10%, 396 at 14%, 523 at 20%, 1140 at 50%, independent bits).  They
// meet near 11%.  The line lies at one bit in eight: at 4096 x 1024 x 4096, where
// the split of B weighs more, 14% is 107 against 112 us.
//
// Two launches.  k_f32_prep writes the mask stream; its other workgroups
// estimate the density from the same 1024 words of A each and, where it is
// above the line, write the three planes of B in MFMA fragment order.  The
// product reads the decision and runs either tile; both take 256 x 256 outputs
// and 16 waves, so neither case pays for an idle launch of the other's kernel.
//
// The planes' unit is a block of 32 K rows x 16 columns, 1 KiB, in which lane l
// of a wave finds its 8 K values (rows 8(l/16) .. +7 of column l % 16) as 16
// contiguous bytes: copies into LDS and fragment reads are linear, without
// swizzle or transpose.
//
// B out of the planes' range (infinities, NaN, values from 2^96 on, whose sums may
// overflow, and nonzero ones below 2^-100, whose parts lose bits): the split marks
// its 64 columns, and every 256 x 256 output over marked columns takes the
// streamed tile, which adds B itself.  A dense mask then costs what it does there
// and the 22 us of the split (4096³, 50%: 1.2 ms for such columns); summed again
// output by output after the product, one NaN in B took 1.9 ms and a B of 1e-35
// 53 ms.
#include "split3.hpp"
#include "stream_tile.hpp"

namespace bws {
namespace {

// The matrix tile: 256 x 128 outputs, 4 x 4 waves of 64 x 32 each, two 32-row K
// steps per LDS stage and three stages (150 KiB: one workgroup per CU, four waves
// per SIMD); a workgroup takes the two halves of a 256 x 256 tile in turn.  With
// one K step per stage, so with twice the additions to the accumulators, the
// product at 4096³ was up to 15% further from the 64-bit one than the streamed
// tile (2.45e-7 against 2.13e-7 of its norm at 14%, B over six decades).
constexpr int kPA = 4, kPB = 2;                    // MFMA tiles per wave, down and across
constexpr int kPWaves = 4;                         // waves each way
constexpr int kPM = kPWaves * kPA * 16, kPN = kPWaves * kPB * 16;
constexpr int kPK = 2, kPBuf = 3;                  // K steps per stage, stages
constexpr int kPStage = kPN / 16 * kPK * kPlanes * 1024;  // B bytes per stage
constexpr int kPWords = kPM * kPK;                 // bitmap words per stage
constexpr int kPLanes = kPWords / (kPWaves * kPWaves);    // of which a wave copies
constexpr int kPLds = kPBuf * (kPStage + kPWords * 4);
static_assert(kPM == kQRows && 2 * kPN == kQBN && kPWaves * kPWaves == kQW, "one grid for both tiles");
static_assert(kPN / 16 * kPK == kQW && kPLanes <= 64, "a step of a column block per wave");

// 16 bytes per lane from base + lane_off (base wave-uniform) to lds + 16 * lane
__device__ __forceinline__ void dma16_lin(uint32_t lane_off, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(lane_off), "s"(base), "s"(lds)
               : "memory", "m0");
}

// Rows m0 .. +255 and columns n0 .. +127 of C.
__device__ __forceinline__ void planes_tile(const uint32_t* __restrict__ W, int64_t M, int64_t K,
                                            int64_t ldw, const uint8_t* __restrict__ planes,
                                            int64_t N, float* __restrict__ C, int64_t ldc,
                                            float alpha, float beta, int64_t m0, int64_t n0,
                                            uint8_t* smem) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / kPWaves, wn = wave % kPWaves;
  const int j = lane & 15, q = lane >> 4;
  const int64_t nks = ceil_div(K, 32), nst = ceil_div(nks, kPK);
  const int64_t ncb = ceil_div(N, 16);
  uint8_t* const sB = smem;
  uint32_t* const sA = reinterpret_cast<uint32_t*>(smem + kPBuf * kPStage);
  const uint32_t sB0 = lds_u32(sB), sA0 = lds_u32(sA);
  const uint32_t lane16 = 16u * lane;

  // this wave's share of a stage: the three planes of step wave % kPK of column
  // block wave / kPK, and kPLanes words: word (step, row) at step * kPM + row
  const int64_t gc = n0 / 16 + wave / kPK < ncb ? n0 / 16 + wave / kPK : ncb - 1;  // past N: unused
  const uint8_t* bsrc = planes + gc * nks * (kPlanes * 1024);
  const int ai = wave * kPLanes + (lane < kPLanes ? lane : 0);
  const int64_t arow = m0 + ai % kPM;
  const uint32_t* asrc = W + (arow < M ? arow : M - 1) * ldw;
  auto issue = [&](int64_t st) {
    const int buf = (int)(st % kPBuf);
    int64_t s = st * kPK + wave % kPK;
    s = s < nks ? s : nks - 1;  // past K: meets zero bits
#pragma unroll
    for (int t = 0; t < kPlanes; ++t)
      dma16_lin(lane16, bsrc + (s * kPlanes + t) * 1024,
                sB0 + (uint32_t)(buf * kPStage + (wave * kPlanes + t) * 1024));
    int64_t w = st * kPK + ai / kPM;
    w = w < nks ? w : nks - 1;
    if (lane < kPLanes) dma4(asrc + w, sA0 + (uint32_t)((buf * kPWords + wave * kPLanes) * 4));
  };

  f32x4 acc[kPA][kPB];
#pragma unroll
  for (int a = 0; a < kPA; ++a)
#pragma unroll
    for (int b = 0; b < kPB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int p = 0; p < kPBuf - 1; ++p)
    if (p < nst) issue(p);

  for (int64_t st = 0; st < nst; ++st) {
    const int buf = (int)(st % kPBuf);
    if (st + kPBuf - 2 < nst) wait_vmcnt<(kPBuf - 2) * (kPlanes + 1)>();
    else wait_vmcnt<0>();
    // every wave's copies of stage st have landed, and every wave has read
    // what the next copies overwrite
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (st + kPBuf - 1 < nst) issue(st + kPBuf - 1);
    uint32_t wr[kPK][kPA], any = 0;
#pragma unroll
    for (int x = 0; x < kPK; ++x) {
      const uint32_t vb = valid_bits(st * kPK + x, K);
#pragma unroll
      for (int a = 0; a < kPA; ++a) {
        wr[x][a] = sA[buf * kPWords + x * kPM + (wm * kPA + a) * 16 + j] & vb;
        any |= wr[x][a];
      }
    }
    if (__ballot(any != 0u) == 0ull) continue;
    __builtin_amdgcn_s_setprio(1);
    uint4 af[kPK][kPA];
#pragma unroll
    for (int x = 0; x < kPK; ++x)
#pragma unroll
      for (int a = 0; a < kPA; ++a) af[x][a] = a_frag01(wr[x][a], q);
    const uint8_t* src = sB + buf * kPStage + wn * kPB * (kPK * kPlanes * 1024) + lane16;
    uint4 bf[kPlanes][kPK];
#pragma unroll
    for (int p = kPlanes - 1; p >= 0; --p)
#pragma unroll
      for (int x = 0; x < kPK; ++x)
        bf[p][x] = *reinterpret_cast<const uint4*>(src + (x * kPlanes + p) * 1024);
#pragma unroll
    for (int b = 0; b < kPB; ++b) {
      f32x4 t[kPA];
#pragma unroll
      for (int a = 0; a < kPA; ++a) t[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = kPlanes - 1; p >= 0; --p)
#pragma unroll
        for (int x = 0; x < kPK; ++x) {
#pragma unroll
          for (int a = 0; a < kPA; ++a) t[a] = mfma<1>(bf[p][x], af[x][a], t[a]);
          if (b + 1 < kPB)
            bf[p][x] = *reinterpret_cast<const uint4*>(
                src + (((b + 1) * kPK + x) * kPlanes + p) * 1024);
        }
#pragma unroll
      for (int a = 0; a < kPA; ++a) acc[a][b] += t[a];
    }
    __builtin_amdgcn_s_setprio(0);
  }

  // lane (j, q) holds row 16a + j, columns 16b + 4q .. +3 of the wave's tile
  // (N a multiple of 4 and 16-byte rows of C, as the streamed tile needs)
#pragma unroll
  for (int a = 0; a < kPA; ++a) {
    const int64_t row = m0 + (wm * kPA + a) * 16 + j;
#pragma unroll
    for (int b = 0; b < kPB; ++b) {
      const int64_t col = n0 + (wn * kPB + b) * 16 + 4 * q;
      if (row >= M || col >= N) continue;
      float4* c = reinterpret_cast<float4*>(C + row * ldc + col);
      f32x4 v = acc[a][b] * alpha;
      if (beta != 0.0f) {
        const float4 o = *c;
        v.x = fmaf(beta, o.x, v.x);
        v.y = fmaf(beta, o.y, v.y);
        v.z = fmaf(beta, o.z, v.z);
        v.w = fmaf(beta, o.w, v.w);
      }
      *c = make_float4(v.x, v.y, v.z, v.w);
    }
  }
}

// Whether columns n0 .. n0 + 255 hold a marked value (marks: planes_block).
__device__ __forceinline__ bool cols_marked(const uint32_t* __restrict__ marks, int64_t nks,
                                            int64_t n0, int64_t N) {
  const int64_t first = n0 / 64 * nks;
  const int64_t last = (n0 + kQBN < N ? (n0 + kQBN) / 64 : ceil_div(N, 64)) * nks;
  uint32_t any = 0u;
  for (int64_t i = first + threadIdx.x; i < last; i += kQW * 64) any |= marks[i];
  return __syncthreads_or(any != 0u) != 0;
}

__global__ void __launch_bounds__(kQW * 64)
k_spmm_f32(const uint32_t* __restrict__ dense, const uint32_t* __restrict__ S,
           const uint8_t* __restrict__ planes, const uint32_t* __restrict__ marks,
           const uint32_t* __restrict__ W, int64_t M, int64_t K, int64_t ldw,
           const float* __restrict__ B, int64_t ldb, int64_t N, float* __restrict__ C,
           int64_t ldc, float alpha, float beta, int64_t row_blocks, int64_t col_blocks,
           int64_t per_xcd) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kPLds > kStreamLds ? kPLds : kStreamLds];
  const int64_t tile = xcd_tile(blockIdx.x, per_xcd);
  if (tile >= row_blocks * col_blocks) return;
  const int64_t m0 = (tile % row_blocks) * kQRows, n0 = (tile / row_blocks) * kQBN;
  if (dense[0] != 0u && !cols_marked(marks, ceil_div(K, 32), n0, N)) {
    for (int64_t n = n0; n < n0 + kQBN && n < N; n += kPN) {
      planes_tile(W, M, K, ldw, planes, N, C, ldc, alpha, beta, m0, n, smem);
      __syncthreads();  // the next half writes the stages
    }
  } else
    stream_tile<false>(S, nullptr, M, ceil_div(K, 64), B, ldb, K, N, C, ldc, alpha, beta, tile,
                       row_blocks, smem);
}

// hi, mid and lo of b, each in the low 16 bits.
__device__ __forceinline__ void split3(float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const uint32_t h = __float_as_uint(b) & 0xFFFF0000u;
  const float r = b - __uint_as_float(h);  // exact
  const uint32_t m = __float_as_uint(r) & 0xFFFF0000u;
  const float l = r - __uint_as_float(m);  // exact, 8 bits
  hi = h >> 16;
  mid = m >> 16;
  lo = __float_as_uint(l) >> 16;
}

// The planes of B over 32 K rows (step s) x 64 columns (group cg): wave q takes
// K rows 8q .. 8q+7, a lane one column (each load instruction 256 contiguous
// bytes).  Rows past K and columns past N are zero.  mark: a byte per wave, whether
// any of its values is out of the planes' range.
__device__ __forceinline__ void planes_block(const float* __restrict__ B, int64_t ldb, int64_t K,
                                             int64_t N, int64_t nks, int64_t ncb, int64_t s,
                                             int64_t cg, uint8_t* __restrict__ planes,
                                             uint8_t* __restrict__ mark) {
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int64_t col = cg * 64 + lane, k0 = s * 32 + 8 * q;
  const int64_t cblk = col >> 4;
  float v[8];
  const float* p = B + (col < N ? col : N - 1);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = p[(k0 + e < K ? k0 + e : K - 1) * ldb];
  uint32_t o[kPlanes][4];
  bool out = false;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (k0 + e >= K || col >= N) v[e] = 0.0f;
    const uint32_t mag = __float_as_uint(v[e]) & 0x7FFFFFFFu;
    out |= mag != 0u && mag - kTinyBits >= kHugeBits - kTinyBits;  // wraps below the range
  }
  const uint64_t outs = __ballot(out);
  if (lane == 0) mark[q] = outs != 0ull ? 1 : 0;
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    uint32_t h0, m0, l0, h1, m1, l1;
    split3(v[e], h0, m0, l0);
    split3(v[e + 1], h1, m1, l1);
    o[0][e / 2] = h0 | (h1 << 16);
    o[1][e / 2] = m0 | (m1 << 16);
    o[2][e / 2] = l0 | (l1 << 16);
  }
  if (cblk >= ncb) return;
  uint8_t* dst = planes + ((cblk * nks + s) * kPlanes) * 1024 + (q * 16 + (lane & 15)) * 16;
#pragma unroll
  for (int x = 0; x < kPlanes; ++x)
    *reinterpret_cast<uint4*>(dst + x * 1024) = make_uint4(o[x][0], o[x][1], o[x][2], o[x][3]);
}

// Whether more than one in eight of A's bits are set, by 256 groups of 4 words
// spread over its rows and, by a multiplicative hash, along them (the same in
// every workgroup; 32768 bits of independent density 1/8 are 0.2% off).  1024
// scattered words cost the sparse side 4 us, these 1.
__device__ __forceinline__ bool mask_dense(const uint32_t* __restrict__ W, int64_t M, int64_t K,
                                           int64_t ldw) {
  __shared__ int32_t sums[4];
  const int64_t wpr = words_for(K);
  int32_t excess = 0;  // 8 * set bits - bits
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t n = (threadIdx.x >> 2) + 64u * i;
    const int64_t r = (int64_t)n * M / 256;
    int64_t w = (int64_t)((n * 2654435761u) >> 8) % wpr + (threadIdx.x & 3);
    w = w < wpr ? w : wpr - 1;
    const uint32_t vb = valid_bits(w, K);
    excess += 8 * __popc(W[r * ldw + w] & vb) - __popc(vb);
  }
  excess = wave_sum(excess);
  if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = excess;
  __syncthreads();
  return sums[0] + sums[1] + sums[2] + sums[3] > 0;
}

// Workgroups [0, mask_wgs): the mask stream, 256 rows x kMaskStages stages each.  The
// others: the decision (written by the first of them) and, for a dense mask,
// the planes, units of 32 rows x 64 columns in turn.
__global__ void __launch_bounds__(256)
k_f32_prep(const uint32_t* __restrict__ W, int64_t M, int64_t K, int64_t ldw,
           const float* __restrict__ B, int64_t ldb, int64_t N, int64_t mask_wgs,
           int64_t mask_cols, uint32_t* __restrict__ S, uint8_t* __restrict__ planes,
           uint32_t* __restrict__ marks, uint32_t* __restrict__ dense) {
  const int64_t g = blockIdx.x;
  if (g < mask_wgs) {
    mask_stream_block<2>(W, M, K, ldw, ceil_div(K, 64), g % mask_cols, g / mask_cols, S);
    return;
  }
  const bool d = mask_dense(W, M, K, ldw);
  if (g == mask_wgs && threadIdx.x == 0) dense[0] = d ? 1u : 0u;
  if (!d) return;
  const int64_t nks = ceil_div(K, 32), ncb = ceil_div(N, 16), units = nks * ceil_div(N, 64);
  for (int64_t u = g - mask_wgs; u < units; u += gridDim.x - mask_wgs)
    planes_block(B, ldb, K, N, nks, ncb, u % nks, u / nks, planes,
                 reinterpret_cast<uint8_t*>(marks + u));
}

// A byte per wave of planes_block, a word per unit: units of one column group together.
size_t marks_bytes(int64_t K, int64_t N) {
  return (size_t)ceil_div(K, 32) * ceil_div(N, 64) * sizeof(uint32_t);
}
size_t planes_bytes(int64_t K, int64_t N) {
  return (size_t)ceil_div(K, 32) * ceil_div(N, 16) * kPlanes * 1024;
}

}  // namespace

// [decision, 256 bytes][mask stream][marks][planes]
size_t f32_routed_bytes(int64_t M, int64_t K, int64_t N) {
  return 256 + align_up(mask_stream_bytes(M, K), 256) + align_up(marks_bytes(K, N), 256) +
         planes_bytes(K, N);
}

bws_status launch_spmm_f32_routed(const bws_bitmap* A, void* ws, const float* B, int64_t ldb,
                                  int64_t N, float* C, int64_t ldc, float alpha, float beta,
                                  hipStream_t s) {
  const int64_t M = A->rows, K = A->cols;
  Carve cv(ws);
  uint32_t* dense = cv.take<uint32_t>(1);
  uint32_t* S = cv.take<uint32_t>(mask_stream_bytes(M, K) / 4);
  uint32_t* marks = cv.take<uint32_t>(marks_bytes(K, N) / 4);
  uint8_t* planes = cv.take<uint8_t>(planes_bytes(K, N));
  const int64_t mask_cols = ceil_div(ceil_div(K, 64), kMaskStages);
  const int64_t row_blocks = ceil_div(M, kQRows), col_blocks = ceil_div(N, kQBN);
  const int64_t mask_wgs = mask_cols * row_blocks;
  const int64_t units = ceil_div(K, 32) * ceil_div(N, 64);
  const int64_t split_wgs = units < 1024 ? units : 1024;
  const int64_t per_xcd = ceil_div(row_blocks * col_blocks, 8);
  if (mask_wgs + split_wgs > kMaxGrid || 8 * per_xcd > kMaxGrid) return BWS_ECAPACITY;
  hipLaunchKernelGGL(k_f32_prep, dim3((unsigned)(mask_wgs + split_wgs)), dim3(256), 0, s, A->words,
                     M, K, A->ldw, B, ldb, N, mask_wgs, mask_cols, S, planes, marks, dense);
  BWS_TRY(launch_check());
  hipLaunchKernelGGL(k_spmm_f32, dim3((unsigned)(8 * per_xcd)), dim3(kQW * 64), 0, s, dense, S,
                     planes, marks, A->words, M, K, A->ldw, B, ldb, N, C, ldc, alpha, beta, row_blocks,
                     col_blocks, per_xcd);
  return launch_check();
}

}  // namespace bws
