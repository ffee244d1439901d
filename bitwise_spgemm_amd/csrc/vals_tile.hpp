// vals_tile.hpp — the output tile of the FP32 SpMM of a value-carrying bitmap
// (gfx950): C = alpha * A·B + beta * C, one fused multiply-add per set bit and
// column, in ascending k.
//
// Workgroup: 16 waves, 16 VR rows x 256 columns of C (VR = 4, 8 or 16); a wave
// owns VR rows, a lane 4 columns of each (VR float4 accumulators).  K is walked in
// stages of 64 rows: a stage's 64 x 256 panel of B goes HBM -> LDS by
// global_load_lds (no registers) into one of two ring slots while the other is
// used; every slot starts with a row of zeros.
//
// Bound: vector issue.  A set bit costs four multiply-adds and the address of its
// B row; everything else is kept off the vector unit:
//  - row masks are walked with s_ff1 / s_bitset0 (two readlanes per row and stage);
//  - a row's values of a stage are one buffer load whose size is the row's bit
//    count, so lanes past it get zeros without a compare, a branch or traffic;
//  - they are written to a wave's own LDS strip (four rows at a time, no barrier:
//    a wave's LDS accesses are in order) and read back as one broadcast read per
//    four bits, which costs no vector instruction.  A readlane per bit and the
//    wait for its scalar result, as before, was a third of the loop;
//  - words are loaded by every lane at a clamped address and masked a stage
//    later: a load under a condition was waited for on the spot, with the
//    next stage's B copies behind it (45 us of 280 at 4096² x 2048, 10%).
// The first F bits of every row are taken without a branch, the next row's reads in
// flight (an empty mask gives k = -1, the zero row, and meets the value zero): F = 1
// below 1.3 bits per row and stage, else 2 (4096² x 2048: 120 us against 127 at 1%,
// 152 against 148 at 3%; F = 4 gains 1% at 10% and loses 27% at 1%).
//
// 4096² x 2048: 120 us at 1%, 242 at 10%, 365 at 20%, 733 at 50% density; the tile
// before (values by readlane) 136, 326, 534, 1143.  The slope is 5.5 CU cycles a
// bit and 256 columns of the 5 its vector instructions need; 100 us are the copies of
// B into LDS and the row and stage bookkeeping.
#pragma once

#include "mfma_common.hpp"

namespace bws {
namespace {

constexpr int kVW = 16;            // waves per workgroup
constexpr int kVBN = 256;          // columns per workgroup (4 per lane)
constexpr int kVS = 64;            // K rows per stage
constexpr int kVB = 4;             // rows whose values are in LDS together
constexpr uint32_t kVSlot = (kVS + 1) * 1024;               // the zero row, then kVS rows
constexpr uint32_t kVPitch = (kVS + 4) * 4;
constexpr uint32_t kVWaveVals = kVB * kVPitch;              // one wave's values
constexpr int kValsLds = 2 * kVSlot + kVW * kVWaveVals;

__device__ __forceinline__ int take_lowest(uint64_t& m) {
  int k;
  asm volatile("s_ff1_i32_b64 %0, %1\n\ts_bitset0_b64 %1, %0" : "=&s"(k), "+s"(m));
  return k;
}
__device__ __forceinline__ int count_bits(uint64_t m) {
  int n;
  asm("s_bcnt1_i32_b64 %0, %1" : "=s"(n) : "s"(m) : "scc");
  return n;
}
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <class T>
__device__ __forceinline__ T lds_at(uint32_t a) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>((uintptr_t)a);
}
__device__ __forceinline__ f32x4 vals_row(uint32_t vbase, int k) {
  return lds_at<f32x4>(vbase + ((uint32_t)k << 10));
}
__device__ __forceinline__ void vfma(f32x4& a, float v, const f32x4& b) {
  a.x = fmaf(v, b.x, a.x);
  a.y = fmaf(v, b.y, a.y);
  a.z = fmaf(v, b.z, a.z);
  a.w = fmaf(v, b.w, a.w);
}
__device__ __forceinline__ void pin4(f32x4& a) { asm volatile("" : "+v"(a)); }

// The set bits left in m: their B rows times the values at va, va + 4, ...
__device__ __forceinline__ void vals_walk(f32x4& acc, uint64_t m, uint32_t vbase, uint32_t va) {
  int n = count_bits(m);
  while (n >= 4) {
    const f32x4 v = lds_at<f32x4>(va);
    const int k0 = take_lowest(m), k1 = take_lowest(m), k2 = take_lowest(m), k3 = take_lowest(m);
    const f32x4 b0 = vals_row(vbase, k0), b1 = vals_row(vbase, k1), b2 = vals_row(vbase, k2),
                b3 = vals_row(vbase, k3);
    vfma(acc, v.x, b0);
    vfma(acc, v.y, b1);
    vfma(acc, v.z, b2);
    vfma(acc, v.w, b3);
    n -= 4;
    va += 16;
  }
  if (n >= 2) {
    const f32x2 v = lds_at<f32x2>(va);
    const int k0 = take_lowest(m), k1 = take_lowest(m);
    const f32x4 b0 = vals_row(vbase, k0), b1 = vals_row(vbase, k1);
    vfma(acc, v.x, b0);
    vfma(acc, v.y, b1);
    n -= 2;
    va += 8;
  }
  if (n) {
    const float v = lds_at<float>(va);
    vfma(acc, v, vals_row(vbase, take_lowest(m)));
  }
}

// 16-byte pieces of B's rows can be copied (the rows' 4 columns per lane).
__device__ __forceinline__ bool vals_vec_b(const float* B, int64_t ldb, int64_t N) {
  return N >= 4 && N % 4 == 0 && ldb % 4 == 0 && (reinterpret_cast<uintptr_t>(B) & 15u) == 0;
}

// wvals: the wave's first value; off: byte offset of row `lane` from there.
template <int VR, int F>
__device__ __forceinline__ void vals_tile_f(const uint32_t* __restrict__ W, int64_t M, int64_t K,
                                          int64_t ldw, const float* __restrict__ wvals,
                                          uint32_t off, const float* __restrict__ B, int64_t ldb, int64_t N,
                                          float* __restrict__ C, int64_t ldc, float alpha,
                                          float beta, int64_t tile, int64_t row_blocks,
                                          uint8_t* smem) {
  static_assert(F == 1 || F == 2, "one aligned read of the F values");
  constexpr int kOff = 4 - F;  // slots left free, so that the values after the first F are 16-byte aligned
  using VT = __attribute__((ext_vector_type(F))) float;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t cb = tile / row_blocks, rb = tile - cb * row_blocks;
  const int64_t n0 = cb * kVBN;
  const int64_t mw = rb * (kVW * VR) + (int64_t)wave * VR;
  const int64_t nst = ceil_div(K, kVS), wpr = words_for(K);
  const uint32_t lds0 = lds_u32(smem);
  const uint32_t vals0 = lds0 + 2 * kVSlot + (uint32_t)wave * kVWaveVals;
  if (wave < 2)
    reinterpret_cast<float4*>(smem + wave * kVSlot)[lane] = make_float4(0.f, 0.f, 0.f, 0.f);
  __syncthreads();

  // lane l < VR: word 0 of row mw + l, lane 32 + l: word 1
  const int rl = lane & 31;
  const bool row_lane = rl < VR && mw + rl < M;
  const int64_t wrow = row_lane ? (mw + rl) * ldw : 0;
  const bool vec = vals_vec_b(B, ldb, N);
  // copied columns, clamped: four neighbours per lane, or one of each 64
  const float* bcol[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int64_t n = vec ? n0 + 4 * lane : n0 + 64 * i + lane;
    const int64_t last = vec ? N - 4 : N - 1;
    bcol[i] = B + (n < last ? n : last);
  }

  // copy stage st's B rows of this wave (st kVS + wave + 16j; rows past K read
  // row K - 1 and meet no bits); rows that are not 16-byte pieces take four
  // copies of 64 columns each instead of one of 256, to the same places
  const int64_t row_step = (int64_t)kVW * ldb;
  auto issue = [&](int64_t st, uint32_t base) {
    const uint32_t m0 = base + (uint32_t)wave * 1024u;
    if (vec && (st + 1) * kVS <= K) {
      const float* p = bcol[0] + (st * kVS + wave) * ldb;
#pragma unroll
      for (int j = 0; j < kVS / kVW; ++j)
        dma16(p + j * row_step, m0 + (uint32_t)(j * kVW) * 1024u);
    } else {
#pragma unroll
      for (int j = 0; j < kVS / kVW; ++j) {
        int64_t k = st * kVS + wave + kVW * j;
        k = (k < K ? k : K - 1) * ldb;
        const uint32_t d = m0 + (uint32_t)(j * kVW) * 1024u;
        if (vec) {
          dma16(bcol[0] + k, d);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) dma4(bcol[i] + k, d + 256u * i);
        }
      }
    }
  };
  // bitmap words: lanes without a row and words past the last read some word
  const uint32_t in_row = row_lane ? ~0u : 0u;
  const uint32_t in_last = row_lane ? valid_bits(2 * (nst - 1) + (lane >> 5), K) : 0u;
  const uint32_t* wp = W + wrow;
  auto load_words = [&](int64_t st) -> uint32_t {
    const int64_t w = 2 * st + (lane >> 5);
    return wp[w < wpr ? w : wpr - 1];
  };
  // values of the rows' set bits, zero past the last
  float vv[VR];
  auto load_vals = [&](uint32_t bytes_v) {
#pragma unroll
    for (int r = 0; r < VR; ++r) {
      const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)off, r);
      const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)bytes_v, r);
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<char*>(reinterpret_cast<const char*>(wvals)) + o, 0, c, 0x00027000);
      vv[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, 4 * lane, 0, 0));
    }
  };
  // the row masks of a stage, lowest bit first (lane r: row r)
  auto masks = [&](int64_t st, uint32_t w, uint32_t& lo, uint32_t& hi) {
    w &= st < nst - 1 ? in_row : st == nst - 1 ? in_last : 0u;
    const uint32_t o = (uint32_t)__shfl_xor((int)w, 32, 64);
    lo = __brev(w);
    hi = __brev(o);
  };

  f32x4 acc[VR];
#pragma unroll
  for (int r = 0; r < VR; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};

  issue(0, lds0 + 1024u);
  uint32_t wnext = load_words(1);
  uint32_t lo, hi;
  masks(0, load_words(0), lo, hi);
  uint32_t bytes_v = 4u * (uint32_t)(__popc(lo) + __popc(hi));
  load_vals(bytes_v);

  auto stage = [&](int64_t st, uint32_t cur, uint32_t nxt) {
    wait_vmcnt<0>();  // this wave's copies and loads have landed
    asm volatile("" : "+v"(wnext));
#pragma unroll
    for (int r = 0; r < VR; ++r) asm volatile("" : "+v"(vv[r]));
    __builtin_amdgcn_s_barrier();  // everyone's have; the other slot is free
    asm volatile("" ::: "memory");
    if (st + 1 < nst) issue(st + 1, nxt);
    const uint32_t wn2 = load_words(st + 2);
    const uint32_t vbase = cur + (uint32_t)lane * 16u;
    off += bytes_v;
    uint32_t nlo, nhi;
    masks(st + 1, wnext, nlo, nhi);
    const uint32_t nbytes = 4u * (uint32_t)(__popc(nlo) + __popc(nhi));
#pragma unroll
    for (int r0 = 0; r0 < VR; r0 += kVB) {
#pragma unroll
      for (int r = 0; r < kVB; ++r)
        *reinterpret_cast<__attribute__((address_space(3))) float*>(
            (uintptr_t)(vals0 + (uint32_t)r * kVPitch + (uint32_t)(lane + kOff) * 4u)) = vv[r0 + r];
      if (r0 + kVB == VR) load_vals(nbytes);
      uint64_t m[kVB];
#pragma unroll
      for (int r = 0; r < kVB; ++r)
        m[r] = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, r0 + r) << 32) |
               (uint32_t)__builtin_amdgcn_readlane((int)lo, r0 + r);
      // F bits of each row, the next row's reads in flight
      VT v[2];
      f32x4 b[2][F];
      auto read = [&](int r) {
        v[r & 1] = lds_at<VT>(vals0 + (uint32_t)r * kVPitch + 4 * kOff);
#pragma unroll
        for (int i = 0; i < F; ++i) b[r & 1][i] = vals_row(vbase, take_lowest(m[r]));
      };
      read(0);
#pragma unroll
      for (int r = 0; r < kVB; ++r) {
        __builtin_amdgcn_sched_barrier(0);
        if (r + 1 < kVB) read(r + 1);
#pragma unroll
        for (int i = 0; i < F; ++i) vfma(acc[r0 + r], v[r & 1][i], b[r & 1][i]);
        pin4(acc[r0 + r]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < kVB; ++r)
        if (m[r] != 0) vals_walk(acc[r0 + r], m[r], vbase, vals0 + (uint32_t)r * kVPitch + 4 * (F + kOff));
    }
    lo = nlo;
    hi = nhi;
    bytes_v = nbytes;
    wnext = wn2;
  };
  for (int64_t st = 0; st < nst; st += 2) {
    stage(st, lds0 + 1024u, lds0 + kVSlot + 1024u);
    if (st + 1 < nst) stage(st + 1, lds0 + kVSlot + 1024u, lds0 + 1024u);
  }

  const int64_t n = n0 + 4 * lane;
  if (n >= N) return;
  const bool vec_c = n + 4 <= N && ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15u) == 0;
#pragma unroll
  for (int r = 0; r < VR; ++r) {
    const int64_t row = mw + r;
    if (row >= M) break;
    float* c = C + row * ldc + n;
    f32x4 v = acc[r] * alpha;
    if (vec_c) {
      f32x4* c4 = reinterpret_cast<f32x4*>(c);
      if (beta != 0.0f) vfma(v, beta, *c4);
      *c4 = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < N) c[i] = beta != 0.0f ? fmaf(beta, c[i], v[i]) : v[i];
    }
  }
}

// One tile (tile index column-block-major).  Byte offsets of a wave's values are
// 32 bits wide: K <= kValsMaxK (checked by the launchers).
constexpr int64_t kValsMaxK = (int64_t)1 << 25;

template <int VR>
__device__ __forceinline__ void vals_tile(const uint32_t* __restrict__ W, int64_t M, int64_t K,
                                          int64_t ldw, const int64_t* __restrict__ row_ptr,
                                          const float* __restrict__ values,
                                          const float* __restrict__ B, int64_t ldb, int64_t N,
                                          float* __restrict__ C, int64_t ldc, float alpha,
                                          float beta, int64_t tile, int64_t row_blocks,
                                          uint8_t* smem) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t mw = (tile % row_blocks) * (kVW * VR) + (int64_t)wave * VR;
  const int64_t r0 = mw < M ? mw : M, r1 = mw + VR < M ? mw + VR : M;
  const int64_t e0 = row_ptr[r0], bits = row_ptr[r1] - e0;
  const int64_t rl = mw + (threadIdx.x & 31);
  const uint32_t off = rl < r1 ? (uint32_t)(row_ptr[rl] - e0) * 4u : 0u;
  // (every wave meets the same barriers on either side)
  if (10 * bits < 13 * VR * ceil_div(K, kVS))
    vals_tile_f<VR, 1>(W, M, K, ldw, values + e0, off, B, ldb, N, C, ldc, alpha, beta, tile,
                       row_blocks, smem);
  else
    vals_tile_f<VR, 2>(W, M, K, ldw, values + e0, off, B, ldb, N, C, ldc, alpha, beta, tile,
                       row_blocks, smem);
}

}  // namespace
}  // namespace bws
