// The compressor's fp32 projections of a prefill chunk (wkv and wgate of dsv41/model.py:593-600): out_i = x w_i^T with
// bf16 x and fp32 weights, both weights in one launch.  The product runs on the bf16 matrix units without losing a
// bit of the weights: an fp32 value is the sum of three bf16 ones (its leading, middle and last 8 significant bits,
// by truncation), their products with bf16 x are exact, and the MFMA accumulates in fp32 -- three MFMAs for one, at
// 16 times the fp32 matrix rate.
//
// 128 rows x 128 columns a workgroup, 8 waves of 64 x 32; 64 k of x rows and weights come to LDS by direct-to-LDS loads
// two stages ahead; the two waves of a SIMD alternate between barriers, one reads its operands and splits half of its
// weights while the other splits the rest and multiplies (all of the split on either side of the barrier: 2 to 4 %
// slower).  Bound: the MFMAs, 48 a wave and stage, and what they wait for of the split: without two of the three
// pieces the kernel takes half of its time.  One workgroup a CU, so the time is the same from 1 to 256 workgroups.
// Two weights of 512 columns, 5120 k, against the two library fp32 products and the fp32 copy of x that they need:
// 3000 rows 122 us (265), 2048 rows 120 (167), 1500 rows 120 (137), 1000 rows 119 (98), 6000 rows 243 (483).  Relative
// error against 64 bits 1.8e-7 at every size (one fp32 chain over all of K, as fast: 7.9e-7); the library's 1.2e-6 to
// 1.3e-6 from 300 rows on, 6.4e-7 below.
#include <type_traits>

#include "common.h"

namespace {

struct F32ProjArgs {
  const uint16_t* x;  // bf16 rows, row stride ldx
  long ldx;
  const float* w[2];  // [N, K]
  float* out[2];      // [M, N]
  int M, N, K, mtiles;
};

DSV41_DEV void f32p_dma16(const void* base, uint32_t off, uint32_t lds_addr) {
  const uint32_t m = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(m) : "memory", "m0");
}

// The leading, middle and last 8 significant bits of a pair of weights.
DSV41_DEV void split2(uint32_t u0, uint32_t u1, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
  const uint32_t r0 = __float_as_uint(__uint_as_float(u0) - __uint_as_float(u0 & 0xffff0000u));
  const uint32_t r1 = __float_as_uint(__uint_as_float(u1) - __uint_as_float(u1 & 0xffff0000u));
  mid = __builtin_amdgcn_perm(r1, r0, 0x07060302u);
  const uint32_t q0 = __float_as_uint(__uint_as_float(r0) - __uint_as_float(r0 & 0xffff0000u));
  const uint32_t q1 = __float_as_uint(__uint_as_float(r1) - __uint_as_float(r1 & 0xffff0000u));
  lo = __builtin_amdgcn_perm(q1, q0, 0x07060302u);
}

// A pair of weights as bf16 with every bit that was cut off in the last one: zero, infinite or NaN exactly where the
// weight is, and of its sign.
DSV41_DEV uint32_t sticky2(uint32_t u0, uint32_t u1) {
  u0 |= min(u0 & 0xffffu, 1u) << 16;
  u1 |= min(u1 & 0xffffu, 1u) << 16;
  return __builtin_amdgcn_perm(u1, u0, 0x07060302u);
}

constexpr int kFpM = 128, kFpN = 128, kFpBuf = 3;

__global__ void __launch_bounds__(512) f32_proj_kernel(const F32ProjArgs a) {
  constexpr int NT = 512, WM = 2, WN = 4;
  constexpr int MT = kFpM / WM / 16, CT = kFpN / WN / 16;
  constexpr int XB = kFpM * 128, WB = kFpN * 256, UNIT = XB + WB;  // bytes of 64 k
  constexpr int XL = XB / 16 / NT, WL = WB / 16 / NT, LPT = XL + WL;
  __shared__ __align__(16) uint8_t buf[kFpBuf * UNIT];
  __shared__ int again;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int wm = wave / WN, wn = wave - wm * WN;
  const int m0 = (int)(blockIdx.x % a.mtiles) * kFpM, n0 = (int)(blockIdx.x / a.mtiles) * kFpN, wi = blockIdx.y;
  const int nk = a.K / 64;
  const uint8_t* xb = (const uint8_t*)(a.x + (long)m0 * a.ldx);
  const uint8_t* wb = (const uint8_t*)(a.w[wi] + (long)n0 * a.K);
  // 16-byte chunk c of a weight row r (256 bytes) sits at c ^ (r & 15), of an x row (128) at c ^ (r / 2 & 7): 16 lanes
  // that read one chunk of 16 rows meet all 64 banks once (c ^ (r & 7) conflicted in half of the reads' cycles)
  uint32_t xo[XL], wo[WL];
#pragma unroll
  for (int u = 0; u < XL; ++u) {
    const int c = u * NT + tid, r = c >> 3;
    xo[u] = (uint32_t)((long)(min(m0 + r, a.M - 1) - m0) * a.ldx * 2) + ((c & 7) ^ (r >> 1 & 7)) * 16;
  }
#pragma unroll
  for (int u = 0; u < WL; ++u) {
    const int c = u * NT + tid, r = c >> 4;
    wo[u] = (uint32_t)((long)r * a.K * 4) + ((c & 15) ^ (r & 15)) * 16;
  }
  const uint32_t lds0 = lds_addr_of(buf) + (uint32_t)(wave * 64 * 16);
  auto issue = [&](int kt, int b) {
    const uint32_t l = lds0 + (uint32_t)(b * UNIT);
#pragma unroll
    for (int u = 0; u < XL; ++u) f32p_dma16(xb + (long)kt * 128, xo[u], l + u * NT * 16);
#pragma unroll
    for (int u = 0; u < WL; ++u) f32p_dma16(wb + (long)kt * 256, wo[u], l + XB + u * NT * 16);
  };
  auto landed = [&](int kt) {  // this wave's loads of stage kt have landed (the one after it may not)
    if (kt + 1 < nk) __builtin_amdgcn_s_waitcnt(vmcnt_imm(LPT));
    else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  };
  f32x4_t acc[MT][CT], sum[MT][CT];  // chains of 256 k, and their sum
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = sum[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        sum[i][j] += acc[i][j];
        acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
  };
  const int xr = wm * (kFpM / WM) + l16, wr = wn * (kFpN / WN) + l16;
  const bool late = wave >= 4;
  if (tid == 0) again = 0;
  // One pass over K, into acc and sum; KINDS: with weights of one piece, into acc alone, of which only whether it is
  // an infinity or NaN is of use.
  // phases between barriers: [early: read kt | late: MFMAs kt - 1] [early: MFMAs kt | late: read kt]; both groups
  // refill stage kt's buffer in the phase after the one in which the late waves read it
  auto pass = [&](auto kinds) {
    constexpr bool KINDS = decltype(kinds)::value;
    issue(0, 0);
    if (nk > 1) issue(1, 1);
    landed(0);
    __syncthreads();
    if (late) {
      if (nk > 2) issue(2, 2);
      lds_barrier();
    }
    int bi = 0;
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
      const uint8_t* u = buf + bi * UNIT;
      uint4 x[MT][2], w[CT][4];  // k 16 g .. 16 g + 15
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          w[j][q] = *(const uint4*)(u + XB + (wr + 16 * j) * 256 + ((4 * g + q) ^ (wr & 15)) * 16);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) x[i][h] = *(const uint4*)(u + (xr + 16 * i) * 128 + ((2 * g + h) ^ (xr >> 1 & 7)) * 16);
      if (!late && kt + 2 < nk) issue(kt + 2, bi == 0 ? 2 : bi - 1);
      if (!KINDS && (kt & 3) == 0) fold();
      uint4 p[CT][2][3];
      auto split = [&](int h) {
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const uint4 w0 = w[j][2 * h], w1 = w[j][2 * h + 1];
          if constexpr (KINDS) {
            p[j][h][0] = make_uint4(sticky2(w0.x, w0.y), sticky2(w0.z, w0.w), sticky2(w1.x, w1.y), sticky2(w1.z, w1.w));
            continue;
          }
          split2(w0.x, w0.y, p[j][h][0].x, p[j][h][1].x, p[j][h][2].x);
          split2(w0.z, w0.w, p[j][h][0].y, p[j][h][1].y, p[j][h][2].y);
          split2(w1.x, w1.y, p[j][h][0].z, p[j][h][1].z, p[j][h][2].z);
          split2(w1.z, w1.w, p[j][h][0].w, p[j][h][1].w, p[j][h][2].w);
        }
      };
      split(0);
      if (late) landed(kt + 1);
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (late && kt + 3 < nk) issue(kt + 3, bi);
      __builtin_amdgcn_s_setprio(1);
      split(1);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int s = KINDS ? 0 : 2; s >= 0; --s)  // (the small parts first)
#pragma unroll
          for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i][j] = mfma_bf16_16x16x32(p[j][h][s], x[i][h], acc[i][j]);
      __builtin_amdgcn_s_setprio(0);
      if (!late) landed(kt + 1);
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
      bi = bi + 1 == kFpBuf ? 0 : bi + 1;
    }
    if (!late) lds_barrier();
  };
  pass(std::false_type{});
  fold();
  // An infinity has no pieces and meets pieces of 0, so a sum that came out as NaN may be an infinity: a workgroup that
  // holds one goes over its tile once more for their kinds (3000 rows 125 -> 200 us, wherever and however many they
  // are; one lane to a sum: 0.35 ms for one infinity, 6.9 ms for a NaN at the end of every row).  A finite result of
  // that pass says nothing.
  bool nan = false;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) nan |= sum[i][j][e] != sum[i][j][e];
  if (nan) again = 1;
  __syncthreads();  // (and every wave is past its last read of the buffers)
  if (again) {
    pass(std::true_type{});
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float k = acc[i][j][e];
          if (sum[i][j][e] != sum[i][j][e] && fabsf(k) == __builtin_inff()) sum[i][j][e] = k;
        }
  }
  // lane (l16, g) holds rows m = 16 i + l16, columns 16 j + 4 g .. + 3
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + wm * (kFpM / WM) + 16 * i + l16;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < CT; ++j)
      *(f32x4_t*)(a.out[wi] + (long)m * a.N + n0 + wn * (kFpN / WN) + 16 * j + 4 * g) = sum[i][j];
  }
}

}  // namespace

extern "C" {

int dsv41_f32_proj2(const void* x, long ldx, const float* w0, const float* w1, int M, int N, int K, float* out0,
                    float* out1, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 64 != 0 || N % kFpN != 0 || ldx < K || ldx % 8 != 0 || !x || !w0 || !w1 || !out0 || !out1 ||
      (((uintptr_t)x | (uintptr_t)w0 | (uintptr_t)w1 | (uintptr_t)out0 | (uintptr_t)out1) & 15) != 0 ||
      kFpM * ldx * 2 >= (1l << 31) || (long)kFpN * K * 4 >= (1l << 31))
    return (int)hipErrorInvalidValue;
  F32ProjArgs a{(const uint16_t*)x, ldx, {w0, w1}, {out0, out1}, M, N, K, (M + kFpM - 1) / kFpM};
  const long tiles = (long)a.mtiles * (N / kFpN);
  if (tiles >= (1l << 31)) return (int)hipErrorInvalidValue;
  f32_proj_kernel<<<dim3((unsigned)tiles, 2), 512, 0, (hipStream_t)stream>>>(a);
  DSV41_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
