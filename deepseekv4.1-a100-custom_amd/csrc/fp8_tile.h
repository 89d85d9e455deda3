// Tile kernel of the FP8 block-scaled projections for more rows than the streaming kernels of fp8_gemm.hip take
// (serving batches, prefill chunks): the same product, bf16 x against e4m3 weights decoded to bf16 with their block
// scale (exact), bf16 MFMA, fp32 accumulation.  x rows and weight bytes come to LDS by direct-to-LDS loads several
// stages ahead, so the weights are read once per BM rows and no register holds a load in flight.
#pragma once
#include "common.h"

namespace {

struct TileArgs {
  const uint16_t* x;  // bf16 rows, row stride ldx; output row m, column n reads x row m * xr_mul + n / group_cols
  long ldx;
  const uint8_t* w8;  // [N, K] e4m3 bits, 16-k groups in the kPermK byte order
  const uint8_t* s8;  // [ceil(N / 32), Kc] E8M0
  int M, N, K, Kc, group_cols, xr_mul;
  uint16_t* out;  // bf16 [M, ldo]
  long ldo;
  float* outf;  // optional fp32 copy [M, ldo]
  int mtiles, ntiles;
  int vec;     // rows of out (and outf) take 4-column stores
  int splits;  // K slices of kslice units (64 k); more than one: fp32 partials [splits, M, ldp] for tile_sum_kernel
  int kslice;
  int chain;   // units summed in one MFMA chain; a multiple of the shape's units per stage
  float* part;
  long ldp;
};

constexpr int kTileMaxK = 16384;  // (the block scales of a column tile are held in LDS)

DSV41_DEV float tile_e8m0(uint32_t s) { return s ? __uint_as_float(s << 23) : __uint_as_float(0x00400000u); }

typedef __bf16 tile_bf2_t __attribute__((ext_vector_type(2)));
DSV41_DEV uint32_t tile_pack(float a, float b) {  // two fp32 to bf16, round to nearest even
  return __builtin_bit_cast(uint32_t, tile_bf2_t{(__bf16)a, (__bf16)b});
}

// Direct-to-LDS load of 16 bytes from base + off (lane i writes lds_addr + 16 i); callers wait with vmcnt counts.
DSV41_DEV void tile_dma16(const void* base, uint32_t off, uint32_t lds_addr) {
  const uint32_t m = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(m) : "memory", "m0");
}

// 8 of a lane's 16 weight bytes (one 16-k group) as bf16, block scale applied; byte word i holds k (2i, 2i + 1) in its
// low half and (2i + 8, 2i + 9) in its high half.  Part h of the k order of x: words' low (h = 0: k 0..7) or high
// halves (k 8..15).  Part h of the byte order: words 2h and 2h + 1.
DSV41_DEV uint32_t tile_cvt(uint32_t w, float sc, int hi) {
  return hi ? __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, sc, true))
            : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, sc, false));
}
DSV41_DEV uint4 tile_decode_k(uint4 w, float sc, int h) {
  return make_uint4(tile_cvt(w.x, sc, h), tile_cvt(w.y, sc, h), tile_cvt(w.z, sc, h), tile_cvt(w.w, sc, h));
}
DSV41_DEV uint4 tile_decode_b(uint4 w, float sc, int h) {
  const uint32_t a = h ? w.z : w.x, b = h ? w.w : w.y;
  return make_uint4(tile_cvt(a, sc, 0), tile_cvt(a, sc, 1), tile_cvt(b, sc, 0), tile_cvt(b, sc, 1));
}

// WM x WN waves of (BM / WM) rows x (BN / WN) columns; NBUF LDS buffers of KU units of 64 k (128 bytes of an x row,
// 64 of a weight row each).  The weights are the MFMA's row operand, so a lane ends with 4 adjacent columns of a row.
// One barrier per stage; two workgroups per CU (one of the 32-row tiles) cover each other's waits, KU > 1 for the small
// tiles: the chain of barrier, weight read, decode and MFMA is then paid once per KU units; K slices when the tiles
// leave CUs idle.  Bound: what stands between the MFMAs of a stage (LDS reads, weight decode, the barrier): 2048 rows in
// 128 x 128 tiles, [32768 x 1280] 237 us, [8192 x 4096] 158 us (0.87 PFLOP/s), [5120 x 8192] 209 us; the 64-row stream
// 3849, 3119 and 4672 us.
// Every sum is made of chains as short as the streaming kernel's K slices, so a lane holds its sums twice and 128 x 128
// is the largest tile.  Not kept: 192 x 256 and 256 x 256 with one chain over all of K, 194, 130 and 180 us, but 1.7e-4,
// 2.9e-4 and 4.2e-4 of the bf16 results off the rounded product (1.5e-4, 1.9e-4, 2.0e-4 in short chains); 192 x 256 with
// the second sums as bf16 and the remainder carried on: 230 us and more at equal error.
//   SAME: the streaming kernel's sums bit for bit: its k order inside an MFMA (8 register moves a 16-row operand; 5 to
//       10 % of the time) and its K slices as chains.
template <int BM, int BN, int WM, int WN, int NBUF, int KU, bool SAME>
__global__ void __launch_bounds__(64 * WM * WN) fp8_tile_kernel(const TileArgs a) {
  constexpr int NT = 64 * WM * WN;
  constexpr int MT = BM / WM / 16, CT = BN / WN / 16;  // 16-row and 16-column tiles of a wave
  constexpr int XB = BM * 128, WB = BN * 64, UNIT = XB + WB;
  constexpr int XL = XB / 16 / NT, WL = WB / 16 / NT, LPT = XL + WL;  // loads per thread and unit
  static_assert(XL * NT * 16 == XB && WL * NT * 16 == WB && (BN / WN) % 32 == 0, "tile shape");
  static_assert((NBUF - 2) * KU * LPT < 64, "vmcnt immediate");
  __shared__ __align__(16) uint8_t buf[NBUF * KU * UNIT];
  __shared__ uint8_t scl[BN / 32][kTileMaxK / 32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int wm = wave / WN, wn = wave - wm * WN;
  // contiguous tile ranges per XCD, rows fastest: the x rows stay in the XCD's L2 while its weights stream once
  const int per = gridDim.x / kXcds;
  const int id = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
  if (id >= a.mtiles * a.ntiles) return;
  const int m0 = id % a.mtiles * BM, n0 = id / a.mtiles * BN;
  const int u0 = blockIdx.y * a.kslice;            // first unit of this K slice
  const int nu = min(a.K / 64 - u0, a.kslice);     // units (a multiple of KU)
  const int nk = nu / KU;                          // stages

  const long xrow0 = (long)m0 * a.xr_mul + (a.group_cols > 0 ? n0 / a.group_cols : 0);
  const uint8_t* xb = (const uint8_t*)(a.x + xrow0 * a.ldx) + (long)u0 * 128;
  const uint8_t* wb = a.w8 + (long)n0 * a.K + (long)u0 * 64;
  // chunk c of a 128-byte row r sits at c ^ (r & 7), of a 64-byte row at c ^ ((r >> 2) & 3): the 8 lanes of an LDS
  // read cycle (8 rows, one chunk) then hit 8 different 16-byte bank groups
  uint32_t xo[XL], wo[WL];
#pragma unroll
  for (int u = 0; u < XL; ++u) {
    const int c = u * NT + tid, r = c >> 3;
    const int m = min(m0 + r, a.M - 1) - m0;  // (rows past M read row M - 1 and are not stored)
    xo[u] = (uint32_t)((long)m * a.xr_mul * a.ldx * 2) + ((c & 7) ^ (r & 7)) * 16;
  }
#pragma unroll
  for (int u = 0; u < WL; ++u) {
    const int c = u * NT + tid, r = c >> 2;
    const int n = min(n0 + r, a.N - 1) - n0;
    wo[u] = (uint32_t)((long)n * a.K) + ((c & 3) ^ ((r >> 2) & 3)) * 16;
  }
  const uint32_t lds0 = lds_addr_of(buf) + (uint32_t)(wave * 64 * 16);
  auto issue = [&](int kt, int b) {
#pragma unroll
    for (int q = 0; q < KU; ++q) {
      const uint8_t* xp = xb + (long)(kt * KU + q) * 128;
      const uint8_t* wp = wb + (long)(kt * KU + q) * 64;
      const uint32_t l = lds0 + (uint32_t)((b * KU + q) * UNIT);
#pragma unroll
      for (int u = 0; u < XL; ++u) tile_dma16(xp, xo[u], l + u * NT * 16);
#pragma unroll
      for (int u = 0; u < WL; ++u) tile_dma16(wp, wo[u], l + XB + u * NT * 16);
    }
  };
  {
    const int ks = nu * 2, nb = (a.N + 31) / 32;
    for (int e = tid; e < BN / 32 * ks; e += NT) {
      const int b = e / ks, k = e - b * ks;
      scl[b][k] = a.s8[(long)min(n0 / 32 + b, nb - 1) * a.Kc + u0 * 2 + k];
    }
  }
#pragma unroll
  for (int p = 0; p < NBUF - 1; ++p)
    if (p < nk) issue(p, p);

  f32x4_t acc[MT][CT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const int xr = wm * (BM / WM) + l16, wr = wn * (BN / WN) + l16;  // (16-row steps keep the swizzles' row bits)
  const int xc0 = ((2 * g) ^ (xr & 7)) * 16, xc1 = ((2 * g + 1) ^ (xr & 7)) * 16, wc = (g ^ ((wr >> 2) & 3)) * 16;
  const uint8_t* sp = &scl[wn * (BN / WN / 32)][g >> 1];
  struct Ops {  // a lane's operands of a unit: k 16 g .. 16 g + 15 of its x rows and weight rows, the block scales
    uint4 x0[MT], x1[MT], w[CT];
    uint32_t s[CT / 2];
  };
  auto read = [&](int b, int q, int unit, Ops& o) {
    const uint8_t* u = buf + (b * KU + q) * UNIT;
#pragma unroll
    for (int j = 0; j < CT / 2; ++j) o.s[j] = sp[j * (kTileMaxK / 32) + 2 * unit];
#pragma unroll
    for (int j = 0; j < CT; ++j) o.w[j] = *(const uint4*)(u + XB + (wr + 16 * j) * 64 + wc);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      o.x0[i] = *(const uint4*)(u + (xr + 16 * i) * 128 + xc0);
      o.x1[i] = *(const uint4*)(u + (xr + 16 * i) * 128 + xc1);
    }
  };
  auto mul = [&](const Ops& o) {  // each half column tile is decoded while the previous one's MFMAs run
#pragma unroll
    for (int jh = 0; jh < 2 * CT; ++jh) {
      const int j = jh >> 1, h = jh & 1;
      const float sc = tile_e8m0(o.s[j / 2]);
      const uint4 wf = SAME ? tile_decode_b(o.w[j], sc, h) : tile_decode_k(o.w[j], sc, h);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const uint4 xb = h ? make_uint4(o.x0[i].z, o.x1[i].z, o.x0[i].w, o.x1[i].w)
                           : make_uint4(o.x0[i].x, o.x1[i].x, o.x0[i].y, o.x1[i].y);  // the byte order
        acc[i][j] = mfma_bf16_16x16x32(wf, SAME ? xb : h ? o.x1[i] : o.x0[i], acc[i][j]);
      }
    }
  };
  auto landed = [&](int kt) {  // this wave's loads of stage kt have landed (the NBUF - 2 stages after it may not)
    constexpr int n = (NBUF - 2) * KU * LPT;
    if (kt + NBUF - 2 < nk) __builtin_amdgcn_s_waitcnt(vmcnt_imm(n));
    else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  };
  // every a.chain units the sums move to a second set, chains as short as the streaming kernel's K slices (fp32
  // relative error 1.4e-7 at K 1280 in both; in one chain 2.3e-7)
  int bi = 0, left = 0;
  f32x4_t tot[MT][CT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) tot[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
  for (int kt = 0; kt < nk; ++kt) {
    landed(kt);
    lds_barrier();  // stage kt is there for every wave, and every wave has read stage kt - 1
    if (kt + NBUF - 1 < nk) issue(kt + NBUF - 1, bi == 0 ? NBUF - 1 : bi - 1);
    if (left == 0) {
      left = a.chain;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          tot[i][j] += acc[i][j];
          acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    Ops o[KU];
#pragma unroll
    for (int q = 0; q < KU; ++q) read(bi, q, kt * KU + q, o[q]);
#pragma unroll
    for (int q = 0; q < KU; ++q) mul(o[q]);
    left -= KU;
    bi = bi + 1 == NBUF ? 0 : bi + 1;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] += tot[i][j];
  // lane (l16, g) holds rows m = 16 i + l16, columns 16 j + 4 g .. + 3
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + wm * (BM / WM) + 16 * i + l16;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int n = n0 + wn * (BN / WN) + 16 * j + 4 * g;
      const f32x4_t v = acc[i][j];
      if (a.splits > 1) {  // (ldp is a multiple of 4 that covers N)
        if (n < a.N) *(f32x4_t*)(a.part + ((long)blockIdx.y * a.M + m) * a.ldp + n) = v;
      } else if (a.vec && n + 4 <= a.N) {
        *(uint2*)(a.out + (long)m * a.ldo + n) = make_uint2(tile_pack(v[0], v[1]), tile_pack(v[2], v[3]));
        if (a.outf) *(f32x4_t*)(a.outf + (long)m * a.ldo + n) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < a.N) {
            a.out[(long)m * a.ldo + n + e] = (uint16_t)tile_pack(v[e], 0.0f);
            if (a.outf) a.outf[(long)m * a.ldo + n + e] = v[e];
          }
      }
    }
  }
}

// The K slices' partials summed in slice order, one thread per 4 columns of a row.
__global__ void __launch_bounds__(256) tile_sum_kernel(const TileArgs a) {
  const long q = a.ldp / 4, e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= q * a.M) return;
  const long m = e / q;
  const int n = (int)(e - m * q) * 4;
  f32x4_t v = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
  for (int s = 0; s < a.splits; ++s) v += *(const f32x4_t*)(a.part + ((long)s * a.M + m) * a.ldp + n);
  if (a.vec && n + 4 <= a.N) {
    *(uint2*)(a.out + m * a.ldo + n) = make_uint2(tile_pack(v[0], v[1]), tile_pack(v[2], v[3]));
    if (a.outf) *(f32x4_t*)(a.outf + m * a.ldo + n) = v;
  } else {
    for (int i = 0; i < 4 && n + i < a.N; ++i) {
      a.out[m * a.ldo + n + i] = (uint16_t)tile_pack(v[i], 0.0f);
      if (a.outf) a.outf[m * a.ldo + n + i] = v[i];
    }
  }
}

}  // namespace
