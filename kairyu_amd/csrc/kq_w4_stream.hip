// W4A16 GEMM for 17 to 48 rows on tiled weights, the activations read in place.
//
// Bound: at these row counts the weights come from HBM once (0.5 byte per
// weight) and the activations reach every workgroup through its CU's vector
// L1, which delivered about 25 KB per us here, weights and all (M = 48, 224
// workgroups N = 28672 K = 4096: 154 MB in 27.6 us; 256 N = 4096 K = 14336: 121 MB
// in 18.6), however the rows were walked (K order rotated per workgroup: no
// change); the LDS-staged tile kernel paid a
// staging pass of 4.5 us per call, one barrier per 128 k and 64-row tiles.
// So a workgroup's four waves divide its K range and meet once, in LDS, at the
// end; each wave owns all of the workgroup's NT column tiles for its stages
// (more columns per activation byte), and keeps one whole 128-k stage of
// weights, activations and scales in flight in registers while it dequantizes
// and multiplies the stage before.  No barrier and no LDS in the K loop.
// One wave per SIMD: a stage pair and 16 * NT * MT accumulators take up to 512
// registers.  (8 waves of half the K range each: no faster at NT = 4; a loop
// whose prefetch is conditional keeps a third stage alive and spills.)
//
// The weight and scale/zero words are the tiled operand's; dequantization is
// fp16((q - z) * s), products accumulate in fp32, waves are added in K order.
// Against the staged tile kernel, graph replay with the weights out of cache,
// fp16, M = 17 / 32 / 48, us before -> after: N = 4096 K = 4096
// 13.0 -> 9.0 / 13.9 -> 9.8 / 15.4 -> 12.2; N = 4096 K = 14336
// 22.0 -> 13.5 / 22.5 -> 15.6 / 23.8 -> 19.8; N = 22016 K = 4096
// 30.1 -> 16.6 / 30.6 -> 17.1 / 31.1 -> 21.4; SwiGLU I = 14336 K = 4096
// 33.4 -> 22.1 / 35.2 -> 22.2 / 35.7 -> 26.0; SwiGLU I = 18944 K = 3584
// 53.6 -> 24.9 / 55.0 -> 25.1 / 56.1 -> 31.1.
#include "kq_w4_stream.h"

#include <algorithm>

namespace kq {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

KQ_DEV uint32_t w4s_and_or(uint32_t x, uint32_t mask, uint32_t magic) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(magic));
  return r;
}
KQ_DEV uint32_t w4s_sub_mul(uint32_t q, uint32_t z, uint32_t s) {
  f16x2 r = (__builtin_bit_cast(f16x2, q) - __builtin_bit_cast(f16x2, z)) * __builtin_bit_cast(f16x2, s);
  return __builtin_bit_cast(uint32_t, r);
}
// bf16 pair -> fp16 pair, finite values saturating (act_to_f16)
KQ_DEV uint32_t w4s_cvt(uint32_t raw) {
  const float a = __uint_as_float(raw << 16), b = __uint_as_float(raw & 0xffff0000u);
  const float ac = __builtin_amdgcn_fmed3f(a, -65504.0f, 65504.0f), bc = __builtin_amdgcn_fmed3f(b, -65504.0f, 65504.0f);
  const _Float16 lo = (_Float16)(__builtin_amdgcn_classf(a, 0x207) ? a : ac);
  const _Float16 hi = (_Float16)(__builtin_amdgcn_classf(b, 0x207) ? b : bc);
  return (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
}

// The same for a pair below 65536 in magnitude, which only rounds.
KQ_DEV uint32_t w4s_cvt_small(uint32_t raw) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  const f32x2_t f{__uint_as_float(raw << 16), __uint_as_float(raw & 0xffff0000u)};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
}

template <int MT, int NT>
struct W4sBuf {
  u32x4 w[NT];
  u32x4 x[4][MT];
  uint32_t t[NT];
};

constexpr int kW4sWaves = 4;

template <int MT, int NT, bool BF16>
__global__ void __launch_bounds__(64 * kW4sWaves)
w4a16_stream_kernel(W4StreamArgs a) {
  constexpr int NW = kW4sWaves;
  __shared__ __attribute__((aligned(16))) f32x4 red[2][NW][NT][64];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int c = lane & 15, g = lane >> 4;
  const int split = blockIdx.x % a.ksplit, nb = blockIdx.x / a.ksplit;
  const int t0 = nb * NT, ntiles = (a.N + 15) / 16;
  const int nst = a.K / 128, pairs = a.pairs, gst = a.G / 128;
  const int part = split * NW + wave, parts = a.ksplit * NW;
  const int kb0 = (int)((int64_t)nst * part / parts), kb1 = (int)((int64_t)nst * (part + 1) / parts);

  // rows past M read row M - 1 and tiles past N the last one; neither is stored
  uint32_t xoff[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xoff[i] = (uint32_t)(min(i * 16 + c, a.M - 1) * a.ldx + g * 8) * 2;
  // table words of a lane: zu, one word of two groups' scales; else one of the
  // group's scale and zero
  const int tstride = a.zu ? 16 : 32;
  const uint32_t toff = a.zu ? c * 4 : c * 8;
  const uint32_t zmask = a.zu ? 0 : 0xffffu, zadd = a.zu ? a.zoff : 0;

  auto load = [&](W4sBuf<MT, NT>& b, int kb) {
    const int grp = kb / gst;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = min(t0 + n, ntiles - 1);
      b.w[n] = __builtin_nontemporal_load((const u32x4*)(a.w + ((int64_t)t * nst + kb) * 1024 + lane * 16));
      const uint32_t* tp = a.table + ((int64_t)t * pairs + (grp >> 1)) * tstride + (a.zu ? 0 : (grp & 1));
      b.t[n] = *(const uint32_t*)((const uint8_t*)tp + toff);
    }
    const uint8_t* xp = (const uint8_t*)a.x + (int64_t)kb * 256;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < MT; ++i) b.x[s][i] = *(const u32x4*)(xp + xoff[i] + s * 64);
  };

  const uint32_t m0 = __builtin_amdgcn_readfirstlane(0x000f000fu), m1 = __builtin_amdgcn_readfirstlane(0x00f000f0u);
  const uint32_t c0 = 0x64006400u + (uint32_t)(lane & 0), c1 = 0x54005400u + (uint32_t)(lane & 0);

  f32x4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[n][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // weights are the MFMA's A operand, x its B operand: lane (c, g) ends with row
  // c and four consecutive columns 4g.  x is put in the [0,4,1,5,2,6,3,7] order
  // of the nibble pairs.  The fence keeps the steps' fragments apart (without it
  // NT = 8 spills).
  auto compute = [&](W4sBuf<MT, NT>& b, int kb) {
    const int sh = a.zu && ((kb / gst) & 1) ? 16 : 0;
    uint32_t zq0[NT], zq1[NT], sq[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const uint32_t z = ((b.t[n] >> 16) & zmask) + zadd;
      zq0[n] = c0 + z * 0x00010001u;
      zq1[n] = c1 + z * 0x00100010u;
      sq[n] = ((b.t[n] >> sh) & 0xffffu) * 0x00010001u;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      // a step whose values are all below 65536 needs no saturation (bf16 has
      // no value between 65504 and that)
      bool big = false;
      if constexpr (BF16) {
        u16x2 top{0, 0};
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, b.x[s][i][q] & 0x7fff7fffu));
        big = __any(top[0] >= 0x4780 || top[1] >= 0x4780);
      }
      f16x8 B[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        u32x4 r = b.x[s][i];
        if constexpr (BF16) {
          if (big) r = u32x4{w4s_cvt(r[0]), w4s_cvt(r[1]), w4s_cvt(r[2]), w4s_cvt(r[3])};
          else r = u32x4{w4s_cvt_small(r[0]), w4s_cvt_small(r[1]), w4s_cvt_small(r[2]), w4s_cvt_small(r[3])};
        }
        B[i] = __builtin_bit_cast(
            f16x8, u32x4{__builtin_amdgcn_perm(r[2], r[0], 0x05040100u), __builtin_amdgcn_perm(r[2], r[0], 0x07060302u),
                         __builtin_amdgcn_perm(r[3], r[1], 0x05040100u), __builtin_amdgcn_perm(r[3], r[1], 0x07060302u)});
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const uint32_t w = b.w[n][s], y = w >> 8;
        const f16x8 A = __builtin_bit_cast(
            f16x8, u32x4{w4s_sub_mul(w4s_and_or(w, m0, c0), zq0[n], sq[n]), w4s_sub_mul(w4s_and_or(w, m1, c1), zq1[n], sq[n]),
                         w4s_sub_mul(w4s_and_or(y, m0, c0), zq0[n], sq[n]), w4s_sub_mul(w4s_and_or(y, m1, c1), zq1[n], sq[n])});
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[n][i] = mfma_f16(A, B[i], acc[n][i]);
      }
    }
  };

  {
    W4sBuf<MT, NT> b0, b1;
    if (kb0 < kb1) {
      load(b0, kb0);
      int kb = kb0;
      for (; kb + 2 < kb1; kb += 2) {
        load(b1, kb + 1);
        compute(b0, kb);
        load(b0, kb + 2);
        compute(b1, kb + 1);
      }
      if (kb + 1 < kb1) {
        load(b1, kb + 1);
        compute(b0, kb);
        compute(b1, kb + 1);
      } else {
        compute(b0, kb);
      }
    }
  }

  // the waves' sums meet a row tile at a time (two buffers: one barrier each)
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int n = 0; n < NT; ++n) red[i & 1][wave][n][lane] = acc[n][i];
    __syncthreads();
    const int m = i * 16 + c;
    auto total = [&](int n) {
      f32x4 v = red[i & 1][0][n][lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += red[i & 1][w][n][lane];
      return v;
    };
    auto biased = [&](f32x4 v, int n) {
      if (a.bias_dtype != KQ_DTYPE_NONE)
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = __fadd_rn(v[q], load_as_f32(a.bias, a.bias_dtype, n + q));
      return v;
    };
    if (a.swiglu) {
      for (int p = wave; p < NT / 2; p += NW) {
        const f32x4 gt = total(2 * p), up = total(2 * p + 1);
        const int n = (t0 + 2 * p) * 16 + 4 * g;  // gate column; its up column is 16 on
        if (m >= a.M || n >= a.N) continue;
        const f32x4 gv = biased(gt, n), uv = biased(up, n + 16);
        *(u32x2*)(a.out + (int64_t)m * (a.N / 2) + (t0 / 2 + p) * 16 + 4 * g) =
            u32x2{swiglu_bits2(gv[0], uv[0], gv[1], uv[1], a.out_dtype),
                  swiglu_bits2(gv[2], uv[2], gv[3], uv[3], a.out_dtype)};
      }
      continue;
    }
    for (int n = wave; n < NT; n += NW) {
      const f32x4 v = total(n);
      const int col = (t0 + n) * 16 + 4 * g;
      if (m >= a.M || col >= a.N) continue;
      if (a.ksplit > 1) {
        *(f32x4*)(a.partials + ((int64_t)split * a.M + m) * a.N + col) = v;
        continue;
      }
      const f32x4 o = biased(v, col);
      *(u32x2*)(a.out + (int64_t)m * a.N + col) =
          u32x2{(uint32_t)f32_to_out(o[0], a.out_dtype) | ((uint32_t)f32_to_out(o[1], a.out_dtype) << 16),
                (uint32_t)f32_to_out(o[2], a.out_dtype) | ((uint32_t)f32_to_out(o[3], a.out_dtype) << 16)};
    }
  }
}

// Up to 48 rows (MT = 4 at 64 rows: SwiGLU I = 14336 31.4 against 35.7 us in
// fp16 but 43 against 36 in bf16, N = 4096 K = 14336 30.2 against 27.3).  Above
// 32 rows the fp16 rows of a narrow, long-K layer still gain (19.8 against 23.8
// us at N = 4096, K = 14336), but rows converted in the loop or gathered first
// do not past K = 8192 where K is split: bf16 N = 4096 K = 14336 23.3 / 23.9,
// N = 3584 K = 18944 28.1 / 26.3, gathered N = 4096 K = 14336 24.7 / 25.3.  And
// with K whole on less than two thirds of the CUs, where the tile kernel splits
// it three ways, rows converted in the loop stop gaining at K = 4096 (N = 8448,
// M = 33, K = 3072 17.4 / 17.7, 4096 21.0 / 19.9, 8192 36.0 / 28.8), gathered ones
// at K = 6144 and 41 rows (M = 48, K = 4096 20.5 / 21.5, 6144 27.2 / 25.9; M = 33
// 23.6 / 24.9).
//
// Columns: the NT with the least rounds of workgroups over the CUs times
// columns, the wider one of two that tie (N = 28672: 8 26.0 us, 6 41, 4 37;
// N = 37888: 10 31.1 us, 8 44.7; N = 57344 K = 8192: 8 82 us, 10 104).  CUs
// left over take K splits, down to one stage per wave (N = 1024 K = 4096,
// M = 32: 8 splits 7.9 us, 4 8.3; N = 4096 K = 4096: 4 splits 9.8 us, 2 11.1).
//
// SwiGLU here keeps K whole; where the plain product would split it, that with
// the elementwise pass (about 3.5 us more) is the faster one as soon as the
// split saves more than that.  A wave's stage of 128 k takes about 0.85 us of
// fp16 rows up to 32 (0.72 where they were gathered just before), 1.2 above, and
// 1.3 / 1.8 of rows converted in the loop:
// fused against two passes, us, I = 1536 M = 17 / 33, fp16 K = 2048 9.6 / 12.4
// and 10.2 / 11.6, K = 4096 13.0 / 17.1 and 11.9 / 13.7; bf16 K = 2048 11.4 / 15.3
// and 10.8 / 12.4, K = 8192 27.1 / 36.7 and 16.1 / 19.4 (the tile kernel's two
// passes 19.6 / 21.1); I = 3072 fp16 K = 4096 13.2 / 17.4 and 13.8 / 16.2.
bool w4_stream_form(int M, int N, int K, W4Rows rows, int swiglu, int cus, int max_splits, W4StreamForm* f) {
  if (M > 48) return false;
  const int tiles = (N + 15) / 16, nst = K / 128;
  f->nt = 4;
  int best = 0;
  for (int nt : {4, 6, 8, 10}) {
    const int cost = ((tiles + nt - 1) / nt + cus - 1) / cus * nt;
    if (best == 0 || cost <= best) {
      best = cost;
      f->nt = nt;
    }
  }
  const int blocks = (tiles + f->nt - 1) / f->nt;
  const int splits = std::max(1, std::min(cus / blocks, nst / kW4sWaves));
  if (swiglu) {
    f->ksplit = 1;
    const float stage = rows == kW4RowsConverted ? (M > 32 ? 1.8f : 1.3f) : (M > 32 ? 1.2f : rows == kW4RowsGathered ? 0.72f : 0.85f);
    return (nst - nst / splits) * stage < 3.5f * kW4sWaves;
  }
  f->ksplit = std::max(1, std::min(splits, max_splits));
  if (M <= 32 || rows == kW4RowsInPlace) return true;
  if (f->ksplit > 1) return K <= 8192;
  const bool idle = 3 * ((N + 127) / 128) <= cus;
  return !idle || (rows == kW4RowsConverted ? K < 4096 : M <= 40 || K < 6144);
}

template <int MT, bool BF16>
static void launch_w4s(const W4StreamArgs& a, const W4StreamForm& f, hipStream_t stream) {
  const int tiles = (a.N + 15) / 16;
  const dim3 grid((unsigned)((tiles + f.nt - 1) / f.nt * f.ksplit)), block(64 * kW4sWaves);
  switch (f.nt) {
    case 4: hipLaunchKernelGGL((w4a16_stream_kernel<MT, 4, BF16>), grid, block, 0, stream, a); break;
    case 6: hipLaunchKernelGGL((w4a16_stream_kernel<MT, 6, BF16>), grid, block, 0, stream, a); break;
    case 8: hipLaunchKernelGGL((w4a16_stream_kernel<MT, 8, BF16>), grid, block, 0, stream, a); break;
    default: hipLaunchKernelGGL((w4a16_stream_kernel<MT, 10, BF16>), grid, block, 0, stream, a); break;
  }
}

void launch_w4_stream(const W4StreamArgs& a, const W4StreamForm& f, hipStream_t stream) {
  if (a.M <= 32) {
    if (a.x_bf16) launch_w4s<2, true>(a, f, stream);
    else launch_w4s<2, false>(a, f, stream);
  } else {
    if (a.x_bf16) launch_w4s<3, true>(a, f, stream);
    else launch_w4s<3, false>(a, f, stream);
  }
}

}  // namespace kq
