// Panel GEMM for tens to a few hundred activation rows (gfx950): INT8, FP8
// and block-scaled FP8 weights, the products of kq_stream_gemm.h.
//
// Between the decode batches, which are bound by the weight stream alone, and
// prefill, which fills the matrix cores with 256 x 256 tiles, a GEMM is bound
// by what its workgroups copy into LDS: the weights once per row tile and the
// activations once per weight panel.  So a workgroup takes every row it can
// (BM = 16 * MTW * WM, up to 256) against a panel of 16 * NT weight rows:
//   * wave w owns the 16 * MTW activation rows 16 * MTW * w ... and all the
//     panel's columns.  Its activation rows are its own part of a stage (it
//     copies them and alone reads them); the panel's weight rows are copied by
//     all waves and read by all.
//   * K advances in stages of 128 bytes through a ring of R slots filled by
//     LDS DMA in whole lines, R - 1 stages ahead, one barrier per stage: it
//     both publishes stage i and frees the slot of stage i - 1.
//   * Weights are the MFMA A operand: a lane's four results are four
//     consecutive columns of one row (one activation scale).
//   * Few panels split K over workgroups; raw accumulators go to `partials`
//     and the split-K reduce adds them in order.
#pragma once

#include "kq_common.h"
#include "kq_stream_gemm.h"

#include <algorithm>

namespace kq {

struct PanelArgs {
  StreamArgs s;        // quantized activations; table, gather, RAW fields unused
  int splits;          // K split over this many workgroups per panel
  uint32_t* partials;  // [splits][M][P] raw accumulators, P = N (SW: 2N, up columns from N)
};

template <int FMT, int MTW, int WM, int NT, int R, bool SW>
struct PgLds {
  static constexpr int BM = 16 * MTW * WM;
  static constexpr int W = NT * 2048;
  static constexpr int X = BM * 128;
  static constexpr int Xs = FMT == kSgBlock ? WM * 256 : 0;  // a wave's 16 * MTW block scales in 64 slots
  static constexpr int Stage = W + X + Xs;
  // block FP8: weight scales of the panel's 128-row blocks, up to 128 K blocks
  static constexpr int WsRows = SW ? 2 : (16 * NT + 127) / 128;
  static constexpr int Ws = R * Stage;
  static constexpr int EpiXs = Ws;                           // INT8, FP8: a wave's row scales in 64 slots
  static constexpr int EpiWs = EpiXs + WM * 256;             // column scales (SW: gate's, then up's)
  static constexpr int WsParts = ((SW ? 8 : 16) * NT + 63) / 64;  // in copies of 64
  static constexpr int Bytes = FMT == kSgBlock ? Ws + WsRows * 512 : EpiWs + (SW ? 2 : 1) * WsParts * 256;
};

template <int FMT, int MTW, int WM, int NT, int R, bool SW>
__global__ void __launch_bounds__(64 * WM) panel_gemm_kernel(PanelArgs pa) {
  const StreamArgs& a = pa.s;
  using L = PgLds<FMT, MTW, WM, NT, R, SW>;
  using Acc = typename SgAcc<FMT>::T;
  constexpr bool BLOCK = FMT == kSgBlock;
  constexpr int TF = FMT == kSgI8 ? kTgI8 : kTgFp8;
  constexpr int COLS = (SW ? 8 : 16) * NT;
  static_assert(2 * NT % WM == 0, "every wave copies as many weight rows");
  static_assert(!BLOCK || (COLS & (COLS - 1)) == 0, "a panel's columns lie in whole scale blocks or in one");
  static_assert(L::Bytes <= 160 * 1024, "the ring exceeds a CU's 160 KB of LDS");
  constexpr int WI = 2 * NT / WM, XI = 2 * MTW;
  constexpr int OPS = WI + XI + (BLOCK ? 1 : 0);
  static_assert((R - 1) * OPS <= 63, "vmcnt counts to 63");
  __shared__ __attribute__((aligned(16))) uint8_t smem[L::Bytes];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int j = lane & 15, kg = lane >> 4;
  const int K = a.K, KB = (K + 127) / 128;
  const int ktail = K - (KB - 1) * 128;
  const int c0 = (int)blockIdx.x * COLS;
  const int row0 = (int)blockIdx.y * L::BM;
  const int split = blockIdx.z;
  const int kb0 = (int)((int64_t)KB * split / pa.splits), kb1 = (int)((int64_t)KB * (split + 1) / pa.splits);
  const int n = kb1 - kb0;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;

  // copies: weight instruction q = wave * WI + i covers 8 rows, half q & 1 of
  // tile q >> 1 (SW: the halves are gate and up rows)
  const uint32_t wbytes = (uint32_t)min(COLS, a.N - c0) * (uint32_t)K;
  const i32x4 rw = make_rsrc(a.w + (int64_t)c0 * K, wbytes);
  const i32x4 ru = SW ? make_rsrc(a.w_up + (int64_t)c0 * K, wbytes) : rw;
  const i32x4 rx = make_rsrc(a.x, a.x_bytes);
  const i32x4 rxs = make_rsrc(a.xs, BLOCK ? (uint32_t)((uint64_t)a.x_rows * KB * 4) : 0u);
  int chunk[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) chunk[h] = tg_chunk<TF>(8 * h + (lane >> 3), lane & 7);
  int32_t vw[WI], vx[XI], vxs = kTgOob;
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int q = wave * WI + i, h = q & 1, t = q >> 1;
    const int row = SW ? 8 * t + (lane >> 3) : 16 * t + 8 * h + (lane >> 3);
    const int ch = h ? chunk[1] : chunk[0];
    vw[i] = c0 + row < a.N ? row * K + ch * 16 : kTgOob;
  }
  const int wrow0 = row0 + 16 * MTW * wave;  // the wave's first row
#pragma unroll
  for (int h = 0; h < XI; ++h) {
    const int r = wrow0 + 8 * h + (lane >> 3);
    vx[h] = r < a.M ? r * K + chunk[h & 1] * 16 : kTgOob;
  }
  if (BLOCK && lane < 16 * MTW && wrow0 + lane < a.M) vxs = (wrow0 + lane) * KB * 4;
  auto issue = [&](int i, int slot) {
    const int kb = kb0 + i;
    const int32_t so = __builtin_amdgcn_readfirstlane(kb * 128);
    const bool tail = !BLOCK && ktail != 128 && kb == KB - 1;
    const uint32_t b = lds0 + slot * L::Stage;
#pragma unroll
    for (int e = 0; e < WI; ++e) {
      const int q = wave * WI + e;
      const int ch = (q & 1) ? chunk[1] : chunk[0];
      tg_dma16nt(SW && (q & 1) ? ru : rw, b + q * 1024, tail && ch * 16 >= ktail ? kTgOob : vw[e], so);
    }
#pragma unroll
    for (int h = 0; h < XI; ++h)
      tg_dma16(rx, b + L::W + (wave * XI + h) * 1024, tail && chunk[h & 1] * 16 >= ktail ? kTgOob : vx[h], so);
    if constexpr (BLOCK)
      tg_dma4(rxs, b + L::W + L::X + wave * 256, vxs, __builtin_amdgcn_readfirstlane(kb * 4));
  };

  // scales that the K loop or the epilogue reads, ahead of the first stage
  if constexpr (BLOCK) {
    if (wave < 2 * L::WsRows) {  // half of a scale row each
      const int wr = wave >> 1, half = wave & 1;
      const float* src = SW && wr ? a.ws_up : a.ws;
      const int nb = min(c0 / 128 + (SW ? 0 : wr), (a.N + 127) / 128 - 1);
      const int kb = half * 64 + lane;
      tg_dma4(make_rsrc(src + (int64_t)nb * KB, (uint32_t)KB * 4u), lds0 + L::Ws + wr * 512 + half * 256,
              kb < KB ? kb * 4 : kTgOob, 0);
    }
  } else {
    const int r = wrow0 + lane;
    tg_dma4(make_rsrc(a.xs, (uint32_t)a.M * 4u), lds0 + L::EpiXs + wave * 256,
            lane < 16 * MTW && r < a.M ? r * 4 : kTgOob, 0);
    for (int q = wave; q < (SW ? 2 : 1) * L::WsParts; q += WM) {
      const int c = q % L::WsParts * 64 + lane;
      const bool live = c < COLS && c0 + c < a.N;
      const uint32_t bytes = a.ws_per_channel ? (uint32_t)min(COLS, a.N - c0) * 4u : 4u;
      tg_dma4(make_rsrc((q >= L::WsParts ? a.ws_up : a.ws) + (a.ws_per_channel ? c0 : 0), bytes),
              lds0 + L::EpiWs + q * 256, !live ? kTgOob : a.ws_per_channel ? c * 4 : 0, 0);
    }
  }

#pragma unroll
  for (int i = 0; i < R - 1; ++i)
    if (i < n) issue(i, i);

  const int o_lo = j * 128 + (tg_chunk<TF>(j, TF == kTgFp8 ? 2 * kg : kg) << 4);
  const int o_hi = j * 128 + (tg_chunk<TF>(j, TF == kTgFp8 ? 2 * kg + 1 : 4 + kg) << 4);
  Acc acc[NT][MTW];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int t = 0; t < MTW; ++t) acc[nt][t] = Acc{0, 0, 0, 0};
  const bool rows = wrow0 < a.M;  // waves past the last row copy weights only

  for (int i = 0; i < n; ++i) {
    sg_wait_stages<OPS, R - 2>(min(R - 2, n - 1 - i));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (i + R - 1 < n) issue(i + R - 1, (i + R - 1) % R);
    if (!rows) continue;
    const uint8_t* q = smem + (i % R) * L::Stage;
    const uint8_t* xq = q + L::W + wave * (MTW * 2048);
    i32x4 xl[MTW], xh[MTW];
    float sx[MTW], sw[L::WsRows];
#pragma unroll
    for (int t = 0; t < MTW; ++t) {
      xl[t] = *(const i32x4*)(xq + t * 2048 + o_lo);
      xh[t] = *(const i32x4*)(xq + t * 2048 + o_hi);
    }
    if constexpr (BLOCK) {
#pragma unroll
      for (int t = 0; t < MTW; ++t) sx[t] = *(const float*)(q + L::W + L::X + wave * 256 + (16 * t + j) * 4);
#pragma unroll
      for (int w2 = 0; w2 < L::WsRows; ++w2) sw[w2] = *(const float*)(smem + L::Ws + w2 * 512 + (kb0 + i) * 4);
      // lane rows 4 kg ... of a tile: gate rows for kg < 2, up rows beyond
      if constexpr (SW) sw[0] = kg < 2 ? sw[0] : sw[1];
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const i32x4 wl = *(const i32x4*)(q + nt * 2048 + o_lo), wh = *(const i32x4*)(q + nt * 2048 + o_hi);
      const i32x8 wv = i32x8{wl[0], wl[1], wl[2], wl[3], wh[0], wh[1], wh[2], wh[3]};
#pragma unroll
      for (int t = 0; t < MTW; ++t) {
        if constexpr (FMT == kSgI8) {
          acc[nt][t] = mfma_i8(wh, xh[t], mfma_i8(wl, xl[t], acc[nt][t]));
        } else {
          const i32x8 xv = i32x8{xl[t][0], xl[t][1], xl[t][2], xl[t][3], xh[t][0], xh[t][1], xh[t][2], xh[t][3]};
          if constexpr (BLOCK) {
            const f32x4 p = mfma_fp8(wv, xv, f32x4{0.f, 0.f, 0.f, 0.f});
            const float c = sx[t] * sw[SW ? 0 : nt / 8];
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[nt][t][r] = fmaf(p[r], c, acc[nt][t][r]);
          } else {
            acc[nt][t] = mfma_fp8(wv, xv, acc[nt][t]);
          }
        }
      }
    }
  }
  if (!rows) return;

  const float* epi_xs = (const float*)(smem + L::EpiXs) + wave * 64;  // landed before stage 0
  const float* epi_ws = (const float*)(smem + L::EpiWs);
  const int P = SW ? 2 * a.N : a.N;
#pragma unroll
  for (int t = 0; t < MTW; ++t) {
    const int m = wrow0 + 16 * t + j;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      // lane (j, kg): columns cl ... cl + 3 of row m (SW: of gate for kg < 2, of up beyond)
      const int cl = SW ? 8 * nt + 4 * (kg & 1) : 16 * nt + 4 * kg;
      const int c = c0 + cl;
      const bool up_lane = SW && kg >= 2;
      if (pa.splits > 1) {
        if (m < a.M) {
          uint32_t* part = pa.partials + ((int64_t)split * a.M + m) * P + (up_lane ? a.N : 0) + c;
          if (c + 4 <= a.N && (a.N & 3) == 0) {
            *(u32x4*)part = u32x4{sg_bits(acc[nt][t], 0), sg_bits(acc[nt][t], 1), sg_bits(acc[nt][t], 2),
                                  sg_bits(acc[nt][t], 3)};
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (c + r < a.N) part[r] = sg_bits(acc[nt][t], r);
          }
        }
        continue;
      }
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = (float)acc[nt][t][r];
        if constexpr (!BLOCK) {
          v[r] = __fmul_rn(__fmul_rn(v[r], epi_xs[16 * t + j]), epi_ws[(up_lane ? L::WsParts * 64 : 0) + cl + r]);
        }
        if (a.bias_dtype != KQ_DTYPE_NONE && c + r < a.N)
          v[r] = __fadd_rn(v[r], load_as_f32(up_lane ? a.bias_up : a.bias, a.bias_dtype, c + r));
      }
      if constexpr (SW) {
        // the halves of the wave swap two columns: gate lanes finish columns
        // cl, cl + 1, up lanes cl + 2, cl + 3
        const float s0 = __shfl_xor(up_lane ? v[0] : v[2], 32, 64), s1 = __shfl_xor(up_lane ? v[1] : v[3], 32, 64);
        const uint32_t o = up_lane ? swiglu_bits2(s0, v[2], s1, v[3], a.out_dtype)
                                   : swiglu_bits2(v[0], s0, v[1], s1, a.out_dtype);
        const int oc = c + (up_lane ? 2 : 0);
        if (m < a.M) {
          uint16_t* dst = (uint16_t*)a.out + (int64_t)m * a.N + oc;
          if (oc + 1 < a.N && ((uintptr_t)dst & 3) == 0) {
            *(uint32_t*)dst = o;
          } else {
            if (oc < a.N) dst[0] = (uint16_t)o;
            if (oc + 1 < a.N) dst[1] = (uint16_t)(o >> 16);
          }
        }
      } else if (m < a.M) {
        if constexpr (FMT == kSgI8) {
          if (a.acc_out) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (c + r < a.N) a.acc_out[(int64_t)m * a.N + c + r] = acc[nt][t][r];
          }
        }
        uint16_t* o = (uint16_t*)a.out + (int64_t)m * a.N + c;
        if (c + 4 <= a.N && (((uintptr_t)o) & 7) == 0) {
          *(u32x2*)o = u32x2{pack_act2(v[0], v[1], a.out_dtype), pack_act2(v[2], v[3], a.out_dtype)};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (c + r < a.N) o[r] = f32_to_out(v[r], a.out_dtype);
        }
      }
    }
  }
}

// ------------------------------------------------------------------ launch
struct PanelForm {
  int nt;      // weight tiles per panel
  int mtw;     // row tiles per wave (4 waves at nt = 4, else 8)
  int splits;
};

// Form for M rows (65 to 256) of `tiles` 16-row weight tiles and KB K blocks;
// nt = 0: another kernel.  One round of workgroups over most CUs at the widest
// panel that gives it, since a panel's activations are copied once: 8 tiles,
// and up to 128 rows 12 or 16 where those of 8 are more than the CUs.  (Beyond
// 128 rows wider panels only match the tile engine: I = 18944 K = 3584 M = 200
// 68.7 us with 12 tiles, 67.0.)
//
// Fewer panels than half the CUs: panels of 4 tiles against 128 rows, split
// over K while that leaves CUs idle, with at least 7 K blocks each, 12 where the
// halves fill the CUs (N = 4096 M = 256, FP8, K = 2048 17.5 us whole and 18.3 in
// two of 8; INT8, K = 3072 23.9 and 22.2); panels of 8 tiles split over K where K
// is long, 64 blocks, or 48 where the panels of 4 are more than half the CUs and
// would run unsplit, 40 up to 160 rows (N = 4096 M = 256 K = 4096 / 6144 / 8192
// INT8 in panels of 4, split in two, against 8: 23.9 / 30.2 / 34.9 and 27.2 /
// 30.0 / 31.7; N = 7168 K = 5120 unsplit against panels of 8 split 4 ways: FP8 M =
// 129 / 256 30.1 / 33.0 and 28.2 / 35.6, N = 8192 K = 6144 INT8 39.1 / 41.2 and
// 32.4 / 37.2).  Measured, INT8 with its quantizer (us, weights out of cache; the
// tile engine in brackets): N = K = 4096 M = 128 / 256 18.7 / 23.9 [29 / 34],
// N = 3456 K = 5120 M = 129 23.6 [30], N = 8192 K = 7168 M = 65 / 190 28.8 / 35.3
// [38 / 46].
static inline PanelForm pg_form(int64_t M, int64_t tiles, int KB) {
  const int64_t cus = tg_device_cus();
  const int big_m = M > 128 ? 2 : 1;
  auto panels = [&](int nt) { return (tiles + nt - 1) / nt; };
  if (panels(8) > cus / 2) {
    int nt = panels(8) <= cus ? 8 : 0;
    if (nt == 0 && M <= 128) nt = panels(12) <= cus ? 12 : panels(16) <= cus ? 16 : 0;
    return PanelForm{nt, big_m, 1};
  }
  const int64_t units = panels(4) * ((M + 127) / 128);
  if (KB >= (2 * units <= cus ? 64 : M > 128 && M <= 160 ? 40 : 48)) return PanelForm{8, big_m, (int)std::min<int64_t>(8, cus / panels(8))};
  if (M > 128 && units > cus) return PanelForm{0, 0, 1};
  const int64_t s = std::min<int64_t>({4, cus / units, KB / (units < 96 ? 7 : 12)});
  return PanelForm{4, 2, (int)std::max<int64_t>(1, s)};
}

template <int FMT, int MTW, int WM, int NT, int R, bool SW>
static void pg_launch_form(const PanelArgs& a, hipStream_t stream) {
  constexpr int cols = (SW ? 8 : 16) * NT, bm = 16 * MTW * WM;
  const dim3 grid((unsigned)((a.s.N + cols - 1) / cols), (unsigned)((a.s.M + bm - 1) / bm), (unsigned)a.splits);
  hipLaunchKernelGGL((panel_gemm_kernel<FMT, MTW, WM, NT, R, SW>), grid, dim3(64 * WM), 0, stream, a);
}

// INT8 / FP8 (a.splits from the form; partials are reduced by the caller).
template <int FMT, bool SW>
static void pg_launch(const PanelArgs& a, const PanelForm& f, hipStream_t stream) {
  if (f.nt == 4) pg_launch_form<FMT, 2, 4, 4, 4, SW>(a, stream);
  else if (f.mtw == 1) {
    if (f.nt == 8) pg_launch_form<FMT, 1, 8, 8, 3, SW>(a, stream);
    else if (f.nt == 12) pg_launch_form<FMT, 1, 8, 12, 3, SW>(a, stream);
    else pg_launch_form<FMT, 1, 8, 16, 3, SW>(a, stream);
  } else {
    pg_launch_form<FMT, 2, 8, 8, 3, SW>(a, stream);
  }
}

// Whether block FP8 rows (at most 256) of an unfused product run here or in
// the streaming kernel; else the tile engine.  A panel of 8 tiles takes a CU's
// LDS, so past one round of them the second is paid in full: N = 16384 /
// 16512, M = 256, us, panels against tile engine, K = 2048 31 / 40 and 53 / 40,
// K = 4096 50 / 70 and 90 / 71, K = 8192 88 / 127 and 158 / 126; N = 32768 /
// 33024, M = 128, K = 4096 51 / 68 and 88 / 68.  The streaming kernel meets the
// tile engine later: N = 37888 / 57344 (296 and 448 panels), M = 64, K = 4096
// 62 / 65 and 81 / 74, M = 49 56 / 64 and 73 / 73.
static inline bool pg_block_applies(int64_t m, int64_t n) {
  const int64_t panels = (n + 127) / 128, cus = tg_device_cus();
  return m <= 48 || (m <= 64 ? 2 * panels <= 3 * cus : panels * ((m + 127) / 128) <= cus);
}

// Block FP8, 65 to 256 rows (no split K): panels of 8, 4 or 2 tiles against
// 128 rows, the widest that gives half the CUs a workgroup.  M = 200, us, with
// the quantizer: N = K = 4096 30.5 with 2 tiles (the tile engine 66); 12288
// rows K = 4096 47.7 with 8 (68).  Every form adds an element's K blocks in
// one order, so a SwiGLU launch gives the bits of its two projections.
static inline int pg_block_tiles(int64_t m, int64_t n, bool sw) {
  auto units = [&](int nt) {
    const int cols = (sw ? 8 : 16) * nt;
    return (n + cols - 1) / cols * ((m + 127) / 128);
  };
  const int64_t need = tg_device_cus() / 2;
  return units(8) >= need ? 8 : units(4) >= need ? 4 : 2;
}
template <bool SW>
static inline void pg_launch_block(const StreamArgs& s, hipStream_t stream) {
  const PanelArgs a{s, 1, nullptr};
  const int nt = pg_block_tiles(s.M, s.N, SW);
  if (nt == 8) pg_launch_form<kSgBlock, 2, 4, 8, 3, SW>(a, stream);
  else if (nt == 4) pg_launch_form<kSgBlock, 2, 4, 4, 4, SW>(a, stream);
  else pg_launch_form<kSgBlock, 2, 4, 2, 4, SW>(a, stream);
}

// 33 to 64 rows against more than two weight tiles per CU: panels of 4 tiles,
// several workgroups per CU (FP8, M = 64, SwiGLU I = 14336 K = 4096 30.9 us, the
// streaming kernel 41.3; I = 18944 K = 3584 39.0 and 51.2).
static inline bool pg_64_applies(int64_t m, int64_t tiles) { return m > 32 && tiles > 2 * (int64_t)tg_device_cus(); }
template <int FMT, bool SW>
static void pg_launch_64(const PanelArgs& a, hipStream_t stream) {
  pg_launch_form<FMT, 1, 4, 4, 3, SW>(a, stream);
}

}  // namespace kq
