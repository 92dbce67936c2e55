// Weight-streaming GEMM for few activation rows (gfx950): INT8, FP8 and
// block-scaled FP8 weights.
//
//   INT8, FP8 : out[m, n] = ((xq[m] . wq[n]) * xs[m]) * ws[n] (+ bias[n])
//   block FP8 : out[m, n] = sum_b xs[m][b] * ws[n/128][b] * (xq . wq over block b) (+ bias[n])
//
// for row tiles of 16 * MT rows: decode batches of the dense linears and the
// MoE experts of a few rows each.  Bound by the HBM stream of the weights, so
// everything else is arranged around keeping that stream full:
//   * A workgroup owns 16 * NT output columns; its NW waves take K blocks
//     (128 bytes of K, one scale block) wave, wave + NW, ...: the waves of a
//     workgroup stream neighbouring lines of the same weight rows (but where
//     the rows' pitch would put those on the same memory channels: sg_apart).
//   * Every wave keeps a private ring of R stages in LDS, filled by LDS DMA
//     in whole 128-byte lines (8 rows x 128 B per instruction) and read back
//     as MFMA fragments through the tile engine's chunk swizzle.  A wave only
//     waits (vmcnt) for its own stage: no barrier in the K loop, and every
//     staged byte is read from LDS once.
//   * NT column tiles share each activation fragment, so the activation
//     traffic (M rows per workgroup, from L2) falls with NT.
//   * RAW (block FP8): the activations are the fp16 / bf16 rows themselves; a
//     1x128 block is exactly one stage's slice of a row, so each wave
//     quantizes the slice it has staged (amax over the 8 lanes of a row, the
//     quantizer's bytes and scale) and no quantization launch runs.
//   * RAW (INT8, FP8; one row): every workgroup reads the row once for its
//     amax while its first weight copies are in flight, then the waves
//     quantize their slices.  (With more rows the repeated amax pass costs
//     what the quantization launch does.)
//   * SW: column tile t holds 8 gate columns [8t, 8t + 8) and the matching 8
//     up columns; the epilogue stores silu(gate) * up with torch's roundings.
//   * The waves' partial sums meet in LDS (in their own rings' space) and are
//     added in wave order: deterministic.
#pragma once

#include "kq_common.h"
#include "kq_tile_gemm.h"

namespace kq {

enum { kSgI8 = 0, kSgFp8 = 1, kSgBlock = 2 };

struct StreamArgs {
  const void* x;          // RAW: 16-bit activations [rows][ldx]; else bytes [rows][K]
  int ldx;                // RAW: row pitch in elements
  uint32_t x_bytes;       // bytes addressable through x
  const float* xs;        // INT8, FP8: [rows]; block FP8: [rows][K/128] (not RAW)
  int x_rows;             // rows of xs
  const uint8_t* w;       // [E][N][K]; SW: the gate rows
  const uint8_t* w_up;    // SW: the up rows (same expert pitch)
  int64_t w_pitch;        // bytes between experts
  const float* ws;        // INT8, FP8: [N], or [1]; block FP8: [E][ceil(N/128)][K/128]; SW: gate's
  const float* ws_up;     // SW
  int ws_per_channel;     // INT8, FP8
  int64_t ws_pitch;       // floats between experts
  const int32_t* gather;  // routed row -> row of x; null: identity
  const int32_t* table;   // row tiles [][4] (expert, first row, end row, 0); null: dense
  const int32_t* count;   // row tiles in use (device)
  int M, N, K;            // N: output columns (SW: activation columns I)
  const void* bias;       // [N] (SW: of the gate columns) or null
  const void* bias_up;
  int bias_dtype;
  void* out;              // [rows][N]
  int out_dtype;
  int32_t* acc_out;       // INT8, not SW: raw accumulators [M][N], or null
  int splits;             // SPLIT: blockIdx.z's, and the K blocks of each
  int split_blocks;
  uint32_t* partials;     // SPLIT: [splits][M][P] raw accumulators, P = N (SW: 2N, up columns from N)
  int scale_mode;         // RAW INT8, FP8: 0 dynamic, 1 scale_in[0], 2 scale_in[row]
  const float* scale_in;
};

template <int N_>
KQ_DEV void sg_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_) : "memory");
}

// Waits until at most `stages` * OPS vector-memory operations are in flight.
template <int OPS, int MAX>
KQ_DEV void sg_wait_stages(int stages) {
  if constexpr (MAX >= 5) { if (stages >= 5) { sg_wait_vm<5 * OPS>(); return; } }
  if constexpr (MAX >= 4) { if (stages >= 4) { sg_wait_vm<4 * OPS>(); return; } }
  if constexpr (MAX >= 3) { if (stages >= 3) { sg_wait_vm<3 * OPS>(); return; } }
  if constexpr (MAX >= 2) { if (stages >= 2) { sg_wait_vm<2 * OPS>(); return; } }
  if (stages >= 1) sg_wait_vm<OPS>();
  else sg_wait_vm<0>();
}

// The larger of each 16-bit half; the four words' largest 16-bit magnitudes;
// half h of a word of fp16 / bf16 pairs as fp32.
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
KQ_DEV uint32_t sg_max_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
KQ_DEV uint32_t sg_abs_max4(u32x4 r) {
  return sg_max_u16(sg_max_u16(r[0] & 0x7fff7fffu, r[1] & 0x7fff7fffu),
                    sg_max_u16(r[2] & 0x7fff7fffu, r[3] & 0x7fff7fffu));
}
template <int DT>
KQ_DEV float sg_widen(uint32_t w, int h) {
  if constexpr (DT == KQ_DTYPE_BF16) return __uint_as_float(h ? w & 0xffff0000u : w << 16);
  else return f16_to_f32((uint16_t)(h ? w >> 16 : w & 0xffffu));
}

KQ_DEV uint32_t sg_bits(i32x4 a, int r) { return (uint32_t)(int)a[r]; }
KQ_DEV uint32_t sg_bits(f32x4 a, int r) { return __float_as_uint((float)a[r]); }

// The e4m3 bytes of 16 consecutive elements of a 1x128 block (r0, r1), one
// block per 8 consecutive lanes, and the block's scale to *scale unless null:
// act_quant_fp8_blocks_kernel's scale and (but for the sign of a zero) bytes.
// The amax is an integer max of the 16-bit magnitudes (they order inf and NaN
// above every finite value), two elements per instruction, over the 8 lanes:
// quad exchanges, then the half-row mirror.  Finite blocks take the reciprocal
// with an fma remainder step (div_by_recip) without its clamp: |v / s| is at
// most an ulp over 448, which rounds to 448.
template <int DT>
KQ_DEV u32x4 sg_quant16(u32x4 r0, u32x4 r1, float* scale) {
  uint32_t ab = sg_max_u16(sg_abs_max4(r0), sg_abs_max4(r1));
  ab = max(ab & 0xffffu, ab >> 16);
  ab = dpp_max_u32<0xB1>(ab);
  ab = dpp_max_u32<0x4E>(ab);
  ab = dpp_max_u32<0x141>(ab);
  float v[16];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    v[2 * d] = sg_widen<DT>(r0[d], 0);
    v[2 * d + 1] = sg_widen<DT>(r0[d], 1);
    v[8 + 2 * d] = sg_widen<DT>(r1[d], 0);
    v[9 + 2 * d] = sg_widen<DT>(r1[d], 1);
  }
  const float s = __fdiv_rn(max_keep_nan(sg_widen<DT>(ab, 0), 1e-12f), 448.0f);
  if (scale) *scale = s;
  u32x4 o;
  if (__ballot(ab >= (DT == KQ_DTYPE_BF16 ? 0x7f80u : 0x7c00u)) == 0) {
    const float rs = __fdiv_rn(1.0f, s);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float q0 = v[e] * rs;
      v[e] = fmaf(fmaf(-q0, s, v[e]), rs, q0);
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = pack4_e4m3(v[4 * d], v[4 * d + 1], v[4 * d + 2], v[4 * d + 3]);
  } else {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t p = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        p |= f32_to_e4m3(clamp_keep_nan(__fdiv_rn(v[4 * d + e], s), 448.0f)) << (8 * e);
      o[d] = p;
    }
  }
  return o;
}

// Two elements of a row quantized by its scale s (rs = RN(1 / s)): the
// per-token quantizer's bytes.  Finite elements under a scale for which it is
// exact (`ok`) take the reciprocal path, decided per wave: there both give the
// same byte.
template <int FMT, int DT>
KQ_DEV uint16_t sg_quant2(uint32_t raw, float s, float rs, bool ok) {
  constexpr float QMAX = FMT == kSgFp8 ? 448.0f : 127.0f;
  const float lo = sg_widen<DT>(raw, 0), hi = sg_widen<DT>(raw, 1);
  const bool fast = ok && (__float_as_uint(lo) & 0x7fffffffu) < 0x7f800000u &&
                    (__float_as_uint(hi) & 0x7fffffffu) < 0x7f800000u;
  if (__ballot(!fast) == 0) {
    const float a = fminf(fmaxf(div_by_recip(lo, s, rs), -QMAX), QMAX);
    const float b = fminf(fmaxf(div_by_recip(hi, s, rs), -QMAX), QMAX);
    if constexpr (FMT == kSgFp8) return (uint16_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    else return (uint16_t)(((uint32_t)(int32_t)__builtin_rintf(a) & 0xffu) | ((uint32_t)(int32_t)__builtin_rintf(b) << 8));
  }
  const float a = clamp_keep_nan(__fdiv_rn(lo, s), QMAX), b = clamp_keep_nan(__fdiv_rn(hi, s), QMAX);
  if constexpr (FMT == kSgFp8) return (uint16_t)(f32_to_e4m3(a) | (f32_to_e4m3(b) << 8));
  else return (uint16_t)(((uint32_t)(int32_t)__builtin_rintf(a) & 0xffu) | (((uint32_t)(int32_t)__builtin_rintf(b) & 0xffu) << 8));
}

// Bytes of one wave's LDS: R stages of NT weight tiles (2 KB each) and the
// activations (RAW: 256-byte rows, 8 * XH of them; else 128-byte rows and 64
// scales), plus the quantized fragment and its scales (RAW).
template <int FMT, bool RAW, int MT, int NT, int R, int XH, bool SW>
struct SgLds {
  static constexpr int W = NT * 2048;
  static constexpr int X = !RAW ? MT * 2048 : FMT == kSgBlock ? XH * 2048 : 1024;
  static constexpr int Xs = FMT == kSgBlock && !RAW ? 256 : 0;
  static constexpr int Stage = W + X + Xs;
  static constexpr int Rows = FMT == kSgBlock ? 8 * XH : 1;         // RAW: rows quantized
  static constexpr int Frag = R * Stage;              // RAW: their bytes of one K block
  static constexpr int Zero = Frag + (RAW ? Rows * 128 : 0);        // RAW: the other fragment rows
  static constexpr int Sc = Zero + (RAW && Rows < 16 ? 128 : 0);    // RAW: 16 row scales
  static constexpr int Ws = Sc + (RAW ? 64 : 0);      // block: this wave's K blocks' weight scales
  static constexpr int Ring = Ws + (FMT != kSgBlock ? 0 : SW ? 512 : 256);
  static constexpr int Gat = (R - 1) * Stage;         // routed rows' sources: the slot that the loop
                                                      // fills first, after they are read
  static constexpr int Red = MT * NT * 1024;          // the wave's partial sums
  static constexpr int Wave = (Ring > Red ? Ring : Red);
  // past the waves': INT8, FP8 the epilogue's row scales (64) and column
  // scales (64; SW 2 x 64), RAW the waves' maxima (16)
  static constexpr int ShWs = 256;
  static constexpr int ShMax = ShWs + (SW ? 512 : 256);
  static constexpr int Shared = FMT == kSgBlock ? 0 : ShMax + (RAW ? 64 : 0);
};

template <int FMT> struct SgAcc { using T = f32x4; };
template <> struct SgAcc<kSgI8> { using T = i32x4; };

// XH: with RAW block FP8, activation rows present in units of 8 (M <= 8: 1).
// DT: with RAW, the activations' dtype.
// SPLIT (INT8, FP8, quantized rows): blockIdx.z takes a range of the K blocks
// and stores raw accumulators.
// APART (INT8, FP8; NW divides the K blocks): a wave takes neighbouring K
// blocks, not blocks wave, wave + NW, ...
template <int FMT, bool RAW, int MT, int NT, int NW, int R, int XH, bool SW, int DT, bool SPLIT, bool APART>
__global__ void __launch_bounds__(64 * NW) stream_gemm_kernel(StreamArgs a) {
  static_assert(!RAW || MT == 1, "at most one row tile quantizes in the launch");
  static_assert(!SPLIT || (FMT != kSgBlock && !RAW), "quantized INT8 / FP8 rows split");
  static_assert(!APART || (FMT != kSgBlock && !SPLIT), "block scales are slotted by wave");
  using L = SgLds<FMT, RAW, MT, NT, R, XH, SW>;
  using Acc = typename SgAcc<FMT>::T;
  constexpr bool BLOCK = FMT == kSgBlock;
  constexpr int COLS = (SW ? 8 : 16) * NT;  // output columns of the workgroup
  constexpr int TF = FMT == kSgI8 ? kTgI8 : kTgFp8;
  static_assert(L::Wave * NW + L::Shared <= 160 * 1024, "the rings exceed a CU's 160 KB of LDS");
  constexpr int XI = !RAW ? 2 * MT : BLOCK ? 2 * XH : 1;  // row-data instructions per stage
  constexpr int OPS = 2 * NT + XI + (BLOCK && !RAW ? 1 : 0);
  static_assert((R - 1) * OPS <= 63, "vmcnt counts to 63");
  // One array for everything: with several, the compiler tells them apart by
  // alias scopes and makes every LDS read wait for copies into another array
  // (N = 4096 K = 14336 M = 8: 13.1 -> 11.6 us for one wait in the K loop).
  __shared__ __attribute__((aligned(16))) uint8_t smem[NW * L::Wave + L::Shared];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int j = lane & 15, kg = lane >> 4;
  const int K = a.K, KB = (K + 127) / 128;
  const int ktail = K - (KB - 1) * 128;  // bytes of K in the last block (16..128)
  const int ct0 = blockIdx.x * NT;       // first 16-row weight tile of the workgroup

  int expert = 0, row0 = (int)blockIdx.y * 16 * MT, row_end = min(a.M, row0 + 16 * MT);
  if (a.table) {
    if ((int)blockIdx.y >= *a.count) return;
    const int32_t* t = a.table + 4 * (int64_t)blockIdx.y;
    expert = __builtin_amdgcn_readfirstlane(t[0]);
    row0 = __builtin_amdgcn_readfirstlane(t[1]);
    row_end = __builtin_amdgcn_readfirstlane(t[2]);
  }

  // weight rows: (tile, 8-row half, lane / 8); SW halves are gate and up rows
  const int c0 = SW ? 8 * ct0 : 16 * ct0;  // first output column
  const uint8_t* wb = a.w + expert * a.w_pitch + (int64_t)c0 * K;
  const uint8_t* wu = SW ? a.w_up + expert * a.w_pitch + (int64_t)c0 * K : wb;
  const uint32_t wbytes = (uint32_t)min(COLS, a.N - c0) * (uint32_t)K;
  const i32x4 rw = make_rsrc(wb, wbytes);
  const i32x4 ru = SW ? make_rsrc(wu, wbytes) : rw;
  int32_t vw[NT][2];
  int chunk[2];  // the K chunk this lane copies, per 8-row half
#pragma unroll
  for (int h = 0; h < 2; ++h) chunk[h] = tg_chunk<TF>(8 * h + (lane >> 3), lane & 7);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = SW ? 8 * nt + (lane >> 3) : 16 * nt + 8 * h + (lane >> 3);  // from c0
      vw[nt][h] = c0 + row < a.N ? row * K + chunk[h] * 16 : kTgOob;
    }
  uint8_t* const mine = smem + wave * L::Wave;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint32_t lds0 = lds_base + wave * L::Wave;

  // this wave's K blocks: kbeg + i * kstep
  constexpr int kstep = APART ? 1 : NW;
  int kbeg = APART ? wave * (KB / NW) : wave, nblocks = KB;
  if constexpr (SPLIT) {
    const int lo = (int)blockIdx.z * a.split_blocks;
    nblocks = min(KB - lo, a.split_blocks);
    kbeg += lo;
  }
  const int nmy = wave < nblocks ? (nblocks - wave + NW - 1) / NW : 0;
  // Block scales of this wave's K blocks (slot i: block wave + i * NW) and the
  // routed rows' sources go through LDS by DMA, ahead of the weights: a load
  // into a register would make the compiler wait for every copy in flight.
  if (a.gather) {
    const i32x4 rg = make_rsrc(a.gather + row0, (uint32_t)(row_end - row0) * 4u);
    tg_dma4(rg, lds0 + L::Gat, lane < row_end - row0 ? lane * 4 : kTgOob, 0);
  }
  if constexpr (BLOCK) {
    const int64_t at = expert * a.ws_pitch + (int64_t)(c0 / 128) * KB;
    const int kb = wave + lane * NW;
    tg_dma4(make_rsrc(a.ws + at, (uint32_t)KB * 4u), lds0 + L::Ws, kb < KB ? kb * 4 : kTgOob, 0);
    if constexpr (SW)
      tg_dma4(make_rsrc(a.ws_up + at, (uint32_t)KB * 4u), lds0 + L::Ws + 256, kb < KB ? kb * 4 : kTgOob, 0);
  }
  // INT8, FP8: the epilogue's scales, by wave 0, so that no load follows the
  // K loop (row slots from row0, column slots from c0)
  const float* epi_xs = (const float*)(smem + NW * L::Wave);
  const float* epi_ws = (const float*)(smem + NW * L::Wave + L::ShWs);
  if constexpr (!BLOCK) {
    if (wave == 0) {
      const uint32_t lds = lds_base + NW * L::Wave;
      if constexpr (!RAW)
        tg_dma4(make_rsrc(a.xs + row0, (uint32_t)(row_end - row0) * 4u), lds,
                lane < row_end - row0 ? lane * 4 : kTgOob, 0);
      // slot c: column c0 + c of the workgroup's 16 NT (SW: 8 NT), gate's then up's
      const bool live = lane < COLS && c0 + lane < a.N;
      const int off = !live ? kTgOob : a.ws_per_channel ? lane * 4 : 0;
      const int64_t at = a.ws_per_channel ? c0 : 0;
      const uint32_t bytes = a.ws_per_channel ? (uint32_t)min(COLS, a.N - c0) * 4u : 4u;
      tg_dma4(make_rsrc(a.ws + at, bytes), lds + L::ShWs, off, 0);
      if constexpr (SW) tg_dma4(make_rsrc(a.ws_up + at, bytes), lds + L::ShWs + 256, off, 0);
    }
  }
  // K tails (K % 128 != 0): the last block's chunks past K are not fetched
  // (zeros), in the weights as in the activations
  auto issue_w = [&](int i, int q, bool none) {
    const int kb = kbeg + i * kstep;
    const int32_t so = __builtin_amdgcn_readfirstlane(none ? 0 : kb * 128);
    const bool tail = !BLOCK && ktail != 128 && kb == KB - 1;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        tg_dma16nt(SW && h ? ru : rw, lds0 + q * L::Stage + nt * 2048 + h * 1024,
                   none || (tail && chunk[h] * 16 >= ktail) ? kTgOob : vw[nt][h], so);
  };
  // (Weights carry the non-temporal hint: FP8 M = 8 N = 4096 K = 14336 with
  // its quantizer 16.2 -> 14.5 us, I = 18944 K = 3584 30.2 -> 26.5.)
  // The first R - 1 stages leave without a branch (one past this wave's last
  // copies nothing), the weights before the routed rows are looked up.
#pragma unroll
  for (int i = 0; i < R - 1; ++i) issue_w(i, i, i >= nmy);

  const i32x4 rx = make_rsrc(a.x, a.x_bytes);
  const i32x4 rxs = make_rsrc(a.xs, BLOCK && !RAW ? (uint32_t)((uint64_t)a.x_rows * KB * 4) : 0u);
  if (a.gather) sg_wait_vm<(R - 1) * 2 * NT>();
  const int32_t* gat = (const int32_t*)(mine + L::Gat);
  int32_t vx[XI], vxs = kTgOob;
#pragma unroll
  for (int h = 0; h < XI; ++h) {
    // RAW: 4 rows of 256 bytes, LDS slot s of row r holds 16-byte chunk
    // 2 (s & 7) + ((s >> 3) ^ (r & 1)): the two reads of a quantizing lane
    // then cover all banks; else 8 rows of 128 bytes in the fragment swizzle
    // (RAW, one row: its 256 bytes in order)
    const int r = RAW ? 4 * h + (lane >> 4) : 8 * h + (lane >> 3);
    vx[h] = kTgOob;
    if (row0 + r < row_end) {
      const int src = a.gather ? gat[r] : row0 + r;
      if constexpr (RAW && !BLOCK) {
        vx[h] = (src * a.ldx + (lane & 15) * 8) * 2;
      } else if constexpr (RAW) {
        const int s = lane & 15, c = 2 * (s & 7) + ((s >> 3) ^ (r & 1));
        vx[h] = (src * a.ldx + c * 8) * 2;
      } else {
        vx[h] = src * K + chunk[h & 1] * 16;
      }
    }
  }
  if constexpr (BLOCK && !RAW) {
    if (lane < 16 * MT && row0 + lane < row_end) vxs = (a.gather ? gat[lane] : row0 + lane) * KB * 4;
  }
  auto issue_x = [&](int i, int q, bool none) {
    const int kb = none ? 0 : kbeg + i * kstep;
    const uint32_t b = lds0 + q * L::Stage + L::W;
    const int32_t so = __builtin_amdgcn_readfirstlane(kb * (RAW ? 256 : 128));
    const bool tail = !BLOCK && ktail != 128 && kb == KB - 1;
#pragma unroll
    for (int h = 0; h < XI; ++h)
      tg_dma16(rx, b + h * 1024, none || (!RAW && tail && chunk[h & 1] * 16 >= ktail) ? kTgOob : vx[h], so);
    if constexpr (BLOCK && !RAW)
      tg_dma4(rxs, b + L::X, none ? kTgOob : vxs, __builtin_amdgcn_readfirstlane(kb * 4));
  };
#pragma unroll
  for (int i = 0; i < R - 1; ++i) issue_x(i, i, i >= nmy);

  int o_lo = j * 128 + (tg_chunk<TF>(j, TF == kTgFp8 ? 2 * kg : kg) << 4);
  int o_hi = j * 128 + (tg_chunk<TF>(j, TF == kTgFp8 ? 2 * kg + 1 : 4 + kg) << 4);
  int xo_lo = o_lo, xo_hi = o_hi;
  if constexpr (RAW && L::Rows < 16) {  // the other fragment rows read zeros, with zero scales
    if (lane < 8) *(i32x4*)(mine + L::Zero + lane * 16) = i32x4{0, 0, 0, 0};
    if (lane >= L::Rows && lane < 16) *(float*)(mine + L::Sc + lane * 4) = 0.0f;
    if (j >= L::Rows) {
      xo_lo = L::Zero - L::Frag + (o_lo & 127);
      xo_hi = L::Zero - L::Frag + (o_hi & 127);
    }
  }
  float row_s = 1.0f, row_rs = 1.0f;  // RAW INT8, FP8: the row's scale
  if constexpr (RAW && !BLOCK) {
    constexpr float QMAX = FMT == kSgFp8 ? 448.0f : 127.0f;
    if (a.scale_mode == 0) {
      const uint16_t* x = (const uint16_t*)a.x + (int64_t)row0 * a.ldx;
      uint32_t mx = 0;
      for (int c = (int)threadIdx.x; c < K / 8; c += 64 * NW) mx = sg_max_u16(mx, sg_abs_max4(*(const u32x4*)(x + c * 8)));
      mx = wave_max_u32_dpp(max(mx & 0xffffu, mx >> 16));
      uint32_t* wmax = (uint32_t*)(smem + NW * L::Wave + L::ShMax);
      if (lane == 0) wmax[wave] = mx;
      __syncthreads();
      mx = wmax[0];
#pragma unroll
      for (int w2 = 1; w2 < NW; ++w2) mx = max(mx, wmax[w2]);
      row_s = __fdiv_rn(max_keep_nan(sg_widen<DT>(mx, 0), 1e-12f), QMAX);
    } else {
      row_s = a.scale_in[a.scale_mode == 1 ? 0 : row0];
    }
    row_rs = __fdiv_rn(1.0f, row_s);
  }
  // the reciprocal path's bytes equal IEEE division's for such scales
  const bool row_ok = row_s >= 0x1p-60f && row_s <= 3.4028235e38f;

  Acc acc[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[t][nt] = Acc{0, 0, 0, 0};

  for (int i = 0; i < nmy; ++i) {
    // stage i + R - 1 takes the slot read in iteration i - 1
    if (i + R - 1 < nmy) {
      issue_w(i + R - 1, (i + R - 1) % R, false);
      issue_x(i + R - 1, (i + R - 1) % R, false);
    }
    // the first R - 1 stages' weights were issued before all their activations
    const int issued = min(nmy, i + R);
    sg_wait_stages<OPS, R - 1>(i < R - 1 ? issued - (R - 1) : issued - 1 - i);
    const uint8_t* q = mine + (i % R) * L::Stage;
    const uint8_t* xf = q + L::W;
    if constexpr (RAW && !BLOCK) {
      uint8_t* frag = mine + L::Frag;
      const uint16_t q2 = sg_quant2<FMT, DT>(*(const uint32_t*)(xf + lane * 4), row_s, row_rs, row_ok);
      // zeros past K whatever the scale: 0 / 0 under a given scale of zero is NaN
      *(uint16_t*)(frag + lane * 2) = (kbeg + i * kstep) * 128 + lane * 2 < K ? q2 : (uint16_t)0;
      xf = frag;
    } else if constexpr (RAW) {
      uint8_t* frag = mine + L::Frag;
#pragma unroll
      for (int h = 0; h < XH; ++h) {
        const int r = 8 * h + (lane >> 3), sub = lane & 7;
        const uint8_t* src = xf + r * 256 + sub * 16;
        const u32x4 r0 = *(const u32x4*)(src + ((r & 1) << 7)), r1 = *(const u32x4*)(src + (((r & 1) ^ 1) << 7));
        *(u32x4*)(frag + r * 128 + (tg_chunk<TF>(r, sub) << 4)) =
            sg_quant16<DT>(r0, r1, sub == 0 ? (float*)(mine + L::Sc + r * 4) : nullptr);
      }
      xf = frag;
    }
    i32x4 wl[NT], wh[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      wl[nt] = *(const i32x4*)(q + nt * 2048 + o_lo);
      wh[nt] = *(const i32x4*)(q + nt * 2048 + o_hi);
    }
    float wsv = 0.0f;
    if constexpr (BLOCK) wsv = *(const float*)(mine + L::Ws + (SW && j >= 8 ? 256 : 0) + i * 4);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const i32x4 xl = *(const i32x4*)(xf + t * 2048 + xo_lo), xh = *(const i32x4*)(xf + t * 2048 + xo_hi);
      if constexpr (FMT == kSgI8) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[t][nt] = mfma_i8(xh, wh[nt], mfma_i8(xl, wl[nt], acc[t][nt]));
      } else {
        const i32x8 xv = i32x8{xl[0], xl[1], xl[2], xl[3], xh[0], xh[1], xh[2], xh[3]};
        float c[4];
        if constexpr (BLOCK) {
          const f32x4 sc = *(const f32x4*)((RAW ? mine + L::Sc : q + L::W + L::X + t * 64) + kg * 16);
#pragma unroll
          for (int r = 0; r < 4; ++r) c[r] = sc[r] * wsv;
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const i32x8 wv = i32x8{wl[nt][0], wl[nt][1], wl[nt][2], wl[nt][3], wh[nt][0], wh[nt][1], wh[nt][2], wh[nt][3]};
          if constexpr (BLOCK) {
            const f32x4 p = mfma_fp8(xv, wv, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][nt][r] = fmaf(p[r], c[r], acc[t][nt][r]);
          } else {
            acc[t][nt] = mfma_fp8(xv, wv, acc[t][nt]);
          }
        }
      }
    }
  }

  // the waves' sums, added in wave order (each parked in its own ring)
  uint32_t* red = (uint32_t*)mine;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((t * NT + nt) * 4 + r) * 64 + lane] = sg_bits(acc[t][nt], r);
  __syncthreads();
  for (int u = wave; u < MT * NT * 4; u += NW) {
    const uint32_t* p = (const uint32_t*)smem + u * 64 + lane;
    uint32_t part[NW];
#pragma unroll
    for (int w2 = 0; w2 < NW; ++w2) part[w2] = p[w2 * (L::Wave / 4)];
    const int blk = u >> 2, r = u & 3, t = blk / NT, nt = blk - t * NT;
    const int m = row0 + 16 * t + 4 * kg + r;
    const int n = SW ? c0 + 8 * nt + (j & 7) : c0 + 16 * nt + j;
    const bool live = n < a.N && m < row_end;
    float v;
    const bool up_lane = SW && j >= 8;
    uint32_t raw;
    if constexpr (FMT == kSgI8) {
      int sum = (int)part[0];
#pragma unroll
      for (int w2 = 1; w2 < NW; ++w2) sum += (int)part[w2];
      raw = (uint32_t)sum;
      v = (float)sum;
    } else {
      v = __uint_as_float(part[0]);
#pragma unroll
      for (int w2 = 1; w2 < NW; ++w2) v = __fadd_rn(v, __uint_as_float(part[w2]));
      raw = __float_as_uint(v);
    }
    if constexpr (SPLIT) {
      if (live) a.partials[((int64_t)blockIdx.z * a.M + m) * (SW ? 2 * a.N : a.N) + (up_lane ? a.N : 0) + n] = raw;
      continue;
    }
    if constexpr (FMT == kSgI8 && !SW) {
      if (a.acc_out && live) a.acc_out[(int64_t)m * a.N + n] = (int)raw;
    }
    if (live) {
      if constexpr (!BLOCK) {
        v = __fmul_rn(__fmul_rn(v, RAW ? row_s : epi_xs[m - row0]), epi_ws[(up_lane ? 64 : 0) + n - c0]);
      }
      if (a.bias_dtype != KQ_DTYPE_NONE)
        v = __fadd_rn(v, load_as_f32(up_lane ? a.bias_up : a.bias, a.bias_dtype, n));
    }
    if constexpr (SW) {
      const float up = __shfl_xor(v, 8, 64);
      if (j < 8 && live) ((uint16_t*)a.out)[(int64_t)m * a.N + n] = swiglu_bits(v, up, a.out_dtype);
    } else {
      if (live) ((uint16_t*)a.out)[(int64_t)m * a.N + n] = f32_to_out(v, a.out_dtype);
    }
  }
}

// ------------------------------------------------------------------ launch
// Form of a launch over `tiles` 16-row weight tiles: how many of them a
// workgroup takes (NT) and its waves (NW).  Up to half a tile per CU and one
// row, one tile and 16 waves: a wave has few K blocks then, and each waits for
// memory.  (FP8, us, 16 waves against 8: one row N = 1024 K = 4096 4.6 / 4.8, K =
// 8192 6.4 / 6.8, but N = 256 K = 2048 3.5 / 3.3, a K block a wave; with more
// rows the waves' sums cost what their loads gain: N = 512 M = 8 K = 4096 6.8 /
// 6.7, K = 16384 13.7 / 13.1.)  Block FP8 takes them from a K block a wave, up to
// 16 rows (8 where the launch quantizes).  Up to one tile per CU, one tile and 8
// waves, so that every CU streams; up to two, two tiles (one round of
// workgroups); beyond, two tiles and 4 waves, several workgroups per CU, so
// that one's prologue and epilogue run under another's stream.  Measured, FP8
// (us; graph replay, weights rotating past the MALL): N = K = 4096 M = 8 5.6,
// 16 6.1, 32 6.7, 64 8.9; N = 4096 K = 14336 10.7 / 12.2 / 15.6 / 22.1;
// N = 4608 K = 3584 5.6 with two tiles, 6.1 with one; SwiGLU I = 14336
// K = 4096 21.0 with two tiles and 4 waves, 20.2 with one, 26.3 with two and
// 8 waves at M = 8, and 26.8 / 36.8 / 30.0 at M = 32.  The form depends on the
// row tiles, `tiles` and K alone, and a SwiGLU pack has as many tiles as its
// packed linear, so both add the K blocks in one order.
struct SgForm {
  int nt, nw;  // weight tiles and waves of a workgroup
};
// mt: row tiles of 16; few: the launch has the form of 16 waves.
static inline SgForm sg_form(int64_t tiles, int mt, bool few) {
  const int64_t cus = tg_device_cus();
  if (few && 2 * tiles <= cus) return SgForm{1, 16};
  const int nw = mt <= 2 ? 8 : 4;
  return tiles <= cus ? SgForm{1, nw} : tiles <= 2 * cus ? SgForm{2, nw} : SgForm{2, nw / 2};
}
static inline int64_t sg_tiles(int64_t n, bool sw) { return sw ? (n + 7) / 8 : (n + 15) / 16; }
// Form of a launch on quantized rows (at most 64) of n columns (SwiGLU: I).
static inline SgForm sg_quantized_form(bool block, int64_t m, int64_t n, int K, bool sw) {
  return sg_form(sg_tiles(n, sw), (int)((m + 15) / 16), block ? m <= 16 && K >= 2048 : m == 1 && K > 2048);
}

// Whether the waves of a launch of at most 16 rows take K apart: with rows a
// multiple of 4 KB long the 16 rows of a tile lie on the same memory channels
// at one K, and NW waves at neighbouring K meet there; apart they do not.  INT8,
// us, weights out of cache, together / apart: M = 2 N = 4096 K = 4096 9.1 / 8.7,
// K = 8192 12.2 / 11.8, K = 16384 20.9 / 17.5, N = 8192 K = 16384 35.3 / 28.4, but
// N = 1024 K = 8192 9.9 / 10.0 and N = 4096 K = 12288 15.0 / 15.1; M = 24
// N = 4096 K = 16384 22.4 / 22.6.
static inline bool sg_apart(int64_t n, int K, bool sw) {
  return K % 4096 == 0 && sg_tiles(n, sw) >= tg_device_cus();
}

template <int FMT, bool RAW, int MT, int NT, int NW, int R, int XH, bool SW, int DT, bool SPLIT = false,
          bool APART = false>
static void sg_launch_form(const StreamArgs& a, int row_tiles, hipStream_t stream) {
  constexpr int cols = (SW ? 8 : 16) * NT;
  const dim3 grid((unsigned)((a.N + cols - 1) / cols), (unsigned)row_tiles, SPLIT ? (unsigned)a.splits : 1u);
  hipLaunchKernelGGL((stream_gemm_kernel<FMT, RAW, MT, NT, NW, R, XH, SW, DT, SPLIT, APART>), grid, dim3(64 * NW), 0, stream, a);
}

template <int FMT, bool RAW, int MT, int XH, bool SW, int DT>
static void sg_launch_rows(const StreamArgs& a, SgForm f, int row_tiles, hipStream_t stream) {
  if constexpr (MT == 1 && XH == 1) {
    if (f.nw == 16) {
      sg_launch_form<FMT, RAW, MT, 1, 16, 2, XH, SW, DT>(a, row_tiles, stream);
      return;
    }
  }
  if constexpr (FMT != kSgBlock && !RAW && MT >= 2) {
    if (a.splits > 1) {  // (narrow products: one tile a workgroup)
      if constexpr (MT == 2) sg_launch_form<FMT, RAW, MT, 1, 8, 2, XH, SW, DT, true>(a, row_tiles, stream);
      else sg_launch_form<FMT, RAW, MT, 1, 4, 3, XH, SW, DT, true>(a, row_tiles, stream);
      return;
    }
  }
  if constexpr (FMT != kSgBlock && MT == 1) {
    if (sg_apart(a.N, a.K, SW)) {
      if (f.nt == 1) sg_launch_form<FMT, RAW, MT, 1, 8, 2, XH, SW, DT, false, true>(a, row_tiles, stream);
      else if (f.nw == 8) sg_launch_form<FMT, RAW, MT, 2, 8, 2, XH, SW, DT, false, true>(a, row_tiles, stream);
      else sg_launch_form<FMT, RAW, MT, 2, 4, 2, XH, SW, DT, false, true>(a, row_tiles, stream);
      return;
    }
  }
  if constexpr (MT <= 2) {
    if (f.nt == 1) sg_launch_form<FMT, RAW, MT, 1, 8, 2, XH, SW, DT>(a, row_tiles, stream);
    else if (f.nw == 8) sg_launch_form<FMT, RAW, MT, 2, 8, 2, XH, SW, DT>(a, row_tiles, stream);
    else sg_launch_form<FMT, RAW, MT, 2, 4, 2, XH, SW, DT>(a, row_tiles, stream);
  } else {
    if (f.nt == 1) sg_launch_form<FMT, RAW, MT, 1, 4, 3, XH, SW, DT>(a, row_tiles, stream);
    else if (f.nw == 4) sg_launch_form<FMT, RAW, MT, 2, 4, 3, XH, SW, DT>(a, row_tiles, stream);
    else sg_launch_form<FMT, RAW, MT, 2, 2, 2, XH, SW, DT>(a, row_tiles, stream);
  }
}

// Quantized activations of a.M <= 64 rows.
template <int FMT, bool SW>
static void sg_launch(const StreamArgs& a, hipStream_t stream) {
  const SgForm form = sg_quantized_form(FMT == kSgBlock, a.M, a.N, a.K, SW);
  constexpr int DT = KQ_DTYPE_BF16;
  if (a.M <= 16) sg_launch_rows<FMT, false, 1, 1, SW, DT>(a, form, 1, stream);
  else if (a.M <= 32) sg_launch_rows<FMT, false, 2, 1, SW, DT>(a, form, 1, stream);
  else if (a.M <= 48) sg_launch_rows<FMT, false, 3, 1, SW, DT>(a, form, 1, stream);
  else sg_launch_rows<FMT, false, 4, 1, SW, DT>(a, form, 1, stream);
}

// Form of a launch that quantizes its rows: INT8 and FP8 one row, block FP8
// up to 16.
static inline SgForm sg_raw_form(bool block, int64_t m, int64_t n, int K, bool sw) {
  return sg_form(sg_tiles(n, sw), 1, block ? m <= 8 && K >= 2048 : K > 2048);
}

// fp16 / bf16 activations quantized in the launch.
template <int FMT, bool SW>
static void sg_launch_raw(const StreamArgs& a, int x_dtype, hipStream_t stream) {
  const SgForm form = sg_raw_form(FMT == kSgBlock, a.M, a.N, a.K, SW);
  if constexpr (FMT == kSgBlock) {
    if (a.M > 8) {
      if (x_dtype == KQ_DTYPE_BF16) sg_launch_rows<FMT, true, 1, 2, SW, KQ_DTYPE_BF16>(a, form, 1, stream);
      else sg_launch_rows<FMT, true, 1, 2, SW, KQ_DTYPE_F16>(a, form, 1, stream);
      return;
    }
  }
  if (x_dtype == KQ_DTYPE_BF16) sg_launch_rows<FMT, true, 1, 1, SW, KQ_DTYPE_BF16>(a, form, 1, stream);
  else sg_launch_rows<FMT, true, 1, 1, SW, KQ_DTYPE_F16>(a, form, 1, stream);
}

}  // namespace kq
