// W8A8 GEMMs for gfx950: INT8 (v_mfma_i32_16x16x64_i8) and FP8 e4m3
// (v_mfma_scale_f32_16x16x128_f8f6f4 with unit scales).
//
//   out[m, n] = epilogue( sum_k xq[m, k] * w[n, k] )
//   INT8: fp32(acc) * xscale[m] * wscale[n] (+ bias[n]), int32 accumulation
//         exact; each multiply/add rounded separately (no FMA contraction), the
//         CPU oracle's op order (kairyu/quant/int8.py:33-41, linear.py:547-553).
//   FP8 : acc (fp32) * xscale[m] * wscale[n or 0] (+ bias[n])
//         (kairyu/quant/fp8.py:48-56, linear.py:463-469).
//
// Kernels:
//   * M <= 64: the weight-streaming kernel of kq_stream_gemm.h, HBM-bound;
//     narrow products of 17 rows up split K over workgroups (stream_splits).
//   * M <= 256: the panel kernel of kq_panel_gemm.h (and 33 to 64 rows against
//     many weight rows), K split over workgroups where its panels leave half the
//     CUs idle (pg_form).
//   * other M > 64 with one 256x256 tile per CU, or half as many units with K
//     split: the persistent tile engine of kq_tile_gemm.h (LDS DMA double
//     buffering, XCD-grouped tiles).
//   * the rest: 128x128x128 workgroup tiles, 4 waves of 64x64, LDS
//     double buffer with an XOR chunk swizzle (twice the workgroups of the
//     256x256 engine for shapes that would leave CUs idle).
// The raw accumulators of every K split are added in split order by one reduce
// launch with the epilogue (kq_splitk.h).
#include "kq_common.h"
#include "kq_panel_gemm.h"
#include "kq_splitk.h"
#include "kq_stream_gemm.h"
#include "kq_tile_gemm.h"

#include <cstring>

namespace kq {

enum { kFmtI8 = 0, kFmtFp8 = 1 };

template <int FMT> struct W8Traits;
template <> struct W8Traits<kFmtI8> {
  static constexpr int kStep = 64;   // K per MFMA
  static constexpr int kLane = 16;   // bytes per lane per operand
  using Acc = i32x4;
  using Frag = i32x4;
};
template <> struct W8Traits<kFmtFp8> {
  static constexpr int kStep = 128;
  static constexpr int kLane = 32;
  using Acc = f32x4;
  using Frag = i32x8;
};

struct Epi {
  const float* xscale;
  const float* wscale;
  int ws_per_channel;
  const void* bias;
  int bias_dtype;
  void* out;
  int out_dtype;
  int32_t* acc_out;
  int M, N;
  // streaming and panel kernels: N = 2I packed gate / up weight rows [gate; up], the
  // output out[M][I] = silu(gate) * up (SwiGLU epilogue); 0: out[M][N]
  int swiglu;
};

template <int FMT>
KQ_DEV void epi_store(const Epi& ep, int m, int n, typename W8Traits<FMT>::Acc acc, int r) {
  if (m >= ep.M || n >= ep.N) return;
  float v;
  if constexpr (FMT == kFmtI8) {
    if (ep.acc_out) ep.acc_out[(int64_t)m * ep.N + n] = acc[r];
    v = (float)acc[r];
  } else {
    v = acc[r];
  }
  v = __fmul_rn(v, ep.xscale[m]);
  v = __fmul_rn(v, ep.ws_per_channel ? ep.wscale[n] : ep.wscale[0]);
  if (ep.bias_dtype != KQ_DTYPE_NONE) v = __fadd_rn(v, load_as_f32(ep.bias, ep.bias_dtype, n));
  ((uint16_t*)ep.out)[(int64_t)m * ep.N + n] = f32_to_out(v, ep.out_dtype);
}

template <int FMT>
KQ_DEV typename W8Traits<FMT>::Acc mfma_w8(typename W8Traits<FMT>::Frag a,
                                           typename W8Traits<FMT>::Frag b,
                                           typename W8Traits<FMT>::Acc c) {
  if constexpr (FMT == kFmtI8) return mfma_i8(a, b, c);
  else return mfma_fp8(a, b, c);
}

// ------------------------------------------------------------------- tiled
constexpr int kTile = 128;      // BM = BN = BK(bytes) = 128
constexpr int kTileBytes = kTile * kTile;

// byte offset of 16-byte chunk `c` (0..7) of row `r` in a swizzled tile
KQ_DEV int swz(int r, int c) { return r * kTile + ((c ^ (r & 7)) << 4); }

template <int FMT>
__global__ void __launch_bounds__(256)
w8a8_tile_kernel(const uint8_t* __restrict__ xq, const uint8_t* __restrict__ w, int K,
                 int tiles_n, Epi ep) {
  using T = W8Traits<FMT>;
  using Acc = typename T::Acc;
  using Frag = typename T::Frag;
  __shared__ __attribute__((aligned(16))) uint8_t smem[2][2][kTileBytes];

  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int j = lane & 15, kg = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;
  // grouped tile order: 8 row-tiles share each sweep over column tiles
  const int nblocks = gridDim.x;
  const int pid = xcd_swizzle(blockIdx.x, nblocks);
  const int tiles_m = (ep.M + kTile - 1) / kTile;
  const int group = 8 * tiles_n;
  const int gid = pid / group;
  const int first_m = gid * 8;
  const int gsize = min(tiles_m - first_m, 8);
  const int tm = first_m + (pid % group) % gsize;
  const int tn = (pid % group) / gsize;
  const int m0 = tm * kTile, n0 = tn * kTile;

  Acc acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = Acc{0, 0, 0, 0};

  i32x4 ra[4], rb[4];
  auto gload = [&](int k0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = tid + 256 * q;
      const int row = c >> 3, ch = c & 7;
      const int kc = k0 + ch * 16;
      const int m = m0 + row, n = n0 + row;
      ra[q] = (m < ep.M && kc < K) ? *(const i32x4*)(xq + (int64_t)m * K + kc) : i32x4{0, 0, 0, 0};
      rb[q] = (n < ep.N && kc < K) ? *(const i32x4*)(w + (int64_t)n * K + kc) : i32x4{0, 0, 0, 0};
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = tid + 256 * q;
      const int row = c >> 3, ch = c & 7;
      *(i32x4*)(&smem[buf][0][swz(row, ch)]) = ra[q];
      *(i32x4*)(&smem[buf][1][swz(row, ch)]) = rb[q];
    }
  };
  auto lfrag = [&](const uint8_t* s, int row, int ch0) -> Frag {
    if constexpr (FMT == kFmtI8) {
      return *(const i32x4*)(s + swz(row, ch0));
    } else {
      i32x4 lo = *(const i32x4*)(s + swz(row, ch0));
      i32x4 hi = *(const i32x4*)(s + swz(row, ch0 + 1));
      return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
  };

  const int nk = (K + kTile - 1) / kTile;
  gload(0);
  sstore(0);
  __syncthreads();
  for (int s = 0; s < nk; ++s) {
    const int cur = s & 1;
    if (s + 1 < nk) gload((s + 1) * kTile);
    const uint8_t* sa = smem[cur][0];
    const uint8_t* sb = smem[cur][1];
    constexpr int kSteps = kTile / T::kStep;
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) {
      const int ch0 = ks * (T::kStep / 16) + kg * (T::kLane / 16);
      Frag fa[4], fb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) fa[i] = lfrag(sa, wm * 64 + i * 16 + j, ch0);
#pragma unroll
      for (int i = 0; i < 4; ++i) fb[i] = lfrag(sb, wn * 64 + i * 16 + j, ch0);
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = mfma_w8<FMT>(fa[a], fb[b], acc[a][b]);
    }
    if (s + 1 < nk) sstore(cur ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        epi_store<FMT>(ep, m0 + wm * 64 + a * 16 + kg * 4 + r, n0 + wn * 64 + b * 16 + j,
                       acc[a][b], r);
}

// --------------------------------------------------------------- generic
// One thread per output; any K.  Used only when K is not a multiple of 16.
template <int FMT>
__global__ void w8a8_generic_kernel(const uint8_t* __restrict__ xq, const uint8_t* __restrict__ w,
                                    int K, Epi ep) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)ep.M * ep.N) return;
  const int m = (int)(idx / ep.N), n = (int)(idx % ep.N);
  typename W8Traits<FMT>::Acc acc = {0, 0, 0, 0};
  if constexpr (FMT == kFmtI8) {
    int s = 0;
    for (int k = 0; k < K; ++k)
      s += (int)(int8_t)xq[(int64_t)m * K + k] * (int)(int8_t)w[(int64_t)n * K + k];
    acc[0] = s;
  } else {
    float s = 0.0f;
    for (int k = 0; k < K; ++k)
      s = __fadd_rn(s, __fmul_rn(e4m3_to_f32(xq[(int64_t)m * K + k]),
                                 e4m3_to_f32(w[(int64_t)n * K + k])));
    acc[0] = s;
  }
  epi_store<FMT>(ep, m, n, acc, 0);
}

// ------------------------------------------------------------------ host
// Few rows (M <= 64, K % 16 == 0): the weight-streaming kernel.
static StreamArgs stream_args(const uint8_t* w, int K, const Epi& ep) {
  StreamArgs a{};
  const int I = ep.N / 2, up = ep.swiglu ? I : 0;  // first up row of a packed gate / up weight
  a.w = w; a.w_up = w + (int64_t)up * K;
  a.ws = ep.wscale; a.ws_up = ep.wscale + (ep.ws_per_channel ? up : 0);
  a.ws_per_channel = ep.ws_per_channel;
  a.M = ep.M; a.N = ep.swiglu ? I : ep.N; a.K = K;
  a.bias = ep.bias; a.bias_dtype = ep.bias_dtype;
  a.bias_up = ep.bias ? (const char*)ep.bias + (int64_t)up * (ep.bias_dtype == KQ_DTYPE_F32 ? 4 : 2) : nullptr;
  a.out = ep.out; a.out_dtype = ep.out_dtype; a.acc_out = ep.acc_out;
  return a;
}

// Adds the raw accumulators of `splits` K ranges in order, with the epilogue.
template <int FMT>
static void reduce_splits(const void* partials, int splits, const Epi& ep, hipStream_t stream) {
  ReduceArgs r{partials, splits, ep.M, ep.N, ep.xscale, ep.wscale, ep.ws_per_channel,
               ep.bias, ep.bias_dtype, ep.out, ep.out_dtype, ep.acc_out, ep.swiglu};
  launch_splitk_reduce(FMT == kFmtI8 ? kReduceI8 : kReduceFp8, r, stream);
}

// K splits of a streaming launch (17 to 64 rows) over workgroups.  Narrow
// products leave most CUs idle, and with long K the few that work walk it
// alone; a split costs the reduce launch, about 1.5 us.  INT8 with its
// quantizer, weights out of cache, us, whole / 4 / 8 splits: N = 512 M = 17
// K = 4096 9.0 / 9.8 / 10.8, K = 8192 12.0 / 11.0 / 11.7, K = 16384 17.1 / 13.0 /
// 13.1; M = 33 N = 1024 K = 4096 10.1 / 10.7; M = 64 N = 512 12.0 / 11.1 / 12.1,
// 17.1 / 13.0 / 13.4, 26.4 / 16.6 / 15.6; N = 1536 (whole / 2) M = 17 K = 8192
// 12.3 / 12.7, K = 12288 15.7 / 14.7.
static int stream_splits(int64_t m, int64_t n, int64_t k) {
  if (m <= 16) return 1;
  const int64_t room = tg_device_cus() / ((n + 15) / 16), kb = (k + 127) / 128;
  if (room >= 8 && kb >= (m > 32 ? 96 : 128)) return 8;
  if (room >= 4 && kb >= (m > 48 ? 32 : m > 32 ? 40 : 64)) return 4;
  return room >= 2 && kb >= 96 ? 2 : 1;
}

template <int FMT>
static void launch_stream(const uint8_t* xq, const uint8_t* w, int K, const Epi& ep, void* workspace,
                          size_t ws_bytes, hipStream_t stream) {
  constexpr int SF = FMT == kFmtI8 ? kSgI8 : kSgFp8;
  StreamArgs a = stream_args(w, K, ep);
  a.x = xq; a.x_bytes = (uint32_t)((int64_t)ep.M * K); a.xs = ep.xscale;
  if (pg_64_applies(ep.M, (ep.N + 15) / 16)) {
    const PanelArgs p{a, 1, nullptr};
    if (ep.swiglu) pg_launch_64<SF, true>(p, stream);
    else pg_launch_64<SF, false>(p, stream);
    return;
  }
  a.splits = stream_splits(ep.M, ep.N, K);
  if (!workspace || (size_t)a.splits * (size_t)ep.M * (size_t)ep.N * 4 > ws_bytes) a.splits = 1;
  a.split_blocks = ((K + 127) / 128 + a.splits - 1) / a.splits;  // (at least 4: none is empty)
  a.partials = (uint32_t*)workspace;
  if (ep.swiglu) sg_launch<SF, true>(a, stream);
  else sg_launch<SF, false>(a, stream);
  if (a.splits > 1) reduce_splits<FMT>(workspace, a.splits, ep, stream);
}

// 65 to 256 rows: the panel kernel's form, nt = 0 where the tile engine or
// the 128x128 kernel runs instead.
static PanelForm panel_form(int64_t m, int64_t n, int64_t k) {
  if (m <= 64 || m > 256 || k % 16 != 0 || k > 65536) return PanelForm{0, 0, 1};
  return pg_form(m, (n + 15) / 16, (int)((k + 127) / 128));
}

template <int FMT>
static void launch_panel(const uint8_t* xq, const uint8_t* w, int K, const Epi& ep, PanelForm f,
                         void* workspace, size_t ws_bytes, hipStream_t stream) {
  constexpr int SF = FMT == kFmtI8 ? kSgI8 : kSgFp8;
  if (!workspace || (size_t)f.splits * (size_t)ep.M * (size_t)ep.N * 4 > ws_bytes) f.splits = 1;
  PanelArgs p{stream_args(w, K, ep), f.splits, (uint32_t*)workspace};
  p.s.x = xq; p.s.x_bytes = (uint32_t)((int64_t)ep.M * K); p.s.xs = ep.xscale;
  if (ep.swiglu) pg_launch<SF, true>(p, f, stream);
  else pg_launch<SF, false>(p, f, stream);
  if (f.splits > 1) reduce_splits<FMT>(workspace, f.splits, ep, stream);
}

// One fp16 / bf16 row, quantized in the launch.
template <int FMT>
static void launch_stream_raw(const void* x, int x_dtype, int scale_mode, const float* scale_in,
                              const uint8_t* w, int K, const Epi& ep, hipStream_t stream) {
  constexpr int SF = FMT == kFmtI8 ? kSgI8 : kSgFp8;
  StreamArgs a = stream_args(w, K, ep);
  a.x = x; a.ldx = K; a.x_bytes = (uint32_t)K * 2u;
  a.scale_mode = scale_mode; a.scale_in = scale_in;
  if (ep.swiglu) sg_launch_raw<SF, true>(a, x_dtype, stream);
  else sg_launch_raw<SF, false>(a, x_dtype, stream);
}

// Work units per 256x256 tile for the tile engine at M > 64, 0 when it does
// not apply: 1 with at least one tile per CU; otherwise the K range is split
// (2..4 ways, >= 8 K blocks each) when that fills at least half the CUs, else
// up to 8 ways with >= 4 K blocks each, where the workspace holds the
// fp32/int32 partials.  Shapes it declines take the 128x128 kernel.
static int tile_engine_splits(int64_t m, int64_t n, int K, const void* workspace, size_t ws_bytes) {
  if (m * K >= ((int64_t)1 << 31) || n * K >= ((int64_t)1 << 31)) return 0;
  const int64_t tiles = ((m + kTgBM - 1) / kTgBM) * ((n + kTgBN - 1) / kTgBN);
  const int cus = tg_device_cus();
  if (tiles >= cus) return 1;
  const int kb = (K + kTgBK - 1) / kTgBK;
  for (int s = (int)std::min<int64_t>(4, cus / tiles); s >= 2; --s)
    if (kb / s >= 8 && tiles * s * 2 >= cus && workspace &&
        (size_t)s * (size_t)(m * n) * 4 <= ws_bytes)
      return s;
  // Too few tiles to fill half the CUs that way: split K up to 8 ways (at
  // least 4 K blocks per unit) rather than run the 128x128 kernel with a
  // workgroup per 128x128 tile.  N = K = 4096 (same process, outputs
  // bit-identical): FP8 M = 128 56.1 -> 26.4 us, M = 256 55.7 -> 28.9, INT8
  // M = 128 51.1 -> 27.2; N = 1024 M = 512 45.9 -> 28.9.  (Where the rule
  // above applies, 8 ways were slower: M = 512 34.8 -> 38.8 us.)
  for (int s = (int)std::min<int64_t>(8, cus / tiles); s >= 2; --s)
    if (kb / s >= 4 && workspace && (size_t)s * (size_t)(m * n) * 4 <= ws_bytes) return s;
  return 0;
}

template <int FMT>
static int run_w8a8(const char* what, const uint8_t* xq, const uint8_t* w, int64_t m,
                    int64_t n, int64_t k, const Epi& ep, void* workspace, size_t ws_bytes,
                    hipStream_t stream) {
  if (m < 0 || n < 1 || k < 1 || m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff ||
      m * k > 0x7fffffffffffLL) {
    set_error("%s: bad shape m=%lld n=%lld k=%lld", what, (long long)m, (long long)n,
              (long long)k);
    return KQ_EINVAL;
  }
  if (ep.out_dtype != KQ_DTYPE_F16 && ep.out_dtype != KQ_DTYPE_BF16) {
    set_error("%s: output dtype must be fp16 or bf16", what);
    return KQ_EUNSUPPORTED;
  }
  if (m == 0) return KQ_OK;
  const int K = (int)k;
  const PanelForm panel = panel_form(m, n, k);
  if (ep.swiglu && !((m <= 64 || panel.nt) && K % 16 == 0 && ((uintptr_t)xq % 16) == 0 && ((uintptr_t)w % 16) == 0 &&
                     n * k < ((int64_t)1 << 31) && m * k < ((int64_t)1 << 31))) {
    set_error("%s: the SwiGLU epilogue runs in the streaming and panel kernels only (m=%lld k=%lld)",
              what, (long long)m, (long long)k);
    return KQ_EINVAL;
  }
  if ((K % 16) != 0 || ((uintptr_t)xq % 16) || ((uintptr_t)w % 16)) {
    const int64_t total = m * n;
    hipLaunchKernelGGL(w8a8_generic_kernel<FMT>, dim3((unsigned)((total + 255) / 256)),
                       dim3(256), 0, stream, xq, w, K, ep);
    return check_launch(what);
  }
  if (m <= 64 && (n * k >= ((int64_t)1 << 32) || m * k >= ((int64_t)1 << 32))) {
    set_error("%s: weight or activation exceeds the 4 GiB addressing of the streaming kernel", what);
    return KQ_EINVAL;
  }
  if (m <= 64 && m * k < ((int64_t)1 << 31) && k < ((int64_t)1 << 26)) {
    launch_stream<FMT>(xq, w, K, ep, workspace, ws_bytes, stream);
  } else if (panel.nt) {
    launch_panel<FMT>(xq, w, K, ep, panel, workspace, ws_bytes, stream);
  }
  else if (const int splits = tile_engine_splits(m, n, K, workspace, ws_bytes)) {
    // persistent 256x256 MFMA tiles (kq_tile_gemm.h), scales in the epilogue;
    // with fewer tiles than CUs each tile's K range is split over `splits`
    // work units whose raw accumulators the split-K reduce sums in order
    TileGemmArgs a{};
    a.x = xq; a.x_rows = (int)m; a.xs = ep.xscale; a.gather = nullptr;
    a.w = w; a.ws = ep.wscale; a.ws_per_channel = ep.ws_per_channel;
    a.mtile_table = nullptr; a.mtile_count = nullptr;
    a.M = (int)m; a.N = (int)n; a.K = K; a.I = 0;
    a.mtiles = (int)((m + kTgBM - 1) / kTgBM);
    a.ntiles = (int)((n + kTgBN - 1) / kTgBN);
    a.out = ep.out; a.out_dtype = ep.out_dtype; a.bias = ep.bias; a.bias_dtype = ep.bias_dtype;
    a.acc_out = ep.acc_out;
    a.ksplit = splits;
    a.partials = splits > 1 ? (uint32_t*)workspace : nullptr;
    tg_launch<FMT == kFmtI8 ? kTgI8 : kTgFp8, false, kTgEpiStore>(a, stream);
    if (splits > 1) {
      reduce_splits<FMT>(workspace, splits, ep, stream);
    }
  } else {
    const int tiles_m = (int)((m + kTile - 1) / kTile);
    const int tiles_n = (int)((n + kTile - 1) / kTile);
    hipLaunchKernelGGL(w8a8_tile_kernel<FMT>, dim3(tiles_m * tiles_n), dim3(256), 0, stream, xq,
                       w, K, tiles_n, ep);
  }
  return check_launch(what);
}

}  // namespace kq

using namespace kq;

// Quantize + GEMM: one launch for one row, otherwise the
// per-token quantizer into the workspace (bytes, then fp32 row scales) and
// the GEMM dispatch of run_w8a8 on the rest of the workspace.
template <int FMT>
static int run_linear(const char* what, const void* x, int x_dtype, int64_t ldx, int scale_mode,
                      const float* scale_in, const uint8_t* w, int64_t m, int64_t n, int64_t k,
                      Epi ep, void* workspace, size_t ws_bytes, hipStream_t stream) {
  if (x_dtype != KQ_DTYPE_F16 && x_dtype != KQ_DTYPE_BF16) {
    set_error("%s: activation dtype must be fp16 or bf16 (code %d)", what, x_dtype);
    return KQ_EUNSUPPORTED;
  }
  if (m < 0 || n < 1 || k < 1 || ldx < k || m > 0x7fffffff || n > 0x7fffffff || k > 65536) {
    set_error("%s: bad shape m=%lld n=%lld k=%lld ldx=%lld", what, (long long)m, (long long)n,
              (long long)k, (long long)ldx);
    return KQ_EINVAL;
  }
  if (ep.out_dtype != KQ_DTYPE_F16 && ep.out_dtype != KQ_DTYPE_BF16) {
    set_error("%s: output dtype must be fp16 or bf16", what);
    return KQ_EUNSUPPORTED;
  }
  if (m == 0) return KQ_OK;
  if (m > 0 && x == nullptr) {
    set_error("%s: null activation", what);
    return KQ_EINVAL;
  }
  const int K = (int)k;
  // One row is quantized inside the GEMM launch (its bytes, and the order of
  // the sums, are those of the two launches); more rows take the quantizer
  // first: the row maxima that every workgroup would repeat cost what the
  // launch does (graph replay, N = 4096 K = 14336 and I = 18944 K = 3584: FP8
  // 14.2 against 16.2 us, INT8 15.9 against 17.1 at one row, even at two).
  if (m == 1 && K % 16 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0 &&
      n * k < ((int64_t)1 << 32)) {
    launch_stream_raw<FMT>(x, x_dtype, scale_mode, scale_in, w, K, ep, stream);
    return check_launch(what);
  }
  const size_t xq_bytes = ((size_t)m * (size_t)k + 255) / 256 * 256;
  const size_t xs_bytes = ((size_t)m * 4 + 255) / 256 * 256;
  if (workspace == nullptr || ws_bytes < xq_bytes + xs_bytes) {
    set_error("%s: workspace of %zu bytes is smaller than the %zu bytes this call needs", what,
              workspace ? ws_bytes : (size_t)0, xq_bytes + xs_bytes);
    return KQ_EWORKSPACE;
  }
  uint8_t* xq = (uint8_t*)workspace;
  float* xs = (float*)(xq + xq_bytes);
  const int rc = FMT == kFmtI8
                     ? kq_act_quant_i8(x, x_dtype, m, k, ldx, (int8_t*)xq, xs, stream)
                     : kq_act_quant_fp8(x, x_dtype, m, k, ldx, scale_in, scale_mode, xq, xs, stream);
  if (rc != KQ_OK) return rc;
  ep.xscale = xs;
  return run_w8a8<FMT>(what, xq, w, m, n, k, ep, xq + xq_bytes + xs_bytes,
                       ws_bytes - xq_bytes - xs_bytes, stream);
}

extern "C" size_t kq_w8a8_workspace_size(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0 || m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff) return 0;
  const size_t plane = (size_t)m * (size_t)n * 4;
  if (m <= 64) {
    const int s = k % 16 == 0 ? stream_splits(m, n, k) : 1;
    return s > 1 ? plane * (size_t)s : 0;
  }
  const PanelForm panel = panel_form(m, n, k);
  const int s = std::max(panel.nt ? panel.splits : 1, tile_engine_splits(m, n, (int)k, (const void*)1, (size_t)-1));
  return s > 1 ? plane * (size_t)s : 0;
}

extern "C" int kq_w8a8_route(int64_t m, int64_t n, int64_t k, int swiglu, int32_t* route) {
  if (m < 1 || n < 1 || k < 1 || m > 0x7fffffff || n > 0x7fffffff || k > 65536 || (swiglu && n % 2) || !route) {
    set_error("kq_w8a8_route: bad shape m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k);
    return KQ_EINVAL;
  }
  const int K = (int)k;
  const PanelForm panel = panel_form(m, n, k);
  int32_t r[4] = {KQ_ROUTE_GENERIC, 0, 0, 1};
  if (K % 16 != 0) {
  } else if (m <= 64 && pg_64_applies(m, (n + 15) / 16)) {
    r[0] = KQ_ROUTE_PANEL; r[1] = 4; r[2] = 4;
  } else if (m <= 64) {
    const SgForm f = sg_quantized_form(false, m, swiglu ? n / 2 : n, K, swiglu);
    r[0] = KQ_ROUTE_STREAM; r[1] = f.nt; r[2] = f.nw; r[3] = stream_splits(m, n, k);
  } else if (panel.nt) {
    r[0] = KQ_ROUTE_PANEL; r[1] = panel.nt; r[2] = panel.nt == 4 ? 4 : 8; r[3] = panel.splits;
  } else {
    const int s = tile_engine_splits(m, n, K, (const void*)1, (size_t)-1);
    r[0] = s ? KQ_ROUTE_TILE : KQ_ROUTE_SQUARE; r[1] = s ? 16 : 8; r[2] = s ? 8 : 4; r[3] = s ? s : 1;
  }
  memcpy(route, r, sizeof(r));
  return KQ_OK;
}

extern "C" int kq_w8a8_i8_gemm(const int8_t* xq, const float* xscale, const int8_t* w,
                               const float* wscale, const void* bias, int bias_dtype,
                               void* out, int out_dtype, int32_t* acc_out, int64_t m, int64_t n,
                               int64_t k, void* workspace, size_t workspace_bytes,
                               void* stream) {
  Epi ep{xscale, wscale, 1, bias, bias_dtype, out, out_dtype, acc_out, (int)m, (int)n};
  return run_w8a8<kFmtI8>("kq_w8a8_i8_gemm", (const uint8_t*)xq, (const uint8_t*)w, m, n, k, ep,
                          workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int kq_w8a8_fp8_gemm(const uint8_t* xq, const float* xscale, const uint8_t* w,
                                const float* wscale, int wscale_per_channel, const void* bias,
                                int bias_dtype, void* out, int out_dtype, int64_t m, int64_t n,
                                int64_t k, void* workspace, size_t workspace_bytes,
                                void* stream) {
  Epi ep{xscale, wscale, wscale_per_channel, bias, bias_dtype, out, out_dtype, nullptr,
         (int)m, (int)n};
  return run_w8a8<kFmtFp8>("kq_w8a8_fp8_gemm", xq, w, m, n, k, ep, workspace, workspace_bytes,
                           (hipStream_t)stream);
}

extern "C" size_t kq_w8a8_linear_workspace_size(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  return ((size_t)m * (size_t)k + 255) / 256 * 256 + ((size_t)m * 4 + 255) / 256 * 256 +
         kq_w8a8_workspace_size(m, n, k);
}

extern "C" int kq_w8a8_i8_linear(const void* x, int x_dtype, int64_t ldx, const int8_t* w,
                                 const float* wscale, const void* bias, int bias_dtype, void* out,
                                 int out_dtype, int32_t* acc_out, int64_t m, int64_t n, int64_t k,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  Epi ep{nullptr, wscale, 1, bias, bias_dtype, out, out_dtype, acc_out, (int)m, (int)n};
  return run_linear<kFmtI8>("kq_w8a8_i8_linear", x, x_dtype, ldx, 0, nullptr,
                            (const uint8_t*)w, m, n, k, ep, workspace, workspace_bytes,
                            (hipStream_t)stream);
}

extern "C" int kq_w8a8_fp8_linear(const void* x, int x_dtype, int64_t ldx, const float* scale_in,
                                  int scale_mode, const uint8_t* w, const float* wscale,
                                  int wscale_per_channel, const void* bias, int bias_dtype,
                                  void* out, int out_dtype, int64_t m, int64_t n, int64_t k,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  if (scale_mode < 0 || scale_mode > 2 || (scale_mode != 0 && scale_in == nullptr)) {
    set_error("kq_w8a8_fp8_linear: bad scale_mode %d", scale_mode);
    return KQ_EINVAL;
  }
  Epi ep{nullptr, wscale, wscale_per_channel, bias, bias_dtype, out, out_dtype, nullptr, (int)m,
         (int)n};
  return run_linear<kFmtFp8>("kq_w8a8_fp8_linear", x, x_dtype, ldx, scale_mode, scale_in, w, m, n,
                             k, ep, workspace, workspace_bytes, (hipStream_t)stream);
}

// ------------------------------------------------------------------ SwiGLU
// A packed (gate, up) projection with SwiGLU, out[m][c] = silu(g) * up for
// gate column c and up column I + c of the packed weight w [2I][K] (the
// reference MLP's act_fn(gate(x)) * up(x), kairyu/models/layers.py:243-244,
// over its packed projections, kairyu/models/packed_linear.py:58-149).
// Prefill shapes (M > 64, I % 128 == 0, enough 256 x 256 tiles for half the
// CUs) run the tile engine with the SwiGLU store epilogue: each tile pairs
// gate columns [n0, n0 + 128) with up columns [I + n0, I + n0 + 128), so the
// [M, 2I] projection output never reaches memory.  Shapes of M <= 64 run the
// weight-streaming kernel, up to 256 rows the panel kernel, with the SwiGLU
// epilogue (each 16-row weight tile is 8 gate rows and the matching 8 up rows),
// which a split K puts off to the reduce.  Other shapes run the packed
// linear into the workspace and the elementwise pass.  All produce the bits
// of the packed linear followed by kq_swiglu.
static bool swiglu_fused_applies(int64_t m, int64_t i_width, int64_t k, const void* x, int64_t ldx,
                                 const void* w) {
  if (m <= 64 || i_width % 128 != 0 || k % 16 != 0 || ((uintptr_t)w % 16) != 0) return false;
  if (m * k >= ((int64_t)1 << 31) || 2 * i_width * k >= ((int64_t)1 << 31)) return false;
  const int64_t tiles = ((m + kTgBM - 1) / kTgBM) * (i_width / 128);
  return 2 * tiles >= tg_device_cus();
}

template <int FMT>
static int run_swiglu_linear(const char* what, const void* x, int x_dtype, int64_t ldx, int scale_mode,
                             const float* scale_in, const uint8_t* w, const float* wscale,
                             int ws_per_channel, const void* bias, int bias_dtype, void* out,
                             int64_t m, int64_t i_width, int64_t k, void* workspace, size_t ws_bytes,
                             hipStream_t stream) {
  if (i_width < 1 || i_width > 0x3fffffff) {
    set_error("%s: bad width %lld", what, (long long)i_width);
    return KQ_EINVAL;
  }
  const int64_t n = 2 * i_width;
  Epi ep{nullptr, wscale, ws_per_channel, bias, bias_dtype, out, x_dtype, nullptr, (int)m, (int)n};
  const bool panel = panel_form(m, n, k).nt != 0;
  if (m > 0 && m <= 0x7fffffff && k >= 1 && k <= 65536 && ldx >= k && x != nullptr &&
      (x_dtype == KQ_DTYPE_F16 || x_dtype == KQ_DTYPE_BF16) && !panel &&
      swiglu_fused_applies(m, i_width, k, x, ldx, w)) {
    const size_t xq_bytes = ((size_t)m * (size_t)k + 255) / 256 * 256;
    const size_t xs_bytes = ((size_t)m * 4 + 255) / 256 * 256;
    if (workspace == nullptr || ws_bytes < xq_bytes + xs_bytes) {
      set_error("%s: workspace of %zu bytes is smaller than the %zu bytes this call needs", what,
                workspace ? ws_bytes : (size_t)0, xq_bytes + xs_bytes);
      return KQ_EWORKSPACE;
    }
    uint8_t* xq = (uint8_t*)workspace;
    float* xs = (float*)(xq + xq_bytes);
    const int rc = FMT == kFmtI8
                       ? kq_act_quant_i8(x, x_dtype, m, k, ldx, (int8_t*)xq, xs, stream)
                       : kq_act_quant_fp8(x, x_dtype, m, k, ldx, scale_in, scale_mode, xq, xs, stream);
    if (rc != KQ_OK) return rc;
    TileGemmArgs a{};
    a.x = xq; a.x_rows = (int)m; a.xs = xs; a.gather = nullptr;
    a.w = w; a.ws = wscale; a.ws_per_channel = ws_per_channel;
    a.mtile_table = nullptr; a.mtile_count = nullptr;
    a.M = (int)m; a.N = (int)n; a.K = (int)k; a.I = (int)i_width;
    a.mtiles = (int)((m + kTgBM - 1) / kTgBM);
    a.ntiles = (int)(i_width / 128);
    a.out = out; a.out_dtype = x_dtype; a.bias = bias; a.bias_dtype = bias_dtype;
    a.acc_out = nullptr;
    a.ksplit = 1;
    tg_launch<FMT == kFmtI8 ? kTgI8 : kTgFp8, false, kTgEpiSwiGluStore>(a, stream);
    return check_launch(what);
  }
  if (m >= 1 && (m <= 64 || panel) && k % 16 == 0 && k <= 65536 && ((uintptr_t)w % 16) == 0 &&
      ((uintptr_t)workspace % 16) == 0 && n * k < ((int64_t)1 << 31)) {
    // few rows: the streaming and panel kernels (one-row fused quantization
    // or the per-token quantizer first) with the SwiGLU epilogue
    ep.swiglu = 1;
    return run_linear<FMT>(what, x, x_dtype, ldx, scale_mode, scale_in, w, m, n, k, ep, workspace,
                           ws_bytes, stream);
  }
  // two passes: the packed projection [m][2I] in the activation dtype, then SwiGLU
  const size_t tmp_bytes = ((size_t)(m > 0 ? m : 0) * (size_t)n * 2 + 255) / 256 * 256;
  if (m > 0 && (workspace == nullptr || ws_bytes < tmp_bytes)) {
    set_error("%s: workspace of %zu bytes is smaller than the %zu bytes this call needs", what,
              workspace ? ws_bytes : (size_t)0, tmp_bytes);
    return KQ_EWORKSPACE;
  }
  ep.out = workspace;
  const int rc = run_linear<FMT>(what, x, x_dtype, ldx, scale_mode, scale_in, w, m, n, k, ep,
                                 (uint8_t*)workspace + tmp_bytes, ws_bytes - tmp_bytes, stream);
  if (rc != KQ_OK || m == 0) return rc;
  return kq_swiglu(workspace, n, 0, x_dtype, out, m, i_width, stream);
}

extern "C" size_t kq_w8a8_swiglu_workspace_size(int64_t m, int64_t i_width, int64_t k) {
  if (m <= 0 || i_width <= 0 || k <= 0) return 0;
  const size_t fused = ((size_t)m * (size_t)k + 255) / 256 * 256 + ((size_t)m * 4 + 255) / 256 * 256;
  const size_t tmp = ((size_t)m * (size_t)(2 * i_width) * 2 + 255) / 256 * 256;
  return std::max(fused, tmp + kq_w8a8_linear_workspace_size(m, 2 * i_width, k));
}

extern "C" int kq_w8a8_i8_swiglu_linear(const void* x, int x_dtype, int64_t ldx, const int8_t* w,
                                        const float* wscale, const void* bias, int bias_dtype, void* out,
                                        int64_t m, int64_t i_width, int64_t k, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  return run_swiglu_linear<kFmtI8>("kq_w8a8_i8_swiglu_linear", x, x_dtype, ldx, 0, nullptr,
                                   (const uint8_t*)w, wscale, 1, bias, bias_dtype, out, m, i_width, k,
                                   workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int kq_w8a8_fp8_swiglu_linear(const void* x, int x_dtype, int64_t ldx, const float* scale_in,
                                         int scale_mode, const uint8_t* w, const float* wscale,
                                         int wscale_per_channel, const void* bias, int bias_dtype,
                                         void* out, int64_t m, int64_t i_width, int64_t k,
                                         void* workspace, size_t workspace_bytes, void* stream) {
  if (scale_mode < 0 || scale_mode > 2 || (scale_mode != 0 && scale_in == nullptr)) {
    set_error("kq_w8a8_fp8_swiglu_linear: bad scale_mode %d", scale_mode);
    return KQ_EINVAL;
  }
  return run_swiglu_linear<kFmtFp8>("kq_w8a8_fp8_swiglu_linear", x, x_dtype, ldx, scale_mode, scale_in,
                                    w, wscale, wscale_per_channel, bias, bias_dtype, out, m, i_width, k,
                                    workspace, workspace_bytes, (hipStream_t)stream);
}
