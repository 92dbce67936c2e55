// Dense block-FP8 linear for gfx950: e4m3 weights with fp32 scales per 128x128
// block, activations quantized per token per 128-wide K block (the convention
// of finegrained_fp8_linear, deepseek_v4_moe_gpu.py:60-74).
//
//   * M <= 64: the weight-streaming kernel of kq_stream_gemm.h, HBM-bound; up
//     to 16 rows it quantizes the activations itself.
//   * M <= 256: the panel kernel of kq_panel_gemm.h.  A SwiGLU launch goes up to
//     128 rows: a layer's projections at 65 / 128 rows, two projections and
//     elementwise passes before -> now, 4096 / 12288 203.3 -> 194.9 us / 237.7 ->
//     227.3, 5120 / 6912 (a shard) 186.4 -> 168.6 / 224.1 -> 197.3; at 200 rows
//     4096 / 12288 lost 2% (276.4 -> 281.0), its two row tiles reading the
//     activations once per 64 columns and not once per 128.
//   * M > 256, or more columns than one round of panels holds
//     (pg_block_applies): the persistent tile engine of kq_tile_gemm.h.
#include "kq_common.h"
#include "kq_panel_gemm.h"
#include "kq_stream_gemm.h"
#include "kq_tile_gemm.h"

namespace kq {

static bool block_dtype_ok(int d) { return d == KQ_DTYPE_F16 || d == KQ_DTYPE_BF16; }

static int block_check_shape(const char* name, int64_t m, int64_t n, int64_t k) {
  if (m < 0 || n < 1 || k < kTgBK || (k % kTgBK) != 0 || k > kTgBK * kTgMaxKB || m > 0x7fffffffLL ||
      n > 0x7fffffffLL || n * k > 0x7fffffffLL || m * k > 0x7fffffffLL) {
    set_error("%s: bad shape m=%lld n=%lld k=%lld (k must be a multiple of 128)", name, (long long)m,
              (long long)n, (long long)k);
    return KQ_EINVAL;
  }
  return KQ_OK;
}

// Rows whose activations the streaming kernel quantizes itself.  Every
// workgroup then repeats the quantization of its M rows, about 1 us per 32 K
// blocks and 8 rows, against 4.6 us for the quantization launch (graph
// replay, K = 4096 M = 8: 6.4 us against 5.6 + 4.6; M = 16 8.9 against 5.8 +
// 4.6; K = 12288 M = 8 12.4 against 10.6 + 4.6, but M = 16 18.8 against
// 12.1 + 4.6).
static bool block_raw_applies(int64_t m, int64_t k) { return m <= 8 || (m <= 16 && k <= 8192); }

static bool block_raw_operands(const void* x, int64_t m, int64_t k, int64_t ldx) {
  return ((uintptr_t)x % 16) == 0 && (ldx % 8) == 0 && ((m - 1) * ldx + k) * 2 < ((int64_t)1 << 31);
}

static StreamArgs block_stream_args(const uint8_t* w, const float* ws, const void* bias, int bias_dtype, void* out,
                                    int out_dtype, int64_t m, int64_t n, int64_t k) {
  StreamArgs a{};
  a.w = w; a.ws = ws; a.bias = bias; a.bias_dtype = bias_dtype;
  a.out = out; a.out_dtype = out_dtype;
  a.M = (int)m; a.N = (int)n; a.K = (int)k;
  return a;
}

static void block_quantized(StreamArgs& a, const uint8_t* xq, const float* xs) {
  a.x = xq; a.x_bytes = (uint32_t)((int64_t)a.M * a.K); a.xs = xs; a.x_rows = a.M;
}

static void block_raw(StreamArgs& a, const void* x, int64_t ldx) {
  a.x = x; a.ldx = (int)ldx; a.x_bytes = (uint32_t)(((int64_t)(a.M - 1) * ldx + a.K) * 2);
}

// Quantized rows: the streaming kernel up to 64 rows, the panel kernel up to
// 256.  (Panels of 4 tiles from 33 rows up against many weight tiles, which
// INT8 and FP8 take, gain nothing here: a layer of 4096 / 12288 at 33 / 48 / 64
// rows 103.2 / 114.4 / 130.7 us streamed, 104.7 / 114.9 / 129.7 in panels.)
template <bool SW>
static void block_launch(const StreamArgs& a, hipStream_t st) {
  if (a.M > 64) pg_launch_block<SW>(a, st);
  else sg_launch<kSgBlock, SW>(a, st);
}

// e4m3 rows, then their block scales, in the workspace
static size_t block_xq_bytes(int64_t m, int64_t k) { return ((size_t)m * (size_t)k + 255) / 256 * 256; }
static size_t block_quant_bytes(int64_t m, int64_t k) {
  return block_xq_bytes(m, k) + ((size_t)m * (size_t)(k / 128) * 4 + 255) / 256 * 256;
}

static int block_quantize(const char* name, const void* x, int x_dtype, int64_t ldx, int64_t m, int64_t k,
                          void* workspace, size_t workspace_bytes, hipStream_t st) {
  if (workspace == nullptr || workspace_bytes < block_quant_bytes(m, k)) {
    set_error("%s: workspace of %zu bytes is smaller than the %zu bytes this call needs", name,
              workspace ? workspace_bytes : (size_t)0, block_quant_bytes(m, k));
    return KQ_EWORKSPACE;
  }
  return kq_act_quant_fp8_blocks(x, x_dtype, m, k, ldx, (uint8_t*)workspace,
                                 (float*)((uint8_t*)workspace + block_xq_bytes(m, k)), st);
}

}  // namespace kq

using namespace kq;

extern "C" int kq_block_fp8_gemm(const uint8_t* xq, const float* xs, const uint8_t* w,
                                 const float* ws, const void* bias, int bias_dtype, void* out,
                                 int out_dtype, int64_t m, int64_t n, int64_t k, void* stream) {
  if (!block_dtype_ok(out_dtype)) {
    set_error("kq_block_fp8_gemm: output dtype must be fp16 or bf16");
    return KQ_EUNSUPPORTED;
  }
  const int bad = block_check_shape("kq_block_fp8_gemm", m, n, k);
  if (bad != KQ_OK || m == 0) return bad;
  if (m <= 256 && pg_block_applies(m, n)) {
    StreamArgs a = block_stream_args(w, ws, bias, bias_dtype, out, out_dtype, m, n, k);
    block_quantized(a, xq, xs);
    block_launch<false>(a, (hipStream_t)stream);
    return check_launch("kq_block_fp8_gemm");
  }
  TileGemmArgs a{};
  a.x = xq; a.xs = xs; a.x_rows = (int)m; a.gather = nullptr;
  a.w = w; a.ws = ws; a.mtile_table = nullptr; a.mtile_count = nullptr;
  a.M = (int)m; a.N = (int)n; a.K = (int)k; a.I = 0;
  a.mtiles = (int)((m + kTgBM - 1) / kTgBM);
  a.ntiles = (int)((n + kTgBN - 1) / kTgBN);
  a.out = out; a.out_dtype = out_dtype; a.bias = bias; a.bias_dtype = bias_dtype;
  tg_launch<kTgFp8, true, kTgEpiStore>(a, (hipStream_t)stream);
  return check_launch("kq_block_fp8_gemm");
}

extern "C" int kq_block_fp8_route(int64_t m, int64_t n, int64_t k, int swiglu, int32_t* route) {
  if (m < 1 || (swiglu && m > 128) || !route || block_check_shape("kq_block_fp8_route", m, n, k) != KQ_OK) {
    if (m < 1 || (swiglu && m > 128) || !route) set_error("kq_block_fp8_route: bad shape m=%lld", (long long)m);
    return KQ_EINVAL;
  }
  route[3] = 1;
  if (m > 256 || !(swiglu || pg_block_applies(m, n))) {
    route[0] = KQ_ROUTE_TILE; route[1] = 16; route[2] = 8;
  } else if (m <= 64) {
    const SgForm f = block_raw_applies(m, k) ? sg_raw_form(true, m, n, (int)k, swiglu)
                                             : sg_quantized_form(true, m, n, (int)k, swiglu);
    route[0] = KQ_ROUTE_STREAM; route[1] = f.nt; route[2] = f.nw;
  } else {
    route[0] = KQ_ROUTE_PANEL; route[1] = pg_block_tiles(m, n, swiglu); route[2] = 4;
  }
  return KQ_OK;
}

extern "C" size_t kq_block_fp8_workspace_size(int64_t m, int64_t k) {
  return m > 0 && k > 0 ? block_quant_bytes(m, k) : 0;
}

extern "C" int kq_block_fp8_linear(const void* x, int x_dtype, int64_t ldx, const uint8_t* w, const float* ws,
                                   const void* bias, int bias_dtype, void* out, int64_t m, int64_t n, int64_t k,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  if (!block_dtype_ok(x_dtype)) {
    set_error("kq_block_fp8_linear: activation dtype must be fp16 or bf16");
    return KQ_EUNSUPPORTED;
  }
  const int bad = block_check_shape("kq_block_fp8_linear", m, n, k);
  if (bad != KQ_OK || m == 0) return bad;
  if (ldx < k) {
    set_error("kq_block_fp8_linear: row pitch %lld below k=%lld", (long long)ldx, (long long)k);
    return KQ_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  if (block_raw_applies(m, k) && block_raw_operands(x, m, k, ldx)) {
    StreamArgs a = block_stream_args(w, ws, bias, bias_dtype, out, x_dtype, m, n, k);
    block_raw(a, x, ldx);
    sg_launch_raw<kSgBlock, false>(a, x_dtype, st);
    return check_launch("kq_block_fp8_linear");
  }
  const int rc = block_quantize("kq_block_fp8_linear", x, x_dtype, ldx, m, k, workspace, workspace_bytes, st);
  if (rc != KQ_OK) return rc;
  return kq_block_fp8_gemm((const uint8_t*)workspace, (const float*)((uint8_t*)workspace + block_xq_bytes(m, k)), w,
                           ws, bias, bias_dtype, out, x_dtype, m, n, k, stream);
}

extern "C" int kq_block_fp8_swiglu_linear(const void* x, int x_dtype, int64_t ldx, const uint8_t* w_gate,
                                          const float* s_gate, const uint8_t* w_up, const float* s_up,
                                          const void* bias_gate, const void* bias_up, int bias_dtype, void* out,
                                          int64_t m, int64_t i_width, int64_t k, void* workspace,
                                          size_t workspace_bytes, void* stream) {
  if (!block_dtype_ok(x_dtype)) {
    set_error("kq_block_fp8_swiglu_linear: activation dtype must be fp16 or bf16");
    return KQ_EUNSUPPORTED;
  }
  const int bad = block_check_shape("kq_block_fp8_swiglu_linear", m, i_width, k);
  if (bad != KQ_OK || m == 0) return bad;
  if (m > 128 || ldx < k) {
    set_error("kq_block_fp8_swiglu_linear: at most 128 rows of pitch >= k (m=%lld ldx=%lld)", (long long)m,
              (long long)ldx);
    return KQ_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  StreamArgs a = block_stream_args(w_gate, s_gate, bias_gate, bias_dtype, out, x_dtype, m, i_width, k);
  a.w_up = w_up; a.ws_up = s_up; a.bias_up = bias_up;
  if (block_raw_applies(m, k) && block_raw_operands(x, m, k, ldx)) {
    block_raw(a, x, ldx);
    sg_launch_raw<kSgBlock, true>(a, x_dtype, st);
    return check_launch("kq_block_fp8_swiglu_linear");
  }
  const int rc = block_quantize("kq_block_fp8_swiglu_linear", x, x_dtype, ldx, m, k, workspace, workspace_bytes, st);
  if (rc != KQ_OK) return rc;
  block_quantized(a, (const uint8_t*)workspace, (const float*)((uint8_t*)workspace + block_xq_bytes(m, k)));
  block_launch<true>(a, st);
  return check_launch("kq_block_fp8_swiglu_linear");
}
