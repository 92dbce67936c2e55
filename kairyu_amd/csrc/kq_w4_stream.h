// Launch interface of the W4A16 streaming GEMM (kq_w4_stream.hip), called by
// the W4A16 entry points.
#pragma once
#include "kq_common.h"

namespace kq {

struct W4StreamArgs {
  const uint16_t* x;       // [M] rows of K fp16 / bf16 values in natural k order, 16-byte aligned
  int ldx;
  int x_bf16;
  const uint8_t* w;        // tiled words: 16-column tiles of 1 KB stages
  const uint32_t* table;   // scale/zero table behind them
  int zu;                  // the table holds scales alone
  uint32_t zoff;           // the zero of such a table
  const void* bias;
  int bias_dtype;
  uint16_t* out;           // [M][N], SwiGLU [M][N / 2]
  int out_dtype;
  int M, N, K, G;
  int pairs;               // group pairs of a tile in the table
  int swiglu;              // N interleaves gate and up by 16
  int ksplit;
  float* partials;         // [ksplit][M][N] when ksplit > 1
};

struct W4StreamForm {
  int nt, ksplit;          // column tiles of a workgroup, K splits
};
// How the rows reach the launch: fp16 read where they are, bf16 read where they
// are and converted in the loop, or gathered (as fp16) through a permutation.
enum W4Rows { kW4RowsInPlace, kW4RowsConverted, kW4RowsGathered };
// Whether the streaming GEMM is the faster one for these sizes (17 rows up),
// and its form, with at most max_splits K splits.
bool w4_stream_form(int M, int N, int K, W4Rows rows, int swiglu, int cus, int max_splits, W4StreamForm* f);
void launch_w4_stream(const W4StreamArgs& a, const W4StreamForm& f, hipStream_t stream);

}  // namespace kq
