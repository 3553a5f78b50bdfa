// Few-row int8 linears (gemm_q8_rows.hip): y = epilogue(x W^T) for up to ROWS_MAX rows, the activations given as int8
// rows, or as bf16 rows that the kernel quantizes (per row or per group of 256 columns) itself.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cohere_rows_gemm {

constexpr int ROWS_MAX = 96;

constexpr int UNIT = 256;    // K of one unit of a wave's work, and of a scale group
constexpr int MAX_UNITS = 24;  // a workgroup's tiles of all units within 64 KB of LDS

// where the int8 activations come from
enum XMode {
  X_Q8 = 0,     // int8 rows with one scale per row
  X_Q8G = 1,    // int8 rows with one scale per row and 256 columns
  X_BF = 2,     // bf16 rows, quantized here as quantize_rows does
  X_BFG = 3,    // bf16 rows, quantized here per 256 columns as the SILU_Q8 epilogue does
};

struct Args {
  const void* X;          // [M, K] int8 or bf16, row stride ldx elements
  const float* sx;        // X_Q8, X_Q8G: scales, row stride ldsx
  const int8_t* W;        // dense [N, K]; 2:4 kept values [N, K/2], or the stage-tiled records (tiled)
  const int32_t* E;       // 2:4 selectors [N, K/32] (row-major kept values only)
  const float* sw;        // [N]
  const uint16_t* bias;   // [N] bf16 or null
  uint16_t* Y;            // bf16 [M, N] ([M, N/2] for GLU), row stride ldy
  const uint16_t* R;      // residual, row stride ldr (may be Y)
  int64_t ldx, ldsx, ldy, ldr;
  int M, N, K;
  int tiled;
  float alpha;
};

// whether the kernel takes these sizes at all (alignments as the tile GEMM's)
bool fits(int64_t M, int64_t N, int64_t K);
// whether it is also the faster one for int8 rows
bool better_than_tiles(int64_t M, int64_t N, int64_t K, bool grouped);
// launches it; epi: the EPI_* ids BIAS, RESID, GLU (RESID only unless X_Q8). false when there is no such kernel
bool launch(XMode xm, bool sparse, int epi, const Args& p, hipStream_t s);

}  // namespace cohere_rows_gemm
