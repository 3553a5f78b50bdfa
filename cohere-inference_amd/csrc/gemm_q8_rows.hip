// Few-row W8A8 linears for gfx950 (dense and 2:4 sparse), the encoder's layers over one short utterance: with at most
// a few dozen rows the tile GEMM (gemm_q8.h) leaves most CUs idle -- its smallest tile gives the 1280-wide linears 20
// workgroups -- and each of them walks K one stage after another.
//
//  * A workgroup owns 16 rows and NS strips of 16 channels over the whole K, its waves each whole units of 256 K. A
//    wave loads its operands straight into registers (no LDS ring: every byte is used once by the workgroup), UB units
//    at a time with every load issued before the first matrix instruction: one or two memory round trips in all.
//  * The sums are int32 and meet in LDS, so the result has the tile GEMM's bits: per-row scales sum the waves' tiles
//    (exact in any order); grouped scales keep each unit's tile and fold them in group order with the same fma chain.
//  * The activations' quantization can ride along (X_BF, X_BFG): a lane holds 64 values of one row per unit, the
//    row's (or group's) maximum meets across the four lanes of the row and, per row, across the waves in LDS. Every
//    workgroup repeats it for its own 16 rows, which costs a fraction of the launch that it replaces. The feed-forward's
//    hidden rows then stay bf16 between its two linears, so that the first one needs no 256-column workgroups.
//  * Operand layouts as in gemm_q8.h: lane l holds row / channel l % 16; a dense instruction takes K 16 (l / 16) .. + 15
//    of its 64, a 2:4 one two such chunks of its 128 and 16 kept values with their selector word.
#include "common.h"
#include "gemm_q8.h"
#include "gemm_q8_rows.h"

namespace cohere_rows_gemm {

namespace {

using cohere_gemm::EPI_BIAS;
using cohere_gemm::EPI_GLU;
using cohere_gemm::EPI_RESID;
using cohere_gemm::TILED_REC;

constexpr int MAX_WAVES = 10;
// the modes that keep a row's values for its statistics hold one unit a wave, in up to 256 registers
constexpr int MAX_WAVES_ONE = 8;
constexpr bool one_unit(int xm) { return xm == X_BF; }

// a lane's activations of one unit: 4 chunks (64 K each) of 16 consecutive K
template <bool BF>
struct XRaw {
  uint4 v[BF ? 8 : 4];
};

// maximum over the four lanes of a row (l, l ^ 16, l ^ 32, l ^ 48) of non-negative values
DEVI float row4_max(float v) { return xor32_max_pos(xor16_max_pos(v)); }

DEVI float bf_at(const uint4* v, int k) {  // value k of consecutive bf16
  const uint32_t w = reinterpret_cast<const uint32_t*>(v)[k >> 1];
  return __uint_as_float(k & 1 ? w & 0xffff0000u : w << 16);
}

// NS strips of 16 channels; UB units loaded at once
template <int XM, bool SPARSE, int EPI, int NS, int UB>
__global__ void __launch_bounds__((one_unit(XM) ? MAX_WAVES_ONE : MAX_WAVES) * 64) rows_gemm_kernel(const Args p) {
  constexpr bool BF = XM == X_BF || XM == X_BFG;
  constexpr bool GROUPED = XM == X_Q8G || XM == X_BFG;
  constexpr int COLS = NS * 16, LDR = COLS + 4;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int nw = blockDim.x >> 6, units = p.K / UNIT;
  auto red = reinterpret_cast<int32_t(*)[16][LDR]>(smem);  // [waves, or units when grouped][16 rows][channels]
  float* scale = reinterpret_cast<float*>(smem + (GROUPED ? units : nw) * 16 * LDR * 4);  // [1 or units][16 rows]
  float* part = scale + 16 * (GROUPED ? units : 1);                                       // [waves][16 rows]
  const int lane = threadIdx.x & 63, wave = wave_id(), h = lane >> 4, c16 = lane & 15;
  const int n0 = blockIdx.x * COLS, m0 = blockIdx.y * 16;
  const int row = min(m0 + c16, p.M - 1);  // rows past M repeat the last one and are not written

  v4i acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = v4i{0, 0, 0, 0};

  XRaw<BF> xr[UB];
  v4i wr[UB][NS][SPARSE ? 2 : 4];
  int ix[UB][NS][SPARSE ? 2 : 1];
  auto load_x = [&](int b, int u) {
    const int64_t at = (int64_t)row * p.ldx + u * UNIT + 16 * h;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      if constexpr (BF) {
        const uint16_t* src = static_cast<const uint16_t*>(p.X) + at + 64 * d;
        xr[b].v[2 * d] = *reinterpret_cast<const uint4*>(src);
        xr[b].v[2 * d + 1] = *reinterpret_cast<const uint4*>(src + 8);
      } else {
        xr[b].v[d] = *reinterpret_cast<const uint4*>(static_cast<const int8_t*>(p.X) + at + 64 * d);
      }
    }
  };
  auto load_w = [&](int b, int u) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int64_t n = n0 + s * 16 + c16;
      if constexpr (!SPARSE) {
#pragma unroll
        for (int d = 0; d < 4; ++d)
          wr[b][s][d] = *reinterpret_cast<const v4i*>(p.W + n * p.K + u * UNIT + 64 * d + 16 * h);
      } else if (p.tiled) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const int8_t* rec = p.W + ((int64_t)(n0 / 16 + s) * (p.K / 128) + 2 * u + d) * TILED_REC;
          wr[b][s][d] = *reinterpret_cast<const v4i*>(rec + 16 * (4 * c16 + (h ^ ((c16 >> 1) & 3))));
          ix[b][s][d] = *reinterpret_cast<const int*>(rec + 1024 + 16 * c16 + 4 * (h ^ ((c16 & 8) >> 2)));
        }
      } else {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          wr[b][s][d] = *reinterpret_cast<const v4i*>(p.W + n * (p.K / 2) + u * (UNIT / 2) + 64 * d + 16 * h);
          ix[b][s][d] = p.E[n * (p.K / 32) + u * (UNIT / 32) + 4 * d + h];
        }
      }
    }
  };
  // a unit's products from its int8 chunks
  auto products = [&](int b, const v4i (&x)[4]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if constexpr (!SPARSE) {
#pragma unroll
        for (int d = 0; d < 4; ++d) acc[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wr[b][s][d], x[d], acc[s], 0, 0, 0);
      } else {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const v4i a = x[2 * d], c = x[2 * d + 1];
          acc[s] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(wr[b][s][d], v8i{a[0], a[1], a[2], a[3], c[0], c[1], c[2],
                                                                             c[3]}, acc[s], ix[b][s][d], 0, 0);
        }
      }
    }
  };
  auto store_acc = [&](int slot) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      *reinterpret_cast<v4i*>(&red[slot][c16][s * 16 + 4 * h]) = acc[s];
      acc[s] = v4i{0, 0, 0, 0};
    }
  };
  // 64 values of the row as int8 with the scale's reciprocal
  auto quantize = [&](auto value, float inv, v4i (&x)[4]) {
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = 16 * d + 4 * q;
        x[d][q] = (int)q8x4(value(k), value(k + 1), value(k + 2), value(k + 3), inv);
      }
  };
  auto row_max = [&](auto value) {
    float mx = 0.f;
#pragma unroll
    for (int k = 0; k < 64; ++k) mx = fmaxf(mx, fabsf(value(k)));
    return row4_max(mx);
  };
  // the row's maximum over the waves, in every lane of the row
  auto over_waves = [&](float v) {
    if (h == 0) part[wave * 16 + c16] = v;
    __syncthreads();
    float t = part[c16];
    for (int w = 1; w < nw; ++w) t = fmaxf(t, part[w * 16 + c16]);
    return t;
  };

  if constexpr (one_unit(XM)) {
    // one unit per wave (the launch sees to it): the row's values wait in registers for its statistics
    const int u = wave;
    load_x(0, u);
    load_w(0, u);
    __builtin_amdgcn_sched_barrier(0);  // every load is issued before the first is waited for
    auto value = [&](int k) { return bf_at(xr[0].v, k); };
    const float mx = over_waves(row_max(value));
    const float sc = mx > 0.f ? mx / 127.f : 1.f;
    v4i x[4];
    quantize(value, 1.f / sc, x);
    if (wave == 0 && h == 0) scale[c16] = sc;
    products(0, x);
    store_acc(wave);
  } else {
    for (int u0 = wave; u0 < units; u0 += nw * UB) {
#pragma unroll
      for (int b = 0; b < UB; ++b) load_x(b, min(u0 + b * nw, units - 1));
#pragma unroll
      for (int b = 0; b < UB; ++b) load_w(b, min(u0 + b * nw, units - 1));
      __builtin_amdgcn_sched_barrier(0);  // every load is issued before the first is waited for
#pragma unroll
      for (int b = 0; b < UB; ++b) {
        const int u = u0 + b * nw;
        if (u >= units) break;
        v4i x[4];
        if constexpr (XM == X_BFG) {
          auto value = [&](int k) { return bf_at(xr[b].v, k); };
          const float mx = row_max(value), sc = mx > 0.f ? mx / 127.f : 1.f;
          quantize(value, 1.f / sc, x);
          if (h == 0) scale[u * 16 + c16] = sc;
        } else {
#pragma unroll
          for (int d = 0; d < 4; ++d) x[d] = __builtin_bit_cast(v4i, xr[b].v[d]);
        }
        products(b, x);
        if constexpr (GROUPED) store_acc(u);
      }
    }
    if constexpr (!GROUPED) store_acc(wave);
  }
  __syncthreads();

  // a thread per output (GLU: per pair), consecutive threads along the channels
  auto result = [&](int r, int c) {
    float v;
    if constexpr (GROUPED) {
      v = 0.f;
      for (int u = 0; u < units; ++u) {
        const float s = XM == X_BFG ? scale[u * 16 + r] : p.sx[(int64_t)(m0 + r) * p.ldsx + u];
        v = __builtin_fmaf((float)red[u][r][c], s, v);
      }
    } else {
      int t = red[0][r][c];
      for (int w = 1; w < nw; ++w) t += red[w][r][c];
      v = (float)t * (BF ? scale[r] : p.sx[(int64_t)(m0 + r) * p.ldsx]);
    }
    return __builtin_fmaf(v, p.sw[n0 + c], p.bias ? bf2f(p.bias[n0 + c]) : -0.f);
  };
  const int rows = min(16, p.M - m0);
  constexpr int OUT = EPI == EPI_GLU ? COLS / 2 : COLS;
  for (int i = threadIdx.x; i < rows * OUT; i += blockDim.x) {
    const int r = i / OUT, c = i % OUT;
    uint16_t* y = p.Y + (int64_t)(m0 + r) * p.ldy + (EPI == EPI_GLU ? n0 / 2 : n0) + c;
    float v;
    if constexpr (EPI == EPI_GLU) {
      v = round_bf(result(r, 2 * c)) * sigmoid_fast(round_bf(result(r, 2 * c + 1)));
    } else {
      v = result(r, c);
      if constexpr (EPI == EPI_RESID) {
        v = __builtin_fmaf(p.alpha, round_bf(v), bf2f(p.R[(int64_t)(m0 + r) * p.ldr + n0 + c]));
      }
    }
    *y = f2bf(v);
  }
}

template <int XM, bool SPARSE, int EPI, int NS>
void launch_ns(const Args& p, hipStream_t s) {
  constexpr bool GROUPED = XM == X_Q8G || XM == X_BFG, BF = XM == X_BF || XM == X_BFG;
  const int units = p.K / UNIT;
  // waves: one unit each up to MAX_WAVES, else as many as share the units evenly; at least 4, units or not, so that a
  // thread has one output and the residual's old value is one memory round trip (with one wave four in a row: K 256,
  // 32 x 1280 with residual 4.3 us, the tiles 3.3)
  int nw = units < MAX_WAVES ? units : MAX_WAVES;
  while (units % nw) --nw;
  if (nw < 4 && !one_unit(XM)) nw = 4;
  constexpr int UB = BF ? 1 : 2;
  const size_t lds = ((GROUPED ? units : nw) * 16 * (NS * 16 + 4) + 16 * (GROUPED ? units : 1) + nw * 16) * 4;
  rows_gemm_kernel<XM, SPARSE, EPI, NS, UB>
      <<<dim3(p.N / (16 * NS), (p.M + 15) / 16), nw * 64, lds, s>>>(p);
}

template <int XM, bool SPARSE, int EPI>
bool launch_epi(const Args& p, hipStream_t s) {
  // one strip a workgroup while those give at most one workgroup per CU, two strips beyond: the activations are then
  // fetched (and quantized) half as often (K 5120 quantized here: 64 rows 16.5 -> 9.5 us, 26 rows 9.5 -> 9.9)
  if (p.N / 16 * ((p.M + 15) / 16) > 256 && p.N % 32 == 0) launch_ns<XM, SPARSE, EPI, 2>(p, s);
  else launch_ns<XM, SPARSE, EPI, 1>(p, s);
  return true;
}

}  // namespace

bool fits(int64_t M, int64_t N, int64_t K) {
  return M > 0 && N % 16 == 0 && K % UNIT == 0 && K / UNIT <= MAX_UNITS;
}

// Up to ROWS_MAX rows. Against the 64 x 64 tile, whose time is its K stages (about 3 us + 0.33 us per 128 K) at any few
// rows, this kernel's grows with its workgroups: N 1280, K 1280 5.1 us against 5.8 at 32 rows, 7.8 against 5.8 at 64;
// N 3840, K 1280 7.0 against 5.4 at 26 rows; K 5120 (grouped) 9.5 against 16.2 at 26 and at 64 rows. From K 3072 on it
// is the faster one at every size up to 512 workgroups (N 256 .. 5120, 1 to 96 rows: 0.37 to 1.01 of the tiles' time);
// K 2560 with scales per row beyond 256 workgroups, two strips each, 8.4 us against 7.4.
bool better_than_tiles(int64_t M, int64_t N, int64_t K, bool grouped) {
  const int64_t most = K < 2560 ? 192 : K < 3072 && !grouped ? 256 : 512;
  return M <= ROWS_MAX && fits(M, N, K) && N / 16 * ((M + 15) / 16) <= most;
}

bool launch(XMode xm, bool sparse, int epi, const Args& p, hipStream_t s) {
#define XM_EPI(XM, E) if (xm == XM && epi == E) return sparse ? launch_epi<XM, true, E>(p, s) : launch_epi<XM, false, E>(p, s)
  if (!fits(p.M, p.N, p.K) || (one_unit(xm) && p.K / UNIT > MAX_WAVES_ONE)) return false;
  XM_EPI(X_Q8, EPI_BIAS);
  XM_EPI(X_Q8, EPI_RESID);
  XM_EPI(X_Q8, EPI_GLU);
  XM_EPI(X_Q8G, EPI_RESID);
  XM_EPI(X_BF, EPI_RESID);
  XM_EPI(X_BFG, EPI_RESID);
#undef XM_EPI
  return false;
}

}  // namespace cohere_rows_gemm
