// The encoder's front end on gfx950: normalized log-mel features of packed audio pieces and the subsampling stem's
// convolutions (the stem's pointwise convolutions and final projection are bf16 GEMMs, gemm_bf16.hip).
//
// Reference: kernels/features.py + kernels/csrc/features.cu (log-mel), kernels/csrc/encoder_ops.cu:339-448 and
// kernels/fast_encoder.py:185-202 (subsampling), whose semantics follow transformers' CohereAsrFeatureExtractor and
// ParakeetEncoderSubsamplingConv2D.
//
// logmel_kernel: one wavefront per frame, four frames per workgroup, everything between the samples and the log-mel
// values in registers and LDS -- no frame buffer and no spectrum in HBM. The 512-sample real frame is transformed as a
// 256-point complex FFT of (even, odd) sample pairs: four radix-4 Stockham passes (one butterfly per lane per pass,
// natural order out, no bit reversal) through a per-wave LDS ping-pong buffer, twiddles from a 512-entry table
// computed once per workgroup in double precision; then the usual split into the 257 bins of the real transform,
// |X|^2, the mel bands over their nonzero bins, and log.
#include "cohere_hip.h"
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int NFFT = 512, HOP = 160, BINS = NFFT / 2 + 1, MELS = 128, NZ = NFFT / 2;
constexpr int FPW = 4;  // frames (waves) per workgroup

struct Cx {
  float re, im;
};
DEVI Cx cadd(Cx a, Cx b) { return {a.re + b.re, a.im + b.im}; }
DEVI Cx csub(Cx a, Cx b) { return {a.re - b.re, a.im - b.im}; }
DEVI Cx cmul(Cx a, Cx b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
DEVI Cx mul_mi(Cx a) { return {a.im, -a.re}; }  // a * (-i)

// this wave's LDS accesses so far are done, and none after is moved before
DEVI void wave_lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// the piece holding flat frame f: the last p with frame_start[p] <= f
DEVI int piece_of(const int64_t* frame_start, int pieces, int64_t f) {
  int lo = 0, hi = pieces - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (frame_start[mid] <= f) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Bound by no one unit: over 12,800 frames (27.8 us; 29 with one frame per wave, tables per frame and a branch around each
// sample load) the counters give 600 vector instructions a frame, a wave's tables among them, 4 cycles each: 12.5 us of
// issue over the 1024 SIMDs, 45 %; the 15 MB take 3 us. The rest is latency: a wave's passes one after another through
// LDS, and its first samples and tables.
// A wave takes `per_wave` consecutive frames, so that the twiddle table (computed in double) and the mel weights in LDS
// are made once for FPW * per_wave frames; the samples of its next frame are loaded while one is transformed. Its
// FFT buffers are its own: between the passes it waits for its own LDS accesses only.
constexpr int MTAPS = 16;  // a band's first weights, held in LDS (the extractor's bands have at most 13)
__global__ void __launch_bounds__(FPW * 64) logmel_kernel(const float* __restrict__ x, const int64_t* __restrict__ meta,
                                                          int pieces, int64_t total_frames, int per_wave,
                                                          const float* __restrict__ window,
                                                          const float* __restrict__ mel, const int* __restrict__ band,
                                                          float preemph, float* __restrict__ logmel) {
  __shared__ Cx tw[NFFT];            // e^{-2 pi i k / 512}
  __shared__ Cx buf[FPW][2][NZ];     // Stockham ping-pong, per wave
  __shared__ float power[FPW][BINS + 3];
  __shared__ float mw[MTAPS][MELS];
  const int lane = threadIdx.x & 63, w = wave_id();
  const int64_t* sample_start = meta;
  const int64_t* lens = meta + pieces;
  const int64_t* frame_start = meta + 2 * pieces;
  const int64_t first = ((int64_t)blockIdx.x * FPW + w) * per_wave, end = min(first + per_wave, total_frames);

  // lane j holds z[j + 64 r] = frame[2 (j + 64 r)] + i frame[2 (j + 64 r) + 1], r = 0..3; frame[j] is sample
  // 160 t - 256 + j of the piece, pre-emphasised (x[s] - p x[s-1], the product rounded first), zero outside it, times
  // the centred window
  int p = first < end ? piece_of(frame_start, pieces, first) : 0;
  // samples j - 1, j, j + 1 of the lane's four pairs; the frame's samples [jlo, jhi) are the piece's, the others load
  // one of these (a guarded load would be a branch, and each branch a memory round trip of its own)
  float raw[4][3];
  int nlo = 0, nhi = 0, n0 = -1;
  auto load = [&](int64_t f) {
    while (p + 1 < pieces && frame_start[p + 1] <= f) ++p;  // pieces without frames are passed over
    const int64_t s0 = (f - frame_start[p]) * HOP - NFFT / 2, n = lens[p];  // the frame's first sample
    nlo = (int)min(max(-s0, (int64_t)0), (int64_t)NFFT);
    nhi = (int)min(max(n - s0, (int64_t)0), (int64_t)NFFT);
    n0 = s0 <= 0 ? nlo : -1;  // sample 0's place in the frame
    const bool has = n > 0 && nhi > 0 && nlo < NFFT;
    const int from = s0 > 0 ? -1 : nlo, to = nhi - 1;  // readable: [from, to]
    const float* xp = x + sample_start[p] + s0;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int j = 2 * (lane + 64 * r) - 1 + k;
        raw[r][k] = has ? xp[min(max(j, from), to)] : 0.f;
      }
  };
  if (first < end) load(first);
  float win[4][2];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int k = 0; k < 2; ++k) win[r][k] = window[2 * (lane + 64 * r) + k];
  int k0[2], k1[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    k0[h] = band[2 * (lane + 64 * h)];
    k1[h] = band[2 * (lane + 64 * h) + 1];
  }
  for (int i = threadIdx.x; i < MTAPS * MELS; i += FPW * 64) {
    const int m = i % MELS, k = band[2 * m] + i / MELS;
    mw[i / MELS][m] = k < band[2 * m + 1] ? mel[(int64_t)m * BINS + k] : 0.f;
  }
  for (int k = threadIdx.x; k < NFFT; k += FPW * 64) {
    double s, c;
    sincospi(-(double)k / 256.0, &s, &c);
    tw[k] = {(float)c, (float)s};
  }
  __syncthreads();  // twiddle table and mel weights

  // the lane's twiddles of the passes and of the split: the same for every frame
  Cx wp[3][3], ws[4];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int Ns = 4 << (2 * i);
#pragma unroll
    for (int r = 1; r < 4; ++r) wp[i][r - 1] = tw[(r * (lane % Ns) * (128 / Ns)) & (NFFT - 1)];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) ws[q] = tw[lane + 64 * q];

  for (int64_t f = first; f < end; ++f) {
    const int jlo = nlo, jhi = nhi, j0 = n0;
    Cx v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float e[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int j = 2 * (lane + 64 * r) + k;
        float y = __fsub_rn(raw[r][k + 1], __fmul_rn(preemph, raw[r][k]));
        if (j == j0) y = raw[r][k + 1];  // sample 0 has no predecessor
        e[k] = __fmul_rn(j >= jlo && j < jhi ? y : 0.f, win[r][k]);
      }
      v[r] = {e[0], e[1]};
    }
    if (f + 1 < end) load(f + 1);

    // radix-4 Stockham passes, Ns = 1, 4, 16, 64: lane j combines in[j + 64 r] (twiddled by W_{4 Ns}^{r (j % Ns)}) and
    // writes out[(j / Ns) 4 Ns + j % Ns + r Ns]
    int cur = 0;
#pragma unroll
    for (int Ns = 1; Ns < NZ; Ns *= 4) {
      const int jm = lane % Ns;
      if (Ns > 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = buf[w][cur][lane + 64 * r];
#pragma unroll
        for (int r = 1; r < 4; ++r) v[r] = cmul(v[r], wp[Ns == 4 ? 0 : (Ns == 16 ? 1 : 2)][r - 1]);
        cur ^= 1;
      }
      const Cx a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]), a2 = cadd(v[1], v[3]), a3 = mul_mi(csub(v[1], v[3]));
      const int o = (lane / Ns) * 4 * Ns + jm;
      buf[w][cur][o] = cadd(a0, a2);
      buf[w][cur][o + Ns] = cadd(a1, a3);
      buf[w][cur][o + 2 * Ns] = csub(a0, a2);
      buf[w][cur][o + 3 * Ns] = csub(a1, a3);
      wave_lds_sync();
    }
    // Z = buf[w][cur] in natural order. Bins of the real transform: X[k] = E[k] + W_512^k O[k] with
    // E = (Z[k] + conj Z[256-k]) / 2, O = (Z[k] - conj Z[256-k]) / 2i; X[256] = E[0] - O[0]. Power as the extractor:
    // |X| then squared.
    const Cx* Z = buf[w][cur];
    float* pw = power[w];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = lane + 64 * q;
      const Cx zk = Z[k], zc0 = Z[(NZ - k) & (NZ - 1)];
      const Cx zc = {zc0.re, -zc0.im};
      const Cx e = {0.5f * (zk.re + zc.re), 0.5f * (zk.im + zc.im)};
      const Cx d = csub(zk, zc);
      const Cx o = {0.5f * d.im, -0.5f * d.re};  // d / 2i
      const Cx X = cadd(e, cmul(ws[q], o));
      const float a = __fsqrt_rn(__fadd_rn(__fmul_rn(X.re, X.re), __fmul_rn(X.im, X.im)));
      pw[k] = __fmul_rn(a, a);
      if (k == 0) {
        const float x256 = e.re - o.re;  // E[0] and O[0] are real
        const float a2 = __fsqrt_rn(__fmul_rn(x256, x256));
        pw[NZ] = __fmul_rn(a2, a2);
      }
    }
    wave_lds_sync();
    // mel bands m = lane and lane + 64 (a narrow low band with a wide high one), fp32 over the band's nonzero bins in
    // order; log(mel + 2^-24)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int m = lane + 64 * h, near = min(k1[h], k0[h] + MTAPS);
      float acc = 0.f;
      for (int k = k0[h]; k < near; ++k) acc = __builtin_fmaf(mw[k - k0[h]][m], pw[k], acc);
      for (int k = near; k < k1[h]; ++k) acc = __builtin_fmaf(mel[(int64_t)m * BINS + k], pw[k], acc);
      logmel[f * MELS + m] = logf(__fadd_rn(acc, 5.9604644775390625e-8f));
    }
    wave_lds_sync();  // the powers are read before the next frame's
  }
}

// per piece and mel band: mean and unbiased variance over the piece's valid frames (fp64 sums in a fixed order), then
// (v - mean) / (std + 1e-5) as bf16 into out (pieces, T, 128) at the piece's first frames.
// Bound by memory latency: the bytes are few (6.6 MB read, 3.3 MB written for eight pieces of 2 to 30 s) and a piece's
// two sums come one after the other. A workgroup takes 8 bands of a piece: thread (f, q) holds bands 4 q .. 4 q + 3 of
// frames f, f + 512, ... in registers, so the values are read once for both sums and the output, 512 frames in flight
// (only past NKEEP * 512 frames, 30.7 s, are they read again). 16 bands of 16 frames in flight, read three times over,
// took 101 us there, this 15 us. The 16 workgroups of a piece run on one XCD (contiguous items of the remapped
// index), whose L2 then merges their 16-byte parts of each output row.
// four floats, two or four bf16 values, read or written whole at their own alignment
typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32_any __attribute__((aligned(2)));
typedef uint32_t b4_any __attribute__((ext_vector_type(2), aligned(2)));
constexpr int NB = 8, NQ = NB / 4, NTHR = 1024, NFR = NTHR / NQ, NKEEP = 6;
// one piece's 8 bands by one workgroup, KEEP frames a thread held in registers. Pieces of at most NFR frames (5.1 s) take
// KEEP = 1 and only the waves that have frames sum (the others' sums are zeros): sixteen waves' shuffles and LDS reads,
// and the code of six held frames, cost 9.4 us whatever the size (0.5 s 4.0 us now, 2 s 5.7).
template <int KEEP>
DEVI void normalize_bands(const float* __restrict__ v, int64_t nv, uint16_t* __restrict__ o,
                          double (&part)[NTHR / 64][NB]) {
  constexpr int NW = NTHR / 64;
  const int tid = threadIdx.x, q = tid % NQ, f = tid / NQ, wave = wave_id();
  const int nw = KEEP == 1 ? (int)((nv + NFR / NW - 1) / (NFR / NW)) : NW;  // waves with frames
  v4f keep[KEEP];
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int64_t t = f + (int64_t)i * NFR;
    keep[i] = t < nv ? (v4f) * reinterpret_cast<const f4_any*>(v + t * MELS) : v4f{0.f, 0.f, 0.f, 0.f};
  }
  // the workgroup's sum of each band, in every thread of that band: over the wave's lanes of equal q, then its waves
  auto total_of = [&](double (&s)[4]) {
    if (wave < nw) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int d = NQ; d < 64; d <<= 1) s[k] += __shfl_xor(s[k], d, 64);
      }
    }
    __syncthreads();  // the last sums are read
    if (wave < nw && (tid & 63) < NQ)
#pragma unroll
      for (int k = 0; k < 4; ++k) part[wave][4 * q + k] = s[k];
    __syncthreads();
    if (wave < nw) {
      double t[4] = {0.0, 0.0, 0.0, 0.0};
      auto add = [&](int w) {
#pragma unroll
        for (int k = 0; k < 4; ++k) t[k] += part[w][4 * q + k];
      };
      if constexpr (KEEP == 1) {
        for (int w = 0; w < nw; ++w) add(w);
      } else {
#pragma unroll
        for (int w = 0; w < NW; ++w) add(w);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) s[k] = t[k];
    }
  };
  auto each = [&](auto fn) {  // this thread's frames, the kept ones first
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
      const int64_t t = f + (int64_t)i * NFR;
      if (t < nv) fn(t, keep[i]);
    }
    if constexpr (KEEP > 1)  // (KEEP = 1: the piece has no more)
      for (int64_t t = f + (int64_t)KEEP * NFR; t < nv; t += NFR)
        fn(t, (v4f) * reinterpret_cast<const f4_any*>(v + t * MELS));
  };
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  each([&](int64_t, const v4f& x) {
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] += x[k];
  });
  total_of(s);
  float mean[4], den[4];
  double m2[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 4; ++k) mean[k] = (float)(s[k] / (double)nv);
  each([&](int64_t, const v4f& x) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double d = (double)x[k] - (double)mean[k];
      m2[k] += d * d;
    }
  });
  total_of(m2);
#pragma unroll
  for (int k = 0; k < 4; ++k) den[k] = __fadd_rn((float)sqrt(m2[k] / (double)(nv - 1)), 1e-5f);
  each([&](int64_t t, const v4f& x) {
    float y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = __fdiv_rn(__fsub_rn(x[k], mean[k]), den[k]);
    *reinterpret_cast<b4_any*>(o + t * MELS) = b4_any{pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3])};
  });
}

__global__ void __launch_bounds__(NTHR) normalize_kernel(const float* __restrict__ logmel,
                                                         const int64_t* __restrict__ frame_start, int64_t T,
                                                         uint16_t* __restrict__ out) {
  __shared__ double part[NTHR / 64][NB];
  const int total = (int)gridDim.x, xcd = (int)blockIdx.x % 8;  // workgroup b runs on XCD b % 8
  const int item = xcd * (total / 8) + min(xcd, total % 8) + (int)blockIdx.x / 8;
  const int p = item / (MELS / NB), b0 = item % (MELS / NB) * NB;
  const int q = threadIdx.x % NQ;
  const int64_t f0 = frame_start[p], nv = frame_start[p + 1] - f0;
  if (nv == 0) return;
  const float* v = logmel + f0 * MELS + b0 + 4 * q;
  uint16_t* o = out + (int64_t)p * T * MELS + b0 + 4 * q;
  if (nv <= NFR) normalize_bands<1>(v, nv, o, part);
  else normalize_bands<NKEEP>(v, nv, o, part);
}

// ---- subsampling convolutions ------------------------------------------------------------------------------------
// ParakeetEncoderSubsamplingConv2D on one sequence at a time (its masking of padded frames after every convolution
// is zero padding at the sequence's ends), channels-last. Roundings as PyTorch's bf16 convolutions: conv0's sum is
// rounded, its bias added and rounded again (cuDNN adds the bias after), ReLU; the depthwise convolutions add the bias
// in fp32 and round once.

// conv0 (1 -> C, 3x3, stride 2, padding 1) + bias + ReLU, then the first depthwise 3x3 stride-2 convolution + bias,
// for one output row (sequence, t2) per workgroup and one channel per thread: out [rows, 32, C] bf16. The 7 mel rows
// the row needs (4 t2 - 3 .. 4 t2 + 3) are staged in LDS as fp32 with a zero column on the left (mel column c at index
// c + 1), so conv0 column f1 reads the float2 at index 2 f1 and the first value of the next.
constexpr int SUB_F1 = 64, SUB_F2 = 32, SUB_LD = MELS + 4;
__global__ void __launch_bounds__(1024) sub_conv0_dw_kernel(const uint16_t* __restrict__ feats, int64_t ld_seq,
                                                            const int* __restrict__ mel_len,
                                                            const int* __restrict__ rows, const float* __restrict__ w0,
                                                            const float* __restrict__ b0, const float* __restrict__ w2,
                                                            const float* __restrict__ b2, uint16_t* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) float mrow[7][SUB_LD];
  const int seq = rows[2 * blockIdx.x], t2 = rows[2 * blockIdx.x + 1];
  const int c = threadIdx.x, C = blockDim.x;
  const int L = mel_len[seq], T1 = (L - 1) / 2 + 1;
  const uint16_t* xs = feats + (int64_t)seq * ld_seq;
  for (int i = threadIdx.x; i < 7 * SUB_LD; i += C) {
    const int r = 4 * t2 - 3 + i / SUB_LD, col = i % SUB_LD - 1;
    mrow[i / SUB_LD][i % SUB_LD] = (r >= 0 && r < L && col >= 0 && col < MELS) ? bf2f(xs[(int64_t)r * MELS + col]) : 0.f;
  }
  float k0[9], kd[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    k0[i] = w0[c * 9 + i];
    kd[i] = w2[c * 9 + i];
  }
  const float bias0 = b0[c];
  float acc[SUB_F2];
#pragma unroll
  for (int i = 0; i < SUB_F2; ++i) acc[i] = b2[c];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 3; ++r) {  // conv0 row t1 = 2 t2 - 1 + r is the depthwise tap row r
    const int t1 = 2 * t2 - 1 + r;
    if (t1 < 0 || t1 >= T1) continue;
    const float* m0 = mrow[2 * r];
    const float* m1 = mrow[2 * r + 1];
    const float* m2 = mrow[2 * r + 2];
    float2 p0 = *reinterpret_cast<const float2*>(m0), p1 = *reinterpret_cast<const float2*>(m1),
           p2 = *reinterpret_cast<const float2*>(m2);
#pragma unroll
    for (int f1 = 0; f1 < SUB_F1; ++f1) {
      // mel columns 2 f1 - 1, 2 f1, 2 f1 + 1
      const float2 n0 = *reinterpret_cast<const float2*>(m0 + 2 * f1 + 2);
      const float2 n1 = *reinterpret_cast<const float2*>(m1 + 2 * f1 + 2);
      const float2 n2 = *reinterpret_cast<const float2*>(m2 + 2 * f1 + 2);
      float s = 0.f;
      s = __builtin_fmaf(k0[0], p0.x, s);
      s = __builtin_fmaf(k0[1], p0.y, s);
      s = __builtin_fmaf(k0[2], n0.x, s);
      s = __builtin_fmaf(k0[3], p1.x, s);
      s = __builtin_fmaf(k0[4], p1.y, s);
      s = __builtin_fmaf(k0[5], n1.x, s);
      s = __builtin_fmaf(k0[6], p2.x, s);
      s = __builtin_fmaf(k0[7], p2.y, s);
      s = __builtin_fmaf(k0[8], n2.x, s);
      const float a = fmaxf(round_bf(round_bf(s) + bias0), 0.f);
      // depthwise output f2 reads conv0 columns 2 f2 - 1, 2 f2, 2 f2 + 1 (taps 0, 1, 2): f1 ascending adds each
      // output's taps in order
      if (f1 & 1) {
        if ((f1 + 1) / 2 < SUB_F2) acc[(f1 + 1) / 2] = __builtin_fmaf(kd[3 * r], a, acc[(f1 + 1) / 2]);
        acc[(f1 - 1) / 2] = __builtin_fmaf(kd[3 * r + 2], a, acc[(f1 - 1) / 2]);
      } else {
        acc[f1 / 2] = __builtin_fmaf(kd[3 * r + 1], a, acc[f1 / 2]);
      }
      p0 = n0;
      p1 = n1;
      p2 = n2;
    }
  }
  uint16_t* o = out + (int64_t)blockIdx.x * SUB_F2 * C + c;
#pragma unroll
  for (int i = 0; i < SUB_F2; ++i) o[(int64_t)i * C] = f2bf(acc[i]);
}

// The pointwise convolution of POS positions x 256 channels held in LDS (bf16, rows of 512 bytes, 16-byte chunk c of
// position r at c ^ (r & 15)): out = relu(bf16(sum) + bias), as the bf16 GEMM's CONV_RELU computes it -- the same
// matrix instruction, operand roles and K order, so the same bits. NW waves of 256 / NW output channels; the weights go
// straight from L2 into registers, two K steps ahead. The results replace the operand in LDS and leave as whole rows.
constexpr int PW_C = 256;
DEVI int pw_slot(int r, int c) { return r * (2 * PW_C) + ((c ^ (r & 15)) << 4); }  // byte offset of chunk c

template <int POS, int NW>
DEVI void pointwise(char* tile, const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias,
                    uint16_t* __restrict__ out, int64_t n_pos) {
  constexpr int MI = POS / 16, NI = 16 / NW, KS = PW_C / 32;
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id(), c16 = lane & 15, h = lane >> 4;
  const int n0 = wave * (16 * NI);
  v8bf wf[3][NI];
  auto load_w = [&](int b, int ks) {
#pragma unroll
    for (int j = 0; j < NI; ++j)
      wf[b][j] = *reinterpret_cast<const v8bf*>(w + (n0 + j * 16 + c16) * PW_C + ks * 32 + 8 * h);
  };
  load_w(0, 0);
  load_w(1, 1);
  uint2 braw[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) braw[j] = *reinterpret_cast<const uint2*>(bias + n0 + j * 16 + 4 * h);
  v4f acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = v4f{0.f, 0.f, 0.f, 0.f};
  __syncthreads();  // the tile
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    if (ks + 2 < KS) load_w((ks + 2) % 3, ks + 2);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const v8bf x = *reinterpret_cast<const v8bf*>(tile + pw_slot(i * 16 + c16, ks * 4 + h));
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ks % 3][j], x, acc[j][i], 0, 0, 0);
    }
  }
  __syncthreads();  // every wave has read the operand
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const float b4[4] = {__uint_as_float(braw[j].x << 16), __uint_as_float(braw[j].x & 0xffff0000u),
                         __uint_as_float(braw[j].y << 16), __uint_as_float(braw[j].y & 0xffff0000u)};
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = fmaxf(round_bf(acc[j][i][k]) + b4[k], 0.f);
      const int col = n0 + j * 16 + 4 * h;  // four channels: half of a 16-byte chunk
      *reinterpret_cast<uint2*>(tile + pw_slot(i * 16 + c16, col >> 3) + (col & 4) * 2) =
          make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
    }
  }
  __syncthreads();
  for (int i = tid; i < POS * 32; i += NW * 64) {
    const int r = i >> 5, c = i & 31;
    if (r < n_pos)
      *reinterpret_cast<uint4*>(out + (int64_t)r * PW_C + c * 8) = *reinterpret_cast<const uint4*>(tile + pw_slot(r, c));
  }
}

// The same two convolutions and the pointwise one that follows, for C = 256, SUB_T output rows (sequence, t2) per
// workgroup; the same bits as the two launches. On the vector units a conv0 value takes 9 multiply-adds and 7 more
// instructions, and that issue is all of the kernel above (129 us for 8 pieces of 30 s; with conv0 rows shared between
// output rows and the pointwise convolution behind it 153). So conv0's multiply-adds run on the matrix cores, one
// instruction a tap: with K = 1 in fp32 it adds each position's product to the sum before it with one rounding, the
// fma of the chain above. (All taps in one bf16 instruction, a weight as three exact bf16 parts, sums them in another
// order, with 1.4 times the rounding error where mel values span many powers of two.) 8 pieces of 30 s: 115 us
// for what the two launches take 169; what is left is the vector work after the sums (about 60 us).
//  * The matrix instruction's four blocks of 16 rows are the 64 positions of a conv0 row: row m of block pb is position
//    16 (m / 4) + 4 pb + m % 4, so a lane holds 16 consecutive positions of a channel and the depthwise taps need one
//    value from another lane.
//  * Where the next row of the list is t2 + 1 of the same sequence (the stem's lists), conv0 row 2 t2 + 1 is computed
//    once and added to both rows' sums.
//  * The rows stay in LDS as the pointwise convolution's operand; only its output is written.
constexpr int SUB_T = 4, SUB_W = 8, SUB_J = 16 / SUB_W;  // output rows, waves, 16-channel blocks of a wave
constexpr int MEL_LD = MELS + 8;
typedef float v16f __attribute__((ext_vector_type(16)));
__global__ void __launch_bounds__(SUB_W * 64) __attribute__((amdgpu_waves_per_eu(4))) sub_conv0_dw_pw_kernel(
    const uint16_t* __restrict__ feats, int64_t ld_seq, const int* __restrict__ mel_len, const int* __restrict__ rows,
    int n_rows, const float* __restrict__ w0, const float* __restrict__ b0, const float* __restrict__ w2,
    const float* __restrict__ b2, const uint16_t* __restrict__ wp, const uint16_t* __restrict__ bp,
    uint16_t* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) char tile[SUB_T * SUB_F2 * 2 * PW_C];
  // mel rows 4 t2 - 3 .. 4 t2 + 3, column c at c + 1, zeros outside
  __shared__ __attribute__((aligned(8))) uint16_t mel[SUB_T][7][MEL_LD];
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id(), c16 = lane & 15, h = lane >> 4;
  const int i0 = blockIdx.x * SUB_T, nt = min(SUB_T, n_rows - i0);
  // one thread per pair of columns of the seven rows, every load unguarded (a row outside the sequence loads row 0)
  static_assert(7 * (MELS / 2) <= SUB_W * 64 && SUB_T * 7 * (MEL_LD - MELS) <= SUB_W * 64, "one pass");
  const int mr = min(tid / (MELS / 2), 6), mc = tid % (MELS / 2) * 2;
  uint32_t mv[SUB_T];
#pragma unroll
  for (int k = 0; k < SUB_T; ++k) {
    const int i = min(i0 + k, n_rows - 1), seq = rows[2 * i], r = 4 * rows[2 * i + 1] - 3 + mr;
    const bool in = r >= 0 && r < mel_len[seq];
    const u32_any v = *reinterpret_cast<const u32_any*>(feats + (int64_t)seq * ld_seq + (in ? (int64_t)r * MELS : 0) + mc);
    mv[k] = in ? (uint32_t)v : 0u;
  }
  // this lane's channels (wave * SUB_J + j) * 16 + c16: conv0 weights (the B operand, the same in all four blocks) and
  // depthwise taps
  float wf[SUB_J][9], kd[SUB_J][9], bias0[SUB_J], bias2[SUB_J];
#pragma unroll
  for (int j = 0; j < SUB_J; ++j) {
    const int c = (wave * SUB_J + j) * 16 + c16;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      wf[j][i] = w0[c * 9 + i];
      kd[j][i] = w2[c * 9 + i];
    }
    bias0[j] = b0[c];
    bias2[j] = b2[c];
  }
  const int f1 = 16 * (c16 >> 2) + 4 * h + (c16 & 3);  // this lane's position as A operand: row c16 of block h
  float acc[SUB_J][8], acc2[SUB_J][8];  // depthwise sums of this lane's channels at f2 = 8 h + o, this output row's and the next's
  // the conv0 row of output row k's tap row r, added as that tap row (and, both, to the next output row as tap row 0)
  auto conv_row = [&](int k, int r, bool both) {
    float x[9];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t* m = reinterpret_cast<const uint32_t*>(&mel[k][2 * r + i][2 * f1]);
      const uint32_t lo = m[0], hi = m[1];
      x[3 * i] = __uint_as_float(lo << 16);
      x[3 * i + 1] = __uint_as_float(lo & 0xffff0000u);
      x[3 * i + 2] = __uint_as_float(hi << 16);
    }
#pragma unroll
    for (int j = 0; j < SUB_J; ++j) {
      v16f d = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 9; ++i) d = __builtin_amdgcn_mfma_f32_16x16x1f32(x[i], wf[j][i], d, 0, 0, 0);
      float v[16];
#pragma unroll
      for (int q = 0; q < 16; q += 2) {
        const uint32_t u = pack_bf2(d[q], d[q + 1]);  // rounded, then the bias, ReLU and the second rounding
        v[q] = round_bf_valu(fmaxf(__uint_as_float(u << 16) + bias0[j], 0.f));
        v[q + 1] = round_bf_valu(fmaxf(__uint_as_float(u & 0xffff0000u) + bias0[j], 0.f));
      }
      // position 16 h - 1: the last one of the lane 16 below (none for h = 0)
      const float left = __shfl(v[15], (lane - 16) & 63, 64);
      const float t0 = r == 0 ? kd[j][0] : r == 1 ? kd[j][3] : kd[j][6], t1 = r == 0 ? kd[j][1] : r == 1 ? kd[j][4] : kd[j][7],
                  t2 = r == 0 ? kd[j][2] : r == 1 ? kd[j][5] : kd[j][8];
      auto add = [&](float (&s)[8], float k0, float k1, float k2) {
#pragma unroll
        for (int o = 0; o < 8; ++o) {
          if (o == 0) {
            const float y = __builtin_fmaf(k0, left, s[0]);
            s[0] = h > 0 ? y : s[0];
          } else {
            s[o] = __builtin_fmaf(k0, v[2 * o - 1], s[o]);
          }
          s[o] = __builtin_fmaf(k1, v[2 * o], s[o]);
          s[o] = __builtin_fmaf(k2, v[2 * o + 1], s[o]);
        }
      };
      add(acc[j], t0, t1, t2);
      if (both) add(acc2[j], kd[j][0], kd[j][1], kd[j][2]);
    }
  };
  auto clear = [&](float (&s)[SUB_J][8]) {
#pragma unroll
    for (int j = 0; j < SUB_J; ++j)
#pragma unroll
      for (int o = 0; o < 8; ++o) s[j][o] = bias2[j];
  };
  auto follows = [&](int k) {  // output row k + 1 is the next one of the same sequence
    return k + 1 < nt && rows[2 * (i0 + k) + 2] == rows[2 * (i0 + k)] &&
           rows[2 * (i0 + k) + 3] == rows[2 * (i0 + k) + 1] + 1;
  };
  if (tid < 7 * (MELS / 2)) {
#pragma unroll
    for (int k = 0; k < SUB_T; ++k) {
      mel[k][mr][mc + 1] = (uint16_t)mv[k];
      mel[k][mr][mc + 2] = (uint16_t)(mv[k] >> 16);
    }
  }
  if (tid < SUB_T * 7 * (MEL_LD - MELS)) {  // the zero columns
    const int row = tid / (MEL_LD - MELS), e = tid % (MEL_LD - MELS);
    mel[row / 7][row % 7][e == 0 ? 0 : MELS + e] = 0;
  }
  __syncthreads();  // mel rows
  bool carried = false;  // acc holds this row's tap row 0
  clear(acc);
  for (int k = 0; k < nt; ++k) {
    const int seq = rows[2 * (i0 + k)], t2 = rows[2 * (i0 + k) + 1], T1 = (mel_len[seq] - 1) / 2 + 1;
    const bool next = follows(k);
    for (int r = carried ? 1 : 0; r < 3; ++r) {
      const int t1 = 2 * t2 - 1 + r;
      if (r == 2 && next) clear(acc2);
      if (t1 >= 0 && t1 < T1) conv_row(k, r, r == 2 && next);
    }
#pragma unroll
    for (int j = 0; j < SUB_J; ++j)
#pragma unroll
      for (int o = 0; o < 8; ++o) {
        const int c = (wave * SUB_J + j) * 16 + c16;
        *reinterpret_cast<uint16_t*>(tile + pw_slot(k * SUB_F2 + 8 * h + o, c >> 3) + (c & 7) * 2) = f2bf(acc[j][o]);
      }
    carried = next;
#pragma unroll
    for (int j = 0; j < SUB_J; ++j)
#pragma unroll
      for (int o = 0; o < 8; ++o) acc[j][o] = next ? acc2[j][o] : bias2[j];
  }
  pointwise<SUB_T * SUB_F2, SUB_W>(tile, wp, bp, out + (int64_t)i0 * SUB_F2 * PW_C, (int64_t)nt * SUB_F2);
}

// depthwise 3x3 stride-2 convolution + bias on channels-last sequences x [sum T_in, F_in, C]: output row
// (sequence, t) = rows[i] into out [n, F_in / 2, C]; a thread per (row, frequency, 8 channels)
__global__ void __launch_bounds__(256) sub_dw_kernel(const uint16_t* __restrict__ x, const int* __restrict__ in_start,
                                                     const int* __restrict__ in_len, const int* __restrict__ rows,
                                                     const float* __restrict__ w, const float* __restrict__ b,
                                                     uint16_t* __restrict__ out, int64_t n, int F_in, int C) {
  const int F_out = F_in / 2, chunks = C / 8;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n * F_out * chunks) return;
  const int c = (int)(id % chunks) * 8, fo = (int)((id / chunks) % F_out);
  const int64_t i = id / chunks / F_out;
  const int seq = rows[2 * i], t = rows[2 * i + 1];
  // this thread's 8 channels x 9 taps are 72 consecutive floats of the (C, 9) layout: 18 16-byte loads, issued
  // with the bias before the row's own loads (not one 4-byte load per tap inside the guarded loops)
  float wk[8 * 9], acc[8];
#pragma unroll
  for (int v = 0; v < 18; ++v)
    *reinterpret_cast<float4*>(wk + 4 * v) = *reinterpret_cast<const float4*>(w + (int64_t)c * 9 + 4 * v);
  *reinterpret_cast<float4*>(acc) = *reinterpret_cast<const float4*>(b + c);
  *reinterpret_cast<float4*>(acc + 4) = *reinterpret_cast<const float4*>(b + c + 4);
  const int start = in_start[seq], len = in_len[seq];
  // the 3 x 3 input chunks (zero outside the sequence or the frequency range), all loaded before the first use
  uint4 u[9];
#pragma unroll
  for (int di = 0; di < 3; ++di)
#pragma unroll
    for (int dj = 0; dj < 3; ++dj) {
      const int ti = 2 * t - 1 + di, fi = 2 * fo - 1 + dj;
      const bool in = ti >= 0 && ti < len && fi >= 0 && fi < F_in;
      const int64_t off = in ? (((int64_t)start + ti) * F_in + fi) * C + c : 0;
      u[di * 3 + dj] = *reinterpret_cast<const uint4*>(x + off);
      if (!in) u[di * 3 + dj] = make_uint4(0, 0, 0, 0);
    }
  // the taps in the same order as before (missing taps skipped, not added as zeros: the fma chain is unchanged)
#pragma unroll
  for (int di = 0; di < 3; ++di) {
    const int ti = 2 * t - 1 + di;
    if (ti < 0 || ti >= len) continue;
#pragma unroll
    for (int dj = 0; dj < 3; ++dj) {
      const int fi = 2 * fo - 1 + dj;
      if (fi < 0 || fi >= F_in) continue;
      const uint4 v = u[di * 3 + dj];
      const uint32_t e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float xv = __uint_as_float(k & 1 ? e[k / 2] & 0xffff0000u : e[k / 2] << 16);
        acc[k] = __builtin_fmaf(wk[k * 9 + di * 3 + dj], xv, acc[k]);
      }
    }
  }
  uint4 o;
  o.x = pack_bf2(acc[0], acc[1]);
  o.y = pack_bf2(acc[2], acc[3]);
  o.z = pack_bf2(acc[4], acc[5]);
  o.w = pack_bf2(acc[6], acc[7]);
  *reinterpret_cast<uint4*>(out + ((int64_t)i * F_out + fo) * C + c) = o;
}

// The same depthwise convolution and the pointwise one that follows, for F_in = 32 and C = 256: a workgroup takes DWP_T
// output rows x 16 frequencies. A thread keeps its 8 channels' 72 taps for 8 outputs (sub_dw_kernel reads them, 320
// bytes, for each output of 144 input bytes) and two neighbouring frequencies share a column of inputs. 8 pieces of
// 30 s: 33 us for what the two launches took 58.
constexpr int DWP_T = 4, DWP_F = 16;
__global__ void __launch_bounds__(256) sub_dw_pw_kernel(const uint16_t* __restrict__ x, const int* __restrict__ in_start,
                                                        const int* __restrict__ in_len, const int* __restrict__ rows,
                                                        const float* __restrict__ w, const float* __restrict__ b,
                                                        const uint16_t* __restrict__ wp, const uint16_t* __restrict__ bp,
                                                        uint16_t* __restrict__ out, int n_rows) {
  __shared__ __attribute__((aligned(16))) char tile[DWP_T * DWP_F * 2 * PW_C];
  constexpr int F_in = 2 * DWP_F;
  const int i0 = blockIdx.x * DWP_T, nt = min(DWP_T, n_rows - i0), chunk = threadIdx.x & 31, pl = threadIdx.x >> 5;
  const int c = chunk * 8, f0 = 4 * pl - 1;  // outputs 2 pl, 2 pl + 1 read input frequencies f0 .. f0 + 4
  float wk[8 * 9], bias[8];
#pragma unroll
  for (int v = 0; v < 18; ++v)
    *reinterpret_cast<float4*>(wk + 4 * v) = *reinterpret_cast<const float4*>(w + c * 9 + 4 * v);
  *reinterpret_cast<float4*>(bias) = *reinterpret_cast<const float4*>(b + c);
  *reinterpret_cast<float4*>(bias + 4) = *reinterpret_cast<const float4*>(b + c + 4);
  for (int k = 0; k < nt; ++k) {
    const int seq = rows[2 * (i0 + k)], t = rows[2 * (i0 + k) + 1], start = in_start[seq], len = in_len[seq];
    float acc[2][8];
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[o][e] = bias[e];
    uint4 u[3][5];
#pragma unroll
    for (int di = 0; di < 3; ++di) {
      const int ti = 2 * t - 1 + di;  // for a row outside the sequence row 0 is loaded and not used
      const int64_t row = ti >= 0 && ti < len ? (int64_t)start + ti : 0;
#pragma unroll
      for (int dj = 0; dj < 5; ++dj)
        u[di][dj] = *reinterpret_cast<const uint4*>(x + (row * F_in + max(f0 + dj, 0)) * PW_C + c);
    }
    // the taps in order, missing ones skipped (not added as zeros)
#pragma unroll
    for (int di = 0; di < 3; ++di) {
      const int ti = 2 * t - 1 + di;
      if (ti < 0 || ti >= len) continue;
#pragma unroll
      for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int dj = 0; dj < 3; ++dj) {
          const uint4 v = u[di][2 * o + dj];
          const uint32_t q[4] = {v.x, v.y, v.z, v.w};
          const bool in = o > 0 || dj > 0 || f0 >= 0;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float xv = __uint_as_float(e & 1 ? q[e / 2] & 0xffff0000u : q[e / 2] << 16);
            const float s = __builtin_fmaf(wk[e * 9 + di * 3 + dj], xv, acc[o][e]);
            acc[o][e] = in ? s : acc[o][e];
          }
        }
    }
#pragma unroll
    for (int o = 0; o < 2; ++o)
      *reinterpret_cast<uint4*>(tile + pw_slot(k * DWP_F + 2 * pl + o, chunk)) =
          make_uint4(pack_bf2(acc[o][0], acc[o][1]), pack_bf2(acc[o][2], acc[o][3]), pack_bf2(acc[o][4], acc[o][5]),
                     pack_bf2(acc[o][6], acc[o][7]));
  }
  pointwise<DWP_T * DWP_F, 4>(tile, wp, bp, out + (int64_t)i0 * DWP_F * PW_C, (int64_t)nt * DWP_F);
}

// ---- packed pieces ---------------------------------------------------------------------------------------------------
// For packed pieces of count[b] rows each, every row's piece (its id) and its row within the piece. The counts travel as
// kernel arguments: no upload, so nothing to pin, to wait for or to keep until a copy has run. A workgroup per piece.
constexpr int PIECES = 128;  // of one launch
struct Pieces {
  int32_t id[PIECES], start[PIECES + 1];
};
__global__ void __launch_bounds__(256) piece_rows_kernel(const Pieces p, int32_t* __restrict__ piece_of,
                                                         int32_t* __restrict__ row_of, int64_t stride) {
  const int b = blockIdx.x, id = p.id[b], start = p.start[b], n = p.start[b + 1] - start;
  for (int r = threadIdx.x; r < n; r += 256) {
    piece_of[(start + r) * stride] = id;
    row_of[(start + r) * stride] = r;
  }
}

bool aligned(const void* q, int a) { return (reinterpret_cast<uintptr_t>(q) % a) == 0; }

}  // namespace

extern "C" int64_t cohere_logmel_workspace_bytes(int64_t total_frames) {
  return total_frames < 0 ? -1 : total_frames * MELS * (int64_t)sizeof(float);
}

extern "C" int cohere_logmel_features(const float* x, const int64_t* meta, int64_t pieces, int64_t total_frames,
                                      const float* window, const float* mel, const int32_t* band, float preemph,
                                      uint16_t* out, int64_t T, float* work, void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(pieces >= 0 && total_frames >= 0 && T >= 0 && pieces < (1 << 30), "logmel_features: bad sizes");
  if (total_frames == 0 || pieces == 0) return 0;
  COHERE_REQUIRE(x && meta && window && mel && band && out && work, "logmel_features: null pointer");
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // frames per wave: as many as keep four workgroups for each of 256 CUs (a workgroup's tables cost about as much as
  // three frames)
  const int64_t per_wave = std::min<int64_t>(8, std::max<int64_t>(1, total_frames / (FPW * 1024)));
  const int64_t blocks = (total_frames + FPW * per_wave - 1) / (FPW * per_wave);
  COHERE_REQUIRE(blocks < (1LL << 31), "logmel_features: too many frames");
  logmel_kernel<<<(unsigned)blocks, FPW * 64, 0, s>>>(x, meta, (int)pieces, total_frames, (int)per_wave, window, mel,
                                                       band, preemph, work);
  constexpr int64_t most = (1LL << 17);  // a launch's threads are counted in 32 bits
  for (int64_t p = 0; p < pieces; p += most)
    normalize_kernel<<<(unsigned)(std::min(most, pieces - p) * (MELS / NB)), NTHR, 0, s>>>(
        work, meta + 2 * pieces + p, T, out + p * T * MELS);
  return cohere::check_launch("logmel_features");
}

extern "C" int cohere_sub_conv0_dw(const uint16_t* feats, int64_t ld_seq, const int32_t* mel_len, const int32_t* rows,
                                   int64_t n_rows, const float* w0, const float* b0, const float* w2, const float* b2,
                                   uint16_t* out, int64_t C, void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(n_rows >= 0 && n_rows < (1LL << 31), "sub_conv0_dw: bad row count");
  COHERE_REQUIRE(C >= 64 && C <= 1024 && C % 64 == 0, "sub_conv0_dw: channels must be a multiple of 64, at most 1024");
  if (n_rows == 0) return 0;
  COHERE_REQUIRE(feats && mel_len && rows && w0 && b0 && w2 && b2 && out, "sub_conv0_dw: null pointer");
  sub_conv0_dw_kernel<<<(unsigned)n_rows, (unsigned)C, 0, reinterpret_cast<hipStream_t>(stream)>>>(
      feats, ld_seq, mel_len, rows, w0, b0, w2, b2, out);
  return cohere::check_launch("sub_conv0_dw");
}

extern "C" int cohere_sub_dw(const uint16_t* x, const int32_t* in_start, const int32_t* in_len, const int32_t* rows,
                             int64_t n_rows, const float* w, const float* b, uint16_t* out, int64_t F_in, int64_t C,
                             void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(n_rows >= 0 && F_in >= 2 && F_in <= 4096 && C > 0 && C % 8 == 0 && C <= 65536,
                 "sub_dw: bad sizes (C % 8 == 0)");
  if (n_rows == 0) return 0;
  COHERE_REQUIRE(x && in_start && in_len && rows && w && b && out, "sub_dw: null pointer");
  COHERE_REQUIRE(aligned(x, 16) && aligned(out, 16) && aligned(w, 16) && aligned(b, 16),
                 "sub_dw: x, out, the taps and the bias must be 16-byte aligned");
  const int64_t total = n_rows * (F_in / 2) * (C / 8);
  COHERE_REQUIRE((total + 255) / 256 < (1LL << 31), "sub_dw: too many rows");
  sub_dw_kernel<<<(unsigned)((total + 255) / 256), 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(
      x, in_start, in_len, rows, w, b, out, n_rows, (int)F_in, (int)C);
  return cohere::check_launch("sub_dw");
}

extern "C" int cohere_sub_conv0_dw_pw(const uint16_t* feats, int64_t ld_seq, const int32_t* mel_len,
                                      const int32_t* rows, int64_t n_rows, const float* w0, const float* b0,
                                      const float* w2, const float* b2, const uint16_t* wp, const uint16_t* bp,
                                      uint16_t* out, void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(n_rows >= 0 && n_rows < (1LL << 30), "sub_conv0_dw_pw: bad row count");
  if (n_rows == 0) return 0;
  COHERE_REQUIRE(feats && mel_len && rows && w0 && b0 && w2 && b2 && wp && bp && out, "sub_conv0_dw_pw: null pointer");
  COHERE_REQUIRE(aligned(wp, 16) && aligned(bp, 8) && aligned(out, 16),
                 "sub_conv0_dw_pw: the pointwise weights and out must be 16-byte aligned, its bias 8-byte aligned");
  sub_conv0_dw_pw_kernel<<<(unsigned)((n_rows + SUB_T - 1) / SUB_T), SUB_W * 64, 0, reinterpret_cast<hipStream_t>(stream)>>>(
      feats, ld_seq, mel_len, rows, (int)n_rows, w0, b0, w2, b2, wp, bp, out);
  return cohere::check_launch("sub_conv0_dw_pw");
}

extern "C" int cohere_sub_dw_pw(const uint16_t* x, const int32_t* in_start, const int32_t* in_len, const int32_t* rows,
                                int64_t n_rows, const float* w, const float* b, const uint16_t* wp, const uint16_t* bp,
                                uint16_t* out, void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(n_rows >= 0 && n_rows < (1LL << 30), "sub_dw_pw: bad row count");
  if (n_rows == 0) return 0;
  COHERE_REQUIRE(x && in_start && in_len && rows && w && b && wp && bp && out, "sub_dw_pw: null pointer");
  COHERE_REQUIRE(aligned(x, 16) && aligned(out, 16) && aligned(w, 16) && aligned(b, 16) && aligned(wp, 16) &&
                     aligned(bp, 8),
                 "sub_dw_pw: x, out, the taps, the biases and the weights must be 16-byte aligned");
  sub_dw_pw_kernel<<<(unsigned)((n_rows + DWP_T - 1) / DWP_T), 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(
      x, in_start, in_len, rows, w, b, wp, bp, out, (int)n_rows);
  return cohere::check_launch("sub_dw_pw");
}

extern "C" int cohere_piece_rows(const int32_t* ids, const int32_t* counts, int64_t n, int32_t* piece_of, int32_t* row_of,
                                 int64_t stride, void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(n >= 0 && stride >= 1, "piece_rows: bad sizes");
  COHERE_REQUIRE(n == 0 || (counts && piece_of && row_of), "piece_rows: null pointer");
  int64_t total = 0;
  for (int64_t b = 0; b < n; ++b) {
    COHERE_REQUIRE(counts[b] >= 0, "piece_rows: repeats can not be negative");
    total += counts[b];
  }
  COHERE_REQUIRE(total < (1LL << 31), "piece_rows: too many rows");
  int64_t row = 0;
  for (int64_t b0 = 0; b0 < n; b0 += PIECES) {
    const int m = (int)std::min<int64_t>(PIECES, n - b0);
    Pieces p;
    p.start[0] = 0;
    for (int b = 0; b < m; ++b) {
      p.id[b] = ids ? ids[b0 + b] : (int32_t)(b0 + b);
      p.start[b + 1] = p.start[b] + counts[b0 + b];
    }
    if (p.start[m] > 0)
      piece_rows_kernel<<<(unsigned)m, 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(p, piece_of + row * stride,
                                                                                        row_of + row * stride, stride);
    row += p.start[m];
  }
  return cohere::check_launch("piece_rows");
}
