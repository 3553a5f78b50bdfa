// C ABI of the W8A8 int8 GEMMs (include/cohere_hip.h): argument checks, the reference's config-id semantics, the
// choice of gfx950 tile, and dispatch to the kernel instantiations (gemm_q8.h, gemm_q8_dense.hip, gemm_q8_sparse.hip).
#include "cohere_hip.h"
#include "gemm_q8.h"
#include "gemm_q8_rows.h"

#include <algorithm>
#include <cstring>
#include <string>

namespace {

using namespace cohere_gemm;

int g_tile_override = -1;

int num_cus() {
  static int n = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) !=
                                                  hipSuccess || v <= 0)
      v = 256;
    return v;
  }();
  return n;
}

// The time of a round of workgroups, one per CU, on each tile, in microseconds: c per 128-byte K stage, f for the launch,
// the first stage and the epilogue, q8 for SILU_Q8's. 64x64 tiles (per_cu 2): two share a CU, each stage then taking
// 1.25 to 1.35 times as long (the more, the more CUs hold two), and what is more than that counts by half rounds. (As
// whole rounds of two with one workgroup's time, 7000 grouped rows x 1280 x 5120 took 64x64 tiles, 110 us, where 128x128
// ones take 83.)
// Fitted to graph replays of every tile at 889 products of each kind (int8; 2:4 row-major and stage-tiled; bf16; 781 with
// grouped scales): 100 to 9024 rows, N 256 to 8192, K 256 to 5120, the encoder's, the stem's and the caches' among them.
// The choice is within 4 % of the fastest tile at all but 8 stage-tiled, 9 row-major, 6 bf16 and 1 grouped of them, int8
// aside (EIGHT_WAVES). Against the largest tile that gives 64 % of the CUs a workgroup (the former rule), 5245 products,
// half of them of other sizes than the fit's (111 to 8000 rows, N 320 to 6144, K 640 to 3072), take 0.96 of the time on
// average; 5 take more than 1.05 times it, at most 1.08. Some: bf16 1892 x 1280 x 5120 62.2 -> 39.1 us, 1892 x 5120 x 1280
// SILU 48.3 -> 39.7, 1892 x 1280 x 1280 21.4 -> 13.9, 3000 x 1024 x 1280 15.0 -> 12.6; int8 3000 x 1280 x 1280 12.2 -> 9.5,
// grouped 1892 x 1280 x 5120 42.7 -> 28.3.
struct TileCost {
  int id;
  int per_cu;
  double c, f, q8;
};
constexpr TileCost BF16_COST[] = {{6, 1, 1.28, 10.9, 0.0}, {15, 1, 1.335, 10.0, 0.0}, {8, 1, .695, 7.5, 0.0},
                                  {9, 1, .69, 6.6, 0.0},   {17, 1, .42, 4.5, 0.0},    {3, 1, .325, 4.1, 0.0},
                                  {7, 2, .265, 3.0, 0.0}};
constexpr TileCost DENSE_COST[] = {{6, 1, 1.28, 10.9, 8.0}, {15, 1, 1.285, 10.5, 6.2}, {8, 1, .695, 7.5, 3.0},
                                   {9, 1, .69, 6.6, 3.0},   {17, 1, .42, 4.5, 2.0},    {4, 1, .6, 4.2, 3.3},
                                   {3, 1, .335, 3.3, 2.0},  {5, 1, .27, 3.1, 2.0},     {7, 2, .268, 3.0, 2.0}};
// int8 over several rounds: alone the 8-wave tiles (doubled fragments) are up to 18 % faster than 256x256 on 16 waves, but
// whole layers that ran on them were up to 4 % slower, kernels that had not changed among them (2 blocks of 16 clips of
// 200 to 376 frames 835 -> 860 us, of 24 x 376 1356 -> 1378; the attention 40.7 -> 44.9, the depthwise convolution 18.6 ->
// 19.2): the chip's clock falls under the denser matrix work. Counted a quarter longer such products keep the 256x256
// tile: 836 and 1355 us. How much it is depends on the card: with the GLU product of 8401 rows on 128x256 a block took 628
// us against 632 on one, and on another 666 where the former rule took 657. (Over one round they stay: 8 x 375 frames
// 522 -> 509. bf16 layers gained at every size.)
constexpr double EIGHT_WAVES = 1.25;
// stage-tiled 2:4 weights
constexpr TileCost SPARSE_COST[] = {{10, 1, .902, 9.5, 7.0}, {15, 1, 1.25, 11.0, 7.0}, {8, 1, .589, 5.5, 3.5},
                                    {9, 1, .442, 6.5, 3.5},  {17, 1, .555, 2.76, 2.0}, {0, 1, .409, 4.25, 2.0},
                                    {4, 1, .492, 3.4, 4.1},  {3, 1, .296, 3.3, 2.0},   {5, 1, .27, 2.9, 2.0},
                                    {7, 2, .2425, 3.0, 2.0}};
// row-major 2:4 weights: 16 waves of 256x256 lose little to them, the 8-wave tiles over a long K much (with the tiled
// weights' costs 3000 x 4096 x 4096 went to 128x256 tiles, 54 us, where 256x256 take 42)
constexpr TileCost SPARSE_ROWS_COST[] = {{15, 1, .85, 9.9, 7.0},  {8, 1, .522, 5.83, 3.5}, {9, 1, .52, 6.7, 3.5},
                                         {17, 1, .435, 3.4, 2.0}, {0, 1, .437, 3.6, 2.0},  {4, 1, .447, 3.4, 4.1},
                                         {3, 1, .268, 3.5, 2.0},  {5, 1, .27, 2.9, 2.0},   {7, 2, .25, 3.0, 2.0}};
// grouped scales (each group's fold is most of a stage); the larger 8-wave tiles spill
constexpr TileCost GROUPED_COST[] = {{17, 1, .62, 3.6, 2.0}, {4, 1, .75, 3.5, 3.3},  {3, 1, .47, 3.4, 2.0},
                                     {5, 1, .35, 3.1, 2.0},  {7, 2, .34, 3.0, 2.0}};
// and row-major 2:4 weights (3000 x 640 x 5120 64x64 tiles 24.9 us, 64x128 22.9)
constexpr TileCost GROUPED_ROWS_COST[] = {{17, 1, .62, 3.6, 2.0},  {4, 1, .75, 3.5, 3.3}, {3, 1, .44, 3.5, 2.0},
                                          {5, 1, .35, 3.1, 2.0},   {7, 2, .34, 3.0, 2.0}};

int choose_tile(const GemmArgs& p, bool grouped, bool bf = false) {
  auto fits = [&](int id) {
    const TileInfo& t = TILES[id];
    if (bf && !bf16_tile(id)) return false;
    if ((p.epi == EPI_KV || p.epi == EPI_KV8) && !kv_tile(id)) return false;
    if (p.N % t.bn) return false;
    if (grouped && !t.grouped_ok) return false;
    if (p.epi == EPI_SILU_Q8 && t.bn % p.qgroup) return false;
    return true;
  };
  if (g_tile_override >= 0 && g_tile_override < N_TILES && fits(g_tile_override)) return g_tile_override;
  // the tile whose model time is least
  const double stages = p.K / 128.0;
  const int64_t cus = num_cus();
  int best = -1;
  double least = 0.0;
  const bool dense = !grouped && !p.E && !bf;
  auto consider = [&](const auto& table) {
    for (const TileCost& t : table) {
      if (!fits(t.id)) continue;
      const int64_t n = (int64_t)((p.M + TILES[t.id].bm - 1) / TILES[t.id].bm) * (p.N / TILES[t.id].bn);
      const double rounds = (double)((n + cus - 1) / cus), once = t.f + (p.epi == EPI_SILU_Q8 ? t.q8 : 0.0);
      double us = t.per_cu == 1 || n <= cus ? rounds * (t.c * stages + once)
                                            : rounds / 2 * ((1.25 + .1 * std::min(1.0, (n - cus) / (double)cus)) *
                                                                t.c * stages + once);
      if (dense && n > cus && (t.id == 8 || t.id == 9 || t.id == 17)) us *= EIGHT_WAVES;
      if (best < 0 || us < least) best = t.id, least = us;
    }
  };
  const bool rows24 = p.E && !p.tiled;
  if (grouped) rows24 ? consider(GROUPED_ROWS_COST) : consider(GROUPED_COST);
  else if (rows24) consider(SPARSE_ROWS_COST);
  else if (p.E) consider(SPARSE_COST);
  else if (bf) consider(BF16_COST);
  else consider(DENSE_COST);
  return best;
}

// the SILU_Q8 output group of each of the reference's int8 configs (its BN, gemm_int8.cu:321-345); -2 = unknown id
int ref_cfg_group(int cfg) {
  switch (cfg) {
    case -1: return 256;
    case 0: case 1: case 3: case 7: case 10: return 128;
    case 4: case 6: case 8: return 256;
    case 5: case 9: return 64;
    default: return -2;
  }
}

// Few rows go to the few-row kernel where it is the faster one (the same bits; a forced tile keeps the tile GEMM)
bool rows_gemm(const GemmArgs& p, bool sparse, bool grouped, hipStream_t s) {
  namespace R = cohere_rows_gemm;
  if (g_tile_override >= 0 || !R::better_than_tiles(p.M, p.N, p.K, grouped)) return false;
  if (p.epi != EPI_BIAS && p.epi != EPI_RESID && p.epi != EPI_GLU) return false;
  if (grouped && p.group != R::UNIT) return false;
  R::Args a{};
  a.X = p.X; a.sx = p.sx; a.W = p.W; a.E = p.E; a.sw = p.sw; a.bias = p.bias;
  a.Y = static_cast<uint16_t*>(p.C); a.R = p.R;
  a.ldx = p.ldx; a.ldsx = p.ldsx; a.ldy = p.ldc; a.ldr = p.ldr;
  a.M = p.M; a.N = p.N; a.K = p.K; a.tiled = p.tiled; a.alpha = p.alpha;
  return R::launch(grouped ? R::X_Q8G : R::X_Q8, sparse, p.epi, a, s);
}

bool aligned16(const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; }

template <bool SPARSE>
int gemm_entry(GemmArgs& p, int64_t group, int64_t lda_k_req, hipStream_t s, const char* name) {
  const std::string nm(name);
  COHERE_REQUIRE(p.M >= 0 && p.N > 0 && p.K > 0, nm + ": bad sizes");
  COHERE_REQUIRE(p.X && p.sx && p.W && p.sw && p.C, nm + ": null pointer");
  COHERE_REQUIRE(!SPARSE || p.E, nm + ": null selectors");
  COHERE_REQUIRE(p.K % lda_k_req == 0, nm + ": K=" + std::to_string(p.K) + " not a multiple of " +
                                           std::to_string(lda_k_req));
  COHERE_REQUIRE(group > 0 && group % lda_k_req == 0 && p.K % group == 0,
                 nm + ": group must divide K and be a multiple of " + std::to_string(lda_k_req));
  COHERE_REQUIRE(p.N % 64 == 0, nm + ": N must be a multiple of 64");
  COHERE_REQUIRE(p.epi == EPI_BIAS || p.epi == EPI_RESID || p.epi == EPI_GLU || p.epi == EPI_SILU_Q8 ||
                     p.epi == EPI_I32,
                 nm + ": unsupported epilogue " + std::to_string(p.epi));
  COHERE_REQUIRE(p.epi != EPI_RESID || p.R, nm + ": residual epilogue needs resid");
  COHERE_REQUIRE(p.epi != EPI_SILU_Q8 || p.qs, nm + ": SILU_Q8 needs qs");
  const bool grouped = group < p.K;
  COHERE_REQUIRE(!(grouped && p.epi == EPI_I32), nm + ": the int32 hook takes per-row scales only");
  COHERE_REQUIRE(p.ldx % 16 == 0 && aligned16(p.X), nm + ": tokens rows must be 16-byte aligned");
  COHERE_REQUIRE(aligned16(p.W) && aligned16(p.sw), nm + ": weights must be 16-byte aligned");
  COHERE_REQUIRE(!SPARSE || aligned16(p.E), nm + ": selectors must be 16-byte aligned");
  COHERE_REQUIRE(!p.bias || (reinterpret_cast<uintptr_t>(p.bias) & 7) == 0, nm + ": bias must be 8-byte aligned");
  const int out_align = 16;  // the staged epilogues write 16-byte chunks of output rows
  const int esize = p.epi == EPI_SILU_Q8 ? 1 : (p.epi == EPI_I32 ? 4 : 2);
  COHERE_REQUIRE((reinterpret_cast<uintptr_t>(p.C) % out_align) == 0 && (p.ldc * esize) % out_align == 0,
                 nm + ": output rows must be aligned");
  COHERE_REQUIRE(p.epi != EPI_RESID || (aligned16(p.R) && p.ldr % 8 == 0), nm + ": residual rows must be aligned");
  if (p.M == 0) return 0;
  p.group = (int)group;
  if (rows_gemm(p, SPARSE, grouped, s)) return cohere::check_launch(name);
  const int tile = choose_tile(p, grouped);
  COHERE_REQUIRE(tile >= 0, nm + ": no gfx950 tile fits N=" + std::to_string(p.N));
  if (!launch_gemm<SPARSE>(tile, p.epi, grouped, p, s)) {
    cohere::set_error(nm + ": tile " + std::to_string(tile) + " has no kernel for this epilogue");
    return 1;
  }
  return cohere::check_launch(name);
}

}  // namespace

int cohere_gemm::ref_config_group(int cfg) { return ref_cfg_group(cfg); }

extern "C" int cohere_set_gemm_tile(int32_t tile) {
  if (tile == -2 || tile == -3) {  // the XCD split off / on
    cohere_gemm::g_xcd_split = tile == -3;
    return N_TILES;
  }
  g_tile_override = tile;
  return N_TILES;
}

extern "C" int cohere_gemm_tile(int32_t kind, int32_t epi, int64_t M, int64_t N, int64_t K, int64_t group) {
  if (kind < 0 || kind > 4 || M <= 0 || N <= 0 || K <= 0 || M >= (1LL << 31) || N >= (1LL << 31) || K >= (1LL << 30) ||
      N % 64)
    return -1;
  const bool bf = kind >= 3;
  GemmArgs p{};
  p.M = (int)M; p.N = (int)N; p.K = (int)(bf ? 2 * K : K); p.epi = kind == 4 ? EPI_KV : epi; p.qgroup = 256;
  p.E = kind == 1 || kind == 2 ? reinterpret_cast<const int32_t*>(&p) : nullptr; p.tiled = kind == 2;
  return choose_tile(p, !bf && group < K, bf);
}

extern "C" int cohere_gemm_i8(const int8_t* a, int64_t lda, const float* sa, int64_t ldsa, int64_t group,
                              const int8_t* w, const float* sw, const uint16_t* bias, void* out, int64_t ldc,
                              int32_t epi, const uint16_t* resid, int64_t ldr, float alpha, float* qs, int64_t ldqs,
                              int64_t M, int64_t N, int64_t K, int32_t cfg, void* stream) {
  cohere::clear_error();
  const int qg = ref_cfg_group(cfg);
  COHERE_REQUIRE(qg != -2, "gemm_i8: unknown config " + std::to_string(cfg));
  GemmArgs p{};
  p.X = a; p.sx = sa; p.W = w; p.E = nullptr; p.sw = sw; p.bias = bias; p.C = out; p.R = resid; p.qs = qs;
  p.ldx = lda; p.ldsx = ldsa; p.ldc = ldc; p.ldr = ldr; p.ldqs = ldqs;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.qgroup = qg; p.epi = epi; p.alpha = alpha;
  return gemm_entry<false>(p, group, 64, reinterpret_cast<hipStream_t>(stream), "gemm_i8");
}

extern "C" int cohere_gemm_sp(const int8_t* x, int64_t ldx, const float* sx, int64_t ldsx, int64_t group,
                              const int8_t* wc, const int32_t* e, const float* sw, const uint16_t* bias, void* out,
                              int64_t ldc, int32_t epi, const uint16_t* resid, int64_t ldr, float alpha, float* qs,
                              int64_t ldqs, int64_t M, int64_t N, int64_t K, int32_t cfg, void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(cfg >= -1 && cfg <= 4, "gemm_sp: unknown config " + std::to_string(cfg));
  GemmArgs p{};
  p.X = x; p.sx = sx; p.W = wc; p.E = e; p.sw = sw; p.bias = bias; p.C = out; p.R = resid; p.qs = qs;
  p.ldx = ldx; p.ldsx = ldsx; p.ldc = ldc; p.ldr = ldr; p.ldqs = ldqs;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.qgroup = 256; p.epi = epi; p.alpha = alpha;
  return gemm_entry<true>(p, group, 128, reinterpret_cast<hipStream_t>(stream), "gemm_sp");
}

extern "C" int cohere_gemm_sp_tiled(const int8_t* x, int64_t ldx, const float* sx, int64_t ldsx, int64_t group,
                                    const uint8_t* wt, const float* sw, const uint16_t* bias, void* out, int64_t ldc,
                                    int32_t epi, const uint16_t* resid, int64_t ldr, float alpha, float* qs,
                                    int64_t ldqs, int64_t M, int64_t N, int64_t K, int32_t cfg, void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(cfg >= -1 && cfg <= 4, "gemm_sp_tiled: unknown config " + std::to_string(cfg));
  GemmArgs p{};
  p.X = x; p.sx = sx; p.W = reinterpret_cast<const int8_t*>(wt); p.E = reinterpret_cast<const int32_t*>(wt);
  p.sw = sw; p.bias = bias; p.C = out; p.R = resid; p.qs = qs; p.tiled = 1;
  p.ldx = ldx; p.ldsx = ldsx; p.ldc = ldc; p.ldr = ldr; p.ldqs = ldqs;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.qgroup = 256; p.epi = epi; p.alpha = alpha;
  return gemm_entry<true>(p, group, 128, reinterpret_cast<hipStream_t>(stream), "gemm_sp_tiled");
}

extern "C" int64_t cohere_pack_24_tiled_bytes(int64_t N, int64_t K) {
  if (N <= 0 || K <= 0 || N % 16 || K % 128) return -1;
  return N / 16 * (K / 128) * TILED_REC;
}

extern "C" int cohere_pack_24_tiled(const int8_t* wc, const int32_t* e, int64_t N, int64_t K, uint8_t* out) {
  cohere::clear_error();
  COHERE_REQUIRE(wc && e && out, "pack_24_tiled: null pointer");
  COHERE_REQUIRE(N > 0 && K > 0 && N % 16 == 0 && K % 128 == 0, "pack_24_tiled: N % 16 and K % 128 must be 0");
  const int64_t KT = K / 128;
  for (int64_t rb = 0; rb < N / 16; ++rb)
    for (int64_t kt = 0; kt < KT; ++kt) {
      uint8_t* rec = out + (rb * KT + kt) * TILED_REC;
      for (int i = 0; i < 64; ++i) {
        const int64_t row = rb * 16 + i / 4;
        const int c = (i % 4) ^ ((i / 8) % 4);
        std::memcpy(rec + 16 * i, wc + row * (K / 2) + kt * 64 + c * 16, 16);
      }
      // row r's four selector words, words 0-1 and 2-3 swapped in rows 8-15 (see TILED_REC)
      for (int r = 0; r < 16; ++r)
        for (int w = 0; w < 4; ++w)
          std::memcpy(rec + 1024 + 16 * r + 4 * (w ^ (r & 8 ? 2 : 0)), e + (rb * 16 + r) * (K / 32) + kt * 4 + w, 4);
    }
  return 0;
}

extern "C" int cohere_gemm_bf16(const uint16_t* a, int64_t lda, const uint16_t* w, const uint16_t* bias, uint16_t* out,
                                int64_t ldc, int32_t epi, const uint16_t* resid, int64_t ldr, float alpha, int64_t M,
                                int64_t N, int64_t K, int32_t cfg, void* stream) {
  cohere::clear_error();
  COHERE_REQUIRE(cfg == 3 || cfg == 5 || cfg == 8, "gemm: unknown config " + std::to_string(cfg));
  COHERE_REQUIRE(M >= 0 && N > 0 && K > 0 && M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 30),
                 "gemm: bad sizes");
  COHERE_REQUIRE(a && w && out, "gemm: null pointer");
  COHERE_REQUIRE(K % 32 == 0, "gemm: K must match and be a multiple of 32");
  COHERE_REQUIRE(N % 64 == 0, "gemm: N must be a multiple of 64");
  COHERE_REQUIRE(epi == EPI_BIAS || epi == EPI_SILU || epi == EPI_RELU || epi == EPI_RESID || epi == EPI_GLU ||
                     epi == EPI_CONV_RELU,
                 "gemm: unknown epilogue " + std::to_string(epi));
  COHERE_REQUIRE(epi != EPI_RESID || resid, "gemm: residual epilogue needs resid");
  COHERE_REQUIRE(lda % 8 == 0 && aligned16(a) && aligned16(w), "gemm: operand rows must be 16-byte aligned");
  COHERE_REQUIRE(!bias || (reinterpret_cast<uintptr_t>(bias) & 7) == 0, "gemm: bias must be 8-byte aligned");
  COHERE_REQUIRE(aligned16(out) && ldc % 8 == 0, "gemm: output rows must be 16-byte aligned");
  COHERE_REQUIRE(epi != EPI_RESID || (aligned16(resid) && ldr % 8 == 0), "gemm: residual rows must be aligned");
  if (M == 0) return 0;
  GemmArgs p{};
  // the int8 kernel's byte addressing: K and the row stride in bytes
  p.X = reinterpret_cast<const int8_t*>(a); p.W = reinterpret_cast<const int8_t*>(w); p.bias = bias; p.C = out;
  p.R = resid; p.ldx = 2 * lda; p.ldc = ldc; p.ldr = ldr;
  p.M = (int)M; p.N = (int)N; p.K = (int)(2 * K); p.group = p.K; p.qgroup = 256; p.epi = epi; p.alpha = alpha;
  const int tile = choose_tile(p, false, true);
  COHERE_REQUIRE(tile >= 0, "gemm: no gfx950 tile fits N=" + std::to_string(p.N));
  if (!launch_gemm_bf16(tile, epi, p, reinterpret_cast<hipStream_t>(stream))) {
    cohere::set_error("gemm: tile " + std::to_string(tile) + " has no bf16 kernel for this epilogue");
    return 1;
  }
  return cohere::check_launch("gemm");
}

namespace {
int gemm_kv_entry(bool q8, const uint16_t* a, int64_t lda, const uint16_t* w, const uint16_t* bias, int64_t M, int64_t K,
                  const int32_t* slot_of, const int32_t* frame_of, void* ck, void* cv, float* cks, float* cvs, int64_t L,
                  int64_t S, int64_t H, int64_t T, void* stream, const char* name) {
  const std::string nm(name);
  COHERE_REQUIRE(M >= 0 && K > 0 && M < (1LL << 31) && K < (1LL << 30) && L > 0 && S > 0 && H > 0 && T > 0 &&
                     L * H < (1LL << 22) && S < (1LL << 31) && T < (1LL << 31),
                 nm + ": bad sizes");
  COHERE_REQUIRE(K % 32 == 0, nm + ": K must be a multiple of 32");
  COHERE_REQUIRE(a && w && slot_of && frame_of && ck && cv && (!q8 || (cks && cvs)), nm + ": null pointer");
  COHERE_REQUIRE(lda % 8 == 0 && aligned16(a) && aligned16(w), nm + ": operand rows must be 16-byte aligned");
  COHERE_REQUIRE(!bias || (reinterpret_cast<uintptr_t>(bias) & 7) == 0, nm + ": bias must be 8-byte aligned");
  COHERE_REQUIRE(aligned16(ck) && aligned16(cv), nm + ": caches must be 16-byte aligned");
  if (M == 0) return 0;
  GemmArgs p{};
  p.X = reinterpret_cast<const int8_t*>(a); p.W = reinterpret_cast<const int8_t*>(w); p.bias = bias;
  p.ldx = 2 * lda; p.M = (int)M; p.N = (int)(L * 2 * H * 128); p.K = (int)(2 * K); p.group = p.K; p.qgroup = 256;
  p.alpha = 1.f; p.epi = q8 ? EPI_KV8 : EPI_KV; p.kc = ck; p.vc = cv; p.ks = cks; p.vs = cvs; p.slot_of = slot_of;
  p.frame_of = frame_of; p.S = (int)S; p.H = (int)H; p.T = (int)T;
  const int tile = choose_tile(p, false, true);
  COHERE_REQUIRE(tile >= 0, nm + ": no gfx950 tile fits");
  if (!launch_gemm_bf16(tile, p.epi, p, reinterpret_cast<hipStream_t>(stream))) {
    cohere::set_error(nm + ": tile " + std::to_string(tile) + " has no cache epilogue");
    return 1;
  }
  return cohere::check_launch(name);
}
}  // namespace

extern "C" int cohere_gemm_kv(const uint16_t* a, int64_t lda, const uint16_t* w, const uint16_t* bias, int64_t M,
                              int64_t K, const int32_t* slot_of, const int32_t* frame_of, uint16_t* ck, uint16_t* cv,
                              int64_t L, int64_t S, int64_t H, int64_t T, void* stream) {
  cohere::clear_error();
  return gemm_kv_entry(false, a, lda, w, bias, M, K, slot_of, frame_of, ck, cv, nullptr, nullptr, L, S, H, T, stream,
                       "gemm_kv");
}

extern "C" int cohere_gemm_kv_q8(const uint16_t* a, int64_t lda, const uint16_t* w, const uint16_t* bias, int64_t M,
                                 int64_t K, const int32_t* slot_of, const int32_t* frame_of, int8_t* ck, int8_t* cv,
                                 float* cks, float* cvs, int64_t L, int64_t S, int64_t H, int64_t T, void* stream) {
  cohere::clear_error();
  return gemm_kv_entry(true, a, lda, w, bias, M, K, slot_of, frame_of, ck, cv, cks, cvs, L, S, H, T, stream,
                       "gemm_kv_q8");
}
