// Both products of a backward pass in one launch.
#include <math.h>

#include "gemm_device.h"

namespace hot {

// ---- two products in one launch -----------------------------------------------------------------------
//
// The two products of a backward pass do not depend on each other.  Launched one after the other each leaves CUs
// idle in its last round, and a lone workgroup per CU leaves the matrix cores idle while it fills its ring and while it
// stores; here both share a grid and two workgroups share a CU (at most 80 KiB of LDS and 256 registers each), so that
// one's loads and stores lie under the other's MFMAs.  The g_W tiles come first: they run longest, and g_x tiles fill
// in behind them.  Two tilings, g_x / g_W:
//   128 x 128 (2 stages) / 64 x 128 (3 stages): while the g_W product makes fewer than 256 tiles of 192 x 128, i.e.
//     one long tile per CU would be its latency.  Measured against one after the other by gemm_plan_impl (us,
//     bf16 results): 12608 x 768 x 3072 INT4 + 3072 x 768 x 7092: 50.2 / 57.5; 768 wide (proj): 21.4 / 31.0; 25216 x 768
//     x 3072 + 3072 x 768 x 7092: 69.1 / 86.1; 3003 x 520 x 1000 + 1000 x 520 x 3003: 11.8 / 19.3; 128 tokens: 5.3 / 10.0
//   192 x 128 / 192 x 128 (2 stages): from there on.  8192 x 4096 x 11008 INT4 + 11008 x 4096 x 4096: 409 / 456;
//     8192 x 11008 x 4096 + 4096 x 11008 x 2080: 348 / 424; 8192 x 4096 x 4096 + 4096^3: 174 / 187
// (Taken with ordinary stores on both sides; the streaming ones take another 3 to 19 % off the pair, gemm_epilogue_staged.)
// (the tilings the other way round: 49.1 for qkv at 12608 tokens against 42.4, 183 for the last pair against 174; the products
// alone, launched over and over: inside a step INT8 products with full rounds of 256 x 256 tiles come out ahead, gemm_pair_pays).
struct PairArgs {
  GemmArgs w, x;
  uint32_t w_blocks;      // a multiple of 8: blockIdx % 8 stays the XCD of the second product's tiles
};

template <int XBITS, bool LARGE, typename OutT>
__global__ void __launch_bounds__(G_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_pair_kernel(const PairArgs p) {
  constexpr int XM = LARGE ? 3 : 2, WM = LARGE ? 3 : 2, WN = LARGE ? 2 : 1, WGM = LARGE ? 2 : 1, WGN = LARGE ? 2 : 4, WS = LARGE ? 2 : 3;
  constexpr int LX = slot_ring_bytes<XM, 2, 2, 2, 2, 128>(), LW = slot_ring_bytes<WM, WN, WGM, WGN, WS, 128>();
  static_assert(LX <= 80 * 1024 && LW <= 80 * 1024, "two workgroups per CU");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[LX > LW ? LX : LW];
  // (the arguments are read inside the branch that uses them: both products' would overflow the scalar registers)
  typedef const __attribute__((address_space(4))) PairArgs* segment_t;
  segment_t k = (segment_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(k));
  const PairArgs& q = *(const PairArgs*)k;
  if (blockIdx.x < p.w_blocks) {
    if ((int)blockIdx.x < q.w.tiles_m * q.w.tiles_n) gemm_slot_body<WM, WN, WGM, WGN, 8, WS, 128, OutT, true>(q.w, (int)blockIdx.x, ring);
  } else {
    gemm_slot_body<XM, 2, 2, 2, XBITS, 2, 128, OutT, true>(q.x, (int)(blockIdx.x - p.w_blocks), ring);
  }
}

static void pair_tiles(GemmArgs& g, int bm, int bn) {
  g.tiles_m = (int)((g.M + bm - 1) / bm);
  g.tiles_n = (int)((g.N + bn - 1) / bn);
  g.group_m = pick_group_m(g.tiles_m, g.tiles_n, 2);
}

template <int XBITS, bool LARGE, typename OutT>
static int launch_pair(PairArgs& p, hipStream_t st) {
  pair_tiles(p.w, LARGE ? 192 : 64, 128);
  pair_tiles(p.x, LARGE ? 192 : 128, 128);
  p.w_blocks = (uint32_t)round_up((int64_t)p.w.tiles_m * p.w.tiles_n, 8);
  const int64_t total = (int64_t)p.w_blocks + (int64_t)p.x.tiles_m * p.x.tiles_n;
  if (total > (1 << 30)) return fail(HOT_ERR_UNSUPPORTED, "hot_gemm_i8: too many tiles");
  hipLaunchKernelGGL((gemm_pair_kernel<XBITS, LARGE, OutT>), dim3((unsigned)total), dim3(G_THREADS), 0, st, p);
  return check_launch("gemm_pair_kernel");
}

bool gemm_pair_possible(const GemmProduct& w, const GemmProduct& x) {
  auto fits = [](const GemmProduct& p) {
    int e;
    return p.M > 0 && p.N > 0 && p.K > 0 && (round_up(p.K, GEMM_KTILE) * p.bits / 8) % 128 == 0 && p.M * p.lda < (1ll << 32) && p.N * p.ldb < (1ll << 32) &&
           frexpf(p.post_scale, &e) == 0.5f && p.post_scale <= 1.f && p.post_scale >= FOLD_POST_MIN;   // (a power of two: acc_value, fold_exact)
  };
  return w.bits == 8 && fits(w) && fits(x);
}

// A g_x product of few tiles with a long K is a chain of stages that nothing else in the pair covers (0.9 us for each
// 256 codes of a 128 x 128 INT4 tile): such a product goes by itself, cut into K ranges or into shorter tiles by its own
// plan.  The line is where 168 shapes of 49 .. 16383 tokens and 64 .. 10624 channels are at most 14 % and on average 0.4 %
// slower than the better of the two; us of both products, pair / apart: 2758 x 128 x 8520 INT4 32.0 / 26.2, 197 x 1024 x
// 10624 45.1 / 29.3, INT8 63.7 / 34.1, 1001 x 768 x 3072 INT8 23.8 / 19.0; 2758 x 768 x 3072 INT4 20.6 / 28.5,
// 4583 x 128 x 4096 21.4 / 27.6, 8191 x 128 x 8520 35.4 / 45.2.
//
// What the pair gains is idle CUs filled and stores hidden; what it gives up is the 256 x 256 tile, which asks the L2 for 0.6
// of the operand bytes per operation.  With INT8 operands of g_x two products that take that tile, fill 94 % of its rounds and
// have few stores for their operations (K of g_x no shorter than 2/3 of its width, 14 stages and more in g_W) have nothing to
// gain.  us of the whole backward, bf16, gradients with outliers, pair / apart: 3584 x 10752 x 8960 652 / 624, 9216 x 8704 x
// 3584 688 / 661, 11264 x 4096 x 4096 340 / 324, 8192 x 11008 x 4096 in blocks of 8192 tokens 734 / 704; beside the lines
// 2048 x 8192 x 8064 313 / 329, 3200 x 8576 x 9856 540 / 587, 9472 x 5760 x 4992 472 / 484.  (Of 70 shapes none that goes apart
// is slower for it by more than 1 %.)  INT4 operands halve the bytes in question and stay in the pair: 8192 x 11008 x 4096
// 551 / 560 at work, 639 / 623 over the first 20 calls of an idle GPU.
bool gemm_pair_pays(const GemmProduct& w, const GemmProduct& x) {
  auto stages = [](const GemmProduct& p) { return round_up(p.K, GEMM_KTILE) * p.bits / 8 / 128; };
  const int64_t x_tiles = ((x.M + 127) / 128) * ((x.N + 127) / 128);
  if (x_tiles <= 192 && stages(x) >= 14 && stages(x) >= 2 * stages(w)) return false;
  auto tile256 = [](const GemmProduct& p) { return gemm_plan_impl(p.M, p.N, p.K, p.bits, p.lda, p.ldb, 0) == HOT_GEMM_SLOT_256; };
  if (x.bits == 4 || 3 * x.K < 2 * x.N || stages(w) < 14 || !tile256(w) || !tile256(x)) return true;
  auto rounds = [](const GemmProduct& p) { return (double)((((p.M + 255) / 256) * ((p.N + 255) / 256) + 255) / 256) * (double)p.K; };
  const double done = ((double)w.M * w.N * w.K + (double)x.M * x.N * x.K) / (256.0 * 65536.0);
  return done < 0.94 * (rounds(w) + rounds(x));
}

bool gemm_pair_large(const GemmProduct& w) { return ((w.M + 191) / 192) * ((w.N + 127) / 128) >= 256; }

int gemm_pair_impl(const GemmProduct& w, const GemmProduct& x, int out_dtype, hipStream_t st) {
  PairArgs p;
  if (int rc = gemm_fill(p.w, w, out_dtype, nullptr)) return rc;
  if (int rc = gemm_fill(p.x, x, out_dtype, nullptr)) return rc;
  if (!gemm_pair_possible(w, x)) return fail(HOT_ERR_UNSUPPORTED, "hot_gemm_i8: the paired kernel takes rows of whole 128-byte lines");
  const bool large = gemm_pair_large(w);
#define HOT_PAIR_CASE(OUT)                                                                                          \
  return x.bits == 4 ? (large ? launch_pair<4, true, OUT>(p, st) : launch_pair<4, false, OUT>(p, st))               \
                     : (large ? launch_pair<8, true, OUT>(p, st) : launch_pair<8, false, OUT>(p, st))
  switch (out_dtype) {
    case HOT_F32: HOT_PAIR_CASE(float);
    case HOT_BF16: HOT_PAIR_CASE(bf16_t);
    case HOT_F16: HOT_PAIR_CASE(f16_t);
    default: return fail(HOT_ERR_INVALID, "hot_gemm_i8: bad out dtype %d", out_dtype);
  }
#undef HOT_PAIR_CASE
}

}  // namespace hot
