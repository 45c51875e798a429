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
// in behind them.  Three tilings, g_x / g_W (us of the whole backward, tokens x out x in, bf16, INT4 unless noted: the three tilings in
// this order / one after the other by gemm_plan_impl; gemm_pair_tiling chooses):
//   64 x 64 both (4 stages): products that leave CUs idle in larger tiles, where the time is a chain of stages: a stage of
//     64 x 64 is 0.2 us of it, one of 128 x 128 0.45 (half the operands to wait for, and four of them under way instead of two).
//     112 x 896 x 1912 19.4 / 23.2 / 26.0 / 31.0; 15360 x 128 x 824 INT8 30.5 / 37.0 / 63.5 / 42.0; 49 x 3072 x 768 fp32 26.6 / 29.8 / 32.8 /
//     36.2; 3003 x 1000 x 520 fp16 25.7 / 26.9 / 38.0 / 34.5
//   128 x 128 (2 stages) / 64 x 128 (3 stages): what fills the chip but would make few tiles of 192 x 128.  12608 x 3072 x 768
//     118 / 105 / 114 / 117; 2304 wide fp32 121 / 111 / 129 / 119; 999 x 720 x 3696 fp16 32.4 / 30.9 / 31.8 / 35.0
//   192 x 128 both (2 stages): many tiles.  12608 x 768 x 3072 INT8 112 / 83.5 / 80.3 / 91.6; 25216 x 768 x 3072 179 / 117 / 110 / 114;
//     5376 x 4736 x 10240 666 / 514 / 464 / 527; 8192 x 11008 x 4096, blocks of 16 tokens 757 / 578 / 529 / 520 (the last one: gemm_pair_pays)
struct PairArgs {
  GemmArgs w, x;
  uint32_t w_blocks;      // a multiple of 8: blockIdx % 8 stays the XCD of the second product's tiles
};

enum { PAIR_64, PAIR_128, PAIR_192 };   // tilings of the launch
template <int XBITS, int TILING, typename OutT>
__global__ void __launch_bounds__(G_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_pair_kernel(const PairArgs p) {
  constexpr bool LARGE = TILING == PAIR_192, SMALL = TILING == PAIR_64;
  constexpr int XM = LARGE ? 3 : SMALL ? 1 : 2, XN = SMALL ? 1 : 2, XS = SMALL ? 4 : 2;
  constexpr int WM = LARGE ? 3 : SMALL ? 1 : 2, WN = LARGE ? 2 : 1, WGM = LARGE || SMALL ? 2 : 1, WGN = LARGE || SMALL ? 2 : 4, WS = LARGE ? 2 : SMALL ? 4 : 3;
  constexpr int LX = slot_ring_bytes<XM, XN, 2, 2, XS, 128>(), LW = slot_ring_bytes<WM, WN, WGM, WGN, WS, 128>();
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
    gemm_slot_body<XM, XN, 2, 2, XBITS, XS, 128, OutT, true>(q.x, (int)(blockIdx.x - p.w_blocks), ring);
  }
}

static void pair_tiles(GemmArgs& g, int bm, int bn) {
  g.tiles_m = (int)((g.M + bm - 1) / bm);
  g.tiles_n = (int)((g.N + bn - 1) / bn);
  g.group_m = pick_group_m(g.tiles_m, g.tiles_n, 2);
}

template <int XBITS, int TILING, typename OutT>
static int launch_pair(PairArgs& p, hipStream_t st) {
  pair_tiles(p.w, TILING == PAIR_192 ? 192 : 64, TILING == PAIR_64 ? 64 : 128);
  pair_tiles(p.x, TILING == PAIR_192 ? 192 : TILING == PAIR_64 ? 64 : 128, TILING == PAIR_64 ? 64 : 128);
  p.w_blocks = (uint32_t)round_up((int64_t)p.w.tiles_m * p.w.tiles_n, 8);
  const int64_t total = (int64_t)p.w_blocks + (int64_t)p.x.tiles_m * p.x.tiles_n;
  if (total > (1 << 30)) return fail(HOT_ERR_UNSUPPORTED, "hot_gemm_i8: too many tiles");
  hipLaunchKernelGGL((gemm_pair_kernel<XBITS, TILING, OutT>), dim3((unsigned)total), dim3(G_THREADS), 0, st, p);
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
// plan.  Over 170 shapes of 49 .. 16383 tokens and 64 .. 10624 channels, INT4 and INT8, the choice is on average 0.35 % slower
// than the better of the two and at most 4 %, but for INT4 products of 14 or 15 stages and a handful of tiles, where the launches
// that going apart adds cost more than the chain (240 x 3808 x 160 30.5 / 38.6, 80 x 3392 x 64 31.9 / 40.2).  us of the whole
// backward, tokens x out x in, bf16, pair / apart: 2758 x 8520 x 128 INT4 86.6 / 82.2, 197 x 10624 x 1024 66.9 / 50.9, INT8
// 90.0 / 57.9, 1001 x 3072 x 768 INT8 39.7 / 35.1; beside the line 2758 x 3072 x 768 INT4 47.1 / 55.1, 4583 x 4096 x 128
// 58.2 / 65.9, 8191 x 8520 x 128 147 / 162.
//
// What the pair gains is idle CUs filled and stores hidden; what it gives up is the 256 x 256 tile, which asks the L2 for 0.6
// of the operand bytes per operation.  With INT8 operands of g_x two products that take that tile, fill 94 % of its rounds and
// have few stores for their operations (K of g_x no shorter than 2/3 of its width, 14 stages and more in g_W) have nothing to
// gain.  us of the whole backward, tokens x out x in, blocks of 16 tokens, bf16, gradients with outliers, half a second of each,
// pair / apart: 3584 x 10752 x 8960 632 / 581, 9216 x 8704 x 3584 510 / 478, 11264 x 4096 x 4096 335 / 310, 8192 x 11008 x 4096
// 657 / 602, in one block of 8192 tokens 723 / 670; beside the lines 2048 x 8192 x 8064 292 / 305, 3200 x 8576 x 9856 518 / 555,
// 9472 x 5760 x 4992 467 / 463.  (Of 60 more shapes the one that goes apart gains 8 %; of those that stay in the pair 1792 x 9728
// x 2048 would gain 7 %, 3584 x 5632 x 9216 and 11008 x 5120 x 5632 4 %, three others 2 to 3 %.)  INT4 operands halve the bytes
// in question and stay in the pair, which was the faster order there while its results were stored through the L2: now
// 8192 x 11008 x 4096 537 / 523, in one block 620 / 597, 8192 x 4096 x 4096 223 / 215, but 8192 x 4096 x 11008 488 / 532.
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

// The tiling: from 256 tiles of 192 x 128 of g_W on that one, below them the one of the least time by this model.  A launch takes as
// long as the work of all tiles on the 512 places there are for them (two to a CU), or as the stages of one tile one after the other,
// whichever is longer, and a quarter of the other.  us for each stage of 128 bytes a row in that chain and with the chip full, and for the
// start and end of a tile, g_x and g_W; with INT8 operands a stage of g_x has half the multiplications: x_int8 of it.  Fitted to
// 157 shapes of 49 .. 25216 tokens and 64 .. 11008 channels, INT4 and INT8, all types, each timed in all three tilings: the choice is on
// average 0.3 % slower than the best of the three (two tilings and the line alone: 5.1 %).  On the wrong side of the line 128 x 2304 x 5248
// 49.0 / 46.5 / 52.0 and 512 x 4352 x 7336 127 / 118 / 127.  (1700 further shapes, the narrow ones among them: 0.5 %.)
// Up to 256 out-features a tile of g_x is little but its own store, which the model does not see: tiles of 192 rows, two to a CU, wait
// for theirs.  Where it would take them, us of the whole backward in 128 / 192: 15199 x 128 x 7848 160 / 215, 10496 x 80 x 5520 INT8 65 / 80,
// 11776 x 168 x 4992 52 / 61, 9728 x 256 x 9856 81.5 / 82.8 (24 such shapes: 6 % on average, the worst 7424 x 144 x 8168 78.6 / 74.3).
constexpr int64_t PAIR_192_LEAST_K = 256;
static int gemm_pair_tiling(const GemmProduct& w, const GemmProduct& x) {
  struct Tiling { int xm, xn, wm, wn; double chain_x, chain_w, full_x, full_w, ends_x, ends_w, x_int8; };
  static const Tiling tilings[3] = {{64, 64, 64, 64, 0.20, 0.16, 0.22, 0.18, 2.0, 1.5, 0.8},
                                    {128, 128, 64, 128, 0.45, 0.24, 0.95, 0.37, 3.3, 1.7, 0.7},
                                    {192, 128, 192, 128, 0.60, 0.48, 1.08, 1.00, 3.9, 4.8, 0.8}};
  auto tiles = [](const GemmProduct& p, int m, int n) { return (double)((p.M + m - 1) / m) * (double)((p.N + n - 1) / n); };
  auto stages = [](const GemmProduct& p) { return (double)(round_up(p.K, GEMM_KTILE) * p.bits / 8 / 128); };
  if (tiles(w, 192, 128) >= 256) return PAIR_192;
  int best = PAIR_128;
  double least = 0.0;
  for (int k = PAIR_64; k <= (x.K > PAIR_192_LEAST_K ? PAIR_192 : PAIR_128); ++k) {
    const Tiling& t = tilings[k];
    const double sx = stages(x) * (x.bits == 8 ? t.x_int8 : 1.0), sw = stages(w);
    const double full = (tiles(x, t.xm, t.xn) * (sx * t.full_x + t.ends_x) + tiles(w, t.wm, t.wn) * (sw * t.full_w + t.ends_w)) / 512.0;
    const double chain = fmax(sx * t.chain_x + t.ends_x, sw * t.chain_w + t.ends_w);
    const double us = fmax(full, chain) + 0.25 * fmin(full, chain);
    if (k == PAIR_64 || us < least) { best = k; least = us; }
  }
  return best;
}
int gemm_pair_tile_rows(const GemmProduct& w, const GemmProduct& x) {
  const int t = gemm_pair_tiling(w, x);
  return t == PAIR_192 ? 192 : t == PAIR_128 ? 128 : 64;
}

int gemm_pair_impl(const GemmProduct& w, const GemmProduct& x, int out_dtype, hipStream_t st) {
  PairArgs p;
  if (int rc = gemm_fill(p.w, w, out_dtype, nullptr)) return rc;
  if (int rc = gemm_fill(p.x, x, out_dtype, nullptr)) return rc;
  if (!gemm_pair_possible(w, x)) return fail(HOT_ERR_UNSUPPORTED, "hot_gemm_i8: the paired kernel takes rows of whole 128-byte lines");
  const int tiling = gemm_pair_tiling(w, x);
#define HOT_PAIR_TILING(BITS, OUT) \
  (tiling == PAIR_64 ? launch_pair<BITS, PAIR_64, OUT>(p, st) : tiling == PAIR_128 ? launch_pair<BITS, PAIR_128, OUT>(p, st) : launch_pair<BITS, PAIR_192, OUT>(p, st))
#define HOT_PAIR_CASE(OUT) return x.bits == 4 ? HOT_PAIR_TILING(4, OUT) : HOT_PAIR_TILING(8, OUT)
  switch (out_dtype) {
    case HOT_F32: HOT_PAIR_CASE(float);
    case HOT_BF16: HOT_PAIR_CASE(bf16_t);
    case HOT_F16: HOT_PAIR_CASE(f16_t);
    default: return fail(HOT_ERR_INVALID, "hot_gemm_i8: bad out dtype %d", out_dtype);
  }
#undef HOT_PAIR_CASE
#undef HOT_PAIR_TILING
}

}  // namespace hot
