// C ABI of libhot_gfx950 and the fused HOT linear backward.
//
// hot_linear_backward sequences the kernels of the path on one HIP stream in
// the stage order of the reference op backward_cuda
// (cuda_measure/HLQ_backward_kernel.cu:457-737: transform -> quantise ->
// low-rank -> GEMM x2 -> dequantise) with the numerics of FLinearQ.backward,
// scheme gih_gwlr (utils/quant_matmul.py:215-348).  hot_abc_forward is the
// forward-side activation buffer of FLinearQ.setup_context (:178-212).
#include <string.h>

#include <mutex>
#include <vector>

#include "phase.h"

namespace hot {

static thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int check_hip(hipError_t e, const char* what) {
  if (e == hipSuccess) return HOT_OK;
  return fail(HOT_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

int check_launch(const char* what) { return check_hip(hipGetLastError(), what); }

static const int32_t* cfg_rows(const hot_config* c) { return c->hla_n > HOT_MAX_HLA_N ? c->hla_rows_big : c->hla_rows; }

static int check_cfg(const hot_config* c, const char* who) {
  if (!c) return fail(HOT_ERR_INVALID, "%s: null config", who);
  if (c->n_o < 1 || c->n_o > 64 || (c->n_o & (c->n_o - 1))) return fail(HOT_ERR_UNSUPPORTED, "%s: n_o=%d (a power of two up to 64)", who, c->n_o);
  if (c->hla_n < 1 || c->hla_n > HOT_MAX_HLA_BIG || (c->hla_n & (c->hla_n - 1))) return fail(HOT_ERR_UNSUPPORTED, "%s: hla_n=%d (power of two up to %d)", who, c->hla_n, HOT_MAX_HLA_BIG);
  if (c->hla_n > HOT_MAX_HLA_N && !c->hla_rows_big) return fail(HOT_ERR_INVALID, "%s: hla_n=%d needs hla_rows_big", who, c->hla_n);
  if (c->hla_r < 1 || c->hla_r > c->hla_n) return fail(HOT_ERR_INVALID, "%s: hla_r=%d outside [1, %d]", who, c->hla_r, c->hla_n);
  if (c->streams < 0 || c->streams > 2) return fail(HOT_ERR_INVALID, "%s: streams=%d (0 = the library's rule, 1 or 2)", who, c->streams);
  const int bits[4] = {c->gx_bits, c->w_bits, c->gw_bits, c->act_bits};
  for (int i = 0; i < 4; ++i)
    if (bits[i] != 4 && bits[i] != 8) return fail(HOT_ERR_UNSUPPORTED, "%s: quantiser width %d (4 or 8)", who, bits[i]);
  return HOT_OK;
}

// The quantiser of g_y for the g_x product and the results' type, whichever kernels will serve them: refused before anything
// is launched (the quantisers of the column-wise passes are checked where their jobs are filled).
static int check_gx_modes(const hot_config* c, int out_dtype, const char* who) {
  if (c->gx_round != HOT_ROUND_NEAREST && c->gx_round != HOT_ROUND_STOCH) return fail(HOT_ERR_INVALID, "%s: bad rounding %d", who, c->gx_round);
  if (c->gx_scale != HOT_SCALE_TENSOR && c->gx_scale != HOT_SCALE_ROW) return fail(HOT_ERR_UNSUPPORTED, "%s: g_y scale mode %d (tensor or row)", who, c->gx_scale);
  if (out_dtype != HOT_F32 && out_dtype != HOT_BF16 && out_dtype != HOT_F16) return fail(HOT_ERR_INVALID, "%s: bad out dtype %d", who, out_dtype);
  return HOT_OK;
}

struct BwdLayout {
  int64_t ld_g, ld_w, ld_gp;                       // code pitches in bytes
  size_t off_hq, off_colw, off_colg, off_sg, off_sw, off_sgp, off_qg, off_qw, off_qgp, off_split, off_colsum, total;
  int64_t colsum_strips;                         // room for that many rows of partial column sums of g_y (bias gradient)
  size_t split_bytes;                            // split-K workspace shared by the two GEMMs
};

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

static BwdLayout bwd_layout(int64_t L, int64_t O, int64_t I, const hot_config* c) {
  BwdLayout b;
  const int64_t lp = (L / c->hla_n) * c->hla_r;
  b.ld_g = round_up(O * c->gx_bits / 8, 128);      // whole 128-byte lines (what is past O is zero)
  b.ld_w = round_up(O * c->w_bits / 8, 128);
  b.ld_gp = round_up(lp, GEMM_KTILE);
  size_t o = 0;
  b.off_hq = o;   o += STAT_SLOT_BYTES;
  b.off_colw = o; o += align256(colwise_workspace_bytes_impl(I));
  b.off_colg = o; o += align256(hla_workspace_bytes_impl(L, O, c->hla_n, c->hla_r));
  b.off_sg = o;   o += align256((size_t)L * 4);
  b.off_sw = o;   o += 256;
  b.off_sgp = o;  o += align256((size_t)O * 4);
  b.off_qg = o;   o += align256((size_t)L * b.ld_g);
  b.off_qw = o;   o += align256((size_t)I * b.ld_w);
  b.off_qgp = o;  o += align256((size_t)O * b.ld_gp);
  const GemmSplit px = gemm_split_plan(L, I, b.ld_g * 8 / c->gx_bits, c->gx_bits), pw = gemm_split_plan(O, I, lp, 8);
  b.split_bytes = px.ws_bytes > pw.ws_bytes ? px.ws_bytes : pw.ws_bytes;
  b.off_split = o; o += align256(b.split_bytes);
  {  // the workspace query knows no input type: room for the larger partition of the two element sizes
    const int64_t s2 = colsum_strips_impl(L, O, c->hla_n, c->hla_r, 0, c->gw_scale, 2);
    const int64_t s4 = colsum_strips_impl(L, O, c->hla_n, c->hla_r, 0, c->gw_scale, 4);
    b.colsum_strips = s2 > s4 ? s2 : s4;
  }
  b.off_colsum = o; o += align256((size_t)b.colsum_strips * (size_t)O * 4);
  b.total = o;
  return b;
}

// The two products, g_x = (qG . qW^T) sG sW / n_o and g_W = (qGp . xq^T) sGp sx / hla_n: their sizes, without operands.
static GemmProduct gx_product(const BwdLayout& b, int64_t L, int64_t O, int64_t I, const hot_config* c) {
  return {nullptr, b.ld_g, nullptr, b.ld_w, c->gx_bits, L, I, b.ld_g * 8 / c->gx_bits, O, nullptr, c->gx_scale == HOT_SCALE_ROW, nullptr,
          1.0f / (float)c->n_o, nullptr, I};
}
static GemmProduct gw_product(const BwdLayout& b, int64_t L, int64_t O, int64_t I, const hot_config* c) {
  const int64_t lp = (L / c->hla_n) * c->hla_r;
  return {nullptr, b.ld_gp, nullptr, b.ld_gp, 8, O, I, lp, lp, nullptr, c->gw_scale == HOT_SCALE_ROW, nullptr, 1.0f / (float)c->hla_n, nullptr, I};
}

// One stream or two, for products that cannot share a launch.  The transform + quantise work is two launches either way; the
// second stream carries the g_x product beside the g_W product.  Forking and joining it costs the host two event record /
// wait pairs, 21 us (measured), which only long calls hide: calls with little arithmetic (both products together below
// 30 GOP, e.g. ViT-B proj at 12608 tokens) keep everything on the caller's stream.
static int backward_streams(int64_t L, int64_t O, int64_t I, const hot_config* c) {
  if (c->streams == 1 || c->streams == 2) return c->streams;
  const double lp = (double)((L / c->hla_n) * c->hla_r);
  const double ops = 2.0 * (double)O * (double)I * ((double)L + lp);
  return ops < 3.0e10 ? 1 : 2;
}

// Whether the products share a launch (calls that time every kernel on its own aside).
static bool pairs(const GemmProduct& w, const GemmProduct& x, const hot_config* c) {
  return c->streams != 2 && gemm_pair_possible(w, x) && gemm_pair_pays(w, x);
}

static const int32_t* identity_rows() {
  struct Rows { int32_t v[HOT_MAX_HLA_N]; Rows() { for (int i = 0; i < HOT_MAX_HLA_N; ++i) v[i] = i; } };
  static const Rows rows;   // initialised once, thread-safe
  return rows.v;
}

// The job that adds up the partial column sums of g_y: as many rows as the statistics pass writes, which the workspace has room for.
static int colsum_args(ColsumArgs& s, const float* partial, int64_t O, int64_t strips, int64_t room, void* out, int out_dtype, const char* who) {
  if (strips > room) return fail(HOT_ERR_WORKSPACE, "%s: %lld rows of partial column sums, room for %lld", who, (long long)strips, (long long)room);
  s.partial = partial; s.C = O; s.out = out; s.out_dtype = out_dtype; s.strips = (int32_t)strips;
  return HOT_OK;
}

// Whether W's job shares the launches of a phase (Hadamard blocks of up to 16; with stochastic rounding of 16).
static bool w_joins_phase(const hot_config* c) { return c->w_round == HOT_ROUND_STOCH ? c->n_o == CW_ROWS : c->n_o <= CW_ROWS; }

}  // namespace hot

using namespace hot;

extern "C" {

const char* hot_last_error(void) { return g_err; }
int hot_abi_version(void) { return HOT_ABI_VERSION; }
int hot_backward_streams(int64_t L, int64_t O, int64_t I, const hot_config* cfg) {
  if (check_cfg(cfg, "hot_backward_streams") || L <= 0 || O <= 0 || I <= 0) return 0;
  return backward_streams(L, O, I, cfg);
}
int hot_backward_pair_rows(int64_t L, int64_t O, int64_t I, const hot_config* cfg) {
  if (hot_backward_products(L, O, I, cfg) <= HOT_PRODUCTS_APART) return 0;
  const BwdLayout b = bwd_layout(L, O, I, cfg);
  return gemm_pair_tile_rows(gw_product(b, L, O, I, cfg), gx_product(b, L, O, I, cfg));
}
int hot_backward_products(int64_t L, int64_t O, int64_t I, const hot_config* cfg) {
  if (check_cfg(cfg, "hot_backward_products") || L <= 0 || O <= 0 || I <= 0 || L % cfg->hla_n || O % cfg->n_o || O % 8 || I % 8 || cfg->gx_bits != cfg->w_bits) return 0;
  const BwdLayout b = bwd_layout(L, O, I, cfg);
  const GemmProduct px = gx_product(b, L, O, I, cfg), pw = gw_product(b, L, O, I, cfg);
  if (!pairs(pw, px, cfg)) return HOT_PRODUCTS_APART;
  return gemm_pair_tile_rows(pw, px) == 192 ? HOT_PRODUCTS_PAIR_192 : HOT_PRODUCTS_PAIR_128;
}
int64_t hot_kpad(int64_t k) { return round_up(k, GEMM_KTILE); }

int hot_gemm_splits(int64_t M, int64_t N, int64_t K, int bits) {
  if (bits != 4 && bits != 8) return 1;
  const GemmSplit sp = gemm_split_plan(M, N, K, bits);
  const int64_t pitch = round_up(K, GEMM_KTILE) * bits / 8;
  return gemm_plan_impl(M, N, K, bits, pitch, pitch, sp.ws_bytes) == HOT_GEMM_DMA_128_SPLITK ? sp.splits : 1;
}

int hot_hq_rowwise(const void* in, int dtype, int64_t M, int64_t K, int n, int bits, int rounding,
                   uint64_t seed, uint32_t rng_stream, int scale_mode, void* codes_out, float* scales_out,
                   void* workspace, size_t workspace_bytes, void* hip_stream) {
  const int64_t ld = (bits == 4 || bits == 8) ? K * bits / 8 : 0;
  return hq_rowwise_impl(in, dtype, M, K, n, bits, rounding, seed, rng_stream, scale_mode, codes_out, ld,
                         scales_out, workspace, workspace_bytes, (hipStream_t)hip_stream);
}

size_t hot_colwise_workspace_bytes(int64_t C) { return colwise_workspace_bytes_impl(C > 0 ? C : 0); }

size_t hot_hla_workspace_bytes(int64_t R, int64_t C, int n, int r) {
  if (R <= 0 || C <= 0 || n < 1 || r < 1) return 0;
  return hla_workspace_bytes_impl(R, C, n, r);
}

int hot_hla_tokenwise(const void* in, int dtype, int64_t R, int64_t C, int n, const int32_t* rows, int r,
                      int bits, int rounding, uint64_t seed, uint32_t rng_stream, int scale_mode,
                      void* codes_out, int64_t ld_out, float* scales_out, void* workspace,
                      size_t workspace_bytes, void* hip_stream) {
  return colwise_quant_impl(in, dtype, R, C, n, rows, r, bits, rounding, seed, rng_stream, scale_mode,
                            codes_out, ld_out, /*store4=*/0, scales_out, workspace, workspace_bytes,
                            (hipStream_t)hip_stream, "hot_hla_tokenwise");
}

int hot_wq_colwise(const void* in, int dtype, int64_t O, int64_t I, int n, int bits, int rounding,
                   uint64_t seed, uint32_t rng_stream, int scale_mode, void* codes_out, int64_t ld_out,
                   float* scales_out, void* workspace, size_t workspace_bytes, void* hip_stream) {
  if (n != 16 && n != 32 && n != 64) return fail(HOT_ERR_UNSUPPORTED, "hot_wq_colwise: Hadamard block %d (16, 32 or 64)", n);
  return colwise_quant_impl(in, dtype, O, I, n, identity_rows(), n, bits, rounding, seed, rng_stream, scale_mode,
                            codes_out, ld_out, /*store4=*/bits == 4, scales_out, workspace, workspace_bytes,
                            (hipStream_t)hip_stream, "hot_wq_colwise");
}

int hot_gemm_i8(const void* A, int64_t lda, const void* B, int64_t ldb, int bits, int64_t M, int64_t N,
                int64_t K, const float* scale_a, int a_per_row, const float* scale_b, float post_scale,
                void* out, int out_dtype, int64_t ldo, int32_t* acc_out, void* hip_stream) {
  return gemm_i8_impl(A, lda, B, ldb, bits, M, N, K, scale_a, a_per_row, scale_b, post_scale, out, out_dtype,
                      ldo, acc_out, (hipStream_t)hip_stream);
}

int hot_gemm_bf16(const void* A, int64_t lda, const void* B, int64_t ldb, int64_t M, int64_t N, int64_t K,
                  const void* bias, void* out, int out_dtype, int64_t ldo, int variant, void* hip_stream) {
  return gemm_bf16_impl(A, lda, B, ldb, M, N, K, bias, out, out_dtype, ldo, (hipStream_t)hip_stream, variant);
}

int hot_gemm_plan(int64_t M, int64_t N, int64_t K, int bits, int64_t lda, int64_t ldb, size_t workspace_bytes) {
  return gemm_plan_impl(M, N, K, bits, lda, ldb, workspace_bytes);
}

size_t hot_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int bits) {
  if (bits != 4 && bits != 8) return 0;
  return gemm_split_plan(M, N, K, bits).ws_bytes;
}

int hot_gemm_i8_variant(const void* A, int64_t lda, const void* B, int64_t ldb, int bits, int64_t M, int64_t N,
                        int64_t K, const float* scale_a, int a_per_row, const float* scale_b, float post_scale,
                        void* out, int out_dtype, int64_t ldo, int32_t* acc_out, int variant, void* workspace,
                        size_t workspace_bytes, void* hip_stream) {
  return gemm_i8_impl(A, lda, B, ldb, bits, M, N, K, scale_a, a_per_row, scale_b, post_scale, out, out_dtype,
                      ldo, acc_out, (hipStream_t)hip_stream, workspace, workspace_bytes, variant);
}

size_t hot_abc_workspace_bytes(int64_t L, int64_t I, const hot_config* cfg) {
  if (!cfg || L <= 0 || I <= 0) return colwise_workspace_bytes_impl(I > 0 ? I : 0);
  return hla_workspace_bytes_impl(L, I, cfg->hla_n, cfg->hla_r);
}

int hot_abc_forward(const void* x, int dtype, int64_t L, int64_t I, const hot_config* cfg, void* xq_out,
                    float* sx_out, void* workspace, size_t workspace_bytes, void* hip_stream) {
  if (int e = check_cfg(cfg, "hot_abc_forward")) return e;
  if (L <= 0 || I <= 0 || L % cfg->hla_n) return fail(HOT_ERR_INVALID, "hot_abc_forward: L=%lld must be a positive multiple of hla_n=%d", (long long)L, cfg->hla_n);
  if (cfg->act_scale == HOT_SCALE_ROW) return fail(HOT_ERR_UNSUPPORTED, "hot_abc_forward: the activation buffer uses one step per tensor");
  const int64_t lp = (L / cfg->hla_n) * cfg->hla_r;
  return colwise_quant_impl(x, dtype, L, I, cfg->hla_n, cfg_rows(cfg), cfg->hla_r, cfg->act_bits, cfg->act_round,
                            cfg->seed, HOT_STREAM_ACT, cfg->act_scale, xq_out, round_up(lp, GEMM_KTILE), 0,
                            sx_out, workspace, workspace_bytes, (hipStream_t)hip_stream, "hot_abc_forward");
}

size_t hot_backward_workspace_bytes(int64_t L, int64_t O, int64_t I, const hot_config* cfg) {
  if (check_cfg(cfg, "hot_backward_workspace_bytes") || L <= 0 || O <= 0 || I <= 0) return 0;
  return bwd_layout(L, O, I, cfg).total;
}

// Slots of the per-kernel timing of one backward (hot_linear_backward_kernels).
enum {
  K_CLEAR = 0,      // statistics cleared
  K_GY_STATS = 1,   // token-wise statistics pass over g_y (also the row-wise absmax when fused)
  K_GY_HLA = 2,     // token-wise quantise pass over g_y  -> g_W operand
  K_GY_HQ = 3,      // row-wise pass(es) over g_y          -> g_x operand
  K_W_STATS = 4,    // statistics pass over W
  K_W_QUANT = 5,    // quantise pass over W
  K_GEMM_GX = 6,
  K_GEMM_GW = 7,
  K_COUNT = 8
};
// Slots of the stage timing (hot_linear_backward with times4)
enum { STAGE_STATS = 0, STAGE_QUANT = 1, STAGE_GEMM = 2, STAGE_COUNT = 3 };

// The side stream of the g_x product.  One per device with its two events, created on first use (default
// priority) and kept for the life of the process; a mutex keeps the fork / join of one call together.
struct SideLane {
  hipStream_t stream = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  bool tried = false, ok = false;
};
static std::mutex g_side_mutex;
static SideLane g_side[64];

static SideLane* side_lane_locked() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  SideLane& s = g_side[dev];
  if (!s.tried) {
    s.tried = true;
    s.ok = hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) == hipSuccess &&
           hipEventCreateWithFlags(&s.fork, hipEventDisableTiming) == hipSuccess &&
           hipEventCreateWithFlags(&s.join, hipEventDisableTiming) == hipSuccess;
    if (!s.ok) (void)hipGetLastError();
  }
  return s.ok ? &s : nullptr;
}

// Events recorded along a timed call: event i + 1 follows the i-th group of launches, slot_of[i] names the group.
struct Marks {
  hipEvent_t* ev;
  int* slot_of;
  bool split;        // one group per kernel (every job launched on its own) instead of one per stage
  int seq = 0;
};

// The fewest workgroups of a column-wise job (col_jobs_want) from those of all jobs of the quantise phase: W's, g_y's along the tokens,
// and as many as g_y's row-wise quantiser takes by itself, which stand for it also where another kernel or another launch has it.
static int64_t flat_want(int64_t L, int64_t O, int64_t I, const hot_config* c, int dtype) {
  const int elem = dtype == HOT_F32 ? 4 : 2;
  const int64_t w = col_job_workgroups(O, I, c->n_o, c->n_o, c->w_bits == 4, c->w_scale, elem);
  const int64_t g = c->hla_n > COL_MAX_N ? 0 : col_job_workgroups(L, O, c->hla_n, c->hla_r, 0, c->gw_scale, elem);
  return col_jobs_want(w + g + L * O / (256 * HQ_UNROLL * EPL));
}

// g_y along the tokens, in blocks of up to 128: of a call, and of one with steps per sample.
static int flat_gy_job(ColJob& job, const void* gy, int dtype, int64_t L, int64_t O, const hot_config* c, const BwdLayout& b, uint8_t* ws,
                       int64_t want, bool bias, const char* who) {
  return col_job_impl(job, gy, dtype, L, O, c->hla_n, cfg_rows(c), c->hla_r, c->gw_bits, c->gw_round, c->seed, HOT_STREAM_GW, c->gw_scale,
                      ws + b.off_qgp, b.ld_gp, 0, (float*)(ws + b.off_sgp), ws + b.off_colg, colwise_workspace_bytes_impl(O), who,
                      1, 0, false, false, want, bias);
}

static int run_backward(const void* gy, const void* w, int dtype, const void* xq, const float* sx, int64_t L,
                        int64_t O, int64_t I, const hot_config* cfg, void* gx, void* gw, int out_dtype,
                        void* workspace, size_t workspace_bytes, Marks* marks, hipStream_t st,
                        void* gb = nullptr /* [O] of out_dtype: column sums of g_y, or null */) {
  const char* who = "hot_linear_backward";
  if (int e = check_cfg(cfg, who)) return e;
  if (!gy || !w || !xq || !sx || !gx || !gw) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
  if (L <= 0 || O <= 0 || I <= 0) return fail(HOT_ERR_INVALID, "%s: bad shape L=%lld O=%lld I=%lld", who, (long long)L, (long long)O, (long long)I);
  if (O % cfg->n_o) return fail(HOT_ERR_INVALID, "%s: O=%lld is not a multiple of n_o=%d", who, (long long)O, cfg->n_o);
  if (L % cfg->hla_n) return fail(HOT_ERR_INVALID, "%s: L=%lld is not a multiple of hla_n=%d", who, (long long)L, cfg->hla_n);
  if (cfg->gx_bits != cfg->w_bits) return fail(HOT_ERR_UNSUPPORTED, "%s: gx_bits (%d) and w_bits (%d) must match", who, cfg->gx_bits, cfg->w_bits);
  if (cfg->gx_scale == HOT_SCALE_SAWB) return fail(HOT_ERR_UNSUPPORTED, "%s: SAWB applies to W and x only", who);
  if (cfg->w_scale == HOT_SCALE_ROW) return fail(HOT_ERR_UNSUPPORTED, "%s: W uses one step per tensor", who);
  if (cfg->gw_scale == HOT_SCALE_SAWB) return fail(HOT_ERR_UNSUPPORTED, "%s: SAWB applies to W and x only", who);
  // limits of the stages, checked here so that nothing has been launched when one of them refuses
  if (int e = check_gx_modes(cfg, out_dtype, who)) return e;
  if (O % 8 || I % 8) return fail(HOT_ERR_UNSUPPORTED, "%s: O=%lld and I=%lld must be multiples of 8", who, (long long)O, (long long)I);
  if (O * I * 4 >= (1ll << 32)) return fail(HOT_ERR_UNSUPPORTED, "%s: W of %lld x %lld elements exceeds the 32-bit offsets of the loader", who, (long long)O, (long long)I);
  if (cfg->hla_n <= COL_MAX_N && L * O * 4 >= (1ll << 32)) return fail(HOT_ERR_UNSUPPORTED, "%s: g_y of %lld x %lld elements exceeds the 32-bit offsets of the loader", who, (long long)L, (long long)O);
  if (L >= (1ll << 31)) return fail(HOT_ERR_UNSUPPORTED, "%s: L too large", who);
  if (((uintptr_t)gy & 15) || ((uintptr_t)w & 15) || ((uintptr_t)xq & 15)) return fail(HOT_ERR_INVALID, "%s: gy, w and xq must be 16-byte aligned", who);
  const BwdLayout b = bwd_layout(L, O, I, cfg);
  if (!workspace || workspace_bytes < b.total) return fail(HOT_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, b.total, workspace_bytes);
  if ((uintptr_t)workspace & 255) return fail(HOT_ERR_INVALID, "%s: workspace must be 256-byte aligned", who);
  uint8_t* ws = (uint8_t*)workspace;
  float* sg = (float*)(ws + b.off_sg);
  float* sw = (float*)(ws + b.off_sw);
  float* sgp = (float*)(ws + b.off_sgp);
  if (marks) (void)hipEventRecord(marks->ev[0], st);
  auto mark = [&](int slot) {
    if (!marks) return;
    marks->slot_of[marks->seq] = slot;
    (void)hipEventRecord(marks->ev[++marks->seq], st);
  };
  const bool split = marks && marks->split;
  int rc;
  // The jobs.  g_y: HLA along tokens + quantise, transposed (g_W operand); Hadamard along O + quantise (g_x operand).
  // W: Hadamard along O + quantise, stored [I, O].  Blocks of up to 128 tokens and Hadamard blocks of up to 16 share
  // the launches of the two phases (phase.h); larger ones have kernels of their own.
  const bool big = cfg->hla_n > COL_MAX_N, w_short = w_joins_phase(cfg);
  ColJob gj, wj;
  const int64_t want = flat_want(L, O, I, cfg, dtype);
  rc = col_job_impl(wj, w, dtype, O, I, cfg->n_o, identity_rows(), cfg->n_o, cfg->w_bits, cfg->w_round, cfg->seed, HOT_STREAM_W,
                    cfg->w_scale, ws + b.off_qw, b.ld_w, cfg->w_bits == 4, sw, ws + b.off_colw, colwise_workspace_bytes_impl(I), who,
                    1, 0, false, w_short, want);
  if (rc) return rc;
  // With one step per tensor both quantisers of g_y need the absmax of their transform first: the statistics pass of
  // the token-wise job delivers both from a single read of g_y.
  const bool row_tensor = cfg->gx_scale == HOT_SCALE_TENSOR;
  const bool hq_job = cfg->n_o <= CW_ROWS && (row_tensor ? (!big || (cfg->n_o == 16 && O % 16 == 0)) : O <= HQ_ROW_MAX_K);
  const bool row_fused = hq_job && row_tensor;
  float* const slots = (float*)(ws + b.off_hq);
  if (!big) {
    rc = flat_gy_job(gj, gy, dtype, L, O, cfg, b, ws, want, gb != nullptr, who);
    if (rc) return rc;
    if (row_fused) col_job_row_stat(gj, cfg->n_o);
    if (gb) gj.a.colsum = (float*)(ws + b.off_colsum);
  }
  HqArgs hj;
  if (hq_job) {
    const float* stat = !row_tensor ? nullptr : big ? slots : gj.a.row_absmax;
    rc = hq_job_impl(hj, gy, L, O, cfg->n_o, cfg->gx_bits, cfg->gx_round, cfg->seed, HOT_STREAM_GX, cfg->gx_scale, ws + b.off_qg, b.ld_g, sg,
                     stat, big ? 1 : row_tensor ? gj.a.npart : 0, 1, 1);
    if (rc) return rc;
  }
  ColsumArgs sj;
  if (gb) {
    const int64_t strips = big ? colsum_strips_impl(L, O, cfg->hla_n, cfg->hla_r, 0, cfg->gw_scale, dtype == HOT_F32 ? 4 : 2) : col_job_strips(gj);
    if (int e = colsum_args(sj, (const float*)(ws + b.off_colsum), O, strips, b.colsum_strips, gb, out_dtype, who)) return e;
  }

  // statistics
  if (!big) col_job_clear(gj, st);
  if (split) mark(K_CLEAR);
  const bool w_joins = w_short && !split;
  if (!big) {
    rc = phase_launch(0, dtype, &gj, w_joins ? &wj : nullptr, nullptr, nullptr, st);
    if (rc) return rc;
    if (split) mark(K_GY_STATS);
  } else if (w_joins) {
    rc = phase_launch(0, dtype, nullptr, &wj, nullptr, nullptr, st);
    if (rc) return rc;
  }
  auto w_alone = [&](int pass) { return w_short ? phase_launch(pass, dtype, nullptr, &wj, nullptr, nullptr, st) : phase_launch(pass, dtype, &wj, nullptr, nullptr, nullptr, st); };
  if (!w_joins && (rc = w_alone(0))) return rc;
  if (split) mark(K_W_STATS);
  if (marks && !split) mark(STAGE_STATS);

  // transform + quantise
  if (big) {
    rc = colwise_quant_impl(gy, dtype, L, O, cfg->hla_n, cfg_rows(cfg), cfg->hla_r, cfg->gw_bits, cfg->gw_round, cfg->seed, HOT_STREAM_GW,
                            cfg->gw_scale, ws + b.off_qgp, b.ld_gp, 0, sgp, ws + b.off_colg,
                            hla_workspace_bytes_impl(L, O, cfg->hla_n, cfg->hla_r), st, who, row_fused ? slots : nullptr,
                            gb ? (float*)(ws + b.off_colsum) : nullptr);
    if (rc) return rc;
  }
  if (split) {
    if (!big && (rc = phase_launch(1, dtype, &gj, nullptr, nullptr, gb ? &sj : nullptr, st))) return rc;
    if (big && gb && (rc = colsum_finish_impl(sj, st))) return rc;
    mark(K_GY_HLA);
    if (hq_job && (rc = phase_launch(1, dtype, nullptr, nullptr, &hj, nullptr, st))) return rc;
  } else {
    rc = phase_launch(1, dtype, big ? nullptr : &gj, w_joins ? &wj : nullptr, hq_job ? &hj : nullptr, gb ? &sj : nullptr, st);
    if (rc) return rc;
  }
  if (!hq_job) {
    rc = hq_rowwise_impl(gy, dtype, L, O, cfg->n_o, cfg->gx_bits, cfg->gx_round, cfg->seed, HOT_STREAM_GX, cfg->gx_scale, ws + b.off_qg,
                         b.ld_g, sg, slots, STAT_SLOT_BYTES, st);
    if (rc) return rc;
  }
  if (split) mark(K_GY_HQ);
  if (!w_joins && (rc = w_alone(1))) return rc;
  if (split) mark(K_W_QUANT);
  if (marks && !split) mark(STAGE_QUANT);

  // the products
  GemmProduct px = gx_product(b, L, O, I, cfg), pw = gw_product(b, L, O, I, cfg);
  px.A = ws + b.off_qg; px.B = ws + b.off_qw; px.scale_a = sg; px.scale_b = sw; px.out = gx;
  pw.A = ws + b.off_qgp; pw.B = xq; pw.scale_a = sgp; pw.scale_b = sx; pw.out = gw;
  if (!split && pairs(pw, px, cfg)) {
    rc = gemm_pair_impl(pw, px, out_dtype, st);
    if (!rc && marks) mark(STAGE_GEMM);
    return rc;
  }
  auto run_gemm = [&](const GemmProduct& p, hipStream_t s2) {
    // (no split on the side stream: the split workspace belongs to the g_W product)
    return gemm_i8_impl(p, out_dtype, nullptr, s2, s2 == st && b.split_bytes ? ws + b.off_split : nullptr, s2 == st ? b.split_bytes : 0);
  };
  // Beside the g_W product when that has fewer tiles than the chip has CUs and cannot fill it alone (two large products
  // only get in each other's way), and only where the caller asks for it or an operand is too large for the paired kernel.  A
  // g_x product that could pair but is better off alone has few tiles and a long K: the fork is 10 us of GPU time and as much
  // of the host's that its neighbour does not cover, and the split workspace stays behind (us of the whole backward, INT8,
  // forked / one after the other: 3904 x 10496 x 384 113 / 101, 8128 x 9984 x 320 182 / 172, 4032 x 5120 x 640 82 / 69).
  std::unique_lock<std::mutex> side_guard(g_side_mutex, std::defer_lock);
  SideLane* side = nullptr;
  if (!marks && (cfg->streams == 2 || !gemm_pair_possible(pw, px)) && backward_streams(L, O, I, cfg) == 2 && ((O + 127) / 128) * ((I + 127) / 128) < 256) {
    side_guard.lock();
    side = side_lane_locked();
    if (!side) side_guard.unlock();
  }
  // Once the side stream has been forked, every way out of this function joins it again: the caller's stream waits
  // for what the side stream was given, also when a launch refuses, so that no kernel of the call still runs (on the
  // workspace) behind work the caller queues next, and a capture of the caller's stream is never left with an unjoined branch.
  struct SideJoin {
    SideLane* side = nullptr;
    hipStream_t st = nullptr;
    ~SideJoin() {
      if (!side) return;
      if (hipEventRecord(side->join, side->stream) == hipSuccess) (void)hipStreamWaitEvent(st, side->join, 0);
    }
  } side_join;
  if (side) {
    rc = check_hip(hipEventRecord(side->fork, st), "hipEventRecord");
    if (!rc) rc = check_hip(hipStreamWaitEvent(side->stream, side->fork, 0), "hipStreamWaitEvent");
    if (rc) return rc;
    side_join.side = side; side_join.st = st;
    rc = run_gemm(px, side->stream);
    if (rc) return rc;
  }
  rc = run_gemm(pw, st);
  if (rc) return rc;
  if (split) mark(K_GEMM_GW);
  if (!side && (rc = run_gemm(px, st))) return rc;
  if (split) mark(K_GEMM_GX);
  if (marks && !split) mark(STAGE_GEMM);
  return HOT_OK;
}

// Timing events, kept for the next timed call: a set is taken for the length of a call and put back after it.
struct EventSet { int dev; hipEvent_t ev[K_COUNT + 1]; };
static std::mutex g_event_mutex;
static std::vector<EventSet> g_event_sets;
constexpr size_t EVENT_SETS_KEPT = 16;

static int take_events(EventSet* out) {
  int dev = 0;
  if (int rc = check_hip(hipGetDevice(&dev), "hipGetDevice")) return rc;
  {
    std::lock_guard<std::mutex> lock(g_event_mutex);
    for (size_t i = 0; i < g_event_sets.size(); ++i)
      if (g_event_sets[i].dev == dev) {
        *out = g_event_sets[i];
        g_event_sets[i] = g_event_sets.back();
        g_event_sets.pop_back();
        return HOT_OK;
      }
  }
  out->dev = dev;
  for (int i = 0; i <= K_COUNT; ++i) {
    if (int rc = check_hip(hipEventCreate(&out->ev[i]), "hipEventCreate")) {
      while (i-- > 0) (void)hipEventDestroy(out->ev[i]);
      return rc;
    }
  }
  return HOT_OK;
}

static void put_events(const EventSet& s) {
  {
    std::lock_guard<std::mutex> lock(g_event_mutex);
    if (g_event_sets.size() < EVENT_SETS_KEPT) { g_event_sets.push_back(s); return; }
  }
  for (int i = 0; i <= K_COUNT; ++i) (void)hipEventDestroy(s.ev[i]);
}

// Runs the backward with an event after every group of launches (split: every kernel, else every stage) and returns
// the durations of the `slots` groups in seconds.
static int run_backward_timed(const void* gy, const void* w, int dtype, const void* xq, const float* sx, int64_t L,
                              int64_t O, int64_t I, const hot_config* cfg, void* gx, void* gw, int out_dtype,
                              void* workspace, size_t workspace_bytes, bool split, float* secs, int slots, hipStream_t st) {
  EventSet set;
  int slot_of[K_COUNT];
  for (int i = 0; i < slots; ++i) secs[i] = 0.f;
  if (int rc = take_events(&set)) return rc;
  Marks marks{set.ev, slot_of, split};
  int rc = run_backward(gy, w, dtype, xq, sx, L, O, I, cfg, gx, gw, out_dtype, workspace, workspace_bytes, &marks, st);
  if (!rc) rc = check_hip(hipEventSynchronize(set.ev[marks.seq]), "hipEventSynchronize");
  if (!rc) {
    for (int i = 0; i < marks.seq; ++i) {
      float ms = 0.f;
      (void)hipEventElapsedTime(&ms, set.ev[i], set.ev[i + 1]);
      secs[slot_of[i]] += ms * 1e-3f;
    }
  }
  put_events(set);
  return rc;
}

int hot_linear_backward(const void* gy, const void* w, int dtype, const void* xq, const float* sx, int64_t L,
                        int64_t O, int64_t I, const hot_config* cfg, void* gx, void* gw, int out_dtype,
                        void* workspace, size_t workspace_bytes, float* times4, void* hip_stream) {
  if (!times4)
    return run_backward(gy, w, dtype, xq, sx, L, O, I, cfg, gx, gw, out_dtype, workspace, workspace_bytes, nullptr,
                        (hipStream_t)hip_stream);
  // the reference op returns {fwht, quant, gemm, dequant} (HLQ_backward_kernel.cu:729-733): here the launches that
  // only measure, those that transform and quantise (with blocks above 128 tokens these hold g_y's statistics too), both
  // products, and 0 for the dequantisation, which is the products' epilogue
  const int rc = run_backward_timed(gy, w, dtype, xq, sx, L, O, I, cfg, gx, gw, out_dtype, workspace, workspace_bytes,
                                    false, times4, STAGE_COUNT, (hipStream_t)hip_stream);
  times4[3] = 0.f;
  return rc;
}

int hot_linear_backward_bias(const void* gy, const void* w, int dtype, const void* xq, const float* sx, int64_t L,
                             int64_t O, int64_t I, const hot_config* cfg, void* gx, void* gw, void* gb, int out_dtype,
                             void* workspace, size_t workspace_bytes, void* hip_stream) {
  if (!gb) return fail(HOT_ERR_INVALID, "hot_linear_backward_bias: null pointer");
  return run_backward(gy, w, dtype, xq, sx, L, O, I, cfg, gx, gw, out_dtype, workspace, workspace_bytes, nullptr,
                      (hipStream_t)hip_stream, gb);
}

// ---- g_x through a low-rank projection along the tokens ---------------------------------------------
// transform_scheme "low_rank" and "gilr_gwh" (utils/quant_matmul.py:229-233, 263-266, 288-290, 334-337):
// g_x = P^T ( q(P g_y) . q(W) ) s_g s_w / n, W untransformed.  The token-wise kernels store q(P g_y)
// untransposed ([L', O], K along the channels), W goes through the column-wise kernel with blocks of
// one row (quantise + transpose), the product lands in fp32 in the workspace and the expansion pass
// takes it back to L tokens.  Kept for completeness of the reference's scheme list: four kernels on
// one stream, not tuned.  The g_W side of those schemes is the g_W side of "gih_gwlr" / "hadamard".

struct LowrankLayout {
  int64_t lp, ld_g, ld_w;
  size_t off_colg, off_colw, off_sg, off_sw, off_qg, off_qw, off_t, off_exp, off_proj, colg_bytes, exp_bytes, total;
};

static LowrankLayout lowrank_layout(int64_t L, int64_t O, int64_t I, const hot_config* c) {
  LowrankLayout b;
  b.lp = (L / c->hla_n) * c->hla_r;
  b.ld_g = round_up(O, GEMM_KTILE) * c->gx_bits / 8;
  b.ld_w = round_up(O, GEMM_KTILE) * c->w_bits / 8;
  size_t o = 0;
  // blocks above 128 tokens: the two-level token-wise path and the two-pass expansion, each with an
  // fp32 intermediate of the tensor's size in the workspace
  b.colg_bytes = hla_workspace_bytes_impl(L, O, c->hla_n, c->hla_r);
  b.exp_bytes = c->hla_n > 128 ? hla_expand_big_workspace_bytes_impl(L / c->hla_n, I, c->hla_n) : 0;
  b.off_colg = o; o += align256(b.colg_bytes);
  b.off_colw = o; o += align256(colwise_workspace_bytes_impl(I));
  // a step per coefficient row (gx_scale ROW): lp steps, and the unquantised projection [L', O] in fp32
  const bool per_row = c->gx_scale == HOT_SCALE_ROW;
  b.off_sg = o;   o += per_row ? align256((size_t)b.lp * 4) : 256;
  b.off_sw = o;   o += 256;
  b.off_qg = o;   o += align256((size_t)b.lp * b.ld_g);
  b.off_qw = o;   o += align256((size_t)I * b.ld_w);
  b.off_t = o;    o += align256((size_t)b.lp * (size_t)I * 4);
  b.off_exp = o;  o += align256(b.exp_bytes);
  b.off_proj = o; o += per_row ? align256((size_t)b.lp * (size_t)O * 4) : 0;
  b.total = o;
  return b;
}

static int check_lowrank(const hot_config* cfg, int64_t L, int64_t O, int64_t I, const char* who) {
  if (int e = check_cfg(cfg, who)) return e;
  if (L <= 0 || O <= 0 || I <= 0 || O % 8 || I % 8) return fail(HOT_ERR_INVALID, "%s: L=%lld, O=%lld and I=%lld must be positive, O and I multiples of 8", who, (long long)L, (long long)O, (long long)I);
  if (L % cfg->hla_n) return fail(HOT_ERR_INVALID, "%s: L=%lld is not a multiple of hla_n=%d", who, (long long)L, cfg->hla_n);
  if (cfg->gx_bits != cfg->w_bits) return fail(HOT_ERR_UNSUPPORTED, "%s: gx_bits (%d) and w_bits (%d) must match", who, cfg->gx_bits, cfg->w_bits);
  if (cfg->gx_scale == HOT_SCALE_SAWB) return fail(HOT_ERR_UNSUPPORTED, "%s: the projected g_y takes absmax steps (one for the tensor or one per coefficient row)", who);
  if (cfg->gx_scale == HOT_SCALE_ROW && cfg->hla_n > 128) return fail(HOT_ERR_UNSUPPORTED, "%s: a step per coefficient row takes token blocks up to 128", who);
  if (cfg->w_scale == HOT_SCALE_ROW) return fail(HOT_ERR_UNSUPPORTED, "%s: W uses one step per tensor", who);
  return HOT_OK;
}

size_t hot_gx_lowrank_workspace_bytes(int64_t L, int64_t O, int64_t I, const hot_config* cfg) {
  if (check_lowrank(cfg, L, O, I, "hot_gx_lowrank_workspace_bytes")) return 0;
  return lowrank_layout(L, O, I, cfg).total;
}

int hot_gx_lowrank(const void* gy, const void* w, int dtype, int64_t L, int64_t O, int64_t I, const hot_config* cfg,
                   void* gx, int out_dtype, void* workspace, size_t workspace_bytes, void* hip_stream) {
  const char* who = "hot_gx_lowrank";
  if (int e = check_lowrank(cfg, L, O, I, who)) return e;
  if (!gy || !w || !gx) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
  if (L * O * 4 >= (1ll << 32) || O * I * 4 >= (1ll << 32)) return fail(HOT_ERR_UNSUPPORTED, "%s: tensors exceed the 32-bit offsets of the loader", who);
  const LowrankLayout b = lowrank_layout(L, O, I, cfg);
  if (!workspace || workspace_bytes < b.total) return fail(HOT_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, b.total, workspace_bytes);
  if ((uintptr_t)workspace & 255) return fail(HOT_ERR_INVALID, "%s: workspace must be 256-byte aligned", who);
  hipStream_t st = (hipStream_t)hip_stream;
  uint8_t* ws = (uint8_t*)workspace;
  float* sg = (float*)(ws + b.off_sg);
  float* sw = (float*)(ws + b.off_sw);
  const int bits = cfg->gx_bits;
  // q(P g_y), untransposed [L', O]; the K padding of every row is cleared apart
  int rc;
  const bool per_row = cfg->gx_scale == HOT_SCALE_ROW;
  if (per_row) {
    // a step per coefficient row (norm_quantizer on [L', O], utils/quant_matmul.py:19-37,244-255): the
    // projection unquantised in fp32, then the row-wise quantiser without a transform (elements numbered
    // row-major for stochastic rounding)
    float* proj = (float*)(ws + b.off_proj);
    rc = hla_project_impl(gy, dtype, L, O, cfg->hla_n, cfg_rows(cfg), cfg->hla_r, proj, O, st, true);
    if (!rc) rc = hq_rowwise_impl(proj, HOT_F32, b.lp, O, 1, bits, cfg->gx_round, cfg->seed, HOT_STREAM_GX, HOT_SCALE_ROW,
                                  ws + b.off_qg, b.ld_g, sg, nullptr, 0, st);
  } else {
    rc = colwise_quant_impl(gy, dtype, L, O, cfg->hla_n, cfg_rows(cfg), cfg->hla_r, bits, cfg->gx_round, cfg->seed,
                            HOT_STREAM_GX, HOT_SCALE_TENSOR, ws + b.off_qg, b.ld_g, bits == 4, sg, ws + b.off_colg,
                            b.colg_bytes, st, who, nullptr, nullptr, 1, 0, true);
  }
  if (rc) return rc;
  zero_pad_impl(ws + b.off_qg, b.lp, O * bits / 8, b.ld_g, st);
  // q(W), stored [I, O]: blocks of one row, nothing transformed
  rc = colwise_quant_impl(w, dtype, O, I, 1, identity_rows(), 1, cfg->w_bits, cfg->w_round, cfg->seed, HOT_STREAM_W,
                          cfg->w_scale, ws + b.off_qw, b.ld_w, cfg->w_bits == 4, sw, ws + b.off_colw,
                          colwise_workspace_bytes_impl(I), st, who);
  if (rc) return rc;
  float* t = (float*)(ws + b.off_t);
  rc = gemm_i8_impl(ws + b.off_qg, b.ld_g, ws + b.off_qw, b.ld_w, bits, b.lp, I, O, sg, per_row ? 1 : 0, sw, 1.0f, t, HOT_F32, I, nullptr, st);
  if (rc) return rc;
  if (cfg->hla_n > 128)
    return hla_expand_big_impl(t, L / cfg->hla_n, I, cfg->hla_n, cfg_rows(cfg), cfg->hla_r, 1.0f / (float)cfg->hla_n, gx,
                               out_dtype, ws + b.off_exp, b.exp_bytes, st);
  return hla_expand_impl(t, L / cfg->hla_n, I, cfg->hla_n, cfg_rows(cfg), cfg->hla_r, 1.0f / (float)cfg->hla_n, gx, out_dtype, st);
}

// ---- g_x with the logarithmic quantiser on g_y -----------------------------------------------------
// quantBWDGogi = "luq" (utils/quant_matmul.py:238,252-253,270,276-285,288-290,343): g_y blkdiag(H) through
// luq_quantizer_BWD, blkdiag(H) W through the weight quantiser, their integer product, the two steps,
// / n_o.  The LUQ codes are powers of two up to 2^(lev + 1) and travel as two INT8 planes (q = 16 a + b);
// W's INT4-range codes are stored as bytes and doubled into [16 w | w]; one INT8 product over twice the K.

struct LuqLayout {
  int64_t kp;
  size_t off_colw, off_slots, off_sg, off_sw, off_qg, off_qw, off_qw2, total;
};

static LuqLayout luq_layout(int64_t L, int64_t O, int64_t I) {
  LuqLayout b;
  b.kp = round_up(O, GEMM_KTILE);
  size_t o = 0;
  b.off_colw = o;  o += align256(colwise_workspace_bytes_impl(I));
  b.off_slots = o; o += STAT_SLOT_BYTES;
  b.off_sg = o;    o += 256;
  b.off_sw = o;    o += 256;
  b.off_qg = o;    o += align256((size_t)L * 2 * b.kp);
  b.off_qw = o;    o += align256((size_t)I * b.kp);
  b.off_qw2 = o;   o += align256((size_t)I * 2 * b.kp);
  b.total = o;
  return b;
}

static int check_luq(const hot_config* cfg, int64_t L, int64_t O, int64_t I, const char* who) {
  if (int e = check_cfg(cfg, who)) return e;
  if (L <= 0 || O <= 0 || I <= 0 || O % 8 || I % 8) return fail(HOT_ERR_INVALID, "%s: L=%lld, O=%lld and I=%lld must be positive, O and I multiples of 8", who, (long long)L, (long long)O, (long long)I);
  if (O % cfg->n_o) return fail(HOT_ERR_INVALID, "%s: O=%lld is not a multiple of n_o=%d", who, (long long)O, cfg->n_o);
  if (cfg->gx_bits != 4 || cfg->w_bits != 4) return fail(HOT_ERR_UNSUPPORTED, "%s: the logarithmic quantiser runs at 4 bits against 4-bit weights", who);
  if (cfg->w_scale == HOT_SCALE_ROW) return fail(HOT_ERR_UNSUPPORTED, "%s: W uses one step per tensor", who);
  return HOT_OK;
}

size_t hot_gx_luq_workspace_bytes(int64_t L, int64_t O, int64_t I, const hot_config* cfg) {
  if (check_luq(cfg, L, O, I, "hot_gx_luq_workspace_bytes")) return 0;
  return luq_layout(L, O, I).total;
}

int hot_gx_luq(const void* gy, const void* w, int dtype, int64_t L, int64_t O, int64_t I, const hot_config* cfg,
               void* gx, int out_dtype, void* workspace, size_t workspace_bytes, void* hip_stream) {
  const char* who = "hot_gx_luq";
  if (int e = check_luq(cfg, L, O, I, who)) return e;
  if (!gy || !w || !gx) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
  if (O * I * 4 >= (1ll << 32)) return fail(HOT_ERR_UNSUPPORTED, "%s: W exceeds the 32-bit offsets of the loader", who);
  const LuqLayout b = luq_layout(L, O, I);
  if (!workspace || workspace_bytes < b.total) return fail(HOT_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, b.total, workspace_bytes);
  if ((uintptr_t)workspace & 255) return fail(HOT_ERR_INVALID, "%s: workspace must be 256-byte aligned", who);
  hipStream_t st = (hipStream_t)hip_stream;
  uint8_t* ws = (uint8_t*)workspace;
  float* sg = (float*)(ws + b.off_sg);
  float* sw = (float*)(ws + b.off_sw);
  // W: Hadamard along O + 4-bit quantiser, codes kept one per byte, stored [I, kp]; then [16 w | w]
  int rc = colwise_quant_impl(w, dtype, O, I, cfg->n_o, identity_rows(), cfg->n_o, cfg->w_bits, cfg->w_round, cfg->seed,
                              HOT_STREAM_W, cfg->w_scale, ws + b.off_qw, b.kp, 0, sw, ws + b.off_colw,
                              colwise_workspace_bytes_impl(I), st, who);
  if (rc) return rc;
  rc = luq_pair_impl(ws + b.off_qw, I, b.kp, ws + b.off_qw2, st);
  if (rc) return rc;
  rc = hq_luq_impl(gy, dtype, L, O, cfg->n_o, cfg->gx_bits, cfg->seed, ws + b.off_qg, b.kp, sg, ws + b.off_slots,
                   STAT_SLOT_BYTES, st);
  if (rc) return rc;
  return gemm_i8_impl(ws + b.off_qg, 2 * b.kp, ws + b.off_qw2, 2 * b.kp, 8, L, I, 2 * b.kp, sg, 0, sw,
                      1.0f / (float)cfg->n_o, gx, out_dtype, I, nullptr, st);
}

// ---- g_W with the logarithmic quantiser on the projected g_y ------------------------------------------
// quantBWDGogw = "luq", or luq_quantizer picked for a layer's g_W under quantAuto (utils/quant_matmul.py:
// 296-301, 307-314, 322-324): g_W = (luq((P g_y)^T) . q(P x)) s s_x / n.  The projection is computed
// unquantised in fp32 ([O, L'], rows padded with zeros to a multiple of 8: a zero draws code 0), the
// quantiser runs on its rows (element e = o K8 + k draws the uniforms 2 e, 2 e + 1 of stream 5), and the
// two planes of the codes (q = 16 a + b) meet the INT8 activation buffer in two products whose integer
// sums a last kernel combines: 16 acc_a + acc_b is the exact sum of q x.  Kept for completeness.

struct GwLuqLayout {
  int64_t lp, k8, kp;
  size_t off_slots, off_sg, off_proj, off_codes, off_acca, off_accb, total;
};

static GwLuqLayout gw_luq_layout(int64_t L, int64_t O, int64_t I, const hot_config* c) {
  GwLuqLayout b;
  b.lp = (L / c->hla_n) * c->hla_r;
  b.k8 = round_up(b.lp, 8);
  b.kp = round_up(b.lp, GEMM_KTILE);
  size_t o = 0;
  b.off_slots = o; o += STAT_SLOT_BYTES;
  b.off_sg = o;    o += 256;
  b.off_proj = o;  o += align256((size_t)O * b.k8 * 4);
  b.off_codes = o; o += align256((size_t)O * 2 * b.kp);
  b.off_acca = o;  o += align256((size_t)O * I * 4);
  b.off_accb = o;  o += align256((size_t)O * I * 4);
  b.total = o;
  return b;
}

static int check_gw_luq(const hot_config* cfg, int64_t L, int64_t O, int64_t I, const char* who) {
  if (int e = check_cfg(cfg, who)) return e;
  if (L <= 0 || O <= 0 || I <= 0 || I % 8) return fail(HOT_ERR_INVALID, "%s: L=%lld, O=%lld and I=%lld must be positive, I a multiple of 8", who, (long long)L, (long long)O, (long long)I);
  if (cfg->hla_n > 128) return fail(HOT_ERR_UNSUPPORTED, "%s: token blocks up to 128 (the projection pass holds a block per thread)", who);
  if (L % cfg->hla_n) return fail(HOT_ERR_INVALID, "%s: L=%lld is not a multiple of hla_n=%d", who, (long long)L, cfg->hla_n);
  if (cfg->gw_bits != 4) return fail(HOT_ERR_UNSUPPORTED, "%s: the logarithmic quantiser runs at 4 bits (gw_bits)", who);
  if ((L / cfg->hla_n) * cfg->hla_r > 16384) return fail(HOT_ERR_UNSUPPORTED, "%s: more than 16384 coefficients per channel overflow the int32 sums", who);
  return HOT_OK;
}

size_t hot_gw_luq_workspace_bytes(int64_t L, int64_t O, int64_t I, const hot_config* cfg) {
  if (check_gw_luq(cfg, L, O, I, "hot_gw_luq_workspace_bytes")) return 0;
  return gw_luq_layout(L, O, I, cfg).total;
}

int hot_gw_luq(const void* gy, int dtype, const void* xq, const float* sx, int64_t L, int64_t O, int64_t I,
               const hot_config* cfg, void* gw, int out_dtype, void* workspace, size_t workspace_bytes, void* hip_stream) {
  const char* who = "hot_gw_luq";
  if (int e = check_gw_luq(cfg, L, O, I, who)) return e;
  if (!gy || !xq || !sx || !gw) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
  const GwLuqLayout b = gw_luq_layout(L, O, I, cfg);
  if (!workspace || workspace_bytes < b.total) return fail(HOT_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, b.total, workspace_bytes);
  if ((uintptr_t)workspace & 255) return fail(HOT_ERR_INVALID, "%s: workspace must be 256-byte aligned", who);
  hipStream_t st = (hipStream_t)hip_stream;
  uint8_t* ws = (uint8_t*)workspace;
  float* sg = (float*)(ws + b.off_sg);
  float* proj = (float*)(ws + b.off_proj);
  int8_t* codes = (int8_t*)(ws + b.off_codes);
  int32_t* acc_a = (int32_t*)(ws + b.off_acca);
  int32_t* acc_b = (int32_t*)(ws + b.off_accb);
  int rc = hla_project_impl(gy, dtype, L, O, cfg->hla_n, cfg_rows(cfg), cfg->hla_r, proj, b.k8, st);
  if (rc) return rc;
  rc = hq_luq_impl(proj, HOT_F32, O, b.k8, 1, cfg->gw_bits, cfg->seed, codes, b.kp, sg, ws + b.off_slots, STAT_SLOT_BYTES, st,
                   HOT_STREAM_LUQ_GW);
  if (rc) return rc;
  const float post = 1.0f / (float)cfg->hla_n;
  rc = gemm_i8_impl(codes, 2 * b.kp, xq, b.kp, 8, O, I, b.lp, sg, 0, sx, post, gw, out_dtype, I, acc_a, st);
  if (rc) return rc;
  rc = gemm_i8_impl(codes + b.kp, 2 * b.kp, xq, b.kp, 8, O, I, b.lp, sg, 0, sx, post, gw, out_dtype, I, acc_b, st);
  if (rc) return rc;
  return luq_combine_impl(acc_a, acc_b, O, I, sg, sx, post, gw, out_dtype, st);
}

// ---- 3-D activations: one set of steps per sample --------------------------------------------------
// The reference vmaps its quantisers over the batch dimension of [B, T, C] tensors
// (utils/quant_matmul.py:33-37,102-106,118-122), applies the token-wise transform inside each sample
// (utils/hadamard_matmul.py:143-161, 3-D branch) and returns one weight gradient per sample, which
// autograd sums (utils/quant_matmul.py:288-290,322-324).  Here the B samples are the rows [b T, (b+1) T)
// of the flattened tensors; the codes of sample b occupy K range [b kg, (b+1) kg) of the g_W operands,
// kg = hot_kpad_group(T') = T' rounded up to 128 codes, and the g_W product dequantises every sample's
// integer sums with that sample's steps before adding them up in fp32, in sample order.

struct BatchedLayout {
  int64_t ld_g, ld_w, kg, ld_gp;
  int64_t colsum_strips;                         // as in BwdLayout
  size_t off_colw, off_colg, off_hq, off_sg, off_sw, off_sgp, off_qg, off_qw, off_qgp, off_part, part_bytes, off_colsum, total;
};

static int64_t kpad_group(int64_t T, const hot_config* c) { return round_up((T / c->hla_n) * c->hla_r, 128); }

static BatchedLayout batched_layout(int64_t B, int64_t T, int64_t O, int64_t I, const hot_config* c) {
  BatchedLayout b;
  const int64_t L = B * T;
  b.ld_g = round_up(O, GEMM_KTILE) * c->gx_bits / 8;
  b.ld_w = round_up(O, GEMM_KTILE) * c->w_bits / 8;
  b.kg = kpad_group(T, c);
  b.ld_gp = B * b.kg;
  size_t o = 0;
  b.off_colw = o; o += align256(colwise_workspace_bytes_impl(I));
  b.off_colg = o; o += align256(colwise_group_workspace_bytes_impl(O, (int)B));
  b.off_hq = o;   o += align256((size_t)B * 128 > STAT_SLOT_BYTES ? (size_t)B * 128 : STAT_SLOT_BYTES);
  b.off_sg = o;   o += align256((size_t)L * 4);
  b.off_sw = o;   o += 256;
  b.off_sgp = o;  o += align256((size_t)B * (size_t)O * 4);
  b.off_qg = o;   o += align256((size_t)L * b.ld_g);
  b.off_qw = o;   o += align256((size_t)I * b.ld_w);
  b.off_qgp = o;  o += align256((size_t)O * b.ld_gp);
  b.part_bytes = gemm_grouped_workspace_bytes_impl(O, I, (int)B, b.kg);
  b.off_part = o; o += align256(b.part_bytes);
  // partial column sums of g_y (bias gradient); the query knows no input type: room for either element size
  const int64_t s2 = colsum_strips_impl(L, O, c->hla_n, c->hla_r, 0, c->gw_scale, 2, B);
  const int64_t s4 = colsum_strips_impl(L, O, c->hla_n, c->hla_r, 0, c->gw_scale, 4, B);
  b.colsum_strips = s2 > s4 ? s2 : s4;
  b.off_colsum = o; o += align256((size_t)b.colsum_strips * (size_t)O * 4);
  b.total = o;
  return b;
}

static int check_batched(const hot_config* cfg, int64_t B, int64_t T, const char* who) {
  if (int e = check_cfg(cfg, who)) return e;
  if (B < 1 || B > 65535 || T < 1) return fail(HOT_ERR_INVALID, "%s: bad batch %lld x %lld tokens", who, (long long)B, (long long)T);
  if (cfg->hla_n > COL_MAX_N) return fail(HOT_ERR_UNSUPPORTED, "%s: token blocks up to %d inside a sample", who, COL_MAX_N);
  if (T % cfg->hla_n) return fail(HOT_ERR_INVALID, "%s: T=%lld is not a multiple of hla_n=%d", who, (long long)T, cfg->hla_n);
  return HOT_OK;
}

int64_t hot_kpad_group(int64_t T, const hot_config* cfg) {
  if (!cfg || cfg->hla_n < 1 || T < 1) return 0;
  return kpad_group(T, cfg);
}

size_t hot_abc_batched_workspace_bytes(int64_t B, int64_t T, int64_t I, const hot_config* cfg) {
  (void)T; (void)cfg;
  return colwise_group_workspace_bytes_impl(I > 0 ? I : 0, B > 0 ? (int)B : 1);
}

int hot_abc_forward_batched(const void* x, int dtype, int64_t B, int64_t T, int64_t I, const hot_config* cfg,
                            void* xq_out, float* sx_out, void* workspace, size_t workspace_bytes, void* hip_stream) {
  const char* who = "hot_abc_forward_batched";
  if (int e = check_batched(cfg, B, T, who)) return e;
  if (I <= 0) return fail(HOT_ERR_INVALID, "%s: bad shape I=%lld", who, (long long)I);
  if (cfg->act_scale == HOT_SCALE_ROW) return fail(HOT_ERR_UNSUPPORTED, "%s: the activation buffer uses one step per sample", who);
  const int64_t kg = kpad_group(T, cfg);
  return colwise_quant_impl(x, dtype, B * T, I, cfg->hla_n, cfg_rows(cfg), cfg->hla_r, cfg->act_bits, cfg->act_round, cfg->seed,
                            HOT_STREAM_ACT, cfg->act_scale, xq_out, B * kg, 0, sx_out, workspace, workspace_bytes,
                            (hipStream_t)hip_stream, who, nullptr, nullptr, (int)B, kg);
}

int hot_backward_batched_ranges(int64_t B, int64_t T, int64_t O, int64_t I, const hot_config* cfg) {
  if (check_batched(cfg, B, T, "hot_backward_batched_ranges") || O <= 0 || I <= 0) return 0;
  return gemm_grouped_splits_impl(O, I, (int)B, kpad_group(T, cfg));
}

size_t hot_backward_batched_workspace_bytes(int64_t B, int64_t T, int64_t O, int64_t I, const hot_config* cfg) {
  if (check_batched(cfg, B, T, "hot_backward_batched_workspace_bytes") || O <= 0 || I <= 0) return 0;
  return batched_layout(B, T, O, I, cfg).total;
}

static int batched_gy_job(ColJob& job, const void* gy, int dtype, int64_t B, int64_t T, int64_t O, const hot_config* c, const BatchedLayout& b,
                          uint8_t* ws, bool bias, const char* who) {
  return col_job_impl(job, gy, dtype, B * T, O, c->hla_n, cfg_rows(c), c->hla_r, c->gw_bits, c->gw_round, c->seed, HOT_STREAM_GW, c->gw_scale,
                      ws + b.off_qgp, b.ld_gp, 0, (float*)(ws + b.off_sgp), ws + b.off_colg, colwise_group_workspace_bytes_impl(O, (int)B),
                      who, (int)B, b.kg, false, false, 0, bias);
}

int hot_backward_gy_runs(int64_t B, int64_t T, int64_t O, int64_t I, const hot_config* cfg, int dtype, int bias, int32_t* out4) {
  const char* who = "hot_backward_gy_runs";
  if (!out4) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
  if (int e = B ? check_batched(cfg, B, T, who) : check_cfg(cfg, who)) return e;
  if (T <= 0 || O <= 0 || I <= 0 || O % cfg->n_o || I % 8) return fail(HOT_ERR_INVALID, "%s: bad shape T=%lld O=%lld I=%lld", who, (long long)T, (long long)O, (long long)I);
  // (the job is filled and nothing launched: any aligned address does for its operands)
  uint8_t* const at = (uint8_t*)4096;
  ColJob g;
  const int rc = B ? batched_gy_job(g, at, dtype, B, T, O, cfg, batched_layout(B, T, O, I, cfg), at, bias != 0, who)
                   : flat_gy_job(g, at, dtype, T, O, cfg, bwd_layout(T, O, I, cfg), at, flat_want(T, O, I, cfg, dtype), bias != 0, who);
  if (rc) return rc;
  out4[0] = g.runs[0];
  out4[1] = g.runs[1];
  out4[2] = g.a.colmax_own ? g.a.ncolmax : 0;
  out4[3] = g.tall_gx != 0;
  return HOT_OK;
}

// gb: [O] of out_dtype, the column sums of g_y (bias gradient), or null.  They come out of the statistics pass, which
// holds the sum of every token block, and a job of the quantise phase adds them up: training step of
// 64 x 197 tokens 768 -> 768 bf16 197 us with a reduction of g_y behind the call, 188 with this; 128 x 197, 768 -> 3072 727 / 669.
static int run_backward_batched(const char* who, const void* gy, const void* w, int dtype, const void* xq, const float* sx, int64_t B,
                                int64_t T, int64_t O, int64_t I, const hot_config* cfg, void* gx, void* gw, void* gb, int out_dtype,
                                void* workspace, size_t workspace_bytes, void* hip_stream) {
  if (int e = check_batched(cfg, B, T, who)) return e;
  if (!gy || !w || !xq || !sx || !gx || !gw) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
  if (O <= 0 || I <= 0 || O % 8 || I % 8) return fail(HOT_ERR_INVALID, "%s: O=%lld and I=%lld must be positive multiples of 8", who, (long long)O, (long long)I);
  if (O % cfg->n_o) return fail(HOT_ERR_INVALID, "%s: O=%lld is not a multiple of n_o=%d", who, (long long)O, cfg->n_o);
  if (cfg->gx_bits != cfg->w_bits) return fail(HOT_ERR_UNSUPPORTED, "%s: gx_bits (%d) and w_bits (%d) must match", who, cfg->gx_bits, cfg->w_bits);
  if (cfg->gx_scale == HOT_SCALE_SAWB || cfg->gw_scale == HOT_SCALE_SAWB) return fail(HOT_ERR_UNSUPPORTED, "%s: SAWB applies to W and x only", who);
  if (cfg->w_scale == HOT_SCALE_ROW) return fail(HOT_ERR_UNSUPPORTED, "%s: W uses one step per tensor", who);
  if (int e = check_gx_modes(cfg, out_dtype, who)) return e;
  const int64_t L = B * T;
  if (L * O * 4 >= (1ll << 32) || O * I * 4 >= (1ll << 32)) return fail(HOT_ERR_UNSUPPORTED, "%s: tensors exceed the 32-bit offsets of the loader", who);
  const BatchedLayout b = batched_layout(B, T, O, I, cfg);
  if (!workspace || workspace_bytes < b.total) return fail(HOT_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, b.total, workspace_bytes);
  if ((uintptr_t)workspace & 255) return fail(HOT_ERR_INVALID, "%s: workspace must be 256-byte aligned", who);
  hipStream_t st = (hipStream_t)hip_stream;
  uint8_t* ws = (uint8_t*)workspace;
  float* sg = (float*)(ws + b.off_sg);
  float* sw = (float*)(ws + b.off_sw);
  float* sgp = (float*)(ws + b.off_sgp);
  // W: Hadamard along O + quantise, stored [I, O].  g_y: HLA inside every sample, one step per sample (or per sample
  // and channel), transposed -> g_W operand; Hadamard along O, one step per sample (or per token) -> g_x operand, whose
  // product reads a step per row.  Two phases of independent jobs (phase.h).
  const bool w_short = w_joins_phase(cfg), row_tensor = cfg->gx_scale == HOT_SCALE_TENSOR;
  const bool hq_job = cfg->n_o <= CW_ROWS && (row_tensor || O <= HQ_ROW_MAX_K);
  ColJob gj, wj;
  int rc = col_job_impl(wj, w, dtype, O, I, cfg->n_o, identity_rows(), cfg->n_o, cfg->w_bits, cfg->w_round, cfg->seed, HOT_STREAM_W,
                        cfg->w_scale, ws + b.off_qw, b.ld_w, cfg->w_bits == 4, sw, ws + b.off_colw, colwise_workspace_bytes_impl(I), who,
                        1, 0, false, w_short);
  if (!rc) rc = batched_gy_job(gj, gy, dtype, B, T, O, cfg, b, ws, gb != nullptr, who);
  if (rc) return rc;
  HqArgs hj;
  if (hq_job) {
    if (row_tensor) col_job_row_stat(gj, cfg->n_o);
    rc = hq_job_impl(hj, gy, L, O, cfg->n_o, cfg->gx_bits, cfg->gx_round, cfg->seed, HOT_STREAM_GX, cfg->gx_scale, ws + b.off_qg, b.ld_g, sg,
                     gj.a.row_absmax, gj.a.npart, 1, B);
    if (rc) return rc;
  }
  ColsumArgs sj;
  if (gb) {
    gj.a.colsum = (float*)(ws + b.off_colsum);
    if ((rc = colsum_args(sj, gj.a.colsum, O, col_job_strips(gj), b.colsum_strips, gb, out_dtype, who))) return rc;
  }
  col_job_clear(gj, st);
  rc = phase_launch(0, dtype, &gj, w_short ? &wj : nullptr, nullptr, nullptr, st);
  if (!rc && !w_short) rc = phase_launch(0, dtype, &wj, nullptr, nullptr, nullptr, st);
  if (!rc) rc = phase_launch(1, dtype, &gj, w_short ? &wj : nullptr, hq_job ? &hj : nullptr, gb ? &sj : nullptr, st);
  if (!rc && !w_short) rc = phase_launch(1, dtype, &wj, nullptr, nullptr, nullptr, st);
  if (!rc && !hq_job)
    rc = hq_rowwise_impl(gy, dtype, L, O, cfg->n_o, cfg->gx_bits, cfg->gx_round, cfg->seed, HOT_STREAM_GX, cfg->gx_scale,
                         ws + b.off_qg, b.ld_g, sg, ws + b.off_hq, b.off_sg - b.off_hq, st, row_tensor ? T : 0);
  if (rc) return rc;
  rc = gemm_i8_impl(ws + b.off_qg, b.ld_g, ws + b.off_qw, b.ld_w, cfg->gx_bits, L, I, O, sg, cfg->gx_scale == HOT_SCALE_ROW || B > 1 || !hq_job, sw,
                    1.0f / (float)cfg->n_o, gx, out_dtype, I, nullptr, st);   // (one sample: one step for the whole operand)
  if (rc) return rc;
  // g_W = sum over samples of (qGp_b . xq_b^T) sGp_b sx_b / hla_n
  return gemm_i8_grouped_impl(ws + b.off_qgp, b.ld_gp, xq, b.ld_gp, O, I, (int)B, b.kg, sgp, cfg->gw_scale == HOT_SCALE_ROW, sx,
                              1.0f / (float)cfg->hla_n, gw, out_dtype, I, ws + b.off_part, b.part_bytes, st);
}

int hot_linear_backward_batched(const void* gy, const void* w, int dtype, const void* xq, const float* sx, int64_t B,
                                int64_t T, int64_t O, int64_t I, const hot_config* cfg, void* gx, void* gw, int out_dtype,
                                void* workspace, size_t workspace_bytes, void* hip_stream) {
  return run_backward_batched("hot_linear_backward_batched", gy, w, dtype, xq, sx, B, T, O, I, cfg, gx, gw, nullptr, out_dtype,
                              workspace, workspace_bytes, hip_stream);
}

int hot_linear_backward_batched_bias(const void* gy, const void* w, int dtype, const void* xq, const float* sx, int64_t B,
                                     int64_t T, int64_t O, int64_t I, const hot_config* cfg, void* gx, void* gw, void* gb,
                                     int out_dtype, void* workspace, size_t workspace_bytes, void* hip_stream) {
  const char* who = "hot_linear_backward_batched_bias";
  if (!gb) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
  return run_backward_batched(who, gy, w, dtype, xq, sx, B, T, O, I, cfg, gx, gw, gb, out_dtype, workspace, workspace_bytes, hip_stream);
}

int hot_linear_backward_kernels(const void* gy, const void* w, int dtype, const void* xq, const float* sx, int64_t L,
                                int64_t O, int64_t I, const hot_config* cfg, void* gx, void* gw, int out_dtype,
                                void* workspace, size_t workspace_bytes, float* times8, void* hip_stream) {
  if (!times8) return fail(HOT_ERR_INVALID, "hot_linear_backward_kernels: null times8");
  return run_backward_timed(gy, w, dtype, xq, sx, L, O, I, cfg, gx, gw, out_dtype, workspace, workspace_bytes, true, times8,
                            K_COUNT, (hipStream_t)hip_stream);
}

}  // extern "C"
