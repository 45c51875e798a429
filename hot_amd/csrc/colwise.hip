// colwise: Hadamard transform along the ROW (strided) dimension of a row-major
// matrix, optional low-rank selection of r of the n coefficients of each
// block, quantisation, and a transposed (K-major) store for the int8 GEMM.
//
// One kernel family serves
//   * HLA of g_y and of x along the token dimension
//     (lowering_matmul_back(P, .), utils/hadamard_matmul.py:143-161 with
//      P = make_WHT :209-226; used at utils/quant_matmul.py:190 and :301), and
//   * the block-Hadamard of W along O
//     (lowering_matmul_back(H_16, W), utils/quant_matmul.py:270),
// followed by int/stoch/norm/sawb_quantizer_BWD (utils/quant_matmul.py:19-55,
// 86-122) and by the transposes the reference op feeds its GEMMs with
// (cuda_measure/HLQ_backward_kernel.cu:561,610-611).
//
// Data movement.  A workgroup owns 256 adjacent channels (columns) and a run
// of token blocks.  Rows arrive 16 at a time through coalesced 16-byte loads
// (each row of the tile is one contiguous segment of HBM) in a ring of up to
// four LDS buffers, and every thread then pulls ITS channel's 16
// values out of LDS: from there on a thread holds whole columns, so the
// butterflies (stage order h = 1, 2, 4, ..., the canonical fp32 order) need
// no cross-lane traffic.  Quantised codes are staged in LDS as [channel][k]
// and leave the CU as one contiguous K-run per channel.  Two passes over the
// input (statistics, then quantise): the step of a tensor depends on all of it.
//
// HBM traffic per input element: 2 * sizeof(in) read + (r/n) * bits/8 written.
#include <string.h>

#include <mutex>

#include "phase.h"

namespace hot {

// The SAWB passes (their statistic is a pair of sums instead of a maximum); every other step mode runs in the
// phase kernels (phase_kernels.h).
template <typename T, int N, int PASS, int ROUND, typename SEL>
__global__ void __launch_bounds__(CW) colwise_sawb_kernel(const ColArgs a) {
  extern __shared__ __align__(16) uint8_t lds[];
  colwise_body<T, N, PASS, ROUND, 1, SEL>(a, blockIdx.x, lds);
}

// Per-channel maxima that the atomics of a statistics pass need zeroed
__global__ void colwise_clear_kernel(float* colmax, int64_t ncolmax) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ncolmax) colmax[i] = 0.f;
}

// ---- column sums ------------------------------------------------------------------

// Sums of a strip of rows per channel, thread = channel: the stand-alone form of what the statistics
// pass of the phase kernels delivers for free (used when the token blocks take the two-level path).
template <typename T>
__global__ void __launch_bounds__(256) colsum_strip_kernel(const void* in, int64_t R, int64_t C, int64_t rows_per_wg,
                                                            float* partial) {
  typedef typename raw_of<T>::type raw_t;
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= C) return;
  const int64_t r0 = (int64_t)blockIdx.y * rows_per_wg;
  const int64_t r1 = r0 + rows_per_wg < R ? r0 + rows_per_wg : R;
  const raw_t* p = reinterpret_cast<const raw_t*>(in) + r0 * C + c;
  float acc = 0.f;
  int64_t r = r0;
  for (; r + 8 <= r1; r += 8, p += 8 * C) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = cvt_raw<T>(p[i * C]);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc += v[i];
  }
  for (; r < r1; ++r, p += C) acc += cvt_raw<T>(*p);
  partial[(int64_t)blockIdx.y * C + c] = acc;
}

__global__ void __launch_bounds__(256) colsum_finish_kernel(const ColsumArgs a) {
  __shared__ __align__(16) uint8_t lds[CS_GROUPS * CS_CHANS * 4];
  colsum_finish_body(a, blockIdx.x, lds);
}

// ---- host ---------------------------------------------------------------------

size_t hla_workspace_bytes_impl(int64_t R, int64_t C, int n, int r) {
  return n > COL_MAX_N ? hla_big_workspace_bytes_impl(R, C, n, r) : colwise_workspace_bytes_impl(C);
}

constexpr int64_t COL_MAX_WGS = 65536;   // workgroups of a pass
size_t colwise_workspace_bytes_impl(int64_t C) {
  // per-channel max | a statistic per workgroup: two doubles (SAWB), or an absmax and a row-wise absmax
  return (size_t)round_up(C * 4 * COLMAX_COPIES, 256) + (size_t)(2 * sizeof(double)) * COL_MAX_WGS;
}

// with sample groups: per-sample per-channel max | a statistic per workgroup
static size_t colmax_bytes(int64_t C, int groups) { return (size_t)round_up(C * 4 * (groups > 1 ? (int64_t)groups : COLMAX_COPIES), 256); }
size_t colwise_group_workspace_bytes_impl(int64_t C, int groups) {
  if (groups <= 1) return colwise_workspace_bytes_impl(C);
  return colmax_bytes(C, groups) + (size_t)(2 * sizeof(double)) * COL_MAX_WGS;
}

// Token blocks per workgroup of the quantise pass (tb) and of an absmax statistics pass (tb0).
// The staged run of a channel (tb * r codes) must be a whole number of output dwords and cover the blocks that share a 16-row step.
// In a launch that fills the chip it is 32 bytes and more (shorter runs of W, 3072 x 768, beside g_y: W's own kernel 8 us instead of 11,
// but four times as many workgroups in the way of g_y's, and the step 2 us longer), and grows up to 128 bytes while the grid keeps four
// workgroups per CU and the staging area does not cost a resident workgroup: the quantise pass lost a quarter of its speed each time
// a longer run took one of three away (measured at 8192 x 11008 and 11008 x 4096; the L2 of an XCD merges the short runs of
// neighbouring workgroups anyway).  Every ring counts with all its buffers there: that those of one or two steps are shorter
// (col_ring_bytes) lets more workgroups share a CU, but with the shorter runs that would go with it the stores lose more (us of the whole
// backward, fp32, runs of 64 / 32 tokens: 6879 x 7424 x 1232 328 / 348, 2561 x 9280 x 2432 203 / 210, 64 x 577 x 1464 x 200 271 / 280).
// With fewer workgroups than `want` the runs go below 32 bytes, down to one step or one output word: a workgroup's time is then
// a chain (rows on their way, transform, store), and two workgroups on two CUs take half of it each (col_jobs_want).
// Absmax statistics stage nothing: while the grid has fewer than 2048 workgroups they take shorter workgroups, down to 64 rows
// (measured 1 us faster at 12608 x 3072).
// Sums depend on the partition, in their last bits: those of SAWB steps and of a bias gradient (keep_stat) take one that `want` does
// not move.
struct ColShape { int n, r, store4, mode; int64_t C, NB; int elem_bytes; };
static int col_bps(const ColShape& s) { return s.n >= CW_ROWS ? 1 : CW_ROWS / s.n; }       // blocks that share a 16-row step
// (runs are powers of two blocks)
static int64_t col_wgs(const ColShape& s, int t) { return (s.C + CW - 1) / CW * ((s.NB + t - 1) >> __builtin_ctz(t)); }
static int col_least(const ColShape& s) {
  int t = col_bps(s);
  while ((t * s.r) % (s.store4 ? 8 : 4) != 0) t <<= 1;
  return t;
}
static int col_long_run(const ColShape& s) {
  auto run_bytes = [&](int t) { return s.store4 ? t * s.r / 2 : t * s.r; };   // t * r is a multiple of 8 when store4
  auto resident = [&](int t) {   // workgroups of the quantise pass per CU, as far as LDS decides (three are enough)
    const unsigned per = (unsigned)col_ring_bytes(4 * CW_ROWS, s.elem_bytes) + CW * (t * s.r + 4) + 256;
    const int k = (int)(160u * 1024u / per);
    return k > 3 ? 3 : k;
  };
  int t = col_least(s);
  while (run_bytes(t) < 32) t <<= 1;
  while (run_bytes(t) < 128 && col_wgs(s, 2 * t) >= 1024 && resident(2 * t) >= resident(t)) t <<= 1;
  return t;
}
// of an absmax statistics pass, from those of a quantise pass
static int col_stat_run(const ColShape& s, int t) {
  const int least = col_bps(s);
  if (s.mode != HOT_SCALE_SAWB)
    while (t > least && (t & 1) == 0 && t * s.n > 64 && col_wgs(s, t) < 2048) t >>= 1;
  return t;
}
struct ColPartition { int tb, tb0; };
static ColPartition col_partition(const ColShape& s, int64_t want, bool keep_stat) {
  const int whole = col_long_run(s);
  int tb = whole;
  if (s.mode != HOT_SCALE_SAWB)
    for (const int least = col_least(s); tb > least && col_wgs(s, tb) < want;) tb >>= 1;
  return {tb, col_stat_run(s, keep_stat ? whole : tb)};
}

// The fewest workgroups that each column-wise job of a launch should have, given how many all jobs of the launch have while none
// is cut up.  us of the whole backward, runs of 32 bytes and more / cut, bf16, tokens x out x in: 272 x 128 x 80 23.1 / 19.0,
// 197 x 632 x 2048 27.2 / 23.5, 4334 x 640 x 72 31.9 / 27.6, 2048 x 1024 x 1024 48.9 / 45.2, 779 x 7504 x 448 52.9 / 49.9, 4096 x 720 x
// 6528 fp32 76.2 / 72.0.  A launch that is full without it only gets more starts and ends of workgroups: 4137 x 7808 x 64 129.5 /
// 131.3; on the wrong side 323 x 3456 x 6144 INT8 67.8 / 70.7, 1505 x 1056 x 3200 38.9 / 40.1, 5216 x 384 x 784 26.0 / 26.4.
// (48 shapes of 64 .. 16384 tokens and 64 .. 11008 channels: 4.5 % on average, with the shorter rings.)
int64_t col_jobs_want(int64_t workgroups) { return workgroups < 2048 ? 256 : 128; }

int64_t col_job_workgroups(int64_t R, int64_t C, int n, int r, int store4, int mode, int elem_bytes) {
  const ColShape s = {n, r, store4, mode, C, R / n, elem_bytes};
  return col_wgs(s, col_long_run(s));
}

// ---- jobs -----------------------------------------------------------------------

template <typename SEL, int N>
static bool matches(const ColArgs& a) {
  for (int i = 0; i < N; ++i)
    if (a.slot[i] != SEL::slot(i)) return false;
  return true;
}

// The instance for a.slot of a block of n rows with r kept ones.
static ColSel pick_sel(ColArgs& a, int n, bool as_short) {
  const int r = a.r;
  if (!as_short) {
    switch (n) {
      case 1: return COL_ONE;
      case 2: return COL_RT2;
      case 4: return COL_RT4;
      case 8: return COL_RT8;
      case 16:
        if (r == 16 && matches<SelFull<16>, 16>(a)) return COL_FULL16;
        if (r == 8 && matches<SelPaper16, 16>(a)) return COL_PAPER16;
        return COL_RT16;
      case 32: return r == 32 && matches<SelFull<32>, 32>(a) ? COL_FULL32 : COL_RT32;
      case 64:
        if (r == 36 && matches<SelPy64, 64>(a)) return COL_PY64;
        return r == 64 && matches<SelFull<64>, 64>(a) ? COL_FULL64 : COL_RT64;
      case 128: return r == 36 && matches<SelPy128, 128>(a) ? COL_PY128 : COL_RT128;
      default: break;
    }
  }
  return COL_SHORT;
}

int col_job_impl(ColJob& job, const void* in, int dtype, int64_t R, int64_t C, int n, const int32_t* rows, int r, int bits,
                 int rounding, uint64_t seed, uint32_t rng_stream, int scale_mode, void* codes_out, int64_t ld_out, int store4,
                 float* scales_out, void* workspace, size_t workspace_bytes, const char* who, int groups, int64_t kpad_group,
                 bool rowmajor, bool as_short, int64_t want, bool keep_stat) {
  if (!in || !codes_out || !scales_out || !rows) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
  if (rowmajor && (groups > 1 || scale_mode == HOT_SCALE_ROW))
    return fail(HOT_ERR_UNSUPPORTED, "%s: the untransposed store takes one step for the tensor", who);
  if (R <= 0 || C <= 0) return fail(HOT_ERR_INVALID, "%s: bad shape R=%lld C=%lld", who, (long long)R, (long long)C);
  if (groups < 1) return fail(HOT_ERR_INVALID, "%s: %d sample groups", who, groups);
  if (groups > 1) {
    if (store4) return fail(HOT_ERR_UNSUPPORTED, "%s: per-sample steps take INT8 storage", who);
    if (n < 1 || R % ((int64_t)n * groups)) return fail(HOT_ERR_INVALID, "%s: R=%lld is not %d samples of whole blocks of %d", who, (long long)R, groups, n);
    if (kpad_group < (R / n / groups) * r || (kpad_group & 15)) return fail(HOT_ERR_INVALID, "%s: %lld code bytes per sample must be a multiple of 16 and hold the sample's codes", who, (long long)kpad_group);
  }
  if (n < 1 || n > COL_MAX_N || (n & (n - 1))) return fail(HOT_ERR_UNSUPPORTED, "%s: block size %d (a power of two up to %d)", who, n, COL_MAX_N);
  if (R % n) return fail(HOT_ERR_INVALID, "%s: R=%lld is not a multiple of the block %d", who, (long long)R, n);
  if (r < 1 || r > n) return fail(HOT_ERR_INVALID, "%s: r=%d outside [1, %d]", who, r, n);
  if (bits != 4 && bits != 8) return fail(HOT_ERR_UNSUPPORTED, "%s: bits=%d (4 or 8)", who, bits);
  if (rounding != HOT_ROUND_NEAREST && rounding != HOT_ROUND_STOCH) return fail(HOT_ERR_INVALID, "%s: bad rounding %d", who, rounding);
  if (scale_mode < HOT_SCALE_TENSOR || scale_mode > HOT_SCALE_SAWB) return fail(HOT_ERR_INVALID, "%s: bad scale mode %d", who, scale_mode);
  if (dtype != HOT_F32 && dtype != HOT_BF16 && dtype != HOT_F16) return fail(HOT_ERR_INVALID, "%s: bad dtype %d", who, dtype);
  if (C % 8) return fail(HOT_ERR_UNSUPPORTED, "%s: channel count %lld must be a multiple of 8", who, (long long)C);
  if (((uintptr_t)in & 15) || ((uintptr_t)codes_out & 15)) return fail(HOT_ERR_INVALID, "%s: pointers must be 16-byte aligned", who);
  if (R * C * 4 >= (1ll << 32)) return fail(HOT_ERR_UNSUPPORTED, "%s: input of %lld x %lld elements exceeds the 32-bit offsets of the loader", who, (long long)R, (long long)C);

  ColArgs& a = job.a;
  memset(&a, 0, sizeof(a));
  a.in = in; a.R = R; a.C = C; a.NB = R / n; a.Kout = a.NB * r; a.Rs = R / groups;
  a.out = (int8_t*)codes_out; a.ld_out = ld_out;
  a.seed = seed; a.stream = rng_stream;
  a.r = r; a.rpad = (r + 7) & ~7; a.bits = bits; a.rounding = rounding; a.mode = scale_mode;
  for (int i = 0; i < COL_MAX_N; ++i) a.slot[i] = -1;
  for (int k = 0; k < r; ++k) {
    if (rows[k] < 0 || rows[k] >= n) return fail(HOT_ERR_INVALID, "%s: rows[%d]=%d outside [0, %d)", who, k, rows[k], n);
    if (a.slot[rows[k]] != -1) return fail(HOT_ERR_INVALID, "%s: rows[%d]=%d listed twice", who, k, rows[k]);
    a.slot[rows[k]] = (int8_t)k;
  }
  const int64_t row_bytes = rowmajor ? (store4 ? C / 2 : C) : groups > 1 ? kpad_group * groups : (store4 ? a.Kout / 2 : a.Kout);
  // packed INT4 pairs codes along K: a channel's codes must come in whole bytes (pairs along the channels
  // when the store is untransposed: C is a multiple of 8)
  if (store4 && !rowmajor && (a.Kout & 1)) return fail(HOT_ERR_UNSUPPORTED, "%s: packed INT4 output needs an even number of codes per channel", who);
  if (ld_out < row_bytes || (ld_out & 15)) return fail(HOT_ERR_INVALID, "%s: ld_out=%lld must be a multiple of 16 and >= %lld", who, (long long)ld_out, (long long)row_bytes);
  if (!workspace || workspace_bytes < colwise_group_workspace_bytes_impl(C, groups)) return fail(HOT_ERR_WORKSPACE, "%s: workspace of %zu bytes needed", who, colwise_group_workspace_bytes_impl(C, groups));
  if ((uintptr_t)workspace & 255) return fail(HOT_ERR_INVALID, "%s: workspace must be 256-byte aligned", who);
  a.store4 = store4;
  uint8_t* ws = (uint8_t*)workspace;
  a.colmax = (float*)ws;
  a.partial = (double*)(ws + colmax_bytes(C, groups));
  a.pmax = (float*)a.partial;
  a.rowmajor = rowmajor ? 1 : 0;
  a.groups = groups; a.NBs = a.NB / groups; a.Kpad = groups > 1 ? kpad_group : ld_out;
  a.scales_out = scales_out;

  // grids: strips of channels x runs of token blocks, per sample group (a run never leaves its sample)
  const int elem = dtype == HOT_F32 ? 4 : 2;
  const ColPartition cp = col_partition({n, r, store4, scale_mode, C, a.NB, elem}, groups > 1 ? 0 : want, keep_stat);
  const int64_t gx = (C + CW - 1) / CW, runs = (a.NBs + cp.tb - 1) / cp.tb;
  int tb0 = cp.tb0;
  int64_t runs0 = (a.NBs + tb0 - 1) / tb0;
  if (runs * groups > 65535 || gx * runs * groups > COL_MAX_WGS || gx * runs0 * groups > COL_MAX_WGS)
    return fail(HOT_ERR_UNSUPPORTED, "%s: grid %lld x %lld too large", who, (long long)gx, (long long)(runs * groups));
  const int64_t tall_gx = (C + 63) / 64, room = (int64_t)colmax_bytes(C, groups) / 4 + 3 * COL_MAX_WGS;
  // (the tall statistics pass below: longer runs while it keeps 2048 waves, or 1024 to get below 32 arrays of maxima, which every
  // workgroup of the quantise pass reads: us of the whole backward, runs of 64 rows / these: 12608 x 768 x 3072 INT8 89.7 / 88.1,
  // 16383 x 512 x 512 fp32 69.1 / 67.5)
  if (scale_mode == HOT_SCALE_ROW && groups == 1 && (runs0 > COLMAX_OWN || runs0 * C > room) && !keep_stat)
    for (; runs0 > 32 && tall_gx * runs0 >= (runs0 > 128 ? 2048 : 4096); runs0 = (a.NBs + tb0 - 1) / tb0) tb0 *= 2;
  job.lds[0] = col_ring_bytes(tb0 * n, elem);
  job.lds[1] = col_ring_bytes(cp.tb * n, elem) + (size_t)CW * (cp.tb * r + 4);
  if (job.lds[1] > 150 * 1024) return fail(HOT_ERR_UNSUPPORTED, "colwise: staging does not fit LDS");
  job.sel = pick_sel(a, n, as_short);
  a.gx = (uint32_t)gx;
  job.tb[0] = tb0; job.tb[1] = cp.tb;
  job.runs[0] = (int)runs0; job.runs[1] = (int)runs;
  if (job.sel == COL_SHORT) {
    // 16 rows at a time (the partition takes whole groups of them)
    const int per = CW_ROWS / n;
    a.nrt = n;
    a.r = per * r;
    a.NBs = (a.NBs + per - 1) / per;
    job.tb[0] /= per; job.tb[1] /= per;
  }
  // Per-channel maxima: every row of workgroups of the statistics pass has an array of its own, up to COLMAX_OWN of them (every
  // workgroup of the quantise pass reads them all) and as far as they find room beside the row-wise maxima; where there are more
  // runs a workgroup takes four of them and 64 channels (tall).  Else atomics update a few copies, which a launch clears.
  // us of the whole backward, cleared and updated / own: 197 x 632 x 2048 24.7 / 21.9, 49 x 3072 x 768 fp32 26.5 / 24.5, 4096 x 768 x 768
  // 27.4 / 24.6, 1505 x 1056 x 3200 38.8 / 36.0; tall: 12608 x 768 x 3072 INT8 92.0 / 88.1, 16383 x 512 x 512 fp32 75.2 / 67.5.
  a.ncolmax = groups > 1 ? 1 : COLMAX_COPIES;
  job.tall_gx = job.tall_gy = 0;
  if (scale_mode == HOT_SCALE_ROW) {
    const int64_t tall_gy = (runs0 + 3) / 4;
    if (runs0 <= COLMAX_OWN && runs0 * groups * C <= room) {
      a.ncolmax = (int32_t)runs0;
      a.colmax_own = 1;
    } else if (groups == 1 && tall_gy <= COLMAX_OWN && tall_gy * C <= room && tall_gx * tall_gy <= COL_MAX_WGS) {
      a.ncolmax = (int32_t)tall_gy;
      a.colmax_own = 1;
      job.tall_gx = (uint32_t)tall_gx; job.tall_gy = (uint32_t)tall_gy;
    }
  }
  a.npart = (int32_t)(scale_mode == HOT_SCALE_SAWB ? gx * runs : job.tall_gx ? (int64_t)job.tall_gx * job.tall_gy : gx * runs0);
  return HOT_OK;
}

void col_job_row_stat(ColJob& job, int n_o) {
  ColArgs& a = job.a;
  a.rs_n = n_o;
  a.row_absmax = a.pmax + 3 * COL_MAX_WGS;
}

int64_t col_job_strips(const ColJob& job) { return (int64_t)job.runs[0] * job.a.groups; }

uint32_t col_job_blocks(const ColJob& job, int pass) {
  if (pass == 0 && job.tall_gx) return (uint32_t)round_up((int64_t)job.tall_gx * job.tall_gy, 8);
  return (uint32_t)round_up((int64_t)job.a.gx * job.runs[pass] * job.a.groups, 8);
}

ColArgs col_job_args(const ColJob& job, int pass) {
  ColArgs a = job.a;
  a.tb = job.tb[pass]; a.runs = job.runs[pass];
  a.gy = (uint32_t)(job.runs[pass] * a.groups);
  if (pass == 0 && job.tall_gx) { a.tall = 1; a.gx = job.tall_gx; a.gy = job.tall_gy; }
  return a;
}

void col_job_clear(const ColJob& job, hipStream_t st) {
  const ColArgs& a = job.a;
  const int64_t n = a.mode == HOT_SCALE_ROW && !a.colmax_own ? a.C * a.ncolmax * a.groups : 0;
  if (n > 0) hipLaunchKernelGGL(colwise_clear_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a.colmax, n);
}

template <typename T, int N, typename SEL>
static int launch_sawb(const ColJob& job, int pass, hipStream_t st) {
  const ColArgs a = col_job_args(job, pass);
  const dim3 grid(col_job_blocks(job, pass));
  // one-time per instantiation; later calls only read the outcome
  static std::once_flag attr_once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(attr_once, [] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(&colwise_sawb_kernel<T, N, 1, 0, SEL>), hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
    if (attr_err == hipSuccess)
      attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(&colwise_sawb_kernel<T, N, 1, 1, SEL>), hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
  });
  if (attr_err != hipSuccess) return check_hip(attr_err, "hipFuncSetAttribute(colwise_sawb_kernel)");
  if (pass == 0) hipLaunchKernelGGL((colwise_sawb_kernel<T, N, 0, 0, SEL>), grid, dim3(CW), job.lds[0], st, a);
  else if (a.rounding == HOT_ROUND_STOCH) hipLaunchKernelGGL((colwise_sawb_kernel<T, N, 1, 1, SEL>), grid, dim3(CW), job.lds[1], st, a);
  else hipLaunchKernelGGL((colwise_sawb_kernel<T, N, 1, 0, SEL>), grid, dim3(CW), job.lds[1], st, a);
  return check_launch("colwise_sawb_kernel");
}

template <typename T>
static int dispatch_sawb(const ColJob& job, int pass, hipStream_t st) {
  switch (job.sel) {
    case COL_ONE: return launch_sawb<T, 1, SelFull<1>>(job, pass, st);
    case COL_SHORT: break;      // (W's slot of a phase)
    case COL_RT2: return launch_sawb<T, 2, SelRuntime>(job, pass, st);
    case COL_RT4: return launch_sawb<T, 4, SelRuntime>(job, pass, st);
    case COL_RT8: return launch_sawb<T, 8, SelRuntime>(job, pass, st);
    case COL_RT16: return launch_sawb<T, 16, SelRuntime>(job, pass, st);
    case COL_PAPER16: return launch_sawb<T, 16, SelPaper16>(job, pass, st);
    case COL_FULL16: return launch_sawb<T, 16, SelFull<16>>(job, pass, st);
    case COL_RT32: return launch_sawb<T, 32, SelRuntime>(job, pass, st);
    case COL_FULL32: return launch_sawb<T, 32, SelFull<32>>(job, pass, st);
    case COL_RT64: return launch_sawb<T, 64, SelRuntime>(job, pass, st);
    case COL_PY64: return launch_sawb<T, 64, SelPy64>(job, pass, st);
    case COL_FULL64: return launch_sawb<T, 64, SelFull<64>>(job, pass, st);
    case COL_RT128: return launch_sawb<T, 128, SelRuntime>(job, pass, st);
    case COL_PY128: return launch_sawb<T, 128, SelPy128>(job, pass, st);
  }
  return fail(HOT_ERR_INVALID, "colwise: bad selection %d", (int)job.sel);
}

// Whether the workgroups of a token-wise quantise pass run the row-wise quantiser of the same tensor too: from three of
// them per CU on, where they fill the chip alone (us of the quantise phase, joined / as a job of its own: 12608 x 3072
// bf16 39 / 46.5, 12608 x 2304 fp32 47.5 / 55, 8192 x 11008 bf16 101 / 130; below that the separate workgroups are what
// fills it: 3003 x 1000 fp16 13.6 / 12.9).
static bool row_job_joins(const ColJob& g, const HqArgs& h) {
  if (col_job_blocks(g, 1) < 768) return false;
  if (g.sel == COL_RT32 || g.sel == COL_RT64 || g.sel == COL_RT128) return false;   // (no registers to spare)
  return !h.per_row && h.groups == 1 && g.a.groups == 1 && g.a.in == h.in && g.a.R == h.M && g.a.C == h.K;
}

int phase_launch(int pass, int dtype, const ColJob* g, const ColJob* w, const HqArgs* h, const ColsumArgs* s, hipStream_t st) {
  if (g && g->a.mode == HOT_SCALE_SAWB) {
    // a SAWB token-wise job has kernels of its own and comes alone
    if (w || h || s) return fail(HOT_ERR_INVALID, "phase: a SAWB token-wise job takes no company");
    switch (dtype) {
      case HOT_F32: return dispatch_sawb<float>(*g, pass, st);
      case HOT_BF16: return dispatch_sawb<bf16_t>(*g, pass, st);
      default: return dispatch_sawb<f16_t>(*g, pass, st);
    }
  }
  // (the rounding is the kernel's, and one kernel serves both)
  if (g && h && g->a.rounding != h->rounding) {
    if (int rc = phase_launch(pass, dtype, g, w, nullptr, s, st)) return rc;
    return phase_launch(pass, dtype, nullptr, nullptr, h, nullptr, st);
  }
  if (w && w->a.rounding == HOT_ROUND_STOCH && w->a.nrt != CW_ROWS) return fail(HOT_ERR_INVALID, "phase: short blocks with stochastic rounding belong in the g slot");
  PhaseArgs p;
  memset(&p, 0, sizeof(p));
  size_t lds = 0;
  if (g) { p.g = col_job_args(*g, pass); p.g_blocks = col_job_blocks(*g, pass); lds = g->lds[pass]; }
  if (w) { p.w = col_job_args(*w, pass); p.w_blocks = col_job_blocks(*w, pass); if (w->lds[pass] > lds) lds = w->lds[pass]; }
  if (h) {
    p.h = *h;
    if (g && row_job_joins(*g, *h)) p.h_in_g = 1;
    else p.h_blocks = (uint32_t)hq_body_blocks(*h);
  }
  if (s) { p.s = *s; p.s_blocks = (uint32_t)((s->C + CS_CHANS - 1) / CS_CHANS); if (lds < CS_GROUPS * CS_CHANS * 4) lds = CS_GROUPS * CS_CHANS * 4; }
  const ColSel sel = g ? g->sel : COL_SHORT;
  switch (dtype) {
    case HOT_F32: return phase_launch_impl<float>(pass, sel, p, lds, st);
    case HOT_BF16: return phase_launch_impl<bf16_t>(pass, sel, p, lds, st);
    default: return phase_launch_impl<f16_t>(pass, sel, p, lds, st);
  }
}

// Rows of the partial column sums a token-wise call writes: one per run of token blocks of its
// statistics pass; the stand-alone kernel of the large-block path takes strips of at least 64 rows,
// about 2048 workgroups in all.
static int64_t colsum_strip_rows_big(int64_t R, int64_t C) {
  const int64_t gx = (C + 255) / 256;
  const int64_t want = 2048 / gx > 0 ? 2048 / gx : 1;
  const int64_t rows = round_up((R + want - 1) / want, 16);
  return rows < 64 ? 64 : rows;
}

int64_t colsum_strips_impl(int64_t R, int64_t C, int n, int r, int store4, int mode, int elem_bytes, int64_t groups) {
  if (R <= 0 || C <= 0 || n < 1 || r < 1) return 0;
  if (n > COL_MAX_N) {
    const int64_t rows = colsum_strip_rows_big(R, C);
    return (R + rows - 1) / rows;
  }
  const ColShape s = {n, r, store4, mode, C, R / n, elem_bytes};
  const int tb0 = col_stat_run(s, col_long_run(s));
  return (s.NB / groups + tb0 - 1) / tb0 * groups;
}

int colsum_finish_impl(const ColsumArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(colsum_finish_kernel, dim3((unsigned)((a.C + CS_CHANS - 1) / CS_CHANS)), dim3(CS_GROUPS * CS_CHANS), 0, st, a);
  return check_launch("colsum_finish_kernel");
}

int colwise_quant_impl(const void* in, int dtype, int64_t R, int64_t C, int n, const int32_t* rows, int r,
                       int bits, int rounding, uint64_t seed, uint32_t rng_stream, int scale_mode,
                       void* codes_out, int64_t ld_out, int store4, float* scales_out, void* workspace,
                       size_t workspace_bytes, hipStream_t st, const char* who, float* row16_absmax_out,
                       float* colsum_partial, int groups, int64_t kpad_group, bool rowmajor) {
  if (n > COL_MAX_N) {
    // blocks one thread cannot hold: the two-level path
    if (!in || !codes_out || !scales_out || !rows) return fail(HOT_ERR_INVALID, "%s: null pointer", who);
    if (R <= 0 || C <= 0) return fail(HOT_ERR_INVALID, "%s: bad shape R=%lld C=%lld", who, (long long)R, (long long)C);
    if (groups != 1) return fail(HOT_ERR_UNSUPPORTED, "%s: per-sample steps take token blocks up to %d", who, COL_MAX_N);
    if (rowmajor && (scale_mode == HOT_SCALE_ROW || row16_absmax_out || colsum_partial))
      return fail(HOT_ERR_UNSUPPORTED, "%s: the untransposed store takes one step for the tensor and no fused statistics", who);
    if (store4 && !rowmajor) return fail(HOT_ERR_UNSUPPORTED, "%s: blocks above %d tokens have no transposed packed-INT4 store", who, COL_MAX_N);
    if (R % n) return fail(HOT_ERR_INVALID, "%s: R=%lld is not a multiple of the block %d", who, (long long)R, n);
    if (r < 1 || r > n) return fail(HOT_ERR_INVALID, "%s: r=%d outside [1, %d]", who, r, n);
    if (bits != 4 && bits != 8) return fail(HOT_ERR_UNSUPPORTED, "%s: bits=%d (4 or 8)", who, bits);
    if (rounding != HOT_ROUND_NEAREST && rounding != HOT_ROUND_STOCH) return fail(HOT_ERR_INVALID, "%s: bad rounding %d", who, rounding);
    if (scale_mode < HOT_SCALE_TENSOR || scale_mode > HOT_SCALE_SAWB) return fail(HOT_ERR_INVALID, "%s: bad scale mode %d", who, scale_mode);
    if (colsum_partial) {
      const int64_t rows_per = colsum_strip_rows_big(R, C);
      const dim3 grid((unsigned)((C + 255) / 256), (unsigned)((R + rows_per - 1) / rows_per));
      switch (dtype) {
        case HOT_F32: hipLaunchKernelGGL(colsum_strip_kernel<float>, grid, dim3(256), 0, st, in, R, C, rows_per, colsum_partial); break;
        case HOT_BF16: hipLaunchKernelGGL(colsum_strip_kernel<bf16_t>, grid, dim3(256), 0, st, in, R, C, rows_per, colsum_partial); break;
        case HOT_F16: hipLaunchKernelGGL(colsum_strip_kernel<f16_t>, grid, dim3(256), 0, st, in, R, C, rows_per, colsum_partial); break;
        default: return fail(HOT_ERR_INVALID, "%s: bad dtype %d", who, dtype);
      }
    }
    return hla_big_impl(in, dtype, R, C, n, rows, r, bits, rounding, seed, rng_stream, scale_mode, codes_out, ld_out,
                        scales_out, workspace, workspace_bytes, st, who, row16_absmax_out, rowmajor, store4);
  }
  if (row16_absmax_out || colsum_partial) return fail(HOT_ERR_INVALID, "%s: fused statistics of short blocks belong to a phase", who);
  ColJob job;
  if (int rc = col_job_impl(job, in, dtype, R, C, n, rows, r, bits, rounding, seed, rng_stream, scale_mode, codes_out, ld_out, store4,
                            scales_out, workspace, workspace_bytes, who, groups, kpad_group, rowmajor, false,
                            col_jobs_want(0), false)) return rc;
  col_job_clear(job, st);
  if (int rc = phase_launch(0, dtype, &job, nullptr, nullptr, nullptr, st)) return rc;
  return phase_launch(1, dtype, &job, nullptr, nullptr, nullptr, st);
}

// ---- the entry point that allocates nothing ---------------------------------------
//
// hot_hla_tokenwise needs a workspace (per-channel maxima, a statistic per workgroup).
// For callers that cannot allocate one, the same kernels run on a fixed array in device memory
// that is part of the library's code object: every GPU that loads the library holds one copy of
// it until the process ends.  Its size fixes the largest channel count the entry point takes.
constexpr int64_t STATIC_MAX_C = HOT_STATIC_MAX_CHANNELS;
constexpr size_t STATIC_SCRATCH_BYTES =
    (size_t)STATIC_MAX_C * 4 * COLMAX_COPIES + (size_t)(2 * sizeof(double)) * 65536;
static_assert((STATIC_MAX_C * 4 * COLMAX_COPIES) % 256 == 0, "the per-channel maxima end on a 256-byte boundary");
static __device__ __align__(256) uint8_t scratch[STATIC_SCRATCH_BYTES];

// Device address of `scratch` on the current device.  In host code the array's name is only a
// handle for the runtime, never an address a kernel could use; the address is asked for once per
// device (with that device current) and kept.
static int static_scratch_ptr(uint8_t** out, const char* who) {
  static std::mutex mu;
  static uint8_t* ptr[64] = {};
  int dev = -1;
  if (int rc = check_hip(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (dev < 0 || dev >= 64) return fail(HOT_ERR_UNSUPPORTED, "%s: device index %d outside [0, 64)", who, dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    if (int rc = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return rc;
    if (!p || ((uintptr_t)p & 255)) return fail(HOT_ERR_HIP, "%s: the scratch array has no usable device address", who);
    ptr[dev] = (uint8_t*)p;
  }
  *out = ptr[dev];
  return HOT_OK;
}

}  // namespace hot

extern "C" int hot_hla_tokenwise_static(const void* in, int dtype, int64_t R, int64_t C, int n, const int32_t* rows,
                                        int r, int bits, int rounding, uint64_t seed, uint32_t rng_stream,
                                        int scale_mode, void* codes_out, int64_t ld_out, float* scales_out,
                                        void* hip_stream) {
  using namespace hot;
  const char* who = "hot_hla_tokenwise_static";
  if (n > COL_MAX_N)
    return fail(HOT_ERR_UNSUPPORTED, "%s: token blocks above %d need a workspace as large as the input; use hot_hla_tokenwise", who, COL_MAX_N);
  if (C > STATIC_MAX_C)
    return fail(HOT_ERR_UNSUPPORTED, "%s: %lld channels exceed the %lld the built-in scratch array holds; use hot_hla_tokenwise", who,
                (long long)C, (long long)STATIC_MAX_C);
  uint8_t* ws = nullptr;
  if (int rc = static_scratch_ptr(&ws, who)) return rc;
  // (per-channel maxima that runs share are cleared by the first kernel of the call, everything else is written before it is read)
  return colwise_quant_impl(in, dtype, R, C, n, rows, r, bits, rounding, seed, rng_stream, scale_mode, codes_out,
                            ld_out, /*store4=*/0, scales_out, ws, STATIC_SCRATCH_BYTES, (hipStream_t)hip_stream, who);
}
