// Device side of the column-wise transform: the body that the kernels of phase_kernels.h (absmax steps)
// and colwise.hip (SAWB steps) run.  What the transform does, which part of the reference it follows and how
// the data moves is described in colwise.hip.
#pragma once

#include "hq_device.h"

#include <type_traits>


namespace hot {

constexpr int CW = 256;        // threads per workgroup = channels per workgroup
constexpr int COLMAX_COPIES = 8;  // per-channel maxima: workgroup row y folds into copy y % 8 (fewer atomics per line) ...
constexpr int COLMAX_OWN = 64;    // ... or, up to that many workgroup rows (per sample), each has a copy of its own: nothing to clear, a launch less
constexpr int CW_ROWS = 16;    // rows staged per step

struct ColArgs {
  const void* in;
  int64_t R, C;       // input rows (transform dim) and channels
  int64_t NB;         // token blocks = R / N
  int64_t Kout;       // NB * r codes per output row
  int8_t* out;
  int64_t ld_out;     // bytes
  // Statistics of the whole tensor: every workgroup of the statistics pass leaves its own value (nothing to
  // clear beforehand, no updates queueing on one address) and every workgroup of the quantise pass reduces them.
  float* pmax;        // TENSOR: absmax per workgroup, npart of them (per sample group)
  double* partial;    // SAWB: 2 doubles per workgroup, npart of them (per sample group)
  int32_t npart;
  float* colmax;      // ROW: per-channel absmax, ncolmax arrays of C floats per sample group
  int32_t ncolmax;    // own: one per row of workgroups of the statistics pass; else updated by atomics, COLMAX_COPIES (sample groups: 1)
  int32_t colmax_own;
  int32_t tall;       // statistics pass: a workgroup is 64 channels x four runs of token blocks, a run to a wave, instead of 256 channels x one
  float* scales_out;
  float* row_absmax;  // statistics pass with RS: absmax of the row-wise block Hadamard, one per workgroup
  int32_t rs_n;       // ... its block along the channels (1, 2, 4, 8 or 16)
  float* colsum;      // statistics pass: NULL or per-channel sums of the input, one row of C floats per run of token blocks
  uint64_t seed;
  uint32_t stream;
  int32_t r, rpad, bits, store4, rounding, mode, tb;
  int32_t nrt;         // SelShortFull: the block length (1 .. 16)
  uint32_t gx, gy;     // logical grid: channel strips x runs of token blocks
  // Sample groups (3-D activations: one step per sample).  The R rows are `groups` samples of NBs
  // token blocks each; a workgroup's run of blocks never leaves its sample (`runs` runs per sample),
  // the codes of a sample take Kpad bytes of every output row (the tail zeroed), and the statistics
  // are kept per sample: its workgroups are neighbours in pmax, and it has ncolmax arrays of maxima per channel.
  // groups == 1: the whole input is one group with Kpad = ld_out.
  int32_t groups, runs;
  int64_t NBs, Kpad, Rs;  // Rs: rows per sample
  // rowmajor: the codes are stored untransposed, [NB r, C] with ld_out bytes per coefficient row
  // (the A operand of a product whose K runs along the channels), instead of [C, NB r]
  int32_t rowmajor;
  int8_t slot[COL_MAX_N];  // output position of natural row i, -1 = dropped
};

// Which coefficients of a block are kept and where they go.  The generic policy reads the table
// from the kernel arguments; the presets make it a compile-time constant, which removes the
// per-coefficient scalar branches and lets the compiler drop the butterflies that only feed
// discarded coefficients.
struct SelRuntime { static constexpr bool STATIC = false; };
// Blocks of 1 .. 16 rows, their length known at run time, every row kept in order (W): 16 rows at a time, r, tb, NBs and
// runs count whole groups of 16 rows then, the last one may be cut short.  Stochastic rounding with it: blocks of 16.
struct SelShortFull {
  static constexpr bool STATIC = true;
  static constexpr int slot(int i) { return i; }
};
template <int N> struct SelFull {
  static constexpr bool STATIC = true;
  static constexpr int slot(int i) { return i; }
};
struct SelPy64 {  // make_WHT rule for n = 64: 36 coefficients, sequency order
  static constexpr bool STATIC = true;
  static constexpr int8_t TABLE[64] = {0,  35, 25, 26, 14, 33, 15, 32, 7,  -1, -1, -1, -1, -1, -1, -1, 3,  -1, 22, 29, 11, -1,
                                       18, -1, 4,  -1, 21, -1, 10, -1, 19, -1, 1,  -1, 24, 27, 13, 34, 16, 31, 6,  -1, -1, -1,
                                       8,  -1, -1, -1, 2,  -1, 23, 28, 12, -1, 17, 30, 5,  -1, -1, -1, 9,  -1, 20, -1};
  static constexpr int slot(int i) { return TABLE[i]; }
};
struct SelPy128 {  // make_WHT rule for n = 128: the n = 64 selection on the even rows, no odd row
  static constexpr bool STATIC = true;
  static constexpr int slot(int i) { return (i & 1) ? -1 : SelPy64::TABLE[i >> 1]; }
};
struct SelPaper16 {  // the 8 lowest sequencies of a 16-block
  static constexpr bool STATIC = true;
  static constexpr int8_t TABLE[16] = {0, -1, 7, -1, 3, -1, 4, -1, 1, -1, 6, -1, 2, -1, 5, -1};
  static constexpr int slot(int i) { return TABLE[i]; }
};

template <typename T> struct raw_of { typedef uint16_t type; };
template <> struct raw_of<float> { typedef uint32_t type; };

template <typename T> __device__ __forceinline__ float cvt_raw(typename raw_of<T>::type v);
template <> __device__ __forceinline__ float cvt_raw<float>(uint32_t v) { return as_f(v); }
template <> __device__ __forceinline__ float cvt_raw<bf16_t>(uint16_t v) { return as_f((uint32_t)v << 16); }
template <> __device__ __forceinline__ float cvt_raw<f16_t>(uint16_t v) { return (float)__builtin_bit_cast(_Float16, v); }

// Unnormalised FWHT of the N-point groups of v[0..LEN), stages h = H0, 2 H0, 4 H0, ... (H0 = 2: the
// caller has run the first stage already)
template <int N, int LEN, int H0 = 1>
__device__ __forceinline__ void fwht_regs(float (&v)[LEN]) {
#pragma unroll
  for (int h = H0; h < N; h <<= 1) {
#pragma unroll
    for (int i = 0; i < LEN; ++i) {
      if ((i & h) == 0) {
        const float a = v[i], b = v[i + h];
        v[i] = a + b;
        v[i + h] = a - b;
      }
    }
  }
}

// The same for groups of n = 1, 2, 4, 8 or 16 of sixteen values, n known at run time
__device__ __forceinline__ void fwht_short(float (&v)[16], int n, int h0) {
#pragma unroll
  for (int h = 1; h < 16; h <<= 1) {
    if (h >= h0 && h < n) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if ((i & h) == 0) {
          const float a = v[i], b = v[i + h];
          v[i] = a + b;
          v[i + h] = a - b;
        }
      }
    }
  }
}

// Streams the rows of the workgroup's tile through a ring of LDS buffers with
// direct global -> LDS loads (16 bytes per lane, no registers in between).
// Step s covers rows [row0 + 16 s, +16); a buffer holds them as one
// [16 rows][64 channels] slice per wave.  A wave-wide load fills one contiguous
// KiB of the wave's own slice, i.e. 1024 / (64 sizeof(T)) rows.  Rows past the
// end of the input and channels past C are redirected to valid addresses: what
// they deliver is never consumed.
// LDS buffers in the ring (steps in flight behind the one in use = depth - 1): four for 16-bit
// inputs; 32-bit rows are twice as large, and three buffers keep a second workgroup on the CU.
template <typename T> constexpr int ring_depth() { return sizeof(T) == 4 ? 3 : 4; }
// ... and the bytes of the ring of a workgroup that covers `rows` rows: no more buffers than it has steps
__host__ __device__ inline int col_ring_bytes(int rows, int elem_bytes) {
  const int depth = elem_bytes == 4 ? 3 : 4, steps = (rows + CW_ROWS - 1) / CW_ROWS;
  return (steps < depth ? steps : depth) * CW_ROWS * CW * elem_bytes;
}

template <typename T>
struct RowStream {
  static constexpr int RB = 64 * (int)sizeof(T);                 // bytes per staged row of ONE wave (64 channels)
  static constexpr int WAVE_BYTES = CW_ROWS * RB;                // one wave's share of a step
  static constexpr int BUF_BYTES = (CW / 64) * WAVE_BYTES;       // all waves' shares of a step
  static constexpr int LPW = WAVE_BYTES / 1024;                  // DMA instructions per wave per step
  static constexpr int VPR = RB / 16;                            // 16-byte vectors per staged row
  static constexpr int RPC = 1024 / RB;                          // rows per KiB chunk (one DMA instruction)
  const uint8_t* base;   // &in[0][first channel of this wave] (or of the workgroup when the wave has none)
  uint32_t pitch;        // bytes per input row
  int64_t rows_total;
  int64_t row0;
  int nvec_row;          // valid 16-byte vectors per row for this wave (at least 1)
};

// s_waitcnt vmcnt(VM) lgkmcnt(0); vmcnt is split over bits 3:0 and 15:14
template <int VM>
__device__ __forceinline__ void wait_stream() {
  __builtin_amdgcn_s_waitcnt((VM & 0xF) | ((VM >> 4) << 14) | (0x7 << 4) | (0x0 << 8));
}

__device__ __forceinline__ void dma16_to_lds(uint32_t lds_addr, uint32_t voff, const uint8_t* sbase) {
  // lds_addr and sbase are wave-uniform by construction; said explicitly, since the instruction takes
  // them in scalar registers and the compiler keeps a uniform value in a vector register when it was
  // computed past lane-dependent control flow.  (The builtin returns a signed int: every half goes
  // through uint32_t, or a low half with its top bit set would sign-extend over the high half.)
  const uint64_t b64 = (uint64_t)(uintptr_t)sbase;
  const uint32_t b_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b64 >> 32));
  const uint32_t b_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b64);
  const uint8_t* base = reinterpret_cast<const uint8_t*>(((uint64_t)b_hi << 32) | (uint64_t)b_lo);
  const uint32_t lds_u = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_u), "v"(voff), "s"(base)
               : "memory", "m0");
}

// Every wave streams the rows of its own 64 channels into its own slice of each ring buffer
// ([16 rows][64 channels]), so a wave waits for nothing but its own loads: no workgroup barrier
// in the streaming loop, and the four waves of a workgroup drift apart freely.
template <typename T>
__device__ __forceinline__ void rs_issue(const RowStream<T>& rs, uint32_t wave_lds, int step, int lane) {
  constexpr int VPR = RowStream<T>::VPR, RPC = RowStream<T>::RPC;
#pragma unroll
  for (int i = 0; i < RowStream<T>::LPW; ++i) {
    int64_t row = rs.row0 + (int64_t)step * CW_ROWS + i * RPC + lane / VPR;
    if (row >= rs.rows_total) row = rs.rows_total - 1;
    int vec = lane % VPR;
    if (vec >= rs.nvec_row) vec = rs.nvec_row - 1;
    dma16_to_lds(wave_lds + i * 1024, (uint32_t)row * rs.pitch + (uint32_t)vec * 16, rs.base);
  }
}

template <typename T>
__device__ __forceinline__ void rs_column(const uint8_t* wave_buf, int lane, float* v) {
  typedef typename raw_of<T>::type raw_t;
  const raw_t* p = reinterpret_cast<const raw_t*>(wave_buf) + lane;
#pragma unroll
  for (int i = 0; i < CW_ROWS; ++i) v[i] = cvt_raw<T>(p[i * 64]);
}

// ---- the kernel: PASS 0 = statistics, PASS 1 = quantise + transposed store ----

// RS (statistics pass only): when non-zero the pass also tracks the absmax of the ROW-wise block
// Hadamard (block RS along the channels) of the same input, so that the row-wise quantiser of g_y
// needs no statistics pass of its own.  Adjacent lanes hold adjacent channels, hence the row-wise
// butterflies run across lanes.
// ROUND and SAWB: 0 / 1, or 2 = as the arguments say.
// HQ (quantise pass): with `hq` the pass is the row-wise quantiser of the same input as well (one step per tensor,
// Hadamard blocks of up to 16, the rounding of this pass): a wave takes the rows of a step a second time from its
// slice of the ring, lane = 16 channels of one row, instead of the input being read again by workgroups of their own
// (quantise phase at 12608 x 3072 bf16 46.5 -> 39 us, at 8192 x 11008 130 -> 101 us; 19 vector instructions per element
// and the K-major stores bound it now: without the stores 34 and 84 us).
constexpr int RUNTIME = 2;
template <typename T, int N, int PASS, int ROUND, int SAWB, typename SEL, bool RS = false, bool HQ = false>
__device__ __forceinline__ void colwise_body(const ColArgs& args, unsigned block, uint8_t* lds, const HqArgs* hq = nullptr) {
  // A copy, so that every argument is loaded once: read through the reference they would be loaded again at each use behind
  // the memory clobber of a DMA instruction, 59 scalar loads and waits in the loop of <bf16, 1, 1, stochastic>.  Blocks of
  // 128 leave no registers for it (a copy costs the pass 30 spilled ones), and the selection of the other lengths is read
  // where it is used: as a part of the copy it overflows the scalar registers (500 of them spilled).
  typename std::conditional<(N < COL_MAX_N), const ColArgs, const ColArgs&>::type a = args;
  constexpr bool SHORT = std::is_same<SEL, SelShortFull>::value;
  static_assert(!SHORT || N == CW_ROWS, "short blocks are handled 16 rows at a time");
  constexpr int SPB = N >= CW_ROWS ? N / CW_ROWS : 1;        // steps per token block
  constexpr int BPS = N >= CW_ROWS ? 1 : CW_ROWS / N;        // token blocks per step
  constexpr int XL = N >= CW_ROWS ? N : CW_ROWS;             // values a thread holds
  constexpr int BUF = RowStream<T>::BUF_BYTES;
  __shared__ float s_max[CW / 64];
  __shared__ double s_sum[2][CW / 64];
  constexpr int CW_DEPTH = ring_depth<T>();
  uint8_t* const stage = lds;                                // PASS 1: codes [channel][k], before the ring
  const bool sawb = SAWB == RUNTIME ? a.mode == HOT_SCALE_SAWB : SAWB != 0;
  const bool nearest = ROUND == RUNTIME ? a.rounding == HOT_ROUND_NEAREST : ROUND == HOT_ROUND_NEAREST;

  // One-dimensional launch.  The hardware deals consecutive workgroups to the eight XCDs in turn;
  // each XCD takes a contiguous chunk of the logical order, which runs along the token blocks
  // of one channel strip: the workgroups an XCD runs side by side then write neighbouring runs
  // of the same output rows, and its L2 merges their partial lines.
  // (The statistics pass stores nothing and keeps the plain order, strips fastest.)
  const unsigned ngrid = a.gx * a.gy, chunk = (ngrid + 7u) >> 3;
  const unsigned wg_lin = PASS == 1 ? (block & 7u) * chunk + (block >> 3) : block;
  if (wg_lin >= ngrid) return;
  const unsigned bx = PASS == 1 ? wg_lin / a.gy : wg_lin % a.gx;
  const unsigned by = PASS == 1 ? wg_lin - bx * a.gy : wg_lin / a.gx;
  const unsigned wg_id = by * a.gx + bx;     // the numbering the ordered reductions use
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool tall = PASS == 0 && !SHORT && SAWB != 1 && a.tall;
  const int64_t cg0 = (int64_t)bx * (tall ? 64 : CW);
  const int64_t cw0 = tall ? cg0 : cg0 + 64 * wave;        // first channel of this wave
  // Fused row statistic: within each group of 16 lanes the channels are dealt out so that the four
  // stages of the 16-point row transform pair lanes at the distances a single DPP operand reaches
  // (channel bit 0 <-> lane xor 1, bit 1 <-> xor 2, bit 2 <-> xor 15, bit 3 <-> xor 8).
  constexpr bool RSP = PASS == 0 && RS;
  const int chan = RSP ? (tid ^ ((tid & 4) ? 0xB : 0)) : tid;   // channel of this thread within the workgroup
  const int64_t c = cw0 + (chan & 63);
  const bool active = c < a.C;
  const int sample = a.groups > 1 ? (int)(by / (unsigned)a.runs) : 0;
  const int run = tall ? (int)by * (CW / 64) + wave : (int)by - sample * a.runs;
  const int64_t blk_in = (int64_t)run * a.tb;                    // first block of the run within its sample
  const int64_t blk0 = (int64_t)sample * a.NBs + blk_in;
  const int64_t row0 = blk0 * N;
  int nblk = (int)((a.NBs - blk_in) < a.tb ? (a.NBs - blk_in) : a.tb);
  if (tall && nblk < 0) nblk = 0;                          // (a wave past the last run: no steps, maxima of 0)
  const int nsteps = (nblk * N + CW_ROWS - 1) / CW_ROWS;
  // (short blocks: the last group of 16 rows may be cut short; what its missing rows deliver is not consumed)
  const int rows_wg = SHORT && a.Rs - blk_in * N < (int64_t)nblk * N ? (int)(a.Rs - blk_in * N) : nblk * N;
  const int qmax = (1 << (a.bits - 1)) - 1;
  const int sb = a.tb * a.r;        // staged code bytes per channel
  const int pitch = sb + 4;
  // (the ring behind it: as many buffers as col_ring_bytes says)
  uint8_t* const ring = lds + (PASS == 1 ? CW * pitch : 0) + wave * RowStream<T>::WAVE_BYTES;       // this wave's slice of buffer 0

  RowStream<T> rs;
  rs.pitch = (uint32_t)(a.C * (int64_t)sizeof(T));
  rs.rows_total = a.R;
  rs.row0 = row0;
  {
    // channels of this wave that exist; a wave past the end streams the workgroup's first
    // channels instead (valid addresses, never consumed)
    int64_t first = cw0;
    int64_t chans = a.C - first;
    if (chans <= 0) { first = cg0; chans = a.C - cg0; }
    if (chans > 64) chans = 64;
    rs.base = reinterpret_cast<const uint8_t*>(a.in) + first * (int64_t)sizeof(T);
    rs.nvec_row = (int)(chans * (int64_t)sizeof(T) / 16);
  }

  // ring of CW_DEPTH LDS buffers: steps s+1 .. s+CW_DEPTH-1 are in flight while step s is consumed
  constexpr int LPW = RowStream<T>::LPW;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)ring;
  const uint8_t* const my = ring;
#pragma unroll
  for (int s = 0; s < CW_DEPTH - 1; ++s)
    if (s < nsteps) rs_issue<T>(rs, lds0 + s * BUF, s, lane);

  float d = 1.f, rcp = 1.f, clip = 0.f;
  if constexpr (PASS == 1) {
    // the steps come from the statistics themselves (no kernel in between), read behind the first
    // rows' way here; the first workgroup publishes them
    if (sawb) {
      // sums of the statistics pass, added in a fixed order: 256 strided chains, then a tree
      double* s_q = reinterpret_cast<double*>(stage), *s_b = s_q + CW;
      const double* part = a.partial + (int64_t)sample * a.npart * 2;
      double q = 0.0, b = 0.0;
      int i = tid;
      for (; i + 3 * CW < a.npart; i += 4 * CW) {      // (four loads in flight, added one by one)
        double2 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = reinterpret_cast<const double2*>(part)[i + u * CW];
#pragma unroll
        for (int u = 0; u < 4; ++u) { q += v[u].x; b += v[u].y; }
      }
      for (; i < a.npart; i += CW) { q += part[2 * i]; b += part[2 * i + 1]; }
      s_q[tid] = q; s_b[tid] = b;
      __syncthreads();
#pragma unroll
      for (int h = CW / 2; h >= 64; h >>= 1) {
        if (tid < h) { s_q[tid] += s_q[tid + h]; s_b[tid] += s_b[tid + h]; }
        __syncthreads();
      }
      q = wave_sum(s_q[lane]);
      b = wave_sum(s_b[lane]);
      __syncthreads();                 // (the area is the staging area again)
      const double cnt = (double)(a.Kout / a.groups) * (double)a.C;
      clip = (float)(12.1 * sqrt(q / cnt) - 12.2 * (b / cnt));
      const float sc = clip / (float)qmax;
      d = sc + 1e-11f;
      if (bx == 0 && run == 0 && tid == 0) a.scales_out[sample] = sc;
    } else if (a.mode == HOT_SCALE_ROW) {
      float cm = 0.f;
      if (active) {
        const float* cmx = a.colmax + (int64_t)sample * a.ncolmax * a.C + c;
        auto fold = [&](auto under_way) {                            // (that many loads at a time)
          constexpr int W = decltype(under_way)::value;
          for (int k0 = 0; k0 < a.ncolmax; k0 += W) {
            float v[W];
#pragma unroll
            for (int k = 0; k < W; ++k) v[k] = cmx[(k0 + k < a.ncolmax ? k0 + k : a.ncolmax - 1) * a.C];
#pragma unroll
            for (int k = 0; k < W; ++k) cm = fmaxf(cm, v[k]);
          }
        };
        if (a.ncolmax <= 8) fold(std::integral_constant<int, 8>{});
        else fold(std::integral_constant<int, 32>{});
      }
      const float sc = cm / (float)qmax;
      d = active ? sc + 1e-11f : 1.f;
      if (active && run == 0) a.scales_out[(int64_t)sample * a.C + c] = sc;
    } else {
      float m = wave_max(part_max(a.pmax + (int64_t)sample * a.npart, a.npart, 1, tid));
      if (lane == 0) s_max[wave] = m;
      __syncthreads();
      m = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
      const float sc = m / (float)qmax;
      d = sc + 1e-11f;
      if (bx == 0 && run == 0 && tid == 0) a.scales_out[sample] = sc;
    }
    rcp = 1.0f / d;
    // gaps of partial groups must read as 0; a workgroup with all its channels and blocks writes
    // every staged byte itself
    if (nblk < a.tb || cg0 + CW > a.C || rows_wg < nblk * N) {
      uint32_t* l32 = reinterpret_cast<uint32_t*>(stage);
      for (int i = tid; i < CW * pitch / 4; i += CW) l32[i] = 0u;
      __syncthreads();
    }
  }
  const float rcpk = rcp * 65536.0f;       // stochastic rounding works in units of 2^-16

  // row-wise quantiser: lane = 16 channels (two chunks) of row lane / 4 of a step
  constexpr bool HQP = PASS == 1 && HQ;
  float hd = 1.f, hrcp = 1.f;
  int8_t* hout = nullptr;
  int64_t hstep = 0;
  uint64_t hoct = 0;
  int hvalid = 0, hpad = 0, hcb = 0;   // chunks of this lane that exist; bytes to clear behind a row (the last strip's); bytes of a chunk
  if constexpr (HQP) {
    if (hq) {
      __shared__ float s_hq[CW / 64];
      float m = wave_max(part_max(hq->stat, hq->nstat, hq->stat_stride, tid));
      if (lane == 0) s_hq[wave] = m;
      __syncthreads();
      m = fmaxf(fmaxf(s_hq[0], s_hq[1]), fmaxf(s_hq[2], s_hq[3]));
      const float sc = m / (float)((1 << (hq->bits - 1)) - 1);
      hd = sc + 1e-11f;
      hrcp = 1.0f / hd;
      if (wg_lin == 0 && tid == 0) hq->scales[0] = sc;
      const int64_t row = row0 + (lane >> 2), ch = cg0 + 64 * wave + (lane & 3) * 16;
      const int64_t left = (a.C - ch) / EPL;
      hvalid = left <= 0 ? 0 : left == 1 ? 1 : 2;
      hcb = hq->bits;
      hout = hq->codes + row * hq->ld + ch / EPL * hcb;
      hstep = CW_ROWS * hq->ld;
      hoct = ((uint64_t)row * (uint64_t)a.C + (uint64_t)ch) >> 3;
      if (bx + 1 == a.gx && wave == 0) hpad = (int)(hq->ld - a.C / EPL * hcb);
    }
  }
  auto row_quant = [&](int s) {
    const T* p = reinterpret_cast<const T*>(my + (s % CW_DEPTH) * BUF) + (lane >> 2) * 64 + (lane & 3) * 16;
    float y[16];
    load_chunk<T>(p, y);
    load_chunk<T>(p + EPL, y + EPL);
    fwht_short(y, hq->n, 1);
    uint32_t q[16];
    if constexpr (ROUND == HOT_ROUND_NEAREST) {
      const rint_rcp hb = rint_bounds(hrcp);
      uint32_t unsure = 0, any = 0;
#pragma unroll
      for (int j = 0; j < 16; ++j) q[j] = rint_div_bits(y[j], hb, unsure, any);
      if (__builtin_expect((unsure | rint_nan<T>(any)) != 0, 0)) {
#pragma unroll
        for (int j = 0; j < 16; ++j) q[j] = rint_div_exact(y[j], hd, hrcp);
      }
    } else {
      const int hmax = (1 << (hq->bits - 1)) - 1;
      quant_stoch(y, hrcp, hoct << 3, hq->seed, hq->stream, hmax, q);
      quant_stoch(y + EPL, hrcp, (hoct + 1) << 3, hq->seed, hq->stream, hmax, q + EPL);
      hoct += (uint64_t)a.C * (CW_ROWS / EPL);
    }
    const bool row_in = s * CW_ROWS + (lane >> 2) < rows_wg;
    if (hcb == 4) {
      uint2 w;
      w.x = pack_codes4(q);
      w.y = pack_codes4(q + EPL);
      if (row_in && hvalid == 2) *reinterpret_cast<uint2*>(hout) = w;
      else if (row_in && hvalid == 1) *reinterpret_cast<uint32_t*>(hout) = w.x;
    } else {
      const uint2 w0 = pack_codes8(q), w1 = pack_codes8(q + EPL);
      if (row_in && hvalid == 2) *reinterpret_cast<uint4*>(hout) = make_uint4(w0.x, w0.y, w1.x, w1.y);
      else if (row_in && hvalid == 1) *reinterpret_cast<uint2*>(hout) = w0;
    }
    if (hpad && row_in) {
      int8_t* const tail = hout + (a.C - cg0) / EPL * hcb - (lane & 3) * 2 * hcb;
      for (int b = (lane & 3) * 4; b < hpad; b += 16) *reinterpret_cast<uint32_t*>(tail + b) = 0u;
    }
    hout += hstep;
  };

  float cmax = 0.f, rmax = 0.f, csum = 0.f;
  double ssq = 0.0, sab = 0.0;
  float x[XL];

  // Transforms and consumes the token blocks held in x; `bl` is the group-local index of the first.
  philox_words u1 = {0u, 0u, 0u, 0u};
  // Kept coefficients of one block at x[base ..]: measured (PASS 0) or quantised into the staging area (PASS 1).
  // valid: coefficients that exist (short blocks in the last, partial group of 16 rows; else all N).
  auto block_body = [&](auto partial, int base, int blk, int valid) {
    constexpr bool PARTIAL = decltype(partial)::value;
    auto place = [&](int i) -> int {
      if constexpr (PARTIAL) if (i >= valid) return -1;
      if constexpr (SEL::STATIC) return SEL::slot(i);
      else return args.slot[i];
    };
    if constexpr (PASS == 0) {
      if (!sawb) {
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (place(i) >= 0) cmax = fmaxf(cmax, fabsf(x[base + i]));
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (place(i) >= 0) {
            const float v = x[base + i];
            ssq += (double)v * (double)v;
            sab += (double)fabsf(v);
          }
      }
    } else {
      uint8_t* const row = stage + tid * pitch + blk * a.r;
      if (sawb) {
#pragma unroll
        for (int i = 0; i < N; ++i) x[base + i] = fminf(fmaxf(x[base + i], -clip), clip);
      }
      if (nearest) {
        // |v / d| <= qmax (1 + 2^-22) by construction of d (absmax) or of the clip (SAWB): the rounded code cannot
        // leave [-qmax, qmax]
        const rint_rcp b = rint_bounds(rcp);
        uint32_t unsure = 0, any = 0;
        if constexpr (N >= 64 && SEL::STATIC) {
          // the coefficients are complete here: the compiler would sink the last butterfly stage into both
          // branches and hold its inputs until then (half as many registers again)
#pragma unroll
          for (int i = 0; i < N; ++i)
            if (SEL::slot(i) >= 0) asm volatile("" : "+v"(x[base + i]));
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const int sl = place(i);
          if (sl >= 0) row[sl] = (uint8_t)rint_div_bits(x[base + i], b, unsure, any);
        }
        if (__builtin_expect((unsure | rint_nan<T>(any)) != 0, 0)) {
#pragma unroll
          for (int i = 0; i < N; ++i) {
            const int sl = place(i);
            if (sl >= 0) row[sl] = (uint8_t)rint_div_exact(x[base + i], d, rcp);
          }
        }
      } else if constexpr (SHORT) {
        // whole blocks of 16: eight coefficients to a generator call
        uint32_t u[8];
#pragma unroll
        for (int i = 0; i < N; ++i) {
          if ((i & 7) == 0) sr_bits8(((uint64_t)c * (uint64_t)a.NB + (uint64_t)(blk0 + blk)) * (uint64_t)(N / 8) + (uint64_t)(i >> 3), a.seed, a.stream, u);
          if (place(i) >= 0) row[i] = (uint8_t)q_stoch_fix(x[base + i], rcpk, u[i & 7], qmax);
        }
      } else {
        int visited = 0;      // kept coefficients of this block quantised so far
        uint32_t u[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};   // 16-bit uniform integers of eight visits
        if constexpr (N == 1) {
          // blocks of one token keep their one coefficient: element number = channel * NB + block, so
          // eight consecutive blocks of a channel share a generator call (u1 lives across the blocks
          // of this step; a new call at the first block and wherever the number passes a multiple of 8)
          const uint64_t e = (uint64_t)c * (uint64_t)a.NB + (uint64_t)(blk0 + blk);
          if (base == 0 || (e & 7u) == 0) u1 = sr_octet_words(e >> 3, a.seed, a.stream);
          u[0] = sr_bits_of(u1, (uint32_t)e);
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const int sl = place(i);
          if (sl >= 0) {
            // counter = ((channel * NB + block) * rpad + visit index) / 8, slot = visit index % 8
            // (blocks of one token: u[0] was drawn above)
            if (N > 1 && (visited & 7) == 0) {
              if (a.r == 1) {
                // a single kept coefficient per block: numbered channel * NB + block, like the
                // one-token blocks above
                const uint64_t e = (uint64_t)c * (uint64_t)a.NB + (uint64_t)(blk0 + blk);
                u[0] = sr_bits_of(sr_octet_words(e >> 3, a.seed, a.stream), (uint32_t)e);
              } else {
                const uint64_t oct = ((uint64_t)c * (uint64_t)a.NB + (uint64_t)(blk0 + blk)) * (uint64_t)(a.rpad >> 3) +
                                     (uint64_t)(visited >> 3);
                sr_bits8(oct, a.seed, a.stream, u);
              }
            }
            row[sl] = (uint8_t)q_stoch_fix(x[base + i], rcpk, u[visited & 7], qmax);   // (the minimum inside: floor + 1 may step past qmax at the very top)
            ++visited;
          }
        }
      }
    }
  };
  // Sixteen neighbouring codes of a channel (blocks of one token, or whole groups of W's rows) leave in four words, with one look at
  // `unsure` for all of them; codes from `left` on do not exist.  us of the whole backward, byte by byte (and a branch each
  // for blocks of one token) / so: 4645 x 4592 x 80 63.1 / 60.0, 14381 x 1424 x 80 71.7 / 67.4, 1264 x 1536 x 8120 59.2 / 57.7; the activation
  // buffer of 12609 x 3072 50.8 / 44.8.
  auto sixteen = [&](int bl, int left) {
    static_assert(XL == 16 || !(N == 1 || SHORT), "a step of sixteen rows");
    uint32_t q[16], unsure = 0, any = 0;
    const rint_rcp b = rint_bounds(rcp);
#pragma unroll
    for (int i = 0; i < 16; ++i) q[i] = rint_div_bits(x[i], b, unsure, any);
    if (__builtin_expect((unsure | rint_nan<T>(any)) != 0, 0)) {
#pragma unroll
      for (int i = 0; i < 16; ++i) q[i] = rint_div_exact(x[i], d, rcp);
    }
    if (left < 16) {
#pragma unroll
      for (int i = 0; i < 16; ++i) q[i] = i < left ? q[i] : 0u;
    }
    uint32_t* const row = reinterpret_cast<uint32_t*>(stage + tid * pitch + bl);
#pragma unroll
    for (int i = 0; i < 4; ++i) row[i] = pack_bytes(q[4 * i], q[4 * i + 1], q[4 * i + 2], q[4 * i + 3]);
  };
  auto consume = [&](int bl) {
    if constexpr (PASS == 1 && (N == 1 || SHORT)) {
      if (nearest) {
        if constexpr (SHORT) fwht_short(x, a.nrt, 1);
        if (sawb) {
#pragma unroll
          for (int i = 0; i < 16; ++i) x[i] = fminf(fmaxf(x[i], -clip), clip);
        }
        sixteen(bl * N, (N == 1 ? nblk : rows_wg) - bl * N);
        return;
      }
    }
    if constexpr (SHORT) fwht_short(x, a.nrt, 1);
    else fwht_regs<N, XL, (RSP && N >= 2) ? 2 : 1>(x);   // the fused statistics pass runs stage h = 1 while loading
    if constexpr (SHORT) {
      const int valid = rows_wg - bl * N;
      if (valid >= N) block_body(std::false_type{}, 0, bl, N);
      else block_body(std::true_type{}, 0, bl, valid);
    } else {
#pragma unroll
      for (int g = 0; g < BPS; ++g) {
        const int blk = bl + g;
        if (blk < nblk) {
          if constexpr (PASS == 0) csum += x[g * N];     // (coefficient 0 of a block: the sum of its tokens, row 0 of H is all ones)
          block_body(std::false_type{}, g * N, blk, N);
        }
      }
    }
  };

  // one step: wait for its rows, let the ring advance, pull this thread's 16 values into x[xo..]
  // -1 on the lane that holds the upper channel of a pair, per channel bit
  const float sg1 = (chan & 1) ? -1.f : 1.f, sg2 = (chan & 2) ? -1.f : 1.f;
  const float sg4 = (chan & 4) ? -1.f : 1.f, sg8 = (chan & 8) ? -1.f : 1.f;
  auto step = [&](int s, float* dst) {
    // this wave's rows of step s have landed, and its LDS reads of step s-1 are complete: the
    // slice that held step s-1 may be refilled.  Steps s+1 .. s+CW_DEPTH-2 may still be in flight.  (Row stores sit
    // among them and only make the wait a little stricter: counting them in changed nothing measurable.)
    if (CW_DEPTH >= 4 && s + 2 < nsteps) wait_stream<2 * LPW>();
    else if (CW_DEPTH >= 3 && s + 1 < nsteps) wait_stream<LPW>();
    else wait_stream<0>();
    if (s + CW_DEPTH - 1 < nsteps) rs_issue<T>(rs, lds0 + ((s + CW_DEPTH - 1) % CW_DEPTH) * BUF, s + CW_DEPTH - 1, lane);
    if constexpr (RSP) {
      // Row-wise 16-point transform across lanes, magnitudes only.  A stage computes
      // own + s * partner with s = +1 on the lane of the lower channel of a pair (own + partner) and
      // -1 on the other (own - partner = -(partner - own)): a lane's value may come out negated,
      // but paired lanes agree in all lower channel bits and so carry the same sign, every value
      // stays +-(the true coefficient), and the product with +-1 is exact: the magnitudes are those
      // of the add/sub butterflies.  One v_fmac with a DPP operand per stage; the stages run
      // row-major over the 16 rows, so no DPP read follows the write of its register within two
      // instructions (and two wait states separate the rows' last writes from the first stage).
      // The raw rows are consumed here, so the first token-wise stage (rows 2j and 2j+1, always
      // within a step) is taken from them first.
      static_assert(CW_ROWS == 16, "the operand list below names sixteen rows");
      float t[CW_ROWS];
      rs_column<T>(my + (s % CW_DEPTH) * BUF, chan & 63, t);
      if (N >= 2) {
#pragma unroll
        for (int j = 0; j < CW_ROWS; j += 2) { dst[j] = t[j] + t[j + 1]; dst[j + 1] = t[j] - t[j + 1]; }
      } else {
#pragma unroll
        for (int j = 0; j < CW_ROWS; ++j) dst[j] = t[j];
      }
      // the first token-wise stage is complete before the rows are overwritten (else the compiler
      // keeps copies of them)
      asm volatile(""
                   : "+v"(dst[0]), "+v"(dst[1]), "+v"(dst[2]), "+v"(dst[3]), "+v"(dst[4]), "+v"(dst[5]), "+v"(dst[6]),
                     "+v"(dst[7]), "+v"(dst[8]), "+v"(dst[9]), "+v"(dst[10]), "+v"(dst[11]), "+v"(dst[12]),
                     "+v"(dst[13]), "+v"(dst[14]), "+v"(dst[15]));
      // every row is in its register before the first DPP read (the hazard check of the compiler
      // does not look into asm statements): the statement below takes all sixteen as operands
      asm volatile("s_nop 1"
                   : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]), "+v"(t[4]), "+v"(t[5]), "+v"(t[6]), "+v"(t[7]),
                     "+v"(t[8]), "+v"(t[9]), "+v"(t[10]), "+v"(t[11]), "+v"(t[12]), "+v"(t[13]), "+v"(t[14]), "+v"(t[15]));
      if (a.rs_n >= 2) {
#pragma unroll
        for (int i = 0; i < CW_ROWS; ++i)
          asm volatile("v_fmac_f32_dpp %0, %0, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf" : "+v"(t[i]) : "v"(sg1));
      }
      if (a.rs_n >= 4) {
#pragma unroll
        for (int i = 0; i < CW_ROWS; ++i)
          asm volatile("v_fmac_f32_dpp %0, %0, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf" : "+v"(t[i]) : "v"(sg2));
      }
      if (a.rs_n >= 8) {
#pragma unroll
        for (int i = 0; i < CW_ROWS; ++i)
          asm volatile("v_fmac_f32_dpp %0, %0, %1 row_mirror row_mask:0xf bank_mask:0xf" : "+v"(t[i]) : "v"(sg4));
      }
      if (a.rs_n >= 16) {
#pragma unroll
        for (int i = 0; i < CW_ROWS; ++i)
          asm volatile("v_fmac_f32_dpp %0, %0, %1 row_ror:8 row_mask:0xf bank_mask:0xf" : "+v"(t[i]) : "v"(sg8));
      }
      const int valid = rows_wg - s * CW_ROWS;     // (rows past the end of the input are copies of its last row)
      if (a.groups == 1 || valid >= CW_ROWS) {
#pragma unroll
        for (int i = 0; i < CW_ROWS; ++i) rmax = fmaxf(rmax, fabsf(t[i]));
      } else {
#pragma unroll
        for (int i = 0; i < CW_ROWS; ++i)
          if (i < valid) rmax = fmaxf(rmax, fabsf(t[i]));
      }
      return;
    }
    if constexpr (HQP) {
      if (hq) row_quant(s);
      __builtin_amdgcn_sched_barrier(0);     // (its registers are free again before the columns are read)
    }
    rs_column<T>(my + (s % CW_DEPTH) * BUF, lane, dst);
  };
  if constexpr (N >= CW_ROWS) {
    for (int bl = 0; bl < nblk; ++bl) {
#pragma unroll
      for (int p = 0; p < SPB; ++p) step(bl * SPB + p, x + p * CW_ROWS);
      consume(bl);
    }
  } else {
    for (int s = 0; s < nsteps; ++s) {
      step(s, x);
      consume(s * BPS);
    }
  }

  if constexpr (PASS == 0) {
    if (a.colsum && active && nblk > 0) a.colsum[(tall ? (int64_t)run : (int64_t)by) * a.C + c] = csum;
    if constexpr (RS) {
      // rows past the end of the input were redirected to real rows and channels past C form whole
      // inactive blocks, so only the latter need masking
      float m = wave_max(active ? rmax : 0.f);
      if (lane == 0) s_max[wave] = m;
      __syncthreads();
      if (tid == 0) {
        float mm = s_max[0];
        for (int i = 1; i < CW / 64; ++i) mm = fmaxf(mm, s_max[i]);
        a.row_absmax[wg_id] = mm;
      }
      __syncthreads();
    }
    if (a.mode == HOT_SCALE_ROW) {
      if (tall) {
        // the four runs meet in the ring, whose rows every wave has read
        float* const s_cm = reinterpret_cast<float*>(lds);
        __syncthreads();
        s_cm[tid] = cmax;
        __syncthreads();
        if (wave == 0 && active) a.colmax[by * a.C + c] = fmaxf(fmaxf(cmax, s_cm[lane + 64]), fmaxf(s_cm[lane + 128], s_cm[lane + 192]));
        return;
      }
      if (active) {
        if (a.colmax_own) a.colmax[by * a.C + c] = cmax;
        else if (a.groups > 1) atomic_max_nonneg(a.colmax + (int64_t)sample * a.C + c, cmax);
        else atomic_max_nonneg(a.colmax + (by % COLMAX_COPIES) * a.C + c, cmax);
      }
      return;
    }
    if (a.mode == HOT_SCALE_TENSOR) {
      float m = wave_max(active ? cmax : 0.f);
      if (lane == 0) s_max[wave] = m;
      __syncthreads();
      if (tid == 0) {
        float mm = s_max[0];
        for (int i = 1; i < CW / 64; ++i) mm = fmaxf(mm, s_max[i]);
        a.pmax[wg_id] = mm;
      }
      return;
    }
    // SAWB: per-workgroup partial sums, reduced in a fixed order by every workgroup of the quantise pass
    ssq = wave_sum(active ? ssq : 0.0);
    sab = wave_sum(active ? sab : 0.0);
    if (lane == 0) { s_sum[0][wave] = ssq; s_sum[1][wave] = sab; }
    __syncthreads();
    if (tid == 0) {
      double q = 0.0, b = 0.0;
      for (int i = 0; i < CW / 64; ++i) { q += s_sum[0][i]; b += s_sum[1][i]; }
      const int64_t wg = (int64_t)wg_id;
      a.partial[2 * wg] = q;
      a.partial[2 * wg + 1] = b;
    }
  } else {
    // the codes that a lane reads below are its wave's, which carries out its LDS accesses in order
    asm volatile("" ::: "memory");
    if (a.rowmajor) {
      // untransposed store: coefficient row (blk0 + b) r + k takes one code of every channel; a
      // wave writes 64 adjacent bytes (INT8) or, two channels to a byte, 32 (packed INT4: the even
      // channel in bits 3:0)
      const int krun = nblk * a.r;      // (groups of short blocks, whose last one may hold fewer, are never stored this way)
      int8_t* orow = a.out + blk0 * a.r * a.ld_out;
      for (int k = 0; k < krun; ++k, orow += a.ld_out) {
        const int code = stage[tid * pitch + k];
        if (a.store4) {
          const int hi = __shfl_xor(code, 1, 64);
          if (active && !(tid & 1)) orow[c >> 1] = (int8_t)((code & 0xF) | ((hi & 0xF) << 4));
        } else if (active) {
          orow[c] = (int8_t)code;
        }
      }
      return;
    }
    // flush: each channel's staged run is one contiguous global segment; a wave writes those of its own 64 channels, without waiting
    // for the others, and what has to be zero behind the last run in a loop of its own that reads nothing (through the same loop as
    // the codes it was 0.35 us a round: 64 x 512 x 512, one block of tokens and 92 bytes of zeros to a channel, 23.3 / 21.4 us).  Two or
    // four units under way at once are slower (fc2's buffer 39.6 / 40.3 / 40.8): these passes feel the length of their code.
    const bool last = blk_in + a.tb >= a.NBs;       // the run that ends its sample also zeroes the sample's tail
    const int out_sb = a.store4 ? sb / 2 : sb;
    const int64_t seg0 = (int64_t)sample * a.Kpad + (int64_t)run * out_sb;      // byte offset in the output row
    const int64_t seg_end = last ? (int64_t)(sample + 1) * a.Kpad : seg0 + out_sb;
    const int ndw = (int)((seg_end - seg0) / 4);            // output dwords per channel
    const int sdw = out_sb / 4 < ndw ? out_sb / 4 : ndw;    // of which staged
    const int64_t ch0 = cg0 + 64 * wave;                    // this wave's first channel
    const int nch = (int)(a.C - ch0 < 64 ? a.C - ch0 : 64);
    if (nch <= 0) return;
    const uint8_t* const wstage = stage + 64 * wave * pitch;
    int8_t* const wout = a.out + ch0 * a.ld_out + seg0;
    // output dword jd of a staged channel row (packing two codes per byte when store4)
    auto word = [&](const uint32_t* row, int jd) -> uint32_t {
      if (a.store4) {
        const uint32_t lo = row[2 * jd], hi = row[2 * jd + 1];
        // bytes b0..b7 -> nibbles: byte j of the result = (b[2j+1] << 4) | (b[2j] & 15)
        const uint32_t l = (lo & 0x0F) | ((lo >> 4) & 0xF0) | ((lo >> 8) & 0x0F00) | ((lo >> 12) & 0xF000);
        const uint32_t h = (hi & 0x0F) | ((hi >> 4) & 0xF0) | ((hi >> 8) & 0x0F00) | ((hi >> 12) & 0xF000);
        return (l & 0xFFFF) | (h << 16);
      }
      return row[jd];
    };
    // consecutive lanes walk along K within a channel, then on to the next channel; (ch, jd) of position p = lane + 64 k advance by a
    // fixed step, so the loop carries them instead of dividing.  Units of 8 bytes when the segments allow it (half the store
    // instructions), else of 4.
    const int unit = ((out_sb & 7) == 0 && (ndw & 1) == 0) ? 2 : 1;      // dwords per store
    {
      const int nun = sdw / unit;                                        // units per channel
      const int total = nch * nun;
      const int step_ch = 64 / nun, step_jd = 64 - step_ch * nun;
      int ch = lane / nun, jd = lane - ch * nun;
      int8_t* at = wout + ch * a.ld_out + (int64_t)jd * (4 * unit);
      const int64_t step_at = step_ch * a.ld_out + (int64_t)step_jd * (4 * unit), wrap_at = a.ld_out - (int64_t)nun * (4 * unit);
      for (int p = lane; p < total; p += 64, ch += step_ch, jd += step_jd, at += step_at) {
        if (jd >= nun) { jd -= nun; ++ch; at += wrap_at; }
        const uint32_t* row = reinterpret_cast<const uint32_t*>(wstage + ch * pitch);
        if (unit == 2) {
          uint2 w2;
          w2.x = word(row, 2 * jd);
          w2.y = word(row, 2 * jd + 1);
          *reinterpret_cast<uint2*>(at) = w2;
        } else {
          *reinterpret_cast<uint32_t*>(at) = word(row, jd);
        }
      }
    }
    if (ndw > sdw) {
      const int nun = (ndw - sdw) / unit, total = nch * nun;
      const int step_ch = 64 / nun, step_jd = 64 - step_ch * nun;
      const int ch = lane / nun;
      int jd = lane - ch * nun;
      int8_t* at = wout + 4 * sdw + ch * a.ld_out + (int64_t)jd * (4 * unit);
      const int64_t step_at = step_ch * a.ld_out + (int64_t)step_jd * (4 * unit), wrap_at = a.ld_out - (int64_t)nun * (4 * unit);
      for (int p = lane; p < total; p += 64, jd += step_jd, at += step_at) {
        if (jd >= nun) { jd -= nun; at += wrap_at; }
        if (unit == 2) *reinterpret_cast<uint2*>(at) = make_uint2(0u, 0u);
        else *reinterpret_cast<uint32_t*>(at) = 0u;
      }
    }
  }
}

}  // namespace hot
