// A phase of a backward pass: independent jobs in ONE launch, each on a range of the grid.
//
// The transform + quantise work of a linear layer comes in two phases with a dependence between them -- first
// the statistics (of g_y token-wise and row-wise, of W, of x), then everything that needs a step -- but within a
// phase nothing depends on anything.  Launched one by one, each small job pays a launch (2.7 us of host time, 1.3 us
// of idle GPU) and leaves the chip partly empty; forked onto a second stream, every event record / wait pair
// costs the host 10 us (measured).  One launch per phase costs neither, and the jobs fill each other's last rounds.
#pragma once

#include "colwise_device.h"
#include "hq_device.h"

namespace hot {

// Column sums of g_y (the bias gradient) from the rows of partial sums that a statistics pass left.
struct ColsumArgs {
  const float* partial;
  int64_t C;
  void* out;
  int32_t strips, out_dtype;
};
// out[c] = sum of partial[s][c] over the strips s, rounded once to the output type, in a fixed order:
// eight groups of threads take the strips s = g, g + 8, g + 16, ... of a channel (eight loads in
// flight each, added in strip order), then the eight group sums are added in group order.  A
// workgroup covers 32 channels, so that a few hundred strips are a short chain of loads per thread.
constexpr int CS_GROUPS = 8, CS_CHANS = 32;
__device__ __forceinline__ void colsum_finish_body(const ColsumArgs& a, unsigned block, uint8_t* lds) {
  float (*s_part)[CS_CHANS] = reinterpret_cast<float (*)[CS_CHANS]>(lds);
  const int ch = threadIdx.x % CS_CHANS, g = threadIdx.x / CS_CHANS;
  const int64_t c = (int64_t)block * CS_CHANS + ch;
  float acc = 0.f;
  if (c < a.C) {
    int s = g;
    for (; s + 7 * CS_GROUPS < a.strips; s += 8 * CS_GROUPS) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = a.partial[(int64_t)(s + i * CS_GROUPS) * a.C + c];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc += v[i];
    }
    for (; s < a.strips; s += CS_GROUPS) acc += a.partial[(int64_t)s * a.C + c];
  }
  s_part[g][ch] = acc;
  __syncthreads();
  if (g == 0 && c < a.C) {
    float t = s_part[0][ch];
#pragma unroll
    for (int i = 1; i < CS_GROUPS; ++i) t += s_part[i][ch];
    if (a.out_dtype == HOT_F32) store_scalar<float>((float*)a.out + c, t);
    else if (a.out_dtype == HOT_BF16) store_scalar<bf16_t>((bf16_t*)a.out + c, t);
    else store_scalar<f16_t>((f16_t*)a.out + c, t);
  }
}

struct PhaseArgs {
  ColArgs g;            // the token-wise job (its n and selection pick the kernel)
  ColArgs w;            // the column-wise job with short blocks (W): SelShortFull
  HqArgs h;             // the row-wise job and
  ColsumArgs s;         // the bias gradient (quantise phase only)
  uint32_t g_blocks, w_blocks, h_blocks, s_blocks;   // workgroups of each; 0 = absent (g and w: multiples of 8, so that
                                                     // a job's workgroup number modulo 8 stays its XCD)
  int32_t h_in_g;       // quantise phase: g's workgroups run the row-wise job too (h_blocks = 0)
};

// Which instance a block length and selection takes; the caller has filled a.slot.
enum ColSel { COL_SHORT, COL_ONE, COL_RT2, COL_RT4, COL_RT8, COL_RT16, COL_PAPER16, COL_FULL16, COL_RT32, COL_FULL32, COL_RT64, COL_PY64, COL_FULL64, COL_RT128, COL_PY128 };

// A column-wise job: the arguments of both passes, and what differs between them.
struct ColJob {
  ColArgs a;
  ColSel sel;
  int tb[2], runs[2];
  size_t lds[2];
  uint32_t tall_gx, tall_gy;   // grid of the statistics pass in its tall form, else 0
};
// Fills a job (blocks of up to 128 rows) and checks everything a pass would refuse.  as_short: for the w slot of a
// phase (blocks of up to 16 rows).
int col_job_impl(ColJob& job, const void* in, int dtype, int64_t R, int64_t C, int n, const int32_t* rows, int r, int bits,
                 int rounding, uint64_t seed, uint32_t rng_stream, int scale_mode, void* codes_out, int64_t ld_out, int store4,
                 float* scales_out, void* workspace, size_t workspace_bytes, const char* who, int groups, int64_t kpad_group,
                 bool rowmajor, bool as_short, int64_t want = 0, bool keep_stat = false);
// want: the fewest workgroups it should have (one group, absmax steps; 0: as many as long runs give).  keep_stat: the statistics
// pass keeps a partition that depends on the shape alone, and with it the order of the column sums.
int64_t col_jobs_want(int64_t workgroups);
// Workgroups of the quantise pass with want = 0.
int64_t col_job_workgroups(int64_t R, int64_t C, int n, int r, int store4, int mode, int elem_bytes);
// The statistics pass also delivers the absmax of the row-wise Hadamard of blocks of n_o (1 .. 16) of the same input.
void col_job_row_stat(ColJob& job, int n_o);
// Rows of partial column sums that its statistics pass writes (a.colsum): one per run of token blocks.
int64_t col_job_strips(const ColJob& job);
// Zeroes what the statistics pass updates by atomics (nothing for most jobs).
void col_job_clear(const ColJob& job, hipStream_t st);
ColArgs col_job_args(const ColJob& job, int pass);
uint32_t col_job_blocks(const ColJob& job, int pass);

// One phase of the given jobs (null: absent), in one launch when g and h round alike; dtype is that of every input.
// w with stochastic rounding: blocks of 16 only.
int phase_launch(int pass, int dtype, const ColJob* g, const ColJob* w, const HqArgs* h, const ColsumArgs* s, hipStream_t st);

// Launches one phase (pass 0: statistics, 1: quantise) with `lds` bytes of dynamic LDS.
template <typename T> int phase_launch_impl(int pass, ColSel sel, const PhaseArgs& p, size_t lds, hipStream_t st);
extern template int phase_launch_impl<float>(int, ColSel, const PhaseArgs&, size_t, hipStream_t);
extern template int phase_launch_impl<bf16_t>(int, ColSel, const PhaseArgs&, size_t, hipStream_t);
extern template int phase_launch_impl<f16_t>(int, ColSel, const PhaseArgs&, size_t, hipStream_t);

}  // namespace hot
