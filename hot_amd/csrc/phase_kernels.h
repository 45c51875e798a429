// The phase kernels (phase.h) for one input type: included by phase_bf16.hip, phase_f16.hip and phase_f32.hip.
#pragma once

#include <mutex>

#include "phase.h"

namespace hot {

// The arguments as they lie in the kernel's argument segment, read from here on: each job loads its own inside its
// branch.  (Loaded at the kernel's entry, three jobs' arguments overflow the scalar registers.)
__device__ __forceinline__ const PhaseArgs& phase_args() {
  typedef const __attribute__((address_space(4))) PhaseArgs* segment_t;
  segment_t k = (segment_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(k));
  return *(const PhaseArgs*)k;
}

// Wavefronts per SIMD that the registers leave room for: three (what the LDS allows in the quantise pass) wherever a
// thread's block and its selection are small enough to be held.  The quantise pass over blocks of 128 rounding to nearest is at
// the edge: 16-bit inputs spill 6 registers and are faster so than with two waves (the backward of 25216 x 3072 -> 768 bf16
// 155 / 170 us), fp32 inputs would spill 21 (25216 x 2304 207 / 181 with 51 spilled / two waves).
template <typename T, int N, int PASS, int ROUND, typename SEL> constexpr int phase_waves() {
  if (sizeof(T) == 4 && N == 128 && PASS == 1 && ROUND == HOT_ROUND_NEAREST && SEL::STATIC) return 2;
  return !std::is_same<SEL, SelRuntime>::value ? 3 : N <= 32 ? 3 : N == 64 ? 2 : 1;
}
template <typename T, int N, int PASS, int ROUND, typename SEL, bool RS>
__global__ void __launch_bounds__(CW, (phase_waves<T, N, PASS, ROUND, SEL>())) phase_kernel(const PhaseArgs p) {
  extern __shared__ __align__(16) uint8_t lds[];
  unsigned b = blockIdx.x;
  // the short jobs first: they end early and the long one's workgroups fill in behind them
  if (b < p.w_blocks) {
    colwise_body<T, 16, PASS, RUNTIME, RUNTIME, SelShortFull>(phase_args().w, b, lds);
    return;
  }
  b -= p.w_blocks;
  if (PASS == 0 || b < p.g_blocks) {
    constexpr bool HQ = PASS == 1 && (N <= CW_ROWS || !std::is_same<SEL, SelRuntime>::value);      // (row_job_joins)
    colwise_body<T, N, PASS, ROUND, 0, SEL, RS, HQ>(phase_args().g, b, lds, p.h_in_g ? &phase_args().h : nullptr);
    return;
  }
  if constexpr (PASS == 1) {
    b -= p.g_blocks;
    if (b < p.s_blocks) {
      colsum_finish_body(phase_args().s, b, lds);
      return;
    }
    hq_body<T, ROUND>(phase_args().h, b - p.s_blocks);
  }
}

template <typename T, int N, int PASS, int ROUND, typename SEL, bool RS>
static int launch_phase(const PhaseArgs& p, size_t lds, hipStream_t st) {
  // one-time per instantiation; later calls only read the outcome
  static std::once_flag attr_once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(attr_once, [] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(&phase_kernel<T, N, PASS, ROUND, SEL, RS>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
  });
  if (attr_err != hipSuccess) return check_hip(attr_err, "hipFuncSetAttribute(phase_kernel)");
  const uint32_t total = p.w_blocks + p.g_blocks + p.s_blocks + p.h_blocks;
  if (total == 0) return HOT_OK;
  hipLaunchKernelGGL((phase_kernel<T, N, PASS, ROUND, SEL, RS>), dim3(total), dim3(CW), lds, st, p);
  return check_launch("phase_kernel");
}

template <typename T, int N, typename SEL>
static int launch_phase_sel(int pass, const PhaseArgs& p, size_t lds, hipStream_t st) {
  if (pass == 0)
    return p.g.row_absmax ? launch_phase<T, N, 0, 0, SEL, true>(p, lds, st) : launch_phase<T, N, 0, 0, SEL, false>(p, lds, st);
  return (p.g_blocks ? p.g.rounding : p.h.rounding) == HOT_ROUND_STOCH ? launch_phase<T, N, 1, HOT_ROUND_STOCH, SEL, false>(p, lds, st)
                                         : launch_phase<T, N, 1, HOT_ROUND_NEAREST, SEL, false>(p, lds, st);
}

template <typename T>
int phase_launch_impl(int pass, ColSel sel, const PhaseArgs& p, size_t lds, hipStream_t st) {
  switch (sel) {
    case COL_ONE: return launch_phase_sel<T, 1, SelFull<1>>(pass, p, lds, st);
    case COL_RT2: return launch_phase_sel<T, 2, SelRuntime>(pass, p, lds, st);
    case COL_RT4: return launch_phase_sel<T, 4, SelRuntime>(pass, p, lds, st);
    case COL_RT8: return launch_phase_sel<T, 8, SelRuntime>(pass, p, lds, st);
    case COL_RT16: return launch_phase_sel<T, 16, SelRuntime>(pass, p, lds, st);
    case COL_SHORT:                     // (no token-wise job: any instance runs the others)
    case COL_PAPER16: return launch_phase_sel<T, 16, SelPaper16>(pass, p, lds, st);
    case COL_FULL16: return launch_phase_sel<T, 16, SelFull<16>>(pass, p, lds, st);
    case COL_RT32: return launch_phase_sel<T, 32, SelRuntime>(pass, p, lds, st);
    case COL_FULL32: return launch_phase_sel<T, 32, SelFull<32>>(pass, p, lds, st);
    case COL_RT64: return launch_phase_sel<T, 64, SelRuntime>(pass, p, lds, st);
    case COL_PY64: return launch_phase_sel<T, 64, SelPy64>(pass, p, lds, st);
    case COL_FULL64: return launch_phase_sel<T, 64, SelFull<64>>(pass, p, lds, st);
    case COL_RT128: return launch_phase_sel<T, 128, SelRuntime>(pass, p, lds, st);
    case COL_PY128: return launch_phase_sel<T, 128, SelPy128>(pass, p, lds, st);
  }
  return fail(HOT_ERR_INVALID, "phase: bad selection %d", (int)sel);
}

}  // namespace hot
