// Device side of the integer products (gemm_i8.hip, gemm_pair.hip): arguments, tile order, epilogues, and the body of the
// slot-scheduled kernels.  What the products compute and which part of the reference they follow is described in gemm_i8.hip.
#pragma once

#include <type_traits>
#include <utility>

#include "hot_device.h"
#include "hot_host.h"

namespace hot {

constexpr int G_THREADS = 256;
constexpr int G_BK = 128;            // int8 bytes of K per stage in LDS

struct GemmArgs {
  const uint8_t* A;
  const uint8_t* B;
  int64_t lda, ldb;  // bytes
  int64_t M, N;
  int32_t ktiles;    // stages of G_BK codes
  const float* scale_a;
  const float* scale_b;
  float post_scale;
  int32_t a_per_row;
  void* out;
  int64_t ldo;
  const void* bias;  // 16-bit floating operands only (BITS = 16): NULL or N elements of the output type, added per column
  int32_t* acc_out;
  int32_t tiles_m, tiles_n;
  int32_t group_m;   // tile rows per group of the launch order (tile_of)
  int32_t vec_out;   // out and ldo allow aligned four-element stores
  int32_t vec16;     // out and its row pitch are 16-byte aligned (staged epilogue)
  int32_t splits;    // K is cut into this many ranges, one workgroup each (1 = no split)
  v4i* partials;     // [tile][range][wave][fragment quad][lane]: raw accumulators of the ranges
  // K groups (gemm_i8_grouped_kernel; 3-D activations: a group is a sample with steps of its own).
  // The integer sums of every group are dequantised with the group's steps and added, in group
  // order, to fp32 accumulators:
  //   out = (sum over groups of (float(acc_g) * sa_g[row or 0]) * sb_g) * post_scale.
  // With gsplits > 1 the groups are cut into gsplits contiguous ranges, one workgroup each; every
  // range leaves its fp32 sum in gpart and a second kernel adds the ranges in order.
  int32_t groups;
  int32_t group_stages;     // 128-byte stages per group
  int32_t gsplits, gper;    // ranges and groups per range
  const float* gscale_a;    // [groups] or, with a_per_row, [groups][M]
  const float* gscale_b;    // [groups]
  float* gpart;             // [gsplits][M][ldp] fp32
  int64_t ldp;
};

// Workgroup -> tile.  Hardware deals consecutive workgroup ids round-robin to the 8 XCDs, each with
// its own L2.  XCD x takes a contiguous chunk of the launch order, and the launch order walks the
// tile grid in groups of group_m tile rows, row index fastest inside a group, so the workgroups that
// are resident in one XCD at the same time form a compact block of tiles: they stream few distinct
// A and B row panels, and most of their loads hit in that XCD's L2.
// Position of workgroup `wg` in a launch order of `total` units in which XCD x (= wg % 8) takes the
// x-th contiguous chunk.
__device__ __forceinline__ int xcd_chunk_position(int total, int wg) {
  const int x = wg & 7, idx = wg >> 3;
  const int q = total >> 3, rem = total & 7;
  return x * q + (x < rem ? x : rem) + idx;
}

// Tile of position t in the grouped walk of the tile grid.
__device__ __forceinline__ void grouped_tile(const GemmArgs& g, int t, int& tm, int& tn) {
  const int per_group = g.group_m * g.tiles_n;
  const int grp = t / per_group, j = t - grp * per_group;
  const int rows = min(g.group_m, g.tiles_m - grp * g.group_m);
  tm = grp * g.group_m + j % rows;
  tn = j / rows;
}

__device__ __forceinline__ void tile_of(const GemmArgs& g, int wg, int& tm, int& tn) {
  const int total = g.tiles_m * g.tiles_n;
  const int t = xcd_chunk_position(total, wg);
  const int per_group = g.group_m * g.tiles_n;
  const int grp = t / per_group, j = t - grp * per_group;
  const int rows = min(g.group_m, g.tiles_m - grp * g.group_m);
  tm = grp * g.group_m + j % rows;
  tn = j / rows;
}

// Rows per group: about the square root of the tiles one XCD holds at a time.
inline int pick_group_m(int tiles_m, int tiles_n, int wgs_per_cu) {
  const int64_t total = (int64_t)tiles_m * tiles_n;
  int64_t conc = total / 8 < 32 * wgs_per_cu ? total / 8 : 32 * wgs_per_cu;
  if (conc < 1) conc = 1;
  int gm = 1;
  while ((int64_t)(gm + 1) * (gm + 1) <= conc) ++gm;
  if (gm > tiles_m) gm = tiles_m;
  return gm;
}


// Fused dequantisation epilogue, shared by all kernels but the grouped ones.  The MFMAs are issued with the operands
// swapped (B fragment first), so a 32x32 accumulator tile holds the TRANSPOSED product: lane l owns
// output row l % 32 and, in registers 4 q .. 4 q + 3, the four adjacent output columns
// 8 q + 4 (l / 32) .. + 3.  Each lane therefore stores four adjacent outputs at a time (8 bytes of
// bf16 / f16, 16 bytes of fp32), and lanes l and l + 32 fill neighbouring quads of one row.
template <typename OutT> struct Quad;
template <> struct Quad<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct Quad<bf16_t> { typedef uint16_t type __attribute__((ext_vector_type(4))); };
template <> struct Quad<f16_t> { typedef _Float16 type __attribute__((ext_vector_type(4))); };
template <typename OutT> __device__ __forceinline__ void quad_set(typename Quad<OutT>::type& q, int t, float v);
template <> __device__ __forceinline__ void quad_set<float>(Quad<float>::type& q, int t, float v) { q[t] = v; }
template <> __device__ __forceinline__ void quad_set<bf16_t>(Quad<bf16_t>::type& q, int t, float v) { q[t] = f32_to_bf16_rne(v); }
template <> __device__ __forceinline__ void quad_set<f16_t>(Quad<f16_t>::type& q, int t, float v) { q[t] = (_Float16)v; }

// The quantisation steps of this lane's output rows; loaded before the K loop so that the loads'
// latency is hidden behind it.
template <int WM>
__device__ __forceinline__ void load_row_scales(const GemmArgs& g, int64_t row_base, int lane, float (&sa_row)[WM]) {
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int64_t row = row_base + i * 32 + (lane & 31);
    sa_row[i] = g.a_per_row ? g.scale_a[row < g.M ? row : g.M - 1] : g.scale_a[0];
  }
}

// Output value of one accumulator register.  Integer codes: ((float(acc) * s_a) * s_b) * post_scale
// (packed INT4 accumulates 256 x the product).  BITS = 16 (bf16 operands): the register holds the
// fp32 sum itself, and `bias` (the column's bias, 0 without one) is added.
// FOLD (post_scale is a power of two): the caller passes s_b * post_scale, and with INT4 s_a / 256, which saves a product per
// output and with INT4 a shift (5.5 vector instructions to 3.5, INT8 4.5 to 3.5; the epilogue issues little else).  A power of
// two commutes with a rounding as long as nothing on the way overflows or is subnormal, and float(acc) of 256 x a sum below
// 2^23 is exact: the value is the same for the steps that fold_exact admits.
template <int BITS, bool FOLD, typename OutT>
__device__ __forceinline__ float acc_value(int a, float sa, float sb, float post, float bias) {
  if constexpr (BITS == 16) return __builtin_bit_cast(float, a) + bias;
  if constexpr (FOLD) {
    float v = ((float)a * sa) * sb;
    // (rounded to fp32 before it is rounded to the result's type: the compiler would make one v_fma_mixlo_f16 of the two)
    if constexpr (std::is_same<OutT, f16_t>::value) asm volatile("" : "+v"(v));
    return v;
  }
  if constexpr (BITS == 4) a >>= 8;
  return (((float)a * sa) * sb) * post;
}

// Whether a step leaves the folded form exact, whatever the other step and the sum: with the magnitudes of both in [2^-48, 2^47)
// and a post_scale in [2^-30, 1] (FOLD_POST_MIN, checked by the host) every nonzero |acc| < 2^31 keeps each factor, product and
// result between 2^-126 and 2^126.  A step of 0 (a row of zeros) gives zeros in either form.  Infinite and NaN steps are not
// admitted.  (On the bits: a few instructions a tile and no branches.  A build without the check / with it, us of the whole
// backward: 12608 x 3072 x 768 104.0 / 104.5, 12608 x 2304 x 768 fp32 112.5 / 112.6, 12608 x 768 x 3072 INT8 91.7 / 91.7, both
// before the direct epilogue formed its values once.)
constexpr float FOLD_POST_MIN = 0x1p-30f;
__device__ __forceinline__ bool fold_exact(float step) {
  const uint32_t lo = (127u - 48u) << 23, hi = (127u + 47u) << 23;
  const uint32_t u = __builtin_bit_cast(uint32_t, step) & 0x7FFFFFFFu;
  return (u - lo < hi - lo) | (u == 0u);
}

template <typename OutT> __device__ __forceinline__ float bias_at(const void* bias, int64_t col);
template <> __device__ __forceinline__ float bias_at<float>(const void* bias, int64_t col) { return bias ? reinterpret_cast<const float*>(bias)[col] : 0.f; }
template <> __device__ __forceinline__ float bias_at<bf16_t>(const void* bias, int64_t col) {
  return bias ? as_f((uint32_t)reinterpret_cast<const uint16_t*>(bias)[col] << 16) : 0.f;
}
template <> __device__ __forceinline__ float bias_at<f16_t>(const void* bias, int64_t col) {
  return bias ? (float)reinterpret_cast<const _Float16*>(bias)[col] : 0.f;
}

// FOLD: the tiles of a paired launch that do not take the folded epilogue (cut ones, and steps that fold_exact does not admit):
// post_scale stays apart; with INT4 the caller passes s_a / 256 (exact: a step below 2^-118 has no codes but zeros).  The values
// are formed once, before the choice between a store of four and four single ones: code that is rarely run, but its length is
// felt by the code beside it (us of the whole backward, formed for either store / once: 12608 x 3072 x 768 106.0 / 105.3, 12608 x
// 2304 x 768 fp32 113.8 / 113.0, 12608 x 768 x 3072 INT8 96.3 / 95.7).
template <int WM, int WN, int BITS, typename OutT, bool FOLD = false>
__device__ __forceinline__ void gemm_epilogue(const v16i (&acc)[WM][WN], const GemmArgs& g, int64_t row_base,
                                              int64_t col_base, int lane, const float (&sa_row)[WM], float sb) {
  OutT* out = reinterpret_cast<OutT*>(g.out);
  const int half = lane >> 5;
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int64_t row = row_base + i * 32 + (lane & 31);
    if (row >= g.M) continue;
    const float sa = sa_row[i];
#pragma unroll
    for (int j = 0; j < WN; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t col = col_base + j * 32 + 8 * q + 4 * half;
        if (col >= g.N) continue;
        int a[4];
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          a[t] = acc[i][j][4 * q + t];
          if constexpr (BITS == 16) bv[t] = col + t < g.N ? bias_at<OutT>(g.bias, col + t) : 0.f;
        }
        if (g.acc_out) {
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (col + t < g.N) g.acc_out[row * g.N + col + t] = BITS == 4 ? a[t] >> 8 : a[t];
        }
        float once[4];
        if constexpr (FOLD) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            once[t] = acc_value<8, false, OutT>(a[t], sa, sb, g.post_scale, 0.f);
            asm volatile("" : "+v"(once[t]));
          }
        }
        auto value = [&](int t) {
          if constexpr (FOLD) return once[t];
          else return acc_value<BITS, false, OutT>(a[t], sa, sb, g.post_scale, bv[t]);
        };
        if (g.vec_out && col + 3 < g.N) {
          typename Quad<OutT>::type v;
#pragma unroll
          for (int t = 0; t < 4; ++t) quad_set<OutT>(v, t, value(t));
          *reinterpret_cast<typename Quad<OutT>::type*>(out + row * g.ldo + col) = v;
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (col + t < g.N) store_scalar<OutT>(out + row * g.ldo + col + t, value(t));
        }
      }
    }
  }
}

// Epilogue through LDS for tiles that lie fully inside the output: a wave turns one row of its
// fragments (32 output rows x WN * 32 columns) into output values, parks them row-major in a
// wave-private LDS area and writes them back out 16 bytes per lane along the rows, so a store
// instruction covers whole 128-byte lines (with one fragment column of 16-bit results, the 64 x 128 tiles of g_W and the
// 32 .. 96 x 128 ones, half lines, whose other half a neighbouring wave stores), where the direct epilogue hands the memory
// system 16-byte pieces of 32 different rows per instruction.  Wave-private, and a wave's LDS accesses are carried out in the order
// in which it issues them: a read finds what the writes before it left, the next fragment row may overwrite the area
// behind the reads, and nothing waits between them but a store for its own data.
// The stores are marked as streaming: nothing in the launch reads a result again, and as ordinary stores they push the
// operands that other workgroups share out of the L2.  MiB fetched by a launch of both products, ordinary / streaming: 25216
// tokens, 768 -> 3072 INT4 (155 MB of results) 123 / 100, 12608 tokens INT8 133 / 126, fp32 107 / 95, 3072 -> 768 137 / 134.
// (That last one writes 0.6 MiB more for its half lines.)  us of the whole backward, bf16: 25216 tokens, 768 -> 3072 128 / 116,
// 12608 80.7 / 76.5, INT8 86.6 / 83.5, 3072 -> 768 106.9 / 107.7, 8192 tokens, 11008 -> 4096 537 / 529, INT8 674 / 664; fp32:
// 25216 173 / 151, 12608 105 / 90, 3072 -> 768 136.5 / 133.1, 11008 -> 4096 653 / 634.  Single products launched over and over:
// 0 to 7 % faster (hot_gemm_bf16 0 to 15 %), the slowest 12608 x 3072 x 768 INT4 to fp32 at 41.0 / 41.5.
// `area` must hold 32 * (WN * 32 * sizeof(OutT) + 16) bytes.
template <int WM, int WN, int BITS, typename OutT, bool FOLD = false>
__device__ __forceinline__ void gemm_epilogue_staged(const v16i (&acc)[WM][WN], const GemmArgs& g, int64_t row_base,
                                                     int64_t col_base, int lane, const float (&sa_row)[WM], float sb,
                                                     uint8_t* area) {
  constexpr int ROWB = WN * 32 * (int)sizeof(OutT);     // bytes of one staged row
  constexpr int PITCH = ROWB + 16;
  constexpr int CPR = ROWB / 16;                        // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;                         // rows one wave-wide store covers
  static_assert(64 % CPR == 0 && 32 % RPI == 0, "a store covers whole rows of the fragment, and no row past it");
  typedef typename Quad<OutT>::type quad_t;
  OutT* out = reinterpret_cast<OutT*>(g.out);
  const int m = lane & 31, half = lane >> 5;
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const float sa = sa_row[i];
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        quad_t v;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          float bv = 0.f;     // (the staged epilogue runs on whole tiles only: every column exists)
          if constexpr (BITS == 16) bv = bias_at<OutT>(g.bias, col_base + j * 32 + 8 * q + 4 * half + t);
          quad_set<OutT>(v, t, acc_value<BITS, FOLD, OutT>(acc[i][j][4 * q + t], sa, sb, g.post_scale, bv));
        }
        *reinterpret_cast<quad_t*>(area + m * PITCH + (j * 32 + 8 * q + 4 * half) * (int)sizeof(OutT)) = v;
      }
    asm volatile("" ::: "memory");                      // (the accesses stay in this order)
#pragma unroll
    for (int r0 = 0; r0 < 32; r0 += RPI) {
      const int r = r0 + lane / CPR, c = lane % CPR;
      const v4i chunk = *reinterpret_cast<const v4i*>(area + r * PITCH + c * 16);
      __builtin_nontemporal_store(chunk, reinterpret_cast<v4i*>(reinterpret_cast<uint8_t*>(out + (row_base + i * 32 + r) * g.ldo + col_base) + c * 16));
    }
    asm volatile("" ::: "memory");
  }
}

// s_waitcnt vmcnt(VM) alone (expcnt and lgkmcnt untouched); vmcnt is split over bits 3:0 and 15:14
template <int VM>
__device__ __forceinline__ void wait_dma() {
  __builtin_amdgcn_s_waitcnt((VM & 0xF) | ((VM >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// s_waitcnt vmcnt(VM) lgkmcnt(0): the DMA wait plus "this wave's LDS reads have all returned"
template <int VM>
__device__ __forceinline__ void wait_dma_lds() {
  __builtin_amdgcn_s_waitcnt((VM & 0xF) | ((VM >> 4) << 14) | (0x7 << 4) | (0x0 << 8));
}

// vmcnt wait that lets `tiles` (0 .. MAXT) groups of LPW loads stay in flight
template <int MAXT, int LPW, bool LDS = false>
__device__ __forceinline__ void wait_dma_upto(int tiles) {
  if constexpr (MAXT <= 0) {
    if constexpr (LDS) wait_dma_lds<0>(); else wait_dma<0>();
  } else {
    if (tiles >= MAXT) { if constexpr (LDS) wait_dma_lds<MAXT * LPW>(); else wait_dma<MAXT * LPW>(); }
    else wait_dma_upto<MAXT - 1, LPW, LDS>(tiles);
  }
}

template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) { static_for_impl(std::make_integer_sequence<int, N>{}, f); }

// One wave-wide 16-byte-per-lane load from global memory straight into LDS:
// lane l's 16 bytes land at lds_addr + 16 l.  `lds_addr` and `sbase` must be
// wave-uniform.  Written as inline assembly so that the explicit vmcnt waits
// of the pipeline below are the only ones: the compiler cannot tell which LDS
// stage a DMA targets and would otherwise drain all of them before every
// fragment read.
__device__ __forceinline__ void dma16(uint32_t lds_addr, uint32_t voff, const uint8_t* sbase) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_addr), "v"(voff), "s"(sbase)
               : "memory", "m0");
}

__device__ __forceinline__ uint32_t lds_offset(const uint8_t* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p;
}

// ---------------------------------------------------------------------------
// Slot-scheduled variant.  Same data path as the pipelined kernel (gemm_i8_pipe_kernel: operand tiles HBM -> LDS by
// DMA through a ring of S stages, packed INT4 expanded after the fragment read), but the K loop is
// laid out by hand as a sequence of "slots", one MFMA each, fenced from one another, so that
// everything else rides in the shadow of the matrix pipe instead of between its blocks:
//   * the fragment reads of the NEXT round are issued in the first slots of the current round (in
//     the order the next round first uses them), so they have all returned when it starts;
//   * packed INT4: the low-nibble operands of the next round are expanded in the second half of the
//     current round, the high-nibble operands (in place) in the first half of their own round;
//   * the DMA instructions that refill a stage go out one per slot behind the barrier;
//   * a stage is refilled as soon as its second round is in registers (S - 1 tiles in flight).
// The wave grid is GM x GN (2 x 2, 1 x 4 or 4 x 1), a wave owns (32 WM) x (32 WN) outputs, so
// block tiles of any multiple of 32 rows exist (160 x 256 gives ViT-B's 12608 tokens x 768 one
// balanced round of 237 tiles on 256 CUs).  A stage's KiB chunks (1024 / RB rows each) are dealt round-
// robin to the four waves; when they do not come out even the spare DMA slots fetch into a
// spare KiB, so that every wave issues the same number of loads and one vmcnt serves all.
// ---------------------------------------------------------------------------
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// LDS of the kernel: S stages, and a spare KiB when the chunks of a stage do not come out even
template <int WM, int WN, int GM, int GN, int S, int RB>
constexpr int slot_ring_bytes() {
  const int rows = 32 * (WM * GM + WN * GN), chunks = rows * RB / 1024;
  return S * rows * RB + (chunks % 4 ? 1024 : 0);
}

template <int WM, int WN, int GM, int GN, int BITS, int S, int RB, typename OutT, bool FOLD = false>
__device__ __forceinline__ void gemm_slot_body(const GemmArgs& g, int block, uint8_t* ring) {
  static_assert(64 * GM * GN == G_THREADS, "the waves of a workgroup of the kernels' launch bounds, four");
  static_assert(RB == 64 || RB == 128, "stage rows of 64 or 128 bytes");
  constexpr int BM = 32 * WM * GM, BN = 32 * WN * GN;
  constexpr int SPR = RB / 16;                      // 16-byte slots per stage row
  constexpr int RPC = 1024 / RB;                    // rows per KiB chunk (one DMA instruction)
  constexpr int RPS = RB / 32;                      // rounds per stage: a round consumes 32 bytes of every row
  constexpr int ROWS = BM + BN, CHUNKS = ROWS / RPC, LPW = (CHUNKS + 3) / 4;
  constexpr bool SPARE = LPW * 4 != CHUNKS;
  constexpr int STAGE_BYTES = ROWS * RB;
  constexpr int RING_BYTES = slot_ring_bytes<WM, WN, GM, GN, S, RB>();
  static_assert(S >= 2 && RING_BYTES <= 160 * 1024, "two or more LDS stages within 160 KiB");
  constexpr int NF = WM * WN;                       // accumulator fragments per wave
  constexpr int NM = NF * (BITS == 4 ? 2 : 1);      // MFMAs (slots) per round
  constexpr int NR = WM + WN;                       // fragment reads per round
  constexpr int H = NM / 2;                         // slots per half round
  constexpr int DPS = (LPW + NM - 1) / NM;          // DMA instructions per slot of the refilling round
  constexpr int RS_ = BITS == 4 ? H : NM;           // slots the fragment reads go out in (INT4: the second half expands them)
  constexpr int RPSL = (NR + RS_ - 1) / RS_;        // fragment reads per slot

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / GN, wn = wave % GN;
  int tm, tn;
  tile_of(g, block, tm, tn);
  const int64_t row0 = (int64_t)tm * BM, col0 = (int64_t)tn * BN;
  constexpr bool EARLY_SCALES = NF <= 4 && BITS != 16;
  float sa_row[WM];
  float sb = 0.f;
  if constexpr (EARLY_SCALES) {
    load_row_scales<WM>(g, row0 + wm * WM * 32, lane, sa_row);
    sb = g.scale_b[0];
  }
  if constexpr (BITS == 16) {
#pragma unroll
    for (int i = 0; i < WM; ++i) sa_row[i] = 1.f;
  }

  // LDS stage layout: rows of RB bytes = SPR slots of 16 bytes; logical slot s of row r sits at
  // physical slot s ^ swz(r), swz(r) = (r >> 2) & 3 for 64-byte rows, (r >> 1) & 7 for 128-byte
  // rows: the fragment reads of 16 consecutive rows (same logical slot) then fall into 16 different
  // 16-byte bank groups.  DMA instruction i of this wave fills KiB chunk c = 4 i + wave of the
  // stage: rows RPC c .. RPC c + RPC - 1 (A rows first, then B rows); lane l fills physical slot
  // l % SPR of row l / SPR of the chunk.  Chunks past the end of the stage go to the spare KiB.
  uint32_t goff[LPW], ldst[LPW];
  uint32_t is_b = 0;                                // bit i: instruction i reads B
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    int c = 4 * i + wave;
    const bool spare = SPARE && c >= CHUNKS;
    ldst[i] = spare ? (uint32_t)(S * STAGE_BYTES) : (uint32_t)c * 1024u;
    if (spare) c = 0;
    const int r = c * RPC + lane / SPR;
    const int swz = RB == 64 ? (r >> 2) & 3 : (r >> 1) & 7;
    const int slot = (lane % SPR) ^ swz;
    if (c * RPC < BM) {
      int64_t gr = row0 + r;
      if (gr >= g.M) gr = g.M - 1;
      goff[i] = (uint32_t)(gr * g.lda + slot * 16);
    } else {
      int64_t gr = col0 + (r - BM);
      if (gr >= g.N) gr = g.N - 1;
      goff[i] = (uint32_t)(gr * g.ldb + slot * 16);
      is_b |= 1u << i;
    }
  }
  is_b = __builtin_amdgcn_readfirstlane(is_b);
  const uint32_t ring0 = lds_offset(ring);
  const int KT = g.ktiles * (G_BK * BITS / 8) / RB;               // stages of RB bytes per row
  // (copies in registers: selecting between the two kernel arguments by a run-time bit would reload
  // the pointer from the argument segment at every DMA instruction, and wait for it)
  const uint8_t* a_base = g.A;
  const uint8_t* b_base = g.B;
  asm volatile("" : "+s"(a_base), "+s"(b_base));
  auto dma_one = [&](int stage_off, int kt, int i) {
    // (wave-uniform by construction; said explicitly, since the instruction takes it in scalar registers)
    const uint64_t b64 = (uint64_t)(uintptr_t)(((is_b >> i) & 1u ? b_base : a_base) + (int64_t)kt * RB);
    // (the builtin returns a signed int: both halves go through uint32_t, or a low half with its top
    // bit set would sign-extend over the high half)
    const uint32_t b_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b64 >> 32));
    const uint32_t b_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b64);
    const uint8_t* base = reinterpret_cast<const uint8_t*>(((uint64_t)b_hi << 32) | (uint64_t)b_lo);
    const bool spare = SPARE && ldst[i] == (uint32_t)(S * STAGE_BYTES);
    dma16(ring0 + (spare ? 0u : (uint32_t)stage_off) + ldst[i], goff[i], base);
  };

  v16i acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

  // Fragments of two consecutive rounds: fr[p][t], p = parity of the round within its stage, t in the
  // order of first use by the MFMAs (A fragment 0, the WN B fragments, then A fragments 1 .. WM - 1).
  // Packed INT4: lo[p][t] holds the low-nibble operands, fr[p][t] turns into the high-nibble operands
  // in place.  In round d of a stage the lanes of half h (= lane / 32) read logical slot 2 d + h of
  // their row: 16 int8 codes (one MFMA) or 32 packed INT4 codes (two MFMAs: the low nibbles, then the
  // high nibbles; both operands alike, so every product pairs equal k).
  v4i fr[2][NR], lo[2][BITS == 4 ? NR : 1];
  const int frow = lane & 31, fhalf = lane >> 5;
  const int sw = RB == 64 ? (frow >> 2) & 3 : (frow >> 1) & 7;     // same for rows r and r + 32 k
  const int offA = (wm * 32 * WM + frow) * RB, offB = (BM + wn * 32 * WN + frow) * RB;
  auto frag_off = [&](int t) {            // byte offset of fragment t within a stage, without the slot
    return t == 0 ? offA : (t <= WN ? offB + (t - 1) * 32 * RB : offA + (t - WN) * 32 * RB);
  };
  auto read_frag = [&](const uint8_t* stage, int d, int t) {
    const int so = ((2 * d + fhalf) ^ sw) * 16;
    fr[d & 1][t] = *reinterpret_cast<const v4i*>(stage + frag_off(t) + so);
  };
  auto a_of = [](int i) { return i == 0 ? 0 : WN + i; };   // fragment index of A fragment i
  auto b_of = [](int j) { return 1 + j; };
  // MFMA m of a round of parity p
  auto mfma_slot = [&](int p, int m) {
    const int mm = m % NF, i = mm / WN, j = mm % WN;
    if constexpr (BITS == 16) {
      // bf16 operands: the same 16 bytes per lane are eight bf16 of K, the accumulator registers hold fp32
      acc[i][j] = __builtin_bit_cast(v16i, __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                               __builtin_bit_cast(v8bf, fr[p][b_of(j)]), __builtin_bit_cast(v8bf, fr[p][a_of(i)]),
                                               __builtin_bit_cast(v16f, acc[i][j]), 0, 0, 0));
    } else if constexpr (BITS == 8) {
      acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[p][b_of(j)], fr[p][a_of(i)], acc[i][j], 0, 0, 0);
    } else {
      if (m < NF) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(lo[p][b_of(j)], lo[p][a_of(i)], acc[i][j], 0, 0, 0);
      else acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[p][b_of(j)], fr[p][a_of(i)], acc[i][j], 0, 0, 0);
    }
  };
  // dword items [e0, e1) of the expansions of the round of parity p: e = 4 t + dword
  auto expand_lo = [&](int p, int e0, int e1) {
#pragma unroll
    for (int e = e0; e < e1 && e < 4 * NR; ++e) lo[p][e >> 2][e & 3] = (fr[p][e >> 2][e & 3] << 4) & (int)0xF0F0F0F0;
  };
  auto expand_hi = [&](int p, int e0, int e1) {
#pragma unroll
    for (int e = e0; e < e1 && e < 4 * NR; ++e) fr[p][e >> 2][e & 3] &= (int)0xF0F0F0F0;
  };
  constexpr int EPS_ = BITS == 4 ? (4 * NR + H - 1) / H : 0;     // expansion items per slot of a half round

  // prologue: S tiles in flight, tile 0 landed and visible, its first round in registers
  static_for<S>([&](auto k) {
    if (k.value < KT) {
#pragma unroll
      for (int i = 0; i < LPW; ++i) dma_one(k.value * STAGE_BYTES, k.value, i);
    }
  });
  wait_dma_upto<S - 1, LPW>((KT < S ? KT : S) - 1);
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int t = 0; t < NR; ++t) read_frag(ring, 0, t);
  if constexpr (BITS == 4) expand_lo(0, 0, 4 * NR);
  __builtin_amdgcn_sched_barrier(0);

  // One K tile in stage `cur` (tile kt + 1 in `nxt`).  `steady`: every predicate below is true.
  auto ktile = [&](auto steady, auto cur_off, auto nxt_off, int kt) {
    constexpr bool ST = decltype(steady)::value;
    constexpr int CUR = decltype(cur_off)::value, NXT = decltype(nxt_off)::value;
    const uint8_t* cur = ring + CUR;
    const uint8_t* nxt = ring + NXT;
    const bool more = ST || kt + 1 < KT;        // there is a tile kt + 1
    const bool refill = ST || kt + S < KT;      // ... and a tile kt + S to fetch into this stage
    static_for<RPS>([&](auto rc) {
      constexpr int r = decltype(rc)::value, p = r & 1;
      constexpr bool LAST = r == RPS - 1;
      if constexpr (LAST) {
        if (more) {
          // tile kt + 1 has landed (this wave's share) and this wave's reads of the stage are in ...
          if constexpr (ST) wait_dma_lds<(S - 2) * LPW>();
          else wait_dma_upto<S - 2, LPW, true>((kt + S - 1 < KT - 1 ? kt + S - 1 : KT - 1) - (kt + 1));
          __builtin_amdgcn_s_barrier();         // ... and everybody's: tile kt + 1 is visible, stage `cur` is free
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // a round: reads of the next round (of this stage, or round 0 of the next tile), the refill of
      // this stage behind the barrier; INT4: high nibbles of this round, then low nibbles of the next
      static_for<NM>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        if constexpr (LAST) {
#pragma unroll
          for (int i = m * DPS; i < (m + 1) * DPS && i < LPW; ++i)
            if (refill) dma_one(CUR, kt + S, i);
        }
        // fragment reads of the next round: one per slot from the first slot on, or, when a wave owns
        // fewer MFMAs than fragments (tiles of one fragment row or column per wave), RPSL per slot
        static_for<RPSL>([&](auto tc) {
          constexpr int t = m * RPSL + decltype(tc)::value;
          if constexpr (t < NR) {
            if constexpr (!LAST) read_frag(cur, r + 1, t);
            else if (more) read_frag(nxt, 0, t);
          }
        });
        if constexpr (BITS == 4) {
          if constexpr (m < H) expand_hi(p, m * EPS_, (m + 1) * EPS_);
          else if (!LAST || more) expand_lo(p ^ 1, (m - H) * EPS_, (m - H + 1) * EPS_);
        }
        mfma_slot(p, m);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  auto rotation = [&](auto steady, int kt0) {
    static_for<S>([&](auto k) {
      constexpr int K = decltype(k)::value;
      if (decltype(steady)::value || kt0 + K < KT)
        ktile(steady, std::integral_constant<int, K * STAGE_BYTES>{}, std::integral_constant<int, ((K + 1) % S) * STAGE_BYTES>{},
              kt0 + K);
    });
  };
  int kt0 = 0;
  for (; kt0 + 2 * S - 1 < KT; kt0 += S) rotation(std::true_type{}, kt0);   // every tile inside has a tile kt + S
  for (; kt0 < KT; kt0 += S) rotation(std::false_type{}, kt0);

  if constexpr (!EARLY_SCALES && BITS != 16) {
    load_row_scales<WM>(g, row0 + wm * WM * 32, lane, sa_row);
    sb = g.scale_b[0];
  }
  // FOLD: a tile with a step outside the range in which the folded values are the same takes the direct epilogue like a cut one,
  // so that a result does not depend on the launch that made it.
  bool exact = true;
  float sa_fold[WM], sb_fold = sb;
#pragma unroll
  for (int i = 0; i < WM; ++i) sa_fold[i] = sa_row[i];
  if constexpr (FOLD) {
    // (sb stays in a vector register: moved to a scalar one for the comparison, its load would be waited for before the first DMA)
    asm volatile("" : "+v"(sb));
    exact = fold_exact(sb);
    sb_fold = sb * g.post_scale;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      exact = exact & fold_exact(sa_row[i]);
      if constexpr (BITS == 4) sa_fold[i] = sa_row[i] * 0.00390625f;
    }
    exact = __all(exact);
  }
  constexpr int AREA = 32 * (WN * 32 * (int)sizeof(OutT) + 16);
  if (4 * AREA <= S * STAGE_BYTES && g.vec16 && !g.acc_out && row0 + BM <= g.M && col0 + BN <= g.N) {
    __syncthreads();                                     // every wave is done with the ring
    if (exact) {
      gemm_epilogue_staged<WM, WN, BITS, OutT, FOLD>(acc, g, row0 + wm * WM * 32, col0 + wn * WN * 32, lane, sa_fold, sb_fold,
                                                     ring + wave * AREA);
      return;
    }
  }
  gemm_epilogue<WM, WN, BITS, OutT, FOLD>(acc, g, row0 + wm * WM * 32, col0 + wn * WN * 32, lane, sa_fold, sb);
}

// Checks a product and fills the arguments that every kernel takes.
int gemm_fill(GemmArgs& g, const GemmProduct& p, int out_dtype, int32_t* acc_out);

}  // namespace hot
