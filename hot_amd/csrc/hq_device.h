// Device side of the row-wise block-Hadamard quantiser: the pieces that the kernels of hq_rowwise.hip are made
// of, and the body that a quantise phase runs beside the column-wise passes (phase_kernels.h).  What the
// quantiser does and which part of the reference it follows is described in hq_rowwise.hip.
#pragma once

#include "hot_device.h"
#include "hot_host.h"

namespace hot {

constexpr int EPL = 8;  // elements per lane-chunk

template <typename T>
__device__ __forceinline__ void load_chunk(const T* p, float* x) {
  constexpr int EPV = vec_traits<T>::EPV;
  const uint4* v = reinterpret_cast<const uint4*>(p);
#pragma unroll
  for (int i = 0; i < EPL / EPV; ++i) {
    const uint4 raw = v[i];
    unpack_vec<T>(raw, x + i * EPV);
  }
}

// FWHT of the N-element blocks formed by N/EPL adjacent lanes.  N = 8 stands for every block that
// fits one lane's chunk: its actual size `nrt` (1, 2, 4 or 8) arrives at run time.
template <int N>
__device__ __forceinline__ void fwht_lanes(float* x, int lane, int nrt) {
#pragma unroll
  for (int h = 1; h < EPL; h <<= 1) {
    if (N > EPL || h < nrt) {   // no early exit: the stage loop must unroll for x to stay in registers
#pragma unroll
      for (int j = 0; j < EPL; ++j) {
        if ((j & h) == 0) {
          const float a = x[j], b = x[j + h];
          x[j] = a + b;
          x[j + h] = a - b;
        }
      }
    }
  }
  // lower lane: own + partner ; upper lane: partner - own  ==  partner + (-own)
  if constexpr (N >= 16) {
    const uint32_t sg = (lane & 1) ? 0x80000000u : 0u;
#pragma unroll
    for (int j = 0; j < EPL; ++j) x[j] = as_f(as_u(x[j]) ^ sg) + lane_xor<1>(x[j]);
  }
  if constexpr (N >= 32) {
    const uint32_t sg = (lane & 2) ? 0x80000000u : 0u;
#pragma unroll
    for (int j = 0; j < EPL; ++j) x[j] = as_f(as_u(x[j]) ^ sg) + lane_xor<2>(x[j]);
  }
  if constexpr (N >= 64) {
    const uint32_t sg = (lane & 4) ? 0x80000000u : 0u;
#pragma unroll
    for (int j = 0; j < EPL; ++j) x[j] = as_f(as_u(x[j]) ^ sg) + lane_xor<4>(x[j]);
  }
}

// Codes of a chunk of an input of type T, in the low bits of q.
template <typename T>
__device__ __forceinline__ void quant_nearest(const float* x, float d, float rcp, uint32_t* q) {
  // |x / d| <= qmax (1 + 2^-22) because d comes from the absmax: no clamp needed
  const rint_rcp r = rint_bounds(rcp);
  uint32_t unsure = 0, any = 0;
#pragma unroll
  for (int j = 0; j < EPL; ++j) q[j] = rint_div_bits(x[j], r, unsure, any);
  if (__builtin_expect((unsure | rint_nan<T>(any)) != 0, 0)) {
#pragma unroll
    for (int j = 0; j < EPL; ++j) q[j] = rint_div_exact(x[j], d, rcp);
  }
}
__device__ __forceinline__ void quant_stoch(const float* x, float rcp, uint64_t e0, uint64_t seed, uint32_t stream, int qmax, uint32_t* q) {
  uint32_t r[EPL];
  sr_bits8(e0 >> 3, seed, stream, r);          // e0 is a multiple of EPL = 8
  const float rcpk = rcp * 65536.0f;
#pragma unroll
  for (int j = 0; j < EPL; ++j) q[j] = (uint32_t)q_stoch_fix(x[j], rcpk, r[j], qmax);
}
// bytes 0 of four registers
__device__ __forceinline__ uint32_t pack_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x0C0C0400u), hi = __builtin_amdgcn_perm(d, c, 0x04000C0Cu);
  return lo | hi;
}
__device__ __forceinline__ uint32_t pack_codes4(const uint32_t* q) {
  const uint32_t ev = pack_bytes(q[0], q[2], q[4], q[6]), od = pack_bytes(q[1], q[3], q[5], q[7]);
  return (ev & 0x0F0F0F0Fu) | ((od << 4) & 0xF0F0F0F0u);
}
__device__ __forceinline__ uint2 pack_codes8(const uint32_t* q) {
  return make_uint2(pack_bytes(q[0], q[1], q[2], q[3]), pack_bytes(q[4], q[5], q[6], q[7]));
}
__device__ __forceinline__ void store_codes4(const uint32_t* q, int8_t* out) { *reinterpret_cast<uint32_t*>(out) = pack_codes4(q); }
__device__ __forceinline__ void store_codes8(const uint32_t* q, int8_t* out) { *reinterpret_cast<uint2*>(out) = pack_codes8(q); }

template <typename T, int BITS, int ROUND>
__device__ __forceinline__ void quant_store_chunk(const float* x, float d, float rcp, uint64_t e0, uint64_t seed,
                                                  uint32_t stream, int8_t* out_row_chunk) {
  uint32_t q[EPL];
  if constexpr (ROUND == 0) quant_nearest<T>(x, d, rcp, q);
  else quant_stoch(x, rcp, e0, seed, stream, (1 << (BITS - 1)) - 1, q);
  if constexpr (BITS == 4) store_codes4(q, out_row_chunk);
  else store_codes8(q, out_row_chunk);
}

// ---- the row-wise quantiser as a part of a larger launch ---------------------------------------------
// Workgroups of 256 threads; Hadamard blocks of 1 .. 16 elements.  One step per tensor or per sample: a workgroup
// takes HQ_UNROLL x 256 consecutive chunks, all loaded before the first is used.  One step per row: rows of up to
// 4096 elements are a wave's (no barrier, the row in registers), longer ones, up to 16384, a workgroup's; a wave skips the
// chunks of its instance that its row does not reach (12608 rows of 768, two of three: the call 103.5 -> 101.5 us).  The
// padding of every row (up to the K tile of the product) is zeroed by the threads that hold the row's end.
constexpr int HQ_UNROLL = 4;
constexpr int64_t HQ_ROW_MAX_K = 16384;

struct HqArgs {
  const void* in;
  int8_t* codes;
  float* scales;          // per tensor [1], per sample or row [M]
  int64_t M, K, ld;       // rows, elements and code pitch (bytes) of a row
  uint32_t nch_row, div_m, div_s;   // chunks per row, and the multiplier and shift that divide by it
  uint32_t chunks;        // per sample (the tensor when there is one)
  uint32_t wgs;           // workgroups per sample
  int64_t rows;           // per sample
  int32_t n, bits, rounding, per_row, groups;
  const float* stat;      // absmax: nstat values stat_stride floats apart (per sample, those of one after the other)
  int32_t nstat, stat_stride;
  uint64_t seed;
  uint32_t stream;
};

// ch / nch_row for ch < 2^31: div_m = floor(2^(31 + s) / d) + 1, s = ceil(log2 d), div_s = s - 1 (d = 1: div_m = 0)
__device__ __forceinline__ uint32_t hq_row_of(const HqArgs& a, uint32_t ch) {
  return a.div_m ? __umulhi(ch, a.div_m) >> a.div_s : ch;
}

// FWHT of blocks of n = 1, 2, 4, 8 or 16 elements, n known at run time
__device__ __forceinline__ void fwht_lanes_short(float* x, int lane, int n) {
  fwht_lanes<8>(x, lane, n);
  if (n == 16) {
    const uint32_t sg = (lane & 1) ? 0x80000000u : 0u;
#pragma unroll
    for (int j = 0; j < EPL; ++j) x[j] = as_f(as_u(x[j]) ^ sg) + lane_xor<1>(x[j]);
  }
}

template <typename T, int ROUND>
__device__ __forceinline__ void hq_store_chunk(const HqArgs& a, const float* x, float d, float rcp, uint64_t e0, int8_t* out) {
  uint32_t q[EPL];
  if constexpr (ROUND == HOT_ROUND_NEAREST) quant_nearest<T>(x, d, rcp, q);
  else quant_stoch(x, rcp, e0, a.seed, a.stream, (1 << (a.bits - 1)) - 1, q);
  if (a.bits == 4) store_codes4(q, out);
  else store_codes8(q, out);
}

template <typename T> struct raw_chunk { uint4 v[EPL / vec_traits<T>::EPV]; };
template <typename T>
__device__ __forceinline__ raw_chunk<T> load_raw(const T* p) {
  raw_chunk<T> r;
#pragma unroll
  for (int i = 0; i < EPL / vec_traits<T>::EPV; ++i) r.v[i] = reinterpret_cast<const uint4*>(p)[i];
  return r;
}
template <typename T>
__device__ __forceinline__ void unpack_raw(const raw_chunk<T>& r, float* x) {
#pragma unroll
  for (int i = 0; i < EPL / vec_traits<T>::EPV; ++i) unpack_vec<T>(r.v[i], x + i * vec_traits<T>::EPV);
}

template <typename T, int ROUND, int C>
__device__ __forceinline__ void hq_row_body(const HqArgs& a, int64_t row, int lanes, int t, float* s_red) {
  const int lane = threadIdx.x & 63;
  const int nch = (int)a.nch_row;
  const T* rp = reinterpret_cast<const T*>(a.in) + row * a.K;
  const int t0 = __builtin_amdgcn_readfirstlane(t);                       // of the wave's first lane: a wave without a c-th chunk skips it
  raw_chunk<T> raw[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if (t0 + c * lanes >= nch) break;
    const int ch = t + c * lanes;
    raw[c] = load_raw<T>(rp + (int64_t)(ch < nch ? ch : 0) * EPL);       // (the first chunk again where there is none: never used)
  }
  float x[C][EPL], mx = 0.f;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if (t0 + c * lanes >= nch) break;
    unpack_raw<T>(raw[c], x[c]);
    fwht_lanes_short(x[c], lane, a.n);
    if (t + c * lanes < nch) {
#pragma unroll
      for (int j = 0; j < EPL; ++j) mx = fmaxf(mx, fabsf(x[c][j]));
    }
  }
  mx = wave_max(mx);
  if (lanes > 64) {
    if (lane == 0) s_red[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  }
  const float s = mx / (float)((1 << (a.bits - 1)) - 1);
  const float d = s + 1e-11f, rcp = 1.0f / d;
  if (t == 0) a.scales[row] = s;
  int8_t* orow = a.codes + row * a.ld;
  const int cb = EPL * a.bits / 8;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if (t0 + c * lanes >= nch) break;
    const int ch = t + c * lanes;
    if (ch < nch) hq_store_chunk<T, ROUND>(a, x[c], d, rcp, (uint64_t)row * (uint64_t)a.K + (uint64_t)ch * EPL, orow + (int64_t)ch * cb);
  }
  const int pad0 = nch * cb, pad = (int)(a.ld - pad0) / 4;
  for (int i = t; i < pad; i += lanes) *reinterpret_cast<uint32_t*>(orow + pad0 + i * 4) = 0u;
}

// workgroups of the body for a tensor
inline int64_t hq_body_blocks(const HqArgs& a) {
  if (a.per_row) return a.nch_row <= 512 ? (a.M + 3) / 4 : a.M;
  return (int64_t)a.wgs * a.groups;
}

template <typename T, int ROUND>
__device__ __forceinline__ void hq_body(const HqArgs& a, unsigned block) {
  __shared__ float s_red[4];
  const int tid = threadIdx.x, lane = tid & 63;
  if (a.per_row) {
    const bool wide = a.nch_row > 512;                 // more than a wave holds
    const int64_t row = wide ? (int64_t)block : (int64_t)block * 4 + (tid >> 6);
    if (row >= a.M) return;
    const int lanes = wide ? 256 : 64, t = wide ? tid : lane;
    const int c = (int)(a.nch_row + lanes - 1) / lanes;
    if (c <= 3) hq_row_body<T, ROUND, 3>(a, row, lanes, t, s_red);
    else if (c <= 6) hq_row_body<T, ROUND, 6>(a, row, lanes, t, s_red);
    else hq_row_body<T, ROUND, 8>(a, row, lanes, t, s_red);
    return;
  }
  const unsigned g = a.groups > 1 ? block / a.wgs : 0u, b = block - g * a.wgs;
  const uint32_t c0 = b * (256u * HQ_UNROLL) + tid;
  const T* in = reinterpret_cast<const T*>(a.in) + (int64_t)g * a.chunks * EPL;
  raw_chunk<T> raw[HQ_UNROLL];
#pragma unroll
  for (int u = 0; u < HQ_UNROLL; ++u) {
    const uint32_t ch = c0 + u * 256u;
    raw[u] = load_raw<T>(in + (int64_t)(ch < a.chunks ? ch : a.chunks - 1) * EPL);   // (the last chunk again past the end: never stored)
  }
  float m = wave_max(part_max(a.stat + (int64_t)g * a.nstat * a.stat_stride, a.nstat, a.stat_stride, tid));
  if (lane == 0) s_red[tid >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  const float s = m / (float)((1 << (a.bits - 1)) - 1);
  const float d = s + 1e-11f, rcp = 1.0f / d;
  if (a.groups == 1 && b == 0 && tid == 0) a.scales[0] = s;
  const int cb = EPL * a.bits / 8;
  const bool dense = a.groups == 1 && a.ld == (int64_t)a.nch_row * cb;
#pragma unroll
  for (int u = 0; u < HQ_UNROLL; ++u) {
    const uint32_t ch = c0 + u * 256u;
    float x[EPL];
    unpack_raw<T>(raw[u], x);
    fwht_lanes_short(x, lane, a.n);
    if (ch >= a.chunks) continue;
    const uint64_t cht = (uint64_t)g * a.chunks + ch;
    if (dense) {
      hq_store_chunk<T, ROUND>(a, x, d, rcp, cht * EPL, a.codes + (int64_t)cht * cb);
      continue;
    }
    const uint32_t row = hq_row_of(a, ch), col = ch - row * a.nch_row;
    const int64_t grow = (int64_t)g * a.rows + row;
    int8_t* orow = a.codes + grow * a.ld;
    if (a.groups > 1 && col == 0) a.scales[grow] = s;
    hq_store_chunk<T, ROUND>(a, x, d, rcp, cht * EPL, orow + (int64_t)col * cb);
    if (col + 1 == a.nch_row)
      for (int64_t p = (int64_t)a.nch_row * cb; p < a.ld; p += 4) *reinterpret_cast<uint32_t*>(orow + p) = 0u;
  }
}

}  // namespace hot
