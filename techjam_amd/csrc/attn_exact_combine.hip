// Adds the key parts of the exact-attention kernel (attn_parts_kernel). A unit
// of its own, with IEEE NaN semantics: a NaN sum has to reach its row whatever
// the other parts hold, and the units of the attention kernels are built with
// -fno-honor-nans for their max chains. Bound by the parts' round trip through
// memory, this kernel has nothing to gain from that.
#include "attn_exact_kernel.h"

namespace tj {
namespace {

// Adds the parts of one query tile: out = sum_p 2^(m_p - M) O_p / sum_p
// 2^(m_p - M) l_p (+ v bias), zero for rows at or past the valid length. One
// row per HD / 4 lanes and thread, the loads of several parts in flight: with
// a tile's rows and parts one after another its latency was most of the call.
template <typename T, int HD>
__global__ __launch_bounds__(NT) void combine_parts_kernel(AttnArgs a) {
  constexpr int LPR = HD / 4, RPB = NT / LPR;  // lanes per row, rows per workgroup
  const int tile = blockIdx.x / (128 / RPB);
  const int bh = tile / a.n_mtiles, mt = tile % a.n_mtiles;
  const int nk = (a.S + 63) / 64;
  const int r = blockIdx.x % (128 / RPB) * RPB + threadIdx.x / LPR, qi = mt * 128 + r;
  if (tile_parts(mt, nk, a.part_tiles, a.causal) == 1 || qi >= a.S) return;
  const int b = bh / a.H, h = bh % a.H;
  int L = a.S;
  if (a.valid_len != nullptr) L = min(a.S, max(0, a.valid_len[b]));
  const int c = 4 * (threadIdx.x % LPR);
  float4_t y = {0.f, 0.f, 0.f, 0.f};
  if (qi < L) {
    using float2_t = float __attribute__((ext_vector_type(2)));
    const int64_t slot0 = int64_t(bh) * a.n_parts + first_part(mt, nk, a.part_tiles, a.causal);
    const float2_t* ml = reinterpret_cast<const float2_t*>(a.part_ml) + slot0 * 128 + r;
    const float* po = a.part_o + (slot0 * 128 + r) * HD + c;
    const int np = live_parts(mt, L, a.part_tiles, a.causal);
    float m = -__builtin_inff();
#pragma unroll 8
    for (int p = 0; p < np; ++p) {
      const float2_t x = ml[p * 128];
      m = has_keys(x[1]) ? fmaxf(m, x[0]) : m;
    }
    float l = 0.f;
#pragma unroll 4
    for (int p = 0; p < np; ++p) {
      const float2_t x = ml[p * 128];
      const float4_t o = *reinterpret_cast<const float4_t*>(po + (int64_t)p * 128 * HD);
      const float wgt = has_keys(x[1]) ? fast_exp2(x[0] - m) : 0.f;  // a part without keys holds zeros
      l += wgt * x[1];
      y += wgt * o;
    }
    const float4_t bv = a.v_bias != nullptr ? *reinterpret_cast<const float4_t*>(a.v_bias + h * HD + c) : float4_t{0.f, 0.f, 0.f, 0.f};
    const bool live = l > 0.f;
    const float inv = live ? 1.f / l : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = y[e] * inv + (live ? bv[e] : 0.f);  // NaN stays NaN, as in one sweep
  }
  T* op = reinterpret_cast<T*>(a.o) + a.vo.row(b, h, qi) + c;
  if constexpr (sizeof(T) == 4) *reinterpret_cast<float4_t*>(op) = y;
  else *reinterpret_cast<half4_t*>(op) = half4_t{(half_t)y[0], (half_t)y[1], (half_t)y[2], (half_t)y[3]};
}

template <typename T, int HD>
int launch(const AttnArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL((combine_parts_kernel<T, HD>), dim3(uint32_t(int64_t(a.B) * a.H * a.n_mtiles * (HD / 8))), dim3(NT),
                     0, stream, a);
  return tjh::launch_status();
}

template <typename T>
int dispatch(const AttnArgs& a, int64_t D, hipStream_t stream) {
  switch (D) {
    case 32: return launch<T, 32>(a, stream);
    case 64: return launch<T, 64>(a, stream);
    case 128: return launch<T, 128>(a, stream);
    default: return launch<T, 256>(a, stream);
  }
}

}  // namespace

int combine_parts_f32(const AttnArgs& a, int64_t D, hipStream_t stream) { return dispatch<float>(a, D, stream); }
int combine_parts_f16(const AttnArgs& a, int64_t D, hipStream_t stream) { return dispatch<half_t>(a, D, stream); }

}  // namespace tj
