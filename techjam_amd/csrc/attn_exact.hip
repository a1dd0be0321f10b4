// Exact causal / right-padded scaled-dot-product attention for gfx950: the
// C ABI entry points and the choice of kernel instance per call (query rows
// per workgroup, key tile width, split scores). The kernel itself, its
// work decomposition and numerics are in attn_exact_kernel.h.
#include "attn_exact_kernel.h"

namespace tj {
namespace {

// Shortest part, in key tiles, and the tiles a sweep must be longer than a part
// for the split to pay for the partial sums and the second kernel.
constexpr int64_t kMinPart = 8;
constexpr int64_t kPartGain = 12;

// Two query blocks per wave halve LDS operand traffic and staging per MFMA.
// They fit the register budget for head_dim <= 64 (with split scores only at
// head_dim 64 with 32-key tiles, fp32 inputs), and need sequences long enough
// to fill 256-row tiles. Launches with fewer than 1024 such tiles (two per CU)
// keep 128-row tiles: there the heaviest tile sets the time, and a 32-row
// block per wave halves its per-key-tile work.
template <typename T, int HD>
int launch(const AttnArgs& a, hipStream_t stream) {
  if constexpr (HD <= 64) {
    const int64_t wide_tiles = int64_t(a.B) * a.H * ((a.S + 255) / 256);
    if (a.S >= 512 && wide_tiles >= 1024) {
      if (a.qk_split == nullptr) return launch_qb<T, HD, 2>(a, stream);
      // Split scores carry K's low half and Q's as well: two query blocks
      // per wave fit only with 32-key tiles (fp32 inputs, head_dim 64).
      if constexpr (HD == 64 && sizeof(T) == 4) return launch_split_wide(a, stream);
    }
  }
  // Wide fp32 heads on 32-key tiles where 64-key tiles do not fit the
  // registers: head_dim 256 spilled 49 of its 512 (B=64 H=4 S=128 41.5 -> 32.1
  // us, B=4 H=16 S=4096 causal 2243 -> 1298 us, not causal 4589 -> 2541), and
  // split scores at 128 took 363, one wave per SIMD (same shapes 22.8 -> 20.1,
  // 887 -> 706, 1658 -> 1262). Plain head_dim 128 fits and stays on 64 keys
  // (413 us against 439 on 32).
  if constexpr (sizeof(T) == 4 && HD == 256) {
    return launch_qb<T, HD, 1, 32>(a, stream);
  } else {
    if constexpr (sizeof(T) == 4 && HD == 128)
      if (a.qk_split != nullptr) return launch_qb<T, HD, 1, 32>(a, stream);
    return launch_qb<T, HD, 1>(a, stream);
  }
}

// Key parts, where the longest key sweep of a 128-row query tile is at least
// 2.5 times what an even split of all key tiles over the chip's workgroup
// slots gives, and (below head_dim 256) longer than a part by two key tiles and
// one for every 18 parts whose sums go through memory; part_tiles 0: none. Measured (us, one
// sweep -> parts, causal, head_dim 64 fp32): 1 head of 2048 33 -> 16, of 8192
// 114 -> 31, of 16 384 224 -> 74; 4 heads of 4096 61 -> 31, 8 of 2048 34 -> 25.
// Past the first line the parts cost as much as they save: 16 heads of 4096
// fp32 73 -> 73, fp16 68 -> 69, head_dim 128 121 -> 132 and 105 -> 121; 32 of
// 2048 40 -> 46, fp16 36 -> 43. The second is that of 1400 random calls near it
// (all head dims and types, half of them padded): without it 137 were slower in
// parts, 16 heads of 1375 not causal 26 -> 32, 12 of 2014 x 128 62 -> 66; with
// it 11, all padded to about twice their length, and none at head_dim 256
// either way.
struct PartPlan {
  int part_tiles = 0, n_parts = 0, n_mtiles = 0;
};

PartPlan plan_parts(int64_t B, int64_t H, int64_t S, int64_t D, int causal) {
  PartPlan p;
  const int64_t nm = (S + 127) / 128, nk = (S + 63) / 64, bhn = B * H;
  if (bhn * nm > 4096) return p;
  // Two workgroups on each of 256 CUs; one at head_dim 256.
  const int64_t slots = D == 256 ? 256 : 512;
  const int64_t all = bhn * (causal ? nm * (nm + 1) : nm * nk);
  int64_t part = (all + slots - 1) / slots;
  part = part < kMinPart ? kMinPart : part;
  part += part & 1;  // whole 128-row steps
  if (nk < part + kPartGain || 2 * nk < 5 * part) return p;
  const int64_t n_parts = first_part((int)nm, (int)nk, (int)part, causal);
  const int64_t whole = causal ? (nm < part / 2 ? nm : part / 2) : 0;  // tiles of one part
  if (D != 256 && 18 * (nk - part - 2) < bhn * (n_parts - whole)) return p;
  p.part_tiles = (int)part;
  p.n_mtiles = (int)nm;
  p.n_parts = (int)n_parts;
  return p;
}

template <typename T>
int dispatch_hd(const AttnArgs& a, int64_t D, hipStream_t stream) {
  switch (D) {
    case 32: return launch<T, 32>(a, stream);
    case 64: return launch<T, 64>(a, stream);
    case 128: return launch<T, 128>(a, stream);
    case 256: return a.qk_split != nullptr ? TJ_ERR_UNSUPPORTED : launch<T, 256>(a, stream);
    default: return TJ_ERR_UNSUPPORTED;
  }
}

}  // namespace
}  // namespace tj

namespace {

int attn_fwd(const void* q, const void* k, const void* v, void* o, int dtype, int64_t B, int64_t H, int64_t S,
             int64_t D, const int64_t q_strides[4], const int64_t k_strides[4], const int64_t v_strides[4],
             const int64_t o_strides[4], float scale, int causal, const int32_t* valid_len,
             const int32_t* row_limit, const int32_t* qk_split, const float* q_bias, const float* v_bias,
             void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (dtype != TJ_F32 && dtype != TJ_F16) return TJ_ERR_DTYPE;
  if (B < 0 || H <= 0 || S < 0 || D <= 0) return TJ_ERR_SHAPE;
  // Tile indices fit 31 bits; the launch also checks that its grid fits the
  // 32-bit dispatch size.
  if (S >= (int64_t(1) << 30) || !tjh::product_below(int64_t(1) << 31, {B, H, (S + 127) / 128})) return TJ_ERR_SHAPE;
  if (D != 32 && D != 64 && D != 128 && D != 256) return TJ_ERR_UNSUPPORTED;
  if (B == 0 || S == 0) return TJ_OK;
  if (!q || !k || !v || !o) return TJ_ERR_SHAPE;
  if (!tjh::view_ok(q, q_strides, dtype) || !tjh::view_ok(k, k_strides, dtype) ||
      !tjh::view_ok(v, v_strides, dtype) || !tjh::view_ok(o, o_strides, dtype))
    return TJ_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(q_bias) | reinterpret_cast<uintptr_t>(v_bias)) & 15u) return TJ_ERR_ALIGN;
  // K and V rows of one (b, h) are addressed with 31-bit byte offsets.
  for (const int64_t* st : {k_strides, v_strides})
    if (!tjh::span_below_2g(S, st[2], D, tjh::elem_size(dtype))) return TJ_ERR_UNSUPPORTED;

  tj::AttnArgs a;
  a.q = q; a.k = k; a.v = v; a.o = o;
  a.vq = {q_strides[0], q_strides[1], q_strides[2]};
  a.vk = {k_strides[0], k_strides[1], k_strides[2]};
  a.vv = {v_strides[0], v_strides[1], v_strides[2]};
  a.vo = {o_strides[0], o_strides[1], o_strides[2]};
  a.B = (int)B; a.H = (int)H; a.S = (int)S;
  a.qscale = scale * 1.4426950408889634f;
  a.causal = causal ? 1 : 0;
  a.valid_len = valid_len;
  a.row_limit = row_limit;
  a.qk_split = qk_split;
  a.q_bias = q_bias;
  a.v_bias = v_bias;
  const tj::PartPlan plan = workspace != nullptr ? tj::plan_parts(B, H, S, D, a.causal) : tj::PartPlan();
  if (plan.part_tiles > 0) {
    if (workspace_bytes < tj_attn_workspace_bytes(B, H, S, D, causal) || !tjh::aligned16(workspace)) return TJ_ERR_WORKSPACE;
    a.part_tiles = plan.part_tiles;
    a.n_parts = plan.n_parts;
    a.n_mtiles = plan.n_mtiles;
    a.part_o = static_cast<float*>(workspace);
    a.part_ml = a.part_o + B * H * plan.n_parts * 128 * D;
    return dtype == TJ_F32 ? tj::dispatch_parts_f32(a, D, stream) : tj::dispatch_parts_f16(a, D, stream);
  }
  if (dtype == TJ_F32) return tj::dispatch_hd<float>(a, D, stream);
  return tj::dispatch_hd<half_t>(a, D, stream);
}

}  // namespace

extern "C" int tj_attn_fwd(const void* q, const void* k, const void* v, void* o, int dtype,
                           int64_t B, int64_t H, int64_t S, int64_t D,
                           const int64_t q_strides[4], const int64_t k_strides[4],
                           const int64_t v_strides[4], const int64_t o_strides[4],
                           float scale, int causal, const int32_t* valid_len,
                           const int32_t* row_limit, const int32_t* qk_split, hipStream_t stream) {
  return attn_fwd(q, k, v, o, dtype, B, H, S, D, q_strides, k_strides, v_strides, o_strides, scale, causal,
                  valid_len, row_limit, qk_split, nullptr, nullptr, nullptr, 0, stream);
}

extern "C" int tj_attn_fwd_proj_bias(const void* q, const void* k, const void* v, void* o, int dtype,
                                     int64_t B, int64_t H, int64_t S, int64_t D,
                                     const int64_t q_strides[4], const int64_t k_strides[4],
                                     const int64_t v_strides[4], const int64_t o_strides[4],
                                     float scale, int causal, const int32_t* valid_len,
                                     const float* q_bias, const float* v_bias, hipStream_t stream) {
  return attn_fwd(q, k, v, o, dtype, B, H, S, D, q_strides, k_strides, v_strides, o_strides, scale, causal,
                  valid_len, nullptr, nullptr, q_bias, v_bias, nullptr, 0, stream);
}

extern "C" size_t tj_attn_workspace_bytes(int64_t B, int64_t H, int64_t S, int64_t D, int causal) {
  if (B <= 0 || H <= 0 || S <= 0 || S >= (int64_t(1) << 30) || (D != 32 && D != 64 && D != 128 && D != 256)) return 0;
  if (!tjh::product_below(int64_t(1) << 31, {B, H, (S + 127) / 128})) return 0;
  const tj::PartPlan p = tj::plan_parts(B, H, S, D, causal);
  if (p.part_tiles == 0) return 0;
  return size_t(B) * size_t(H) * size_t(p.n_parts) * 128 * size_t(D + 2) * sizeof(float);
}

extern "C" int tj_attn_fwd_ws(const void* q, const void* k, const void* v, void* o, int dtype,
                              int64_t B, int64_t H, int64_t S, int64_t D,
                              const int64_t q_strides[4], const int64_t k_strides[4],
                              const int64_t v_strides[4], const int64_t o_strides[4],
                              float scale, int causal, const int32_t* valid_len, const int32_t* qk_split,
                              const float* q_bias, const float* v_bias,
                              void* workspace, size_t workspace_bytes, hipStream_t stream) {
  return attn_fwd(q, k, v, o, dtype, B, H, S, D, q_strides, k_strides, v_strides, o_strides, scale, causal,
                  valid_len, nullptr, qk_split, q_bias, v_bias, workspace, workspace_bytes, stream);
}
