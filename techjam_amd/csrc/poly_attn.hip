// Chunked causal degree-2 polynomial linear attention for gfx950 (D = 64, chunk 512).
//
// Replaces the reference's chunk scan (src/implementations/poly_reference.py:162-249)
// and its Triton kernels quad_apply / quad_update / causal_diag
// (src/kernels/poly_attention_triton.py:151-257, :420-591). With a = q*sqrt(scale),
// b = k*sqrt(scale) (fp16) and per-head coefficients (c0, c1, c2), chunk
// [t0, t1) emits for each row i
//   num = c0*S_const + c1*a.S_lin + c2*phi2(a).S_quad + sum_{t0<=j<=i} exp(a_i.b_j) v_j
//   den = c0*t0      + c1*a.z    + c2*a^T G a        + sum_{t0<=j<=i} exp(a_i.b_j)
// and the states fold in the chunk afterwards:
//   S_quad[(i,j), v] += sum_t b_ti b_tj v_tv,  S_lin[j, v] += sum_t b_tj v_tv,
//   G[i, j] += sum_t b_ti b_tj,  z[j] += sum_t b_tj,  S_const[v] += sum_t v_tv.
//
// Launches advance one window of KG = 16 chunks at a time; in launch L every
// head owns workgroups with five roles (P, 1 or 2, is the split below):
//   * apply (2 per chunk, 256 rows each, for the KG chunks whose start
//     states the previous launch produced): quadratic term as
//       y^T = sum_i S_i^T (a_i * a^T)  (S_i = rows (i, .) of S_quad),
//     i.e. 64 MFMA GEMMs whose B operand is the fp16 product a_i*a_j built in
//     registers -- phi2(a) never exists in memory; linear and denominator terms
//     as three more small GEMMs; the exact diagonal block like the exact
//     kernel (S^T = b a^T in registers, no max subtraction).
//   * state update (6 quad + 1 small per head and part): S_i += (b_i * b)^T v
//     over the tokens of the part's KG / P chunks of window L, accumulated
//     straight into MFMA accumulators that hold the fp32 state in its register
//     image (the state's memory layout IS the accumulator layout, so loading
//     and storing it is straight 16-byte copies); S_lin, G, z, S_const
//     likewise. A part starts from the state at the window's start plus the
//     sums of the parts before it; the last part stores the next window's
//     start. After each chunk it writes the fp16 shadow of the state the apply
//     of the next chunk reads.
//   * part sums (7 per head for each part of window L + 1 but the last, when
//     P > 1): the same folding from zero, without shadows, into an fp32 sum.
//   * token images (KG per head): b = k*sqrt(scale) and v of a later window
//     (L + 1; L + 2 when P > 1), converted once to fp16 tiles laid out as
//     the LDS image the state roles and the applies' diagonal blocks then
//     stream with direct global->LDS copies.
// State c (before chunk c) lives in shadow slot c % (2 KG): a launch reads
// the slots of states KG L - KG + 1 .. KG L and writes those of KG L + 1 ..
// KG L + KG, so applies and updates of one launch never touch the same slot.
// Window starts, part sums and images are buffered by window, so that no role
// of a launch writes what another one reads.
// More chunks per launch load and store each state less often and need
// fewer launches (the polynomial call on 64 heads of 65536 tokens: 4 -> 8
// chunks 5.8-6.1 -> 5.4-5.5 ms; the extreme step with 8 -> 16 chunks
// 8.99-9.02 -> 8.78-8.83 ms, 10.2 MiB more workspace per head).
//
// Parts. A window is a chain of KG * 8 token tiles for each update workgroup
// (~0.8 us a tile), while seven of them per head leave the chip idle for a
// few heads. P parts fold KG / P chunks each, all at once, at the price of
// folding all but one part twice; see parts_for().
#include <type_traits>

#include "tj_common.h"

namespace tj {
namespace {

constexpr int PD = 64;         // head dim (d = dv)
constexpr int PC = 512;        // chunk length
constexpr int PT = 256;        // threads per workgroup
constexpr int NAPPLY = 2;      // apply workgroups per head and chunk (256 rows each)
constexpr int NUPD = 6;        // quad-update workgroups per head (4 for i < 32, 2 for i >= 32)
constexpr int KG = 16;         // chunks per launch (update sub-chunks, apply groups)
constexpr int NSLOT = 2 * KG;  // shadow slots: state_c lives in slot c % NSLOT
constexpr int NCONV = KG;      // token-image workgroups per head (one chunk each)
constexpr int NSTATE = NUPD + 1;  // state-update workgroups per head and part
constexpr int PMAX = 2;        // most parts of a window
constexpr int NIMG = 4;        // token-image buffers: window w in buffer w % NIMG
constexpr int kBufferFlags = 0x00020000;  // raw (untyped) buffer resource word 3 on gfx950

// One state (byte offsets): S_quad without the j < 32 blocks of i >= 32, which
// nothing reads (S_ij = S_ji), in accumulator images of [64 lanes][16] fp32.
constexpr uint32_t kImg = 64 * 16 * 4;
constexpr uint32_t kStQuad = 0;                        // [i < 32][2 jb][2 vb], then [i >= 32][2 vb] (jb = 1)
constexpr uint32_t kStLin = (32 * 4 + 32 * 2) * kImg;  // [2 jb][2 vb]
constexpr uint32_t kStGram = kStLin + 4 * kImg;        // [2 ib][2 jb]
constexpr uint32_t kStZs = kStGram + 4 * kImg;         // fp32 z[64], S_const[64]
constexpr uint32_t kStateBytes = kStZs + 128 * 4;
__host__ __device__ constexpr uint32_t quad_img(int i, int jb, int vb) {
  return kStQuad + (i < 32 ? (i * 2 + jb) * 2 + vb : 128 + (i - 32) * 2 + vb) * kImg;
}
// fp16 quad shadow of one state, piece-major: for each i the pieces q = j / 8
// >= 2 (i / 16) that the apply reads, [q][64 v][8 j] (1 KiB each).
__host__ __device__ constexpr uint32_t quad_shadow(int i) {
  const int ib = i >> 4;
  return 1024u * (16 * (9 * ib - ib * ib) + (i & 15) * (8 - 2 * ib));
}
constexpr uint32_t kShadowBytes = quad_shadow(64);
static_assert(quad_shadow(16) == 1024 * 128 && quad_shadow(32) == 1024 * 224 && kShadowBytes == 1024 * 320, "pieces");

// Workspace of one head (byte offsets).
constexpr uint32_t kStart = 0;                                  // window starts [2][kStateBytes]
constexpr uint32_t kPart = kStart + 2 * kStateBytes;             // part sums [2][PMAX - 1][kStateBytes]
constexpr uint32_t kQuadShadow = kPart + 2 * (PMAX - 1) * kStateBytes;  // fp16 [NSLOT][kShadowBytes]
constexpr uint32_t kLinShadow = kQuadShadow + NSLOT * kShadowBytes;     // fp16 [NSLOT][64 v][64 j]
constexpr uint32_t kGramShadow = kLinShadow + NSLOT * PD * PD * 2;      // fp16 [NSLOT][64][64] (symmetric)
constexpr uint32_t kZsShadow = kGramShadow + NSLOT * PD * PD * 2;       // fp32 [NSLOT][128]
// Token images: the k (scaled) and v tiles of a window, as fp16 LDS images
// (see TokTile).
constexpr int kTileImg = 2 * PD * 64 * 2;                            // [b^T | v^T] of 64 tokens
constexpr uint32_t kTokImgBytes = uint32_t(KG) * (PC / 64) * kTileImg;  // one window: 2 MiB
constexpr uint32_t kTokImg = (kZsShadow + NSLOT * 128 * 4 + 255) & ~255u;  // [NIMG][kTokImgBytes]
constexpr size_t kPerHead = size_t(kTokImg) + NIMG * kTokImgBytes;

// LDS: apply = quad-state ring, then token tiles; updates = token tiles
// (three stages of 16 KiB each).
constexpr int kRing = 3;                        // quad-state stages in flight
constexpr int kRingStage = 2 * PD * PD * 2;     // one stage: rows of two i, [2][64 v][64 j] fp16
constexpr int kStageBytes = kRing * kRingStage;
static_assert(kPerHead < (size_t(1) << 31), "workspace offsets of one head fit a buffer resource");
constexpr int kSmemBytes = kStageBytes;

struct PolyArgs {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  View4 vq, vk, vv, vo;
  int H, S;
  float rs;             // sqrt(scale)
  int launch;           // launch index L: applies chunks (KG (L-1), KG L], updates [KG L, KG L + KG)
  int parts;            // P
  int n_chunks;
  int prefix_end;       // rows below are left to the exact kernel
  const float* coeffs;  // [M][3]
  const int32_t* flags; // [M] or null
  char* ws;
  int M;                // B * H
};

// One direct global->LDS copy of a wave: 16 bytes per lane from byte offset
// soff + voff of the head's workspace to lds + 16 * lane. A buffer load, not
// global_load_lds: the compiler counts that one as a FLAT access, and while
// one is in flight turns every wait for an LDS read into lgkmcnt(0), so that
// reads issued ahead of the MFMAs they feed would be waited for at once.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t head_rsrc(const char* ws) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(ws), (short)0, (int)kPerHead, kBufferFlags);
}
__device__ __forceinline__ void copy_to_lds(__amdgpu_buffer_rsrc_t r, char* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}

__device__ __forceinline__ float4_t ld4(const float* p) { return *reinterpret_cast<const float4_t*>(p); }

template <typename T>
__device__ __forceinline__ void load_row4(const T* p, float out[4]) {
  if constexpr (sizeof(T) == 4) {
    const float4_t x = *reinterpret_cast<const float4_t*>(p);
    out[0] = x[0]; out[1] = x[1]; out[2] = x[2]; out[3] = x[3];
  } else {
    const half4_t x = *reinterpret_cast<const half4_t*>(p);
    out[0] = (float)x[0]; out[1] = (float)x[1]; out[2] = (float)x[2]; out[3] = (float)x[3];
  }
}

// Global -> registers of one 64-token x 64-dim tile of k and v. Unit =
// (4-token group g, 4-dim group c); one unit per thread. Rows are read with
// bounds-checked buffer loads (one resource per (b, h) spanning rows 0..S-1),
// so tokens at or past S read as zeros without a branch, and nothing waits
// on the loads before the tile is stored: k is scaled by rs at the store.
template <typename T>
struct TokTile {
  // Raw rows as loaded (fp32 or fp16), converted at the stores: fp16 input
  // holds half the registers.
  using Raw = std::conditional_t<sizeof(T) == 4, float4_t, half4_t>;
  Raw kx[4];
  Raw vx[4];
  __amdgpu_buffer_rsrc_t rk, rv;
  uint32_t koff, voff, kstep, vstep;
  __device__ __forceinline__ static void coords(int tid, int& g, int& c) {
    g = (tid >> 2) & 15;
    c = (tid & 3) | ((tid >> 6) << 2);
  }
  __device__ __forceinline__ void init(const PolyArgs& a, int b, int h, int tid) {
    int g, c;
    coords(tid, g, c);
    const T* kp = reinterpret_cast<const T*>(a.k) + a.vk.row(b, h, 0);
    const T* vp = reinterpret_cast<const T*>(a.v) + a.vv.row(b, h, 0);
    kstep = (uint32_t)(a.vk.ss * (int64_t)sizeof(T));
    vstep = (uint32_t)(a.vv.ss * (int64_t)sizeof(T));
    const int kbytes = (int)((int64_t)(a.S - 1) * kstep + PD * (int64_t)sizeof(T));
    const int vbytes = (int)((int64_t)(a.S - 1) * vstep + PD * (int64_t)sizeof(T));
    rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(kp), (short)0, kbytes, kBufferFlags);
    rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(vp), (short)0, vbytes, kBufferFlags);
    koff = 4 * g * kstep + 4 * c * (uint32_t)sizeof(T);
    voff = 4 * g * vstep + 4 * c * (uint32_t)sizeof(T);
  }
  __device__ __forceinline__ void load(int tok0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (sizeof(T) == 4) {
        const float4_t x = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, koff, (tok0 + r) * kstep, 0));
        const float4_t y = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, voff, (tok0 + r) * vstep, 0));
        kx[r] = x;
        vx[r] = y;
      } else {
        const half4_t x = __builtin_bit_cast(half4_t, __builtin_amdgcn_raw_buffer_load_b64(rk, koff, (tok0 + r) * kstep, 0));
        const half4_t y = __builtin_bit_cast(half4_t, __builtin_amdgcn_raw_buffer_load_b64(rv, voff, (tok0 + r) * vstep, 0));
        kx[r] = x;
        vx[r] = y;
      }
    }
  }
  // The tile's LDS image for the update roles, stored to global memory:
  // [b^T | v^T], each 64 dim rows of 128 bytes (64 tokens), the eight
  // 16-byte pieces of row d at position piece ^ ((d >> 1) & 7) so that 16
  // lanes reading one piece column of 16 consecutive rows hit distinct banks.
  __device__ __forceinline__ void store_image(char* dst, float rs, int tid) const {
    int g, c;
    coords(tid, g, c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = 4 * c + e;
      const int off = d * 128 + 16 * ((g >> 1) ^ ((d >> 1) & 7)) + 8 * (g & 1);
      *reinterpret_cast<half4_t*>(dst + off) =
          half4_t{(half_t)((float)kx[0][e] * rs), (half_t)((float)kx[1][e] * rs), (half_t)((float)kx[2][e] * rs),
                  (half_t)((float)kx[3][e] * rs)};
      *reinterpret_cast<half4_t*>(dst + PD * 128 + off) =
          half4_t{(half_t)vx[0][e], (half_t)vx[1][e], (half_t)vx[2][e], (half_t)vx[3][e]};
    }
  }
};

// x * s as four packed multiplies. (Element by element the compiler emits
// eight scalar multiplies and four packs.)
__device__ __forceinline__ half8_t mul8(half8_t x, half_t s) { return x * half8_t{s, s, s, s, s, s, s, s}; }

// Three LDS stages of one token image each.
struct TokRing {
  char s0[kTileImg];
  char s1[kTileImg];
  char s2[kTileImg];
};
static_assert(sizeof(TokRing) <= kStageBytes, "the token ring must fit the ring area");

// Tokens 8 pc .. 8 pc + 7 of dim row `row` of a tile image.
__device__ __forceinline__ half8_t img_piece(const half_t* base, int row, int pc) {
  return *reinterpret_cast<const half8_t*>(reinterpret_cast<const char*>(base) + row * 128 + 16 * (pc ^ ((row >> 1) & 7)));
}

// Eight dims d0 .. d0 + 7 (d0 = 16 ks + 8 (lane / 32)) of one token of a b^T
// image per lane: the A operand of a score MFMA, by two transposing reads (16
// lanes read 4 dim rows of 16 tokens and get one token's 4 dims each). Lane
// row rho = lane % 32 gets token tok0 + rho with bits 2 and 3 of rho swapped,
// so that accumulator element r of the scores holds token tok0 + 16 (r / 8) +
// 8 (lane / 32) + r % 8: eight consecutive tokens per 16-token step, the k-slots
// that img_piece gives the V^T operand.
__device__ __forceinline__ half8_t img_tokens(const half_t* bT, int tok0, int ks) {
  using s4 = short __attribute__((ext_vector_type(4)));
  using u4 = half4_t;
  const int lane = threadIdx.x % kWave, i = lane % 16, m = i % 4;
  const int tok = tok0 + (lane & 16) + 4 * (((m & 1) << 1) | (m >> 1));
  half8_t r;
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int d = 16 * ks + 8 * (lane / 32) + 4 * x + i / 4;
    const char* p = reinterpret_cast<const char*>(bT) + d * 128 + 16 * ((tok >> 3) ^ ((d >> 1) & 7)) + 2 * (tok & 4);
    const u4 v = __builtin_bit_cast(
        u4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)const_cast<char*>(p)));
#pragma unroll
    for (int j = 0; j < 4; ++j) r[4 * x + j] = v[j];
  }
  return r;
}

// ---------------------------------------------------------------------------
// Apply role: rows [row0, row0 + 256) of the chunk; each wave owns RB = 2
// blocks of 32 consecutive rows, so every state fragment read from LDS feeds
// two MFMAs and every ring stage serves 256 rows.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void apply_role(const PolyArgs& a, const char* ws, int b, int h, int m, int c, int qt, char* smem) {
  constexpr int RB = 2;
  constexpr int WROWS = 32 * RB;
  const int t0 = c * PC, t1 = min(a.S, t0 + PC), slot = c % NSLOT;
  const int row0 = t0 + 4 * WROWS * qt;
  if (row0 >= t1 || row0 + 4 * WROWS <= a.prefix_end) return;
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave, hl = lane / 32, ln = lane % 32;
  const int qw0 = row0 + WROWS * w;

  // a = fp16(q * rs); B operand slots (hl, j) <-> dim 16*ks + 8*hl + j.
  half8_t aB[RB][4];
  {
    const T* qp = reinterpret_cast<const T*>(a.q);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int qi = qw0 + 32 * rb + ln;
      const bool in = qi < t1;
      const int64_t base = a.vq.row(b, h, in ? qi : t0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        float x[8];
        load_row4<T>(qp + base + 16 * ks + 8 * hl, x);
        load_row4<T>(qp + base + 16 * ks + 8 * hl + 4, x + 4);
#pragma unroll
        for (int j = 0; j < 8; ++j) aB[rb][ks][j] = in ? (half_t)(x[j] * a.rs) : (half_t)0.f;
      }
    }
  }
  // Linear denominator a.z (z = S_lin's row sums, fp32 in the slot's small
  // shadow), taken while few registers are live.
  const float* zs = reinterpret_cast<const float*>(ws + kZsShadow) + slot * 128;
  float den_l[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    float dl = 0.f;
    if (c > 0)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) dl += (float)aB[rb][ks][j] * zs[16 * ks + 8 * hl + j];
    den_l[rb] = pair_sum(dl);
  }
  // a_i, a_i+1 (i = 2p) of this lane's query: dword p & 3 of aB[rb][p >> 3],
  // held by the lane half (p >> 2) & 1; the lane-pair swap hands it to both
  // (r[0] from the lower-half lane, r[1] from the upper, as in pair_values).
  auto a_pair = [&](int rb, int p) -> half2_t {
    using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
    const uint32_t u = __builtin_bit_cast(u32x4, aB[rb][p >> 3])[p & 3];
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __builtin_bit_cast(half2_t, ((p >> 2) & 1) ? r[1] : r[0]);
  };

  const __amdgpu_buffer_rsrc_t rws = head_rsrc(ws);
  const uint32_t qshadow = kQuadShadow + slot * kShadowBytes;
  // The quad shadow streams through a ring of kRing LDS stages by direct
  // global->LDS copies two stages ahead of the MFMAs (no registers held).
  // Pair p (i = 2p, 2p + 1) has the pieces q >= 2 ib, ib = p >> 3 (S is
  // symmetric, see the step), np = 8 - 2 ib of them per i, so a stage holds
  // G pairs (G = 1, 1, 2, 4 for ib = 0 .. 3, at most 16 KiB), contiguous in
  // the shadow: [2 gp + ii][q - 2 ib][64 v] 16-byte pieces, filled by 2 G np
  // copy instructions of 1 KiB (wave w issues k = w, w + 4, ...): 37.5 % fewer
  // bytes than whole rows, 22 stages instead of 32, and 16 lanes reading one
  // piece column of 16 consecutive rows touch 256 contiguous bytes. The stages
  // are distinct members addressed with compile-time indices, so the compiler
  // can tell the copies into one stage from reads of another and does not wait
  // for every copy in flight.
  struct Ring {
    char s0[kRingStage];
    char s1[kRingStage];
    char s2[kRingStage];
  };
  static_assert(kRing == 3, "the ring below has three members");
  Ring& ring = *reinterpret_cast<Ring*>(smem);
  auto stage_ptr = [&](auto st) -> char* {
    if constexpr (decltype(st)::value == 0) return ring.s0;
    else if constexpr (decltype(st)::value == 1) return ring.s1;
    else return ring.s2;
  };
  constexpr int kSteps = 22;
  auto step_p0 = [](int st) constexpr { return st < 16 ? st : (st < 20 ? 16 + 2 * (st - 16) : 24 + 4 * (st - 20)); };
  auto step_g = [](int st) constexpr { return st < 16 ? 1 : (st < 20 ? 2 : 4); };
  auto issue = [&](auto sc, auto st) {
    constexpr int p0 = step_p0(decltype(sc)::value), G = step_g(decltype(sc)::value);
    constexpr int ib = p0 >> 3, np = 8 - 2 * ib;
    static_assert(G * np * 2 <= 16, "a stage holds at most 16 KiB");
    char* base = stage_ptr(st);
#pragma unroll
    for (int it = 0; it < G * np / 2; ++it) {
      const int k = w + 4 * it;
      copy_to_lds(rws, base + k * 1024, lane * 16, qshadow + quad_shadow(2 * p0) + k * 1024);
    }
  };

  // accq: the quadratic numerator first; after the ring, scaled by c2 and
  // joined by c1 times the linear term and by the exact diagonal block.
  float16_t accq[RB][2];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int vb = 0; vb < 2; ++vb)
#pragma unroll
      for (int r = 0; r < 16; ++r) accq[rb][vb][r] = 0.f;

  // One ring step: MFMAs on the pairs of stage sc, after issuing stage sc + 2.
  auto step = [&](auto sc) {
    constexpr int si = decltype(sc)::value;
    constexpr int p0 = step_p0(si), G = step_g(si);
    constexpr int ib = p0 >> 3, np = 8 - 2 * ib;  // 16-block of every i of the stage
    if constexpr (si + 2 < kSteps) issue(std::integral_constant<int, si + 2>{}, std::integral_constant<int, (si + 2) % kRing>{});
    const char* base = stage_ptr(std::integral_constant<int, si % kRing>{});
    // phi2(a).S = sum_i a_i sum_j a_j S_ij with S_ij = S_ji (the update forms
    // both from the same fp16 products b_i b_j in the same order): the j-block
    // holding i counts once, j-blocks above it twice (a_i doubled, exact in
    // fp16), j-blocks below it not at -- 37.5 % fewer MFMAs.
#pragma unroll
    for (int gp = 0; gp < G; ++gp) {
      const int p = p0 + gp;
      half2_t ap[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) ap[rb] = a_pair(rb, p);
#pragma unroll
      for (int ii = 0; ii < 2; ++ii) {
#pragma unroll
        for (int ks = ib; ks < 4; ++ks) {
          const int k = (2 * gp + ii) * np + 2 * ks + hl - 2 * ib;
          half8_t sa[2];
#pragma unroll
          for (int vb = 0; vb < 2; ++vb) sa[vb] = *reinterpret_cast<const half8_t*>(base + k * 1024 + (32 * vb + ln) * 16);
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) {
            const half_t ai = ap[rb][ii];
            const half8_t bop = mul8(aB[rb][ks], ks == ib ? ai : (half_t)(ai + ai));
#pragma unroll
            for (int vb = 0; vb < 2; ++vb) accq[rb][vb] = mfma32(sa[vb], bop, accq[rb][vb]);
          }
        }
      }
    }
    // Stage sc + 1 (this wave's copies) must have landed before the barrier;
    // stage sc + 2 (G np / 2 copies of this wave) may stay in flight. A plain
    // barrier: __syncthreads() would also wait for every copy in flight.
    if constexpr (si + 2 < kSteps) {
      constexpr int in_flight = step_g(si + 2) * (8 - 2 * (step_p0(si + 2) >> 3)) / 2;
      __builtin_amdgcn_s_waitcnt(0x0070 | in_flight);  // vmcnt(in_flight) lgkmcnt(0)
    } else {
      __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    }
    lds_barrier();
  };
  if (c > 0) {  // the state before chunk 0 is zero, and no launch wrote it
    issue(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    issue(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
    __builtin_amdgcn_s_waitcnt(0x0074);  // stage 0 landed (stage 1: four copies in flight)
    lds_barrier();
    static_for<0, kSteps>(step);
  }

  // Exact diagonal block: keys [t0, min(t1, row0 + 256)), no max subtraction;
  // the weighted values accumulate straight into accq. The chunk's token
  // images, written by an earlier launch for the state updates, serve as its
  // K and V tiles through the same LDS area (fp32 K and V read again and
  // converted by every apply: 20 of its 69 us, and 2 GB per call of the
  // extreme workload). The first two copies go out before the linear terms.
  const int key_end = min(t1, row0 + 4 * WROWS);
  const int n_kt = (key_end - t0 + 63) / 64;
  const uint32_t img = kTokImg + uint32_t(c / KG % NIMG) * kTokImgBytes + uint32_t(c % KG) * (PC / 64) * kTileImg;
  TokRing& tiles = *reinterpret_cast<TokRing*>(smem);
  auto tile_ptr = [&](auto st) -> char* {
    if constexpr (decltype(st)::value == 0) return tiles.s0;
    else if constexpr (decltype(st)::value == 1) return tiles.s1;
    else return tiles.s2;
  };
  auto issue_tile = [&](int kt, auto st) {
#pragma unroll
    for (int it = 0; it < 4; ++it)
      copy_to_lds(rws, tile_ptr(st) + (4 * it + w) * 1024, lane * 16, img + kt * kTileImg + (4 * it + w) * 1024);
  };
  issue_tile(0, std::integral_constant<int, 0>{});
  if (n_kt > 1) issue_tile(1, std::integral_constant<int, 1>{});

  // Linear numerator term S_lin^T a^T and the quadratic denominator G a^T
  // (operands straight from the L2-resident shadows). G's rows are read in
  // the order that swaps bits 2 and 3 of the row index, so that accumulator
  // element r of this lane holds row 32 blk + 16 (r / 8) + 8 hl + r % 8 --
  // the dims this lane's own aB[rb][2 blk + r / 8][r % 8] holds -- and
  // a^T G a needs no other lane's a.
  const float c0 = a.coeffs[3 * m], c1 = a.coeffs[3 * m + 1], c2 = a.coeffs[3 * m + 2];
  const half_t* lsh = reinterpret_cast<const half_t*>(ws + kLinShadow) + size_t(slot) * PD * PD;
  const half_t* gsh = reinterpret_cast<const half_t*>(ws + kGramShadow) + size_t(slot) * PD * PD;
  const int grow = (ln & 0x13) | ((ln & 4) << 1) | ((ln & 8) >> 1);
  float den_q[RB], den_d[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) den_q[rb] = den_d[rb] = 0.f;
  // One 32-row block of S_lin^T (output block blk = v block) and of G at a time,
  // each fragment feeding both query blocks.
#pragma unroll
  for (int blk = 0; blk < (c > 0 ? 2 : 0); ++blk) {
    half8_t la[4], ga[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      la[ks] = *reinterpret_cast<const half8_t*>(lsh + (32 * blk + ln) * PD + 16 * ks + 8 * hl);
      ga[ks] = *reinterpret_cast<const half8_t*>(gsh + (32 * blk + grow) * PD + 16 * ks + 8 * hl);
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float16_t tl, tg;
#pragma unroll
      for (int r = 0; r < 16; ++r) tl[r] = tg[r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        tl = mfma32(la[ks], aB[rb][ks], tl);
        tg = mfma32(ga[ks], aB[rb][ks], tg);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        den_q[rb] += (float)aB[rb][2 * blk + r / 8][r % 8] * tg[r];
        accq[rb][blk][r] = c2 * accq[rb][blk][r] + c1 * tl[r];
      }
    }
  }
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) den_q[rb] = pair_sum(den_q[rb]);

  // Tile kt + 1 (this wave's four copies) must have landed before the barrier.
  auto wait_tile = [&](int kt) {
    if (kt + 2 < n_kt) __builtin_amdgcn_s_waitcnt(0x0074);  // vmcnt(4) lgkmcnt(0)
    else __builtin_amdgcn_s_waitcnt(0x0070);                // vmcnt(0) lgkmcnt(0)
    lds_barrier();
  };
  auto diag_tile = [&](int kt, auto st) {
    constexpr int sv = decltype(st)::value;
    if (kt + 2 < n_kt) issue_tile(kt + 2, std::integral_constant<int, (sv + 2) % 3>{});
    const half_t* bT = reinterpret_cast<const half_t*>(tile_ptr(st));
    const half_t* vT = bT + PD * 64;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      const int k0 = t0 + 64 * kt + 32 * kh;
      // Rows that all precede the 32 keys skip them.
      if (k0 > min(qw0 + WROWS - 1, key_end - 1)) continue;
      half8_t kf[4], vf[2][2];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) kf[ks] = img_tokens(bT, 32 * kh, ks);
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int vb = 0; vb < 2; ++vb) vf[x][vb] = img_piece(vT, 32 * vb + ln, 4 * kh + 2 * x + hl);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int qb0 = qw0 + 32 * rb;
        if (k0 > min(qb0 + 31, key_end - 1)) continue;
        float16_t sc;
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) sc = mfma32(kf[ks], aB[rb][ks], sc);
        half8_t pf[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) pf[r / 8][r % 8] = (half_t)fast_exp2(sc[r] * 1.4426950408889634f);
        if (k0 + 31 > qb0) {  // the causal edge crosses this block
          const int lim = qb0 + ln - k0 - 8 * hl;
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (16 * (r / 8) + r % 8 > lim) pf[r / 8][r % 8] = (half_t)0.f;
        }
        // den sums the rounded weights, as the value product multiplies them.
#pragma unroll
        for (int r = 0; r < 16; r += 2)
          den_d[rb] = __builtin_amdgcn_fdot2(half2_t{pf[r / 8][r % 8], pf[r / 8][r % 8 + 1]},
                                             half2_t{(half_t)1.f, (half_t)1.f}, den_d[rb], false);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int vb = 0; vb < 2; ++vb) accq[rb][vb] = mfma32(vf[x][vb], pf[x], accq[rb][vb]);
      }
    }
    wait_tile(kt);
  };
  wait_tile(-1);
  for (int kt = 0; kt < n_kt; kt += 3) {
    diag_tile(kt, std::integral_constant<int, 0>{});
    if (kt + 1 < n_kt) diag_tile(kt + 1, std::integral_constant<int, 1>{});
    if (kt + 2 < n_kt) diag_tile(kt + 2, std::integral_constant<int, 2>{});
  }

#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int qi = qw0 + 32 * rb + ln;
    const float dd = pair_sum(den_d[rb]);
    if (qi >= t1 || qi < a.prefix_end) continue;
    const float den = c0 * (float)t0 + c1 * den_l[rb] + c2 * den_q[rb] + dd;
    const float inv = 1.f / den;
    T* op = reinterpret_cast<T*>(a.o) + a.vo.row(b, h, qi);
#pragma unroll
    for (int vb = 0; vb < 2; ++vb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int v0 = 32 * vb + 8 * g + 4 * hl;
        const float4_t sc = c > 0 ? ld4(zs + 64 + v0) : float4_t{0.f, 0.f, 0.f, 0.f};
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = (c0 * sc[e] + accq[rb][vb][4 * g + e]) * inv;
        if constexpr (sizeof(T) == 4) {
          *reinterpret_cast<float4_t*>(op + v0) = float4_t{y[0], y[1], y[2], y[3]};
        } else {
          *reinterpret_cast<half4_t*>(op + v0) = half4_t{(half_t)y[0], (half_t)y[1], (half_t)y[2], (half_t)y[3]};
        }
      }
  }
}

// ---------------------------------------------------------------------------
// Update roles: fold the chunk's tokens into the states.
// ---------------------------------------------------------------------------

// The token images of the chunks this launch folds in stream through a ring
// of three LDS stages by direct global->LDS copies issued two tiles ahead (no
// registers held). A 64-token tile is four MFMA k-steps; load(bT, vT, ks)
// reads one step's operands (b^T and v^T, 64 dim rows of 128 bytes with
// XOR-placed 16-byte pieces, see img_piece) and mma(ops) consumes them. The
// operands of step ks + 1 -- across the tile boundary too -- are read before
// step ks's MFMAs, so the LDS latency is under them: with one or two waves
// per SIMD nothing else hides it (a tile took ~3000 cycles against 1024 of
// MFMA when each step read its own operands first). chunk_end(j) runs after
// the last tile of the launch's j-th chunk, once the
// workgroup has passed that tile's barrier: its global stores then complete
// under the next tile instead of holding up the wait for the copies (issued
// before them) that the barrier needs. The stages are
// distinct members addressed with compile-time indices, so the compiler can
// tell the copies into one stage from the reads of another.
template <typename Load, typename Mma, typename ChunkEnd>
__device__ __forceinline__ void stream_image(const char* ws, uint32_t img, int n_chunk, char* smem, Load&& load,
                                             Mma&& mma, ChunkEnd&& chunk_end) {
  constexpr int kTiles = PC / 64;
  TokRing& ring = *reinterpret_cast<TokRing*>(smem);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int n = n_chunk * kTiles;
  const __amdgpu_buffer_rsrc_t rws = head_rsrc(ws);
  auto stage_ptr = [&](auto st) -> char* {
    if constexpr (decltype(st)::value == 0) return ring.s0;
    else if constexpr (decltype(st)::value == 1) return ring.s1;
    else return ring.s2;
  };
  // Copy instruction `it` of wave w moves 1 KiB slot 4 it + w of the tile.
  auto issue = [&](int t, auto st) {
    char* base = stage_ptr(st);
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int slot = 4 * it + w;
      copy_to_lds(rws, base + slot * 1024, lane * 16, img + t * kTileImg + slot * 1024);
    }
  };
  // Tile t + 1 (this wave's four copies) must have landed before the barrier;
  // tile t + 2 may stay in flight (anything issued after it only makes the
  // wait longer). A plain barrier: __syncthreads() would also wait for every
  // copy in flight.
  auto wait_next = [&](int t) {
    if (t + 2 < n) __builtin_amdgcn_s_waitcnt(0x0074);  // vmcnt(4) lgkmcnt(0)
    else __builtin_amdgcn_s_waitcnt(0x0070);            // vmcnt(0) lgkmcnt(0)
    lds_barrier();
  };
  using Ops = decltype(load((const half_t*)nullptr, (const half_t*)nullptr, 0));
  Ops ops[2];
  auto load_ks = [&](char* base, int ks) {
    return load(reinterpret_cast<const half_t*>(base), reinterpret_cast<const half_t*>(base + PD * 128), ks);
  };
  auto step = [&](int t, auto st) {
    constexpr int sv = decltype(st)::value;
    if (t + 2 < n) issue(t + 2, std::integral_constant<int, (sv + 2) % 3>{});
    char* base = stage_ptr(st);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) {
        ops[(ks + 1) & 1] = load_ks(base, ks + 1);
      } else {
        // This wave's last operands of tile t are in registers (lgkmcnt(0)),
        // so past the barrier the tile's stage may be refilled.
        wait_next(t);
        if (t + 1 < n) ops[0] = load_ks(stage_ptr(std::integral_constant<int, (sv + 1) % 3>{}), 0);
      }
      // This step's operands are there; the next step's may stay in flight.
      if (ks < 3 || t + 1 < n) __builtin_amdgcn_s_waitcnt(0xC07F | (sizeof(Ops) / 16) << 8);
      __builtin_amdgcn_sched_barrier(0);
      mma(ops[ks & 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if ((t + 1) % kTiles == 0) chunk_end(t / kTiles);
  };
  if (n == 0) return;
  issue(0, std::integral_constant<int, 0>{});
  if (n > 1) issue(1, std::integral_constant<int, 1>{});
  wait_next(-1);
  ops[0] = load_ks(ring.s0, 0);
  for (int t = 0; t < n; t += 3) {
    step(t, std::integral_constant<int, 0>{});
    if (t + 1 < n) step(t + 1, std::integral_constant<int, 1>{});
    if (t + 2 < n) step(t + 2, std::integral_constant<int, 2>{});
  }
}

__device__ __forceinline__ void add_img(const char* img, float16_t& acc) {
  const int lane = threadIdx.x % kWave;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4_t x = ld4(reinterpret_cast<const float*>(img) + lane * 16 + 4 * q);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[4 * q + e] += x[e];
  }
}

__device__ __forceinline__ void store_img(char* dst, const float16_t& acc) {
  float* img = reinterpret_cast<float*>(dst);
  const int lane = threadIdx.x % kWave;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<float4_t*>(img + lane * 16 + 4 * q) = float4_t{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
}

// acc holds D[row][col] of a 32x32 block (rows 32*rb + ..., column 32*cb + ln);
// writes it transposed as fp16 into dst[col][row] (row-contiguous, 4 rows per store).
__device__ __forceinline__ void store_shadow_t(half_t* dst, const float16_t& acc, int rb, int cb) {
  const int lane = threadIdx.x % kWave, hl = lane / 32, ln = lane % 32;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int row = 32 * rb + 8 * g + 4 * hl;
    *reinterpret_cast<half4_t*>(dst + (32 * cb + ln) * PD + row) =
        half4_t{(half_t)acc[4 * g], (half_t)acc[4 * g + 1], (half_t)acc[4 * g + 2], (half_t)acc[4 * g + 3]};
  }
}

// The same block written into the piece-major quad shadow of S_i (dst, whose
// first piece is q0), [q - q0][64 v][8 j], as the apply's ring reads it; row
// groups before piece q0 are skipped (j = 32 rb .. 32 rb + 15 for odd i / 16).
__device__ __forceinline__ void store_quad_shadow(half_t* dst, const float16_t& acc, int rb, int cb, int q0) {
  const int lane = threadIdx.x % kWave, hl = lane / 32, ln = lane % 32;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int j = 32 * rb + 8 * g + 4 * hl;  // four consecutive j, one piece
    if (4 * rb + g < q0) continue;
    *reinterpret_cast<half4_t*>(dst + ((4 * rb + g - q0) * 64 + 32 * cb + ln) * 8 + (j & 7)) =
        half4_t{(half_t)acc[4 * g], (half_t)acc[4 * g + 1], (half_t)acc[4 * g + 2], (half_t)acc[4 * g + 3]};
  }
}

// What one state workgroup folds: chunks [c0, c1) of window c0 / KG onto the
// states listed, and where the result goes.
struct Fold {
  int c0, c1;
  uint32_t tok;         // its token images (workspace offset)
  uint32_t start;       // the window's start state, 0xffffffff for none (zero)
  uint32_t part;        // part sums added to it: n_part states from here
  int n_part;
  uint32_t dst;         // the folded state, 0xffffffff if nobody reads it
  bool shadow;          // write the fp16 shadow after every chunk

  // f(state) for every state the fold starts from.
  template <typename F>
  __device__ __forceinline__ void sources(const char* ws, F&& f) const {
    if (start != 0xffffffffu) f(ws + start);
    for (int i = 0; i < n_part; ++i) f(ws + part + i * kStateBytes);
  }
};

// Update of part p of window L, or (sum) the part's sum for window L + 1. The
// final chunk's update is never needed; false when nothing is left to fold.
__device__ __forceinline__ bool make_fold(const PolyArgs& a, int p, bool sum, Fold& f) {
  const int win = a.launch + (sum ? 1 : 0), len = KG / a.parts;
  const int last = a.n_chunks - 1;
  if (win < 0) return false;
  f.c0 = KG * win + p * len;
  f.c1 = min(f.c0 + len, last);
  // A sum is wanted only if the part after it has chunks.
  if (f.c0 >= f.c1 || (sum && f.c0 + len >= last)) return false;
  const uint32_t parts = kPart + (win & 1) * (PMAX - 1) * kStateBytes;
  f.tok = kTokImg + uint32_t(win % NIMG) * kTokImgBytes + uint32_t(p * len) * (PC / 64) * kTileImg;
  f.start = sum || win == 0 ? 0xffffffffu : kStart + (win & 1) * kStateBytes;
  f.part = parts;
  f.n_part = sum ? 0 : p;
  f.dst = sum ? parts + p * kStateBytes
              : (p == a.parts - 1 && KG * (win + 1) < last ? kStart + ((win + 1) & 1) * kStateBytes : 0xffffffffu);
  f.shadow = !sum;
  return true;
}

// One wave folds four slices i0 .. i0 + 3 on one 32-row j-block: eight MFMAs
// per 16-token step from four LDS reads -- b_j, two of v, and one that gives
// lane l the piece of slice i0 + l % 4, whose four values are then spread
// over each row of 16 lanes by DPP moves. The LDS reads, 16 cycles each for
// the whole CU, are what bounds a tile: with two slices on two j-blocks (or
// four on one) and each slice's piece read by itself it took 6 (7) reads,
// 1536 (1792) cycles a workgroup against 1024 of MFMA.
__device__ __forceinline__ half8_t row_bcast(half8_t x, int i) {
  using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
  const u32x4 u = __builtin_bit_cast(u32x4, x);
  u32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    switch (i) {  // DPP row_newbcast:i
      case 0: r[e] = __builtin_amdgcn_update_dpp(0, u[e], 0x150, 0xf, 0xf, true); break;
      case 1: r[e] = __builtin_amdgcn_update_dpp(0, u[e], 0x151, 0xf, 0xf, true); break;
      case 2: r[e] = __builtin_amdgcn_update_dpp(0, u[e], 0x152, 0xf, 0xf, true); break;
      default: r[e] = __builtin_amdgcn_update_dpp(0, u[e], 0x153, 0xf, 0xf, true); break;
    }
  }
  return __builtin_bit_cast(half8_t, r);
}

// Workgroups 0 .. 3: i < 32, one j-block per half; 4 and 5: i >= 32, j >= 32
// only (the apply never reads j < 32 there: S is symmetric).
__device__ __forceinline__ void quad_update_role(const Fold& f, char* ws, int ug, char* smem) {
  constexpr int NI = 4;
  struct Ops {
    half8_t bj, vv[2], bi;
  };
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave, hl = lane / 32, ln = lane % 32;
  const int i0 = ug < 4 ? 16 * (ug >> 1) + 4 * w : 32 + 16 * (ug - 4) + 4 * w;
  const int jb = ug < 4 ? ug & 1 : 1;
  // acc[ii][vb] = D[j][v] block of S_{i0+ii}. The fp32 state stays in these
  // registers across the fold's chunks.
  float16_t acc[NI][2];
  auto blocks = [&](auto&& g) {
#pragma unroll
    for (int ii = 0; ii < NI; ++ii)
#pragma unroll
      for (int vb = 0; vb < 2; ++vb) g(i0 + ii, vb, acc[ii][vb]);
  };
  blocks([](int, int, float16_t& x) {
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = 0.f;
  });
  f.sources(ws, [&](const char* st) {
    blocks([&](int i, int vb, float16_t& x) { add_img(st + quad_img(i, jb, vb), x); });
  });

  stream_image(
      ws, f.tok, f.c1 - f.c0, smem,
      [&](const half_t* bT, const half_t* vT, int ks) {
        const int pc = 2 * ks + hl;  // tokens 16 ks + 8 hl .. +7 of the tile
        Ops o;
        o.bi = img_piece(bT, i0 + (lane & 3), pc);
        o.bj = img_piece(bT, 32 * jb + ln, pc);
#pragma unroll
        for (int x = 0; x < 2; ++x) o.vv[x] = img_piece(vT, 32 * x + ln, pc);
        return o;
      },
      [&](const Ops& o) {
        // Issue order: the eight VALU operations of slice ii + 1's product go
        // four and four after slice ii's two MFMAs. A wave issues in order, so
        // behind both MFMAs they would wait for the second to leave the pipe
        // and then hold up the third.
        half8_t phi = o.bj * row_bcast(o.bi, 0);
#pragma unroll
        for (int ii = 0; ii < NI; ++ii) {
          acc[ii][0] = mfma32(phi, o.vv[0], acc[ii][0]);
          acc[ii][1] = mfma32(phi, o.vv[1], acc[ii][1]);
          if (ii + 1 < NI) phi = o.bj * row_bcast(o.bi, ii + 1);
        }
        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);  // VALU
#pragma unroll
        for (int x = 0; x < 2 * (NI - 1); ++x) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
      },
      [&](int j) {
        // fp16 shadow of state_{c+1} for the applies of the next launch: only
        // the pieces the apply reads.
        if (!f.shadow) return;
        char* sh = ws + kQuadShadow + uint32_t((f.c0 + j + 1) % NSLOT) * kShadowBytes;
        blocks([&](int i, int vb, const float16_t& x) {
          store_quad_shadow(reinterpret_cast<half_t*>(sh + quad_shadow(i)), x, jb, vb, 2 * (i >> 4));
        });
      });
  if (f.dst != 0xffffffffu)
    blocks([&](int i, int vb, const float16_t& x) { store_img(ws + f.dst + quad_img(i, jb, vb), x); });
}

// One wave each: S_lin[j][v] = sum_t b_tj v_tv, G[i][j] = sum_t b_ti b_tj (as
// 2x2 accumulator blocks each), z[d] = sum_t b_td and S_const[d] = sum_t v_td
// (lane = dim; four running sums, so the adds do not wait on one another).
template <bool GRAM>
__device__ __forceinline__ void small_mfma_wave(const Fold& f, char* ws, char* smem) {
  struct Ops {
    half8_t r[2], c[2];
  };
  const int lane = threadIdx.x % kWave, hl = lane / 32, ln = lane % 32;
  constexpr uint32_t img = GRAM ? kStGram : kStLin;
  float16_t acc[2][2];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b >> 1][b & 1][r] = 0.f;
  f.sources(ws, [&](const char* st) {
#pragma unroll
    for (int b = 0; b < 4; ++b) add_img(st + img + b * kImg, acc[b >> 1][b & 1]);
  });
  stream_image(
      ws, f.tok, f.c1 - f.c0, smem,
      [&](const half_t* bT, const half_t* vT, int ks) {
        const int pc = 2 * ks + hl;
        Ops o;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          o.r[x] = img_piece(bT, 32 * x + ln, pc);
          if constexpr (!GRAM) o.c[x] = img_piece(vT, 32 * x + ln, pc);
        }
        return o;
      },
      [&](const Ops& o) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) acc[rb][cb] = mfma32(o.r[rb], GRAM ? o.r[cb] : o.c[cb], acc[rb][cb]);
      },
      [&](int j) {
        if (!f.shadow) return;
        const int nxt = (f.c0 + j + 1) % NSLOT;  // S_lin as [v][j]; G is symmetric
        half_t* sh = reinterpret_cast<half_t*>(ws + (GRAM ? kGramShadow : kLinShadow)) + size_t(nxt) * PD * PD;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) store_shadow_t(sh, acc[rb][cb], rb, cb);
      });
  if (f.dst == 0xffffffffu) return;
#pragma unroll
  for (int b = 0; b < 4; ++b) store_img(ws + f.dst + img + b * kImg, acc[b >> 1][b & 1]);
}

template <bool CONST>
__device__ __forceinline__ void small_sum_wave(const Fold& f, char* ws, char* smem) {
  struct Ops {
    half8_t x[2];
  };
  const int lane = threadIdx.x % kWave;
  constexpr uint32_t at = kStZs + (CONST ? 64 * 4 : 0);
  float total = 0.f;
  f.sources(ws, [&](const char* st) { total += reinterpret_cast<const float*>(st + at)[lane]; });
  float part[4] = {0.f, 0.f, 0.f, 0.f};
  stream_image(
      ws, f.tok, f.c1 - f.c0, smem,
      [&](const half_t* bT, const half_t* vT, int ks) {
        Ops o;
#pragma unroll
        for (int x = 0; x < 2; ++x) o.x[x] = img_piece(CONST ? vT : bT, lane, 2 * ks + x);
        return o;
      },
      [&](const Ops& o) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          part[j & 1] += (float)o.x[0][j];
          part[2 + (j & 1)] += (float)o.x[1][j];
        }
      },
      [&](int j) {
        total += (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
        for (int x = 0; x < 4; ++x) part[x] = 0.f;
        if (f.shadow)
          reinterpret_cast<float*>(ws + kZsShadow)[(f.c0 + j + 1) % NSLOT * 128 + (CONST ? 64 : 0) + lane] = total;
      });
  if (f.dst != 0xffffffffu) reinterpret_cast<float*>(ws + f.dst + at)[lane] = total;
}

__device__ __forceinline__ void small_update_role(const Fold& f, char* ws, char* smem) {
  // The waves take different code (a scalar branch) but the same barriers,
  // one per tile.
  switch (__builtin_amdgcn_readfirstlane(threadIdx.x / kWave)) {
    case 0: small_mfma_wave<false>(f, ws, smem); break;
    case 1: small_mfma_wave<true>(f, ws, smem); break;
    case 2: small_sum_wave<false>(f, ws, smem); break;
    default: small_sum_wave<true>(f, ws, smem); break;
  }
}

// Windows between the images a launch writes and its own: the updates read
// window L, the part sums window L + 1.
__host__ __device__ constexpr int image_lag(int parts) { return parts > 1 ? 2 : 1; }

// Token images of chunk j of a later window: eight 64-token tiles, loads of
// the next tile in flight while the current one is stored.
template <typename T>
__device__ void image_role(const PolyArgs& a, char* ws, int b, int h, int j) {
  const int win = a.launch + image_lag(a.parts);
  const int c = KG * win + j;
  if (c >= a.n_chunks) return;
  char* dst = ws + kTokImg + uint32_t(win % NIMG) * kTokImgBytes + uint32_t(j) * (PC / 64) * kTileImg;
  const int tid = threadIdx.x;
  TokTile<T> x0, x1;
  x0.init(a, b, h, tid);
  x1.init(a, b, h, tid);
  x0.load(c * PC);
#pragma unroll
  for (int blk = 0; blk < PC / 64; blk += 2) {
    x1.load(c * PC + 64 * (blk + 1));
    x0.store_image(dst + blk * kTileImg, a.rs, tid);
    if (blk + 2 < PC / 64) x0.load(c * PC + 64 * (blk + 2));
    x1.store_image(dst + (blk + 1) * kTileImg, a.rs, tid);
  }
}

// Roles of one head in launch L, longest first: NSTATE workgroups for each of
// the P update parts of window L and of the P - 1 part sums of window L + 1;
// KG * NAPPLY apply workgroups (chunk KG (L-1) + 1 + j / NAPPLY, row block
// j % NAPPLY; launch 0 applies chunk 0 only); NCONV workgroups writing token
// images. Launches below 0 only prepare sums and images.
// Head m runs on XCD m % 8 (its roles share that L2); each XCD issues the
// roles of its heads role-major in that order.
__host__ __device__ constexpr int n_roles(int parts) { return (2 * parts - 1) * NSTATE + KG * NAPPLY + NCONV; }

template <typename T>
__global__ __launch_bounds__(PT, 2) void poly_chunk_kernel(PolyArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[kSmemBytes];
  const int x = blockIdx.x % kNumXcd, k = blockIdx.x / kNumXcd;
  const int nh = x < a.M ? (a.M - x + kNumXcd - 1) / kNumXcd : 0;  // heads on this XCD
  if (k >= nh * n_roles(a.parts)) return;
  int rr = k / nh;
  const int m = x + kNumXcd * (k % nh);
  if (a.flags != nullptr && a.flags[m] == 0) return;
  const int b = m / a.H, h = m % a.H;
  char* ws = a.ws + size_t(m) * kPerHead;
  const int n_state = (2 * a.parts - 1) * NSTATE;
  if (rr < n_state) {
    const bool sum = rr >= a.parts * NSTATE;
    if (sum) rr -= a.parts * NSTATE;
    Fold f;
    if (!make_fold(a, rr / NSTATE, sum, f)) return;
    if (rr % NSTATE < NUPD) quad_update_role(f, ws, rr % NSTATE, smem);
    else small_update_role(f, ws, smem);
    return;
  }
  rr -= n_state;
  if (rr >= KG * NAPPLY) {
    image_role<T>(a, ws, b, h, rr - KG * NAPPLY);
  } else if (a.launch >= 0) {
    const int g = rr / NAPPLY;
    const int c = a.launch == 0 ? (g == 0 ? 0 : -1) : KG * (a.launch - 1) + 1 + g;
    if (c >= 0 && c < a.n_chunks) apply_role<T>(a, ws, b, h, m, c, rr % NAPPLY, smem);
  }
}

// Parts of a window by the number of heads M. Two parts while the update
// chain sets the time, one where the chip is busy anyway (polynomial rows
// alone, us with one / two / four parts, fp32 unless said: 1 head of 100 000 tokens
// 1687 / 1110 / 1183, 2 of 60 000 1036 / 720 / 728, 8 of 60 000 1113 / 798 /
// 815, 16 of 30 000 687 / 693 / 719, 24 of 40 000 1079 / 1246 / 1390, 64 of
// 65536 4388 / 5259 / 5967; four parts are never worth their sums).
int parts_for(int M) { return M < 16 ? 2 : 1; }

template <typename T>
int run(PolyArgs a, size_t ws_bytes, hipStream_t stream) {
  (void)ws_bytes;
  a.parts = parts_for(a.M);
  const dim3 grid(unsigned(kNumXcd * ((a.M + kNumXcd - 1) / kNumXcd) * n_roles(a.parts)));
  // Token images and part sums of the first windows.
  for (int L = -image_lag(a.parts); L < 0; ++L) {
    if (L > -image_lag(a.parts) && a.n_chunks == 1) continue;
    a.launch = L;
    hipLaunchKernelGGL(poly_chunk_kernel<T>, grid, dim3(PT), 0, stream, a);
    if (hipGetLastError() != hipSuccess) return TJ_ERR_LAUNCH;
  }
  // Launch L applies chunks (KG (L-1), KG L] and folds in chunks [KG L, KG L + KG).
  const int n_launch = 1 + (a.n_chunks - 1 + KG - 1) / KG;
  for (int L = 0; L < n_launch; ++L) {
    const int last_applied = min(KG * L, a.n_chunks - 1);
    const bool emits = min(a.S, (last_applied + 1) * PC) > a.prefix_end;
    const bool updates = KG * L < a.n_chunks - 1;
    if (!emits && !updates) continue;
    a.launch = L;
    hipLaunchKernelGGL(poly_chunk_kernel<T>, grid, dim3(PT), 0, stream, a);
    if (hipGetLastError() != hipSuccess) return TJ_ERR_LAUNCH;
  }
  return TJ_OK;
}

}  // namespace
}  // namespace tj

extern "C" size_t tj_poly_workspace_bytes(int64_t B, int64_t H, int64_t S, int64_t D, int64_t chunk) {
  (void)S;
  (void)chunk;
  if (B <= 0 || H <= 0 || D != tj::PD) return 0;
  if (!tjh::product_below(std::numeric_limits<int64_t>::max() / int64_t(tj::kPerHead), {B, H})) return 0;
  return size_t(B * H) * tj::kPerHead;
}

extern "C" int tj_poly_attn_fwd(const void* q, const void* k, const void* v, void* o, int dtype,
                                int64_t B, int64_t H, int64_t S, int64_t D,
                                const int64_t q_strides[4], const int64_t k_strides[4],
                                const int64_t v_strides[4], const int64_t o_strides[4],
                                float scale, int64_t chunk, int64_t exact_prefix,
                                const float* coeffs, const int32_t* flags,
                                void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (dtype != TJ_F32 && dtype != TJ_F16) return TJ_ERR_DTYPE;
  if (B < 0 || H <= 0 || S < 0 || D <= 0 || chunk <= 0 || exact_prefix < 0 || !(scale > 0.f)) return TJ_ERR_SHAPE;
  if (D != tj::PD || chunk != tj::PC) return TJ_ERR_UNSUPPORTED;
  if (B == 0 || S == 0 || exact_prefix >= S) return TJ_OK;
  if (S >= (int64_t(1) << 30) ||
      !tjh::product_below((int64_t(1) << 31) / tj::n_roles(1) - tj::kNumXcd, {B, H}))
    return TJ_ERR_SHAPE;
  if (!q || !k || !v || !o || !coeffs) return TJ_ERR_SHAPE;
  if (!tjh::view_ok(q, q_strides, dtype) || !tjh::view_ok(k, k_strides, dtype) ||
      !tjh::view_ok(v, v_strides, dtype) || !tjh::view_ok(o, o_strides, dtype))
    return TJ_ERR_ALIGN;
  // K and V rows of one (b, h) are addressed with 31-bit byte offsets.
  for (const int64_t* st : {k_strides, v_strides})
    if (!tjh::span_below_2g(S, st[2], D, tjh::elem_size(dtype))) return TJ_ERR_UNSUPPORTED;
  const size_t need = size_t(B * H) * tj::kPerHead;
  if (workspace == nullptr || workspace_bytes < need || !tjh::aligned16(workspace)) return TJ_ERR_WORKSPACE;

  tj::PolyArgs a;
  a.q = q; a.k = k; a.v = v; a.o = o;
  a.vq = {q_strides[0], q_strides[1], q_strides[2]};
  a.vk = {k_strides[0], k_strides[1], k_strides[2]};
  a.vv = {v_strides[0], v_strides[1], v_strides[2]};
  a.vo = {o_strides[0], o_strides[1], o_strides[2]};
  a.H = (int)H; a.S = (int)S;
  a.rs = sqrtf(scale);
  a.prefix_end = (int)exact_prefix;
  a.coeffs = coeffs;
  a.flags = flags;
  a.ws = static_cast<char*>(workspace);
  a.M = (int)(B * H);
  a.n_chunks = (int)((S + tj::PC - 1) / tj::PC);
  if (dtype == TJ_F32) return tj::run<float>(a, need, stream);
  return tj::run<half_t>(a, need, stream);
}
