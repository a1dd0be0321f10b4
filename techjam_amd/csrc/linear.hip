// Dense layers of the encoder block, y = x W^T in fp32 on bf16 MFMAs, with the
// passes that follow them folded in (the projections of
// torch_transformer_benchmark.py:75-145).
//
// Every fp32 operand is split as it is loaded, v = hi + lo with both parts
// rounded to bf16, and each product is three MFMAs, hi.hi + hi.lo + lo.hi, in
// fp32 accumulators: the arithmetic of the GEMM library's fast float32 mode,
// for which these kernels stand in where it is slower (kernels/linear.py has
// the rules). Relative error against 64 bits over M = 1 .. 200 000, N and K
// 64 .. 4096: 4.0e-6 to 4.8e-6, to 5.5e-6 at one row, the library's to two
// digits. An infinity or a value past bf16's largest makes its row NaN (its
// low part is inf - inf), in that mode as here.
//
//   * linear_rows_kernel: one workgroup per 32 x 32 outputs, its 4 (8 from K =
//     512 on) waves each taking a share of K straight from global memory into
//     MFMA operands (a lane loads 32 contiguous bytes of one row), partial
//     sums added through LDS. For few tokens, where a launch is latency: no
//     staging barrier, every load of a wave's first steps in flight at once,
//     and enough workgroups to cover the chip. 256 x 256 x 256: 26.0 us by
//     the library, 4.5 us here; 256 x 128 x 512: 28.7 and 6.3 us.
//   * narrow_kernel: layers of width 128 (x, W and y all 128 wide), any number
//     of tokens. W is split once per workgroup into LDS and stays there; each
//     wave then takes 32 tokens at a time, its rows of x straight from global
//     memory, without another barrier. Outputs come out transposed (a lane
//     holds 64 of one token's 128 values), so a row's LayerNorm is lane-local
//     plus one lane-pair swap, and the FFN's hidden activations convert in
//     place into the second product's operand: the whole FFN half of a block
//     reads two [tokens, 128] tensors and writes two. Bound by HBM for many
//     tokens: at 65 536 (26 us for its bytes at the copy rate) the q, k, v
//     projections take 36 us (52 as three library products), out_proj +
//     residual + norm 31 (38), the FFN half 41 (66; 49 with erff in its GELU).
#include "tj_common.h"

namespace tj {
namespace {

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf4_t __attribute__((ext_vector_type(4)));

enum Act { ACT_NONE, ACT_GELU, ACT_RELU };

struct LinArgs {
  const float* x;
  const float* w[3];
  float* out[3];
  int64_t M;
  int N, K, n_w;
  const float* bias;
};

__device__ __forceinline__ float16_t mfma_bf16(bf8_t a, bf8_t b, float16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// hi + lo ~ v, both bf16 (round to nearest even).
template <typename B, typename V>
__device__ __forceinline__ void split(V v, B& hi, B& lo) {
  hi = __builtin_convertvector(v, B);
  lo = __builtin_convertvector(v - __builtin_convertvector(hi, V), B);
}

// Eight floats from a 16-byte aligned address.
__device__ __forceinline__ float8_t load8(const float* p) {
  const float4_t a = *reinterpret_cast<const float4_t*>(p), b = *reinterpret_cast<const float4_t*>(p + 4);
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <Act A>
__device__ __forceinline__ float activate(float t) {
  if constexpr (A == ACT_GELU) return gelu_erf(t);
  else if constexpr (A == ACT_RELU) return t > 0.f ? t : 0.f;
  else return t;
}

// Output tiles are dealt so that each XCD takes a contiguous range, columns
// fastest: the workgroups that read one row block share an L2.
__device__ __forceinline__ bool tile_of_block(int64_t tiles, int64_t& t) {
  const int64_t per = (tiles + kNumXcd - 1) / kNumXcd;
  t = (blockIdx.x % kNumXcd) * per + blockIdx.x / kNumXcd;
  return blockIdx.x / kNumXcd < per && t < tiles;
}

template <Act A, int NW>
__global__ __launch_bounds__(NW* kWave) void linear_rows_kernel(LinArgs a) {
  __shared__ __attribute__((aligned(16))) float part[NW][32][36];
  const int nt = a.N / 32;
  int64_t t;
  if (!tile_of_block((a.M + 31) / 32 * nt * a.n_w, t)) return;
  const int col = (int)(t % (nt * a.n_w));
  const int64_t m0 = t / (nt * a.n_w) * 32;
  const int wi = col / nt, n0 = col % nt * 32;
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave, hl = lane / 32, ln = lane % 32;

  // This wave's share of K, in 16-wide steps; rows past M repeat the last.
  const int kq = a.K / NW, steps = kq / 16;
  const float* xp = a.x + (m0 + ln < a.M ? m0 + ln : a.M - 1) * a.K + w * kq + 8 * hl;
  const float* wp = a.w[wi] + (int64_t)(n0 + ln) * a.K + w * kq + 8 * hl;
  constexpr int U = 4;  // steps in flight, twice
  float8_t xa[2][U], wa[2][U];
  auto load = [&](int s0, int buf) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s0 + u < steps) {
        xa[buf][u] = load8(xp + (s0 + u) * 16);
        wa[buf][u] = load8(wp + (s0 + u) * 16);
      }
  };
  float16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  auto mma = [&](int s0, int buf) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s0 + u < steps) {
        bf8_t xh, xl, wh, wl;
        split(xa[buf][u], xh, xl);
        split(wa[buf][u], wh, wl);
        acc = mfma_bf16(xl, wh, acc);
        acc = mfma_bf16(xh, wl, acc);
        acc = mfma_bf16(xh, wh, acc);
      }
  };
  load(0, 0);
  for (int s = 0; s < steps; s += 2 * U) {
    load(s + U, 1);
    mma(s, 0);
    load(s + 2 * U, 0);
    mma(s + U, 1);
  }
  // acc: rows 8 (r / 4) + 4 hl + r % 4, column ln.
#pragma unroll
  for (int r = 0; r < 16; ++r) part[w][8 * (r / 4) + 4 * hl + (r % 4)][ln] = acc[r];
  __syncthreads();
  const int row = tid / 8, c = 4 * (tid % 8);
  if (row >= 32 || m0 + row >= a.M) return;
  float4_t y = *reinterpret_cast<const float4_t*>(&part[0][row][c]);
#pragma unroll
  for (int p = 1; p < NW; ++p) y += *reinterpret_cast<const float4_t*>(&part[p][row][c]);
  if constexpr (A != ACT_NONE) {
    y += *reinterpret_cast<const float4_t*>(a.bias + n0 + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = activate<A>(y[e]);
  }
  *reinterpret_cast<float4_t*>(a.out[wi] + (m0 + row) * a.N + n0 + c) = y;
}

// ---------------------------------------------------------------------------
// Width 128
// ---------------------------------------------------------------------------
constexpr int NWD = 128;       // the width
constexpr int NWP = NWD + 8;   // padded LDS row of W (272 bytes: 16 rows hit 16 distinct 16-byte slots)

struct NarrowArgs {
  const float* x;
  const float* w[3];   // PLAIN: the weights, one per blockIdx.y; RES: out_proj; FFN: ffn_in, ffn_out
  float* out[3];       // PLAIN: one per weight; RES / FFN: out[0], the new residual stream (or null)
  int64_t M;
  const float* bias;   // of the (last) projection
  const float* bias_in;  // FFN: of ffn_in
  const float* resid;
  const int32_t* valid_len;
  int64_t seq_len;
  int mode, zero_ln;
  const float* gamma;
  const float* beta;
  float* ln_out;
  float eps;
};

enum NarrowKind { NARROW_PLAIN, NARROW_RES, NARROW_FFN };

struct SplitW {
  __bf16 h[NWD][NWP], l[NWD][NWP];
};

// Split W [128][128] into LDS. With SLOTS the columns of each 16 are stored
// in key_slot order: a step's operand is then the 8 columns whose activations
// one lane of a transposed product holds.
template <bool SLOTS, int NT>
__device__ __forceinline__ void stage_weight(SplitW& s, const float* w) {
#pragma unroll
  for (int i = 0; i < NWD * NWD / 4 / NT; ++i) {
    const int e = threadIdx.x + i * NT, n = e / (NWD / 4), k = 4 * (e % (NWD / 4));
    bf4_t h, l;
    split(*reinterpret_cast<const float4_t*>(w + n * NWD + k), h, l);
    const int c = SLOTS ? key_slot(k) : k;
    *reinterpret_cast<bf4_t*>(&s.h[n][c]) = h;
    *reinterpret_cast<bf4_t*>(&s.l[n][c]) = l;
  }
}

// acc[nb] += W x^T (rows n = 32 nb + .., columns tokens) over the eight
// k-steps, or with ROWS x W^T (rows tokens, columns n = 32 nb + ..).
template <bool ROWS = false>
__device__ __forceinline__ void narrow_product(const SplitW& s, const bf8_t (&xh)[8], const bf8_t (&xl)[8],
                                               float16_t (&acc)[4]) {
  const int lane = threadIdx.x % kWave, hl = lane / 32, ln = lane % 32;
#pragma unroll
  for (int ks = 0; ks < 8; ++ks)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const bf8_t wh = *reinterpret_cast<const bf8_t*>(&s.h[32 * nb + ln][16 * ks + 8 * hl]);
      const bf8_t wl = *reinterpret_cast<const bf8_t*>(&s.l[32 * nb + ln][16 * ks + 8 * hl]);
      if constexpr (ROWS) {
        acc[nb] = mfma_bf16(xh[ks], wl, acc[nb]);
        acc[nb] = mfma_bf16(xl[ks], wh, acc[nb]);
        acc[nb] = mfma_bf16(xh[ks], wh, acc[nb]);
      } else {
        acc[nb] = mfma_bf16(wl, xh[ks], acc[nb]);
        acc[nb] = mfma_bf16(wh, xl[ks], acc[nb]);
        acc[nb] = mfma_bf16(wh, xh[ks], acc[nb]);
      }
    }
}

template <NarrowKind KIND, Act A, int NT>
__global__ __launch_bounds__(NT, KIND == NARROW_FFN ? 1 : 2) void narrow_kernel(NarrowArgs a) {
  __shared__ __attribute__((aligned(16))) SplitW sw[KIND == NARROW_FFN ? 2 : 1];
  constexpr int NWV = NT / kWave;
  const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave, hl = lane / 32, ln = lane % 32;
  const int64_t tiles = (a.M + 31) / 32;  // of 32 tokens, one per wave at a time
  int64_t tile = blockIdx.x * (int64_t)NWV + w;
  const int64_t stride = gridDim.x * (int64_t)NWV;

  // x^T as the B operand: lane holds token ln, dims 16 ks + 8 hl .. + 7.
  float8_t xr[8];
  auto load_x = [&](int64_t t) {
    const int64_t m = t * 32 + ln;
    const float* p = a.x + (m < a.M ? m : a.M - 1) * NWD + 8 * hl;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) xr[ks] = load8(p + 16 * ks);
  };
  if (tile < tiles) load_x(tile);
  stage_weight<false, NT>(sw[0], a.w[KIND == NARROW_PLAIN ? blockIdx.y : 0]);
  if constexpr (KIND == NARROW_FFN) stage_weight<true, NT>(sw[1], a.w[1]);
  __syncthreads();

  for (; tile < tiles; tile += stride) {
    // The weights in LDS and the vectors are read anew for every tile: kept in
    // registers across tiles, as the compiler would, they do not fit.
    asm volatile("" ::: "memory");
    bf8_t xh[8], xl[8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) split(xr[ks], xh[ks], xl[ks]);
    if (KIND != NARROW_FFN && tile + stride < tiles) load_x(tile + stride);
    float16_t acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[nb][r] = 0.f;
    narrow_product<KIND == NARROW_PLAIN>(sw[0], xh, xl, acc);

    if constexpr (KIND == NARROW_FFN) {
      // Hidden activations: element r of block nb is f = 32 nb + 8 (r / 4) +
      // 4 hl + r % 4 of this lane's token; elements 8 x .. 8 x + 7 are the
      // k-slots of step 2 nb + x in the key_slot order W2 is staged in.
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        __builtin_amdgcn_sched_barrier(0);  // one block's temporaries at a time
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4_t b = *reinterpret_cast<const float4_t*>(a.bias_in + 32 * nb + 8 * g + 4 * hl);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[nb][4 * g + e] = activate<A>(acc[nb][4 * g + e] + b[e]);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          float8_t v;
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = acc[nb][8 * x + e];
          split(v, xh[2 * nb + x], xl[2 * nb + x]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");  // the next tile's rows not before the activations
      if (tile + stride < tiles) load_x(tile + stride);
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[nb][r] = 0.f;
      narrow_product(sw[1], xh, xl, acc);
    }

    const int64_t row = tile * 32 + ln;
    const bool live = row < a.M;
    const int64_t at = (live ? row : a.M - 1) * NWD + 4 * hl;
    if constexpr (KIND == NARROW_PLAIN) {
      // Element r of block nb: token tile * 32 + 8 (r / 4) + 4 hl + r % 4,
      // column 32 nb + ln: every store writes two whole 128-byte lines.
      const int64_t left = a.M - tile * 32 - 4 * hl;
      float* o = a.out[blockIdx.y] + (tile * 32 + 4 * hl) * NWD + ln;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int tok = 8 * (r / 4) + (r % 4);
        if (tok < left)
#pragma unroll
          for (int nb = 0; nb < 4; ++nb) o[tok * NWD + 32 * nb] = acc[nb][r];
      }
    } else {
      const bool valid = a.valid_len == nullptr || (live ? row : 0) % a.seq_len < (int64_t)a.valid_len[(live ? row : 0) / a.seq_len];
      const bool ok = a.mode == 0 || valid;
      float sum = 0.f;
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4_t xv = *reinterpret_cast<const float4_t*>(a.resid + at + 32 * nb + 8 * g);
          const float4_t b = *reinterpret_cast<const float4_t*>(a.bias + 32 * nb + 8 * g + 4 * hl);
          float4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float y = acc[nb][4 * g + e] + b[e];
            v[e] = a.mode == 2 ? (ok ? xv[e] + y : 0.f) : xv[e] + (ok ? y : 0.f);
            acc[nb][4 * g + e] = v[e];
            sum += v[e];
          }
          if (live && a.out[0] != nullptr) *reinterpret_cast<float4_t*>(a.out[0] + at + 32 * nb + 8 * g) = v;
        }
      // Two exact passes over the row, as torch.nn.LayerNorm defines them.
      const float mean = pair_sum(sum) / (float)NWD;
      float sq = 0.f;
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) sq += (acc[nb][r] - mean) * (acc[nb][r] - mean);
      const float rstd = 1.f / sqrtf(pair_sum(sq) / (float)NWD + a.eps);
      const bool zero = a.zero_ln != 0 && !valid;
      if (live) {
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float4_t gv = *reinterpret_cast<const float4_t*>(a.gamma + 32 * nb + 8 * g + 4 * hl);
            const float4_t hv = *reinterpret_cast<const float4_t*>(a.beta + 32 * nb + 8 * g + 4 * hl);
            float4_t n;
#pragma unroll
            for (int e = 0; e < 4; ++e) n[e] = zero ? 0.f : (acc[nb][4 * g + e] - mean) * rstd * gv[e] + hv[e];
            *reinterpret_cast<float4_t*>(a.ln_out + at + 32 * nb + 8 * g) = n;
          }
      }
    }
  }
}

// Workgroups per weight, n_w weights side by side: never more in all than are
// resident at once, two of four waves per CU, or one of eight (two weights in
// LDS). One more (171 x 3 for q, k, v) would start its whole share of the
// tokens when the others end.
constexpr int64_t narrow_slots(bool ffn, int n_w) { return (ffn ? 256 : 512) / n_w; }
static_assert(narrow_slots(true, 1) <= 256 && narrow_slots(false, 1) <= 512 && 2 * narrow_slots(false, 2) <= 512 &&
              3 * narrow_slots(false, 3) <= 512, "resident workgroups");

template <NarrowKind KIND, Act A>
int launch_narrow(const NarrowArgs& a, int n_w, hipStream_t stream) {
  constexpr int NT = KIND == NARROW_FFN ? 512 : 256;
  const int64_t full = (a.M + NT / 2 - 1) / (NT / 2);  // 32 tokens a wave
  const int64_t per = narrow_slots(KIND == NARROW_FFN, n_w);
  hipLaunchKernelGGL((narrow_kernel<KIND, A, NT>), dim3((unsigned)(full < per ? full : per), (unsigned)n_w), dim3(NT), 0,
                     stream, a);
  return tjh::launch_status();
}

template <Act A>
int launch_rows(const LinArgs& a, hipStream_t stream) {
  const int64_t tiles = (a.M + 31) / 32 * (a.N / 32) * a.n_w;
  const int64_t grid = (tiles + kNumXcd - 1) / kNumXcd * kNumXcd;
  const bool deep = a.K >= 512 && a.K % 128 == 0;
  if (grid * 512 >= (int64_t(1) << 32)) return TJ_ERR_SHAPE;
  if (deep) hipLaunchKernelGGL((linear_rows_kernel<A, 8>), dim3((unsigned)grid), dim3(512), 0, stream, a);
  else hipLaunchKernelGGL((linear_rows_kernel<A, 4>), dim3((unsigned)grid), dim3(256), 0, stream, a);
  return tjh::launch_status();
}

// [p, p + pn) and [q, q + qn) floats share no byte.
bool apart(const void* p, int64_t pn, const void* q, int64_t qn) {
  const int64_t a = (int64_t)p, b = (int64_t)q;
  return a + pn * 4 <= b || b + qn * 4 <= a;
}

// Shapes within the kernels' index types.
bool sizes_ok(int64_t M, int64_t N, int64_t K) {
  return M >= 0 && N > 0 && K > 0 && tjh::product_below(int64_t(1) << 40, {M, N}) &&
         tjh::product_below(int64_t(1) << 40, {M, K}) && tjh::product_below(int64_t(1) << 31, {N, K});
}

// What the two residual entry points share: everything but the products.
int check_residual(const float* x, const float* bias, const float* resid, const float* out, int64_t M, int64_t seq_len,
                   const int32_t* valid_len, int mode, const float* gamma, const float* beta, const float* ln_out,
                   float eps, int zero_ln_padded) {
  if (!sizes_ok(M, NWD, NWD) || seq_len <= 0 || mode < 0 || mode > 2 || !(eps >= 0.f)) return TJ_ERR_SHAPE;
  if ((mode != 0 || zero_ln_padded) && valid_len != nullptr && M % seq_len != 0) return TJ_ERR_SHAPE;
  if (M == 0) return TJ_OK;
  if (!x || !bias || !resid || !gamma || !beta || !ln_out) return TJ_ERR_SHAPE;  // out may be null
  for (const void* p : {x, bias, resid, out, gamma, beta, ln_out})
    if (!tjh::aligned16(p)) return TJ_ERR_ALIGN;
  // A wave writes its rows while others still read theirs: outputs apart from
  // the inputs, except that out may be resid itself (a row is its wave's own).
  const int64_t n = M * NWD;
  if (!apart(ln_out, n, x, n) || !apart(ln_out, n, resid, n) || (out && !apart(ln_out, n, out, n))) return TJ_ERR_SHAPE;
  if (out && (!apart(out, n, x, n) || (out != resid && !apart(out, n, resid, n)))) return TJ_ERR_SHAPE;
  return TJ_OK;
}

NarrowArgs residual_args(const float* x, const float* bias, const float* resid, float* out, int64_t M, int64_t seq_len,
                         const int32_t* valid_len, int mode, const float* gamma, const float* beta, float* ln_out,
                         float eps, int zero_ln_padded) {
  NarrowArgs a = {};
  a.x = x; a.out[0] = out; a.M = M; a.bias = bias; a.resid = resid;
  a.valid_len = (mode == 0 && !zero_ln_padded) ? nullptr : valid_len;
  a.seq_len = seq_len; a.mode = mode; a.zero_ln = zero_ln_padded;
  a.gamma = gamma; a.beta = beta; a.ln_out = ln_out; a.eps = eps;
  return a;
}

}  // namespace
}  // namespace tj

extern "C" int tj_linear(const float* x, const float* w0, const float* w1, const float* w2, float* out0, float* out1,
                         float* out2, int64_t M, int64_t N, int64_t K, const float* bias, int act, int narrow,
                         hipStream_t stream) {
  const float* w[3] = {w0, w1, w2};
  float* out[3] = {out0, out1, out2};
  const int n_w = w2 != nullptr ? 3 : (w1 != nullptr ? 2 : 1);
  if (act < 0 || act > 2 || (act != 0) != (bias != nullptr) || (act != 0 && (n_w != 1 || narrow))) return TJ_ERR_SHAPE;
  if (!tj::sizes_ok(M, N, K)) return TJ_ERR_SHAPE;
  if (narrow ? (N != tj::NWD || K != tj::NWD) : (N % 32 != 0 || K % 64 != 0)) return TJ_ERR_UNSUPPORTED;
  if (M == 0) return TJ_OK;
  if (x == nullptr) return TJ_ERR_SHAPE;
  if (!tjh::aligned16(x) || !tjh::aligned16(bias)) return TJ_ERR_ALIGN;
  for (int i = 0; i < n_w; ++i) {
    if (w[i] == nullptr || out[i] == nullptr || !tj::apart(out[i], M * N, x, M * K)) return TJ_ERR_SHAPE;
    if (!tjh::aligned16(w[i]) || !tjh::aligned16(out[i])) return TJ_ERR_ALIGN;
  }
  if (narrow) {
    tj::NarrowArgs a = {};
    a.x = x; a.M = M;
    for (int i = 0; i < n_w; ++i) { a.w[i] = w[i]; a.out[i] = out[i]; }
    return tj::launch_narrow<tj::NARROW_PLAIN, tj::ACT_NONE>(a, n_w, stream);
  }
  tj::LinArgs a = {};
  a.x = x; a.bias = bias; a.n_w = n_w;
  for (int i = 0; i < n_w; ++i) { a.w[i] = w[i]; a.out[i] = out[i]; }
  a.M = M; a.N = (int)N; a.K = (int)K;
  if (act == 0) return tj::launch_rows<tj::ACT_NONE>(a, stream);
  if (act == 1) return tj::launch_rows<tj::ACT_GELU>(a, stream);
  return tj::launch_rows<tj::ACT_RELU>(a, stream);
}

extern "C" int tj_narrow_residual_norm(const float* x, const float* w, const float* bias, const float* resid, float* out,
                                       int64_t M, int64_t seq_len, const int32_t* valid_len, int mode,
                                       const float* gamma, const float* beta, float* ln_out, float eps,
                                       int zero_ln_padded, hipStream_t stream) {
  const int rc = tj::check_residual(x, bias, resid, out, M, seq_len, valid_len, mode, gamma, beta, ln_out, eps, zero_ln_padded);
  if (rc != TJ_OK || M == 0) return rc;
  if (w == nullptr) return TJ_ERR_SHAPE;
  if (!tjh::aligned16(w)) return TJ_ERR_ALIGN;
  tj::NarrowArgs a = tj::residual_args(x, bias, resid, out, M, seq_len, valid_len, mode, gamma, beta, ln_out, eps, zero_ln_padded);
  a.w[0] = w;
  return tj::launch_narrow<tj::NARROW_RES, tj::ACT_NONE>(a, 1, stream);
}

extern "C" int tj_narrow_ffn_norm(const float* x, const float* w_in, const float* bias_in, int act, const float* w_out,
                                  const float* bias, const float* resid, float* out, int64_t M, int64_t seq_len,
                                  const int32_t* valid_len, int mode, const float* gamma, const float* beta,
                                  float* ln_out, float eps, int zero_ln_padded, hipStream_t stream) {
  if (act != 1 && act != 2) return TJ_ERR_SHAPE;
  const int rc = tj::check_residual(x, bias, resid, out, M, seq_len, valid_len, mode, gamma, beta, ln_out, eps, zero_ln_padded);
  if (rc != TJ_OK || M == 0) return rc;
  if (!w_in || !w_out || !bias_in) return TJ_ERR_SHAPE;
  if (!tjh::aligned16(w_in) || !tjh::aligned16(w_out) || !tjh::aligned16(bias_in)) return TJ_ERR_ALIGN;
  tj::NarrowArgs a = tj::residual_args(x, bias, resid, out, M, seq_len, valid_len, mode, gamma, beta, ln_out, eps, zero_ln_padded);
  a.w[0] = w_in; a.w[1] = w_out; a.bias_in = bias_in;
  if (act == 1) return tj::launch_narrow<tj::NARROW_FFN, tj::ACT_GELU>(a, 1, stream);
  return tj::launch_narrow<tj::NARROW_FFN, tj::ACT_RELU>(a, 1, stream);
}
