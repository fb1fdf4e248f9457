// Residual add + LayerNorm on feature-major activations, the glue between the sparse products of the
// encoder-layer configuration (the reference's model code keeps these in torch on token-major tensors,
// reference end2end/sspmm_e2e/end_to_end.py:58-75; the SpMM wants and returns [features, tokens], and
// normalising that layout through torch costs two transposed copies per LayerNorm).
//
//   out[h, t] = (s[h, t] - mean_t) * rsqrt(var_t + eps) * gamma[h] + beta[h],   s = fp16(x + a)
//
// with mean and (biased) variance over the H features of token t, in fp32.  HBM-bound: x and a read once, out
// written once (6 * H * T bytes); a workgroup of eight waves owns 16 tokens (32 bytes of every row), has the loads of
// six rows per thread in flight together, keeps the H x 16 sums in LDS as fp16 and makes its passes (mean,
// variance, result) over LDS.  The four workgroups that share the 128-byte lines of 64 consecutive tokens get
// workgroup ids that the hardware's round-robin deal puts on one XCD, so a line crosses the fabric once.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "lane_ops.h"
#include "layer_kernels.h"

namespace sspmm {

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// TOK tokens per workgroup (TOK / 4 lanes of four tokens each), THREADS threads, TRIP rows per thread whose loads are
// in flight together.
template <int TOK, int THREADS, int TRIP>
struct LnShape {
  static constexpr int kLanes = TOK / 4;
  static constexpr int kRowGroups = THREADS / kLanes;
  static constexpr int kParts = 64 / TOK;  // workgroups that share the 128-byte lines of 64 consecutive tokens
};

// Sum over the workgroup's row groups of one value per token group: across the row groups of a wave with lane
// exchanges, across the waves through LDS.  Contains barriers.
template <int LANES, int THREADS>
__device__ __forceinline__ floatx4 block_sum_per_token(floatx4 v, floatx4 *red, int tl) {
#pragma unroll
  for (int d = LANES; d < 64; d <<= 1)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += __shfl_xor(v[i], d, 64);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();  // red may still be read from the call before
  if (lane < LANES) red[wave * LANES + tl] = v;
  __syncthreads();
  floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < THREADS / 64; ++w) s += red[w * LANES + tl];
  return s;
}

// RAGGED: T any number of tokens, rows at any element (such calls had torch's LayerNorm between two transposed copies: 768 x 4000
// 46 us a call where this takes 9, 768 x 1665 29 and 12, of which the host is most).
template <int TOK, int THREADS, int TRIP, bool RAGGED>
__global__ __launch_bounds__(THREADS) void add_layernorm_kernel(int H, int T, const _Float16 *__restrict__ x,
                                                                 const _Float16 *__restrict__ a,
                                                                 const _Float16 *__restrict__ gamma,
                                                                 const _Float16 *__restrict__ beta, float eps,
                                                                 _Float16 *__restrict__ out) {
  typedef LnShape<TOK, THREADS, TRIP> S;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  half4 *sums = reinterpret_cast<half4 *>(lds_raw);                            // [H][S::kLanes] groups of four tokens
  floatx4 *red = reinterpret_cast<floatx4 *>(lds_raw + (size_t)H * TOK * 2);  // [waves][S::kLanes]
  const int tl = threadIdx.x % S::kLanes, rg = threadIdx.x / S::kLanes;
  // workgroup id -> token group: ids congruent modulo 8 share an XCD, and the parts of a 64-token line group go to
  // ids 8 apart, so the workgroups that share 128-byte lines share an L2
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int first = (((idx / S::kParts) * 8 + xcd) * S::kParts + (idx % S::kParts)) * TOK;
  if (first >= T) return;  // (the whole workgroup: the grid is padded to eight line groups)
  const int t0 = first + 4 * tl;
  const bool live = t0 < T;
  const int left = T - t0;  // (at least 4 where T is a multiple of it)
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  // (the loads of TRIP rows are issued together: the kernel is bound by how many bytes its workgroups keep in flight)
  for (int h0 = rg; h0 < H; h0 += S::kRowGroups * TRIP) {
    half4 xs[TRIP], as[TRIP];
#pragma unroll
    for (int u = 0; u < TRIP; ++u) {
      const int h = h0 + u * S::kRowGroups;
      xs[u] = half4{0, 0, 0, 0};
      as[u] = half4{0, 0, 0, 0};
      if (live && h < H) {
        xs[u] = load_four<RAGGED, true>(x + (size_t)h * T + t0, left);
        if (a) as[u] = load_four<RAGGED, true>(a + (size_t)h * T + t0, left);
      }
    }
#pragma unroll
    for (int u = 0; u < TRIP; ++u) {
      const int h = h0 + u * S::kRowGroups;
      if (h < H) {
        const half4 s = xs[u] + as[u];  // fp16 sum, as the unfused add gives
        sums[h * S::kLanes + tl] = s;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += (float)s[i];
      }
    }
  }
  floatx4 mean = block_sum_per_token<S::kLanes, THREADS>(acc, red, tl);
  mean *= 1.0f / (float)H;
  acc = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int h = rg; h < H; h += S::kRowGroups) {
    const half4 s = sums[h * S::kLanes + tl];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = (float)s[i] - mean[i];
      acc[i] += d * d;
    }
  }
  floatx4 rstd = block_sum_per_token<S::kLanes, THREADS>(acc, red, tl);
#pragma unroll
  for (int i = 0; i < 4; ++i) rstd[i] = rsqrtf(rstd[i] / (float)H + eps);
  if (!live) return;
  for (int h = rg; h < H; h += S::kRowGroups) {
    const half4 s = sums[h * S::kLanes + tl];
    const float w = gamma ? (float)gamma[h] : 1.0f, b = beta ? (float)beta[h] : 0.0f;
    half4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (_Float16)(((float)s[i] - mean[i]) * rstd[i] * w + b);
    store_four<RAGGED>(out + (size_t)h * T + t0, o, left);
  }
}

// The same for up to 128 * TRIP features with the sums kept in registers: no pass over LDS, two barriers (one per
// reduction) and the reductions on lane moves of the vector unit.  A workgroup's loads, gamma and beta among them, are all
// in flight together.  768 x 4096: 7.2 us against 8.7, 512 x 4096 5.6 against 6.9, 1024 x 8192 18.3 against 19.7.
template <int TRIP, bool RAGGED>
__global__ __launch_bounds__(512) void add_layernorm_held_kernel(int H, int T, const _Float16 *__restrict__ x, const _Float16 *__restrict__ a,
                                                                 const _Float16 *__restrict__ gamma, const _Float16 *__restrict__ beta,
                                                                 float eps, _Float16 *__restrict__ out) {
  typedef LnShape<16, 512, TRIP> S;
  __shared__ floatx4 red[2][8][S::kLanes];
  const int tl = threadIdx.x % S::kLanes, rg = threadIdx.x / S::kLanes, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;  // (as above)
  const int first = (((idx / S::kParts) * 8 + xcd) * S::kParts + (idx % S::kParts)) * 16;
  if (first >= T) return;
  const int t0 = first + 4 * tl;
  const bool live = t0 < T;
  const int left = T - t0;
  half4 s[TRIP], r[TRIP];
  float w[TRIP], b[TRIP];
#pragma unroll
  for (int u = 0; u < TRIP; ++u) {
    const int h = rg + u * S::kRowGroups;
    s[u] = half4{0, 0, 0, 0};
    r[u] = half4{0, 0, 0, 0};
    if (live && h < H) {
      s[u] = load_four<RAGGED, true>(x + (size_t)h * T + t0, left);
      if (a) r[u] = load_four<RAGGED, true>(a + (size_t)h * T + t0, left);
    }
  }
#pragma unroll
  for (int u = 0; u < TRIP; ++u) {
    const int h = rg + u * S::kRowGroups;
    w[u] = gamma && h < H ? (float)gamma[h] : 1.0f;
    b[u] = beta && h < H ? (float)beta[h] : 0.0f;
  }
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < TRIP; ++u) {
    s[u] = s[u] + r[u];  // fp16 sum, as the unfused add gives
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += (float)s[u][i];
  }
  floatx4 stat[2];  // mean, 1 / deviation
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = sum_over_quads(acc[i]);
    if (lane < S::kLanes) red[pass][wave][tl] = acc;
    __syncthreads();
    floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < 8; ++v) sum += red[pass][v][tl];
    stat[pass] = sum;
    if (pass == 0) {
      stat[0] *= 1.0f / (float)H;
      acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < TRIP; ++u) {
        if (rg + u * S::kRowGroups < H) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float d = (float)s[u][i] - stat[0][i];
            acc[i] += d * d;
          }
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) stat[1][i] = rsqrtf(stat[1][i] / (float)H + eps);
  if (!live) return;
#pragma unroll
  for (int u = 0; u < TRIP; ++u) {
    const int h = rg + u * S::kRowGroups;
    if (h >= H) break;
    half4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (_Float16)(((float)s[u][i] - stat[0][i]) * stat[1][i] * w[u] + b[u]);
    store_four<RAGGED>(out + (size_t)h * T + t0, o, left);
  }
}
template <int TRIP, bool RAGGED>
static hipError_t launch_ln_held(int H, int T, const uint16_t *x, const uint16_t *a, const uint16_t *gamma, const uint16_t *beta, float eps,
                                 uint16_t *out, hipStream_t stream) {
  const int line_groups = (T + 63) / 64, blocks = ((line_groups + 7) / 8) * 8 * 4;
  hipLaunchKernelGGL((add_layernorm_held_kernel<TRIP, RAGGED>), dim3(blocks), dim3(512), 0, stream, H, T, reinterpret_cast<const _Float16 *>(x),
                     reinterpret_cast<const _Float16 *>(a), reinterpret_cast<const _Float16 *>(gamma),
                     reinterpret_cast<const _Float16 *>(beta), eps, reinterpret_cast<_Float16 *>(out));
  return hipGetLastError();
}

template <int TOK, int THREADS, int TRIP, bool RAGGED>
static hipError_t launch_ln(int H, int T, const uint16_t *x, const uint16_t *a, const uint16_t *gamma, const uint16_t *beta,
                            float eps, uint16_t *out, hipStream_t stream) {
  const size_t lds = (size_t)H * TOK * 2 + (size_t)(THREADS / 64) * (TOK / 4) * 16;
  auto kern = add_layernorm_kernel<TOK, THREADS, TRIP, RAGGED>;
  if (lds > 64 * 1024) {
    // the runtime is told once per device and size
    static int raised[16] = {};
    static std::mutex raised_mutex;
    std::lock_guard<std::mutex> lock(raised_mutex);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) dev = -1;
    if (dev < 0 || raised[dev] < (int)lds) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
      if (dev >= 0) raised[dev] = (int)lds;
    }
  }
  const int line_groups = (T + 63) / 64;
  const int blocks = ((line_groups + 7) / 8) * 8 * (64 / TOK);
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(THREADS), lds, stream, H, T, reinterpret_cast<const _Float16 *>(x),
                     reinterpret_cast<const _Float16 *>(a), reinterpret_cast<const _Float16 *>(gamma),
                     reinterpret_cast<const _Float16 *>(beta), eps, reinterpret_cast<_Float16 *>(out));
  return hipGetLastError();
}

template <bool RAGGED>
static hipError_t launch_ln_any(int H, int T, const uint16_t *x, const uint16_t *a, const uint16_t *gamma,
                                const uint16_t *beta, float eps, uint16_t *out, hipStream_t stream) {
  // 16 tokens and eight waves per workgroup, six rows per thread in flight (measured on 768 x 4096 against 32 and 64
  // tokens, 4 to 16 waves, 3 to 12 rows: 8.5 us against 9-15); up to 1024 features the sums fit the registers of that shape,
  // beyond they take the pass over LDS.  So do most calls of 40 MiB and more, which is more than the L2 holds: the held sums'
  // registers leave fewer workgroups on a CU (three instead of four up to 512 features, two beyond; held to fewer they spill,
  // 512 x 8192 8.0 -> 8.8 us).  Held / over LDS, with a residual: 256 x 32768 23.7 / 20.5 us, 320 x 24576 21.6 / 19.8, 512 x 16384 21.5 /
  // 19.3, 512 x 65536 96 / 94, 448 x 24576 30.2 / 31.5; without: 384 x 32768 25.2 / 22.3, 512 x 32768 32.7 / 29.0, 640 x 32768 39.7 / 36.1,
  // 1024 x 16384 31.1 / 24.8.  On the other side: 384 x 16384 12.4 / 13.9, 512 x 8192 8.0 / 9.6, 128 x 65536 23.9 / 25.4 and, without,
  // 160 x 131072 41.4 / 47.0; more than 512 features with a residual, 640 x 32768 55.0 / 58.5, 1024 x 32768 84.9 / 91.2.
  const bool large = (int64_t)H * T * (a ? 6 : 4) >= (40 << 20);
  const bool held = H <= 1024 && !(large && H >= 256 && (H <= 512 || !a));
  if (held && H <= 512) return launch_ln_held<4, RAGGED>(H, T, x, a, gamma, beta, eps, out, stream);
  if (held && H <= 768) return launch_ln_held<6, RAGGED>(H, T, x, a, gamma, beta, eps, out, stream);
  if (held) return launch_ln_held<8, RAGGED>(H, T, x, a, gamma, beta, eps, out, stream);
  return launch_ln<16, 512, 6, RAGGED>(H, T, x, a, gamma, beta, eps, out, stream);
}
// (T a multiple of 4 with rows at multiples of 8 bytes keeps the kernels without the tests for a row's end)
hipError_t launch_add_layernorm(int H, int T, const uint16_t *x, const uint16_t *a, const uint16_t *gamma,
                                const uint16_t *beta, float eps, uint16_t *out, hipStream_t stream) {
  const bool whole = T % 4 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(out)) & 7u) == 0;
  return whole ? launch_ln_any<false>(H, T, x, a, gamma, beta, eps, out, stream) : launch_ln_any<true>(H, T, x, a, gamma, beta, eps, out, stream);
}

// ------------------------------------------------------------------------------------------
// Residual add + LayerNorm on token-major rows (the sparse attention encoder's activations [seq, batch, E]):
//   s = fp16(a + x) (a may be null: s = x),  out = LayerNorm(s),  and s itself where the next step wants it.
// HBM-bound (2 E bytes per row and operand).  LPR lanes hold a row, 8 x CH features each in 16-byte pieces: a row is
// loaded once, both passes of the statistics run on registers in fp32, and the sums cross the row's lanes with
// exchanges.  Rows shorter than 512 features share a wave, so that every lane carries a full piece (64 lanes on one
// row of 256 features would move 8 bytes each).  x may be a [seq, batch] view with strides of its own (the embedding
// is batch-major); everything else is dense.  32768 rows of 256 features: 11.9 us with the residual and (every other call) the
// sum, 4.6 TB/s; torch's LayerNorm took 37.6 us on them and its add another 8.4.
template <int LPR, int CH>
__global__ __launch_bounds__(256) void add_layernorm_rows_kernel(const AddLayerNormRows p) {
  constexpr int E = LPR * CH * 8, kRows = 256 / LPR;
  const int sub = threadIdx.x % LPR;
  const long long row = (long long)blockIdx.x * kRows + threadIdx.x / LPR;
  const bool live = row < p.rows;
  const long long r = live ? row : p.rows - 1;  // (lanes beyond the last row repeat it, without storing)
  const long long outer = r / p.inner, in = r - outer * p.inner;
  const _Float16 *xr = reinterpret_cast<const _Float16 *>(p.x) + outer * p.x_outer + in * p.x_inner + sub * 8;
  half8 s[CH], w[CH], b[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) s[c] = *reinterpret_cast<const half8 *>(xr + c * (LPR * 8));
  if (p.a) {
    const _Float16 *ar = reinterpret_cast<const _Float16 *>(p.a) + r * E + sub * 8;
#pragma unroll
    for (int c = 0; c < CH; ++c) s[c] = *reinterpret_cast<const half8 *>(ar + c * (LPR * 8)) + s[c];  // fp16 sum, as the unfused add gives
  }
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const half8 one = {1, 1, 1, 1, 1, 1, 1, 1}, zero = {0, 0, 0, 0, 0, 0, 0, 0};
    w[c] = p.gamma ? *reinterpret_cast<const half8 *>(reinterpret_cast<const _Float16 *>(p.gamma) + (c * LPR + sub) * 8) : one;
    b[c] = p.beta ? *reinterpret_cast<const half8 *>(reinterpret_cast<const _Float16 *>(p.beta) + (c * LPR + sub) * 8) : zero;
  }
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) sum += (float)s[c][i];
#pragma unroll
  for (int d = 1; d < LPR; d <<= 1) sum += __shfl_xor(sum, d, 64);
  const float mean = sum * (1.0f / (float)E);
  float sq = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float d = (float)s[c][i] - mean;
      sq += d * d;
    }
#pragma unroll
  for (int d = 1; d < LPR; d <<= 1) sq += __shfl_xor(sq, d, 64);
  const float rstd = rsqrtf(sq * (1.0f / (float)E) + p.eps);
  if (!live) return;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const long long at = row * E + (c * LPR + sub) * 8;
    half8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = (_Float16)(((float)s[c][i] - mean) * rstd * (float)w[c][i] + (float)b[c][i]);
    if (p.sum) *reinterpret_cast<half8 *>(reinterpret_cast<_Float16 *>(p.sum) + at) = s[c];
    *reinterpret_cast<half8 *>(reinterpret_cast<_Float16 *>(p.out) + at) = o;
  }
}

template <int LPR, int CH>
static hipError_t launch_ln_rows(const AddLayerNormRows &p, hipStream_t stream) {
  const long long blocks = (p.rows + 256 / LPR - 1) / (256 / LPR);
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((add_layernorm_rows_kernel<LPR, CH>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_add_layernorm_rows(int E, const AddLayerNormRows &p, hipStream_t stream) {
  switch (E) {
    case 64: return launch_ln_rows<8, 1>(p, stream);
    case 128: return launch_ln_rows<16, 1>(p, stream);
    case 256: return launch_ln_rows<32, 1>(p, stream);
    case 512: return launch_ln_rows<64, 1>(p, stream);
    case 1024: return launch_ln_rows<64, 2>(p, stream);
    case 2048: return launch_ln_rows<64, 4>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

// ------------------------------------------------------------------------------------------
// Dense softmax(Q^T K / sqrt(d)) attention on feature-major activations (the dense attention of the
// reference's comparison block, reference end2end/sspmm_e2e/end_to_end.py:84-97, which runs it in torch on
// token-major tensors).  The SpMM that produces q, k, v leaves them as [features, tokens]; torch's attention
// wants [batch, heads, tokens, head size] with the head size contiguous, which costs one transposed copy of all
// three before it and one of the context behind it.  Here a workgroup of four waves owns 64 queries of one
// (batch element, head): its 64 columns of Q go to LDS once, and the head's K and V pass through LDS in blocks of
// 64 keys (64 features x 64 tokens each, as they lie in memory; two buffers, the next block's loads in flight in
// registers while the current one is computed, one barrier per block), 45 KB of LDS in all, so three workgroups
// share a CU.  Each wave computes for 32 queries (two sets of 16) and half of every block's keys
//     scores^T[key, query] = sum_d K[d, key] Q[d, query]          (MFMA; both operands by transpose reads)
//     out[d, query]        = sum_key V[d, key] P[query, key]       (MFMA; V read directly, P from registers)
// per block with the running maximum and sum of the usual one-pass softmax.  The scores come out of the first
// product with a query per lane and four consecutive keys per accumulator, which is the second product's operand
// layout once its contraction slots are numbered accordingly (slots 0-3 and 4-7 of lane group g = keys 4g .. 4g+3
// of two neighbouring 16-key tiles; V is read with the same numbering), so the probabilities never leave the
// registers.  The context goes back through LDS and is written feature-major in whole 128-byte lines.  Bound by
// HBM in bytes (q, k, v read once, out written once: 8 * hidden * tokens bytes; a head's K and V are re-read by its
// seq / 64 workgroups from L2), by the exponentials and the LDS reads in time.
// 8 x 512 tokens, 12 heads, inside the layer: 18.0 -> 16.8 to 17.5 us with the maxima exchanged by lane swaps instead of permutes through the LDS and
// V's operands read ahead of the exponentials.  (Sums of the probabilities as fp16 holds them, four dot products for eight additions, are level:
// 17.0 and 17.1 in the same two runs.)
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

static constexpr int kAttThreads = 256;
static constexpr int kAttD = 64;          // head size
static constexpr int kAttQueries = 64;    // per workgroup, 16 per wave
static constexpr int kAttKeys = 64;       // per block of the softmax
// Row pitches in bytes, chosen so that the rows one LDS pass touches fall into different banks.  Q and K are read by
// transpose reads, 32 lanes = eight consecutive rows of 32 bytes per pass: 160-byte rows put them at bank offsets
// 0, 40, 16, 56, 32, 8, 48, 24 (of 64 four-byte banks), each eight banks wide.  V is read eight bytes per lane from
// sixteen consecutive rows: 144-byte rows put those at sixteen different multiples of four banks.
static constexpr uint32_t kAttPitchK = 64 * 2 + 32;
static constexpr uint32_t kAttPitchV = 64 * 2 + 16;
static constexpr uint32_t kAttTileK = kAttD * kAttPitchK, kAttTileV = kAttD * kAttPitchV;
static constexpr size_t kAttLds = 3 * (size_t)kAttTileK + 2 * (size_t)kAttTileV;  // Q, two K blocks, two V blocks
static constexpr int kAttMaxSeq = 16384;

union AttOperand {
  half8 h;
  uint32_t u[4];
};

__device__ __forceinline__ uint32_t att_pack(float lo, float hi) {
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  const half2v h = {(_Float16)lo, (_Float16)hi};
  return __builtin_bit_cast(uint32_t, h);
}

// v with its infinities (and NaN) replaced by the largest finite number.
__device__ __forceinline__ half8 att_bounded(half8 v) {
  const _Float16 x = (_Float16)65504;
  const half8 most = {x, x, x, x, x, x, x, x};
  return __builtin_elementwise_max(__builtin_elementwise_min(v, most), -most);
}

struct AttentionArgs {
  const _Float16 *q, *k, *v;
  _Float16 *out;
  long long ld, ld_out;  // elements between consecutive features
  int S, heads, units;  // units = batch elements x heads
  float scale_log2e;
};

// A piece of eight tokens of which `left` are inside the sequence.  RAGGED: rows begin at any element, and what lies behind
// the sequence (another one's tokens, or nothing) is neither read nor written.
typedef uint32_t uintx4_any __attribute__((ext_vector_type(4), aligned(2)));
template <bool RAGGED>
__device__ __forceinline__ uintx4 att_load(const _Float16 *p, int left) {
  if constexpr (RAGGED) {
    if (left >= 8) return *reinterpret_cast<const uintx4_any *>(p);
    half8 h = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 7; ++i)
      if (i < left) h[i] = p[i];
    return __builtin_bit_cast(uintx4, h);
  } else {
    return *reinterpret_cast<const uintx4 *>(p);
  }
}
template <bool RAGGED>
__device__ __forceinline__ void att_store(_Float16 *p, uintx4 v, int left) {
  if constexpr (RAGGED) {
    if (left >= 8) {
      *reinterpret_cast<uintx4_any *>(p) = v;
      return;
    }
    const half8 h = __builtin_bit_cast(half8, v);
#pragma unroll
    for (int i = 0; i < 7; ++i)
      if (i < left) p[i] = h[i];
  } else {
    *reinterpret_cast<uintx4 *>(p) = v;
  }
}

// RAGGED: sequences of any length and rows at any element.  The last block of keys is filled up with zeros, whose
// probabilities are set to zero; the last block of queries likewise, without being stored.  Such calls ran on torch's attention
// between two relayout copies, whose error against float64 is 2.7e-4 (12 heads, 500 tokens) where this kernel's is 2.9e-4, the
// probabilities' rounding for the most part; so RAGGED adds what that rounding leaves as a second product: 2.1e-4, the rounding
// of the result.  8 x 500 tokens: 25 us (21 without it, 15 for 8 x 512) against 69.
template <bool RAGGED>
__global__ __launch_bounds__(kAttThreads, 3) void attention_fm_kernel(const AttentionArgs p) {
  __shared__ __align__(16) unsigned char lds[kAttLds + (RAGGED ? 16 : 0)];
  int *const again = reinterpret_cast<int *>(lds + kAttLds);  // (RAGGED)
  const int S = p.S, qblocks = (S + kAttQueries - 1) / kAttQueries, blocks = (S + kAttKeys - 1) / kAttKeys;
  // Workgroup ids go round-robin to the 8 XCDs, each with its own L2: the query blocks of one (batch element, head)
  // take ids 8 apart, so that the head's K and V are fetched from memory once and found in that L2 by the others.
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int qb = idx % qblocks, unit = (idx / qblocks) * 8 + xcd;
  if (unit >= p.units) return;  // (the grid is padded to a multiple of eight units)
  const int head = unit % p.heads, b = unit / p.heads;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char *const q_tile = lds;
  unsigned char *const k_tiles = lds + kAttTileK;      // buffer i at k_tiles + i * kAttTileK
  unsigned char *const v_tiles = lds + 3 * kAttTileK;  // buffer i at v_tiles + i * kAttTileV
  const long long tok0 = (long long)b * S;
  const _Float16 *qg = p.q + (long long)(head * kAttD) * p.ld + tok0 + qb * kAttQueries;
  const _Float16 *kg = p.k + (long long)(head * kAttD) * p.ld + tok0;
  const _Float16 *vg = p.v + (long long)(head * kAttD) * p.ld + tok0;

  // A 64 x 64 fp16 tile is 512 pieces of 16 bytes, two per thread: rows r0 and r0 + 32, piece pc.
  const int r0 = tid >> 3, pc = tid & 7;
  const long long g0 = (long long)r0 * p.ld + pc * 8, g1 = g0 + 32 * p.ld;
  const uint32_t l0 = r0 * kAttPitchK + pc * 16, l1 = l0 + 32 * kAttPitchK;    // in a Q or K tile
  const uint32_t lv0 = r0 * kAttPitchV + pc * 16, lv1 = lv0 + 32 * kAttPitchV;  // in a V tile
  const int left = S - pc * 8, left_q = left - qb * kAttQueries;  // tokens of the sequence from the thread's piece on
  uintx4 kk[2], vv[2];
  kk[0] = att_load<RAGGED>(kg + g0, left);
  kk[1] = att_load<RAGGED>(kg + g1, left);
  vv[0] = att_load<RAGGED>(vg + g0, left);
  vv[1] = att_load<RAGGED>(vg + g1, left);
  *reinterpret_cast<uintx4 *>(q_tile + l0) = att_load<RAGGED>(qg + g0, left_q);
  *reinterpret_cast<uintx4 *>(q_tile + l1) = att_load<RAGGED>(qg + g1, left_q);
  *reinterpret_cast<uintx4 *>(k_tiles + l0) = kk[0];
  *reinterpret_cast<uintx4 *>(k_tiles + l1) = kk[1];
  *reinterpret_cast<uintx4 *>(v_tiles + lv0) = vv[0];
  *reinterpret_cast<uintx4 *>(v_tiles + lv1) = vv[1];
  if (RAGGED && tid == 0) *again = 0;
  __syncthreads();

  // ---- Wave w works on queries 32 * (w / 2) .. + 31 of the workgroup's 64 (two sets of 16) against keys
  // 32 * (w % 2) .. + 31 of every block: an operand read of K or V then serves two products (the two query sets),
  // which halves the LDS reads per product, and the two waves that share queries merge their softmax states at the end.
  // The contraction slots of the first product are numbered so that a transpose read of 32 lanes touches eight
  // consecutive rows: slots 0-3 of lane group g are features 32u + 4g .. + 3, slots 4-7 features 32u + 16 + 4g .. + 3
  // (the same numbering for Q and K).
  const int qhalf = wave >> 1, khalf = wave & 1;
  AttOperand qop[2][2];  // [query set][u]: lane (m, g) holds its slots of query 32 * qhalf + 16 * set + m
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const unsigned char *a = q_tile + (32 * u + 4 * g + (m >> 2)) * kAttPitchK + (32 * qhalf + 16 * j) * 2 + (m & 3) * 8;
      const uintx2 lo = lds_read_tr(a), hi = lds_read_tr(a + 16 * kAttPitchK);
      qop[j][u].u[0] = lo[0]; qop[j][u].u[1] = lo[1]; qop[j][u].u[2] = hi[0]; qop[j][u].u[3] = hi[1];
    }

  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 o[2][4] = {{zero, zero, zero, zero}, {zero, zero, zero, zero}};  // [set][dt], lane (m, g): features 16dt + 4g .. + 3 of query m
  // per query set, of query m: the largest raw score so far, and this lane's share of the sum of
  // 2^((score - max) * scale_log2e), over the keys of this wave
  float run_max[2] = {-3.0e38f, -3.0e38f}, run_sum[2] = {0.f, 0.f};
  const float c = p.scale_log2e;  // > 0: the largest scaled score is the scaled largest score
  const uint32_t k_rd = (4 * g + (m >> 2)) * kAttPitchK + (m & 3) * 8 + (32 * khalf) * 2;
  const uint32_t v_rd = m * kAttPitchV + (4 * g) * 2 + (32 * khalf) * 2;
  // what the two waves of a query half exchange at the end
  floatx4 *const xo = reinterpret_cast<floatx4 *>(k_tiles) + qhalf * (2 * 4 * 64);  // [set][dt][lane]
  float *const xs = reinterpret_cast<float *>(k_tiles + 2 * (2 * 4 * 64) * 16) + qhalf * (2 * 2 * 64);  // [set][max, sum][lane]
  // What the rounding of the probabilities leaves (RAGGED) is of either sign or zero: against an infinite value it makes NaN where the
  // probability alone makes infinity.  A workgroup with a NaN goes over its keys once more with V bounded in that product.
  // 8 x 500 tokens: 24.2 us without the test for NaN, 25.4 with it; bounded the first time 26.7, a second copy of the loop 25.6.
  for (bool bounded = false;; bounded = true) {
    for (int kb = 0; kb < blocks; ++kb) {
      const unsigned char *const k_tile = k_tiles + (kb & 1) * kAttTileK;
      const unsigned char *const v_tile = v_tiles + (kb & 1) * kAttTileV;
      const bool more = kb + 1 < blocks;  // uniform
      if (more) {
        const int off = (kb + 1) * kAttKeys;
        kk[0] = att_load<RAGGED>(kg + g0 + off, left - off);
        kk[1] = att_load<RAGGED>(kg + g1 + off, left - off);
        vv[0] = att_load<RAGGED>(vg + g0 + off, left - off);
        vv[1] = att_load<RAGGED>(vg + g1 + off, left - off);
      }
      // scores^T: s[set][kt], lane (m, g): keys 32 * khalf + 16kt + 4g .. + 3 of the block against query m of the set
      floatx4 s[2][2] = {{zero, zero}, {zero, zero}};
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const unsigned char *a = k_tile + k_rd + (32 * u) * kAttPitchK + (16 * kt) * 2;
          const uintx2 lo = lds_read_tr(a), hi = lds_read_tr(a + 16 * kAttPitchK);
          AttOperand kop;
          kop.u[0] = lo[0]; kop.u[1] = lo[1]; kop.u[2] = hi[0]; kop.u[3] = hi[1];
#pragma unroll
          for (int j = 0; j < 2; ++j) s[j][kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop.h, qop[j][u].h, s[j][kt], 0, 0, 0);
        }
      }
      // keys of this lane's accumulators that lie in the sequence: those below (all of them in every block but the last)
      const int keys_left = S - kb * kAttKeys - 32 * khalf - 4 * g;
      const bool cut = RAGGED && (kb + 1) * kAttKeys > S;  // uniform
      if (cut) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (16 * kt + r >= keys_left) s[0][kt][r] = s[1][kt][r] = -3.0e38f;
      }
      // V's operands are read ahead of the exponentials (RAGGED, whose products take more registers, reads them where it uses them)
      AttOperand vops[4];
      const auto read_v = [&](int dt) {
        const unsigned char *a = v_tile + v_rd + (16 * dt) * kAttPitchV;
        const uintx2 lo = *reinterpret_cast<const uintx2 *>(a), hi = *reinterpret_cast<const uintx2 *>(a + 32);
        vops[dt].u[0] = lo[0]; vops[dt].u[1] = lo[1]; vops[dt].u[2] = hi[0]; vops[dt].u[3] = hi[1];
      };
      if constexpr (!RAGGED) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) read_v(dt);
        __builtin_amdgcn_sched_barrier(0);
      }
      AttOperand rest[2];  // (RAGGED) what the rounding of the probabilities leaves
      AttOperand pop[2];  // per set: contraction slots 0-3 = keys 4g .. + 3 of tile 0, slots 4-7 = the same keys of tile 1
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float mx = s[j][0][0];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[j][kt][r]);
        if constexpr (RAGGED) {  // (25.9 us at 8 x 500 tokens, 26.2 with the lane swaps)
          mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
          mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        } else {
          mx = max_over_rows(mx);
        }
        // The reference point of the exponentials moves only when some query's maximum has grown by more than 8 in
        // the base-2 domain (a wave-uniform decision): until then the probabilities are at most 2^8 times too large,
        // which fp16 holds, the running sums and the context stay consistent with the old reference point, and the
        // rescaling of the accumulators, which after the first block is nearly always by 1, is skipped.
        const float new_max = fmaxf(run_max[j], mx);
        if (__ballot((new_max - run_max[j]) * c > 8.0f) != 0) {
          const float alpha = __builtin_amdgcn_exp2f(fmaxf((run_max[j] - new_max) * c, -126.0f));
          run_max[j] = new_max;
          run_sum[j] *= alpha;
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) o[j][dt] *= alpha;
        }
        const float shift = -run_max[j] * c;
        float part = 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            s[j][kt][r] = __builtin_amdgcn_exp2f(fmaf(s[j][kt][r], c, shift));
            if (cut && 16 * kt + r >= keys_left) s[j][kt][r] = 0.f;  // (a wave may have had no key at all yet)
            part += s[j][kt][r];
          }
        run_sum[j] += part;
        pop[j].u[0] = att_pack(s[j][0][0], s[j][0][1]);
        pop[j].u[1] = att_pack(s[j][0][2], s[j][0][3]);
        pop[j].u[2] = att_pack(s[j][1][0], s[j][1][1]);
        pop[j].u[3] = att_pack(s[j][1][2], s[j][1][3]);
        if constexpr (RAGGED) {
#pragma unroll
          for (int i = 0; i < 8; ++i) rest[j].h[i] = (_Float16)(s[j][i >> 2][i & 3] - (float)pop[j].h[i]);
        }
      }
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        if (RAGGED) read_v(dt);
        const AttOperand vop = vops[dt];
        half8 vrest = vop.h;
        if (RAGGED && __builtin_expect(bounded, 0)) vrest = att_bounded(vrest);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if constexpr (RAGGED) o[j][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vrest, rest[j].h, o[j][dt], 0, 0, 0);
          o[j][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop.h, pop[j].h, o[j][dt], 0, 0, 0);
        }
      }
      if (more) {  // the other buffer: every wave finished reading it before the barrier that ended the previous block
        unsigned char *const kn = k_tiles + ((kb + 1) & 1) * kAttTileK, *const vn = v_tiles + ((kb + 1) & 1) * kAttTileV;
        *reinterpret_cast<uintx4 *>(kn + l0) = kk[0];
        *reinterpret_cast<uintx4 *>(kn + l1) = kk[1];
        *reinterpret_cast<uintx4 *>(vn + lv0) = vv[0];
        *reinterpret_cast<uintx4 *>(vn + lv1) = vv[1];
      }
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      run_sum[j] += __shfl_xor(run_sum[j], 16, 64);
      run_sum[j] += __shfl_xor(run_sum[j], 32, 64);
    }

    // ---- The two waves of a query half merge: the one with the upper keys leaves its state in LDS (over the K tiles:
    // the loop's last barrier is behind every read of them), the other adds it to its own.
    if constexpr (RAGGED) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) sum += (o[j][dt][0] + o[j][dt][1]) + (o[j][dt][2] + o[j][dt][3]);
      const bool nan = sum != sum;  // (or infinities of both signs)
      if (__ballot(nan) != 0 && lane == 0) *again = 1;
    }
    if (khalf == 1) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) xo[(j * 4 + dt) * 64 + lane] = o[j][dt];
        xs[(j * 2 + 0) * 64 + lane] = run_max[j];
        xs[(j * 2 + 1) * 64 + lane] = run_sum[j];
      }
    }
    __syncthreads();
    if (!RAGGED || bounded || __builtin_amdgcn_readfirstlane(*again) == 0) break;
    __syncthreads();
    *reinterpret_cast<uintx4 *>(k_tiles + l0) = att_load<RAGGED>(kg + g0, left);
    *reinterpret_cast<uintx4 *>(k_tiles + l1) = att_load<RAGGED>(kg + g1, left);
    *reinterpret_cast<uintx4 *>(v_tiles + lv0) = att_load<RAGGED>(vg + g0, left);
    *reinterpret_cast<uintx4 *>(v_tiles + lv1) = att_load<RAGGED>(vg + g1, left);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      run_max[j] = -3.0e38f;
      run_sum[j] = 0.f;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[j][dt] = zero;
    }
    __syncthreads();
  }
  if (khalf == 0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float m1 = xs[(j * 2 + 0) * 64 + lane], l1 = xs[(j * 2 + 1) * 64 + lane];
      const float mm = fmaxf(run_max[j], m1);
      const float a0 = __builtin_amdgcn_exp2f(fmaxf((run_max[j] - mm) * c, -126.0f));
      const float a1 = __builtin_amdgcn_exp2f(fmaxf((m1 - mm) * c, -126.0f));
      const float inv = 1.0f / (run_sum[j] * a0 + l1 * a1);
      // the context through LDS (over the query tile: every wave read its queries before the first barrier of the
      // loop) and out in whole lines
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const floatx4 other = xo[(j * 4 + dt) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *reinterpret_cast<_Float16 *>(q_tile + (16 * dt + 4 * g + r) * kAttPitchK + (32 * qhalf + 16 * j + m) * 2) =
              (_Float16)((o[j][dt][r] * a0 + other[r] * a1) * inv);
      }
    }
  }
  __syncthreads();
  _Float16 *og = p.out + (long long)(head * kAttD) * p.ld_out + tok0 + qb * kAttQueries;
  att_store<RAGGED>(og + (long long)r0 * p.ld_out + pc * 8, *reinterpret_cast<const uintx4 *>(q_tile + l0), left_q);
  att_store<RAGGED>(og + (long long)(r0 + 32) * p.ld_out + pc * 8, *reinterpret_cast<const uintx4 *>(q_tile + l1), left_q);
}

bool attention_fm_applies(int batch, int heads, int seq, int head_dim, const void *q, const void *k, const void *v,
                          long long ld, const void *out, long long ld_out) {
  const auto aligned = [](const void *x) { return (reinterpret_cast<uintptr_t>(x) & 15u) == 0; };
  return batch > 0 && heads > 0 && head_dim == kAttD && seq >= kAttQueries && seq % kAttQueries == 0 && seq <= kAttMaxSeq &&
         ld % 8 == 0 && ld_out % 8 == 0 && aligned(q) && aligned(k) && aligned(v) && aligned(out) &&
         ((long long)batch * heads + 7) * (seq / kAttQueries) <= 0x7fffffffLL;
}

bool attention_fm_ragged_applies(int batch, int heads, int seq, int head_dim, const void *q, const void *k, const void *v, const void *out) {
  const auto aligned = [](const void *x) { return (reinterpret_cast<uintptr_t>(x) & 1u) == 0; };
  return batch > 0 && heads > 0 && head_dim == kAttD && seq >= 1 && seq <= kAttMaxSeq && aligned(q) && aligned(k) && aligned(v) &&
         aligned(out) && ((long long)batch * heads + 7) * ((seq + kAttQueries - 1) / kAttQueries) <= 0x7fffffffLL;
}

hipError_t launch_attention_fm(int batch, int heads, int seq, const uint16_t *q, const uint16_t *k, const uint16_t *v,
                               long long ld, uint16_t *out, long long ld_out, float scale, hipStream_t stream) {
  AttentionArgs a;
  a.q = reinterpret_cast<const _Float16 *>(q);
  a.k = reinterpret_cast<const _Float16 *>(k);
  a.v = reinterpret_cast<const _Float16 *>(v);
  a.out = reinterpret_cast<_Float16 *>(out);
  a.ld = ld;
  a.ld_out = ld_out;
  a.S = seq;
  a.heads = heads;
  a.units = batch * heads;
  a.scale_log2e = scale * 1.4426950408889634f;
  const long long units_padded = (((long long)batch * heads + 7) / 8) * 8;
  const unsigned blocks = (unsigned)(units_padded * ((seq + kAttQueries - 1) / kAttQueries));
  // (whole tiles at aligned rows keep the kernel without the tests for what lies behind a sequence)
  if (attention_fm_applies(batch, heads, seq, kAttD, q, k, v, ld, out, ld_out))
    hipLaunchKernelGGL(attention_fm_kernel<false>, dim3(blocks), dim3(kAttThreads), 0, stream, a);
  else
    hipLaunchKernelGGL(attention_fm_kernel<true>, dim3(blocks), dim3(kAttThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace sspmm
