// The dense part of a sparse attention block in one launch (the reference runs it as torch modules, reference
// end2end/sspmm_e2e/end_to_end.py:58-75: output projection, + x, LayerNorm, two linear layers, + x, and the next
// block's LayerNorm and input projection).
//
// As separate launches every one of these reads and writes an activation of tokens x 256 to 1024 features, and the
// matrix products are then bound by those bytes, not by the matrix units.  Here a workgroup keeps TM tokens from the
// attention's output to the next block's projection: four waves split the output features of every product, the
// activations pass between the products through LDS as fp16, and the accumulators of the second linear layer stay in
// registers while the hidden features are made and used 256 at a time.
//
// Orientation: out^T[feature, token] = W (MFMA operand A, 16 features x 32 k) * act^T (operand B, 32 k x 16 tokens).
// Both operands then are eight consecutive k per lane: W comes straight from global memory (row-major as torch keeps it;
// a wave reads only the rows of its own features, so nothing is loaded twice by a workgroup and LDS is not involved),
// act from LDS rows padded by 32 bytes (by 16 both layers took 59 us at 32768 tokens, by 32 or 48 56 to 58).  The rows of a wave's feature
// tiles are dealt so that two tiles leave a lane eight consecutive features of one token (feature 32 (j / 2) + 8 g + 4 (j % 2)
// + i of tile j, accumulator i, lane group g): residual loads, LDS writes and stores are 16-byte pieces, of which the
// four lane groups make 64 consecutive bytes.
//
// There is nothing between the two linear layers, so the encoder's forward pass has them multiplied first (fold_rows, once a pass)
// where that makes fewer weights: 0.39 M products a token in the place of 0.79, and 0.79 MB of weights to stream instead of
// 1.6.  W2 W1 comes as two fp16 matrices, what it is rounded to and what the rounding left.  The layers one after the other take W1 and W2
// as they are and round what comes out of W1, after all that W1 cancels (a mean along its rows against the LayerNorm's output, a bias
// against beta): one rounded matrix, whose elements know nothing of that, misses float64 by up to fifteen times as much (256 x 1024, rows of
// W1 with a mean of sixteen deviations: rms of x' 3.3e-3, the layers 3.6e-4), the two by less than the layers (2.9e-4), for 0.065 M products a token.
// 256 features, 1024 hidden ones, in a model, both layers / one matrix / two: 8192 tokens 26.7 / 16.3 / 17.7 us a launch, 32768 tokens 61 / 38.3 / 40.0;
// what packs the weights and multiplies them takes 13 us a pass for four blocks, where packing all took 7.6.  (Both layers, where they are the
// narrower ones and for callers that bring them packed: the rest of this paragraph.)
//
// The launch in front of the first block looks the tokens up in the embedding's table itself: as a launch of its own the lookup wrote
// and this one read tokens x E halfs that no one else wants (256 features, four blocks: 8192 tokens 194 -> 180 us the forward pass,
// 32768 tokens 546 -> 507).
//
// The weights a workgroup streams from L2 are 1.6 MB at 256 features and 1024 hidden ones, 25k cycles at the 64 bytes a
// cycle of a CU, whatever TM, and the products 384 cycles per token.  The loads of the next two units (eight 16-byte
// loads of a wave each) are in flight throughout, also across the products' boundaries; four units, at 64 registers more, were
// level at best and slower where they make the compiler spill (512 features, 32768 tokens: 164 us, with two 149).  The matrices are packed by
// a launch of their own first (7 us for the 6.7 MB of a model of four blocks), so that a load instruction reads 1 KB in a
// row: from torch's layout it reads 64 bytes of each of sixteen rows, which lie 512 to 2048 bytes apart on a few of the L2's
// channels, and 32 tokens per workgroup took 61 us instead of 27 (8192 tokens).
//
// 256 features, 1024 hidden, 768 out, with the LayerNorms, both layers / folded (this paragraph: one matrix): 8192 tokens 25.7 / 16.5 us, 32768 tokens 62.6 / 38.5,
// against 104 (the host) and 121 for the four library products and two LayerNorm launches.  Where a folded launch's cycles go: 8192 tokens
// 26 000: 4000 until the attention's output is there, 2400 to 2700 a product of 256 x 256 (2048 at 64 bytes of weights a cycle), 1900 a LayerNorm, 1300 the
// stores of 256 outputs; 32768 tokens 58 000, 12 to 13 000 of them until all workgroups' 33 MB are there, and the stores at the end, 7 us of them, as
// exposed.  Without gain: loads of x and the attention's output in front of the first weights, the weights fetched into L2 ahead by a load a thread,
// four units of the last product's weights in flight, the last product's bias in its accumulators (its load waits for the stores).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "block_kernels.h"
#include "lane_ops.h"

namespace sspmm {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

constexpr int kChunk = 256;  // hidden (or output) features a workgroup makes at a time, 64 per wave

template <int NJ>
struct Unit {  // what is loaded together: NJ tiles of 16 features x K values of k
  static constexpr int K = NJ == 8 ? 32 : 64;
  static constexpr uint32_t kBytes = 32u * NJ * K;
};

// A wave's share of a packed weight matrix: its 16 * NJ rows, from column k0 on.  Every unit that is asked for lies inside
// the matrix.
struct Weights {
  __amdgpu_buffer_rsrc_t srd;
  uint32_t base;
};
template <int NJ>
__device__ __forceinline__ Weights weights(const uint16_t *w, int rows, int cols, int row0, int k0) {
  Weights r;
  r.srd = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(w), 0, (int)((uint32_t)rows * (uint32_t)cols * 2u), 0x00020000);
  r.base = (uint32_t)row0 * (uint32_t)cols * 2u + (uint32_t)(k0 / Unit<NJ>::K) * Unit<NJ>::kBytes;
  return r;
}
template <int NJ>
__device__ __forceinline__ void issue(uintx4 (&w)[8], const Weights &a, int unit) {
  const uint32_t lane16 = (threadIdx.x & 63u) * 16u;
#pragma unroll
  for (int i = 0; i < (int)(Unit<NJ>::kBytes / 1024u); ++i)
    w[i] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(a.srd, lane16 + (i & 3) * 1024u,
                                                                            a.base + unit * Unit<NJ>::kBytes + (i >> 2) * 4096u, 0));
}
template <int NJ, int D>
__device__ __forceinline__ void issue_first(uintx4 (&w)[D][8], const Weights &a) {
#pragma unroll
  for (int u = 0; u < D; ++u) issue<NJ>(w[u], a, u);
}

// acc[tile of 16 tokens][tile of 16 features] += W * act^T over K.  The first D units of `cur` are in `w` or on their way;
// on return those of `next` (tiles of NEXT) are.  act: the lane's address in the LDS rows (row lane % 16, k = 8 (lane / 16)).
template <int TT, int NJ, int K, int PITCH, int NEXT, int D>
__device__ __forceinline__ void gemm(floatx4 (&acc)[TT][NJ], const unsigned char *act, const Weights &cur, const Weights &next,
                                     uintx4 (&w)[D][8]) {
  constexpr int KU = Unit<NJ>::K, U = K / KU;
  static_assert(U % D == 0, "the units of a product rotate through the buffers whole");
  constexpr int S = KU / 32;  // steps of a unit
  half8 b[2][TT];
#pragma unroll
  for (int t = 0; t < TT; ++t) b[0][t] = *reinterpret_cast<const half8 *>(act + t * 16 * PITCH);
#pragma unroll
  for (int s = 0; s < U * S; ++s) {
    const int u = s / S;
    if (s + 1 < U * S) {
#pragma unroll
      for (int t = 0; t < TT; ++t) b[(s + 1) & 1][t] = *reinterpret_cast<const half8 *>(act + t * 16 * PITCH + (s + 1) * 64);
    }
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        acc[t][j] =
            __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, w[u % D][(s % S) * NJ + j]), b[s & 1][t], acc[t][j], 0, 0, 0);
    if (s % S == S - 1) {
      if (u + D < U)
        issue<NJ>(w[u % D], cur, u + D);
      else
        issue<NEXT>(w[u % D], next, u + D - U);
    }
    // (left alone, the scheduler pulls the reads of many steps ahead and spills)
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The lane's 4 * NJ values of one row (16-byte pieces, 32 features apart) as they lie in memory, and one of them widened.
template <int NJ>
__device__ __forceinline__ void load_row(half8 (&v)[NJ / 2], const uint16_t *p) {
#pragma unroll
  for (int j = 0; j < NJ / 2; ++j) v[j] = *reinterpret_cast<const half8 *>(p + 32 * j);
}
template <int N>
__device__ __forceinline__ float value(const half8 (&v)[N], int j, int i) { return (float)v[j / 2][(j & 1) * 4 + i]; }
// Per-feature values (bias, gamma, beta); `none` where there is no such vector.
template <int NJ>
__device__ __forceinline__ void feature_values(half8 (&v)[NJ / 2], const uint16_t *p, int first, float none) {
  if (p) {
    load_row<NJ>(v, p + first);
  } else {
#pragma unroll
    for (int j = 0; j < NJ / 2; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) v[j][i] = (_Float16)none;
  }
}

// A lane's 4 * NJ features of one token as 16-byte pieces.
template <int NJ>
__device__ __forceinline__ void put_row(unsigned char *p, const floatx4 (&v)[NJ]) {
#pragma unroll
  for (int j = 0; j < NJ; j += 2) {
    half8 h;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      h[i] = (_Float16)v[j][i];
      h[4 + i] = (_Float16)v[j + 1][i];
    }
    *reinterpret_cast<half8 *>(p + j * 32) = h;
  }
}

// v = LayerNorm(v) over the E features of every token, statistics in fp32.  s: the lane's sums of v.  A wave takes the mean of its E / 4
// features of a token and the squares' sum about it, and the four waves' pairs are put together as Chan, Golub and LeVeque do (1979): one
// exchange through `part` [4][TM] and one barrier, where the mean first and then the squares about it took two.  At 8192 tokens of 256
// features nothing runs beside it: with lane permutes, two exchanges, and gamma and beta loaded here, behind the weights in flight, the two LayerNorms took
// 2680 and 2340 of a workgroup's 27 300 cycles, now (lane swaps, gamma and beta in LDS from the start) 1880 and 1930.
template <int TT, int NJ, int E>
__device__ __forceinline__ void layer_norm(floatx4 (&v)[TT][NJ], float (&s)[TT], const uint16_t *gamma_beta, float eps, int first, floatx2 *part,
                                           int wave, int lane) {
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    s[t] = sum_over_rows(s[t]) * (4.0f / (float)E);
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[t][j][i] -= s[t];
        q = __builtin_fmaf(v[t][j][i], v[t][j][i], q);
      }
    part[wave * (TT * 16) + t * 16 + (lane & 15)] = floatx2{s[t], sum_over_rows(q)};  // (the four lane groups hold the same)
  }
  lds_barrier();
  half8 w[NJ / 2], b[NJ / 2];
  load_row<NJ>(w, gamma_beta + first);
  load_row<NJ>(b, gamma_beta + E + first);
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    const floatx2 *const at = part + t * 16 + (lane & 15);
    const floatx2 x0 = at[0], x1 = at[TT * 16], x2 = at[2 * TT * 16], x3 = at[3 * TT * 16];
    const float mean = ((x0[0] + x1[0]) + (x2[0] + x3[0])) * 0.25f;
    const float d0 = x0[0] - mean, d1 = x1[0] - mean, d2 = x2[0] - mean, d3 = x3[0] - mean;
    const float between = (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
    const float q = (x0[1] + x1[1]) + (x2[1] + x3[1]);
    const float rstd = rsqrtf(q * (1.0f / (float)E) + between * 0.25f + eps), shift = (s[t] - mean) * rstd;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[t][j][i] = __builtin_fmaf(v[t][j][i], rstd, shift) * value(w, j, i) + value(b, j, i);
  }
}

constexpr int block_waves(int E, int TM) { return TM == 16 || (TM == 64 && E < 512) ? 2 : 1; }  // per SIMD

enum Part { kNoAttention, kTwoLayers, kFolded };  // what lies in front of the last LayerNorm

template <int E, int TM, Part PART>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(block_waves(E, TM), block_waves(E, TM)))) void block_dense_kernel(const BlockDenseArgs p) {
  constexpr int NT = E / 64, TT = TM / 16, D = 2;
  constexpr int kPitchA = E * 2 + 32, kPitchH = kChunk * 2 + 32;
  __shared__ __align__(16) unsigned char act[TM * kPitchA];  // attention's output, then n, then h
  __shared__ __align__(16) unsigned char hid[PART == kTwoLayers ? TM * kPitchH : 16];  // kChunk hidden features
  __shared__ __align__(16) float affine[PART == kFolded ? 2 * E : 4];
  __shared__ __align__(16) uint16_t norms[4 * E];  // gamma and beta of both LayerNorms
  __shared__ __align__(8) floatx2 part[4 * TM];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m = lane & 15, g = lane >> 4;
  const long long t0 = (long long)blockIdx.x * TM;
  const int left = (int)min((long long)TM, p.tokens - t0);  // >= 1: tokens beyond the last repeat it, without storing
  const int first = wave * (16 * NT) + g * 8;  // the lane's first feature of E
  const int chunk_first = wave * 64 + g * 8;         // and of a chunk
  const unsigned char *const act_op = act + m * kPitchA + g * 16, *const hid_op = hid + m * kPitchH + g * 16;

  float one = 1.f;  // (the compiler does not see it: a product with it and a sum are one instruction that takes halfs as they are)
  asm("" : "+s"(one));

  uintx4 w[D][8];
  const int t_row = p.wt && wave * 64 < p.n_out ? wave * 64 : 0;
  // (where nothing follows, the loads ahead go to the matrix at hand once more)
  const Weights tail = p.wt ? weights<4>(p.wt, p.n_out, E, t_row, 0)
                       : PART == kFolded ? weights<4>(p.w2, E, E, 0, 0) : weights<4>(p.w1, p.mlp, E, wave * 64, 0);
  const Weights wo = weights<NT>(p.wo, E, E, wave * (16 * NT), 0);
  if constexpr (PART != kNoAttention)
    issue_first<NT, D>(w, wo);
  else if (p.wt)
    issue_first<4, D>(w, tail);

  // token / inner, of the workgroup's first and of a number below inner + 64 (a product with 2^(31 + l) / inner, l = log2 inner rounded up, which is
  // exact below 2^31; the division takes the scalar unit 150 instructions and a lane 20, with nothing beside them)
  const auto outer_of = [&](long long t) -> long long {
    if (p.inner == 1) return t;
    return p.inner_magic ? (long long)(__umulhi((uint32_t)t, p.inner_magic) >> p.inner_shift) : t / p.inner;
  };
  const auto inner_of = [&](uint32_t r) -> uint32_t {
    if (p.inner == 1) return r;
    return p.inner_magic ? __umulhi(r, p.inner_magic) >> p.inner_shift : r / (uint32_t)p.inner;
  };

#pragma unroll
  for (int i = 0; i < 4 * E; i += 256 * 8) {  // (256 features: 128 threads take a piece each)
    const int at = i + (int)threadIdx.x * 8, which = at / E;
    if (at < 4 * E && (PART != kNoAttention || which >= 2)) {
      const uint16_t *const from = which == 0 ? p.gamma2 : which == 1 ? p.beta2 : which == 2 ? p.gamma_n : p.beta_n;
      const uint32_t none = which & 1 ? 0u : 0x3c003c00u;
      *reinterpret_cast<uintx4 *>(norms + at) = from ? *reinterpret_cast<const uintx4 *>(from + at % E) : uintx4{none, none, none, none};
    }
  }

  // the lane's share of x, fetched once
  half8 x[TT][NT / 2];
  if (p.x_inner == E && p.x_outer == p.inner * E && !p.pos) {
#pragma unroll
    for (int t = 0; t < TT; ++t) load_row<NT>(x[t], p.x + (t0 + min(t * 16 + m, left - 1)) * E + first);
  } else {
    const long long q0 = outer_of(t0);
    const uint32_t r0 = (uint32_t)(t0 - q0 * p.inner);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const uint32_t r = r0 + (uint32_t)min(t * 16 + m, left - 1), q = inner_of(r);
      const long long at = (q0 + q) * p.x_outer + (long long)(r - q * (uint32_t)p.inner) * p.x_inner;
      if (PART == kNoAttention && p.ids) {  // (uniform)
        const long long id = p.wide_ids ? static_cast<const long long *>(p.ids)[at] : static_cast<const int *>(p.ids)[at];
        const bool there = id >= 0 && id < p.vocab;
        load_row<NT>(x[t], p.x + (there ? id : 0) * E + first);
        if (!there) {
          if (p.ids_ok) *p.ids_ok = 0;
#pragma unroll
          for (int j = 0; j < NT / 2; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) x[t][j][i] = (_Float16)__builtin_nanf("");
        }
      } else {
        load_row<NT>(x[t], p.x + at + first);
      }
      if (p.pos) {  // (uniform) fp16(x * scale) + pos, rounded as an activation in between
        half8 at[NT / 2];
        load_row<NT>(at, p.pos + (q0 + q) * E + first);
#pragma unroll
        for (int j = 0; j < NT / 2; ++j) {
#pragma unroll
          for (int i = 0; i < 8; ++i) x[t][j][i] = (_Float16)((float)x[t][j][i] * p.x_scale);
          x[t][j] += at[j];
        }
      }
    }
  }

  floatx4 v[TT][NT];
  if constexpr (PART != kNoAttention) {
    const Weights w1 = PART == kFolded ? Weights() : weights<4>(p.w1, p.mlp, E, wave * 64, 0);
    const Weights w2 = weights<NT>(p.w2, E, PART == kFolded ? E : p.mlp, wave * (16 * NT), 0);
    // (without it w2 twice, at half its scale: a branch around the product costs registers that spill at 512 features)
    const Weights rest = PART == kFolded && p.rest ? weights<NT>(p.rest, E, E, wave * (16 * NT), 0) : w2;
    const float share = p.rest ? 1.f : 0.5f;
    half8 bias[NT / 2], bias2[NT / 2];
    feature_values<NT>(bias, p.bo, first, 0.f);
    if constexpr (PART == kFolded) {
#pragma unroll
      for (int i = 0; i < 2 * E; i += 1024)
        if (i + 4 * (int)threadIdx.x < 2 * E)
          *reinterpret_cast<floatx4 *>(affine + i + 4 * threadIdx.x) = *reinterpret_cast<const floatx4 *>(p.affine + i + 4 * threadIdx.x);
    } else {
      feature_values<NT>(bias2, p.b2, first, 0.f);
    }
    constexpr int kPieces = E / 8, kRows = 256 / kPieces;
    const int piece = threadIdx.x % kPieces, row0 = threadIdx.x / kPieces;
#pragma unroll
    for (int r = 0; r < TM; r += kRows)
      *reinterpret_cast<uintx4 *>(act + (r + row0) * kPitchA + piece * 16) =
          *reinterpret_cast<const uintx4 *>(p.attn + (t0 + min(r + row0, left - 1)) * E + piece * 8);
    lds_barrier();
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[t][j][i] = __builtin_fmaf(value(bias, j, i), one, value(x[t], j, i));
    // (or the compiler keeps the widened values for the second use, at twice the registers)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < NT / 2; ++j) asm("" : "+v"(x[t][j]));
    gemm<TT, NT, E, kPitchA, PART == kFolded ? NT : 4, D>(v, act_op, wo, PART == kFolded ? rest : w1, w);
    float s[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      s[t] = 0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j) s[t] += (v[t][j][0] + v[t][j][1]) + (v[t][j][2] + v[t][j][3]);
    }
    layer_norm<TT, NT, E>(v, s, norms, p.eps2, first, part, wave, lane);
    // (every wave is past its product: the sums' barrier lies in between)
#pragma unroll
    for (int t = 0; t < TT; ++t) put_row<NT>(act + (t * 16 + m) * kPitchA + first * 2, v[t]);
    lds_barrier();
    if constexpr (PART == kFolded) {
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int j = 0; j < NT; ++j) v[t][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      gemm<TT, NT, E, kPitchA, NT, D>(v, act_op, rest, w2, w);
      gemm<TT, NT, E, kPitchA, 4, D>(v, act_op, w2, tail, w);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int f = first + 32 * (j >> 1) + 4 * (j & 1);
        const floatx4 scale = *reinterpret_cast<const floatx4 *>(affine + f) * share, shift = *reinterpret_cast<const floatx4 *>(affine + E + f);
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) v[t][j][i] = __builtin_fmaf(v[t][j][i], scale[i], __builtin_fmaf(value(x[t], j, i), one, shift[i]));
      }
    } else {
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) v[t][j][i] = __builtin_fmaf(value(bias2, j, i), one, value(x[t], j, i));
      for (int c = 0; c < p.mlp; c += kChunk) {
        floatx4 h[TT][4];
        half8 bias1[2];
        feature_values<4>(bias1, p.b1, c + chunk_first, 0.f);
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int j = 0; j < 4; ++j) h[t][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        Weights up = w1, down = w2, then = tail;
        up.base += (uint32_t)c * (E * 2u);
        down.base += (uint32_t)(c / Unit<NT>::K) * Unit<NT>::kBytes;
        if (c + kChunk < p.mlp) {
          then = up;
          then.base += kChunk * (E * 2u);
        }
        gemm<TT, 4, E, kPitchA, NT, D>(h, act_op, up, down, w);
        lds_barrier();  // the previous chunk has been read
#pragma unroll
        for (int t = 0; t < TT; ++t) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) h[t][j][i] += value(bias1, j, i);
          put_row<4>(hid + (t * 16 + m) * kPitchH + chunk_first * 2, h[t]);
        }
        lds_barrier();
        gemm<TT, NT, kChunk, kPitchH, 4, D>(v, hid_op, down, then, w);
      }
    }
  } else {
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[t][j][i] = value(x[t], j, i);
  }
  // x' as it is stored is what its LayerNorm reads
  float s[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    s[t] = 0.f;
#pragma unroll
    for (int j = 0; j < NT; j += 2) {
      half8 h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        h[i] = (_Float16)v[t][j][i];
        h[4 + i] = (_Float16)v[t][j + 1][i];
      }
      if (p.x_out && t * 16 + m < left) *reinterpret_cast<half8 *>(p.x_out + (t0 + t * 16 + m) * E + first + j * 16) = h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[t][j][i] = (float)h[i];
        v[t][j + 1][i] = (float)h[4 + i];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) s[t] = __builtin_fmaf((float)h[i], one, s[t]);
    }
  }

  layer_norm<TT, NT, E>(v, s, norms + 2 * E, p.eps_n, first, part, wave, lane);
  if (!p.wt) {
#pragma unroll
    for (int t = 0; t < TT; ++t)
      if (t * 16 + m < left) put_row<NT>(reinterpret_cast<unsigned char *>(p.norm_out + (t0 + t * 16 + m) * E + first), v[t]);
    return;
  }
#pragma unroll
  for (int t = 0; t < TT; ++t) put_row<NT>(act + (t * 16 + m) * kPitchA + first * 2, v[t]);
  lds_barrier();
  Weights cur = tail;
  const long long outer = p.outer, q0 = p.head_dim ? outer_of(t0) : 0;
  const uint32_t r0 = (uint32_t)(t0 - q0 * p.inner);
  const int head_shift = p.head_dim ? __builtin_ctz((unsigned)p.head_dim) : 0;
  for (int c = wave * 64; c < p.n_out; c += kChunk) {  // (no barrier from here on)
    floatx4 o[TT][4];
    half8 bias[2];
    feature_values<4>(bias, p.bt, c + g * 8, 0.f);
    uint32_t r_first = r0;
    asm volatile("" : "+s"(r_first));  // (the rows' places are made anew for every chunk: kept, they cost registers that spill)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) o[t][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    Weights then = cur;
    if (c + kChunk < p.n_out) then.base += kChunk * (E * 2u);
    gemm<TT, 4, E, kPitchA, 4, D>(o, act_op, cur, then, w);
    cur = then;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[t][j][i] += value(bias, j, i);
      if (t * 16 + m < left) {
        if (p.head_dim == 0) {
          put_row<4>(reinterpret_cast<unsigned char *>(p.out + (t0 + t * 16 + m) * p.n_out + c + g * 8), o[t]);
        } else {  // (a head is at least as wide as the 32 features of two tiles)
          const uint32_t r = r_first + (uint32_t)(t * 16 + m), i = inner_of(r);  // token (q0 + i, r - i * inner)
          uint16_t *const row = p.out + (r - i * (uint32_t)p.inner) * (E * outer) + (q0 + i) * p.head_dim + g * 8;
#pragma unroll
          for (int j = 0; j < 4; j += 2) {
            const int f = c + 16 * j, in_part = f % E;
            const floatx4 pair[2] = {o[t][j], o[t][j + 1]};
            put_row<2>(reinterpret_cast<unsigned char *>(row + (f / E) * (p.inner * outer * E) + (in_part >> head_shift) * (outer * p.head_dim) +
                                                         (in_part & (p.head_dim - 1))),
                       pair);
          }
        }
      }
    }
  }
}

// Up to BlockPackArgs::kMost matrices into the order in which the waves above load them: groups of 16 * NJ rows, in each units of
// K columns, in each a 1 KB piece per step of 32 columns and tile, in that the 16 bytes of every lane.
__device__ __forceinline__ void pack_piece(const BlockPackArgs &p, uint32_t block, uint32_t threads) {
  int i = 0;
  while (i + 1 < p.count && block >= p.m[i + 1].first_block) ++i;
  const BlockPackArgs::Matrix &a = p.m[i];
  const uint32_t at = (block - a.first_block) * threads + threadIdx.x;  // 16-byte piece of the packed matrix
  const uint32_t cols = a.cols, nj = a.group / 16u, ku = nj == 8 ? 32u : 64u;
  if (at >= (uint32_t)a.rows * (cols / 8u)) return;
  const uint32_t lane = at & 63u, m = lane & 15u, g = lane >> 4, frag = at >> 6;
  const uint32_t per_unit = nj * ku / 32u, in_unit = frag % per_unit, unit = frag / per_unit;
  const uint32_t units = cols / ku, group = unit / units;
  const uint32_t row = group * a.group + 32u * (in_unit % nj / 2u) + 8u * (m >> 2) + 4u * (in_unit & 1u) + (m & 3u);
  const uint32_t k = (unit % units) * ku + (in_unit / nj) * 32u + 8u * g;
  reinterpret_cast<uintx4 *>(a.dst)[at] = *reinterpret_cast<const uintx4 *>(a.src + (size_t)row * cols + k);
}

__global__ __launch_bounds__(256) void block_pack_kernel(const BlockPackArgs p) { pack_piece(p, blockIdx.x, 256); }

// Sixteen rows of W2 W1, and of W2 b1 + b2.  Sixteen waves: E / 64 of them take 64 columns each, and as many groups of them as that
// leaves a share of the hidden features each; the shares are added up in LDS in their order.  A wave's 32 rows of W1 pass through an
// LDS stage of its own, whose transpose reads make the operand (32 hidden features x 16 columns); W2's rows are the operand as they lie.
// A row is scaled by a power of two before it is rounded to fp16, which needs its largest element: a workgroup therefore makes whole rows
// and streams all of W1 through one CU, 512 KB for 256 x 1024: 5 of the 12.5 us at 64 bytes a cycle, some 3 for the sums and 2 to start.
// Four steps of loads ahead instead of two are level (12.7), loads without a condition, the last ones repeated, slower (13.5).
constexpr uint32_t kFoldPitch = 160;
template <int E>
__device__ void fold_rows(const BlockFoldArgs::Pair &a, int row0, unsigned char *lds) {
  constexpr int CG = E / 64, KS = 16 / CG, DEPTH = 2, PER = E / 64;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), m = lane & 15, g = lane >> 4;
  const int cg = wave % CG, ks = wave / CG, share = a.mlp / KS;
  const uint16_t *const left = a.w2 + (size_t)(row0 + m) * a.mlp + ks * share + 8 * g;
  const uint16_t *const right = a.w1 + (size_t)(ks * share + (lane >> 3)) * E + cg * 64 + (lane & 7) * 8;
  unsigned char *const stage = lds + wave * (32 * kFoldPitch);
  unsigned char *const dst = stage + (lane >> 3) * kFoldPitch + (lane & 7) * 16;
  const unsigned char *const src = stage + (8 * g + (m >> 2)) * kFoldPitch + (m & 3) * 8;
  uintx4 l[DEPTH], r[DEPTH][4];
  const auto fetch = [&](int d, int k) {
    l[d] = *reinterpret_cast<const uintx4 *>(left + k);
#pragma unroll
    for (int i = 0; i < 4; ++i) r[d][i] = *reinterpret_cast<const uintx4 *>(right + (size_t)(k + 8 * i) * E);
  };
  floatx4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (32 * d < share) fetch(d, 32 * d);
  for (int k = 0; k < share; k += 32 * DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int at = k + 32 * d;
      if (32 * DEPTH > 256 / KS && at >= share) continue;  // (uniform; a share is a multiple of 256 / KS)
      // (LDS operations of a wave execute in order: these writes land behind the previous step's reads)
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<uintx4 *>(dst + 8 * i * kFoldPitch) = r[d][i];
      const half8 w = __builtin_bit_cast(half8, l[d]);
      if (at + 32 * DEPTH < share) fetch(d, at + 32 * DEPTH);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const two_words lo = lds_read_tr(src + 32 * t), hi = lds_read_tr(src + 4 * kFoldPitch + 32 * t);
        const uintx4 b = {lo[0], lo[1], hi[0], hi[1]};
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, __builtin_bit_cast(half8, b), acc[t], 0, 0, 0);
      }
    }
  }
  const int row = row0 + wave;
  const uint16_t *const w2 = a.w2 + (size_t)row * a.mlp;
  float shift = 0.f;
  if (a.b1)
    for (int k = lane * 8; k < a.mlp; k += 512) {
      const half8 w = *reinterpret_cast<const half8 *>(w2 + k), b = *reinterpret_cast<const half8 *>(a.b1 + k);
#pragma unroll
      for (int i = 0; i < 8; ++i) shift += (float)w[i] * (float)b[i];
    }
  shift = wave_sum_all(shift);
  __syncthreads();
  constexpr int kSums = E + 16;  // (the four rows a store touches at different banks)
  float *const sums = reinterpret_cast<float *>(lds);  // [KS][16][kSums]
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[(ks * 16 + 4 * g + i) * kSums + cg * 64 + 16 * t + m] = acc[t][i];
  __syncthreads();
  // a wave per row, PER columns per lane
  float c[PER], most = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    c[i] = 0.f;
#pragma unroll
    for (int q = 0; q < KS; ++q) c[i] += sums[(q * 16 + wave) * kSums + lane * PER + i];
    most = fmaxf(most, fabsf(c[i]));
  }
  most = wave_max_all(most);
  // (a row of zeros, and one with an infinity or a NaN, as they are)
  const int up = most > 0.f && most < INFINITY ? min(max(13 - (int)((__float_as_uint(most) >> 23) - 127u), -100), 100) : 0;
  const float factor = __uint_as_float((uint32_t)(127 + up) << 23);
  if (lane == 0) {
    a.affine[row] = __uint_as_float((uint32_t)(127 - up) << 23);
    a.affine[E + row] = shift + (a.b2 ? (float)*reinterpret_cast<const _Float16 *>(a.b2 + row) : 0.f);
  }
  // where block_pack_kernel puts element (row, k)
  constexpr uint32_t kGroup = E / 4, NJ = kGroup / 16, KU = NJ == 8 ? 32 : 64;
  const uint32_t in_group = (uint32_t)row % kGroup, k = (uint32_t)lane * PER;
  const uint32_t tile = in_group / 32u * 2u + ((in_group >> 2) & 1u), mm = ((in_group >> 3) & 3u) * 4u + (in_group & 3u);
  const uint32_t piece = ((uint32_t)row / kGroup * (E / KU) + k / KU) * (NJ * KU / 32u) + (k % KU) / 32u * NJ + tile;
  _Float16 *const out = reinterpret_cast<_Float16 *>(a.dst) + piece * 512u + ((k % 32u) / 8u * 16u + mm) * 8u + k % 8u;
  typedef _Float16 halves __attribute__((ext_vector_type(PER)));
  halves h, rest;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    h[i] = (_Float16)(c[i] * factor);
    const float left = c[i] * factor - (float)h[i];  // (exact; of an infinity or a NaN nothing is left)
    rest[i] = fabsf(left) < INFINITY ? (_Float16)left : (_Float16)0;
  }
  *reinterpret_cast<halves *>(out) = h;
  if (a.rest) *reinterpret_cast<halves *>(reinterpret_cast<_Float16 *>(a.rest) + (out - reinterpret_cast<_Float16 *>(a.dst))) = rest;
}

template <int E>
__global__ __launch_bounds__(1024) void block_prepare_kernel(const BlockFoldArgs f, const BlockPackArgs p) {
  __shared__ __align__(16) unsigned char lds[16 * 32 * kFoldPitch];
  const uint32_t folds = (uint32_t)f.count * (E / 16);
  if (f.ids_ok && blockIdx.x == 0 && threadIdx.x == 0) *f.ids_ok = 1;
  if (blockIdx.x < folds) {
    // (workgroups eight apart share an XCD: one pair's on as few of them as can be, each of which fetches W1 once)
    const uint32_t id = (blockIdx.x & 7u) * (folds / 8u) + (blockIdx.x >> 3);
    fold_rows<E>(f.m[id / (E / 16)], (int)(id % (E / 16)) * 16, lds);
  } else {
    pack_piece(p, blockIdx.x - folds, 1024);
  }
}

template <int E, int TM>
hipError_t launch(const BlockDenseArgs &p, hipStream_t stream) {
  const long long blocks = (p.tokens + TM - 1) / TM;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  if (!p.attn)
    hipLaunchKernelGGL((block_dense_kernel<E, TM, kNoAttention>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
  else if (p.affine)
    hipLaunchKernelGGL((block_dense_kernel<E, TM, kFolded>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((block_dense_kernel<E, TM, kTwoLayers>), dim3((unsigned)blocks), dim3(256), 0, stream, p);
  return hipGetLastError();
}

// 64 tokens per workgroup, two workgroups per CU (where the registers of 512 features allow one): one's LayerNorms and LDS
// passes run under the other's products.  32768 tokens of 256 features: 58 us, with one workgroup per CU 69, with one of
// 128 tokens 64; of 128 features 32, 39 and 35.  Up to 8192 tokens those are at most 128 workgroups, and 32 tokens give every
// CU one: 8192 tokens of 128, 256, 512 features 15, 26, 56 us against 18, 30, 73; 10000 tokens 25, 43, 101 against 18, 31, 73.
// Up to 4096 tokens 16 do the same, and a workgroup's chain of products and LayerNorms is shorter: 2048 tokens 10.0, 17.5, 43 us
// against 12.3, 20.1, 48 with 32 (without attention 4.6, 7.4, 17 against 5.6, 9.2, 20), 4096 tokens 10.9, 19.3, 46 against 12.6, 21.2,
// 49; 8192 tokens without attention 7.6, 14.2, 36 against 6.6, 11.1, 25.  (Both linear layers, LayerNorms of two exchanges.)  Folded, replayed,
// 16 / 32 / 64 tokens, 128 features: 4096 tokens 6.7 / 7.6 / 10.3, 8192 9.1 / 8.3 / 10.8, 10000 12.6 / 13.7 / 11.2, 32768 28.5 / 27.3 / 17.3; 256: 12.7 / 13.8 / 18.6,
// 20.1 / 15.7 / 19.8, 27.7 / 25.5 / 20.3, 68 / 53 / 37.3; 512: 36.6 / 37.2 / 47.5, 65.6 / 43.0 / 48.9, 91.8 / 74.0 / 50.0, 243 / 157 / 115.
template <int E>
hipError_t launch_for_width(const BlockDenseArgs &p, hipStream_t stream) {
  if (p.tokens <= 256 * 16) return launch<E, 16>(p, stream);
  return p.tokens <= 256 * 32 ? launch<E, 32>(p, stream) : launch<E, 64>(p, stream);
}

}  // namespace

bool block_dense_applies(int E, int mlp, int n_out) {
  // (a weight matrix is addressed with 32-bit byte offsets)
  return (E == 128 || E == 256 || E == 512) && mlp > 0 && mlp % kChunk == 0 && mlp <= (1 << 20) && n_out >= 0 && n_out % 64 == 0 &&
         n_out <= (1 << 20);
}

hipError_t launch_block_pack(const BlockPackArgs &p, uint32_t blocks, hipStream_t stream) {
  hipLaunchKernelGGL(block_pack_kernel, dim3(blocks), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_block_prepare(int E, const BlockFoldArgs &folds, const BlockPackArgs &packs, uint32_t pack_blocks, hipStream_t stream) {
  const dim3 grid((uint32_t)folds.count * (uint32_t)(E / 16) + pack_blocks);
  if (grid.x == 0) return hipSuccess;
  switch (E) {
    case 128: hipLaunchKernelGGL(block_prepare_kernel<128>, grid, dim3(1024), 0, stream, folds, packs); break;
    case 256: hipLaunchKernelGGL(block_prepare_kernel<256>, grid, dim3(1024), 0, stream, folds, packs); break;
    case 512: hipLaunchKernelGGL(block_prepare_kernel<512>, grid, dim3(1024), 0, stream, folds, packs); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_block_dense(int E, const BlockDenseArgs &args, hipStream_t stream) {
  BlockDenseArgs p = args;
  p.outer = p.tokens / p.inner;
  p.inner_magic = 0;
  p.inner_shift = 0;
  if (p.inner > 1 && p.tokens < (1ll << 31) && p.inner < (1ll << 31) - 64) {
    int l = 1;
    while ((1ll << l) < p.inner) ++l;
    p.inner_magic = (uint32_t)((1ull << (31 + l)) / (unsigned long long)p.inner + 1u);
    p.inner_shift = l - 1;
  }
  switch (E) {
    case 128: return launch_for_width<128>(p, stream);
    case 256: return launch_for_width<256>(p, stream);
    case 512: return launch_for_width<512>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace sspmm
