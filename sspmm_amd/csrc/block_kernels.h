// Launch interface of the dense part of a sparse attention block on token-major activations.
#ifndef SSPMM_AMD_BLOCK_KERNELS_H
#define SSPMM_AMD_BLOCK_KERNELS_H

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace sspmm {

// Everything between one block's attention and the next one's, for rows (tokens) of E features:
//   s  = attn Wo^T + bo + x            n = LayerNorm2(s)
//   x' = (n W1^T + b1) W2^T + b2 + x   h = LayerNormN(x')
// and from h either h itself (norm_out) or out = h Wt^T + bt.  Without attn: x' = x.  The weights are packed: wo and w2 in
// groups of E / 4 rows, w1 and wt of 64.  Row i of x is at x + (i / inner) * x_outer + (i % inner) * x_inner
// elements; the other activations are dense.  16-byte aligned pointers, x strides multiples of 8.
struct BlockDenseArgs {
  long long tokens, inner;
  const uint16_t *x;
  long long x_outer, x_inner;
  const uint16_t *pos;                       // nullable: x is an embedding, fp16(x * x_scale) + pos[token / inner] in its place
  float x_scale;
  const uint16_t *attn;                      // nullable, and the next two lines with it
  const uint16_t *wo, *bo, *gamma2, *beta2;
  const uint16_t *w1, *b1, *w2, *b2;
  const uint16_t *gamma_n, *beta_n;
  const uint16_t *wt, *bt;                   // nullable: norm_out in their place
  float eps2, eps_n;
  int mlp, n_out;
  int head_dim;                              // out as [n_out / E, inner, E / head_dim, tokens / inner, head_dim]; 0: as [tokens, n_out]
  uint16_t *x_out;                           // nullable: x' is not needed
  uint16_t *norm_out, *out;
};

// Weight matrices [out features, in features] as torch.nn.Linear keeps them, in the order in which block_dense loads them.
struct BlockPackArgs {
  static constexpr int kMost = 48;
  struct Matrix {
    const uint16_t *src;
    uint16_t *dst;
    int rows, cols, group;  // group = 32, 64 or 128; rows a multiple of it, cols of 64
    uint32_t first_block;   // of 256 16-byte pieces each
  } m[kMost];
  int count;
};
hipError_t launch_block_pack(const BlockPackArgs &args, uint32_t blocks, hipStream_t stream);

// E = 128, 256 or 512, mlp a multiple of 256, n_out a multiple of 64.
bool block_dense_applies(int E, int mlp, int n_out);
hipError_t launch_block_dense(int E, const BlockDenseArgs &args, hipStream_t stream);

}  // namespace sspmm
#endif
