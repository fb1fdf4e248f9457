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
  const void *ids;                           // nullable (without attn, with pos): row i of x is row ids[(i / inner) * x_outer + (i % inner) * x_inner]
  int wide_ids;                              // of `vocab` rows at x, NaN where there is none; int64 instead of int32
  long long vocab;
  int *ids_ok;                               // nullable: becomes 0 where there is no such row
  const uint16_t *attn;                      // nullable, and the next two lines with it
  const uint16_t *wo, *bo, *gamma2, *beta2;
  const uint16_t *w1, *b1, *w2, *b2;
  const uint16_t *gamma_n, *beta_n;
  const uint16_t *wt, *bt;                   // nullable: norm_out in their place
  float eps2, eps_n;
  int mlp, n_out;
  const float *affine;                       // nullable: w2 is the product W2 W1 of E x E, see launch_block_prepare; [2][E]: what undoes a row's
                                             // scaling, and W2 b1 + b2; w1, b1, b2 and mlp are not looked at
  const uint16_t *rest;                      // nullable, with affine: what the rounding of w2's rows left
  int head_dim;                              // out as [n_out / E, inner, E / head_dim, tokens / inner, head_dim]; 0: as [tokens, n_out]
  uint16_t *x_out;                           // nullable: x' is not needed
  uint16_t *norm_out, *out;
  long long outer;                           // (these three by launch_block_dense) tokens / inner
  uint32_t inner_magic;                      // 0: a division
  int inner_shift;
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

// The same, first_block counting 1024 pieces each, and with it the products of pairs of linear layers with nothing between them:
// n -> (n W1^T + b1) W2^T + b2 as one matrix [E, E], packed in groups of E / 4 rows, row o times 2^s(o) (its largest element then is
// between 2^13 and 2^14, so that fp16 keeps what fp32 sums give whatever the weights' size), what that rounding to fp16 leaves as a second
// matrix, rounded to fp16 in turn, packed and scaled alike, and affine = [2][E]: 2^-s and W2 b1 + b2.
struct BlockFoldArgs {
  static constexpr int kMost = 16;
  struct Pair {
    const uint16_t *w1, *b1, *w2, *b2;  // W1 [mlp, E], W2 [E, mlp]; b1 and b2 nullable
    uint16_t *dst, *rest;               // rest nullable
    float *affine;
    int mlp;                            // a multiple of 256
  } m[kMost];
  int count;
  int *ids_ok;                          // nullable: set to 1, for BlockDenseArgs::ids_ok of a launch behind this one
};
hipError_t launch_block_prepare(int E, const BlockFoldArgs &folds, const BlockPackArgs &packs, uint32_t pack_blocks, hipStream_t stream);

// E = 128, 256 or 512, mlp a multiple of 256, n_out a multiple of 64.
bool block_dense_applies(int E, int mlp, int n_out);
hipError_t launch_block_dense(int E, const BlockDenseArgs &args, hipStream_t stream);

}  // namespace sspmm
#endif
