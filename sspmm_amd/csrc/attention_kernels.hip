// The two steps either side of the batched SpMM in a sparse attention block, in the same
// vector-sparse format, for gfx950 (wave64, MFMA 16x16x32 f16).
//
//   sddmm:   out[j*V + v] = lhs[i*V + v, :] . rhs[col_j, :]   for the vectors j of vector-row i
//            (reference end2end/sspmm_e2e/src/cuda/sddmm_kernel.cu:1161-1295: `sddmm`, `bsddmm`);
//   softmax: per dense row, over its stored entries, exp(x*scaler - max) / sum
//            (reference end2end/sspmm_e2e/src/cuda/softmax_kernel.cu:95-290: `csr_softmax`, `bcsr_softmax`).
//
// Both are bound by memory traffic: the sddmm by the gathers of rows of rhs (F*2 bytes per stored
// vector) and the writes of the values, the softmax by one read and one write of the values.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attention_kernels.h"
#include "lane_ops.h"

namespace sspmm {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));

static constexpr uint32_t kSrdWord3 = 0x00020000u;  // 32-bit raw (untyped) buffer, gfx9 family

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_srd(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, (int)kSrdWord3);
}

// Linear block ids are dealt round-robin to the 8 XCDs by the hardware; each XCD gets one
// contiguous range of the work list so that neighbouring work shares an L2.
__device__ __forceinline__ uint32_t xcd_work_index(uint32_t per_xcd) {
  const uint32_t id = blockIdx.x;
  return (id & 7u) * per_xcd + (id >> 3);
}

}  // namespace

// ------------------------------------------------------------------------------------ sddmm
// One wave per (vector-row, batch element).  The V rows of lhs are the MFMA's first operand and
// stay in registers (lane (m, g) holds features 32c + 8g .. + 7 of row m, c = 0 .. NC-1).  Per
// group of 16 stored vectors the 16 rows of rhs they name are needed in the same layout, lane
// (m, g) holding features 32c + 8g .. of the row of vector m.  Loaded that way, neighbouring
// lanes would read 16 bytes each of sixteen different rows; instead the rows are fetched with
// neighbouring lanes on neighbouring 16-byte pieces of one row (whole 128-byte lines for 64
// features), written to a small LDS stage, and read back in the operand layout.  Rows of the
// stage are padded by 16 bytes (the reads still meet in some banks: a quarter of the LDS cycles at 64 features and 2000 keys).
// NC MFMAs contract the features, and the lane ends up with rows 4g .. 4g+3 of vector m: eight
// contiguous bytes of the output.  The column indices run two groups ahead of the arithmetic, the
// rows of rhs one group (two stages, used alternately).
// WHOLE: F = 32 * NC exactly, no piece to test for: vector instructions are what the kernel waits for (2000 keys, 16 heads,
// 64 features 11.3 -> 10.7 us, 128: 17.5 -> 16.2; 4096 keys, 48 heads, 64: 79.6 -> 76.2; 16 heads, 256: 109 -> 96).  Two groups
// of vectors per step, with twice the rows in flight, measured 3 to 8 % slower.
template <int V, int NC, bool WHOLE, bool SHARED>
__global__ __launch_bounds__(64) void sddmm_kernel(const SddmmArgs p) {
  constexpr uint32_t kStageRow = NC * 64u + 16u;  // bytes: room for 32 * NC features, and the padding
  __shared__ __align__(16) unsigned char stage[2][16 * kStageRow];
  const uint32_t w = xcd_work_index(p.per_xcd);
  if (w >= p.total_work) return;
  const uint32_t r = w % (uint32_t)p.m_vec;
  const uint32_t batch = w / (uint32_t)p.m_vec;
  const int row = p.row_indices ? p.row_indices[r] : (int)r;
  const int beg = p.row_offsets[row], end = p.row_offsets[row + 1];
  if (beg == end) return;

  const int lane = threadIdx.x, m = lane & 15, g = lane >> 4;
  const uint32_t F = WHOLE ? 32u * NC : (uint32_t)p.F;
  const uint16_t *lhs = p.lhs + (int64_t)batch * p.stride_lhs + (int64_t)row * V * F;
  const __amdgpu_buffer_rsrc_t srd_lhs = make_srd(lhs, (uint32_t)V * F * 2u);
  const uint32_t rhs_bytes = (uint32_t)p.n_rhs * F * 2u;
  const __amdgpu_buffer_rsrc_t srd_rhs = make_srd(p.rhs + (int64_t)batch * p.stride_rhs, rhs_bytes);
  const __amdgpu_buffer_rsrc_t srd_cols = make_srd(p.col_idx, (uint32_t)end * 4u);  // past the row: reads 0
  uint16_t *out = p.out + (int64_t)batch * p.stride_out;

  // operand side: feature offsets of this lane's 16-byte pieces; pieces past F (or rows past V) are zeros
  uint32_t op_off[NC];
  bool op_ok[NC];
  half8 a[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const uint32_t f0 = 32u * c + 8u * g;
    op_ok[c] = WHOLE || f0 < F;
    op_off[c] = (uint32_t)m * kStageRow + f0 * 2u;
    const uint32_t off = (m < V && op_ok[c]) ? ((uint32_t)m * F + f0) * 2u : 0xfffffff0u;
    a[c] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(srd_lhs, off, 0, 0));
  }
  // fetch side: piece lane + 64 i of the group's 16 * F / 8 pieces, row-major (piece = 8 features of one row)
  const uint32_t chunks = F / 8u;
  uint32_t ld_row[NC], ld_src[NC], ld_dst[NC];
  bool ld_ok[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const uint32_t piece = (uint32_t)lane + 64u * i;
    ld_row[i] = piece / chunks;
    const uint32_t ch = piece - ld_row[i] * chunks;
    ld_ok[i] = WHOLE || ld_row[i] < 16u;
    ld_src[i] = ch * 16u;
    ld_dst[i] = ld_row[i] * kStageRow + ch * 16u;
  }

  struct Cols {
    uint32_t c[NC];
  };
  struct Pieces {
    uintx4 d[NC];
  };
  // Column indices: one load of 4 bytes a lane per load of rows, the lanes of a row asking for the same index (five cycles of the address unit),
  // or, SHARED, blocks of 64 of them (four groups), one per lane, a block ahead, out of which the lanes pick theirs with a lane permute.  16 heads of
  // 2000 keys, 64 features 10.54 (blocks) / 10.04 us, 512 keys, 8 heads 3.29 / 3.16, 128 features, 2048 keys, 16 heads 15.7 / 15.4, 256 features
  // 30.3 / 28.2; but of 64 features with more waves than are resident at once the address unit is what they wait for: 2048 keys, 48 heads, V = 16
  // 16.2 / 16.6, 4096 keys, 48 heads 77.0 / 78.4 (32 features 18.7 / 18.1, 128 28.2 / 27.7).
  int blk_base = beg;
  uint32_t blk0 = 0, blk1 = 0;
  if constexpr (SHARED) {
    blk0 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(srd_cols, (beg + lane) * 4, 0, 0);
    blk1 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(srd_cols, (beg + 64 + lane) * 4, 0, 0);
  }
  auto load_cols = [&](int kc) {  // (called with kc rising by 16 from beg)
    if (SHARED && kc - blk_base >= 64) {
      blk_base += 64;
      blk0 = blk1;
      blk1 = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(srd_cols, (blk_base + 64 + lane) * 4, 0, 0);
    }
    Cols x;
#pragma unroll
    for (int i = 0; i < NC; ++i)
      x.c[i] = SHARED ? (uint32_t)__builtin_amdgcn_ds_bpermute((kc - blk_base + (int)ld_row[i]) * 4, (int)blk0)
                      : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(srd_cols, (kc + (int)ld_row[i]) * 4, 0, 0);
    return x;
  };
  auto load_rows = [&](Pieces &b, const Cols &x) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const uint32_t off = ld_ok[i] ? __umul24(x.c[i], F * 2u) + ld_src[i] : 0xfffffff0u;
      b.d[i] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(srd_rhs, off, 0, 0));
    }
  };
  auto to_stage = [&](const Pieces &b, unsigned char *st) {
#pragma unroll
    for (int i = 0; i < NC; ++i)
      if (ld_ok[i]) *reinterpret_cast<uintx4 *>(st + ld_dst[i]) = b.d[i];
  };
  // the group's 16 x V products: lane (m, g) gets rows 4g .. 4g+3 of stored vector kc + m, as four halfs
  auto products = [&](const unsigned char *st) {
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      half8 b = {0, 0, 0, 0, 0, 0, 0, 0};
      if (op_ok[c]) b = *reinterpret_cast<const half8 *>(st + op_off[c]);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c], b, acc, 0, 0, 0);
    }
    const half4 h = {(_Float16)acc[0], (_Float16)acc[1], (_Float16)acc[2], (_Float16)acc[3]};  // round to nearest even
    return __builtin_bit_cast(uintx2, h);
  };
  auto store_group = [&](uintx2 h, int kc) {
    if (kc + m < end && 4 * g < V) *reinterpret_cast<uintx2 *>(out + ((int64_t)(kc + m) * V + 4 * g)) = h;
  };
  // Two groups in one store instruction (a store costs the address unit the same sixteen cycles whether its lanes
  // carry 8 or 16 bytes, and this kernel is bound by that unit): the lane groups g and g + 1 exchange halves, so
  // that g even holds rows 8 (g / 2) .. + 7 of vector kc + m and g odd those of vector kc + 16 + m.
  auto store_two_groups = [&](uintx2 first, uintx2 second, int kc) {
    const auto w0 = __builtin_amdgcn_permlane16_swap(first[0], second[0], false, false);
    const auto w1 = __builtin_amdgcn_permlane16_swap(first[1], second[1], false, false);
    const uintx4 v = {(uint32_t)w0[0], (uint32_t)w1[0], (uint32_t)w0[1], (uint32_t)w1[1]};
    const int vec = kc + m + 16 * (g & 1);
    if (vec < end && 8 * (g >> 1) < V) *reinterpret_cast<uintx4 *>(out + ((int64_t)vec * V + 8 * (g >> 1))) = v;
  };
  const bool pair_stores = p.pair_stores != 0;

  // The LDS operations of a wave execute in order, so a stage can be rewritten right after the reads of the group
  // that used it have been issued; no barrier is involved (one wave per workgroup).
  Pieces b0, b1;
  const Cols c_first = load_cols(beg);
  Cols c_next = load_cols(beg + 16);
  load_rows(b0, c_first);
  to_stage(b0, stage[0]);
  int kc = beg;
  for (;;) {
    // stage[0] holds group kc; c_next the columns of group kc + 16
    if (kc + 16 >= end) {
      store_group(products(stage[0]), kc);
      break;
    }
    Cols c_after = load_cols(kc + 32);
    load_rows(b1, c_next);
    const uintx2 first = products(stage[0]);
    if (!pair_stores) store_group(first, kc);
    to_stage(b1, stage[1]);
    kc += 16;
    if (kc + 16 >= end) {
      const uintx2 second = products(stage[1]);
      if (pair_stores) store_two_groups(first, second, kc - 16);
      else store_group(second, kc);
      break;
    }
    c_next = load_cols(kc + 32);
    load_rows(b0, c_after);
    const uintx2 second = products(stage[1]);
    if (pair_stores) store_two_groups(first, second, kc - 16);
    else store_group(second, kc);
    to_stage(b0, stage[0]);
    kc += 16;
  }
}

template <int V, int NC>
static hipError_t launch_sddmm_nc(const SddmmArgs &a, hipStream_t stream) {
  SddmmArgs p = a;
  p.pair_stores = reinterpret_cast<uintptr_t>(a.out) % 16 == 0 && a.stride_out % 8 == 0;
  p.total_work = (uint32_t)a.m_vec * (uint32_t)a.batch;
  p.per_xcd = (p.total_work + 7u) / 8u;
  if (p.total_work == 0) return hipSuccess;
  if (a.F == 32 * NC)
    // (8192 waves: 32 for every CU; 32 heads of 2048 keys, V = 8, are level)
    if (NC == 2 && p.total_work > 8192u)
      hipLaunchKernelGGL((sddmm_kernel<V, NC, true, NC == 2>), dim3(p.per_xcd * 8u), dim3(64), 0, stream, p);
    else
      hipLaunchKernelGGL((sddmm_kernel<V, NC, true, false>), dim3(p.per_xcd * 8u), dim3(64), 0, stream, p);
  else
    hipLaunchKernelGGL((sddmm_kernel<V, NC, false, false>), dim3(p.per_xcd * 8u), dim3(64), 0, stream, p);
  return hipGetLastError();
}

template <int V>
static hipError_t launch_sddmm_v(const SddmmArgs &a, hipStream_t stream) {
  const int nc = (a.F + 31) / 32;
  if (nc <= 1) return launch_sddmm_nc<V, 1>(a, stream);
  if (nc <= 2) return launch_sddmm_nc<V, 2>(a, stream);
  if (nc <= 4) return launch_sddmm_nc<V, 4>(a, stream);
  return launch_sddmm_nc<V, 8>(a, stream);
}

hipError_t launch_sddmm(const SddmmArgs &a, int V, hipStream_t stream) {
  return V == 8 ? launch_sddmm_v<8>(a, stream) : launch_sddmm_v<16>(a, stream);
}

// ---------------------------------------------------------------------------------- softmax
namespace {

__device__ __forceinline__ float wave_max(float x) { return wave_max_all(x); }
__device__ __forceinline__ float wave_sum(float x) { return wave_sum_all(x); }

// The V halfs of one stored vector as packed words.
template <int V>
struct Halfs {
  half8 h[V / 8];
  static __device__ __forceinline__ Halfs load(const uint16_t *p) {
    Halfs x;
#pragma unroll
    for (int i = 0; i < V / 8; ++i) x.h[i] = *reinterpret_cast<const half8 *>(p + 8 * i);
    return x;
  }
  static __device__ __forceinline__ Halfs all(float v) {
    Halfs x;
#pragma unroll
    for (int i = 0; i < V / 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) x.h[i][j] = (_Float16)v;
    return x;
  }
  __device__ __forceinline__ float at(int v) const { return (float)h[v / 8][v % 8]; }
  // (streamed out: ordinary stores would push the values still to be read out of the L2; measured 75 -> 60 us)
  static __device__ __forceinline__ void store(uint16_t *p, const float (&e)[V], const float (&f)[V]) {
#pragma unroll
    for (int i = 0; i < V / 8; ++i) {
      half8 y;
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = (_Float16)(e[8 * i + j] * f[8 * i + j]);
      __builtin_nontemporal_store(y, reinterpret_cast<half8 *>(p + 8 * i));
    }
  }
};

}  // namespace

// One wave per (vector-row, batch element); lane l takes the stored vectors l, l + 64, ... of the
// row, V dense rows at a time.  Three passes over the row's values (maximum, sum of exponentials,
// result).  The first kSoftmaxCached vectors of every lane (512 / 256 vectors of the row for V = 8 / 16) are
// loaded once, all loads in flight together, and stay in registers; only the rest of a longer row is read again (from
// the caches).  As much of the time goes into vector instructions as into memory, so there are few per value: the
// extreme of a row is taken on packed halves (x * scaler is monotonic: the maximum of x for a scaler >= 0, of -x, by its
// sign bit, for a negative one), exp(x * s - max) is one multiply-add of x by s * log2(e) and the base-2 exponential, the exponentials
// of the second pass are kept for the third, and what a short row leaves empty is passed by.  48 heads, 4096 keys, 90 % masked:
// 62 us with the three passes on floats, 54 with the exponentials kept, 48 so; 16 heads, 2000 keys 9.3, 8.3, 7.2.  48 heads
// of 512 rows of 60 vectors 22.5 us on floats, 25.3 with a branch on the scaler's sign at every step and the empty slots
// gone through, 20.7 so.
template <int V>
struct SoftmaxCached {
  static constexpr int value = V == 8 ? 8 : 4;
};

template <int V>
__global__ __launch_bounds__(64) void softmax_kernel(const SoftmaxArgs p) {
  constexpr int KC = SoftmaxCached<V>::value;
  const uint32_t w = xcd_work_index(p.per_xcd);
  if (w >= p.total_work) return;
  const uint32_t r = w % (uint32_t)p.m_vec;
  const uint32_t batch = w / (uint32_t)p.m_vec;
  const int row = p.row_indices ? p.row_indices[r] : (int)r;
  const int beg = p.row_offsets[row], end = p.row_offsets[row + 1];
  if (beg == end) return;
  const int lane = threadIdx.x;
  const uint16_t *in = p.values + (int64_t)batch * p.stride;
  uint16_t *out = p.out + (int64_t)batch * p.stride;
  const float s2 = p.scaler * 1.4426950408889634f;
  const bool falling = p.scaler < 0.f;
  const uint32_t sign = falling ? 0x80008000u : 0u;
  const int tail = beg + lane + 64 * KC;  // the lane's first vector that is not held in registers

  // (a lane past the row's end in a slot that other lanes need: a value that changes no extreme; its exponentials are
  // skipped below)
  Halfs<V> cached[KC];
#pragma unroll
  for (int i = 0; i < KC; ++i) {
    const int j = beg + lane + 64 * i;
    if (beg + 64 * i < end) cached[i] = j < end ? Halfs<V>::load(in + (int64_t)j * V) : Halfs<V>::all(falling ? INFINITY : -INFINITY);
  }
  Halfs<V> top = Halfs<V>::all(-INFINITY);
  const auto fold = [&](const Halfs<V> &x) {
#pragma unroll
    for (int i = 0; i < V / 8; ++i) {
      const uintx4 y = __builtin_bit_cast(uintx4, x.h[i]) ^ uintx4{sign, sign, sign, sign};
      top.h[i] = __builtin_elementwise_max(top.h[i], __builtin_bit_cast(half8, y));
    }
  };
#pragma unroll
  for (int i = 0; i < KC; ++i)
    if (beg + 64 * i < end) fold(cached[i]);
  for (int j = tail; j < end; j += 64) fold(Halfs<V>::load(in + (int64_t)j * V));

  float mx[V], sum[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    mx[v] = wave_max(top.at(v)) * (falling ? -s2 : s2);
    sum[v] = 0.f;
  }
  const auto exponentials = [&](const Halfs<V> &x, float (&e)[V]) {
#pragma unroll
    for (int v = 0; v < V; ++v) e[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(x.at(v), s2, -mx[v]));
  };
  float e[KC][V];
#pragma unroll
  for (int i = 0; i < KC; ++i)
    if (beg + lane + 64 * i < end) {
      exponentials(cached[i], e[i]);
#pragma unroll
      for (int v = 0; v < V; ++v) sum[v] += e[i][v];
    }
  for (int j = tail; j < end; j += 64) {
    float f[V];
    exponentials(Halfs<V>::load(in + (int64_t)j * V), f);
#pragma unroll
    for (int v = 0; v < V; ++v) sum[v] += f[v];
  }
#pragma unroll
  for (int v = 0; v < V; ++v) sum[v] = 1.0f / wave_sum(sum[v]);
#pragma unroll
  for (int i = 0; i < KC; ++i) {
    const int j = beg + lane + 64 * i;
    if (j < end) Halfs<V>::store(out + (int64_t)j * V, e[i], sum);
  }
  for (int j = tail; j < end; j += 64) {
    float f[V];
    exponentials(Halfs<V>::load(in + (int64_t)j * V), f);
    Halfs<V>::store(out + (int64_t)j * V, f, sum);
  }
}

// Long rows of 16-row vectors: the three passes on floats, the exponentials made again in the third.  Such rows' values outgrow the
// L2 between the passes, and this kernel, whose registers are as many, gets more of them from the memory behind it: 512
// rows x 8 heads of 256 vectors 16.0 us against 23.2 with the kernel above, 409 24.6 against 30.2, 600 34.9 against 40.8,
// 1500 109 against 113 (200: 14.7 against 14.0, 100: 10.7 against 10.1).
struct WideVec {
  static __device__ __forceinline__ void load(const uint16_t *p, _Float16 (&x)[16]) {
    const half8 lo = *reinterpret_cast<const half8 *>(p), hi = *reinterpret_cast<const half8 *>(p + 8);
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      x[v] = lo[v];
      x[8 + v] = hi[v];
    }
  }
  static __device__ __forceinline__ void store(uint16_t *p, const _Float16 (&x)[16]) {
    half8 lo, hi;
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      lo[v] = x[v];
      hi[v] = x[8 + v];
    }
    __builtin_nontemporal_store(lo, reinterpret_cast<half8 *>(p));
    __builtin_nontemporal_store(hi, reinterpret_cast<half8 *>(p + 8));
  }
};
__global__ __launch_bounds__(64) void softmax_long_kernel(const SoftmaxArgs p) {
  constexpr int V = 16, KC = SoftmaxCached<V>::value;
  const uint32_t w = xcd_work_index(p.per_xcd);
  if (w >= p.total_work) return;
  const uint32_t r = w % (uint32_t)p.m_vec;
  const uint32_t batch = w / (uint32_t)p.m_vec;
  const int row = p.row_indices ? p.row_indices[r] : (int)r;
  const int beg = p.row_offsets[row], end = p.row_offsets[row + 1];
  if (beg == end) return;
  const int lane = threadIdx.x;
  const uint16_t *in = p.values + (int64_t)batch * p.stride;
  uint16_t *out = p.out + (int64_t)batch * p.stride;
  const float s = p.scaler;
  const int tail = beg + lane + 64 * KC;

  _Float16 cached[KC][V];
#pragma unroll
  for (int i = 0; i < KC; ++i) {
    const int j = beg + lane + 64 * i;
    if (j < end) {
      WideVec::load(in + (int64_t)j * V, cached[i]);
    } else {
#pragma unroll
      for (int v = 0; v < V; ++v) cached[i][v] = (_Float16)0;  // never used: the passes below skip these slots
    }
  }

  float mx[V], sum[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    mx[v] = -INFINITY;
    sum[v] = 0.f;
  }
#pragma unroll
  for (int i = 0; i < KC; ++i)
    if (beg + lane + 64 * i < end) {
#pragma unroll
      for (int v = 0; v < V; ++v) mx[v] = fmaxf(mx[v], (float)cached[i][v] * s);
    }
  for (int j = tail; j < end; j += 64) {
    _Float16 x[V];
    WideVec::load(in + (int64_t)j * V, x);
#pragma unroll
    for (int v = 0; v < V; ++v) mx[v] = fmaxf(mx[v], (float)x[v] * s);
  }
#pragma unroll
  for (int v = 0; v < V; ++v) mx[v] = wave_max(mx[v]);
#pragma unroll
  for (int i = 0; i < KC; ++i)
    if (beg + lane + 64 * i < end) {
#pragma unroll
      for (int v = 0; v < V; ++v) sum[v] += __expf((float)cached[i][v] * s - mx[v]);
    }
  for (int j = tail; j < end; j += 64) {
    _Float16 x[V];
    WideVec::load(in + (int64_t)j * V, x);
#pragma unroll
    for (int v = 0; v < V; ++v) sum[v] += __expf((float)x[v] * s - mx[v]);
  }
#pragma unroll
  for (int v = 0; v < V; ++v) sum[v] = 1.0f / wave_sum(sum[v]);
#pragma unroll
  for (int i = 0; i < KC; ++i) {
    const int j = beg + lane + 64 * i;
    if (j < end) {
      _Float16 y[V];
#pragma unroll
      for (int v = 0; v < V; ++v) y[v] = (_Float16)(__expf((float)cached[i][v] * s - mx[v]) * sum[v]);
      WideVec::store(out + (int64_t)j * V, y);
    }
  }
  for (int j = tail; j < end; j += 64) {
    _Float16 x[V], y[V];
    WideVec::load(in + (int64_t)j * V, x);
#pragma unroll
    for (int v = 0; v < V; ++v) y[v] = (_Float16)(__expf((float)x[v] * s - mx[v]) * sum[v]);
    WideVec::store(out + (int64_t)j * V, y);
  }
}

hipError_t launch_softmax(const SoftmaxArgs &a, int V, hipStream_t stream) {
  SoftmaxArgs p = a;
  p.total_work = (uint32_t)a.m_vec * (uint32_t)a.batch;
  p.per_xcd = (p.total_work + 7u) / 8u;
  if (p.total_work == 0) return hipSuccess;
  // (the batch stride is the number of stored values, so it tells a row's mean length; 0, of a single product, does not)
  const bool long_rows = V == 16 && (a.stride <= 0 || a.stride > (int64_t)a.m_vec * (16 * 208));
  if (V == 8)
    hipLaunchKernelGGL(softmax_kernel<8>, dim3(p.per_xcd * 8u), dim3(64), 0, stream, p);
  else if (long_rows)
    hipLaunchKernelGGL(softmax_long_kernel, dim3(p.per_xcd * 8u), dim3(64), 0, stream, p);
  else
    hipLaunchKernelGGL(softmax_kernel<16>, dim3(p.per_xcd * 8u), dim3(64), 0, stream, p);
  return hipGetLastError();
}

// ---------------------------------------------------------------------- the three steps in one
// softmax(mask(q k^T) * scale) v per vector-row without the scores ever leaving the CU, for heads of 32, 64 or 128
// features (described for 64)
// (the three launches of the block, reference end2end/sspmm_e2e/spattention.py:167-179, move the scores and the
// probabilities through memory twice each: 2 * V bytes per stored vector four times over).
//
// One wave per (vector-row, batch element), a step is 32 stored vectors.  The rows of k and of v the step names
// are fetched as in the staged SpMM kernel (eight lanes on the eight 16-byte pieces of one 128-byte row, lane
// (j, pc) = rows of k slots 4j .. 4j+3, piece pc) and written to an LDS stage with padded rows, k's first and v's behind them.
//   scores:  the staged rows of k are the MFMA's first operand (lane (n, g): features 32c + 8g .. of staged row
//            16t + n), the V rows of q the second, held in registers for the whole row; the lane ends up with the
//            scores of query n against staged rows 16t + 4g + r, r = 0 .. 3, t = 0, 1.
//   softmax: running maximum and running sum per query in base 2 (the scale carries log2 e); a query's scores
//            sit in the four lanes n, n + 16, n + 32, n + 48, which exchange their maxima with two lane swaps.
//            When the maximum moves, the sums so far are scaled down by 2^(old - new).
//   product: the eight probabilities of a lane are, in this order, the second operand's k slots 8g .. 8g+7 of
//            query n; the first operand is the transpose read of the staged rows of v in the matching order
//            (rows 4g .. 4g+3, then 16 + 4g .. 16 + 4g + 3).  Lane (n, g) accumulates features 16u + 4g + r of
//            query n, u = 0 .. 3, divides by the sum at the end and stores four times 8 bytes.
// The probabilities enter the product rounded to fp16 before the division by the sum (the three launches round
// after it); sums are fp32 throughout.
// The launch is bound by the stream of gathered rows from the L2 into the CUs (256 bytes per stored vector and batch
// element; 22 TB/s on 4096 keys, 90 % masked, once there are rows for every wave).  What it can be given is loads in flight: rows in registers
// for one step and one stage that k's and v's pass through in turn take 106 registers and 5 KB of LDS a wave, four waves per SIMD, where two
// sets of rows and two stages (160 registers, two waves) had 20.9 TB/s.  4096 keys, 64 features, 8 / 16 / 32 / 64 (element, head) pairs, V = 8:
// 27.6 / 49.2 / 90.8 / 167.8 -> 25.5 / 44.9 / 82.3 / 153.6 us, V = 16: 15.1 / 27.8 / 51.0 / 97.3 -> 14.7 / 25.8 / 46.0 / 88.1 (sums of rounded probabilities; of the
// exponentials, as now, measures the same, 8 pairs 21.06 / 21.13 replayed, 32 pairs 76.3 / 76.4, V = 16 13.25 / 13.16 and 45.1 / 44.8).  32 features (six waves) 19.0 / 33.1 / 60.6 / 112.7 -> 18.3 / 33.8 / 60.7 / 112.4, 128 (two) 46.2 / 84.3 / 156 / 308
// -> 45.2 / 81.9 / 152 / 302; five waves at 64 features, eight at 32, three at 128 are level or slower, and so are two stages.  Neither what a
// wave computes nor its column indices count: two heads per wave, which share the indices and the addresses, are level (27.6 -> 29, 106 -> 107), and
// indices handed out with lane permutes, as the sddmm kernel does, slower (124 -> 137 us: the permutes queue in the LDS pipe).
// K and V of 256 keys at a time in LDS, every CU fetching all of them for its 64 vector-rows, would read the L2 a seventh as often; it was built and
// is level at 32 pairs (85-93 us) and slower below (36 us at 8): its waves wait for each other at every panel.
constexpr int attention_waves(int F) { return F == 64 ? 4 : F == 32 ? 6 : 2; }  // per SIMD

// F: features per row of q, k and v (32, 64 or 128).  A row is F * 2 bytes = LPR 16-byte pieces, a load instruction
// brings 64 / LPR rows, a step of 32 rows takes L = LPR / 2 of them per operand; lane (jr, pc) fetches piece pc of the
// rows of k slots L * jr .. L * jr + L - 1, whose column indices it reads as L consecutive ints.
template <int V, int F>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(attention_waves(F), attention_waves(F)))) void sparse_attention_kernel(const AttentionArgs p) {
  constexpr int LPR = F / 8, L = LPR / 2, NC = F / 32, NT = F / 16;
  constexpr uint32_t kRowBytes = F * 2u, kPitch = kRowBytes + 32u;  // (sixteen rows' pieces, read four at a time, then touch every bank as often)
  __shared__ __align__(16) unsigned char stage[32 * kPitch];
  const uint32_t w = xcd_work_index(p.per_xcd);
  if (w >= p.total_work) return;
  const uint32_t r = w % (uint32_t)p.m_vec;
  const uint32_t batch = w / (uint32_t)p.m_vec;
  const int row = __builtin_amdgcn_readfirstlane(p.row_indices ? p.row_indices[r] : (int)r);
  const int beg = p.row_offsets[row], end = p.row_offsets[row + 1];
  const int lane = threadIdx.x, n = lane & 15, g = lane >> 4, jr = lane / LPR, pc = lane % LPR;

  const uint32_t elem = batch / (uint32_t)p.heads, head = batch % (uint32_t)p.heads;
  uint16_t *out = p.out + (int64_t)elem * p.stride_out + (int64_t)head * p.head_out + ((int64_t)row * V + n) * p.ld_out + 4 * g;
  if (beg == end) {  // a query that attends to nothing: zeros, as the product with no stored vectors gives
    if (n < V) {
#pragma unroll
      for (int u = 0; u < NT; ++u) *reinterpret_cast<uintx2 *>(out + 16 * u) = uintx2{0u, 0u};
    }
    return;
  }
  // (descriptors end with the last row's bytes; between the rows of a strided operand lies what belongs to other heads)
  const uint32_t q_row = (uint32_t)p.ld_q * 2u, k_row = (uint32_t)p.ld_k * 2u, v_row = (uint32_t)p.ld_v * 2u;
  const __amdgpu_buffer_rsrc_t srd_q = make_srd(p.q + (int64_t)elem * p.stride_q + (int64_t)head * p.head_q + (int64_t)row * V * p.ld_q,
                                                (uint32_t)(V - 1) * q_row + kRowBytes);
  // (no keys at all: descriptors of zero bytes, whatever a pattern then names reads as zeros)
  const uint32_t k_bytes = p.n_keys > 0 ? (uint32_t)(p.n_keys - 1) * k_row + kRowBytes : 0u;
  const uint32_t v_bytes = p.n_keys > 0 ? (uint32_t)(p.n_keys - 1) * v_row + kRowBytes : 0u;
  const __amdgpu_buffer_rsrc_t srd_k = make_srd(p.k + (int64_t)elem * p.stride_k + (int64_t)head * p.head_k, k_bytes);
  const __amdgpu_buffer_rsrc_t srd_v = make_srd(p.v + (int64_t)elem * p.stride_v + (int64_t)head * p.head_v, v_bytes);
  const __amdgpu_buffer_rsrc_t srd_cols = make_srd(p.col_idx, (uint32_t)end * 4u);  // past the row: reads 0

  half8 q[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)  // (rows past V: beyond the descriptor, zeros)
    q[c] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(srd_q, n < V ? (uint32_t)n * q_row + (32u * c + 8u * g) * 2u : 0xfffffff0u, 0, 0));

  unsigned char *const dst = stage + (uint32_t)(L * jr) * kPitch + (uint32_t)pc * 16u;
  const unsigned char *const k_rd = stage + (uint32_t)n * kPitch + (uint32_t)g * 16u;
  const unsigned char *const v_rd = stage + (uint32_t)(4 * g + (n >> 2)) * kPitch + (uint32_t)(n & 3) * 8u;
  const uint32_t piece_off = (uint32_t)pc * 16u;
  const float scale2 = p.scale * 1.4426950408889634f;

  struct Head {
    uint32_t c[L];
  };
  const auto load_head = [&](int kc) {
    Head h;
    const int at = (kc + L * jr) * 4;
    if (L == 2) {
      const uintx2 x = __builtin_bit_cast(uintx2, __builtin_amdgcn_raw_buffer_load_b64(srd_cols, at, 0, 0));
      h.c[0] = x[0]; h.c[1] = x[1];
    } else {
#pragma unroll
      for (int i = 0; i < L; i += 4) {
        const uintx4 x = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(srd_cols, at + 4 * i, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) h.c[(i + e) % L] = x[e];
      }
    }
    return h;
  };
  struct Places {
    uint32_t k[L], v[L];
  };
  const auto places = [&](const Head &h, int kc) {
    Places o;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      o.k[i] = __umul24(h.c[i], k_row) + piece_off;  // (both factors below 2^24: the launcher's caller checks the row pitch)
      o.v[i] = __umul24(h.c[i], v_row) + piece_off;
    }
    if (kc + 32 > end) {  // (uniform) the row's last step: slots past its end fetch zeros
#pragma unroll
      for (int i = 0; i < L; ++i) {
        const bool live = kc + L * jr + i < end;
        o.k[i] = live ? o.k[i] : k_bytes;
        o.v[i] = live ? o.v[i] : v_bytes;
      }
    }
    return o;
  };
  uintx4 k[L], v[L];
  const auto fetch = [&](uintx4 (&rows)[L], const __amdgpu_buffer_rsrc_t &srd, const uint32_t (&at)[L]) {
#pragma unroll
    for (int i = 0; i < L; ++i) rows[i] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(srd, at[i], 0, 0));
  };
  // (LDS operations of a wave execute in order: the writes land behind the reads of what the stage held before)
  const auto put = [&](const uintx4 (&rows)[L]) {
#pragma unroll
    for (int i = 0; i < L; ++i) *reinterpret_cast<uintx4 *>(dst + i * kPitch) = rows[i];
  };

  floatx4 acc[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) acc[u] = floatx4{0.f, 0.f, 0.f, 0.f};
  float run_raw = -INFINITY, run_max = -INFINITY, run_sum = 0.f;  // of query n: maximum before and after the scale; the sum only over this lane's share of the keys
  // Some query's scaled maximum lies beyond 2^10 (uniform).  An exponent x scale2 - run_max misses by the rounding of run_max, the same for every key: beyond 2^28
  // the largest probability would be 2^16 or 0, so there the difference is taken first, which is 0 at the maximum; below 2^10 it is 2^-15 and cancels in the quotient.  Costs 2 us of 507 in
  // a model of 8 x 4096 tokens; taken first everywhere it is the additions that the multiply-add saves.
  bool far = false;

  float x[8];
  const auto scores = [&] {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const half8 a = *reinterpret_cast<const half8 *>(k_rd + (uint32_t)t * (16u * kPitch) + (uint32_t)c * 64u);
        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, q[c], s, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) x[4 * t + i] = s[i];
    }
  };
  const auto softmax_and_product = [&](int kc) {
    if (kc + 32 > end) {  // (uniform)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (kc + 16 * t + 4 * g + i >= end) x[4 * t + i] = -INFINITY;
    }
    float mx = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
    mx = max_over_rows(mx);  // finite: the step's first slot is always a stored vector
    const float new_raw = fmaxf(run_raw, mx);  // (scale2 > 0: the order of the scaled scores)
    if (__builtin_amdgcn_ballot_w64(new_raw > run_raw)) {  // (uniform) some query's maximum moved
      const float alpha = __builtin_amdgcn_exp2f((run_raw - new_raw) * scale2);
      run_sum *= alpha;
#pragma unroll
      for (int u = 0; u < NT; ++u) acc[u] *= alpha;
      run_raw = new_raw;
      run_max = new_raw * scale2;
      far = __builtin_amdgcn_ballot_w64(fabsf(run_max) > 1024.f) != 0;
    }
    if (far) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = (x[i] - run_raw) * scale2;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf(x[i], scale2, -run_max);
    }
    half8 pb;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float e = __builtin_amdgcn_exp2f(x[i]);
      sum += e;  // (before the rounding: many probabilities that fp16 does not hold are a part of it)
      pb[i] = (_Float16)e;
    }
    run_sum += sum;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const uintx2 lo = lds_read_tr(v_rd + 32u * u);
      const uintx2 hi = lds_read_tr(v_rd + 16u * kPitch + 32u * u);
      const uintx4 a = {lo[0], lo[1], hi[0], hi[1]};
      acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), pb, acc[u], 0, 0, 0);
    }
  };

  // Column indices run two steps ahead of the arithmetic, the rows of k and v one: a step's rows pass through the stage, k's and then
  // v's, and the next step's are on their way as soon as the registers are free.
  const auto in_order = [] { asm volatile("" ::: "memory"); };  // (left alone the compiler lets loads sink to their first use)
  const Head now = load_head(beg);
  Head ahead = load_head(beg + 32);
  in_order();
  Places at = places(now, beg);
  fetch(k, srd_k, at.k);
  fetch(v, srd_v, at.v);
  // The last step stands apart, and the loads stay in this order: where loads may or may not have been issued behind those that a write to
  // LDS waits for, it waits for all.  4096 keys, 64 features, replayed, with one loop / now: V = 8, one pair 8.80 / 8.38 us, 2 9.45 / 9.2-9.3, 4 and more
  // level; V = 16, 1 / 2 / 4 / 8 pairs 8.50 / 9.13 / 9.9 / 13.1 -> 8.07 / 8.64 / 9.41 / 13.1, 32 features 7.1 / 7.6 / 7.8 / 9.5 -> 6.7 / 7.15 / 7.4 / 9.4,
  // 128 features 11.9 / 12.7 / 15.0 / 24.0 -> 11.2 / 12.1 / 14.4 / 24.1; 1024 waves on 1024 keys, V = 16 5.33 -> 5.11.
  int kc = beg;
  for (; kc + 32 < end; kc += 32) {
    put(k);
    at = places(ahead, kc + 32);
    fetch(k, srd_k, at.k);
    ahead = load_head(kc + 64);
    scores();
    put(v);
    fetch(v, srd_v, at.v);
    in_order();
    softmax_and_product(kc);
  }
  put(k);
  scores();
  put(v);
  softmax_and_product(kc);

  const float inv = 1.0f / sum_over_rows(run_sum);
  if (n < V) {
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const half4 h = {(_Float16)(acc[u][0] * inv), (_Float16)(acc[u][1] * inv), (_Float16)(acc[u][2] * inv), (_Float16)(acc[u][3] * inv)};
      *reinterpret_cast<uintx2 *>(out + 16 * u) = __builtin_bit_cast(uintx2, h);
    }
  }
}

template <int V>
static void launch_sparse_attention_v(const AttentionArgs &p, int F, hipStream_t stream) {
  const dim3 grid(p.per_xcd * 8u), block(64);
  if (F == 32) hipLaunchKernelGGL((sparse_attention_kernel<V, 32>), grid, block, 0, stream, p);
  else if (F == 64) hipLaunchKernelGGL((sparse_attention_kernel<V, 64>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((sparse_attention_kernel<V, 128>), grid, block, 0, stream, p);
}

hipError_t launch_sparse_attention(const AttentionArgs &a, int V, int F, hipStream_t stream) {
  if (F != 32 && F != 64 && F != 128) return hipErrorInvalidValue;
  AttentionArgs p = a;
  p.total_work = (uint32_t)a.m_vec * (uint32_t)a.batch;
  p.per_xcd = (p.total_work + 7u) / 8u;
  if (p.total_work == 0) return hipSuccess;
  if (V == 8) launch_sparse_attention_v<8>(p, F, stream);
  else launch_sparse_attention_v<16>(p, F, stream);
  return hipGetLastError();
}

}  // namespace sspmm
