// gemm.hip -- prefill GEMM on the matrix cores, and on-device Q8_0
// activation quantization.
//
// Replaces the prefill use of forward_linear_batch
// (swamp-engine/src/executor.rs:106-110 -> linear.rs:176-239): the reference
// runs the batched CPU GEMV token block by token block; here one launch
// computes y[m][r] = sum_k W[r,k] x[m][k] for the whole prompt.
// The bf16 kernel is in gemm_core.hpp; the int8 one in gemm_i8.hip.
#include "gemm_core.hpp"

namespace {

// y = sum of the K pieces' partials, in piece order (deterministic); all
// (at most 8) loads are issued before the adds.
__global__ void split_reduce_kernel(const float *__restrict__ part, float *__restrict__ y,
                                    int splits, size_t n) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float v[8];
#pragma unroll
  for (int p = 0; p < 8; p++) v[p] = p < splits ? part[size_t(p) * n + i] : 0.f;
  float s = v[0];
#pragma unroll
  for (int p = 1; p < 8; p++) s += v[p];  // missing pieces add 0
  y[i] = s;
}

// The same sums, 4 consecutive elements per thread (16-byte loads and
// stores: part, y and n / 4 16-byte aligned); each element takes the
// scalar kernel's additions in the same order, so y is bit-identical.
__global__ void split_reduce4_kernel(const float4 *__restrict__ part, float4 *__restrict__ y,
                                     int splits, size_t n4) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n4) return;
  float4 v[8];
#pragma unroll
  for (int p = 0; p < 8; p++)
    v[p] = p < splits ? part[size_t(p) * n4 + i] : make_float4(0.f, 0.f, 0.f, 0.f);
  float4 s = v[0];
#pragma unroll
  for (int p = 1; p < 8; p++) {
    s.x += v[p].x;
    s.y += v[p].y;
    s.z += v[p].z;
    s.w += v[p].w;
  }
  y[i] = s;
}

// ---- Q8_0 activation quantization ------------------------------------------
// The arithmetic of one block, shared by both kernels: amax over the block,
// d = amax / 127, q = round(v / d) clamped to [-127, 127], d stored as fp16
// (the host quantizer's, byte for byte).
__device__ __forceinline__ float q8_scale(float amax) { return amax / 127.0f; }
__device__ __forceinline__ int q8_code(float v, float d) {
  const float id = d != 0.f ? 1.0f / d : 0.f;
  const float q = fminf(127.f, fmaxf(-127.f, roundf(v * id)));
  return int(q);
}

// Any alignment of dst: one element per thread, 32 lanes per block, byte
// stores.  Also quantizes the blocks [first, n_blocks) left over by the
// vector kernel below.
template <bool kBf16>
__global__ void quantize_q8_0_kernel(const void *__restrict__ src, uint8_t *__restrict__ dst,
                                     size_t first, size_t n_blocks) {
  const size_t gid = first * 32 + size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const size_t blk = gid >> 5;
  const int i = int(gid & 31);
  const bool ok = blk < n_blocks;
  float v = 0.f;
  if (ok) {
    if (kBf16) v = __uint_as_float(uint32_t(static_cast<const uint16_t *>(src)[gid]) << 16);
    else v = static_cast<const float *>(src)[gid];
  }
  float a = fabsf(v);
#pragma unroll
  for (int off = 16; off >= 1; off >>= 1) a = fmaxf(a, __shfl_xor(a, off, 32));
  const float d = q8_scale(a);
  const int q = q8_code(v, d);
  if (ok) {
    uint8_t *b = dst + blk * 34;
    b[2 + i] = uint8_t(int8_t(q));
    if (i == 0) {
      const uint16_t h = __builtin_bit_cast(uint16_t, _Float16(d));
      b[0] = uint8_t(h & 0xFF);
      b[1] = uint8_t(h >> 8);
    }
  }
}

// 4-byte aligned dst: a wave quantizes 8 whole blocks, 4 consecutive
// elements per lane (one 16-byte or 8-byte load), the block's amax over its
// 8 lanes.  The wave's 8 output blocks are 272 contiguous bytes at a 4-byte
// aligned offset (272 = 4 * 68): they are assembled in LDS with 2-byte
// stores (a lane's 4 codes sit at 34 k + 2 + 4 j, 2 mod 4 for even blocks)
// and written out as 68 dwords.  Only whole groups of 8 blocks come here.
template <bool kBf16>
__global__ void __launch_bounds__(256) quantize_q8_0_x8_kernel(const void *__restrict__ src,
                                                               uint8_t *__restrict__ dst,
                                                               size_t n_groups) {
  __shared__ uint32_t stage[4][68];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const size_t grp = size_t(blockIdx.x) * 4 + size_t(w);
  const bool ok = grp < n_groups;  // uniform per wave
  const int k = lane >> 3, j = lane & 7;
  // this workgroup's groups as one buffer range (out-of-range loads read 0)
  const size_t g0 = size_t(blockIdx.x) * 4;
  const uint32_t ebytes = kBf16 ? 2u : 4u;
  const uint32_t range = uint32_t(min(n_groups - g0, size_t(4)) * 256u * ebytes);
  const __amdgpu_buffer_rsrc_t r = swamp::make_rsrc(
      static_cast<const uint8_t *>(src) + g0 * 256u * ebytes, range);
  const uint32_t voff = (uint32_t(w) * 256u + uint32_t(lane) * 4u) * ebytes;
  float v[4];
  if constexpr (kBf16) {
    typedef uint32_t u32x2v_t __attribute__((ext_vector_type(2)));
    const u32x2v_t h = __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, 0);
    v[0] = __uint_as_float(h[0] << 16);
    v[1] = __uint_as_float(h[0] & 0xFFFF0000u);
    v[2] = __uint_as_float(h[1] << 16);
    v[3] = __uint_as_float(h[1] & 0xFFFF0000u);
  } else {
    const u32x4v_t a = __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = __uint_as_float(a[i]);
  }
  float a = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
  for (int off = 4; off >= 1; off >>= 1) a = fmaxf(a, __shfl_xor(a, off, 8));
  const float d = q8_scale(a);
  uint32_t packed = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) packed |= (uint32_t(q8_code(v[i], d)) & 0xFFu) << (8 * i);
  typedef uint16_t __attribute__((may_alias)) u16_alias_t;  // 2-byte view of the dword stage
  u16_alias_t *st = reinterpret_cast<u16_alias_t *>(stage[w]);
  const int o = 17 * k + 1 + 2 * j;  // in 2-byte units: byte 34 k + 2 + 4 j
  st[o] = uint16_t(packed & 0xFFFFu);
  st[o + 1] = uint16_t(packed >> 16);
  if (j == 0) st[17 * k] = __builtin_bit_cast(uint16_t, _Float16(d));
  __syncthreads();
  if (ok) {
    uint32_t *out = reinterpret_cast<uint32_t *>(dst + grp * 272u);
    out[lane] = stage[w][lane];
    if (lane < 4) out[64 + lane] = stage[w][64 + lane];
  }
}

}  // namespace

int swamp_launch_split_reduce(const float *d_part, float *d_y, int pieces, size_t n,
                              hipStream_t s) {
  if (pieces < 1 || pieces > 8) return SWAMP_EINVAL;
  if (n % 4 == 0 && reinterpret_cast<uintptr_t>(d_part) % 16 == 0 &&
      reinterpret_cast<uintptr_t>(d_y) % 16 == 0) {
    const size_t n4 = n / 4;
    split_reduce4_kernel<<<unsigned((n4 + 255) / 256), 256, 0, s>>>(
        reinterpret_cast<const float4 *>(d_part), reinterpret_cast<float4 *>(d_y), pieces, n4);
  } else {
    split_reduce_kernel<<<unsigned((n + 255) / 256), 256, 0, s>>>(d_part, d_y, pieces, n);
  }
  return hipGetLastError() == hipSuccess ? SWAMP_OK : SWAMP_ELAUNCH;
}

size_t swamp_gemm_scratch_bytes(uint32_t dtype, uint32_t x_type, int m, int n_rows, int n_cols,
                                size_t limit) {
  if (m <= 0 || n_rows <= 0 || n_cols <= 0) return 0;
  if (x_type == SWAMP_Q8_0)
    return swamp::scratch_round(swamp_gemm_i8_scratch_bytes(dtype, m, n_rows, n_cols));
  if (x_type != SWAMP_BF16 || n_cols % kBK != 0) return 0;
  if (swamp_gemm_dq_route(dtype, m, n_rows, n_cols)) {
    const size_t dq = swamp_gemm_dq_scratch_bytes(m, n_rows, n_cols);
    if (dq <= limit || dtype == SWAMP_Q6_K) return dq;
  }
  switch (dtype) {
    case SWAMP_Q4_0: return swamp::scratch_round(plan_bf16<SWAMP_Q4_0>(m, n_rows, n_cols).part_bytes);
    case SWAMP_Q8_0: return swamp::scratch_round(plan_bf16<SWAMP_Q8_0>(m, n_rows, n_cols).part_bytes);
    case SWAMP_Q4_K: return swamp::scratch_round(plan_bf16<SWAMP_Q4_K>(m, n_rows, n_cols).part_bytes);
    case SWAMP_Q6_K: return swamp_gemm_q6k_scratch_bytes(m, n_rows, n_cols);
    default: return 0;
  }
}

int swamp_launch_gemm(uint32_t dtype, const void *d_w, const void *d_x, uint32_t x_type,
                      float *d_y, int m, int n_rows, int n_cols, swamp::Scratch &sc,
                      hipStream_t s) {
  if (m == 0 || n_rows == 0) return SWAMP_OK;
  if (x_type == SWAMP_Q8_0)
    return swamp_launch_gemm_i8(dtype, d_w, d_x, d_y, m, n_rows, n_cols, sc, s);
  if (x_type != SWAMP_BF16) return SWAMP_EDTYPE;
  if (n_cols % kBK != 0) return SWAMP_ESHAPE;
  // activation offsets are 32-bit (buffer descriptors)
  if (size_t(m) * size_t(n_cols) * 2 > size_t(UINT32_MAX)) return SWAMP_ESHAPE;
  // long prompts: dequantize once to bf16 and run a plain bf16 GEMM, when
  // the scratch for it is there (else the fused kernel below)
  bool once = swamp_gemm_dq_route(dtype, m, n_rows, n_cols);
  // Q6_K scratch too small for the fused kernel's partial sums may still hold
  // the weights
  if (dtype == SWAMP_Q6_K && sc.cap - sc.used < swamp_gemm_q6k_scratch_bytes(m, n_rows, n_cols))
    once = true;
  if (once && sc.cap - sc.used >= swamp_gemm_dq_scratch_bytes(m, n_rows, n_cols)) {
    const size_t used = sc.used;
    const int rc = swamp_launch_gemm_dq(dtype, d_w, d_x, d_y, m, n_rows, n_cols, sc, s);
    if (rc != kDqUnavailable) return rc;
    sc.used = used;
  }
  if (dtype == SWAMP_Q6_K) return swamp_launch_gemm_q6k(d_w, d_x, d_y, m, n_rows, n_cols, sc, s);
  const uint8_t *w = static_cast<const uint8_t *>(d_w);
  const uint16_t *x = static_cast<const uint16_t *>(d_x);
  switch (dtype) {
    case SWAMP_Q4_0: return launch_bf16<SWAMP_Q4_0>(w, x, d_y, m, n_rows, n_cols, sc, s);
    case SWAMP_Q8_0: return launch_bf16<SWAMP_Q8_0>(w, x, d_y, m, n_rows, n_cols, sc, s);
    case SWAMP_Q4_K: return launch_bf16<SWAMP_Q4_K>(w, x, d_y, m, n_rows, n_cols, sc, s);
    default: return SWAMP_EDTYPE;
  }
}

int swamp_launch_quantize_q8_0(const void *d_x, uint32_t x_type, void *d_q, size_t n,
                               hipStream_t s) {
  const size_t nb = n / 32;
  if (nb == 0) return SWAMP_OK;
  if (x_type != SWAMP_BF16 && x_type != SWAMP_F32) return SWAMP_EDTYPE;
  const bool bf = x_type == SWAMP_BF16;
  uint8_t *q = static_cast<uint8_t *>(d_q);
  // whole groups of 8 blocks by the vector kernel when dst is 4-byte
  // aligned; the rest (and any block of an unaligned dst) one element per thread
  const size_t groups = reinterpret_cast<uintptr_t>(d_q) % 4 == 0 ? nb / 8 : 0;
  if (groups > 0) {
    const unsigned grid = unsigned((groups + 3) / 4);
    if (bf) quantize_q8_0_x8_kernel<true><<<grid, 256, 0, s>>>(d_x, q, groups);
    else quantize_q8_0_x8_kernel<false><<<grid, 256, 0, s>>>(d_x, q, groups);
  }
  const size_t first = groups * 8;
  if (first < nb) {
    const unsigned grid = unsigned(((nb - first) * 32 + 255) / 256);
    if (bf) quantize_q8_0_kernel<true><<<grid, 256, 0, s>>>(d_x, q, first, nb);
    else quantize_q8_0_kernel<false><<<grid, 256, 0, s>>>(d_x, q, first, nb);
  }
  return hipGetLastError() == hipSuccess ? SWAMP_OK : SWAMP_ELAUNCH;
}
