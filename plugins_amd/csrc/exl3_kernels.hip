// exl3_kernels.hip -- HIP kernels for the EXL3 trellis-quantized linear on
// MI355X (gfx950, wave64) and their host launchers.
//
// Kernels (reference roles, paths relative to /root/reference/plugins/):
//  * prepare / finish: the Hadamard-128 rotations around the inner product
//    (sushi_ds41/src/sushi/exl3/expert_exl3_kernels.zig:902-970; contract
//    turboexl3_qwen38/overlay/mlx_serve/abi/quant.zig:52-55);
//  * decode_matrix: whole-matrix decode to f16 (the `q3_exl3_dig_decmat_*`
//    role, turboexl3_ds41/src/exl3/kernels/exl3/q3_exl3_dig_decmat_5120x2304_mul1hk3.metal);
//  * gemv: rows <= 8, weights decoded in registers, split-K over workgroups
//    with the finish fused into the last workgroup of each 128-column group
//    (the decode GEMV role: expert_exl3_kernels.zig:1653-1849,
//    turboexl3_ds41/src/exl3/kernels/exl3/dsv41_exl3_mul1h_k3_2304.metal);
//  * gemm: any rows, weight tiles decoded into LDS as f16 in MFMA operand
//    layout, v_mfma_f32_32x32x16_f16 with f32 accumulation, finish fused
//    (the prefill GEMM role: expert_exl3_kernels.zig:676-750,
//    dsv41_prefill_dig_gemm_5120x2304_gu_xmul1hk3_m128.metal).
//
// Compiled with -ffp-contract=off: every f32 multiply and add rounds on its
// own where the reference's order of operations is reproduced; fused
// multiply-adds are written out where they are meant.
// The rate-templated kernels live in exl3_kern.h; their launchers are
// instantiated once per rate in exl3_rate.hip.
#include <atomic>

#include "exl3_kern.h"

namespace exl3 {

// =================================================================== prepare

// One wave per 128-block of one row, four blocks per workgroup: element i
// of the block lives in lane i/2, register i%2 (had128_pair: the stage on
// index bit 0 in-register, bits 1..6 across lanes; each stage (lo + hi,
// lo - hi) in bit order, as the reference computes it).
// Row r takes suh row r % groups (groups 1: one suh for every row; a grouped
// linear's [rows, G, in] input: group g's suh for its rows).
__global__ __launch_bounds__(256) void prepare_kernel(const void *__restrict__ x, int xdt,
                                                      const uint16_t *__restrict__ suh,
                                                      uint16_t *__restrict__ xp, int in,
                                                      int nblk, int groups) {
  const int lane = threadIdx.x & 63;
  const int blk = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (blk >= nblk) return;  // whole waves
  const size_t base = (size_t)blockIdx.y * in;
  const int k = blk * 128 + 2 * lane;
  // f16(x) * suh in f32 (expert_exl3.zig:490-493; the kernel's
  // float(x) * float(suh), expert_exl3_kernels.zig:908-912).
  const uint32_t su =
      *reinterpret_cast<const uint32_t *>(suh + (size_t)(blockIdx.y % (unsigned)groups) * in + k);
  float v0 = h2f(f2h(load_act(x, base + k, xdt))) * h2f((uint16_t)(su & 0xFFFFu));
  float v1 = h2f(f2h(load_act(x, base + k + 1, xdt))) * h2f((uint16_t)(su >> 16));
  had128_pair(v0, v1, lane);
  *reinterpret_cast<uint32_t *>(xp + base + k) =
      (uint32_t)f2h(v0 * HAD_SCALE) | ((uint32_t)f2h(v1 * HAD_SCALE) << 16);
}

// The same rotation on an f16 [rows, 128-block] of inner products, then
// * svh, rounded to f16, stored in the output dtype
// (expert_exl3_kernels.zig:938-970; expert_exl3.zig:534-544).
__device__ __forceinline__ void finish_row_wave(const uint16_t *z, const uint16_t *svh, void *y,
                                                int ydt, size_t yoff, int lane) {
  float v0 = h2f(z[lane]);
  float v1 = h2f(z[lane + 64]);
#pragma unroll
  for (int bit = 1; bit <= 32; bit <<= 1) {
    const float p0 = xor_lanes(v0, bit), p1 = xor_lanes(v1, bit);
    const float sg = (lane & bit) == 0 ? 1.0f : -1.0f;
    v0 = butterfly(sg, v0, p0);
    v1 = butterfly(sg, v1, p1);
  }
  const float a = v0 + v1, b = v0 - v1;
  const float s0 = a * HAD_SCALE, s1 = b * HAD_SCALE;
  store_out(y, yoff + lane, f2h(s0 * h2f(svh[lane])), ydt);
  store_out(y, yoff + lane + 64, f2h(s1 * h2f(svh[lane + 64])), ydt);
}

__global__ __launch_bounds__(64) void finish_kernel(const uint16_t *__restrict__ z,
                                                    const uint16_t *__restrict__ svh,
                                                    void *__restrict__ y, int ydt, int out) {
  const size_t off = (size_t)blockIdx.y * out + blockIdx.x * 128;
  finish_row_wave(z + off, svh + blockIdx.x * 128, y, ydt, off, threadIdx.x);
}

// prepare_kernel's rotation with 8 elements per lane and 16-byte accesses:
// a 128-block is 16 lanes, element 8 j + i in lane j's register i.  The
// butterflies on element bits 0-2 run in registers, bits 3-6 across the 16
// lanes, in had128_pair's stage order and with its sums (lo + hi, lo - hi),
// so the results are identical.  Block gb of the flattened [rows][in / 128]
// starts at element 128 gb.  x, suh and xp must be 16-byte aligned.
struct SuhSets {
  const uint16_t *p[4];
};
// SETS: grid y is one prepared set per consumer (suh sets.p[y], xp stacked).
// Its own instantiation: one set's suh comes preloaded in SGPRs, the sets'
// pointer from an indexed argument load ahead of suh's own.
template <bool SETS>
__global__ __launch_bounds__(256) void prepare8_kernel(const void *__restrict__ x, int xdt,
                                                       const uint16_t *__restrict__ suh0,
                                                       uint16_t *__restrict__ xp0, int nblk,
                                                       uint32_t nblocks, int groups,
                                                       SuhSets sets) {
  const uint16_t *__restrict__ suh = SETS ? sets.p[blockIdx.y] : suh0;
  uint16_t *__restrict__ xp = SETS ? xp0 + (size_t)blockIdx.y * nblocks * 128 : xp0;
  const int j = threadIdx.x & 15;
  const uint32_t gb0 = blockIdx.x * 16u + (threadIdx.x >> 4);
  const bool valid = gb0 < nblocks;  // a 16-lane group is valid or not as a whole
  const uint32_t gb = valid ? gb0 : nblocks - 1;
  const size_t off = (size_t)gb * 128 + 8 * j;
  const int k = (int)(gb % (uint32_t)nblk) * 128 + 8 * j;
  const size_t ks = (size_t)((gb / (uint32_t)nblk) % (uint32_t)groups) * nblk * 128 + k;
  float v[8];
  if (xdt == OUT_F32) {
    const float4 a = *reinterpret_cast<const float4 *>((const float *)x + off);
    const float4 b = *reinterpret_cast<const float4 *>((const float *)x + off + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else {
    const uint4 w = *reinterpret_cast<const uint4 *>((const uint16_t *)x + off);
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint16_t lo = (uint16_t)(ws[i] & 0xFFFFu), hi = (uint16_t)(ws[i] >> 16);
      v[2 * i] = xdt == OUT_F16 ? h2f(lo) : bf2f(lo);
      v[2 * i + 1] = xdt == OUT_F16 ? h2f(hi) : bf2f(hi);
    }
  }
  const uint4 su = *reinterpret_cast<const uint4 *>(suh + ks);
  const uint32_t ss[4] = {su.x, su.y, su.z, su.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = h2f(f2h(v[2 * i])) * h2f((uint16_t)(ss[i] & 0xFFFFu));
    v[2 * i + 1] = h2f(f2h(v[2 * i + 1])) * h2f((uint16_t)(ss[i] >> 16));
  }
#pragma unroll
  for (int b = 1; b < 8; b <<= 1)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if ((i & b) == 0) {
        const float lo = v[i], hi = v[i + b];
        v[i] = lo + hi;
        v[i + b] = lo - hi;
      }
#pragma unroll
  for (int bit = 1; bit <= 8; bit <<= 1) {
    const float sg = (j & bit) == 0 ? 1.0f : -1.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = butterfly(sg, v[i], xor_lanes(v[i], bit));
  }
  if (valid) {
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = (uint32_t)f2h(v[2 * i] * HAD_SCALE) | ((uint32_t)f2h(v[2 * i + 1] * HAD_SCALE) << 16);
    *reinterpret_cast<uint4 *>(xp + off) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

hipError_t launch_prepare(const void *x, int xdt, const uint16_t *suh, uint16_t *xp, int rows,
                          int in, hipStream_t s, int groups) {
  if (rows <= 0 || in <= 0 || in % 128 != 0 || groups <= 0) return hipErrorInvalidValue;
  if (rows > 65535) return hipErrorInvalidValue;
  const int nblk = in / 128;
  const size_t nblocks = (size_t)rows * nblk;
  const bool aligned = (((uintptr_t)x | (uintptr_t)suh | (uintptr_t)xp) & 15) == 0;
  if (aligned && nblocks * 16 < ((size_t)1 << 31)) {
    hipLaunchKernelGGL(prepare8_kernel<false>, dim3((unsigned)((nblocks + 15) / 16)), dim3(256), 0,
                       s, x, xdt, suh, xp, nblk, (uint32_t)nblocks, groups, SuhSets{});
    return hipGetLastError();
  }
  hipLaunchKernelGGL(prepare_kernel, dim3((nblk + 3) / 4, rows), dim3(256), 0, s, x, xdt, suh, xp,
                     in, nblk, groups);
  return hipGetLastError();
}

hipError_t launch_prepare_sets(const void *x, int xdt, const uint16_t *const *suh, int count,
                               uint16_t *xp, int rows, int in, hipStream_t s) {
  if (rows <= 0 || in <= 0 || in % 128 != 0 || count < 1 || count > 4) return hipErrorInvalidValue;
  const size_t nblocks = (size_t)rows * (in / 128);
  uintptr_t bits = (uintptr_t)x | (uintptr_t)xp;
  SuhSets sets{};
  for (int i = 0; i < count; ++i) {
    sets.p[i] = suh[i];
    bits |= (uintptr_t)suh[i];
  }
  if (count == 1 && rows <= 65535) return launch_prepare(x, xdt, suh[0], xp, rows, in, s, 1);
  if ((bits & 15) == 0 && nblocks * 16 < ((size_t)1 << 31)) {
    hipLaunchKernelGGL(prepare8_kernel<true>, dim3((unsigned)((nblocks + 15) / 16), count),
                       dim3(256), 0, s, x, xdt, suh[0], xp, in / 128, (uint32_t)nblocks, 1, sets);
    return hipGetLastError();
  }
  const size_t xsz = xdt == OUT_F32 ? 4 : 2;
  for (int i = 0; i < count; ++i)
    for (int r0 = 0; r0 < rows; r0 += 65535) {
      const hipError_t e =
          launch_prepare((const char *)x + (size_t)r0 * in * xsz, xdt, suh[i],
                         xp + ((size_t)i * rows + r0) * in, std::min(65535, rows - r0), in, s, 1);
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}

hipError_t launch_finish(const uint16_t *z, const uint16_t *svh, void *y, int ydt, int rows,
                         int out, hipStream_t s) {
  if (rows <= 0 || out <= 0 || out % 128 != 0 || rows > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(finish_kernel, dim3(out / 128, rows), dim3(64), 0, s, z, svh, y, ydt, out);
  return hipGetLastError();
}

// ============================================================ decode matrix

// One wave per (k-tile row tk, 8 consecutive output tiles): lane = 8*tile +
// chunk.  Decoded values are staged in LDS as the 16 x 128 row block and
// written out as contiguous rows of W_inner [in, out].
template <int K, int CB>
__global__ __launch_bounds__(64) void decode_matrix_kernel(const uint32_t *__restrict__ tw,
                                                           uint16_t *__restrict__ w, int out_tiles,
                                                           CbRow d) {
  __shared__ uint32_t blk[16 * 64];  // 16 rows x 128 f16, as dwords
  const int lane = threadIdx.x;
  const int tk = blockIdx.y, cg = blockIdx.x;
  const int tl = lane >> 3, c = lane & 7;
  const size_t tile = (size_t)tk * out_tiles + cg * 8 + tl;
  const uint32_t *tp = tw + tile * (8 * K);
  uint32_t wd[K + 1];
#pragma unroll
  for (int i = 0; i < K; ++i) wd[i + 1] = tp[c * K + i];
  wd[0] = tp[((c + 7) & 7) * K + (K - 1)];
  uint16_t *row16 = reinterpret_cast<uint16_t *>(blk);
  static_for<16>([&](auto P) {
    constexpr int p = decltype(P)::value;
    const uint32_t v = chunk_pair<K, CB, p>(wd, d);
    constexpr int r = chunk_row(2 * p);
    const int col = tl * 16 + c + 8 * chunk_colhalf(2 * p);
    row16[r * 128 + col] = (uint16_t)(v & 0xFFFFu);
    row16[(r + 1) * 128 + col] = (uint16_t)(v >> 16);
  });
  __syncthreads();
  const size_t out = (size_t)out_tiles * 16;
  // 16 rows x 64 dwords: lane writes dword `lane` of every row.
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    uint32_t *dst = reinterpret_cast<uint32_t *>(w + ((size_t)tk * 16 + r) * out + cg * 128);
    dst[lane] = blk[r * 64 + lane];
  }
}

// Any even n: the 8 tiles' dwords are staged in LDS and each lane extracts its
// 32 codewords with run-time windows.
template <int CB>
__global__ __launch_bounds__(64) void decode_matrix_generic_kernel(const uint32_t *__restrict__ tw,
                                                                   uint16_t *__restrict__ w,
                                                                   int out_tiles, int n,
                                                                   CbRow d) {
  __shared__ uint32_t words[8 * 64];
  __shared__ uint32_t blk[16 * 64];
  const int lane = threadIdx.x;
  const int tk = blockIdx.y, cg = blockIdx.x;
  const int nw = n >> 1;
  const uint32_t *src = tw + ((size_t)tk * out_tiles + cg * 8) * nw;
  for (int i = lane; i < 8 * nw; i += 64) words[i] = src[i];
  __syncthreads();
  const int tl = lane >> 3, c = lane & 7;
  const uint32_t *mine = words + tl * nw;
  uint16_t *row16 = reinterpret_cast<uint16_t *>(blk);
  for (int p = 0; p < 16; ++p) {
    const uint32_t t = 32u * c + 2u * p;
    const uint32_t v = decode_pair<CB>(tile_window(mine, n, t), tile_window(mine, n, t + 1u), d);
    const int r = chunk_row(2 * p);
    const int col = tl * 16 + c + 8 * chunk_colhalf(2 * p);
    row16[r * 128 + col] = (uint16_t)(v & 0xFFFFu);
    row16[(r + 1) * 128 + col] = (uint16_t)(v >> 16);
  }
  __syncthreads();
  const size_t out = (size_t)out_tiles * 16;
  for (int r = 0; r < 16; ++r) {
    uint32_t *dst = reinterpret_cast<uint32_t *>(w + ((size_t)tk * 16 + r) * out + cg * 128);
    dst[lane] = blk[r * 64 + lane];
  }
}

template <int CB>
static hipError_t decode_matrix_cb(const uint32_t *tw, const Format &f, int in, int out,
                                   uint16_t *w, hipStream_t s) {
  const dim3 grid(out / 128, in / 16);
  const int ot = out / 16;
  const CbRow m = f.dec();
  switch (f.integer_rate() ? f.n / 16 : 0) {
#define EXL3_DM(KK)                                                                             \
  case KK:                                                                                      \
    hipLaunchKernelGGL((decode_matrix_kernel<KK, CB>), grid, dim3(64), 0, s, tw, w, ot, m); \
    break;
    EXL3_DM(1) EXL3_DM(2) EXL3_DM(3) EXL3_DM(4) EXL3_DM(5) EXL3_DM(6) EXL3_DM(7) EXL3_DM(8)
#undef EXL3_DM
    default:
      hipLaunchKernelGGL((decode_matrix_generic_kernel<CB>), grid, dim3(64), 0, s, tw, w, ot, f.n,
                         m);
  }
  return hipGetLastError();
}

hipError_t launch_decode_matrix(const uint16_t *trellis, const Format &f, int in, int out,
                                uint16_t *w, hipStream_t s) {
  if (in <= 0 || out <= 0 || in % 16 != 0 || out % 128 != 0) return hipErrorInvalidValue;
  if (f.n < 16 || f.n > 128 || (f.n & 1)) return hipErrorInvalidValue;
  if (in / 16 > 65535) return hipErrorInvalidValue;
  const uint32_t *tw = reinterpret_cast<const uint32_t *>(trellis);
  switch (f.codebook) {
    case CB_MCG: return decode_matrix_cb<CB_MCG>(tw, f, in, out, w, s);
    case CB_HASH: return decode_matrix_cb<CB_HASH>(tw, f, in, out, w, s);
    case CB_PAIR1: return decode_matrix_cb<CB_PAIR1>(tw, f, in, out, w, s);
    default: return decode_matrix_cb<CB_MUL1>(tw, f, in, out, w, s);
  }
}

// Every state of a codebook, the table the load-time self-check hashes:
// w[s] = the weight codeword s decodes to (mul1, mcg, the hash-mask tables;
// 65536 f16), through the same device decode the GEMV and GEMM use (pairs of
// codewords, the window's mask applied first).  pair1 decodes a pair of
// weights from one codeword: w[2c], w[2c + 1] for codeword c (131072 f16).
template <int CB>
__global__ __launch_bounds__(256) void decode_states_kernel(uint16_t *__restrict__ w, CbRow d) {
  const uint32_t p = blockIdx.x * 256u + threadIdx.x;  // pair index
  uint32_t v;
  if constexpr (CB == CB_PAIR1)
    v = decode_pair<CB>(0u, p, d);
  else
    v = decode_pair<CB>(2u * p, 2u * p + 1u, d);
  reinterpret_cast<uint32_t *>(w)[p] = v;
}

hipError_t launch_decode_states(const Format &f, uint16_t *w, hipStream_t s) {
  const CbRow d = f.dec();
  switch (f.codebook) {
    case CB_MCG: hipLaunchKernelGGL(decode_states_kernel<CB_MCG>, dim3(128), dim3(256), 0, s, w, d); break;
    case CB_HASH: hipLaunchKernelGGL(decode_states_kernel<CB_HASH>, dim3(128), dim3(256), 0, s, w, d); break;
    case CB_PAIR1: hipLaunchKernelGGL(decode_states_kernel<CB_PAIR1>, dim3(256), dim3(256), 0, s, w, d); break;
    default: hipLaunchKernelGGL(decode_states_kernel<CB_MUL1>, dim3(128), dim3(256), 0, s, w, d);
  }
  return hipGetLastError();
}

// ------------------------------------------------------------ un-rotation

// W_public = diag(suh) H W_inner H diag(svh) / 128 per 128 x 128 block, in
// the reference's order (sushi_ds41/src/sushi/exl3/expert_exl3.zig:440-488,
// `reconstructPublic`): the dense Hadamard over the input index of every
// column (out[r] = sum_k e(r,k) * v[k], e = +-HAD_SCALE by the parity of
// r & k, products and sums in f32 in k order), times suh per row, the dense
// Hadamard over the output index of every row, times svh per column, then
// one rounding to the output type (f16: the reference's value bit for bit).
// e * v is +-(HAD_SCALE * v) exactly and acc + (-p) is acc - p, so each term
// is the scaled value added or subtracted.  A thread keeps 8 sums: rows (or
// columns) o0 + i, i < 8, o0 a multiple of 8, whose sign for k = k8 + j is
// parity(o0 & k8) ^ parity(i & j) -- the second term fixed at compile time.
constexpr int UNROT_THREADS = 256;
constexpr int UNROT_LD = 129;  // padded LDS row (floats)

__device__ __forceinline__ void unrot_eight(const float *hv, int stride, int o0, float (&acc)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
  for (int k8 = 0; k8 < 128; k8 += 8) {
    const uint32_t flip = (uint32_t)(__builtin_popcount((unsigned)(o0 & k8)) & 1) << 31;
    static_for<8>([&](auto J) {
      constexpr int j = decltype(J)::value;
      const float p = bits<float>(bits<uint32_t>(hv[(k8 + j) * stride]) ^ flip);
      static_for<8>([&](auto I) {
        constexpr int i = decltype(I)::value;
        if constexpr (__builtin_popcount(i & j) & 1)
          acc[i] = acc[i] - p;
        else
          acc[i] = acc[i] + p;
      });
    });
  }
}

__global__ __launch_bounds__(UNROT_THREADS) void unrotate_kernel(
    const uint16_t *__restrict__ w, const uint16_t *__restrict__ suh,
    const uint16_t *__restrict__ svh, void *__restrict__ dst, int out, int64_t ld, int ydt) {
  __shared__ __attribute__((aligned(16))) float lds[2 * 128 * UNROT_LD];  // 129 KiB
  float *A = lds;                    // HAD_SCALE * W_inner block [k][c]
  float *B = lds + 128 * UNROT_LD;   // HAD_SCALE * (column Hadamard * suh) [r][k]
  const int tid = threadIdx.x;
  const int rb = blockIdx.y * 128, cb = blockIdx.x * 128;
  for (int e = tid; e < 128 * 128; e += UNROT_THREADS) {
    const int r = e >> 7, c = e & 127;
    A[r * UNROT_LD + c] = f32_value(HAD_SCALE * h2f(w[(size_t)(rb + r) * out + cb + c]));
  }
  __syncthreads();
  {
    // input-index Hadamard: column c, rows o0 .. o0 + 7 at a time
    const int c = tid & 127;
    for (int o0 = (tid >> 7) * 8; o0 < 128; o0 += 16) {
      float acc[8];
      unrot_eight(A + c, UNROT_LD, o0, acc);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float v = f32_value(acc[i] * h2f(suh[rb + o0 + i]));
        B[(o0 + i) * UNROT_LD + c] = f32_value(HAD_SCALE * v);
      }
    }
  }
  __syncthreads();
  {
    // output-index Hadamard: row r, columns o0 .. o0 + 7 at a time
    const int r = tid & 127;
    for (int o0 = (tid >> 7) * 8; o0 < 128; o0 += 16) {
      float acc[8];
      unrot_eight(B + r * UNROT_LD, 1, o0, acc);
      const size_t base = (size_t)(rb + r) * ld + cb + o0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float v = f32_value(acc[i] * h2f(svh[cb + o0 + i]));
        if (ydt == OUT_F16)
          ((uint16_t *)dst)[base + i] = f2h(v);
        else if (ydt == OUT_BF16)
          ((uint16_t *)dst)[base + i] = f2bf(v);
        else
          ((float *)dst)[base + i] = v;
      }
    }
  }
}

hipError_t launch_unrotate(const uint16_t *w_inner, const uint16_t *suh, const uint16_t *svh,
                           int in, int out, void *dst, int64_t ld, int ydt, hipStream_t s) {
  if (in <= 0 || out <= 0 || in % 128 != 0 || out % 128 != 0 || ld < out) return hipErrorInvalidValue;
  if (in / 128 > 65535 || ydt < OUT_F16 || ydt > OUT_F32) return hipErrorInvalidValue;
  hipLaunchKernelGGL(unrotate_kernel, dim3(out / 128, in / 128), dim3(UNROT_THREADS), 0, s, w_inner,
                     suh, svh, dst, out, ld, ydt);
  return hipGetLastError();
}

static std::atomic<int> g_poll_bound{-1};
int splitk_poll_max() {
  const int v = g_poll_bound.load(std::memory_order_relaxed);
  return v >= 0 ? v : PARTIAL_POLL_MAX;
}
void set_splitk_poll_max(int polls) { g_poll_bound.store(polls, std::memory_order_relaxed); }
static std::atomic<int> g_splitk_drop{0};
int splitk_drop() { return g_splitk_drop.load(std::memory_order_relaxed); }
void set_splitk_drop(int on) { g_splitk_drop.store(on != 0, std::memory_order_relaxed); }

// k-splits of a GEMV: whole input Hadamard blocks per split, at most
// GEMV_KSPLIT_MAX splits and tps_max k-tile rows (GEMV_TPS_MAX; the generic
// rate's launchers clamp to 32 afterwards), GEMV_TPS_ONE_ROW_MAX at one or
// two rows.
// * Up to 4 rows, over at most 1024 workgroups: the split count that
//   balances the launch over the 256 CUs, the least (workgroups on the
//   busiest CU) x (blocks a workgroup), ties to fewer splits (fewer partial
//   sums and hand-offs).  Qwen3-8B at one row: q+k+v 16 splits of 2 blocks
//   (768 workgroups, against 11 of 3: 528, 16 CUs holding a third), o 8 of 4
//   (256), down 8 of 12 (256), gate+up 4 of 8 (768); the pass 1.7 % faster
//   than with ~512 workgroups a launch.
// * Else ~512 workgroups over `groups` column groups; above 4 rows at most
//   256 (one round: q+k+v 5 splits, 240 workgroups, against 6 and 288, 0.3 %
//   faster a decode step at 16 rows), whose split-K partial sums (rows x 128
//   floats per workgroup) would otherwise add half the weight bytes again.
void gemv_plan(int in, int out, int groups, int rows, int *ksplit, int *tps, int tps_max) {
  const int nb = in / 128;
  const int cgs = std::max(1, out / 128) * std::max(1, groups);
  if (rows <= 4) {
    const int cap = (rows <= 2 ? std::max(tps_max, GEMV_TPS_ONE_ROW_MAX) : tps_max) / 8;
    long best = -1;
    int bks = 0;
    for (int ks = 1; ks <= std::min(nb, GEMV_KSPLIT_MAX) && (long)cgs * ks <= 1024; ++ks) {
      const int bps = (nb + ks - 1) / ks;
      if (bps > cap || (nb + bps - 1) / bps != ks) continue;  // not the fewest splits of bps
      const long cost = (long)(((long)cgs * ks + 255) / 256) * bps;
      if (best < 0 || cost < best) {
        best = cost;
        bks = ks;
      }
    }
    if (bks > 0) {
      const int bps = (nb + bks - 1) / bks;
      *tps = 8 * bps;
      *ksplit = bks;
      return;
    }
  }
  const int target = rows > 4 ? 256 : 512;
  const int ks0 = std::min(nb, std::max(1, rows > 4 ? target / cgs : (target + cgs - 1) / cgs));
  auto split = [&](int cap, int *ks) {  // blocks per split and splits under a cap
    int bps = std::min(cap, (nb + ks0 - 1) / ks0);
    bps = std::max(bps, (nb + GEMV_KSPLIT_MAX - 1) / GEMV_KSPLIT_MAX);
    *ks = (nb + bps - 1) / bps;
    return bps;
  };
  int bps = split(tps_max / 8, ksplit);
  if (rows > 4 && groups == 1) {
    // longer splits, as far as the prepare's passes hold the rows, where they
    // take less time on the busiest CU: 12288 -> 4096 in 8 splits of 12
    // blocks, 256 workgroups, against 12 of 8, 384: an MLP of 6 rows 38.4 ->
    // 36.9 us.  (Two more prepare passes, for 16 rows of 12 blocks, measured
    // no faster a decode step of 16.)
    int ks2;
    const int bps2 = split(std::min(GEMV_TPS_ONE_ROW_MAX / 8, PREP_PASSES * PREP_GROUPS / rows), &ks2);
    auto cost = [&](int ks, int b) { return (((long)cgs * ks + 255) / 256) * b; };
    if (bps2 > bps && cost(ks2, bps2) < cost(*ksplit, bps)) {
      bps = bps2;
      *ksplit = ks2;
    }
  }
  *tps = 8 * bps;
}

int gemv_ksplit(int in, int out, int groups, int rows) {
  int ks, tps;
  gemv_plan(in, out, groups, rows, &ks, &tps, GEMV_TPS_MAX);
  return ks;
}

void gemv_multi_plan(int in, int total_out, bool generic, int rows, int *ksplit, int *tps) {
  gemv_plan(in, total_out, 1, rows, ksplit, tps, GEMV_TPS_MAX);
  if (generic && *tps > 32) {
    *tps = 32;
    *ksplit = (in / 16 + 31) / 32;
  }
}

// The GEMV kernels' rate of a format (their K): 1..8, -3 and -5 (n = 24, 40)
// or 0.  A half-integer rate's windows are as fixed as an integer rate's; with
// run-time windows out of LDS its GEMV ran 24.0 us on q + k + v of 4096 at n =
// 40, 3 rows, against 11.4.
static int gemv_rate(const Format &f) {
  return f.integer_rate() ? f.n / 16 : f.n == 24 ? -3 : f.n == 40 ? -5 : 0;
}

// Calls launch(integral_constant<int, K>) for K = kk in 1..8, -3, -5, else 0.
template <typename F>
static void rate_dispatch(int kk, F &&launch) {
  switch (kk) {
    case 1: launch(std::integral_constant<int, 1>{}); break;
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 3: launch(std::integral_constant<int, 3>{}); break;
    case 4: launch(std::integral_constant<int, 4>{}); break;
    case 5: launch(std::integral_constant<int, 5>{}); break;
    case 6: launch(std::integral_constant<int, 6>{}); break;
    case 7: launch(std::integral_constant<int, 7>{}); break;
    case 8: launch(std::integral_constant<int, 8>{}); break;
    case -3: launch(std::integral_constant<int, -3>{}); break;
    case -5: launch(std::integral_constant<int, -5>{}); break;
    default: launch(std::integral_constant<int, 0>{});
  }
}

static hipError_t gemv_multi(const GemvLinear *ls, int count, const Format &f, const void *x,
                             int xdt, bool prepared, int ydt, int rows, int in, Scratch *sc,
                             const GemvFuse &fz, hipStream_t s) {
  if (count < 1 || count > GEMV_MAXW || rows < 1 || rows > GEMV_ROWS_MAX) return hipErrorInvalidValue;
  if (in <= 0 || in % 128 != 0) return hipErrorInvalidValue;
  if (f.n < 16 || f.n > 128 || (f.n & 1)) return hipErrorInvalidValue;
  const bool generic = f.gemv_generic();
  int maxout = 0, totcg = 0;
  for (int i = 0; i < count; ++i) {
    if (ls[i].out <= 0 || ls[i].out % 128 != 0) return hipErrorInvalidValue;
    if (ls[i].y == nullptr && ls[i].zout == nullptr && fz.res == nullptr) return hipErrorInvalidValue;
    maxout = std::max(maxout, ls[i].out);
    totcg += ls[i].out / 128;
  }
  if ((int64_t)rows * std::max(in, maxout) >= (int64_t)1 << 31) return hipErrorInvalidValue;
  int ksplit, tps;
  gemv_multi_plan(in, 128 * totcg, generic, rows, &ksplit, &tps);
  if (ksplit > GEMV_KSPLIT_MAX || totcg > 65535) return hipErrorInvalidValue;
  if (in / 16 > 65535) return hipErrorInvalidValue;
  GemvArgs a{};
  const uint32_t *tw[GEMV_MAXW] = {nullptr, nullptr, nullptr, nullptr};
  int cgs[GEMV_MAXW] = {0, 0, 0, 0};
  int cg0 = 0;
  for (int i = 0; i < count; ++i) {
    GemvWeight &w = a.w[i];
    tw[i] = reinterpret_cast<const uint32_t *>(ls[i].trellis);
    w.suh = ls[i].suh;
    w.svh = ls[i].svh;
    w.y = ls[i].y;
    w.zout = ls[i].zout;
    w.expert_words = 0;
    cgs[i] = cg0;
    cg0 += ls[i].out / 128;
    if (ksplit > 1) {
      if (sc[i].partial == nullptr || sc[i].partial_floats < (size_t)ksplit * rows * ls[i].out)
        return hipErrorInvalidValue;
    }
    w.partial = sc[i].partial;
  }
  if (ksplit > 1 && sc[0].status == nullptr) return hipErrorInvalidValue;
  // the unused trellis arguments carry suh pointers, which gemv_kernel's
  // workgroups read without waiting for the argument segment
  if (count == 1) {
    tw[1] = reinterpret_cast<const uint32_t *>(ls[0].suh);
  } else if (count == 2) {
    tw[2] = reinterpret_cast<const uint32_t *>(ls[0].suh);
    tw[3] = reinterpret_cast<const uint32_t *>(ls[1].suh);
  } else if (count == 3) {
    tw[3] = reinterpret_cast<const uint32_t *>(ls[0].suh);
  }
  a.c.status = sc[0].status;
  a.c.poll_max = splitk_poll_max();
  a.c.drop_partials = splitk_drop();
  a.c.ydt = ydt;
  a.c.ptotal = (size_t)rows;
  a.c.ksplit = ksplit;
  a.c.dec = f.dec();
  a.c.nw = f.n / 2;
  a.c.x2 = fz.up;
  a.c.limit = fz.limit;
  a.c.nssq = fz.nssq;
  a.c.nw_norm = fz.norm_w;
  a.c.eps = fz.eps;
  a.c.res = fz.res;
  a.c.res_ssq = fz.res_ssq;
  a.c.attn_part = fz.attn_part;
  a.c.attn_nkv = fz.attn_nkv;
  a.c.attn_g = fz.attn_g;
  a.c.attn_nsplit = fz.attn_nsplit;
  GemvGeo geo{};
  geo.cg1 = cgs[1];
  geo.cg2 = cgs[2];
  geo.cg3 = cgs[3];
  geo.cgend = totcg;
  geo.rows = rows;
  geo.xdt = xdt;
  geo.prepared = prepared || fz.stacked ? 1 : 0;
  geo.stacked = fz.stacked ? 1 : 0;
  geo.in_tiles = in / 16;
  geo.tps = tps;
  uint32_t g0, g1, g2;
  if (!gemv_geo_pack(geo, &g0, &g1, &g2)) return hipErrorInvalidValue;
  const size_t lds = gemv_lds_bytes(rows, tps, generic);
  const dim3 grid(totcg, ksplit);
  const int prep = gemv_prep_form(rows, tps);
  const bool oneb = prep == 0;
  if (fz.nssq != nullptr &&
      (!oneb || xdt != OUT_F32 || prepared || fz.norm_w == nullptr || in / 128 > NORM_MAXBLK))
    return hipErrorInvalidValue;
  if (fz.res != nullptr && (count != 1 || fz.res_ssq == nullptr)) return hipErrorInvalidValue;
  if (fz.stacked && (xdt != OUT_F16 || fz.nssq != nullptr || fz.up != nullptr ||
                     fz.attn_part != nullptr))
    return hipErrorInvalidValue;
  if (fz.attn_part != nullptr &&
      (!oneb || count != 1 || xdt != OUT_F16 || prepared || fz.nssq != nullptr ||
       fz.up != nullptr || fz.attn_nkv < 1 || fz.attn_g < 1 || fz.attn_nsplit < 1 ||
       in != fz.attn_nkv * fz.attn_g * 128))
    return hipErrorInvalidValue;
  rate_dispatch(gemv_rate(f), [&](auto KC) {
    gemv_go<decltype(KC)::value>(f, prep, grid, lds, s, tw, x, g0, g1, g2, a);
  });
  return hipGetLastError();
}

hipError_t launch_gemv_multi(const GemvLinear *ls, int count, const Format &f, const void *x,
                             int xdt, bool prepared, int ydt, int rows, int in, Scratch *sc,
                             hipStream_t s) {
  return gemv_multi(ls, count, f, x, xdt, prepared, ydt, rows, in, sc, GemvFuse{}, s);
}

hipError_t launch_gemv_fused(const GemvLinear *ls, int count, const Format &f, const void *x,
                             int xdt, int ydt, int rows, int in, Scratch *sc, const GemvFuse &fz,
                             hipStream_t s) {
  if (fz.up != nullptr && (xdt != OUT_F16 || fz.nssq != nullptr)) return hipErrorInvalidValue;
  return gemv_multi(ls, count, f, x, xdt, false, ydt, rows, in, sc, fz, s);
}

namespace {
// h = f16(silu(g) * u) elementwise (the prologue's arithmetic, swiglu1).
// h = f16(silu(g) * u) and its prepare with suh (the consumer's), in one
// pass: a 16-lane group per 128-block of the flattened [rows][in] (in a
// multiple of 128), 8 elements a lane; the prepared rows equal what the
// GEMV prologue forms from h (prep_block8).  Groups past the last block
// redo the last one (whole waves), storing nothing.
__global__ __launch_bounds__(256) void swiglu_prepare_kernel(const uint16_t *__restrict__ g,
                                                             const uint16_t *__restrict__ u,
                                                             const uint16_t *__restrict__ suh,
                                                             uint16_t *__restrict__ xp, int nblk,
                                                             uint32_t nblocks, float limit) {
  const int j = threadIdx.x & 15;
  const uint32_t gb0 = blockIdx.x * 16u + (threadIdx.x >> 4);
  const bool valid = gb0 < nblocks;
  const uint32_t gb = valid ? gb0 : nblocks - 1;
  const size_t off = (size_t)gb * 128 + 8 * j;
  const int k = (int)(gb % (uint32_t)nblk) * 128 + 8 * j;
  const uint4 gv = *reinterpret_cast<const uint4 *>(g + off);
  const uint4 uv = *reinterpret_cast<const uint4 *>(u + off);
  const uint4 su = *reinterpret_cast<const uint4 *>(suh + k);
  const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w}, uw[4] = {uv.x, uv.y, uv.z, uv.w};
  uint32_t h[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    h[i] = (uint32_t)f2h(swiglu1((uint16_t)(gw[i] & 0xFFFFu), (uint16_t)(uw[i] & 0xFFFFu), limit)) |
           ((uint32_t)f2h(swiglu1((uint16_t)(gw[i] >> 16), (uint16_t)(uw[i] >> 16), limit)) << 16);
  const uint4 o = prep_block8(h, su, j);
  if (valid) *reinterpret_cast<uint4 *>(xp + off) = o;
}

__global__ __launch_bounds__(256) void swiglu_kernel(const uint16_t *__restrict__ g,
                                                     const uint16_t *__restrict__ u,
                                                     uint16_t *__restrict__ h, size_t n,
                                                     float limit) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    h[i] = f2h(swiglu1(g[i], u[i], limit));
}
}  // namespace

hipError_t launch_gemv_swiglu(const GemvLinear &l, const Format &f, const uint16_t *g,
                              const uint16_t *u, uint16_t *h, float limit, int ydt, int rows,
                              int in, Scratch &sc, hipStream_t s) {
  if (g == nullptr || u == nullptr || !(limit >= 0.0f)) return hipErrorInvalidValue;
  if (rows <= SWIGLU_PROLOGUE_ROWS) {
    GemvFuse fz{};
    fz.up = u;
    fz.limit = limit;
    return gemv_multi(&l, 1, f, g, OUT_F16, false, ydt, rows, in, &sc, fz, s);
  }
  // more rows: every column group would redo the rows' SwiGLU and prepare,
  // so both run once here, into prepared rows
  if (h == nullptr) return hipErrorInvalidValue;
  hipError_t e = launch_swiglu_prepare(g, u, l.suh, h, rows, in, limit, s);
  if (e != hipSuccess) return e;
  GemvFuse fz{};
  fz.stacked = true;
  return gemv_multi(&l, 1, f, h, OUT_F16, false, ydt, rows, in, &sc, fz, s);
}

hipError_t launch_swiglu(const uint16_t *g, const uint16_t *u, uint16_t *h, size_t n, float limit,
                         hipStream_t s) {
  if (n == 0 || !(limit >= 0.0f)) return hipErrorInvalidValue;
  const size_t blocks = std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(swiglu_kernel, dim3((unsigned)blocks), dim3(256), 0, s, g, u, h, n, limit);
  return hipGetLastError();
}

hipError_t launch_swiglu_prepare(const uint16_t *g, const uint16_t *u, const uint16_t *suh,
                                 uint16_t *xp, int rows, int in, float limit, hipStream_t s) {
  if (rows <= 0 || in <= 0 || in % 128 != 0 || !(limit >= 0.0f) || suh == nullptr)
    return hipErrorInvalidValue;
  const int nblk = in / 128;
  const uint32_t nblocks = (uint32_t)rows * (uint32_t)nblk;
  hipLaunchKernelGGL(swiglu_prepare_kernel, dim3((nblocks + 15) / 16), dim3(256), 0, s, g, u, suh,
                     xp, nblk, nblocks, limit);
  return hipGetLastError();
}

bool gemv_one_batch(int in, int total_out, bool generic, int rows) {
  int ks, tps;
  gemv_multi_plan(in, total_out, generic, rows, &ks, &tps);
  return rows * (tps / 8) <= PREP_ITEMS;
}

hipError_t launch_gemv(const uint16_t *trellis, const Format &f, const void *x, int xdt,
                       bool prepared, const uint16_t *suh, const uint16_t *svh, void *y, int ydt,
                       uint16_t *zout, int rows, int in, int out, Scratch &sc, hipStream_t s) {
  GemvLinear l{trellis, suh, svh, y, zout, out};
  return launch_gemv_multi(&l, 1, f, x, xdt, prepared, ydt, rows, in, &sc, s);
}


namespace {
// The end of a split-K GEMM: z = f16(sum of the S planes of kpart, in split
// order), then the finish (Hadamard-128 in the reference's stage order,
// * 1/sqrt(128) * svh, as the GEMV's) or z itself.  One wave per row, lane l
// columns 2 l, 2 l + 1 of the block's 128.
__global__ __launch_bounds__(512) void gemm_splitk_finish_kernel(
    const float *__restrict__ part, int S, int M, int out, const uint16_t *__restrict__ svh,
    void *__restrict__ y, int ydt, uint16_t *__restrict__ zout) {
  const int cg = blockIdx.x, lane = threadIdx.x & 63;
  const int m = blockIdx.y * 8 + (threadIdx.x >> 6);
  if (m >= M) return;
  const size_t plane = (size_t)M * out;
  const float *p = part + (size_t)m * out + cg * 128 + 2 * lane;
  float s0 = 0.0f, s1 = 0.0f;
#pragma unroll 8
  for (int k = 0; k < S; ++k) {
    const float2 v = *reinterpret_cast<const float2 *>(p + (size_t)k * plane);
    s0 += v.x;
    s1 += v.y;
  }
  float v0 = h2f(f2h(s0)), v1 = h2f(f2h(s1));
  const size_t o = (size_t)m * out + cg * 128 + 2 * lane;
  if (y == nullptr) {
    zout[o] = f2h(v0);
    zout[o + 1] = f2h(v1);
    return;
  }
  had128_pair(v0, v1, lane);
  const float sv0 = h2f(svh[cg * 128 + 2 * lane]), sv1 = h2f(svh[cg * 128 + 2 * lane + 1]);
  store_out2(y, o, f2h(v0 * HAD_SCALE * sv0), f2h(v1 * HAD_SCALE * sv1), ydt);
}
}  // namespace

// Split-K of a GEMM whose tiles fill at most half the GPU: S splits (an
// even run of stages each), the most that keep tiles x S within one round
// of the 256 CUs (one workgroup a CU: its LDS); their f32 sums take S planes
// of rows x out floats.  A partial second round costs a whole split's time
// (gate+up at 128 rows: 96 tiles, 45.7 us a call in 2 splits against 57.3 in
// 3, 288 workgroups).  Above 128 tiles the planes' traffic costs more than
// the idle CUs (gate+up at 512 rows: 192 tiles, 547 TFLOP/s split in two
// against 629 whole).
GemmSplit gemm_split(int rows, int in, int out) {
  GemmSplit g;
  const int mblocks = (rows + GM_BM - 1) / GM_BM;
  const int tiles = ((out + GM_BN - 1) / GM_BN) * mblocks;
  const int pairs = in / 16 / 4 / 2;  // stage pairs
  int S = tiles > GM_SPLIT_TILES ? 1 : 256 / tiles;
  S = std::max(1, std::min(S, std::min(pairs, GM_SPLIT_MAX)));
  g.splits = S;
  g.tiles = tiles;
  g.part_floats = S > 1 ? (size_t)S * rows * out : 0;
  return g;
}

// The most rows one GEMM launch takes: the kernel addresses a launch's
// activations with 32-bit byte offsets, so a call past that runs as windows
// of whole row tiles, each its own launch (rows are independent: the same
// results).
static int64_t gemm_window_rows(int in) {
  return std::max<int64_t>(GM_BM, (int64_t)(0xFFFFFFFFull / ((uint64_t)in * 2)) / GM_BM * GM_BM);
}

size_t gemm_kpart_floats(int64_t rows, int in, int out) {
  const int64_t wmax = gemm_window_rows(in);
  const int64_t last = rows > wmax ? (rows - 1) % wmax + 1 : rows;
  size_t need = gemm_split((int)std::min(rows, wmax), in, out).part_floats;
  return std::max(need, gemm_split((int)last, in, out).part_floats);
}

hipError_t launch_gemm(const uint16_t *trellis, const Format &f, const uint16_t *xp,
                       const uint16_t *svh, void *y, int ydt, uint16_t *zout, int rows, int in,
                       int out, float *kpart, size_t kpart_floats, hipStream_t s) {
  if (rows < 1 || in <= 0 || out <= 0 || in % 128 != 0 || out % 128 != 0) return hipErrorInvalidValue;
  if (!f.gemm_rate()) return hipErrorInvalidValue;
  if (y == nullptr && zout == nullptr) return hipErrorInvalidValue;
  const int64_t wmax = gemm_window_rows(in);
  if (rows > wmax) {
    const size_t ysz = ydt == OUT_F32 ? 4 : 2;
    for (int64_t r0 = 0; r0 < rows; r0 += wmax) {
      const int r = (int)std::min<int64_t>(wmax, rows - r0);
      const hipError_t e = launch_gemm(
          trellis, f, xp + (size_t)r0 * in, svh, y ? (char *)y + (size_t)r0 * out * ysz : nullptr,
          ydt, zout ? zout + (size_t)r0 * out : nullptr, r, in, out, kpart, kpart_floats, s);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  const int mblocks = (rows + GM_BM - 1) / GM_BM;
  if (mblocks > 65535) return hipErrorInvalidValue;
  const GemmSplit sp = gemm_split(rows, in, out);
  if (sp.splits > 1 && (kpart == nullptr || kpart_floats < sp.part_floats))
    return hipErrorInvalidValue;
  if (sp.splits > 1 && (rows + 7) / 8 > 65535) return hipErrorInvalidValue;
  const dim3 grid((out + GM_BN - 1) / GM_BN, mblocks, sp.splits);
  const uint32_t *tw = reinterpret_cast<const uint32_t *>(trellis);
  const int it = in / 16, ot = out / 16;
  if (f.n == 24)
    gemm_frac_go<3>(f, grid, s, tw, xp, svh, y, ydt, zout, rows, it, ot, kpart);
  else if (f.n == 40)
    gemm_frac_go<5>(f, grid, s, tw, xp, svh, y, ydt, zout, rows, it, ot, kpart);
  else
    rate_dispatch(f.n / 16, [&](auto KC) {
      constexpr int K = decltype(KC)::value;
      if constexpr (K > 0) gemm_go<K>(f, grid, s, tw, xp, svh, y, ydt, zout, rows, it, ot, kpart);
    });
  if (sp.splits > 1)
    hipLaunchKernelGGL(gemm_splitk_finish_kernel, dim3(out / 128, (rows + 7) / 8), dim3(512), 0, s,
                       kpart, sp.splits, rows, out, svh, y, ydt, zout);
  return hipGetLastError();
}

// ------------------------------------------------- register-decode GEMM

namespace {
// gemm_splitk_finish_kernel over the launch's linears (column groups side by
// side in grid x).
__global__ __launch_bounds__(512) void gemm_rd_finish_kernel(RdArgs a, int S) {
  const int lane = threadIdx.x & 63;
  const int m = blockIdx.y * 8 + (threadIdx.x >> 6);
  if (m >= a.M) return;
  int wi = 0, c0 = 0;
#pragma unroll
  for (int i = 0, c = 0; i < RD_MAXW; ++i) {
    if (i < a.nw && (int)blockIdx.x >= c) {
      wi = i;
      c0 = c;
    }
    c += a.w[i].out_tiles / 8;
  }
  const RdWeight &W = a.w[wi];
  const int col = ((int)blockIdx.x - c0) * 128 + 2 * lane;
  const size_t out = (size_t)W.out_tiles * 16, plane = (size_t)a.M * out, o = (size_t)m * out + col;
  const float *p = W.kpart + o;
  float s0 = 0.0f, s1 = 0.0f;
#pragma unroll 8
  for (int k = 0; k < S; ++k) {
    const float2 v = *reinterpret_cast<const float2 *>(p + (size_t)k * plane);
    s0 += v.x;
    s1 += v.y;
  }
  float v0 = h2f(f2h(s0)), v1 = h2f(f2h(s1));
  if (W.y == nullptr) {
    W.zout[o] = f2h(v0);
    W.zout[o + 1] = f2h(v1);
    return;
  }
  had128_pair(v0, v1, lane);
  store_out2(W.y, o, f2h(v0 * HAD_SCALE * h2f(W.svh[col])),
             f2h(v1 * HAD_SCALE * h2f(W.svh[col + 1])), a.ydt);
}

// Row blocks by the rows (a tile of 128 from 65 on); k-splits to about one
// workgroup a CU (two and more k-part stages a split), which is what the
// planes' traffic and the finish launch allow: 4096 -> 12288 at 40 rows in 2 /
// 4 / 5 / 8 splits 33.9 / 27.0 / 26.2 / 30.8 us.
struct GemmRdPlan {
  int shape, ct, mtiles, splits;
  size_t part_floats;
};
GemmRdPlan gemm_rd_plan(int rows, int in, const int *outs, int count) {
  GemmRdPlan g{};
  g.shape = rows <= 32 ? 0 : rows <= 64 ? 1 : 2;
  const RdShape t = RD_SHAPES[g.shape];
  g.mtiles = (rows + 32 * t.mr - 1) / (32 * t.mr);
  size_t plane = 0;  // floats of one split
  for (int i = 0; i < count; ++i) {
    g.ct += (outs[i] + 64 * t.cw - 1) / (64 * t.cw);
    plane += (size_t)rows * outs[i];
  }
  const int tiles = g.ct * g.mtiles;
  int S = tiles > 128 ? 1 : std::max(1, std::min(256 / tiles, in / 128 / 4));
  // planes within the no-alloc matmul's staging beside the call's prepared
  // rows, whatever scratch the caller has: every entry splits a shape alike
  const size_t xp = ((size_t)rows * in * 2 + 255) & ~(size_t)255;
  const size_t stage = NOALLOC_BYTES - NOALLOC_SLOT_BYTES;
  const size_t room = xp < stage ? stage - xp : 0;
  while (S > 1 && (size_t)S * plane * 4 > room) --S;
  g.splits = S;
  g.part_floats = S > 1 ? (size_t)S * plane : 0;
  return g;
}
}  // namespace

// Against the 256 x 128 tiles, ratios of a call's time (prepare included,
// weights rotated), rates n = 16 .. 128 from row to row:
// * one linear: its splits' planes and its finish launch have to pay, and every
//   128 rows decode the weights once more, so what counts is in x out.  In x
//   out = 2^25 (4096 -> 8192, 8192 -> 4096): 17 / 32 / 64 / 96 rows 0.77-0.85 /
//   0.83-0.93 / 0.97-1.18 / 1.06-1.31; 1.5 x that (4096 -> 12288, 12288 -> 4096):
//   64 / 65 / 96 / 128 rows 0.81-0.97 / 0.91-1.07 / 0.92-1.09 / 0.92-1.08, above
//   1.02 at n < 40 (and past 96 rows into 4096); 2 x (4096 -> 16384, 8192 ->
//   8192): 0.71-0.92 / 0.84-1.03 / 0.84-1.00 / 0.86-1.01; 4 x: at most 0.86.
// * several linears, which the other kernel runs one after the other: while the
//   256 x 128 tiles of them all are at most 192 (0.32-0.96; q + k + v of 4096 at
//   17 / 1024 rows 0.44-0.49 / 0.70-0.75, gate + up of 12288 at 17 / 256 rows
//   0.47-0.54 / 0.79-0.91; 240 tiles of 3 x 640: 1.06-1.11, 384 of 2 x 12288:
//   1.04-1.14) and the workgroups here fill the CUs once (128 x 256 tiles: narrow
//   linears of an odd number of 128 columns waste half a tile; 4 x 128 columns
//   in 256 / 384 workgroups 0.76-0.80 / 1.03-1.07, 384 + 128 in 240 / 288
//   0.94-0.96 / 1.25-1.28).  At 7 and 8 bits past 1024 rows to 120 tiles (128
//   and 136 tiles at 2048 rows: 1.06, 1.03).
// Inputs past its 65535 k-tiles keep the 256 x 128 tiles.
bool gemm_rd_takes(int64_t rows, int in, const int *outs, int count, int n) {
  if (in / 16 > 65535) return false;
  if (count == 1) {
    const int64_t w = (int64_t)in * outs[0], u = (int64_t)1 << 24;
    if (rows <= 32) return w >= 2 * u;
    if (rows <= 64) return w >= 3 * u;
    return rows <= (outs[0] >= 8192 ? 128 : 96) && w >= (n < 40 ? 4 : 3) * u;
  }
  int64_t tiles = 0, wgs = 0;
  for (int i = 0; i < count; ++i) {
    tiles += (outs[i] / 128) * ((rows + 255) / 256);
    wgs += ((outs[i] + 255) / 256) * ((rows + 127) / 128);
  }
  return tiles <= (n > 96 && rows > 1024 ? 120 : 192) && wgs <= 256 &&
         (uint64_t)rows * in * 2 <= 0xFFFFFFFFull;
}

size_t gemm_rd_kpart_floats(int rows, int in, const int *outs, int count) {
  return gemm_rd_plan(rows, in, outs, count).part_floats;
}

hipError_t launch_gemm_rd(const GemmLinear *ls, int count, const Format &f, int ydt, int rows,
                          int in, float *kpart, size_t kpart_floats, hipStream_t s) {
  if (count < 1 || count > GEMM_RD_MAXW || rows < 1 || in <= 0 || in % 128 != 0 ||
      in / 16 > 65535 || !f.gemm_rate())
    return hipErrorInvalidValue;
  // activation offsets (bytes from xp) and a stage's word offsets are 32-bit
  if ((size_t)rows * in * 2 > 0xFFFFFFFFu) return hipErrorInvalidValue;
  int outs[GEMM_RD_MAXW], cgs = 0;
  for (int i = 0; i < count; ++i) {
    outs[i] = ls[i].out;
    if (ls[i].out <= 0 || ls[i].out % 128 != 0 || (ls[i].y == nullptr && ls[i].zout == nullptr) ||
        (((uintptr_t)ls[i].trellis | (uintptr_t)ls[i].xp) & 15) != 0 ||
        (size_t)4 * (ls[i].out / 16) * f.n * 2 > 0xFFFFFFFFu)
      return hipErrorInvalidValue;
    cgs += ls[i].out / 128;
  }
  const GemmRdPlan g = gemm_rd_plan(rows, in, outs, count);
  if (g.mtiles > 65535 || (rows + 7) / 8 > 65535) return hipErrorInvalidValue;
  if (g.splits > 1 && (kpart == nullptr || kpart_floats < g.part_floats)) return hipErrorInvalidValue;
  RdArgs a{};
  a.nw = count;
  a.ydt = ydt;
  a.M = rows;
  a.in_tiles = in / 16;
  a.dec = f.dec();
  int ct = 0;
  for (int i = 0; i < count; ++i) {
    a.w[i] = RdWeight{reinterpret_cast<const uint32_t *>(ls[i].trellis), ls[i].xp, ls[i].svh,
                      ls[i].y, ls[i].zout, kpart, ls[i].out / 16, ct};
    ct += (ls[i].out + 64 * RD_SHAPES[g.shape].cw - 1) / (64 * RD_SHAPES[g.shape].cw);
    if (g.splits > 1) kpart += (size_t)g.splits * rows * ls[i].out;
  }
  const dim3 grid(g.ct, g.mtiles, g.splits);
  if (f.n == 24)
    gemm_rd_go<1, 3>(f, g.shape, grid, s, a);
  else if (f.n == 40)
    gemm_rd_go<1, 5>(f, g.shape, grid, s, a);
  else
    rate_dispatch(f.n / 16, [&](auto KC) {
      constexpr int K = decltype(KC)::value;
      if constexpr (K > 0) gemm_rd_go<K, 0>(f, g.shape, grid, s, a);
    });
  if (g.splits > 1)
    hipLaunchKernelGGL(gemm_rd_finish_kernel, dim3(cgs, (rows + 7) / 8), dim3(512), 0, s, a,
                       g.splits);
  return hipGetLastError();
}

// A grouped linear's prefill: the grouped GEMM over every group's row tiles
// in one launch, items formed from the grid (GemmGroup.groups), each
// group's trellis and svh at its index in the G-bank, the finish fused.
hipError_t launch_gemm_groups(const uint16_t *trellis, const Format &f, const uint16_t *xp,
                              const uint16_t *svh, void *y, int ydt, int rows, int groups,
                              int in, int out, hipStream_t s) {
  if (rows < 1 || groups < 1 || in <= 0 || out <= 0 || in % 128 != 0 || out % 128 != 0)
    return hipErrorInvalidValue;
  if (!f.integer_rate() || y == nullptr) return hipErrorInvalidValue;
  // activation offsets (bytes from xp) are 32-bit in the kernel
  if ((size_t)rows * groups * in * 2 > 0xFFFFFFFFu) return hipErrorInvalidValue;
  const size_t tiles_y = (size_t)groups * ((rows + GM_BM - 1) / GM_BM);
  if (tiles_y > 65535) return hipErrorInvalidValue;
  GemmGroup gg{nullptr, nullptr, nullptr, (size_t)(in / 16) * (out / 16) * (f.n / 2), groups, rows};
  const dim3 grid(out / GM_BN, (unsigned)tiles_y);
  const uint32_t *tw = reinterpret_cast<const uint32_t *>(trellis);
  rate_dispatch(f.n / 16, [&](auto KC) {
    constexpr int K = decltype(KC)::value;
    if constexpr (K > 0) gemm_grouped_go<K>(f, grid, s, tw, xp, svh, y, ydt, in / 16, out / 16, gg);
  });
  return hipGetLastError();
}

// ====================================================================== MoE
//
// Routed SwiGLU experts (sushi_ds41/src/sushi/exl3/expert_exl3_kernels.zig:
// 3151-3206 for the arithmetic; decode chain :2765-3113):
//   1. route: one workgroup counts the (row, k) slots per expert, orders the
//      slots by expert (within an expert in any order: every slot's
//      arithmetic is independent of its position) and emits work items of
//      up to 4 slots of one expert (of 64, 128 or 256 where moe_gemm takes a
//      grouped GEMM, which then stands for the GEMVs);
//   2. grouped GEMV, gate and up in one launch: each work item is the GEMV
//      workgroup above over its expert's packed weights for its slots, the
//      prepare (x[row] * suh[e]) fused, split-K with the fused finish,
//      giving g and u (f16) per slot;
//   3. mid: h = silu(g) * u in f32 (limit > 0: g <= limit, |u| <= limit,
//      turboexl3_ds41/src/exl3/kernels/exl3/q3_exl3_prep_gu_epi.metal:47-56),
//      then the down projection's prepare with suh_down[e];
//   4. grouped GEMV down on the prepared rows, finished per slot (f16);
//   5. combine: y[row] = sum_k score[row, k] * d[slot(row, k)] in f32, in k
//      order, then the output dtype.


constexpr int MOE_ROUTE_THREADS = 1024;

// Exclusive prefix sum over the 1024 threads of a block; *total gets the sum.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t *tmp,
                                                         uint32_t *total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t inc = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t t = __shfl_up(inc, d, 64);
    if (lane >= d) inc += t;
  }
  if (lane == 63) tmp[wave] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t run = 0;
    for (int w = 0; w < MOE_ROUTE_THREADS / 64; ++w) {
      const uint32_t t = tmp[w];
      tmp[w] = run;
      run += t;
    }
    *total = run;
  }
  __syncthreads();
  const uint32_t r = tmp[wave] + inc - v;
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(MOE_ROUTE_THREADS) void moe_route_kernel(
    const uint32_t *__restrict__ inds, int slots, int experts, uint32_t *__restrict__ sorted,
    MoeItem *__restrict__ items, uint32_t *__restrict__ n_items, uint32_t item_rows) {
  __shared__ uint32_t cnt[MOE_ROUTE_THREADS], cur[MOE_ROUTE_THREADS], tmp[MOE_ROUTE_THREADS / 64];
  __shared__ uint32_t total;
  const int t = threadIdx.x;
  cnt[t] = 0;
  __syncthreads();
  for (int s = t; s < slots; s += MOE_ROUTE_THREADS) {
    const uint32_t e = inds ? inds[s] : 0u;
    if (e < (uint32_t)experts) atomicAdd(&cnt[e], 1u);
  }
  __syncthreads();
  const uint32_t c = t < experts ? cnt[t] : 0u;
  const uint32_t off = block_exclusive_scan(c, tmp, &total);
  const uint32_t nit = (c + item_rows - 1) / item_rows;
  const uint32_t ioff = block_exclusive_scan(nit, tmp, &total);
  cur[t] = off;
  __syncthreads();
  for (int s = t; s < slots; s += MOE_ROUTE_THREADS) {
    const uint32_t e = inds ? inds[s] : 0u;
    if (e < (uint32_t)experts) sorted[atomicAdd(&cur[e], 1u)] = (uint32_t)s;
  }
  for (uint32_t r = 0; r < nit; ++r) {
    MoeItem it;
    it.expert = (uint32_t)t;
    it.start = off + r * item_rows;
    it.count = min(item_rows, c - r * item_rows);
    it.pad = 0;
    items[ioff + r] = it;
  }
  if (t == 0) *n_items = total;
}

// Eight consecutive elements at element i of a 2-byte array as dwords; wide:
// the array is 16-byte aligned (i a multiple of 8).
__device__ __forceinline__ uint4 load8_16(const uint16_t *p, size_t i, bool wide) {
  if (wide) return *reinterpret_cast<const uint4 *>(p + i);
  uint32_t w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = (uint32_t)p[i + 2 * e] | ((uint32_t)p[i + 2 * e + 1] << 16);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// The grouped GEMM's gate and up inputs: slot s's row x[s / topk] prepared
// with expert e = inds[s]'s suh of each (as prepare8_kernel: f16(x) * suh,
// Hadamard-128, * 1/sqrt(128), f16), 16 lanes a 128-block of the flattened
// [slots][in / 128].  Bound by its writes (2 x slots x in f16): 16-byte
// accesses, 1024 tokens x top 8 of 7168: 157 -> 88 us against a wave per
// block and 4-byte accesses.  wide: x and both suh are 16-byte aligned.
__global__ __launch_bounds__(256) void moe_prep_kernel(const void *__restrict__ x, int xdt,
                                                       const uint32_t *__restrict__ inds,
                                                       int experts, int topk,
                                                       const uint16_t *__restrict__ suh_g,
                                                       const uint16_t *__restrict__ suh_u,
                                                       uint16_t *__restrict__ xg,
                                                       uint16_t *__restrict__ xu, int in,
                                                       uint32_t nblocks, int wide) {
  const int j = threadIdx.x & 15;
  const uint32_t gb0 = blockIdx.x * 16u + (threadIdx.x >> 4);
  const uint32_t gb = min(gb0, nblocks - 1);  // past the last: redone, not stored
  const uint32_t nblk = (uint32_t)in / 128u;
  const uint32_t slot = gb / nblk;
  const int k = (int)(gb - slot * nblk) * 128 + 8 * j;
  const uint32_t e0 = inds[slot];
  const bool valid = gb0 < nblocks && e0 < (uint32_t)experts;
  const size_t e = valid ? e0 : 0;  // (all lanes take part in the exchanges)
  const size_t xo = (size_t)(slot / (uint32_t)topk) * in + k;
  uint32_t h[4];
  if (xdt == OUT_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      h[i] = (uint32_t)f2h(((const float *)x)[xo + 2 * i]) |
             ((uint32_t)f2h(((const float *)x)[xo + 2 * i + 1]) << 16);
  } else {
    const uint4 w = load8_16((const uint16_t *)x, xo, wide != 0);
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      h[i] = xdt == OUT_F16 ? ws[i]
                            : (uint32_t)f2h(bits<float>(ws[i] << 16)) |
                                  ((uint32_t)f2h(bits<float>(ws[i] & 0xFFFF0000u)) << 16);
  }
  const uint4 g = prep_block8(h, load8_16(suh_g, e * in + k, wide != 0), j);
  const uint4 u = prep_block8(h, load8_16(suh_u, e * in + k, wide != 0), j);
  if (valid) {
    *reinterpret_cast<uint4 *>(xg + (size_t)slot * in + k) = g;
    *reinterpret_cast<uint4 *>(xu + (size_t)slot * in + k) = u;
  }
}

// The mid step: h = silu(g) * u (clamped when limit > 0), then down's
// prepare with suh_d[e] (the shared expert's, sh_suh_d, for e == shared), 16
// lanes a 128-block of the flattened [slots][inter / 128] (16-byte accesses:
// 8192 slots of 2048, 48 -> 33 us against a wave a block and 2-byte ones).
// A down GEMV launch of few workgroups forms the same values, bit for bit,
// in its SwiGLU prologue instead.  wide: the suh arrays are 16-byte aligned.
__global__ __launch_bounds__(256) void moe_mid_kernel(const uint16_t *__restrict__ g,
                                                      const uint16_t *__restrict__ u,
                                                      const uint32_t *__restrict__ inds,
                                                      int experts,
                                                      const uint16_t *__restrict__ suh_d,
                                                      uint16_t *__restrict__ xd, int inter,
                                                      float limit, int shared,
                                                      const uint16_t *__restrict__ sh_suh_d,
                                                      uint32_t nblocks, int wide) {
  const int j = threadIdx.x & 15;
  const uint32_t gb0 = blockIdx.x * 16u + (threadIdx.x >> 4);
  const uint32_t gb = min(gb0, nblocks - 1);
  const uint32_t nblk = (uint32_t)inter / 128u;
  const uint32_t slot = gb / nblk;
  const int k = (int)(gb - slot * nblk) * 128 + 8 * j;
  const uint32_t e0 = inds ? inds[slot] : 0u;
  const bool valid = gb0 < nblocks && e0 < (uint32_t)experts;
  const bool sh = valid && (int)e0 == shared;
  const uint16_t *sud = sh ? sh_suh_d : suh_d + (valid ? (size_t)e0 * inter : 0);
  const size_t off = (size_t)slot * inter + k;
  const uint4 gv = *reinterpret_cast<const uint4 *>(g + off);
  const uint4 uv = *reinterpret_cast<const uint4 *>(u + off);
  const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w}, uw[4] = {uv.x, uv.y, uv.z, uv.w};
  uint32_t h[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    h[i] = (uint32_t)f2h(swiglu1((uint16_t)(gw[i] & 0xFFFFu), (uint16_t)(uw[i] & 0xFFFFu), limit)) |
           ((uint32_t)f2h(swiglu1((uint16_t)(gw[i] >> 16), (uint16_t)(uw[i] >> 16), limit)) << 16);
  const uint4 o = prep_block8(h, load8_16(sud, k, wide != 0), j);
  if (valid) *reinterpret_cast<uint4 *>(xd + off) = o;
}

void launch_moe_mid(const uint16_t *g, const uint16_t *u, const uint32_t *inds, int experts,
                    const uint16_t *suh_d, uint16_t *xd, int slots, int inter, float limit,
                    int shared, const uint16_t *sh_suh_d, hipStream_t s) {
  const uint32_t nblocks = (uint32_t)slots * (uint32_t)(inter / 128);
  const int wide = (((uintptr_t)suh_d | (uintptr_t)sh_suh_d) & 15) == 0;
  hipLaunchKernelGGL(moe_mid_kernel, dim3((nblocks + 15) / 16), dim3(256), 0, s, g, u, inds,
                     experts, suh_d, xd, inter, limit, shared, sh_suh_d, nblocks, wide);
}

// y[row] = sum_k score * d[slot] (f32, k order), in the output dtype: eight
// columns a thread, U slots' loads in flight before their sums (1024 rows x top
// 8 of 7168: 84 -> 24 us against a column a thread).  U: 2, 4 or 8, the least
// that holds topk -- the rest of a wider pass is only more instructions (top 2 of
// 512 columns, 1 row 2.84 us at U = 8, 2.00 at 2; of 4096, 16 rows 3.64 and
// 3.04).  wide: y is 16-byte aligned.
template <int U>
__global__ __launch_bounds__(128) void moe_combine_kernel(const uint16_t *__restrict__ d,
                                                          const uint32_t *__restrict__ inds,
                                                          const void *__restrict__ scores, int sdt,
                                                          int topk, int experts, int hidden,
                                                          void *__restrict__ y, int ydt, int wide) {
  const size_t row = blockIdx.y;
  const int i = 8 * (blockIdx.x * 128 + threadIdx.x);
  if (i >= hidden) return;
  float acc[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = 0.0f;
  for (int k0 = 0; k0 < topk; k0 += U) {
    uint4 v[U];
    float w[U];
    bool on[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const size_t slot = row * topk + min(k0 + q, topk - 1);
      on[q] = k0 + q < topk && (inds ? inds[slot] : 0u) < (uint32_t)experts;
      w[q] = scores ? load_act(scores, slot, sdt) : 1.0f;
      if (on[q]) v[q] = *reinterpret_cast<const uint4 *>(d + slot * hidden + i);
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      if (!on[q]) continue;
      const uint32_t ws[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        acc[2 * c] = acc[2 * c] + f32_value(w[q] * h2f((uint16_t)(ws[c] & 0xFFFFu)));
        acc[2 * c + 1] = acc[2 * c + 1] + f32_value(w[q] * h2f((uint16_t)(ws[c] >> 16)));
      }
    }
  }
  const size_t o = row * hidden + i;
  if (ydt == OUT_F32) {
    float *p = (float *)y + o;
    if (wide) {
      *reinterpret_cast<float4 *>(p) = make_float4(acc[0], acc[1], acc[2], acc[3]);
      *reinterpret_cast<float4 *>(p + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) p[c] = acc[c];
    }
    return;
  }
  uint16_t r[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) r[c] = ydt == OUT_F16 ? f2h(acc[c]) : f2bf(acc[c]);
  uint16_t *p = (uint16_t *)y + o;
  if (wide) {
    *reinterpret_cast<uint4 *>(p) =
        make_uint4((uint32_t)r[0] | ((uint32_t)r[1] << 16), (uint32_t)r[2] | ((uint32_t)r[3] << 16),
                   (uint32_t)r[4] | ((uint32_t)r[5] << 16), (uint32_t)r[6] | ((uint32_t)r[7] << 16));
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) p[c] = r[c];
  }
}

void launch_moe_combine(const MoeArgs &a, const uint16_t *d, hipStream_t s) {
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((a.hidden / 8 + 127) / 128, a.rows), dim3(128), 0, s, d, a.inds,
                       a.scores, a.sdt, a.topk, a.experts, a.hidden, a.y, a.ydt,
                       (int)(((uintptr_t)a.y & 15) == 0));
  };
  if (a.topk <= 2)
    go(moe_combine_kernel<2>);
  else if (a.topk <= 4)
    go(moe_combine_kernel<4>);
  else
    go(moe_combine_kernel<8>);
}

// The routes of a swiglu with a shared expert (launch_moe_shared_route): one
// wave per row.  Top k of a softmax: the same order as the logits' (exp is
// monotonic), so the selection runs on the logits, k rounds of a wave argmax
// (ties: the lower index); the kept probabilities exp(l - max) / sum are
// renormalized to sum 1.
constexpr int SHARED_ROUTE_PER_LANE = 16;  // experts per lane: up to 1024

__device__ __forceinline__ float round_act(float v, int dt) {
  if (dt == OUT_F16) return h2f(f2h(v));
  if (dt == OUT_BF16) return bf2f(f2bf(v));
  return v;
}

// The shared expert's gate of row `row` (one wave; every lane returns it):
// sigmoid of the given logit, or of f(x . gate_vec) summed lane-strided
// then across the wave, rounded to the activation dtype xdt.
__device__ __forceinline__ float shared_gate(size_t row, int lane, const void *logit,
                                             const void *gate_vec, const void *x, int xdt,
                                             int hidden) {
  float lg;
  if (logit != nullptr) {
    lg = load_act(logit, row, xdt);
  } else {
    float d = 0.0f;
    for (int i = lane; i < hidden; i += 64)
      d += load_act(x, row * hidden + i, xdt) * load_act(gate_vec, i, xdt);
    for (int m = 32; m >= 1; m >>= 1) d += __shfl_xor(d, m, 64);
    lg = round_act(d, xdt);
  }
  return round_act(1.0f / (1.0f + expf(-lg)), xdt);
}

__global__ __launch_bounds__(64) void moe_shared_route_kernel(
    const uint32_t *__restrict__ inds, const void *__restrict__ scores, int sdt,
    const void *__restrict__ logits, int E, int k, const void *__restrict__ logit,
    const void *__restrict__ gate_vec, const void *__restrict__ x, int xdt, int hidden,
    uint32_t *__restrict__ inds_out, float *__restrict__ scores_out) {
  const size_t row = blockIdx.x;
  const int lane = threadIdx.x;
  const int kk = k + 1;
  if (logits != nullptr) {
    float l[SHARED_ROUTE_PER_LANE];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < SHARED_ROUTE_PER_LANE; ++i) {
      const int e = lane + 64 * i;
      l[i] = e < E ? load_act(logits, row * E + e, xdt) : -INFINITY;
      mx = fmaxf(mx, l[i]);
    }
    for (int m = 32; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, 64));
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < SHARED_ROUTE_PER_LANE; ++i)
      if (lane + 64 * i < E) sum += expf(l[i] - mx);
    for (int m = 32; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
    uint32_t taken = 0;
    float kept = 0.0f, pk = 0.0f;
    int ek = 0;
    for (int j = 0; j < k; ++j) {
      float bv = -INFINITY;
      int bi = 0x7FFFFFFF;
#pragma unroll
      for (int i = 0; i < SHARED_ROUTE_PER_LANE; ++i) {
        const int e = lane + 64 * i;
        if (e < E && !(taken & (1u << i)) && (l[i] > bv || (l[i] == bv && e < bi))) {
          bv = l[i];
          bi = e;
        }
      }
      for (int m = 32; m >= 1; m >>= 1) {
        const float ov = __shfl_xor(bv, m, 64);
        const int oi = __shfl_xor(bi, m, 64);
        if (ov > bv || (ov == bv && oi < bi)) {
          bv = ov;
          bi = oi;
        }
      }
      if ((bi & 63) == lane) taken |= 1u << (bi >> 6);
      const float p = expf(bv - mx) / sum;
      kept += p;
      if (lane == j) {
        pk = p;
        ek = bi;
      }
    }
    if (lane < k) {
      inds_out[row * kk + lane] = (uint32_t)ek;
      scores_out[row * kk + lane] = pk / kept;
    }
  } else if (lane < k) {
    inds_out[row * kk + lane] = inds[row * k + lane];
    scores_out[row * kk + lane] = load_act(scores, row * k + lane, sdt);
  }
  const float gate = shared_gate(row, lane, logit, gate_vec, x, xdt, hidden);
  if (lane == 0) {
    inds_out[row * kk + k] = (uint32_t)E;
    scores_out[row * kk + k] = gate;
  }
}

// The combine of a one-row swiglu_shared call whose k routes are given
// (no route launch): y[row] = sum over the routed slots j < k (expert below
// experts) of score_j * d[slot j], then + gate * d[slot k], gate the shared
// expert's sigmoid formed here by one wave as moe_shared_route_kernel forms
// it; the same f32 operations in the same order as moe_combine_kernel over
// that kernel's (k + 1)-wide routes, so results are equal bit for bit.
// Two columns a thread; the slots' loads go out before the gate's chain (logit,
// exponential, the workgroup's exchange), behind which they went one slot at a
// time (a DeepSeek-V3-shaped layer at one row 68.8 -> 67.6 us).
// U as moe_combine_kernel's.
template <int U>
__global__ __launch_bounds__(256) void moe_combine_shared_kernel(
    const uint16_t *__restrict__ d, const uint32_t *__restrict__ inds,
    const void *__restrict__ scores, int sdt, int k, int experts,
    const void *__restrict__ logit, const void *__restrict__ gate_vec,
    const void *__restrict__ x, int xdt, int hidden, void *__restrict__ y, int ydt) {
  __shared__ float gsh;
  const size_t row = blockIdx.y;
  const int i = 2 * (blockIdx.x * 256 + threadIdx.x);
  const int ic = min(i, hidden - 2);  // (past the last column: read, not stored)
  const size_t kk = (size_t)k + 1;
  uint32_t v[U];
  float w[U];
  bool on[U];
  auto load = [&](int j0) {
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int j = min(j0 + q, k - 1);
      on[q] = j0 + q < k && inds[row * k + j] < (uint32_t)experts;
      w[q] = load_act(scores, row * k + j, sdt);
      v[q] = on[q] ? *reinterpret_cast<const uint32_t *>(d + (row * kk + j) * hidden + ic) : 0u;
    }
  };
  load(0);
  const uint32_t vs = *reinterpret_cast<const uint32_t *>(d + (row * kk + k) * hidden + ic);
  if (threadIdx.x < 64) {
    const float gate = shared_gate(row, (int)threadIdx.x, logit, gate_vec, x, xdt, hidden);
    if (threadIdx.x == 0) gsh = gate;
  }
  float a0 = 0.0f, a1 = 0.0f;
  for (int j0 = 0; j0 < k; j0 += U) {
    if (j0 > 0) load(j0);
#pragma unroll
    for (int q = 0; q < U; ++q) {
      if (!on[q]) continue;
      a0 = a0 + f32_value(w[q] * h2f((uint16_t)(v[q] & 0xFFFFu)));
      a1 = a1 + f32_value(w[q] * h2f((uint16_t)(v[q] >> 16)));
    }
  }
  __syncthreads();
  a0 = a0 + f32_value(gsh * h2f((uint16_t)(vs & 0xFFFFu)));
  a1 = a1 + f32_value(gsh * h2f((uint16_t)(vs >> 16)));
  if (i >= hidden) return;
  const size_t o = row * hidden + i;
  if (ydt == OUT_F32) {
    ((float *)y)[o] = a0;
    ((float *)y)[o + 1] = a1;
  } else {
    ((uint16_t *)y)[o] = ydt == OUT_F16 ? f2h(a0) : f2bf(a0);
    ((uint16_t *)y)[o + 1] = ydt == OUT_F16 ? f2h(a1) : f2bf(a1);
  }
}

hipError_t launch_moe_shared_route(const uint32_t *inds, const void *scores, int sdt,
                                   const void *logits, int experts, int k, const void *logit,
                                   const void *gate_vec, const void *x, int xdt, int rows,
                                   int hidden, uint32_t *inds_out, float *scores_out,
                                   hipStream_t s) {
  if (rows <= 0 || k <= 0 || k > 63 || experts <= 0 || experts > 64 * SHARED_ROUTE_PER_LANE ||
      (logits == nullptr && (inds == nullptr || scores == nullptr)) ||
      (logit == nullptr && (gate_vec == nullptr || x == nullptr)))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(moe_shared_route_kernel, dim3(rows), dim3(64), 0, s, inds, scores, sdt,
                     logits, experts, k, logit, gate_vec, x, xdt, hidden, inds_out, scores_out);
  return hipGetLastError();
}

namespace {

struct MoeLayout {
  size_t sorted, items, n_items, g, u, xd, d, xg, xu, total;
  size_t partial_floats;  // slots in the separate slot buffer: gate, up, down
  int slots, max_items, ks_gu, ks_d, tps_gu, tps_d;
  bool gemm;  // larger expert batches: grouped GEMMs over items of up to RDG_ROWS slots,
  bool tiles;  // or the 256-slot ones
  bool direct;  // one row, routes given: every slot its own one-row item
  int item_rows;  // slots an item holds at most
};

// Down GEMV launches of at most this many workgroups take the mid step in
// their prepare (measured on the DeepSeek-V3 shape: 1008 workgroups at
// batch 1 gain ~3 us a call, 8064 at batch 16 lose ~11 us).
constexpr size_t MOE_FUSED_MID_MAX_WG = 2048;

// Grouped GEMM items hold up to 64 slots (32-row blocks by two, four
// workgroups a CU) below this average of slots per expert, where few experts
// pass 64; else 128 (two a CU), which decodes an expert's weights half as
// often.  256 experts of 7168 x 2048 at 32 slots: gate + up 1218 against 1343
// us, down 666 against 800; 16 experts of 4096 x 2048 at 64 / 128 / 1024
// slots, a call: 180 against 156, 270 against 253, 1528 against 1373 us.
constexpr int MOE_ITEM64_SLOTS = 48;

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace

namespace {
// The average of slots an expert from which a call counts as prefill-sized:
// swiglu_shared refuses such batches.
constexpr int MOE_PREFILL_SLOTS_PER_EXPERT = 32;

// What a routed call's linears run in: the GEMV items of up to 4 slots, which
// decode an expert's weights once per item; the register-decode grouped GEMM
// (items of up to RDG_ROWS slots); or the 256-slot grouped GEMM.
//
// Below 32 slots an expert: the items' time goes with the weights they decode
// (slots / 4 x 3 hidden inter, ~(its millions / 27)^0.65 x 18 us), the GEMM's
// with its unsplit k, ~21 us + 12.5 ns x (hidden + inter), which is what the
// quadratic bound follows; and few slots or workgroups (gate + up) leave its row
// blocks or the CUs empty, which is what the least averages are for.  The GEMM's
// time over the items' at that edge, K = 3 and 4: 256 experts of 7168 x 2048 at 4
// slots 0.83, of 1024 x 128 at 5 0.90, 64 of 1024 x 512 at 6 0.91, 32 of 7168 x
// 512 at 8 0.80, 16 of 2048 x 512 at 8 0.97, 8 of 4096 x 1024 at 12 0.85, 12 of
// 2048 x 256 at 17 0.72, 8 of 2048 x 512 at 17 0.80; under it 128 of 512 x 128 at
// 4 1.10, 32 of 1024 x 128 at 8 1.11, 16 of 7168 x 512 at 8 1.22, 8 of 1024 x 128
// at 31 1.43.  At 7 and 8 bits the GEMM is the slower for longer (32 of 4096 x
// 1024 at 4 / 6 / 8 slots 1.23 / 1.04 / 0.88), at the other rates alike.
//
// From 32 on the 256-slot GEMM is the other one (0.42-0.95 at 32 and 48 slots).
// In few workgroups over a short k its larger tiles win from 64 slots on:
// 8 experts of 512 x 256 at 64 / 96 / 128 / 200 / 300 slots 1.02 / 1.13 / 1.14 /
// 1.01 / 0.95, 2 of 1024 x 512 0.93 / 1.07 / 1.15 / 1.03 / 0.97; 2 of 4096 x 2048
// at 128 slots 0.95-1.01, at 8 bits 1.14.
//
// Banks that are not 16-byte aligned: the 256-slot GEMM, which reads words by
// dwords, from prefill-sized averages on.  16 experts of 4096 x 2048 at K = 3, 32
// / 64 / 300 slots: 237 / 250 / 535 us against 437 / 777 / 3466 in GEMV items.
enum class MoeGemm { none, rd, tiles };
MoeGemm moe_gemm(const MoeArgs &a, bool gu_generic, bool d_generic) {
  if (gu_generic || d_generic || a.inds == nullptr || a.verify_rows) return MoeGemm::none;
  const int64_t slots = (int64_t)a.rows * a.topk, E = a.experts;
  const bool prefill = slots >= MOE_PREFILL_SLOTS_PER_EXPERT * E;
  if (!a.aligned) return prefill ? MoeGemm::tiles : MoeGemm::none;
  const int64_t wg = E * 2 * ((a.inter + 64 * RDG_CW - 1) / (64 * RDG_CW));
  const double k = (double)a.hidden + a.inter;
  if (prefill)
    return wg < 64 && (k <= 3072 || a.n > 96) && slots >= 64 * E && slots < 256 * E
               ? MoeGemm::tiles
               : MoeGemm::rd;
  const int least = wg >= 1024 ? 4 : wg >= 512 ? 5 : wg >= 256 ? 6 : wg >= 64 ? 8 : 17;
  const double work = 0.75 * (double)slots * a.hidden * a.inter;
  return slots >= least * E && work >= (32e6 + 8.5 * k * k) * (a.n > 96 ? 2.5 : 1.0)
             ? MoeGemm::rd
             : MoeGemm::none;
}
}  // namespace

bool moe_uses_gemm(const MoeArgs &a, bool gu_generic, bool d_generic) {
  return moe_gemm(a, gu_generic, d_generic) != MoeGemm::none;
}

bool moe_prefill_sized(const MoeArgs &a, bool gu_generic, bool d_generic) {
  return !gu_generic && !d_generic &&
         (long)a.rows * a.topk >= (long)MOE_PREFILL_SLOTS_PER_EXPERT * a.experts;
}

namespace {

// A grouped GEMV launch's k-splits: as many as keep the launch within 768
// workgroups (three a CU; the grouped kernel's registers hold two a CU
// resident, and the third starts as the first two end: a further partial
// round and the split-K hand-off cost more than the longer splits;
// DeepSeek-V3's down at one row: 448 workgroups unsplit, 3 % faster a call
// than 896 in two splits), splits of at most MOE_TPS_MAX k-tiles, or
// MOE_DIRECT_TPS_MAX for one-row items (direct: DeepSeek-V3's gate+up at one
// row in 3 splits of 19 blocks, 768 workgroups, ~4 % faster a call than 4
// splits of up to 16 blocks, 1024 workgroups).
constexpr int MOE_RESIDENT_WG = 3 * 256;
void moe_plan(int in, int out, int groups, bool direct, int *ksplit, int *tps) {
  const int nb = in / 128;
  const int cgs = std::max(1, out / 128) * std::max(1, groups);
  const int ks = std::min(nb, std::max(1, MOE_RESIDENT_WG / cgs));
  int bps = std::min((direct ? MOE_DIRECT_TPS_MAX : MOE_TPS_MAX) / 8, (nb + ks - 1) / ks);
  bps = std::max(bps, (nb + GEMV_KSPLIT_MAX - 1) / GEMV_KSPLIT_MAX);
  // splits of even length: the fewest splits of at most bps blocks, then
  // the blocks spread over them (56 blocks at most 32 a split: 28 + 28, not
  // 32 + 24)
  const int nsplit = (nb + bps - 1) / bps;
  bps = (nb + nsplit - 1) / nsplit;
  *tps = 8 * bps;
  *ksplit = (nb + bps - 1) / bps;
}

MoeLayout moe_layout(const MoeArgs &a, bool generic_gu, bool generic_d) {
  MoeLayout L{};
  const int slots = a.rows * a.topk;
  L.slots = slots;
  const MoeGemm kind = moe_gemm(a, generic_gu, generic_d);
  L.gemm = kind != MoeGemm::none;
  L.tiles = kind == MoeGemm::tiles;
  // one row with its routes given: every slot its own work item, read from
  // the routes directly (no route launch; a row's routes name distinct
  // experts, and a repeated one would only be read twice)
  L.direct = !L.gemm && a.rows == 1 && a.inds != nullptr;
  const int item_rows = L.item_rows = !L.gemm   ? MOE_ITEM_ROWS
                                      : L.tiles ? GM_BM
                                      : slots < MOE_ITEM64_SLOTS * a.experts ? RDG_ROWS / 2
                                                                             : RDG_ROWS;
  L.max_items = std::min(a.experts, slots) + (slots + item_rows - 1) / item_rows;
  const int groups = std::max(1, std::min(a.experts, slots));
  moe_plan(a.hidden, a.inter, 2 * groups, L.direct, &L.ks_gu, &L.tps_gu);
  moe_plan(a.inter, a.hidden, groups, L.direct, &L.ks_d, &L.tps_d);
  if (generic_gu && L.tps_gu > 32) {
    L.tps_gu = 32;
    L.ks_gu = (a.hidden / 16 + 31) / 32;
  }
  if (generic_d && L.tps_d > 32) {
    L.tps_d = 32;
    L.ks_d = (a.inter / 16 + 31) / 32;
  }
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += align256(bytes);
    return at;
  };
  L.sorted = take((size_t)slots * 4);
  L.items = take((size_t)L.max_items * sizeof(MoeItem));
  L.n_items = take(4);
  L.g = take((size_t)slots * a.inter * 2);
  L.u = take((size_t)slots * a.inter * 2);
  L.xd = take((size_t)slots * a.inter * 2);
  L.d = take((size_t)slots * a.hidden * 2);
  if (L.gemm) {
    L.xg = take((size_t)slots * a.hidden * 2);
    L.xu = take((size_t)slots * a.hidden * 2);
  }
  L.total = o;
  L.partial_floats = L.gemm ? 1
                            : (size_t)2 * L.ks_gu * slots * a.inter + (size_t)L.ks_d * slots * a.hidden;
  return L;
}

// One grouped GEMV launch over `nweights` banks (gate and up side by side,
// or down); x holds raw rows (slot / topk) or prepared rows (slot); pro
// PRO_SWIGLU: x the slots' gate rows, a.c.x2 their up rows.
struct MoeGemv {
  const uint32_t *tw[2];
  int nweights;
  const void *x;
  int xdt;
  bool prepared;
  int pro;
  int in, out, ksplit, tps;
  int rows = MOE_ITEM_ROWS;  // the rows a workgroup's LDS holds: an item's at most, a
                             // grouped linear's; 1 where items are single slots
  GemvArgs a;
};

// The launch's packed geometry; false when a field does not fit.
bool moe_geo(const MoeGemv &m, dim3 grid, uint32_t *g0, uint32_t *g1, uint32_t *g2) {
  GemvGeo geo{};
  geo.cg1 = m.nweights > 1 ? m.out / 128 : 0;
  geo.cgend = (int)grid.x;
  geo.rows = m.rows;
  geo.xdt = m.xdt;
  geo.prepared = m.prepared ? 1 : 0;
  geo.in_tiles = m.in / 16;
  geo.tps = m.tps;
  return gemv_geo_pack(geo, g0, g1, g2);
}

void moe_gemv_launch(const Format &f, dim3 grid, size_t lds, hipStream_t s, const MoeGemv &m,
                     const uint32_t *sorted, const MoeItem *items, const uint32_t *n_items,
                     int topk) {
  uint32_t g0, g1, g2;
  if (!moe_geo(m, grid, &g0, &g1, &g2)) return;  // checked before the first launch
  rate_dispatch(gemv_rate(f), [&](auto KC) {
    moe_gemv_go<decltype(KC)::value>(f, m.pro, grid, lds, s, m.tw[0], m.tw[1], m.x, g0, g1, g2,
                                     topk, sorted, items, n_items, m.a);
  });
}

GemvWeight moe_weight(const MoeBank &b, uint16_t *y, float *partial) {
  GemvWeight w{};
  w.suh = b.suh;
  w.svh = b.svh;
  w.y = y;
  w.zout = nullptr;
  w.partial = partial;
  w.expert_words = (size_t)(b.in / 16) * (b.out / 16) * (b.f.n / 2);
  return w;
}

MoeGemv moe_gemv(const void *x, int xdt, bool prepared, size_t slots, int in, int out,
                 const Format &f, int ksplit, int tps) {
  MoeGemv m{};
  m.x = x;
  m.xdt = xdt;
  m.prepared = prepared;
  m.in = in;
  m.out = out;
  m.ksplit = ksplit;
  m.tps = tps;
  m.a.c.ydt = OUT_F16;
  m.a.c.ptotal = slots;
  m.a.c.ksplit = ksplit;
  m.a.c.dec = f.dec();
  m.a.c.nw = f.n / 2;
  m.a.c.shared_expert = -1;
  return m;
}

// The k-splits of a grouped linear's GEMV: the dense plan over every group's
// column groups.
void gemv_groups_plan(int rows, int groups, int in, int out, bool generic, int *ks, int *tps) {
  gemv_plan(in, out, groups, rows, ks, tps, GEMV_TPS_MAX);
  if (generic && *tps > 32) {
    *tps = 32;
    *ks = (in / 16 + 31) / 32;
  }
}

}  // namespace

size_t gemv_groups_floats(int rows, int groups, int in, int out, bool generic) {
  int ks, tps;
  gemv_groups_plan(rows, groups, in, out, generic, &ks, &tps);
  return (size_t)ks * rows * groups * out;
}

// One launch of the grouped GEMV, group z its work item z: every group's
// rows read and written in place.  (Per group, a strided copy in, a GEMV and a
// copy out were 24 launches at 8 groups: 8 x 4096 -> 1024 at K = 3, 4 rows,
// 104.7 -> 12.1 us.)
hipError_t launch_gemv_groups(const uint16_t *trellis, const Format &f, const void *x, int xdt,
                              const uint16_t *suh, const uint16_t *svh, void *y, int ydt, int rows,
                              int groups, int in, int out, const Scratch &sc, hipStream_t s) {
  if (rows < 1 || rows > GEMV_ROWS_MAX || groups < 1 || groups > 65535 || in <= 0 || out <= 0 ||
      in % 128 != 0 || out % 128 != 0 || in / 16 > 65535 || out / 128 > 65535 || y == nullptr)
    return hipErrorInvalidValue;
  if (f.n < 16 || f.n > 128 || (f.n & 1)) return hipErrorInvalidValue;
  if ((int64_t)rows * groups * std::max(in, out) >= (int64_t)1 << 31) return hipErrorInvalidValue;
  const bool generic = f.gemv_generic();
  int ks, tps;
  gemv_groups_plan(rows, groups, in, out, generic, &ks, &tps);
  const size_t slots = (size_t)rows * groups;
  // a split's slot planes are addressed with 32-bit byte offsets
  if (ks > GEMV_KSPLIT_MAX || (size_t)ks * slots * out * 4 > 0x7FFFFFFFu)
    return hipErrorInvalidValue;
  if (rows * (tps / 8) > PREP_PASSES * PREP_GROUPS) return hipErrorInvalidValue;
  if (ks > 1 && (sc.partial == nullptr || sc.status == nullptr ||
                 sc.partial_floats < (size_t)ks * slots * out))
    return hipErrorInvalidValue;
  MoeGemv m = moe_gemv(x, xdt, false, slots, in, out, f, ks, tps);
  m.nweights = 1;
  m.rows = rows;
  m.a.c.ydt = ydt;
  m.a.c.status = sc.status;
  m.a.c.poll_max = splitk_poll_max();
  m.a.c.drop_partials = splitk_drop();
  m.tw[0] = m.tw[1] = reinterpret_cast<const uint32_t *>(trellis);
  GemvWeight &w = m.a.w[0];
  w.suh = suh;
  w.svh = svh;
  w.y = y;
  w.partial = sc.partial;
  w.expert_words = (size_t)(in / 16) * (out / 16) * (f.n / 2);
  const dim3 grid(out / 128, ks, groups);
  uint32_t g[3];
  if (!moe_geo(m, grid, &g[0], &g[1], &g[2])) return hipErrorInvalidValue;
  moe_gemv_launch(f, grid, gemv_lds_bytes(rows, tps, generic), s, m, nullptr, nullptr, nullptr,
                  groups);
  return hipGetLastError();
}

bool moe_shared_direct(const MoeArgs &a, bool gu_generic, bool d_generic) {
  if (a.rows != 1 || a.topk <= 0 || a.experts <= 0 || a.hidden % 128 != 0) return false;
  const MoeLayout L = moe_layout(a, gu_generic, d_generic);
  return !L.gemm &&
         (size_t)(a.hidden / 128) * L.ks_d * L.slots <= MOE_FUSED_MID_MAX_WG;
}

size_t moe_scratch_bytes(const MoeArgs &a, bool gu_generic, bool d_generic,
                         size_t *partial_floats) {
  if (a.rows <= 0 || a.topk <= 0) {
    *partial_floats = 1;
    return 256;
  }
  const MoeLayout L = moe_layout(a, gu_generic, d_generic);
  *partial_floats = L.partial_floats;
  return L.total;
}

hipError_t launch_moe(const MoeArgs &a, const MoeBank &gate, const MoeBank &up,
                      const MoeBank &down, void *scratch, size_t scratch_bytes,
                      const Scratch &slots, hipStream_t s, const MoeShared *shared) {
  if (a.rows <= 0 || a.topk <= 0 || a.experts <= 0 || a.experts > MOE_ROUTE_THREADS)
    return hipErrorInvalidValue;
  if (a.hidden % 128 != 0 || a.inter % 128 != 0) return hipErrorInvalidValue;
  if (a.hidden / 16 > 65535 || a.inter / 16 > 65535) return hipErrorInvalidValue;
  if (gate.f.n != up.f.n || !gate.f.same_decode(up.f) ||
      gate.in != a.hidden || up.in != a.hidden || down.out != a.hidden || gate.out != a.inter ||
      up.out != a.inter || down.in != a.inter)
    return hipErrorInvalidValue;
  const bool gu_generic = !gate.f.integer_rate(), d_generic = !down.f.integer_rate();
  const MoeLayout L = moe_layout(a, gu_generic, d_generic);
  if (shared) {
    auto same = [](const MoeBank &b, const MoeBank &r) {
      return b.trellis && b.suh && b.svh && b.in == r.in && b.out == r.out && b.f.n == r.f.n &&
             b.f.same_decode(r.f);
    };
    if (L.gemm || a.inds == nullptr || !same(shared->gate, gate) || !same(shared->up, up) ||
        !same(shared->down, down))
      return hipErrorInvalidValue;
  }
  const int sh_index = shared ? a.experts - 1 : -1;
  // one row, k routes given: slot k is the shared expert, no route launch
  const int routes_k = shared ? shared->routes_k : 0;
  if (routes_k > 0 && (a.rows != 1 || a.inds == nullptr || a.topk != routes_k + 1 ||
                       (shared->logit == nullptr && shared->gate_vec == nullptr)))
    return hipErrorInvalidValue;
  if (scratch_bytes < L.total || slots.status == nullptr || slots.partial == nullptr ||
      slots.partial_floats < L.partial_floats || L.slots > MOE_SLOTS_MAX ||
      L.max_items > 65535 || (int64_t)L.slots * std::max(a.hidden, a.inter) >= (int64_t)1 << 31)
    return hipErrorInvalidValue;
  float *partial = slots.partial;
  char *base = (char *)scratch;
  uint32_t *sorted = (uint32_t *)(base + L.sorted);
  MoeItem *items = (MoeItem *)(base + L.items);
  uint32_t *n_items = (uint32_t *)(base + L.n_items);
  uint16_t *g = (uint16_t *)(base + L.g), *u = (uint16_t *)(base + L.u);
  uint16_t *xd = (uint16_t *)(base + L.xd), *d = (uint16_t *)(base + L.d);
  float *pgu = partial, *pd = partial + (size_t)2 * L.ks_gu * L.slots * a.inter;

  if (L.gemm) {
    // prefill-sized expert batches: per-slot prepared rows, grouped GEMMs
    // gate and up, the mid step, grouped GEMM down, the weighted sum
    hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(MOE_ROUTE_THREADS), 0, s, a.inds, L.slots,
                       a.experts, sorted, items, n_items, (uint32_t)L.item_rows);
    uint16_t *xg = (uint16_t *)(base + L.xg), *xu = (uint16_t *)(base + L.xu);
    const uint32_t nblocks = (uint32_t)L.slots * (uint32_t)(a.hidden / 128);
    const int wide = (((uintptr_t)a.x | (uintptr_t)gate.suh | (uintptr_t)up.suh) & 15) == 0;
    hipLaunchKernelGGL(moe_prep_kernel, dim3((nblocks + 15) / 16), dim3(256), 0, s, a.x, a.xdt,
                       a.inds, a.experts, a.topk, gate.suh, up.suh, xg, xu, a.hidden, nblocks,
                       wide);
    auto grouped = [&](const MoeBank *const *b, const uint16_t *const *xp, uint16_t *const *yo,
                       int nw) {
      if (L.tiles) {
        for (int i = 0; i < nw; ++i) {
          const GemmGroup gg{sorted, items, n_items,
                             (size_t)(b[i]->in / 16) * (b[i]->out / 16) * (b[i]->f.n / 2), 0, 0};
          rate_dispatch(b[i]->f.n / 16, [&](auto KC) {
            constexpr int K = decltype(KC)::value;
            if constexpr (K > 0)
              gemm_grouped_go<K>(b[i]->f, dim3(b[i]->out / GM_BN, L.max_items), s,
                                 reinterpret_cast<const uint32_t *>(b[i]->trellis), xp[i],
                                 b[i]->svh, yo[i], OUT_F16, b[i]->in / 16, b[i]->out / 16, gg);
          });
        }
        return;
      }
      RdGroupArgs r{};
      r.nw = nw;
      r.ydt = OUT_F16;
      r.in_tiles = b[0]->in / 16;
      r.dec = b[0]->f.dec();
      r.sorted = sorted;
      r.items = items;
      r.n_items = n_items;
      for (int i = 0; i < nw; ++i) {
        r.w[i] = RdGroupWeight{reinterpret_cast<const uint32_t *>(b[i]->trellis), xp[i], b[i]->svh,
                               yo[i], (size_t)(b[i]->in / 16) * (b[i]->out / 16) * (b[i]->f.n / 2),
                               b[i]->out / 16, r.ct};
        r.ct += (b[i]->out + 64 * RDG_CW - 1) / (64 * RDG_CW);
      }
      const unsigned grid = (unsigned)r.ct * ((L.max_items + 7) / 8 * 8);
      rate_dispatch(b[0]->f.n / 16, [&](auto KC) {
        constexpr int K = decltype(KC)::value;
        if constexpr (K > 0) gemm_rd_grouped_go<K>(b[0]->f, L.item_rows, grid, s, r);
      });
    };
    const MoeBank *const gub[2] = {&gate, &up}, *const db[1] = {&down};
    const uint16_t *const gux[2] = {xg, xu}, *const dx[1] = {xd};
    uint16_t *const guy[2] = {g, u}, *const dy[1] = {d};
    grouped(gub, gux, guy, 2);
    launch_moe_mid(g, u, a.inds, a.experts, down.suh, xd, L.slots, a.inter, a.limit, -1, nullptr, s);
    grouped(db, dx, dy, 1);
    launch_moe_combine(a, d, s);
    return hipGetLastError();
  }
  const size_t gu_part = (size_t)L.ks_gu * L.slots * a.inter;
  MoeGemv mgu = moe_gemv(a.x, a.xdt, false, L.slots, a.hidden, a.inter, gate.f, L.ks_gu, L.tps_gu);
  mgu.nweights = 2;
  // one-row items (direct) allocate one row of LDS
  const bool direct = L.direct;
  const int nz = direct ? L.slots : L.max_items;
  const dim3 grid_gu(2 * (a.inter / 128), L.ks_gu, nz);
  const dim3 grid_d(a.hidden / 128, L.ks_d, nz);
  // down: in a launch of few workgroups every workgroup forms the mid step
  // (the SwiGLU of its slots' gate and up rows, the down rotation) for its
  // k-slice in its prepare, which costs less than the mid launch; in larger
  // launches the repeats across column groups cost more than the launch
  const bool fused_mid = (size_t)grid_d.x * grid_d.y * grid_d.z <= MOE_FUSED_MID_MAX_WG;
  if (routes_k > 0 && !fused_mid) return hipErrorInvalidValue;
  MoeGemv md = fused_mid ? moe_gemv(g, OUT_F16, false, L.slots, a.inter, a.hidden, down.f, L.ks_d,
                                    L.tps_d)
                         : moe_gemv(xd, OUT_F16, true, L.slots, a.inter, a.hidden, down.f, L.ks_d,
                                    L.tps_d);
  md.nweights = 1;
  const int lds_rows = direct ? 1 : MOE_ITEM_ROWS;
  mgu.rows = md.rows = lds_rows;
  if (fused_mid) {
    md.pro = PRO_SWIGLU;
    md.a.c.x2 = u;
    md.a.c.limit = a.limit;
  }
  mgu.a.c.status = md.a.c.status = slots.status;
  mgu.a.c.poll_max = md.a.c.poll_max = splitk_poll_max();
  mgu.a.c.drop_partials = md.a.c.drop_partials = splitk_drop();
  uint32_t gg[3];
  if (!moe_geo(mgu, grid_gu, &gg[0], &gg[1], &gg[2]) || !moe_geo(md, grid_d, &gg[0], &gg[1], &gg[2]))
    return hipErrorInvalidValue;
  if (!direct)
    hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(MOE_ROUTE_THREADS), 0, s, a.inds, L.slots,
                       a.experts, sorted, items, n_items, (uint32_t)MOE_ITEM_ROWS);
  const uint32_t *isorted = direct ? a.inds : sorted;
  const MoeItem *iitems = direct ? nullptr : items;
  const uint32_t *in_items = direct ? nullptr : n_items;
  mgu.a.c.experts = md.a.c.experts = a.experts;
  mgu.a.c.routes_k = md.a.c.routes_k = routes_k;
  mgu.tw[0] = reinterpret_cast<const uint32_t *>(gate.trellis);
  mgu.tw[1] = reinterpret_cast<const uint32_t *>(up.trellis);
  mgu.a.w[0] = moe_weight(gate, g, pgu);
  mgu.a.w[1] = moe_weight(up, u, pgu + gu_part);
  if (shared) {
    mgu.a.c.shared_expert = md.a.c.shared_expert = sh_index;
    const MoeBank *sb[2] = {&shared->gate, &shared->up};
    for (int i = 0; i < 2; ++i) {
      mgu.a.w[i].sh_tw = reinterpret_cast<const uint32_t *>(sb[i]->trellis);
      mgu.a.w[i].sh_suh = sb[i]->suh;
      mgu.a.w[i].sh_svh = sb[i]->svh;
    }
  }
  moe_gemv_launch(gate.f, grid_gu, gemv_lds_bytes(lds_rows, L.tps_gu, gu_generic), s, mgu,
                  isorted, iitems, in_items, a.topk);
  if (!fused_mid)
    launch_moe_mid(g, u, a.inds, a.experts, down.suh, xd, L.slots, a.inter, a.limit, sh_index,
                   shared ? shared->down.suh : nullptr, s);
  md.tw[0] = md.tw[1] = reinterpret_cast<const uint32_t *>(down.trellis);
  md.a.w[0] = moe_weight(down, d, pd);
  if (shared) {
    md.a.w[0].sh_tw = reinterpret_cast<const uint32_t *>(shared->down.trellis);
    md.a.w[0].sh_suh = shared->down.suh;
    md.a.w[0].sh_svh = shared->down.svh;
  }
  moe_gemv_launch(down.f, grid_d, gemv_lds_bytes(lds_rows, L.tps_d, d_generic), s, md,
                  isorted, iitems, in_items, fused_mid ? 1 : a.topk);
  auto combine_shared = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((a.hidden + 511) / 512, 1), dim3(256), 0, s, d, a.inds, a.scores,
                       a.sdt, routes_k, a.experts, shared->logit, shared->gate_vec, a.x, a.xdt,
                       a.hidden, a.y, a.ydt);
  };
  if (routes_k <= 0)
    launch_moe_combine(a, d, s);
  else if (routes_k <= 2)
    combine_shared(moe_combine_shared_kernel<2>);
  else if (routes_k <= 4)
    combine_shared(moe_combine_shared_kernel<4>);
  else
    combine_shared(moe_combine_shared_kernel<8>);
  return hipGetLastError();
}

}  // namespace exl3
