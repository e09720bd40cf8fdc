// Row-major values <-> the C-stream element order c_layout_atb(., 128, 128) (redline/npu_layouts.py:31-47), optionally
// through a permutation of the columns (the packed weights' channel order, redline/vlm_run.py:363-366).
//
// A workgroup takes 8 rows (a br half of a 16-row band) x 1024 columns without a permutation, or 8 whole rows with one.
// Block f = (column block, rib) of the band is 16 bytes; 16 consecutive lanes hold 16 consecutive blocks of the stream
// and 128 contiguous bytes of each row. With a permutation the 8 rows pass through LDS as bf16, read or written there
// at the permuted column (2-byte accesses), so that both sides in memory stay whole 16-byte accesses. HBM-bound: each
// value read once and written once. A 1536 x 4096 text-encoder input or output took ~10 launches (index arithmetic on
// int64 tensors, gathers, casts) each way and takes one of 15-17 us now: a text-encoder layer with its input and output
// 1621 -> 1076 us.
#include "rlbfp.h"
#include "rlbfp_device.h"
#include "rlbfp_host.h"

namespace rl {

constexpr int kStThreads = 512, kStRows = 8, kStPad = 8;

// Stream block of (row r0 + rib, column block cb) for a band starting at r0 (r0 % 8 == 0)
__device__ __forceinline__ int64_t stream_block(int64_t r0, int cb, int rib, int D) {
  const int64_t g = (r0 >> 9) * (D >> 7) + (cb >> 4);
  return g * 8192 + ((r0 >> 7) & 3) * 2048 + ((r0 >> 4) & 7) * 256 + ((cb >> 1) & 7) * 32 + ((r0 >> 3) & 1) * 16 +
         (cb & 1) * 8 + rib;
}

template <int DT>
__device__ __forceinline__ u32x4 load8_bf16(const void* x, int64_t i) {
  if constexpr (DT == RL_DTYPE_BF16) return *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(x) + i);
  const f32x4* p = reinterpret_cast<const f32x4*>(static_cast<const float*>(x) + i);
  const f32x4 a = p[0], b = p[1];
  return u32x4{pack_bf16_rne(a[0], a[1]), pack_bf16_rne(a[2], a[3]), pack_bf16_rne(b[0], b[1]),
               pack_bf16_rne(b[2], b[3])};
}

template <int DT>
__device__ __forceinline__ void store8_bf16(void* x, int64_t i, u32x4 v) {
  if constexpr (DT == RL_DTYPE_BF16) {
    *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(x) + i) = v;
  } else {
    u32x4* p = reinterpret_cast<u32x4*>(static_cast<float*>(x) + i);
    p[0] = u32x4{v.x << 16, v.x & 0xFFFF0000u, v.y << 16, v.y & 0xFFFF0000u};
    p[1] = u32x4{v.z << 16, v.z & 0xFFFF0000u, v.w << 16, v.w & 0xFFFF0000u};
  }
}

// stream[(r, c)] = bf16(x[r][perm[c]]), rows from `rows` on zero
template <int DT, bool PERM>
__global__ __launch_bounds__(kStThreads) void stream_pack_kernel(const void* __restrict__ x, int64_t rows, int64_t ld,
                                                                 const int64_t* __restrict__ perm, int D,
                                                                 uint16_t* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int64_t r0 = (int64_t)blockIdx.x * kStRows;
  const int tid = threadIdx.x, rib = tid & 7, nb = D >> 3, ldr = D + kStPad;
  const int64_t r = r0 + rib;
  if constexpr (!PERM) {
    const int cb = blockIdx.y * 128 + (tid >> 3);
#pragma unroll
    for (int j = 0; j < 2; j++) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (r < rows) v = load8_bf16<DT>(x, r * ld + (cb + 64 * j) * 8);
      *reinterpret_cast<u32x4*>(out + 8 * stream_block(r0, cb + 64 * j, rib, D)) = v;
    }
  } else {
    // a wave reads one row's consecutive blocks
    const int wr = tid >> 6;
    for (int cb = tid & 63; cb < nb; cb += 64) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (r0 + wr < rows) v = load8_bf16<DT>(x, (r0 + wr) * ld + cb * 8);
      *reinterpret_cast<u32x4*>(lds + wr * ldr + cb * 8) = v;
    }
    __syncthreads();
    for (int cb = tid >> 3; cb < nb; cb += kStThreads / 8) {
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const uint64_t p = (uint64_t)perm[cb * 8 + e];
        const uint32_t b = p < (uint64_t)D ? lds[rib * ldr + (int)p] : 0u;  // the host has checked the range
        w[e >> 1] = e & 1 ? w[e >> 1] | (b << 16) : b;
      }
      *reinterpret_cast<u32x4*>(out + 8 * stream_block(r0, cb, rib, D)) = u32x4{w[0], w[1], w[2], w[3]};
    }
  }
}

// out[r][perm[c]] = stream[(r, c)]
template <int DT, bool PERM>
__global__ __launch_bounds__(kStThreads) void stream_unpack_kernel(const uint16_t* __restrict__ s, int64_t ld,
                                                                   const int64_t* __restrict__ perm, int D,
                                                                   void* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int64_t r0 = (int64_t)blockIdx.x * kStRows;
  const int tid = threadIdx.x, rib = tid & 7, nb = D >> 3, ldr = D + kStPad;
  if constexpr (!PERM) {
    const int cb = blockIdx.y * 128 + (tid >> 3);
#pragma unroll
    for (int j = 0; j < 2; j++)
      store8_bf16<DT>(out, (r0 + rib) * ld + (cb + 64 * j) * 8,
                      *reinterpret_cast<const u32x4*>(s + 8 * stream_block(r0, cb + 64 * j, rib, D)));
  } else {
    for (int cb = tid >> 3; cb < nb; cb += kStThreads / 8) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(s + 8 * stream_block(r0, cb, rib, D));
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const uint64_t p = (uint64_t)perm[cb * 8 + e];
        if (p < (uint64_t)D) lds[rib * ldr + (int)p] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
      }
    }
    __syncthreads();
    const int wr = tid >> 6;
    for (int cb = tid & 63; cb < nb; cb += 64)
      store8_bf16<DT>(out, (r0 + wr) * ld + cb * 8, *reinterpret_cast<const u32x4*>(lds + wr * ldr + cb * 8));
  }
}

static int check_stream(int32_t dtype, int64_t ld, int64_t M, int64_t D, bool perm) {
  if (dtype != RL_DTYPE_F32 && dtype != RL_DTYPE_BF16) return fail(RL_ERR_ARG, "dtype %d unknown", dtype);
  if (M < 512 || M % 512 || M > (1 << 30) || D < 1024 || D % 1024 || D > (perm ? 8192 : 1 << 24))
    return fail(RL_ERR_SHAPE, "M %lld D %lld: need M %% 512 == 0, D %% 1024 == 0 (D <= 8192 with a permutation)",
                (long long)M, (long long)D);
  if (ld < D || ld % 8) return fail(RL_ERR_ALIGN, "ld %lld: need >= D and a multiple of 8", (long long)ld);
  return RL_OK;
}

template <typename K>
static int set_lds(K kernel, int lds) {
  if (lds <= 48 * 1024) return RL_OK;
  const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  return e == hipSuccess ? RL_OK : fail(RL_ERR_DEVICE, "hipFuncSetAttribute: %s", hipGetErrorString(e));
}

}  // namespace rl

extern "C" int rl_stream_pack(const void* x, int32_t dtype, int64_t rows, int64_t ld, const int64_t* perm, int64_t M,
                              int64_t D, uint16_t* out, void* stream) {
  using namespace rl;
  int s = check_stream(dtype, ld, M, D, perm != nullptr);
  if (s) return s;
  if (rows < 0 || rows > M) return fail(RL_ERR_SHAPE, "%lld rows of %lld", (long long)rows, (long long)M);
  if ((!x && rows) || !out) return fail(RL_ERR_NULL, "x or out is NULL");
  if (((uintptr_t)x | (uintptr_t)out) % 16 || (uintptr_t)perm % 8)
    return fail(RL_ERR_ALIGN, "x and out must be 16-byte, perm 8-byte aligned");
  if ((s = check_device())) return s;
  const int lds = perm ? kStRows * ((int)D + kStPad) * 2 : 0;
  const dim3 grid((unsigned)(M / kStRows), perm ? 1u : (unsigned)(D / 1024));
  auto go = [&](auto kernel) {
    if (int e = set_lds(kernel, lds)) return e;
    hipLaunchKernelGGL(kernel, grid, dim3(kStThreads), (unsigned)lds, static_cast<hipStream_t>(stream), x, rows, ld,
                       perm, (int)D, out);
    return launch_status("rl_stream_pack");
  };
  if (dtype == RL_DTYPE_BF16)
    return perm ? go(stream_pack_kernel<RL_DTYPE_BF16, true>) : go(stream_pack_kernel<RL_DTYPE_BF16, false>);
  return perm ? go(stream_pack_kernel<RL_DTYPE_F32, true>) : go(stream_pack_kernel<RL_DTYPE_F32, false>);
}

extern "C" int rl_stream_unpack(const uint16_t* x, const int64_t* perm, int64_t M, int64_t D, void* out, int32_t dtype,
                                int64_t ld, void* stream) {
  using namespace rl;
  int s = check_stream(dtype, ld, M, D, perm != nullptr);
  if (s) return s;
  if (!x || !out) return fail(RL_ERR_NULL, "x or out is NULL");
  if (((uintptr_t)x | (uintptr_t)out) % 16 || (uintptr_t)perm % 8)
    return fail(RL_ERR_ALIGN, "x and out must be 16-byte, perm 8-byte aligned");
  if ((s = check_device())) return s;
  const int lds = perm ? kStRows * ((int)D + kStPad) * 2 : 0;
  const dim3 grid((unsigned)(M / kStRows), perm ? 1u : (unsigned)(D / 1024));
  auto go = [&](auto kernel) {
    if (int e = set_lds(kernel, lds)) return e;
    hipLaunchKernelGGL(kernel, grid, dim3(kStThreads), (unsigned)lds, static_cast<hipStream_t>(stream), x, ld, perm,
                       (int)D, out);
    return launch_status("rl_stream_unpack");
  };
  if (dtype == RL_DTYPE_BF16)
    return perm ? go(stream_unpack_kernel<RL_DTYPE_BF16, true>) : go(stream_unpack_kernel<RL_DTYPE_BF16, false>);
  return perm ? go(stream_unpack_kernel<RL_DTYPE_F32, true>) : go(stream_unpack_kernel<RL_DTYPE_F32, false>);
}
