// Fused residual add + LayerNorm / RMSNorm + modulate, producing the next GEMM's A operand.
//
// Replaces the fused artifact of kernels/glue/ln_design.py:38-118 (microkernels ln_par / ln_p1 / ln_fin / ln_p2,
// kernels/glue/ln_mod.cc:92-204) that run_ln.ln_run drives (redline/run_ln.py:43-57), and its RMSNorm copies
// (kernels/vlm/rms_mod.cc with a bfp16 branch, rms16_mod.cc with a bf16 branch). The NPU kernel streams each 128-row
// tile twice, statistics first and outputs second. Here one wave owns one row and keeps its D values in registers,
// so x and the branch are read once. The kernel is HBM-bound: per value it reads 2 bytes of x and 2 (bf16) or 9/8
// (packed) bytes of branch, and writes 2 bytes of x', 9/8 bytes of packed A and/or 2 bytes of bf16 A.
//
// Lane l of a row's wave owns the 8-value blocks l, l + 64, l + 128, ... of the row, so every load and store is a
// coalesced 16-byte access and a wave covers 1 KB of the row per instruction. The packed output is assembled in LDS
// in output order and written with 16-byte stores. In rowblock order the workgroup's 4 rows are one contiguous span.
// In A-layout order the workgroup takes 16 rows, one 16-row band (sbr) of the 128-row A tiles, which is a contiguous
// 128-block (1152-byte) span per 64-column K tile.
#include <math.h>

#include "rlbfp.h"
#include "rlbfp_device.h"
#include "rlbfp_host.h"

namespace rl {

constexpr int kLnThreads = 256;  // 4 waves
constexpr int kLnMaxNB = 16;     // blocks per lane: D <= 64 lanes * 16 blocks * 8 = 8192

struct LnArgs {
  const uint16_t* x;
  int64_t ldx;
  const void* br;
  int32_t br_fmt;
  int64_t ld_br;
  const uint16_t* params;
  int64_t split_row;
  int32_t norm;
  uint16_t* x_out;
  int64_t ld_xo;
  uint8_t* a_packed;
  int32_t a_order;
  uint16_t* a_deq;
  int64_t ld_a;
  int64_t M;
  int32_t D;
  int32_t rows_wg;  // rows per workgroup: 4, or 16 for the A-layout order
};

template <bool NT>
__device__ __forceinline__ void store_x(uint16_t* p, u32x4 v) {
  if constexpr (NT)
    store_stream(p, v);
  else
    *reinterpret_cast<u32x4*>(p) = v;
}

// Whether x' goes past the caches (br: 0 no branch, 1 bf16, 2 packed). It pays where x and the branch are more than the
// L2s hold (8 x 4 MB): cached x' then pushes out what is still to be read. Cached against past the caches, us, by bytes
// read: 37 MB (2624 x 3520, bf16 branch) 15.3 / 15.7; 36 MB (4352 x 4096, no branch) 21.1 / 21.6; 42 MB (4352 x 3072,
// packed) 19.7 / 18.4; 48 MB (4352 x 3520, packed) 24.4 / 22.3; 61 MB (same, bf16) 28.1 / 23.5; 71 MB (8704 x 4096, no
// branch) 46.6 / 43.0; from 110 MB on the same. On streams (below) it cost nothing at any size, so there it is always so.
static bool past_caches(int64_t M, int64_t D, int br) {
  return M * D * (br == 0 ? 16 : br == 1 ? 32 : 25) / 8 > 40000000;
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}

// Sum over the wave, every lane getting the same value: within rows of 16 by DPP adds (quad swaps, half-row and row
// mirrors), then across the four rows with two lane permutes.
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp_f<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_f<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_f<0x141>(v);  // row_half_mirror
  v += dpp_f<0x140>(v);  // row_mirror
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

__device__ __forceinline__ void unpack8(u32x4 v, float f[8]) {
  f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xFFFF0000u);
  f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xFFFF0000u);
  f[4] = __uint_as_float(v.z << 16); f[5] = __uint_as_float(v.z & 0xFFFF0000u);
  f[6] = __uint_as_float(v.w << 16); f[7] = __uint_as_float(v.w & 0xFFFF0000u);
}


// Template NB = blocks of 8 per lane (D / 512 rounded up); lanes whose block lies past the row end hold zeros and
// skip every access. Up to 8 blocks a row's first-pass loads are all in flight at once (in chunks of up to 6), which
// needs more registers than one block at a time: the register budget per NB is the smallest that compiles without
// spills. For D = 3072 (NB 6) it allows 4 waves per SIMD, so a launch of one wave per row for M = 4352 rows leaves a
// short second round; that costs less than the per-block round trips of the 5-wave form (23.0 -> 22.0 us with a bf16
// branch, 19.9 -> 18.6 us with a packed one, same bits).
template <int NB>
constexpr int ln_waves_per_simd() { return NB <= 2 ? 6 : NB <= 4 ? 5 : NB <= 6 ? 4 : NB <= 8 ? 3 : NB <= 13 ? 4 : 3; }

// BR: the branch's format for NB <= 8 (0 none, 1 bf16, 2 packed); above 8 blocks it is tested at run time (BR = -1)
template <int NB, int BR, bool NT>
__global__ __launch_bounds__(kLnThreads, ln_waves_per_simd<NB>()) void ln_kernel(LnArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t stage[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int D = a.D, nbr = D >> 3;
  const int rpw = a.rows_wg >> 2;
  const int64_t r0 = (int64_t)blockIdx.x * a.rows_wg;
  const bool a_lay = a.a_order == RL_ORDER_A_LAYOUT;

  for (int i = 0; i < rpw; i++) {
    const int lr = wave * rpw + i;  // row within the workgroup
    const int64_t r = r0 + lr;
    if (r >= a.M) break;
    const uint16_t* prm = a.params + (r < a.split_row ? 2 * (int64_t)D : 0);  // [g | sc] row

    // x' = bf16(x + g * branch) of block j from its loaded words, kept as its bf16 bits (two per register: the row
    // stays resident at 4 registers per block); sum for the mean. g * branch is exact in fp32: one rounding in the
    // fma, then RNE to bf16; the mean's sum takes the bf16 pairs with one dot2 against (1, 1).
    u32x4 v[NB];
    float s = 0.f;
    auto first = [&](int j, const u32x4& xw4, const u32x4& gw4, const float (&bf)[8]) {
      const int cb = lane + 64 * j;
      float xf[8], gf[8];
      unpack8(xw4, xf);
      unpack8(gw4, gf);
      uint32_t xw[4];
      const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int i2 = 2 * e;
        xw[e] = pack_bf16_rne(fmaf(gf[i2], bf[i2], xf[i2]), fmaf(gf[i2 + 1], bf[i2 + 1], xf[i2 + 1]));
        s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, xw[e]), one, s, false);
      }
      v[j] = u32x4{xw[0], xw[1], xw[2], xw[3]};
      if (a.x_out) store_x<NT>(a.x_out + r * a.ld_xo + cb * 8, v[j]);
    };
    // a packed branch block from its 12-byte window (block blk starts at byte 9 blk): exact, as from_bfp16
    auto branch_block = [&](int64_t blk, uint32_t w0, uint32_t w1, uint32_t w2, float (&bf)[8]) {
      const uint32_t o = (uint32_t)(blk & 3);  // (9 * blk) % 4
      const uint32_t lo = __builtin_amdgcn_alignbyte(w1, w0, o);
      const uint32_t hi = __builtin_amdgcn_alignbyte(w2, w1, o);
      const int sh = (int)(lo & 0xFFu) - 133;
      const int32_t q[8] = {(int8_t)(lo >> 8), (int8_t)(lo >> 16), (int8_t)(lo >> 24), (int8_t)hi,
                            (int8_t)(hi >> 8), (int8_t)(hi >> 16), (int8_t)(hi >> 24), (int8_t)(w2 >> (8 * o))};
#pragma unroll
      for (int e = 0; e < 8; e++) bf[e] = __builtin_amdgcn_ldexpf((float)q[e], sh);
    };
    if constexpr (NB <= 8) {
      // chunks of at most 6 blocks (4 for 7 or 8 blocks): every load of a chunk (x, the gate row and the branch;
      // for the packed branch the block's 12-byte window in .x .y .z) is issued before any of them is used, so a
      // row takes one or two memory round trips rather than one per block
      constexpr int kMaxC = NB <= 6 ? 6 : 4, kNC = (NB + kMaxC - 1) / kMaxC, kC = (NB + kNC - 1) / kNC;
#pragma unroll
      for (int j0 = 0; j0 < NB; j0 += kC) {
        u32x4 xr[kC], gr[kC], brw[kC];
#pragma unroll
        for (int c = 0; c < kC; c++) {
          const int cb = lane + 64 * (j0 + c);
          xr[c] = gr[c] = brw[c] = u32x4{0u, 0u, 0u, 0u};
          if (j0 + c < NB && cb < nbr) {
            xr[c] = *reinterpret_cast<const u32x4*>(a.x + r * a.ldx + cb * 8);
            gr[c] = *reinterpret_cast<const u32x4*>(prm + cb * 8);
            if constexpr (BR == 1) {
              brw[c] = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.br) + r * a.ld_br + cb * 8);
            } else if constexpr (BR == 2) {
              const Window w = load_window_safe(static_cast<const uint8_t*>(a.br), r * nbr + cb, a.M * nbr);
              brw[c] = u32x4{w.w0, w.w1, w.w2, 0u};
            }
          }
        }
#pragma unroll
        for (int c = 0; c < kC; c++) {
          const int j = j0 + c;
          if (j >= NB) break;
          v[j] = u32x4{0u, 0u, 0u, 0u};
          if (lane + 64 * j < nbr) {
            float bf[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if constexpr (BR == 1) unpack8(brw[c], bf);
            if constexpr (BR == 2) branch_block(r * nbr + lane + 64 * j, brw[c].x, brw[c].y, brw[c].z, bf);
            first(j, xr[c], gr[c], bf);
          }
        }
        // the next chunk's loads stay behind this chunk's math (registers)
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // above 8 blocks: one block at a time, the branch's format tested at run time
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const int cb = lane + 64 * j;
        v[j] = u32x4{0u, 0u, 0u, 0u};
        if (cb < nbr) {
          float bf[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          if (a.br && a.br_fmt == RL_BRANCH_BF16) {
            unpack8(*reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.br) + r * a.ld_br + cb * 8), bf);
          } else if (a.br) {
            const Window w = load_window_safe(static_cast<const uint8_t*>(a.br), r * nbr + cb, a.M * nbr);
            branch_block(r * nbr + cb, w.w0, w.w1, w.w2, bf);
          }
          first(j, *reinterpret_cast<const u32x4*>(a.x + r * a.ldx + cb * 8),
                *reinterpret_cast<const u32x4*>(prm + cb * 8), bf);
        }
      }
    }
    // up to 8 blocks, the scale row's loads go out before the two reductions
    constexpr bool kScaleEarly = NB <= 8;
    u32x4 sr[kScaleEarly ? NB : 1];
    if constexpr (kScaleEarly) {
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const int cb = lane + 64 * j;
        sr[j] = u32x4{0u, 0u, 0u, 0u};
        if (cb < nbr) sr[j] = *reinterpret_cast<const u32x4*>(prm + D + cb * 8);
      }
    }
    s = wave_sum(s);
    const float mean = a.norm == RL_NORM_LAYER ? s / (float)D : 0.f;
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NB; j++) {
      if (lane + 64 * j < nbr) {
        float xf[8];
        unpack8(v[j], xf);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float d = xf[e] - mean;
          ss = fmaf(d, d, ss);
        }
      }
    }
    ss = wave_sum(ss);
    const float rstd = __builtin_amdgcn_rsqf(ss / (float)D + 1e-6f);

    // y = (x' - mean) * rstd * sc -> bfp16
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const int cb = lane + 64 * j;
      if (cb < nbr) {
        float sf[8], xf[8];
        if constexpr (kScaleEarly)
          unpack8(sr[j], sf);
        else
          unpack8(*reinterpret_cast<const u32x4*>(prm + D + cb * 8), sf);
        unpack8(v[j], xf);
        uint32_t u[8];
        int32_t q[8];
        u32x4 bw;
#pragma unroll
        for (int e = 0; e < 8; e++) u[e] = __float_as_uint((xf[e] - mean) * rstd * sf[e]);
        const uint32_t E = encode_block(u, q, bw);
        if (a.a_deq) *reinterpret_cast<u32x4*>(a.a_deq + r * a.ld_a + cb * 8) = bw;
        if (a.a_packed) {
          const int pos = a_lay ? (cb >> 3) * 128 + (cb & 7) * 16 + (lr >> 3) * 8 + (lr & 7) : lr * nbr + cb;
          uint8_t* p = stage + pos * kBlockBytes;
          p[0] = (uint8_t)E;
#pragma unroll
          for (int e = 0; e < 8; e++) p[1 + e] = (uint8_t)(int8_t)q[e];
        }
      }
    }
  }

  if (!a.a_packed) return;
  __syncthreads();
  if (a_lay) {
    // rows r0 .. r0 + 15 = band sbr of A tile mt: for K tile kt, 128 blocks at block ((mt * KT + kt) * 8 + sbr) * 128
    const int KT = D >> 6;
    const int64_t mt = r0 >> 7, sbr = (r0 >> 4) & 7;
    const int chunks = KT * 72;  // 1152 bytes = 72 x 16 per K tile
    for (int c = threadIdx.x; c < chunks; c += kLnThreads) {
      const int kt = c / 72, w = c - kt * 72;
      uint8_t* dst = a.a_packed + (((mt * KT + kt) * 8 + sbr) * 128) * kBlockBytes + 16 * w;
      *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(stage + kt * 1152 + 16 * w);
    }
  } else {
    // rows r0 .. r0 + nrows - 1 are one span; r0 * nbr * 9 is a multiple of 16 (r0 % 4 == 0, nbr % 8 == 0)
    const int64_t nrows = min((int64_t)a.rows_wg, a.M - r0);
    const int bytes = (int)(nrows * nbr * kBlockBytes);
    uint8_t* dst = a.a_packed + r0 * nbr * kBlockBytes;
    const int full = bytes / 16;
    for (int c = threadIdx.x; c < full; c += kLnThreads)
      *reinterpret_cast<u32x4*>(dst + 16 * c) = *reinterpret_cast<const u32x4*>(stage + 16 * c);
    for (int c = full * 16 + threadIdx.x; c < bytes; c += kLnThreads) dst[c] = stage[c];
  }
}

template <int NB, int BR, bool NT>
static int launch_nb_br(const LnArgs& a, hipStream_t st) {
  const int64_t lds = a.a_packed ? (int64_t)a.rows_wg * (a.D / 8) * kBlockBytes : 0;
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&ln_kernel<NB, BR, NT>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail(RL_ERR_DEVICE, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  }
  const dim3 grid((unsigned)((a.M + a.rows_wg - 1) / a.rows_wg));
  hipLaunchKernelGGL((ln_kernel<NB, BR, NT>), grid, dim3(kLnThreads), (unsigned)lds, st, a);
  return launch_status("rl_ln_modulate");
}

// the branch's format is a template parameter, so that the first pass is straight-line code whose loads all issue
// before the first use
template <int NB, bool NT>
static int launch_nb_nt(const LnArgs& a, hipStream_t st) {
  if constexpr (NB > 8) {
    return launch_nb_br<NB, -1, NT>(a, st);
  } else {
    if (!a.br) return launch_nb_br<NB, 0, NT>(a, st);
    if (a.br_fmt == RL_BRANCH_BF16) return launch_nb_br<NB, 1, NT>(a, st);
    return launch_nb_br<NB, 2, NT>(a, st);
  }
}

template <int NB>
static int launch_nb(const LnArgs& a, hipStream_t st) {
  const int br = !a.br ? 0 : a.br_fmt == RL_BRANCH_BF16 ? 1 : 2;
  return a.x_out && past_caches(a.M, a.D, br) ? launch_nb_nt<NB, true>(a, st) : launch_nb_nt<NB, false>(a, st);
}

template <int NB>
static int launch_upto(int nb, const LnArgs& a, hipStream_t st) {
  if constexpr (NB > kLnMaxNB) {
    return fail(RL_ERR_SHAPE, "D %d too large", a.D);
  } else {
    if (nb <= NB) return launch_nb<NB>(a, st);
    return launch_upto<NB + 1>(nb, a, st);
  }
}

// ---- the same op on streams: x, the branch and x' in the C-stream order, A packed in the A layout --------------------
//
// Workgroup = 8 rows (one br half of a 16-row band), 512 threads; thread f + 512 j takes the 8-value block (row rib =
// f & 7, 16-byte column blocks in stream order), so that 16 consecutive lanes hold 16 consecutive blocks of the
// stream: a wave's load or store is four runs of 256 bytes (bf16) or 144 bytes (packed). The two halves of a band
// share their cache lines; xcd_remap puts them on one XCD. A row's values are spread over the lanes of equal rib of
// all 8 waves, so the mean and the variance take a wave reduction, an LDS exchange and a barrier each.
// HBM-bound: 2 + 9/8 (or 2) bytes read and 2 + 9/8 written per value, once. 4096 x 4096 with a packed branch (105 MB)
// replaces index-tensor permutations of x and x', a dequantize pass, the row-major kernel and a copy (1063 us); it takes
// 22.9 us (4.6 TB/s; 28.1 with cached stores of x'). All of a row's loads are issued before the first use; 8 rows x D
// values stay in registers as bf16 pairs (32 VGPRs at D = 4096: the 512 workgroups of 4096 rows are all resident, 2 per
// CU).
constexpr int kLsThreads = 512, kLsRows = 8;

struct LnStreamArgs {
  const uint16_t* x;
  const void* br;
  const uint16_t* params;
  int64_t split_row;
  int32_t norm;
  uint16_t* x_out;
  uint8_t* a_packed;
  int32_t D;
};

// Sum over the 8 lanes of equal lane & 7, every lane getting the result
__device__ __forceinline__ float sum_rib(float v) {
  v += dpp_f<0x128>(v);  // row_ror:8
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// NB = blocks per thread (D / 512); BR: 0 no branch, 1 bf16, 2 packed
template <int NB, int BR>
__global__ __launch_bounds__(kLsThreads, NB <= 8 ? 4 : 2) void ln_stream_kernel(LnStreamArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t stage[];
  __shared__ float red[2][kLsThreads / 64][kLsRows];
  const int tid = threadIdx.x, lane = tid & 63, rib = tid & 7;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int D = a.D;
  const int64_t r0 = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * kLsRows;
  const uint16_t* prm = a.params + (r0 + rib < a.split_row ? 2 * D : 0);  // [g | sc] row
  // stream block of item j: tile column c128 = 4 j + tid / 128 (8192 blocks apart), then sbc, br, bc, rib
  const int sbc = (tid >> 4) & 7, bc = (tid >> 3) & 1;
  const int64_t blk0 = ((r0 >> 9) * (D >> 7) + (tid >> 7)) * 8192 + ((r0 >> 7) & 3) * 2048 + ((r0 >> 4) & 7) * 256 +
                       sbc * 32 + ((r0 >> 3) & 1) * 16 + bc * 8 + rib;
  const int cb0 = (tid >> 7) * 16 + sbc * 2 + bc;  // column block; + 64 j
  constexpr int kStep = 4 * 8192;                  // stream blocks between items j and j + 1

  u32x4 v[NB];
  float s = 0.f;
  constexpr int kC = NB <= 8 ? NB : (NB + 1) / 2;  // loads in flight: whole rows, or two chunks above D = 4096
#pragma unroll
  for (int j0 = 0; j0 < NB; j0 += kC) {
    u32x4 xr[kC], brw[kC];
#pragma unroll
    for (int c = 0; c < kC; c++) {
      if (j0 + c >= NB) break;
      const int64_t blk = blk0 + (int64_t)(j0 + c) * kStep;
      xr[c] = *reinterpret_cast<const u32x4*>(a.x + blk * 8);
      if constexpr (BR == 1) brw[c] = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.br) + blk * 8);
      if constexpr (BR == 2) {
        // the window of a stream's last block (odd index) ends with the block
        const Window w = load_window(static_cast<const uint8_t*>(a.br), blk * 9);
        brw[c] = u32x4{w.w0, w.w1, w.w2, 0u};
      }
    }
#pragma unroll
    for (int c = 0; c < kC; c++) {
      const int j = j0 + c;
      if (j >= NB) break;
      const int64_t blk = blk0 + (int64_t)j * kStep;
      u32x4 xw = xr[c];
      if constexpr (BR != 0) {
        float xf[8], gf[8], bf[8];
        unpack8(xr[c], xf);
        unpack8(*reinterpret_cast<const u32x4*>(prm + (cb0 + 64 * j) * 8), gf);
        if constexpr (BR == 1) {
          unpack8(brw[c], bf);
        } else {
          const uint32_t o = (uint32_t)(rib & 3);  // (9 * blk) % 4: blk % 4 == rib % 4
          const uint32_t lo = __builtin_amdgcn_alignbyte(brw[c].y, brw[c].x, o);
          const uint32_t hi = __builtin_amdgcn_alignbyte(brw[c].z, brw[c].y, o);
          const int sh = (int)(lo & 0xFFu) - 133;
          const int32_t q[8] = {(int8_t)(lo >> 8), (int8_t)(lo >> 16), (int8_t)(lo >> 24), (int8_t)hi,
                                (int8_t)(hi >> 8), (int8_t)(hi >> 16), (int8_t)(hi >> 24),
                                (int8_t)(brw[c].z >> (8 * o))};
#pragma unroll
          for (int e = 0; e < 8; e++) bf[e] = __builtin_amdgcn_ldexpf((float)q[e], sh);
        }
#pragma unroll
        for (int e = 0; e < 4; e++)
          xw[e] = pack_bf16_rne(fmaf(gf[2 * e], bf[2 * e], xf[2 * e]), fmaf(gf[2 * e + 1], bf[2 * e + 1], xf[2 * e + 1]));
      }
      const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t w = xw[e];
        s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), one, s, false);
      }
      v[j] = xw;
      store_stream(a.x_out + blk * 8, xw);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // the scale row's loads go out before the reductions
  u32x4 sr[NB <= 8 ? NB : 1];
  if constexpr (NB <= 8) {
#pragma unroll
    for (int j = 0; j < NB; j++) sr[j] = *reinterpret_cast<const u32x4*>(prm + D + (cb0 + 64 * j) * 8);
  }
  auto row_sum = [&](int i, float p) {
    p = sum_rib(p);
    if (lane < kLsRows) red[i][wave][lane] = p;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < kLsThreads / 64; w++) t += red[i][w][rib];
    return t;
  };
  float mean = 0.f;
  if (a.norm == RL_NORM_LAYER) mean = row_sum(0, s) / (float)D;
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < NB; j++) {
    float xf[8];
    unpack8(v[j], xf);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float d = xf[e] - mean;
      ss = fmaf(d, d, ss);
    }
  }
  const float rstd = __builtin_amdgcn_rsqf(row_sum(1, ss) / (float)D + 1e-6f);

  // y -> bfp16; the 8 rows' blocks of column block cb are 72 consecutive bytes of the A layout, staged at 72 cb
#pragma unroll
  for (int j = 0; j < NB; j++) {
    const int cb = cb0 + 64 * j;
    float sf[8], xf[8];
    if constexpr (NB <= 8)
      unpack8(sr[j], sf);
    else
      unpack8(*reinterpret_cast<const u32x4*>(prm + D + cb * 8), sf);
    unpack8(v[j], xf);
    uint32_t u[8];
    int32_t q[8];
    u32x4 bw;
#pragma unroll
    for (int e = 0; e < 8; e++) u[e] = __float_as_uint((xf[e] - mean) * rstd * sf[e]);
    const uint32_t E = encode_block(u, q, bw);
    uint8_t* p = stage + (cb * 8 + rib) * kBlockBytes;
    p[0] = (uint8_t)E;
#pragma unroll
    for (int e = 0; e < 8; e++) p[1 + e] = (uint8_t)(int8_t)q[e];
  }
  __syncthreads();
  // A tile (mt, kt): 8 bands x 8 column blocks x 144 bytes, of which this workgroup's half is 72
  const int64_t KT = D >> 6;
  uint8_t* dst = a.a_packed + ((r0 >> 7) * KT * 8 + ((r0 >> 4) & 7)) * 1152 + ((r0 >> 3) & 1) * 72;
  for (int c = tid; c < (D >> 3) * 9; c += kLsThreads) {
    const int cb = c / 9, w = c - cb * 9;
    *reinterpret_cast<uint2*>(dst + (cb >> 3) * (8 * 1152) + (cb & 7) * 144 + 8 * w) =
        *reinterpret_cast<const uint2*>(stage + 8 * c);
  }
}

template <int NB>
static int launch_stream(const LnStreamArgs& a, int br, int64_t M, hipStream_t st) {
  const dim3 grid((unsigned)(M / kLsRows)), block(kLsThreads);
  const int lds = a.D * kBlockBytes;  // 8 rows x D / 8 blocks
  auto go = [&](auto kernel) {
    if (lds > 48 * 1024) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return fail(RL_ERR_DEVICE, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    hipLaunchKernelGGL(kernel, grid, block, (unsigned)lds, st, a);
    return launch_status("rl_ln_modulate_stream");
  };
  if (br == 0) return go(ln_stream_kernel<NB, 0>);
  return br == 1 ? go(ln_stream_kernel<NB, 1>) : go(ln_stream_kernel<NB, 2>);
}

}  // namespace rl

extern "C" int rl_ln_modulate(const uint16_t* x, int64_t ldx, const void* branch, int32_t br_fmt, int64_t ld_br,
                              const uint16_t* params, int64_t split_row, int32_t norm, uint16_t* x_out, int64_t ld_xo,
                              uint8_t* a_packed, int32_t a_order, uint16_t* a_deq, int64_t ld_a, int64_t M, int64_t D,
                              void* stream) {
  using namespace rl;
  // the leading dimension of an absent operand is not used
  if (!branch) ld_br = D;
  if (!x_out) ld_xo = D;
  if (!a_deq) ld_a = D;
  int s = rl_validate_ln(ldx, br_fmt, ld_br, norm, ld_xo, a_order, ld_a, split_row, M, D);
  if (s) return s;
  if (!x || !params) return fail(RL_ERR_NULL, "x or params is NULL");
  if (!x_out && !a_packed && !a_deq) return fail(RL_ERR_NULL, "every output is NULL");
  if (((uintptr_t)x | (uintptr_t)params | (uintptr_t)x_out | (uintptr_t)a_deq | (uintptr_t)a_packed) % 16)
    return fail(RL_ERR_ALIGN, "x, params and the outputs must be 16-byte aligned");
  if (branch && (uintptr_t)branch % (br_fmt == RL_BRANCH_BF16 ? 16 : 4))
    return fail(RL_ERR_ALIGN, "branch must be 16-byte (bf16) or 4-byte (packed) aligned");
  if ((s = check_device())) return s;
  LnArgs a;
  a.x = x; a.ldx = ldx;
  a.br = branch; a.br_fmt = br_fmt; a.ld_br = ld_br;
  a.params = params; a.split_row = split_row; a.norm = norm;
  a.x_out = x_out; a.ld_xo = ld_xo;
  a.a_packed = a_packed; a.a_order = a_order;
  a.a_deq = a_deq; a.ld_a = ld_a;
  a.M = M; a.D = (int32_t)D;
  a.rows_wg = (a_packed && a_order == RL_ORDER_A_LAYOUT) ? 16 : 4;
  const int nb = (int)((D / 8 + 63) / 64);
  return launch_upto<1>(nb, a, static_cast<hipStream_t>(stream));
}

extern "C" int rl_ln_modulate_stream(const uint16_t* x, const void* branch, int32_t br_fmt, const uint16_t* params,
                                     int64_t split_row, int32_t norm, uint16_t* x_out, uint8_t* a_packed, int64_t M,
                                     int64_t D, void* stream) {
  using namespace rl;
  int s = rl_validate_ln(D, br_fmt, D, norm, D, RL_ORDER_A_LAYOUT, D, split_row, M, D);
  if (s) return s;
  if (M % 512 || D % 1024)
    return fail(RL_ERR_SHAPE, "M %lld D %lld: the C-stream order needs M %% 512 == 0 and D %% 1024 == 0", (long long)M,
                (long long)D);
  if (!x || !params || !x_out || !a_packed) return fail(RL_ERR_NULL, "x, params, x_out or a_packed is NULL");
  if (((uintptr_t)x | (uintptr_t)params | (uintptr_t)x_out | (uintptr_t)a_packed) % 16)
    return fail(RL_ERR_ALIGN, "x, params and the outputs must be 16-byte aligned");
  if (branch && (uintptr_t)branch % (br_fmt == RL_BRANCH_BF16 ? 16 : 4))
    return fail(RL_ERR_ALIGN, "branch must be 16-byte (bf16) or 4-byte (packed) aligned");
  if ((s = check_device())) return s;
  LnStreamArgs a;
  a.x = x; a.br = branch; a.params = params; a.split_row = split_row; a.norm = norm;
  a.x_out = x_out; a.a_packed = a_packed; a.D = (int32_t)D;
  const int br = !branch ? 0 : br_fmt == RL_BRANCH_BF16 ? 1 : 2;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  switch (D / 1024) {
    case 1: return launch_stream<2>(a, br, M, st);
    case 2: return launch_stream<4>(a, br, M, st);
    case 3: return launch_stream<6>(a, br, M, st);
    case 4: return launch_stream<8>(a, br, M, st);
    case 5: return launch_stream<10>(a, br, M, st);
    case 6: return launch_stream<12>(a, br, M, st);
    case 7: return launch_stream<14>(a, br, M, st);
    default: return launch_stream<16>(a, br, M, st);
  }
}
