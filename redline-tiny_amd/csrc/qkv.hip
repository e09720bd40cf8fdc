// QKV post: the QKV GEMM's output -> attention Q / K / V (per-head RMSNorm * w, RoPE, bfp16 tiles).
//
// Replaces the QKV-post artifact of kernels/glue/qkv_design.py:40-118 (microkernels q_post / k_post / v_post,
// kernels/glue/qkv_post.cc:134-177) that run_qkv.qkv32_npu drives (redline/run_qkv.py:67-82). One workgroup takes
// one part (q, k or v) of one head of one 64-token tile: 64 x 128 values (16 KB of bf16 in), and writes the 9216-byte
// tile the attention kernel reads. The pass is HBM-bound: 2 bytes read and 9/8 bytes written per value (plus 2 per
// value for each bf16 output requested). Small workgroups (9 KB of LDS) keep many tiles in flight per CU.
//
// Q and K: thread (token r, 8-dim block bc) holds 8 dims of one token; the 16 threads of a token (16 lanes of a wave)
// reduce the sum of squares across their lanes. RoPE pairs (2i, 2i + 1) lie inside a block, so each thread rotates
// its own 4 pairs. V: each thread reads the 8 tokens of one dim that a V block holds (and writes them, as one 16-byte
// store, to the optional V^T output). The tile is assembled in LDS in output order and written with 16-byte stores.
#include <math.h>

#include "rlbfp.h"
#include "rlbfp_device.h"
#include "rlbfp_host.h"

namespace rl {

constexpr int kQkvThreads = 256;
constexpr int kHeadDim = 128;
constexpr int kTileTokens = 64;
constexpr int kTileBlocks = kTileTokens * kHeadDim / 8;     // 1024
constexpr int kTile9 = kTileBlocks * kBlockBytes;          // 9216

struct QkvArgs {
  const uint16_t* C;
  int64_t ldc;
  int64_t M;
  int32_t hq, hkv;  // q heads, k / v heads (equal for the DiT; grouped-query attention has hq a multiple of hkv)
  const uint16_t* cos;
  const uint16_t* sin;
  const uint16_t* wq;
  const uint16_t* wk;
  uint8_t* q_tiles;
  uint8_t* kv_tiles;
  uint16_t* q;
  uint16_t* k;
  uint16_t* v;
};

__device__ __forceinline__ void unpack8f(u32x4 v, float f[8]) {
  f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xFFFF0000u);
  f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xFFFF0000u);
  f[4] = __uint_as_float(v.z << 16); f[5] = __uint_as_float(v.z & 0xFFFF0000u);
  f[6] = __uint_as_float(v.w << 16); f[7] = __uint_as_float(v.w & 0xFFFF0000u);
}

// Sum over each row of 16 lanes, every lane of the row getting the same value: quad swaps, then half-row and row
// mirrors, each one v_add_f32 with a DPP operand (no LDS round trip).
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_f<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_f<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_f<0x141>(v);  // row_half_mirror: lane i <- 7 - i within each 8
  v += dpp_f<0x140>(v);  // row_mirror: lane i <- 15 - i
  return v;
}

__device__ __forceinline__ void stage_block(uint8_t* stage, int pos, uint32_t E, const int32_t q[8]) {
  uint8_t* p = stage + pos * kBlockBytes;
  p[0] = (uint8_t)E;
#pragma unroll
  for (int e = 0; e < 8; e++) p[1 + e] = (uint8_t)(int8_t)q[e];
}

// One token's 8 dims of a head (the other 15 blocks in the lanes of its row of 16): rope(x / rms * w) as float32 bits
__device__ __forceinline__ void rms_rope8(const float (&xf)[8], const float (&wf)[8], uint2 cr, uint2 sr,
                                          uint32_t (&u)[8]) {
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) ss = fmaf(xf[e], xf[e], ss);
  ss = row16_sum(ss);  // the token's 16 lanes
  const float inv = __builtin_amdgcn_rsqf(ss / (float)kHeadDim + 1e-6f);
  const float c4[4] = {__uint_as_float(cr.x << 16), __uint_as_float(cr.x & 0xFFFF0000u),
                       __uint_as_float(cr.y << 16), __uint_as_float(cr.y & 0xFFFF0000u)};
  const float s4[4] = {__uint_as_float(sr.x << 16), __uint_as_float(sr.x & 0xFFFF0000u),
                       __uint_as_float(sr.y << 16), __uint_as_float(sr.y & 0xFFFF0000u)};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float ev = xf[2 * i] * inv * wf[2 * i], od = xf[2 * i + 1] * inv * wf[2 * i + 1];
    u[2 * i] = __float_as_uint(ev * c4[i] - od * s4[i]);
    u[2 * i + 1] = __float_as_uint(ev * s4[i] + od * c4[i]);
  }
}

// TILES / NATIVE: whether any tile / any head-major bf16 output is requested (the other's work is compiled out).
template <bool TILES, bool NATIVE>
__global__ __launch_bounds__(kQkvThreads) void qkv_post_kernel(QkvArgs a) {
  __shared__ __attribute__((aligned(16))) uint8_t stage[kTile9];
  const int tid = threadIdx.x;
  // workgroup = (part, head) item j of 64-token tile t; C's columns are [q hq x 128 | k hkv x 128 | v hkv x 128].
  // With hq == hkv the three parts of one (head, tile) are neighbours in launch order (j = 3 h + part); otherwise
  // the q heads come first, then k and v head g side by side.
  const int per_tile = a.hq + 2 * a.hkv;
  const int t = blockIdx.x / per_tile, j = blockIdx.x - t * per_tile;
  int part, h;
  if (a.hq == a.hkv) {
    part = j % 3; h = j / 3;
  } else if (j < a.hq) {
    part = 0; h = j;
  } else {
    part = 1 + ((j - a.hq) & 1); h = (j - a.hq) >> 1;
  }
  const int64_t row0 = (int64_t)t * kTileTokens;
  const int64_t col0 = (part == 0 ? 0 : (int64_t)a.hq * kHeadDim + (part - 1) * (int64_t)a.hkv * kHeadDim) +
                       (int64_t)h * kHeadDim;
  const bool tiles = TILES && (part == 0 ? a.q_tiles != nullptr : a.kv_tiles != nullptr);

  if (part < 2) {
    // Q (part 0) and K (part 1): thread = (token rr + 16 pass, dim block bc)
    const int bc = tid & 15, rr = tid >> 4;
    float wf[8];
    unpack8f(*reinterpret_cast<const u32x4*>((part ? a.wk : a.wq) + bc * 8), wf);
    uint16_t* nat = NATIVE ? (part ? a.k : a.q) : nullptr;
    // every pass's loads (the token's 8 values, its cos and sin) are issued before the first use: the encoder's
    // rarely taken integer path is a branch that later loads are not hoisted over
    u32x4 xr[4];
    uint2 cr4[4], sr4[4];
#pragma unroll
    for (int pass = 0; pass < 4; pass++) {
      const int64_t row = row0 + pass * 16 + rr;
      xr[pass] = *reinterpret_cast<const u32x4*>(a.C + row * a.ldc + col0 + bc * 8);
      cr4[pass] = *reinterpret_cast<const uint2*>(a.cos + row * 64 + bc * 4);
      sr4[pass] = *reinterpret_cast<const uint2*>(a.sin + row * 64 + bc * 4);
    }
#pragma unroll
    for (int pass = 0; pass < 4; pass++) {
      const int r = pass * 16 + rr;
      const int64_t row = row0 + r;
      float xf[8];
      unpack8f(xr[pass], xf);
      uint32_t u[8];
      int32_t q[8];
      u32x4 bw;
      rms_rope8(xf, wf, cr4[pass], sr4[pass], u);
      const uint32_t E = encode_block(u, q, bw);
      if (nat) *reinterpret_cast<u32x4*>(nat + (((int64_t)h * a.M + row) * kHeadDim + bc * 8)) = bw;
      // a_layout(64, 128) for Q and b_layout(K^T, 128, 64) for K order a tile's blocks the same way:
      // 16-token band, 8-dim block, 8-token half, token
      if (tiles) stage_block(stage, (((r >> 4) * 16 + bc) * 2 + ((r >> 3) & 1)) * 8 + (r & 7), E, q);
    }
  } else {
    // V: thread = (dim d, 8-token block kb), reading its 8 tokens of one dim (consecutive lanes read consecutive
    // dims: 128 contiguous bytes of a row per load); b_layout(V, 64, 128): 16-dim band, token block, 8-dim half, dim
    // all four items' loads first, as for Q and K
    uint16_t vr[4][8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int item = tid + kQkvThreads * i, d = item & 127, kb = item >> 7;
#pragma unroll
      for (int e = 0; e < 8; e++) vr[i][e] = a.C[(row0 + kb * 8 + e) * a.ldc + col0 + d];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int item = tid + kQkvThreads * i, d = item & 127, kb = item >> 7;
      uint32_t u[8];
      int32_t q[8];
      u32x4 bw;
#pragma unroll
      for (int e = 0; e < 8; e++) u[e] = (uint32_t)vr[i][e] << 16;
      const uint32_t E = encode_block(u, q, bw);
      if (NATIVE && a.v)  // V^T: the block's 8 tokens are contiguous in row d
        *reinterpret_cast<u32x4*>(a.v + ((int64_t)h * kHeadDim + d) * a.M + row0 + kb * 8) = bw;
      if (tiles) stage_block(stage, (((d >> 4) * 8 + kb) * 2 + ((d >> 3) & 1)) * 8 + (d & 7), E, q);
    }
  }
  if (!tiles) return;
  __syncthreads();
  const int64_t T = a.M / kTileTokens;
  uint8_t* dst = part == 0 ? a.q_tiles + ((int64_t)h * T + t) * kTile9
                           : a.kv_tiles + (((int64_t)h * T + t) * 2 + (part - 1)) * kTile9;
  for (int c = tid; c < kTile9 / 16; c += kQkvThreads)
    *reinterpret_cast<u32x4*>(dst + 16 * c) = *reinterpret_cast<const u32x4*>(&stage[16 * c]);
}

// ---- the same pass on the artifact's own buffers ----------------------------------------------------------------------
//
// C is the QKV GEMM's C stream (bfp16, or bf16 in that element order), cos / sin come from the NPU kernel's table
// (redline/run_qkv.py:52-64). In both orders the 64 x 128 tile of one head is contiguous: 4 row bands x 8 column
// bands x (2 x 2) 8 x 8 blocks, 9216 bytes of bfp16 (16 KB of bf16, 16 KB of table), so a workgroup reads one run of C
// and one of the table and writes one run of tiles. Thread (column block bc = tid & 15, row quad) takes rows 4 quad ..
// + 3 of one 8-dim block: four consecutive blocks of C (36 or 64 bytes), of the table (32 + 32) and of the output tile
// (36 bytes). A token's 16 blocks sit in 16 neighbouring lanes, as in qkv_post_kernel. V goes through a 16 KB LDS tile
// of decoded values, read down the columns.
// HBM-bound: 9/8 (or 2) bytes read and 9/8 written per value. It replaces a decode pass, index passes over the table and
// the row-major kernel: at 4096 x 12288 this kernel takes 30 us (113 MB of tiles and 34 MB of table re-read by every
// head, from L2), and the attention step that holds it went from 1155 to 1025 us.
struct QkvStreamArgs {
  const void* C;
  int32_t n_cols;
  int32_t hq, hkv;
  int64_t M;
  const uint16_t* tabs;  // (M / 64, kTabLen)
  uint8_t* q_tiles;
  uint8_t* kv_tiles;
};
constexpr int kTabLen = 128 * 64 + 2 * 128;

// Four blocks' values, row i's block in u[i] (float32 bits) -> their 36 bytes at p
__device__ __forceinline__ void encode_store4(uint8_t* p, const uint32_t (&u)[4][8]) {
  uint32_t E[4], ql[4], qh[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int32_t q[8];
    u32x4 bw;
    E[i] = encode_block(u[i], q, bw);
    ql[i] = (q[0] & 0xFFu) | ((q[1] & 0xFFu) << 8) | ((q[2] & 0xFFu) << 16) | ((uint32_t)q[3] << 24);
    qh[i] = (q[4] & 0xFFu) | ((q[5] & 0xFFu) << 8) | ((q[6] & 0xFFu) << 16) | ((uint32_t)q[7] << 24);
  }
  store_blocks4(p, E, ql, qh);
}

// PACKED: C as bfp16 blocks, else bf16
template <bool PACKED>
__global__ __launch_bounds__(kQkvThreads) void qkv_stream_kernel(QkvStreamArgs a) {
  typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
  constexpr int kVRow = kHeadDim + 8;  // LDS row of V values: 16 bytes of padding
  __shared__ __attribute__((aligned(16))) uint8_t stage[kTile9];
  __shared__ __attribute__((aligned(16))) uint16_t vals[kTileTokens * kVRow];
  const int tid = threadIdx.x, bc = tid & 15, quad = tid >> 4;  // quad: row 4 quad of the 64
  const int per_tile = a.hq + 2 * a.hkv;
  const int t = blockIdx.x / per_tile, j = blockIdx.x - t * per_tile;
  int part, h;
  if (a.hq == a.hkv) {
    part = j % 3; h = j / 3;
  } else if (j < a.hq) {
    part = 0; h = j;
  } else {
    part = 1 + ((j - a.hq) & 1); h = (j - a.hq) >> 1;
  }
  const int col128 = part == 0 ? h : a.hq + (part - 1) * a.hkv + h;
  // blocks of a tile: row band, column band, row half, column half, row in 8
  const int loc = ((((quad >> 2) * 8 + (bc >> 1)) * 2 + ((quad >> 1) & 1)) * 2 + (bc & 1)) * 8 + (quad & 1) * 4;
  // 64-row tile t of 128-column group col128: row group t / 8, then column groups, 128-row groups, 16-row bands
  const int64_t blk = ((int64_t)(t >> 3) * (a.n_cols >> 7) + col128) * 8192 + (t & 7) * 1024 + loc;
  u32x4 x[4];
  if constexpr (PACKED) {
    const uint8_t* src = static_cast<const uint8_t*>(a.C) + 9 * blk;
    const u32x4 b0 = reinterpret_cast<const u32x4_a4*>(src)[0], b1 = reinterpret_cast<const u32x4_a4*>(src)[1];
    const uint32_t w[9] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w, reinterpret_cast<const uint32_t*>(src)[8]};
#pragma unroll
    for (int i = 0; i < 4; i++)
      x[i] = __builtin_bit_cast(u32x4, decode_window(w[2 * i], w[2 * i + 1], w[2 * i + 2], (uint32_t)i));
  } else {
    const u32x4* src = reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.C) + 8 * blk);
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = src[i];
  }
  uint32_t u[4][8];
  int pos;
  if (part < 2) {
    // the table's block: 8 rows x 4 cos, then 8 rows x 4 sin; its index is loc / 8
    const uint16_t* tab = a.tabs + (int64_t)t * kTabLen + (loc >> 3) * 64 + (quad & 1) * 16;
    uint2 cr4[4], sr4[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      cr4[i] = *reinterpret_cast<const uint2*>(tab + 4 * i);
      sr4[i] = *reinterpret_cast<const uint2*>(tab + 32 + 4 * i);
    }
    float wf[8];
    unpack8f(*reinterpret_cast<const u32x4*>(a.tabs + kTabLen - 256 + part * 128 + bc * 8), wf);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float xf[8];
      unpack8f(x[i], xf);
      rms_rope8(xf, wf, cr4[i], sr4[i], u[i]);
    }
    pos = ((quad >> 2) * 16 + bc) * 16 + (quad & 3) * 4;  // 16-token band, 8-dim block, token
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) *reinterpret_cast<u32x4*>(&vals[(4 * quad + i) * kVRow + 8 * bc]) = x[i];
    __syncthreads();
    // thread (dim quad tid & 31, 8-token block tid >> 5): the 8 tokens of dims 4 dq .. + 3
    const int dq = tid & 31, kb = tid >> 5;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint2 v = *reinterpret_cast<const uint2*>(&vals[(8 * kb + e) * kVRow + 4 * dq]);
      u[0][e] = v.x << 16; u[1][e] = v.x & 0xFFFF0000u;
      u[2][e] = v.y << 16; u[3][e] = v.y & 0xFFFF0000u;
    }
    pos = ((dq >> 2) * 8 + kb) * 16 + (dq & 3) * 4;  // 16-dim band, token block, dim
  }
  encode_store4(stage + pos * kBlockBytes, u);
  __syncthreads();
  const int64_t T = a.M / kTileTokens;
  uint8_t* dst = part == 0 ? a.q_tiles + ((int64_t)h * T + t) * kTile9
                           : a.kv_tiles + (((int64_t)h * T + t) * 2 + (part - 1)) * kTile9;
  for (int c = tid; c < kTile9 / 16; c += kQkvThreads)
    *reinterpret_cast<u32x4*>(dst + 16 * c) = *reinterpret_cast<const u32x4*>(&stage[16 * c]);
}

// ---- attention tiles -> the attention kernel's operands --------------------------------------------------------------
//
// One workgroup decodes one 9216-byte tile: Q and K tiles to 64 rows of 256 bytes (head major), V tiles to 128 rows of
// V^T, 128 bytes each; query tiles past the source range are zeros. Thread t decodes blocks 4 t .. 4 t + 3, a 36-byte
// dword-aligned run (two 16-byte loads and one 4-byte load) holding rows r .. r + 3 (V: dims) of one 8-value block
// column, so each store instruction of a wave fills whole 256-byte (V: 128-byte) rows. HBM-bound: 9/8 bytes read and 2
// written per value; it replaces index-tensor gathers, float32 copies and concatenations of every operand (32 heads, 4096
// queries, 8256 keys: 43 us; with the QKV post's stream form and packed O, the attention step with its two GEMMs took
// 4950 us and takes 1005). Decoding inside the attention kernel instead would cost every workgroup of a head the same
// ~100 VALU instructions per wave and key block, beside 112 of the softmax.
struct TilesArgs {
  const uint8_t* q_tiles;
  int32_t hq, q_all, q_t0, q_n, q_out;  // heads, tiles per head in the source, first tile, tiles there, tiles written
  uint16_t* q;
  const uint8_t* kv[2];  // [head][tile][K | V]; the second may be absent (n = 0)
  int32_t hkv, kv_all[2], kv_t0[2], kv_n[2];
  uint16_t* k;
  uint16_t* vt;
};

__global__ __launch_bounds__(kQkvThreads) void attn_tiles_kernel(TilesArgs a) {
  typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
  const int tid = threadIdx.x;
  const int nkt = a.kv_n[0] + a.kv_n[1];
  const int64_t nk = (int64_t)nkt * kTileTokens;
  int j = blockIdx.x;
  const uint8_t* src;
  uint16_t* dst;
  int64_t ld;
  int row, col;
  bool zero = false;
  const int nq = a.hq * a.q_out;
  if (j < nq || ((j - nq) & 1) == 0) {
    // Q and K: blocks (16-token band, 8-dim block, 8-token half, token)
    row = (tid >> 6) * 16 + (tid & 3) * 4;
    col = (tid >> 2) & 15;
    ld = kHeadDim;
  } else {
    // V: blocks (16-dim band, 8-token block, 8-dim half, dim)
    row = (tid >> 5) * 16 + (tid & 3) * 4;
    col = (tid >> 2) & 7;
    ld = nk;
  }
  if (j < nq) {
    const int h = j / a.q_out, t = j - h * a.q_out;
    zero = t >= a.q_n;
    src = a.q_tiles + ((int64_t)h * a.q_all + a.q_t0 + t) * kTile9;
    dst = a.q + (int64_t)j * kTileTokens * kHeadDim;
  } else {
    j -= nq;
    const int v = j & 1, h = (j >> 1) / nkt, t = (j >> 1) - h * nkt;
    const int b = t >= a.kv_n[0];
    src = a.kv[b] + (((int64_t)h * a.kv_all[b] + a.kv_t0[b] + (b ? t - a.kv_n[0] : t)) * 2 + v) * kTile9;
    dst = v ? a.vt + (int64_t)h * kHeadDim * nk + t * kTileTokens
            : a.k + ((int64_t)h * nk + t * kTileTokens) * kHeadDim;
  }
  u32x4 o[4] = {};
  if (!zero) {
    src += 36 * tid;
    const u32x4 x = reinterpret_cast<const u32x4_a4*>(src)[0], y = reinterpret_cast<const u32x4_a4*>(src)[1];
    const uint32_t w[9] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w, reinterpret_cast<const uint32_t*>(src)[8]};
#pragma unroll
    for (int i = 0; i < 4; i++)
      o[i] = __builtin_bit_cast(u32x4, decode_window(w[2 * i], w[2 * i + 1], w[2 * i + 2], (uint32_t)i));
  }
  dst += row * ld + col * 8;
#pragma unroll
  for (int i = 0; i < 4; i++) *reinterpret_cast<u32x4*>(dst + i * ld) = o[i];
}

}  // namespace rl

extern "C" int rl_qkv_post_gqa(const uint16_t* C, int64_t ldc, int64_t M, int32_t hq, int32_t hkv,
                               const uint16_t* cos, const uint16_t* sin, const uint16_t* wq, const uint16_t* wk,
                               uint8_t* q_tiles, uint8_t* kv_tiles, uint16_t* q, uint16_t* k, uint16_t* v,
                               void* stream) {
  using namespace rl;
  int s = rl_validate_qkv_post_gqa(ldc, M, hq, hkv);
  if (s) return s;
  if (!C || !cos || !sin || !wq || !wk) return fail(RL_ERR_NULL, "C, cos, sin, wq or wk is NULL");
  if (!q_tiles && !kv_tiles && !q && !k && !v) return fail(RL_ERR_NULL, "every output is NULL");
  if (((uintptr_t)C | (uintptr_t)wq | (uintptr_t)wk | (uintptr_t)q_tiles | (uintptr_t)kv_tiles | (uintptr_t)q |
       (uintptr_t)k) % 16)
    return fail(RL_ERR_ALIGN, "C, wq, wk, the tiles and q / k must be 16-byte aligned");
  if ((uintptr_t)v % 16) return fail(RL_ERR_ALIGN, "v must be 16-byte aligned");
  if (((uintptr_t)cos | (uintptr_t)sin) % 8) return fail(RL_ERR_ALIGN, "cos / sin must be 8-byte aligned");
  if ((s = check_device())) return s;
  QkvArgs a;
  a.C = C; a.ldc = ldc; a.M = M; a.hq = hq; a.hkv = hkv;
  a.cos = cos; a.sin = sin; a.wq = wq; a.wk = wk;
  a.q_tiles = q_tiles; a.kv_tiles = kv_tiles; a.q = q; a.k = k; a.v = v;
  const dim3 grid((unsigned)(M / kTileTokens * (hq + 2 * hkv)));
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const bool tiles = q_tiles || kv_tiles, native = q || k || v;
  if (tiles && native)
    hipLaunchKernelGGL((qkv_post_kernel<true, true>), grid, dim3(kQkvThreads), 0, st, a);
  else if (tiles)
    hipLaunchKernelGGL((qkv_post_kernel<true, false>), grid, dim3(kQkvThreads), 0, st, a);
  else
    hipLaunchKernelGGL((qkv_post_kernel<false, true>), grid, dim3(kQkvThreads), 0, st, a);
  return launch_status("rl_qkv_post");
}

extern "C" int rl_qkv_post(const uint16_t* C, int64_t ldc, int64_t M, int32_t heads, const uint16_t* cos,
                           const uint16_t* sin, const uint16_t* wq, const uint16_t* wk, uint8_t* q_tiles,
                           uint8_t* kv_tiles, uint16_t* q, uint16_t* k, uint16_t* v, void* stream) {
  return rl_qkv_post_gqa(C, ldc, M, heads, heads, cos, sin, wq, wk, q_tiles, kv_tiles, q, k, v, stream);
}

extern "C" int rl_attn_tiles(const uint8_t* q_tiles, int32_t hq, int64_t q_all, int64_t q_first, int64_t q_count,
                             int64_t nq, uint16_t* q, const uint8_t* kv0, int64_t all0, int64_t first0, int64_t count0,
                             const uint8_t* kv1, int64_t all1, int64_t first1, int64_t count1, int32_t hkv, uint16_t* k,
                             uint16_t* vt, void* stream) {
  using namespace rl;
  if (hq < 1 || hq > 1024 || hkv < 1 || hkv > 1024) return fail(RL_ERR_SHAPE, "heads %d / %d: need 1..1024", hq, hkv);
  constexpr int64_t kMax = 1 << 18;  // tiles per head: 2^24 tokens
  if (nq < 64 || nq % 64 || nq > 64 * kMax) return fail(RL_ERR_SHAPE, "nq %lld: need a multiple of 64", (long long)nq);
  if (q_first < 0 || q_count < 1 || q_count > nq / 64 || q_all > kMax || q_first > q_all - q_count)
    return fail(RL_ERR_SHAPE, "Q tiles %lld + %lld of %lld", (long long)q_first, (long long)q_count, (long long)q_all);
  if (first0 < 0 || count0 < 1 || all0 > kMax || first0 > all0 - count0)
    return fail(RL_ERR_SHAPE, "KV tiles %lld + %lld of %lld", (long long)first0, (long long)count0, (long long)all0);
  if (count1 && (first1 < 0 || count1 < 1 || all1 > kMax || first1 > all1 - count1))
    return fail(RL_ERR_SHAPE, "second KV tiles %lld + %lld of %lld", (long long)first1, (long long)count1,
                (long long)all1);
  if (count0 + count1 > kMax) return fail(RL_ERR_SHAPE, "%lld KV tiles", (long long)(count0 + count1));
  const int64_t nwg = hq * (nq / 64) + 2 * (int64_t)hkv * (count0 + count1);
  if (nwg > ((int64_t)1 << 31) - 1) return fail(RL_ERR_SHAPE, "more than 2^31 tiles");
  if (!q_tiles || !q || !kv0 || !k || !vt || (count1 && !kv1)) return fail(RL_ERR_NULL, "a buffer is NULL");
  if (((uintptr_t)q_tiles | (uintptr_t)kv0 | (uintptr_t)kv1) % 4 || ((uintptr_t)q | (uintptr_t)k | (uintptr_t)vt) % 16)
    return fail(RL_ERR_ALIGN, "tiles must be 4-byte, q / k / vt 16-byte aligned");
  int s;
  if ((s = check_device())) return s;
  TilesArgs a;
  a.q_tiles = q_tiles; a.hq = hq; a.q_all = (int32_t)q_all; a.q_t0 = (int32_t)q_first; a.q_n = (int32_t)q_count;
  a.q_out = (int32_t)(nq / 64); a.q = q;
  a.kv[0] = kv0; a.kv_all[0] = (int32_t)all0; a.kv_t0[0] = (int32_t)first0; a.kv_n[0] = (int32_t)count0;
  a.kv[1] = kv1; a.kv_all[1] = (int32_t)all1; a.kv_t0[1] = (int32_t)first1; a.kv_n[1] = (int32_t)count1;
  a.hkv = hkv; a.k = k; a.vt = vt;
  hipLaunchKernelGGL(attn_tiles_kernel, dim3((unsigned)nwg), dim3(kQkvThreads), 0, static_cast<hipStream_t>(stream), a);
  return launch_status("rl_attn_tiles");
}

extern "C" int rl_qkv_post_stream(const void* C, int32_t c_packed, int64_t M, int32_t hq, int32_t hkv,
                                  const uint16_t* tabs, uint8_t* q_tiles, uint8_t* kv_tiles, void* stream) {
  using namespace rl;
  const int64_t n = 128 * ((int64_t)hq + 2 * (int64_t)hkv);
  int s = rl_validate_qkv_post_gqa(n, M, hq, hkv);
  if (s) return s;
  if (M % 512 || n % 1024)
    return fail(RL_ERR_SHAPE, "M %lld, %lld columns: the C-stream order needs M %% 512 == 0 and columns %% 1024 == 0",
                (long long)M, (long long)n);
  if (!C || !tabs || !q_tiles || !kv_tiles) return fail(RL_ERR_NULL, "C, tabs or an output is NULL");
  if (((uintptr_t)C | (uintptr_t)tabs | (uintptr_t)q_tiles | (uintptr_t)kv_tiles) % 16)
    return fail(RL_ERR_ALIGN, "C, tabs and the tiles must be 16-byte aligned");
  if ((s = check_device())) return s;
  QkvStreamArgs a;
  a.C = C; a.n_cols = (int32_t)n; a.hq = hq; a.hkv = hkv; a.M = M; a.tabs = tabs; a.q_tiles = q_tiles;
  a.kv_tiles = kv_tiles;
  const dim3 grid((unsigned)(M / kTileTokens * (hq + 2 * hkv)));
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (c_packed)
    hipLaunchKernelGGL(qkv_stream_kernel<true>, grid, dim3(kQkvThreads), 0, st, a);
  else
    hipLaunchKernelGGL(qkv_stream_kernel<false>, grid, dim3(kQkvThreads), 0, st, a);
  return launch_status("rl_qkv_post_stream");
}
