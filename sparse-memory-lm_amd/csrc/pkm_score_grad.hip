// Gradient of the sub-key scores with respect to the keys in training (the einsum's in smlm/pkm.py:117-123):
//   dkeys[h, p, k, :] = sum_n g_p[n, h, k] q[n, h, p half + :]
// g_p (N, H, NK) and q (N, H, 2 half) bf16 as the forward has them, fp32 sums, each output written by one wavefront (the
// same bits on every call).
//
// Bound by the token walk: a contraction over N with few outputs (4 heads, 2 x 1,024 keys of 256: 256 tiles of 64 x 128),
// 17 GFLOP for 4,096 tokens.  The library's two batched products took 58 us there, and 25 more for copies of the query's
// halves and the cast of a bf16 result; this kernel takes 40.
// One workgroup per (head, half, 64 keys, 128 columns) walks the tokens 64 at a time.  Both operands have the contraction
// as their slow dimension, so both come through the transposing LDS reads (ds_read_b64_tr_b16: lane r gets four
// tokens of column r; the token order within a 32-token step is the same for both operands, which is all that the sum
// needs).  Four LDS buffers, three tiles on the way: with one workgroup per CU the walk waits for memory otherwise.
// blockIdx % (2 H) is the (head, half): with 4 heads each XCD's L2 holds one query slice.
#include "pkm_common.h"

namespace smlm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kKgThreads = 512, kKgKeys = 64, kKgCols = 128, kKgTokens = 64, kKgBufs = 4;
constexpr int kKgTileG = kKgTokens * kKgKeys, kKgTile = kKgTileG + kKgTokens * kKgCols;  // elements of a buffer
constexpr int kKgLds = kKgBufs * kKgTile * 2;                                            // 96 KB

// Fragments of four 16-column groups of the query tile (256-byte rows) and two of the gradient tile (128-byte rows) over 32
// tokens: two reads each, 16 tokens apart (the same swizzle).  One asm block with its wait: for the builtin the compiler
// waits until no load into LDS is on its way, the younger tiles' among them.
__device__ __forceinline__ void read_frags(const uint32_t *qa, const uint32_t *ga, uint2 (*x)[2]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %12\n\t"
      "ds_read_b64_tr_b16 %1, %12 offset:4096\n\t"
      "ds_read_b64_tr_b16 %2, %13\n\t"
      "ds_read_b64_tr_b16 %3, %13 offset:4096\n\t"
      "ds_read_b64_tr_b16 %4, %14\n\t"
      "ds_read_b64_tr_b16 %5, %14 offset:4096\n\t"
      "ds_read_b64_tr_b16 %6, %15\n\t"
      "ds_read_b64_tr_b16 %7, %15 offset:4096\n\t"
      "ds_read_b64_tr_b16 %8, %16\n\t"
      "ds_read_b64_tr_b16 %9, %16 offset:2048\n\t"
      "ds_read_b64_tr_b16 %10, %17\n\t"
      "ds_read_b64_tr_b16 %11, %17 offset:2048\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[2][0]), "=&v"(x[2][1]), "=&v"(x[3][0]),
        "=&v"(x[3][1]), "=&v"(x[4][0]), "=&v"(x[4][1]), "=&v"(x[5][0]), "=&v"(x[5][1])
      : "v"(qa[0]), "v"(qa[1]), "v"(qa[2]), "v"(qa[3]), "v"(ga[0]), "v"(ga[1])
      : "memory");
}

// Byte offset within a tile of CPR swizzled 16-byte chunks a row that lane (r, g) reads a 16-column group from.
template <int CPR>
__device__ __forceinline__ uint32_t frag_at(int token0, int col, int r, int g) {
  const int row = token0 + 4 * g + r / 4, c = col + 4 * (r % 4);
  return row * CPR * 16 + (((c / 8) ^ (row % 8)) * 16) + (c % 8) * 2;
}

template <bool OUT_F32>
__global__ void __launch_bounds__(kKgThreads)
    score_keys_grad_kernel(const uint16_t *__restrict__ g1, const uint16_t *__restrict__ g2,
                           const uint16_t *__restrict__ q, int N, int H, int NK, int half, void *__restrict__ dk) {
  extern __shared__ __align__(16) uint16_t lds[];
  const int hp = blockIdx.x % (2 * H), h = hp / 2, p = hp % 2, tile = blockIdx.x / (2 * H);
  const int nd = (half + kKgCols - 1) / kKgCols, k0 = tile / nd * kKgKeys, d0 = tile % nd * kKgCols;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, r = lane & 15, g = lane >> 4;
  // the wavefront's 32 keys and 64 columns of the tile, and its 32 of each 64 tokens
  const int kw = (wave & 1) * 32, dw = (wave / 2 % 2) * 64, ks = wave / 4;
  const uint16_t *gp = p ? g2 : g1;
  floatx4 acc[4][2];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i / 2][i % 2] = floatx4{0.f, 0.f, 0.f, 0.f};

  if (gp) {  // workgroup-uniform; without a gradient the half's result is zero
    const int64_t gs = (int64_t)H * NK, qs = (int64_t)H * 2 * half;
    const int64_t go = (int64_t)h * NK + k0, qo = ((int64_t)h * 2 + p) * half + d0;
    // the records end with the tensors: rows from N on read as zeros, columns past a row's end as its neighbours',
    // which no output uses
    const __amdgpu_buffer_rsrc_t rg =
        __builtin_amdgcn_make_buffer_rsrc((void *)(gp + go), (short)0, (int)((N * gs - go) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rq =
        __builtin_amdgcn_make_buffer_rsrc((void *)(q + qo), (short)0, (int)((N * qs - qo) * 2), 0x00020000);
    auto load_tile = [&](int t) {  // 3 loads per thread, also past the end, so that the counts below hold
      uint16_t *buf = lds + (t % kKgBufs) * kKgTile;
      const int64_t row0 = (int64_t)t * kKgTokens;
      const int grow = tid / 8, gc = (tid % 8) ^ (grow % 8);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rg, (__attribute__((address_space(3))) void *)((char *)buf + wave * kWave * 16), 16,
          (int)(((row0 + grow) * gs + 8 * gc) * 2), 0, 0, 0);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int id = tid + kKgThreads * u, row = id / 16, c = (id % 16) ^ (row % 8);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rq,
            (__attribute__((address_space(3))) void *)((char *)(buf + kKgTileG) + (kKgThreads * u + wave * kWave) * 16),
            16, (int)(((row0 + row) * qs + 8 * c) * 2), 0, 0, 0);
      }
    };
    const int tiles = (N + kKgTokens - 1) / kKgTokens;
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)lds;
    uint32_t qa[4], ga[2];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) qa[mt] = base + kKgTileG * 2 + frag_at<16>(32 * ks, dw + 16 * mt, r, g);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) ga[nt] = base + frag_at<8>(32 * ks, kw + 16 * nt, r, g);
    for (int t = 0; t < kKgBufs - 1; ++t) load_tile(t);
    for (int t = 0; t < tiles; ++t) {
      // this wavefront's part of tile t is in LDS (6 younger loads may be on the way) and its reads of tile t - 1 are
      // done; after the barrier that holds for all of them, and tile t - 1's buffer takes tile t + 3
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0x0076);  // vmcnt(6) lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      load_tile(t + kKgBufs - 1);
      const uint32_t buf = (t % kKgBufs) * kKgTile * 2;
      const uint32_t qt[4] = {qa[0] + buf, qa[1] + buf, qa[2] + buf, qa[3] + buf}, gt[2] = {ga[0] + buf, ga[1] + buf};
      uint2 x[6][2];
      read_frags(qt, gt, x);
      auto frag = [&](int i) {
        return __builtin_bit_cast(bf16x8, uint4{x[i][0].x, x[i][0].y, x[i][1].x, x[i][1].y});
      };
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(mt), frag(4 + nt), acc[mt][nt], 0, 0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0);  // no load is on its way into LDS
  }

  // the two token halves' sums meet in LDS (32 KB of the buffers)
  __syncthreads();
  float4 *sums = (float4 *)lds + (wave % 4) * 8 * kWave + lane;
  if (ks == 1) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const floatx4 v = acc[i / 2][i % 2];
      sums[i * kWave] = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
  __syncthreads();
  if (ks == 1) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float4 v = sums[i * kWave];
    acc[i / 2][i % 2] += floatx4{v.x, v.y, v.z, v.w};
  }

  // lane (r, g) holds columns 4 g .. 4 g + 3 of key r of each 16 x 16 tile
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int key = k0 + kw + 16 * nt + r;
    if (key >= NK) continue;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int d = d0 + dw + 16 * mt + 4 * g;
      if (d >= half) continue;
      const int64_t o = ((int64_t)hp * NK + key) * half + d;
      const floatx4 v = acc[mt][nt];
      if constexpr (OUT_F32) *(float4 *)((float *)dk + o) = make_float4(v[0], v[1], v[2], v[3]);
      else *(uint2 *)((uint16_t *)dk + o) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
  }
}

}  // namespace
}  // namespace smlm

extern "C" int smlm_score_keys_grad(const void *g1, const void *g2, const void *q, int64_t N, int H, int NK, int half,
                                    void *dk, int dk_dtype, void *stream) {
  using namespace smlm;
  if (!q || !dk) return fail(SMLM_EINVAL, "smlm_score_keys_grad: null q or dk pointer");
  if (dk_dtype != SMLM_BF16 && dk_dtype != SMLM_F32)
    return fail(SMLM_EINVAL, "smlm_score_keys_grad: dk must be SMLM_BF16 or SMLM_F32, got %d", dk_dtype);
  if (N < 1 || H < 1 || H > 32768 || NK < 8 || NK % 8 || half < 8 || half % 8)
    return fail(SMLM_EUNSUPPORTED, "smlm_score_keys_grad: N=%lld H=%d NK=%d half=%d (NK and half multiples of 8)",
                (long long)N, H, NK, half);
  if (((uintptr_t)g1 | (uintptr_t)g2 | (uintptr_t)q | (uintptr_t)dk) % 16)
    return fail(SMLM_EINVAL, "smlm_score_keys_grad: g1, g2, q and dk must be 16-byte aligned");
  // byte offsets of 32 bits, up to four tiles past the last row
  const int64_t width = (int64_t)H * (NK > 2 * half ? NK : 2 * half);
  if (N > 0x7FFFFFFFLL || (N + (kKgBufs + 1) * kKgTokens) * width * 2 + 512 > 0x7FFFFFFFLL)
    return fail(SMLM_EUNSUPPORTED, "smlm_score_keys_grad: N=%lld rows of %lld exceed 2 GB", (long long)N,
                (long long)width);
  const int64_t blocks = 2LL * H * ((NK + kKgKeys - 1) / kKgKeys) * ((half + kKgCols - 1) / kKgCols);
  if (blocks > 0x7FFFFFFFLL) return fail(SMLM_EUNSUPPORTED, "smlm_score_keys_grad: too many workgroups");
  const bool f32 = dk_dtype == SMLM_F32;
  const void *kernel = f32 ? (const void *)score_keys_grad_kernel<true> : (const void *)score_keys_grad_kernel<false>;
  const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kKgLds);
  if (e != hipSuccess) return fail(SMLM_EHIP, "smlm_score_keys_grad: %s", hipGetErrorString(e));
  const dim3 grid((unsigned)blocks), block(kKgThreads);
  const uint16_t *a = (const uint16_t *)g1, *b = (const uint16_t *)g2, *x = (const uint16_t *)q;
  hipStream_t s = (hipStream_t)stream;
  if (f32) hipLaunchKernelGGL(score_keys_grad_kernel<true>, grid, block, kKgLds, s, a, b, x, (int)N, H, NK, half, dk);
  else hipLaunchKernelGGL(score_keys_grad_kernel<false>, grid, block, kKgLds, s, a, b, x, (int)N, H, NK, half, dk);
  return launch_status("smlm_score_keys_grad");
}
