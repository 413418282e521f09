// Gate logits of token batches (gfx950): logits[T, E] = x[T, H] wg[E, H]^T with the summation order of k_gate_logits
// (64 partial sums, partial l over k = 512 c + 8 l + i with c, then i ascending; then the xor butterfly 32, 16 .. 1), so
// that routing does not depend on the batch size a token arrives in.
//
// The order leaves the matrix cores usable: a product of depth one (v_mfma_f32_16x16x1_4b_f32: four independent
// 16 x 16 outer products, added to their accumulators) is one fp32 fma per element, and products of two bf16 values are
// exact, so the four blocks carry four partial sums l of 16 gate rows x 16 tokens, one chain step per instruction.
// They do twice the fma's per cycle of the vector unit (without packed fp32), and each operand is unpacked from bf16 once
// per 16 products.  A workgroup of 8 waves takes a tile of 16 tokens x 16 rows; wave w holds the partial sums
// l = 4 w .. 4 w + 3 and l + 32 (its lanes read 64 contiguous bytes of a row).  Step 32 of the butterfly is one add per
// register; the rest is the same binary tree for every element, over the 32 sums that meet in LDS.
//
// What bounds it: one trip to memory and the chain behind it (64 products per wave at 2048 columns), then the matrix cores'
// fp32 rate (3.4 us for 2048 tokens x 64 rows x 2048 columns, which take 12.6; with 8 row-adjacent partial sums per wave, whole
// 128-byte lines, no faster).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "moe_common.h"
#include "moe_kernels.h"
#include "moe_device.h"

typedef float f32x16_t __attribute__((ext_vector_type(16)));

#define GT_TILE 16
// One (token, gate row) pair by one wave: the sum of gate_row_sum (D < 4: rows of at most D chunks)
template <int D>
static __device__ __forceinline__ float gt_row(const uint16_t *xr, const uint16_t *wr, const int H, const int lane) {
  if constexpr (D == 4) return gate_row_sum(xr, wr, H, lane);
  float v = gate_row_partial<D>(xr, wr, H, lane);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = v + __shfl_xor(v, m, 64);
  return v;
}

// D: chunks of 512 columns on their way (rows of at most 512 and 1024 columns need no more than 1 and 2; with the registers
// that saves, 4 and 3 workgroups share a compute unit instead of 2, which cover each other's trip to memory and reduction:
// 4096 tokens x 64 rows x 512 columns 11.4 -> 8.1 us, x 1024 columns 15.3 -> 13.4).
// n_full: row tiles.  Rows behind the last of them (one or two: a shared expert's gate row behind 64 experts) go to one more
// workgroup per token tile, a wave per (token, row), instead of a tile of which one row is used (4096 x 65 x 2048 27.4 -> 24.1
// us, 1024 x 65 x 3584 16.1 -> 12.1, 4096 x 17 x 2048 12.3 -> 9.5).
template <int D>
__global__ __launch_bounds__(512, D == 1 ? 8 : (D == 2 ? 6 : 4)) void k_gate_tiles(const uint16_t *__restrict__ x, const uint16_t *__restrict__ wg,
                                                       const float *__restrict__ bias, const int n_bias,
                                                       float *__restrict__ logits, const int T, const int H, const int E,
                                                       const int ldl, const int n_full) {
  __shared__ __align__(16) float red[32][GT_TILE][GT_TILE];  // [partial sum][token][gate row]
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n = lane & 15, b = lane >> 4;
  const int t0 = blockIdx.x * GT_TILE, e0 = blockIdx.y * GT_TILE;
  if ((int)blockIdx.y >= n_full) {
    for (int q = w; q < GT_TILE * (E - e0); q += 8) {
      const int tt = t0 + q % GT_TILE, ee = e0 + q / GT_TILE;
      if (tt >= T) continue;
      const float v = gt_row<D>(x + (size_t)tt * H, wg + (size_t)ee * H, H, lane);
      if (lane == 0) logits[(size_t)tt * ldl + ee] = ee < n_bias ? v + bias[ee] : v;
    }
    return;
  }
  const int t = min(t0 + n, T - 1), e = min(e0 + n, E - 1);  // past the end: the last one again, not stored
  const int k0 = 8 * (4 * w + b);                            // the lane's columns: 512 c + 256 h + k0 .. + 7
  constexpr int OUT = 0x7fffff00;                            // length of the resources; a load from there on reads zeros
  const rsrc_t rx = make_rsrc(x + (size_t)t0 * H, OUT), rw = make_rsrc(wg + (size_t)e0 * H, OUT);
  const int xo = ((t - t0) * H + k0) * 2, wo = ((e - e0) * H + k0) * 2;
  uint4 xv[D][2], wv[D][2];
  auto load = [&](const int d, const int c) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = 512 * c + 256 * h;
      const bool in = k + k0 < H;                            // (H % 8 == 0; outside: 0 * 0 leaves a sum as it is)
      xv[d][h] = bload16(rx, in ? xo + 2 * k : OUT, 0);
      wv[d][h] = bload16(rw, in ? wo + 2 * k : OUT, 0);
    }
  };
  f32x16_t acc[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[h][i] = 0.f;
  const int nc = (H + 511) >> 9;
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  for (int c0 = 0; c0 < nc; c0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (c0 + d < nc) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const u32 xd = i < 4 ? (i < 2 ? xv[d][h].x : xv[d][h].y) : (i < 6 ? xv[d][h].z : xv[d][h].w);
            const u32 wd = i < 4 ? (i < 2 ? wv[d][h].x : wv[d][h].y) : (i < 6 ? wv[d][h].z : wv[d][h].w);
            acc[h] = __builtin_amdgcn_mfma_f32_16x16x1f32(i & 1 ? bf16hi(wd) : bf16lo(wd), i & 1 ? bf16hi(xd) : bf16lo(xd),
                                                          acc[h], 0, 0, 0);
          }
        load(d, c0 + d + D);
      }
    }
  }
  // element 4 blk + i of a lane: partial sum 4 w + blk, gate row 4 b + i, token n
#pragma unroll
  for (int blk = 0; blk < 4; ++blk) {
    float4 s;
    s.x = acc[0][4 * blk] + acc[1][4 * blk]; s.y = acc[0][4 * blk + 1] + acc[1][4 * blk + 1];
    s.z = acc[0][4 * blk + 2] + acc[1][4 * blk + 2]; s.w = acc[0][4 * blk + 3] + acc[1][4 * blk + 3];
    *(float4 *)&red[4 * w + blk][n][4 * b] = s;
  }
  __syncthreads();
  if (tid < GT_TILE * GT_TILE) {
    const float *p = &red[0][0][0] + tid;
    float v[16];
#pragma unroll
    for (int l = 0; l < 16; ++l) v[l] = p[256 * l] + p[256 * (l + 16)];
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1)
#pragma unroll
      for (int l = 0; l < m; ++l) v[l] = v[l] + v[l + m];
    const int tt = t0 + (tid >> 4), ee = e0 + (tid & 15);
    if (tt < T && ee < E) logits[(size_t)tt * ldl + ee] = ee < n_bias ? v[0] + bias[ee] : v[0];
  }
}

// From this many logits on.  A wave per logit (k_gate_logits) takes 2.3 us and 0.27 ns per logit of 2048 columns (0.16 ns at
// 512), the tiles one trip to memory and the chain of H products, 7.8 us at 2048 columns, 3.9 at 512, up to 512 of them on
// the chip.  us, wave per logit / tiles: 2048 columns, 12800 logits 5.9 / 7.7, 19200 logits 7.6 / 7.8, 32768 logits 11.1 / 7.8;
// 512 columns, 12800 logits 4.4 / 3.9, 18000 logits 5.4 / 4.0.
// The kernel for more than 128 tokens before this one (gate rows in LDS, two tokens per wave) was as fast where its workgroups
// filled the chip exactly (512 tokens x 64 rows x 2048 columns 6.3 / 7.8 us, 2048 x 8 x 2048 6.4 / 6.9) and slower elsewhere:
// 400 x 64 x 2048 9.1 / 7.7, 1024 x 65 x 2048 11.3 / 8.7, 4096 x 65 x 2048 28.7 / 24.1, 4096 x 65 x 512 11.2 / 8.9, 512 x 65 x 3584
// 13.3 / 10.5, 4096 x 8 x 4096 14.7 / 11.2.
bool moe_gate_tiles_take(int T, int H, int E) { return (long long)T * E >= (H <= 1024 ? 13000 : 20000); }

int moe_gate_tiles(const void *x, const void *wg, const float *bias, int n_bias, float *logits, int T, int H, int E, int ldl,
                   hipStream_t s) {
  moe_ktimer_begin(MOE_K_GATE, s);
  // token tiles fastest: the row tiles of one token tile mostly meet on one XCD and share its activations
  const int rest = E % GT_TILE, n_full = rest <= 2 && E >= GT_TILE ? E / GT_TILE : (E + GT_TILE - 1) / GT_TILE;
  const dim3 grid((T + GT_TILE - 1) / GT_TILE, n_full + (n_full * GT_TILE < E ? 1 : 0));
#define GT_LAUNCH(D_) hipLaunchKernelGGL(k_gate_tiles<D_>, grid, dim3(512), 0, s, (const uint16_t *)x, (const uint16_t *)wg, bias, \
                                         bias ? n_bias : 0, logits, T, H, E, ldl, n_full)
  if (H <= 512) GT_LAUNCH(1);
  else if (H <= 1024) GT_LAUNCH(2);
  else GT_LAUNCH(4);
#undef GT_LAUNCH
  moe_ktimer_end(MOE_K_GATE, s);
  return moe_check_launch("k_gate_tiles");
}
