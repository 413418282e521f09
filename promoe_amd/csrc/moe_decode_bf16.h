// Work split and pass of the bf16 decode kernels (moe_decode_bf16.hip; the launch that routes by itself is in
// moe_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "moe_device.h"

typedef __bf16 db_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float db_f32x4_t __attribute__((ext_vector_type(4)));

struct DbClass {
  const uint16_t *act;   // activation rows
  const int *gather;     // row -> activation row, or NULL
  void *out;             // bf16 h rows (w13) or fp32 partial rows (w2)
  long long w_off;       // byte offset of the matrix in the expert image
  int K, act_stride, out_stride;
  int nblk;              // workgroups per unit and window of the reduction
  int set_delta;         // w13: 32-row blocks from gate to up (I / 32)
  int slab_step;         // storage rotation per 128-row group (see the bf16 slot layout)
  int ksplit;            // shared expert's w2 pass: windows of the reduction, partial rows to out + window * T * out_stride
};
#define DB_NO_ROW 0x7fffff00u  // length of the buffer resources and the offset that reads zeros without a memory request

// One pass over up to 16 NT token rows.  rwA / rwB: the two row sets' rows of slabs, rotA / rotB: the position of slab 0
// in them (rotation), slabs kt0 .. kt0 + nk - 1 of a row of Kn slabs.
// row_of(i): the activation row of the pass's row i < mc.
template <bool SWIGLU, int HV, int NT, int DEPTH, typename RowOf>
static __device__ __forceinline__ void db_pass(const DbClass &c, float *red, const rsrc_t rwA, const rsrc_t rwB, const rsrc_t rx,
                                               const int rotA, const int rotB, const int half, const int kt0,
                                               const int nk, const int Kn, const int row_first, const int mc,
                                               const size_t out_row0, const int out_col, const int tid, const RowOf &row_of) {
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, cq = lane >> 4;
  // weights: load (h, m) of a slab = rows 16 h + r, chunk of 8 k number (j, q) = (2 m + cq / 2, cq % 2) of the block
  const int wv = cq * 512 + half * 256 + r * 16;
  int xv[NT];   // activations: the same chunk of token row 16 t + r
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int row = 16 * t + r;
    const int arow = row_of(row < mc ? row : mc - 1);
    xv[t] = row < mc ? (int)((unsigned)arow * (unsigned)c.act_stride * 2u) + 64 * (cq & 1) + 16 * (cq >> 1) : (int)DB_NO_ROW;
  }
  u32x4_t wt[DEPTH][2][HV][2], xb[DEPTH][NT][2];
  auto load = [&](const int d, const int i) {   // this wave's i-th slab: slab 4 i + w of the window
    const int kt = 4 * i + w;
    const bool in = kt < nk;                    // (past the end: zeros, no memory request)
    const int kb = kt0 + (in ? kt : 0);
    const int a = kb + rotA, b = kb + rotB;
    const int sa = (a >= Kn ? a - Kn : a) * 16384, sb = (b >= Kn ? b - Kn : b) * 16384;
    const int v = in ? wv : (int)DB_NO_ROW;
#pragma unroll
    for (int h = 0; h < HV; ++h)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        wt[d][0][h][m] = __builtin_amdgcn_raw_buffer_load_b128(rwA, v + h * 256 + m * 2048, sa, 2);
        wt[d][1][h][m] = __builtin_amdgcn_raw_buffer_load_b128(rwB, v + h * 256 + m * 2048, sb, 2);
      }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < 2; ++m) xb[d][t][m] = __builtin_amdgcn_raw_buffer_load_b128(rx, xv[t] + 32 * m, kb * 128, 0);
  };
  db_f32x4_t acc[2][HV][NT];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int h = 0; h < HV; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[s][h][t] = db_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(d, d);
  const int ni = (nk - w + 3) >> 2;
  for (int i0 = 0; i0 < ni; i0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int h = 0; h < HV; ++h)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              acc[s][h][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(db_bf16x8_t, wt[d][s][h][m]),
                                                                     __builtin_bit_cast(db_bf16x8_t, xb[d][t][m]), acc[s][h][t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      load(d, i0 + d + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the waves' sums: red[wave][set][half][token block][element][lane]
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int h = 0; h < HV; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        *(db_f32x4_t *)(red + ((((w * 2 + s) * HV + h) * NT + t) * 64 + lane) * 4) = acc[s][h][t];
  __syncthreads();
  for (int q = w; q < HV * NT; q += 4) {
    const int h = q / NT, t = q - h * NT;
    db_f32x4_t v[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      v[s] = db_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) v[s] += *(const db_f32x4_t *)(red + ((((ww * 2 + s) * HV + h) * NT + t) * 64 + lane) * 4);
    }
    if (16 * t + r < mc) {
      const size_t orow = (out_row0 + (size_t)(row_first + 16 * t + r)) * c.out_stride;
      if (SWIGLU) {
        u32 o[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float g0 = v[0][2 * i], g1 = v[0][2 * i + 1];
          const float h0 = g0 / (1.f + expf(-g0)) * v[1][2 * i], h1 = g1 / (1.f + expf(-g1)) * v[1][2 * i + 1];
          o[i] = (u32)f32_to_bf16(h0) | ((u32)f32_to_bf16(h1) << 16);
        }
        *(uint2 *)((uint16_t *)c.out + orow + out_col + 16 * h + 4 * cq) = make_uint2(o[0], o[1]);
      } else {
        *(db_f32x4_t *)((float *)c.out + orow + out_col + 16 * h + 4 * cq) = v[0];
        *(db_f32x4_t *)((float *)c.out + orow + out_col + 16 * HV + 16 * h + 4 * cq) = v[1];
      }
    }
  }
}


// The two row sets of workgroup rr of a unit: 32-row blocks (HV = 2) or halves of one (HV = 1)
struct DbSets {
  rsrc_t rwA, rwB;
  int rotA, rotB, half, out_col;
};
template <bool SWIGLU, int HV>
static __device__ __forceinline__ DbSets db_sets(const DbClass &c, const unsigned char *base, const int rr) {
  DbSets t;
  const int Kn = c.K >> 6;
  int nbA, nbB;
  t.half = 0;
  if (SWIGLU) {
    nbA = HV == 2 ? rr : rr >> 1;
    nbB = nbA + c.set_delta;
    if (HV == 1) t.half = rr & 1;
    t.out_col = 32 * nbA + 16 * t.half;
  } else {
    nbA = HV == 2 ? 2 * rr : rr;
    nbB = HV == 2 ? nbA + 1 : nbA;
    t.out_col = 32 * nbA;
  }
  const int gA = nbA >> 2, gB = nbB >> 2;
  t.rotA = (int)((unsigned)(gA * c.slab_step) % (unsigned)Kn); t.rotB = (int)((unsigned)(gB * c.slab_step) % (unsigned)Kn);
  // (64-bit bases: an expert image may have 2 GiB and more, a set's row of slabs has 256 bytes per column)
  auto set_rsrc = [&](const int g, const int nb, const int off) {
    const unsigned long long p = (unsigned long long)(base + c.w_off) + (unsigned long long)g * (unsigned)Kn * 16384u +
                                 (unsigned)((nb & 3) * 4096 + off);
    return make_rsrc((const void *)(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(p >> 32)) << 32) |
                                    (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)p)), DB_NO_ROW);
  };
  t.rwA = set_rsrc(gA, nbA, 0); t.rwB = set_rsrc(gB, nbB, !SWIGLU && HV == 1 ? 256 : 0);
  return t;
}
