// bf16 experts, decode batches of up to 64 tokens (gfx950): the grouped SwiGLU expert product as a weight stream.
//
// What bounds it: with a few rows per expert every weight is read once and used for at most 64 tokens, so the launch
// is as long as its bytes take (about 6 TB/s for plain reads on this chip) plus the chain kernel start -> unit ->
// slot address -> first weights.  The tile kernels of moe_prefill.hip, which took these batches before, stage
// activations through LDS with a barrier per slab for up to 256 rows, hold one workgroup per compute unit, and their
// w2 pass has H / 256 workgroups per expert (40 in all for one token of the Qwen1.5 shape).
//
// Work split: a workgroup of four waves owns two row sets of one unit (w13: the same 16 HV rows of gate and up; w2:
// two adjacent sets), its waves take every fourth 64-wide slab of the reduction and their sums meet in LDS once, at
// the end.  Weights (16 HV rows x 64 k) and activation rows go global -> registers in the operand order of
// v_mfma_f32_16x16x32_bf16, DEPTH slabs ahead; there is no barrier and no LDS in the loop.  The activation rows come
// out of the caches (T rows, read by every workgroup of a unit): HV = 2 reads them half as often as HV = 1 and is
// taken where its workgroups still fill the chip.
//
// Measured (us, both launches, tile kernels / these): Qwen1.5 shape 1 token 73.2 / 31.5, 4 tokens 82.9 / 62.5, 16 tokens
// 155 / 131, 64 tokens 199 / 181; Mixtral shape 1 token 231 / 119, 8 tokens 420 / 355, 64 tokens 480 / 443 (up to 6.4 TB/s);
// 8 experts of 2048 x 4096 that all see every token: 16 tokens 103 / 79, 48 tokens 109 / 99, 64 tokens 111 / 111: there the line.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include "moe_common.h"
#include "moe_kernels.h"
#include "moe_device.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

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
struct DbArgs {
  DbClass c[2];          // 0 = shared expert, 1 = routed experts
  const moe_unit *units;
  const unsigned long long *expert_ptr;
  const unsigned char *shared_base;
  int n_sh_blocks, T;
  int pass_rows;         // most rows of one pass: what the launch has LDS for (16, 32 or 64)
  int *err;
  moe_publish pub;       // w13 pass: the first workgroup takes the unit list to the host (units_host NULL: none does)
};

#define DB_NO_ROW 0x7fffff00u  // length of the buffer resources and the offset that reads zeros without a memory request

// One pass over up to 16 NT token rows.  rwA / rwB: the two row sets' rows of slabs, rotA / rotB: the position of slab 0
// in them (rotation), slabs kt0 .. kt0 + nk - 1 of a row of Kn slabs.
template <bool SWIGLU, int HV, int NT, int DEPTH>
static __device__ __forceinline__ void db_pass(const DbClass &c, float *red, const rsrc_t rwA, const rsrc_t rwB, const rsrc_t rx,
                                               const int rotA, const int rotB, const int half, const int kt0,
                                               const int nk, const int Kn, const int row_first, const int mc,
                                               const size_t out_row0, const int out_col, const int tid) {
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, cq = lane >> 4;
  // weights: load (h, m) of a slab = rows 16 h + r, chunk of 8 k number (j, q) = (2 m + cq / 2, cq % 2) of the block
  const int wv = cq * 512 + half * 256 + r * 16;
  int xv[NT];   // activations: the same chunk of token row 16 t + r
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int row = 16 * t + r;
    const int gr = row_first + (row < mc ? row : mc - 1);
    const int arow = c.gather ? c.gather[gr] : gr;
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
  f32x4_t acc[2][HV][NT];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int h = 0; h < HV; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[s][h][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
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
              acc[s][h][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wt[d][s][h][m]),
                                                                     __builtin_bit_cast(bf16x8_t, xb[d][t][m]), acc[s][h][t], 0, 0, 0);
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
        *(f32x4_t *)(red + ((((w * 2 + s) * HV + h) * NT + t) * 64 + lane) * 4) = acc[s][h][t];
  __syncthreads();
  for (int q = w; q < HV * NT; q += 4) {
    const int h = q / NT, t = q - h * NT;
    f32x4_t v[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      v[s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) v[s] += *(const f32x4_t *)(red + ((((ww * 2 + s) * HV + h) * NT + t) * 64 + lane) * 4);
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
        *(f32x4_t *)((float *)c.out + orow + out_col + 16 * h + 4 * cq) = v[0];
        *(f32x4_t *)((float *)c.out + orow + out_col + 16 * HV + 16 * h + 4 * cq) = v[1];
      }
    }
  }
}

template <bool SWIGLU, int HV>
__global__ __launch_bounds__(256, 2) void k_decode_bf16(const DbArgs a) {
  extern __shared__ __align__(16) float red_db[];
  const int tid = threadIdx.x;
  const bool pub = SWIGLU && a.pub.units_host != nullptr;
  if (pub && blockIdx.x == 0) { publish_units(a.pub, a.units, tid, 256); return; }
  const int bx = (int)blockIdx.x - (pub ? 1 : 0);
  const bool sh = bx < a.n_sh_blocks;
  const DbClass &c = a.c[sh ? 0 : 1];
  int rr = sh ? bx : bx - a.n_sh_blocks;
  int m, row0, win = 0;
  const unsigned char *base;
  if (sh) {
    m = a.T; row0 = 0; base = a.shared_base;
    win = rr / c.nblk; rr -= win * c.nblk;
  } else {
    const int u = rr / c.nblk;
    rr -= u * c.nblk;
    const moe_unit un = a.units[u];
    if (un.m <= 0 || un.expert < 0) return;
    m = un.m; row0 = un.row0;
    base = (const unsigned char *)a.expert_ptr[un.expert];
    if (!base) {
      if (tid == 0) moe_raise_err(a.err);
      return;
    }
  }
  const int Kn = c.K >> 6, nk = Kn / c.ksplit, kt0 = win * nk;
  // the two row sets: 32-row blocks (HV = 2) or halves of one (HV = 1)
  int nbA, nbB, half = 0, out_col;
  if (SWIGLU) {
    nbA = HV == 2 ? rr : rr >> 1;
    nbB = nbA + c.set_delta;
    if (HV == 1) half = rr & 1;
    out_col = 32 * nbA + 16 * half;
  } else {
    nbA = HV == 2 ? 2 * rr : rr;
    nbB = HV == 2 ? nbA + 1 : nbA;
    out_col = 32 * nbA;
  }
  const int gA = nbA >> 2, gB = nbB >> 2;
  const int rotA = (int)((unsigned)(gA * c.slab_step) % (unsigned)Kn), rotB = (int)((unsigned)(gB * c.slab_step) % (unsigned)Kn);
  // (64-bit bases: an expert image may have 2 GiB and more, a set's row of slabs has 256 bytes per column)
  auto set_rsrc = [&](const int g, const int nb, const int off) {
    const unsigned long long p = (unsigned long long)(base + c.w_off) + (unsigned long long)g * (unsigned)Kn * 16384u +
                                 (unsigned)((nb & 3) * 4096 + off);
    return make_rsrc((const void *)(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(p >> 32)) << 32) |
                                    (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)p)), DB_NO_ROW);
  };
  const rsrc_t rwA = set_rsrc(gA, nbA, 0), rwB = set_rsrc(gB, nbB, !SWIGLU && HV == 1 ? 256 : 0);
  const rsrc_t rx = make_rsrc(c.act, DB_NO_ROW);
  const size_t orow0 = (size_t)win * a.T;
  // A unit has more rows than there are tokens where a token holds its expert more than once (a choice among fewer than
  // k finite logits repeats one): then in further passes, each of no more rows than the LDS takes.
  const int mm = __builtin_amdgcn_readfirstlane(m), r_0 = __builtin_amdgcn_readfirstlane(row0);
  for (int p0 = 0; p0 < mm; p0 += a.pass_rows) {
    const int mc = mm - p0 < a.pass_rows ? mm - p0 : a.pass_rows, r0 = r_0 + p0;
    if (p0) __syncthreads();   // the sums of the pass before have been read
#define DB_PASS(NT_, D_) db_pass<SWIGLU, HV, NT_, D_>(c, red_db, rwA, rwB, rx, rotA, rotB, half, kt0, nk, Kn, r0, mc, orow0, out_col, tid)
    if (mc <= 16) DB_PASS(1, HV == 2 ? 4 : 6);
    else if (mc <= 32) DB_PASS(2, 3);
    else DB_PASS(4, 2);
#undef DB_PASS
  }
}

template <int HV>
static int db_launch(bool w13, const DbArgs &a, int grid, hipStream_t s) {
  const size_t lds = (size_t)4 * 2 * HV * (a.pass_rows / 16) * 64 * 16;
  moe_ktimer_begin(w13 ? MOE_K_PREFILL_W13 : MOE_K_PREFILL_W2, s);
  if (w13) hipLaunchKernelGGL((k_decode_bf16<true, HV>), dim3(grid), dim3(256), lds, s, a);
  else hipLaunchKernelGGL((k_decode_bf16<false, HV>), dim3(grid), dim3(256), lds, s, a);
  moe_ktimer_end(w13 ? MOE_K_PREFILL_W13 : MOE_K_PREFILL_W2, s);
  return moe_check_launch("k_decode_bf16");
}

// Whether a batch of T tokens goes to these kernels (a unit of up to 64 rows is one pass).
bool moe_decode_bf16_takes(int T) { return T <= 64; }

// Windows of the shared expert's w2 reduction: few row sets (H / 64) over a long reduction (Qwen1.5 shape: 32 over 88
// slabs) would outlast the routed experts' workgroups, so it is cut until there are 256 workgroups, in windows of at
// least 16 slabs.
int moe_decode_bf16_splits(int H, int I_sh) {
  const int nk = I_sh / 64;
  int s = 1;
  while (s < 8 && (H / 64) * s < 256 && nk % (2 * s) == 0 && nk / (2 * s) >= 16) s *= 2;
  return s;
}

int moe_decode_bf16(const void *x, int T, int H, int I, int I_sh, const moe_unit *units, int max_units, const int *sorted_tok,
                    const uint64_t *expert_ptr, const void *shared_ptr, void *h_r, void *h_s, float *part_r, float *part_s,
                    int pieces, int *err, int phases, const moe_publish *pub, hipStream_t s) {
  DbArgs a;
  memset(&a, 0, sizeof a);
  a.units = units; a.expert_ptr = (const unsigned long long *)expert_ptr; a.shared_base = (const unsigned char *)shared_ptr;
  a.T = T; a.err = err;
  a.pass_rows = T <= 16 ? 16 : (T <= 32 ? 32 : 64);
  if (pub) a.pub = *pub;
  for (int w2 = 0; w2 < 2; ++w2) {
    if (!(phases & (w2 ? 2 : 1))) continue;
    for (int i = 0; i < 2; ++i) {
      DbClass &c = a.c[i];
      const int Ii = i == 0 ? I_sh : I;
      if (!w2) {
        c.act = (const uint16_t *)x; c.gather = i == 0 ? nullptr : sorted_tok; c.act_stride = H; c.out = i == 0 ? h_s : h_r;
        c.out_stride = Ii; c.K = H; c.w_off = 0; c.set_delta = Ii / 32; c.ksplit = 1;
      } else {
        c.act = (const uint16_t *)(i == 0 ? h_s : h_r); c.gather = nullptr; c.act_stride = Ii;
        c.out = i == 0 ? (void *)part_s : (void *)part_r; c.out_stride = H; c.K = Ii;
        c.w_off = (long long)2 * Ii * H * 2; c.set_delta = 0; c.ksplit = i == 0 ? pieces : 1;
      }
      c.slab_step = c.K ? moe_bf16_slab_step(c.K / 64) : 1;
    }
    const int sh_blk = shared_ptr ? (w2 ? H / 64 * pieces : I_sh / 32) : 0, r_blk = w2 ? H / 64 : I / 32;
    // 16-row sets where 32-row sets would leave the chip with under four workgroups per compute unit
    const int hv = sh_blk + max_units * r_blk < 1024 ? 1 : 2;
    const int f = hv == 1 ? 2 : 1;
    a.c[0].nblk = f * (shared_ptr ? sh_blk / (w2 ? pieces : 1) : 0);
    a.c[1].nblk = f * r_blk;
    a.n_sh_blocks = f * sh_blk;
    const int grid = a.n_sh_blocks + max_units * a.c[1].nblk + (!w2 && pub ? 1 : 0);
    if (grid <= 0) continue;
    if (int rc = hv == 1 ? db_launch<1>(!w2, a, grid, s) : db_launch<2>(!w2, a, grid, s)) return rc;
  }
  return MOE_OK;
}
