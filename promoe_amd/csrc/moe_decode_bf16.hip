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
#include "moe_decode_bf16.h"

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
  const DbSets ws = db_sets<SWIGLU, HV>(c, base, rr);
  const rsrc_t rx = make_rsrc(c.act, DB_NO_ROW);
  const size_t orow0 = (size_t)win * a.T;
  // A unit has more rows than there are tokens where a caller's own choices list its expert more than once for a token (the
  // top-k never does): then in further passes, each of no more rows than the LDS takes.
  const int mm = __builtin_amdgcn_readfirstlane(m), r_0 = __builtin_amdgcn_readfirstlane(row0);
  for (int p0 = 0; p0 < mm; p0 += a.pass_rows) {
    const int mc = mm - p0 < a.pass_rows ? mm - p0 : a.pass_rows, r0 = r_0 + p0;
    if (p0) __syncthreads();   // the sums of the pass before have been read
    auto row_of = [&](const int row) { return c.gather ? c.gather[r0 + row] : r0 + row; };
#define DB_PASS(NT_, D_) db_pass<SWIGLU, HV, NT_, D_>(c, red_db, ws.rwA, ws.rwB, rx, ws.rotA, ws.rotB, ws.half, kt0, nk, Kn, r0, mc, \
                                                      orow0, ws.out_col, tid, row_of)
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
