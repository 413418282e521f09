// Prefill-sized expert groups on the matrix cores (gfx950): grouped GEMM over the
// tokens dispatched to each expert, bf16 operands, fp32 accumulation.
//
//   w13 pass: h[rows, I]   = silu(A Wg^T) * (A Wu^T)     A = gathered activations
//   w2  pass: part[rows,H] = h W2^T
//
// bf16 experts: workgroup = 256 threads (4 waves, one per SIMD) -> a tile of up to 256 rows x (128+128)
// columns: for w13 the two column halves are the SAME columns of gate and up (SwiGLU fused in the epilogue),
// for w2 they are adjacent column blocks.  K advances 64 at a time; the activation slab goes global -> LDS
// directly (a ring of four slabs), the weight fragments go global -> registers in operand order and feed
// v_mfma_f32_32x32x16_bf16.  int4 / q4_K experts: four waves on a tile of up to 128 rows, two workgroups per compute unit,
// activations, nibbles and scales through one LDS ring, fragments dequantised in registers between the products (below).
// bf16 batches of up to 64 tokens go to moe_decode_bf16.hip.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>
#include <stdlib.h>
#include <type_traits>

#include "moe_common.h"
#include "moe_kernels.h"
#include "moe_device.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

#define PF_BM 256     // most rows of one tile (8 blocks of 32)
#define PF_BM_SHARED 256     // rows per tile of the dense shared expert in the w13 pass
#define PF_BM_SHARED_W2 128  // and in its w2 pass, which has few column tiles (H/256) and a long K
#define PF_BNH 128   // columns per half
#define PF_BK 64

struct PfTile {
  unsigned long long w_base;  // expert image base (device address)
  int row0;                   // first row (sorted pair order / token order for the shared expert)
  int rows_group;             // bits 0-15 valid rows (<= PF_BM), 16-23 tiles in its group, 24-31 its place in the group
};
static __device__ __forceinline__ int pf_rows(const PfTile &t) { return t.rows_group & 0xffff; }
// one GEMM problem class of a launch (routed experts / shared expert)
struct PfClass {
  const uint16_t *act;  // activations: bf16, or fp16 for the nibble formats (the copy of x, then the h rows)
  const int *gather;    // row -> activation row, or NULL
  void *out;            // h rows in the format of the activations (SWIGLU) or fp32 partial rows
  const PfTile *tiles;
  const int *n_tiles_real;  // device: tiles actually in use (<= n_mtiles, the launch's upper bound)
  long long w_off;      // byte offset of the matrix inside the expert image
  long long half_delta; // weight-row offset of the second column half relative to the first
  long long off_s, off_z; // int4: byte offsets of the scale / zero sections (w_off = the nibble section)
  int act_stride, out_stride, K, n_ntiles, n_mtiles, n_cols_per_tile;
  int shared;           // the shared expert's class
  int slab_step;        // storage rotation per 128-row group: smallest odd s >= 3 coprime with K/64
  int n_blocks;         // n_mtiles * n_ntiles * ksplit, padded (pf_padded)
  int ksplit;           // w2 pass (bf16: the shared expert's): workgroups per tile, each over 1/ksplit of the reduction, partial rows
                        // to out + split * split_stride (0 or 1: the whole reduction)
  long long split_stride;  // elements between the pieces of out
};
struct PfArgs {
  PfClass c[2];
  int n_blocks_total;  // blocks of c[0] come first
};

// silu(g) * u with the hardware's 2^x and reciprocal (1 ulp each; the result is rounded to bf16 by the caller,
// round to nearest even in hardware): a tile's epilogue computes 128 of these per lane
static __device__ __forceinline__ float pf_silu_mul(float g, float u) {
  return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(g * -1.44269504088896f)) * u;
}

// Which block of which class a physical workgroup takes; false: none.  The blocks of class 0 come first, each class
// padded (pf_padded).  Workgroup i runs on XCD i % 8; runs of PF_DEAL consecutive blocks are dealt to the XCDs in turn, so
// that the XCDs get the same number of blocks of every size whatever the row counts are: the list holds the large tiles
// first.  (One contiguous range of the list per XCD, the order before this one, left the XCDs with the popular experts'
// tiles busy alone: 1.4 of 2 waves per SIMD on average over the w13 launch of the DeepSeek shape at 2048 tokens, 1.0 at 379.)
// Inside the list: a group of up to PF_GROUP tiles of one expert goes through all its column tiles, tile fastest, so
// that a run shares either a column tile's weights (many tiles) or the activation rows (one tile) in its XCD's L2.
// EVEN (bf16 kernel: one workgroup per compute unit, so that a run too many is a quarter of a round of its XCD): the blocks
// of a class past its last whole round of 8 runs are spread evenly.  Otherwise class 1 goes on at the XCD where class 0
// ended, and the last round is runs as well: what the nibble kernel's short launches are faster with.
// Measured, us, contiguous ranges / runs / even, w13 and w2 launch:
//   bf16, Qwen1.5 shape    65 tokens 115.5 / 116.2 / 116.7 and 77.6 / 88.3 / 77.8, 379 tokens 135.6 / 136.5 / 136.5 and
//                          91.1 / 93.4 / 91.6, 1999 tokens 228 / 224 / 224 and 132 / 131 / 135
//   bf16, Mixtral shape    1024 tokens 489 / 423 / 424 and 287 / 289 / 287, 2048 tokens 909 / 738 / 737 and 519 / 470 / 467
//   int4, DeepSeek shape   (runs / even) 65 tokens 34.3 / 34.5 and 31.7 / 33.1, 200 tokens 44.9 / 46.5 and 36.4 / 37.6, 2048
//                          tokens 194 / 193 and 109 / 110
#define PF_DEAL 8
#define PF_GROUP 8
template <bool EVEN>
static __device__ __forceinline__ bool pf_block_of(const PfArgs &a, int &ci, int &mt, int &nt, int &split) {
  const int pad0 = a.c[0].n_blocks;
  ci = (int)blockIdx.x >= pad0;
  const int pb = ci ? (int)blockIdx.x - pad0 : (int)blockIdx.x;
  const PfClass &c = a.c[ci];
  const int ks = c.ksplit > 1 ? c.ksplit : 1;
  const int n_tiles = *c.n_tiles_real * c.n_ntiles, n_real = n_tiles * ks;
  int xcd = pb & 7;
  if (!EVEN && ci) {
    const int n0 = *a.c[0].n_tiles_real * a.c[0].n_ntiles * (a.c[0].ksplit > 1 ? a.c[0].ksplit : 1);
    xcd = (xcd - (n0 + PF_DEAL - 1) / PF_DEAL) & 7;
  }
  const int i = pb >> 3, first = i / PF_DEAL * (8 * PF_DEAL), j = i % PF_DEAL;  // first: the round's first block
  int b = first + xcd * PF_DEAL + j;
  if (EVEN && n_real - first < 8 * PF_DEAL) {
    const int each = (n_real - first + 7) >> 3;
    if (j >= each) return false;
    b = first + xcd * each + j;
  }
  if (b >= n_real) return false;
  // a class whose reduction is split has ksplit workgroups per tile: the pieces of one tile are `n_tiles` blocks
  // apart, so that the first piece of every tile starts before the second of any
  split = b / n_tiles;
  b -= split * n_tiles;
  mt = b / c.n_ntiles;
  const int grp = c.tiles[mt].rows_group >> 16, size = grp & 0xff;
  mt -= (grp >> 8) & 0xff;               // the group's first tile
  b -= mt * c.n_ntiles;
  nt = b / size;
  mt += b - nt * size;
  return true;
}

// ---- bf16 experts: main loop of one wave ------------------------------------------------------------
// One wave per SIMD, 512 registers each: wave w owns columns 32w..32w+31 of both column halves and ALL row
// blocks of the tile (up to 8 x 32 rows: 256 accumulator registers, which the compiler keeps in the
// accumulation half of the register file), so every weight fragment is fetched by exactly one wave of the
// workgroup.  The weights lie in HBM in operand order (blocks of 32 rows x 64 k, one contiguous KiB per MFMA
// step; within a 64-wide K slab lane half q = lane / 32 takes k = 32 q + 8 j + 0..7 for MFMA j: both operands
// use the same permutation of k, which a dot product allows) and never touch LDS.
// What a single wave per SIMD needs, since nothing else fills its stalls (each measured on the Qwen1.5 shape
// and in a stand-alone loop of the same structure):
//   * weight fragments and activations are requested three slabs ahead (four register sets of fragments,
//     four activation slabs in LDS);
//   * the requests are spread between the products, at most one behind each, instead of standing in a block
//     at the head of a slab where the matrix core runs dry behind them (stand-alone loop, streaming from HBM:
//     1.29 -> 1.53 PFLOP/s);
//   * the activation fragment of a product is read from LDS four product groups ahead, and nothing may move
//     across the pinned order (left to itself the scheduler puts every read right in front of its own
//     products and waits for it there: an LDS round trip per pair of products);
//   * no vector instruction computes an address inside the loop (buffer addressing: lane offsets that never
//     change, slab offsets in scalars; LDS addresses with compile-time ring slots).
#define PF_ST 4                      // register sets of weight fragments: requested three slabs ahead
#define PF4_SLAB (PF_BM * PF_BK)     // bf16 elements of one activation slab in LDS (rows of 128 bytes, no padding)
#define PF4_RING 4                   // slabs in LDS: one being read, three on their way
#define PF_FD 4                      // LDS reads in flight in front of the products
typedef __attribute__((address_space(3))) void pf_lds_void;
typedef __attribute__((address_space(1))) const void pf_g_void;
// s_waitcnt that waits for all but the N most recent vector-memory operations and for nothing else
#define PF_VMCNT(N) __builtin_amdgcn_s_waitcnt(((N) & 15) | (7 << 4) | (15 << 8) | (((N) >> 4) << 14))

typedef int pf_i32x4_t __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t pf_rsrc_t;

// Activations go global -> LDS directly (no registers, no LDS store instructions): transfer n of wave w
// brings rows 32 n + 8 w .. + 7 of the slab, 8 lanes per row.  An LDS row is 128 bytes = 8 chunks of 16; the
// chunk that holds k = 8 c .. 8 c + 7 of row r sits in slot c ^ ((r >> 1) & 7), so the 16 lanes that a
// ds_read_b128 serves together (16 rows, one chunk index) fall on 16 different bank groups.  The lanes choose
// their global address accordingly; the LDS side of the transfer is fixed (lane l writes 16 bytes at 16 l).
// All addresses are buffer addresses (lane offset in a register that never changes, slab offset in a scalar):
// with one wave per SIMD every vector instruction that is not a product is issue time taken from the products.
// NTW: the weight fragments are read with the non-temporal hint (a routed expert's tile is the only reader of
// its fragments: they only pass through the caches); the shared expert's row tiles all read the same fragments
// and those are requested with plain loads, so that the second-level cache keeps them for the next row tile
// nk slabs of a row of Kn; rot0, rot1: the storage positions of the first one in the two column halves
template <int NB, bool NTW>
static __device__ __forceinline__ void pf_mainloop(f32x16_t (&acc)[8][2], unsigned lds_base, const pf_i32x4_t ra_rsrc,
                                                    const int (&a_voff)[8], const pf_rsrc_t rb, int b_delta1, int nk, int Kn, int rot0,
                                                    int rot1, int tid) {
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, q = lane >> 5;
  constexpr int NL = NB + 8;   // requests of a step: NB activation transfers, 8 weight fragments
  constexpr int NS = 4 * NB;   // groups of two products
  u32x4_t bw[PF_ST][2][4];
  const int b_voff = lane * 16;
  // transfer n of slab kt_ into ring slot `slot` (past the end: the last slab again, into a slot nobody reads)
  auto dma = [&](int n, int kt_, int slot) {
    const int kt = kt_ < nk ? kt_ : nk - 1;
    // Written as assembly on purpose: the compiler, told that a load writes LDS, waits for ALL such loads in
    // front of every barrier and LDS read, which would end the run-ahead; here the waits are placed by hand
    // (PF_VMCNT below).  Its own counts for the fragment loads then include fewer operations than are in
    // flight, which only makes its waits for those loads earlier, never later.
    const unsigned lds_addr = lds_base + (unsigned)(slot * PF4_SLAB + (32 * n + 8 * w) * PF_BK) * 2u;
    __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :: "s"(lds_addr), "v"(a_voff[n]), "s"(ra_rsrc), "s"(kt * (PF_BK * 2)) : "memory", "m0");
  };
  auto bslab = [&](int kt_, int rot) {
    const int kt = kt_ < nk ? kt_ : nk - 1;  // past the end: the last slab once more (never used)
    const int k = kt + rot;                  // slab position inside the 128-row group's storage of Kn slabs
    return (k >= Kn ? k - Kn : k) * 16384;   // bytes
  };
  // LDS byte address of the lane's fragment of MFMA step j in row block 0 of slot 0 (chunk 4 q + j of its row)
  unsigned faddr[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) faddr[j] = lds_base + (unsigned)(fr * PF_BK + (((4 * q + j) ^ ((fr >> 1) & 7)) * 8)) * 2u;
  auto lds_frag = [&](int slot, int g) {
    typedef __attribute__((address_space(3))) const bf16x8_t lds_frag_t;
    return *(lds_frag_t *)(uintptr_t)(faddr[g / NB] + (unsigned)(slot * PF4_SLAB + 32 * (g % NB) * PF_BK) * 2u);
  };
  // slab kt (ring slot S = kt % 4, a compile-time number in the unrolled loop): its weight fragments are in
  // `cur`.  Requested meanwhile, at most one request behind every product: the activations (into slot
  // (S + 3) % 4) and the fragments (into `far`) of slab kt + 3.
  auto step = [&](auto S_, int kt, const u32x4_t(&cur)[2][4], u32x4_t(&far)[2][4]) {
    constexpr int S = decltype(S_)::value;
    const int sb0 = bslab(kt + 3, rot0), sb1 = bslab(kt + 3, rot1) + b_delta1;
    // product group g = MFMA step j = g / NB of row block i = g % NB; its activation fragment is read from LDS
    // PF_FD groups ahead of its products
    bf16x8_t fa[PF_FD + 1];
#pragma unroll
    for (int g = 0; g < PF_FD && g < NS; ++g) fa[g] = lds_frag(S, g);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NS; ++g) {
      acc[g % NB][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[g % (PF_FD + 1)], __builtin_bit_cast(bf16x8_t, cur[0][g / NB]),
                                                               acc[g % NB][0], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (g + PF_FD < NS) fa[(g + PF_FD) % (PF_FD + 1)] = lds_frag(S, g + PF_FD);
      __builtin_amdgcn_sched_barrier(0);
      acc[g % NB][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[g % (PF_FD + 1)], __builtin_bit_cast(bf16x8_t, cur[1][g / NB]),
                                                               acc[g % NB][1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < NL; ++n)
        if (n * NS / NL == g) {  // request n of this step goes out behind product group g
          if (n < NB) dma(n, kt + 3, (S + 3) % PF4_RING);
          else if (n - NB < 4) far[0][n - NB] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_voff + 1024 * (n - NB), sb0, NTW ? 2 : 0);
          else far[1][n - NB - 4] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_voff + 1024 * (n - NB - 4), sb1, NTW ? 2 : 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    // slab kt + 1 must have landed before anybody reads it: its transfers are two steps old, issued before
    // the 8 fragment loads of their own step and the NB + 8 requests of each of the two steps since
    PF_VMCNT(2 * NB + 24);
    __syncthreads();
  };
  auto gloadB = [&](u32x4_t(&b)[2][4], int kt) {
    const int sb0 = bslab(kt, rot0), sb1 = bslab(kt, rot1) + b_delta1;
#pragma unroll
    for (int j = 0; j < 4; ++j) b[0][j] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_voff + 1024 * j, sb0, NTW ? 2 : 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) b[1][j] = __builtin_amdgcn_raw_buffer_load_b128(rb, b_voff + 1024 * j, sb1, NTW ? 2 : 0);
  };
#pragma unroll
  for (int t = 0; t < 3; ++t) {
#pragma unroll
    for (int n = 0; n < NB; ++n) dma(n, t, t);
    gloadB(bw[t], t);
  }
  PF_VMCNT(0);
  __syncthreads();
  typedef std::integral_constant<int, 0> S0; typedef std::integral_constant<int, 1> S1;
  typedef std::integral_constant<int, 2> S2; typedef std::integral_constant<int, 3> S3;
  for (int kt = 0; kt < nk; kt += 4) {  // nk is even; no separate tail: its register assignment would differ
    step(S0(), kt, bw[0], bw[3]);      // from the loop's and the compiler would spill around the loop's back edge
    step(S1(), kt + 1, bw[1], bw[0]);
    if (kt + 2 < nk) {
      step(S2(), kt + 2, bw[2], bw[1]);
      step(S3(), kt + 3, bw[3], bw[2]);
    }
  }
}

template <bool SWIGLU>
__global__ __launch_bounds__(256, 1) void k_prefill_gemm(const PfArgs a) {
  extern __shared__ __align__(16) uint16_t As[];  // [PF4_RING][PF_BM][PF_BK]
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int ci, mt, nt, split;
  if (!pf_block_of<true>(a, ci, mt, nt, split)) return;
  const PfClass &c = a.c[ci];
  const PfTile tile = c.tiles[mt];
  const int rows = pf_rows(tile);
  if (rows <= 0) return;
  // this workgroup's window of the reduction (only the shared expert's w2 pass is ever split)
  const int Kn = c.K / PF_BK, nk = SWIGLU || c.ksplit <= 1 ? Kn : Kn / c.ksplit, kt0 = SWIGLU ? 0 : split * nk;
  const int n0 = nt * c.n_cols_per_tile;
  const uint16_t *W = (const uint16_t *)(tile.w_base + c.w_off);

  // transfer n of this wave brings rows 32 n + 8 w .. + 7, 8 lanes per row; the lane in slot s of row r
  // fetches chunk s ^ ((r >> 1) & 7).  Byte offsets from the activation tensor's base (< 2 GiB, checked by the launcher)
  int a_voff[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int rt = 32 * i + 8 * w + (lane >> 3);
    const int row = rt < rows ? rt : 0;  // rows past the group's end re-read row 0 (never stored)
    const int grow = tile.row0 + row;
    const int arow = c.gather ? c.gather[grow] : grow;
    a_voff[i] = (arow * c.act_stride + (((lane & 7) ^ ((rt >> 1) & 7)) * 8)) * 2;
  }
  pf_i32x4_t ra_rsrc;
  {
    const unsigned long long ab = (unsigned long long)(c.act + kt0 * PF_BK);
    ra_rsrc.x = __builtin_amdgcn_readfirstlane((int)(unsigned)ab);
    ra_rsrc.y = __builtin_amdgcn_readfirstlane((int)(unsigned)(ab >> 32));
    ra_rsrc.z = 0x7fffffff; ra_rsrc.w = 0x00020000;
  }
  // weight blocks of 32 rows x 64 k (4 KiB); the 4 blocks of a 128-row group are adjacent for each k slab, so
  // one slab of a column half is 16 KiB of contiguous memory; wave w reads block w
  const unsigned char *wb = (const unsigned char *)W + ((size_t)(n0 / 128) * Kn * 4 + w) * 4096;
  const unsigned long long wbu = (unsigned long long)wb;
  const pf_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(wbu >> 32)) << 32) |
               (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)wbu)), 0, 0x7fffffff, 0x00020000);
  const int b_delta1 = (int)(c.half_delta / 128) * Kn * 16384;

  f32x16_t acc[8][2];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][h][e] = 0.f;

  const int G0 = n0 / 128, G1 = G0 + (int)(c.half_delta / 128);
  const int rot0 = (int)((unsigned)(G0 * c.slab_step + kt0) % (unsigned)Kn), rot1 = (int)((unsigned)(G1 * c.slab_step + kt0) % (unsigned)Kn);
  const int nb = (rows + 31) >> 5;  // live row blocks (uniform for the workgroup)
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) uint16_t *)As;
#define PF_LOOPS(NTW_)                                                                                          \
  switch (nb) {                                                                                             \
    case 1: pf_mainloop<1, NTW_>(acc, lds_base, ra_rsrc, a_voff, rb, b_delta1, nk, Kn, rot0, rot1, tid); break; \
    case 2: pf_mainloop<2, NTW_>(acc, lds_base, ra_rsrc, a_voff, rb, b_delta1, nk, Kn, rot0, rot1, tid); break; \
    case 3: pf_mainloop<3, NTW_>(acc, lds_base, ra_rsrc, a_voff, rb, b_delta1, nk, Kn, rot0, rot1, tid); break; \
    case 4: pf_mainloop<4, NTW_>(acc, lds_base, ra_rsrc, a_voff, rb, b_delta1, nk, Kn, rot0, rot1, tid); break; \
    case 5: pf_mainloop<5, NTW_>(acc, lds_base, ra_rsrc, a_voff, rb, b_delta1, nk, Kn, rot0, rot1, tid); break; \
    case 6: pf_mainloop<6, NTW_>(acc, lds_base, ra_rsrc, a_voff, rb, b_delta1, nk, Kn, rot0, rot1, tid); break; \
    case 7: pf_mainloop<7, NTW_>(acc, lds_base, ra_rsrc, a_voff, rb, b_delta1, nk, Kn, rot0, rot1, tid); break; \
    default: pf_mainloop<8, NTW_>(acc, lds_base, ra_rsrc, a_voff, rb, b_delta1, nk, Kn, rot0, rot1, tid); break; \
  }
  if (c.shared) { PF_LOOPS(false) } else { PF_LOOPS(true) }
#undef PF_LOOPS
  // epilogue.  acc element e of lane l: row 8*(e/4) + 4*(l/32) + e%4, column l%32
  const int col = 32 * w + (lane & 31);
  if constexpr (SWIGLU) {
    // The h tile (rows x 128 bf16) goes through LDS, so that it leaves in 16-byte stores that cover whole 256-byte
    // rows: straight from the accumulators a lane stores 2 bytes at a time (128 store instructions per lane, each
    // covering two 64-byte pieces of two rows).  The activation ring is free once every wave has left the main loop
    // and the transfers still on their way into it (the slabs requested past the end) have landed.
    constexpr int HS = 2 * PF_BNH + 16;  // padded row stride in bytes
    static_assert((size_t)PF_BM * HS <= (size_t)PF4_RING * PF4_SLAB * 2, "the h tile fits the activation ring");
    unsigned char *hs = (unsigned char *)As;
    PF_VMCNT(0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < nb) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
          *(__bf16 *)(hs + row * HS + col * 2) = (__bf16)pf_silu_mul(acc[i][0][e], acc[i][1][e]);
        }
      }
    __syncthreads();
    const int chunk = tid & 15;
    for (int row = tid >> 4; row < rows; row += 16) {
      const uint4 v = *(const uint4 *)(hs + row * HS + chunk * 16);
      *(uint4 *)((__bf16 *)c.out + (size_t)(tile.row0 + row) * c.out_stride + n0 + 8 * chunk) = v;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
      if (row < rows) {
        float *o = (float *)c.out + (size_t)split * c.split_stride + (size_t)(tile.row0 + row) * c.out_stride + n0 + col;
        o[0] = acc[i][0][e];
        o[PF_BNH] = acc[i][1][e];
      }
    }
}

// ---- int4-g128 and q4_K experts ---------------------------------------------------------
// A workgroup of four waves (one per SIMD, two workgroups per compute unit) computes a tile of up to 128 rows x
// (128 + 128) columns; wave w owns 32 columns of both halves (for w13 the same columns of gate and up, for w2
// adjacent column blocks) and ALL row blocks of the tile, so every weight is dequantised once per tile.  K advances
// 64 at a time (half a quantisation group).  A 16-byte piece of a nibble tile is 32 consecutive k of one weight row;
// lane (n = lane % 32, q = lane / 32) of a fragment takes row n and the slab's k quarter q, so dword j of its piece is
// the B operand of product j with k = 32 q + 8 j + 0..7 (the order in which the activation rows are read as well: a
// dot product allows any).  What goes into the loop and why:
//   * everything from memory goes global -> LDS directly (buffer_load ... lds) into one ring of slabs: the
//     activation rows (fp16, a converted copy of x or the h rows; 128-byte rows with XOR-swizzled 16-byte chunks),
//     and, private to each wave, the two fragments' nibbles, the scale section and the zero section of the slab.
//     All requests are assembly, so that ONE hand-placed counter wait per slab covers them in order and the
//     compiler, which knows of none, adds no waits of its own;
//   * a slab's nibbles and scales are read from LDS in the third quarter of the slab before it, and the first
//     fragments are dequantised in its last quarter: a wave depends on the others only for the activation rows;
//   * dequantisation (three vector operations per pair, deq8_f16) of product step j + 1 is spread between the
//     products of step j, in pieces of one pair (order pinned by sched_barrier);
//   * two workgroups per compute unit cover each other's barriers, prologues and epilogues.
// h rows leave the w13 pass as fp16, so that the w2 pass brings them into LDS as they are.
// Measured (mean of a launch under the profiler, w13 / w2, whole layers one after the other; outside it 5 to 8 % less): DeepSeek
// shape 2048 tokens 221 / 124 us, 379 tokens 65 / 46, Mixtral shape 4096 tokens 1672 / 907, Qwen2-57B shape q4_K 512 tokens 399 /
// 222.  The kernel before (eight waves, the weights of a tile dequantised by two of them each, activations converted and
// nibbles loaded through registers one group ahead; its blocks dealt in contiguous ranges) against this one with the same
// ranges: 305 / 167 and 215 / 121, 115 / 65 and 76 / 49, 2132 / 1038 and 1733 / 991, 577 / 303 and 408 / 219.
// What bounds it: on the Mixtral shape the power limit (matrix cores busy 78 % and 69 % of the cycles of the two launches,
// which run at 1.46 and 1.51 GHz); on the others partly (DeepSeek shape, 2048 tokens: 59 % and 50 % at 1.70 and 1.81 GHz;
// Qwen2-57B shape, 512 tokens: 61 % and 49 % at 1.65 and 1.78 GHz), with 0.8 to 0.9 vector cycles of dequantisation per
// matrix cycle.  Tiles of 256 rows with one workgroup per compute unit halve the dequantisation per product and lose 8 to
// 15 % on all but the Mixtral shape (+1 %).  q4_K tiles of 64 rows: the Qwen2-57B shape takes 635 instead of 553 us a layer at 512
// tokens and 226 instead of 220 at 65.
// int4 on the scaled 6- and 8-bit matrix formats (a nibble is an fp6 number as it is; x and h split into two pieces) takes 0.83 to
// 0.88 of a layer's time, but holds fewer bits of x and h than fp16: with weights that fp16 holds exactly the partial rows are off by
// 1.0e-3 in norm against 64 bits, 2.0e-4 here, and single elements of h by up to 2^-8 of themselves, 2^-11 here.  More pieces do
// not help: three 6-bit pieces of h are 18 bits a value where the rows have 16, two 8-bit pieces of x take the fp16 products' time.
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

#define PN_BM 128                         // most rows of one tile: 4 blocks of 32 (128 accumulator registers)
#define PN_LDS 81920                      // half of a compute unit's LDS
template <bool Q4K> struct PnSlab {       // one ring slot: activations, then per wave 2 KiB of nibbles and the scales
  static constexpr int SB = Q4K ? 512 : 256;                 // scale bytes of one wave
  static constexpr int bytes(int nb) { return nb * 4096 + 4 * (2048 + SB); }
  static constexpr int ring(int nb) { return PN_LDS / bytes(nb) < 8 ? PN_LDS / bytes(nb) : 8; }
};

static __device__ __forceinline__ pf_i32x4_t pn_rsrc(const void *p) {
  const unsigned long long v = (unsigned long long)p;
  pf_i32x4_t r;
  r.x = __builtin_amdgcn_readfirstlane((int)(unsigned)v);
  r.y = __builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
  r.z = 0x7fffffff; r.w = 0x00020000;
  return r;
}
// 64 lanes x 16 (4) bytes from base + voff + soff to LDS address lds + 16 (4) * lane
static __device__ __forceinline__ void pn_dma16(unsigned lds, int voff, const pf_i32x4_t r, int soff) {
  __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                   :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory", "m0");
}
static __device__ __forceinline__ void pn_dma4(unsigned lds, int voff, const pf_i32x4_t r, int soff) {
  __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                   :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory", "m0");
}
template <typename T>
static __device__ __forceinline__ T pn_lds(unsigned addr) {
  typedef __attribute__((address_space(3))) const T lds_t;
  return *(lds_t *)(uintptr_t)addr;
}

// what a wave of a tile reads; offsets in bytes, voff per lane
struct PnSrc {
  // activation matrix; nibbles, scales and (q4_K) super-block scales of the tile's 16 row blocks (64-bit bases: an expert
  // image may have 2 GiB and more)
  pf_i32x4_t ra, rw, rs, rz;
  int a_voff[4];            // row block n: the lane's row and chunk
  int w_voff[2];            // fragment f
  int s_voff, z_voff;       // scale request; q4_K: (d, dmin) request; int4: s_voff covers scales and zeros
  int s_step;               // int4: what s_voff advances by per quantisation group (scales and zeros differ)
};

// acc[i][f]: row block i, fragment (column half) f; slabs kt0 .. kt0 + nk - 1 (64 k each), nk >= 2
template <int NB, bool Q4K>
static __device__ __forceinline__ void pn_mainloop(f32x16_t (&acc)[NB][2], const unsigned lds_base, const PnSrc &m, const int kt0,
                                                   const int nk, const int tid) {
  constexpr int SB = PnSlab<Q4K>::SB, SLOT = PnSlab<Q4K>::bytes(NB), R = PnSlab<Q4K>::ring(NB);
  constexpr int NS_ = Q4K ? 2 : 1;         // scale requests of a slab
  constexpr int NL = NB + 2 + NS_;         // requests of a slab
  static_assert(R >= 3 && (R - 2) * NL < 63, "ring depth");
  constexpr int NG = 4 * NB;               // product groups of a slab (two products each)
  constexpr int FD = NG < 4 ? NG : 4;      // activation fragments read ahead
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, q = lane >> 5;
  const DeqF16Consts dqc = deq_f16_consts();
  const unsigned wbase = lds_base + (unsigned)(NB * 4096 + w * (2048 + SB));   // this wave's nibbles, then scales
  // request r of slab kt (clamped: past the end the last slab again, into a slot nobody reads) into slot offset so
  auto request = [&](int r, int kt_, int so) {
    const int kt = kt0 + (kt_ < nk ? kt_ : nk - 1);
    if (r < NB) pn_dma16(lds_base + (unsigned)(so + (32 * r + 8 * w) * 128), m.a_voff[r], m.ra, kt * 128);
    else if (r < NB + 2) pn_dma16(wbase + (unsigned)(so + 1024 * (r - NB)), m.w_voff[r - NB], m.rw, kt * 512);
    else if (!Q4K) pn_dma4(wbase + (unsigned)(so + 2048), m.s_voff + (kt >> 1) * m.s_step, m.rs, 0);
    else if (r == NB + 2) pn_dma4(wbase + (unsigned)(so + 2048), m.s_voff, m.rs, kt * 64);
    else pn_dma4(wbase + (unsigned)(so + 2048 + 256), m.z_voff, m.rz, (kt >> 2) * 64);
  };
  // LDS addresses in slot 0: the lane's activation chunk of product step j, its nibbles, its scale words
  unsigned fa0[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) fa0[j] = lds_base + (unsigned)(n * 128 + (((4 * q + j) ^ ((n >> 1) & 7)) * 16));
  const unsigned na0 = wbase + (unsigned)lane * 16u;
  const int t0 = n >> 4, r16 = n & 15;   // fragment f reads row r16 of the wave's row block 2 f + t0
  const unsigned sa0 = wbase + 2048u + (unsigned)(Q4K ? t0 * 64 + (16 * q + r16) * 2 : t0 * 32 + r16 * 2);
  const unsigned za0 = wbase + 2048u + (unsigned)(Q4K ? 256 + t0 * 64 + r16 * 4 : 128 + t0 * 8 + (r16 >> 1));
  const int zsh = 4 * (r16 & 1);
  u32x4_t nib[2], nxt[2];
  u32 s2[2], c2[2], sraw[2], zraw[2];
  u32x4_t wd[2][2];                      // [step parity][fragment]: 8 fp16 weights
  auto read_w = [&](u32x4_t(&d)[2], int so) {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      d[f] = pn_lds<u32x4_t>(na0 + (unsigned)(so + 1024 * f));
      if (Q4K) {
        sraw[f] = pn_lds<uint16_t>(sa0 + (unsigned)(so + 128 * f));
        zraw[f] = pn_lds<u32>(za0 + (unsigned)(so + 128 * f));
      } else {
        sraw[f] = pn_lds<uint16_t>(sa0 + (unsigned)(so + 64 * f));
        zraw[f] = pn_lds<unsigned char>(za0 + (unsigned)(so + 16 * f));
      }
    }
  };
  auto prep = [&]() {  // S = 16 s and C of deq8_f16 for the lane's row in both fragments
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      float s16, cz;
      if (Q4K) {
        s16 = 16.f * __builtin_bit_cast(float, h2f_bits(zraw[f] & 0xffffu)) * (float)(sraw[f] & 0xffu);
        cz = -s16 - __builtin_bit_cast(float, h2f_bits(zraw[f] >> 16)) * (float)((sraw[f] >> 8) & 0xffu);
      } else {
        const float sf = __builtin_bit_cast(float, h2f_bits(sraw[f]));
        s16 = 16.f * sf;
        cz = -(16.f + (float)((zraw[f] >> zsh) & 15u)) * sf;
      }
      const u32 sb = f2h_bits(s16), cb = f2h_bits(cz);
      s2[f] = sb | (sb << 16);
      c2[f] = cb | (cb << 16);
    }
  };
  // pair p (0..7) of a step's two fragments: 3 vector operations
  auto deq_piece = [&](u32x4_t(&dst)[2], const u32x4_t(&src)[2], int j, int p) {
    const int f = p >> 2, e = p & 3;
    const u32 d = src[f][j];
    const u32 sh = e == 0 ? d << 6 : (e == 1 ? d << 2 : (e == 2 ? d >> 2 : d >> 6));
    const f16x2_t h = __builtin_bit_cast(f16x2_t, (sh & dqc.M) | dqc.C);
    dst[f][e] = __builtin_bit_cast(u32, __builtin_elementwise_fma(h, __builtin_bit_cast(f16x2_t, s2[f]), __builtin_bit_cast(f16x2_t, c2[f])));
  };

#pragma unroll
  for (int t = 0; t < R - 1; ++t)
#pragma unroll
    for (int r = 0; r < NL; ++r) request(r, t, t * SLOT);
  PF_VMCNT((R - 2) * NL);
  __syncthreads();
  read_w(nib, 0);
  prep();
#pragma unroll
  for (int p = 0; p < 8; ++p) deq_piece(wd[0], nib, 0, p);
  int so = 0, sn = SLOT, sl = (R - 1) * SLOT;   // slot offsets of slab kt, kt + 1 and kt + R - 1
  for (int kt = 0; kt < nk; ++kt) {
    unsigned fb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) fb[j] = fa0[j] + (unsigned)so;
    auto frag = [&](int g) { return pn_lds<f16x8_t>(fb[g / NB] + (unsigned)((g % NB) * 4096)); };
    f16x8_t fa[FD + 1];
#pragma unroll
    for (int g = 0; g < FD; ++g) fa[g] = frag(g);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int j = g / NB, i = g % NB;
      if (g == 2 * NB) {                // the next slab's own requests have landed: nibbles and scales into registers
        PF_VMCNT((R - 2) * NL);
        read_w(nxt, sn);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (g == 3 * NB) prep();
      auto deq = [&](int half) {        // pieces of the next step's fragments behind this product
#pragma unroll
        for (int p = 0; p < 8; ++p)
          if (p * 2 * NB / 8 == 2 * i + half) deq_piece(wd[(j + 1) & 1], j < 3 ? nib : nxt, (j + 1) & 3, p);
      };
      acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[g % (FD + 1)], __builtin_bit_cast(f16x8_t, wd[j & 1][0]), acc[i][0], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (g + FD < NG) fa[(g + FD) % (FD + 1)] = frag(g + FD);
      deq(0);
      __builtin_amdgcn_sched_barrier(0);
      acc[i][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[g % (FD + 1)], __builtin_bit_cast(f16x8_t, wd[j & 1][1]), acc[i][1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      deq(1);
#pragma unroll
      for (int r = 0; r < NL; ++r)      // requests of slab kt + R - 1 in the first half of the step
        if (r * 2 * NB / NL == g) request(r, kt + R - 1, sl);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    nib[0] = nxt[0]; nib[1] = nxt[1];
    so = sn; 
    sn = sn + SLOT == R * SLOT ? 0 : sn + SLOT;
    sl = sl + SLOT == R * SLOT ? 0 : sl + SLOT;
  }
}

template <int NB, bool SWIGLU, bool Q4K>
static __device__ __forceinline__ void pn_tile(const PfClass &c, const PfTile &tile, unsigned char *lds, int nt, int kt0, int nk,
                                               int split, int tid) {
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, q = lane >> 5;
  const int G = c.K >> 7, rows = pf_rows(tile);
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
  PnSrc m;
  m.ra = pn_rsrc(c.act);
  const size_t tile0 = (size_t)16 * nt * G;   // (row block, group) pairs in front of the tile's
  m.rw = pn_rsrc((const void *)(tile.w_base + c.w_off + tile0 * 1024));
  m.rs = pn_rsrc((const void *)(tile.w_base + c.off_s + tile0 * (Q4K ? 128 : 32)));
  m.rz = pn_rsrc((const void *)(tile.w_base + c.off_z + tile0 * (Q4K ? 32 : 8)));
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m.a_voff[i] = 0;
    if (i < NB) {
      // transfer i of this wave brings rows 32 i + 8 w .. + 7, 8 lanes per row; the lane in slot s of row r fetches
      // chunk s ^ ((r >> 1) & 7).  Byte offsets from the activation tensor's base (< 2 GiB, checked by the launcher)
      const int rt = 32 * i + 8 * w + (lane >> 3);
      const int row = rt < rows ? rt : 0;   // rows past the group's end re-read row 0 (never stored)
      const int grow = tile.row0 + row;
      const int arow = c.gather ? c.gather[grow] : grow;
      m.a_voff[i] = arow * c.act_stride * 2 + (((lane & 7) ^ ((rt >> 1) & 7)) * 16);
    }
  }
  // row block t (0..3) of this wave in the tile, t = 2 f + h: fragment f's lanes 16 h .. 16 h + 15 (of 32).  w13: gate blocks
  // (even) are fragment 0, up blocks (odd) fragment 1; w2: column halves 128 apart
  auto rb = [&](int t) { return SWIGLU ? 4 * w + (t >> 1) + 2 * (t & 1) : 2 * w + 8 * (t >> 1) + (t & 1); };
#pragma unroll
  for (int f = 0; f < 2; ++f)
    m.w_voff[f] = rb(2 * f + (n >> 4)) * G * 1024 + (16 * q + (n & 15)) * 16;
  if (Q4K) {
    m.s_voff = rb(lane >> 4) * G * 128 + (lane & 15) * 4;
    m.z_voff = rb(lane >> 4) * (G >> 1) * 64 + (lane & 15) * 4;
    m.s_step = 0;
  } else {
    // lanes 0..31: 8 dwords of scales of each row block; lanes 32..39: 2 dwords of zeros of each; the rest idle copies.
    // The zeros of the tile lie behind its scales (in the image's next section, less than 2 GiB away: the launcher)
    const int l = lane < 40 ? lane : 39;
    const int z0 = (int)(c.off_z - c.off_s - (long long)tile0 * 24);
    m.s_voff = l < 32 ? rb(l >> 3) * G * 32 + (l & 7) * 4 : z0 + rb((l - 32) >> 1) * G * 8 + (l & 1) * 4;
    m.s_step = l < 32 ? 32 : 8;
    m.z_voff = 0;
  }
  f32x16_t acc[NB][2];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][h][e] = 0.f;
  pn_mainloop<NB, Q4K>(acc, lds_base, m, kt0, nk, tid);
  // epilogue.  acc element e of lane l: row 8*(e/4) + 4*(l/32) + e%4 of its block, column l%32
  const int col = 32 * w + n;
  PF_VMCNT(0);   // the transfers past the end have landed: the ring is free, and nothing is in flight at the end
  if constexpr (SWIGLU) {
    // the h tile (rows x 128 fp16) leaves through LDS in 16-byte stores over whole 256-byte rows
    constexpr int HS = 2 * PF_BNH + 16;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = 32 * i + 8 * (e >> 2) + 4 * q + (e & 3);
        *(_Float16 *)(lds + row * HS + col * 2) = (_Float16)pf_silu_mul(acc[i][0][e], acc[i][1][e]);
      }
    __syncthreads();
    const int chunk = tid & 15;
    for (int row = tid >> 4; row < rows; row += 16)
      *(uint4 *)((_Float16 *)c.out + (size_t)(tile.row0 + row) * c.out_stride + nt * PF_BNH + 8 * chunk) =
          *(const uint4 *)(lds + row * HS + chunk * 16);
  } else {
    float *out = (float *)c.out + (size_t)split * c.split_stride + nt * 2 * PF_BNH + col;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = 32 * i + 8 * (e >> 2) + 4 * q + (e & 3);
        if (row < rows) {
          float *o = out + (size_t)(tile.row0 + row) * c.out_stride;
          o[0] = acc[i][0][e];
          o[PF_BNH] = acc[i][1][e];
        }
      }
  }
}

template <bool SWIGLU, bool Q4K>
__global__ __launch_bounds__(256, 2) void k_prefill_nib(const PfArgs a) {
  extern __shared__ __align__(16) unsigned char lds_n[];
  const int tid = threadIdx.x;
  int ci, mt, nt, split;
  if (!pf_block_of<false>(a, ci, mt, nt, split)) return;
  const PfClass &c = a.c[ci];
  const PfTile tile = c.tiles[mt];
  const int rows = pf_rows(tile);
  if (rows <= 0) return;
  const int ks = c.ksplit > 1 ? c.ksplit : 1;
  // this workgroup's window of the reduction (only the w2 pass is ever split)
  const int nk = SWIGLU ? c.K / PF_BK : c.K / PF_BK / ks, kt0 = SWIGLU ? 0 : split * nk;
  switch ((rows + 31) >> 5) {
    case 1: pn_tile<1, SWIGLU, Q4K>(c, tile, lds_n, nt, kt0, nk, split, tid); break;
    case 2: pn_tile<2, SWIGLU, Q4K>(c, tile, lds_n, nt, kt0, nk, split, tid); break;
    case 3: pn_tile<3, SWIGLU, Q4K>(c, tile, lds_n, nt, kt0, nk, split, tid); break;
    default: pn_tile<4, SWIGLU, Q4K>(c, tile, lds_n, nt, kt0, nk, split, tid); break;
  }
}


// Workgroups of a class of `blocks` blocks: whole rounds of 8 runs, or, where less than a round is spread evenly (EVEN), an
// even share per XCD (56 idle workgroups between the shared expert's 8 w2 blocks and the routed ones of a 65-token batch of
// the Qwen1.5 shape made that launch 85 us instead of 78)
static int pf_padded(bool even, int blocks) {
  const int q = even && blocks < 8 * PF_DEAL ? 8 : 8 * PF_DEAL;
  return (blocks + q - 1) / q * q;
}

template <bool Q4K>
static int pn_launch(bool swiglu, const PfArgs &a, hipStream_t s) {
  if (a.n_blocks_total <= 0) return MOE_OK;
  const int grid = a.c[0].n_blocks + a.c[1].n_blocks;
  static bool attr_set = false;
  if (!attr_set) {
    for (const void *f : {(const void *)k_prefill_nib<true, Q4K>, (const void *)k_prefill_nib<false, Q4K>})
      if (int rc = moe_check_hip(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, PN_LDS),
                                 "hipFuncSetAttribute(k_prefill_nib)"))
        return rc;
    attr_set = true;
  }
  moe_ktimer_begin(swiglu ? MOE_K_PREFILL_W13 : MOE_K_PREFILL_W2, s);
  if (swiglu) hipLaunchKernelGGL((k_prefill_nib<true, Q4K>), dim3(grid), dim3(256), PN_LDS, s, a);
  else hipLaunchKernelGGL((k_prefill_nib<false, Q4K>), dim3(grid), dim3(256), PN_LDS, s, a);
  moe_ktimer_end(swiglu ? MOE_K_PREFILL_W13 : MOE_K_PREFILL_W2, s);
  return moe_check_launch("k_prefill_nib");
}

static int pf_launch(bool swiglu, const PfArgs &a, hipStream_t s) {
  if (a.n_blocks_total <= 0) return MOE_OK;
  const int grid = a.c[0].n_blocks + a.c[1].n_blocks;
  const size_t lds = (size_t)PF4_RING * PF4_SLAB * 2;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e1 = hipFuncSetAttribute((const void *)k_prefill_gemm<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipError_t e2 = hipFuncSetAttribute((const void *)k_prefill_gemm<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (int rc = moe_check_hip(e1 != hipSuccess ? e1 : e2, "hipFuncSetAttribute(k_prefill_gemm)")) return rc;
    attr_set = true;
  }
  moe_ktimer_begin(swiglu ? MOE_K_PREFILL_W13 : MOE_K_PREFILL_W2, s);
  if (swiglu) hipLaunchKernelGGL(k_prefill_gemm<true>, dim3(grid), dim3(256), lds, s, a);
  else hipLaunchKernelGGL(k_prefill_gemm<false>, dim3(grid), dim3(256), lds, s, a);
  moe_ktimer_end(swiglu ? MOE_K_PREFILL_W13 : MOE_K_PREFILL_W2, s);
  return moe_check_launch("k_prefill_gemm");
}

// ---- tile list ------------------------------------------------------------------------
// One entry per tile of every active expert's token group (routed list: a group of more rows than a tile holds is
// split evenly), and one per tile of tokens for the shared expert's two passes.  Built on the device from the
// dispatch result, so the host never needs the counts: the launch covers the upper bound on the number of blocks, and
// blocks past the real count find nothing to do.  The routed list is in order of tile height, the tallest first (four
// classes; expert order inside a class), so that no long workgroup starts when the launch is nearly over.
// Nibble formats: the same launch converts x to fp16 for the w13 pass (8 MB read and written for 2048 x 2048, hidden
// behind the 4 us that the list takes).  One more workgroup takes the unit list to the host: two copies and an event
// behind the routing stood in the stream for 9 us a layer.
static __device__ __forceinline__ PfTile pf_make_tile(unsigned long long w_base, int row0, int rows, int i, int n) {
  PfTile t;                                  // tile i of n of one expert
  const int g0 = i / PF_GROUP * PF_GROUP;
  t.w_base = w_base; t.row0 = row0; t.rows_group = rows | (min(PF_GROUP, n - g0) << 16) | ((i - g0) << 24);
  return t;
}
__global__ __launch_bounds__(1024) void k_prefill_tiles(const moe_unit *__restrict__ units, int max_units,
                                                        const unsigned long long *__restrict__ expert_ptr,
                                                        PfTile *__restrict__ tiles, int n_tiles_max,
                                                        PfTile *__restrict__ sh_tiles, int n_sh_tiles,
                                                        PfTile *__restrict__ sh_tiles2, int n_sh_tiles2,
                                                        unsigned long long shared_base, int T, int cap, int cap_s, int cap_s2,
                                                        int *__restrict__ n_real, int *__restrict__ err,
                                                        const u32x4_t *__restrict__ x, u32x4_t *__restrict__ x16, int n16,
                                                        const moe_publish pub) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int conv0 = pub.units_host ? 2 : 1;
  if (blockIdx.x > 0) {  // workgroups behind the first: the unit list to the host, the fp16 copy of the activations
    if ((int)blockIdx.x < conv0) { publish_units(pub, units, tid, 1024); return; }
    const int i = ((int)blockIdx.x - conv0) * 1024 + tid;   // (8 values per thread)
    if (i < n16) {
      const u32x4_t v = x[i];
      x16[i] = u32x4_t{bf16x2_to_f16x2(v.x), bf16x2_to_f16x2(v.y), bf16x2_to_f16x2(v.z), bf16x2_to_f16x2(v.w)};
    }
    return;
  }
  __shared__ int total[4];
  __shared__ unsigned long long wsum[16];
  if (tid < 4) total[tid] = 0;
  for (int i = tid; i < n_sh_tiles; i += 1024)
    sh_tiles[i] = pf_make_tile(shared_base, i * cap_s, min(cap_s, T - i * cap_s), i, n_sh_tiles);
  for (int i = tid; i < n_sh_tiles2; i += 1024)
    sh_tiles2[i] = pf_make_tile(shared_base, i * cap_s2, min(cap_s2, T - i * cap_s2), i, n_sh_tiles2);
  __syncthreads();
  // tiles of unit u: nt of up to `per` rows (a multiple of 32); class 0 = the tallest quarter
  int m = 0, row0 = 0, nt = 0, per = 0, cls = 0;
  unsigned long long wb = 0;
  auto load = [&](int u, bool report) {
    m = 0; wb = 0; row0 = 0;
    if (u < max_units) {
      const moe_unit un = units[u];
      if (un.m > 0 && un.expert >= 0) {
        wb = expert_ptr[un.expert];
        if (wb) { m = un.m; row0 = un.row0; }
        else if (report) moe_raise_err(err);
      }
    }
    nt = (m + cap - 1) / cap;
    per = nt ? ((((m + nt - 1) / nt) + 31) & ~31) : 0;
    cls = nt ? min(3, (cap - per) * 4 / cap) : 0;
  };
  // Tile counts of the four classes travel as 16-bit fields of one word (1024 units of one batch have at most 2^15 + 1024
  // tiles: activation buffers stay under 2 GiB, launcher): one scan instead of four, and the sums over the waves in use.
  // (Counting the totals first and scanning class by class, over 16 waves whatever the number of units, took 4.8 us on 16 experts
  // instead of 3.7, 5.6 instead of 4.8 on 60.)
  const bool once = max_units <= 1024;   // the totals then come out of the only scan
  if (!once)
    for (int base = 0; base < max_units; base += 1024) {
      load(base + tid, true);
      if (nt) atomicAdd(&total[cls], nt);
    }
  __syncthreads();
  int done[4] = {0, total[0], total[0] + total[1], total[0] + total[1] + total[2]};  // first free entry per class
  int n_all = done[3] + total[3];
  for (int base = 0; base < max_units; base += 1024) {
    load(base + tid, once);
    // tiles of the same class in front of this unit's: inside the wave, then the waves before
    unsigned long long v = (unsigned long long)nt << (16 * cls), before = 0, all = 0;
    const unsigned long long own = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned long long o = __shfl_up(v, d);
      if (lane >= d) v += o;
    }
    if (lane == 63) wsum[wave] = v;
    __syncthreads();
    const int waves = min(16, (max_units - base + 63) >> 6);
    for (int w = 0; w < waves; ++w) {
      const unsigned long long o = wsum[w];
      if (w < wave) before += o;
      all += o;
    }
    int in_all[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) in_all[c] = (int)(all >> (16 * c)) & 0xffff;
    if (once) {
      done[1] = in_all[0]; done[2] = done[1] + in_all[1]; done[3] = done[2] + in_all[2];
      n_all = done[3] + in_all[3];
    }
    const int first = (cls < 2 ? (cls ? done[1] : done[0]) : (cls == 2 ? done[2] : done[3])) +
                      ((int)((before + v - own) >> (16 * cls)) & 0xffff);
    for (int i = 0; i < nt; ++i)
      if (first + i < n_tiles_max) tiles[first + i] = pf_make_tile(wb, row0 + i * per, max(0, min(per, m - i * per)), i, nt);
    if (!once) {
#pragma unroll
      for (int c = 0; c < 4; ++c) done[c] += in_all[c];
      __syncthreads();
    }
  }
  if (tid == 0) { n_real[0] = min(n_all, n_tiles_max); n_real[1] = n_sh_tiles; n_real[2] = n_sh_tiles2; }
}

extern "C" int moe_prefill_tile_rows(void) { return PF_BM; }

extern "C" int64_t moe_prefill_workspace_bytes(int T, int k, int max_units) {
  const int64_t P = (int64_t)T * k;
  return (P / 128 + max_units + 2 * ((T + 127) / 128) + 3) * (int64_t)sizeof(PfTile);  // covers every tile height in use (>= 128)
}

// where the fp16 copy of the activations stands in a workspace with room for it (phase bit 2)
static int64_t pf_x16_offset(int T, int k, int max_units) {
  return (moe_prefill_workspace_bytes(T, k, max_units) + 255) & ~(int64_t)255;
}

// Pieces the w2 pass leaves the shared expert's partial rows in (moe_experts_prefill_pieces).  The shared expert's
// workgroups of that pass each reduce over all of I_sh; where there are few of them (ceil(T/128) row tiles x H/256
// column tiles) and the reduction is long, they outlast everything else in the launch: Qwen2-57B shape (H 3584,
// I_sh 20480) at 512 tokens, 56 workgroups over 160 groups each: 371 us for the launch, 285 us with the reduction in 4
// windows (8 windows: no shorter, and the combine reads twice the partial rows).  Then the reduction is cut into 2, 4
// or 8 windows of at least 32 groups, a workgroup per tile and window, until there are 192 of them.
// bf16 batches of decode size have a rule of their own (moe_decode_bf16_splits).
extern "C" int moe_prefill_shared_splits(int fmt, int T, int H, int I_sh) {
  if (fmt == MOE_FMT_BF16 && T > 0 && H > 0 && I_sh > 0 && moe_decode_bf16_takes(T)) return moe_decode_bf16_splits(H, I_sh);
  if ((fmt != MOE_FMT_INT4_G128 && fmt != MOE_FMT_Q4K) || T <= 0 || H <= 0 || I_sh <= 0) return 1;
  const int tiles = ((T + PF_BM_SHARED_W2 - 1) / PF_BM_SHARED_W2) * (H / (2 * PF_BNH));
  const int G = I_sh / 128;
  int s = 1;
  while (s < 8 && tiles * s < 192 && G % (s * 4) == 0 && G / (s * 2) >= 32) s *= 2;
  return s;
}

extern "C" int moe_experts_prefill(const void *x_bf16, int T, int H, int I, int I_sh, int k, int fmt,
                                   const moe_unit *units, int max_units, const int *sorted_tok,
                                   const uint64_t *expert_ptr, const void *shared_ptr, void *h_r, void *h_s,
                                   float *part_r, float *part_s, void *tiles_ws, int *err, int phases,
                                   void *stream) {
  return moe_experts_prefill_pieces(x_bf16, T, H, I, I_sh, k, fmt, units, max_units, sorted_tok, expert_ptr, shared_ptr,
                                    h_r, h_s, part_r, part_s, 1, tiles_ws, err, phases, stream);
}

extern "C" int moe_experts_prefill_pieces(const void *x_bf16, int T, int H, int I, int I_sh, int k, int fmt,
                                          const moe_unit *units, int max_units, const int *sorted_tok,
                                          const uint64_t *expert_ptr, const void *shared_ptr, void *h_r, void *h_s,
                                          float *part_r, float *part_s, int shared_pieces, void *tiles_ws, int *err,
                                          int phases, void *stream) {
  return moe_experts_prefill_publish(x_bf16, T, H, I, I_sh, k, fmt, units, max_units, sorted_tok, expert_ptr, shared_ptr, h_r,
                                     h_s, part_r, part_s, shared_pieces, tiles_ws, err, phases, nullptr, stream);
}

static int experts_prefill(bool windows, const void *x_bf16, int T, int H, int I, int I_sh, int k, int fmt,
                           const moe_unit *units, int max_units, const int *sorted_tok,
                           const uint64_t *expert_ptr, const void *shared_ptr, void *h_r, void *h_s,
                           float *part_r, float *part_s, int shared_pieces, int routed_pieces,
                           void *tiles_ws, int *err, int phases, const moe_publish *pub, void *stream);

extern "C" int moe_experts_prefill_publish(const void *x_bf16, int T, int H, int I, int I_sh, int k, int fmt,
                                           const moe_unit *units, int max_units, const int *sorted_tok,
                                           const uint64_t *expert_ptr, const void *shared_ptr, void *h_r, void *h_s,
                                           float *part_r, float *part_s, int shared_pieces, void *tiles_ws, int *err,
                                           int phases, const moe_publish *pub, void *stream) {
  return experts_prefill(false, x_bf16, T, H, I, I_sh, k, fmt, units, max_units, sorted_tok, expert_ptr, shared_ptr, h_r, h_s,
                         part_r, part_s, shared_pieces, 1, tiles_ws, err, phases, pub, stream);
}

extern "C" int moe_experts_prefill_windows(const void *x_bf16, int T, int H, int I, int I_sh, int k, int fmt,
                                           const moe_unit *units, int max_units, const int *sorted_tok,
                                           const uint64_t *expert_ptr, const void *shared_ptr, void *h_r, void *h_s,
                                           float *part_r, float *part_s, int shared_pieces, int routed_pieces,
                                           void *tiles_ws, int *err, int phases, const moe_publish *pub, void *stream) {
  return experts_prefill(true, x_bf16, T, H, I, I_sh, k, fmt, units, max_units, sorted_tok, expert_ptr, shared_ptr, h_r, h_s,
                         part_r, part_s, shared_pieces, routed_pieces, tiles_ws, err, phases, pub, stream);
}

// windows: moe_experts_prefill_windows, whose pieces are windows of whole slabs; the older entries take the shared expert's
// in pairs of quantisation groups and leave the routed experts' rows whole
static int experts_prefill(bool windows, const void *x_bf16, int T, int H, int I, int I_sh, int k, int fmt,
                           const moe_unit *units, int max_units, const int *sorted_tok,
                           const uint64_t *expert_ptr, const void *shared_ptr, void *h_r, void *h_s,
                           float *part_r, float *part_s, int shared_pieces, int routed_pieces,
                           void *tiles_ws, int *err, int phases, const moe_publish *pub, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  if (pub && (T <= 0 || max_units <= 0 || !(phases & 1) || !moe_publish_ok(pub, max_units))) {
    moe_set_error("moe_experts_prefill_publish: publishing needs tokens, units and the w13 phase (T=%d phases=%d)", T, phases);
    return MOE_EINVAL;
  }
  if (T == 0) return MOE_OK;
  if (shared_pieces != 1 && shared_pieces != 2 && shared_pieces != 4 && shared_pieces != 8) {
    moe_set_error("moe_experts_prefill: shared_pieces = %d (1, 2, 4 or 8)", shared_pieces);
    return MOE_EINVAL;
  }
  const bool bf16_decode = fmt == MOE_FMT_BF16 && moe_decode_bf16_takes(T);
  if (shared_pieces > 1 && bf16_decode && shared_ptr) {
    if ((I_sh / 64) % shared_pieces != 0) {
      moe_set_error("moe_experts_prefill: %d pieces do not divide the bf16 shared expert's I_sh / 64 (I_sh=%d)", shared_pieces, I_sh);
      return MOE_EINVAL;
    }
  } else if (shared_pieces > 1 && windows && fmt == MOE_FMT_BF16) {
    if (!shared_ptr || (I_sh / 64) % (shared_pieces * 2) != 0) {   // (the tile kernel's loop takes an even number of slabs)
      moe_set_error("moe_experts_prefill: %d windows need a bf16 shared expert whose I_sh / 64 is a multiple of %d (I_sh=%d)",
                    shared_pieces, shared_pieces * 2, I_sh);
      return MOE_EINVAL;
    }
  } else if (shared_pieces > 1 && (!shared_ptr || (fmt != MOE_FMT_INT4_G128 && fmt != MOE_FMT_Q4K) ||
                                   (windows ? (I_sh / 64) % shared_pieces || I_sh / 64 / shared_pieces < 2
                                            : (I_sh / 128) % (shared_pieces * 2) != 0))) {
    moe_set_error("moe_experts_prefill: %d pieces need an int4 / q4_K shared expert whose I_sh / %d is a multiple of %d "
                  "(I_sh=%d)", shared_pieces, windows ? 64 : 128, windows ? shared_pieces : shared_pieces * 2, I_sh);
    return MOE_EINVAL;
  }
  if (!x_bf16 || T < 0 || k <= 0 || max_units < 0 || !units || !sorted_tok || !expert_ptr || !tiles_ws || !err ||
      !h_r || !part_r || (shared_ptr && (!h_s || !part_s || I_sh <= 0))) {
    moe_set_error("moe_experts_prefill: NULL or negative argument");
    return MOE_EINVAL;
  }
  if (routed_pieces < 1 || routed_pieces > 8 || (routed_pieces > 1 && (fmt == MOE_FMT_BF16 || I % 64 || (I / 64) % routed_pieces ||
                                                                       I / 64 / routed_pieces < 2))) {
    moe_set_error("moe_experts_prefill: %d windows of a reduction over %d columns of the routed experts (format %d)", routed_pieces, I, fmt);
    return MOE_EINVAL;
  }
  if (fmt != MOE_FMT_BF16 && fmt != MOE_FMT_INT4_G128 && fmt != MOE_FMT_Q4K) {
    moe_set_error("moe_experts_prefill: weight format %d not supported by the prefill kernels", fmt);
    return MOE_EINVAL;
  }
  const bool q4k = fmt == MOE_FMT_Q4K;
  const bool int4 = fmt == MOE_FMT_INT4_G128 || q4k;  // nibble tiles + fp16 operands
  if (q4k && (H % 256 || I % 256 || (shared_ptr && I_sh % 256))) {
    moe_set_error("moe_experts_prefill: q4_K experts need H, I multiples of 256 (H=%d I=%d I_sh=%d)", H, I, I_sh);
    return MOE_EINVAL;
  }
  if (H % 256 || I % 128 || (shared_ptr && I_sh % 128)) {
    moe_set_error("moe_experts_prefill: H %% 256 == 0 and I %% 128 == 0 required (H=%d I=%d I_sh=%d)", H, I, I_sh);
    return MOE_EINVAL;
  }
  if (int rc = moe_check_expert_sizes("moe_experts_prefill", int4, T, k, H, I, shared_ptr ? I_sh : 0)) return rc;
  if (bf16_decode)
    return moe_decode_bf16(x_bf16, T, H, I, I_sh, units, max_units, sorted_tok, expert_ptr, shared_ptr, h_r, h_s, part_r, part_s,
                           shared_pieces, err, phases, pub, s);
  const long long P = (long long)T * k;
  const int cap = int4 ? PN_BM : PF_BM, cap_s = int4 ? PN_BM : PF_BM_SHARED, cap_s2 = PF_BM_SHARED_W2;
  // fp16 copy of x for the nibble formats: behind the tile list where the caller left room, else stream-ordered memory
  void *x16 = nullptr, *x16_own = nullptr;
  const bool convert = int4 && (phases & 1);
  if (convert) {
    if (phases & 4) x16 = (unsigned char *)tiles_ws + pf_x16_offset(T, k, max_units);
    else if (int rc = moe_check_hip(hipMallocAsync(&x16_own, (size_t)T * H * 2, s), "hipMallocAsync(fp16 activations)")) return rc;
    if (x16_own) x16 = x16_own;
  }
  struct FreeX16 {  // on every way out
    void *p; hipStream_t s;
    ~FreeX16() { if (p) (void)hipFreeAsync(p, s); }
  } free_x16{x16_own, s};
  const int n16 = convert ? (int)((long long)T * H / 8) : 0;
  const int n_r = (int)(P / cap) + max_units;
  const int n_s = shared_ptr ? (T + cap_s - 1) / cap_s : 0;
  const int n_s2 = shared_ptr ? (T + cap_s2 - 1) / cap_s2 : 0;
  int *n_real = (int *)tiles_ws;  // [0] routed tiles in use, [1] shared tiles (w13 pass), [2] shared tiles (w2 pass)
  PfTile *tiles = (PfTile *)tiles_ws + 1, *sh_tiles = tiles + n_r, *sh_tiles2 = sh_tiles + n_s;
  hipLaunchKernelGGL(k_prefill_tiles, dim3(1 + (pub ? 1 : 0) + (n16 + 1023) / 1024), dim3(1024), 0, s, units, max_units,
                     (const unsigned long long *)expert_ptr, tiles, n_r, sh_tiles, n_s, sh_tiles2, n_s2,
                     (unsigned long long)(uintptr_t)shared_ptr, T, cap, cap_s, cap_s2, n_real, err, (const u32x4_t *)x_bf16,
                     (u32x4_t *)x16, n16, pub ? *pub : moe_publish{});
  if (int rc = moe_check_launch("k_prefill_tiles")) return rc;
  for (int w2 = 0; w2 < 2; ++w2) {
    if (!(phases & (w2 ? 2 : 1))) continue;
    PfArgs a;
    memset(&a, 0, sizeof a);
    // the shared expert (long K in the w2 pass, dense rows) goes first, the routed groups fill in behind it
    int n = 0;
    for (int shared = 1; shared >= 0; --shared) {
      if (shared && !shared_ptr) continue;
      PfClass &c = a.c[n++];
      const int Ii = shared ? I_sh : I;
      c.tiles = shared ? (w2 ? sh_tiles2 : sh_tiles) : tiles;
      c.n_mtiles = shared ? (w2 ? n_s2 : n_s) : n_r;
      c.n_tiles_real = n_real + (shared ? (w2 ? 2 : 1) : 0);
      c.shared = shared;
      if (!w2) {  // w13 [2I, H]: gate rows 0..I-1, up rows I..2I-1
        c.act = (const uint16_t *)(int4 ? x16 : x_bf16); c.gather = shared ? nullptr : sorted_tok; c.act_stride = H;
        c.out = shared ? h_s : h_r; c.out_stride = Ii;
        c.K = H; c.w_off = 0; c.half_delta = Ii; c.n_cols_per_tile = PF_BNH; c.n_ntiles = Ii / PF_BNH;
      } else {    // w2 [H, I] after w13 in the expert image
        c.act = (const uint16_t *)(shared ? h_s : h_r); c.gather = nullptr; c.act_stride = Ii;
        c.out = shared ? (void *)part_s : (void *)part_r; c.out_stride = H;
        c.K = Ii; c.w_off = (long long)2 * Ii * H * 2; c.half_delta = PF_BNH; c.n_cols_per_tile = 2 * PF_BNH;
        c.n_ntiles = H / (2 * PF_BNH);
      }
      if (int4) {
        moe_int4_layout lay;
        if (int rc = q4k ? moe_q4k_layout_make(H, Ii, &lay) : moe_int4_layout_make(H, Ii, &lay)) return rc;
        c.w_off = w2 ? lay.off2_q : lay.off13_q;
        c.off_s = w2 ? lay.off2_s : lay.off13_s;
        c.off_z = w2 ? lay.off2_z : lay.off13_z;
        if (!q4k && c.off_z - c.off_s >= (1ll << 31) - (1ll << 24)) {  // (pn_tile: the zeros are addressed from the scales)
          moe_set_error("moe_experts_prefill: the scales of an expert of %d x %d take 2 GiB or more", H, Ii);
          return MOE_EINVAL;
        }
      }
      c.ksplit = !w2 ? 1 : (shared ? shared_pieces : routed_pieces);
      c.split_stride = (shared ? (long long)T : P) * H;
      c.n_blocks = pf_padded(!int4, c.n_mtiles * c.n_ntiles * c.ksplit);
      c.slab_step = moe_bf16_slab_step(c.K / PF_BK);
      a.n_blocks_total += c.n_blocks;
    }
    if (int rc = q4k ? pn_launch<true>(!w2, a, s) : (int4 ? pn_launch<false>(!w2, a, s) : pf_launch(!w2, a, s))) return rc;
  }
  return MOE_OK;
}
