// int4-g128 experts of a prefill-sized batch on the scaled matrix instructions of gfx950 (included by moe_prefill.hip,
// whose tile list, block order and request helpers it uses).
//
// A nibble q = 0..15, zero-extended to six bits, IS the fp6 number q / 8 (e2m3: codes 0..7 are subnormal), so a weight
// needs no dequantisation: a lane's 32 nibbles become an operand of v_mfma_scale_f32_32x32x64_f8f6f4 by spreading four dwords
// over six (half an operation per weight).  The group's scale s multiplies the group's sum, one fma per output and
// group, and the zero points go in as one small product in front of the loop: sum_k s (q - z) x = s sum_k q x - (s z) X with
// X the sum of x over the group.  Weights and scales are thereby exact.
// Activations are split into two numbers of few bits with one power-of-two scale per 32 (the instruction's block scale):
//   x (w13 pass):  hi e4m3 + lo e3m2: the 8 significant bits of a bf16 are kept exactly down to 2^-5 of the block's largest
//                  value, below that to 2^-13 of it;
//   h (w2 pass):   hi e2m3 + lo e2m3 at 2^-5: 2^-11 of the block's largest value, and hi's product at twice the rate of fp8.
// Per 64 x 32 x 32 products: 96 (w13) and 64 (w2) matrix cycles, 128 as fp16; a loop of the products and folds alone reaches 2.24
// and 2.67 PFLOP/s of the product on this chip, the fp16 products alone 1.70 (all three at the power limit).
// Error against 64 bits (2-norm of the partial rows): 2048 x 1408 1.04e-3, 4096 x 4096 1.06e-3, where dequantising to fp16
// had 3.17e-3 and 3.18e-3 (the rounding of -(16 + z) s, common to the 128 weights of a group's row).
// Measured against that kernel (four waves, dequantisation between the products; w13 / w2 launch under the profiler, us):
// Mixtral shape 4096 tokens 1349 / 667 (1658 / 891), DeepSeek shape 2048 tokens 173 / 93 (200 / 114), 379 tokens 49 / 34
// (64 / 45).
// What bounds it (a build whose launches took 1437 / 710 and 182 / 102; Mixtral shape, then DeepSeek shape): without the requests in
// the loop 1142 / 562 and 148 / 81, without the folds 1331 / 686 and 172 / 99.  The Mixtral launches run at 1.74 GHz (power), the
// others at 2.0 to 2.2 with the matrix cores 41 and 23 % busy, two waves per SIMD that wait a sixth of the time for a group to
// arrive; the split of the h rows is 13 % of a DeepSeek w13 launch.
#pragma once

typedef int p6_i32x8_t __attribute__((ext_vector_type(8)));
typedef u32 p6_u32x2_t __attribute__((ext_vector_type(2)));
typedef u32 p6_u32x6_t __attribute__((ext_vector_type(6)));
typedef float p6_f32x2_t __attribute__((ext_vector_type(2)));
typedef float p6_f32x32_t __attribute__((ext_vector_type(32)));

// ---- split activation rows ------------------------------------------------------------------------
// Records of 256 bytes, one per (group of 128, row), group after group: record (g, row) at (g rows + row) * 256.  A matrix takes
// the room of 16-bit values, the rows of a tile lie on all memory channels (with the rows of a matrix one after the other
// every row of a tile began on the same channel: strides of 4 and 8 KiB), and gathered rows are whole cache lines.
// Record: two slabs of SLAB bytes (64 k each), the dword of the group's block scales, and from byte 240 on, in records of
// groups g % 4 = 0, the sums of the row's groups g .. g + 3 (two bf16 each: the sum and what rounding it left).
// Slab: pieces of 16 bytes that lane half h of an operand reads:
//   W13 (112 bytes): 0, 16 hi fields 0..15 and 16..31 of block 0 | 32, 48 the same of block 1 | 64 + 16 h lo dwords 0..3 of
//                    block h | 96 + 8 h lo dwords 4, 5 of block h
//     (the fp8 operand's lane half h takes the k slots 16 h + 0..15 and 32 + 16 h + 0..15, the 6-bit ones 32 h + 0..31)
//   W2 (96 bytes):   16 h hi dwords 0..3 of block h | 32 + 16 h lo dwords 0..3 | 64 + 8 h hi dwords 4, 5 | 80 + 8 h lo dwords 4, 5
// Scale dword: bytes of blocks 0, 2, 1, 3, so that lane half h reads those of the group's two slabs side by side.
#define P6_REC 256
#define P6_SUMS 240
template <bool W13> struct P6Row {
  static constexpr int SLAB = W13 ? 112 : 96, SCALES = 2 * SLAB, UNITS = SCALES / 16 + 1;   // 16-byte units that the kernel reads
};
#define P6_SCALE_Q 130          // block scale of the weights: 2^3 (the codes are q / 8)
#define P6_LO_X (P6_SCALE_Q - 1)  // of lo of x (stored in units of half hi's scale)
#define P6_LO_H (P6_SCALE_Q - 5)  // of lo of h

// order of the k of 16 in the operands: field f holds k = p6_k(f) (what p6_spread below makes of the nibble order)
static __host__ __device__ constexpr int p6_k16(int f) {
  constexpr int t[16] = {0, 2, 6, 1, 5, 7, 10, 12, 9, 11, 15, 8, 4, 14, 3, 13};
  return t[f];
}
static __host__ __device__ constexpr int p6_k(int f) { return (f & 16) | p6_k16(f & 15); }

// 16 nibbles in the image's order (a, b: one 8-byte piece of a tile) -> 16 six-bit fields (three dwords)
static __device__ __forceinline__ void p6_spread(u32 a, u32 b, int &d0, int &d1, int &d2) {
  const u32 a2 = a << 2;                                        // nibbles at 4, 16 -> 6, 18; the top one's low half -> 30
  const u32 b2 = __builtin_amdgcn_alignbit(b, a, 30);           // b << 2, and the top nibble's high half of a -> 0
  d0 = (int)((a & 0x0f00f00fu) | (a2 & 0xc03c03c0u));
  d1 = (int)((b & 0xf00f00f0u) | (b2 & 0x03c03c03u));
  d2 = (int)((a & 0x00f00f00u) | (b2 & 0x3c03c03cu));
}

// biased exponent of a block scale from the largest magnitude's bits; hi's largest binade is 2^TOP, both scales stay normal
template <int TOP> static __device__ __forceinline__ int p6_scale_of(u32 amax, bool round_up) {
  const int e = (int)(amax >> 23) - TOP + (round_up ? 1 : 0);
  return e < 8 ? 8 : e;
}
// the sum of a group as two bf16 (sum in the low half); a block with an infinity or a NaN makes it NaN, which makes every
// output of that row NaN through the zero-point product
static __device__ __forceinline__ u32 p6_sum_pair(float s) {
  const u32 hi = f32_to_bf16(s);
  const float left = s - __uint_as_float(hi << 16);
  const u32 v = hi | ((u32)f32_to_bf16(left) << 16);
  return s - s == 0.f ? v : 0x7fc07fc0u;
}

// One block of 32 values v (in k order): operands of x.  Returns the scale byte, sum = the sum of what hi and lo hold.
static __device__ __forceinline__ int p6_split_x(const float (&v)[32], u32 (&hi)[8], u32 (&lo)[6], float &sum) {
  u32 am = 0;
#pragma unroll
  for (int k = 0; k < 32; ++k) am = max(am, __float_as_uint(v[k]) & 0x7fffffffu);
  const int e = p6_scale_of<7>(am, false);
  const float s = __uint_as_float((u32)e << 23), s2 = __uint_as_float((u32)(e - 1) << 23);
  typedef short v2s __attribute__((ext_vector_type(2)));
  f32x16_t r0, r1;
  float t = 0.f;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    v2s o = {0, 0};
    o = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(o, v[p6_k(4 * d)], v[p6_k(4 * d + 1)], s, false);
    o = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(o, v[p6_k(4 * d + 2)], v[p6_k(4 * d + 3)], s, true);
    hi[d] = __builtin_bit_cast(u32, o);
    const p6_f32x2_t a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi[d], s, false);
    const p6_f32x2_t b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi[d], s, true);
    r0[2 * d] = v[p6_k(4 * d)] - a.x;          // fields 2 j and 2 j + 1 of the 6-bit conversion come from its two sources
    r1[2 * d] = v[p6_k(4 * d + 1)] - a.y;
    r0[2 * d + 1] = v[p6_k(4 * d + 2)] - b.x;
    r1[2 * d + 1] = v[p6_k(4 * d + 3)] - b.y;
    t += (a.x + a.y) + (b.x + b.y);
  }
  const p6_u32x6_t l = __builtin_bit_cast(p6_u32x6_t, __builtin_amdgcn_cvt_scalef32_2xpk16_bf6_f32(r0, r1, s2));
  const p6_f32x32_t q = __builtin_amdgcn_cvt_scalef32_pk32_f32_bf6(l, s2);
#pragma unroll
  for (int d = 0; d < 6; ++d) lo[d] = l[d];
  float u = 0.f;
#pragma unroll
  for (int k = 0; k < 32; ++k) u += q[k];
  sum = (am >> 23) == 255u ? __uint_as_float(0x7fc00000u) : t + u;
  return e;
}
// The same of h: hi's grid ends at 7.5, so a block whose largest value would round past it moves up by one binade.
static __device__ __forceinline__ int p6_split_h(const float (&v)[32], u32 (&hi)[6], u32 (&lo)[6], float &sum) {
  u32 am = 0;
#pragma unroll
  for (int k = 0; k < 32; ++k) am = max(am, __float_as_uint(v[k]) & 0x7fffffffu);
  const int e = p6_scale_of<2>(am, (am & 0x7fffffu) >= 0x780000u);   // 7.75
  const float s = __uint_as_float((u32)min(e, 254) << 23), s2 = __uint_as_float((u32)(min(e, 254) - 5) << 23);
  f32x16_t a, b;
#pragma unroll
  for (int j = 0; j < 16; ++j) { a[j] = v[p6_k(2 * j)]; b[j] = v[p6_k(2 * j + 1)]; }
  const p6_u32x6_t p = __builtin_bit_cast(p6_u32x6_t, __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(a, b, s));
  const p6_f32x32_t q = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(p, s);
  float t = 0.f;
#pragma unroll
  for (int j = 0; j < 16; ++j) { t += q[2 * j] + q[2 * j + 1]; a[j] -= q[2 * j]; b[j] -= q[2 * j + 1]; }
  const p6_u32x6_t l = __builtin_bit_cast(p6_u32x6_t, __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(a, b, s2));
  const p6_f32x32_t ql = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(l, s2);
#pragma unroll
  for (int d = 0; d < 6; ++d) { hi[d] = p[d]; lo[d] = l[d]; }
  float u = 0.f;
#pragma unroll
  for (int j = 0; j < 32; ++j) u += ql[j];
  sum = (am >> 23) == 255u ? __uint_as_float(0x7fc00000u) : t + u;
  return e;
}

// x [rows, K] bf16 -> records, one thread per block of 32 (four consecutive threads a group)
static __device__ __forceinline__ void p6_convert_x(const u32x4_t *__restrict__ x, unsigned char *__restrict__ out, int K, int rows, int i) {
  const int per = K / 32;
  const bool on = i < rows * per;
  const int ii = on ? i : 0, row = ii / per, b = ii - row * per;
  float v[32];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const u32x4_t d = x[(size_t)ii * 4 + c];
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[8 * c + 2 * j] = bf16lo(d[j]); v[8 * c + 2 * j + 1] = bf16hi(d[j]); }
  }
  u32 hi[8], lo[6];
  float sum;
  const int e = p6_split_x(v, hi, lo, sum);
  sum += __shfl_xor(sum, 1);
  sum += __shfl_xor(sum, 2);
  u32 sc = (u32)e << (8 * (((b & 1) << 1) | ((b >> 1) & 1)));
  sc |= __shfl_xor(sc, 1);
  sc |= __shfl_xor(sc, 2);
  if (!on) return;
  const int g = b >> 2, h = b & 1;
  unsigned char *r = out + ((size_t)g * rows + row) * P6_REC, *sl = r + ((b >> 1) & 1) * P6Row<true>::SLAB;
  *(u32x4_t *)(sl + 32 * h) = u32x4_t{hi[0], hi[1], hi[2], hi[3]};
  *(u32x4_t *)(sl + 32 * h + 16) = u32x4_t{hi[4], hi[5], hi[6], hi[7]};
  *(u32x4_t *)(sl + 64 + 16 * h) = u32x4_t{lo[0], lo[1], lo[2], lo[3]};
  *(p6_u32x2_t *)(sl + 96 + 8 * h) = p6_u32x2_t{lo[4], lo[5]};
  if ((b & 3) == 0) {
    *(u32 *)(r + P6Row<true>::SCALES) = sc;
    *(u32 *)(out + ((size_t)(g & ~3) * rows + row) * P6_REC + P6_SUMS + 4 * (g & 3)) = p6_sum_pair(sum);
  }
}

// ---- the tile kernel ------------------------------------------------------------------------------------
// Four waves, two workgroups per compute unit, tiles of up to 128 rows x (128 + 128) columns as k_prefill_nib: wave w owns 32
// columns of both halves and ALL NB row blocks.  K advances a quantisation group (128) at a time: the two 64-wide slabs
// of a row block go through the matrix cores into 2 x 16 registers, which the group's scales fold into the
// accumulators.  From memory everything goes global -> LDS directly: the group's activation pieces and block scales into
// RA slots that the workgroup shares (one barrier per group), and, private to each wave, its four nibble tiles and
// scales into RW slots; a wave has spread its nibbles over the operands by the end of the group's first row block and
// requests the next ones into the same slot.
template <int NB, bool W13> struct P6Lds {
  static constexpr int U = P6Row<W13>::UNITS, ROW = U * 16;   // (an odd number of pieces: 16 rows on 16 bank groups)
  static constexpr int A = NB * 32 * ROW;
  static constexpr int W = 4 * 4096, S = 4 * 256;             // nibbles, scales of the four waves
  static constexpr int RA = NB == 1 ? 3 : 2;
  static constexpr int RW = NB == 1 ? 3 : (NB == 2 ? (W13 ? 2 : 3) : (NB == 3 ? 2 : 1));
  static constexpr int W0 = RA * A, S0 = W0 + RW * W, BYTES = S0 + RW * S;
  static constexpr int PER_WAVE = 8 * NB * U;                 // 16-byte units of a group that a wave requests
  static constexpr int Q = (PER_WAVE + 63) / 64;              // requests for them; the last one in LAST lanes
  static constexpr int LAST = PER_WAVE - 64 * (Q - 1);
  static constexpr int NA = Q, NW = 5;                // requests of a group
  // newest requests that may still be on their way when group g is needed: those behind its activations (the nibbles requested
  // in the same iteration, then whole iterations) and those behind its nibbles
  static constexpr bool W_FIRST = RW == 1;                    // order of an iteration's requests
  static constexpr int PEND_A = (W_FIRST ? 0 : NW) + (RA - 2) * (NA + NW), PEND_W = (W_FIRST ? NA : 0) + (RW - 1) * (NA + NW);
  static constexpr int PEND = PEND_A < PEND_W ? PEND_A : PEND_W;
  static_assert(BYTES <= PN_LDS && PEND < 63, "LDS, counter");
};

static __device__ __forceinline__ void p6_dma16(unsigned lds, int voff, const pf_i32x4_t r, int soff, unsigned long long lanes) {
  __asm__ volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\ts_mov_b64 exec, -1"
                   :: "s"(lds), "v"(voff), "s"(r), "s"(soff), "s"(lanes) : "memory", "m0");
}
static __device__ __forceinline__ void p6_dma4(unsigned lds, int voff, const pf_i32x4_t r, int soff, unsigned long long lanes) {
  __asm__ volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %4\n\tbuffer_load_dword %1, %2, %3 offen lds\n\ts_mov_b64 exec, -1"
                   :: "s"(lds), "v"(voff), "s"(r), "s"(soff), "s"(lanes) : "memory", "m0");
}
template <int N> static constexpr unsigned long long P6_LANES = N >= 64 ? ~0ull : (1ull << (N & 63)) - 1;

template <int NB, bool SWIGLU>
static __device__ __forceinline__ void p6_tile(const PfClass &c, const PfTile &tile, unsigned char *lds, int nt, int g0, int ng,
                                               int split, int tid) {
  constexpr bool W13 = SWIGLU;
  typedef P6Lds<NB, W13> M;
  typedef P6Row<W13> R;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5, r16 = n & 15;
  const int K = c.K, G = K >> 7, rows = pf_rows(tile);
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
  const pf_i32x4_t ra = pn_rsrc(c.act);
  const size_t tile0 = (size_t)16 * nt * G;   // (row block, group) pairs in front of the tile's
  const pf_i32x4_t rw = pn_rsrc((const void *)(tile.w_base + c.w_off + tile0 * 1024));
  const pf_i32x4_t rs = pn_rsrc((const void *)(tile.w_base + c.off_s + tile0 * 32));
  // row block t = 2 f + (n / 16) of this wave in the tile, as in pn_tile
  auto rb = [&](int t) { return SWIGLU ? 4 * w + (t >> 1) + 2 * (t & 1) : 2 * w + 8 * (t >> 1) + (t & 1); };
  auto act_row = [&](int r) {                 // byte offset of row r's record of group 0 (rows past the end: row 0, never stored)
    const int grow = tile.row0 + (r < rows ? r : 0);
    return (c.gather ? c.gather[grow] : grow) * P6_REC;
  };
  const int g_step = c.act_rows * P6_REC;     // from a record to the next group's
  const int w_voff = lane * 16;
  const int s_voff = rb(n >> 3) * G * 32 + (n & 7) * 4;
  // request t of a group's nibbles (t = 4: the scales); past the end: the last group again, into a slot that nobody reads
  auto req_w = [&](int t, int g_, int slot) {
    const int g = g0 + (g_ < ng ? g_ : ng - 1);
    if (t < 4) p6_dma16(lds0 + (unsigned)(M::W0 + slot * M::W + w * 4096 + t * 1024), w_voff, rw, (rb(t) * G + g) * 1024, ~0ull);
    else p6_dma4(lds0 + (unsigned)(M::S0 + slot * M::S + w * 256), s_voff, rs, g * 32, P6_LANES<32>);
  };
  int a_voff[M::Q];                           // unit u = row u / U, piece u % U
#pragma unroll
  for (int q = 0; q < M::Q; ++q) {
    const int u = M::PER_WAVE * w + 64 * q + lane, r = u / M::U;
    a_voff[q] = act_row(r) + (u - r * M::U) * 16;
  }
  // zero points (below): CH groups' sums a time, request rq of this wave = 64 (quad, row) pairs
  constexpr int CH = NB >= 3 ? 16 : 8, CQ = CH / 4, XR = (CQ * NB + 7) / 8;
  int x_voff[XR];
#pragma unroll
  for (int rq = 0; rq < XR; ++rq) x_voff[rq] = act_row((64 * (4 * rq + w) + lane) % (32 * NB)) + P6_SUMS;
  // (the rows' loads are waited for here: behind a request in assembly their wait would be for that one too)
#pragma unroll
  for (int q = 0; q < M::Q; ++q) __asm__ volatile("" : "+v"(a_voff[q]));
#pragma unroll
  for (int rq = 0; rq < XR; ++rq) __asm__ volatile("" : "+v"(x_voff[rq]));
  // request q of a group's activations
  auto req_a = [&](int q, int g_, int slot) {
    const int g = g0 + (g_ < ng ? g_ : ng - 1);
    p6_dma16(lds0 + (unsigned)(slot * M::A + (M::PER_WAVE * w + 64 * q) * 16), a_voff[q], ra, g * g_step,
             q + 1 < M::Q ? ~0ull : P6_LANES<M::LAST>);
  };
  // a chunk of the zero points' operands, into the slot of the activations' ring that is filled last
  constexpr int X0 = (M::RA - 1) * M::A, ZS = X0 + CQ * 32 * NB * 16, ZZ = ZS + 4 * 4 * CH * 32;
  static_assert(ZZ + 4 * 4 * CH * 8 <= X0 + M::A, "the slot holds a chunk");
  const int z0 = (int)(c.off_z - c.off_s - (long long)tile0 * 24);   // from the tile's scales to its zeros (launcher: below 2 GiB)
  const int q_last = (g0 + ng - 1) >> 2;
  auto req_zero = [&](int q0) {
#pragma unroll
    for (int rq = 0; rq < XR; ++rq) {     // 64 rows' sums of four groups
      const int req = 4 * rq + w;
      if (req < CQ * NB / 2) {
        const int q = (64 * req + lane) / (32 * NB);
        p6_dma16(lds0 + (unsigned)(X0 + 1024 * req), x_voff[rq] + 4 * min(q0 + q, q_last) * g_step, ra, 0, ~0ull);
      }
    }
#pragma unroll
    for (int rq = 0; rq < CH / 8; ++rq) {  // scales: 2 CH pieces of 16 bytes per row block; zeros: 2 CH dwords
      const int u = 64 * rq + lane, t = u / (2 * CH), v = u - t * 2 * CH;
      const int b = rb(t) * G + min(4 * q0 + (v >> 1), G - 1);
      p6_dma16(lds0 + (unsigned)(ZS + w * 4 * CH * 32 + 1024 * rq), b * 32 + (v & 1) * 16, rs, 0, ~0ull);
      p6_dma4(lds0 + (unsigned)(ZZ + w * 4 * CH * 8 + 256 * rq), z0 + b * 8 + (v & 1) * 4, rs, 0, ~0ull);
    }
  };
  // what the zero points and group 0 need, then the groups behind it
  req_zero(g0 >> 2);
#pragma unroll
  for (int q = 0; q < M::NA; ++q) req_a(q, 0, 0);
#pragma unroll
  for (int t = 0; t < M::NW; ++t) req_w(t, 0, 0);
#pragma unroll
  for (int g = 1; g < M::RA - 1; ++g)
#pragma unroll
    for (int q = 0; q < M::NA; ++q) req_a(q, g, g);
#pragma unroll
  for (int g = 1; g < M::RW; ++g)
#pragma unroll
    for (int t = 0; t < M::NW; ++t) req_w(t, g, g);
  f32x16_t acc[NB][2];
  // zero points: acc = - sum_g (s z) X as products of the two bf16 pieces of either, four groups an instruction (lane
  // half h: groups 4 p + 2 h, + 1).  Sums, scales and zeros of CH groups come together, through LDS, in front of group 0, which
  // is on its way meanwhile.  (Loaded by every wave into registers, the sums four times and behind the first groups' requests, this
  // took 17 of 178 us of the w13 launch of the DeepSeek shape at 2048 tokens and 12 of 99 of the w2 launch: now 173 and 93.5;
  // Mixtral shape 4096 tokens 1395 / 690 -> 1349 / 667, 379 tokens 51.5 / 35.5 -> 49.4 / 34.1.)
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][f][e] = 0.f;
  {
    const unsigned xr = lds0 + (unsigned)(X0 + n * 16 + 8 * h);
    const unsigned sr = lds0 + (unsigned)(ZS + (w * 4 + (n >> 4)) * CH * 32 + 64 * h + r16 * 2);
    const unsigned zr = lds0 + (unsigned)(ZZ + (w * 4 + (n >> 4)) * CH * 8 + 16 * h + (r16 >> 1));
    const int zsh = 4 * (r16 & 1);
    for (int q0 = g0 >> 2; q0 <= q_last; q0 += CQ) {
      if (q0 > g0 >> 2) {
        __syncthreads();     // the chunk before has been read
        req_zero(q0);
        PF_VMCNT(0);
      } else PF_VMCNT((M::RA - 1) * M::NA + M::RW * M::NW);   // all but the groups' requests behind it
      __syncthreads();
#pragma unroll
      for (int q = 0; q < CQ; ++q) {
        if (q0 + q > q_last) break;
        u32x4_t xa[NB], wb[2];
        bool on[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int g = 4 * (q0 + q) + 2 * h + j;
          on[j] = g >= g0 && g < g0 + ng;    // (groups past the end have no sum)
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            const float sc = half_bits_to_f32(pn_lds<uint16_t>(sr + (unsigned)(2 * f * CH * 32 + 128 * q + 32 * j)));
            const u32 z = (pn_lds<unsigned char>(zr + (unsigned)(2 * f * CH * 8 + 32 * q + 8 * j)) >> zsh) & 15u;
            const float v = on[j] ? -sc * (float)z : 0.f;   // 15 significant bits: its upper half and what that leaves are bf16
            const u32 v1 = __float_as_uint(v), v2 = __float_as_uint(v - __uint_as_float(v1 & 0xffff0000u));
            wb[f][2 * j] = __builtin_amdgcn_perm(v1, v1, 0x03020302u);
            wb[f][2 * j + 1] = __builtin_amdgcn_perm(v2, v2, 0x03020302u);
          }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const p6_u32x2_t xv = pn_lds<p6_u32x2_t>(xr + (unsigned)((q * 32 * NB + 32 * i) * 16));
          const u32 x0 = on[0] ? xv.x : 0u, x1 = on[1] ? xv.y : 0u;
          xa[i] = u32x4_t{x0, x0, x1, x1};
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int f = 0; f < 2; ++f)
            acc[i][f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, xa[i]), __builtin_bit_cast(bf16x8_t, wb[f]),
                                                                acc[i][f], 0, 0, 0);
      }
    }
  }
  PF_VMCNT((M::RA - 2) * M::NA + (M::RW - 1) * M::NW);   // group 0 is there (the loop's first barrier follows)
  // LDS addresses: the lane's pieces of a slab's row, its block scales, its nibbles and scales
  const unsigned fa = lds0 + (unsigned)(n * M::ROW + 16 * h), fb = lds0 + (unsigned)(n * M::ROW + (W13 ? 96 : 64) + 8 * h);
  const unsigned fs = lds0 + (unsigned)(n * M::ROW + R::SCALES + 2 * h);
  const unsigned nw = lds0 + (unsigned)(M::W0 + w * 4096 + (n >> 4) * 1024 + (16 * h + r16) * 16);
  const unsigned sw = lds0 + (unsigned)(M::S0 + w * 256 + (n >> 4) * 32 + r16 * 2);
  struct Frag { u32x4_t hi0, hi1, lo0; p6_u32x2_t hi2, lo1; };
  auto read_frag = [&](int so, int i, int s) {
    Frag f;
    const unsigned o = (unsigned)(so + s * R::SLAB + i * 32 * M::ROW);
    f.hi0 = pn_lds<u32x4_t>(fa + o);
    if (W13) {
      f.hi1 = pn_lds<u32x4_t>(fa + o + 32u);
      f.lo0 = pn_lds<u32x4_t>(fa + o + 64u);
      f.lo1 = pn_lds<p6_u32x2_t>(fb + o);
    } else {
      f.hi2 = pn_lds<p6_u32x2_t>(fb + o);
      f.lo0 = pn_lds<u32x4_t>(fa + o + 32u);
      f.lo1 = pn_lds<p6_u32x2_t>(fb + o + 16u);
    }
    return f;
  };
  auto hi_of = [&](const Frag &f) {
    if (W13) return p6_i32x8_t{(int)f.hi0.x, (int)f.hi0.y, (int)f.hi0.z, (int)f.hi0.w, (int)f.hi1.x, (int)f.hi1.y, (int)f.hi1.z, (int)f.hi1.w};
    return p6_i32x8_t{(int)f.hi0.x, (int)f.hi0.y, (int)f.hi0.z, (int)f.hi0.w, (int)f.hi2.x, (int)f.hi2.y, 0, 0};
  };
  auto lo_of = [&](const Frag &f) { return p6_i32x8_t{(int)f.lo0.x, (int)f.lo0.y, (int)f.lo0.z, (int)f.lo0.w, (int)f.lo1.x, (int)f.lo1.y, 0, 0}; };
  constexpr int FH = W13 ? 0 : 2, FL = W13 ? 3 : 2;    // operand formats: e4m3, e2m3, e3m2
  const int q_hi = P6_SCALE_Q, q_lo = W13 ? P6_LO_X : P6_LO_H;
  int sa = 0, sn = (M::RA - 1) % M::RA, sb = 0;        // slots of group g, of g + RA - 1, of the nibbles
  // Order of a group: for every row block the four products of half 0 (hi and lo of both slabs, one chain), then those of half
  // 1.  A chain's sum is folded into its accumulators behind the products of the next chain, the last one's of a group behind
  // the first of the next group; a slab's fragment is read anew as soon as half 1 has used it.
  f32x16_t d[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) d[1][e] = 0.f;
  float s[2] = {0.f, 0.f};
  for (int g = 0; g < ng; ++g) {
    PF_VMCNT(M::PEND);
    __syncthreads();
    const int so = sa * M::A;
    const float s_old = s[1];
    u32 raw_s[2], bs[NB];
    u32x4_t raw[2][2];                                 // [slab][half]
    p6_i32x8_t code[2][2];
    Frag fr[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) raw[t][0] = pn_lds<u32x4_t>(nw + (unsigned)(sb * M::W + t * 512));
    bs[0] = pn_lds<uint16_t>(fs + (unsigned)so);
    fr[0] = read_frag(so, 0, 0);
    fr[1] = read_frag(so, 0, 1);
#pragma unroll
    for (int t = 0; t < 2; ++t) raw[t][1] = pn_lds<u32x4_t>(nw + (unsigned)(sb * M::W + 2048 + t * 512));
#pragma unroll
    for (int f = 0; f < 2; ++f) raw_s[f] = pn_lds<uint16_t>(sw + (unsigned)(sb * M::S + 64 * f));
#pragma unroll
    for (int i = 1; i < NB; ++i) bs[i] = pn_lds<uint16_t>(fs + (unsigned)(so + i * 32 * M::ROW));
    __builtin_amdgcn_sched_barrier(0);
    auto spread = [&](int t, int f) {
      const u32x4_t v = raw[t][f];
      int k0, k1, k2, k3, k4, k5;
      p6_spread(v.x, v.y, k0, k1, k2);
      p6_spread(v.z, v.w, k3, k4, k5);
      code[t][f] = p6_i32x8_t{k0, k1, k2, k3, k4, k5, 0, 0};
    };
    spread(0, 0);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        auto fold = [&](int e0) {                      // four sums of the chain before this one
          const int pi = f ? i : (i ? i - 1 : NB - 1);
          const float ps = f ? s[0] : (i ? s[1] : s_old);
#pragma unroll
          for (int e = e0; e < e0 + 4; ++e) acc[pi][f ^ 1][e] = __builtin_fmaf(d[f ^ 1][e], ps, acc[pi][f ^ 1][e]);
        };
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          f32x16_t z;
#pragma unroll
          for (int e = 0; e < 16; ++e) z[e] = 0.f;
          d[f] = t == 0 ? __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(hi_of(fr[t]), code[t][f], z, FH, 2, 0, (int)bs[i], 0, q_hi)
                        : __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(hi_of(fr[t]), code[t][f], d[f], FH, 2, 1, (int)bs[i], 0, q_hi);
          __builtin_amdgcn_sched_barrier(0);
          if (i == 0 && f == 0) spread(t == 0 ? 1 : 0, t == 0 ? 0 : 1);
          fold(8 * t);
          __builtin_amdgcn_sched_barrier(0);
          d[f] = t == 0 ? __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(lo_of(fr[t]), code[t][f], d[f], FL, 2, 0, (int)bs[i], 0, q_lo)
                        : __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(lo_of(fr[t]), code[t][f], d[f], FL, 2, 1, (int)bs[i], 0, q_lo);
          __builtin_amdgcn_sched_barrier(0);
          if (i == 0 && f == 0 && t == 1) spread(1, 1);
          fold(8 * t + 4);
          if (f == 1 && i + 1 < NB) fr[t] = read_frag(so, i + 1, t);
          if (i == 0 && f == 0 && t == 1) {
#pragma unroll
            for (int k = 0; k < 2; ++k) { s[k] = half_bits_to_f32((uint16_t)raw_s[k]); __asm__ volatile("" : "+v"(s[k])); }
          }
          // the requests, spread over the products behind the first chain (by then the nibbles and scales have been read: the
          // codes are made)
          constexpr int SLOTS = NB > 1 ? 2 * NB - 1 : 2, NR = M::NA + M::NW;
          const int slot = 2 * (2 * i + f - 1) + t;
          if (slot >= 0) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < NR; ++q)
              if (q * SLOTS / NR == slot) {
                const int qa = M::W_FIRST ? q - M::NW : q, qw = M::W_FIRST ? q : q - M::NA;
                if (qa >= 0 && qa < M::NA) req_a(qa, g + M::RA - 1, sn);
                if (qw >= 0 && qw < M::NW) req_w(qw, g + M::RW, sb);
              }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    sa = sa + 1 == M::RA ? 0 : sa + 1;
    sn = sn + 1 == M::RA ? 0 : sn + 1;
    sb = sb + 1 == M::RW ? 0 : sb + 1;
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[NB - 1][1][e] = __builtin_fmaf(d[1][e], s[1], acc[NB - 1][1][e]);
  PF_VMCNT(0);   // the transfers past the end have landed: the slots are free, and nothing is in flight at the end
  // acc element e of lane l: row 8*(e/4) + 4*(l/32) + e%4 of its block, column l%32
  if constexpr (SWIGLU) {
    // A wave's 32 columns of h are one block of every row's group nt: through LDS a lane gets a row's 32 values.
    constexpr int HS = 36;                             // floats per row: 16-byte pieces on different banks
    static_assert(4 * 32 * NB * HS * 4 + 2 * 512 * NB <= PN_LDS, "the h tile fits");
    __syncthreads();
    float *hs = (float *)lds + w * (32 * NB * HS);
    u32 *xsum = (u32 *)(lds + 4 * 32 * NB * HS * 4), *xsc = xsum + 128 * NB;   // [wave][row]
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        hs[(32 * i + 8 * (e >> 2) + 4 * h + (e & 3)) * HS + n] = pf_silu_mul(acc[i][0][e], acc[i][1][e]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    unsigned char *out = (unsigned char *)c.out + ((size_t)nt * c.out_rows + tile.row0) * P6_REC;
#pragma unroll
    for (int p = 0; p < (NB + 1) / 2; ++p) {
      const int r = 64 * p + lane;
      if (r < 32 * NB) {
        float v[32];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float4 q = *(const float4 *)(hs + r * HS + 4 * j);
          v[4 * j] = q.x; v[4 * j + 1] = q.y; v[4 * j + 2] = q.z; v[4 * j + 3] = q.w;
        }
        u32 hi[6], lo[6];
        float sum;
        const int e = p6_split_h(v, hi, lo, sum);
        xsum[w * 32 * NB + r] = __float_as_uint(sum);
        xsc[w * 32 * NB + r] = (u32)e;
        if (r < rows) {
          unsigned char *sl = out + r * P6_REC + (w >> 1) * P6Row<false>::SLAB;
          const int k = w & 1;
          *(u32x4_t *)(sl + 16 * k) = u32x4_t{hi[0], hi[1], hi[2], hi[3]};
          *(u32x4_t *)(sl + 32 + 16 * k) = u32x4_t{lo[0], lo[1], lo[2], lo[3]};
          *(p6_u32x2_t *)(sl + 64 + 8 * k) = p6_u32x2_t{hi[4], hi[5]};
          *(p6_u32x2_t *)(sl + 80 + 8 * k) = p6_u32x2_t{lo[4], lo[5]};
        }
      }
    }
    __syncthreads();
    if (tid < rows) {
      u32 e[4];
      float sum = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        e[k] = xsc[k * 32 * NB + tid];
        sum += __uint_as_float(xsum[k * 32 * NB + tid]);
      }
      *(u32 *)(out + tid * P6_REC + P6Row<false>::SCALES) = e[0] | (e[2] << 8) | (e[1] << 16) | (e[3] << 24);
      *(u32 *)((unsigned char *)c.out + ((size_t)(nt & ~3) * c.out_rows + tile.row0 + tid) * P6_REC + P6_SUMS + 4 * (nt & 3)) = p6_sum_pair(sum);
    }
  } else {
    const int col = 32 * w + n;
    float *out = (float *)c.out + (size_t)split * c.split_stride + nt * 2 * PF_BNH + col;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
        if (row < rows) {
          float *o = out + (size_t)(tile.row0 + row) * c.out_stride;
          o[0] = acc[i][0][e];
          o[PF_BNH] = acc[i][1][e];
        }
      }
  }
}

template <bool SWIGLU>
__global__ __launch_bounds__(256, 2) void k_prefill_int4(const PfArgs a) {
  extern __shared__ __align__(16) unsigned char lds_6[];
  const int tid = threadIdx.x;
  int ci, mt, nt, split;
  if (!pf_block_of<false>(a, ci, mt, nt, split)) return;
  const PfClass &c = a.c[ci];
  const PfTile tile = c.tiles[mt];
  const int rows = pf_rows(tile);
  if (rows <= 0) return;
  const int ks = c.ksplit > 1 ? c.ksplit : 1;
  const int ng = SWIGLU ? c.K >> 7 : (c.K >> 7) / ks, g0 = SWIGLU ? 0 : split * ng;   // this workgroup's window of groups
  switch ((rows + 31) >> 5) {
    case 1: p6_tile<1, SWIGLU>(c, tile, lds_6, nt, g0, ng, split, tid); break;
    case 2: p6_tile<2, SWIGLU>(c, tile, lds_6, nt, g0, ng, split, tid); break;
    case 3: p6_tile<3, SWIGLU>(c, tile, lds_6, nt, g0, ng, split, tid); break;
    default: p6_tile<4, SWIGLU>(c, tile, lds_6, nt, g0, ng, split, tid); break;
  }
}
