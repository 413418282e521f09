// Shared host-side helpers of the library (error string, launch check).
#pragma once
#include <hip/hip_runtime.h>

#include "moe_kernels.h"

void moe_set_error(const char *fmt, ...) __attribute__((format(printf, 1, 2)));
int moe_check_launch(const char *what);
int moe_check_hip(hipError_t e, const char *what);

// Optional per-kernel timing with HIP events on the launch stream (moe_kernel_timing*).
enum MoeKernelId { MOE_K_GATE = 0, MOE_K_TOPK, MOE_K_DISPATCH, MOE_K_W13, MOE_K_W2, MOE_K_COMBINE,
                   MOE_K_PREFILL_W13, MOE_K_PREFILL_W2, MOE_K_COUNT };
void moe_ktimer_begin(int kid, hipStream_t s);
void moe_ktimer_end(int kid, hipStream_t s);

// A kernel met a selected expert whose slot-table entry is 0: it skips the unit and raises the caller's
// error word.  A system-scope store (every raiser writes the same value), so the word may live in device
// memory or in pinned host memory that the host polls without a copy.
static __device__ __forceinline__ void moe_raise_err(int *err) {
  __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// what the entry points that publish a unit list ask of their descriptor
static inline bool moe_publish_ok(const moe_publish *p, int max_units) {
  return p->n_active && p->units_host && p->n_active_host && p->seq_host && p->max_units > 0 && p->max_units <= max_units;
}

// Sizes past the expert kernels' 32-bit offsets: activation buffers of 2 GiB (x, h, of the routed pairs and of the shared
// expert), rows of 2^24 columns (bf16: 2^23: offsets inside a 128-row group of a bf16 matrix, 256 bytes per column, and inside 16
// row blocks of nibbles, 128).  I_sh: 0 without a shared expert.  An error, set, or MOE_OK.
static inline int moe_check_expert_sizes(const char *who, bool nibbles, int T, int k, int H, int I, int I_sh) {
  const long long widest = I > H ? I : H, rows = (long long)T * (k > 1 ? k : 1);
  if (rows * widest * 2 >= (1ll << 31) || (I_sh > 0 && (long long)T * (I_sh > H ? I_sh : H) * 2 >= (1ll << 31))) {
    moe_set_error("%s: activation buffers of 2 GiB or more are not supported (T=%d k=%d)", who, T, k);
    return MOE_EINVAL;
  }
  const int most = nibbles ? 1 << 24 : 1 << 23;
  if (H >= most || I >= most || I_sh >= most) {
    moe_set_error("%s: rows of %d columns and more are not supported (H=%d I=%d I_sh=%d)", who, most, H, I, I_sh);
    return MOE_EINVAL;
  }
  return MOE_OK;
}

// Storage rotation of a bf16 matrix per 128-row group of nk slabs: smallest odd s >= 3 coprime with nk (the slot layout)
static inline int moe_bf16_slab_step(int nk) {
  for (int s = 3;; s += 2) {
    int a = s, b = nk;
    while (b) { const int r = a % b; a = b; b = r; }
    if (a == 1) return s;
  }
}

// bf16 expert product of a decode batch (moe_decode_bf16.hip), behind moe_experts_prefill for batches it takes
bool moe_decode_bf16_takes(int T);
int moe_decode_bf16_splits(int H, int I_sh);
int moe_decode_bf16(const void *x, int T, int H, int I, int I_sh, const moe_unit *units, int max_units, const int *sorted_tok,
                    const uint64_t *expert_ptr, const void *shared_ptr, void *h_r, void *h_s, float *part_r, float *part_s,
                    int pieces, int *err, int phases, const moe_publish *pub, hipStream_t s);

// gate logits on the matrix cores (moe_gate.hip), behind moe_gate_logits for the batches it takes; same bits.  The first
// n_bias rows get the bias.
bool moe_gate_tiles_take(int T, int H, int E);
int moe_gate_tiles(const void *x, const void *wg, const float *bias, int n_bias, float *logits, int T, int H, int E, int ldl,
                   hipStream_t s);
