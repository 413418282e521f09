// moe_forward's bookkeeping of unit lists on their way to the host, on the CPU: the engine with its HIP backend over a
// stand-in of the HIP runtime (memory is malloc, copies happen at once, any call can be told to fail) and kernel entry
// points that do what the real ones promise the host: they store the unit list and the sequence word, or refuse.
// A forward that fails on its way (the refresh of the slot table, the expert launch) must leave no slot waiting for a word
// that nobody writes: the forwards after it, and the drain, go on at once, and count every hit.  A refresh of the slot table
// that failed stays due: the launches after it find the slots' addresses.
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

#include "moe_engine.h"
#include "moe_kernels.h"

// ---- the HIP runtime, as far as the engine uses it ----
static int g_fail_copies = 0;   // that many host-to-device copies on the compute stream fail
static hipStream_t g_compute = (hipStream_t)0x10;
extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)0x20; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)0x30; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = calloc(1, n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
  if (st == g_compute && k == hipMemcpyHostToDevice && g_fail_copies > 0) { --g_fail_copies; return hipErrorUnknown; }
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) { memset(a, 0, sizeof *a); a->type = hipMemoryTypeHost; return hipSuccess; }
}

// ---- kernel entry points of the path under test; every batch uses all E experts ----
static const int E = 8, K = 2, H = 256, I = 128;
static int g_refuse = 0;        // that many expert launches are refused
static uint64_t g_first_slot_seen = 0;
extern "C" {
int moe_gate_logits_bias_rows(const void *, const void *, const float *, int, float *, int, int, int, int, void *) { return MOE_OK; }
int moe_topk_dispatch_ws(const float *, int T, int, int, int, int, int *, float *, int *, int *, int *, int *, int *, moe_unit *units,
                         int *n_active, int64_t *, int max_units, void *, int64_t, int *, void *) {
  for (int u = 0; u < max_units; ++u) units[u] = moe_unit{u, T * K / E, u * (T * K / E), 0};
  *n_active = max_units;
  return MOE_OK;
}
int moe_experts_prefill_publish(const void *, int, int, int, int, int, int, const moe_unit *units, int, const int *,
                                const uint64_t *table, const void *, void *, void *, float *, float *, int, void *, int *,
                                int, const moe_publish *pub, void *) {
  if (g_refuse > 0) { --g_refuse; return MOE_EINVAL; }
  g_first_slot_seen = table[0];
  if (pub) {
    for (int u = 0; u < *pub->n_active; ++u) pub->units_host[u] = units[u];
    *pub->n_active_host = *pub->n_active;
    *pub->seq_host = pub->seq_value;
  }
  return MOE_OK;
}
int moe_combine_splits(const float *, const float *, const float *, const int *, const float *, int, void *, int, int, int, int, void *) {
  return MOE_OK;
}
}

#define CK(call)                                                                         \
  do {                                                                                   \
    const int rc_ = (call);                                                              \
    if (rc_ != 0) { printf("%s failed (%d): %s\n", #call, rc_, moe_last_error()); return 1; } \
  } while (0)

int main(int argc, char **argv) {
  // which step of the forward fails: table | launch | windows (an entry point this build has no stand-in for but the stub)
  const std::string what = argc > 1 ? argv[1] : "table";
  const bool windows = what == "windows";
  moe_cfg *cfg = moe_cfg_create(1, E);
  const char *names[1] = {"w"};
  CK(moe_cfg_set_params(cfg, names, 1));
  CK(moe_cfg_set(cfg, "num_expert_per_token", "2"));
  CK(moe_cfg_set(cfg, "cache_rate", "1.0"));
  CK(moe_cfg_set(cfg, "cache_policy", "lru"));
  setenv("SPARSE_CACHE_PHYSICAL_MEM_IMPL", "slab", 1);   // (one allocation: the stand-in maps no memory)
  CK(moe_cfg_finalize(cfg));
  moe_engine *eng = nullptr;
  CK(moe_engine_create(cfg, MOE_BACKEND_HIP, g_compute, &eng));
  std::vector<std::vector<uint8_t>> bufs;
  for (int e = 0; e < E; ++e) {
    bufs.emplace_back(512, (uint8_t)e);
    CK(moe_register_param(eng, 0, e, 0, bufs.back().data(), bufs.back().size(), 0));
  }
  CK(moe_init_slots(eng));
  std::vector<uint16_t> gate((size_t)E * H), x((size_t)100 * H), y((size_t)100 * H), shared(windows ? 3 * 5120 * H : 1);
  moe_layer_desc d;
  memset(&d, 0, sizeof d);
  d.H = H; d.I = I; d.top_k = K; d.fmt = MOE_FMT_BF16; d.gate_w = gate.data();
  if (windows) { d.I_sh = 5120; d.shared = shared.data(); }   // (w2 reduction in windows from 65 tokens on)
  CK(moe_set_layer(eng, 0, &d));
  CK(moe_forward_prepare(eng, 100));
  CK(moe_launch(eng));
  // every expert into its slot through the module hooks, which leave the slot table's copy on the device as it was
  std::vector<int64_t> ids(E);
  for (int e = 0; e < E; ++e) ids[e] = e;
  CK(moe_report_layer_logits(eng, 0, nullptr, 1, 40, H));
  CK(moe_report_one_layer(eng, 0, ids.data(), E));
  for (int64_t e : ids) {
    CK(moe_wait_expert(eng, 0, (int)e));
    CK(moe_expert_launched(eng, 0, (int)e));
  }
  CK(moe_layer_done(eng, 0));
  CK(moe_drain(eng));
  moe_counters c0, c1;
  CK(moe_get_counters(eng, &c0));
  if (what == "table") g_fail_copies = 1;
  if (what == "launch") g_refuse = 1;
  if (moe_forward(eng, 0, x.data(), windows ? 100 : 40, y.data()) == MOE_OK) { printf("the forward that was to fail did not\n"); return 1; }
  if (g_fail_copies || g_refuse) { printf("the failure was not met\n"); return 1; }
  const auto t0 = std::chrono::steady_clock::now();
  const int n = 20;   // more than there are slots
  for (int i = 0; i < n; ++i) CK(moe_forward(eng, 0, x.data(), 40, y.data()));
  CK(moe_drain(eng));
  CK(moe_get_counters(eng, &c1));
  const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  printf("hits %llu of %d, %.3f s, table %s\n", (unsigned long long)(c1.hit - c0.hit), n * E, s, g_first_slot_seen ? "filled" : "empty");
  moe_engine_destroy(eng);
  moe_cfg_destroy(cfg);
  return c1.hit - c0.hit == (uint64_t)(n * E) && s < 2.0 && g_first_slot_seen ? 0 : 1;
}
