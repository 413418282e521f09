#include "moe_common.h"

#include <stdarg.h>
#include <stdio.h>

static thread_local char g_err[512] = "";

void moe_set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
}

extern "C" const char *moe_last_error(void) { return g_err; }

int moe_check_hip(hipError_t e, const char *what) {
  if (e == hipSuccess) return MOE_OK;
  moe_set_error("%s: %s", what, hipGetErrorString(e));
  return MOE_EHIP;
}

int moe_check_launch(const char *what) { return moe_check_hip(hipGetLastError(), what); }

// ---- per-kernel timing -----------------------------------------------------
#include <mutex>
#include <vector>
namespace {
struct KRec { int kid; hipEvent_t a, b; };
std::mutex g_kt_mu;
bool g_kt_on = false;
std::vector<KRec> g_kt_recs;
std::vector<hipEvent_t> g_kt_free;
hipEvent_t g_kt_open[MOE_K_COUNT];
const size_t kMaxRecs = 1 << 15;
hipEvent_t kt_event() {
  if (!g_kt_free.empty()) { hipEvent_t e = g_kt_free.back(); g_kt_free.pop_back(); return e; }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}
}  // namespace

void moe_ktimer_begin(int kid, hipStream_t s) {
  if (!g_kt_on) return;
  std::lock_guard<std::mutex> lk(g_kt_mu);
  if (g_kt_recs.size() >= kMaxRecs) return;
  hipEvent_t e = kt_event();
  if (!e) return;
  (void)hipEventRecord(e, s);
  g_kt_open[kid] = e;
}
void moe_ktimer_end(int kid, hipStream_t s) {
  if (!g_kt_on) return;
  std::lock_guard<std::mutex> lk(g_kt_mu);
  if (!g_kt_open[kid]) return;
  hipEvent_t e = kt_event();
  if (!e) return;
  (void)hipEventRecord(e, s);
  g_kt_recs.push_back(KRec{kid, g_kt_open[kid], e});
  g_kt_open[kid] = nullptr;
}

extern "C" int moe_kernel_timing(int enable) {
  std::lock_guard<std::mutex> lk(g_kt_mu);
  g_kt_on = enable != 0;
  for (auto &r : g_kt_recs) { g_kt_free.push_back(r.a); g_kt_free.push_back(r.b); }
  g_kt_recs.clear();
  for (auto &e : g_kt_open) e = nullptr;
  return MOE_OK;
}

extern "C" int moe_kernel_timing_read(int kernel_id, double *total_ms, int *calls) {
  if (kernel_id < 0 || kernel_id >= MOE_K_COUNT || !total_ms || !calls) { moe_set_error("moe_kernel_timing_read: bad argument"); return MOE_EINVAL; }
  std::lock_guard<std::mutex> lk(g_kt_mu);
  double tot = 0;
  int n = 0;
  for (auto &r : g_kt_recs) {
    if (r.kid != kernel_id) continue;
    if (hipEventSynchronize(r.b) != hipSuccess) continue;
    float ms = 0;
    if (hipEventElapsedTime(&ms, r.a, r.b) == hipSuccess) { tot += ms; ++n; }
  }
  *total_ms = tot;
  *calls = n;
  return MOE_OK;
}

// Pieces the w2 pass leaves the routed experts' partial rows in (moe_experts_prefill_windows).  A few wide experts have few
// tiles of a long reduction (Mixtral shape, 256 tokens: 128 workgroups over 224 slabs, half the chip idle for 190 us; 2048
// tokens: 592 workgroups for 512 places, 80 of them in a second round of 290 us).  Windows of at least 32 slabs while the launch
// has no more workgroups than the chip has places (two per compute unit; an expert has at least one tile, and one more per 128
// rows); past that only windows of 96 slabs and more, up to three per compute unit: the rows of more pieces cost the launch and the
// combine more than the last round has left.  us a layer, 1 / 2 / 4 / 8 pieces, Mixtral shape int4: 128 tokens 272 / 230 / 224 / 230, 379
// 382 / 333 / 328 / 343, 512 470 / 453 / 446 / 456, 1024 777 / 744 / 744 / 778, 2048 1454 / 1427 / 1431 / 1504, 4096 2589 / 2569 / 2627 / 2778.  q4_K,
// passes and combine, 1 / 2 / 4: the same shape 65 tokens 247 / 190 / 193, 128 276 / 225 / 229, 512 464 / 440 / 433, 1024 758 / 730 / 721, 2048 1380 /
// 1337 / 1358; 2048 x 8192, 16 experts top-2 128 tokens 141 / 117 / 115, 512 189 / 154 / 156; 32 experts top-4 65 tokens 217 / 208 / 216, 1024
// 506 / 497 / 503.  A chip that is full already loses: 2048 x 4096, 64 experts top-6 q4_K 65 tokens 207 / 213, 128 205 / 210, 512 260 / 274;
// 4096 x 4096, 32 experts top-4 65 tokens int4 202 / 207, q4_K 206 / 214; 2048 x 8192, 64 experts 512 tokens int4 513 / 527, q4_K 533 / 539, 32
// experts 1536 tokens 648 / 654, 660 / 671 (16 experts 4096 tokens, left whole as well, would gain: 825 / 812, 834 / 818).  So do short
// reductions: DeepSeek shape (22 slabs) 128 tokens 91.1 / 93.8, 2048 367 / 392; Qwen2-57B shape (40 slabs) 128 tokens 312 / 312 / 322,
// 512 610 / 620 / 663.
extern "C" int moe_prefill_routed_windows(int fmt, int T, int k, int E, int H, int I) {
  if ((fmt != MOE_FMT_INT4_G128 && fmt != MOE_FMT_Q4K) || T <= 0 || k <= 0 || E <= 0 || H <= 0 || I <= 0) return 1;
  const long long P = (long long)T * k, wgs = ((P < E ? P : E) + P / 128) * (H / 256);
  const int nk = I / 64;
  int s = 1;
  while (s < 4 && nk % (s * 2) == 0 && nk / (s * 2) >= 32 && wgs * s <= (nk / (s * 2) >= 96 ? 767 : 512)) s *= 2;
  return s;
}

// Pieces for the shared expert's partial rows of moe_experts_prefill_windows beside routed experts of I columns: those of
// moe_prefill_shared_splits, and two for an int4 shared expert of 32 slabs and more in a launch of few of its tiles.  There its
// workgroups, which have every token's row where the routed experts' have a few, are the last to end (DeepSeek shape, 128 tokens: 8
// workgroups of 44 slabs, 36 us, beside 280 of 22 slabs).  us a layer, one piece / two, DeepSeek shape: 65 tokens 85.9 / 73.4, 128
// 104.2 / 91.2, 200 115.7 / 103.0, 379 145.3 / 133.3, 512 156.3 / 152.8; past 32 tiles the shared expert's workgroups start a full round and the
// pieces only cost the combine: 1024 tokens 229.9 / 232.4, 2048 367.2 / 374.1.  It pays beside routed experts of the same length too (w13
// and w2 passes and combine, 65 / 128 / 512 tokens): 2048 columns both, 16 experts top-2 63.0 / 57.0, 66.6 / 59.7, 81.1 / 78.3; 2816 both
// 71.6 / 64.2, 76.7 / 67.3, 94.5 / 91.6; with 64 experts top-6, whose launches fill the chip, within 3 % (2816 both 163.4 / 159.5, 162.6 /
// 165.1, 208.8 / 206.4) but where the launch just fits it at once without them (2048 both, 65 tokens: 120 / 127).
// bf16 past 64 tokens (tile kernel, one workgroup per compute unit): from 64 slabs on, windows of an even number, at least 20, while
// there are at most 16 workgroups and one of them has a longer reduction than the routed experts'.  Qwen1.5 shape, 128 tokens: 8
// workgroups of 88 slabs took 85 us beside two rounds of 33 us of the routed experts' 22 slabs.  us a layer, 1 / 2 / 4 pieces: 65
// tokens 222.1 / 213.1 / 210.3, 128 230.4 / 221.3 / 217.2, 256 243.8 / 233.7 / 248.3, 379 255.2 / 256.2 / 261.7, 1024 325.3 / 327.8 / 340.9.  44 slabs beside 22
// (2048 x 1408, shared 2816): 65 tokens 149.2 / 151.2, 256 180.8 / 183.3.  128 tokens, passes and combine, 60 experts top-4, shared beside
// routed columns: 5632 beside 2816 387.2 / 368.5 / 370.4, beside 4096 505.5 / 499.1 / 501.7, beside 5632 675.5 / 676.1 / 684.1; 4096 beside
// 2048 280.8 / 267.8 / 268.5, beside 4096 493.9 / 494.2 / 499.6.
extern "C" int moe_prefill_shared_windows_beside(int fmt, int T, int H, int I, int I_sh) {
  int s = moe_prefill_shared_splits(fmt, T, H, I_sh);
  const int tiles = (T + 127) / 128 * (H / 256), nk = I_sh / 64;
  if (fmt == MOE_FMT_BF16 && T > 64 && H > 0 && I_sh > 0) {
    while (s < 4 && tiles * s <= 16 && nk % (4 * s) == 0 && nk >= 64 && nk / (2 * s) >= 20 && I_sh / s > I) s *= 2;
    return s;
  }
  if (s > 1 || fmt != MOE_FMT_INT4_G128 || T <= 0 || H <= 0 || I_sh <= 0) return s;
  return tiles <= 32 && nk % 2 == 0 && nk >= 32 ? 2 : 1;
}

// the most of them, whatever the routed experts
extern "C" int moe_prefill_shared_windows(int fmt, int T, int H, int I_sh) { return moe_prefill_shared_windows_beside(fmt, T, H, 0, I_sh); }
