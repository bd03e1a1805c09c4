// A device of one lane in host memory, for tests of the engine's host code
// (hvm64_api.cpp) without a GPU: the HIP calls it makes and the launches it
// asks for.  Launches run the same rules as the kernels (hvm64_rules.h, host
// build); a reduction runs its redexes one after another.  The lane's
// registers that a kernel keeps on chip stand in front of guard words, so a
// register index past them is seen (fake_guard_intact).
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <vector>

#include "hvm64_rules.h"
#include "fake_device.h"

using namespace hvm;

namespace {
const u64 GUARD = 0x5AFE5AFE5AFE5AFEull;
const u32 GUARD_WORDS = 64 * 64;
std::vector<u64> chip_regs(LDS_SLOTS * 64 + GUARD_WORDS, GUARD);
pair chip_links[LINK_CAP * 64];
int sync_failures = 0;
Params ring;  // the ring of the last launch that used it

// A lane as a one-wave kernel sets it up: `regs`: with registers on chip.
void lane_on_chip(Lane &L, const Params &P, bool regs) {
  lane_init(L, P, 0, 0);
  L.PL = chip_links;
  if (regs) L.T_lds = chip_regs.data();
}

void lane_done(Lane &L) {
  lane_finish(L);
  for (u32 k = 0; k < RW_SLOTS; k++) L.P->g->rw[k] += L.rw[k];
}
}  // namespace

bool fake_guard_intact() {
  for (u32 i = 0; i < GUARD_WORDS; i++)
    if (chip_regs[LDS_SLOTS * 64 + i] != GUARD) return false;
  return true;
}
void fake_fail_next_sync() { sync_failures = 1; }
bool fake_ring_clear() {
  for (u64 i = 0; i < 1024; i++)  // (a test's redexes are in its first slots)
    if (ring.queue[2 * i] || ring.queue[2 * i + 1]) return false;
  return true;
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------
namespace hvm {
hipError_t launch_fill(u64 *words, u64 n, u64 value, hipStream_t) {
  for (u64 i = 0; i < n; i++)
    if (words[i] != value) words[i] = value;  // (untouched zero pages stay so)
  return hipSuccess;
}
hipError_t launch_mirror(const Params &P, hipStream_t) {
  std::memcpy(P.g_host, P.g, sizeof(Globals));
  return hipSuccess;
}
hipError_t launch_exec(const Params &P, u32 def, u64 t0, u32 count_dref, hipStream_t st) {
  Lane L;
  lane_on_chip(L, P, true);
  if (count_dref) L.rw[RW_DREF]++;
  run_def(L, def, t0);
  lane_done(L);
  return launch_mirror(P, st);
}
hipError_t launch_expand(const Params &P, u64 old_root_cell, hipStream_t) {
  Lane L;
  lane_on_chip(L, P, false);
  const u64 r2 = alloc_node(L);
  st2(L, r2, P_NONE, var_port(r2));
  u32 np = 0;
  push_link(L, np, var_port(old_root_cell), expand_ref(r2 + 8));
  flush_links(L, np);
  lane_done(L);
  P.g->root = r2;
  return hipSuccess;
}
hipError_t launch_prepare(const Params &P, hipStream_t) {
  std::memset(P.g->st, 0, sizeof(P.g->st));
  P.g->done = 0;
  return hipSuccess;
}
hipError_t launch_reset(const Params &P, u64 q0, u64 q1, hipStream_t) {
  for (u64 i = q0; i < q1; i++)
    for (u64 k = 0; k < 2; k++)
      if (P.queue[(i & P.qmask) * 2 + k]) P.queue[(i & P.qmask) * 2 + k] = 0;
  std::memset((void *)P.g, 0, sizeof(Globals));
  std::memset(P.alloc_pos, 0, (size_t)P.total_waves * 64 * 8);
  P.heap[ROOT0_WORD] = P_NONE;
  return hipSuccess;
}
hipError_t launch_reduce(const Params &P, u32, hipStream_t) {
  ring = P;
  Lane L;
  lane_on_chip(L, P, true);
  while (P.g->q_head < P.g->q_tail && P.g->err == 0 && P.g->done < P.limit) {
    u64 *const slot = P.queue + (P.g->q_head++ & P.qmask) * 2;
    const u64 a = slot[0], b = slot[1];
    slot[0] = slot[1] = 0;
    P.g->S -= 1ull << 32;
    P.g->done++;
    L.rw[RW_POPS]++;
    run_tasks(L, redex_class(a, b, nullptr, false, P.ndefs), true, a, b, false, 0, 0, 0);
    lane_report(L);
  }
  lane_done(L);
  return hipSuccess;
}
hipError_t launch_boot_batch(const Params &, u32, const u32 *, u64 *, u32, hipStream_t) { return hipErrorNotSupported; }
hipError_t launch_expand_batch(const Params &, u32, u64 *, u32, hipStream_t) { return hipErrorNotSupported; }
hipError_t launch_root_ports(const Params &, u32, const u64 *, u64 *, hipStream_t) { return hipErrorNotSupported; }
hipError_t launch_batch_reset(const Params &, u64, u64, hipStream_t) { return hipErrorNotSupported; }
hipError_t launch_readback(const Params &, u64, u64, u64, u64 *, u64, u64 *, u64, hipStream_t) {
  return hipErrorNotSupported;
}
u32 reduce_waves_per_block() { return WAVES_PER_BLOCK; }
u32 reduce_book_lds_words() { return BOOK_LDS_WORDS; }
u32 reduce_lds_slots() { return LDS_SLOTS; }
hipError_t reduce_occupancy(int *blocks_per_cu) {
  *blocks_per_cu = 1;
  return hipSuccess;
}
hipError_t noalloc_scratch(u64 **out) {
  static u64 scratch[1];
  *out = scratch;
  return hipSuccess;
}
u32 noalloc_nets() { return 0; }
}  // namespace hvm

// ---------------------------------------------------------------------------
// HIP
// ---------------------------------------------------------------------------
extern "C" {
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
  std::memset((void *)p, 0, sizeof *p);
  p->multiProcessorCount = 1;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 100000;
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  *p = std::calloc(n ? n : 1, 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void **d, void *p, unsigned) {
  *d = p;
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void *d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  if (sync_failures == 0) return hipSuccess;
  sync_failures--;
  return hipErrorUnknown;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error of the test device"; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}
