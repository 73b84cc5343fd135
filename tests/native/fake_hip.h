// A HIP runtime and a set of kernels for CPU tests of the host engine
// (sapporo2_amd/csrc/engine.cpp): one in-order queue that runs as late as the
// engine's waits allow, so that host memory the engine reuses too early is seen
// changed.  Device memory is host memory.  The "kernels" move staged rows into
// the store, copy a call's inputs and write the completion word; no forces.
// A kernel that reads host memory takes a copy of it at its launch and compares
// when it runs.  Requests can be made to fail by count.
#pragma once

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "kernels.h"

namespace fake {

using Op = std::function<void()>;
inline std::deque<Op> queue;
inline uint64_t queued = 0, ran = 0;
inline std::vector<Op>* capture = nullptr;
inline std::map<void*, size_t> device_mem;     // hipMalloc'd, bytes
inline size_t device_bytes = 0;
inline int host_allocs = 0, violations = 0;
inline std::map<std::string, int> fail_in;     // name -> calls until one fails (1: the next)
inline std::map<std::string, int> calls;
inline sapk::ForceConfig last_cfg{};
inline sapk::ForceArgs last_force{};
inline sapk::StoreView last_store{};

// true when the request named so is to fail now
inline bool fails(const char* name) {
  ++calls[name];
  auto f = fail_in.find(name);
  return f != fail_in.end() && f->second > 0 && --f->second == 0;
}
inline void violation(const char* what) {
  if (violations++ < 10) std::printf("violation: %s\n", what);
}
inline void submit(Op op) {
  if (capture) { capture->push_back(std::move(op)); return; }
  queue.push_back(std::move(op));
  ++queued;
}
inline void run_to(uint64_t pos) {
  while (ran < pos && !queue.empty()) {
    Op op = std::move(queue.front());
    queue.pop_front();
    ++ran;
    op();
  }
}
inline void run_all() { run_to(queued); }

// Host memory as it is now; check() when the kernel runs.
struct Seen {
  const char* p = nullptr;
  std::vector<char> copy;
  Seen(const void* q, size_t n) : p(static_cast<const char*>(q)) {
    if (q) copy.assign(p, p + n);
  }
  void check(const char* what) const {
    if (p && std::memcmp(p, copy.data(), copy.size()) != 0) violation(what);
  }
};

inline size_t bytes_from(const void* p) {  // of a device allocation, from p to its end
  auto it = device_mem.upper_bound(const_cast<void*>(p));
  if (it == device_mem.begin()) return 0;
  --it;
  const size_t off = (size_t)(static_cast<const char*>(p) - static_cast<char*>(it->first));
  return off < it->second ? it->second - off : 0;
}

// One staged row into the store; ids only where the launch writes them.
inline void apply_row(const sapk::StoreView& st, int nf, const double* u, bool ids) {
  int pair[2];
  std::memcpy(pair, u + nf, sizeof pair);
  if (pair[0] < 0 || pair[0] >= st.cap) return violation("row address");
  for (int f = 0; f < nf; ++f) st.raw[(size_t)f * st.cap + pair[0]] = u[f];
  if (ids) st.id[pair[0]] = pair[1];
  else if (st.id[pair[0]] != pair[1]) violation("an id changes in a launch that writes none");
}

// The partial rows of a launch lie within their arrays.
inline int check_rows(const sapk::ForceArgs& a, int rows, int order) {
  const size_t n = (size_t)rows * a.grid_ni;
  if (bytes_from(a.part) < n * sapk::part_fields(order) * 8 || bytes_from(a.part_ds2) < n * 8 ||
      bytes_from(a.part_addr) < n * 4) {
    violation("partial rows beyond their arrays");
    return -1;
  }
  return 0;
}

}  // namespace fake

// ------------------------------------------------------------------ runtime
struct ihipStream_t { int x; };
struct ihipEvent_t { uint64_t pos; };
struct ihipGraph { std::vector<fake::Op> ops; };
struct hipGraphExec { std::vector<fake::Op> ops; };

extern "C" {
inline ihipStream_t g_fake_stream;
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "injected"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = &g_fake_stream; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  if (fake::capture) fake::violation("synchronization under capture");
  ++fake::calls["sync"];
  fake::run_all();
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { fake::run_all(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new ihipEvent_t{0}; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  if (fake::fails("event")) return hipErrorUnknown;
  e->pos = fake::queued;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { fake::run_to(e->pos); return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { fake::run_to(e->pos); return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  if (fake::fails("malloc")) return hipErrorOutOfMemory;
  *p = std::calloc(1, n);
  fake::device_mem[*p] = n;
  fake::device_bytes += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  fake::run_all();
  fake::device_bytes -= fake::device_mem[p];
  fake::device_mem.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++fake::host_allocs;
  if (fake::fails("hostmalloc")) return hipErrorOutOfMemory;
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  if (fake::fails("memcpy")) return hipErrorUnknown;
  // a host source may be written again behind the copy: rows are copied anew then
  fake::submit([=] { if (n) std::memcpy(d, s, n); });
  (void)k;
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  if (fake::capture) fake::violation("memset under capture");
  fake::submit([=] { std::memset(d, v, n); });
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  fake::capture = new std::vector<fake::Op>;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = new ihipGraph{std::move(*fake::capture)};
  delete fake::capture;
  fake::capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *x = new hipGraphExec{g->ops};
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) {
  if (fake::fails("graph")) return hipErrorUnknown;
  for (auto& op : x->ops) fake::submit(op);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { delete x; return hipSuccess; }
}

// ------------------------------------------------------------------ kernels
namespace sapk {

bool force_p_supported(int P) { return P >= 1 && P <= 64 && (P & (P - 1)) == 0; }

int launch_scatter(hipStream_t, int, bool, const ScatterArgs& a) {
  fake::last_store = a.st;
  fake::submit([=] {
    for (int k = 0; k < a.cd->nupd; ++k) fake::apply_row(a.st, a.nf, a.upd + (size_t)k * (a.nf + 1), true);
  });
  return 0;
}

int launch_predict(hipStream_t, int, bool, const PredictArgs& a) {
  fake::submit([=] { if (a.desc_out) *a.desc_out = a.desc; });
  return 0;
}

int launch_prep(hipStream_t, int order, bool, const PrepArgs& a) {
  if (fake::fails("prep")) return -1;
  const int nf = raw_fields(order), nr = nf + 1;
  fake::last_store = a.st;
  auto rows = std::make_shared<fake::Seen>(a.nupd > a.nd ? a.rows_h + (size_t)a.nd * nr : nullptr,
                                           a.nupd > a.nd ? (size_t)(a.nupd - a.nd) * nr * 8 : 0);
  auto bits = std::make_shared<fake::Seen>(a.nbits ? a.bits : nullptr, (size_t)a.nbits / 8);
  std::vector<std::shared_ptr<fake::Seen>> in;
  for (const CopySeg& g : a.seg) in.push_back(std::make_shared<fake::Seen>(g.n16 ? g.src : nullptr, (size_t)g.n16 * 16));
  fake::submit([=] {
    rows->check("staged rows changed before the launch that reads them had run");
    bits->check("update bits changed before the launch that reads them had run");
    for (auto& s : in) s->check("call inputs changed before the launch that reads them had run");
    for (int k = 0; k < a.nupd; ++k) {
      const double* u = (k < a.nd ? a.rows_d : a.rows_h) + (size_t)k * nr;
      int addr;
      std::memcpy(&addr, u + nf, sizeof addr);
      // the predictor leaves out marked addresses, and only those
      if (a.pred_j1 > 0 && addr < a.pred_j1 && !(addr < a.nbits && (a.bits[addr >> 5] >> (addr & 31) & 1u)))
        fake::violation("an update the predictor does not leave out");
      fake::apply_row(a.st, nf, u, a.new_ids != 0);
    }
    for (const CopySeg& g : a.seg)
      if (g.n16) std::memcpy(g.dst, g.src, (size_t)g.n16 * 16);
    for (int k = 0; k < a.ni_reset; ++k) a.ngb_cnt[k] = 0;
  });
  return 0;
}

int launch_force(hipStream_t, int order, bool, const ForceArgs& a, const ForceConfig& c) {
  if (fake::fails("force")) return -1;
  fake::last_cfg = c;
  fake::last_force = a;
  if ((long)c.S * c.jchunk < a.nj) fake::violation("splits do not cover the j");
  return fake::check_rows(a, partial_rows(c), order);
}

int launch_force_small(hipStream_t, int order, bool, const SmallArgs& a, const ForceConfig& c, bool) {
  if (fake::fails("small")) return -1;
  const int nf = raw_fields(order), nr = nf + 1;
  fake::last_store = a.st;
  fake::last_cfg = c;
  auto rows = std::make_shared<fake::Seen>(a.nupd ? a.rows_h : nullptr, (size_t)a.nupd * nr * 8);
  auto bits = std::make_shared<fake::Seen>(a.nbits ? a.bits : nullptr, (size_t)a.nbits / 8);
  auto in = std::make_shared<fake::Seen>(a.f.ibuf, (size_t)a.ni * 6 * 8);
  fake::submit([=] {
    rows->check("staged rows changed before the small call that reads them had run");
    bits->check("update bits changed before the small call that reads them had run");
    in->check("call inputs changed before the small call that reads them had run");
    for (int k = 0; k < a.nupd; ++k) fake::apply_row(a.st, nf, a.rows_h + (size_t)k * nr, false);
    for (int k = 0; k < a.ni; ++k) {
      if (a.f.ngb_on && a.f.ngb_cnt[k] != 0) fake::violation("neighbour counters not cleared");
      if (a.f.ngb_on) a.f.ngb_cnt[k] = 1;
    }
    for (int k = 0; k < SMALL_NI; ++k) a.cnt_clear[k] = 0;
  });
  return fake::check_rows(a.f, partial_rows(c), order);
}

int launch_finalize(hipStream_t, int, bool, const FinalizeArgs& a) {
  if (fake::fails("finalize")) return -1;
  fake::submit([=] { if (a.done) *a.done = a.cd ? a.cd->seq : a.seq; });
  return 0;
}

int launch_force_ens(hipStream_t, int order, bool, const EnsArgs& a, const FinalizeArgs& f, int) {
  if (fake::fails("ens")) return -1;
  (void)f;
  const size_t n = (size_t)a.nitems * 64;
  if (fake::bytes_from(a.part) < n * part_fields(order) * 8 || fake::bytes_from(a.part_ds2) < n * 8)
    fake::violation("ensemble rows beyond their arrays");
  return 0;
}

int launch_gather_pred(hipStream_t, int, bool, const GatherArgs& a) {
  fake::submit([=] {
    if (a.addr)
      for (int k = 0; k < a.n; ++k)
        for (int d = 0; d < 3; ++d) a.out[(size_t)d * a.n + k] = a.st.raw[(size_t)(RF_X + d) * a.st.cap + a.addr[k]];
    if (a.done) *a.done = a.seq;
  });
  return 0;
}

int launch_ens_idesc(hipStream_t, const EnsGroup*, int, int, int4*) { return fake::fails("idesc") ? -1 : 0; }
int launch_write_desc(hipStream_t, CallDesc* cd, const CallDesc& v) {
  fake::submit([=] { *cd = v; });
  return 0;
}

}  // namespace sapk
