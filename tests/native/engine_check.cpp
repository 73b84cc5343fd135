// Checks of the host engine against a HIP runtime of the test's own (fake_hip.h):
// one check per argument.
#include "fake_hip.h"

#include <chrono>
#include <set>

#include "engine.h"

using namespace sap;
using namespace sapk;

namespace {

int bad = 0;
#define EXPECT(c, ...)                                            \
  do {                                                            \
    if (!(c)) {                                                   \
      ++bad;                                                      \
      std::printf("%s:%d: " #c " does not hold: ", __FILE__, __LINE__); \
      std::printf(__VA_ARGS__);                                   \
      std::printf("\n");                                          \
    }                                                             \
  } while (0)

// A program: n particles, each send recorded so that the store can be compared.
struct Program {
  Engine e;
  int order;
  std::vector<double> x;  // last x sent, by address
  std::vector<int> id;
  Program(int n, int order_ = ORDER_H4, int prec = PREC_DS) : order(order_), x(n, 0.0), id(n, 0) {
    if (e.open(0, order, prec) != 0) std::abort();
    if (n == 0) return;
    std::vector<int> a(n);
    std::vector<double> m(n, 1.0), p(3 * (size_t)n);
    for (int k = 0; k < n; ++k) { a[k] = k; id[k] = 10 + k; x[k] = p[3 * (size_t)k] = k; }
    if (e.set_j_particles(n, a.data(), id.data(), nullptr, nullptr, m.data(), nullptr, nullptr, nullptr, p.data(),
                          nullptr, nullptr, nullptr) != 0)
      std::abort();
    e.set_time(0.0);
    if (e.force_prediction(n) != 0) std::abort();
  }
  void send(int a, double v, int new_id = -1) {
    if (new_id >= 0) id[a] = new_id;
    x[a] = v;
    const double p[3] = {v, 0, 0}, z[3] = {0, 0, 0};
    EXPECT(e.set_j_particle(a, id[a], 0, 0, 1, z, z, z, p, z, z, 0) == 0, "send %d", a);
  }
  void batch(const std::vector<int>& a, double v) {
    const int n = (int)a.size();
    std::vector<int> ids(n);
    std::vector<double> m(n, 1.0), p(3 * (size_t)n, 0.0);
    for (int k = 0; k < n; ++k) { ids[k] = id[a[k]]; p[3 * (size_t)k] = x[a[k]] = v + k; }
    EXPECT(e.set_j_particles(n, a.data(), ids.data(), nullptr, nullptr, m.data(), nullptr, nullptr, nullptr, p.data(),
                             nullptr, nullptr, nullptr) == 0, "batch of %d", n);
  }
  int call(int nj, int ni, bool lists = false, bool predict = true) {
    std::vector<int> ids(ni, -5);
    std::vector<double> p(3 * (size_t)ni, 0.5), h(ni, 1.0);
    predict ? e.set_time(1.0) : e.set_no_time();
    const auto* v = reinterpret_cast<const double(*)[3]>(p.data());
    return e.start_grav_calc(nj, ni, ids.data(), v, v, v, 1e-4, lists ? h.data() : nullptr);
  }
  int results(int nj, int ni) {
    std::vector<double> a(3 * (size_t)ni);
    return e.get_grav_results(nj, ni, reinterpret_cast<double(*)[3]>(a.data()), nullptr, nullptr, nullptr, nullptr,
                              nullptr, nullptr, false);
  }
  // the store holds what was sent
  void check(const char* label) {
    EXPECT(e.force_prediction(0) == 0, "%s", label);
    EXPECT(e.synchronize() == 0, "%s", label);
    const StoreView& st = fake::last_store;
    int wrong = 0;
    for (size_t a = 0; a < x.size(); ++a)
      wrong += st.raw[(size_t)RF_X * st.cap + a] != x[a] || st.id[a] != id[a];
    EXPECT(wrong == 0, "%s: %d addresses of the store differ from what was sent", label, wrong);
    EXPECT(fake::violations == 0, "%s", label);
    fake::violations = 0;
  }
};

int ens_call(Program& p, const std::vector<int>& nj, int per) {
  std::vector<int> c, ids;
  for (size_t k = 0; k < nj.size(); ++k)
    for (int i = 0; i < per; ++i) { c.push_back((int)k); ids.push_back(-5); }
  const int ni = (int)c.size();
  std::vector<double> x(3 * (size_t)ni, 0.5), eps(nj.size(), 1e-4);
  const auto* v = reinterpret_cast<const double(*)[3]>(x.data());
  p.e.set_time(1.0);
  return p.e.start_grav_calc_clusters(ni, c.data(), ids.data(), v, v, v, eps.data(), nullptr);
}

}  // namespace

struct Fault {
  const char* what;  // fake::fails name, and which of the call's requests of that name fails
  int nth, ni, lists;
  bool ens;
};

// Calls that fail, each followed by sends into both stages and by calls that succeed.
void fail_and_go_on(const Fault* at, int cases) {
  for (int q = 0; q < cases; ++q) {
    const Fault& f = at[q];
    Program p(std::max(3000, f.ni));
    const int np = (int)p.x.size();
    const std::vector<int> cl(4, 700);
    if (f.ens) EXPECT(p.e.set_clusters(4, cl.data()) == 0, "clusters");
    char label[96];
    std::snprintf(label, sizeof label, "%s %d of a call of %d%s", f.what, f.nth, f.ni, f.ens ? " (ensemble)" : "");
    bool reached = false;
    for (int r = 0; r < 3; ++r) {
      // "prep" 2: ids change, so that updates and prediction are two launches
      const bool ids = f.nth == 2 && std::strcmp(f.what, "prep") == 0;
      for (int k = 0; k < 40; ++k) p.send(3 * k + r, 1000.0 * r + k, ids ? 90000 + 100 * r + k : -1);
      fake::fail_in[f.what] = f.nth;
      const int rc = f.ens ? ens_call(p, cl, f.ni) : p.call(np, f.ni, f.lists != 0);
      const bool hit = fake::fail_in[f.what] == 0;  // memory that is there is not asked for again
      fake::fail_in.clear();
      reached |= hit;
      EXPECT((rc != 0) == hit, "%s: returns %d", label, rc);
      for (int k = 0; k < 40; ++k) p.send(3 * k + 1, -1.0 - k - 50 * r);
      EXPECT(p.e.force_prediction(0) == 0, "%s: flush", label);
      for (int k = 0; k < 40; ++k) p.send(3 * k + 2, -2.0 - k - 50 * r);
      EXPECT((f.ens ? ens_call(p, cl, 40) : p.call(np, 70, f.lists != 0)) == 0, "%s: the next call", label);
      EXPECT(p.results(np, 3) == 0, "%s: the next results", label);
      EXPECT(p.call(np, 5, true) == 0 && p.results(np, 5) == 0, "%s: a small call", label);
    }
    EXPECT(reached || f.nth > 3, "%s: not reached", label);
    p.check(label);
  }
}

// A call that fails after device work was queued: the memory which that work reads
// is not written before it has run, and the next calls are as any other.
void failed_calls() {
  const Fault at[] = {{"idesc", 1, 3, 0, true},      {"ens", 1, 3, 0, true},       {"event", 1, 3, 0, true},
                      {"force", 1, 100, 0, false},   {"finalize", 1, 100, 1, false}, {"event", 1, 5000, 0, false},
                      {"small", 1, 5, 1, false},     {"finalize", 1, 5, 1, false}, {"prep", 1, 100, 1, false},
                      {"prep", 2, 100, 0, false}};
  fail_and_go_on(at, sizeof at / sizeof *at);
}

// Memory that a growing buffer does not get: the buffer is not used at a size it no
// longer has.
void failed_growth() {
  std::vector<Fault> at;
  for (int nth = 1; nth <= 8; ++nth) {  // no call makes as many requests
    at.push_back({"malloc", nth, 700, 1, true});
    at.push_back({"malloc", nth, 5000, 0, true});
    at.push_back({"malloc", nth, 16384, 1, false});
    at.push_back({"hostmalloc", nth, 5000, 0, true});
  }
  at.push_back({"hostmalloc", 1, 700, 0, true});
  at.push_back({"hostmalloc", 1, 16384, 1, false});
  fail_and_go_on(at.data(), (int)at.size());
}

// A program that sends its particles one by one has its addresses released on its own
// thread, however many: the host threads (started at their first use) are not.
void send_release() {
  const int n = 131072;
  Program p(0);
  p.x.assign(n, 0.0);
  p.id.assign(n, 7);
  for (int r = 0; r < 2; ++r) {
    for (int a = 0; a < n; ++a) p.send(a, 1.0 + r + a);
    EXPECT(p.call(n, 100) == 0 && p.results(n, 100) == 0, "call");
  }
  int threads = 0;
  if (FILE* f = std::fopen("/proc/self/status", "r")) {
    char line[256];
    while (std::fgets(line, sizeof line, f)) std::sscanf(line, "Threads: %d", &threads);
    std::fclose(f);
  }
  EXPECT(threads == 1, "%d threads", threads);
  p.check("sends");
}

// A load takes the dump's capacity: addresses beyond it are refused as on an engine
// that never held more, whatever this one held before.
void load_capacity() {
  Program small(1000);
  std::vector<char> dump((size_t)small.e.state_bytes());
  EXPECT(small.e.save_state(dump.data(), (long long)dump.size()) == 0, "save");
  Program p(60000);
  EXPECT(p.e.load_state(dump.data(), (long long)dump.size()) == 0, "load");
  const double z[3] = {0, 0, 0};
  for (Engine* e : {&small.e, &p.e})
    EXPECT(e->set_j_particle(50000, 1, 0, 0, 1, z, z, z, z, z, z, 0) != 0, "address beyond the dump's capacity");
  p.x.assign(1000, 0.0);
  p.id.assign(1000, 0);
  for (int k = 0; k < 1000; ++k) { p.x[k] = k; p.id[k] = 10 + k; }
  p.send(999, 5.0, 12);
  p.check("after a load");
}

// A send that fails leaves its address's id as it was: the next send of that id writes it.
void failed_send() {
  const int n = 1500;
  Program p(0);
  p.x.assign(n, 0.0);
  p.id.assign(n, 7);
  for (int a = 0; a < n; ++a) {
    p.send(a, a);
    if (a % 500 == 499) EXPECT(p.e.force_prediction(0) == 0, "flush");
  }
  int failed = 0;
  for (int a = 0; a < n; ++a) {
    // 1024 rows are staged: this send asks for more
    if (a == 1024) fake::fail_in["hostmalloc"] = 1;
    const double x[3] = {p.x[a] = 3.0 * a, 0, 0}, z[3] = {0, 0, 0};
    p.id[a] = 50000 + a;
    if (p.e.set_j_particle(a, p.id[a], 0, 0, 1, z, z, z, x, z, z, 0) != 0) {
      ++failed;
      EXPECT(p.e.force_prediction(0) == 0, "flush");
      p.send(a, p.x[a]);
      EXPECT(p.call(n, 5) == 0 && p.results(n, 5) == 0, "call");
    }
  }
  fake::fail_in.clear();
  EXPECT(failed == 1, "%d sends failed", failed);
  p.check("after a failed send");
}

// Work-groups go to the 8 XCDs in turn: the j that a launch gives them.
double xcd_balance(const ForceConfig& c, int ni, int nj) {
  const int G = (ni + c.P - 1) / c.P, nb = c.S / 4;
  const Splits sp = make_splits(c.P, c.S, nj);
  std::vector<double> j(8, 0.0);
  for (int g = 0; g < G; ++g)
    for (int b = 0; b < nb; ++b)
      j[(size_t)(g * nb + b) % 8] += std::min(nj, sp.begin(4 * b + 4)) - std::min(nj, sp.begin(4 * b));
  double top = 0, sum = 0;
  for (double v : j) { top = std::max(top, v); sum += v; }
  return top * 8 / sum;
}

// Large calls of any size give the 8 XCDs the same work, to the ranges' unit; splits
// cover the j once, in order.
void xcd_shapes() {
  for (int f64 = 0; f64 < 2; ++f64) {
    Engine e;
    EXPECT(e.open(0, ORDER_H4, f64 ? PREC_DOUBLE : PREC_DS) == 0, "open");
    for (int nj : {65536, 100003, 131072, 200003, 262144, 1048577})
      for (int ni = 2000; ni <= NPIPES; ni += 237) {
        const ForceConfig c = e.choose_config(ni, nj, true);
        const double b = xcd_balance(c, ni, nj);
        EXPECT(b < 1.02, "%d i x %d j, S = %d: the busiest XCD has %.3f of the mean", ni, nj, c.S, b);
      }
    for (int nj : {1, 15, 16, 17, 63, 64, 65, 1000, 4097, 131071})
      for (int S : {1, 3, 16, 33, 200, 1000})
        for (int P : {64, 16, 4, 1}) {
          e.set_force_override(P, S);
          const ForceConfig c = e.choose_config(100, nj, true);
          const Splits sp = make_splits(c.P, c.S, nj);
          int longest = 0;
          for (int k = 0; k < c.S; ++k) {
            EXPECT(sp.begin(k + 1) >= sp.begin(k), "order");
            longest = std::max(longest, sp.begin(k + 1) - sp.begin(k));
          }
          EXPECT(sp.begin(0) == 0 && sp.begin(c.S) >= nj && sp.begin(c.S) - nj < sp.unit, "cover %d", nj);
          EXPECT(longest == c.jchunk, "longest range %d, jchunk %d", longest, c.jchunk);
        }
  }
}

// The allocation-free call: rows within the scratch region, and no fewer splits than a
// halving needs for that (a split count that is no whole work-group writes four times
// the rows).
void noalloc_shapes() {
  const size_t bytes = size_t(64) << 20;
  std::vector<char> scratch(bytes);
  fake::device_mem[scratch.data()] = bytes;
  std::vector<int> ids(NPIPES, 1);
  std::vector<double> in(10 * NPIPES, 0.0), out(13 * NPIPES);
  for (int order : {ORDER_H4, ORDER_H6}) {
    Program p(1000, order);
    for (int nj : {100003, 131072, 200003, 300000}) {
      std::vector<int> a(1, nj - 1), id(1, 5);
      std::vector<double> m(1, 1.0), x(3, 0.0);
      EXPECT(p.e.set_j_particles(1, a.data(), id.data(), nullptr, nullptr, m.data(), nullptr, nullptr, nullptr, x.data(),
                                 nullptr, nullptr, nullptr) == 0, "send");
      p.e.set_time(0.0);
      EXPECT(p.e.force_prediction(nj) == 0, "flush");
      for (int ni : {65, 1000, 4096, 5000, 8192, 12345, 15000, 16384}) {
        const ForceConfig direct = p.e.choose_config(ni, nj, false);
        p.e.set_time(1.0);
        EXPECT(p.e.grav_calc_scratch(scratch.data(), bytes, nj, ni, ids.data(), in.data(), 1e-4, out.data(), nullptr) == 0,
               "%d x %d", ni, nj);
        const ForceConfig c = fake::last_cfg;
        const double row = ni * (8.0 * (part_fields(order) + 1) + 4), rows = partial_rows(c);
        EXPECT(c.S == direct.S || rows * 2.3 * row > (double)bytes, "%d x %d: %d splits, %g rows of %g", ni, nj, c.S,
               rows, row);
        EXPECT(xcd_balance(c, ni, nj) < 1.02, "%d x %d: XCDs", ni, nj);
        p.e.synchronize();
      }
    }
  }
  fake::device_mem.erase(scratch.data());
  EXPECT(fake::violations == 0, "rows");
}

// Picking up the active particles of a step asks for no memory, between calls with and
// without graphs; more than a call's worth of them does once.
void pick_up() {
  const int n = 40000;
  for (int graphs = 0; graphs < 2; ++graphs) {
    Program p(n);
    p.e.set_graphs(graphs != 0);
    for (int m : {1, 2500, NPIPES, 30000}) {
      p.send(m / 2, 4.0 * m);
      EXPECT(p.call(n, 100) == 0, "call");
      std::vector<int> a(m);
      for (int k = 0; k < m; ++k) a[k] = m - 1 - k;
      std::vector<double> x(3 * (size_t)m), mass(m);
      const int before = fake::host_allocs;
      const size_t bytes = fake::device_bytes;
      EXPECT(p.e.retrieve_predicted_j_particles(m, a.data(), mass.data(), reinterpret_cast<double(*)[3]>(x.data()),
                                                nullptr, nullptr) == 0, "pick-up of %d", m);
      EXPECT((fake::host_allocs == before) == (m <= NPIPES), "%d: %d pinned allocations", m, fake::host_allocs - before);
      EXPECT(fake::device_bytes == bytes, "%d: device memory", m);
      int wrong = 0;
      for (int k = 0; k < m; ++k) wrong += x[3 * (size_t)k] != p.x[a[k]];
      EXPECT(wrong == 0, "%d of %d rows", wrong, m);
      EXPECT(p.results(n, 100) == 0 && p.call(n, 5) == 0 && p.results(n, 5) == 0, "calls after it");
    }
    p.check("pick-up");
  }
}

// An engine's partial rows take what its calls write.
void scratch_size() {
  for (int ni : {100, 5000, 16384}) {
    Program p(131072);
    EXPECT(p.call(131072, ni) == 0 && p.results(131072, ni) == 0, "call");
    const size_t want = (size_t)partial_rows(fake::last_cfg) * ni * part_fields(ORDER_H4) * 8;
    const size_t got = fake::bytes_from(fake::last_force.part);
    EXPECT(got == want, "%d: %zu bytes of rows, %zu are written", ni, got, want);
    p.check("rows");
  }
}

// Split-major order and pipelined list stores keep the general shapes at every active
// count: at least 512 j a split (split-major launches write a row for each).
void mode_shapes() {
  Engine e;
  EXPECT(e.open(0, ORDER_H4, PREC_DS) == 0, "open");
  for (int mode = 0; mode < 2; ++mode) {
    e.set_split_major(mode == 0);
    e.set_ngb_pipeline(mode == 1);
    for (int ni : {1, 20, 33, 64, 65, 333, 5000, 16384}) {
      const ForceConfig c = e.choose_config(ni, 131072, true);
      EXPECT(c.small == 0 && c.jchunk >= 512, "%d i: %d splits of %d", ni, c.S, c.jchunk);
    }
  }
}

// A batch with an address that no store can hold is refused, large batches like small
// ones, and leaves the engine as it was.
void batch_range() {
  Program p(9000);
  for (int n : {3, 7000}) {
    std::vector<int> a(n), id(n, 1);
    std::vector<double> m(n, 1.0), x(3 * (size_t)n, 0.0);
    for (int k = 0; k < n; ++k) a[k] = k;
    for (int wrong : {INT_MAX, -1}) {
      a[0] = wrong;  // first: nothing of the batch is staged
      EXPECT(p.e.set_j_particles(n, a.data(), id.data(), nullptr, nullptr, m.data(), nullptr, nullptr, nullptr, x.data(),
                                 nullptr, nullptr, nullptr) != 0, "address %d in a batch of %d", wrong, n);
    }
  }
  p.send(8999, 2.0, 3);
  std::vector<int> a(7000);
  for (int k = 0; k < 7000; ++k) a[k] = 2 * k % 9000 + (k >= 4500);
  p.batch(a, 0.5);
  EXPECT(p.call(9000, 100) == 0 && p.results(9000, 100) == 0, "call");
  p.check("after refused batches");
}

int main(int argc, char** argv) {
  const std::string want = argc > 1 ? argv[1] : "";
  const struct { const char* name; void (*f)(); } checks[] = {
      {"failed_calls", failed_calls},
      {"failed_growth", failed_growth},
      {"send_release", send_release},
      {"load_capacity", load_capacity},
      {"failed_send", failed_send},
      {"xcd_shapes", xcd_shapes},
      {"noalloc_shapes", noalloc_shapes},
      {"pick_up", pick_up},
      {"scratch_size", scratch_size},
      {"mode_shapes", mode_shapes},
      {"batch_range", batch_range},
  };
  int ran = 0;
  for (const auto& c : checks)
    if (want.empty() || want == c.name) {
      c.f();
      ++ran;
    }
  std::printf("%s: %s\n", want.c_str(), bad || !ran || fake::violations ? "FAIL" : "ok");
  return bad || !ran || fake::violations;
}
