// Chunks forced past a small level budget must end where they do when levels
// are measured whole (the device and the queries of sched_measure.cpp).
#pragma GCC diagnostic push
#pragma GCC diagnostic ignored "-Wreturn-type"  // its main, under another name and not called
#define main sched_measure_main
#include "sched_measure.cpp"
#undef main
#pragma GCC diagnostic pop

namespace {

struct Run {
  std::string chunks;
  gemh::SchedStats st;
  uint64_t measured;
};

Run run(uint64_t cap, uint64_t budget, uint64_t force, uint64_t units) {
  Backend be;
  std::vector<gemh::SQuery<Buf>> qs(5);
  std::vector<gemh::SQuery<Buf> *> ptrs;
  for (size_t i = 0; i < qs.size(); ++i) {
    gemh::SQuery<Buf> &Q = qs[i];
    Q.nv = 3 + (uint32_t)i;
    Q.nb.assign(Q.nv, i % 2 ? 2 : 1);
    Q.level_rows.assign(Q.nv, 0);
    const uint64_t n0 = i ? 777 * i * i : 63;
    gemh::SLevel<Buf> L;
    L.level = 1;
    L.rows = std::make_shared<Buf>(Buf{4 * n0, n0, i + 1});
    L.nrows = n0;
    L.k = 1;
    Q.stack.push_back(std::move(L));
    ptrs.push_back(&Q);
  }
  gemh::SchedConfig cfg;
  cfg.cap = cap;
  cfg.budget = budget;
  cfg.force_chunk = force;
  cfg.max_chunk = 4ull << 20;
  cfg.max_active = 3;
  cfg.final_piece = 50000;
  cfg.measure_units = units;
  Run r;
  gemh::run_schedule(be, ptrs, cfg, &r.st);
  r.chunks = be.log;
  r.measured = be.measured;
  return r;
}

}  // namespace

int main(int argc, char **argv) {
  const uint64_t cap = std::stoull(argv[argc - 1]);
  uint64_t forced = 0;
  for (uint64_t budget : {1ull << 16, 1ull << 18, 1ull << 20, 1ull << 22})
    for (uint64_t force : {0ull, 1ull << 15, 1ull << 20, 1ull << 26}) {
      const Run whole = run(cap, budget, force, 0);
      forced += whole.st.forced;
      for (uint64_t units : {1ull, 3ull, 64ull, 4096ull}) {
        const Run r = run(cap, budget, force, units);
        if (r.chunks != whole.chunks || r.st.forced != whole.st.forced ||
            r.st.max_overshoot != whole.st.max_overshoot) {
          std::printf("budget %llu force %llu units %llu: %llu iterations, whole %llu; %llu forced, whole %llu\n",
                      (unsigned long long)budget, (unsigned long long)force, (unsigned long long)units,
                      (unsigned long long)r.st.iterations, (unsigned long long)whole.st.iterations,
                      (unsigned long long)r.st.forced, (unsigned long long)whole.st.forced);
          return 1;
        }
      }
    }
  std::printf("%llu forced\n", (unsigned long long)forced);
  if (cap >= 5000000 && !forced) return 1;
  std::printf("ok\n");
}
