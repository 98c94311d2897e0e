// The scheduler with levels measured in parts (SchedConfig::measure_units) must
// hand the backend the same chunks as with levels measured whole, over a
// simulated device: levels are row counts, output bounds and survivors come
// from a hash of (level, unit).
#include <cstdio>
#include <memory>
#include <string>
#include <vector>

#include "vsched.h"

namespace {

uint64_t mix(uint64_t x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  return x ^ (x >> 31);
}

struct Buf {
  uint64_t bytes = 0, nrows = 0, id = 0;
};

struct Backend {
  using Buf = ::Buf;
  std::string log;          // chunks in order
  uint64_t measured = 0;    // units
  static uint64_t buf_bytes(const Buf &b) { return b.bytes; }
  std::shared_ptr<Buf> alloc(uint64_t bytes) { return std::make_shared<Buf>(Buf{bytes, 0, 0}); }
  std::shared_ptr<Buf> shrink(const std::shared_ptr<Buf> &f, uint64_t bytes) {
    f->bytes = bytes;
    return f;
  }
  static uint64_t bound(const Buf &b, uint64_t u) {
    const uint64_t h = mix(b.id * 1000003 + u);
    return (b.nrows - u * 64 < 64 ? b.nrows - u * 64 : 64) * (h % 97 == 0 ? 3000 : h % 4);
  }
  void length_pass(const std::vector<gemh::SItem<Buf>> &items, std::vector<std::vector<uint64_t>> *prefix) {
    prefix->clear();
    for (const auto &x : items) {
      std::vector<uint64_t> P{0};
      for (uint64_t u = x.row_begin / 64; u * 64 < x.row_end; ++u) P.push_back(P.back() + bound(*x.rows, u));
      measured += P.size() - 1;
      prefix->push_back(std::move(P));
    }
  }
  void extend(const std::vector<gemh::SItem<Buf>> &wr, const std::vector<gemh::SItem<Buf>> &fin,
              std::vector<uint64_t> *got_wr, std::vector<uint64_t> *got_fin) {
    auto walk = [&](const gemh::SItem<Buf> &x, char kind) {
      uint64_t n = 0;
      for (uint64_t u = x.row_begin / 64; u * 64 < x.row_end; ++u) n += bound(*x.rows, u) / 2;
      log += kind + std::to_string(x.q) + "." + std::to_string(x.level) + ":" + std::to_string(x.row_begin) + "-" +
             std::to_string(x.row_end) + " ";
      return n;
    };
    got_wr->clear();
    got_fin->clear();
    for (const auto &x : wr) {
      got_wr->push_back(walk(x, 'w'));
      x.out->nrows = got_wr->back();
      x.out->id = mix(x.rows->id + x.row_begin);
    }
    for (const auto &x : fin) got_fin->push_back(walk(x, 'f'));
  }
  void on_iteration(uint64_t, size_t, uint64_t, uint64_t) {}
  bool restart(uint32_t) { return false; }
  bool prolong(uint32_t) { return false; }
  bool ready(uint32_t) { return true; }
  void wait_ready(uint32_t) {}
  std::shared_ptr<void> swap_out(const Buf &, uint64_t) { return {}; }
  std::shared_ptr<Buf> swap_in(const std::shared_ptr<void> &, uint64_t) { return {}; }
  void admit(uint32_t) {}
};

}  // namespace

int main(int argc, char **argv) {
  const uint64_t cap = std::stoull(argv[argc - 1]);
  std::string first, counts0;
  uint64_t whole = 0;
  for (uint64_t mu : {0ull, 1ull, 3ull, 64ull, 4096ull}) {
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
    cfg.budget = 64ull << 20;
    cfg.max_chunk = 4ull << 20;
    cfg.max_active = 3;
    cfg.final_piece = 50000;
    cfg.measure_units = mu;
    gemh::SchedStats st;
    gemh::run_schedule(be, ptrs, cfg, &st);
    std::string counts;
    for (auto &Q : qs) counts += std::to_string(Q.count) + (Q.saturated ? "s " : " ");
    if (!mu) {
      first = be.log;
      counts0 = counts;
      whole = be.measured;
      std::printf("%zu bytes of chunks, %llu units, %s\n", first.size(), (unsigned long long)whole, counts.c_str());
    } else if (be.log != first || counts != counts0) {
      std::printf("units %llu: other chunks, %s\n", (unsigned long long)mu, counts.c_str());
      return 1;
    } else if (mu == 64 && cap < 10000000 && be.measured >= whole) {
      std::printf("units %llu: %llu measured, %llu whole\n", (unsigned long long)mu, (unsigned long long)be.measured,
                  (unsigned long long)whole);
      return 1;
    }
  }
  std::printf("ok\n");
}
