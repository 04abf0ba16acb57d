// Checks of mlp_dvnd's host logic against a runtime of the host (fake_hip.h).
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "fake_hip.h"
#include "mlp_gpu.h"

namespace {

#define CHECK(c, ...)                              \
  do {                                             \
    if (!(c)) {                                    \
      printf("%s:%d: ", __FILE__, __LINE__);       \
      printf(__VA_ARGS__);                         \
      printf("\n");                                \
      return 1;                                    \
    }                                              \
  } while (0)

struct Run {
  mlp_ctx* ctx = nullptr;
  std::vector<int32_t> slots;
  explicit Run(const std::vector<int>& ns) {
    mlp_ctx_create(0, &ctx);
    for (int n : ns) {
      std::vector<int32_t> x(n), y(n);
      for (int c = 0; c < n; ++c) {
        x[c] = c;
        y[c] = 7 * c % 101;
      }
      int32_t inst = -1, s = -1;
      mlp_instance_create(ctx, x.data(), y.data(), n, 1, &inst);
      mlp_slot_create(ctx, inst, &s);
      slots.push_back(s);
    }
  }
  ~Run() { mlp_ctx_destroy(ctx); }
  int dvnd(int rowmap, int max_rounds, std::vector<int32_t>* rounds = nullptr) {
    std::vector<int32_t> r(slots.size());
    const int st = mlp_dvnd(ctx, slots.data(), (int)slots.size(), rowmap, max_rounds, r.data());
    if (rounds) *rounds = r;
    return st;
  }
};

// A call repeated on the same slots replays its chunks' graphs: from its third
// time on nothing is launched one by one (a chunk is seen, then captured) and
// no graph is made.
int graphs() {
  for (const std::vector<int>& ns : {std::vector<int>{150}, {600}, {600, 150}, {600, 500, 90}})
    for (int rowmap = 0; rowmap < 2; ++rowmap)
      for (int max_rounds = 0; max_rounds <= 17; ++max_rounds) {
        rounds_of_slot = [](int) { return 30; };
        Run r(ns);
        for (int call = 0; call < 5; ++call) {
          counts = Counts();
          std::vector<int32_t> rounds;
          CHECK(r.dvnd(rowmap, max_rounds, &rounds) == MLP_OK, "%s", mlp_ctx_error(r.ctx));
          for (int32_t k : rounds) CHECK(k == (max_rounds ? max_rounds : 30), "%d rounds", k);
          if (call < 2) continue;
          CHECK(counts.instantiated == 0 && counts.eager <= counts.fills && counts.replayed > 0,
                "%d slots, n = %d, row map %d, max_rounds %d, call %d: %d launches one by one, %d graphs made, %d replayed",
                (int)ns.size(), ns[0], rowmap, max_rounds, call, counts.eager, counts.instantiated,
                counts.replayed);
        }
      }
  return 0;
}

// Rows that a failed call left incomplete cannot be read as if they were whole.
int failed_rows() {
  int left = 0;
  for (const std::vector<int>& ns : {std::vector<int>{600}, {600, 300}, {600, 90}})
    for (int max_rounds : {0, 7, 30})
      for (int at = 1; at < 40; ++at) {
        rounds_of_slot = [](int N) { return N > 400 ? 18 : 11; };
        Run r(ns);
        fail_sync = 0;
        if (r.dvnd(0, 0)) return 1;
        fail_sync = at;
        const int st = r.dvnd(0, max_rounds);
        const bool failed = fail_sync == 0;
        fail_sync = 0;
        CHECK(failed == (st != MLP_OK), "synchronisation %d: status %d", at, st);
        for (int32_t s : r.slots)
          for (int nb = 0; nb < 5; ++nb) {
            std::vector<int64_t> cost(MLP_MAX_N);
            std::vector<int32_t> i(MLP_MAX_N), j(MLP_MAX_N);
            int32_t rows = 0;
            const int got = mlp_get_rows(r.ctx, s, nb, cost.data(), i.data(), j.data(), &rows);
            left += left_out(s);
            CHECK(got == MLP_OK ? !left_out(s) : failed && got == MLP_ESTATE,
                  "max_rounds %d, synchronisation %d: rows of slot %d, neighborhood %d: %d", max_rounds, at, s, nb,
                  got);
          }
      }
  CHECK(left > 0, "no run failed with rows left out");
  return 0;
}

// A slot evaluates each neighborhood once a round, and once more after its last
// one if rows were left out there; a slot that stops in its first round (a tour
// at its optimum) does not.
int evaluations() {
  for (const std::vector<int>& ns : {std::vector<int>{150}, {600}, {600, 150}, {600, 500, 90}})
    for (int rowmap = 0; rowmap < 2; ++rowmap)
      for (int max_rounds : {0, 1, 2, 3, 4, 5, 9})
        for (int large = 1; large < 8; ++large)
          for (int small = 1; small < 8; small += 3) {
            rounds_of_slot = [=](int N) { return N > 400 ? large : small; };
            Run r(ns);
            for (int call = 0; call < 3; ++call) {
              counts = Counts();
              std::vector<int32_t> rounds;
              CHECK(r.dvnd(rowmap, max_rounds, &rounds) == MLP_OK, "%s", mlp_ctx_error(r.ctx));
              int least = 0, most = 0;
              for (int32_t k : rounds) {
                least += 5 * k;
                most += 5 * (k > 1 && k != max_rounds ? k + 1 : k);
              }
              CHECK(counts.worked >= least && counts.worked <= most,
                    "%d slots, n = %d, row map %d, max_rounds %d, %d and %d rounds: %d evaluations, expected %d to %d",
                    (int)ns.size(), ns[0], rowmap, max_rounds, large, small, counts.worked, least, most);
            }
          }
  return 0;
}

// Between mlp_timing_begin and mlp_timing_end every evaluation of a round
// launched outside a graph is timed, also of rounds that leave rows out, and no
// other: a ring of that many launches is enough.
int timed() {
  for (const std::vector<int>& ns : {std::vector<int>{150}, {600}, {600, 150}})
    for (int rowmap = 0; rowmap < 2; ++rowmap) {
      rounds_of_slot = [](int) { return 6; };
      Run r(ns);
      mlp_dvnd_config(r.ctx, 4, 0, 0);
      counts = Counts();
      CHECK(mlp_timing_begin(r.ctx, (int)ns.size() * 40) == MLP_OK && r.dvnd(rowmap, 0) == MLP_OK, "%s", mlp_ctx_error(r.ctx));
      double ms = 0;
      int32_t launches = 0;
      CHECK(mlp_timing_end(r.ctx, &ms, &launches) == MLP_OK, "%s", mlp_ctx_error(r.ctx));
      const int ran = counts.evals + counts.pruned;
      CHECK(launches == ran, "%d slots, n = %d, row map %d: %d of %d launches timed", (int)ns.size(), ns[0], rowmap,
            launches, ran);
    }
  return 0;
}

// A fused round's launch has no more workgroups than its dynamic and static LDS
// leave room for at once.
int fused_grid() {
  for (int n = 100; n < 5000; n += 50) {
    rounds_of_slot = [](int) { return 2; };
    Run r({n, n - 20});
    mlp_dvnd_fused(r.ctx, 1);
    counts = Counts();
    CHECK(r.dvnd(0, 0) == MLP_OK, "%s", mlp_ctx_error(r.ctx));
    const int fit = 256 * (int)(160 * 1024 / counts.fused_lds);
    CHECK(counts.fused_grid > 0 && counts.fused_grid <= fit, "n = %d: %d workgroups, %d fit", n, counts.fused_grid, fit);
  }
  return 0;
}

// Merges of more slots than the GPU has CUs (256) say so to their launch.
int wide_merges() {
  for (int count : {1, 255, 256, 257, 300}) {
    Run r(std::vector<int>(count, 20));
    counts = Counts();
    CHECK(mlp_eval(r.ctx, r.slots.data(), count, 3, 0, 0) == MLP_OK &&
              mlp_merge_apply(r.ctx, r.slots.data(), count, 1) == MLP_OK,
          "%s", mlp_ctx_error(r.ctx));
    CHECK(counts.wide == (count > 256) && counts.narrow == (count <= 256), "%d slots: %d wide, %d not", count,
          counts.wide, counts.narrow);
  }
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  const int bad = what == "graphs" ? graphs() : what == "failed_rows" ? failed_rows()
                  : what == "evaluations" ? evaluations()
                  : what == "timed" ? timed()
                  : what == "fused_grid" ? fused_grid()
                  : what == "wide_merges" ? wide_merges() : 2;
  if (!bad) printf("%s ok\n", what.c_str());
  return bad;
}
