// Host check of the flexible chains chosen for least waiting time
// and with the work around them (csrc/flex_chain.hpp, FlexWait): the replay of
// flex_chain_host.cpp over small, large and chip-filling batches, and the threads a member gets: at least as many as
// for least work, and at most the butterflies or 16.
#define main flex_chain_main
#include "flex_chain_host.cpp"
#undef main

int main() {
  long count = 0, more = 0;
  const int cfg[][3] = {{20, 512, 8}, {20, 1024, 8}, {16, 256, 16}, {16, 512, 16}};
  for (const auto &c : cfg)
    for (int64_t n = 2; n <= 2048; ++n) {
      FlexDesc least, d;
      if (!flex_choose(n, c[0], c[1], c[2], 160 * 1024, 0, &least)) continue;
      const FlexWait full = {0, 0, c[2] == 8 ? 20. : 8., 0, false};
      CHECK(flex_choose(n, c[0], c[1], c[2], 160 * 1024, 0, &d, &full));
      check(n, c[0], c[1], c[2], d);
      for (int64_t members : {1, 40, 1000, 30000})
        for (int kind = 0; kind < 3; ++kind) {
          const FlexWait w = {members, c[2] == 8 ? 131072 : 65536, kind == 1 ? 130. : 55.,
                              kind == 2 ? 300. : 0., kind > 0};
          CHECK(flex_choose(n, c[0], c[1], c[2], 160 * 1024, 0, &d, &w));
          check(n, c[0], c[1], c[2], d);
          int64_t most = w.spare ? 16 : 1;
          for (int s = 0; s < d.ns; ++s) most = d.st[s].nb > most ? d.st[s].nb : most;
          CHECK(d.tpt <= most);
          if (members == 1 && kind == 1) {
            CHECK(d.tpt >= least.tpt);
            more += d.tpt > least.tpt;
          }
          ++count;
        }
    }
  std::printf("%ld chains, %ld with more threads\n", count, more);
  return 0;
}
