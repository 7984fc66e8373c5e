// Replays the readout's walk over the bricks of particle grids with the
// kernel's own index code (flowpm_amd/csrc/brick_index.h): four rounds of 512
// threads, as k_readout_box makes them.  Every offset has to be that of the
// particle, and that of the brick's first particle past the brick's end, so
// that no load leaves the brick.
#include <cstdio>
#include <cstdlib>

#include "../../flowpm_amd/csrc/brick_index.h"

using namespace pmx;

static long check(int gx, int gy, int gz) {
  constexpr int T = 512;
  const BrickGrid g = make_brick_grid(gx, gy, gz, 1);
  long bad = 0, past = 0;
  for (int bid = 0; bid < g.nbricks; ++bid) {
    int q0[3], cnt[3];
    brick_block(g, bid, q0, cnt);
    const BrickWalk w = brick_walk(g, cnt, T);
    const int n = cnt[0] * cnt[1] * cnt[2];
    const long long o0 = ((long long)q0[0] * gy + q0[1]) * gz + q0[2];
    auto want = [&](int t) -> unsigned {
      if (t >= n) return 0u;
      const int lz = t % cnt[2], q = t / cnt[2], lx = q % cnt[0],
                ly = q / cnt[0];
      return (unsigned)((lx * gy + ly) * gz + lz);
    };
    for (int parts = 1; parts <= 4; parts *= 2)
      for (int part = 0; part < parts; ++part)
        for (int tid = 0; tid < T; ++tid) {
          const int ua = part * 4 / parts, ub = ua + 4 / parts;
          unsigned o = walk_at(w, tid + ua * T);
          for (int u = ua; u < ub; ++u) {
            const int t = tid + u * T;
            bad += o != want(t);
            past += o0 + o >= (long long)gx * gy * gz;
            o = walk_next(w, o, t);
          }
        }
  }
  std::printf("%d x %d x %d: %d bricks, %ld wrong, %ld past the end\n", gx, gy,
              gz, g.nbricks, bad, past);
  return bad;
}

int main() {
  long bad = 0;
  const int cubes[] = {8, 12, 16, 20, 24, 32, 40, 48, 60, 64, 80, 96, 100,
                       120, 128, 160, 200, 240};
  for (int n : cubes) bad += check(n, n, n);
  bad += check(40, 24, 60) + check(20, 24, 12) + check(64, 80, 48) +
         check(100, 24, 40) + check(4, 200, 8) + check(8, 1000, 16);
  std::puts(bad ? "WRONG" : "ok");
  return bad != 0;
}
