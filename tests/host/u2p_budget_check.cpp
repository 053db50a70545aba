// The W inversion of koral_amd/csrc/dev_cell.hpp under a budget of residual
// evaluations, built for the host.
//
// usage: u2p_budget_check BATCH BUDGET OUT   (BATCH: params, n, pp[n][nv],
// uu[n][nv], g20[n][20], G20[n][20]; OUT: the n return values as int32)
#define KD_HOST_CHECK 1
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "dev_cell.hpp"

using namespace kd;

static void rd(FILE *f, void *p, size_t n)
{
  if (fread(p, 1, n, f) != n) exit(2);
}

int main(int argc, char **argv)
{
  if (argc < 4) return 2;
  FILE *f = fopen(argv[1], "rb");
  if (!f) return 2;
  koral_params P;
  long n = 0;
  rd(f, &P, sizeof P);
  rd(f, &n, sizeof n);
  constexpr int NV = Lay<1, 0>::NV;
  std::vector<double> pp(NV * n), uu(NV * n), g20(20 * n), G20(20 * n);
  rd(f, pp.data(), 8 * pp.size());
  rd(f, uu.data(), 8 * uu.size());
  rd(f, g20.data(), 8 * g20.size());
  rd(f, G20.data(), 8 * G20.size());
  fclose(f);
  std::vector<int> r(n);
  for (long i = 0; i < n; i++) {
    Geom g;
    load_geom(g, [&](int c) { return g20[20 * i + c]; }, [&](int c) { return G20[20 * i + c]; });
    r[i] = u2p_solver_W<1, 0>(P, &uu[NV * i], &pp[NV * i], g, 0, 0., nullptr, atoi(argv[2]));
  }
  FILE *o = fopen(argv[3], "wb");
  if (!o) return 2;
  fwrite(r.data(), 4, n, o);
  fclose(o);
  return 0;
}
