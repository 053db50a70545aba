// Host build of the batched u2p's per-point function (calc_primitives_point
// of koral_amd/csrc/dev_cell.hpp) over a batch of points, counting how often
// it reads a point's state and metric.
//
// usage: u2p_point_check BATCH OUT   (BATCH: params, n, pp[n][nv], uu[n][nv],
// g20[n][20], G20[n][20]; OUT: pp[n][nv], uu[n][nv], then per point int32 ret,
// entropy, entropy2, hd and rad flags, reads of the state, reads of the metric)
#define KD_HOST_CHECK 1
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "dev_cell.hpp"

using namespace kd;

static void rd(FILE *f, void *p, size_t n)
{
  if (fread(p, 1, n, f) != n) {
    fprintf(stderr, "u2p_point_check: short read\n");
    exit(2);
  }
}

template <int MAG, int RAD>
static void all(const koral_params &P, long n, std::vector<double> &pp, std::vector<double> &uu,
                const std::vector<double> &g20, const std::vector<double> &G20, std::vector<int> &out)
{
  constexpr int NV = Lay<MAG, RAD>::NV;
#pragma omp parallel for schedule(dynamic, 64)
  for (long i = 0; i < n; i++) {
    int states = 0, metrics = 0;
    double p[NV], u[NV];
    CpFlags fl;
    const int r = calc_primitives_point<MAG, RAD>(
        P,
        [&](Geom &g) {
          metrics++;
          load_geom(g, [&](int c) { return g20[20 * i + c]; }, [&](int c) { return G20[20 * i + c]; });
        },
        [&](double *us, double *ps) {
          states++;
          for (int v = 0; v < NV; v++) {
            ps[v] = pp[NV * i + v];
            us[v] = uu[NV * i + v];
          }
        },
        u, p, fl);
    for (int v = 0; v < NV; v++) {
      pp[NV * i + v] = p[v];
      uu[NV * i + v] = u[v];
    }
    const int o[7] = {r, fl.entr, fl.entr2, fl.hd, fl.rad, states, metrics};
    for (int k = 0; k < 7; k++) out[7 * i + k] = o[k];
  }
}

int main(int argc, char **argv)
{
  if (argc < 3) return 2;
  FILE *f = fopen(argv[1], "rb");
  if (!f) return 2;
  koral_params P;
  long n = 0;
  rd(f, &P, sizeof P);
  rd(f, &n, sizeof n);
  const int nv = P.nv;
  std::vector<double> pp(nv * n), uu(nv * n), g20(20 * n), G20(20 * n);
  rd(f, pp.data(), 8 * pp.size());
  rd(f, uu.data(), 8 * uu.size());
  rd(f, g20.data(), 8 * g20.size());
  rd(f, G20.data(), 8 * G20.size());
  fclose(f);
  std::vector<int> out(7 * n);
  if (P.mag && P.rad)
    all<1, 1>(P, n, pp, uu, g20, G20, out);
  else if (P.mag)
    all<1, 0>(P, n, pp, uu, g20, G20, out);
  else if (P.rad)
    all<0, 1>(P, n, pp, uu, g20, G20, out);
  else
    all<0, 0>(P, n, pp, uu, g20, G20, out);
  FILE *o = fopen(argv[2], "wb");
  if (!o) return 2;
  fwrite(pp.data(), 8, pp.size(), o);
  fwrite(uu.data(), 8, uu.size(), o);
  fwrite(out.data(), 4, out.size(), o);
  fclose(o);
  return 0;
}
