// CPU build of the SOA loop's two forms (chain_device.hpp) for
// tests/test_soa_run.py: the general sub-step dev::soa_tick<false> and the
// one on bounded inputs, dev::soa_run_tick.  Test infrastructure only.
#include <cmath>

#include "../../mam4xx_amd/csrc/chain_device.hpp"

using namespace mam4x;

// in: n rows of SOAG, 4 SOA, 4 uptake rates, 4 oxygenated POM, g0; out: n rows
// of SOAG, 4 SOA, mean SOAG, sub-steps.  fast: the bounded form, whose ok[i]
// says whether its result stands.
extern "C" void soa_run_host(int n, double dtfull, int fast, const double *in, double *out,
                             int *ok) {
  for (int i = 0; i < n; ++i) {
    const double *p = in + 14 * i;
    double *o = out + 7 * i;
    dev::SoaIn<double> c = {p[0], {p[1], p[2], p[3], p[4]}, {p[5], p[6], p[7], p[8]},
                            {p[9], p[10], p[11], p[12]}, p[13]};
    if (fast) {
      dev::SoaRun<4> s;
      dev::soa_run_init(s, c, dtfull);
      while (s.run) dev::soa_run_tick(s, dtfull);
      ok[i] = s.low >= dev::kSoaLowMin;
      o[0] = s.g;
      for (int m = 0; m < 4; ++m) o[1 + m] = s.a[m];
      o[5] = dev::kmax(0.0, s.avg / s.dtsum);
      o[6] = s.niter;
    } else {
      dev::SoaState<double> s;
      dev::soa_init(s, c);
      while (dev::soa_tick<false>(s, dtfull)) {
      }
      ok[i] = 1;
      o[0] = s.g;
      for (int m = 0; m < 4; ++m) o[1 + m] = s.a[m];
      o[5] = dev::soa_gavg(s);
      o[6] = s.niter;
    }
  }
}
