// CPU build of the work queue's claims (queue_claims.hpp) for
// tests/test_queue_claims.py.  Test infrastructure only.
#include "../../mam4xx_amd/csrc/queue_claims.hpp"

#include <vector>

using namespace mam4x;

// nwave waves take entries in turn from a queue of nq, the first nsplit of them
// its long part, until it is over for all; seen[i] counts how often entry i was
// handed out.  Returns the largest range taken at once.
extern "C" int claims_host(int soa_chunk, int soa_short_chunk, unsigned nwave, unsigned nq,
                           unsigned nsplit, unsigned char *seen) {
  mam4x_config c{};
  c.soa_chunk = soa_chunk;
  c.soa_short_chunk = soa_short_chunk;
  const QueueShape qs = queue_shape(c);
  QueueCtl ctl{};
  std::vector<Claims> waves(nwave);
  for (unsigned w = 0; w < nwave; ++w) {
    Claims &cl = waves[w];
    cl.nq = nq;
    cl.nsplit = nsplit;
    cl.chunk = (unsigned)qs.chunk;
    cl.short_chunk = (unsigned)qs.short_chunk;
    cl.ctl = &ctl;
    cl.lane = 0;
    cl.init(w, nwave);
  }
  unsigned most = 0;
  for (bool any = true; any;) {
    any = false;
    for (Claims &cl : waves) {
      unsigned b, e;
      cl.next(b, e);
      if (b == e) continue;
      any = true;
      if (e > nq || b > e) return -1;
      most = e - b > most ? e - b : most;
      for (unsigned i = b; i < e; ++i) seen[i] = (unsigned char)(seen[i] < 255 ? seen[i] + 1 : 255);
    }
  }
  return (int)most;
}
