// The SOA work queue's counters and how a wave claims entries from it.
#pragma once

#include "../../include/mam4x.h"

#if defined(__HIP__)
#include <hip/hip_runtime.h>
#else
// plain C++ compilers see the device annotations as no-ops (the test suite
// builds this file for the CPU: tests/cpp/claims_host.cpp)
#ifndef __device__
#define __device__
#define __forceinline__ inline
#endif
#endif

namespace mam4x {

constexpr int kNBucket = 24;  // half-octave cost buckets: 2 log2(1 + predicted sub-steps)
#ifndef MAM4X_QUEUE_CHUNK
#define MAM4X_QUEUE_CHUNK 64
#endif
constexpr int kChunk = MAM4X_QUEUE_CHUNK;  // default queue entries a wave takes per refill
// Waves whose first chunk comes from buckets >= kLongBucket (predicted >= ~180
// sub-steps) raise their issue priority: a cell's sub-steps are a serial
// chain, so the longest cells set the kernel's critical path and should not
// yield issue slots to the bulk.
constexpr int kLongBucket = 15;
// Refills cost a device-scope atomic on a queue counter, and those atomics
// serialise across the device (tens of ns each), so the kernel keeps their
// number down: every wave's first chunk is assigned statically (chunk = wave
// index: the longest cells go to the first-dispatched, oldest waves), and the
// cells of buckets < kShortBucket (predicted <= ~30 sub-steps) form a second
// part of the queue taken kShortChunk at a time -- holding a few short cells
// back in a busy wave costs little.
#ifndef MAM4X_SHORT_BUCKET
#define MAM4X_SHORT_BUCKET 10
#endif
#ifndef MAM4X_SHORT_CHUNK
#define MAM4X_SHORT_CHUNK 256
#endif
constexpr int kShortBucket = MAM4X_SHORT_BUCKET;
constexpr int kShortChunk = MAM4X_SHORT_CHUNK;
constexpr int kSeg = 32;      // records staged at a time

struct QueueCtl {
  unsigned hist[kNBucket];  // cells per bucket
  unsigned fill[kNBucket];  // scatter cursor per bucket
  unsigned head;            // next free slot of the long part of the queue
  unsigned pad[31];         // the two counters on separate cache lines
  unsigned shead;           // next free slot of the short part
};

// The queue's granularity (mam4x_config.soa_chunk, soa_short_chunk,
// soa_short_bucket; performance only): queue entries a wave takes per refill
// from the long part and from the short part, the first bucket of the long
// part, and the first bucket whose waves raise their issue priority.
struct QueueShape {
  int chunk, short_chunk, short_bucket, long_bucket;
};

// Claims are counted in 32 bits, and every wave's last ones run past the end of
// the queue: with at most 2^13 waves (32 a CU) and 2^31 cells no sum passes
// 2^32, up to 2^18 entries a claim.  (2^20 entries a claim and 2^12 waves wrap
// the counter, and cells are handed out twice.)
constexpr int kMaxClaim = 1 << 18;

static inline QueueShape queue_shape(const mam4x_config &c) {
  const auto claim = [](int n) { return n < kMaxClaim ? n : kMaxClaim; };
  QueueShape q;
  q.chunk = claim(c.soa_chunk > 0 ? c.soa_chunk : kChunk);
  q.short_chunk = claim(c.soa_short_chunk > 0 ? c.soa_short_chunk : kShortChunk);
  q.short_bucket = c.soa_short_bucket > 0 ? c.soa_short_bucket : kShortBucket;
  q.long_bucket = kLongBucket;
  return q;
}

#if defined(__HIP__)
__device__ __forceinline__ unsigned fetch_add(unsigned *p, unsigned n) { return atomicAdd(p, n); }
__device__ __forceinline__ unsigned first_lane(unsigned v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_readfirstlane(v);
#else
  return v;
#endif
}
#else
inline unsigned fetch_add(unsigned *p, unsigned n) {
  const unsigned v = *p;
  *p += n;
  return v;
}
inline unsigned first_lane(unsigned v) { return v; }
#endif
__device__ __forceinline__ unsigned least(unsigned a, unsigned b) { return a < b ? a : b; }

// The wave's source of queue entries: a claimed range, the next claim's
// atomic in flight.  The long part of the queue first (the first claim of
// every wave static: claim = wave index), then the short part.
struct Claims {
  unsigned beg, end;  // what is left of the claimed range (wave-uniform)
  unsigned pend;      // lane 0: the outstanding atomic's result
  bool longs, over;
  unsigned nq, nsplit, chunk, short_chunk, first;
  QueueCtl *ctl;
  int lane;
  __device__ __forceinline__ void ask() {
    if (lane == 0)
      pend = fetch_add(longs ? &ctl->head : &ctl->shead, longs ? chunk : short_chunk);
  }
  __device__ __forceinline__ void init(unsigned wid, unsigned nwave) {
    first = nwave * chunk;
    longs = true;
    over = false;
    pend = 0;
    beg = least(wid * chunk, nsplit);
    end = least(beg + chunk, nsplit);
    if (first >= nsplit) longs = false;  // the static claims cover the long part
    if (!longs && nsplit == nq)
      over = beg == end;
    else
      ask();
  }
  // the next range of at most kSeg entries (empty: none left)
  __device__ __forceinline__ void next(unsigned &b, unsigned &e) {
    while (beg == end && !over) {
      if (!longs && nsplit == nq) {
        over = true;
        break;
      }
      const unsigned v = first_lane(pend) + (longs ? first : nsplit);
      const unsigned lim = longs ? nsplit : nq;
      if (v < lim) {
        beg = v;
        end = least(v + (longs ? chunk : short_chunk), lim);
        ask();
      } else if (longs) {
        longs = false;
        if (nsplit < nq) ask();
      } else {
        over = true;
      }
    }
    b = beg;
    e = least(beg + kSeg, end);
    beg = e;
  }
};

}  // namespace mam4x
