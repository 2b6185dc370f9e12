// Which workgroup of a launch does what: block index -> (head, job within the head), and the grid that goes with it.  Plain
// arithmetic, on the host and in the kernels.
//
// Every workgroup of every attention kernel begins with this, in front of its first load, and a compute unit has no divider: a
// division of two launch arguments is a chain of some 30 dependent instructions, one of 64-bit numbers of 120, and a start
// had ten of them (770 instructions in front of the first tile load of ring_split_kernel).  So the divisors come with their
// reciprocals, made once per launch, and a quotient is a multiplication and a shift: 300 instructions, and 0.4 to 0.5 us less a
// workgroup (us a launch before and after, one behind the other: 4 ranks x 128 tokens, d = 64 6.46, 6.00; 4 heads x 256, d = 128 7.79,
// 7.31; the 19 steps of a rank of 12 heads x 300 rows 128, 122).
#pragma once
#include <stdint.h>
#ifdef __HIPCC__
#define RINGATTN_BOTH __host__ __device__ __forceinline__
#else
#define RINGATTN_BOTH inline
#endif

namespace ringattn {

// n / d = (n * mul) >> shift for 0 <= n < 2^31.  With 2^(l-1) < d <= 2^l and mul = ceil(2^(31+l) / d), mul d exceeds 2^(31+l) by
// e < d, and the product exceeds n / d by n e / (d 2^(31+l)) < 1 / d: too little to reach the next integer.
struct Divisor {
  unsigned mul, shift;
};
inline Divisor divisor(unsigned d) {
  unsigned l = 0;
  while (l < 31 && (1u << l) < d) ++l;
  return Divisor{(unsigned)((((uint64_t)1 << (31 + l)) + d - 1) / d), 31 + l};
}
RINGATTN_BOTH int quotient(int n, Divisor d) { return (int)(((uint64_t)(unsigned)n * d.mul) >> d.shift); }

// An XCD's jobs: those of `lead_heads` heads of its own one head after the other, then those of its last tail_heads heads together
// with its part of the heads that are shared (job_map says why).
struct JobMap {
  int per_head;       // jobs of a head
  int full, rem;      // heads = 8 full + rem
  int tail_heads;
  int lead, own;      // jobs of the heads that run one after the other; of the others of its own
  int log_sets;       // the shared heads fall to 2^log_sets sets of XCDs ...
  int shared_heads;   // ... so many to each
  int most;           // shared jobs of the first XCD of a set: the others have as many, or one fewer
  unsigned pace[2];   // of 2^32 jobs that are not in the lead, how many are shared (with `most` of them, with one fewer)
  Divisor by_head, by_tail, by_shared;
};

// `masked`: the q tiles of a head differ in length, longest first.  Heads are dealt to the eight XCDs and run one after the
// other; what is left of them, heads mod 8, is shared out tile by tile: with rem of them, gcd(8, rem) sets of XCDs take rem / gcd
// heads each and split their tiles round-robin, so that one head (or any number) still fills all XCDs.  Under the mask the last
// heads of an XCD, as many as make up 64 jobs (two for each of its 32 compute units), and its part of the shared ones go
// through their tiles together: one after the other, the longest tile of the last head would start when little else is left.
// Returns the workgroups of the launch: 8 x the jobs of the busiest XCD.
inline int64_t job_map(JobMap& m, int heads, int64_t per_head, bool masked) {
  m = JobMap{};
  m.per_head = (int)per_head;
  m.full = heads / 8;
  m.rem = heads & 7;
  if (masked && per_head > 0) {
    const int64_t g = (64 + per_head - 1) / per_head;
    m.tail_heads = (int)(g < m.full ? g : m.full);
  }
  m.lead = (int)((m.full - m.tail_heads) * per_head);
  m.own = (int)(m.tail_heads * per_head);
  int64_t per_xcd = m.full * per_head;
  if (m.rem) {
    const int sets = m.rem & -m.rem;
    m.log_sets = sets == 4 ? 2 : sets - 1;
    m.shared_heads = m.rem / sets;
    const int64_t all = m.shared_heads * per_head;
    m.most = (int)((all * sets + 7) / 8);
    per_xcd += m.most;
    for (int i = 0; i < 2; ++i) {  // (rounded up: after own + shared jobs exactly `shared` of them have been shared ones)
      const int64_t shared = m.most - i;
      m.pace[i] = m.own > 0 && shared > 0 ? (unsigned)((((uint64_t)shared << 32) + (uint64_t)(m.own + shared) - 1) / (uint64_t)(m.own + shared)) : 0;
    }
  }
  m.by_head = divisor(m.per_head > 0 ? m.per_head : 1);
  m.by_tail = divisor(m.tail_heads > 0 ? m.tail_heads : 1);
  m.by_shared = divisor(m.shared_heads > 0 ? m.shared_heads : 1);
  return 8 * per_xcd;
}

// The w-th job of XCD `xcd`: which head, and which of its jobs.  False for the holes of the grid.
RINGATTN_BOTH bool job_of(const JobMap& m, bool masked, int xcd, int w, int& head, int& job) {
  if (w < m.lead) {
    const int i = quotient(w, m.by_head);
    head = 8 * i + xcd;
    job = w - i * m.per_head;
    return true;
  }
  int p = w - m.lead, from_shared = 0;
  if (m.rem) {
    const int log_share = 3 - m.log_sets, share = 1 << log_share, sub = xcd >> m.log_sets;
    const int shared = (m.shared_heads * m.per_head - sub + share - 1) >> log_share;  // this XCD's jobs of the shared heads
    if (p >= m.own + shared) return false;
    // the p-th of both lists merged in proportion
    const uint64_t pace = m.own == 0 ? (uint64_t)1 << 32 : m.pace[shared == m.most ? 0 : 1];
    from_shared = (int)((uint64_t)(unsigned)p * pace >> 32);
    if ((int)((uint64_t)(unsigned)(p + 1) * pace >> 32) > from_shared) {
      const int j = (from_shared << log_share) + sub;
      const int i = masked ? quotient(j, m.by_shared) : quotient(j, m.by_head);
      const int rest = j - i * (masked ? m.shared_heads : m.per_head);
      job = masked ? i : rest;
      head = 8 * m.full + (xcd & ((1 << m.log_sets) - 1)) + ((masked ? rest : i) << m.log_sets);
      return true;
    }
  } else if (p >= m.own) {
    return false;
  }
  p -= from_shared;
  job = quotient(p, m.by_tail);
  head = 8 * (m.full - m.tail_heads + p - job * m.tail_heads) + xcd;
  return true;
}

}  // namespace ringattn
