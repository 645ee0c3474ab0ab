// The plan of the reference-order LU-SGS sweeps in one workgroup (sweep.h):
// passes, steps and LDS slots, formed on the host from the order alone.  A
// file of its own so that a host compiler builds it.
#pragma once

#include <hip/hip_vector_types.h>

#include <algorithm>
#include <cstddef>
#include <vector>

namespace ufx {

constexpr int SW_WAVES = 4;      // one wave per SIMD: the loads ahead take its registers
constexpr int SW_WIDTH = 64;     // nodes of a pass, lanes of a wave
constexpr int SW_THREADS = SW_WAVES * SW_WIDTH;
constexpr int SW_MAXE = 5;       // entries of a node that are loaded ahead
constexpr int SW_REC = 9;        // doubles per LDS slot: dq (4), rho, u, v, p, E + p
constexpr int SW_GREC = 10;      // doubles per stored record (the same, whole 16-byte loads)
// LDS slots of a sweep with a ring of `ring`: the ring, the fetched records
// of each wave, a record of zeros (what unused entries read); a multiple of
// 64.  The LDS holds value i of slot s at [i][s]: neighbours of consecutive
// nodes are mostly consecutive, and so are their banks.
constexpr int sw_zero_slot(int ring) { return ring + SW_THREADS; }
constexpr int sw_slots(int ring) { return (sw_zero_slot(ring) + 64) / 64 * 64; }
// When a stored record may be read.  After its update of pass p (wave p mod
// 4) a wave stores that pass's results, then loads the stream of its pass
// p + 8 and the records that pass reads.  A wave's vector memory operations
// complete in order, so its update of pass y, which waits for what it loaded
// after pass y - 8, shows its stores of pass y - 8 done, and the barrier that
// ends the step of pass y passes this on.  Records for pass p are loaded
// after the step of pass p - 8: the stores of pass p - 16 and before are
// done.  So a record that is fetched is at least SW_GAP passes old.  (One
// that a pass reads from memory itself could be 8 passes younger.)
constexpr int SW_GAP = 16;

// What the kernel's offsets hold: 32 bits for 32 bytes a node (both sweeps'
// positions), and 15 bits of a position's head for its count of entries.
constexpr size_t SW_MAX_POS = (size_t)1 << 27;
constexpr size_t SW_MAX_CNT = (1 << 15) - 1;

// Host side: the passes and slots of both sweeps.  verts: the nodes of the
// forward levels, then of the backward levels; off: offsets of the levels
// (both sweeps, into verts); per position the entries [eptr[s], eptr[s + 1])
// of nb, each a neighbour's position; out: where a position's result goes.
// A node with more neighbours beyond the ring than a pass can fetch (a hub of
// a mesh, of any number) reads those that have no slot from their stored
// records, a bit-inverted place there in `more`; never one of its first
// SW_MAXE entries, which take at most as many of its pass's SW_WIDTH slots.
// No passes: the nodes or a node's entries are more than the kernel takes,
// and the caller sweeps by level launches.
struct SweepPlan {
  std::vector<int4> pass, head;  // as SweepDev has them
  std::vector<int> far, more;
  int npass[2] = {0, 0}, nstep[2] = {0, 0};  // of the forward and the backward sweep
  int q = SW_MAXE;     // the most entries of a node, at least SW_MAXE
  bool spill = false;  // some entries are read from their stored records
};

// The least steps that the levels with offsets `off` can take (known before
// the plan).
inline size_t sweep_least_steps(const std::vector<int>& off) {
  size_t n = 0;
  for (size_t l = 0; l + 1 < off.size(); ++l)
    n += ((size_t)(off[l + 1] - off[l]) + SW_THREADS - 1) / SW_THREADS;
  return n;
}

inline SweepPlan sweep_plan(int n, const std::vector<int>& off_f, const std::vector<int>& off_b,
                            const std::vector<size_t>& eptr, const std::vector<int>& nb,
                            const std::vector<int>& out, int ring) {
  static_assert(SW_MAXE == 5 && SW_MAXE <= SW_WIDTH, "what a head holds; and has slots");
  SweepPlan p;
  const size_t np = 2 * (size_t)n;
  if (np > SW_MAX_POS) return p;
  size_t q = SW_MAXE;
  for (size_t s = 0; s < np; ++s) q = std::max(q, eptr[s + 1] - eptr[s]);
  if (q > SW_MAX_CNT) return p;
  p.q = (int)q;
  const int zero = sw_zero_slot(ring);
  p.head.resize(np);
  p.more.assign((q - SW_MAXE) * np, zero);
  for (int dir = 0; dir < 2; ++dir) {
    const std::vector<int>& off = dir == 0 ? off_f : off_b;
    const int base = dir == 0 ? 0 : n;  // ring slots count from the sweep's first position
    const int at0 = (int)p.pass.size();
    int step = -1;
    for (size_t l = 0; l + 1 < off.size(); ++l) {
      if (off[l + 1] > off[l]) ++step;
      for (int b = off[l]; b < off[l + 1];) {
        // as many nodes of the level as fit: at most SW_WIDTH, and at most
        // SW_WIDTH fetched records, unless the first node alone has more.
        // The ring is short of what the passes of the same step write.
        const int at = (int)p.pass.size(), most = std::min(off[l + 1] - b, SW_WIDTH);
        const int lim = b + SW_THREADS - ring;
        // a wave's passes are in different steps
        if (at - at0 >= SW_WAVES) step = std::max(step, p.pass[at - SW_WAVES].z + 1);
        p.far.resize((size_t)(at + 1) * SW_WIDTH, -1);
        int* far = &p.far[(size_t)at * SW_WIDTH];
        int cnt_far = 0, m = 0, mc = 0;
        for (; m < most; ++m) {
          const size_t s = (size_t)b + m;
          int need = 0;
          for (size_t j = eptr[s]; j < eptr[s + 1]; ++j) need += nb[j] < lim;
          if (cnt_far + need > SW_WIDTH && m > 0) break;
          const int cnt = (int)(eptr[s + 1] - eptr[s]);
          int sl[SW_MAXE] = {zero, zero, zero, zero, zero};
          for (int k = 0; k < cnt; ++k) {
            const int o = nb[eptr[s] + k];
            int at_slot;
            if (o >= lim) {
              at_slot = (o - base) % ring;
            } else {
              p.head[o].z |= (int)0x80000000;
              if (cnt_far < SW_WIDTH) {
                at_slot = ring + (at - at0) % SW_WAVES * SW_WIDTH + cnt_far;
                far[cnt_far++] = o - base;
              } else {
                at_slot = ~(o - base);
                p.spill = true;
              }
            }
            if (k < SW_MAXE) sl[k] = at_slot;
            else p.more[(size_t)(k - SW_MAXE) * np + s] = at_slot;
          }
          p.head[s] = make_int4(sl[0] | sl[1] << 16, sl[2] | sl[3] << 16, sl[4] | cnt << 16, out[s]);
          mc = std::max(mc, cnt);
        }
        p.pass.push_back(make_int4(b, m, step, mc));
        b += m;
      }
    }
    // whole groups of eight passes (two to each wave; the kernel's loop has
    // no exit inside one): the last pass again, whose inputs are still in place
    while (((int)p.pass.size() - at0) % (2 * SW_WAVES) != 0) {
      int4 w = p.pass.back();
      w.z = ++step;
      p.pass.push_back(w);
      p.far.resize(p.pass.size() * SW_WIDTH, -1);
    }
    p.npass[dir] = (int)p.pass.size() - at0;
    p.nstep[dir] = step + 1;
  }
  return p;
}

}  // namespace ufx
