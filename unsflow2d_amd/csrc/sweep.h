// The reference-order LU-SGS sweeps of both solvers in one workgroup
// (gfx950).  Included by cc_kernels.h and nc_kernels.h.
//
// A sequential sweep (CCFVM/lusgs.F90:244-310, NCFVM/lusgs.f90:46-122) updates
// the nodes in number order, each from the neighbours already swept.  Nodes
// grouped by dependency level update concurrently and the sweep equals the
// reference's, but the levels are a chain: some hundred to some thousand of
// them, each of a hundred nodes or so.  Between the levels of a chain only
// one CU can hand results over in less than a microsecond (its LDS; another
// CU sees them after a write to L2 or, on another XCD, to memory), so the
// whole sweep runs in one workgroup and what a level costs is latency: the
// reads that a node's update waits for, its arithmetic and the barrier.
// Therefore
//   - everything that does not depend on the sweep is written beforehand in
//     the sweep's order by a parallel pass (position-major, so that a wave's
//     loads are whole lines) and loaded into registers passes ahead;
//   - a node leaves what its neighbours need of it -- the increment, and the
//     density, velocities, pressure and total enthalpy of its new state, so
//     that their divisions are done once per node and not once per edge --
//     in an LDS ring of the last SW_RING positions;
//   - a neighbour further back (1 to 3 % of the reads on an O-grid of 125 000
//     vertices, 6 to 10 % on 500 000, a third on two million) is fetched from
//     its stored record passes ahead into a second LDS area, at a slot that
//     the host has assigned: inside a pass every read is an LDS read (but for
//     nodes with more neighbours further back than a pass can fetch);
//   - the four waves take the passes in turn: while one (or, in a wide level,
//     several) updates its nodes, the others store the results of their last
//     pass and issue the loads of their next ones, which would otherwise stand
//     in the chain;
//   - the barrier waits for LDS only, so the loads ahead stay in flight.
// A pass is a level, or a piece of a level of at most SW_WIDTH nodes; a step
// is the passes between two barriers.
//
// Measured per sweep, forward / backward.  The CC solver on 40 000 triangles
// (563 levels, 568 steps): 350 / 412 us, 0.62 and 0.73 us a step, where the
// level launches took 7.2 us each, 4 ms a sweep.  The NC solver on 125 000
// vertices (1240 steps): 1444 / 1496 us, 1.2 us a step, where one workgroup
// of 1024 threads with an LDS ring of dq alone, which formed each neighbour's
// new state again at every edge, took 4350 us.  A whole iteration takes 3.0,
// 12.5 and 61 ms on 125 000, 500 000 and two million vertices (2.4 steps a
// level there), where that one took 8.6, 25.5 and 71.7; 9.8 and 41.8 ms on
// 500 000 and two million cells, where the level launches took 37 and 92.
// Half of a step is the
// arithmetic of one wave (an NC node is some 600 double precision
// instructions of four cycles), the rest LDS latency and the barrier; the
// bytes (about 1.2 KB a node) would take a tenth.  Tried and slower: two
// groups of 128 threads in turn (371 / 436 and 1647 / 1726 us), records as
// structures in LDS (their reads conflict: 2808 us), the loads of a pass
// under branches of its entry counts (the compiler then waits for all of
// them).
#pragma once

#include <hip/hip_runtime.h>

#include "sweep_plan.h"

namespace ufx {

// Device side of a plan.  Positions: the forward sweep's nodes in its order,
// then the backward sweep's; np = 2 nodes.  rows: the most entries of a node,
// at least 3.
struct SweepDev {
  int np = 0;
  const int4* pass = nullptr;  // first position, count, its step, most entries of a node
  const int* far = nullptr;    // [passes][SW_WIDTH] position whose record the lane fetches, or -1
  const int4* head = nullptr;  // [np] the first five entries' LDS slots (16 bits each); then in z
                               // the entry count << 16 and the sign bit if the node's record is
                               // read from memory by some pass; in w where its result goes (forward: the
                               // node's place in the backward order; backward: the node)
  const int* more = nullptr;   // [rows - 5][np] LDS slot of each entry past the fifth, or
                               // bit-inverted the place of its stored record
  const int2* pe = nullptr;    // [rows][np] (edge, neighbour) for the preparing pass
  const int* node = nullptr;   // [np] node of each position
  double2* ent = nullptr;      // [rows][S::NE][np] the entries' data
  double2* own = nullptr;      // [4][np] the node's residual negated (2), its old state (2)
  double2* diag = nullptr;     // [np] diagonal and its reciprocal
  double* fwd = nullptr;       // [nodes][4] the forward sweep's dq in backward order
  double* rec = nullptr;       // [nodes + 1][SW_GREC] stored records (by position within the sweep)
};

// ---------------------------------------------------------------- kernels
// What a sweep reads in its order: per position the node's residual (negated),
// its old state and diagonal, per entry its data (S::entry).  The
// entries' geometry is written once at set-up.
template <typename S>
__global__ __launch_bounds__(256) void k_sweep_prep(S sc, SweepDev d, const double* res,
                                                    const double* qold, const double* lam,
                                                    const int* err) {
  const int s = (int)(blockIdx.x * 256 + threadIdx.x);
  const size_t np = (size_t)d.np;
  if (s >= d.np || (err && err[0])) return;
  const int v = d.node[s];
  const double2* qo = reinterpret_cast<const double2*>(qold);
  const int cnt = (d.head[s].z >> 16) & 0x7fff;
  for (int k = 0; k < cnt; ++k) {
    const int2 pe = d.pe[(size_t)k * np + s];
    double2* en = d.ent + (size_t)k * S::NE * np + s;
    const double2 a = qo[2 * (size_t)pe.y], b = qo[2 * (size_t)pe.y + 1];
    const double q[4] = {a.x, a.y, b.x, b.y};
    sc.entry(q, 1.5 * lam[pe.x], en, np);
  }
  const double2* rr = reinterpret_cast<const double2*>(res) + 2 * (size_t)v;
  const double2 r01 = rr[0], r23 = rr[1];
  d.own[s] = make_double2(-r01.x, -r01.y);
  d.own[np + s] = make_double2(-r23.x, -r23.y);
  d.own[2 * np + s] = qo[2 * (size_t)v];
  d.own[3 * np + s] = qo[2 * (size_t)v + 1];
  const double dg = sc.diag(v);
  d.diag[s] = make_double2(dg, 1.0 / dg);
}

// What is loaded ahead of one position, and its pass.
template <int ME, int NE>
struct SweepStage {
  int b, n, step, mc;  // uniform
  int4 head;
  double2 r01, r23, q01, q23, e[ME][NE], p01, p23, dd;
};

// Every lane of a pass loads, computes and stores, the ones past the pass's
// last node as that node again (the same values to the same places), and the
// first three entries whether nodes have them or not (rows of zeros, with the
// record of zeros): the number of memory operations of a pass is then nearly
// fixed, which is what lets a wait for older loads leave the younger ones in
// flight.
template <typename T>
__device__ __forceinline__ T sweep_ld(const T* base, unsigned bytes) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + bytes);
}
template <typename S, int ME, int DIR>
__device__ __forceinline__ void sweep_load(const SweepDev& d, int l, SweepStage<ME, S::NE>& st) {
  const size_t np = (size_t)d.np;
  // uniform bases and 32-bit lane offsets (a plan has at most SW_MAX_POS positions)
  const unsigned s = (unsigned)(st.b + min(l, st.n - 1));
  st.head = sweep_ld(d.head, s * 16);
#pragma unroll
  for (int k = 0; k < ME; ++k)
    if (k < 3 || k < st.mc)
#pragma unroll
      for (int i = 0; i < S::NE; ++i)
        st.e[k][i] = sweep_ld((const double2*)d.ent + (k * S::NE + i) * np, s * 16);
  if (DIR == 0) {
    st.r01 = sweep_ld((const double2*)d.own, s * 16);
    st.r23 = sweep_ld((const double2*)d.own + np, s * 16);
  }
  if (DIR == 1) {
    const double2* f = reinterpret_cast<const double2*>(d.fwd);
    const unsigned sf = (s - (unsigned)(np / 2)) * 32;
    st.p01 = sweep_ld(f, sf);
    st.p23 = sweep_ld(f + 1, sf);
  }
  st.q01 = sweep_ld((const double2*)d.own + 2 * np, s * 16);
  st.q23 = sweep_ld((const double2*)d.own + 3 * np, s * 16);
  st.dd = sweep_ld((const double2*)d.diag, s * 16);
}

// LDS accesses done, then the barrier; global memory operations stay in
// flight.
__device__ __forceinline__ void sweep_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// a / b from y = 1 / b correctly rounded: two of Markstein's corrections, the
// first bringing the quotient within an ulp, the second rounding it as the
// division does (IBM J. Res. Dev. 34 (1990) 111), in five dependent
// operations where the division takes about twenty.  Not finite where the
// operands are not; then the division itself.
__device__ __forceinline__ double sweep_div(double a, double b, double y) {
  double q = a * y;
  q = __builtin_fma(__builtin_fma(-b, q, a), y, q);
  return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}
__device__ __forceinline__ void sweep_div4(const double* a, double b, double y, double* o) {
  bool ok = true;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[i] = sweep_div(a[i], b, y);
    ok = ok && __builtin_isfinite(o[i]);
  }
  if (!ok)
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = a[i] / b;
}

// One sweep over npass passes (a multiple of 8) in nstep steps.  S: the
// solver's terms (term), update (update) and primitives (prims).  ME entries
// of a node are loaded ahead; TAIL 1: some have more; 2: and some of those are
// read from their stored records (SweepPlan::spill; a kernel of its own: the
// branch costs the others half a per cent).
template <typename S, int ME, int TAIL, int RING, int DIR>
__global__ __launch_bounds__(SW_THREADS, 1) void k_sweep(S sc, SweepDev d, int pass0, int npass,
                                                         int nstep, double* qc, const int* err) {
  static_assert((TAIL ? ME == SW_MAXE : ME <= SW_MAXE) && RING >= SW_THREADS + SW_GAP * SW_WIDTH,
                "records out of the ring are SW_GAP passes old");
  constexpr int NE = S::NE, NS = sw_slots(RING);
  __shared__ double lds[SW_REC * NS];
  if (err && err[0]) return;
  const int t = (int)threadIdx.x, l = t % SW_WIDTH;
  const int wave = __builtin_amdgcn_readfirstlane(t / SW_WIDTH);
  const int base = DIR == 0 ? 0 : d.np / 2, last = npass - 1;
  const double2* recs = reinterpret_cast<const double2*>(d.rec);
  int zero = 0;
  asm volatile("" : "+v"(zero));  // (per lane: vector loads, whose wait the LDS does not share)
  const int4* pass = d.pass + pass0 + zero;
  const int* far = d.far + (size_t)pass0 * SW_WIDTH + l;
  if (t < SW_REC) lds[t * NS + sw_zero_slot(RING)] = 0.0;
  auto uniform = [&](int4 w, SweepStage<ME, NE>& st) {
    st.b = __builtin_amdgcn_readfirstlane(w.x);
    st.n = __builtin_amdgcn_readfirstlane(w.y);
    st.step = __builtin_amdgcn_readfirstlane(w.z);
    st.mc = __builtin_amdgcn_readfirstlane(w.w);
  };
  SweepStage<ME, NE> st[2];
  double2 fr[5] = {};  // stored records of the wave's next pass but one
  int fv = -1;         // whether fr holds one
  // of the pass after that: where its records are, and its descriptor
  int fi = far[(size_t)min(wave + 2 * SW_WAVES, last) * SW_WIDTH];
  int4 w = pass[min(wave + 2 * SW_WAVES, last)];
  uniform(pass[wave], st[0]);
  uniform(pass[wave + SW_WAVES], st[1]);
#pragma unroll
  for (int i = 0; i < 2; ++i) sweep_load<S, ME, DIR>(d, l, st[i]);
  // (the waits inside the loop then count the loop's own loads)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0);
  sweep_barrier();
  int step = 0;
  auto one = [&](int p, SweepStage<ME, NE>& sg) {
    for (; step < sg.step; ++step) sweep_barrier();
    const int ll = min(l, sg.n - 1);
    double cres[4] = {0.0, 0.0, 0.0, 0.0};
    // the terms in entry order; the entries that no node of the pass has are
    // passed over
    auto add = [&](int sl, const double2* e) {
      double nb[SW_REC];
#pragma unroll
      for (int i = 0; i < SW_REC; ++i) nb[i] = lds[i * NS + sl];
      sc.term(nb, e, cres);
    };
#pragma unroll
    for (int k = 0; k < ME; ++k)
      if (k < 3 || k < sg.mc) {
        const int h = k < 2 ? sg.head.x : k < 4 ? sg.head.y : sg.head.z;
        add((k & 1) ? (int)((unsigned)h >> 16) : h & 0xffff, sg.e[k]);
      }
    if (TAIL > 0)
      for (int k = ME; k < ((sg.head.z >> 16) & 0x7fff); ++k) {
        const size_t np = (size_t)d.np, s = (size_t)sg.b + ll;
        double2 e[NE];
#pragma unroll
        for (int i = 0; i < NE; ++i) e[i] = d.ent[((size_t)k * NE + i) * np + s];
        const int sl = d.more[(size_t)(k - SW_MAXE) * np + s];
        if (TAIL == 1 || sl >= 0) {
          add(sl, e);
        } else {
          const double2* rec = recs + 5 * (size_t)~sl;
          double nb[SW_REC + 1];
#pragma unroll
          for (int i = 0; i < 5; ++i) {
            nb[2 * i] = rec[i].x;
            nb[2 * i + 1] = rec[i].y;
          }
          sc.term(nb, e, cres);
        }
      }
    const double res[4] = {sg.r01.x, sg.r01.y, sg.r23.x, sg.r23.y};
    const double pd[4] = {sg.p01.x, sg.p01.y, sg.p23.x, sg.p23.y};
    const double qo[4] = {sg.q01.x, sg.q01.y, sg.q23.x, sg.q23.y};
    double o[SW_REC + 1], q[4];
    sc.template update<DIR>(res, pd, cres, sg.dd.x, sg.dd.y, o);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = qo[i] + o[i];
    sc.prims(q, o + 4);
    o[SW_REC] = 0.0;
    {
      int sl = (sg.b - base) % RING + ll;
      sl = sl >= RING ? sl - RING : sl;
#pragma unroll
      for (int i = 0; i < SW_REC; ++i) lds[i * NS + sl] = o[i];
    }
    sweep_barrier();
    ++step;
    // beside the other waves' steps: this pass's results to memory, the
    // records of the wave's next pass into its LDS slots, and the loads for
    // the pass after that
    double2* out = reinterpret_cast<double2*>(DIR == 0 ? d.fwd : qc) + 2 * (size_t)sg.head.w;
    const double* ov = DIR == 0 ? o : q;
    out[0] = make_double2(ov[0], ov[1]);
    out[1] = make_double2(ov[2], ov[3]);
    if (sg.head.z < 0) {
      double2* rec = reinterpret_cast<double2*>(d.rec) + 5 * (size_t)(sg.b + ll - base);
#pragma unroll
      for (int i = 0; i < 5; ++i) rec[i] = make_double2(o[2 * i], o[2 * i + 1]);
    }
    if (fv >= 0) {
      double* r = lds + RING + wave * SW_WIDTH + l;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[2 * i * NS] = fr[i].x;
        r[(2 * i + 1) * NS] = fr[i].y;
      }
      r[8 * NS] = fr[4].x;
    }
    fv = p + 2 * SW_WAVES <= last ? fi : -1;
    if (fv >= 0) {
      const double2* rec = recs + 5 * (size_t)fv;
#pragma unroll
      for (int i = 0; i < 5; ++i) fr[i] = rec[i];
    }
    uniform(w, sg);
    fi = far[(size_t)min(p + 3 * SW_WAVES, last) * SW_WIDTH];
    w = pass[min(p + 3 * SW_WAVES, last)];
    sweep_load<S, ME, DIR>(d, l, sg);
  };
  for (int p = wave; p < npass; p += 2 * SW_WAVES) {
    one(p, st[0]);
    one(p + SW_WAVES, st[1]);
  }
  for (; step < nstep; ++step) sweep_barrier();
}

}  // namespace ufx
