// Replays the plan of the one-workgroup LU-SGS sweeps (sweep_plan.h) step by
// step on the host and checks everything that the kernel's synchronisation
// rests on.  Prints one line per sweep; exit status 1 on the first violation.
//
//   sweep_plan_replay RING grid NI NJ | cells NI NJ | shuffled NI NJ SEED |
//                     layers WIDTH COUNT BACK | hub N WHERE | limits
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <random>
#include <string>

#include "sweep_plan.h"

using namespace ufx;

static int bad(const char* what, long a = 0, long b = 0, long c = 0) {
  std::printf("violated: %s (%ld %ld %ld)\n", what, a, b, c);
  return 1;
}

struct Graph {
  int n = 0;
  std::vector<std::vector<int>> adj;
  explicit Graph(int n) : n(n), adj(n) {}
  void edge(int a, int b) {
    adj[a].push_back(b);
    adj[b].push_back(a);
  }
};

// vertices of a triangulated O-grid, round the circle first
static Graph grid(int ni, int nj) {
  Graph g(ni * nj);
  for (int j = 0; j < nj; ++j)
    for (int i = 0; i < ni; ++i) {
      const int v = j * ni + i, r = j * ni + (i + 1) % ni;
      g.edge(v, r);
      if (j + 1 < nj) {
        g.edge(v, v + ni);
        g.edge(r, v + ni);
      }
    }
  return g;
}

// cells of a triangulated channel: two to a square, at most three neighbours
static Graph cells(int ni, int nj) {
  Graph g(2 * ni * nj);
  for (int j = 0; j < nj; ++j)
    for (int i = 0; i < ni; ++i) {
      const int lo = 2 * (j * ni + i), up = lo + 1;
      g.edge(lo, up);
      if (i + 1 < ni) g.edge(up, lo + 2);
      if (j + 1 < nj) g.edge(up, lo + 2 * ni);
    }
  return g;
}

static Graph renumbered(const Graph& a, unsigned seed) {
  std::vector<int> num(a.n);
  std::iota(num.begin(), num.end(), 0);
  std::shuffle(num.begin(), num.end(), std::mt19937(seed));
  Graph g(a.n);
  for (int v = 0; v < a.n; ++v)
    for (int o : a.adj[v])
      if (o > v) g.edge(num[v], num[o]);
  return g;
}

// `count` levels of `width` nodes, each joined to the level before and to the
// one `back` levels before (reads far behind the ring)
static Graph layers(int width, int count, int back) {
  Graph g(width * count);
  for (int l = 1; l < count; ++l)
    for (int i = 0; i < width; ++i) {
      g.edge(l * width + i, (l - 1) * width + i);
      if (width > 1) g.edge(l * width + i, (l - 1) * width + (i + 1) % width);
      if (back > 1 && l >= back) g.edge(l * width + i, (l - back) * width + (i * 7) % width);
    }
  return g;
}

// a chain, and one node at place `where` joined to all the others
static Graph hub(int n, int where) {
  Graph g(n);
  for (int v = 0; v + 1 < n; ++v)
    if (v != where && v + 1 != where) g.edge(v, v + 1);
  for (int v = 0; v < n; ++v)
    if (v != where) g.edge(v, where);
  return g;
}

static int replay(const Graph& g, int ring) {
  const int n = g.n;
  std::vector<int> verts(2 * (size_t)n), pos(2 * (size_t)n), off[2], nb, out(2 * (size_t)n);
  for (int dir = 0; dir < 2; ++dir) {
    std::vector<int> lev(n, 0), cnt(n, 0);
    int nl = 0;
    for (int i = 0; i < n; ++i) {
      const int v = dir == 0 ? i : n - 1 - i;
      for (int o : g.adj[v])
        if (dir == 0 ? o < v : o > v) {
          lev[v] = std::max(lev[v], lev[o] + 1);
          ++cnt[v];
        }
      nl = std::max(nl, lev[v] + 1);
    }
    off[dir].assign(nl + 1, 0);
    for (int v = 0; v < n; ++v) off[dir][lev[v] + 1]++;
    for (int l = 0; l < nl; ++l) off[dir][l + 1] += off[dir][l];
    for (int& o : off[dir]) o += dir * n;
    std::vector<int> order(n);
    std::iota(order.begin(), order.end(), 0);
    // (the solvers order a level by the neighbour counts, most first)
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
      return lev[a] != lev[b] ? lev[a] < lev[b] : cnt[a] > cnt[b];
    });
    for (int i = 0; i < n; ++i) {
      verts[(size_t)dir * n + i] = order[i];
      pos[(size_t)dir * n + order[i]] = dir * n + i;
    }
  }
  std::vector<size_t> eptr(1, 0);
  for (size_t s = 0; s < 2 * (size_t)n; ++s) {
    const int v = verts[s], dir = s < (size_t)n ? 0 : 1;
    for (int o : g.adj[v])
      if (dir == 0 ? o < v : o > v) nb.push_back(pos[(size_t)dir * n + o]);
    eptr.push_back(nb.size());
    out[s] = dir == 0 ? pos[(size_t)n + v] - n : v;
  }
  const SweepPlan p = sweep_plan(n, off[0], off[1], eptr, nb, out, ring);
  const size_t np = 2 * (size_t)n;
  auto slot = [&](int k, int s) {
    if (k >= SW_MAXE) return p.more[(size_t)(k - SW_MAXE) * np + s];
    const int4 h = p.head[s];
    const int w = k < 2 ? h.x : k < 4 ? h.y : h.z & 0xffff;
    return k % 2 ? (int)((unsigned)w >> 16) : w & 0xffff;
  };
  if (!p.npass[0] || !p.npass[1]) return bad("a plan");
  if (p.far.size() != p.pass.size() * SW_WIDTH) return bad("far size", p.far.size());
  if (sw_slots(ring) > 65536) return bad("slots fit 16 bits");
  for (int dir = 0; dir < 2; ++dir) {
    const int base = dir * n, p0 = dir == 0 ? 0 : p.npass[0], npass = p.npass[dir];
    if (sweep_least_steps(off[dir]) > (size_t)p.nstep[dir]) return bad("least steps", dir);
    if (npass % (2 * SW_WAVES)) return bad("whole groups of passes", npass);
    std::vector<int> pass_of(n, -1), lev_of(n);
    for (size_t l = 0; l + 1 < off[dir].size(); ++l)
      for (int s = off[dir][l]; s < off[dir][l + 1]; ++s) lev_of[s - base] = (int)l;
    // the passes cover the positions in order, then the last one again
    int next = base, real = 0;
    for (int i = 0; i < npass; ++i) {
      const int4 w = p.pass[p0 + i];
      if (w.y < 1 || w.y > SW_WIDTH) return bad("nodes of a pass", i, w.y);
      if (next < base + n) {
        if (w.x != next) return bad("passes in order", i, w.x, next);
        for (int s = w.x; s < w.x + w.y; ++s) {
          if (lev_of[s - base] != lev_of[w.x - base]) return bad("one level to a pass", i);
          pass_of[s - base] = i;
        }
        next += w.y;
        real = i + 1;
      } else if (w.x + w.y != base + n) {
        return bad("repeated pass", i);
      }
      if (i >= SW_WAVES && w.z <= p.pass[p0 + i - SW_WAVES].z)
        return bad("a wave's passes in different steps", i);
      if (i > 0 && w.z < p.pass[p0 + i - 1].z) return bad("steps ascend", i);
      if (w.z >= p.nstep[dir]) return bad("step count", i, w.z, p.nstep[dir]);
    }
    if (next != base + n) return bad("all positions", next);
    std::vector<int> tag(ring, -1), writer(ring, -1);  // position in a slot; step that last wrote it
    long far_reads = 0, spilt = 0, reads = 0;
    for (int i0 = 0; i0 < npass;) {
      int i1 = i0;
      while (i1 < npass && p.pass[p0 + i1].z == p.pass[p0 + i0].z) ++i1;
      const int step = p.pass[p0 + i0].z;
      // the writes of a step's passes may land before another's reads
      for (int i = i0; i < i1; ++i)
        for (int s = p.pass[p0 + i].x; s < p.pass[p0 + i].x + p.pass[p0 + i].y; ++s)
          writer[(s - base) % ring] = step;
      for (int i = i0; i < i1; ++i) {
        const int4 w = p.pass[p0 + i];
        const int own = std::min(i, real - 1);  // (a repeated pass reads what the last one did)
        int mc = 0;
        for (int s = w.x; s < w.x + w.y; ++s) {
          const int cnt = (int)(eptr[s + 1] - eptr[s]);
          const int4 h = p.head[s];
          mc = std::max(mc, cnt);
          if (((h.z >> 16) & 0x7fff) != cnt) return bad("entry count", s, cnt);
          if (h.w != out[s]) return bad("place of the result", s);
          for (int k = 0; k < cnt; ++k) {
            const int o = nb[eptr[s] + k], po = pass_of[o - base];
            const int sl = slot(k, s);
            reads += i < real;
            if (po >= i || p.pass[p0 + po].z >= step) return bad("dependency", s, o);
            if (sl >= sw_slots(ring)) return bad("slot in the LDS", s, k, sl);
            if (sl >= 0 && sl < ring) {
              if (tag[sl] != o) return bad("ring slot holds the neighbour", s, o, tag[sl]);
              if (writer[sl] == step && !(i >= real)) return bad("ring slot written while read", s, o);
              continue;
            }
            // stored records
            if (po > own - SW_GAP) return bad("age of a stored record", s, own - po);
            if (p.head[o].z >= 0) return bad("record stored", o);
            if (sl < 0) {
              if (k < SW_MAXE) return bad("entry loaded ahead reads memory", s, k);
              if (!p.spill) return bad("a plan that says so", s, k);
              if (~sl != o - base) return bad("record read from memory", s, o, ~sl);
              spilt += i < real;
            } else {
              const int lane = sl - ring - own % SW_WAVES * SW_WIDTH;
              if (lane < 0 || lane >= SW_WIDTH) return bad("the wave's own fetch slot", s, k, sl);
              if (p.far[(size_t)(p0 + own) * SW_WIDTH + lane] != o - base)
                return bad("fetched record", s, o);
              far_reads += i < real;
            }
          }
          for (int k = cnt; k < p.q; ++k)
            if (slot(k, s) != sw_zero_slot(ring)) return bad("unused entry", s, k);
        }
        if (mc != w.w) return bad("most entries", i, mc, w.w);
        for (int l = 0; l < SW_WIDTH; ++l) {
          const int f = p.far[(size_t)(p0 + i) * SW_WIDTH + l];
          if (f >= 0 && (i >= real || f >= n || i < 2 * SW_WAVES)) return bad("fetch", i, l, f);
        }
      }
      for (int i = i0; i < i1; ++i)
        for (int s = p.pass[p0 + i].x; s < p.pass[p0 + i].x + p.pass[p0 + i].y; ++s)
          tag[(s - base) % ring] = s;
      i0 = i1;
    }
    std::printf("%s: %zu levels, %d passes, %d steps, %.2f %% of %ld reads fetched, %ld from memory\n",
                dir == 0 ? "forward" : "backward", off[dir].size() - 1, real, p.nstep[dir],
                100.0 * far_reads / std::max(1L, reads), reads, spilt);
  }
  return 0;
}

// no plan past what the kernel's 32-bit offsets and 15-bit counts hold
static int limits(int ring) {
  const std::vector<int> none(1, 0);
  if (sweep_plan((1 << 26) + 1, none, none, {}, none, none, ring).npass[0])
    return bad("no plan of more than 2^27 positions");
  // node 0 last in the backward sweep, with 2^15 neighbours; one level a sweep is enough here
  const int n = (1 << 15) + 1;
  std::vector<int> f(2), b(3), nb(2 * (size_t)(n - 1), 0), out(2 * (size_t)n, 0);
  f = {0, 1, n};
  b = {n, 2 * n - 1, 2 * n};
  std::vector<size_t> eptr(1, 0);
  for (int s = 0; s < 2 * n; ++s) eptr.push_back(eptr.back() + (s == 0 || (s >= n && s < 2 * n - 1) ? 0 : s < n ? 1 : n - 1));
  for (int i = 0; i < n - 1; ++i) nb[(size_t)n - 1 + i] = n + i;
  if (sweep_plan(n, f, b, eptr, nb, out, ring).npass[0])
    return bad("no plan of a node with 2^15 neighbours");
  return 0;
}

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  const int ring = std::atoi(argv[1]);
  const std::string kind = argv[2];
  auto a = [&](int i) { return i < argc ? std::atoi(argv[i]) : 0; };
  if (kind == "grid") return replay(grid(a(3), a(4)), ring);
  if (kind == "cells") return replay(cells(a(3), a(4)), ring);
  if (kind == "shuffled") return replay(renumbered(grid(a(3), a(4)), (unsigned)a(5)), ring);
  if (kind == "layers") return replay(layers(a(3), a(4), a(5)), ring);
  if (kind == "limits") return limits(ring);
  if (kind == "hub") return replay(hub(a(3), a(4)), ring);
  return 2;
}
