// Plan of the one-launch triangular sweeps (host only; see sweepplan.h).
#include "sweepplan.h"

#include <algorithm>
#include <atomic>
#include <functional>
#include <thread>

#include "threads.h"

namespace fvk {

namespace {

// f(i) for i in [0, n), shared between threads in runs of consecutive i
template <class F>
void parallel_for(int n, int grain, F f) {
  const int hw = std::max(1u, std::thread::hardware_concurrency());
  const int nt = std::max(1, std::min({hw, 8, n / std::max(1, grain)}));
  on_threads(nt, [&](int t) {
    const int a = (int)((long)n * t / nt), b = (int)((long)n * (t + 1) / nt);
    for (int i = a; i < b; ++i) f(i);
  });
}

// An entry of rank distance x is of a direction's: within a quarter of its
// distance, so that rows left out, added or out of order, which shift the
// distances between lines and planes, do not hide a structured numbering.
inline bool near_distance(int x, int d) { return std::abs(x - d) <= d / 4; }

// The (at most three) rank distances that carry most lower entries, when
// they carry nearly all of them: a structured numbering.  exact: without the
// quarter.  Sampled rows, one of every `step` at no fixed distance: every 224th
// row of a box 224 cells wide has no neighbour at distance 1.
int main_distances(const SweepGraph &g, int (&d)[3], bool &exact) {
  constexpr int T = 64;
  int key[T], cnt[T], same[T], used = 0;
  long total = 0;
  const int step = std::max(1, g.n / 50021);
  unsigned h = 1;
  for (int k0 = 0; k0 < g.n; k0 += step) {
    h = h * 1664525u + 1013904223u;
    const int k = std::min(g.n - 1, k0 + (int)((h >> 8) % (unsigned)step));
    for (int q = g.lptr[k]; q < g.lptr[k + 1]; ++q) {
      const int x = k - g.lcol[q];
      ++total;
      int s = 0;
      while (s < used && !near_distance(x, key[s])) ++s;
      if (s == used) {
        if (used == T) continue;
        key[used] = x;
        cnt[used] = same[used] = 0;
        ++used;
      }
      ++cnt[s];
      same[s] += x == key[s];
    }
  }
  int m = 0;
  long sum = 0, alike = 0;
  while (m < 3) {
    int best = -1;
    for (int s = 0; s < used; ++s)
      if (cnt[s] > 0 && (best < 0 || cnt[s] > cnt[best])) best = s;
    if (best < 0 || cnt[best] * 20L < total) break;
    d[m++] = key[best];
    sum += cnt[best];
    alike += same[best];
    cnt[best] = 0;
  }
  exact = alike * 10 >= total * 9;
  return m > 1 && sum * 10 >= total * 9 ? m : 0;
}

}  // namespace

// The chunks on the longest path through a grid of bricks of these sides
// (cells each), as one compute wave a brick runs them: the chunks of the last
// brick, and for every crossing in a direction the chunks by which a brick
// lags behind the one before it plus the crossing itself.
// kCross: a crossing in chunks (1.4 us against 0.1 us, from boxes of 12^3 to
// 96^3 cut into bricks of 8^3 and 12^3).
static double brick_path(int m, const int *side, const int *cells) {
  constexpr double kCross = 14.0;
  // rows of a brick by level, and the chunks up to a level
  std::vector<int> cnt(1, 1);
  for (int c = 0; c < m; ++c) {
    const int had = (int)cnt.size();
    std::vector<int> t(had + side[c] - 1);
    for (int l = 0, sum = 0; l < (int)t.size(); ++l) {
      if (l < had) sum += cnt[l];
      if (l >= side[c]) sum -= cnt[l - side[c]];
      t[l] = sum;
    }
    cnt.swap(t);
  }
  int all = 0;
  for (int &v : cnt) v = all += (v + kChunk - 1) / kChunk;
  double path = all;
  for (int c = 0; c < m; ++c) {
    int lag = 0;
    for (size_t l = 0; l + side[c] - 1 < cnt.size(); ++l)
      lag = std::max(lag, cnt[l + side[c] - 1] - (l ? cnt[l - 1] : 0));
    path += (cells[c] - 1) * (lag + kCross);
  }
  return path;
}

// Parts.  An acyclic split with few crossings on a path: for each of the
// main rank distances d, phi_d(row) is the largest number of entries of
// distance d (near_distance) on any path that ends at the row.  Each phi_d never decreases
// along an entry, so cells of a grid over the phi_d ("bricks") depend on
// each other only in the direction of growing cell indices, and taking them
// by the sum of the indices is a valid order.  On a box in natural order
// the phi_d are the cell's coordinates, and a path through it crosses a few
// bricks in each direction instead of one range of consecutive rows per
// plane.  The sides are those with the shortest path: few crossings, but no
// levels much wider than a chunk, which the one compute wave runs one after
// the other and which the next brick waits for.  On boxes that gives 8 x 8
// columns (whose levels have at most 64 rows) of up to kBrickRows rows (DIC,
// both sweeps, 24^3 / 96^3 / 128^3, with two halo waves: 35.3 / 153 / 235 us;
// cubes of at most 1728 rows 38 / 163 / 250, of 512 rows 37 / 173).
// Without main distances (unstructured numberings) the parts are ranges of
// consecutive rows, of whichever size sweep_plan_us finds faster: a path through
// triangles crosses them about once a level anyway, and short ones are loaded
// sooner (DIC, both sweeps, 20k / 40k / 200k triangles in RCM order: ranges of
// 512 rows 53 / 65 / 93 us, 1024 45 / 57 / 87, 2048 51 / 61 / 92), where long
// ones save crossings elsewhere (an iteration of CG on 24k tetrahedra 172 -> 123
// us, on a 64^3 box of which a fiftieth is numbered at random 1090 -> 574).
constexpr int kBrickRows = 4096;
constexpr int kRangeRows[] = {1024, 2048};

static bool brick_parts(const SweepGraph &g, int max_rows, std::vector<int> &part, int &P, bool &exact) {
  max_rows = std::min(max_rows, kBrickRows);
  int dist[3] = {0, 0, 0};
  const int m = main_distances(g, dist, exact), n = g.n;
  if (m == 0) return false;
  std::vector<int> phi[3];
  int ext[3] = {1, 1, 1};
  for (int c = 0; c < m; ++c) {
    std::vector<int> &f = phi[c];
    f.assign(n, 0);
    int top = 0;
    for (int k = 0; k < n; ++k) {
      int v = f[k];
      for (int q = g.lptr[k]; q < g.lptr[k + 1]; ++q) {
        const int j = g.lcol[q];
        v = std::max(v, f[j] + (near_distance(k - j, dist[c]) ? 1 : 0));
      }
      f[k] = v;
      top = std::max(top, v);
      if (!g.symmetric)
        for (int q = g.uptr[k]; q < g.uptr[k + 1]; ++q) {
          const int i = g.ucol[q];
          f[i] = std::max(f[i], v + (near_distance(i - k, dist[c]) ? 1 : 0));
        }
    }
    ext[c] = top + 1;
  }
  // sides: the shortest path of all that are even within a direction and have
  // at most `rows` rows a brick of a box; fewer when a brick then has more than
  // max_rows after all, as on irregular numberings
  int side[3] = {1, 1, 1}, cells[3] = {1, 1, 1};
  std::vector<int> cand[3], cnt;
  for (int c = 0; c < 3; ++c)
    for (int w = 1; w <= ext[c]; ++w) {
      const int k = (ext[c] + w - 1) / w, e = (ext[c] + k - 1) / k;
      if (e == w && (w >= 4 || w == ext[c])) cand[c].push_back(w);
    }
  long grid = 1;
  part.resize(n);
  for (int rows = max_rows;; rows = rows * 3 / 4) {
    double best = -1.0;
    for (int s0 : cand[0])
      for (int s1 : cand[1]) {
        if ((long)s0 * s1 > rows) break;
        for (int s2 : cand[2]) {
          if ((long)s0 * s1 * s2 > rows) break;
          const int s[3] = {s0, s1, s2};
          int k[3];
          for (int c = 0; c < 3; ++c) k[c] = (ext[c] + s[c] - 1) / s[c];
          const double t = brick_path(m, s, k);
          if (best < 0 || t < best) {
            best = t;
            std::copy(s, s + 3, side);
          }
        }
      }
    if (best < 0) return false;
    grid = 1;
    for (int c = 0; c < m; ++c) {
      cells[c] = (ext[c] + side[c] - 1) / side[c];
      grid *= cells[c];
    }
    if (grid > n) return false;
    cnt.assign(grid, 0);
    for (int k = 0; k < n; ++k) {
      int id = 0;
      for (int c = m - 1; c >= 0; --c) id = id * cells[c] + phi[c][k] / side[c];
      part[k] = id;
      ++cnt[id];
    }
    if (*std::max_element(cnt.begin(), cnt.end()) <= max_rows) break;
    if (rows < max_rows / 8) return false;
  }
  std::vector<std::pair<int, int>> order;
  for (int id = 0; id < (int)grid; ++id) {
    if (!cnt[id]) continue;
    int s = 0, r = id;
    for (int c = 0; c < m; ++c) {
      s += r % cells[c];
      r /= cells[c];
    }
    order.emplace_back(s, id);
  }
  std::sort(order.begin(), order.end());
  P = (int)order.size();
  std::vector<int> to(grid, -1);
  for (int t = 0; t < P; ++t) to[order[t].second] = t;
  for (int k = 0; k < n; ++k) part[k] = to[part[k]];
  return true;
}

enum PlanEnd { PLAN_OK, PLAN_LDS, PLAN_POSITIONS, PLAN_NONE };
// range_rows 0: bricks
static PlanEnd plan_with(const SweepGraph &g, int max_rows, int range_rows, long limit, SweepPlan &p, bool &exact) {
  const int n = g.n;
  std::vector<int> part;
  int P = 0;
  p.bricks = range_rows == 0;
  if (p.bricks) {
    if (!brick_parts(g, max_rows, part, P, exact)) return PLAN_NONE;
  } else {
    const int rows = std::min(max_rows, range_rows);
    part.resize(n);
    for (int k = 0; k < n; ++k) part[k] = k / rows;
    P = (n + rows - 1) / rows;
  }
  p.n = n;
  p.P = P;
  // dependency levels, and the rows of each part by level (ties by rank)
  std::vector<int> lev(n, 0);
  int nl = 0;
  for (int k = 0; k < n; ++k) {
    int l = lev[k];
    for (int q = g.lptr[k]; q < g.lptr[k + 1]; ++q) l = std::max(l, lev[g.lcol[q]] + 1);
    lev[k] = l;
    nl = std::max(nl, l + 1);
    if (!g.symmetric)
      for (int q = g.uptr[k]; q < g.uptr[k + 1]; ++q) lev[g.ucol[q]] = std::max(lev[g.ucol[q]], l + 1);
  }
  p.levels = nl;
  std::vector<int> order(n), pbeg(P + 1, 0);
  {
    std::vector<int> at(nl + 1, 0), tmp(n);
    for (int k = 0; k < n; ++k) ++at[lev[k] + 1];
    for (int l = 0; l < nl; ++l) at[l + 1] += at[l];
    for (int k = 0; k < n; ++k) tmp[at[lev[k]]++] = k;
    for (int k = 0; k < n; ++k) ++pbeg[part[k] + 1];
    for (int q = 0; q < P; ++q) pbeg[q + 1] += pbeg[q];
    std::vector<int> to(pbeg.begin(), pbeg.end() - 1);
    for (int k : tmp) order[to[part[k]]++] = k;
  }
  // asymmetric patterns: who reads a row in each direction
  std::vector<unsigned char> rd[2];
  if (!g.symmetric) {
    rd[0].assign(n, 0);
    rd[1].assign(n, 0);
    for (int k = 0; k < n; ++k) {
      for (int q = g.lptr[k]; q < g.lptr[k + 1]; ++q)
        if (part[g.lcol[q]] != part[k]) rd[0][g.lcol[q]] = 1;
      for (int q = g.uptr[k]; q < g.uptr[k + 1]; ++q)
        if (part[g.ucol[q]] != part[k]) rd[1][g.ucol[q]] = 1;
    }
  }
  auto exported = [&](int k, int dir) {
    if (!g.symmetric) return rd[dir][k] != 0;
    // read in the forward sweep by the rows of its upper entries
    const std::vector<int> &ptr = dir == 0 ? g.uptr : g.lptr, &col = dir == 0 ? g.ucol : g.lcol;
    for (int q = ptr[k]; q < ptr[k + 1]; ++q)
      if (part[col[q]] != part[k]) return true;
    return false;
  };
  // chunks: rows in level order; a new chunk when one is full or the next
  // row depends on a row of the chunk being filled
  std::vector<int> chunk(n), lane(n), slot(n), nch(P);
  std::vector<int> dep(g.symmetric ? 0 : n);  // asymmetric: newest chunk that reaches a row from an upper entry
  std::vector<int> ne[2] = {std::vector<int>(P), std::vector<int>(P)};
  for (p.width = kChunk;; p.width /= 2) {
    const int width = p.width;
    std::fill(dep.begin(), dep.end(), -1);
    parallel_for(P, 8, [&](int q) {
      int c = 0, fill = 0, e0 = 0, e1 = 0;
      for (int t = pbeg[q]; t < pbeg[q + 1]; ++t) {
        const int k = order[t];
        bool next = fill == width;
        for (int z = g.lptr[k]; !next && z < g.lptr[k + 1]; ++z) {
          const int j = g.lcol[z];
          next = part[j] == q && chunk[j] == c;
        }
        if (!next && !g.symmetric) next = dep[k] == c;
        if (next) {
          ++c;
          fill = 0;
        }
        chunk[k] = c;
        lane[k] = fill++;
        slot[k] = t - pbeg[q];
        if (!g.symmetric)
          for (int z = g.uptr[k]; z < g.uptr[k + 1]; ++z)
            if (part[g.ucol[z]] == q) dep[g.ucol[z]] = c;
        e0 += exported(k, 0);
        e1 += exported(k, 1);
      }
      nch[q] = c + 1;
      ne[0][q] = e0;
      ne[1][q] = e1;
    });
    long positions = 0;
    for (int q = 0; q < P; ++q) positions += (long)nch[q] * width;
    if (positions <= (long)kPadding * n || width <= kPadding) break;
  }
  std::vector<int> cb(P + 1, 0);
  for (int q = 0; q < P; ++q) cb[q + 1] = cb[q] + nch[q];
  const int width = p.width;
  if ((long)cb[P] * width > limit) return PLAN_POSITIONS;
  p.np = cb[P] * width;
  // exports, numbered part by part in the order the direction runs
  std::vector<int> eslot[2];
  for (int dir = 0; dir < 2; ++dir) {
    std::vector<int> eb(P + 1, 0);
    for (int q = 0; q < P; ++q) eb[q + 1] = eb[q] + ne[dir][q];
    p.d[dir].NE = eb[P];
    eslot[dir].assign(n, -1);
    parallel_for(P, 8, [&](int q) {
      int e = eb[q];
      const int a = pbeg[q], b = pbeg[q + 1];
      for (int t = a; t < b; ++t) {
        const int k = order[dir == 0 ? t : a + b - 1 - t];
        if (exported(k, dir)) eslot[dir][k] = e++;
      }
    });
  }
  // halos and entry offsets
  p.slots = 0;
  const int MW = p.MW, NI = p.nrec(), ND = p.at_need();
  const size_t np = p.np;
  p.part.assign((size_t)8 * P, 0);
  p.tval.assign((size_t)MW * np, -1);
  std::atomic<int> slots{0};
  for (int dir = 0; dir < 2; ++dir) {
    SweepPlan::Dir &D = p.d[dir];
    const std::vector<int> &ptr = dir == 0 ? g.lptr : g.uptr, &col = dir == 0 ? g.lcol : g.ucol,
                           &val = dir == 0 ? g.lval : g.uval;
    D.rec.assign((size_t)NI * np, 0);
    D.val.assign((size_t)MW * np, -1);
    std::vector<std::vector<int>> halo(P);
    parallel_for(P, 8, [&](int q) {
      std::vector<int> &h = halo[q];
      const int a = pbeg[q], b = pbeg[q + 1], nr = b - a;
      std::vector<int> need(nch[q], 0);
      // open addressing: row -> halo slot
      size_t cap = 64;
      std::vector<std::pair<int, int>> tab(cap, {-1, 0});
      auto find = [&](int j) -> int & {
        if (h.size() * 2 >= cap) {
          cap *= 2;
          std::vector<std::pair<int, int>> t2(cap, {-1, 0});
          for (auto &e : tab)
            if (e.first >= 0) {
              size_t i = (unsigned)e.first * 2654435761u & (cap - 1);
              while (t2[i].first >= 0) i = (i + 1) & (cap - 1);
              t2[i] = e;
            }
          tab.swap(t2);
        }
        size_t i = (unsigned)j * 2654435761u & (cap - 1);
        while (tab[i].first >= 0 && tab[i].first != j) i = (i + 1) & (cap - 1);
        if (tab[i].first < 0) {
          tab[i] = {j, (int)h.size()};
          h.push_back(j);
        }
        return tab[i].second;
      };
      for (int s = a; s < b; ++s) {
        const int k = order[dir == 0 ? s : a + b - 1 - s];
        const size_t pos = (size_t)(cb[q] + chunk[k]) * width + lane[k];
        unsigned short *ix = &D.rec[pos * NI];
        ix[0] = (unsigned short)(slot[k] * 8);
        ix[ND + 1] = (unsigned short)((unsigned)eslot[dir][k] & 0xffffu);
        ix[ND + 2] = (unsigned short)((unsigned)eslot[dir][k] >> 16);
        for (int z = ptr[k], t = 0; z < ptr[k + 1]; ++z, ++t) {
          const int j = col[z];
          ix[1 + t] = (unsigned short)((part[j] == q ? slot[j] : nr + find(j)) * 8);
          D.val[(size_t)t * np + pos] = val[z];
          if (dir == 0) p.tval[(size_t)t * np + pos] = g.tval[z];
        }
        need[chunk[k]] = (int)h.size();
      }
      const int zero = nr + (int)h.size(), used = zero + 2;
      int seen = slots.load();
      while (used > seen && !slots.compare_exchange_weak(seen, used)) {
      }
      if (used * 8 > 65535) return;  // no plan: see below
      // padding entries read the zero slot; the need is the chunk's in every lane
      for (int c = 0; c < nch[q]; ++c)
        for (int l = 0; l < width; ++l) {
          const size_t pos = (size_t)(cb[q] + c) * width + l;
          unsigned short *ix = &D.rec[pos * NI];
          ix[ND] = (unsigned short)need[c];
          int t = 0;
          while (t < MW && D.val[(size_t)t * np + pos] >= 0) ++t;
          for (; t < MW; ++t) ix[1 + t] = (unsigned short)(zero * 8);
        }
    });
    if (slots.load() * 8 > 65535) return PLAN_LDS;
    // lanes without a row write the last slot and export nothing
    parallel_for(P, 8, [&](int q) {
      const int other = (pbeg[q + 1] - pbeg[q] + (int)halo[q].size() + 1) * 8;
      std::vector<int> fill(nch[q], 0);
      for (int t = pbeg[q]; t < pbeg[q + 1]; ++t) fill[chunk[order[t]]] = lane[order[t]] + 1;
      for (int c = 0; c < nch[q]; ++c)
        for (int l = fill[c]; l < width; ++l) {
          unsigned short *ix = &D.rec[((size_t)(cb[q] + c) * width + l) * NI];
          ix[0] = (unsigned short)other;
          ix[ND + 1] = ix[ND + 2] = 0xffffu;
        }
    });
    size_t hb = 0;
    for (int q = 0; q < P; ++q) {
      p.part[8 * q + 4 + 2 * dir] = (int)hb;
      p.part[8 * q + 5 + 2 * dir] = (int)halo[q].size();
      p.maxh = std::max(p.maxh, (int)halo[q].size());
      hb += halo[q].size();
    }
    D.hsrc.resize(hb);
    parallel_for(P, 8, [&](int q) {
      int *o = D.hsrc.data() + p.part[8 * q + 4 + 2 * dir];
      for (int j : halo[q]) *o++ = eslot[dir][j];
    });
  }
  p.slots = slots.load();
  if (p.lds(3) > (size_t)kSweepLds) return PLAN_LDS;
  // rows of each part by device row
  p.prow.resize(n);
  p.ppos.resize(n);
  p.pslot.resize(n);
  parallel_for(P, 8, [&](int q) {
    p.part[8 * q] = cb[q];
    p.part[8 * q + 1] = nch[q];
    p.part[8 * q + 2] = pbeg[q];
    p.part[8 * q + 3] = pbeg[q + 1] - pbeg[q];
    std::vector<std::pair<int, int>> r;
    r.reserve(pbeg[q + 1] - pbeg[q]);
    for (int t = pbeg[q]; t < pbeg[q + 1]; ++t) r.emplace_back(g.row[order[t]], order[t]);
    std::sort(r.begin(), r.end());
    for (size_t t = 0; t < r.size(); ++t) {
      const int k = r[t].second;
      p.prow[pbeg[q] + t] = r[t].first;
      p.ppos[pbeg[q] + t] = (cb[q] + chunk[k]) * width + lane[k];
      p.pslot[pbeg[q] + t] = (unsigned short)(slot[k] * 8);
    }
  });
  return PLAN_OK;
}

// Time of both sweeps with one right-hand side in us, by walking the plan as
// the kernels do: blocks take parts as they come free, a chunk takes 0.1 us
// from the one before or from its last halo value, a lane of the halo wave
// fetches one value in 0.5 us, 0.7 us after it was passed on at the earliest,
// and a part is loaded and stored in 1.4 us.  Within 10 % of the sweeps in 50
// patterns (boxes, triangles, tetrahedra; natural, RCM, Morton, red-black and
// random orders) with ranges of 256 to 4096 rows, from 10 us to 9.5 ms, and low
// by up to 1.7 where many blocks wait long, as polls then hinder each other.
// Chunks of the level order (sweep.h) take 4.2 us a level for both sweeps, 3 to
// 5.4 in those patterns, or 0.32 ns a row.  They are the faster form where a
// part needs many values from many others: an iteration of CG, parts / chunks:
// 48^3 box numbered at random 408 / 116 us, 80^3 949 / 214, 200k triangles at
// random 248 / 91, 64^3 in RCM order 821 / 608; but 60k triangles as they are
// 85 / 121, 64^3 in natural order 112 / 1028.
double sweep_plan_us(const SweepPlan &p) {
  constexpr int kCus = 256;
  const int NI = p.nrec(), ND = p.at_need();
  const int blocks = std::min(p.P, kCus * std::max(1, std::min(4, (int)(163840 / (p.lds(1) + 512)))));
  double sum = 0;
  for (int dir = 0; dir < 2; ++dir) {
    const SweepPlan::Dir &D = p.d[dir];
    std::vector<float> passed(D.NE, 0.f);    // when a value was passed on
    std::vector<double> idle(blocks, 0.0);   // when a block comes free, the first at the heap's head
    double end = 0;
    for (int o = 0; o < p.P; ++o) {
      const int q = dir == 0 ? o : p.P - 1 - o, *Q = &p.part[8 * q];
      const int *src = D.hsrc.data() + Q[4 + 2 * dir];
      std::pop_heap(idle.begin(), idle.end(), std::greater<double>());
      double t = idle.back() + 1.4, there = t, lane[64];
      std::fill(lane, lane + 64, t);
      int have = 0;
      for (int c = 0; c < Q[1]; ++c) {
        const int ch = Q[0] + (dir == 0 ? c : Q[1] - 1 - c);
        const unsigned short *rec = &D.rec[(size_t)ch * p.width * NI];
        for (; have < rec[ND]; ++have) {
          double &l = lane[have % 64];
          l = std::max(l + 0.5, passed[src[have]] + 0.7);
          there = std::max(there, l);
        }
        t = std::max(t, there) + 0.1;
        for (int k = 0; k < p.width; ++k) {
          const int e = (int)((unsigned)rec[k * NI + ND + 1] | (unsigned)rec[k * NI + ND + 2] << 16);
          if (e >= 0) passed[e] = (float)t;
        }
      }
      idle.back() = t + 1.4;
      std::push_heap(idle.begin(), idle.end(), std::greater<double>());
      end = std::max(end, t);
    }
    sum += end;
  }
  return sum;
}

std::string sweep_plan(const SweepGraph &g, int max_rows, SweepPlan &p, long limit) {
  int W = 1;
  for (int k = 0; k < g.n; ++k) W = std::max({W, g.lptr[k + 1] - g.lptr[k], g.uptr[k + 1] - g.uptr[k]});
  if (W > 8) return "a row has more lower or upper entries than one launch holds";
  const int MW = W <= 3 ? 3 : W <= 4 ? 4 : 8;
  // smaller parts until every part and its halo fit the LDS (a part of R
  // rows has at most 8 R halo values, so this ends)
  bool exact = false;
  auto fit = [&](int range, SweepPlan &q) {
    for (int r = range ? std::min(max_rows, range) : max_rows; r >= 64; r /= 2) {
      q = SweepPlan();
      q.W = W;
      q.MW = W <= 3 ? 3 : W <= 4 ? 4 : 8;
      const long most = (1L << 32) / (2 * q.nrec());
      const PlanEnd e = plan_with(g, r, range, limit > 0 ? std::min(limit, most) : most, q, exact);
      if (e == PLAN_OK && !(range == 0 && exact)) q.us = sweep_plan_us(q);
      if (e != PLAN_LDS) return e;
    }
    return PLAN_NONE;
  };
  // bricks of an exactly structured numbering, else the fastest of the forms
  PlanEnd e = fit(0, p);
  if (e != PLAN_OK || !exact)
    for (int range : kRangeRows) {
      if (range > kRangeRows[0] && (e == PLAN_POSITIONS || max_rows <= kRangeRows[0] || p.P == 1)) break;
      SweepPlan q;
      const PlanEnd f = fit(range, q);
      if (f == PLAN_OK && (e != PLAN_OK || q.us < p.us)) p = std::move(q);
      if (e != PLAN_OK) e = f;
    }
  if (e == PLAN_POSITIONS) return "the pattern needs more positions than the sweep tables hold";
  if (e != PLAN_OK) return "no plan";
  p.chunk_us = std::max(4.2 * p.levels, 3.2e-4 * p.n);
  return "";
}

std::string sweep_plan_check(const SweepGraph &g, const SweepPlan &p) {
  const int NI = p.nrec(), ND = p.at_need();
  if ((long)p.np * 2 * NI > 1L << 32) return "a record's byte offset";
  // rank at each position
  std::vector<int> rank_of_row(g.n, -1), rank_at(p.np, -1);
  for (int k = 0; k < g.n; ++k) rank_of_row[g.row[k]] = k;
  for (int t = 0; t < g.n; ++t) {
    const int k = rank_of_row[p.prow[t]];
    if (k < 0 || p.ppos[t] < 0 || p.ppos[t] >= p.np || rank_at[p.ppos[t]] >= 0) return "a row is not run once";
    rank_at[p.ppos[t]] = k;
  }
  for (int dir = 0; dir < 2; ++dir) {
    const SweepPlan::Dir &D = p.d[dir];
    const std::vector<int> &ptr = dir == 0 ? g.lptr : g.uptr, &col = dir == 0 ? g.lcol : g.ucol,
                           &val = dir == 0 ? g.lval : g.uval;
    std::vector<int> exported(D.NE, -1);
    std::vector<int> lds(p.slots);
    for (int o = 0; o < p.P; ++o) {
      const int q = dir == 0 ? o : p.P - 1 - o, *Q = &p.part[8 * q];
      std::fill(lds.begin(), lds.end(), -1);
      const int h0 = Q[4 + 2 * dir], nh = Q[5 + 2 * dir], zero = Q[3] + nh;
      if (h0 < 0 || h0 + nh > (int)D.hsrc.size() || nh > p.maxh || zero + 2 > p.slots) return "halo size";
      int have = 0;
      for (int c = 0; c < Q[1]; ++c) {
        const int ch = Q[0] + (dir == 0 ? c : Q[1] - 1 - c);
        const int need = D.rec[(size_t)ch * p.width * NI + ND];
        if (need > nh) return "halo count";
        for (; have < need; ++have) {
          const int e = D.hsrc[h0 + have];
          if (e < 0 || e >= D.NE || exported[e] < 0) return "a halo value of a part not taken before";
          lds[Q[3] + have] = exported[e];
        }
        for (int l = 0; l < p.width; ++l) {
          const size_t pos = (size_t)ch * p.width + l;
          const int k = rank_at[pos];
          const unsigned short *ix = &D.rec[pos * NI];
          if (ix[ND] != need) return "the need differs between lanes";
          if (k < 0) {
            if (ix[0] / 8 != zero + 1 || ix[ND + 1] != 0xffffu || ix[ND + 2] != 0xffffu) return "padding lane";
            continue;
          }
          int t = 0;
          for (int z = ptr[k]; z < ptr[k + 1]; ++z, ++t)
            if (lds[ix[1 + t] / 8] != col[z] || D.val[(size_t)t * p.np + pos] != val[z] ||
                (dir == 0 && p.tval[(size_t)t * p.np + pos] != g.tval[z]))
              return "an entry reads the wrong value";
          for (; t < p.MW; ++t)
            if (ix[1 + t] / 8 != zero || D.val[(size_t)t * p.np + pos] >= 0) return "padding entry";
        }
        for (int l = 0; l < p.width; ++l) {
          const size_t pos = (size_t)ch * p.width + l;
          const int k = rank_at[pos];
          if (k < 0) continue;
          const unsigned short *ix = &D.rec[pos * NI];
          lds[ix[0] / 8] = k;
          const int e = (int)((unsigned)ix[ND + 1] | (unsigned)ix[ND + 2] << 16);
          if (e < -1 || e >= D.NE || (e >= 0 && exported[e] >= 0)) return "an export index";
          if (e >= 0) exported[e] = k;
        }
      }
    }
    for (int e : exported)
      if (e < 0) return "an export without a value";
  }
  for (int t = 0; t < g.n; ++t)
    if (p.d[0].rec[(size_t)p.ppos[t] * NI] != p.pslot[t] || p.d[1].rec[(size_t)p.ppos[t] * NI] != p.pslot[t])
      return "a row's slot";
  return "";
}

}  // namespace fvk
