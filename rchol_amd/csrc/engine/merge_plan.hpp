// Host plan of the merged levels of the persistent sweep (k_sptrsv).
// Included by engine.hip inside its anonymous namespace, after analysis.hpp.
//
// A dependency level costs a handshake between compute units (1.5 to 2 us
// on MI355X) however few rows it holds, and most levels of a factor hold few
// (256^3: 461 of 487 hold 4% of the rows).  Consecutive narrow levels are
// therefore merged into one group: a row's dependencies inside the group are
// eliminated on the host,
//
//   x_i = (b_i - sum_j L_ij x_j) / d_i,   j in the group:
//   L_ij x_j = (L_ij / d_j) (b_j - sum_k L_jk x_k),
//
// until the row reads only rows of earlier groups (merged entries) and
// right-hand sides of its own group.  The group is then one level: one
// handshake instead of as many as it holds levels, for rows that are longer.
//
// Only factors whose off-diagonal entries have the sign opposite to their
// row's pivot are merged (every rchol factor: L_ij <= 0 < d_i).  Then every
// product added to a merged entry has the same sign, so the elimination
// cancels nothing and a merged row is as accurate as the substitution it
// replaces.
#pragma once

// What a handshake and an entry cost, for the choice of the groups
// (microseconds): the handshake of a narrow level and the throughput of
// gathered entries measured with all waves busy.
#ifndef RCHOL_AMD_MERGE_HOP
#define RCHOL_AMD_MERGE_HOP 2.0
#endif
#ifndef RCHOL_AMD_MERGE_PS
#define RCHOL_AMD_MERGE_PS 5.0
#endif
constexpr double kHopUs = RCHOL_AMD_MERGE_HOP;
constexpr double kEntryUs = RCHOL_AMD_MERGE_PS * 1e-6;
// How far a level is merged: microseconds of entries that merging may add to
// it, mean entries of its merged rows; most levels of a sweep that is merged;
// largest coefficient of a merged row, in pivots of the row.
struct MergeLimits {
  double cap_us, len;
  int levels;
  double ratio;
};
constexpr int kMergeMaxLevels = 1 << 20;  // (fits the sort key of a merged entry)
#ifndef RCHOL_AMD_MERGE_CAP
#define RCHOL_AMD_MERGE_CAP 0.2
#endif
#ifndef RCHOL_AMD_MERGE_LEN
#define RCHOL_AMD_MERGE_LEN 1024
#endif
// A deep factor (thousands of narrow levels) has few rows per level: deeper
// groups, to rows that grow at most kDeepGrowth-fold on average (24^3 in
// natural order, 2929 levels, FP64: 48-fold 7.5 ms per solve and 40 ms of
// planning, 96-fold 5.7 and 55; static 64^3, 8216 levels: 54 and 51 ms).
// Planning grows with the levels and stays out beyond kDeepMaxLevels.  That
// line bounds the upload, not the gain: at static 96^3 (17126 levels) and 128^3
// (21937) planning would take 0.46 and 0.68 s, the chunks' 0.11 and 0.22, for
// sweeps of 5.6 and 9.9 ms an application instead of 9.0 and 15.1; at 256^3
// (104163) 4.5 s, for sweeps that the chunks win.
#ifndef RCHOL_AMD_MERGE_DEEP_CAP
#define RCHOL_AMD_MERGE_DEEP_CAP 0.05
#endif
#ifndef RCHOL_AMD_MERGE_DEEP_LEN
#define RCHOL_AMD_MERGE_DEEP_LEN 2048
#endif
constexpr double kDeepGrowth = 96.0;
constexpr int kDeepMaxLevels = 16384;
// Largest coefficient of a merged row in pivots of the row.  Beyond the
// reciprocal of the unit roundoff a term x_k c / d says nothing of a result of
// ordinary size: the row's terms cancel.  The substitution cancels them one
// dependency at a time; merged, each is formed whole, and in FP32 c x_k may
// pass the largest number.
constexpr double kMergeRatio32 = 1e8;
MergeLimits merge_limits(bool deep, size_t n, size_t nnz, int precision) {
  const double ratio = precision == RCHOL_AMD_FP32 ? kMergeRatio32 : HUGE_VAL;
  if (!deep) return {RCHOL_AMD_MERGE_CAP, RCHOL_AMD_MERGE_LEN, kMergeMaxLevels, ratio};
  return {RCHOL_AMD_MERGE_DEEP_CAP,
          std::min<double>(RCHOL_AMD_MERGE_DEEP_LEN, kDeepGrowth * (double)nnz / (double)n),
          kDeepMaxLevels, ratio};
}

struct MergePlan {
  std::vector<int> gptr;  // group g: levels [gptr[g], gptr[g + 1])
  int m0 = 0, m1 = 0;     // slots that may hold merged rows
  IntVec rp;              // merged row of slot s at [rp[s - m0], rp[s - m0 + 1])
  IntVec ci;              // x of row c: c;  right-hand side of row c: -2 - c
  DblVec cv;
  ProxyVec proxy;  // per slot of [m0, m1): row_proxy over groups
  double est_us = 0.0;
  bool any() const { return m1 > m0; }
};

// Column -> value map of one row under elimination, in insertion order.  Up to
// kDirectMap rows a place per column; beyond, open addressing.  `at` lists the
// used places so that clearing costs the row's length.
constexpr size_t kDirectMap = (size_t)1 << 20;
struct RowMap {
  struct Place {
    int key, pos;  // key == c: column c is cols[pos]
  };
  std::vector<Place> tab;
  std::vector<int> at, cols;
  std::vector<double> vals;
  bool direct;
  size_t mask = 1023;
  explicit RowMap(size_t n) : tab(n <= kDirectMap ? n : 1024, Place{-1, 0}), direct(n <= kDirectMap) {}
  size_t find(int c) const {
    if (direct) return (size_t)c;
    size_t p = (size_t)((unsigned)c * 2654435761u >> 7) & mask;
    while (tab[p].key != -1 && tab[p].key != c) p = (p + 1) & mask;
    return p;
  }
  void clear() {
    for (int p : at) tab[p].key = -1;
    at.clear();
    cols.clear();
    vals.clear();
  }
  void put(size_t p, int c, int k) {
    tab[p] = Place{c, k};
    at.push_back((int)p);
  }
  // Adds v to column c and returns its place in cols / vals; fresh: new.
  int add(int c, double v, bool &fresh) {
    const size_t p = find(c);
    fresh = tab[p].key == -1;
    if (!fresh) {
      vals[tab[p].pos] += v;
      return tab[p].pos;
    }
    const int k = (int)cols.size();
    cols.push_back(c);
    vals.push_back(v);
    if (!direct && 2 * cols.size() > mask) {
      mask = 4 * (mask + 1) - 1;
      tab.assign(mask + 1, Place{-1, 0});
      at.clear();
      for (int q = 0; q <= k; q++) put(find(cols[q]), cols[q], q);
    } else {
      put(p, c, k);
    }
    return k;
  }
};

// One row under elimination: its entries outside levels [l0, lev(i)) and its
// dependencies inside them.
struct RowElim {
  RowMap map;
  std::vector<std::vector<int>> bucket;  // map positions of the dependencies per level - l0
  int depth = 0;
  explicit RowElim(size_t n) : map(n) {}

  // Eliminate row i (level m) of the group that starts at level l0.  With
  // values: map holds every column's merged coefficient (dependencies inside
  // the group: their coefficient before division).  Returns the row's merged
  // entries plus right-hand sides.
  int run(const HostSweep &h, const IntVec &lev, int i, int l0, bool values) {
    map.clear();
    const int m = lev[i];
    depth = m - l0;
    if ((int)bucket.size() < depth) bucket.resize(depth);
    for (int q = 0; q < depth; q++) bucket[q].clear();
    const DblVec &dg = *h.nat_diag;
    auto take = [&](int r, double f) {
      for (int e = h.nat_rp[r]; e < h.nat_rp[r + 1]; e++) {
        const int j = h.nat_ci[e];
        bool fresh;
        const int p = map.add(j, values ? f * h.nat_cv[e] : 0.0, fresh);
        if (fresh && lev[j] >= l0) bucket[lev[j] - l0].push_back(p);
      }
    };
    take(i, 1.0);
    for (int q = depth - 1; q >= 0; q--)
      for (size_t t = 0; t < bucket[q].size(); t++) {
        const int p = bucket[q][t];
        const int k = map.cols[p];
        take(k, values ? -(map.vals[p] / dg[k]) : 0.0);
      }
    return (int)map.cols.size();
  }
};

// Sort key of a merged entry: level (20 bits) | column (31) | place (13).
constexpr int kKeyPos = 13, kKeyLevel = 44;
static_assert(kKeyLevel + 20 == 64 && kMergeMaxLevels == 1 << 20, "sort key");
constexpr int kMergeMaxRow = 1 << kKeyPos;
// Largest merged coefficient: one beyond it (pivots that differ by tens of
// orders of magnitude) could overflow where the substitution does not.
constexpr double kMergeMaxAbs = 1e30;
// Most merged entries of a sweep, in entries and rows of the factor.  The
// limit on a group's mean row says nothing of it: a chain of 300 rows, or 604
// levels of a 32 x 32 grid in natural order, fit one group of rows of several
// hundred entries.  A plan beyond it is made again with shorter rows.
constexpr long long kMergeMaxGrowth = 64;
constexpr double kMergeMinLen = 8;  // rows too short to be worth a plan
constexpr int kMergeCuts = 6;

// Whether every off-diagonal entry of the sweep has the sign opposite to its
// row's pivot (or is zero).
bool merge_signs(const HostSweep &h, size_t n) {
  std::atomic<bool> ok{true};
  const DblVec &dg = *h.nat_diag;
  par_for(n, [&](size_t r0, size_t r1) {
    bool good = true;
    for (size_t r = r0; r < r1 && good; r++) {
      const bool pos = dg[r] > 0.0;
      for (int e = h.nat_rp[r]; e < h.nat_rp[r + 1]; e++)
        good &= pos ? h.nat_cv[e] <= 0.0 : h.nat_cv[e] >= 0.0;
    }
    if (!good) ok = false;
  });
  return ok;
}

// Groups of consecutive levels [a, b): a group grows by its next levels (an
// eighth of its depth at a time) while their rows, merged, stay within lim.len
// entries on average and the entries that merging adds to a level cost less
// than lim.cap_us.  Merged lengths come from a sample of the rows of the last
// level.  Neighbouring groups are about as deep as each other, so the search
// starts at the depth of the last one and goes up or down from there.
constexpr int kMergeSample = 6;

void plan_groups(const HostSweep &h, const IntVec &lev, int a, int b, const MergeLimits &lim,
                 std::vector<int> &gptr) {
  const std::vector<int> &lp = h.level_ptr;
  RowElim el(h.nat_rp.size() - 1);
  double merged = 0.0, plain = 0.0;  // mean entries of the rows that fits() looked at last
  auto mean_merged = [&](int m, int l0) {
    const int w = lp[m + 1] - lp[m], k = std::min(w, kMergeSample);
    merged = plain = 0.0;
    for (int t = 0; t < k; t++) {
      const int i = h.slot_row[lp[m] + (int)((2LL * t + 1) * w / (2 * k))];
      merged += el.run(h, lev, i, l0, false);
      plain += h.nat_rp[i + 1] - h.nat_rp[i];
    }
    merged /= k;
    plain /= k;
  };
  auto widest = [&](int l0, int l1) {
    int w = 0;
    for (int q = l0; q < l1; q++) w = std::max(w, lp[q + 1] - lp[q]);
    return (double)w;
  };
  // whether the group [l, e) may hold its last levels (a ninth of them)
  auto fits = [&](int l, int e, double cap_us) {
    mean_merged(e - 1, l);
    return merged <= lim.len &&
           (merged - plain) * widest(e - std::max(1, (e - l) / 9), e) * kEntryUs <= cap_us;
  };
  int depth = 1;
  for (int l = a; l < b;) {
    const int guess = std::min(b, l + depth);
    int e = guess;
    while (e - l > 1 && !fits(l, e, lim.cap_us)) e = std::max(l + 1, e - std::max(1, (e - l) / 8));
    // the levels below the last: their rows are no longer than the last one's,
    // but a level may be wider.  One of up to twice the limit is left in, where
    // it costs less than the handshake of cutting there (solves cut at the limit
    // itself: natural 24^3 5.64 -> 5.74 ms, 32^3 2.53 -> 2.56)
    const double longest = merged, cap = 2.0 * lim.cap_us;
    for (int q = l + 1; q < e;) {
      const int m = std::min(e, q + std::max(1, (q - l) / 8));
      if (m < e && longest * widest(q, m) * kEntryUs > cap && !fits(l, m, cap)) e = q;
      q = m;
    }
    while (e >= guess && e < b) {
      const int m = std::min(b, e + std::max(1, (e - l) / 8));
      if (!fits(l, m, lim.cap_us)) break;
      e = m;
    }
    depth = e - l;
    gptr.push_back(l);
    l = e;
  }
}

// Merged rows of the groups out.gptr (grp: each level's group) into out: blocks
// of slots, each into its own arrays, then in order.  A row's entries:
// right-hand sides, then values by level and column, so that the latest come
// last and neighbouring columns are gathered together (in the order the
// elimination meets them: sweeps 4 to 18% slower).  bad[g]: lowered to the
// lowest level of group g with a row that cannot be merged (which is left
// out).  False: more merged entries than kMergeMaxGrowth allows.
bool merge_rows(const HostSweep &h, size_t n, const IntVec &lev, const IntVec &grp, double ratio,
                std::vector<std::atomic<int>> &bad, MergePlan &out) {
  const int M = out.m1 - out.m0;
  constexpr int kBlk = 64;
  const int B = (M + kBlk - 1) / kBlk;
  struct Block {
    std::vector<int> ci;
    std::vector<double> cv;
  };
  std::vector<Block> blk(B);
  IntVec len(M);
  out.proxy.resize(M);
  std::atomic<int> next{0};
  std::atomic<long long> total{0};
  std::atomic<bool> over{false};  // too many merged entries
  const long long most = std::min<long long>(kMergeMaxGrowth * (h.rp[n] + (long long)n), INT_MAX / 2);
  par_run(std::min(host_threads(), std::max(1, B / 4)), [&](int) {
    RowElim el(n);
    Block o;
    std::vector<unsigned long long> key;  // level | column | map position
    for (int b; (b = next.fetch_add(1)) < B && !over;) {
      o.ci.clear();
      o.cv.clear();
      for (int s = out.m0 + b * kBlk; s < std::min(out.m1, out.m0 + (b + 1) * kBlk); s++) {
        const int i = h.slot_row[s], g = grp[lev[i]], l0 = out.gptr[g];
        len[s - out.m0] = 0;
        out.proxy[s - out.m0] = 0;
        if (lev[i] == l0) continue;  // reads nothing inside its group: its plain row
        el.run(h, lev, i, l0, true);
        const RowMap &m = el.map;
        bool fits = (int)m.cols.size() <= kMergeMaxRow;
        const double most_v = std::min(kMergeMaxAbs, ratio * std::fabs((*h.nat_diag)[i]));
        for (double v : m.vals) fits &= std::fabs(v) <= most_v;
        for (int p = 0; p < (int)m.cols.size(); p++)
          if (lev[m.cols[p]] >= l0)
            fits &= std::fabs(m.vals[p] / (*h.nat_diag)[m.cols[p]]) <= kMergeMaxAbs;
        if (!fits) {
          for (int l = bad[g]; lev[i] < l && !bad[g].compare_exchange_weak(l, lev[i]);) {
          }
          continue;
        }
        const size_t at = o.ci.size();
        key.clear();
        for (int p = 0; p < (int)m.cols.size(); p++) {
          const int j = m.cols[p], l = lev[j];
          if (l >= l0) {
            o.ci.push_back(-2 - j);
            o.cv.push_back(m.vals[p] / (*h.nat_diag)[j]);
          } else {
            key.push_back(((unsigned long long)l << kKeyLevel) | ((unsigned long long)j << kKeyPos) |
                          (unsigned)p);
          }
        }
        std::sort(key.begin(), key.end());
        for (unsigned long long q : key) {
          const int p = (int)(q & ((1u << kKeyPos) - 1));
          o.ci.push_back(m.cols[p]);
          o.cv.push_back(m.vals[p]);
        }
        len[s - out.m0] = (int)(o.ci.size() - at);
        out.proxy[s - out.m0] =
            row_proxy(g, (int)key.size(), [&](int u) { return grp[(int)(key[u] >> kKeyLevel)]; });
      }
      blk[b].ci.assign(o.ci.begin(), o.ci.end());
      blk[b].cv.assign(o.cv.begin(), o.cv.end());
      if (total.fetch_add((long long)o.ci.size()) + (long long)o.ci.size() > most) over = true;
    }
  });
  if (over) return false;
  par_prefix((size_t)M, [&](size_t s) { return len[s]; }, out.rp);
  out.ci.resize(out.rp[M]);
  out.cv.resize(out.rp[M]);
  par_for((size_t)B, [&](size_t b0, size_t b1) {
    for (size_t b = b0; b < b1; b++) {
      const int o = out.rp[b * kBlk];
      std::copy(blk[b].ci.begin(), blk[b].ci.end(), out.ci.begin() + o);
      std::copy(blk[b].cv.begin(), blk[b].cv.end(), out.cv.begin() + o);
    }
  }, 64);
  return true;
}

// The groups and merged rows of one sweep within the limits (empty when no two
// levels are worth merging).  A group with rows that cannot be merged (longer
// than kMergeMaxRow, a coefficient too large) is cut where the lowest
// of them stands, up to kMergeCuts times; what is left of it then stays as its
// plain levels.  False: more merged entries than kMergeMaxGrowth allows.
bool plan_within(const HostSweep &h, size_t n, const IntVec &lev, const MergeLimits &lim,
                 MergePlan &out) {
  const std::vector<int> &lp = h.level_ptr;
  const int nl = h.nlevels;
  out = MergePlan();
  // groups, in runs of levels of about equal work planned in parallel (a
  // fixed number, so the plan does not depend on the threads): half of a
  // run's share counted in entries, half in levels, since the narrow levels
  // hold few entries and most of the planning
  {
    const long long total = h.rp[n];
    const int S = (int)std::max<long long>(1, std::min<long long>({16, total / 500000, nl / 8}));
    std::vector<int> cut{0};
    for (int k = 1; k < S; k++) {
      const double goal = (double)k / S;
      int l = cut.back();
      while (l < nl && 0.5 * ((double)h.rp[lp[l]] / total + (double)l / nl) < goal) l++;
      if (l > cut.back() && l < nl) cut.push_back(l);
    }
    cut.push_back(nl);
    const int R = (int)cut.size() - 1;
    std::vector<std::vector<int>> part(R);
    std::atomic<int> next{0};
    par_run(std::min(host_threads(), R), [&](int) {
      for (int k; (k = next.fetch_add(1)) < R;)
        plan_groups(h, lev, cut[k], cut[k + 1], lim, part[k]);
    });
    for (auto &p : part) out.gptr.insert(out.gptr.end(), p.begin(), p.end());
    out.gptr.push_back(nl);
  }
  IntVec grp(nl);  // group of each level
  for (int cuts = 0;; cuts++) {
    const int G = (int)out.gptr.size() - 1;
    if (G == nl) {
      out = MergePlan();
      return true;
    }
    int first = -1, last = -1;
    for (int g = 0; g < G; g++) {
      for (int l = out.gptr[g]; l < out.gptr[g + 1]; l++) grp[l] = g;
      if (out.gptr[g + 1] - out.gptr[g] > 1) {
        if (first < 0) first = g;
        last = g;
      }
    }
    out.m0 = lp[out.gptr[first] + 1];  // a group's first level reads nothing inside it
    out.m1 = lp[out.gptr[last + 1]];
    std::vector<std::atomic<int>> bad(G);
    for (auto &l : bad) l = nl;
    if (!merge_rows(h, n, lev, grp, lim.ratio, bad, out)) {
      out = MergePlan();
      return false;
    }
    std::vector<int> gptr;
    for (int g = 0; g < G; g++) {
      gptr.push_back(out.gptr[g]);
      if (bad[g] == nl) continue;
      for (int l = bad[g]; l < (cuts < kMergeCuts ? bad[g] + 1 : out.gptr[g + 1]); l++)
        gptr.push_back(l);
    }
    gptr.push_back(nl);
    const bool done = gptr.size() == out.gptr.size();
    out.gptr = std::move(gptr);
    if (done) break;
  }
  // the sweep's estimate: a handshake per group and the entries it reads
  long long ents = h.rp[n] + (long long)out.ci.size();
  for (int s = out.m0; s < out.m1; s++)
    if (out.rp[s - out.m0 + 1] > out.rp[s - out.m0]) ents -= h.rp[s + 1] - h.rp[s];
  out.est_us = (out.gptr.size() - 1) * kHopUs + ents * kEntryUs;
  return true;
}

// Merge plan of one sweep (empty when no two levels are worth merging).
void plan_merge(const HostSweep &h, size_t n, const MergeLimits &lim, MergePlan &out) {
  const std::vector<int> &lp = h.level_ptr;
  const int nl = h.nlevels;
  out = MergePlan();
  if (nl < 2 || nl > lim.levels || !merge_signs(h, n)) return;
  IntVec lev(n);
  par_for((size_t)nl, [&](size_t l0, size_t l1) {
    for (size_t l = l0; l < l1; l++)
      for (int s = lp[l]; s < lp[l + 1]; s++) lev[h.slot_row[s]] = (int)l;
  }, 32);
  // too many merged entries: rows of at most the mean that the limit leaves,
  // then half as long, and so on (each attempt stops at the limit)
  const double share = (double)kMergeMaxGrowth * ((double)h.rp[n] + (double)n) / (double)n;
  for (MergeLimits l = lim; l.len >= kMergeMinLen; l.len = std::min(0.5 * l.len, share))
    if (plan_within(h, n, lev, l, out)) return;
}

// One sweep as the device runs it: groups in order, a merged row from the
// rows of earlier groups and right-hand sides, any other row as it is.
// Checks that a row reads only rows of earlier groups.
int simulate_merge(const HostSweep &h, const MergePlan &p, size_t n, const double *rhs, double *x) {
  const std::vector<int> &lp = h.level_ptr;
  std::vector<char> done(n, 0);
  std::vector<int> gp = p.gptr;
  if (!p.any()) {
    gp.resize(h.nlevels + 1);
    for (int l = 0; l <= h.nlevels; l++) gp[l] = l;
  }
  for (size_t g = 0; g + 1 < gp.size(); g++) {
    for (int s = lp[gp[g]]; s < lp[gp[g + 1]]; s++) {
      const int i = h.slot_row[s];
      const bool merged = s >= lp[gp[g] + 1];
      const int k = s - p.m0;
      const int e0 = merged ? p.rp[k] : h.nat_rp[i], e1 = merged ? p.rp[k + 1] : h.nat_rp[i + 1];
      double acc = 0.0;
      for (int e = e0; e < e1; e++) {
        const int j = merged ? p.ci[e] : h.nat_ci[e];
        if (j < 0) {
          acc += p.cv[e] * rhs[-2 - j];
          continue;
        }
        if (!done[j])
          return fail(RCHOL_AMD_EINVAL, "merged row %d reads row %d of its own or a later group", i, j);
        acc += (merged ? p.cv[e] : h.nat_cv[e]) * x[j];
      }
      x[i] = (rhs[i] - acc) / (*h.nat_diag)[i];
    }
    for (int s = lp[gp[g]]; s < lp[gp[g + 1]]; s++) done[h.slot_row[s]] = 1;
  }
  return RCHOL_AMD_OK;
}
