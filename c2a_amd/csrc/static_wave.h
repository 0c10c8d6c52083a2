// static_wave.h -- the depth-first static queries whose entry test does not
// change during the search (the triangle-contact form of C2A_Collide,
// C2A_Tolerance with qsize <= 2, C2A_Distance_At_ContactSpace;
// C2A/src/C2A_PQP.cpp:798-968, :1282-1604) with one wavefront per query.
//
// Which pairs such a search enters depends on the pair alone, so the
// wavefront expands the next 32 pairs of the depth-first order at once, one
// child per lane.  What the order decides -- the contact list's order, the
// first pair found and the test counts up to it -- follows from the pairs'
// visiting keys: one bit per level from the top, 0 for the child visited
// first, so keys compare as the reference's depth-first order does.
//
// Why: with one thread per query (static_query.h) a batch takes as long as
// its longest search on one lane, and the lanes of a wavefront wait for each
// other in every branch.  MI355X, host to host, two 8192-triangle knots:
// 2048 contact lists 194 ms with one thread and 8.9 ms with one wavefront per
// query, 4096 tolerance queries 8.0 and 0.7 ms (with the workspace kept
// between calls).  A single query is one lane's search against 32 pairs a turn
// and a second pass for the counts: 24 contact-space queries one by one 0.87
// and 0.27 ms on average, the shortest 0.16 and 0.22.
//
// Stack bound: a batch pops the stack's top, so pairs of depth d are pushed
// only when every deeper one has been popped, by at most 32 parents of depth
// d - 1 each leaving one more pair than it was: at most 32 * depth + 1 pairs
// wait at any time.
#pragma once

#include "ccd_core.h"
#include "static_query.h"

namespace c2a {

// Keys have 64 bits, one per level.
constexpr int kSqWaveDepth = 62;
// Contact lists up to this length are kept sorted by the wavefront.
constexpr int kSqWavePairs = 2048;

struct SqWaveEntry {   // a pair waiting to be expanded
  double R[9], T[3];
  uint64_t key;
  int32_t b1, b2, lev, pad;
};

struct SqHit {         // a contact found
  uint64_t key;
  int32_t t1, t2;
};

// Per-wavefront LDS.
struct SqWaveLds {
  double Rrel[9], Trel[3];
  double d, p[3], q[3];   // the first pair found (tolerance, contact space)
  int32_t t1, t2;
  int64_t ticket;
};

// Per-wavefront workspace: the stack, then (contact lists) two hit buffers.
C2A_HD int64_t sq_wave_stack(int depth_sum) { return 32 * ((int64_t)depth_sum + 1) + 64; }
C2A_HD int64_t sq_wave_hits(int kind, int pair_cap) {
  return kind == SQ_COLLIDE ? 2 * (int64_t)pair_cap + 64 : 0;
}
C2A_HD int64_t sq_wave_bytes(int kind, int depth_sum, int pair_cap) {
  return sq_wave_stack(depth_sum) * (int64_t)sizeof(SqWaveEntry) +
         2 * sq_wave_hits(kind, pair_cap) * (int64_t)sizeof(SqHit);
}

// Orders the n hits by key and keeps the first `keep`; returns the number
// kept.  Every lane counts the smaller keys of its hits.
C2A_HD int sq_sort_hits(SqHit* hits, SqHit* tmp, int n, int keep, int lane) {
  for (int i = lane; i < n; i += 64) {
    const SqHit h = hits[i];
    int r = 0;
    for (int k = 0; k < n; k++) r += hits[k].key < h.key ? 1 : 0;
    if (r < keep) tmp[r] = h;
  }
  mem_sync();
  const int m = n < keep ? n : keep;
  for (int i = lane; i < m; i += 64) hits[i] = tmp[i];
  mem_sync();
  return m;
}

// 64-bit value of one lane in every lane.
C2A_HD uint64_t lane_read64(uint64_t v, int src) {
  return ((uint64_t)(uint32_t)lane_read((int32_t)(v >> 32), src) << 32) |
         (uint32_t)lane_read((int32_t)(uint32_t)v, src);
}

// One search over a query.  best: visiting key of the first pair found so far
// (all ones: none); pairs behind it are not entered.  count = false looks for
// the first pair, or lists the contacts; count = true counts the tests made
// up to the final best.
template <int KIND>
C2A_HD void sq_wave_search(const StaticArgs& a, SqWaveLds& g, const MeshDev& M1,
                           const MeshDev& M2, const StaticQueryDev& q, SqWaveEntry* st,
                           SqHit* hits, SqHit* tmp, bool count, uint64_t& best, int64_t& bv,
                           int64_t& tri, int& found, int& nhits, int lane) {
  const GpuNode* N1 = M1.nodes;
  const GpuNode* N2 = M2.nodes;
  node_ptr G1 = nodes_of(M1), G2 = nodes_of(M2);
  const double lim = (KIND == SQ_TOLERANCE && q.param < 0.0) ? 0.0 : q.param;   // :1786
  const bool list = KIND == SQ_COLLIDE && a.flag != 2;
  uint64_t last = ~0ull;   // contacts behind this key are past the list's end
  nhits = 0;
  bv = 0;
  tri = 0;
  found = 0;
  // the pair a lane tests: the root (first turn), then one child of a pair
  double R[9], T[3], Rr[9], Tr[3];
  sq_root(N1, N2, q, Rr, Tr, R, T);
  if (lane == 0) {
    for (int i = 0; i < 9; i++) g.Rrel[i] = Rr[i];
    for (int i = 0; i < 3; i++) g.Trel[i] = Tr[i];
  }
  lane_sync();
  int n = 0;
  for (bool root = true; root || n > 0; root = false) {
    int b1 = 0, b2 = 0, lev = 0;
    uint64_t key = 0;
    bool act = lane == 0;
    if (!root) {
      const int np = n < 32 ? n : 32;
      act = (lane >> 1) < np;
      C2A_CHECK(n <= sq_wave_stack(a.depth_sum));
      const SqWaveEntry C2A_GLOBAL* e = gp(st) + (n - 1 - (act ? lane >> 1 : 0));
      for (int i = 0; i < 9; i++) R[i] = e->R[i];
      for (int i = 0; i < 3; i++) T[i] = e->T[i];
      key = e->key;
      b1 = e->b1;
      b2 = e->b2;
      lev = e->lev;
      n -= np;
      mem_sync();   // entries are read before new ones take their places
      act = act && key <= best;
      if (KIND != SQ_COLLIDE)   // two tests per pair expanded
        bv += 2 * (int64_t)__builtin_popcountll(wave_ballot(act && !(lane & 1)));
      NodeHead h1 = head_of(G1 + b1), h2 = head_of(G2 + b2);
      descend_h(G1, G2, b1, b2, h1, h2, lane & 1, R, T);
      lev++;
    }
    node_ptr A = G1 + b1, B = G2 + b2;
    const int fc1 = A->first_child, fc2 = B->first_child;
    const bool leaf = fc1 < 0 && fc2 < 0;
    const double rr = A->r + B->r;
    double S[3];
    const double la[2] = {A->l[0], A->l[1]}, lb[2] = {B->l[0], B->l[1]};
    double d = rect_dist(R, T, la, lb, S);
    bool enter, second = (lane & 1) != 0;
    if (KIND == SQ_COLLIDE) {
      enter = d <= rr;   // BV_Overlap (:807); the first child first
    } else {
      d -= rr;
      d = (d < 0.0) ? 0.0 : d;
      const double ds = lane_xor1d(d, lane);   // the closer child first
      second = (lane & 1) ? !(d < ds) : ds < d;
      // the contact-space search enters its root untested (:1410)
      enter = KIND == SQ_TOLERANCE ? d <= lim : (root || d < lim);
    }
    if (!root && second) key |= 1ull << (64 - lev);
    act = act && key <= best;
    if (KIND == SQ_COLLIDE) bv += __builtin_popcountll(wave_ballot(act));   // one per pair popped
    enter = enter && act;
    const bool test = enter && leaf;
    const uint64_t testm = wave_ballot(test);
    tri += __builtin_popcountll(testm);
    if (testm && !count) {
      bool hit = false;
      const int t1 = -fc1 - 1, t2 = -fc2 - 1;
      double p[3], qq[3], dt = 0.0;
      if (test) {
        double ta[9], tb[9], Rg[9], Tg[3];
        gdouble_ptr g1 = tris_of(M1) + 9 * (int64_t)t1;
        gdouble_ptr g2 = tris_of(M2) + 9 * (int64_t)t2;
        for (int i = 0; i < 9; i++) {
          ta[i] = g1[i];
          tb[i] = g2[i];
          Rg[i] = g.Rrel[i];
        }
        for (int i = 0; i < 3; i++) Tg[i] = g.Trel[i];
        if (KIND == SQ_COLLIDE) {
          double qv[9];
          mxvpv(qv + 0, Rg, tb + 0, Tg);
          mxvpv(qv + 3, Rg, tb + 3, Tg);
          mxvpv(qv + 6, Rg, tb + 6, Tg);
          hit = tri_contact(ta, ta + 3, ta + 6, qv, qv + 3, qv + 6);
        } else {
          dt = tri_distance(Rg, Tg, ta, tb, p, qq, nullptr);
          hit = KIND == SQ_TOLERANCE ? dt <= lim : dt < lim;
        }
      }
      const uint64_t hm = wave_ballot(hit), sm = wave_ballot(second);
      if (hm && list) {
        found += (int)__builtin_popcountll(hm);
        const uint64_t km = wave_ballot(hit && a.pair_cap > 0 && key <= last);
        if (hit && ((km >> lane) & 1)) {
          SqHit C2A_GLOBAL* o = gp(hits) + nhits + lanes_below(km, lane);
          o->key = key;
          o->t1 = t1;
          o->t2 = t2;
        }
        nhits += (int)__builtin_popcountll(km);
        mem_sync();
        if (nhits > 2 * a.pair_cap) {   // the list's candidates so far
          nhits = sq_sort_hits(hits, tmp, nhits, a.pair_cap, lane);
          last = hits[nhits - 1].key;
          mem_sync();
        }
      } else if (hm) {
        // the earliest: lanes hold pairs in visiting order, children by `second`
        int w = (int)__builtin_ctzll(hm);
        if (!(w & 1) && ((hm >> (w + 1)) & 1) && ((sm >> w) & 1)) w++;
        const uint64_t hk = lane_read64(key, w);
        if (found == 0 || hk < best) {
          best = hk;
          found = 1;
          lane_sync();
          if (lane == w) {
            g.d = dt;
            for (int i = 0; i < 3 && KIND != SQ_COLLIDE; i++) {
              g.p[i] = p[i];
              g.q[i] = qq[i];
            }
            g.t1 = t1;
            g.t2 = t2;
          }
          lane_sync();
        }
      }
    }
    const bool push = enter && !leaf && key <= best;
    const uint64_t pm = wave_ballot(push);
    const int total = (int)__builtin_popcountll(pm);
    if (push) {
      const int pair = lane & ~1;
      const int rank = (int)__builtin_popcountll(pm & ((1ull << pair) - 1)) +
                       ((second && ((pm >> (lane ^ 1)) & 1)) ? 1 : 0);
      SqWaveEntry C2A_GLOBAL* e = gp(st) + (n + total - 1 - rank);
      for (int i = 0; i < 9; i++) e->R[i] = R[i];
      for (int i = 0; i < 3; i++) e->T[i] = T[i];
      e->key = key;
      e->b1 = b1;
      e->b2 = b2;
      e->lev = lev;
    }
    n += total;
    mem_sync();
  }
}

// One query; ws: this wavefront's sq_wave_bytes.
template <int KIND>
C2A_HD void sq_wave_query(const StaticArgs& a, int64_t qi, SqWaveLds& g, unsigned char* ws,
                          int lane) {
  const StaticQueryDev& q = a.q[qi];
  const MeshDev& M1 = a.meshes[q.mesh[0]];
  const MeshDev& M2 = a.meshes[q.mesh[1]];
  SqWaveEntry* st = (SqWaveEntry*)ws;
  SqHit* hits = (SqHit*)(ws + sq_wave_stack(a.depth_sum) * (int64_t)sizeof(SqWaveEntry));
  SqHit* tmp = hits + sq_wave_hits(KIND, a.pair_cap);
  uint64_t best = ~0ull;
  int64_t bv, tri;
  int found, nhits, dummy;
  sq_wave_search<KIND>(a, g, M1, M2, q, st, hits, tmp, false, best, bv, tri, found, nhits, lane);
  const bool list = KIND == SQ_COLLIDE && a.flag != 2;
  if (!list && found) {
    uint64_t b = best;
    int f;
    sq_wave_search<KIND>(a, g, M1, M2, q, st, hits, tmp, true, b, bv, tri, f, dummy, lane);
  }
  if (KIND == SQ_COLLIDE) {
    int32_t C2A_GLOBAL* pl = gp(a.pairs) + 2 * (int64_t)a.pair_cap * qi;
    if (list) {
      nhits = sq_sort_hits(hits, tmp, nhits, a.pair_cap, lane);
      for (int i = lane; i < nhits; i += 64) {
        pl[2 * i] = hits[i].t1;
        pl[2 * i + 1] = hits[i].t2;
      }
    } else if (found && a.pair_cap > 0 && lane == 0) {
      pl[0] = g.t1;
      pl[1] = g.t2;
    }
  }
  if (lane == 0) {
    StaticOut o;
    const bool pts = KIND != SQ_COLLIDE && found;
    o.distance = pts ? g.d : (KIND == SQ_DISTANCE_CS ? q.param : 0.0);
    double u[3], p2[3] = {0.0, 0.0, 0.0};
    if (pts) {   // p2 into model 2's frame (C2A_PQP.cpp:1043-1047)
      const double Rr[9] = {g.Rrel[0], g.Rrel[1], g.Rrel[2], g.Rrel[3], g.Rrel[4],
                            g.Rrel[5], g.Rrel[6], g.Rrel[7], g.Rrel[8]};
      sub3(u, g.q, g.Trel);
      mtxv(p2, Rr, u);
    }
    for (int i = 0; i < 3; i++) {
      o.p1[i] = pts ? g.p[i] : 0.0;
      o.p2[i] = p2[i];
    }
    o.bv_tests = bv;
    o.tri_tests = tri;
    o.tri[0] = pts ? g.t1 : (KIND == SQ_TOLERANCE ? -1 : q.seed[0]);
    o.tri[1] = pts ? g.t2 : (KIND == SQ_TOLERANCE ? -1 : q.seed[1]);
    o.found = found;
    o.flags = 0;
    a.out[qi] = o;
  }
  lane_sync();
}

}  // namespace c2a
