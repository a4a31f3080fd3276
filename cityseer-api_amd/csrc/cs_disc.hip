// cs_disc.hip -- shortest-path centrality, one workgroup per source with the
// search's distances in LDS.
//
// The search settles rounds of nodes in parallel. With L the smallest (seconds
// + shortest in-edge) over the discovered, unsettled nodes, nothing relaxed from
// now on offers less than L, so every node below L by more than the widest tie
// band of a fold is final and no offer still to come can reach its band; they
// settle together. When L leaves no such node (a very short edge at the front)
// the first node in settle order settles alone, the serial search's own step. A
// round is as wide as the front's own edges allow, not as the network's shortest
// edge does.
//
//  * A settling node's row (in- and out-edge of each neighbour side by side,
//    four neighbours per 64-byte block, four lanes per block) serves both
//    directions at once: the in-edges offer seconds to the neighbours (an LDS
//    atomic min), the out-edges to neighbours already settled before it are the
//    candidates of its predecessor fold (centrality.rs:1413-1437), whose order
//    only matters between candidates within the tie band. One such candidate,
//    the usual case, is the predecessor; several replay the fold in settle order.
//  * LDS holds 4 bytes per node of the touched pages (runs of 2^ps nodes of the
//    Hilbert order, found through a byte table): no per-source clearing, and the
//    result passes walk nodes in address order, 64 neighbouring words per atomic.
//  * Betweenness keeps 8 bytes per settled node in scratch and back-propagates
//    (centrality.rs:823-873) one (threshold, kind) array per wave, dependencies
//    in LDS over the distances, for the nodes that precede another only.
//
// A round is a chain of LDS and L2 round trips (front, page, distance, offer):
// waits are 75% of a wave's cycles on the city below; workgroups in flight hide them, so
// the layout counts LDS in the units a CU gives out. Against a wave per source
// with its state in scratch (cs_search.hip), kernel ms: 32,400 sources, four
// thresholds to 5,000 m, both measures (reach 3,960) 24.8 -> 19.3; 30,406
// sources, closeness to 800 m on 20 m pieces (reach 1,003) 3.85 -> 2.42; 676
// sources to 800 m (reach 93) 0.122 -> 0.079; 64 sources 0.089 -> 0.046.
#include "cs_internal.hpp"
#include "cs_wave.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace cs {

namespace {

constexpr uint32_t kQuad = 4;                 // neighbours of a row block = lanes of an item
constexpr uint32_t kMaxBlocks = 4;            // row blocks of a node at most (16 neighbours)
constexpr uint32_t kMaxWaves = 4;
constexpr uint32_t kNoNb = 0x3fffffffu;       // padding entry of a row
constexpr uint32_t kNone = 0xffu, kClaimed = 0xfeu;  // page table: not touched, being opened
constexpr uint32_t kMaxPages = 253;
constexpr uint32_t kStart = 0x8000u;          // record: first node of a round
constexpr uint32_t kMulti = 0xffffu;          // record: several predecessors
constexpr uint32_t kNoSlot = 0x7fffu;         // record: no predecessor (the source)
constexpr uint32_t kMaxSlots = 0x7ff0u;
constexpr uint32_t kInf = 0x7f800000u;
constexpr uint32_t kFailRoom = 1u, kFailInternal = 2u;

// One (graph, request) pair of a launch.
struct DiscJob {
  const uint4 *row;       // [N][blocks][4] {neighbour | counts << 30, seconds neighbour->node, seconds
                          // node->neighbour, neighbour's shortest in-edge | its further blocks in the low bits}
  const uint32_t *orig;   // original index of each node (exact ties)
  const uint8_t *eligible;
  const uint32_t *sources;
  const float *src_wt, *src_cyc;
  double *acc;            // [7][tstride][N]
  uint32_t *reach;
  uint32_t N, blocks, tstride, flags;  // 1 closeness, 2 betweenness, 4 track reach
  float maxsec, speed, clear;
  double far_max;
  float dist[kMaxT];      // beyond the job's own thresholds: -1
  float beta[kMaxT];
};
typedef __attribute__((address_space(4))) const DiscJob CDiscJob;

struct DiscArgs {
  const DiscJob *jobs;
  const uint2 *items;     // {job, source position}; null: job 0, position = item
  uint32_t n_items;
  uint32_t P, ps, F, S;   // pages, page shift, front entries, settled nodes of a source at most
  uint32_t n_pt;          // page table bytes (a multiple of 4)
  uint32_t maxp;          // predecessors of a node at most
  uint32_t o_front, o_items, o_bits, o_pt, o_pl;  // LDS offsets (distances at 0)
  uint32_t dcap;          // f64 words of the back-propagation overlay (from 0 up to the bits)
  uint32_t o_iid, o_ext, o_ratio;  // scratch offsets (records at 0)
  char *ws;               // [blocks][stride] scratch, never cleared
  size_t stride;
  unsigned long long *stats;
  uint32_t *next;         // [kXcd] item counters
  uint32_t xbeg[kXcd + 1];
  uint32_t *fail_list, *n_fail, *fail_flags;
  uint32_t *progress;
};

// LDS control words of a workgroup.
struct Ctl {
  unsigned long long first;  // single step: {original index << 32 | slot} of the first node
  uint32_t lim[2], low[2];   // smallest (seconds + in-edge) and smallest seconds of the front, by round parity
  uint32_t cnt[2];           // entries of the front being built
  uint32_t ns, np, ni, nmulti, fail, item;
  uint32_t nband[kMaxT], eband[kMaxT];
};

// A workgroup barrier for LDS: no wait for the scratch stores under way.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// Orders one wave's memory accesses for the compiler (the hardware keeps one
// wave's accesses to an address in order).
__device__ __forceinline__ void order() {
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) { return __ockl_wfred_min_u32(v); }
__device__ __forceinline__ float fbits(uint32_t b) { return __uint_as_float(b); }
// f32 exponential of the reference's host library (see cs_search.hip).
__device__ __forceinline__ float exp_host(float x) { return (float)exp((double)x); }

// Front entry: slot | further row blocks << 16 | upper 14 bits of a lower bound
// on the node's shortest in-edge.
__device__ __forceinline__ uint32_t front_entry(uint32_t slot, uint32_t wm) {
  return slot | ((wm & 3u) << 16) | (wm & 0xfffc0000u);
}

struct Disc {
  uint32_t *D;        // LDS [P << ps] seconds of each node (f32 bits), infinite: not reached
  uint32_t *front;    // LDS [2][F]
  uint8_t *its;       // LDS [waves][256] items of a wave: lane | block << 6
  uint32_t *cand;     // LDS [waves][64] candidates of each settling node: count << 20 + slots
  uint32_t *bits;     // LDS node precedes another
  uint8_t *pt;
  uint32_t *pl;       // LDS page number of each touched page
  Ctl *c;
  char *ws;
};

__device__ __forceinline__ uint32_t node_of(const DiscArgs &a, const Disc &q, uint32_t slot) {
  return (q.pl[slot >> a.ps] << a.ps) | (slot & ((1u << a.ps) - 1u));
}

// Page of a node for the lanes that `want` it, opened where it has not been
// touched: one lane claims the table byte, clears the page and publishes it;
// lanes that meet a claimed byte look again (the claimant never waits).
__device__ __forceinline__ uint32_t open_pages(const DiscArgs &a, const Disc &q, uint32_t pg, bool want) {
  const uint32_t lane = lane_id();
  uint32_t b = want ? lds_ld8(&q.pt[pg]) : 0u;
  while (__ballot(want && b >= kClaimed)) {
    uint32_t id = kNone;
    if (want && b == kNone) {
      uint32_t *word = reinterpret_cast<uint32_t *>(q.pt) + (pg >> 2);
      const uint32_t sh = (pg & 3u) * 8u;
      uint32_t w = lds_ld(word);
      if (((w >> sh) & 0xffu) == kNone &&
          __hip_atomic_compare_exchange_strong(word, &w, w & ~(1u << sh), __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP)) {
        id = lds_add(&q.c->np, 1u);
        if (id >= a.P) {  // no room: the source fails; a harmless page lets the others go on
          lds_or(&q.c->fail, kFailRoom);
          id = 0x100u;
        } else {
          q.pl[id] = pg;
        }
      }
    }
    // the claimed pages, cleared by the whole wave, then published
    for (uint64_t m = __ballot(id < kNone); m; m &= m - 1) {
      const uint32_t p = (uint32_t)__builtin_amdgcn_readlane(id, __builtin_ctzll(m));
      for (uint32_t i = lane; i < (1u << a.ps); i += kWave) q.D[(p << a.ps) + i] = kInf;
    }
    order();
    if (id != kNone) lds_st8(&q.pt[pg], (uint8_t)(id & 0xffu));
    order();
    if (want && b >= kClaimed) b = lds_ld8(&q.pt[pg]);
  }
  return b;
}

// The reference's ordered fold over the near candidates of node v (two or more;
// centrality.rs:1413-1437), by one lane: selection passes in settle order
// (seconds, original index), parallel edges in row order. Leaves the
// predecessors' slots in x: count, slots. False when the fold does not end at
// the node's seconds.
__device__ bool fold_several(const DiscArgs &a, CDiscJob &j, const Disc &q, uint32_t v, uint32_t nblk, float sv,
                             uint32_t n_near, uint16_t *x) {
  const float one_m = 1.0f - kTieEps, one_p = 1.0f + kTieEps;
  const uint4 *row = j.row + (size_t)v * j.blocks * kQuad;
  const uint32_t deg = nblk * kQuad;
  const double thr = (double)sv * j.far_max;
  float best = INFINITY, lsu = 0.0f;
  uint32_t mask = 0, lo = 0, lj = 0;
  bool have = false;
  for (uint32_t step = 0; step < n_near; ++step) {
    bool found = false;
    float psu = INFINITY, pcs = 0.0f;
    uint32_t po = 0, pj = 0, pu = 0;
    for (uint32_t k = 0; k < deg; ++k) {
      const uint4 e = row[k];
      const uint32_t u = e.x & kNoNb;
      if (u == kNoNb || u == v) continue;
      const uint32_t pg = lds_ld8(&q.pt[u >> a.ps]);
      if (pg >= kClaimed) continue;
      const float su = fbits(lds_ld(&q.D[(pg << a.ps) | (u & ((1u << a.ps) - 1u))]));
      if (!(su <= sv)) continue;
      const uint32_t ou = j.orig[u];
      if (su == sv && !(ou < j.orig[v])) continue;
      const float cs = su + fbits(e.z);
      if (!(cs <= j.maxsec) || (double)cs > thr) continue;
      if (have && !(lsu < su || (lsu == su && (lo < ou || (lo == ou && k > lj))))) continue;
      if (!found || su < psu || (su == psu && (ou < po || (ou == po && k < pj)))) {
        found = true;
        psu = su;
        pcs = cs;
        po = ou;
        pj = k;
        pu = u;
      }
    }
    if (!found) return false;
    if (pcs < best) {
      mask = pcs < best * one_m ? 1u << pj : mask | (1u << pj);
      best = pcs;
    } else if (pcs <= best * one_p) {
      bool has = false;
      for (uint32_t k = 0; k < deg; ++k)
        if (((mask >> k) & 1u) && (row[k].x & kNoNb) == pu) has = true;
      if (!has) mask |= 1u << pj;
    }
    have = true;
    lsu = psu;
    lo = po;
    lj = pj;
  }
  uint32_t n = 0;
  for (uint32_t k = 0; k < deg; ++k)
    if ((mask >> k) & 1u) {
      const uint32_t u = row[k].x & kNoNb;
      st_u16(&x[1 + n++], (uint16_t)((lds_ld8(&q.pt[u >> a.ps]) << a.ps) | (u & ((1u << a.ps) - 1u))));
    }
  st_u16(&x[0], (uint16_t)n);
  return best == sv;
}

// A settled node that takes its place as a predecessor gets the next number
// among the inner nodes, once.
__device__ __forceinline__ void number_inner(const DiscArgs &a, const Disc &q, uint32_t slot) {
  const uint32_t b = 1u << (slot & 31u);
  if (!(__hip_atomic_fetch_or(&q.bits[slot >> 5], b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & b))
    st_u16(reinterpret_cast<uint16_t *>(q.ws + a.o_iid) + slot, (uint16_t)lds_add(&q.c->ni, 1u));
}

// The job's fields a round reads, held in registers over the search (left to
// itself the compiler loads them again at each use, 17 scalar loads and their
// waits per wave and round).
template <int NT>
struct Hot {
  const uint4 *row;
  const uint32_t *orig;
  const uint8_t *eligible;
  uint32_t blocks, flags;
  float maxsec, speed;
  double far_max;
  float dist[NT];
};
template <typename T>
__device__ __forceinline__ T held(T x) {
  if constexpr (sizeof(T) == 8) {
    uint64_t b = __builtin_bit_cast(uint64_t, x);
    asm volatile("" : "+s"(b));
    return __builtin_bit_cast(T, b);
  } else {
    uint32_t b = __builtin_bit_cast(uint32_t, x);
    asm volatile("" : "+s"(b));
    return __builtin_bit_cast(T, b);
  }
}

// Settles and relaxes the wave's selected lanes (slot, seconds, further blocks);
// newly reached nodes join the front `nxt` (its count in *cnt). ns0: settled
// nodes when the round began.
template <int NT>
__device__ __forceinline__ void settle(const DiscArgs &a, CDiscJob &j, const Hot<NT> &h, const Disc &q, bool sel, uint32_t slot,
                                       uint32_t more, uint32_t sb, uint32_t ns0, uint32_t *nxt, uint32_t *cnt,
                                       uint32_t (&eband)[NT], uint32_t &st_edges) {
  const uint32_t lane = lane_id(), wib = threadIdx.x / kWave;
  const bool betw = (h.flags & 2u) != 0, close = (h.flags & 1u) != 0;
  uint8_t *its = q.its + wib * 256;
  uint32_t *cand = q.cand + wib * kWave;
  const uint64_t ms = __ballot(sel), m1 = __ballot(sel && (more & 1u)), m2 = __ballot(sel && (more & 2u));
  const uint32_t n = (uint32_t)__popcll(ms);
  const uint32_t tot = n + (uint32_t)__popcll(m1) + 2u * (uint32_t)__popcll(m2);
  uint32_t base = 0;
  if (lane == 0) base = lds_add(&q.c->ns, n);
  const uint32_t v = sel ? node_of(a, q, slot) : 0u;
  uint32_t el = 0;
  if (sel) {
    const uint32_t at = rank_below(ms) + rank_below(m1) + 2u * rank_below(m2);
    for (uint32_t k = 0; k <= more; ++k) its[at + k] = (uint8_t)(lane | (k << 6));
    cand[lane] = 0u;
    if (betw) el = h.eligible[v];
  }
  order();
  for (uint32_t c0 = 0; c0 < tot; c0 += kWave / kQuad) {
    const uint32_t k = c0 + lane / kQuad;
    const bool has = k < tot;
    const uint32_t it = has ? its[k] : 0u;
    const uint32_t l = it & 63u;
    const uint32_t sv = (uint32_t)__shfl((int)v, (int)l);
    const uint32_t ss = (uint32_t)__shfl((int)sb, (int)l);
    const float s = fbits(ss);
    uint4 e = make_uint4(kNoNb, kInf, kInf, 0u);
    if (has) e = h.row[((size_t)sv * h.blocks + (it >> 6)) * kQuad + lane % kQuad];
    const uint32_t nb = e.x & kNoNb;
    const bool act = nb != kNoNb;
    const float cs = s + fbits(e.y);
    const bool want = act && cs <= h.maxsec;
    if (act && e.y != kInf) ++st_edges;
    // (a neighbour whose page nobody has opened, or is just opening, is not settled)
    uint32_t page = act ? lds_ld8(&q.pt[nb >> a.ps]) : kNone;
    if (__ballot(want && page >= kClaimed)) {
      const uint32_t opened = open_pages(a, q, nb >> a.ps, want);
      if (want) page = opened;
    }
    const bool there = act && page < kClaimed;
    const uint32_t ns = (page << a.ps) | (nb & ((1u << a.ps) - 1u));
    uint32_t db = kInf;
    if (there) db = lds_ld(&q.D[ns]);
    const float d = fbits(db);
    bool found = false;
    if (want && cs < d) found = lds_min(&q.D[ns], __float_as_uint(cs)) == kInf;
    // neighbours settled before the node: they close its undirected edges
    // (circuit rank) and are its possible predecessors
    bool before = d < s;
    if (there && d == s && nb != sv) before = h.orig[nb] < h.orig[sv];
    if (before) {
      if (close) {
        const uint32_t edges = e.x >> 30;
        if (edges) {
          const float route = s * h.speed;
#pragma unroll
          for (int t = 0; t < NT; ++t) eband[t] += route <= h.dist[t] ? edges : 0u;
        }
      }
      if (betw) {
        const float cp = d + fbits(e.z);
        if (cp <= h.maxsec && (double)cp <= (double)s * h.far_max)
          __hip_atomic_fetch_add(&cand[l], (1u << 20) | ns, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    const uint64_t mf = __ballot(found);
    if (mf) {
      uint32_t fb = 0;
      if (lane == 0) fb = lds_add(cnt, (uint32_t)__popcll(mf));
      fb = uniform(fb) + rank_below(mf);
      if (found) {
        if (fb < a.F) nxt[fb] = front_entry(ns, e.w);
        else lds_or(&q.c->fail, kFailRoom);
      }
    }
  }
  if (!betw) return;
  order();
  // ---- a record per settled node: its predecessor
  base = uniform(base);
  if (sel) {
    const uint32_t idx = base + rank_below(ms);
    const uint32_t x = cand[lane], nn = x >> 20;
    uint32_t pred = x & 0xffffu;
    if (idx >= a.S) {
      lds_or(&q.c->fail, kFailRoom);
    } else {
      if (idx == 0) {
        pred = kNoSlot;
      } else if (nn == 1) {
        number_inner(a, q, pred);
      } else {
        uint16_t *pl = reinterpret_cast<uint16_t *>(q.ws + a.o_ext) + (size_t)slot * (a.maxp + 1);
        if (nn == 0 || !fold_several(a, j, q, v, more + 1u, fbits(sb), nn, pl)) {
          lds_or(&q.c->fail, kFailInternal);
        } else {
          const uint32_t np = ld_u16(&pl[0]);
          for (uint32_t k = 1; k <= np; ++k) number_inner(a, q, ld_u16(&pl[k]));
          pred = np == 1 ? ld_u16(&pl[1]) : kMulti;
          if (np > 1) lds_add(&q.c->nmulti, 1u);
        }
      }
      // seconds are never negative: their sign carries the eligibility
      st64(reinterpret_cast<uint64_t *>(q.ws) + idx,
           ((uint64_t)(sb | (el ? 0x80000000u : 0u)) << 32) | (pred << 16) | slot | (idx == ns0 ? kStart : 0u));
    }
  }
}

// Path counts where some node has several predecessors: by one wave, rounds in
// settle order; the shares of each such node's predecessors go to its ratios.
__device__ __forceinline__ void path_shares(const DiscArgs &a, const Disc &q, uint32_t ns, double *sig) {
  const uint32_t lane = lane_id();
  uint16_t *no = reinterpret_cast<uint16_t *>(q.D);  // path count number of each slot, 0: one path
  uint32_t nsig = 0;
  auto load = [&](uint32_t w) { return w + lane < ns ? ld64(reinterpret_cast<uint64_t *>(q.ws) + w + lane) : 0ull; };
  uint64_t r1 = load(0), r2 = load(kWave);
  for (uint32_t w0 = 0; w0 < ns; w0 += kWave) {
    const uint64_t r = r1;
    r1 = r2;
    r2 = load(w0 + 2 * kWave);
    uint64_t starts = __ballot(w0 + lane < ns && ((uint32_t)r & kStart));
    uint32_t lo = 0;
    const uint32_t end = ns - w0 < kWave ? ns - w0 : kWave;
    while (lo < end) {
      const uint64_t above = lo + 1 < 64 ? starts & ~((2ull << lo) - 1ull) : 0ull;
      uint32_t hi = above ? (uint32_t)__builtin_ctzll(above) : end;
      hi = hi < end ? hi : end;
      const bool on = lane >= lo && lane < hi;
      const uint32_t slot = (uint32_t)r & (kStart - 1u), pred = ((uint32_t)r >> 16) & 0xffffu;
      const bool multi = on && pred == kMulti;
      const uint64_t mm = __ballot(multi);
      uint32_t mine = 0;
      if (on && !multi && pred != kNoSlot) mine = no[pred];
      if (multi) {
        const uint16_t *pl = reinterpret_cast<const uint16_t *>(q.ws + a.o_ext) + (size_t)slot * (a.maxp + 1);
        double *ratio = reinterpret_cast<double *>(q.ws + a.o_ratio) + (size_t)slot * a.maxp;
        const uint32_t np = ld_u16(&pl[0]);
        double s = 0.0;
        for (uint32_t k = 1; k <= np; ++k) {
          const uint32_t c = no[ld_u16(&pl[k])];
          s += c ? ldd(&sig[c - 1]) : 1.0;
        }
        for (uint32_t k = 1; k <= np; ++k) {
          const uint32_t c = no[ld_u16(&pl[k])];
          std_(&ratio[k - 1], (c ? ldd(&sig[c - 1]) : 1.0) / s);
        }
        mine = nsig + rank_below(mm) + 1u;
        std_(&sig[mine - 1], s);
      }
      nsig += (uint32_t)__popcll(mm);
      order();
      if (on) no[slot] = (uint16_t)mine;
      order();
      lo = hi;
    }
  }
}

// One dependency array: threshold t, plain or beta-weighted, for the settled
// nodes before `top`, dependencies dep[0 .. room) of the first `room` inner
// nodes. Leaves each one's credit in its place.
__device__ __forceinline__ void sweep(const DiscArgs &a, CDiscJob &j, const Disc &q, double *dep, uint32_t room,
                                      uint32_t top, float dist, bool weighted, float beta) {
  const uint32_t lane = lane_id();
  const uint16_t *iid = reinterpret_cast<const uint16_t *>(q.ws + a.o_iid);
  for (uint32_t i = lane; i < room; i += kWave) dep[i] = 0.0;
  order();
  if (!top) return;
  // records load two windows ahead, the numbers they name one window ahead
  auto load = [&](int w) {
    return w >= 0 && (uint32_t)w + lane < top ? ld64(reinterpret_cast<uint64_t *>(q.ws) + w + lane) : (uint64_t)kNoSlot << 16;
  };
  uint32_t on = 0xffffu, pn = 0xffffu;
  auto load_ids = [&](uint64_t r) {
    const uint32_t slot = (uint32_t)r & (kStart - 1u), pred = ((uint32_t)r >> 16) & 0xffffu;
    on = pn = 0xffffu;
    if ((q.bits[slot >> 5] >> (slot & 31u)) & 1u) on = ld_u16(&iid[slot]);
    if (pred < kNoSlot) pn = ld_u16(&iid[pred]);
  };
  const int last = (int)((top - 1) & ~(kWave - 1u));
  uint64_t r1 = load(last), r2 = load(last - (int)kWave);
  load_ids(r1);
  for (int w0 = last; w0 >= 0; w0 -= (int)kWave) {
    const uint64_t r = r1;
    const uint32_t own = on, pred = pn;
    r1 = r2;
    r2 = load(w0 - 2 * (int)kWave);
    load_ids(r1);
    const bool in = (uint32_t)w0 + lane < top;
    const uint64_t starts = __ballot(in && ((uint32_t)r & kStart));
    const uint32_t sb = (uint32_t)(r >> 32);
    const float route = fbits(sb & 0x7fffffffu) * j.speed;
    const bool within = in && route <= dist;
    double seed = (sb & 0x80000000u) ? 0.5 : 1.0;
    if (weighted) seed = seed * exp(-(double)beta * (double)route);
    const bool multi = in && (((uint32_t)r >> 16) & 0xffffu) == kMulti;
    uint32_t hi = top - (uint32_t)w0 < kWave ? top - (uint32_t)w0 : kWave;
    while (hi > 0) {
      const uint64_t below = hi < 64 ? starts & ((1ull << hi) - 1ull) : starts;
      const uint32_t lo = below ? 63u - (uint32_t)__builtin_clzll(below) : 0u;
      if (lane >= lo && lane < hi) {
        double total = 0.0;
        if (within) total = seed;
        if (own < room) {
          if (within) total = seed + dep[own];
          dep[own] = within ? total - seed : 0.0;  // the node's credit
        }
        if (total != 0.0) {
          if (pred < room) {
            wadd_f64(&dep[pred], total);
          } else if (multi) {
            const uint32_t slot = (uint32_t)r & (kStart - 1u);
            const uint16_t *pl = reinterpret_cast<const uint16_t *>(q.ws + a.o_ext) + (size_t)slot * (a.maxp + 1);
            const double *ratio = reinterpret_cast<const double *>(q.ws + a.o_ratio) + (size_t)slot * a.maxp;
            const uint32_t np = ld_u16(&pl[0]);
            for (uint32_t k = 1; k <= np; ++k) {
              const uint32_t p = ld_u16(&iid[ld_u16(&pl[k])]);
              if (p < room) wadd_f64(&dep[p], ldd(&ratio[k - 1]) * total);
            }
          }
        }
      }
      order();
      hi = lo;
    }
  }
}

// Next item for a workgroup on XCD x: its own share first, then the others'.
__device__ __forceinline__ uint32_t next_item(const DiscArgs &a, uint32_t x) {
  for (uint32_t k = 0; k < kXcd; ++k) {
    const uint32_t xx = (x + k) % kXcd;
    const uint32_t len = a.xbeg[xx + 1] - a.xbeg[xx];
    if (__hip_atomic_load(&a.next[xx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= len) continue;
    const uint32_t i = atomicAdd(&a.next[xx], 1u);
    if (i < len) return a.xbeg[xx] + i;
  }
  return a.n_items;
}

template <int NT>
__global__ __launch_bounds__(kMaxWaves *kWave) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_disc(DiscArgs a) {
  extern __shared__ __align__(16) char disc_lds[];
  __shared__ Ctl ctl;
  const uint32_t tid = threadIdx.x, B = blockDim.x, lane = lane_id(), wib = uniform(tid / kWave);
  const uint32_t waves = B / kWave;
  Disc q;
  q.D = reinterpret_cast<uint32_t *>(disc_lds);
  q.front = reinterpret_cast<uint32_t *>(disc_lds + a.o_front);
  q.its = reinterpret_cast<uint8_t *>(disc_lds + a.o_items);
  q.cand = reinterpret_cast<uint32_t *>(disc_lds + a.o_items + waves * 256);
  q.bits = reinterpret_cast<uint32_t *>(disc_lds + a.o_bits);
  q.pt = reinterpret_cast<uint8_t *>(disc_lds + a.o_pt);
  q.pl = reinterpret_cast<uint32_t *>(disc_lds + a.o_pl);
  q.c = &ctl;
  q.ws = a.ws + (size_t)blockIdx.x * a.stride;
  for (uint32_t i = tid; i < a.n_pt / 4; i += B) reinterpret_cast<uint32_t *>(q.pt)[i] = 0xffffffffu;
  uint32_t pdone = a.progress && tid == 0 ? __hip_atomic_load(&a.progress[blockIdx.x], __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_SYSTEM) : 0u;
  unsigned long long st_reached = 0, st_within = 0;
  uint32_t st_edges = 0;
  for (;;) {
    __syncthreads();
    if (tid == 0) {
      ctl.item = next_item(a, blockIdx.x % kXcd);
      ctl.lim[0] = ctl.lim[1] = ctl.low[0] = ctl.low[1] = kInf;
      ctl.cnt[0] = ctl.cnt[1] = 0;
      ctl.ns = ctl.np = ctl.ni = ctl.nmulti = ctl.fail = 0;
      ctl.first = ~0ull;
    }
    if (tid < kMaxT) ctl.nband[tid] = ctl.eband[tid] = 0;
    for (uint32_t i = tid; i < ((a.P << a.ps) + 31) / 32; i += B) q.bits[i] = 0;
    __syncthreads();
    const uint32_t item = uniform(ctl.item);
    if (item >= a.n_items) break;
    uint32_t job = 0, si = item;
    if (a.items) {
      const uint2 it = a.items[item];
      job = uniform(it.x);
      si = uniform(it.y);
    }
    CDiscJob &j = ((CDiscJob *)a.jobs)[job];
    const uint32_t src = j.sources[si];
    Hot<NT> h;
    h.row = held(j.row);
    h.orig = held(j.orig);
    h.eligible = held(j.eligible);
    h.blocks = held(j.blocks);
    h.flags = held(j.flags);
    h.maxsec = held(j.maxsec);
    h.speed = held(j.speed);
    h.far_max = held(j.far_max);
#pragma unroll
    for (int t = 0; t < NT; ++t) h.dist[t] = held(j.dist[t]);
    const float clear = held(j.clear);
    const bool betw = (h.flags & 2u) != 0;
    uint32_t eband[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) eband[t] = 0;
    // ---- the source: page 0, the front's one entry (alone in its round)
    if (wib == 0) {
      open_pages(a, q, src >> a.ps, lane == 0);
      order();
      if (lane == 0) {
        const uint32_t slot = src & ((1u << a.ps) - 1u);
        q.D[slot] = 0u;
        uint32_t more = 0;
        while (more + 1 < j.blocks && (j.row[((size_t)src * j.blocks + more + 1) * kQuad].x & kNoNb) != kNoNb) ++more;
        q.front[0] = slot | (more << 16);
      }
    }
    lds_barrier();
    uint32_t nf = 1, ns0 = 0;
    // per threshold: settled nodes by the end of the last round that holds one
    // within it (rounds are in order of distance), and inner nodes by then
    uint32_t top[NT], room[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) top[t] = room[t] = 0;
    for (uint32_t par = 0;; par ^= 1u) {
      const uint32_t *cur = q.front + par * a.F;
      uint32_t *nxt = q.front + (par ^ 1u) * a.F;
      // ---- how far the front is safe
      uint32_t lim = kInf, low = kInf;
      for (uint32_t i = tid; i < nf; i += B) {
        const uint32_t e = cur[i], db = q.D[e & 0xffffu];
        const uint32_t x = __float_as_uint(fbits(db) + fbits(e & 0xfffc0000u));
        lim = x < lim ? x : lim;
        low = db < low ? db : low;
      }
      lim = wave_min_u32(lim);
      low = wave_min_u32(low);
      if (lane == 0 && low != kInf) {
        lds_min(&ctl.lim[par], lim);
        lds_min(&ctl.low[par], low);
      }
      lds_barrier();
      const float L = fbits(uniform(lds_ld(&ctl.lim[par]))) * clear;
      const uint32_t lowb = uniform(lds_ld(&ctl.low[par]));
      if (tid == 0) {  // the other parity's words: everyone has read them
        lds_st(&ctl.lim[par ^ 1u], kInf);
        lds_st(&ctl.low[par ^ 1u], kInf);
        lds_st(&ctl.cnt[par ^ 1u], 0u);
      }
      // none safe: the first node in settle order, alone
      const bool single = !(fbits(lowb) < L);
      uint32_t only = 0;
      if (single) {
        for (uint32_t i = tid; i < nf; i += B) {
          const uint32_t slot = cur[i] & 0xffffu;
          if (q.D[slot] == lowb)
            __hip_atomic_fetch_min(&ctl.first, ((unsigned long long)j.orig[node_of(a, q, slot)] << 32) | slot,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        lds_barrier();
        only = uniform((uint32_t)__hip_atomic_load(&ctl.first, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        lds_barrier();
        if (tid == 0) ctl.first = ~0ull;
      }
      // ---- each wave keeps, or settles and relaxes, its part of the front
      uint32_t *cnt = &ctl.cnt[par];
      const uint32_t part = (nf + waves - 1) / waves, i1 = (wib + 1) * part < nf ? (wib + 1) * part : nf;
      for (uint32_t i0 = wib * part; i0 < i1; i0 += kWave) {
        const uint32_t i = i0 + lane;
        uint32_t e = 0, db = kInf;
        if (i < i1) {
          e = cur[i];
          db = lds_ld(&q.D[e & 0xffffu]);
        }
        const bool sel = i < i1 && (single ? (e & 0xffffu) == only : fbits(db) < L);
        const bool keep = i < i1 && !sel;
        const uint64_t mk = __ballot(keep);
        if (mk) {
          uint32_t kb = 0;
          if (lane == 0) kb = lds_add(cnt, (uint32_t)__popcll(mk));
          kb = uniform(kb) + rank_below(mk);
          if (keep) {
            if (kb < a.F) nxt[kb] = e;
            else lds_or(&ctl.fail, kFailRoom);
          }
        }
        if (__ballot(sel))
          settle<NT>(a, j, h, q, sel, e & 0xffffu, (e >> 16) & 3u, db, ns0, nxt, cnt, eband, st_edges);
        order();
      }
      lds_barrier();
      nf = uniform(lds_ld(cnt));
      const uint32_t ns = uniform(lds_ld(&ctl.ns));
      if (uniform(lds_ld(&ctl.fail))) break;
      const uint32_t ni = uniform(lds_ld(&ctl.ni));
      const float low_route = fbits(lowb) * h.speed;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (low_route <= h.dist[t]) {
          top[t] = ns;
          room[t] = ni;
        }
      ns0 = ns;
      if (nf == 0) break;
    }
    uint32_t fail = uniform(lds_ld(&ctl.fail));
    if (betw && uniform(lds_ld(&ctl.ni)) > a.dcap) fail |= kFailRoom;
    if (fail & kFailRoom) fail = kFailRoom;  // without room the rest of the round means nothing
    if (fail) {
      if (tid == 0) {
        const uint32_t k = atomicAdd(a.n_fail, 1u);
        a.fail_list[k] = item;
        atomicOr(a.fail_flags, fail);
      }
      lds_barrier();
      for (uint32_t i = tid; i < a.n_pt / 4; i += B) reinterpret_cast<uint32_t *>(q.pt)[i] = 0xffffffffu;
      continue;
    }
    const uint32_t ns = ns0, np = uniform(lds_ld(&ctl.np)), slots = np << a.ps;
    if (tid == 0) st_reached += ns;
    const float wt = j.src_wt[si];
    const size_t N = j.N, ts = j.tstride;
    // ---- nodes and undirected edges within each threshold (circuit rank, reach)
    {
      uint32_t nb[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) nb[t] = 0;
      for (uint32_t s = tid; s < slots; s += B) {
        const float route = fbits(q.D[s]) * j.speed;
#pragma unroll
        for (int t = 0; t < NT; ++t) nb[t] += route <= j.dist[t] ? 1u : 0u;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint32_t x = wave_sum(nb[t]), y = wave_sum(eband[t]);
        if (lane == 0 && x) lds_add(&ctl.nband[t], x);
        if (lane == 0 && y) lds_add(&ctl.eband[t], y);
      }
    }
    lds_barrier();
    float rank[NT];
    const float cyc = j.src_cyc[si];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint32_t nn = uniform(lds_ld(&ctl.nband[t])), ee = uniform(lds_ld(&ctl.eband[t]));
      const int r = (int)ee - (int)nn + 1;
      rank[t] = nn == 0 ? 0.0f : (float)(r > 0 ? r : 0);
      const uint32_t others = nn ? nn - 1 : 0u;
      if (tid == 0) {
        st_within += others;
        if ((j.flags & 5u) == 5u && others) atomicAdd(&j.reach[t], others);
      }
    }
    // ---- closeness terms of every reached node, in address order (centrality.rs:1736-1779)
    if (j.flags & 1u) {
      for (uint32_t s = tid; s < slots; s += B) {
        const uint32_t db = q.D[s];
        const uint32_t v = node_of(a, q, s);
        if (db == kInf || v == src) continue;
        const float route = fbits(db) * j.speed;
        double *accv = j.acc + v;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          if (!(route <= j.dist[t])) continue;
          gadd_f64(&accv[((size_t)0 * ts + t) * N], (double)wt);
          gadd_f64(&accv[((size_t)1 * ts + t) * N], (double)(route * wt));
          gadd_f64(&accv[((size_t)2 * ts + t) * N], (double)(rank[t] * cyc));
          gadd_f64(&accv[((size_t)3 * ts + t) * N], (double)((1.0f / route) * wt));
          gadd_f64(&accv[((size_t)4 * ts + t) * N], (double)(exp_host(-j.beta[t] * route) * wt));
        }
      }
    }
    // ---- betweenness: dependency arrays packed over the distances, one a wave
    if (betw) {
      __syncthreads();  // records, numbers and rounds of every wave
      if (uniform(lds_ld(&ctl.nmulti))) {
        if (wib == 0) path_shares(a, q, ns, reinterpret_cast<double *>(q.ws + a.o_ratio) + ((size_t)a.P << a.ps) * a.maxp);
        __syncthreads();
      }
      double *dep = reinterpret_cast<double *>(disc_lds);
      // arrays k = 2t + kind, taken in passes that fill the overlay; within a
      // pass array number i is wave i's (mod waves)
      uint32_t todo = 0;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (top[t] > 1) todo |= 3u << (2 * t);
      while (todo) {
        uint32_t used = 0, take = 0, cnt = 0;
        uint32_t at[2 * NT];
#pragma unroll
        for (int k = 2 * NT - 1; k >= 0; --k) {
          at[k] = 0;
          if (((todo >> k) & 1u) && used + room[k / 2] <= a.dcap) {
            at[k] = used;
            used += room[k / 2];
            take |= 1u << k;
          }
        }
        lds_barrier();
#pragma unroll
        for (int k = 2 * NT - 1; k >= 0; --k) {
          if (!((take >> k) & 1u)) continue;
          if (cnt++ % waves == wib)
            sweep(a, j, q, dep + at[k], room[k / 2], top[k / 2], j.dist[k / 2], (k & 1) != 0, j.beta[k / 2]);
        }
        lds_barrier();
        // credits in address order (centrality.rs:848-866)
        const uint16_t *iid = reinterpret_cast<const uint16_t *>(q.ws + a.o_iid);
        for (uint32_t s = tid; s < slots; s += B) {
          if (!((q.bits[s >> 5] >> (s & 31u)) & 1u)) continue;
          const uint32_t v = node_of(a, q, s);
          if (v == src) continue;
          const uint32_t id = ld_u16(&iid[s]);
#pragma unroll
          for (int k = 0; k < 2 * NT; ++k) {
            if (!((take >> k) & 1u) || id >= room[k / 2]) continue;
            const double c = dep[at[k] + id];
            if (c > 0.0) gadd_f64(&j.acc[((size_t)(5 + (k & 1)) * ts + k / 2) * N + v], c * (double)wt);
          }
        }
        todo &= ~take;  // (every array fits the overlay alone: the inner nodes do)
      }
    }
    lds_barrier();
    for (uint32_t i = tid; i < np; i += B) lds_st8(&q.pt[q.pl[i]], (uint8_t)kNone);
    if (a.progress && tid == 0)
      __hip_atomic_store(&a.progress[blockIdx.x], ++pdone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  const unsigned long long edges = wave_sum((unsigned long long)st_edges);
  if (lane == 0) atomicAdd(&a.stats[1], edges);
  if (tid == 0) {
    atomicAdd(&a.stats[0], st_reached);
    atomicAdd(&a.stats[2], st_within);
  }
}

// A node's row: its out-edges in their order, each beside an in-edge from the
// same neighbour, then the in-edges left over. f(neighbour, edges counted
// there, in-edge seconds, out-edge seconds) for each; their number. (At most
// 16 edges each way.)
template <typename F>
__device__ __forceinline__ uint32_t each_neighbour(const uint4 r, const uint2 *rev, const uint2 *fwd, F f) {
  const uint32_t nr = r.w - r.z;
  uint32_t used = 0, n = 0;
  for (uint32_t i = r.x; i < r.y; ++i) {
    const uint2 o = fwd[i];
    const uint32_t u = o.x & ~kCanonBit;
    uint32_t edges = o.x >> 31, in = kInf;
    for (uint32_t k = 0; k < nr; ++k) {
      const uint2 x = rev[r.z + k];
      if (((used >> k) & 1u) || (x.x & ~kCanonBit) != u) continue;
      used |= 1u << k;
      in = x.y;
      edges += x.x >> 31;
      break;
    }
    f(n++, u, edges, in, o.y);
  }
  for (uint32_t k = 0; k < nr; ++k) {
    if ((used >> k) & 1u) continue;
    const uint2 x = rev[r.z + k];
    f(n++, x.x & ~kCanonBit, x.x >> 31, x.y, kInf);
  }
  return n;
}

// Per node: its shortest in-edge from another node and its row's entries.
// info: most entries of a row, costs the search does not take, then the nodes
// by shortest in-edge in powers of two of a millisecond [64].
__global__ void k_disc_measure(const uint4 *rows, const uint2 *rev, const uint2 *fwd, uint32_t N, uint2 *meas, uint32_t *info) {
  __shared__ uint32_t hist[66];
  for (uint32_t i = threadIdx.x; i < 66; i += blockDim.x) hist[i] = 0;
  __syncthreads();
  const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < N) {
    float shortest = INFINITY;
    bool bad = false;
    const uint32_t n = each_neighbour(rows[v], rev, fwd, [&](uint32_t, uint32_t u, uint32_t, uint32_t in, uint32_t out) {
      const float a = fbits(in), b = fbits(out);
      if (!(a >= 0.0f) || !(b >= 0.0f)) bad = true;
      if (u != v && a < shortest) shortest = a;
    });
    meas[v] = make_uint2(__float_as_uint(shortest), n);
    atomicMax(&hist[0], n);
    if (bad) atomicOr(&hist[1], 1u);
    if (shortest < INFINITY) {
      int k = 0;
      (void)frexp((double)shortest * 1000.0, &k);
      atomicAdd(&hist[2 + (k < 0 ? 0 : k > 63 ? 63 : k)], 1u);
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < 66; i += blockDim.x) {
    if (!hist[i]) continue;
    if (i == 0) atomicMax(&info[0], hist[0]);
    else if (i == 1) atomicOr(&info[1], hist[1]);
    else atomicAdd(&info[i], hist[i]);
  }
}

// The rows, a node a thread.
__global__ void k_disc_rows(const uint4 *rows, const uint2 *rev, const uint2 *fwd, uint32_t N, uint32_t blocks,
                            const uint2 *meas, uint4 *row) {
  const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= N) return;
  uint4 *out = row + (size_t)v * blocks * kQuad;
  const uint32_t n = each_neighbour(rows[v], rev, fwd, [&](uint32_t at, uint32_t u, uint32_t edges, uint32_t in, uint32_t o) {
    const uint2 m = meas[u];
    out[at] = make_uint4(u | (edges << 30), in, o, (m.x & ~3u) | (m.y ? (m.y - 1) / kQuad : 0u));
  });
  for (uint32_t k = n; k < blocks * kQuad; ++k) out[k] = make_uint4(kNoNb, kInf, kInf, 0u);
}

// Probed sources: eight spread over the node order and one in its middle, which
// on the Hilbert curve of a town as wide as its searches is the town's.
constexpr uint32_t kProbes = 9, kProbeList = 65536, kProbeStop = 40000, kProbeWords = 16;
constexpr uint32_t kProbePages = 10;  // page shifts of a probe's table: 4 .. 9

struct ProbeArgs {
  const uint4 *row;
  uint32_t N, blocks;
  float maxsec;
  uint32_t *secs;    // [kProbes][N], infinite
  uint32_t *mark;    // [kProbes][N + pages], 0: round a node was last queued in; touched pages
  uint32_t *lists;   // [kProbes][5][cap]: seen, two of the band, two beyond
  uint32_t cap;      // entries of a list: all nodes, or more than a probe goes on with
  uint32_t pages;    // words of the page marks
  uint32_t *out;     // [kProbes][kProbeWords]: nodes, front, inner, pages from shift 4 on
};

__global__ void k_fill32(uint32_t *p, size_t n, uint32_t v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// What a search takes, for a few sources spread over the node order, one a
// workgroup, of each request (grid's y): bands of seconds, within a band a node again whenever its seconds
// drop, lists in memory. Stops past what LDS holds. Each step is a round trip to
// memory: 0.4 ms for a reach of 4,300 nodes (the same on the host from a copy of
// the rows 3.8 ms).
__global__ __launch_bounds__(512) void k_disc_probe(const ProbeArgs *args) {
  const ProbeArgs a = args[blockIdx.y];
  constexpr uint32_t kBands = 32;
  __shared__ uint32_t n_seen, n_next, n_far, kept, inner, pages[kProbePages];
  const uint32_t tid = threadIdx.x, B = blockDim.x;
  const uint32_t src = blockIdx.x + 1 == kProbes ? a.N / 2
                                                 : (uint32_t)(((uint64_t)2 * blockIdx.x + 1) * a.N / (2 * (kProbes - 1)));
  uint32_t *secs = a.secs + (size_t)blockIdx.x * a.N;
  uint32_t *mark = a.mark + (size_t)blockIdx.x * (a.N + a.pages), *pmark = mark + a.N;
  uint32_t *seen = a.lists + (size_t)blockIdx.x * 5 * a.cap;
  uint32_t *cur = seen + a.cap, *next = cur + a.cap, *far = next + a.cap, *far2 = far + a.cap;
  if (tid == 0) {
    n_seen = 1;
    n_far = inner = 0;
    seen[0] = cur[0] = src;
    atomicExch(&secs[src], 0u);
  }
  if (tid < kProbePages) pages[tid] = 0;
  uint32_t n_cur = 1, front = 0, round = 0;
  const float step = a.maxsec / kBands;
  float lim = step;
  for (uint32_t b = 0; b < kBands; ++b) {
    const bool last = b + 1 == kBands;
    while (n_cur) {
      ++round;
      __syncthreads();
      if (tid == 0) n_next = 0;
      __syncthreads();
      // four lanes a row block; a node's further blocks in turn
      for (uint32_t i = tid / kQuad; i < n_cur; i += B / kQuad) {
        const uint32_t v = cur[i];
        const float s = fbits(__hip_atomic_load(&secs[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        for (uint32_t k = 0; k < a.blocks; ++k) {
          const uint4 e = a.row[((size_t)v * a.blocks + k) * kQuad + tid % kQuad];
          const uint32_t u = e.x & kNoNb;
          if (u == kNoNb) continue;
          const float cs = s + fbits(e.y);
          if (!(cs <= a.maxsec)) continue;
          const uint32_t was = atomicMin(&secs[u], __float_as_uint(cs));
          if (was <= __float_as_uint(cs)) continue;
          if (was == kInf) {
            const uint32_t at = atomicAdd(&n_seen, 1u);
            if (at < a.cap) seen[at] = u;
          }
          if (last || cs < lim) {
            if (atomicExch(&mark[u], round) != round) {
              const uint32_t at = atomicAdd(&n_next, 1u);
              if (at < a.cap) next[at] = u;
            }
          } else if (was == kInf) {
            const uint32_t at = atomicAdd(&n_far, 1u);
            if (at < a.cap) far[at] = u;
          }
        }
      }
      __syncthreads();
      n_cur = n_next;
      uint32_t *t = cur;
      cur = next;
      next = t;
      if (n_seen > kProbeStop) break;
    }
    __syncthreads();
    const uint32_t seen_now = n_seen, nfar = n_far;
    __syncthreads();
    if (seen_now > kProbeStop || nfar == 0) break;
    // the nodes beyond the band: the front. Those of the next band are its list.
    if (tid == 0) n_next = n_far = kept = 0;
    __syncthreads();
    const float beyond = lim + step;
    for (uint32_t i = tid; i < nfar; i += B) {
      const uint32_t u = far[i];
      const float s = fbits(__hip_atomic_load(&secs[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      if (s < lim) continue;  // came nearer, and settled
      atomicAdd(&kept, 1u);
      if (b + 2 == kBands || s < beyond) cur[atomicAdd(&n_next, 1u)] = u;
      else far2[atomicAdd(&n_far, 1u)] = u;
    }
    __syncthreads();
    n_cur = n_next;
    front = kept > front ? kept : front;
    lim = beyond;
    uint32_t *t = far;
    far = far2;
    far2 = t;
  }
  __syncthreads();
  const uint32_t n = n_seen < a.cap ? n_seen : a.cap;
  for (uint32_t i = tid; i < n; i += B) {
    const uint32_t v = seen[i];
    uint32_t at = 0;
    for (uint32_t ps = 4; ps < kProbePages; ++ps) {
      if (!atomicExch(&pmark[at + (v >> ps)], 1u)) atomicAdd(&pages[ps], 1u);
      at += (a.N >> ps) + 1;
    }
    // does it precede another?
    const float s = fbits(__hip_atomic_load(&secs[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    bool before = false;
    for (uint32_t k = 0; k < a.blocks * kQuad && !before; ++k) {
      const uint4 e = a.row[(size_t)v * a.blocks * kQuad + k];
      const uint32_t u = e.x & kNoNb;
      if (u == kNoNb) break;
      const float cs = s + fbits(e.y);
      before = cs <= a.maxsec && cs == fbits(__hip_atomic_load(&secs[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
    if (before) atomicAdd(&inner, 1u);
  }
  __syncthreads();
  if (tid == 0) {
    uint32_t *o = a.out + blockIdx.x * kProbeWords;
    o[0] = n;
    o[1] = front;
    o[2] = inner;
    for (uint32_t ps = 4; ps < kProbePages; ++ps) o[ps - 1] = pages[ps];
  }
}

__global__ void k_disc_zero(uint64_t *p, uint32_t n) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0;
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// The graphs' rows for this kernel, built once per speed, on the device from the
// edge arrays they hold, all that are missing at once. They are there when this
// returns: another call may read them on its own stream as soon as the caller
// lets go of the graph's disc_mu, and `tmp` may go to another call.
void disc_graphs(const std::vector<JobSpec> &specs, DevVec &tmp, hipStream_t stream) {
  constexpr uint32_t kInfo = 66, most = kMaxBlocks * kQuad;
  struct New {
    const JobSpec *js;
    std::unique_ptr<DiscGraph> w;
    size_t meas;  // words from the start of tmp
  };
  std::vector<New> todo;
  size_t words = 0;
  for (const JobSpec &js : specs) {
    const Graph &g = *js.g;
    if (!js.n_sources || js.de->disc) continue;
    bool there = false;
    for (const New &x : todo) there = there || x.js->de == js.de;
    if (there) continue;
    if (!(g.n > 0 && g.n < (1u << 24) && !(js.de->min_es <= 0.0f) && g.max_out_deg <= most && g.max_in_deg <= most)) {
      js.de->disc = std::make_unique<DiscGraph>();
      continue;
    }
    todo.push_back({&js, std::make_unique<DiscGraph>(), words});
    words += 2 * (size_t)g.n;
  }
  if (todo.empty()) return;
  uint32_t *meas = static_cast<uint32_t *>(tmp.get(4 * (words + kInfo * todo.size()), "row measures")), *info = meas + words;
  const dim3 block(256);
  hipLaunchKernelGGL(k_fill32, dim3(1), block, 0, stream, info, kInfo * todo.size(), 0u);
  for (size_t i = 0; i < todo.size(); ++i) {
    const JobSpec &js = *todo[i].js;
    hipLaunchKernelGGL(k_disc_measure, dim3((js.g->n + 255) / 256), block, 0, stream, js.dg->rows, js.de->rev_adj,
                       js.de->fwd_adj, js.g->n, reinterpret_cast<uint2 *>(meas + todo[i].meas), info + kInfo * i);
  }
  hip_check(hipGetLastError(), "row measures launch");
  std::vector<uint32_t> host(kInfo * todo.size());
  hip_check(hipMemcpyAsync(host.data(), info, 4 * host.size(), hipMemcpyDeviceToHost, stream), "copy");
  hip_check(hipStreamSynchronize(stream), "sync");
  for (size_t i = 0; i < todo.size(); ++i) {
    const JobSpec &js = *todo[i].js;
    DiscGraph &w = *todo[i].w;
    const uint32_t *h = &host[kInfo * i], n = js.g->n;
    w.blocks = std::max(1u, (h[0] + kQuad - 1) / kQuad);
    w.maxp = std::max(1u, js.g->max_out_deg);
    w.spans.assign(h + 2, h + kInfo);
    w.usable = !h[1] && w.blocks <= kMaxBlocks;
    if (!w.usable) continue;
    hip_check(hipMalloc(&w.row, sizeof(uint4) * n * w.blocks * kQuad), "hipMalloc rows");
    hipLaunchKernelGGL(k_disc_rows, dim3((n + 255) / 256), block, 0, stream, js.dg->rows, js.de->rev_adj, js.de->fwd_adj, n,
                       w.blocks, reinterpret_cast<const uint2 *>(meas + todo[i].meas), w.row);
  }
  hip_check(hipGetLastError(), "rows launch");
  hip_check(hipStreamSynchronize(stream), "sync");
  for (New &x : todo) x.js->de->disc = std::move(x.w);
}

// What the requests' searches take, the most over the probed sources of each, for
// those not probed before: together, in as few launches as 256 MB of scratch
// allow (a launch lasts as long as its longest chain of steps).
void disc_probe(const std::vector<const JobSpec *> &asked, DevVec &tmp, hipStream_t stream) {
  std::vector<const JobSpec *> todo;
  for (const JobSpec *js : asked) {
    bool there = js->de->disc->reach.count(js->cs.maxsec) != 0;
    for (const JobSpec *x : todo) there = there || (x->de == js->de && x->cs.maxsec == js->cs.maxsec);
    if (!there) todo.push_back(js);
  }
  auto pages_of = [](uint32_t n) {
    uint32_t pages = 0;
    for (uint32_t ps = 4; ps < kProbePages; ++ps) pages += (n >> ps) + 1;
    return pages;
  };
  auto words_of = [&](uint32_t n) {
    return (size_t)kProbes * (2 * (size_t)n + pages_of(n) + 5 * (size_t)std::min(n, kProbeList));
  };
  for (size_t i0 = 0; i0 < todo.size();) {
    size_t i1 = i0, words = 0;
    while (i1 < todo.size() && i1 - i0 < 4096 && (i1 == i0 || words + words_of(todo[i1]->g->n) <= (64u << 20))) words += words_of(todo[i1++]->g->n);
    const size_t k = i1 - i0, table = (sizeof(ProbeArgs) * k + 3) / 4, out = k * kProbes * kProbeWords;
    uint32_t *d = static_cast<uint32_t *>(tmp.get(4 * (table + out + words), "probe scratch"));
    uint32_t *at = d + table + out;
    std::vector<ProbeArgs> args(k);
    size_t secs = 0, marks = 0;
    for (size_t i = 0; i < k; ++i) secs += kProbes * (size_t)todo[i0 + i]->g->n;
    for (size_t i = 0; i < k; ++i) marks += kProbes * (size_t)(todo[i0 + i]->g->n + pages_of(todo[i0 + i]->g->n));
    size_t o_secs = 0, o_marks = secs, o_lists = secs + marks;
    for (size_t i = 0; i < k; ++i) {
      const JobSpec &js = *todo[i0 + i];
      ProbeArgs &a = args[i];
      a.row = js.de->disc->row;
      a.N = js.g->n;
      a.blocks = js.de->disc->blocks;
      a.maxsec = js.cs.maxsec;
      a.pages = pages_of(a.N);
      a.cap = std::min(a.N, kProbeList);
      a.secs = at + o_secs;
      a.mark = at + o_marks;
      a.lists = at + o_lists;
      a.out = d + table + i * kProbes * kProbeWords;
      o_secs += kProbes * (size_t)a.N;
      o_marks += kProbes * (size_t)(a.N + a.pages);
      o_lists += (size_t)kProbes * 5 * a.cap;
    }
    hip_check(hipMemcpyAsync(d, args.data(), sizeof(ProbeArgs) * k, hipMemcpyHostToDevice, stream), "copy");
    hipLaunchKernelGGL(k_fill32, dim3(256), dim3(256), 0, stream, at, secs, kInf);
    hipLaunchKernelGGL(k_fill32, dim3(256), dim3(256), 0, stream, at + secs, marks, 0u);
    hipLaunchKernelGGL(k_disc_probe, dim3(kProbes, (uint32_t)k), dim3(512), 0, stream, reinterpret_cast<const ProbeArgs *>(d));
    hip_check(hipGetLastError(), "probe launch");
    std::vector<uint32_t> h(out);
    hip_check(hipMemcpyAsync(h.data(), d + table, 4 * out, hipMemcpyDeviceToHost, stream), "copy");
    hip_check(hipStreamSynchronize(stream), "sync");
    for (size_t i = 0; i < k; ++i) {
      DiscGraph::Reach r;
      for (uint32_t q = 0; q < kProbes; ++q) {
        const uint32_t *o = &h[(i * kProbes + q) * kProbeWords];
        r.nodes = std::max(r.nodes, o[0]);
        r.front = std::max(r.front, o[1]);
        if (q + 1 < kProbes) r.spread = std::max(r.spread, o[1]);
        r.inner = std::max(r.inner, o[2]);
        for (uint32_t ps = 4; ps < kProbePages; ++ps) r.pages[ps] = std::max(r.pages[ps], o[ps - 1]);
      }
      auto &known = todo[i0 + i]->de->disc->reach;
      if (known.size() >= 64) known.clear();
      known[todo[i0 + i]->cs.maxsec] = r;
    }
    i0 = i1;
  }
  if (tmp.bytes > (64u << 20)) tmp.release();
}

constexpr uint32_t kLdsMax = 159u * 1024u;  // (a workgroup's control words lie beside it)

// LDS layout for searches of reach r with `room` times its sizes; false when it
// does not fit.
bool disc_layout(DiscArgs &a, uint32_t N, const DiscGraph::Reach &r, bool betw, uint32_t waves, double room, uint32_t cap,
                 uint32_t *lds) {
  uint32_t best = 0xffffffffu;
  DiscArgs pick = a;
  for (uint32_t ps = 4; ps < 10; ++ps) {
    DiscArgs b = a;
    b.ps = ps;
    const uint32_t all = (N + (1u << ps) - 1) >> ps;
    b.P = std::min<uint32_t>(all, (uint32_t)(r.pages[ps] * 1.04 * room) + 2);
    if (b.P > kMaxPages || (b.P << ps) > kMaxSlots) continue;
    b.n_pt = (all + 3) & ~3u;
    b.F = std::min<uint32_t>(N, (uint32_t)(r.front * 1.2 * room) + 32);
    b.S = std::min<uint32_t>(N, (uint32_t)(r.nodes * 1.3 * room) + 64);
    if (cap) b.S = std::min(b.S, cap);
    const uint32_t slots = b.P << ps;
    uint32_t o = 4 * slots;
    auto take = [&](uint32_t bytes) {
      const uint32_t at = o;
      o = (o + bytes + 15) & ~15u;
      return at;
    };
    b.o_front = take(8 * b.F);
    b.o_items = take(512 * waves);
    if (betw) o = std::max(o, (uint32_t)((8 * (size_t)std::min<uint32_t>(N, (uint32_t)(r.inner * 1.06 * room) + 16) + 15) & ~15u));
    b.dcap = o / 8;
    b.o_bits = take((slots + 31) / 32 * 4);
    b.o_pt = take(b.n_pt);
    b.o_pl = take(4 * b.P);
    if (o < best) {
      best = o;
      pick = b;
    }
  }
  if (best > kLdsMax) return false;
  a = pick;
  *lds = best;
  return true;
}

// Workgroups of a CU by its LDS, which is given out in units of 1,280 bytes (the
// runtime's occupancy query does not count them).
uint32_t blocks_by_lds(uint32_t lds) {
  const uint32_t unit = 1280, need = (lds + (uint32_t)sizeof(Ctl) + unit - 1) / unit * unit;
  return 160u * 1024u / need;
}

const void *disc_kernel(uint32_t NT) {
  return NT <= 1   ? reinterpret_cast<const void *>(k_disc<1>)
         : NT <= 2 ? reinterpret_cast<const void *>(k_disc<2>)
         : NT <= 4 ? reinterpret_cast<const void *>(k_disc<4>)
                   : reinterpret_cast<const void *>(k_disc<8>);
}

struct DiscWorkspace {
  DevVec scratch, ctl, jobs, items, fail, tmp;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  std::mutex mu;
  void release() {
    for (DevVec *d : {&scratch, &ctl, &jobs, &items, &fail, &tmp}) d->release();
  }
  ~DiscWorkspace() {
    release();
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
  }
};
std::mutex g_disc_mu;
std::map<int, std::vector<std::unique_ptr<DiscWorkspace>>> g_disc;

// A workspace of the device's pool, locked for the caller (one per concurrent call).
DiscWorkspace *acquire_disc(int device) {
  std::lock_guard<std::mutex> lk(g_disc_mu);
  auto &v = g_disc[device];
  for (auto &w : v)
    if (w->mu.try_lock()) return w.get();
  v.emplace_back(new DiscWorkspace());
  v.back()->mu.lock();
  return v.back().get();
}

}  // namespace

// Jobs of one launch: searches of similar size.
struct DiscClass {
  DiscArgs a;
  uint32_t lds = 0, waves = 1, NT = 1, N = 0;
  bool betw = false;
  // searches that ran out of room before: the first launch's searches, workgroups
  // and time, and the time of the tries since
  bool again = false;
  uint32_t first_n = 0, first_blocks = 0;
  double first_ms = 0.0, tries_ms = 0.0;
  double room = 1.0;
  double most = 0.0, all = 0.0;  // expected time of its slowest search, of all its searches one by one (ms)
  double load = 0.0;             // `all` on the workgroups the device holds
  DiscGraph::Reach reach;  // the most over its jobs
  std::vector<DiscJob> jobs;
  std::vector<uint32_t> which;  // the caller's job of each
  std::vector<uint2> items;     // {job of this launch, source position}; empty: all of the one job
  uint32_t n = 0;
};

// Waves of a workgroup: a round settles most of the front, sixteen nodes a wave.
// (Lines from two workloads:)
// Front 52 (closeness on 20 m pieces to 800 m): one wave 2.65 ms, two 2.42, four
// 2.99. Eight towns to 1,600 m: 3.04 ms by this rule, 3.14 with the lines at 64
// and 160, 3.44 at 24 and 48. (The front of a town's middle, which only its few
// nearest sources have, is not what they are about: with it 3,095 sources to
// 2,750 m on a 62x62 town take four waves and 0.68 ms, without it two and 0.59.)
static uint32_t disc_waves(uint32_t front) { return front <= 40 ? 1u : front <= 100 ? 2u : 4u; }

// ... as far as the request itself tells.
static bool disc_may(const JobSpec &js) {
  if (js.d_od_off || js.extra_records) return false;
  if (js.cs.betweenness && js.cs.tolerance > kTieEps) return false;  // predecessors rebuilt from final distances (Phase 2)
  return js.cs.maxsec >= 0.0f;
}

// Can this request search in LDS (its other work is the caller's)? Its graph's
// rows are built.
static bool disc_takes(const JobSpec &js) {
  if (!disc_may(js)) return false;
  const DiscGraph &w = *js.de->disc;
  if (!w.usable) return false;
  // where many nodes have an in-edge shorter than the tie bands at the search's
  // far end, they would settle one at a time
  const uint32_t deg = std::max(js.g->max_out_deg, js.g->max_in_deg) + 3;
  const double gap = (double)js.cs.maxsec * 1.02e-4 * deg;
  uint64_t few = 0, all = 0;
  for (int i = 0; i < 64; ++i) {
    all += w.spans[i];
    if (std::ldexp(0.001, i) <= gap) few += w.spans[i];
  }
  return few * 8 <= all;
}

// Is a workgroup per source, at `lds` bytes each, the faster search? Its rate
// falls with the waves its workgroups put on a CU; a wave per source with its
// state in scratch has twenty a CU whatever the reach. Both measured, kernel ms
// here | there (L: 300x300 lattice, P: 39,000 nodes in 20 m pieces, both with
// workgroups of four waves).
// Betweenness, 16 waves a CU:
//   L reach 5,027: 1,600 sources 1.75 | 2.82,  6,400 5.49 | 7.54,  70,000 54.4 | 61.4
// 12 waves:
//   L 6,480: 1,600 2.79 | 3.65,  3,200 4.74 | 5.03,  6,400 8.63 | 9.71,  70,000 87.6 | 79.3
//   P 5,035: 3,200 2.85 | 3.06,  6,400 5.26 | 5.91,  12,000 9.45 | 9.79
// 8 waves:
//   L 8,090: 800 2.39 | 3.71,  1,600 4.29 | 4.58,  3,200 7.69 | 6.26
//   P 6,150: 800 1.44 | 1.86,  1,600 2.53 | 2.37,  3,200 4.48 | 3.69
// 4 waves:
//   P 11,400: 300 2.08 | 2.98,  800 3.94 | 3.39,  1,600 7.16 | 4.31
// Closeness, 8 waves:
//   L 9,830: 1,600 1.55 | 2.53,  70,000 51.3 | 59.4;  P 8,620: 3,200 2.71 | 2.82,  12,000 9.35 | 8.98
// 4 waves:
//   P 14,380: 800 2.10 | 2.09,  1,600 3.64 | 3.11,  3,200 6.77 | 4.58
static bool disc_pays(uint32_t lds, uint32_t waves, bool betw, uint32_t n, uint32_t cus) {
  const uint32_t per_cu = blocks_by_lds(lds) * waves;
  if (!betw) return per_cu >= 8 || n <= 4 * cus;
  return per_cu >= 16 || n <= (per_cu >= 12 ? 28 : per_cu >= 8 ? 5 : 2) * cus;
}

// Lays a launch out and estimates it: 0.05 ms and 0.17 us a node for a search
// (0.06 us without betweenness; the 250x250 lattice to 5,000 m, 38 searches after
// one another on five workgroups a CU: 25.7 and 8.6 ms), twenty waves a CU at
// most. False when the layout does not fit.
static bool disc_estimate(DiscClass &d, uint32_t cap, uint32_t cus) {
  DiscArgs a;
  std::memset(&a, 0, sizeof(a));
  if (!disc_layout(a, d.N, d.reach, d.betw, d.waves, 1.0, cap, &d.lds)) return false;
  d.load = d.all / ((double)cus * std::max(1u, std::min(blocks_by_lds(d.lds), 20u / d.waves)));
  return true;
}

// Two launches as one, without their jobs.
static DiscClass disc_pair(const DiscClass &x, const DiscClass &y) {
  DiscClass d;
  std::memset(&d.a, 0, sizeof(d.a));
  d.NT = x.NT;
  d.N = std::max(x.N, y.N);
  d.n = x.n + y.n;
  d.betw = x.betw || y.betw;
  d.reach.nodes = std::max(x.reach.nodes, y.reach.nodes);
  d.reach.front = std::max(x.reach.front, y.reach.front);
  d.reach.inner = std::max(x.reach.inner, y.reach.inner);
  for (int p = 0; p < 10; ++p) d.reach.pages[p] = std::max(x.reach.pages[p], y.reach.pages[p]);
  d.a.maxp = std::max(x.a.maxp, y.a.maxp);
  d.waves = std::max(x.waves, y.waves);
  d.most = std::max(x.most, y.most);
  d.all = x.all + y.all;
  return d;
}

// Expected time of a launch: of its slowest search, or of its load with the
// device running empty at its end.
static double disc_time(const DiscClass &d) { return std::max(d.most, d.load + 0.5 * d.most); }

// Joins launches, neighbours in size, while that shortens their time after one
// another.
static void disc_join(std::vector<DiscClass> &v, uint32_t cap, uint32_t cus) {
  std::sort(v.begin(), v.end(), [](const DiscClass &x, const DiscClass &y) { return x.lds < y.lds; });
  // what joining each with its next saves
  std::vector<double> saves;
  auto saved = [&](size_t k) {
    DiscClass m = disc_pair(v[k], v[k + 1]);
    return disc_estimate(m, cap, cus) ? disc_time(v[k]) + disc_time(v[k + 1]) - disc_time(m) : -INFINITY;
  };
  for (size_t k = 0; k + 1 < v.size(); ++k) saves.push_back(saved(k));
  while (v.size() > 1) {
    const size_t k = (size_t)(std::max_element(saves.begin(), saves.end()) - saves.begin());
    if (!(saves[k] > 0.0)) break;
    DiscClass m = disc_pair(v[k], v[k + 1]);
    (void)disc_estimate(m, cap, cus);
    for (DiscClass *x : {&v[k], &v[k + 1]}) {
      m.which.insert(m.which.end(), x->which.begin(), x->which.end());
      m.jobs.insert(m.jobs.end(), x->jobs.begin(), x->jobs.end());
    }
    v[k] = std::move(m);
    v.erase(v.begin() + k + 1);
    saves.erase(saves.begin() + k);
    if (k < saves.size()) saves[k] = saved(k);
    if (k) saves[k - 1] = saved(k - 1);
  }
}

// Splits the jobs' items into launches; what cannot search in LDS goes to rest.
// A launch is laid out for its largest search, so jobs share one where their
// sizes are alike or all their sources run at once anyway: seven towns of 9x9 to
// 28x28 to 1,200 m 0.50 ms as seven launches after one another, 0.24 with a wave
// per source in one launch.
static std::vector<DiscClass> disc_plan(const std::vector<JobSpec> &specs, uint32_t NT, uint32_t cap, DevVec &tmp,
                                        hipStream_t stream, std::vector<uint2> *rest) {
  std::vector<DiscClass> out;
  int n_cu = 0;
  hip_check(hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, specs[0].dg->device), "attribute");
  const uint32_t cus = (uint32_t)n_cu;
  // what the graphs keep, in one order for all callers
  std::vector<DevEdges *> des;
  for (const JobSpec &js : specs) des.push_back(js.de);
  std::sort(des.begin(), des.end(), std::less<DevEdges *>());
  des.erase(std::unique(des.begin(), des.end()), des.end());
  std::vector<std::unique_lock<std::mutex>> locks;
  for (DevEdges *de : des) locks.emplace_back(de->disc_mu);
  {
    std::vector<JobSpec> may;
    for (const JobSpec &js : specs)
      if (disc_may(js)) may.push_back(js);
    disc_graphs(may, tmp, stream);
  }
  struct Size {
    bool takes = false, whole = false;
    DiscGraph::Reach r;
    uint32_t waves = 1, lds = 0;
  };
  std::vector<Size> sizes(specs.size());
  std::vector<const JobSpec *> asked;
  for (size_t i = 0; i < specs.size(); ++i) {
    const JobSpec &js = specs[i];
    Size &z = sizes[i];
    z.takes = js.n_sources && disc_takes(js);
    if (!z.takes) continue;
    // a network so small that every source runs at once with room for all of
    // it needs no probes (they took a fifth of a first call on 676 nodes)
    DiscArgs a;
    std::memset(&a, 0, sizeof(a));
    z.r.nodes = z.r.front = z.r.inner = js.g->n;
    for (uint32_t ps = 4; ps < kProbePages; ++ps) z.r.pages[ps] = (js.g->n + (1u << ps) - 1) >> ps;
    z.waves = disc_waves((uint32_t)(2.0 * std::sqrt((double)js.g->n)));
    z.whole = disc_layout(a, js.g->n, z.r, js.cs.betweenness, z.waves, 1.0, cap, &z.lds) &&
              js.n_sources <= cus * blocks_by_lds(z.lds);
    if (!z.whole) asked.push_back(&js);
  }
  disc_probe(asked, tmp, stream);
  for (size_t i = 0; i < specs.size(); ++i) {
    const JobSpec &js = specs[i];
    if (!sizes[i].takes) continue;
    DiscGraph &w = *js.de->disc;
    DiscGraph::Reach &r = sizes[i].r;
    uint32_t &waves = sizes[i].waves, &lds = sizes[i].lds;
    if (!sizes[i].whole) {
      DiscArgs a;
      std::memset(&a, 0, sizeof(a));
      if (!w.reach.count(js.cs.maxsec)) disc_probe({&js}, tmp, stream);  // (forgotten over more than 64 others)
      r = w.reach.at(js.cs.maxsec);
      waves = disc_waves(r.spread);
      if (!disc_layout(a, js.g->n, r, js.cs.betweenness, waves, 1.0, cap, &lds)) continue;
    }
    if (!disc_pays(lds, waves, js.cs.betweenness, js.n_sources, cus)) continue;
    DiscClass d;
    std::memset(&d.a, 0, sizeof(d.a));
    d.waves = waves;
    d.NT = NT;
    d.betw = js.cs.betweenness;
    d.which.push_back((uint32_t)i);
    d.N = js.g->n;
    d.n = js.n_sources;
    d.reach = r;
    d.a.maxp = std::max(1u, w.maxp);
    d.most = 0.05 + (d.betw ? 1.7e-4 : 6e-5) * r.nodes;
    d.all = d.n * d.most;
    DiscJob j;
    std::memset(&j, 0, sizeof(j));
    j.row = w.row;
    j.orig = js.dg->orig;
    j.eligible = js.d_eligible;
    j.sources = js.d_sources;
    j.src_wt = js.d_wt;
    j.src_cyc = js.d_cyc;
    j.acc = js.d_acc;
    j.reach = js.d_reach;
    j.N = js.g->n;
    j.blocks = w.blocks;
    j.tstride = js.tstride ? js.tstride : NT;
    j.flags = (js.cs.closeness ? 1u : 0u) | (js.cs.betweenness ? 2u : 0u) | (js.cs.track_reach ? 4u : 0u);
    j.maxsec = js.cs.maxsec;
    j.speed = js.cs.speed;
    j.far_max = 1.0;
    for (uint32_t k = 0; k < js.g->max_out_deg + 3; ++k) j.far_max *= 1.00010002;
    j.clear = (float)((1.0 - 4e-6) / j.far_max);
    for (uint32_t t = 0; t < kMaxT; ++t) {
      j.dist[t] = t < js.cs.T ? js.cs.dist[t] : -1.0f;
      j.beta[t] = t < js.cs.T ? js.cs.beta[t] : 0.0f;
    }
    d.jobs.push_back(j);
    if (disc_estimate(d, cap, cus)) out.push_back(std::move(d));
  }
  if (out.empty()) return out;
  disc_join(out, cap, cus);
  // (jobs that paid for their few sources alone may be many together)
  out.erase(std::remove_if(out.begin(), out.end(),
                           [&](const DiscClass &d) { return !disc_pays(d.lds, d.waves, d.betw, d.n, cus); }),
            out.end());
  if (out.empty()) return out;
  // items in the callers' order; one whole job alone needs no list
  if (specs.size() == 1) return out;
  std::vector<int> cls(specs.size(), -1);
  std::vector<uint32_t> local(specs.size(), 0);
  for (size_t c = 0; c < out.size(); ++c)
    for (size_t k = 0; k < out[c].which.size(); ++k) {
      cls[out[c].which[k]] = (int)c;
      local[out[c].which[k]] = (uint32_t)k;
    }
  for (uint32_t i = 0; i < specs.size(); ++i)
    for (uint32_t k = 0; k < specs[i].n_sources; ++k) {
      if (cls[i] < 0) rest->push_back(make_uint2(i, k));
      else out[cls[i]].items.push_back(make_uint2(local[i], k));
    }
  return out;
}

// Shapes a launch: LDS layout, workgroups, scratch. The first launch of a class
// takes the most room that costs it no resident workgroup: a source that runs
// out of it is searched twice. False when the layout does not fit.
static bool disc_shape(DiscClass &d, uint32_t cap, int dev, bool first, uint32_t *blocks) {
  const uint32_t maxp = d.a.maxp;
  const void *f = disc_kernel(d.NT);
  hip_check(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax), "LDS size");
  int cus = 0;
  hip_check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "attribute");
  uint32_t resident = 0;
  auto lay = [&](double room) {
    std::memset(&d.a, 0, sizeof(d.a));
    d.a.maxp = maxp;
    if (!disc_layout(d.a, d.N, d.reach, d.betw, d.waves, room, cap, &d.lds)) return false;
    int per_cu = 0;
    hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, (int)(d.waves * kWave), d.lds), "occupancy");
    resident = std::min<uint32_t>(d.n, (uint32_t)cus * (uint32_t)std::max(1, std::min(per_cu, (int)blocks_by_lds(d.lds))));
    return true;
  };
  if (!lay(d.room)) return false;
  if (first) {
    // (steps of 1.08 from the probed sizes left a city without 0.7 ms for a few
    // sources searched twice, or with them, as its probes fell)
    const uint32_t most = resident;
    double room = d.room, above = 2.0 * d.room;
    for (double r = above; above - room > 0.015; r = 0.5 * (room + above)) {
      if (lay(r) && resident == most) room = r;
      else above = r;
      if (room == above) break;
    }
    d.room = room;
    lay(room);
  }
  *blocks = resident;
  // scratch of a workgroup: records | inner numbers | predecessor lists | their shares, path counts
  const size_t slots = (size_t)d.a.P << d.a.ps;
  size_t o = 0;
  if (d.betw) {
    o = align256(8ull * d.a.S);
    auto take = [&](size_t bytes) {
      const size_t at = o;
      o = align256(o + bytes);
      return (uint32_t)at;
    };
    d.a.o_iid = take(2 * slots);
    d.a.o_ext = take(2 * slots * (maxp + 1));
    d.a.o_ratio = take(8 * (slots * maxp + d.a.S));
  }
  d.a.stride = std::max<size_t>(o, 256);
  return true;
}

// A launch's 256 bytes of control words, zero when it starts.
static void disc_ctl(DiscArgs &a, char *ctl) {
  a.stats = reinterpret_cast<unsigned long long *>(ctl + 128);
  a.next = reinterpret_cast<uint32_t *>(ctl);
  a.n_fail = a.next + kXcd;
  a.fail_flags = a.next + kXcd + 1;
}

static void disc_args(DiscClass &d, char *ctl, uint32_t *fail, const uint2 *items, const DiscJob *jobs, char *scratch,
                      uint32_t *progress, uint32_t blocks) {
  DiscArgs &a = d.a;
  a.jobs = jobs;
  a.items = d.items.empty() ? nullptr : items;
  a.n_items = d.n;
  a.ws = scratch;
  disc_ctl(a, ctl);
  a.fail_list = fail;
  for (uint32_t x = 0; x <= kXcd; ++x) a.xbeg[x] = (uint32_t)((uint64_t)d.n * x / kXcd);
  a.progress = progress_room(progress, blocks);
}

static void disc_enqueue(const DiscClass &d, uint32_t blocks, hipStream_t stream) {
  const dim3 grid(blocks), block(d.waves * kWave);
  if (d.NT <= 1) hipLaunchKernelGGL(k_disc<1>, grid, block, d.lds, stream, d.a);
  else if (d.NT <= 2) hipLaunchKernelGGL(k_disc<2>, grid, block, d.lds, stream, d.a);
  else if (d.NT <= 4) hipLaunchKernelGGL(k_disc<4>, grid, block, d.lds, stream, d.a);
  else hipLaunchKernelGGL(k_disc<8>, grid, block, d.lds, stream, d.a);
}

// The tries of a request's searches ended with room for all. Later calls give it
// to every search from the start where the workgroups that costs are expected to
// cost less time than the tries took.
static void disc_learn(const DiscClass &d, const JobSpec &js, uint32_t cus) {
  DiscClass g = disc_pair(d, d);
  auto up = [&](uint32_t x, uint32_t most) { return (uint32_t)std::min<double>(most, std::ceil(x * d.room)); };
  g.reach.nodes = up(d.reach.nodes, d.N);
  g.reach.front = up(d.reach.front, d.N);
  g.reach.inner = up(d.reach.inner, d.N);
  for (uint32_t ps = 4; ps < kProbePages; ++ps) g.reach.pages[ps] = up(d.reach.pages[ps], (d.N + (1u << ps) - 1) >> ps);
  if (!disc_estimate(g, 0, cus)) return;
  const double had = std::min(d.first_n, d.first_blocks);
  const double has = std::min(d.first_n, cus * std::max(1u, std::min(blocks_by_lds(g.lds), 20u / g.waves)));
  if (d.first_ms * (had / has - 1.0) > d.tries_ms) return;
  std::lock_guard<std::mutex> lk(js.de->disc_mu);
  const auto it = js.de->disc->reach.find(js.cs.maxsec);
  if (it != js.de->disc->reach.end() && it->second.nodes <= g.reach.nodes) it->second = g.reach;
}

bool launch_disc(const std::vector<JobSpec> &specs, uint32_t NT, uint32_t cap, hipStream_t stream, cs_stats &st,
                 uint32_t *progress, std::vector<uint2> *rest) {
  const int dev = specs[0].dg->device;
  int n_cu = 0;
  hip_check(hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev), "attribute");
  const uint32_t cus = (uint32_t)n_cu;
  DiscWorkspace *ws = acquire_disc(dev);
  std::lock_guard<std::mutex> guard(ws->mu, std::adopt_lock);
  std::vector<DiscClass> work = disc_plan(specs, NT, cap, ws->tmp, stream, rest);
  if (work.empty()) return false;
  if (!ws->e0) {
    hip_check(hipEventCreate(&ws->e0), "event");
    hip_check(hipEventCreate(&ws->e1), "event");
  }
  char *ctl = static_cast<char *>(ws->ctl.get(256, "control words"));
  while (!work.empty()) {
    DiscClass d = std::move(work.back());
    work.pop_back();
    uint32_t blocks = 0;
    if (!disc_shape(d, cap, dev, d.room == 1.0, &blocks)) {
      // (a launch of several jobs together may not fit where each alone did)
      for (uint32_t i = 0; i < d.n; ++i) {
        const uint2 x = d.items.empty() ? make_uint2(0u, i) : d.items[i];
        rest->push_back(make_uint2(d.which[x.x], x.y));
      }
      continue;
    }
    if (d.a.stride * blocks > ws->scratch.bytes) {
      size_t free_b = 0, total_b = 0;
      hip_check(hipMemGetInfo(&free_b, &total_b), "meminfo");
      blocks = (uint32_t)std::min<size_t>(blocks, std::max<size_t>(1, (free_b / 4 + ws->scratch.bytes) / d.a.stride));
    }
    char *scratch = static_cast<char *>(ws->scratch.get(d.a.stride * blocks, "search scratch"));
    DiscJob *jobs = static_cast<DiscJob *>(ws->jobs.get(sizeof(DiscJob) * d.jobs.size(), "job table"));
    hip_check(hipMemcpyAsync(jobs, d.jobs.data(), sizeof(DiscJob) * d.jobs.size(), hipMemcpyHostToDevice, stream), "copy");
    uint2 *items = nullptr;
    if (!d.items.empty()) {
      items = static_cast<uint2 *>(ws->items.get(sizeof(uint2) * d.n, "items"));
      hip_check(hipMemcpyAsync(items, d.items.data(), sizeof(uint2) * d.n, hipMemcpyHostToDevice, stream), "copy");
    }
    uint32_t *fail_list = static_cast<uint32_t *>(ws->fail.get(4ull * d.n, "failure list"));
    disc_args(d, ctl, fail_list, items, jobs, scratch, progress, blocks);
    hip_check(hipEventRecord(ws->e0, stream), "event");
    hipLaunchKernelGGL(k_disc_zero, dim3(1), dim3(kWave), 0, stream, reinterpret_cast<uint64_t *>(ctl), 32u);
    disc_enqueue(d, blocks, stream);
    hip_check(hipGetLastError(), "k_disc launch");
    hip_check(hipEventRecord(ws->e1, stream), "event");
    uint32_t h[64];
    hip_check(hipMemcpyAsync(h, ctl, 256, hipMemcpyDeviceToHost, stream), "copy");
    hip_check(hipStreamSynchronize(stream), "sync");
    float ms = 0.0f;
    hip_check(hipEventElapsedTime(&ms, ws->e0, ws->e1), "elapsed");
    unsigned long long stv[4];
    std::memcpy(stv, h + 32, 32);
    st.kernel_ms += ms;
    st.waves = std::max<uint32_t>(st.waves, blocks * d.waves);
    st.nodes_reached += stv[0];
    st.edges_scanned += stv[1];
    st.within_sum += stv[2];
    const uint32_t n_failed = h[kXcd];
    thread_lds_searches() += d.n - n_failed;
    if (d.again) {
      d.tries_ms += ms;
    } else {
      d.first_n = d.n;
      d.first_blocks = blocks;
      d.first_ms = ms;
    }
    if (!n_failed) {
      if (d.again && !cap && d.which.size() == 1) disc_learn(d, specs[d.which[0]], cus);
      continue;
    }
    if (h[kXcd + 1] & kFailInternal) fail(CS_EINTERNAL, "search invariant violated (settle order)");
    std::vector<uint32_t> fl(n_failed);
    hip_check(hipMemcpy(fl.data(), fail_list, 4ull * n_failed, hipMemcpyDeviceToHost), "copy");
    std::vector<uint2> left(n_failed);
    for (uint32_t i = 0; i < n_failed; ++i) left[i] = d.items.empty() ? make_uint2(0u, fl[i]) : d.items[fl[i]];
    st.retries += n_failed;
    // again with more room while LDS has it: as much as leaves them all running
    // at once, or half as much again
    DiscClass e = d;
    e.again = true;
    e.items = left;
    e.n = n_failed;
    bool wider = false;
    double room = d.room;
    for (double f = d.room * 1.5; f < 40.0; f *= 1.5) {
      e.room = f;
      uint32_t b = 0;
      if (!disc_shape(e, cap, dev, false, &b) || (wider && b < n_failed)) break;
      wider = wider || e.a.S > d.a.S || e.a.P > d.a.P || e.a.F > d.a.F;
      room = f;
    }
    e.room = room;
    if (wider && !cap) {
      work.push_back(std::move(e));
    } else {
      for (const uint2 &x : left) rest->push_back(make_uint2(d.which[x.x], x.y));
    }
  }
  return true;
}

// The launches of a fixed set of jobs, for a batch that replays them from a
// graph: memory of their own, nothing of it changed between runs. They follow
// one another: beside one another on four branches of the graph a replay was 3
// to 20% shorter, but each branch has a stream of its own made first, and a
// batch's first run took 1 to 5 ms more.
struct DiscBatch {
  struct Part {
    DiscClass d;
    uint32_t blocks = 0;
    uint32_t *fail = nullptr;
  };
  std::vector<Part> parts;
  std::vector<void *> bufs;
  uint32_t waves = 0;
  ~DiscBatch() {
    for (void *q : bufs) (void)hipFree(q);
  }
  void *mem(size_t bytes) {
    void *q = nullptr;
    hip_check(hipMalloc(&q, std::max<size_t>(bytes, 1)), "hipMalloc batch");
    bufs.push_back(q);
    return q;
  }
};

DiscBatch *disc_batch_new(const std::vector<JobSpec> &specs, uint32_t NT, int device, hipStream_t stream,
                          std::vector<uint2> *rest) {
  auto b = std::make_unique<DiscBatch>();
  DevVec tmp;
  struct Release {
    DevVec &v;
    ~Release() { v.release(); }
  } release{tmp};
  std::vector<DiscClass> work = disc_plan(specs, NT, 0, tmp, stream, rest);
  size_t scratch = 0;
  for (DiscClass &c : work) {
    DiscBatch::Part p;
    p.d = std::move(c);
    if (!disc_shape(p.d, 0, device, true, &p.blocks)) {
      for (uint32_t i = 0; i < p.d.n; ++i) {
        const uint2 x = p.d.items.empty() ? make_uint2(0u, i) : p.d.items[i];
        rest->push_back(make_uint2(p.d.which[x.x], x.y));
      }
      continue;
    }
    size_t free_b = 0, total_b = 0;
    hip_check(hipMemGetInfo(&free_b, &total_b), "meminfo");
    p.blocks = (uint32_t)std::min<size_t>(p.blocks, std::max<size_t>(1, free_b / 4 / p.d.a.stride));
    scratch = std::max(scratch, p.d.a.stride * p.blocks);
    b->waves = std::max(b->waves, p.blocks * p.d.waves);
    b->parts.push_back(std::move(p));
  }
  if (b->parts.empty()) return nullptr;
  char *ws = static_cast<char *>(b->mem(scratch));
  for (DiscBatch::Part &p : b->parts) {
    p.fail = static_cast<uint32_t *>(b->mem(4ull * p.d.n));
    DiscJob *jobs = static_cast<DiscJob *>(b->mem(sizeof(DiscJob) * p.d.jobs.size()));
    hip_check(hipMemcpy(jobs, p.d.jobs.data(), sizeof(DiscJob) * p.d.jobs.size(), hipMemcpyHostToDevice), "copy");
    uint2 *items = nullptr;
    if (!p.d.items.empty()) {
      items = static_cast<uint2 *>(b->mem(sizeof(uint2) * p.d.n));
      hip_check(hipMemcpy(items, p.d.items.data(), sizeof(uint2) * p.d.n, hipMemcpyHostToDevice), "copy");
    }
    disc_args(p.d, nullptr, p.fail, items, jobs, ws, nullptr, p.blocks);
  }
  return b.release();
}

void disc_batch_delete(DiscBatch *b) { delete b; }

size_t disc_batch_ctl(const DiscBatch &b) { return 256 * b.parts.size(); }

void disc_batch_enqueue(DiscBatch &b, char *ctl, hipStream_t stream) {
  for (size_t i = 0; i < b.parts.size(); ++i) {
    disc_ctl(b.parts[i].d.a, ctl + 256 * i);
    disc_enqueue(b.parts[i].d, b.parts[i].blocks, stream);
  }
}

void disc_batch_collect(const DiscBatch &b, const char *ctl, cs_stats &st, std::vector<uint2> *retry) {
  st.waves = std::max(st.waves, b.waves);
  for (size_t i = 0; i < b.parts.size(); ++i) {
    const DiscBatch::Part &p = b.parts[i];
    uint32_t c[64];
    std::memcpy(c, ctl + 256 * i, 256);
    unsigned long long stv[4];
    std::memcpy(stv, c + 32, 32);
    st.nodes_reached += stv[0];
    st.edges_scanned += stv[1];
    st.within_sum += stv[2];
    const uint32_t n_failed = c[kXcd];
    thread_lds_searches() += p.d.n - n_failed;
    if (!n_failed) continue;
    if (c[kXcd + 1] & kFailInternal) fail(CS_EINTERNAL, "search invariant violated (settle order)");
    std::vector<uint32_t> fl(n_failed);
    hip_check(hipMemcpy(fl.data(), p.fail, 4ull * n_failed, hipMemcpyDeviceToHost), "copy");
    for (uint32_t k : fl) {
      const uint2 x = p.d.items.empty() ? make_uint2(0u, k) : p.d.items[k];
      retry->push_back(make_uint2(p.d.which[x.x], x.y));
    }
  }
}

bool disc_more_room(DevEdges &de, float maxsec, uint32_t N) {
  std::lock_guard<std::mutex> lk(de.disc_mu);
  if (!de.disc) return false;
  const auto it = de.disc->reach.find(maxsec);
  if (it == de.disc->reach.end()) return false;
  DiscGraph::Reach &r = it->second;
  bool more = false;
  auto up = [&](uint32_t &x, uint32_t most) {
    const uint32_t y = std::min(most, x + x / 4 + 1);
    more = more || y > x;
    x = std::max(x, y);
  };
  for (uint32_t *x : {&r.nodes, &r.front, &r.inner}) up(*x, N);
  for (uint32_t ps = 4; ps < kProbePages; ++ps) up(r.pages[ps], (N + (1u << ps) - 1) >> ps);
  return more;
}

uint32_t disc_nodes(const DevEdges &de, float maxsec) {
  std::lock_guard<std::mutex> lk(de.disc_mu);
  if (!de.disc) return 0;
  const auto it = de.disc->reach.find(maxsec);
  if (it == de.disc->reach.end()) return 0;
  const uint32_t n = it->second.nodes;
  return n > kProbeStop ? 4 * 16384u : n + n / 4;
}

DiscGraph::~DiscGraph() { (void)hipFree(row); }

void release_disc_workspaces() {
  std::lock_guard<std::mutex> lk(g_disc_mu);
  for (auto &dv : g_disc)
    for (auto &w : dv.second) {
      std::lock_guard<std::mutex> wl(w->mu);
      w->release();
    }
}

}  // namespace cs
