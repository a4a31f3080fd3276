// cs_angwave.hip -- simplest-path (angular) centrality, one wave per source
// with the whole search state in LDS.
//
// The search is the reference's (centrality.rs:577-705): states settle in the
// order (route, seconds at push, state), and every relaxation folds into its
// target in that order, so predecessor lists, path counts, routes and seconds
// are the serial search's bit for bit. What runs in parallel is what that
// order leaves free:
//
//  * Let L be the smallest (route + smallest usable route increment) over the
//    unsettled states. Whatever is relaxed from now on offers at least L, so
//    the states whose route lies below L by more than the tie band settle
//    together: none of them can reach another's band. When the smallest route
//    itself is not that far below L (straight continuations cost almost
//    nothing), it settles alone, which is the serial search's own step.
//  * The settled states get their positions in the order of the lanes they were
//    found in, which within a batch is no settle order, and their out-edges
//    relax one per lane. Lanes whose targets are the same node take turns in
//    settle order: by the route of the state they leave, then its seconds at
//    push, then its original number.
//
// A lane-per-source search keeps its maps, records and queue in HBM and pays a
// chain of dependent cache misses per state; here a source's state is a few
// tens of KiB of LDS and only the adjacency rows and the settle records touch
// memory. Nodes are laid out along a Hilbert curve; LDS holds the pages (runs
// of 2^ps nodes) a search has touched, found through a page table, so a lookup
// needs no hash and the result passes walk nodes in address order, 64
// neighbouring words per atomic instruction.
//
// LDS per node of a touched page: the routes of its two states (8 B) and two
// 16-bit words; every other word is scratch in HBM (L2 mostly) that is written
// and forgotten, or read where its latency overlaps another load's. Not stored
// because they follow from what is: a node's best route and seconds (the smaller
// of its states' until an offer falls in the tie band of the best; from then on
// explicit words), a state's seconds at push (its seconds, until a tied offer
// lowers them), its path count (that of its one predecessor; a state with
// several gets a numbered count), predecessor lists (the one predecessor's
// settle position; several: a list). Dependencies of the back-propagation lie
// over the routes, for the states that precede another only (63% on a lattice).
//
// What bounds it: the latency of one batch's instructions and LDS accesses
// (about 8 states, 27 edges; waits are 57% of a wave's cycles on the dual below),
// times the waves a CU's LDS holds. On the dual of
// the 150x150 lattice at [500, 1000, 2000] m (32.5k sources, 1,870 states each)
// 20 KiB per wave run eight waves per CU: 20.2 ms, against 55.1 ms for the
// lane-per-source kernel; with seconds, lists and page numbers in LDS too (30
// KiB, five waves) 25.7 ms; with the state words in HBM as well (eleven waves)
// 20.2 ms. The 30x30 dual at [400, 800] m: 0.29 ms against 2.65; the dual of an
// 18x18 lattice cut to 20 m pieces, where nearly every state settles alone:
// 15.0 ms against 37.9.
#include "cs_internal.hpp"
#include "cs_wave.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <queue>

namespace cs {

namespace {

constexpr uint32_t kRow = 4;                  // out-edges of a state's row
constexpr uint32_t kChunk = kWave / kRow;     // states relaxed together
constexpr uint32_t kNoEdge = 0xffffffffu;     // padding entry of a row
constexpr uint32_t kRowSpill = 0xfffffffeu;   // first entry of a row whose edges lie in the spill list {.., begin, count}
constexpr uint32_t kNearGoal = 56;            // a refill brings the near set up to this many states where routes allow
                                              // (an earlier layout, 24.3 ms on the 150x150 dual: with 28, 40, 52 27.3, 25.1, 24.3)
constexpr uint32_t kOwn = 128;                // conflict table entries
constexpr uint32_t kPage = 3;                 // a page: a run of 8 nodes
constexpr uint32_t kLdsStage = 8 * kOwn, kLdsRoutes = kLdsStage + 16 * kWave;
constexpr uint32_t kNoSuper = 0xffu, kNoPage = 0xffffu;  // page tables: not touched
constexpr uint32_t kMaxSupers = 254, kMaxPages = 4096;
constexpr uint32_t kNoInner = 0xffffu;        // a state that precedes no other
constexpr uint32_t kNoState = 0xffffffffu;
constexpr uint32_t kIdxMask = 0x1fffu;        // settle position in a state word
constexpr uint32_t kNoPred = 0x1fffu;         // ... of a state without predecessor (the source's)
constexpr uint32_t kMaxStates = 0x1ff0u;      // settled states per source at most
constexpr uint32_t kEqBit = 0x2000u;          // the predecessor's route equals the state's (lists: set as the state settles)
constexpr uint32_t kMultiBit = 0x4000u;       // several predecessors (list in scratch)
constexpr uint32_t kSpillBit = 0x8000u;       // first state's word: the node's best lies in scratch
constexpr uint32_t kSign = 0x80000000u;
constexpr uint32_t kFree = 0xffffffffu;       // near lane without a state
constexpr uint32_t kPassT = 4;                // thresholds one back-propagation pass holds at most
constexpr uint32_t kFarRegs = 8;              // far-list entries per lane a refill holds in registers
// Below L by this much a state is out of every tie band an offer of L or more
// can open (1e-4 on either side of a best route itself within 1e-4 of the
// state's, and f32 rounding).
constexpr float kClear = 1.0f - 4e-4f;
constexpr uint32_t kFailRoom = 1u, kFailPreds = 2u;

// One (graph, request) pair of a launch.
struct WaveJob {
  const uint4 *row;       // [2N][kRow] {target | slot << 31, seconds, angle, 1e-6 length}, kNoEdge pads
  const float *row_wm;    // [2N][kRow] smallest increment out of the entry's target state
  const uint4 *spill;     // rows of more than kRow edges
  const float *spill_wm;
  const float *wm;        // [2N] smallest increment out of a state
  const uint32_t *perm;   // original node -> node
  const uint32_t *orig;   // node -> original node
  const uint8_t *eligible;  // by original node
  const uint32_t *sources;  // original nodes
  const float *src_wt;
  double *acc;            // [4][T][N]
  uint32_t *reach;
  uint32_t N, T, flags;   // 1 closeness, 2 betweenness, 4 track reach
  float maxsec, tol, unit, offset, step;  // step: first width of the near list's route range
  float sec_thr[kMaxT];
};
typedef __attribute__((address_space(4))) const WaveJob CWaveJob;

struct WaveArgs {
  const WaveJob *jobs;
  const uint2 *items;     // {job, source position}; null: job 0, position = item
  uint32_t n_items;
  uint32_t P, Q, ss, S, F;  // pages, superpages (2^ss nodes), settled states and far-list entries of a source
  uint32_t n_pt;          // superpage table entries
  uint32_t maxp;          // predecessors of one state at most
  uint32_t o_pw, o_pt, o_pt2;  // LDS offsets (conflict table, exchange and routes at fixed ones)
  uint32_t dcap;          // f64 words of the back-propagation overlay (from 0 up to the state words)
  char *ws;               // [waves][stride] scratch, never cleared
  size_t stride;
  uint32_t o_secs, o_far, o_pl, o_iid, o_seed, o_ext, o_psec, o_best, o_sig;  // scratch offsets (records at 0)
  unsigned long long *stats;  // reached, settled states, node-threshold pairs
  uint32_t *next;         // [kXcd] item counters
  uint32_t xbeg[kXcd + 1];
  uint32_t *fail_list, *n_fail, *fail_flags;
  uint32_t *progress;
};

// Orders one wave's memory accesses for the compiler. LDS and vector memory
// serve a single wave's accesses to an address in the order it issues them
// (wavefront scope needs no waits), and nothing here is shared between waves.
__device__ __forceinline__ void order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ float lane_f(float v, uint32_t l) {
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), l));
}
__device__ __forceinline__ uint32_t lane_u(uint32_t v, uint32_t l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float pos(float x) { return __uint_as_float(__float_as_uint(x) & ~kSign); }
__device__ __forceinline__ bool neg(float x) { return (__float_as_uint(x) & kSign) != 0; }
// Wave-wide minimum of a non-negative (or infinite) float.
__device__ __forceinline__ float wave_min_pos(float v) {
  return __uint_as_float(__ockl_wfred_min_u32(__float_as_uint(v)));
}

// One source's search state: LDS arrays, scratch arrays and wave-uniform counts.
struct Search {
  float *R;       // LDS [2 NS] route of each state, sign = settled; infinite: not reached
  uint32_t *PW;   // LDS [NS] two state words: predecessor (unsettled) or own settle position, with bits
  uint8_t *pt;    // LDS superpage table
  uint16_t *pt2;  // LDS [Q][2^(ss - kPage)] pages of each touched superpage
  uint32_t *pl;   // page number of each touched page
  uint16_t *fr;   // far list: states
  unsigned long long *own;  // LDS conflict table
  uint4 *stage;   // LDS [64] exchange between lanes
  char *ws;       // scratch: records [S] {state slot (kSign: a back-propagation group starts here),
                  // predecessor word | path count number << 16, seconds, route} in settle order
  uint32_t np, nq, nf, ns, nsig, ni;
  float Rb;       // every unsettled state with a route below this is in the near set
  uint32_t fail;
  // the near set, one state per lane: slot, {node << 1 | state} id, smallest increment out of it
  uint32_t n_st, n_ds;
  float n_wm;
};

template <typename T>
__device__ __forceinline__ T *at(const Search &q, uint32_t off) { return reinterpret_cast<T *>(q.ws + off); }
__device__ __forceinline__ float *secs_of(const WaveArgs &a, const Search &q) { return at<float>(q, a.o_secs); }
__device__ __forceinline__ uint16_t *preds_of(const WaveArgs &a, const Search &q, uint32_t st) {
  return at<uint16_t>(q, a.o_ext) + (size_t)st * (a.maxp + 1);
}
__device__ __forceinline__ double path_count(const WaveArgs &a, const Search &q, uint32_t number) {
  return number ? ldd(&at<double>(q, a.o_sig)[number - 1]) : 1.0;
}
// Path count number, and route, of the state settled at position p.
__device__ __forceinline__ uint32_t count_no(const Search &q, uint32_t p) { return ld32(&at<uint4>(q, 0)[p].y) >> 16; }
__device__ __forceinline__ float route_at(const Search &q, uint32_t p) {
  return __uint_as_float(ld32(&at<uint4>(q, 0)[p].w));
}
__device__ __forceinline__ uint32_t node_of(const Search &q, uint32_t slot) {
  return (q.pl[slot >> kPage] << kPage) | (slot & ((1u << kPage) - 1u));
}
// Seconds at push, by which states at one route settle.
__device__ __forceinline__ float push_secs(const WaveArgs &a, const Search &q, uint32_t st) {
  const float s = ld_f(&secs_of(a, q)[st]);
  return neg(s) ? ld_f(&at<float>(q, a.o_psec)[st]) : s;
}
__device__ __forceinline__ uint32_t orig_state(CWaveJob &jb, uint32_t ds) { return 2 * jb.orig[ds >> 1] + (ds & 1u); }

__device__ __forceinline__ uint32_t page_of(const WaveArgs &a, const Search &q, uint32_t v) {
  const uint32_t sp = q.pt[v >> a.ss];
  return sp == kNoSuper ? kNoPage : q.pt2[(sp << (a.ss - kPage)) | ((v >> kPage) & ((1u << (a.ss - kPage)) - 1u))];
}

// The page of node v, met for the first time: all its states unreached. False
// without room, and then nothing is touched: a superpage is only ever taken with
// a page of it, which is how the clean-up after a search finds its table byte.
__device__ __forceinline__ bool open_page(const WaveArgs &a, Search &q, uint32_t v) {
  const uint32_t lane = lane_id(), rs = a.ss - kPage;
  if (q.np == a.P) return false;
  uint32_t sp = uniform(q.pt[v >> a.ss]);
  if (sp == kNoSuper) {
    if (q.nq == a.Q) return false;
    sp = q.nq++;
    if (lane < (1u << rs)) q.pt2[(sp << rs) + lane] = (uint16_t)kNoPage;
    if (lane == 0) q.pt[v >> a.ss] = (uint8_t)sp;
    order();
  }
  const uint32_t id = q.np++;
  if (lane < (1u << kPage)) {
    *reinterpret_cast<float2 *>(&q.R[2 * ((id << kPage) + lane)]) = make_float2(INFINITY, INFINITY);
    q.PW[(id << kPage) + lane] = 0u;
  }
  if (lane == 0) {
    q.pt2[(sp << rs) | ((v >> kPage) & ((1u << rs) - 1u))] = (uint16_t)id;
    q.pl[id] = v >> kPage;
  }
  order();
  return true;
}

// Puts the lanes' states `want` (slot st, id ds, smallest increment out wm) into free lanes of the near set; what finds no room goes to the far
// list, and the near set's range shrinks to below it.
__device__ __forceinline__ void to_near_set(const WaveArgs &a, Search &q, bool want, uint32_t st, uint32_t ds,
                                            float wm) {
  const uint64_t mw = __ballot(want);
  if (!mw) return;
  const uint64_t mf = __ballot(q.n_st == kFree);
  const uint32_t k = rank_below(mw), room = (uint32_t)__popcll(mf), cnt = (uint32_t)__popcll(mw);
  order();
  if (want && k < room) q.stage[k] = make_uint4(st, ds, __float_as_uint(wm), 0u);
  order();
  if (q.n_st == kFree && rank_below(mf) < cnt) {
    const uint4 x = q.stage[rank_below(mf)];
    q.n_st = x.x;
    q.n_ds = x.y;
    q.n_wm = __uint_as_float(x.z);
  }
  order();
  if (cnt > room) {
    const bool out = want && k >= room;
    if (q.nf + (cnt - room) > a.F) {
      q.fail |= kFailRoom;
      return;
    }
    if (out) q.fr[q.nf + (k - room)] = (uint16_t)st;
    q.nf += cnt - room;
    q.Rb = fminf(q.Rb, wave_min_pos(out ? q.R[st] : INFINITY));
  }
}

// Relaxes one edge per active lane. e: the edge, wm: the smallest increment out
// of its target, ui/ur/us: settle position, route and seconds of the state
// u_ds (slot u_st) that it leaves. Of the lanes whose targets share a conflict
// table entry (one node's always do) the one whose state settles first goes
// first; one state's edges go in row order = lane order, its lanes next to each
// other: four lanes a state (ui kNoState: none), or with `solo` all of one state.
__device__ __forceinline__ void relax(const WaveArgs &a, CWaveJob &jb, Search &q, uint4 e, float wm, uint32_t ui, float ur,
                                      float us, uint32_t u_st, uint32_t u_ds, bool solo) {
  const float one_m = 1.0f - kTieEps, one_p = 1.0f + kTieEps;
  const uint32_t lane = lane_id();
  const float cs = pos(us) + __uint_as_float(e.y);
  const bool act = e.x != kNoEdge && !(cs > jb.maxsec);
  const uint32_t v = e.x & 0x7fffffffu, end = e.x >> 31;
  uint32_t page = act ? page_of(a, q, v) : 0u;
  for (uint64_t m = __ballot(page == kNoPage); m; m = __ballot(page == kNoPage)) {
    const uint32_t lv = lane_u(v, (uint32_t)__builtin_ctzll(m));
    const uint32_t id = q.np;
    if (!open_page(a, q, lv)) {
      q.fail |= kFailRoom;
      return;
    }
    if (page == kNoPage && (v >> kPage) == (lv >> kPage)) page = id;
  }
  const uint32_t slot = (page << kPage) | (v & ((1u << kPage) - 1u));
  const uint32_t st = 2 * slot + end;
  unsigned long long *own = &q.own[slot & (kOwn - 1u)];
  float cr = ur + __uint_as_float(e.z);
  cr = cr + __uint_as_float(e.w);
  unsigned long long key = ((unsigned long long)__float_as_uint(ur) << 32) | lane;
  bool pend = act, ranked = false;
  bool near = false, far = false, took = false;
  order();
  while (__ballot(pend)) {
    if (pend) __hip_atomic_fetch_min(own, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    order();
    // the target's words load with the table's answer
    unsigned long long first = key;
    float2 r2 = make_float2(0.0f, 0.0f);
    uint32_t pw2 = 0;
    if (pend) {
      first = *own;
      r2 = *reinterpret_cast<const float2 *>(&q.R[2 * slot]);
      pw2 = q.PW[slot];
    }
    order();
    if (pend) *own = ~0ull;
    const bool win = pend && first == key;
    if (!ranked) {
      // two states at one route: their order is by seconds at push, then by id
      const bool even = pend && !win && (uint32_t)(first >> 32) == (uint32_t)(key >> 32);
      if (__ballot(even)) {
        const uint32_t other = (uint32_t)__shfl((int)u_ds, even ? (int)((uint32_t)first & 63u) : (int)lane);
        if (__ballot(even && other != u_ds)) {
          const float ps = act ? (neg(us) ? ld_f(&at<float>(q, a.o_psec)[u_st]) : us) : INFINITY;
          const uint32_t os = act ? orig_state(jb, u_ds) : 0xffffffffu;
          const float rr = act ? ur : INFINITY;
          uint32_t rk = 0;
          for (uint32_t j = 0; j < kWave; ++j) {
            const float rj = lane_f(rr, j), pj = lane_f(ps, j);
            const uint32_t oj = lane_u(os, j);
            rk += (rj < rr || (rj == rr && (pj < ps || (pj == ps && oj < os)))) ? 1u : 0u;
          }
          key = ((unsigned long long)rk << 32) | lane;
          ranked = true;
          order();
          continue;
        }
      }
    }
    const float cur = end ? r2.y : r2.x;
    if (win && !neg(cur)) {
      const float b = fminf(cur, pos(end ? r2.x : r2.y));
      uint32_t pw = end ? pw2 >> 16 : pw2 & 0xffffu;
      const uint32_t mine = ui | (cr == ur ? kEqBit : 0u);
      const bool clear = cr < cur * one_m;
      uint32_t spill = 0;
      // the node's best route and seconds (centrality.rs:695-703): the smaller
      // of its states' until an offer ties with it
      if ((pw2 & kSpillBit) || (!(cr < b * one_m) && cr <= b * one_p)) {
        float2 *bp = &at<float2>(q, a.o_best)[slot];
        if (pw2 & kSpillBit) {
          const float2 bb = ld_f2(bp);
          if (cr < bb.x * one_m) st_f2(bp, make_float2(cr, cs));
          else if (cr <= bb.x * one_p) st_f2(bp, make_float2(bb.x, fminf(bb.y, cs)));
        } else {
          const float bs = pos(ld_f(&secs_of(a, q)[2 * slot + (cur == b ? end : 1u - end)]));
          st_f2(bp, make_float2(b, fminf(bs, cs)));
          spill = kSpillBit;
        }
      }
      if (clear) {
        // a clear improvement: one predecessor, new route and seconds
        took = true;
        pw = mine | (pw & (end ? 0u : kSpillBit));
      } else if (cr <= cur * one_p) {
        // within the tie band: joins the predecessors (once)
        uint16_t *x = preds_of(a, q, st);
        const bool better = cr < cur;
        uint32_t k = 1;
        bool has = false;
        if (pw & kMultiBit) {
          k = ld_u16(&x[0]);
          if (!better)
            for (uint32_t i = 1; i <= k; ++i) has = has || (ld_u16(&x[i]) & kIdxMask) == ui;
        } else {
          has = !better && (pw & kIdxMask) == ui;
          st_u16(&x[1], (uint16_t)(pw & (kIdxMask | kEqBit)));
        }
        if (!has) {
          if (!better) {
            const float old = ld_f(&secs_of(a, q)[st]);
            if (cs < pos(old)) {
              if (!neg(old)) st_f(&at<float>(q, a.o_psec)[st], old);
              st_f(&secs_of(a, q)[st], __uint_as_float(__float_as_uint(cs) | kSign));
            }
          }
          if (k >= a.maxp) {
            q.fail |= kFailPreds;
          } else {
            st_u16(&x[k + 1], (uint16_t)mine);
            st_u16(&x[0], (uint16_t)(k + 1));
            pw |= kMultiBit;
            took = true;
          }
        }
      }
      if (cr < cur) {
        q.R[st] = cr;
        st_f(&secs_of(a, q)[st], cs);
        near = cr < q.Rb && !(cur < q.Rb);
        far = cur == INFINITY && !near;
      }
      q.PW[slot] = (end ? (pw2 & 0xffffu) | (pw << 16) : (pw2 & 0xffff0000u) | pw) | spill;
    }
    pend = pend && !win;
    order();
  }
  if (__ballot(q.fail != 0)) {
    q.fail = wave_or(q.fail);
    return;
  }
  // a state whose offer was taken gets a number among the inner states, which
  // the back-propagation keeps dependencies for; its first lane notes it
  {
    const uint64_t mt = __ballot(took);
    if (solo) {
      // one state's lanes, perhaps not its first: keep a number it has
      uint16_t *id = &at<uint16_t>(q, a.o_iid)[uniform(ui)];
      if (mt && uniform(ld_u16(id)) == kNoInner) {
        if (lane == 0) st_u16(id, (uint16_t)q.ni);
        ++q.ni;
      }
    } else {
      const bool inner = ((mt >> (lane & ~(kRow - 1u))) & ((1u << kRow) - 1u)) != 0;
      const uint64_t ml = __ballot(inner && lane % kRow == 0);
      if (ui != kNoState && lane % kRow == 0)
        st_u16(&at<uint16_t>(q, a.o_iid)[ui], (uint16_t)(inner ? q.ni + rank_below(ml) : kNoInner));
      q.ni += (uint32_t)__popcll(ml);
    }
    if (q.ni > a.dcap) {
      q.fail |= kFailRoom;
      return;
    }
  }
  // newly reached and improved states join the near set or the far list
  const uint64_t mf = __ballot(far);
  if (mf) {
    if (q.nf + (uint32_t)__popcll(mf) > a.F) {
      q.fail |= kFailRoom;
      return;
    }
    if (far) q.fr[q.nf + rank_below(mf)] = (uint16_t)st;
    q.nf += (uint32_t)__popcll(mf);
  }
  to_near_set(a, q, near, st, 2 * v + end, wm);
  order();
}

// Moves the states with the smallest routes from the far list into the near
// set, about kNearGoal of them; none of the near set lies below Rb. `step` is
// the width of routes that brought about that many last time.
__device__ __forceinline__ void refill(const WaveArgs &a, CWaveJob &jb, Search &q, float &step) {
  const uint32_t lane = lane_id();
  // what is left in the near set (an overflow had shrunk its range) goes back
  {
    const uint64_t m = __ballot(q.n_st != kFree);
    if (m) {
      if (q.nf + (uint32_t)__popcll(m) > a.F) {
        q.fail |= kFailRoom;
        return;
      }
      if (q.n_st != kFree) q.fr[q.nf + rank_below(m)] = (uint16_t)q.n_st;
      q.nf += (uint32_t)__popcll(m);
      q.n_st = kFree;
      order();
    }
  }
  // the list's first kFarRegs * 64 entries in registers (infinite: settled)
  float r[kFarRegs];
  uint32_t st[kFarRegs];
  float rm = INFINITY;
#pragma unroll
  for (uint32_t k = 0; k < kFarRegs; ++k) {
    const uint32_t i = k * kWave + lane;
    st[k] = 0;
    r[k] = INFINITY;
    if (k * kWave < q.nf && i < q.nf) st[k] = q.fr[i];
  }
#pragma unroll
  for (uint32_t k = 0; k < kFarRegs; ++k) {
    const uint32_t i = k * kWave + lane;
    if (k * kWave < q.nf && i < q.nf) {
      const float x = q.R[st[k]];
      r[k] = neg(x) ? INFINITY : x;
      rm = fminf(rm, r[k]);
    }
  }
  for (uint32_t b = kFarRegs * kWave; b < q.nf; b += kWave)
    if (b + lane < q.nf) {
      const float x = q.R[q.fr[b + lane]];
      if (!neg(x)) rm = fminf(rm, x);
    }
  const float r0 = wave_min_pos(rm);
  if (r0 == INFINITY) {  // every state listed has settled
    q.nf = 0;
    return;
  }
  float lim = INFINITY;
  for (;;) {
    lim = r0 + step;
    if (!(lim > r0)) lim = __uint_as_float(__float_as_uint(r0) + 1u);  // the next f32: r0 alone
    uint32_t cnt = 0;
#pragma unroll
    for (uint32_t k = 0; k < kFarRegs; ++k)
      if (k * kWave < q.nf) cnt += (uint32_t)__popcll(__ballot(r[k] < lim));
    for (uint32_t b = kFarRegs * kWave; b < q.nf; b += kWave) {
      const float x = b + lane < q.nf ? q.R[q.fr[b + lane]] : INFINITY;
      cnt += (uint32_t)__popcll(__ballot(!neg(x) && x < lim));
    }
    if (cnt <= kNearGoal) {
      if (cnt < kNearGoal / 3) step *= 2.0f;
      break;
    }
    if (lim == __uint_as_float(__float_as_uint(r0) + 1u)) {  // that many states at one route
      if (cnt <= kWave) break;
      q.fail |= kFailRoom;
      return;
    }
    step *= 0.5f;
  }
  q.Rb = lim;
  // keep the rest; those taken (at most 64) go through the stage to the lanes
  uint32_t out = 0, got = 0;
  auto place = [&](uint32_t s, float x) {
    const bool go = x < lim, stay = x < INFINITY && !go;
    const uint64_t mg = __ballot(go), ms = __ballot(stay);
    if (stay) q.fr[out + rank_below(ms)] = (uint16_t)s;
    if (go) q.stage[got + rank_below(mg)].x = s;
    out += (uint32_t)__popcll(ms);
    got += (uint32_t)__popcll(mg);
    order();
  };
  order();
#pragma unroll
  for (uint32_t k = 0; k < kFarRegs; ++k)
    if (k * kWave < q.nf) place(st[k], r[k]);
  for (uint32_t b = kFarRegs * kWave; b < q.nf; b += kWave) {
    uint32_t s = 0;
    float x = INFINITY;
    if (b + lane < q.nf) {
      s = q.fr[b + lane];
      x = q.R[s];
      if (neg(x)) x = INFINITY;
    }
    order();
    place(s, x);
  }
  q.nf = out;
  if (lane < got) {
    q.n_st = q.stage[lane].x;
    q.n_ds = 2 * node_of(q, q.n_st >> 1) + (q.n_st & 1u);
    q.n_wm = jb.wm[q.n_ds];
  }
  order();
}

// The forward search of one source (a node of the launch's order).
__device__ __forceinline__ void search(const WaveArgs &a, CWaveJob &jb, Search &q, uint32_t src) {
  const uint32_t lane = lane_id();
  q.np = q.nq = q.nf = q.ns = q.nsig = q.ni = q.fail = 0;
  q.n_st = kFree;
  q.n_ds = 0;
  q.n_wm = 0.0f;
  if (!open_page(a, q, src)) {
    q.fail |= kFailRoom;
    return;
  }
  order();
  {
    const uint32_t slot = src & ((1u << kPage) - 1u);
    if (lane < 2) {
      q.R[2 * slot + lane] = 0.0f;
      st_f(&secs_of(a, q)[2 * slot + lane], 0.0f);
      q.n_st = 2 * slot + lane;
      q.n_ds = 2 * src + lane;
      q.n_wm = jb.wm[q.n_ds];
    }
    if (lane == 0) q.PW[slot] = kNoPred | (kNoPred << 16);
  }
  float step = jb.step;
  q.Rb = step;
  order();
  uint32_t gstart = 0;  // first state of the current back-propagation group
  for (;;) {
    // ---- how far the routes are safe (the seconds are wanted further down)
    float r = INFINITY, us = 0.0f;
    if (q.n_st != kFree) {
      us = ld_f(&secs_of(a, q)[q.n_st]);
      r = q.R[q.n_st];
      if (neg(r)) {  // settled through another lane
        q.n_st = kFree;
        r = INFINITY;
      }
    }
    const float rmin = wave_min_pos(r), lmin = wave_min_pos(r + q.n_wm);
    if (!(rmin < q.Rb)) {
      if (rmin == INFINITY && q.nf == 0) break;
      refill(a, jb, q, step);
      if (q.fail) return;
      continue;
    }
    float L = fminf(lmin * kClear, q.Rb);
    uint64_t ms = __ballot(r < L);
    for (uint32_t tries = 0; (uint32_t)__popcll(ms) > kChunk && tries < 40; ++tries) {
      L = rmin + (L - rmin) * 0.5f;
      ms = __ballot(r < L);
    }
    if (!ms || (uint32_t)__popcll(ms) > kChunk) {
      // none is safe (or none apart) but the first in settle order
      ms = __ballot(r == rmin);
      if (ms & (ms - 1)) {
        const float ps = r == rmin ? push_secs(a, q, q.n_st) : INFINITY;
        ms = __ballot(ps == wave_min_pos(ps));
        if (ms & (ms - 1)) {
          const uint32_t os = (ms >> lane) & 1ull ? orig_state(jb, q.n_ds) : 0xffffffffu;
          ms = __ballot(os == __ockl_wfred_min_u32(os));
        }
      }
      ms &= ~ms + 1;
    }
    // ---- settle. A state may sit in two lanes (an overflow of the near set):
    // the first to set its sign has it.
    const uint32_t my_st = q.n_st, slot = my_st >> 1, shift = (my_st & 1u) * 16u;
    bool on = (ms >> lane) & 1ull;
    uint32_t pw = 0;
    if (on) {
      const uint32_t old = __hip_atomic_fetch_or(reinterpret_cast<uint32_t *>(&q.R[my_st]), kSign, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP);
      pw = (q.PW[slot] >> shift) & 0xffffu;
      q.n_st = kFree;
      on = !(old & kSign);
    }
    ms = __ballot(on);
    const uint32_t n = (uint32_t)__popcll(ms);
    if (q.ns + n > a.S) {
      q.fail |= kFailRoom;
      return;
    }
    const uint32_t rank = rank_below(ms), idx = q.ns + rank;
    order();
    if (on) {
      q.stage[2 * rank] = make_uint4(my_st, q.n_ds, idx, __float_as_uint(r));
      q.stage[2 * rank + 1].x = __float_as_uint(us);
    }
    order();
    // ---- their rows: four lanes a state
    const bool has = lane / kRow < n;
    uint4 x = make_uint4(0u, 0u, 0u, 0u), e = make_uint4(kNoEdge, 0u, 0u, 0u);
    float w = 0.0f, xs = 0.0f;
    if (has) {
      x = q.stage[2 * (lane / kRow)];
      xs = __uint_as_float(q.stage[2 * (lane / kRow) + 1].x);
      e = jb.row[(size_t)x.y * kRow + lane % kRow];
      w = jb.row_wm[(size_t)x.y * kRow + lane % kRow];
    }
    order();
    // ---- while they load: a record and a path count
    {
      const bool multi = on && (pw & kMultiBit);
      const bool single = on && !multi && (pw & kIdxMask) != kNoPred;
      uint32_t sn = 0;
      // a back-propagation group goes on while no state's predecessor is in it
      bool inside = single && (pw & kIdxMask) >= gstart;
      // with no state of several predecessors so far every path count is one
      if (q.nsig && single) sn = count_no(q, pw & kIdxMask);
      const uint64_t mm = __ballot(multi);
      if (mm) {
        if (multi) {
          uint16_t *pl = preds_of(a, q, my_st);
          const uint32_t k = ld_u16(&pl[0]);
          double sg = 0.0;
          for (uint32_t i = 1; i <= k; ++i) {
            const uint32_t p = ld_u16(&pl[i]) & kIdxMask;
            sg += path_count(a, q, count_no(q, p));
            st_u16(&pl[i], (uint16_t)(p | (route_at(q, p) == r ? kEqBit : 0u)));
            inside = inside || p >= gstart;
          }
          sn = q.nsig + rank_below(mm) + 1;
          std_(&at<double>(q, a.o_sig)[sn - 1], sg);
        }
        q.nsig += (uint32_t)__popcll(mm);
      }
      const bool fresh = __ballot(inside) != 0;
      if (fresh) gstart = q.ns;
      if (on) {
        at<uint4>(q, 0)[idx] = make_uint4(my_st | (fresh && rank == 0 ? kSign : 0u),
                                          (pw & (kIdxMask | kEqBit | kMultiBit)) | (sn << 16),
                                          __float_as_uint(pos(us)), __float_as_uint(r));
        // the state's half of its node's words holds its own position now
        reinterpret_cast<uint16_t *>(q.PW)[my_st] = (uint16_t)((pw & kSpillBit) | idx);
      }
    }
    q.ns += n;
    order();
    const uint64_t msp = __ballot(e.x == kRowSpill);
    if (!msp) {
      relax(a, jb, q, e, w, has ? x.z : kNoState, __uint_as_float(x.w), xs, x.x, x.y, false);
      if (q.fail) return;
      continue;
    }
    // some state has a longer row: one state at a time, in settle order
    uint32_t rk = 0;
    {
      const float rr = __uint_as_float(x.w);
      const float ps = has ? (neg(xs) ? ld_f(&at<float>(q, a.o_psec)[x.x]) : xs) : INFINITY;
      const uint32_t os = has ? orig_state(jb, x.y) : 0xffffffffu;
      for (uint32_t k = 0; k < n; ++k) {
        const float rj = lane_f(rr, k * kRow), pj = lane_f(ps, k * kRow);
        const uint32_t oj = lane_u(os, k * kRow);
        rk += (rj < rr || (rj == rr && (pj < ps || (pj == ps && oj < os)))) ? 1u : 0u;
      }
    }
#pragma unroll 1
    for (uint32_t k = 0; k < n; ++k) {
      const uint32_t l = (uint32_t)__builtin_ctzll(__ballot(has && rk == k));
      const uint32_t kst = lane_u(x.x, l), kds = lane_u(x.y, l), ki = lane_u(x.z, l);
      const float kr = lane_f(__uint_as_float(x.w), l), ks = lane_f(xs, l);
      const bool sp = (msp >> l) & 1ull;
      if (lane == 0) st_u16(&at<uint16_t>(q, a.o_iid)[ki], (uint16_t)kNoInner);
      order();
      const uint32_t beg = sp ? lane_u(e.y, l) : 0u, cnt = sp ? lane_u(e.z, l) : kRow;
#pragma unroll 1
      for (uint32_t j = 0; j < cnt; j += kWave) {
        uint4 f = make_uint4(kNoEdge, 0u, 0u, 0u);
        float fw = 0.0f;
        if (j + lane < cnt) {
          f = sp ? jb.spill[beg + j + lane] : jb.row[(size_t)kds * kRow + lane];
          fw = sp ? jb.spill_wm[beg + j + lane] : jb.row_wm[(size_t)kds * kRow + lane];
        }
        relax(a, jb, q, f, fw, ki, kr, ks, kst, kds, true);
        if (q.fail) return;
      }
    }
  }
}

// Next item for a wave on XCD x: its own share first, then the others'.
__device__ __forceinline__ uint32_t next_item(const WaveArgs &a, uint32_t x) {
  uint32_t si = a.n_items;
  if (lane_id() == 0) {
    for (uint32_t k = 0; k < kXcd; ++k) {
      const uint32_t xx = (x + k) % kXcd;
      const uint32_t len = a.xbeg[xx + 1] - a.xbeg[xx];
      if (__hip_atomic_load(&a.next[xx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= len) continue;
      const uint32_t i = atomicAdd(&a.next[xx], 1u);
      if (i < len) {
        si = a.xbeg[xx] + i;
        break;
      }
    }
  }
  return uniform(si);
}

__global__ __launch_bounds__(kWave) void k_angular_wave(WaveArgs a) {
  extern __shared__ __align__(16) char wave_lds[];
  const uint32_t lane = lane_id();
  Search q;
  q.own = reinterpret_cast<unsigned long long *>(wave_lds);
  q.stage = reinterpret_cast<uint4 *>(wave_lds + kLdsStage);
  q.R = reinterpret_cast<float *>(wave_lds + kLdsRoutes);
  q.PW = reinterpret_cast<uint32_t *>(wave_lds + a.o_pw);
  q.pt = reinterpret_cast<uint8_t *>(wave_lds + a.o_pt);
  q.pt2 = reinterpret_cast<uint16_t *>(wave_lds + a.o_pt2);
  q.ws = a.ws + (size_t)blockIdx.x * a.stride;
  q.fr = at<uint16_t>(q, a.o_far);
  q.pl = at<uint32_t>(q, a.o_pl);
  for (uint32_t i = lane; i < a.n_pt; i += kWave) q.pt[i] = (uint8_t)kNoSuper;
  uint32_t pdone = a.progress ? uniform(__hip_atomic_load(&a.progress[blockIdx.x], __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_SYSTEM)) : 0u;
  unsigned long long st_reached = 0, st_states = 0, st_within = 0;
  for (;;) {
    const uint32_t item = next_item(a, blockIdx.x % kXcd);
    if (item >= a.n_items) break;
    uint32_t job = 0, si = item;
    if (a.items) {
      const uint2 it = a.items[item];
      job = uniform(it.x);
      si = uniform(it.y);
    }
    CWaveJob &jb = ((CWaveJob *)a.jobs)[job];
    const uint32_t src = uniform(jb.perm[jb.sources[si]]);
    const float wt = jb.src_wt[si];
    for (uint32_t i = lane; i < kOwn; i += kWave) q.own[i] = ~0ull;  // (the back-propagation lies over it)
    order();
    search(a, jb, q, src);
    if (q.fail) {
      if (lane == 0) {
        const uint32_t k = atomicAdd(a.n_fail, 1u);
        a.fail_list[k] = item;
        atomicOr(a.fail_flags, q.fail);
      }
      for (uint32_t i = lane; i < q.np; i += kWave) q.pt[q.pl[i] >> (a.ss - kPage)] = (uint8_t)kNoSuper;
      order();
      continue;
    }
    order();
    const uint32_t T = jb.T, ns = q.ns, slots = q.np << kPage, ni = q.ni;
    const size_t NN = jb.N;
    double *seed = at<double>(q, a.o_seed);
    // ---- every reached node in address order: closeness terms
    // (centrality.rs:1995-2033) and its terminal states' seeds
    // (best_angular_target_states, :793-821)
    for (uint32_t s0 = 0; s0 < slots; s0 += kWave) {
      const uint32_t slot = s0 + lane;
      bool hit = false;
      float r0 = INFINITY, r1 = INFINITY;
      uint32_t v = 0, pw2 = 0;
      if (slot < slots) {
        v = node_of(q, slot);
        const float2 r2 = *reinterpret_cast<const float2 *>(&q.R[2 * slot]);
        r0 = pos(r2.x);
        r1 = pos(r2.y);
        pw2 = q.PW[slot];
        hit = fminf(r0, r1) < INFINITY;
      }
      st_reached += (uint32_t)__popcll(__ballot(hit));
      if (!hit) continue;
      const float2 c2 = ld_f2(&at<float2>(q, a.o_secs)[slot]);
      const float c0 = pos(c2.x), c1 = pos(c2.y);
      float br = r0 <= r1 ? r0 : r1, bs = r0 <= r1 ? c0 : c1;
      if (pw2 & kSpillBit) {
        const float2 bb = ld_f2(&at<float2>(q, a.o_best)[slot]);
        br = bb.x;
        bs = bb.y;
      }
      const bool other = v != src && isfinite(bs);
      if (other) {
        double *accv = jb.acc + v;
        const float far_ang = jb.offset + (br / jb.unit);
        const float harm_ang = 1.0f + (br / jb.unit);
        for (uint32_t t = 0; t < T; ++t) {
          if (!(bs <= jb.sec_thr[t])) continue;
          ++st_within;
          if (jb.flags & 4u) atomicAdd(&jb.reach[t], 1u);
          if (jb.flags & 1u) {
            gadd_f64(&accv[((size_t)0 * T + t) * NN], (double)wt);
            gadd_f64(&accv[((size_t)1 * T + t) * NN], (double)(far_ang * wt));
            gadd_f64(&accv[((size_t)2 * T + t) * NN], (double)((1.0f / harm_ang) * wt));
          }
        }
      }
      if (jb.flags & 2u) {
        const bool h0 = r0 < INFINITY, h1 = r1 < INFINITY;
        const uint32_t i0 = pw2 & kIdxMask, i1 = (pw2 >> 16) & kIdxMask;
        const double pc = other ? (jb.eligible[jb.orig[v]] ? 0.5 : 1.0) : 0.0;
        const float lim = br * (1.0f + jb.tol);
        const bool u0 = other && h0 && r0 <= lim, u1 = other && h1 && r1 <= lim;
        double g0 = 1.0, g1 = 1.0;
        if (u0 && u1) {  // the split needs the path counts
          g0 = path_count(a, q, count_no(q, i0));
          g1 = path_count(a, q, count_no(q, i1));
        }
        for (uint32_t t = 0; t < T; ++t) {
          const float lt = jb.sec_thr[t];
          const bool in = bs <= lt;
          const bool w0 = in && u0 && !(c0 > lt), w1 = in && u1 && !(c1 > lt);
          const double tot = (w0 ? g0 : 0.0) + (w1 ? g1 : 0.0);
          if (h0) std_(&seed[(size_t)t * a.S + i0], w0 ? (w1 ? pc * (g0 / tot) : pc) : 0.0);
          if (h1) std_(&seed[(size_t)t * a.S + i1], w1 ? (w0 ? pc * (g1 / tot) : pc) : 0.0);
        }
      }
    }
    // ---- betweenness (centrality.rs:2037-2096, 823-873): dependencies over the
    // settled states in reverse groups; no state of a group precedes another.
    // A predecessor at an equal route is visited before its successor in the
    // reference's order (equal routes in settle order), so what the successor
    // passes on never counts: kEqBit skips it.
    if (jb.flags & 2u) {
      order();
      double *dep = reinterpret_cast<double *>(wave_lds);
      const uint4 *rec = at<uint4>(q, 0);
      const uint16_t *iid = at<uint16_t>(q, a.o_iid);
      const uint32_t fit = a.dcap / (ni ? ni : 1u);
      const uint32_t per = fit < 1u ? 1u : (fit < kPassT ? fit : kPassT);
      for (uint32_t t0 = 0; t0 < T; t0 += per) {
        const uint32_t nt = T - t0 < per ? T - t0 : per;
        order();
        for (uint32_t i = lane; i < nt * ni; i += kWave) dep[i] = 0.0;
        order();
        const uint32_t last = (ns - 1) & ~(kWave - 1u);
        uint4 rn = make_uint4(0u, 0u, __float_as_uint(INFINITY), 0u);
        uint32_t in = kNoInner, pn = kNoInner;  // the state's own number and its predecessor's
        double gn[kPassT];
        auto load = [&](uint32_t w) {
          rn = make_uint4(0u, 0u, __float_as_uint(INFINITY), 0u);
          in = pn = kNoInner;
          if (w + lane < ns) {
            rn = rec[w + lane];
            in = ld_u16(&iid[w + lane]);
#pragma unroll
            for (uint32_t k = 0; k < kPassT; ++k)
              if (k < nt) gn[k] = ldd(&seed[(size_t)(t0 + k) * a.S + w + lane]);
          }
        };
        // the predecessors' numbers, once the records are there
        auto load_preds = [&]() {
          const uint32_t p = rn.y;
          if (__uint_as_float(rn.z) < INFINITY && !(p & (kMultiBit | kEqBit)) && (p & kIdxMask) != kNoPred) pn = ld_u16(&iid[p & kIdxMask]);
        };
#pragma unroll
        for (uint32_t k = 0; k < kPassT; ++k) gn[k] = 0.0;
        load(last);
        load_preds();
        for (int w0 = (int)last; w0 >= 0; w0 -= (int)kWave) {
          const uint32_t rx = rn.x, rw = rn.y;
          const float secs = __uint_as_float(rn.z);
          const uint32_t own = in, pred = pn;
          double sd[kPassT];
#pragma unroll
          for (uint32_t k = 0; k < kPassT; ++k) sd[k] = gn[k];
          if (w0 > 0) load((uint32_t)w0 - kWave);  // the next window, in flight over this one's groups
          const uint32_t idx = (uint32_t)w0 + lane;
          const uint64_t starts = __ballot(idx < ns && (rx & kSign));
          const uint32_t sg = rw >> 16;
          const bool multi = (rw & kMultiBit) != 0;
          uint32_t hi = ns - (uint32_t)w0 < kWave ? ns - (uint32_t)w0 : kWave;
          while (hi > 0) {
            const uint64_t below = hi < 64 ? starts & ((1ull << hi) - 1ull) : starts;
            const uint32_t lo = below ? 63u - (uint32_t)__builtin_clzll(below) : 0u;
            if (lane >= lo && lane < hi) {
#pragma unroll
              for (uint32_t k = 0; k < kPassT; ++k) {
                if (k >= nt) continue;
                double *d = dep + (size_t)k * ni;
                if (!(secs <= jb.sec_thr[t0 + k])) {  // beyond the threshold: takes part in nothing
                  if (own != kNoInner) d[own] = 0.0;
                  continue;
                }
                double total = sd[k];
                if (own != kNoInner) {
                  total = sd[k] + d[own];
                  d[own] = total - sd[k];  // the state's credit
                }
                if (total == 0.0) continue;
                if (!multi) {
                  if (pred != kNoInner) wadd_f64(&d[pred], total);
                } else {
                  const uint16_t *x = preds_of(a, q, rx & ~kSign);
                  const uint32_t np = ld_u16(&x[0]);
                  const double sw = path_count(a, q, sg);
                  for (uint32_t i = 1; i <= np; ++i) {
                    const uint32_t p = ld_u16(&x[i]);
                    if (p & kEqBit) continue;
                    const double sv = path_count(a, q, count_no(q, p & kIdxMask));
                    wadd_f64(&d[ld_u16(&iid[p & kIdxMask])], (sv / sw) * total);
                  }
                }
              }
            }
            order();
            hi = lo;
          }
          if (w0 > 0) load_preds();
        }
        // the credits of a node's two states, in address order
        for (uint32_t slot = lane; slot < slots; slot += kWave) {
          const uint32_t pw2 = q.PW[slot];
          const uint32_t v = node_of(q, slot);
          if (v == src) continue;
          // position 0 is a state of the source, so 0 marks a state not reached
          const uint32_t i0 = pw2 & kIdxMask, i1 = (pw2 >> 16) & kIdxMask;
          const uint32_t j0 = i0 ? ld_u16(&iid[i0]) : kNoInner, j1 = i1 ? ld_u16(&iid[i1]) : kNoInner;
#pragma unroll
          for (uint32_t k = 0; k < kPassT; ++k) {
            if (k >= nt) continue;
            const double x0 = j0 != kNoInner ? dep[(size_t)k * ni + j0] : 0.0;
            const double x1 = j1 != kNoInner ? dep[(size_t)k * ni + j1] : 0.0;
            double c = 0.0;
            if (x0 > 0.0) c += x0 * (double)wt;
            if (x1 > 0.0) c += x1 * (double)wt;
            if (c != 0.0) gadd_f64(&jb.acc[((size_t)3 * T + t0 + k) * NN + v], c);
          }
        }
      }
    }
    st_states += ns;
    order();
    for (uint32_t i = lane; i < q.np; i += kWave) q.pt[q.pl[i] >> (a.ss - kPage)] = (uint8_t)kNoSuper;
    order();
    if (a.progress) {
      ++pdone;
      if (lane == 0)
        __hip_atomic_store(&a.progress[blockIdx.x], pdone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  const unsigned long long within = wave_sum(st_within);
  if (lane == 0) {
    atomicAdd(&a.stats[0], st_reached);
    atomicAdd(&a.stats[1], st_states);
    atomicAdd(&a.stats[2], within);
  }
}

// dst[m][t][orig[d]] += src[m][t][d], dst rows of stride tstride thresholds
__global__ void k_wave_rows(double *dst, const double *src, const uint32_t *orig, uint32_t N, uint32_t T,
                            uint32_t tstride) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)N * 4 * T) return;
  const size_t r = i / N, d = i - r * N, m = r / T, t = r - m * T;
  const double v = src[i];
  if (v != 0.0) dst[(m * tstride + t) * N + orig[d]] += v;
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct WaveWorkspace {
  DevVec scratch, acc, ctl, jobs, items, fail;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  std::mutex mu;
};
std::mutex g_wave_mu;
std::map<int, std::unique_ptr<WaveWorkspace>> g_wave;

WaveWorkspace &wave_ws(int device) {
  std::lock_guard<std::mutex> lk(g_wave_mu);
  auto &p = g_wave[device];
  if (!p) p = std::make_unique<WaveWorkspace>();
  return *p;
}

template <typename T>
void to_device(const std::vector<T> &v, T **p) {
  hip_check(hipMalloc(p, sizeof(T) * std::max<size_t>(v.size(), 1)), "hipMalloc angular rows");
  if (!v.empty()) hip_check(hipMemcpy(*p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice), "upload");
}

uint32_t bits(float x) {
  uint32_t b;
  std::memcpy(&b, &x, 4);
  return b;
}

// The graph's rows for the LDS search, built once per speed.
AngWaveGraph &wave_graph(Graph &g, DevEdges &de) {
  if (de.ang_wave) return *de.ang_wave;
  auto w = std::make_unique<AngWaveGraph>();
  const uint32_t n = g.n;
  bool ok = n > 0 && n <= (1u << 22) && g.max_in_deg <= 64;
  std::vector<uint32_t> perm(n), orig(n);
  for (uint32_t v = 0; v < n; ++v) {
    perm[v] = g.ang_perm.empty() ? v : g.ang_perm[v];
    orig[perm[v]] = v;
  }
  std::vector<uint4> ent(ok ? g.m : 0);
  std::vector<float> wm(ok ? 2 * (size_t)n : 0, INFINITY);
  for (uint32_t v = 0; v < n && ok; ++v)
    for (uint32_t j = g.fwd_off[v]; j < g.fwd_off[v + 1]; ++j) {
      const uint32_t e = g.fwd_eid[j];
      const uint32_t u = g.edst[e];
      const float es = edge_seconds(g, v, u, e, de.speed, false), tb = kAngularTieBreak * g.elen[e], ang = g.eang[e];
      if (!(es >= 0.0f) || !(ang >= 0.0f) || !(tb >= 0.0f) || !std::isfinite(es) || !std::isfinite(ang) ||
          !std::isfinite(tb)) {
        ok = false;  // the parallel settling needs increments that never lower a route
        break;
      }
      ent[j] = make_uint4(perm[u] | ((uint32_t)g.slot_dst[e] << 31), bits(es), bits(ang), bits(tb));
      // the state 2v + entry leaves through its other endpoint: source slot 1 - entry
      float &m = wm[2 * (size_t)perm[v] + (1u - (uint32_t)g.slot_src[e])];
      m = std::min(m, ang + tb);
      w->max_w = std::max(w->max_w, ang + tb);
    }
  if (ok) {
    const uint4 pad = make_uint4(kNoEdge, 0u, 0u, 0u);
    std::vector<uint4> row(2 * (size_t)n * kRow, pad), spill;
    std::vector<float> row_wm(2 * (size_t)n * kRow, INFINITY), spill_wm;
    std::vector<uint4> use;
    for (uint32_t v = 0; v < n; ++v)
      for (uint32_t entry = 0; entry < 2; ++entry) {
        use.clear();
        for (uint32_t j = g.fwd_off[v]; j < g.fwd_off[v + 1]; ++j)
          if ((uint32_t)g.slot_src[g.fwd_eid[j]] == 1u - entry) use.push_back(ent[j]);
        const size_t at = (2 * (size_t)perm[v] + entry) * kRow;
        auto target = [&](const uint4 &e) { return wm[2 * (size_t)(e.x & 0x7fffffffu) + (e.x >> 31)]; };
        if (use.size() <= kRow) {
          for (size_t k = 0; k < use.size(); ++k) {
            row[at + k] = use[k];
            row_wm[at + k] = target(use[k]);
          }
        } else {
          row[at] = make_uint4(kRowSpill, (uint32_t)spill.size(), (uint32_t)use.size(), 0u);
          for (const uint4 &e : use) {
            spill.push_back(e);
            spill_wm.push_back(target(e));
          }
        }
      }
    to_device(row, &w->row);
    to_device(row_wm, &w->row_wm);
    to_device(spill, &w->spill);
    to_device(spill_wm, &w->spill_wm);
    to_device(wm, &w->wm);
    to_device(perm, &w->perm);
    to_device(orig, &w->orig);
  }
  if (ok) {
    // A search's time per reached node, which hangs on how many states settle
    // together. The smallest increment out of any state of the front bounds that:
    // its likely size is what two in a hundred states lie below. Measured on
    // duals of lattices with their nodes moved by up to 20, 8, 3, 1 and 0.3 m and
    // of streets cut into pieces (300 sources, about 1,000 nodes each), that
    // increment over the largest and the time: 4e-3 0.96 us, 1.8e-3 1.14, 7.6e-4
    // 1.34, 2.7e-4 2.15, 8.4e-5 3.5, 5e-7 3.1 to 4.2.
    std::vector<float> out;
    for (const float x : wm)
      if (std::isfinite(x)) out.push_back(x);
    float low = 0.0f;
    if (!out.empty() && w->max_w > 0.0f) {
      std::nth_element(out.begin(), out.begin() + out.size() / 50, out.end());
      low = out[out.size() / 50] / w->max_w;
    }
    w->state_ms = 0.95e-3f * std::clamp(std::pow(4e-3f / std::max(low, 1e-9f), 0.3f), 1.0f, 4.4f);
  }
  w->usable = ok;
  de.ang_wave = std::move(w);
  return *de.ang_wave;
}

// Nodes and pages that searches up to maxsec reach: the most over a few sources
// spread over the node order, by plain shortest time (a simplest route takes no
// less), stopped once a search is past what LDS could hold.
const AngWaveGraph::Reach &wave_reach(Graph &g, const DevEdges &de, AngWaveGraph &w, float maxsec) {
  auto it = w.reach.find(maxsec);
  if (it != w.reach.end()) return it->second;
  constexpr uint32_t kProbes = 8, kStop = 8192;
  AngWaveGraph::Reach r;
  const uint32_t n = g.n;
  auto perm = [&](uint32_t v) { return g.ang_perm.empty() ? v : g.ang_perm[v]; };
  auto iperm = [&](uint32_t d) { return g.ang_iperm.empty() ? d : g.ang_iperm[d]; };
  std::vector<float> secs(n, INFINITY);
  std::vector<uint32_t> from(n), seen, pg;
  uint64_t inner = 0, all = 0;
  for (uint32_t k = 0; k < kProbes; ++k) {
    const uint32_t src = iperm((uint32_t)(((uint64_t)2 * k + 1) * n / (2 * kProbes)));
    std::priority_queue<std::pair<float, uint32_t>, std::vector<std::pair<float, uint32_t>>, std::greater<>> h;
    secs[src] = 0.0f;
    seen.assign(1, src);
    h.push({0.0f, src});
    while (!h.empty() && seen.size() < kStop) {
      const auto [s, v] = h.top();
      h.pop();
      if (s > secs[v]) continue;
      for (uint32_t j = g.fwd_off[v]; j < g.fwd_off[v + 1]; ++j) {
        const uint32_t e = g.fwd_eid[j], u = g.edst[e];
        const float cs = s + edge_seconds(g, v, u, e, de.speed, false);
        if (cs > maxsec || !(cs < secs[u])) continue;
        if (secs[u] == INFINITY) seen.push_back(u);
        secs[u] = cs;
        from[u] = v;
        h.push({cs, u});
      }
    }
    r.nodes = std::max<uint32_t>(r.nodes, (uint32_t)seen.size());
    for (uint32_t ps = kPage; ps < 10; ++ps) {
      pg.clear();
      for (uint32_t v : seen) pg.push_back(perm(v) >> ps);
      std::sort(pg.begin(), pg.end());
      r.pages[ps] = std::max<uint32_t>(r.pages[ps], (uint32_t)(std::unique(pg.begin(), pg.end()) - pg.begin()));
    }
    for (uint32_t v : seen) secs[v] = INFINITY;
    all += seen.size();
    pg.clear();
    for (size_t i = 1; i < seen.size(); ++i) pg.push_back(from[seen[i]]);
    std::sort(pg.begin(), pg.end());
    inner += (uint64_t)(std::unique(pg.begin(), pg.end()) - pg.begin());
  }
  r.mean = (float)all / (float)kProbes;
  r.chains = (double)inner > 0.75 * (double)all;
  if (w.reach.size() >= 64) w.reach.clear();
  return w.reach[maxsec] = r;
}

constexpr uint32_t kLdsMax = 160u * 1024u;

// LDS layout of a launch whose sources reach `nodes` nodes on pages[k] runs of
// 2^k; false when it does not fit.
bool wave_layout(WaveArgs &a, uint32_t N, uint32_t nodes, const uint32_t *pages, double room, uint32_t cap,
                 bool chains, uint32_t *lds) {
  uint32_t best = 0xffffffffu;
  WaveArgs pick = a;
  const uint32_t rn = std::min<uint32_t>(N, (uint32_t)(nodes * room) + 8);
  for (uint32_t ss = 6; ss < 10; ++ss) {
    WaveArgs b = a;
    b.ss = ss;
    b.n_pt = (N + (1u << ss) - 1) >> ss;
    b.Q = std::min<uint32_t>(b.n_pt, (uint32_t)(pages[ss] * room) + 1);
    b.P = std::min<uint32_t>((N + (1u << kPage) - 1) >> kPage, (uint32_t)(pages[kPage] * room) + 2);
    b.S = std::min<uint32_t>(2 * rn + 2, kMaxStates);
    if (cap) b.S = std::min(b.S, cap);
    if (b.P > kMaxPages || b.Q > kMaxSupers) continue;
    b.F = 2 * rn + 2;  // (each state joins the far list at most once, but for the near set's overflow)
    const uint32_t ns = b.P << kPage;
    uint32_t o = kLdsRoutes + 8 * ns;
    auto take = [&](uint32_t bytes) {
      const uint32_t at = o;
      o = (o + bytes + 15) & ~15u;
      return at;
    };
    // dependencies of the inner states lie over all of this: nearly every state
    // of a network cut into short pieces is one, under two thirds of a lattice's
    o = std::max(o, (8 * (chains ? b.S : b.S / 3 * 2) + 15) & ~15u);
    b.dcap = o / 8;
    b.o_pw = take(4 * ns);
    b.o_pt = take(b.n_pt);
    b.o_pt2 = take(2 * (b.Q << (ss - kPage)));
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

}  // namespace

AngWaveGraph::~AngWaveGraph() {
  for (void *p : {(void *)row, (void *)row_wm, (void *)spill, (void *)spill_wm, (void *)wm, (void *)perm, (void *)orig})
    (void)hipFree(p);
}

void release_angular_wave_workspaces() {
  std::lock_guard<std::mutex> lk(g_wave_mu);
  for (auto &dv : g_wave) {
    WaveWorkspace &w = *dv.second;
    std::lock_guard<std::mutex> wl(w.mu);
    for (DevVec *d : {&w.scratch, &w.acc, &w.ctl, &w.jobs, &w.items, &w.fail}) d->release();
  }
}

namespace {

// Requests whose searches run in one launch, laid out for the largest of them.
struct WaveClass {
  std::vector<uint32_t> specs;  // of the caller's
  uint32_t n = 0;               // searches
  uint32_t N = 1, T = 1, maxp = 1, nodes = 0;
  uint32_t pages[10] = {0};
  bool chains = false, betw = false;
  double mean = 0.0, visits = 0.0;  // nodes of a search (the most over the requests), of all searches
  double most = 0.0, all = 0.0;     // search time of the slowest request's sources, of all sources (ms)
  double lane = 0.0;                // a lane's time per node (lane_cost)
  uint32_t lds = 0;                 // 0: does not fit
  WaveArgs a;
  double ms = 0.0;
};

// Expected time of a launch, n searches on the waves that its LDS leaves room
// for. Beside the time per node a search has a fixed part that grows with the
// waves a CU runs (its results' atomics): 0.045 ms alone, 0.165 at twelve. On
// the 150x150 lattice's dual, all 32,549 sources, expected and measured ms:
// 400 m 2.1, 2.1; 800 m 3.4, 3.1; 2,000 m 17.4, 17.0; 3,200 m 104, 109.
void wave_cost(WaveClass &c, uint32_t cap, uint32_t cus) {
  std::memset(&c.a, 0, sizeof(c.a));
  // a search settles up to two states a node (1.8 where it reaches thousands):
  // past the positions that a state word holds most would fail
  if (2.0 * c.mean > kMaxStates || !wave_layout(c.a, c.N, c.nodes, c.pages, 1.0, cap, c.chains, &c.lds)) {
    c.lds = 0;
    c.ms = INFINITY;
    return;
  }
  const double W = std::min<double>(c.n, (double)cus * std::min(12u, kLdsMax / c.lds));
  const double fixed = 0.045 + 0.01 * std::max(0.0, W / cus - 1.0);
  c.ms = std::max(fixed + c.most, (c.n * fixed + c.all) / W) + 0.15;
}

// Expected time of a lane-per-source launch. At 100 sources and a reach of 1,000
// a lane's search takes `per` us a node (0.64 of it without betweenness), a
// little more the farther it reaches, and with 32,768 sources 3.6 (2.8) times
// that; from there on more sources take in proportion longer. Measured on the
// same dual to 2,000 m (and on one of 20 m pieces to 800 m): 100 sources 14.5
// (11.3) us, 2,000 27.6 (22), 8,000 38 (27.5), 32,549 (30,000) 52.5 (38.8),
// 113,865 (109,880) 139 (115); all sources to 400 m 37, to 3,200 m 58 (to 200 m 32).
double lane_cost(uint32_t n, uint32_t lanes, double per, double mean, double visits, bool betw) {
  const double m = std::min(std::min<double>(n, lanes), 32768.0), k = std::max(m, 100.0) / 100.0;
  const double t = 1e-3 * per * std::pow(std::max(mean, 30.0) / 1000.0, 0.1) * (betw ? std::pow(k, 0.22) : 0.64 * std::pow(k, 0.255));
  return 0.35 + t * std::max(mean, visits / m);
}

void merge(WaveClass &c, const WaveClass &d) {
  c.specs.insert(c.specs.end(), d.specs.begin(), d.specs.end());
  c.n += d.n;
  c.N = std::max(c.N, d.N);
  c.T = std::max(c.T, d.T);
  c.maxp = std::max(c.maxp, d.maxp);
  c.nodes = std::max(c.nodes, d.nodes);
  for (int k = 0; k < 10; ++k) c.pages[k] = std::max(c.pages[k], d.pages[k]);
  c.chains = c.chains || d.chains;
  c.betw = c.betw || d.betw;
  c.mean = std::max(c.mean, d.mean);
  c.visits += d.visits;
  c.most = std::max(c.most, d.most);
  c.all += d.all;
  c.lane = std::max(c.lane, d.lane);
}

// The requests that search in LDS, by launch; the others are the lanes' (their
// numbers in `lanes`). A wave per source is the faster search until many sources
// have to take turns: the 150x150 lattice's dual to 3,200 m (three waves a CU,
// 32,549 sources) 109 ms against 145 with a lane per source, but a dual of 20 m
// pieces to 1,600 m (one wave a CU) 18 against 47 with 100 sources, 125 against
// 86 with 2,000 and 471 against 108 with 8,000. And a lane launch lasts as long
// as its slowest source, so what it can take along is cheap there.
std::vector<WaveClass> wave_plan(const std::vector<AngSpec> &specs, const std::vector<uint32_t> &count, uint32_t cap,
                                 uint32_t cus, std::vector<uint32_t> *lanes) {
  std::vector<WaveClass> cls;
  WaveClass rest;  // the lanes' part
  for (uint32_t i = 0; i < specs.size(); ++i) {
    const AngSpec &sp = specs[i];
    if (!count[i]) continue;
    // (a larger tolerance rebuilds its predecessors from final routes, Phase 2)
    const bool takes = !(sp.cs.betweenness && sp.cs.tolerance > kTieEps) && sp.cs.maxsec >= 0.0f &&
                       wave_graph(*sp.g, *sp.de).usable;
    WaveClass c;
    c.specs = {i};
    c.n = count[i];
    c.N = sp.g->n;
    c.T = sp.cs.T;
    c.maxp = std::max(1u, sp.g->max_in_deg);
    c.betw = sp.cs.betweenness;
    c.lane = 14.7;
    if (takes) {
      AngWaveGraph &w = *sp.de->ang_wave;
      const AngWaveGraph::Reach &r = wave_reach(*sp.g, *sp.de, w, sp.cs.maxsec);
      c.nodes = r.nodes;
      c.mean = r.mean;
      c.chains = r.chains;
      for (uint32_t ps = kPage; ps < 10; ++ps) c.pages[ps] = r.pages[ps];
      c.visits = (double)c.n * r.mean;
      c.most = (double)w.state_ms * r.mean;
      c.all = c.n * c.most;
      if (w.state_ms > 2e-3f) c.lane = 11.1;  // (as on the pieces)
      wave_cost(c, cap, cus);
    }
    if (!takes || !c.lds) merge(rest, c);
    else cls.push_back(std::move(c));
  }
  // neighbours in size share a launch where that is the faster
  std::sort(cls.begin(), cls.end(), [](const WaveClass &x, const WaveClass &y) { return x.nodes < y.nodes; });
  while (cls.size() > 1) {
    double best = 0.0;
    size_t at = cls.size();
    WaveClass both;
    for (size_t k = 0; k + 1 < cls.size(); ++k) {
      WaveClass m = cls[k];
      merge(m, cls[k + 1]);
      wave_cost(m, cap, cus);
      if (m.lds && cls[k].ms + cls[k + 1].ms - m.ms > best) {
        best = cls[k].ms + cls[k + 1].ms - m.ms;
        at = k;
        both = std::move(m);
      }
    }
    if (at == cls.size()) break;
    cls[at] = std::move(both);
    cls.erase(cls.begin() + at + 1);
  }
  // what a lane launch does sooner goes there, the slowest first
  std::sort(cls.begin(), cls.end(), [](const WaveClass &x, const WaveClass &y) { return x.ms > y.ms; });
  auto lane_ms = [&](const WaveClass &c) {
    return c.n ? lane_cost(c.n, angular_lanes(c.N, c.T, c.maxp, c.n, specs[0].dg->device), c.lane, c.mean, c.visits, c.betw) : 0.0;
  };
  double now = lane_ms(rest);
  for (size_t k = 0; k < cls.size();) {
    WaveClass m = rest;
    merge(m, cls[k]);
    const double with = lane_ms(m);
    if (with - now < cls[k].ms) {
      rest = std::move(m);
      now = with;
      cls.erase(cls.begin() + k);
    } else {
      ++k;
    }
  }
  *lanes = rest.specs;
  return cls;
}

// One launch (two, where some of its sources outgrow their room): `items`
// {request of the caller's, source position}, empty for all n of the one
// request. What is left over goes to rest.
void run_class(WaveWorkspace &ws, WaveClass &c, const std::vector<AngSpec> &specs, std::vector<uint2> items, uint32_t cap,
               uint32_t cus, hipStream_t stream, cs_stats &st, uint32_t *progress, std::vector<uint2> *rest) {
  WaveArgs a = c.a;
  uint32_t lds = c.lds;
  // a little room beyond the probed sources, and more where that costs no
  // resident wave of the launch
  double room = 1.0;
  const uint32_t want = std::min<uint32_t>(c.n, cus * (kLdsMax / lds));
  for (double f : {1.02, 1.05, 1.1, 1.2, 1.5, 2.0}) {
    WaveArgs b = a;
    uint32_t bl = 0;
    if (!wave_layout(b, c.N, c.nodes, c.pages, f, cap, c.chains, &bl) || cus * (kLdsMax / bl) < want) break;
    a = b;
    lds = bl;
    room = f;
  }
  static_assert(sizeof(WaveJob) % 4 == 0, "job table");
  uint32_t n_list = c.n;
  if (!ws.e0) {
    hip_check(hipEventCreate(&ws.e0), "event");
    hip_check(hipEventCreate(&ws.e1), "event");
  }
  size_t rows = 0;
  for (const uint32_t i : c.specs) rows += (size_t)4 * specs[i].cs.T * specs[i].g->n;
  double *acc = static_cast<double *>(ws.acc.get(8 * rows, "angular result rows"));
  hip_check(hipMemsetAsync(acc, 0, 8 * rows, stream), "memset");
  std::vector<WaveJob> jobs(specs.size());  // (of the class's requests)
  size_t at = 0;
  for (const uint32_t i : c.specs) {
    const AngSpec &sp = specs[i];
    const AngWaveGraph &w = *sp.de->ang_wave;
    WaveJob &j = jobs[i];
    std::memset(&j, 0, sizeof(j));
    j.row = w.row;
    j.row_wm = w.row_wm;
    j.spill = w.spill;
    j.spill_wm = w.spill_wm;
    j.wm = w.wm;
    j.perm = w.perm;
    j.orig = w.orig;
    j.eligible = sp.d_eligible;
    j.sources = sp.d_sources;
    j.src_wt = sp.d_wt;
    j.acc = acc + at;
    j.reach = sp.d_reach;
    j.N = sp.g->n;
    j.T = sp.cs.T;
    j.flags = (sp.cs.closeness ? 1u : 0u) | (sp.cs.betweenness ? 2u : 0u) | (sp.cs.track_reach ? 4u : 0u);
    j.maxsec = sp.cs.maxsec;
    j.tol = sp.cs.tolerance;
    j.unit = sp.cs.ang_unit;
    j.offset = sp.cs.far_offset;
    j.step = w.max_w > 0.0f ? w.max_w / 32.0f : 1.0f;
    for (uint32_t t = 0; t < kMaxT; ++t) j.sec_thr[t] = t < sp.cs.T ? (float)sp.cs.seconds[t] : -1.0f;
    at += (size_t)4 * sp.cs.T * sp.g->n;
  }
  WaveJob *d_jobs = static_cast<WaveJob *>(ws.jobs.get(sizeof(WaveJob) * jobs.size(), "job table"));
  hip_check(hipMemcpyAsync(d_jobs, jobs.data(), sizeof(WaveJob) * jobs.size(), hipMemcpyHostToDevice, stream), "copy");
  char *ctl = static_cast<char *>(ws.ctl.get(256, "control words"));
  hip_check(hipMemsetAsync(ctl + 128, 0, 32, stream), "memset stats");
  uint32_t *d_fail = static_cast<uint32_t *>(ws.fail.get(4ull * n_list, "failure list"));
  for (int tier = 0; tier < 2; ++tier) {
    a.jobs = d_jobs;
    a.items = nullptr;
    if (!items.empty()) {
      uint2 *d_items = static_cast<uint2 *>(ws.items.get(sizeof(uint2) * items.size(), "items"));
      hip_check(hipMemcpyAsync(d_items, items.data(), sizeof(uint2) * items.size(), hipMemcpyHostToDevice, stream),
                "copy");
      a.items = d_items;
    }
    a.n_items = n_list;
    a.maxp = c.maxp;
    // scratch of a wave: records | seconds | far list | page numbers | inner numbers |
    // seeds | predecessor lists | push seconds | node bests | path counts
    const size_t slots = (size_t)a.P << kPage;
    size_t o = align256(16ull * a.S);
    auto take = [&](size_t bytes) {
      const size_t at = o;
      o = align256(o + bytes);
      return (uint32_t)at;
    };
    a.o_secs = take(8 * slots);
    a.o_far = take(2ull * a.F);
    a.o_pl = take(4ull * a.P);
    a.o_iid = take(2ull * a.S);
    a.o_seed = take(8ull * c.T * a.S);
    a.o_ext = take(4 * slots * (c.maxp + 1));
    a.o_psec = take(8 * slots);
    a.o_best = take(8 * slots);
    a.o_sig = take(8ull * a.S);
    a.stride = o;
    hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(k_angular_wave),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax), "LDS size");
    int per_cu = 0;
    hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_angular_wave, kWave, lds), "occupancy");
    uint32_t waves = std::min<uint32_t>(n_list, cus * (uint32_t)std::max(per_cu, 1));
    size_t free_b = 0, total_b = 0;
    if (a.stride * waves > ws.scratch.bytes) {
      hip_check(hipMemGetInfo(&free_b, &total_b), "meminfo");
      waves = (uint32_t)std::min<size_t>(waves, std::max<size_t>(1, (free_b / 4 + ws.scratch.bytes) / a.stride));
    }
    a.ws = static_cast<char *>(ws.scratch.get(a.stride * waves, "angular search scratch"));
    a.next = reinterpret_cast<uint32_t *>(ctl);
    a.n_fail = a.next + kXcd;
    a.fail_flags = a.next + kXcd + 1;
    a.fail_list = d_fail;
    a.stats = reinterpret_cast<unsigned long long *>(ctl + 128);
    for (uint32_t x = 0; x <= kXcd; ++x) a.xbeg[x] = (uint32_t)((uint64_t)n_list * x / kXcd);
    a.progress = progress_room(progress, waves);
    hip_check(hipMemsetAsync(ctl, 0, 64, stream), "memset ctl");
    hip_check(hipEventRecord(ws.e0, stream), "event");
    hipLaunchKernelGGL(k_angular_wave, dim3(waves), dim3(kWave), lds, stream, a);
    hip_check(hipGetLastError(), "k_angular_wave launch");
    hip_check(hipEventRecord(ws.e1, stream), "event");
    uint32_t hctl[64];
    hip_check(hipMemcpyAsync(hctl, ctl, 256, hipMemcpyDeviceToHost, stream), "copy");
    hip_check(hipStreamSynchronize(stream), "sync");
    float ms = 0.0f;
    hip_check(hipEventElapsedTime(&ms, ws.e0, ws.e1), "elapsed");
    st.kernel_ms += ms;
    st.waves = std::max<uint32_t>(st.waves, waves);
    const uint32_t n_failed = hctl[kXcd];
    thread_lds_searches() += n_list - n_failed;
    std::vector<uint2> left(n_failed);
    if (n_failed) {
      std::vector<uint32_t> fl(n_failed);
      hip_check(hipMemcpy(fl.data(), d_fail, 4ull * n_failed, hipMemcpyDeviceToHost), "copy");
      for (uint32_t i = 0; i < n_failed; ++i) left[i] = items.empty() ? make_uint2(0u, fl[i]) : items[fl[i]];
    }
    items.swap(left);
    n_list = n_failed;
    unsigned long long stv[4];
    std::memcpy(stv, hctl + 32, 32);
    st.retries += n_failed;
    // (no second try where a source may settle as many states as there can be)
    if (tier == 1 || n_failed == 0 || cap || a.S == kMaxStates) {
      st.nodes_reached += stv[0];
      st.edges_scanned += stv[1];
      st.within_sum += stv[2];
      break;
    }
    // (a few searched twice cost less than room for them in every wave)
    if ((uint64_t)n_failed * 32 > c.n)
      for (const uint32_t i : c.specs) {
        const uint32_t n = specs[i].g->n;
        AngWaveGraph::Reach &r = specs[i].de->ang_wave->reach[specs[i].cs.maxsec];
        r.nodes = std::min(n, r.nodes + r.nodes / 4 + 1);
        for (uint32_t ps = kPage; ps < 10; ++ps) r.pages[ps] = std::min((n >> ps) + 1, r.pages[ps] + r.pages[ps] / 4 + 1);
      }
    // the rest once more with as much room as one workgroup per CU has
    double wider = room;
    WaveArgs wide = a;
    uint32_t wide_lds = lds;
    for (double f = room * 1.25; f < 40.0; f *= 1.2) {
      WaveArgs b = a;
      uint32_t bl = 0;
      if (!wave_layout(b, c.N, c.nodes, c.pages, f, 0, true, &bl)) break;
      wide = b;
      wide_lds = bl;
      wider = f;
      // the fewer are left, the more room each can have
      if (cus * (kLdsMax / bl) < n_failed) break;
    }
    if (wider == room) {
      st.nodes_reached += stv[0];
      st.edges_scanned += stv[1];
      st.within_sum += stv[2];
      break;
    }
    a = wide;
    lds = wide_lds;
  }
  for (const uint32_t i : c.specs) {
    const WaveJob &j = jobs[i];
    const size_t n = (size_t)4 * j.T * j.N;
    hipLaunchKernelGGL(k_wave_rows, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, stream, specs[i].d_acc, j.acc,
                       j.orig, j.N, j.T, specs[i].tstride ? specs[i].tstride : specs[i].cs.T);
  }
  hip_check(hipGetLastError(), "k_wave_rows launch");
  // the staging belongs to the next launch, or the next call once the lock is released
  hip_check(hipStreamSynchronize(stream), "sync");
  rest->insert(rest->end(), items.begin(), items.end());
}

}  // namespace

bool launch_simplest_wave(const std::vector<AngSpec> &specs, const std::vector<uint2> *explicit_items, uint32_t n_implicit,
                          hipStream_t stream, cs_stats &st, uint32_t *progress, std::vector<uint2> *rest) {
  const int dev = specs[0].dg->device;
  // (also guards what the device's graphs keep for this search: a served slice
  // comes without the graph's own lock)
  WaveWorkspace &ws = wave_ws(dev);
  std::lock_guard<std::mutex> lk(ws.mu);
  int n_cu = 0;
  hip_check(hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev), "attribute");
  const uint32_t cap = default_tuning().cap, cus = (uint32_t)n_cu;
  std::vector<uint32_t> count(specs.size(), 0), lanes;
  if (explicit_items)
    for (const uint2 &x : *explicit_items) ++count[x.x];
  else
    count[0] = n_implicit;
  std::vector<WaveClass> cls = wave_plan(specs, count, cap, cus, &lanes);
  if (cls.empty()) return false;
  auto of = [&](const std::vector<uint32_t> &which) {  // the items of some requests, in the caller's order
    std::vector<uint8_t> in(specs.size(), 0);
    for (const uint32_t i : which) in[i] = 1;
    std::vector<uint2> out;
    for (const uint2 &x : *explicit_items)
      if (in[x.x]) out.push_back(x);
    return out;
  };
  if (explicit_items && !lanes.empty()) *rest = of(lanes);
  for (WaveClass &c : cls)
    run_class(ws, c, specs, explicit_items ? of(c.specs) : std::vector<uint2>(), cap, cus, stream, st, progress, rest);
  return true;
}

}  // namespace cs
