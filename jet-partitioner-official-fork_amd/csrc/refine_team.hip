// Whole-level Jet refinement by a team of workgroups on one XCD, for levels of
// up to TEAM_MAX_N vertices (reference: jet_refine, src/jet_refiner.hpp:
// 1050-1142, and every step it calls).
//
// What bounds these levels is latency, not bytes: a step is a chain of
// dependent loads that finishes in a microsecond or two, and the multi-kernel
// path pays a kernel boundary (2.6 us, after which L2 is cold) for each of an
// iteration's four to nine kernels and a host round trip for the controller.
// Here one launch runs the level: it builds the connectivity tables, iterates
// and keeps the controller (step choice, best state, counters, temperatures),
// with the team's barriers (team_dev.h) between the steps.
//
// Vertices are owned by workgroups (8 to 64 consecutive ones in turn). A workgroup
// selects among its vertices, keeps its candidates and moves in LDS lists, and
// is the only one that writes its vertices' part, destination and cached
// values, except that any workgroup may clear a cached destination and update
// a connectivity table. The steps compute what the multi-kernel path computes,
// with the same canonical schedule; positions inside a minibucket are counted
// directly or scanned over the chunks, instead of by sorting.
#include "refine_team.h"

#include <algorithm>
#include <mutex>

#include "conn_table.h"
#include "team_dev.h"
#include "wave.h"

namespace jet {

// 512 threads let two workgroups share a CU but take 10-20% longer on levels
// of more than 10,000 vertices (mesh of 65,536: 30 against 22 us an iteration).
constexpr int TM_BLOCK = 1024;
constexpr int TM_WAVES = TM_BLOCK / WAVE;
constexpr int32_t TM_LANES = 16;             // lanes that build a row of at most TM_SMALL edges
constexpr int32_t TM_SMALL = 64;
constexpr int32_t TM_TABLE = 256;            // table slots of a wave: WAVE / TM_LANES * TM_SMALL, and TEAM_MAX_K
static_assert(TM_TABLE >= TEAM_MAX_K && TM_TABLE >= WAVE / TM_LANES * TM_SMALL, "a wave's table");
constexpr int TM_REDRAW_LDS = 1024;
// Ranked members are compared with each other up to this many (R * R / 64
// wave steps over the team); above, when they are in few buckets (isolated
// vertices share one), positions come from per-chunk sums of each bucket.
// R-MAT level of 6,172 vertices (k = 4): 413 us an iteration with comparisons
// only.
constexpr int32_t TM_RANK_DIRECT = 1024;
constexpr int32_t TM_RANK_BUCKETS = 64;

namespace {

struct TeamShared {
    int64_t sizes[TEAM_MAX_K];
    int64_t delta[TEAM_MAX_K];   // the step's part-size changes
    int64_t adjust[TEAM_MAX_K];  // strong: eviction adjustments
    int64_t evict_start[TEAM_MAX_K + 1];
    part_t undersized[TEAM_MAX_K];
    int64_t red[TM_WAVES + 1];
    int64_t bscore[256];
    int32_t bw[256];
    vid_t bv[256];
    int32_t used[TM_WAVES * 4];
    int32_t rbucket[TM_RANK_BUCKETS];
    int32_t cpre[TEAM_MAX_N / WAVE];
    int32_t cnt[6];  // [0] small candidates, [1] big candidates, [2] small moves, [3] big moves, [4] ranked
    int32_t base;
    int32_t nunder;
    int32_t go, size, me;
    int32_t take;
    int32_t done;
    int64_t counter;
    int64_t cc;
    LevelState S;
};

__device__ inline int2 ldr_slot(const int2* p) {
    const uint64_t x = ldr64(reinterpret_cast<const uint64_t*>(p));
    return make_int2((int32_t)(uint32_t)x, (int32_t)(uint32_t)(x >> 32));
}

// for_slots with loads that see the other workgroups' updates
template <class F>
__device__ inline void for_slots_rx(const int2* tab, int32_t sz, F&& f) {
    for (int32_t s0 = 0; s0 < sz; s0 += 4) {
        int2 e[4];
#pragma unroll
        for (int u = 0; u < 4; u++) e[u] = s0 + u < sz ? ldr_slot(&tab[s0 + u]) : make_int2(NULL_PART, 0);
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (s0 + u < sz) f(e[u]);
    }
}

// Appends to an LDS list of TEAM_OWN items: small items from the front, big
// ones from the back.
__device__ inline void own_push(vid_t* list, int32_t* cnt_small, int32_t* cnt_big, bool pred, bool big, vid_t v) {
    const int32_t a = wave_append(cnt_small, pred && !big);
    const int32_t b = wave_append(cnt_big, pred && big);
    if (a >= 0) list[a] = v;
    if (b >= 0) list[TEAM_OWN - 1 - b] = v;
}

// Runs item(v, sub, lanes) over the workgroup's listed items: G lanes for a
// small one, a wave for a big one.
template <class F>
__device__ inline void own_items(const vid_t* list, int32_t ns, int32_t nb, int G, F&& item) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int gsub = threadIdx.x & (G - 1);
    for (int32_t x = threadIdx.x / G; x < ns; x += TM_BLOCK / G) item(list[x], gsub, G);
    for (int32_t x = threadIdx.x / WAVE; x < nb; x += TM_WAVES) item(list[TEAM_OWN - 1 - x], lane, WAVE);
}

__device__ inline int64_t lanes_sum(int64_t v, int G) {
    for (int o = 1; o < G; o <<= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)(uint64_t)v, o, WAVE);
        const uint32_t hi = __shfl_xor((uint32_t)((uint64_t)v >> 32), o, WAVE);
        v += (int64_t)(((uint64_t)hi << 32) | lo);
    }
    return v;
}

// Inserts part p with weight w into an LDS table of cap slots (cap == k:
// direct, else probing from p % cap); counts newly used slots.
__device__ inline void tm_table_add(int2* T, int32_t cap, int32_t k, part_t p, int32_t w, int32_t* used) {
    int32_t po = p % cap;
    if (cap == k) {
        if (T[po].x == NULL_PART && atomicCAS(&T[po].x, NULL_PART, p) == NULL_PART) atomicAdd(used, 1);
    } else {
        for (int32_t guard = 0; guard <= cap; guard++) {
            const int32_t px = T[po].x;
            if (px == p) break;
            if (px == NULL_PART) {
                const int32_t old = atomicCAS(&T[po].x, NULL_PART, p);
                if (old == NULL_PART) {
                    atomicAdd(used, 1);
                    break;
                }
                if (old == p) break;
            }
            po = po + 1 == cap ? 0 : po + 1;
        }
    }
    atomicAdd(&T[po].y, w);
}

// One row's table by `lanes` lanes (all of a wave, or an aligned group of 16
// in lockstep): hashed in T, shrunk into T2 when that pays, and written out
// (jet_refiner.hpp:958-1048).
__device__ inline void tm_build_row(const TeamParams& P, const part_t* part, vid_t i, eoff_t rs, int32_t deg, int sub,
                                    int lanes, int2* T, int2* T2, int32_t* used) {
    const int32_t k = P.k;
    const int32_t cap = deg < k ? deg : k;
    for (int32_t s = sub; s < cap; s += lanes) {
        T[s] = make_int2(NULL_PART, 0);
        T2[s] = make_int2(NULL_PART, 0);
    }
    if (sub == 0) *used = 0;
    wave_sync();
    for (int32_t j = sub; j < deg; j += lanes)
        tm_table_add(T, cap, k, ld_rx(&part[P.g.col[rs + j]]), P.g.ew[rs + j], used);
    wave_sync();
    const int32_t size = shrink_size(*used, cap);
    int2* out = P.conn + rs;
    if (size < cap) {
        for (int32_t s = sub; s < cap; s += lanes) {
            const int2 e = T[s];
            if (e.x == NULL_PART) continue;
            int32_t po = e.x % size;
            for (int32_t guard = 0; guard <= size; guard++) {
                if (T2[po].x == NULL_PART && atomicCAS(&T2[po].x, NULL_PART, e.x) == NULL_PART) {
                    T2[po].y = e.y;
                    break;
                }
                po = po + 1 == size ? 0 : po + 1;
            }
        }
        wave_sync();
    }
    const int2* src = size < cap ? T2 : T;
    for (int32_t s = sub; s < cap; s += lanes) out[s] = src[s];
    if (sub == 0) {
        P.conn_size[i] = size;
        P.dest_cache[i] = NULL_PART;
    }
    wave_sync();
}

// Tables of the workgroup's own rows (marked: only those with a mark, which
// is cleared), from the parts in `part`: 64 vertices at a time, four by each
// wave (16 lanes a row, or one row after another when they are longer).
__device__ inline void tm_build_rows(const TeamParams& P, const part_t* part, bool marked, int2* lds, int32_t* used,
                                     int32_t team, int32_t me) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = threadIdx.x / WAVE;
    const vid_t n = P.g.n;
    const int32_t tcap = TM_TABLE;  // a wave's table: 4 of TM_SMALL slots or one of k
    int2* T = lds + (size_t)(2 * wv) * tcap;
    int2* T2 = T + tcap;
    const int grp = lane / TM_LANES, sub = lane & (TM_LANES - 1);
    for (int32_t x0 = 4 * wv;; x0 += 4 * TM_WAVES) {
        // own vertices x0 .. x0 + 3; ids grow with x, so the first is the smallest
        if (own_vertex(x0, P.own, team, me) >= n) break;
        const int64_t i64 = own_vertex(x0 + grp, P.own, team, me);
        const vid_t i = (vid_t)i64;
        const bool in = i64 < n;
        const eoff_t rs = in ? P.g.rowptr[i] : 0;
        const int32_t deg = in ? (int32_t)(P.g.rowptr[i + 1] - rs) : 0;
        bool want = in;
        if (marked) {
            want = in && ld_rx(&P.mark[i]) != 0;
            if (want && sub == 0) P.mark[i] = 0;
        }
        if (want && deg <= TM_SMALL)
            tm_build_row(P, part, i, rs, deg, sub, TM_LANES, T + grp * TM_SMALL, T2 + grp * TM_SMALL,
                         &used[wv * 4 + grp]);
        uint64_t big = __ballot(want && deg > TM_SMALL && sub == 0);
        while (big) {
            const int b = __ffsll((unsigned long long)big) - 1;
            big &= big - 1;
            const eoff_t rrs = (eoff_t)__shfl((int64_t)rs, b, WAVE);
            const int32_t rdeg = __shfl(deg, b, WAVE);
            const vid_t ri = __shfl(i, b, WAVE);
            tm_build_row(P, part, ri, rrs, rdeg, lane, WAVE, T, T2, &used[wv * 4]);
        }
    }
}

// First index in [lo, hi) whose evict_start exceeds s (hi when none).
__device__ inline int32_t tm_walk(const int64_t* es, int32_t lo, int32_t hi, int64_t s) {
    while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (es[mid] <= s) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// The next step of the temperature loop of :1095-1134: `for (fr : temps) {
// count = 0; while (count++ <= 11) ... }` as the state (temp_idx, count).
__device__ inline void tm_next_step(TeamShared& L, int32_t ntemps, int32_t iter_cap) {
    LevelState& S = L.S;
    if (S.count > 11) {
        S.temp_idx++;
        S.count = 0;
    }
    L.done = S.temp_idx >= ntemps ? 1 : 0;
    if (!L.done && S.iterations >= iter_cap) {
        // the next launch takes this step again, from this state
        S.status = LEVEL_MORE;
        L.done = 1;
        return;
    }
    S.count++;
    if (!L.done) S.iterations++;
}

__device__ inline void tm_publish(const TeamParams& P, const LevelState& S, int32_t err) {
    P.host_out[0] = S.best_cut;
    P.host_out[1] = S.best_imb;
    P.host_out[2] = S.curr_cut;
    P.host_out[3] = S.curr_imb;
    P.host_out[4] = (int64_t)S.lp_iterations << 32 | (uint32_t)S.iterations;
    P.host_out[5] = (int64_t)S.balance_counter << 32 | (uint32_t)err;
    P.host_out[6] = (int64_t)S.count << 48 | (int64_t)S.temp_idx << 32 | S.changed << 16 | S.status;
    __threadfence_system();
    P.host_out[TEAM_OUT_WORDS] = P.seq;  // the host waits for this word
    __threadfence_system();
}

}  // namespace

__global__ void __launch_bounds__(256) k_team_prep(RefineCtl* ctl, int32_t* buckets, int32_t nb, int64_t* sizes,
                                                  const int64_t* best_sizes, int32_t k, int32_t resume) {
    const int32_t t = blockIdx.x * 256 + threadIdx.x;
    constexpr int32_t W = sizeof(RefineCtl) / 4;
    if (t < W) reinterpret_cast<int32_t*>(ctl)[t] = 0;
    for (int32_t x = t; x < nb; x += gridDim.x * 256) buckets[x] = 0;
    if (!resume)
        for (int32_t x = t; x < k; x += gridDim.x * 256) sizes[x] = best_sizes[x];
}

__global__ void __launch_bounds__(TM_BLOCK) k_refine_team(TeamParams P) {
    extern __shared__ __align__(16) int32_t dyn[];  // bucket sums, then their scan; or the build's tables
    __shared__ TeamShared L;
    __shared__ vid_t cand[TEAM_OWN];   // candidates; rebalancing: ranked members
    __shared__ vid_t moves[TEAM_OWN];
    const DGraph g = P.g;
    const vid_t n = g.n;
    const int32_t k = P.k;
    const int t = threadIdx.x;
    const int lane = t & (WAVE - 1);
    const int wv = t / WAVE;
    RefineCtl* C = P.ctl;
    int32_t* err = &C->err;

    // ------------------------------------------------------------ start-up
    if (t == 0) {
        const int32_t st = team_start(C->team, P.xcd, P.team, ceil_div_dev(n, TEAM_OWN), P.start_spins, L.go, L.size, L.me);
        LevelState S{};
        if (st == TEAM_ABANDON) {
            S.status = LEVEL_ABANDONED;
            tm_publish(P, S, 0);
        }
        S = P.start;
        S.status = LEVEL_DONE;
        L.S = S;
    }
    __syncthreads();
    if (!L.go) return;
    const int32_t T = L.size, me = L.me;
    Team team{&C->team, T, me, 0, &L.go};
    // this workgroup's vertices, a wave 64 of them at a time
    auto for_own = [&](auto&& f) {
        for (int32_t x0 = WAVE * wv;; x0 += WAVE * TM_WAVES) {
            if (own_vertex(x0, P.own, T, me) >= n) break;
            const int64_t i = own_vertex(x0 + lane, P.own, T, me);
            f((vid_t)i, i < n);
        }
    };

    // ------------------------------------------------------------ initial state
    if (!P.resume) {
        int32_t mx = 0;
        for_own([&](vid_t i, bool in) {
            if (!in) return;
            P.part[i] = P.best_part[i];
            P.lock[i] = 0;
            mx = max(mx, (int32_t)(g.rowptr[i + 1] - g.rowptr[i]));
        });
        if (g.m > TEAM_REGULAR_M) {
            mx = wave_reduce_max(mx);
            if (lane == 0 && mx > 0) atomicMax(&C->max_deg, mx);
            const bool ok = team.sync();
            if (!ok || ld_rx(&C->max_deg) > TEAM_MAX_DEG) {
                if (me == 0 && t == 0) {
                    L.S.status = ok ? LEVEL_IRREGULAR : LEVEL_STALLED;
                    tm_publish(P, L.S, 0);
                }
                return;
            }
        }
    }
    for (int32_t p = t; p < k; p += TM_BLOCK) L.sizes[p] = P.resume ? P.sizes[p] : P.best_sizes[p];
    if (!P.resume) tm_build_rows(P, P.best_part, false, reinterpret_cast<int2*>(dyn), L.used, T, me);
    if (t < 6) L.cnt[t] = 0;
    for (int32_t p = t; p < k; p += TM_BLOCK) L.delta[p] = 0;
    if (t == 0) {
        L.take = 0;
        L.cc = 0;
        tm_next_step(L, P.ntemps, P.iter_cap);
    }
    bool alive = team.sync();
    int b = 0;  // the step's set of sums

    // the controller's state is the same in every workgroup: each takes the
    // same decisions from the team's sums
    while (alive) {
        if (L.take) {  // the previous step's best state (every write of it precedes the barrier)
            for_own([&](vid_t i, bool in) {
                if (in) P.best_part[i] = ld_rx(&P.part[i]);
            });
            if (me == 0)
                for (int32_t p = t; p < k; p += TM_BLOCK) P.best_sizes[p] = L.sizes[p];
        }
        if (L.done) break;
        const double fr = P.temps[L.S.temp_idx];
        const int kind = L.S.curr_imb <= P.imb_max ? 0 : (L.S.balance_counter < 2 ? 1 : 2);
        const int32_t gen = P.gen0 + L.S.iterations;

        if (kind == 0) {
            // ---------------------------------------------------- jet_lp (:211-268)
            for_own([&](vid_t i, bool in) {
                const part_t cached = in ? ld_rx(&P.dest_cache[i]) : NO_MOVE;
                const int32_t lk = in ? ld_rx(&P.lock[i]) : 0;
                part_t best = cached;
                int32_t gain = 0;
                eoff_t r0 = 0, r1 = 0;
                if (in) {
                    r0 = g.rowptr[i];
                    r1 = g.rowptr[i + 1];
                }
                if (cached == NULL_PART) {
                    const part_t p = ld_rx(&P.part[i]);
                    best = NO_MOVE;
                    int32_t b_conn = 0, p_conn = 0;
                    for_slots_rx(P.conn + r0, ld_rx(&P.conn_size[i]), [&](int2 e) {
                        if (e.y > b_conn && e.x != p) {
                            best = e.x;
                            b_conn = e.y;
                        } else if (e.y == b_conn && b_conn > 0 && e.x != p && e.x < best) {
                            best = e.x;
                        } else if (e.y > 0 && e.x == p) {
                            p_conn = e.y;
                        }
                    });
                    if (best != NO_MOVE) {
                        if (b_conn >= p_conn || ((double)(p_conn - b_conn) < floor(fr * (double)p_conn)))
                            gain = b_conn - p_conn;
                        else best = NO_MOVE;
                    }
                    P.gain_p[i] = gain;
                    P.dest_cache[i] = best;
                } else if (cached != NO_MOVE && lk == 0) {
                    gain = ld_rx(&P.gain_p[i]);
                }
                const bool c = in && best != NO_MOVE && lk == 0;
                if (in) P.dest[i] = c ? best : NO_MOVE;
                if (in && !c && lk) P.lock[i] = 0;
                if (c) P.pregain[i] = gain;
                own_push(cand, &L.cnt[0], &L.cnt[1], c, r1 - r0 > P.big_deg, i);
            });
            if (!(alive = team.sync())) break;
            // ---------------------------------------------------- afterburner (:275-320)
            const int32_t ns = L.cnt[0], nb = L.cnt[1];
            auto burn = [&](vid_t i, int sub, int lanes) -> int64_t {
                const part_t p = ld_rx(&P.part[i]), best = ld_rx(&P.dest[i]);
                const int32_t ig = ld_rx(&P.pregain[i]);
                int64_t change = 0;
                const eoff_t re = g.rowptr[i + 1];
                for (eoff_t j = g.rowptr[i] + sub; j < re; j += lanes) {
                    const vid_t v = g.col[j];
                    const int32_t w = g.ew[j];
                    const part_t vd = ld_rx(&P.dest[v]), vq = ld_rx(&P.part[v]);
                    const int32_t vg = ld_rx(&P.pregain[v]);
                    if (vd == NO_MOVE) continue;
                    if (vg > ig || (vg == ig && v < i)) {  // afterburn_edge
                        if (vd == p) change -= w;
                        else if (vd == best) change += w;
                        if (vq == p) change += w;
                        else if (vq == best) change -= w;
                    }
                }
                return change;
            };
            {
                // the whole workgroup takes the same number of rounds, so the
                // group sums and the list appends see every lane
                const int G = P.lanes;
                const int gsub = t & (G - 1);
                const int32_t ngroups = TM_BLOCK / G;
                for (int32_t x0 = 0; x0 < ns; x0 += ngroups) {
                    const int32_t x = x0 + t / G;
                    const bool have = x < ns;
                    const vid_t i = have ? cand[x] : 0;
                    const int64_t change = lanes_sum(have ? burn(i, gsub, G) : 0, G);
                    const bool keep = have && gsub == 0 && (int64_t)ld_rx(&P.pregain[i]) + change >= 0;
                    if (keep) {
                        P.lock[i] = 1;
                        P.stamp[i] = gen;
                    }
                    own_push(moves, &L.cnt[2], &L.cnt[3], keep, false, i);
                }
            }
            for (int32_t x = wv; x < nb; x += TM_WAVES) {
                const vid_t i = cand[TEAM_OWN - 1 - x];
                const int64_t change = wave_reduce_sum(burn(i, lane, WAVE));
                if (lane == 0 && (int64_t)ld_rx(&P.pregain[i]) + change >= 0) {
                    P.lock[i] = 1;
                    P.stamp[i] = gen;
                    moves[TEAM_OWN - 1 - atomicAdd(&L.cnt[3], 1)] = i;
                }
            }
            __syncthreads();
            if (t == 0 && L.cnt[2] + L.cnt[3]) atomicAdd(&C->moves[b], L.cnt[2] + L.cnt[3]);
            if (!(alive = team.sync())) break;
        } else {
            // ---------------------------------------------------- rebalancing
            const bool strong = kind == 2;
            const int64_t max_dest = strong ? P.max_dest_strong : P.max_dest_weak;
            const int64_t smax = P.size_max;
            const int64_t width = (int64_t)MAX_BUCKETS * P.sections;
            const int32_t nbk = strong ? k * (int32_t)width + 1 : P.nbk;
            int32_t* sbk = dyn;
            for (int32_t q = t; q <= nbk; q += TM_BLOCK) sbk[q] = 0;
            if (wv == 0) {
                if (strong) {
                    // the largest receiver capacity (:440-448)
                    int64_t mx = INT64_MIN;
                    for (int32_t p = lane; p < k; p += WAVE) {
                        const int64_t sz = L.sizes[p];
                        if (sz < max_dest && max_dest - sz > mx) mx = max_dest - sz;
                        if (me == 0) P.evict_adjust[p] = 0;
                    }
                    mx = wave_reduce_max(mx);
                    if (lane == 0) L.counter = mx;
                } else {
                    // undersized parts in increasing id (:578-591)
                    int32_t base = 0;
                    for (int32_t p0 = 0; p0 < k; p0 += WAVE) {
                        const int32_t p = p0 + lane;
                        const bool f = p < k && L.sizes[p] < max_dest;
                        const uint64_t mk = __ballot(f);
                        if (f) L.undersized[base + (int32_t)__popcll(mk & ((1ull << lane) - 1ull))] = p;
                        base += (int32_t)__popcll(mk);
                    }
                    if (lane == 0) L.nunder = base;
                }
            }
            __syncthreads();
            const int32_t tu = L.nunder;
            const int64_t max_vwgt = L.counter;
            // select (:592-643 weak, :449-481 strong)
            for_own([&](vid_t i, bool in) {
                if (!in) return;
                const part_t p = ld_rx(&P.part[i]);
                const int64_t sp = L.sizes[p];
                const int64_t w = g.vw[i];
                int32_t bk = -1;
                if (!strong) {
                    part_t d = p;
                    if (sp > smax && (double)w < 1.5 * (double)(sp - P.opt)) {
                        part_t best = p;
                        int32_t gain = 0, p_gain = 0;
                        for_slots_rx(P.conn + g.rowptr[i], ld_rx(&P.conn_size[i]), [&](int2 e) {
                            if (e.x > NULL_PART && L.sizes[e.x] < max_dest) {
                                if (e.y > gain) {
                                    best = e.x;
                                    gain = e.y;
                                } else if (e.y == gain && gain > 0 && e.x < best) {
                                    best = e.x;
                                }
                            }
                            if (e.x == p) p_gain = e.y;
                        });
                        int64_t sv = 0;
                        if (gain > 0) {
                            d = best;
                            sv = (int64_t)gain - p_gain;
                        } else if (tu > 0) {
                            d = L.undersized[(uint32_t)i % (uint32_t)tu];
                            sv = -(int64_t)p_gain;
                        }
                        if (d != p)
                            bk = (MAX_BUCKETS * p + gain_bucket_fast(sv, w)) * P.sections +
                                 (int32_t)((uint32_t)i % (uint32_t)P.sections);
                    }
                    P.dest[i] = d;
                } else {
                    const bool vw_ok = max_vwgt > 0 && w <= 2 * max_vwgt;
                    if (sp > smax && vw_ok && w < 2 * (sp - P.opt)) {
                        uint64_t tk = 0, tg = 0;
                        int64_t p_gain = 0;
                        for_slots_rx(P.conn + g.rowptr[i], ld_rx(&P.conn_size[i]), [&](int2 e) {
                            if (e.x == p) {
                                p_gain = e.y;
                            } else if (e.x > NULL_PART && L.sizes[e.x] < max_dest) {
                                tg += (uint64_t)e.y;
                                tk += 1;
                            }
                        });
                        if (tk == 0) tk = 1;
                        const int64_t gain = (int64_t)(tg / tk) - p_gain;
                        const int64_t vwgt = w < sp - smax ? w : sp - smax;
                        const int32_t gt = gain_bucket_fast(gain, vwgt);
                        if (gt < MAX_BUCKETS)
                            bk = (MAX_BUCKETS * p + gt) * P.sections + (int32_t)((uint32_t)i % (uint32_t)P.sections) +
                                 1;
                    }
                }
                if (bk >= 0) atomicAdd(&sbk[bk], (int32_t)w);
                P.bid[i] = bk;
            });
            __syncthreads();
            for (int32_t q = t; q < nbk; q += TM_BLOCK)
                if (sbk[q]) atomicAdd(&P.buckets[q], sbk[q]);
            if (!(alive = team.sync())) break;
            // sbk = exclusive offsets (get_evictions, :363-384), in every workgroup
            for (int32_t q = t; q < nbk; q += TM_BLOCK) sbk[q] = ld_rx(&P.buckets[q]);
            __syncthreads();
            {
                const int32_t per = (nbk + TM_BLOCK - 1) / TM_BLOCK;
                const int32_t t0 = t * per;
                int64_t sum = 0;
                for (int32_t j = 0; j < per && t0 + j < nbk; j++) sum += sbk[t0 + j];
                int64_t tot;
                int64_t run = block_excl_scan<int64_t, TM_BLOCK>(sum, tot, L.red);
                for (int32_t j = 0; j < per && t0 + j < nbk; j++) {
                    const int32_t v = sbk[t0 + j];
                    sbk[t0 + j] = (int32_t)run;
                    run += v;
                }
                if (t == 0) sbk[nbk] = (int32_t)tot;
                __syncthreads();
            }
            // classification: whole buckets below a part's limit are evicted
            // (weak) or need their members' positions (strong); a weak bucket
            // that straddles the limit of a part it holds members of needs
            // them too, of all its members (bucket 50 of part q shares its
            // index with part q + 1's first gain bucket)
            auto weak_straddle = [&](int32_t bk, int32_t q) -> bool {
                const int64_t base = (int64_t)sbk[bk] - sbk[(int64_t)q * width];
                const int64_t limit = L.sizes[q] - smax;
                return base < limit && base + ((int64_t)sbk[bk + 1] - sbk[bk]) > limit;
            };
            for_own([&](vid_t i, bool in) {
                const int32_t bk = in ? ld_rx(&P.bid[i]) : -1;
                bool ev = false, rank = false, big = false;
                if (bk >= 0) {
                    const part_t p = ld_rx(&P.part[i]);
                    const int64_t base = (int64_t)sbk[bk] - sbk[(int64_t)p * width];
                    const int64_t limit = L.sizes[p] - smax;
                    if (strong) {
                        rank = base < limit;
                    } else {
                        ev = base + ((int64_t)sbk[bk + 1] - sbk[bk]) <= limit;
                        const int32_t q = (int32_t)(bk / width);
                        rank = (q < k && weak_straddle(bk, q)) ||
                               (q >= 1 && (int64_t)bk - (int64_t)q * width < P.sections && weak_straddle(bk, q - 1));
                    }
                    if (ev) {
                        big = g.rowptr[i + 1] - g.rowptr[i] > P.big_deg;
                        P.stamp[i] = gen;
                    }
                }
                own_push(moves, &L.cnt[2], &L.cnt[3], ev, big, i);
                const int32_t r = wave_append(&L.cnt[4], rank);
                if (r >= 0) cand[r] = i;
            });
            __syncthreads();
            // the ranked members of all workgroups, for their positions
            const int32_t lr = L.cnt[4];
            if (t == 0) L.base = lr ? atomicAdd(&C->ranked, lr) : 0;
            __syncthreads();
            for (int32_t x = t; x < lr; x += TM_BLOCK) {
                const vid_t v = cand[x];
                P.rkey[L.base + x] = ((uint64_t)(uint32_t)ld_rx(&P.bid[v]) << 32) | (uint32_t)v;
                P.rweight[L.base + x] = g.vw[v];
            }
            if (!(alive = team.sync())) break;
            // the bucket sums have been read: zero for the next rebalancing step
            for (int32_t q = me * TM_BLOCK + t; q < nbk; q += T * TM_BLOCK) P.buckets[q] = 0;
            // one member's decision from its position (the weight of its
            // bucket's members of smaller id): 0 kept, 1 evicted, 2 evicted
            // with a long row
            auto decide = [&](vid_t v, int32_t bk, int64_t pos) -> int {
                const part_t p = ld_rx(&P.part[v]);
                const int64_t w = g.vw[v];
                const int64_t base = (int64_t)sbk[bk] - sbk[(int64_t)p * width];
                const int64_t limit = L.sizes[p] - smax;
                // a weak member decides here only when its own part's limit
                // straddles the bucket
                if ((!strong && !weak_straddle(bk, p)) || base + pos >= limit) return 0;
                if (strong) {
                    if (base + pos + w >= limit) P.evict_adjust[p] = base + pos + w;
                    P.score[v] = (int64_t)sbk[bk] + pos;
                }
                P.stamp[v] = gen;
                return g.rowptr[v + 1] - g.rowptr[v] > P.big_deg ? 2 : 1;
            };
            const int32_t R = ld_rx(&C->ranked);
            const int32_t nchunks = (n + WAVE - 1) / WAVE;
            int32_t S = 0;
            if (R > TM_RANK_DIRECT && P.own == WAVE) {
                // the buckets with ranked members, the same list in every workgroup
                auto ranked_bucket = [&](int32_t q) -> bool {
                    if (q >= nbk || sbk[q + 1] == sbk[q]) return false;
                    if (strong) {
                        const int32_t p = (int32_t)((q - 1) / width);
                        return q > 0 && (int64_t)sbk[q] - sbk[(int64_t)p * width] < L.sizes[p] - smax;
                    }
                    const int32_t p = (int32_t)(q / width);
                    return (p < k && weak_straddle(q, p)) ||
                           (p >= 1 && (int64_t)q - (int64_t)p * width < P.sections && weak_straddle(q, p - 1));
                };
                for (int32_t q0 = 0; q0 < nbk && S <= TM_RANK_BUCKETS; q0 += TM_BLOCK) {
                    const int64_t f = ranked_bucket(q0 + t) ? 1 : 0;
                    int64_t tot;
                    const int64_t at = S + block_excl_scan<int64_t, TM_BLOCK>(f, tot, L.red);
                    if (f && at < TM_RANK_BUCKETS) L.rbucket[at] = q0 + t;
                    S += (int32_t)tot;
                }
                __syncthreads();
            }
            if (S > 0 && S <= TM_RANK_BUCKETS) {
                // many members in few buckets: the weight of each bucket in every
                // chunk of 64 vertices, scanned over the chunks
                int32_t* csum = reinterpret_cast<int32_t*>(P.rkey);  // the list is not read
                for_own([&](vid_t i, bool in) {
                    const int32_t bk = in ? ld_rx(&P.bid[i]) : -1;
                    const int32_t w = bk >= 0 ? g.vw[i] : 0;
                    const int32_t c = i / WAVE;
                    for (int32_t s = 0; s < S; s++) {
                        const int32_t q = L.rbucket[s];
                        if (__ballot(bk == q) == 0) {
                            if (lane == 0) csum[(int64_t)s * nchunks + c] = 0;
                            continue;
                        }
                        const int32_t sum = wave_reduce_sum(bk == q ? w : 0);
                        if (lane == 0) csum[(int64_t)s * nchunks + c] = sum;
                    }
                });
                if (!(alive = team.sync())) break;
                for (int32_t s = 0; s < S; s++) {
                    const int32_t q = L.rbucket[s];
                    // nchunks <= TM_BLOCK
                    int64_t tot;
                    const int64_t pre = block_excl_scan<int64_t, TM_BLOCK>(
                        t < nchunks ? ld_rx(&csum[(int64_t)s * nchunks + t]) : 0, tot, L.red);
                    if (t < nchunks) L.cpre[t] = (int32_t)pre;
                    __syncthreads();
                    for_own([&](vid_t i, bool in) {
                        const int32_t bk = in ? ld_rx(&P.bid[i]) : -1;
                        if (__ballot(bk == q) == 0) return;
                        const int32_t w = bk == q ? g.vw[i] : 0;
                        const int32_t inc = wave_incl_scan(w);
                        const int code = bk == q ? decide(i, q, (int64_t)L.cpre[i / WAVE] + inc - w) : 0;
                        own_push(moves, &L.cnt[2], &L.cnt[3], code != 0, code == 2, i);
                    });
                    __syncthreads();
                }
            } else {
                // positions counted directly: a wave per own member against all
                for (int32_t x = wv; x < lr; x += TM_WAVES) {
                    const vid_t v = cand[x];
                    const int32_t bk = ld_rx(&P.bid[v]);
                    const uint64_t key = ((uint64_t)(uint32_t)bk << 32) | (uint32_t)v;
                    const uint64_t first = (uint64_t)(uint32_t)bk << 32;
                    int64_t pos = 0;
                    for (int32_t y0 = 0; y0 < R; y0 += 4 * WAVE) {
                        uint64_t ky[4];
                        int32_t wy[4];
#pragma unroll
                        for (int u = 0; u < 4; u++) {
                            const int32_t y = y0 + u * WAVE + lane;
                            ky[u] = y < R ? ldr64(&P.rkey[y]) : ~0ull;
                            wy[u] = y < R ? ld_rx(&P.rweight[y]) : 0;
                        }
#pragma unroll
                        for (int u = 0; u < 4; u++)
                            if (ky[u] >= first && ky[u] < key) pos += wy[u];
                    }
                    pos = wave_reduce_sum(pos);
                    if (lane == 0) {
                        const int code = decide(v, bk, pos);
                        if (code == 2) moves[TEAM_OWN - 1 - atomicAdd(&L.cnt[3], 1)] = v;
                        else if (code == 1) moves[atomicAdd(&L.cnt[2], 1)] = v;
                    }
                }
            }
            __syncthreads();
            if (t == 0 && L.cnt[2] + L.cnt[3]) atomicAdd(&C->moves[b], L.cnt[2] + L.cnt[3]);
            if (!(alive = team.sync())) break;
            if (strong) {
                // cookie cutter (:491-518): two scans over the parts, in every workgroup
                if (wv == 0) {
                    int64_t run = 0, run2 = 0;
                    for (int32_t p0 = 0; p0 < k; p0 += WAVE) {
                        const int32_t p = p0 + lane;
                        int64_t add = 0, cap = 0;
                        const int64_t begin = (int64_t)MAX_BUCKETS * p * P.sections;
                        if (p < k) {
                            add = ldr64(&P.evict_adjust[p]);
                            if (add == 0) add = (int64_t)sbk[begin + width] - sbk[begin];
                            cap = max_dest > L.sizes[p] ? max_dest - L.sizes[p] : 0;
                        }
                        const int64_t inc = wave_incl_scan(add), inc2 = wave_incl_scan(cap);
                        if (p < k) {
                            L.adjust[p] = (int64_t)sbk[begin] - (run + inc - add);
                            L.evict_start[p + 1] = run2 + inc2;
                        }
                        run += __shfl(inc, WAVE - 1, WAVE);
                        run2 += __shfl(inc2, WAVE - 1, WAVE);
                    }
                    if (lane == 0) {
                        L.evict_start[0] = 0;
                        L.counter = run;
                    }
                }
                __syncthreads();
                // destinations (:519-544): a member takes the chunk that holds at
                // least half of its weight; the others are re-drawn below
                const int32_t ns = L.cnt[2], nb = L.cnt[3];
                for (int32_t x = t; x < ns + nb; x += TM_BLOCK) {
                    const vid_t v = x < ns ? moves[x] : moves[TEAM_OWN - 1 - (x - ns)];
                    const part_t pv = ld_rx(&P.part[v]);
                    const int64_t s = ldr64(&P.score[v]) - L.adjust[pv];
                    const int32_t c = tm_walk(L.evict_start, 0, k + 1, s) - 1;
                    const int64_t w = g.vw[v];
                    part_t d = pv;
                    if (c < k && w / 2 <= L.evict_start[c + 1] - s) {
                        d = c;
                    } else if (c < k) {
                        P.score[v] = s;
                        P.redraw[atomicAdd(&C->redraws, 1)] = v;
                    }
                    P.dest[v] = d;
                }
                if (!(alive = team.sync())) break;
                const int32_t nr = ld_rx(&C->redraws);
                if (nr > 0) {
                    // the re-drawn members in increasing id, one after another, by
                    // the first workgroup (its own LDS lists hold its moves: the
                    // ordered ids go to `cand`, or back to `redraw`)
                    if (me == 0) {
                        const bool in_lds = nr <= TM_REDRAW_LDS;
                        if (in_lds) {
                            // each id's place by counting the smaller ones
                            if (t < nr) cand[TM_REDRAW_LDS + t] = ld_rx(&P.redraw[t]);
                            __syncthreads();
                            if (t < nr) {
                                const vid_t v = cand[TM_REDRAW_LDS + t];
                                int32_t at = 0;
                                for (int32_t q = 0; q < nr; q++) at += cand[TM_REDRAW_LDS + q] < v ? 1 : 0;
                                cand[at] = v;
                            }
                        } else {
                            // marked, then written back in increasing id
                            for (int32_t x = t; x < nr; x += TM_BLOCK) P.mark[ld_rx(&P.redraw[x])] = 1;
                            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                            __syncthreads();
                            int32_t out = 0;
                            for (vid_t v0 = 0; v0 < n; v0 += TM_BLOCK) {
                                const vid_t v = v0 + t;
                                const int64_t f = v < n && ld_rx(&P.mark[v]) != 0 ? 1 : 0;
                                int64_t tot;
                                const int64_t at = block_excl_scan<int64_t, TM_BLOCK>(f, tot, L.red);
                                if (f) {
                                    P.redraw[out + at] = v;
                                    P.mark[v] = 0;
                                }
                                out += (int32_t)tot;
                            }
                            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                        }
                        __syncthreads();
                        int64_t counter = L.counter;  // carried by thread 0
                        for (int32_t x0 = 0; x0 < nr; x0 += 256) {
                            const int32_t nx = min(256, nr - x0);
                            if (t < nx) {
                                const vid_t v = in_lds ? cand[x0 + t] : ld_rx(&P.redraw[x0 + t]);
                                L.bv[t] = v;
                                L.bscore[t] = ldr64(&P.score[v]);
                                L.bw[t] = g.vw[v];
                            }
                            __syncthreads();
                            if (t == 0) {
                                for (int32_t x = 0; x < nx; x++) {
                                    const int64_t w = L.bw[x];
                                    int64_t s = L.bscore[x];
                                    int32_t p = 0;
                                    // every pass with p < k re-draws (s grows) or stops,
                                    // so at most k + 1 passes reach a chunk past the last
                                    for (int32_t guard = 0; p < k; guard++) {
                                        if (guard > 2 * k + 2) {
                                            atomicOr(err, 8);
                                            break;
                                        }
                                        p = tm_walk(L.evict_start, p, k + 1, s) - 1;
                                        if (p < k && w / 2 <= L.evict_start[p + 1] - s) {
                                            P.dest[L.bv[x]] = p;  // else it keeps its part, written above
                                            break;
                                        } else if (p < k) {
                                            s = counter;
                                            counter += w;
                                        }
                                    }
                                }
                            }
                            __syncthreads();
                        }
                    }
                    if (!(alive = team.sync())) break;
                }
            }
        }

        // -------------------------------------------------------- perform_moves (:905-955)
        const int32_t ms = L.cnt[2], mb = L.cnt[3];
        const bool rebuild = ld_rx(&C->moves[b]) > n / 10;  // update_large (:933)
        // part sizes, cached destinations, the whole cut change (from the parts
        // before and after the step; a neighbour moves when it is stamped) and
        // update_small's subtractions, or the rows to rebuild marked
        int64_t cc = 0;
        own_items(moves, ms, mb, P.lanes, [&](vid_t v, int sub, int lanes) {
            const part_t pold = ld_rx(&P.part[v]), pnew = ld_rx(&P.dest[v]);
            const eoff_t rs = g.rowptr[v], re = g.rowptr[v + 1];
            if (sub == 0) {
                P.dest_cache[v] = NULL_PART;
                const unsigned long long w = (unsigned long long)g.vw[v];
                atomicAdd((unsigned long long*)&L.delta[pold], (unsigned long long)(-(long long)w));
                atomicAdd((unsigned long long*)&L.delta[pnew], w);
            }
            for (eoff_t j = rs + sub; j < re; j += lanes) {
                const vid_t u = g.col[j];
                const int32_t w = g.ew[j];
                const part_t pu = ld_rx(&P.part[u]), du = ld_rx(&P.dest[u]);
                const bool su = ld_rx(&P.stamp[u]) == gen;
                const int32_t cs = ld_rx(&P.conn_size[u]);
                const eoff_t co = g.rowptr[u];
                const part_t nu = su ? du : pu;
                cc += (int64_t)w *
                      ((pu == pnew ? 1 : 0) - (pu == pold ? 1 : 0) + (nu == pnew ? 1 : 0) - (nu == pold ? 1 : 0));
                if (rebuild) P.mark[u] = 1;
                else conn_sub(P.conn + co, cs, pold, w, k, err);
            }
        });
        cc = wave_reduce_sum(cc);
        if (lane == 0 && cc) atomicAdd((unsigned long long*)&L.cc, (unsigned long long)cc);
        __syncthreads();
        if (t == 0 && L.cc) atomicAdd((unsigned long long*)&C->cut[b], (unsigned long long)L.cc);
        for (int32_t p = t; p < k; p += TM_BLOCK)
            if (L.delta[p]) atomicAdd((unsigned long long*)&P.sizes[p], (unsigned long long)L.delta[p]);
        if (!(alive = team.sync())) break;
        // the new parts and update_small's additions
        own_items(moves, ms, mb, P.lanes, [&](vid_t v, int sub, int lanes) {
            const part_t pnew = ld_rx(&P.dest[v]);
            if (sub == 0) P.part[v] = pnew;
            if (rebuild) return;
            const eoff_t rs = g.rowptr[v], re = g.rowptr[v + 1];
            for (eoff_t j = rs + sub; j < re; j += lanes) {
                const vid_t u = g.col[j];
                const int32_t w = g.ew[j];
                const eoff_t co = g.rowptr[u];
                const int64_t du = g.rowptr[u + 1] - co;
                P.dest_cache[u] = NULL_PART;
                conn_add(P.conn + co, &P.conn_size[u], (int32_t)(du < k ? du : k), pnew, w, err);
            }
        });
        // the step's results (complete since the barrier) and the controller's
        // decisions (best state: :1117-1132), by the last wave, which has the
        // fewest moves
        if (wv == TM_WAVES - 1) {
            int64_t mx = INT64_MIN;
            for (int32_t p = lane; p < k; p += WAVE) {
                const int64_t sz = ldr64(&P.sizes[p]);
                L.sizes[p] = sz;
                L.delta[p] = 0;
                mx = sz > mx ? sz : mx;
            }
            const int64_t change = ldr64(&C->cut[b]);
            mx = wave_reduce_max(mx);
            if (lane < 6) L.cnt[lane] = 0;
            if (lane == 0) {
                if (me == 0) {  // the other set of sums, and the lists' counts, for the next step
                    C->moves[b ^ 1] = 0;
                    C->cut[b ^ 1] = 0;
                    C->ranked = 0;
                    C->redraws = 0;
                }
                L.cc = 0;
                LevelState& S = L.S;
                S.curr_cut -= change;
                S.curr_imb = mx > P.opt ? mx - P.opt : 0;
                if (kind == 0) {
                    S.balance_counter = 0;
                    S.lp_iterations++;
                } else {
                    S.balance_counter++;
                }
                int take = 0;
                if (S.best_imb > P.imb_max && S.curr_imb < S.best_imb) {
                    take = 1;
                    S.count = 0;
                } else if (S.curr_cut < S.best_cut && (S.curr_imb <= P.imb_max || S.curr_imb <= S.best_imb)) {
                    if ((double)S.curr_cut < P.tol * (double)S.best_cut) S.count = 0;
                    take = 2;
                }
                if (take) {
                    S.best_cut = S.curr_cut;
                    S.best_imb = S.curr_imb;
                    S.changed = 1;
                }
                L.take = take;
                tm_next_step(L, P.ntemps, P.iter_cap);
            }
        }
        if (!(alive = team.sync())) break;
        if (rebuild) {
            tm_build_rows(P, P.part, true, reinterpret_cast<int2*>(dyn), L.used, T, me);
            if (!(alive = team.sync())) break;
        }
        b ^= 1;
    }
    __syncthreads();
    if (me == 0 && t == 0) {
        if (!alive || ld_rx(&C->team.fail)) L.S.status = LEVEL_STALLED;
        tm_publish(P, L.S, ld_rx(err));
    }
}

// ---------------------------------------------------------------- host side
// Levels with more edges leave more work than one XCD's 32 CUs do in the time
// that the whole GPU's launches cost. Measured, microseconds per iteration,
// team against multi-kernel path: 2-D mesh (k = 8) of 65,536 vertices and
// 391,170 edges 22 / 31, of 2,105 vertices 18 / 39; 3-D stencil levels (k =
// 64) of 10,759 vertices and 162,232 edges 32 / 40, of 46,131 and 685,786 44 /
// 43; (k = 2) of 40,627 and 567,136 24 / 33. Long rows cost more, because the
// updates of all their neighbours meet on their tables: over 2,131 levels of
// R-MAT graphs the team is ahead up to 100,000 edges (sum 0.984 / 1.407 s;
// with 50,000-100,000 edges 0.078 / 0.091 s) and behind above (100,000-200,000
// 0.104 / 0.076 s, 200,000-400,000 0.207 / 0.096 s), so above that it takes
// only levels without rows of more than TEAM_MAX_DEG edges, which the kernel
// finds out before it changes anything.
static bool team_pays(int64_t n, int64_t m) { return m <= 400000 || (m <= 600000 && m <= 16 * n); }

bool team_fits(int64_t n, int64_t m, int32_t k, int64_t nbk, int64_t max_n) {
    return team_pays(n, m) && n >= 1 && n <= std::min<int64_t>(max_n, TEAM_MAX_N) && m <= TEAM_MAX_M && k >= 1 && k <= TEAM_MAX_K &&
           nbk < TEAM_MAX_NBK;
}

// One workgroup needs no barrier beyond its own and no place on an XCD: 14
// against 16.4 us an iteration on levels of 300 to 400 vertices, 18 against 21
// on 490; with 1,433 vertices and 25,000 edges 30.5 against 22.1.
int32_t team_size(int64_t n, int64_t m) {
    if (n <= 700 && m <= 7000) return 1;
    if (n > 8192 || m > 40000) return 32;
    return n > 1024 || m > 10000 ? 16 : 8;
}

// Dynamic LDS: nbk + 1 words of bucket sums, or the build's tables (two per
// wave).
static size_t team_lds(const TeamParams& p) {
    const size_t buckets = sizeof(int32_t) * (size_t)(p.nbk + 2);
    const size_t tables = sizeof(int2) * 2 * TM_WAVES * (size_t)TM_TABLE;
    return std::max(buckets, tables);
}

void launch_refine_team(TeamParams p, hipStream_t s) {
    static std::once_flag once[64];
    static hipError_t rc[64];
    int dev = 0;
    JET_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) throw DeviceError("device index beyond 64");
    std::call_once(once[dev], [&] {
        rc[dev] = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_refine_team),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
    });
    JET_HIP(rc[dev]);
    if (!team_fits(p.g.n, p.g.m, p.k, p.nbk, TEAM_MAX_N) || p.ntemps > TEAM_MAX_TEMPS || p.team < 1 ||
        p.team > TEAM_MAX || (int64_t)p.team * TEAM_OWN < p.g.n)
        throw DeviceError("team refinement: level outside the kernel's limits");
    // chunks of 64 vertices keep a wave's loads together; shorter ones when a
    // level would leave workgroups without vertices
    p.own = 64;
    while (p.own > 8 && ceil_div(p.g.n, p.own) < 4 * (int64_t)p.team) p.own /= 2;
    k_team_prep<<<(int)std::max<int64_t>(1, ceil_div(p.nbk + 1, 1024)), 256, 0, s>>>(p.ctl, p.buckets, p.nbk + 1,
                                                                                    p.sizes, p.best_sizes, p.k, p.resume);
    k_refine_team<<<p.team == 1 ? 1 : 8 * p.team, TM_BLOCK, team_lds(p), s>>>(p);
    JET_LAUNCH_CHECK();
}

}  // namespace jet
