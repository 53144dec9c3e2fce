// Matching of one level (coarsen_match, src/heuristics.hpp:427-671) in one
// launch, by a team of workgroups on one XCD (team_dev.h), for levels of up to
// TEAM_MAX_N vertices.
//
// A matching pass is fourteen kernels of about 2 us each and a host read of the
// work list's length, a 2-hop stage a count, a compaction and a radix sort of
// its candidates (some thirty kernels): on a level of a few thousand vertices
// the launches are nearly all of the time. Here the steps are separated by the
// team's barriers. Workgroups own chunks of 64 consecutive vertices in turn and
// keep their part of the work list in LDS. The schedule is the one of the
// kernels in coarsen.hip: commit rounds in which the smallest active u claiming
// v wins, and 2-hop candidates of equal digest paired two at a time in
// increasing id. The pairs are found without sorting: a hash table groups the
// candidates by digest, every member's rank in its group is counted against
// the group's other members (or, in groups of more than GROUP_DIRECT members,
// scanned over the chunks), and odd ranks join the member before them.
#include "coarsen_team.h"

#include <algorithm>
#include <mutex>

#include "coarsen_rules.h"
#include "prims.h"
#include "team_dev.h"
#include "tuning.h"
#include "wave.h"

namespace jet {

namespace {

constexpr int CM_BLOCK = 1024;
constexpr int CM_WAVES = CM_BLOCK / WAVE;
constexpr int32_t CM_CHUNKS = TEAM_MAX_N / WAVE;
constexpr int32_t GROUP_DIRECT = 512;  // members compared one by one up to this
constexpr int32_t GROUP_MAX_BIG = TEAM_MAX_N / GROUP_DIRECT;

struct MatchCtl {
    TeamCtl team;
    int32_t left[2], pad1[30];  // work-list lengths of alternate passes
    int32_t unmatched[3], total[3], nbig[3], pad2[23];
};

struct MatchParams {
    DGraph g;
    int32_t uniform, two_hop, level;
    uint64_t seed;
    int32_t lanes;    // lanes per vertex of a neighbourhood walk: a power of two up to a wave
    int32_t big_deg;  // longer rows take a whole wave
    int32_t team, xcd, start_spins;
    int32_t hmask;    // hash slots - 1 (a power of two above 2 n)
    vid_t* hn;
    vid_t* vcmap;
    int32_t* claim;
    vid_t* map;
    uint64_t* digest;  // n
    int32_t* slots;    // hmask + 1: candidate + 1, 0 empty
    int32_t* count;    // hmask + 1
    int32_t* offset;   // hmask + 1
    vid_t* members;    // n
    int32_t* big;      // GROUP_MAX_BIG: slots of large groups
    int32_t* csum;     // GROUP_MAX_BIG * chunks: members (or roots) per chunk
    int32_t* clast;    // GROUP_MAX_BIG * chunks: a chunk's last member
    MatchCtl* ctl;
    int64_t* host_out;  // nc (-1 abandoned, -2 failed), then the sequence word
    int64_t seq;
};

struct MatchShared {
    int32_t red[CM_WAVES + 1];
    int32_t pre[CM_CHUNKS];
    int32_t last[CM_CHUNKS];
    int32_t go, size, me;
    int32_t n0, n1;  // lengths of the two work lists
    int32_t add;
};

__device__ inline void cm_publish(const MatchParams& P, int64_t nc) {
    P.host_out[0] = nc;
    __threadfence_system();
    P.host_out[1] = P.seq;  // the host waits for this word
    __threadfence_system();
}

}  // namespace

__global__ void k_match_prep(MatchCtl* ctl) {
    const int32_t t = threadIdx.x;
    for (int32_t x = t; x < (int32_t)(sizeof(MatchCtl) / 4); x += blockDim.x) reinterpret_cast<int32_t*>(ctl)[x] = 0;
}

__global__ void __launch_bounds__(CM_BLOCK) k_match_team(MatchParams P) {
    __shared__ MatchShared L;
    __shared__ vid_t list[2][TEAM_OWN];      // the work list's own vertices, this pass's and the next's
    __shared__ int32_t own_slot[TEAM_OWN];   // 2-hop: an own vertex's hash slot (-1: no candidate)
    __shared__ int32_t own_at[TEAM_OWN];     // and its place in the group, in order of arrival
    const DGraph g = P.g;
    const vid_t n = g.n;
    const int t = threadIdx.x;
    const int lane = t & (WAVE - 1);
    const int wv = t / WAVE;
    MatchCtl* C = P.ctl;
    if (t == 0) {
        const int32_t st = team_start(C->team, P.xcd, P.team, ceil_div_dev(n, TEAM_OWN), P.start_spins, L.go, L.size, L.me);
        if (st == TEAM_ABANDON) cm_publish(P, -1);
        L.n0 = L.n1 = 0;
    }
    __syncthreads();
    if (!L.go) return;
    const int32_t T = L.size, me = L.me;
    Team team{&C->team, T, me, 0, &L.go};
    const int32_t nchunks = (n + WAVE - 1) / WAVE;
    // own vertices: f(x, i, in) with x the vertex's place among the own ones
    auto for_own = [&](auto&& f) {
        for (int32_t x0 = WAVE * wv;; x0 += WAVE * CM_WAVES) {
            if (own_vertex(x0, WAVE, T, me) >= n) break;
            const int64_t i = own_vertex(x0 + lane, WAVE, T, me);
            f(x0 + lane, (vid_t)i, i < n);
        }
    };
    // the eligible neighbour pickMatch takes for u (ORD_MAX: none); a vertex
    // whose mark of this pass is not reset yet (ORD_MAX - 1) counts as unmatched
    auto pick = [&](vid_t u, uint32_t pass, bool initial, int sub, int lanes, int64_t& bw, uint32_t& bh, vid_t& bv) {
        const uint32_t r = (uint32_t)rng(P.seed, (uint32_t)P.level, SITE_PICK, pass, (uint32_t)u);
        const eoff_t re = g.rowptr[u + 1];
        for (eoff_t j = g.rowptr[u] + sub; j < re; j += lanes) {
            const vid_t v = g.col[j];
            const int64_t w = P.uniform ? 0 : (int64_t)g.ew[j];
            if (!initial && ld_rx(&P.vcmap[v]) < ORD_MAX - 1) continue;
            if (w < 0) continue;
            pick_better(bw, bh, bv, w, xorshift32((uint32_t)v + r), v);
        }
    };
    auto reduce_pick = [&](int lanes, int64_t& bw, uint32_t& bh, vid_t& bv) {
        for (int d = 1; d < lanes; d <<= 1) {
            const int64_t ow = __shfl_xor(bw, d, WAVE);
            const uint32_t oh = __shfl_xor(bh, d, WAVE);
            const vid_t ov = __shfl_xor(bv, d, WAVE);
            if (ov != ORD_MAX) pick_better(bw, bh, bv, ow, oh, ov);
        }
    };
    // hn of the listed vertices for which want(u) holds: groups of P.lanes
    // lanes for the short rows, then a wave for each long one
    auto pick_all = [&](const vid_t* lst, int32_t len, uint32_t pass, bool initial, auto&& want) {
        const int G = P.lanes;
        const int sub = t & (G - 1);
        for (int32_t x0 = 0; x0 < len; x0 += CM_BLOCK / G) {
            const int32_t x = x0 + t / G;
            const vid_t u = x < len ? lst[x] : 0;
            const bool go = x < len && want(u) && g.rowptr[u + 1] - g.rowptr[u] <= P.big_deg;
            int64_t bw = 0;
            uint32_t bh = 0;
            vid_t bv = ORD_MAX;
            if (go) pick(u, pass, initial, sub, G, bw, bh, bv);
            reduce_pick(G, bw, bh, bv);
            if (go && sub == 0) P.hn[u] = bv;
        }
        for (int32_t x = wv; x < len; x += CM_WAVES) {
            const vid_t u = lst[x];
            if (g.rowptr[u + 1] - g.rowptr[u] <= P.big_deg || !want(u)) continue;
            int64_t bw = 0;
            uint32_t bh = 0;
            vid_t bv = ORD_MAX;
            pick(u, pass, initial, lane, WAVE, bw, bh, bv);
            reduce_pick(WAVE, bw, bh, bv);
            if (lane == 0) P.hn[u] = bv;
        }
    };

    // ------------------------------------------------------------ first choices
    for_own([&](int32_t x, vid_t i, bool in) {
        if (in) {
            list[0][x] = i;
            P.vcmap[i] = ORD_MAX;
            if (P.uniform) {
                const eoff_t s0 = g.rowptr[i];
                const int64_t deg = g.rowptr[i + 1] - s0;
                const uint64_t r = rng(P.seed, (uint32_t)P.level, SITE_MATCH_INIT, 0, (uint32_t)i);
                P.hn[i] = deg > 0 ? g.col[s0 + (int64_t)(r % (uint64_t)deg)] : ORD_MAX;
            }
        }
        // ids grow with x, so the own vertices fill the list's front
        const uint64_t m = __ballot(in);
        if (lane == 0 && m) atomicAdd(&L.n0, (int32_t)__popcll(m));
    });
    __syncthreads();
    int32_t len = L.n0;
    int cur = 0;
    if (!P.uniform) pick_all(list[0], len, 0, true, [](vid_t) { return true; });
    bool alive = team.sync();

    // ------------------------------------------------------------ matching passes (:427-533)
    for (uint32_t pass = 1; alive; pass++) {
        const vid_t* wl = list[cur];
        for (int r = 0; r < 4; r++) {
            for (int32_t x = t; x < len; x += CM_BLOCK) {
                const vid_t u = wl[x];
                vid_t cu = ld_rx(&P.vcmap[u]);
                const vid_t v = ld_rx(&P.hn[u]);
                if (cu == ORD_MAX - 1) cu = ORD_MAX;
                P.claim[u] = ORD_MAX;
                if (v != ORD_MAX && cu == ORD_MAX) {
                    const bool cond = r > 0 ? (pod_hash_i32(u + r) < pod_hash_i32(v + r)) : (u < v);
                    if (!cond) cu = ORD_MAX - 1;
                }
                P.vcmap[u] = cu;
            }
            if (!(alive = team.sync())) break;
            for (int32_t x = t; x < len; x += CM_BLOCK) {
                const vid_t u = wl[x];
                const vid_t v = ld_rx(&P.hn[u]);
                if (v == ORD_MAX || ld_rx(&P.vcmap[u]) != ORD_MAX) continue;
                if (ld_rx(&P.vcmap[v]) == ORD_MAX - 1) atomicMin(&P.claim[v], u);
            }
            if (!(alive = team.sync())) break;
            for (int32_t x = t; x < len; x += CM_BLOCK) {
                const vid_t u = wl[x];
                const vid_t v = ld_rx(&P.hn[u]);
                if (v == ORD_MAX) continue;
                if (ld_rx(&P.claim[v]) == u) {
                    const vid_t cv = u < v ? u : v;
                    P.vcmap[u] = cv;
                    P.vcmap[v] = cv;
                }
            }
            if (!(alive = team.sync())) break;
        }
        if (!alive) break;
        // marks reset, unmatched vertices whose target is matched pick again,
        // and the vertices still to be matched are listed
        for (int32_t x = t; x < len; x += CM_BLOCK)
            if (ld_rx(&P.vcmap[wl[x]]) == ORD_MAX - 1) P.vcmap[wl[x]] = ORD_MAX;
        pick_all(wl, len, pass, false, [&](vid_t u) {
            if (ld_rx(&P.vcmap[u]) < ORD_MAX - 1) return false;
            const vid_t h = ld_rx(&P.hn[u]);
            return h != ORD_MAX && ld_rx(&P.vcmap[h]) < ORD_MAX - 1;
        });
        if (t == 0) L.n1 = 0;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the new choices are read below
        __syncthreads();
        for (int32_t x0 = 0; x0 < len; x0 += CM_BLOCK) {
            const int32_t x = x0 + t;
            const vid_t u = x < len ? wl[x] : 0;
            const bool keep = x < len && ld_rx(&P.vcmap[u]) >= ORD_MAX - 1 && ld_rx(&P.hn[u]) != ORD_MAX;
            const int32_t at = wave_append(&L.n1, keep);
            if (at >= 0) list[cur ^ 1][at] = u;
        }
        __syncthreads();
        len = L.n1;
        cur ^= 1;
        if (t == 0 && len) atomicAdd(&C->left[pass & 1], len);
        if (!(alive = team.sync())) break;
        const int32_t left = ld_rx(&C->left[pass & 1]);
        // the other counter was read a pass ago
        if (me == 0 && t == 0) C->left[(pass & 1) ^ 1] = 0;
        if (left == 0) break;
        if (pass > (uint32_t)n + 8) {
            alive = false;
            break;
        }
    }

    // ------------------------------------------------------------ 2-hop stages (:535-641)
    for (int stage = 0; alive && P.two_hop && stage < 3; stage++) {
        if (t == 0) L.add = 0;
        __syncthreads();
        for_own([&](int32_t, vid_t i, bool in) {
            const uint64_t m = __ballot(in && ld_rx(&P.vcmap[i]) == ORD_MAX);
            if (lane == 0 && m) atomicAdd(&L.add, (int32_t)__popcll(m));
        });
        __syncthreads();
        if (t == 0 && L.add) atomicAdd(&C->unmatched[stage], L.add);
        if (!(alive = team.sync())) break;
        if (!((double)ld_rx(&C->unmatched[stage]) / (double)n > 0.25)) continue;
        for (int32_t x = me * CM_BLOCK + t; x <= P.hmask; x += T * CM_BLOCK) {
            P.slots[x] = 0;
            P.count[x] = 0;
        }
        // candidates: unmatched vertices (leaves first), with their digests:
        // the single neighbour (:551-555); the sum of (y * y + y), y =
        // pod_hash(neighbour) (:580-596); the lowest-degree neighbour, the
        // first heaviest among equals (:611-637)
        for_own([&](int32_t x, vid_t i, bool in) {
            bool c = in && ld_rx(&P.vcmap[i]) == ORD_MAX;
            if (stage == 0) c = c && g.rowptr[i + 1] - g.rowptr[i] == 1;
            own_slot[x] = c ? 0 : -1;
        });
        __syncthreads();
        {
            const int G = P.lanes;
            const int sub = t & (G - 1);
            int32_t own = 0;  // own vertices: those of the chunks me, me + T, ...
            for (int32_t c = me; c < nchunks; c += T) own = (c - me) / T * WAVE + min(WAVE, n - c * WAVE);
            for (int32_t x0 = 0; x0 < own; x0 += CM_BLOCK / G) {
                const int32_t x = x0 + t / G;
                const bool c = x < own && own_slot[x] >= 0;
                const vid_t u = c ? (vid_t)own_vertex(x, WAVE, T, me) : 0;
                const eoff_t rs = c ? g.rowptr[u] : 0, re = c ? g.rowptr[u + 1] : 0;
                if (stage == 0) {
                    if (c && sub == 0) P.digest[u] = (uint64_t)(uint32_t)g.col[rs];
                } else if (stage == 1) {
                    uint64_t h = 0;
                    for (eoff_t j = rs + sub; j < re; j += G) {
                        const uint64_t y = pod_hash_i32(g.col[j]);
                        h += y * y + y;
                    }
                    for (int d = 1; d < G; d <<= 1) h += (uint64_t)__shfl_xor((int64_t)h, d, WAVE);
                    if (c && sub == 0) P.digest[u] = h;
                } else {
                    // least degree, then greatest weight, then the first edge
                    int32_t bd = ORD_MAX, bw = 0;
                    eoff_t bj = -1;
                    for (eoff_t j = rs + sub; j < re; j += G) {
                        const vid_t v = g.col[j];
                        const int32_t vd = (int32_t)(g.rowptr[v + 1] - g.rowptr[v]);
                        const int32_t w = g.ew[j];
                        if (bj < 0 || vd < bd || (vd == bd && w > bw)) {
                            bd = vd;
                            bw = w;
                            bj = j;
                        }
                    }
                    for (int d = 1; d < G; d <<= 1) {
                        const int32_t od = __shfl_xor(bd, d, WAVE), ow = __shfl_xor(bw, d, WAVE);
                        const eoff_t oj = (eoff_t)__shfl_xor((int64_t)bj, d, WAVE);
                        if (oj >= 0 && (bj < 0 || od < bd || (od == bd && (ow > bw || (ow == bw && oj < bj))))) {
                            bd = od;
                            bw = ow;
                            bj = oj;
                        }
                    }
                    if (c && sub == 0) P.digest[u] = bj < 0 ? (uint64_t)(uint32_t)ORD_MAX : (uint64_t)(uint32_t)g.col[bj];
                }
            }
        }
        if (!(alive = team.sync())) break;
        // group by digest: a slot holds its first candidate; equal digests meet
        for_own([&](int32_t x, vid_t i, bool in) {
            if (!in || own_slot[x] < 0) return;
            const uint64_t key = ldr64(&P.digest[i]);
            int32_t h = (int32_t)(mix64(key) & (uint64_t)P.hmask);
            for (;;) {  // at most n of more than 2 n slots are ever taken
                int32_t c = ld_rx(&P.slots[h]);
                if (c == 0) {
                    c = atomicCAS(&P.slots[h], 0, i + 1);
                    if (c == 0) break;
                }
                if (ldr64(&P.digest[c - 1]) == key) break;
                h = (h + 1) & P.hmask;
            }
            own_slot[x] = h;
            own_at[x] = atomicAdd(&P.count[h], 1);
        });
        if (!(alive = team.sync())) break;
        // the first to arrive reserves the group's stretch of the member array
        for_own([&](int32_t x, vid_t, bool in) {
            if (!in || own_slot[x] < 0 || own_at[x] != 0) return;
            const int32_t h = own_slot[x], c = ld_rx(&P.count[h]);
            if (c < 2) return;
            P.offset[h] = atomicAdd(&C->total[stage], c);
            if (c > GROUP_DIRECT) P.big[atomicAdd(&C->nbig[stage], 1)] = h;
        });
        if (!(alive = team.sync())) break;
        const int32_t nbig = ld_rx(&C->nbig[stage]);
        for_own([&](int32_t x, vid_t i, bool in) {
            const int32_t h = in ? own_slot[x] : -1;
            const int32_t c = h >= 0 ? ld_rx(&P.count[h]) : 0;
            if (c >= 2 && c <= GROUP_DIRECT) P.members[ld_rx(&P.offset[h]) + own_at[x]] = i;
            for (int32_t b = 0; b < nbig; b++) {
                const uint64_t m = __ballot(h >= 0 && h == ld_rx(&P.big[b]));
                const int32_t ch = i / WAVE;
                if (lane == 0) {
                    P.csum[(int64_t)b * nchunks + ch] = (int32_t)__popcll(m);
                    P.clast[(int64_t)b * nchunks + ch] = m ? (i & ~(WAVE - 1)) + 63 - __clzll((long long)m) : -1;
                }
            }
        });
        if (!(alive = team.sync())) break;
        // every second member of a group, in increasing id, joins the one before it
        for_own([&](int32_t x, vid_t i, bool in) {
            const int32_t h = in ? own_slot[x] : -1;
            const int32_t c = h >= 0 ? ld_rx(&P.count[h]) : 0;
            if (c < 2 || c > GROUP_DIRECT) return;
            const int32_t off = ld_rx(&P.offset[h]);
            int32_t rank = 0;
            vid_t prev = -1;
            for (int32_t y0 = 0; y0 < c; y0 += 4) {
                vid_t v[4];
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = y0 + q < c ? ld_rx(&P.members[off + y0 + q]) : ORD_MAX;
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (v[q] < i) {
                        rank++;
                        prev = v[q] > prev ? v[q] : prev;
                    }
            }
            if (rank & 1) {
                P.vcmap[i] = prev;
                P.vcmap[prev] = prev;
            }
        });
        for (int32_t b = 0; b < nbig; b++) {
            const int32_t h = ld_rx(&P.big[b]);
            // before each chunk: the group's members, and the last of them
            __syncthreads();
            const int32_t v = t < nchunks ? ld_rx(&P.csum[(int64_t)b * nchunks + t]) : 0;
            int32_t tot;
            const int32_t pre = block_excl_scan<int32_t, CM_BLOCK>(v, tot, L.red);
            if (t < nchunks) {
                L.pre[t] = pre;
                L.last[t] = ld_rx(&P.clast[(int64_t)b * nchunks + t]);
            }
            __syncthreads();
            for_own([&](int32_t x, vid_t i, bool in) {
                const uint64_t m = __ballot(in && own_slot[x] == h);
                if (!((m >> lane) & 1ull)) return;
                const uint64_t below = m & ((1ull << lane) - 1ull);
                const int32_t ch = i / WAVE;
                if (((L.pre[ch] + (int32_t)__popcll(below)) & 1) == 0) return;
                vid_t prev;
                if (below) {
                    prev = (i & ~(WAVE - 1)) + 63 - __clzll((long long)below);
                } else {
                    int32_t q = ch - 1;
                    while (L.last[q] < 0) q--;  // an odd rank: an earlier chunk has a member
                    prev = L.last[q];
                }
                P.vcmap[i] = prev;
                P.vcmap[prev] = prev;
            });
        }
        if (!(alive = team.sync())) break;
    }

    // ------------------------------------------------------------ ids (:147-165, :650-665)
    // roots get dense ids in increasing order; unmatched vertices are roots
    int32_t nc = 0;
    if (alive) {
        for_own([&](int32_t, vid_t i, bool in) {
            vid_t c = in ? ld_rx(&P.vcmap[i]) : -1;
            if (c == ORD_MAX) {
                c = i;
                P.vcmap[i] = i;
            }
            const uint64_t m = __ballot(in && c == i);
            if (lane == 0) P.csum[i / WAVE] = (int32_t)__popcll(m);
        });
        alive = team.sync();
    }
    if (alive) {
        const int32_t v = t < nchunks ? ld_rx(&P.csum[t]) : 0;
        const int32_t pre = block_excl_scan<int32_t, CM_BLOCK>(v, nc, L.red);
        if (t < nchunks) L.pre[t] = pre;
        __syncthreads();
        // claim[] takes the roots' ids
        for_own([&](int32_t, vid_t i, bool in) {
            const bool root = in && ld_rx(&P.vcmap[i]) == i;
            const uint64_t m = __ballot(root);
            if (root) P.claim[i] = L.pre[i / WAVE] + (int32_t)__popcll(m & ((1ull << lane) - 1ull));
        });
        alive = team.sync();
    }
    if (alive)
        for_own([&](int32_t, vid_t i, bool in) {
            if (in) P.map[i] = ld_rx(&P.claim[ld_rx(&P.vcmap[i])]);
        });
    if (me == 0 && t == 0) cm_publish(P, alive && !ld_rx(&C->team.fail) ? nc : -2);
}

// ---------------------------------------------------------------- host side
bool team_match_fits(int64_t n, int64_t m) {
    return n >= 1 && n <= team_max_n() && m <= TEAM_MATCH_M;
}

int32_t coarsen_match_team(const DGraph& g, bool uniform, uint64_t seed, int32_t level, bool two_hop, vid_t* map,
                           Arena& a, hipStream_t s) {
    ArenaScope sc(a);
    const int64_t n = g.n, nchunks = ceil_div(n, (int64_t)WAVE);
    MatchParams P{};
    P.g = g;
    P.uniform = uniform ? 1 : 0;
    P.two_hop = two_hop ? 1 : 0;
    P.level = level;
    P.seed = seed;
    const double avg = n > 0 ? (double)g.m / (double)n : 0.0;
    P.lanes = avg <= 4 ? 4 : avg <= 8 ? 8 : avg <= 16 ? 16 : avg <= 32 ? 32 : 64;
    P.big_deg = 8 * P.lanes;
    P.team = (int32_t)std::max<int64_t>(1, std::min<int64_t>(TEAM_MAX, ceil_div(nchunks, (int64_t)4)));
    int64_t slots = 64;
    while (slots < 2 * n + 1) slots *= 2;
    P.hmask = (int32_t)(slots - 1);
    P.hn = a.alloc<vid_t>(n);
    P.vcmap = a.alloc<vid_t>(n);
    P.claim = a.alloc<int32_t>(n);
    P.map = map;
    P.digest = a.alloc<uint64_t>(n);
    P.slots = a.alloc<int32_t>(slots);
    P.count = a.alloc<int32_t>(slots);
    P.offset = a.alloc<int32_t>(slots);
    P.members = a.alloc<vid_t>(n);
    P.big = a.alloc<int32_t>(GROUP_MAX_BIG);
    P.csum = a.alloc<int32_t>(GROUP_MAX_BIG * nchunks);
    P.clast = a.alloc<int32_t>(GROUP_MAX_BIG * nchunks);
    P.ctl = a.alloc<MatchCtl>(1);
    Mailbox& mb = thread_mailbox();
    P.host_out = mb.dev + 32;
    volatile int64_t* out = mb.host + 32;
    P.seq = ++mb.seq;
    TeamSlot slot(P.team);
    P.xcd = slot.xcd();
    P.start_spins = (int32_t)tuning().team_start_spins;
    k_match_prep<<<1, 256, 0, s>>>(P.ctl);
    k_match_team<<<P.team == 1 ? 1 : 8 * P.team, CM_BLOCK, 0, s>>>(P);
    JET_LAUNCH_CHECK();
    // without a result: no workgroup ran on the wanted XCD
    const int64_t nc = wait_mailbox(&out[1], P.seq, s) ? out[0] : -1;
    if (nc == -2) throw DeviceError("matching made no progress");
    if (nc < 0) team_abandoned();
    return (int32_t)nc;
}

}  // namespace jet
