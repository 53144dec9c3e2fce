// Coarse-graph contraction for gfx950 (reference: src/contract.hpp:347-446).
//
// For a fixed fine->coarse map the coarse adjacency is P^T A P without its
// diagonal, with coarse vertex weights P^T vw. Each coarse row c is built by
// hashing the mapped neighbours of all fine members of c:
//  * rows with at most 128 incident fine edges: one wave per row, open
//    addressing in a per-wave LDS table, ranks by counting;
//  * rows with at most 4096: one workgroup per row, LDS table + bitonic sort;
//  * larger rows (hub aggregates): global spill path, a radix sort of
//    (row, neighbour) keys followed by a reduce-by-key.
// Rows are emitted in increasing neighbour order, which is one of the orders
// the reference's unordered consolidate can produce; weights are integer sums.
#include "contract.h"

#include <algorithm>

#include "contract_dev.h"
#include "contract_team.h"
#include "tuning.h"
#include "prims.h"
#include "wave.h"

namespace jet {

constexpr int32_t T1_MAX = 128;   // hsize bound for the wave tier
constexpr int32_t T1_CAP = 256;   // wave LDS table slots
constexpr int32_t T2_MAX = 4096;  // hsize bound for the workgroup tier
constexpr int32_t T2_CAP = 8192;  // workgroup LDS table slots
// The workgroup tier runs in two sizes, so that its many short rows do not
// hold the long rows' LDS: up to T2S_MAX fine edges a 256-thread workgroup
// with 2048 slots (8 of them fit a CU), above that 1024 threads with 8192
// slots (2 fit). One size of 256 threads and 8192 slots left 8 waves a CU.
constexpr int32_t T2S_MAX = 1024;
constexpr int32_t T2S_CAP = 2048;

__global__ void k_contract_reset(vid_t nc, eoff_t* hsize, wgt_t* cvw, int32_t* moff, int32_t* mfill, int32_t* ucount,
                                 int32_t* cnt) {
    FOR_THREAD(c, (int64_t)nc + 1) {
        hsize[c] = 0;
        moff[c] = 0;
        ucount[c] = 0;
        if (c < nc) {
            cvw[c] = 0;
            mfill[c] = 0;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < 4) cnt[threadIdx.x] = 0;
}

__global__ void k_count(DGraph g, const vid_t* map, eoff_t* hsize, wgt_t* cvw, int32_t* mcount) {
    FOR_THREAD(i, g.n) {
        vid_t c = map[i];
        atomicAdd((unsigned long long*)&hsize[c], (unsigned long long)(g.rowptr[i + 1] - g.rowptr[i]));
        atomicAdd(&cvw[c], g.vw[i]);
        atomicAdd(&mcount[c], 1);
    }
}

__global__ void k_members(vid_t n, const vid_t* map, const int32_t* moff, int32_t* mfill, vid_t* members) {
    FOR_THREAD(i, n) {
        vid_t c = map[i];
        members[moff[c] + atomicAdd(&mfill[c], 1)] = (vid_t)i;
    }
}

__global__ void k_member_degrees(DGraph g, const vid_t* members, int32_t* deg) {
    FOR_THREAD(x, g.n) {
        const vid_t i = members[x];
        deg[x] = (int32_t)(g.rowptr[i + 1] - g.rowptr[i]);
    }
}

__global__ void __launch_bounds__(256)
    k_tiers(vid_t nc, const eoff_t* hoff, vid_t* l1, vid_t* l2, vid_t* l3, vid_t* l4, int32_t* cnt, int32_t t1max,
            int32_t t2max) {
    __shared__ int32_t sh[256 / WAVE + 1];
    FOR_BLOCK_UNIFORM(c, nc) {
        const bool in = c < nc;
        const eoff_t hs = in ? hoff[c + 1] - hoff[c] : 0;
        int32_t a = block_append<256>(&cnt[0], in && hs <= t1max, sh);
        int32_t b = block_append<256>(&cnt[1], in && hs > t1max && hs <= t2max && hs <= T2S_MAX, sh);
        int32_t e = block_append<256>(&cnt[3], in && hs > t1max && hs <= t2max && hs > T2S_MAX, sh);
        int32_t d = block_append<256>(&cnt[2], in && hs > t2max, sh);
        if (a >= 0) l1[a] = (vid_t)c;
        if (b >= 0) l2[b] = (vid_t)c;
        if (d >= 0) l3[d] = (vid_t)c;
        if (e >= 0) l4[e] = (vid_t)c;
    }
}

constexpr int T1_WAVES = 4;

__global__ void __launch_bounds__(T1_WAVES* WAVE)
    k_dedupe_wave(DGraph g, const vid_t* map, const vid_t* members, const int32_t* moff, const eoff_t* hoff,
                  const vid_t* list, const int32_t* cnt, vid_t* tkey, wgt_t* tval, int32_t* ucount) {
    __shared__ int32_t keys[T1_WAVES][T1_CAP];
    __shared__ int32_t vals[T1_WAVES][T1_CAP];
    __shared__ int32_t ukeys[T1_WAVES][T1_CAP];
    __shared__ int32_t uvals[T1_WAVES][T1_CAP];
    __shared__ eoff_t s_ex[T1_WAVES][WAVE];
    __shared__ eoff_t s_rs[T1_WAVES][WAVE];
    const int lane = threadIdx.x & (WAVE - 1);
    const int w = threadIdx.x / WAVE;
    const int32_t nrows = cnt[0];
    for (int32_t r = blockIdx.x * T1_WAVES + w; r < nrows; r += gridDim.x * T1_WAVES) {
        vid_t c = list[r];
        eoff_t hs = hoff[c];
        int32_t hsz = (int32_t)(hoff[c + 1] - hs);
        uint32_t cap = 64;
        while ((int32_t)cap < 2 * hsz) cap <<= 1;
        for (uint32_t t = lane; t < cap; t += WAVE) {
            keys[w][t] = EMPTY;
            vals[w][t] = 0;
        }
        wave_sync();
        int32_t* K = keys[w];
        int32_t* V = vals[w];
        auto member = [&](int32_t x) { return members[x]; };
        wave_row_edges(g, member, moff[c], moff[c + 1], s_ex[w], s_rs[w], [&](eoff_t j) {
            vid_t u = map[g.col[j]];
            if (u != c) lds_insert(K, V, cap - 1, u, g.ew[j]);
        });
        wave_sync();
        // compact unique entries (slot order), then rank by counting
        int32_t base = 0;
        for (uint32_t t0 = 0; t0 < cap; t0 += WAVE) {
            uint32_t t = t0 + lane;
            int32_t k = t < cap ? K[t] : EMPTY;
            bool has = k != EMPTY;
            uint64_t bal = __ballot(has);
            int32_t pos = base + (int32_t)__popcll(bal & ((1ull << lane) - 1ull));
            if (has) {
                ukeys[w][pos] = k;
                uvals[w][pos] = V[t];
            }
            base += (int32_t)__popcll(bal);
        }
        wave_sync();
        const int32_t U = base;
        for (int32_t e = lane; e < U; e += WAVE) {
            int32_t k = ukeys[w][e];
            int32_t rank = 0;
            for (int32_t q = 0; q < U; q++) rank += ukeys[w][q] < k ? 1 : 0;
            tkey[hs + rank] = k;
            tval[hs + rank] = uvals[w][e];
        }
        if (lane == 0) ucount[c] = U;
        wave_sync();
    }
}

// One workgroup per row: hash into LDS, compact the unique entries (they fill
// at most half of the table), then bitonic-sort only those. Sorting the whole
// table took four times the exchanges: 7.5 ms a call on R-MAT 22's levels,
// 4.7 with the entries packed and rows in two sizes, 2.6 with the row's edges
// shared equally by the waves. Bound by the insertions' and the sort's LDS
// round trips.
template <int BLOCK, int CAP>
__global__ void __launch_bounds__(BLOCK)
    k_dedupe_block(DGraph g, const vid_t* map, const vid_t* members, const eoff_t* medge, const int32_t* moff,
                   const eoff_t* hoff, const vid_t* list, int32_t nrows, vid_t* tkey, wgt_t* tval, int32_t* ucount) {
    __shared__ int32_t keys[CAP];
    __shared__ int32_t vals[CAP];
    __shared__ int32_t ws[BLOCK / WAVE + 1];
    __shared__ int32_t s_e[BLOCK / WAVE][WAVE];
    __shared__ eoff_t s_rs[BLOCK / WAVE][WAVE];
    constexpr int PER = CAP / BLOCK;
    for (int32_t r = blockIdx.x; r < nrows; r += gridDim.x) {
        vid_t c = list[r];
        eoff_t hs = hoff[c];
        int32_t hsz = (int32_t)(hoff[c + 1] - hs);
        uint32_t cap = 256;
        while ((int32_t)cap < 2 * hsz) cap <<= 1;
        for (uint32_t t = threadIdx.x; t < cap; t += BLOCK) {
            keys[t] = EMPTY;
            vals[t] = 0;
        }
        __syncthreads();
        // an equal share of the row's edges to each wave, whatever members they
        // are of: a member per wave left most waves waiting for the longest
        const int wid = threadIdx.x / WAVE;
        const int32_t share = (hsz + BLOCK / WAVE * WAVE - 1) / (BLOCK / WAVE * WAVE) * WAVE;
        const eoff_t ea = hs + min(hsz, wid * share), eb = hs + min(hsz, (wid + 1) * share);
        wave_edge_range(g, members, medge, moff[c], moff[c + 1], ea, eb, s_e[wid], s_rs[wid], [&](eoff_t j, eoff_t) {
            const vid_t u = map[g.col[j]];
            if (u != c) lds_insert(keys, vals, cap - 1, u, g.ew[j]);
        });
        __syncthreads();
        // the unique entries, packed to the front through registers
        int32_t rk[PER], rv[PER];
        int32_t mine = 0;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const uint32_t t = threadIdx.x + (uint32_t)q * BLOCK;
            rk[q] = t < cap ? keys[t] : EMPTY;
            rv[q] = t < cap ? vals[t] : 0;
            mine += rk[q] != EMPTY ? 1 : 0;
        }
        int32_t U;
        int32_t at = block_excl_scan<int32_t, BLOCK>(mine, U, ws);
        uint32_t scap = 2;
        while ((int32_t)scap < U) scap <<= 1;
#pragma unroll
        for (int q = 0; q < PER; q++)
            if (rk[q] != EMPTY) {
                keys[at] = rk[q];
                vals[at++] = rv[q];
            }
        // scap <= cap: U <= hsz <= cap / 2
        for (uint32_t t = (uint32_t)U + threadIdx.x; t < scap; t += BLOCK) keys[t] = EMPTY;
        // bitonic sort by key as unsigned (EMPTY last)
        for (uint32_t size = 2; size <= scap; size <<= 1) {
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                __syncthreads();
                for (uint32_t t = threadIdx.x; t < scap / 2; t += BLOCK) {
                    uint32_t lo = 2 * t - (t & (stride - 1));
                    uint32_t hi = lo + stride;
                    bool up = (lo & size) == 0;
                    uint32_t a = (uint32_t)keys[lo], b = (uint32_t)keys[hi];
                    if ((a > b) == up) {
                        keys[lo] = (int32_t)b;
                        keys[hi] = (int32_t)a;
                        int32_t tv = vals[lo];
                        vals[lo] = vals[hi];
                        vals[hi] = tv;
                    }
                }
            }
        }
        __syncthreads();
        for (int32_t e = threadIdx.x; e < U; e += BLOCK) {
            tkey[hs + e] = keys[e];
            tval[hs + e] = vals[e];
        }
        if (threadIdx.x == 0) ucount[c] = U;
        __syncthreads();
    }
}

// ---- spill path: (row rank << nbits | neighbour) keys, all ones for the
// diagonal; radix sort, reduce by key
// A wave takes SPILL_CHUNK consecutive places of the concatenated spilled rows,
// whatever rows and members they are of. (A workgroup per row and a wave per
// member left one wave with the longest member: 2.4 ms a call on R-MAT 22's
// levels and 7.5 on the first; now 0.44 and 0.65.)
constexpr int64_t SPILL_CHUNK = 1024;
__global__ void __launch_bounds__(256)
    k_spill_gather(DGraph g, const vid_t* map, const vid_t* members, const eoff_t* medge, const int32_t* moff,
                   const eoff_t* hoff, const vid_t* list, int32_t n3, const eoff_t* soff, eoff_t len, int nbits,
                   uint64_t* skey, uint32_t* sval) {
    __shared__ int32_t s_e[256 / WAVE][WAVE];
    __shared__ eoff_t s_rs[256 / WAVE][WAVE];
    const int wid = threadIdx.x / WAVE;
    const int64_t stride = (int64_t)gridDim.x * (256 / WAVE) * SPILL_CHUNK;
    for (int64_t t0 = ((int64_t)blockIdx.x * (256 / WAVE) + wid) * SPILL_CHUNK; t0 < len; t0 += stride) {
        const int64_t t1 = min((int64_t)len, t0 + SPILL_CHUNK);
        int32_t r = 0, hi = n3 - 1;  // the row that holds place t0
        while (r < hi) {
            const int32_t mid = (r + hi + 1) >> 1;
            if (soff[mid] <= t0) r = mid;
            else hi = mid - 1;
        }
        for (int64_t t = t0; t < t1; r++) {
            const vid_t c = list[r];
            const eoff_t base = soff[r], end = min((eoff_t)t1, soff[r + 1]), h = hoff[c];
            wave_edge_range(g, members, medge, moff[c], moff[c + 1], h + (t - base), h + (end - base), s_e[wid],
                            s_rs[wid], [&](eoff_t j, eoff_t e) {
                                const vid_t u = map[g.col[j]];
                                const eoff_t at = base + (e - h);
                                skey[at] = u == c ? ~0ull : (((uint64_t)r << nbits) | (uint32_t)u);
                                sval[at] = (uint32_t)g.ew[j];
                            });
            t = end;
        }
    }
}

__global__ void k_spill_heads(const uint64_t* skey, int64_t len, int32_t* head) {
    FOR_THREAD(t, len) {
        uint64_t k = skey[t];
        head[t] = (k != ~0ull && (t == 0 || k != skey[t - 1])) ? 1 : 0;
    }
}

// Sums the runs of equal keys. A hub row's runs are long (one entry per fine
// edge between two aggregates), so each wave first sums its stretch of every
// run with a segmented scan and adds once per wave and run; a row's first
// unique entry is found by its neighbour's key instead of a minimum over the
// row. With an atomic per entry, the entries of the few hub rows met on a few
// addresses: 11.1 ms per call on R-MAT 22's levels (spill_write, which
// counted a row's uniques with an atomic each, 10.5 ms); now 0.34 and 0.29.
__global__ void __launch_bounds__(256)
    k_spill_reduce(const uint64_t* skey, const uint32_t* sval, int64_t len, int nbits, const int32_t* uid_ex, int32_t* ukey,
                   wgt_t* uval, int32_t* urow, int32_t* rowfirst) {
    const int lane = threadIdx.x & (WAVE - 1);
    for (int64_t t0 = blockIdx.x * (int64_t)256 + (threadIdx.x - lane); t0 < len; t0 += (int64_t)gridDim.x * 256) {
        const int64_t t = t0 + lane;
        const uint64_t k = t < len ? skey[t] : ~0ull;
        const uint64_t kp = t > 0 && t < len ? skey[t - 1] : ~0ull;
        const uint64_t kn = t + 1 < len ? skey[t + 1] : ~0ull;
        const bool valid = k != ~0ull;
        const bool head = t == 0 || k != kp;
        wgt_t v = valid ? (wgt_t)sval[t] : 0;
        const int32_t uid = valid ? uid_ex[t + 1] - 1 : 0;
        // inclusive sum since the run's first entry in this wave
        const uint64_t starts = __ballot(head || lane == 0);
        const uint64_t upto = lane == WAVE - 1 ? starts : starts & ((2ull << lane) - 1ull);
        const int start = 63 - __clzll((long long)upto);
#pragma unroll
        for (int d = 1; d < WAVE; d <<= 1) {
            const wgt_t o = __shfl_up(v, d, WAVE);
            if (lane - d >= start) v += o;
        }
        const bool last = lane == WAVE - 1 || kn != k;  // of the wave's stretch of the run
        if (valid && last) atomicAdd(&uval[uid], v);
        if (valid && head) {
            const int32_t r = (int32_t)(k >> nbits);
            ukey[uid] = (int32_t)(k & ((1ull << nbits) - 1ull));
            urow[uid] = r;
            if (t == 0 || (int32_t)(kp >> nbits) != r) rowfirst[r] = uid;
        }
    }
}

__global__ void k_spill_write(int32_t U, const int32_t* ukey, const wgt_t* uval, const int32_t* urow,
                              const int32_t* rowfirst, const vid_t* list, const eoff_t* hoff, vid_t* tkey, wgt_t* tval,
                              int32_t* ucount) {
    FOR_THREAD(e, U) {
        int32_t r = urow[e];
        vid_t c = list[r];
        int32_t off = (int32_t)e - rowfirst[r];
        tkey[hoff[c] + off] = ukey[e];
        tval[hoff[c] + off] = uval[e];
        // the row's last unique entry knows its count
        if (e + 1 == U || urow[e + 1] != r) ucount[c] = off + 1;
    }
}

// A search of all rows per entry was 1.43 ms a call on R-MAT 22's levels, of
// a tile's rows in LDS 0.54 (16 bytes per entry at the copy rate: 0.22).
__global__ void __launch_bounds__(256)
    k_consolidate(vid_t nc, int64_t mc, const eoff_t* crow, const eoff_t* hoff, const vid_t* tkey, const wgt_t* tval,
                  vid_t* col, wgt_t* ew) {
    __shared__ EdgeWalkLds walk;
    block_edges<256>(crow, nc, mc, walk, [&](vid_t r, eoff_t e) {
        const eoff_t src = hoff[r] + (e - crow[r]);
        col[e] = tkey[src];
        ew[e] = tval[src];
    });
}

__global__ void k_spill_sizes(const vid_t* list, int32_t n3, const eoff_t* hoff, eoff_t* ssz) {
    FOR_THREAD(r, n3) {
        vid_t c = list[r];
        ssz[r] = hoff[c + 1] - hoff[c];
    }
}

void contract(const DGraph& g, const vid_t* map, vid_t nc, Arena& persist, Arena& a, hipStream_t s, Level& out) {
    if (team_contract_fits(g.n, g.m, nc) && contract_team(g, map, nc, persist, a, s, out)) return;
    out.n = nc;
    out.rowptr = persist.alloc<eoff_t>((int64_t)nc + 1);
    out.vw = persist.alloc<wgt_t>(nc);
    ArenaScope sc(a);
    eoff_t* hoff = a.alloc<eoff_t>((int64_t)nc + 1);
    int32_t* moff = a.alloc<int32_t>((int64_t)nc + 1);
    int32_t* mfill = a.alloc<int32_t>(nc);
    int32_t* ucount = a.alloc<int32_t>((int64_t)nc + 1);
    vid_t* members = a.alloc<vid_t>(g.n);
    vid_t* lists = a.alloc<vid_t>(4 * (int64_t)nc);
    int32_t* cnt = a.alloc<int32_t>(4);
    k_contract_reset<<<grid_for((int64_t)nc + 1, 256, 8192), 256, 0, s>>>(nc, hoff, out.vw, moff, mfill, ucount, cnt);
    int nb = grid_for(g.n, 256, 8192);
    k_count<<<nb, 256, 0, s>>>(g, map, hoff, out.vw, moff);
    JET_LAUNCH_CHECK();
    excl_scan_i64_i64(hoff, hoff, nc, a, s);
    excl_scan_i32_i32(moff, moff, nc, a, s);
    k_members<<<nb, 256, 0, s>>>(g.n, map, moff, mfill, members);
    vid_t* l1 = lists;
    vid_t* l2 = lists + nc;
    vid_t* l3 = lists + 2 * (int64_t)nc;
    vid_t* l4 = lists + 3 * (int64_t)nc;
    // the tuned tier bounds never exceed T1_MAX / T2_MAX (half of each table)
    const int32_t t1max = (int32_t)std::min<int64_t>(T1_MAX, tuning().ct_wave_max);
    const int32_t t2max = (int32_t)std::min<int64_t>(T2_MAX, std::max<int64_t>(t1max, tuning().ct_block_max));
    k_tiers<<<grid_for(nc, 256, 8192), 256, 0, s>>>(nc, hoff, l1, l2, l3, l4, cnt, t1max, t2max);
    JET_LAUNCH_CHECK();
    int32_t hcnt[4];
    read_i32_words(cnt, 4, hcnt, s);
    eoff_t H = g.m;
    vid_t* tkey = a.alloc<vid_t>(H);
    wgt_t* tval = a.alloc<wgt_t>(H);
    if (hcnt[0] > 0) {
        k_dedupe_wave<<<grid_for(hcnt[0], T1_WAVES, 8192), T1_WAVES * WAVE, 0, s>>>(g, map, members, moff, hoff, l1,
                                                                                   cnt, tkey, tval, ucount);
        JET_LAUNCH_CHECK();
    }
    eoff_t* medge = nullptr;  // the first fine edge of each member, in the rows' concatenated edges
    if (hcnt[1] > 0 || hcnt[2] > 0 || hcnt[3] > 0) {
        medge = a.alloc<eoff_t>((int64_t)g.n + 1);
        ArenaScope scd(a);
        int32_t* deg = a.alloc<int32_t>((int64_t)g.n + 1);
        k_member_degrees<<<nb, 256, 0, s>>>(g, members, deg);
        JET_LAUNCH_CHECK();
        excl_scan_i32_i64(deg, medge, g.n, a, s);
    }
    if (hcnt[1] > 0) {
        k_dedupe_block<256, T2S_CAP><<<std::min(hcnt[1], 8192), 256, 0, s>>>(g, map, members, medge, moff, hoff, l2,
                                                                            hcnt[1], tkey, tval, ucount);
        JET_LAUNCH_CHECK();
    }
    if (hcnt[3] > 0) {
        k_dedupe_block<1024, T2_CAP><<<std::min(hcnt[3], 2048), 1024, 0, s>>>(g, map, members, medge, moff, hoff, l4,
                                                                             hcnt[3], tkey, tval, ucount);
        JET_LAUNCH_CHECK();
    }
    if (hcnt[2] > 0) {
        int32_t n3 = hcnt[2];
        ArenaScope sc3(a);
        eoff_t* soff = a.alloc<eoff_t>((int64_t)n3 + 1);
        k_spill_sizes<<<grid_for(n3, 256, 1024), 256, 0, s>>>(l3, n3, hoff, soff);
        JET_LAUNCH_CHECK();
        excl_scan_i64_i64(soff, soff, n3, a, s);
        eoff_t H3 = read_scalar(soff + n3, s);
        uint64_t* skey = a.alloc<uint64_t>(H3);
        uint32_t* sval = a.alloc<uint32_t>(H3);
        uint64_t* ktmp = a.alloc<uint64_t>(H3);
        uint32_t* vtmp = a.alloc<uint32_t>(H3);
        // keys of as few bits as the rows and neighbours need: four or five radix
        // passes instead of six on R-MAT 22's levels
        int rbits = 1, nbits = 1;
        while ((int64_t(1) << rbits) < n3 + 1) rbits++;
        while ((int64_t(1) << nbits) < nc) nbits++;
        k_spill_gather<<<grid_for(ceil_div(H3, SPILL_CHUNK) * WAVE, 256, 8192), 256, 0, s>>>(
            g, map, members, medge, moff, hoff, l3, n3, soff, H3, nbits, skey, sval);
        JET_LAUNCH_CHECK();
        radix_sort_u64(skey, sval, H3, nbits + rbits, ktmp, vtmp, a, s);
        int32_t* uid = a.alloc<int32_t>(H3 + 1);
        int hb = grid_for(H3, 256, 8192);
        k_spill_heads<<<hb, 256, 0, s>>>(skey, H3, uid);
        JET_LAUNCH_CHECK();
        excl_scan_i32_i32(uid, uid, H3, a, s);
        int32_t U = read_scalar(uid + H3, s);
        int32_t* ukey = a.alloc<int32_t>(U);
        wgt_t* uval = a.alloc<wgt_t>(U);
        int32_t* urow = a.alloc<int32_t>(U);
        int32_t* rowfirst = a.alloc<int32_t>(n3);
        fill_i32(uval, 0, U, s);
        k_spill_reduce<<<hb, 256, 0, s>>>(skey, sval, H3, nbits, uid, ukey, uval, urow, rowfirst);
        JET_LAUNCH_CHECK();
        if (U > 0) {
            k_spill_write<<<grid_for(U, 256, 8192), 256, 0, s>>>(U, ukey, uval, urow, rowfirst, l3, hoff, tkey, tval,
                                                                 ucount);
            JET_LAUNCH_CHECK();
        }
    }
    excl_scan_i32_i64(ucount, out.rowptr, nc, a, s);
    out.m = read_scalar(out.rowptr + nc, s);
    out.col = persist.alloc<vid_t>(out.m);
    out.ew = persist.alloc<wgt_t>(out.m);
    if (out.m > 0) {
        k_consolidate<<<grid_for(ceil_div(out.m, EB_TILE) * 256, 256, 4096), 256, 0, s>>>(nc, out.m, out.rowptr, hoff, tkey, tval, out.col,
                                                                   out.ew);
        JET_LAUNCH_CHECK();
    }
}

}  // namespace jet
