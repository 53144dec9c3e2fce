// Jet refinement for gfx950 (reference: src/jet_refiner.hpp, src/part_stat.hpp,
// src/uncoarsen.hpp).
//
// Connectivity tables keep the reference's mechanics (capacity min(deg, k),
// direct mapping when the table size is k, linear probing from p % size
// otherwise, shrink to used + max(used/4, 3), HASH_RECLAIM slots, dense
// overflow append) so their contents, sizes and zero entries evolve exactly
// as in the reference. Their slot order is not kept: concurrent updates here
// place new parts in whichever free slot they reach first. Every decision
// that reads a table is therefore made independent of slot order: among parts
// with equal connectivity the lowest part id wins. The reference keeps the
// first maximum in slot order (jet_refiner.hpp:226-233, :603-611). For
// direct-mapped rows (table size k) the two rules agree. For hashed rows
// (size < k) they differ whenever the tied parts' slots are not in id order,
// e.g. parts 5 and 2 in a 4-slot table sit in slots 1 and 2 and the reference
// takes 5; such rows are built serially in edge order by the reference when
// the average degree is below 8, so there its choice is fixed and the lowest-id
// choice is not one the reference can make. Rebalancer minibucket positions
// follow increasing vertex id (a stable sort by bucket id), and the strong
// rebalancer's destination re-draws run in increasing vertex id.
#include <algorithm>
#include <chrono>
#include <mutex>
#include <cmath>

#include "prims.h"
#include "prof.h"
#include "conn_table.h"
#include "refine.h"
#include "tuning.h"
#include "wave.h"

namespace jet {

constexpr int32_t SMALL_DEG = 16;       // rows built by one lane
constexpr int32_t WAVE_TABLE_MAX = 1024; // rows with capacity <= this built by one wave
constexpr int64_t SLICE_EDGES = 1024;  // edges of a long moved row that one wave updates
constexpr int32_t BIG_DEG = 64;         // candidates/moves above this degree use one wave
constexpr int32_t MAX_K = 8192;
constexpr int32_t LDS_K = 2048;         // part-size deltas aggregated in LDS up to this k
constexpr int32_t HEAVY_DEG_REFINE = 2048;  // rows above this degree are built by a workgroup

// ---------------------------------------------------------------- helpers
__device__ inline vid_t list_at(const vid_t* list, int32_t nsmall, vid_t nmax, int64_t x) {
    return x < nsmall ? list[x] : list[nmax - 1 - (x - nsmall)];
}

// ---------------------------------------------------------------- statistics
__global__ void k_cut2(DGraph g, const part_t* part, unsigned long long* out) {
    __shared__ int64_t red[256 / WAVE];
    __shared__ EdgeWalkLds walk;
    int64_t c = 0;
    block_edges<256>(g.rowptr, g.n, g.m, walk, [&](vid_t r, eoff_t j) {
        if (part[g.col[j]] != part[r]) c += g.ew ? g.ew[j] : 1;
    });
    c = block_reduce_sum<int64_t, 256>(c, red);
    if (threadIdx.x == 0 && c) atomicAdd(out, (unsigned long long)c);
}

void launch_cut2(const DGraph& g, const part_t* part, unsigned long long* out, hipStream_t s) {
    if (g.n > 0 && g.m > 0) {
        // 1024 workgroups fill the device; each adds to the one sum (12 ns)
        k_cut2<<<grid_for(g.m, EB_TILE, 1024), 256, 0, s>>>(g, part, out);
        JET_LAUNCH_CHECK();
    }
}

int64_t total_cut2(const DGraph& g, const part_t* part, Arena& a, hipStream_t s) {
    ArenaScope sc(a);
    unsigned long long* out = a.alloc<unsigned long long>(1);
    fill_i64(reinterpret_cast<int64_t*>(out), 0, 1, s);
    launch_cut2(g, part, out, s);
    return (int64_t)read_scalar(out, s);
}

__global__ void k_part_sizes(DGraph g, const part_t* part, int32_t k, unsigned long long* sizes) {
    __shared__ unsigned long long ls[LDS_K];
    bool lds = k <= LDS_K;
    if (lds) {
        for (int t = threadIdx.x; t < k; t += blockDim.x) ls[t] = 0;
        __syncthreads();
    }
    FOR_THREAD(i, g.n) {
        if (lds) atomicAdd(&ls[part[i]], (unsigned long long)g.vw[i]);
        else atomicAdd(&sizes[part[i]], (unsigned long long)g.vw[i]);
    }
    if (lds) {
        __syncthreads();
        for (int t = threadIdx.x; t < k; t += blockDim.x)
            if (ls[t]) atomicAdd(&sizes[t], ls[t]);
    }
}

void part_sizes(const DGraph& g, const part_t* part, int32_t k, int64_t* sizes, hipStream_t s) {
    fill_i64(sizes, 0, k, s);
    if (g.n > 0) {
        k_part_sizes<<<grid_for(g.n, 1024, 256), 1024, 0, s>>>(g, part, k, reinterpret_cast<unsigned long long*>(sizes));
        JET_LAUNCH_CHECK();
    }
}

__global__ void k_project(vid_t n, const vid_t* map, const part_t* coarse, part_t* fine) {
    FOR_THREAD(i, n) fine[i] = coarse[map[i]];
}

// A best-state copy due from the previous step, made by the next step's
// selection kernel as it reads every vertex's part (part_out null: none due).
struct BestCopy {
    part_t* part_out;
    int64_t* sizes_out;
    const int64_t* sizes;
    int32_t k;
    __device__ void sizes_block0() const {
        if (part_out && blockIdx.x == 0)
            for (int32_t p = threadIdx.x; p < k; p += blockDim.x) sizes_out[p] = sizes[p];
    }
};

// The controller's best state (jet_refiner.hpp:1117-1132): the partition
// and the part sizes copied in one launch.
__global__ void k_copy_best(part_t* best_part, const part_t* part, vid_t n, int64_t* best_sizes,
                            const int64_t* sizes, int32_t k) {
    FOR_THREAD(i, n) best_part[i] = part[i];
    if (blockIdx.x == 0)
        for (int32_t p = threadIdx.x; p < k; p += blockDim.x) best_sizes[p] = sizes[p];
}

void project(vid_t n_fine, const vid_t* map, const part_t* coarse, part_t* fine, hipStream_t s) {
    if (n_fine <= 0) return;
    k_project<<<grid_for(n_fine, 256, 16384), 256, 0, s>>>(n_fine, map, coarse, fine);
    JET_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- table build
// jet_refiner.hpp:958-1048 and :648-739: capacity min(deg, k); direct slot p
// when the capacity is k, else linear probing from p % cap; shrink to
// used + max(used/4, 3) when that is smaller. The whole capacity is written
// (layout followed by empty slots). `mark` (optional) restricts the build to
// marked rows, clears their mark and their destination cache (update_large,
// :743-777).

__global__ void k_conn_caps(DGraph g, int32_t k, int32_t* caps) {
    FOR_THREAD(i, g.n) {
        int64_t d = g.rowptr[i + 1] - g.rowptr[i];
        caps[i] = (int32_t)(d > k ? k : d);
    }
}

// Table-build tiers (mid: one wave per row, big: one workgroup per row) and
// the rows whose update_small changes are pulled (degree > BIG_DEG): big-tier
// rows and pull_mid rows; hub[] flags both kinds.
__global__ void __launch_bounds__(256) k_conn_tiers(DGraph g, int32_t k, vid_t* mid, vid_t* big, vid_t* pull_mid,
                                                    int32_t* cnt, uint8_t* hub, int32_t small_max,
                                                    int32_t long_deg) {
    __shared__ int32_t sh[256 / WAVE + 1];
    FOR_BLOCK_UNIFORM(i, g.n) {
        const bool in = i < g.n;
        int64_t d = in ? g.rowptr[i + 1] - g.rowptr[i] : 0;
        int64_t cap = d > k ? k : d;
        bool is_mid = d > small_max && d <= HEAVY_DEG_REFINE && cap <= WAVE_TABLE_MAX;
        bool is_big = d > SMALL_DEG && !is_mid;
        bool is_pmid = is_mid && d > BIG_DEG;
        if (in) hub[i] = (is_big || is_pmid) ? 1 : 0;
        if (d > long_deg) atomicAdd(&cnt[4], (int32_t)((d + SLICE_EDGES - 1) / SLICE_EDGES));
        int32_t a = block_append<256>(&cnt[0], is_mid, sh);
        int32_t b = block_append<256>(&cnt[1], is_big, sh);
        int32_t c = block_append<256>(&cnt[3], is_pmid, sh);
        if (a >= 0) mid[a] = (vid_t)i;
        if (b >= 0) big[b] = (vid_t)i;
        if (c >= 0) pull_mid[c] = (vid_t)i;
    }
}

// The rows of more than long_deg edges, SLICE_EDGES edges of one row per entry:
// (vertex, slice). The update passes give each slice of a moved row to a wave.
__global__ void __launch_bounds__(256) k_row_slices(DGraph g, int32_t long_deg, int2* slices, int32_t* cnt) {
    FOR_THREAD(i, g.n) {
        const int64_t d = g.rowptr[i + 1] - g.rowptr[i];
        if (d <= long_deg) continue;
        const int32_t c = (int32_t)((d + SLICE_EDGES - 1) / SLICE_EDGES);
        const int32_t at = atomicAdd(cnt, c);
        for (int32_t q = 0; q < c; q++) slices[at + q] = make_int2((int32_t)i, q);
    }
}

// Counting runs of the profiler only: adds the degrees of the items of a
// list (counters[cs] from the front, counters[cb] from the back of its nmax
// slots) to out[0]; returns at once when *deferred is set.
__global__ void __launch_bounds__(256)
    k_prof_degsum(DGraph g, const vid_t* list, const int32_t* counters, int cs, int cb, vid_t nmax,
                  const int32_t* deferred, unsigned long long* out) {
    __shared__ int64_t red[256 / WAVE];
    if (deferred && *deferred) return;
    const int64_t ns = counters[cs], nb = counters[cb];
    int64_t sum = 0;
    FOR_THREAD(x, ns + nb) {
        const vid_t v = x < ns ? list[x] : list[nmax - 1 - (x - ns)];
        sum += g.rowptr[v + 1] - g.rowptr[v];
    }
    sum = block_reduce_sum<int64_t, 256>(sum, red);
    if (threadIdx.x == 0 && sum) atomicAdd(out, (unsigned long long)sum);
}

constexpr int SB_BLOCK = 256;

__global__ void __launch_bounds__(SB_BLOCK)
    k_conn_build_small(DGraph g, const part_t* part, int32_t k, const eoff_t* conn_off, int2* conn,
                       int32_t* conn_size, int32_t* mark, part_t* dest_cache, const int32_t* gate, int32_t small_max) {
    if (gate && gate[0] == 0) return;
    __shared__ int2 tab[SMALL_DEG][SB_BLOCK];
    const int t = threadIdx.x;
    FOR_THREAD(i, g.n) {
        eoff_t rs = g.rowptr[i], re = g.rowptr[i + 1];
        int32_t deg = (int32_t)(re - rs);
        if (deg > small_max) continue;
        if (mark) {
            if (!mark[i]) continue;
            mark[i] = 0;
            dest_cache[i] = NULL_PART;
        }
        int32_t cap = deg < k ? deg : k;
        for (int32_t s = 0; s < cap; s++) tab[s][t] = make_int2(NULL_PART, 0);
        int32_t used = 0;
        for (eoff_t j = rs; j < re; j++) {
            part_t p = part[g.col[j]];
            int32_t po = p % cap;
            if (cap < k) {
                while (tab[po][t].x != NULL_PART && tab[po][t].x != p) po = (po + 1) % cap;
            }
            if (tab[po][t].x == NULL_PART) {
                tab[po][t].x = p;
                used++;
            }
            tab[po][t].y += g.ew[j];
        }
        int2* out = conn + conn_off[i];
        int32_t size = shrink_size(used, cap);
        if (size < cap) {
            for (int32_t s = 0; s < cap; s++) out[s] = make_int2(NULL_PART, 0);
            for (int32_t s = 0; s < cap; s++) {
                int2 e = tab[s][t];
                if (e.x == NULL_PART) continue;
                int32_t po = e.x % size;
                while (out[po].x != NULL_PART) po = (po + 1) % size;
                out[po] = e;
            }
        } else {
            for (int32_t s = 0; s < cap; s++) out[s] = tab[s][t];
        }
        conn_size[i] = size;
    }
}

// Inserts part p with weight w into an LDS table of `cap` slots (cap == k:
// direct; else probing); counts newly used slots.
__device__ inline void lds_table_add(int2* T, int32_t cap, int32_t k, part_t p, int32_t w, int32_t* used) {
    int32_t po = p % cap;
    if (cap == k) {
        if (T[po].x == NULL_PART && atomicCAS(&T[po].x, NULL_PART, p) == NULL_PART) atomicAdd(used, 1);
    } else {
        for (int32_t guard = 0; guard <= cap; guard++) {
            int32_t px = T[po].x;
            if (px == p) break;
            if (px == NULL_PART) {
                int32_t old = atomicCAS(&T[po].x, NULL_PART, p);
                if (old == NULL_PART) {
                    atomicAdd(used, 1);
                    break;
                }
                if (old == p) break;
            }
            po = (po + 1) % cap;
        }
    }
    atomicAdd(&T[po].y, w);
}

// The edges rs + sub + q * stride of a row by this thread, CB_UNROLL of their
// parts in flight.
constexpr int CB_UNROLL = 4;
__device__ inline void table_add_row(int2* T, int32_t cap, int32_t k, const DGraph& g, eoff_t rs, eoff_t re, int sub,
                                     int stride, const part_t* part, int32_t* used) {
    for (eoff_t b0 = rs + sub; b0 < re; b0 += (eoff_t)CB_UNROLL * stride) {
        vid_t v[CB_UNROLL];
        int32_t w[CB_UNROLL];
        part_t p[CB_UNROLL];
#pragma unroll
        for (int q = 0; q < CB_UNROLL; q++) {
            const eoff_t j = b0 + (eoff_t)q * stride;
            v[q] = j < re ? g.col[j] : -1;
            w[q] = j < re ? g.ew[j] : 0;
        }
#pragma unroll
        for (int q = 0; q < CB_UNROLL; q++) p[q] = v[q] >= 0 ? part[v[q]] : 0;
#pragma unroll
        for (int q = 0; q < CB_UNROLL; q++)
            if (v[q] >= 0) lds_table_add(T, cap, k, p[q], w[q], used);
    }
}

// Re-inserts the entries of T (cap slots) into T2 (size slots, linear probing).
__device__ inline void lds_table_shrink(const int2* T, int32_t cap, int2* T2, int32_t size, int start, int stride) {
    for (int32_t s = start; s < cap; s += stride) {
        int2 e = T[s];
        if (e.x == NULL_PART) continue;
        int32_t po = e.x % size;
        for (int32_t guard = 0; guard <= size; guard++) {
            if (T2[po].x == NULL_PART && atomicCAS(&T2[po].x, NULL_PART, e.x) == NULL_PART) {
                T2[po].y = e.y;
                break;
            }
            po = (po + 1) % size;
        }
    }
}

constexpr int WB_WAVES = 4;

__global__ void __launch_bounds__(WB_WAVES* WAVE)
    k_conn_build_wave(DGraph g, const part_t* part, int32_t k, const eoff_t* conn_off, int2* conn,
                      int32_t* conn_size, int32_t* mark, part_t* dest_cache, const vid_t* list, int32_t nlist,
                      const int32_t* gate) {
    if (gate && gate[0] == 0) return;
    // per wave two tables of tcap = min(k, WAVE_TABLE_MAX) slots, sized at launch
    extern __shared__ int2 tabs[];
    __shared__ int32_t used[WB_WAVES];
    const int lane = threadIdx.x & (WAVE - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int32_t tcap = k < WAVE_TABLE_MAX ? k : WAVE_TABLE_MAX;
    int2* Tw = tabs + (size_t)(2 * w) * tcap;
    int2* T2w = Tw + tcap;
    for (int32_t r = blockIdx.x * WB_WAVES + w; r < nlist; r += gridDim.x * WB_WAVES) {
        vid_t i = list[r];
        if (mark) {
            if (!mark[i]) continue;
        }
        eoff_t rs = g.rowptr[i], re = g.rowptr[i + 1];
        int32_t deg = (int32_t)(re - rs);
        int32_t cap = deg < k ? deg : k;
        for (int32_t s = lane; s < cap; s += WAVE) {
            Tw[s] = make_int2(NULL_PART, 0);
            T2w[s] = make_int2(NULL_PART, 0);
        }
        if (lane == 0) used[w] = 0;
        wave_sync();
        table_add_row(Tw, cap, k, g, rs, re, lane, WAVE, part, &used[w]);
        wave_sync();
        int32_t size = shrink_size(used[w], cap);
        int2* out = conn + conn_off[i];
        if (size < cap) {
            lds_table_shrink(Tw, cap, T2w, size, lane, WAVE);
            wave_sync();
            for (int32_t s = lane; s < cap; s += WAVE) out[s] = T2w[s];
        } else {
            for (int32_t s = lane; s < cap; s += WAVE) out[s] = Tw[s];
        }
        if (lane == 0) {
            conn_size[i] = size;
            if (mark) {
                mark[i] = 0;
                dest_cache[i] = NULL_PART;
            }
        }
        wave_sync();
    }
}

constexpr int BB_BLOCK = 512;

__global__ void __launch_bounds__(BB_BLOCK)
    k_conn_build_block(DGraph g, const part_t* part, int32_t k, const eoff_t* conn_off, int2* conn,
                       int32_t* conn_size, int32_t* mark, part_t* dest_cache, const vid_t* list, int32_t nlist,
                       const int32_t* gate) {
    if (gate && gate[0] == 0) return;
    // two tables of min(k, max degree) slots, sized at launch
    extern __shared__ int2 tabs[];
    const int32_t tcap = k;
    int2* T = tabs;
    int2* T2 = tabs + tcap;
    __shared__ int32_t used;
    for (int32_t r = blockIdx.x; r < nlist; r += gridDim.x) {
        vid_t i = list[r];
        if (mark && !mark[i]) continue;
        eoff_t rs = g.rowptr[i], re = g.rowptr[i + 1];
        int64_t deg = re - rs;
        int32_t cap = (int32_t)(deg < k ? deg : k);
        for (int32_t s = threadIdx.x; s < cap; s += BB_BLOCK) {
            T[s] = make_int2(NULL_PART, 0);
            T2[s] = make_int2(NULL_PART, 0);
        }
        if (threadIdx.x == 0) used = 0;
        __syncthreads();
        table_add_row(T, cap, k, g, rs, re, threadIdx.x, BB_BLOCK, part, &used);
        __syncthreads();
        int32_t size = shrink_size(used, cap);
        int2* out = conn + conn_off[i];
        if (size < cap) {
            lds_table_shrink(T, cap, T2, size, threadIdx.x, BB_BLOCK);
            __syncthreads();
            for (int32_t s = threadIdx.x; s < cap; s += BB_BLOCK) out[s] = T2[s];
        } else {
            for (int32_t s = threadIdx.x; s < cap; s += BB_BLOCK) out[s] = T[s];
        }
        if (threadIdx.x == 0) {
            conn_size[i] = size;
            if (mark) {
                mark[i] = 0;
                dest_cache[i] = NULL_PART;
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- jet_lp
// A table of more than SEL_LONG slots is read by the whole wave in the select
// kernels, one after another of its lanes' long tables: a lane that reads 256
// slots alone takes 64 dependent trips to memory, for which its wave waits.
// That pays where the waves wait for memory anyway: R-MAT 22 (k = 256), LP
// select 1.06 -> 0.86 ms on 4,194,304 vertices and 0.49 -> 0.31 on 756,505, but
// 98 -> 141 us on 370,878; strong select 0.90 -> 0.37, 0.15 -> 0.10 and, on
// 438,484 vertices, 0.08 -> 0.06 ms, but 70 -> 82 us on 370,878. (LP select has
// the variant in its two-pass shape only, above lp_one_pass_n vertices.) The
// weak select's four vertices a lane hide the trips as they are (0.15 -> 0.20 ms
// on 756,505).
constexpr int32_t SEL_LONG = 16;
constexpr int64_t SEL_LONG_N = 400000;

// Calls f(lane's row broadcast) for each lane with `mine` set, the whole wave
// together: f(b) gets the lane's number.
template <class F>
__device__ inline void for_long_rows(bool mine, F&& f) {
    uint64_t mk = __ballot(mine);
    while (mk) {
        const int b = __ffsll((unsigned long long)mk) - 1;
        mk &= mk - 1;
        f(b);
    }
}

__device__ inline uint64_t wave_reduce_max_u64(uint64_t x) {
    for (int d = WAVE / 2; d >= 1; d >>= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)x, d, WAVE);
        const uint32_t hi = __shfl_xor((uint32_t)(x >> 32), d, WAVE);
        const uint64_t y = ((uint64_t)hi << 32) | lo;
        x = y > x ? y : x;
    }
    return x;
}

// The slot of largest positive connectivity among those ok() accepts (ties:
// smaller part id) and part p's connectivity, by a wave; `none` when no slot
// qualifies.
template <class OK>
__device__ inline void wave_best_slot(const int2* tab, int32_t sz, part_t p, part_t none, OK&& ok, part_t& best,
                                      int32_t& gain, int32_t& p_gain) {
    const int lane = threadIdx.x & (WAVE - 1);
    uint64_t key = 0;
    int32_t pg = 0;
    for (int32_t s = lane; s < sz; s += WAVE) {
        const int2 e = tab[s];
        if (e.y > 0 && ok(e)) {
            const uint64_t x = ((uint64_t)(uint32_t)e.y << 32) | (uint32_t)~e.x;
            key = x > key ? x : key;
        }
        if (e.x == p) pg = e.y;
    }
    key = wave_reduce_max_u64(key);
    gain = (int32_t)(key >> 32);
    best = gain > 0 ? (part_t)~(uint32_t)key : none;
    p_gain = wave_reduce_sum(pg);
}

// jet_refiner.hpp:211-268: destination selection, viable-move filter.
// Each wave owns a contiguous chunk of CHW vertices (CHW / WAVE passes);
// candidates are staged in LDS and published with one atomic per workgroup
// of W waves.
constexpr int LS_WAVES = 8;
// Levels up to Tuning::lp_one_pass_n vertices run one pass per wave in
// workgroups of LS_WAVES waves (eight: 0.3 ms less per 128^3 stencil
// partition than four; sixteen is slower there). Larger levels run
// LS_MULTI_CHW vertices per wave in workgroups of LS_MULTI_WAVES waves: few
// enough workgroups appending to the candidate counters, and two passes per
// wave (measured on the 128^3 stencil: 12.1 us per launch on average,
// against 14.2 with eight passes in workgroups of four waves).
constexpr int LS_MULTI_CHW = 128;
constexpr int LS_MULTI_WAVES = 16;

template <int CHW, int W, bool LONG>
__global__ void __launch_bounds__(W* WAVE)
    k_lp_select(DGraph g, const part_t* part, const eoff_t* conn_off, const int2* conn, const int32_t* conn_size,
                part_t* dest_cache, int32_t* gain_p, int32_t* lock, double fr, part_t* dest, int32_t* pregain,
                vid_t* cand, int32_t* counters, vid_t nmax, int32_t* next_counters, uint64_t* cbits, int4* crec,
                unsigned long long* pc, BestCopy bc) {
    constexpr int NPASS = CHW / WAVE;
    __shared__ vid_t sbuf[W * CHW];
    __shared__ int32_t sh[2 * W + 2];
    __shared__ int64_t pred[W];
    // wave-private: the slots (u * WAVE + lane) of the wave's cache misses,
    // and each miss's new destination and gain
    __shared__ int16_t mslot[W][CHW];
    __shared__ part_t mbest[W][CHW];
    __shared__ int32_t mgain[W][CHW];
    int64_t n_miss = 0, n_slot = 0;
    StagedLists<W, CHW> st(sbuf);
    if (blockIdx.x == 0 && threadIdx.x < 8) next_counters[threadIdx.x] = 0;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = threadIdx.x / WAVE;
    const int64_t wbase = ((int64_t)blockIdx.x * W + wv) * CHW;
    const uint64_t lt = (1ull << lane) - 1ull;
    // 1. the cached destinations and locks of all passes, loaded together
    part_t cached[NPASS];
    int32_t locks[NPASS];
#pragma unroll
    for (int u = 0; u < NPASS; u++) {
        const int64_t i = wbase + u * WAVE + lane;
        cached[u] = i < g.n ? dest_cache[i] : NO_MOVE;
        locks[u] = i < g.n ? lock[i] : 0;
    }
    if (bc.part_out) {  // the previous step's best state, with the loads above
#pragma unroll
        for (int u = 0; u < NPASS; u++) {
            const int64_t i = wbase + u * WAVE + lane;
            if (i < g.n) bc.part_out[i] = part[i];
        }
        bc.sizes_block0();
    }
    // 2. the wave's misses, compacted, so that every lane evaluates one
    // table at a time instead of each pass waiting on its own few misses
    int32_t nm = 0;
#pragma unroll
    for (int u = 0; u < NPASS; u++) {
        const bool miss = cached[u] == NULL_PART;
        const uint64_t mk = __ballot(miss);
        if (miss) mslot[wv][nm + (int32_t)__popcll(mk & lt)] = (int16_t)(u * WAVE + lane);
        nm += (int32_t)__popcll(mk);
    }
    wave_sync();
    for (int32_t m0 = 0; m0 < nm; m0 += WAVE) {
        const bool in = m0 + lane < nm;
        const int32_t slot = in ? mslot[wv][m0 + lane] : 0;
        const int64_t i = wbase + slot;
        const part_t p = in ? part[i] : 0;
        part_t best = NO_MOVE;
        int32_t b_conn = 0, p_conn = 0;
        const int32_t sz = in ? conn_size[i] : 0;
        const eoff_t off = in ? conn_off[i] : 0;
        n_miss += in;
        n_slot += sz;
        if (!LONG || sz <= SEL_LONG)
            for_slots(conn + off, sz, [&](int2 e) {
                if (e.y > b_conn && e.x != p) {
                    best = e.x;
                    b_conn = e.y;
                } else if (e.y == b_conn && b_conn > 0 && e.x != p && e.x < best) {
                    best = e.x;
                } else if (e.y > 0 && e.x == p) {
                    p_conn = e.y;
                }
            });
        for_long_rows(LONG && sz > SEL_LONG, [&](int b) {
            const part_t bp = __shfl(p, b, WAVE);
            part_t x;
            int32_t gx, px;
            wave_best_slot(conn + (eoff_t)__shfl((int64_t)off, b, WAVE), __shfl(sz, b, WAVE), bp, NO_MOVE,
                           [&](int2 e) { return e.x != bp; }, x, gx, px);
            if (lane == b) {
                best = x;
                b_conn = gx;
                p_conn = px;
            }
        });
        if (!in) continue;
        int32_t gsv = 0;
        if (best != NO_MOVE) {
            if (b_conn >= p_conn || ((double)(p_conn - b_conn) < floor(fr * (double)p_conn))) gsv = b_conn - p_conn;
            else best = NO_MOVE;
        }
        gain_p[i] = gsv;
        dest_cache[i] = best;
        mbest[wv][slot] = best;
        mgain[wv][slot] = gsv;
    }
    wave_sync();
    // 3. destinations; a vertex that is not a candidate this iteration gets
    // NO_MOVE: the afterburner skips such neighbours before reading their
    // pre-gain, which is then only written for candidates. The candidates'
    // gains and row offsets of all passes are loaded together.
    bool is_cand[NPASS];
    part_t dst[NPASS];
    int32_t gain[NPASS];
    eoff_t r0[NPASS], r1[NPASS];
#pragma unroll
    for (int u = 0; u < NPASS; u++) {
        const int64_t i = wbase + u * WAVE + lane;
        const bool miss = cached[u] == NULL_PART;
        const part_t best = miss ? mbest[wv][u * WAVE + lane] : cached[u];
        is_cand[u] = i < g.n && best != NO_MOVE && locks[u] == 0;
        dst[u] = best;
        if (i < g.n) {
            dest[i] = is_cand[u] ? best : NO_MOVE;
            if (!is_cand[u] && locks[u]) lock[i] = 0;
        }
        gain[u] = 0;
        r0[u] = r1[u] = 0;
        if (is_cand[u]) {
            gain[u] = miss ? mgain[wv][u * WAVE + lane] : gain_p[i];
            r0[u] = g.rowptr[i];
            r1[u] = g.rowptr[i + 1];
        }
    }
#pragma unroll
    for (int u = 0; u < NPASS; u++) {
        const int64_t i = wbase + u * WAVE + lane;
        const eoff_t deg = r1[u] - r0[u];
        if (is_cand[u]) pregain[i] = gain[u];
        if (cbits) {
            const uint64_t mk = __ballot(is_cand[u]);
            if (lane == 0 && i < g.n) cbits[i / WAVE] = mk;
            if (is_cand[u]) crec[i] = make_int4(dst[u], gain[u], part[i], 0);
        }
        st.push(is_cand[u] && deg <= BIG_DEG, is_cand[u] && deg > BIG_DEG, (vid_t)i);
    }
    st.flush(cand, &counters[0], &counters[1], nmax, sh);
    if (pc) {  // counting runs only: evaluated vertices and table slots read
        int64_t v2[2] = {n_miss, n_slot};
        for (int q = 0; q < 2; q++) {
            int64_t v = block_reduce_sum<int64_t, W * WAVE>(v2[q], pred);
            if (threadIdx.x == 0 && v) atomicAdd(&pc[q], (unsigned long long)v);
        }
    }
}

// 16-wave workgroups: each workgroup publishes its moves with one atomic on
// the move counters, and fewer workgroups contend for them (measured 0.9 ms
// less per 128^3 stencil partition than four-wave workgroups)
constexpr int AB_WAVES = 16;
constexpr int AB_CHW = 256;

// A neighbour's term from its record (destination, pre-gain, part), and the
// same behind its candidate bit (a vertex without it contributes nothing).
__device__ inline int64_t burn_term(vid_t v, vid_t i, int32_t ig, int32_t w, part_t p, part_t best, int4 r) {
    int64_t ch = 0;
    if (r.y > ig || (r.y == ig && v < i)) {  // afterburn_edge
        if (r.x == p) ch -= w;
        else if (r.x == best) ch += w;
        if (r.z == p) ch += w;
        else if (r.z == best) ch -= w;
    }
    return ch;
}
__device__ inline int64_t afterburn_rec(vid_t v, vid_t i, int32_t ig, int32_t w, part_t p, part_t best,
                                        const uint32_t* cbits, const int4* crec) {
    if (((cbits[v >> 5] >> (v & 31)) & 1u) == 0) return 0;
    return burn_term(v, i, ig, w, p, best, crec[v]);
}

template <int G, bool REC>
__global__ void __launch_bounds__(AB_WAVES* WAVE)
    k_afterburner_small(DGraph g, const vid_t* cand, const int32_t* counters, const part_t* part, const part_t* dest,
                        const int32_t* pregain, int32_t* lock, vid_t* moves, int32_t* mcounters, vid_t nmax,
                        int32_t* stamp, int32_t gen, const uint32_t* cbits, const int4* crec) {
    __shared__ vid_t sbuf[AB_WAVES * AB_CHW];
    __shared__ int32_t sh[2 * AB_WAVES + 2];
    StagedLists<AB_WAVES, AB_CHW> st(sbuf);
    const int lane = threadIdx.x & (WAVE - 1);
    const int sub = lane & (G - 1);
    // wave w takes candidates w * WAVE/G + [0, WAVE/G), then every tw-th such
    // group (tw = waves in the grid): the mapping does not depend on the
    // count, so a lane's first candidate is loaded together with it. The
    // host launches tw * AB_CHW >= n lanes' worth of waves, so no wave
    // stages more than AB_CHW moves (AB_CHW * G / WAVE rounds).
    const int64_t tw = (int64_t)gridDim.x * AB_WAVES;
    const int64_t wfirst = ((int64_t)blockIdx.x * AB_WAVES + threadIdx.x / WAVE) * (WAVE / G);
    const int64_t x0 = wfirst + lane / G;
    const vid_t c0 = x0 < nmax ? cand[x0] : 0;
    const int32_t nc = counters[0];
    int32_t round = 0;
    for (int64_t xw = wfirst; xw < nc && round < AB_CHW * G / WAVE; xw += tw * (WAVE / G), round++) {
        const int64_t x = xw + lane / G;
        bool keep = false;
        vid_t i = 0;
        if (x < nc) {
            i = round == 0 ? c0 : cand[x];
            part_t p = part[i], best = dest[i];
            int32_t ig = pregain[i];
            int64_t change = 0;
            for (eoff_t j = g.rowptr[i] + sub; j < g.rowptr[i + 1]; j += G)
                change += REC ? afterburn_rec(g.col[j], i, ig, g.ew[j], p, best, cbits, crec)
                              : afterburn_edge(g.col[j], i, ig, g.ew[j], p, best, part, dest, pregain);
#pragma unroll
            for (int d = G / 2; d >= 1; d >>= 1) change += __shfl_xor(change, d, G);
            keep = (int64_t)ig + change >= 0;
            if (keep && sub == 0) lock[i] = 1;
        }
        st.push(keep && sub == 0, false, i);
    }
    st.flush_stamped(moves, &mcounters[2], &mcounters[3], nmax, sh, stamp, gen);
}

// A wave per candidate of degree > BIG_DEG, AB_UNROLL edges per lane in
// flight. A bit per vertex says which neighbours are candidates (n / 8 bytes,
// resident in L2; the others contribute nothing), and a candidate's
// destination, pre-gain and part come in one 16-byte record. A wave appends
// its moves 64 at a time: one atomic per move on the list's counter was the
// bound where a tenth of the vertices move (R-MAT 22, 4,194,304 vertices: 1.55
// ms on average, now 0.38; 756,505: 1.08, now 0.59, bound by the gathers).
// Candidates of degree > long_deg are queued in LDS and taken by the
// whole workgroup afterwards.
constexpr int AB_UNROLL = 4;
constexpr int AB_QUEUE = 1024;
__global__ void __launch_bounds__(AB_WAVES* WAVE)
    k_afterburner_big(DGraph g, const vid_t* cand, const int32_t* counters, const part_t* part, const part_t* dest,
                      const int32_t* pregain, int32_t* lock, vid_t* moves, int32_t* mcounters, vid_t nmax,
                      int32_t* stamp, int32_t gen, int32_t long_deg, const uint32_t* cbits, const int4* crec) {
    __shared__ vid_t queue[AB_QUEUE];
    __shared__ vid_t keeps[AB_WAVES][WAVE];
    __shared__ int32_t nqueue;
    __shared__ int64_t red[AB_WAVES];
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);  // the candidates' state in scalar registers
    const int32_t nb = counters[1];
    if (nb == 0) return;
    if (threadIdx.x == 0) nqueue = 0;
    __syncthreads();
    auto burn = [&](vid_t i, eoff_t rs, eoff_t re, int sub, int stride) -> int64_t {
        const part_t p = part[i], best = dest[i];
        const int32_t ig = pregain[i];
        int64_t change = 0;
        for (eoff_t b0 = rs; b0 < re; b0 += (eoff_t)AB_UNROLL * stride) {
            vid_t v[AB_UNROLL];
            bool c[AB_UNROLL];
            int32_t w[AB_UNROLL];
            int4 r[AB_UNROLL];
#pragma unroll
            for (int q = 0; q < AB_UNROLL; q++) {
                const eoff_t j = b0 + (eoff_t)q * stride + sub;
                v[q] = j < re ? g.col[j] : -1;
            }
#pragma unroll
            for (int q = 0; q < AB_UNROLL; q++) c[q] = v[q] >= 0 && ((cbits[v[q] >> 5] >> (v[q] & 31)) & 1u);
#pragma unroll
            for (int q = 0; q < AB_UNROLL; q++) {
                r[q] = c[q] ? crec[v[q]] : make_int4(0, 0, 0, 0);
                w[q] = c[q] ? g.ew[b0 + (eoff_t)q * stride + sub] : 0;
            }
#pragma unroll
            for (int q = 0; q < AB_UNROLL; q++)
                if (c[q]) change += burn_term(v[q], i, ig, w[q], p, best, r[q]);
        }
        return change;
    };
    // the wave's moves, appended to the list WAVE at a time
    vid_t* kept = keeps[wv];
    int32_t nkept = 0;
    auto flush = [&]() {
        wave_sync();
        int32_t at = 0;
        if (lane == 0) at = atomicAdd(&mcounters[3], nkept);
        at = __shfl(at, 0, WAVE);
        if (lane < nkept) moves[nmax - 1 - (at + lane)] = kept[lane];
        nkept = 0;
        wave_sync();
    };
    auto keep = [&](vid_t i, int64_t change) {  // a wave
        if ((int64_t)pregain[i] + change < 0) return;
        if (lane == 0) {
            lock[i] = 1;
            stamp[i] = gen;
            kept[nkept] = i;
        }
        if (++nkept == WAVE) flush();
    };
    // consecutive candidates go to different workgroups
    for (int64_t x = (int64_t)wv * gridDim.x + blockIdx.x; x < nb; x += (int64_t)gridDim.x * AB_WAVES) {
        const vid_t i = cand[nmax - 1 - x];
        const eoff_t rs = g.rowptr[i], re = g.rowptr[i + 1];
        if (re - rs > long_deg) {
            int32_t slot = 0;
            if (lane == 0) slot = atomicAdd(&nqueue, 1);
            slot = __shfl(slot, 0, WAVE);
            if (slot < AB_QUEUE) {
                if (lane == 0) queue[slot] = i;
                continue;
            }
        }
        keep(i, wave_reduce_sum(burn(i, rs, re, lane, WAVE)));
    }
    __syncthreads();
    const int32_t nq = min(nqueue, AB_QUEUE);
    for (int32_t q = 0; q < nq; q++) {
        const vid_t i = queue[q];
        const int64_t change = block_reduce_sum<int64_t, AB_WAVES * WAVE>(
            burn(i, g.rowptr[i], g.rowptr[i + 1], threadIdx.x, AB_WAVES * WAVE), red);
        if (wv == 0) keep(i, change);
    }
    if (nkept > 0) flush();
}

// ---------------------------------------------------------------- perform_moves
// perform_moves' choice between update_small (push each moved vertex's
// contribution into its neighbours' tables) and update_large (rebuild the
// tables of every neighbour of a moved vertex): rebuild when more than n/10
// vertices move (jet_refiner.hpp:933). The two do not leave the same tables:
// pushing keeps a part whose connectivity falls to 0 in a table of k slots
// (jet_refiner.hpp:806-810) and the rebalancers read such entries, so the
// choice follows the reference exactly.
// Every hub row is scanned for moved neighbours (k_pull_hubs) when more than
// n / PULL_ALL_DIV vertices move, else only those the first pass flags.
constexpr int32_t PULL_ALL_DIV = 512;

// The cut change and the largest part (jet_refiner.hpp:937-948). For a moved
// vertex v the reference adds conn(v, new part) - conn(v, old part) from its
// table before the updates and again after them; each is the sum over v's
// edges (v, u) of w * ([part(u) == new part of v] - [part(u) == old part of v]),
// with the parts before and after the moves, so the first pass computes both
// from the parts and needs no table. It adds each workgroup's sum into one of
// PUB_GROUPS partials (workgroup b into partial b mod PUB_GROUPS), 128 bytes
// apart, so that no line takes more than a sixteenth of the grid's atomics.
// Workgroup 0 of the second pass folds them, takes the largest part and
// writes (cut change, largest part, deferred, rebuild) to the host mailbox. A
// deferred step reports only the deferral.
constexpr int PUB_GROUPS = 16;
constexpr int PUB_STRIDE = 16;  // int64 words: 128 bytes

__device__ inline void add_cut_part2(int64_t* partials, int64_t c2, int64_t* red) {
    c2 = block_reduce_sum<int64_t, 256>(c2, red);
    if (threadIdx.x == 0 && c2)
        atomicAdd((unsigned long long*)&partials[(int64_t)(blockIdx.x % PUB_GROUPS) * PUB_STRIDE],
                  (unsigned long long)c2);
}

// Run by one workgroup (256 threads) after the first pass: folds the
// partials, takes the largest part and writes (cut change, largest part,
// deferred, rebuild) to the host mailbox, then the sequence word the host
// waits for, and clears the accumulators. One workgroup needs no completion
// ticket (a ticket in a many-workgroup kernel needs an agent-scope release
// fence per workgroup, which writes back L2), and the kernel boundary before
// it orders the other kernels' atomics.
// The state a rebalancing step starts from, besides zeroed bucket sums: the
// undersized parts in increasing id (weak, jet_refiner.hpp:578-591) or the
// largest receiver capacity and cleared eviction adjustments (strong,
// :440-448), from the part sizes before the step. One workgroup of 256.
__device__ inline void rebalance_prep_block(const int64_t* sizes, int32_t k, int64_t max_dest, bool strong,
                                            part_t* undersized, int32_t* misc, int64_t* acc, int64_t* evict_adjust,
                                            int64_t* red, int32_t* ws) {
    if (strong) {
        int64_t mx = INT64_MIN;
        for (int t = threadIdx.x; t < k; t += blockDim.x) {
            int64_t sz = sizes[t];
            if (sz < max_dest && max_dest - sz > mx) mx = max_dest - sz;
            evict_adjust[t] = 0;
        }
        mx = block_reduce_max<int64_t, 256>(mx, red);
        if (threadIdx.x == 0) acc[3] = mx;
    } else {
        int32_t base = 0;
        for (int32_t p0 = 0; p0 < k; p0 += 256) {
            int32_t p = p0 + threadIdx.x;
            int32_t f = (p < k && sizes[p] < max_dest) ? 1 : 0;
            int32_t tot;
            int32_t ex = block_excl_scan<int32_t, 256>(f, tot, ws);
            if (f) undersized[base + ex] = p;
            base += tot;
        }
        if (threadIdx.x == 0) misc[0] = base;
    }
}

// What the second update pass prepares for the next step in case it is a
// rebalancing step of the given kind (buckets == nullptr: nothing): its
// bucket sums zeroed (nb entries) and rebalance_prep_block's state, so that
// the step needs no reset launch.
struct RebalPrep {
    int64_t* buckets;
    int64_t nb;
    int64_t max_dest;
    int32_t strong;
    part_t* undersized;
    int32_t* misc;
    int64_t* acc;
    int64_t* evict_adjust;
};

// The first update pass's workgroups add their part-size deltas into one of
// `ncopies` copies of a k-entry array (workgroup b into copy b mod ncopies),
// so that fewer workgroups' atomics meet on one address; the second pass's
// publishing workgroup folds the copies into the sizes and clears them.
constexpr int SIZE_COPIES_MAX = 16;

struct Publish {
    int64_t* partials;
    int64_t* sizes;
    int32_t k;
    int64_t* host_out;
    const int32_t* mc;
    int64_t seq;
    unsigned long long* copies;  // ncopies * k deltas, zero between steps
    int32_t ncopies;
};

__device__ inline void fold_size_copies(const Publish& pb) {
    if (pb.ncopies <= 0) return;
    for (int t = threadIdx.x; t < pb.k; t += blockDim.x) {
        // every copy's load in flight at once, then the clears
        unsigned long long v[SIZE_COPIES_MAX];
#pragma unroll
        for (int c = 0; c < SIZE_COPIES_MAX; c++) v[c] = c < pb.ncopies ? pb.copies[(int64_t)c * pb.k + t] : 0;
        unsigned long long d = 0;
#pragma unroll
        for (int c = 0; c < SIZE_COPIES_MAX; c++) {
            d += v[c];
            if (v[c]) pb.copies[(int64_t)c * pb.k + t] = 0;
        }
        if (d) pb.sizes[t] += (int64_t)d;
    }
    __syncthreads();
}

__device__ inline void publish_step(const Publish& pb, bool deferred, int64_t* red) {
    if (deferred) {
        if (threadIdx.x == 0) {
            pb.host_out[2] = 1;
            __threadfence_system();
            pb.host_out[5] = pb.seq;  // the host waits for this word
            __threadfence_system();
        }
        return;
    }
    int64_t mx = INT64_MIN;
    for (int t = threadIdx.x; t < pb.k; t += blockDim.x) mx = pb.sizes[t] > mx ? pb.sizes[t] : mx;
    mx = block_reduce_max<int64_t, 256>(mx, red);
    int64_t c2 = threadIdx.x < PUB_GROUPS ? pb.partials[(int64_t)threadIdx.x * PUB_STRIDE] : 0;
    c2 = block_reduce_sum<int64_t, 256>(c2, red);
    if (threadIdx.x < PUB_GROUPS) pb.partials[(int64_t)threadIdx.x * PUB_STRIDE] = 0;
    if (threadIdx.x == 0) {
        pb.host_out[0] = c2;
        pb.host_out[1] = mx;
        pb.host_out[2] = 0;
        pb.host_out[3] = pb.mc[6];  // the tables are to be rebuilt (update_large)
        __threadfence_system();
        pb.host_out[5] = pb.seq;  // written after the results: the host waits for it
        __threadfence_system();
    }
}

// One move's record, written by the first pass for the second: the vertex,
// its new part and its row, so that the second pass's chain starts at the
// record (no part, destination or row-offset loads).
struct MoveRec {
    eoff_t rs;
    int32_t deg;
    vid_t v;
    part_t pnew;
    int32_t unused;
};

// One move in either pass, or one slice of it: the edges rs + sub, rs + sub +
// stride, ... before re.
// One edge of a move, its neighbour v no hub: the cut change and the old
// part's subtraction (first pass) or the new part's addition (second).
template <bool ADD>
__device__ inline void update_edge(vid_t v, int32_t w, part_t pold, part_t pnew, bool rebuild, const part_t* part,
                                   const part_t* dest, const eoff_t* conn_off, int2* conn, int32_t* conn_size,
                                   part_t* dest_cache, int32_t k, int32_t* err, int32_t* mark, const int32_t* stamp,
                                   int32_t gen, int64_t& cc) {
    if (!ADD) {
        // loaded together: the neighbour's parts and table
        const part_t pv = part[v], dv = dest[v];
        const bool sv = stamp[v] == gen;
        const eoff_t co = rebuild ? 0 : conn_off[v];
        const int32_t cs = rebuild ? 0 : ld_rx(&conn_size[v]);
        const part_t nv = sv ? dv : pv;
        cc += (int64_t)w *
              ((pv == pnew ? 1 : 0) - (pv == pold ? 1 : 0) + (nv == pnew ? 1 : 0) - (nv == pold ? 1 : 0));
        if (rebuild) mark[v] = 1;
        else conn_sub(conn + co, cs, pold, w, k, err);
    } else {
        const eoff_t co = conn_off[v], ce = conn_off[v + 1];
        dest_cache[v] = NULL_PART;
        conn_add<false>(conn + co, &conn_size[v], (int32_t)(ce - co), pnew, w, err);
    }
}

// A neighbour of degree > BIG_DEG (hub[v]; hub null: the level has none) is
// left to k_pull_hubs, which takes its table update and its share of the cut
// change; unless every hub row is scanned there (pull_all), it is flagged.
template <bool ADD>
__device__ inline void update_move(const DGraph& g, part_t pold, part_t pnew, eoff_t rs, eoff_t re, int sub,
                                   int stride, bool rebuild, bool pull_all, const part_t* part, const part_t* dest,
                                   const eoff_t* conn_off, int2* conn, int32_t* conn_size, part_t* dest_cache,
                                   int32_t k, int32_t* err, int32_t* mark, const uint8_t* hub, uint8_t* hub_dirty,
                                   const int32_t* stamp, int32_t gen, int64_t& cc) {
    for (eoff_t j = rs + sub; j < re; j += stride) {
        const vid_t v = g.col[j];
        const int32_t w = g.ew[j];
        if (hub && hub[v]) {
            if (!ADD && !pull_all) hub_dirty[v] = 1;
            continue;
        }
        update_edge<ADD>(v, w, pold, pnew, rebuild, part, dest, conn_off, conn, conn_size, dest_cache, k, err, mark,
                         stamp, gen, cc);
    }
}

// The moves of a step, in two passes (jet_refiner.hpp:905-955 and
// update_small/update_large, :785-884). A move v goes from part[v] to dest[v];
// the producers of the move list stamp each listed vertex with the step's
// generation, so the new part of any vertex u is dest[u] when stamp[u] == gen
// and part[u] otherwise, before part[] changes.
// ADD == false (first pass): part-size deltas of the moves, the moved
// vertices' cached destinations cleared, the whole cut change (for each edge
// (v, u) of a moved v: w * ([p(u) == new] - [p(u) == old]) with the parts
// before and after the step, the reference's table lookups before and after
// the updates), and the old part's connectivity subtracted from each
// neighbour's table, or, when the tables are rebuilt instead (update_large),
// the neighbours marked; each move's record for the second pass.
// ADD == true (second pass): part[v] = new part and the new part's
// connectivity added (unless rebuilding); workgroup 0 only publishes the
// step, so that its chain of loads does not add to a chain of move updates.
// Each kernel loads the deferral flag, the move counts and its first list
// entry together. G lanes stride the edges of one move.
template <bool ADD, int G>
__global__ void __launch_bounds__(256)
    k_update_small(DGraph g, const vid_t* moves, MoveRec* rec, int32_t* mc, vid_t nmax, part_t* part,
                   const part_t* dest, const eoff_t* conn_off, int2* conn, int32_t* conn_size, part_t* dest_cache,
                   int32_t k, int32_t* err, int32_t* mark, const uint8_t* hub, uint8_t* hub_dirty,
                   const int32_t* deferred, const int32_t* stamp, int32_t gen, unsigned long long* sizes,
                   int64_t* partials, uint32_t* bits, int2* moved, Publish pb, RebalPrep prep) {
    __shared__ int64_t red[256 / WAVE];
    __shared__ int32_t ws[ADD ? 256 / WAVE + 1 : 1];
    __shared__ unsigned long long ls[ADD ? 1 : LDS_K];
    const int sub = threadIdx.x & (G - 1);
    // the second pass's move workgroups are 1 .. gridDim.x - 1
    const int64_t blk = ADD ? (int64_t)blockIdx.x - 1 : (int64_t)blockIdx.x;
    const int64_t nblk = ADD ? (int64_t)gridDim.x - 1 : (int64_t)gridDim.x;
    const int64_t gstride = (nblk * blockDim.x) / G;
    const int64_t x0 = ADD && blockIdx.x == 0 ? nmax : (blk * blockDim.x + threadIdx.x) / G;
    const bool have0 = x0 < nmax;
    const vid_t i0 = !ADD && have0 ? moves[x0] : 0;
    MoveRec r0{};
    if (ADD && have0) r0 = rec[x0];
    const int32_t dfr = *deferred;
    const int32_t ns = mc[2], nbig = mc[3];
    // the second pass's workgroup 0 publishes the step (the first pass, which
    // completes the results, has finished)
    if (ADD && blockIdx.x == 0) {
        // the first pass's size deltas (every copy complete: that pass has
        // finished); no other kernel of this pass touches the sizes
        fold_size_copies(pb);
        publish_step(pb, dfr != 0, red);
        // then the next rebalancing step's start (its kernels run after this one)
        if (!dfr && prep.buckets)
            rebalance_prep_block(pb.sizes, pb.k, prep.max_dest, prep.strong != 0, prep.undersized, prep.misc,
                                 prep.acc, prep.evict_adjust, red, ws);
        return;
    }
    if (dfr) return;
    if (ADD && prep.buckets) {
        // the move workgroups zero the next rebalancing step's bucket sums (the
        // current step's readers have all run before the first pass)
        for (int64_t i = (blk * blockDim.x) + threadIdx.x; i < prep.nb; i += nblk * blockDim.x) prep.buckets[i] = 0;
    }
    const bool rebuild = ns + nbig > g.n / 10;  // jet_refiner.hpp:933
    const bool pull_all = ns + nbig > g.n / PULL_ALL_DIV;
    if (!ADD && rebuild && blockIdx.x == 0 && threadIdx.x == 0) mc[6] = 1;  // the tables are to be rebuilt
    const bool lds = !ADD && k <= LDS_K;
    if (lds) {
        for (int t = threadIdx.x; t < k; t += blockDim.x) ls[t] = 0;
        __syncthreads();
    }
    int64_t cc = 0;
    for (int64_t x = x0; x < ns; x += gstride) {
        if (ADD) {
            const MoveRec r = x == x0 ? r0 : rec[x];
            if (sub == 0) {
                part[r.v] = r.pnew;
                if (bits) bits[r.v >> 5] = 0;
            }
            if (rebuild) continue;
            update_move<true>(g, 0, r.pnew, r.rs, r.rs + r.deg, sub, G, false, pull_all, part, dest, conn_off, conn,
                              conn_size, dest_cache, k, err, mark, hub, hub_dirty, stamp, gen, cc);
        } else {
            const vid_t i = x == x0 ? i0 : moves[x];
            const part_t pold = part[i], pnew = dest[i];
            const eoff_t rs = g.rowptr[i], re = g.rowptr[i + 1];
            if (sub == 0) {
                dest_cache[i] = NULL_PART;
                if (bits) {
                    atomicOr(&bits[i >> 5], 1u << (i & 31));
                    moved[i] = make_int2(pold, pnew);
                }
                rec[x] = MoveRec{rs, (int32_t)(re - rs), i, pnew, 0};
                const unsigned long long w = (unsigned long long)g.vw[i];
                if (lds) {
                    atomicAdd(&ls[pold], (unsigned long long)(-(long long)w));
                    atomicAdd(&ls[pnew], w);
                } else {
                    atomicAdd(&sizes[pold], (unsigned long long)(-(long long)w));
                    atomicAdd(&sizes[pnew], w);
                }
            }
            update_move<false>(g, pold, pnew, rs, re, sub, G, rebuild, pull_all, part, dest, conn_off, conn,
                               conn_size, dest_cache, k, err, mark, hub, hub_dirty, stamp, gen, cc);
        }
    }
    if (!ADD) {
        add_cut_part2(partials, cc, red);
        if (lds) {
            __syncthreads();
            unsigned long long* dst =
                pb.ncopies > 0 ? pb.copies + (int64_t)(blockIdx.x % (uint32_t)pb.ncopies) * k : sizes;
            for (int t = threadIdx.x; t < k; t += blockDim.x)
                if (ls[t]) atomicAdd(&dst[t], ls[t]);
        }
    }
}

// The same for the moves of degree > BIG_DEG (the back of the list): a wave
// per move, UB_UNROLL edges per lane in flight. The rows of more than long_deg
// edges are left to a second loop over the level's row slices (k_row_slices),
// a wave per slice whose row moves, so that no chain of updates is longer than
// SLICE_EDGES / 64 edges.
// A workgroup per long row left chains of hundreds of table updates per lane
// for the longest ones: on R-MAT 22's level of 756,505 vertices a second pass
// that moves them took 4.7 ms, with the slices and an insertion that starts at
// the first free slot seen 2.1 (the level 166 ms, now 130).
//
// Bound: chains of table probes. Of a moved row's neighbours a quarter are no
// hubs, so the edges that do need an update are collected in a queue per wave
// and taken 64 at a time: lanes without work cost as much as the others. The
// part-size deltas meet in LDS first: two atomics per move on k addresses were
// 1.6 ms of a first pass that moves a tenth of 4,194,304 vertices. Averages
// per pass before and now: first 577 and 235 us there, 233 and 143 at 756,505
// vertices; second 293 and 184, 444 and 136.
constexpr int UB_BLOCK = 1024;
constexpr int UB_UNROLL = 4;
template <bool ADD>
__global__ void __launch_bounds__(UB_BLOCK)
    k_update_big(DGraph g, const vid_t* moves, MoveRec* rec, const int32_t* mc, vid_t nmax, part_t* part,
                 const part_t* dest, const eoff_t* conn_off, int2* conn, int32_t* conn_size, part_t* dest_cache,
                 int32_t k, int32_t* err, int32_t* mark, const uint8_t* hub, uint8_t* hub_dirty,
                 const int32_t* deferred, const int32_t* stamp, int32_t gen, unsigned long long* sizes,
                 int64_t* partials, uint32_t* bits, int2* moved, int32_t long_deg, const int2* slices, int32_t nslices,
                 unsigned long long* copies, int32_t ncopies) {
    __shared__ int4 queues[UB_BLOCK / WAVE][2 * WAVE];
    __shared__ unsigned long long ls[ADD ? 1 : LDS_K];
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = threadIdx.x / WAVE;
    constexpr int WAVES = UB_BLOCK / WAVE;
    const int32_t dfr = *deferred;
    const int32_t ns = mc[2], nb = mc[3];
    if (dfr || nb == 0) return;
    const bool rebuild = ns + nb > g.n / 10;  // jet_refiner.hpp:933
    const bool pull_all = ns + nb > g.n / PULL_ALL_DIV;
    const bool lds = !ADD && k <= LDS_K;
    if (lds) {
        for (int t = threadIdx.x; t < k; t += UB_BLOCK) ls[t] = 0;
        __syncthreads();
    }
    int64_t cc = 0;
    // the wave's queue of edges to neighbours that are no hubs: (neighbour,
    // weight, old part, new part)
    int4* queue = queues[wv];
    int32_t nq = 0;
    auto drain = [&](int32_t c) {  // the last c <= WAVE entries
        wave_sync();
        nq -= c;
        if (lane < c) {
            const int4 e = queue[nq + lane];
            update_edge<ADD>(e.x, e.y, e.z, e.w, rebuild, part, dest, conn_off, conn, conn_size, dest_cache, k, err,
                             mark, stamp, gen, cc);
        }
        wave_sync();
    };
    auto edges = [&](part_t pold, part_t pnew, eoff_t rs, eoff_t re) {
        for (eoff_t b0 = rs; b0 < re; b0 += (eoff_t)UB_UNROLL * WAVE) {
            vid_t u[UB_UNROLL];
            uint8_t h[UB_UNROLL];
            int32_t w[UB_UNROLL];
#pragma unroll
            for (int q = 0; q < UB_UNROLL; q++) {
                const eoff_t j = b0 + (eoff_t)q * WAVE + lane;
                u[q] = j < re ? g.col[j] : -1;
                w[q] = j < re ? g.ew[j] : 0;
            }
#pragma unroll
            for (int q = 0; q < UB_UNROLL; q++) h[q] = u[q] >= 0 && hub ? hub[u[q]] : 0;
#pragma unroll
            for (int q = 0; q < UB_UNROLL; q++) {
                if (!ADD && !pull_all && h[q]) hub_dirty[u[q]] = 1;
                const bool in = u[q] >= 0 && !h[q];
                const uint64_t mk = __ballot(in);
                if (in) queue[nq + (int32_t)__popcll(mk & ((1ull << lane) - 1ull))] = make_int4(u[q], w[q], pold, pnew);
                nq += (int32_t)__popcll(mk);
                if (nq >= WAVE) drain(WAVE);
            }
        }
    };
    // consecutive moves, and consecutive slices of a row, go to different workgroups
    const int64_t first = (int64_t)wv * gridDim.x + blockIdx.x, stride = (int64_t)gridDim.x * WAVES;
    for (int64_t x = first; x < nb; x += stride) {
        const int64_t at = nmax - 1 - x;
        if (ADD) {
            const MoveRec r = rec[at];
            if (lane == 0) {
                part[r.v] = r.pnew;
                if (bits) bits[r.v >> 5] = 0;
            }
            if (!rebuild && r.deg <= long_deg) edges(0, r.pnew, r.rs, r.rs + r.deg);
        } else {
            const vid_t i = moves[at];
            const part_t pold = part[i], pnew = dest[i];
            const eoff_t rs = g.rowptr[i], re = g.rowptr[i + 1];
            if (lane == 0) {
                dest_cache[i] = NULL_PART;
                if (bits) {
                    atomicOr(&bits[i >> 5], 1u << (i & 31));
                    moved[i] = make_int2(pold, pnew);
                }
                rec[at] = MoveRec{rs, (int32_t)(re - rs), i, pnew, 0};
                const unsigned long long w = (unsigned long long)g.vw[i];
                if (lds) {
                    atomicAdd(&ls[pold], (unsigned long long)(-(long long)w));
                    atomicAdd(&ls[pnew], w);
                } else {
                    atomicAdd(&sizes[pold], (unsigned long long)(-(long long)w));
                    atomicAdd(&sizes[pnew], w);
                }
            }
            if (re - rs <= long_deg) edges(pold, pnew, rs, re);
        }
    }
    if (!(ADD && rebuild))
        for (int64_t x = first; x < nslices; x += stride) {
            const int2 sl = slices[x];
            if (stamp[sl.x] != gen) continue;
            const eoff_t rs = g.rowptr[sl.x] + (eoff_t)sl.y * SLICE_EDGES;
            const eoff_t re = min(g.rowptr[sl.x + 1], rs + (eoff_t)SLICE_EDGES);
            edges(ADD ? 0 : part[sl.x], dest[sl.x], rs, re);
        }
    if (nq > 0) drain(nq);
    if (!ADD) {
        cc = wave_reduce_sum(cc);
        if (lane == 0 && cc)
            atomicAdd((unsigned long long*)&partials[(int64_t)(blockIdx.x % PUB_GROUPS) * PUB_STRIDE],
                      (unsigned long long)cc);
        if (lds) {
            __syncthreads();
            unsigned long long* dst = ncopies > 0 ? copies + (int64_t)(blockIdx.x % (uint32_t)ncopies) * k : sizes;
            for (int t = threadIdx.x; t < k; t += UB_BLOCK)
                if (ls[t]) atomicAdd(&dst[t], ls[t]);
        }
    }
}

// The step's effect on the rows of degree > BIG_DEG ("hubs": the
// workgroup-built tier and the pull_mid rows), one kernel between the two
// passes: a wave per row (a workgroup per row of the workgroup-built tier)
// scans the row for neighbours that move and adds their share of the cut
// change (the same term the first pass adds for its neighbours, seen from the
// other end of the edge). The row's table is held dense in LDS, connectivity
// by part, so a moved neighbour costs two LDS adds; when the scan has found
// one, the table is written back in increasing part id. It has the content
// and the size that per-edge pushes, subtractions before additions, leave:
// in a table of fewer than k slots a part whose connectivity reaches 0 is
// dropped (jet_refiner.hpp:806-810) and new parts take the free slots before
// the table grows (:828-884); a table of k slots keeps its zero entries.
// Nothing looks a hub row's part up by its slot: select kernels read all
// slots, and only this kernel and the builds write them. When the step
// rebuilds the tables (update_large), the rows with a moved neighbour are
// marked instead.
//
// Bound: the scan streams 4 bytes per edge; which neighbours move is a bit
// per vertex, set by the first pass and cleared by the second, which every
// workgroup holds in LDS (EXACT), so an edge costs an LDS read instead of a
// gather of the generation stamp from L2. On levels of more vertices than
// PH_BITS_MAX bytes hold, an LDS bit stands for 2^shift consecutive vertices
// and only the neighbours whose bit is set look their own bit up in memory
// (n / 8 bytes, resident in L2). Two workgroups fit a CU. Probing and
// updating the hashed table per moved neighbour instead (staged in LDS too)
// was bound by its instructions, a few lanes of a wave active in each.
// R-MAT 22 (k = 256), averages per step: two scans per step with global
// tables 1.36 ms in four launches, one scan probing hashed LDS tables 2.4 ms,
// this kernel 0.32 ms on the levels of up to 438,484 vertices and 0.67 ms
// above (0.90 ms with the stamps gathered there). Those were with one
// workgroup of 80 registers a thread on a CU; with the row's state in scalar
// registers two fit (0.37 and 0.50 ms), and with a moved neighbour's two parts
// in one 8-byte word, written by the first pass, 0.30 and 0.43 ms.
// Steps that move few vertices scan only the rows that the first pass
// flagged; from n / PULL_ALL_DIV moves on, about a third of the rows of
// average degree 190 have a moved neighbour and flagging costs a store per
// edge, so every hub row is scanned.
constexpr int PH_WAVES_MAX = 16;
constexpr int PH_UNROLL = 4;
constexpr size_t PH_BITS_MAX = 56 * 1024;
constexpr size_t PH_LDS_MAX = 96 * 1024;  // tables (at most 34 KB) and bits

// LDS words of one dense table: k connectivities, then a bit per part (the
// part has a slot).
__host__ __device__ inline int32_t ph_table_words(int32_t k) { return k + (k + 31) / 32; }

// Loads the row's table (cap slots at conn) into the dense table, which is
// all zero; lanes start, start + stride, ...
__device__ inline void ph_load(const int2* conn, int32_t cap, int32_t k, int32_t* val, int start, int stride) {
    uint32_t* has = reinterpret_cast<uint32_t*>(val + k);
    for (int32_t q = start; q < cap; q += stride) {
        const int2 e = conn[q];
        if (e.x < 0) continue;
        val[e.x] = e.y;
        atomicOr(&has[e.x >> 5], 1u << (e.x & 31));
    }
}

// Writes the dense table back as the row's table of vsz slots (a wave), and
// zeroes it; returns the new size.
__device__ inline int32_t ph_store(int2* conn, int32_t cap, int32_t vsz, int32_t k, int32_t* val, int lane,
                                   int32_t* err) {
    uint32_t* has = reinterpret_cast<uint32_t*>(val + k);
    int32_t used = 0;
    for (int32_t p0 = 0; p0 < k; p0 += WAVE) {
        const int32_t p = p0 + lane;
        const int32_t y = p < k ? val[p] : 0;
        const bool keep = p < k && (y != 0 || (vsz == k && ((has[p >> 5] >> (p & 31)) & 1u)));
        if (y < 0) atomicOr(err, 1);
        const uint64_t mk = __ballot(keep);
        const int32_t at = used + (int32_t)__popcll(mk & ((1ull << lane) - 1ull));
        if (keep) {
            if (at < cap) conn[at] = make_int2(p, y);
            else atomicOr(err, 2);
        }
        if (p < k) val[p] = 0;
        used += (int32_t)__popcll(mk);
    }
    wave_sync();  // the presence bits are read before they are cleared
    for (int32_t q = lane; q < (k + 31) / 32; q += WAVE) has[q] = 0;
    for (int32_t q = used + lane; q < vsz; q += WAVE) conn[q] = make_int2(NULL_PART, 0);
    return used > vsz ? min(used, cap) : vsz;
}

template <bool EXACT>
__global__ void __launch_bounds__(PH_WAVES_MAX* WAVE, 8)
    k_pull_hubs(DGraph g, const vid_t* big, int32_t nbig, const vid_t* mid, int32_t nmid, const int32_t* mc,
                const uint32_t* bits, int32_t shift, const int2* parts, uint8_t* hub_dirty, const part_t* part,
                const part_t* dest, const eoff_t* conn_off, int2* conn, int32_t* conn_size, part_t* dest_cache,
                int32_t k, int32_t* err, int32_t* mark, const int32_t* deferred, int64_t* partials) {
    extern __shared__ int32_t ph_lds[];  // a dense table per wave, then the bits
    if (*deferred) return;
    const int32_t nm = mc[2] + mc[3];
    if (nm == 0) return;
    const bool rebuild = nm > g.n / 10;  // jet_refiner.hpp:933
    const bool all = nm > g.n / PULL_ALL_DIV;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);  // the rows' state in scalar registers
    const int nwv = blockDim.x / WAVE;
    const int32_t tw = ph_table_words(k);
    uint32_t* lbits = reinterpret_cast<uint32_t*>(ph_lds + (size_t)nwv * tw);
    for (int32_t t = threadIdx.x; t < nwv * tw; t += blockDim.x) ph_lds[t] = 0;
    const int32_t words = (g.n + 31) >> 5;
    if (EXACT) {
        for (int32_t t = threadIdx.x; t < words; t += blockDim.x) lbits[t] = bits[t];
    } else {
        for (int32_t t = threadIdx.x; t < (int32_t)(((int64_t)g.n + (32ll << shift) - 1) >> (5 + shift));
             t += blockDim.x)
            lbits[t] = 0;
        __syncthreads();
        const uint32_t group = shift >= 5 ? ~0u : (1u << (1 << shift)) - 1u;
        for (int32_t t = threadIdx.x; t < words; t += blockDim.x) {
            const uint32_t x = bits[t];
            if (x == 0) continue;
            uint32_t y = 0;  // the word's groups with a bit set, from its group's place in the LDS word
            const int32_t g0 = shift >= 5 ? t >> (shift - 5) : t << (5 - shift);
            for (int32_t q = 0; q < (shift >= 5 ? 1 : 32 >> shift); q++)
                if ((x >> (q << shift)) & group) y |= 1u << q;
            atomicOr(&lbits[g0 >> 5], y << (g0 & 31));
        }
    }
    __syncthreads();
    auto moved = [&](vid_t v) -> bool {
        if (EXACT) return ((lbits[v >> 5] >> (v & 31)) & 1u) != 0;
        return ((lbits[v >> (5 + shift)] >> ((v >> shift) & 31)) & 1u) != 0 && ((bits[v >> 5] >> (v & 31)) & 1u) != 0;
    };
    int64_t cc = 0;
    // the row's edges rs + sub + q * stride by this thread, PH_UNROLL at a
    // time; first() runs before the first moved neighbour of a round (of any
    // lane of the wave) is added to val. Returns whether one was found.
    auto scan = [&](eoff_t rs, eoff_t re, int sub, int stride, part_t pu, part_t nu, int32_t* val, auto&& first) {
        bool any = false;
        const vid_t* col = g.col + rs;
        const int32_t* ew = g.ew + rs;
        const uint32_t deg = (uint32_t)(re - rs);
        for (uint32_t b0 = 0; b0 < deg; b0 += PH_UNROLL * stride) {
            vid_t v[PH_UNROLL];
#pragma unroll
            for (int q = 0; q < PH_UNROLL; q++) {
                const uint32_t j = b0 + q * stride + sub;
                v[q] = j < deg ? col[j] : -1;
            }
            uint32_t hits = 0;
#pragma unroll
            for (int q = 0; q < PH_UNROLL; q++)
                if (v[q] >= 0 && moved(v[q])) hits |= 1u << q;
            if (__ballot(hits != 0) == 0) continue;
            int32_t w[PH_UNROLL];
            part_t po[PH_UNROLL], pn[PH_UNROLL];
#pragma unroll
            for (int q = 0; q < PH_UNROLL; q++) {
                const bool h = (hits >> q) & 1u;
                w[q] = h ? ew[b0 + q * stride + sub] : 0;
                const int2 p = h ? parts[v[q]] : make_int2(0, 0);
                po[q] = p.x;
                pn[q] = p.y;
            }
            if (!any) first();
            any = true;
#pragma unroll
            for (int q = 0; q < PH_UNROLL; q++) {
                if (!((hits >> q) & 1u)) continue;
                cc += (int64_t)w[q] * ((pu == pn[q] ? 1 : 0) - (pu == po[q] ? 1 : 0) + (nu == pn[q] ? 1 : 0) -
                                       (nu == po[q] ? 1 : 0));
                if (!rebuild) {
                    atomicAdd(&val[po[q]], -w[q]);
                    atomicAdd(&val[pn[q]], w[q]);
                }
            }
        }
        return any;
    };
    // rows of the workgroup-built tier first: they are the longest
    for (int32_t r = blockIdx.x; r < nbig; r += gridDim.x) {
        const vid_t u = big[r];
        if (!all && !hub_dirty[u]) continue;  // the same for every thread
        const eoff_t rs = g.rowptr[u], re = g.rowptr[u + 1];
        const eoff_t co = conn_off[u];
        const int32_t cap = (int32_t)(conn_off[u + 1] - co);
        const int32_t vsz = conn_size[u];
        const part_t pu = part[u], nu = moved(u) ? dest[u] : pu;
        int32_t* val = ph_lds;
        if (!rebuild) ph_load(conn + co, cap, k, val, threadIdx.x, blockDim.x);
        __syncthreads();
        const int any = __syncthreads_or(scan(rs, re, threadIdx.x, blockDim.x, pu, nu, val, [] {}) ? 1 : 0);
        if (wv == 0) {
            // an unchanged row's table is written back as it was (the dense
            // table has to be zero again)
            int32_t sz = vsz;
            if (!rebuild) sz = ph_store(conn + co, cap, vsz, k, val, lane, err);
            if (lane == 0) {
                if (any) {
                    if (rebuild) {
                        mark[u] = 1;
                    } else {
                        conn_size[u] = sz;
                        dest_cache[u] = NULL_PART;
                    }
                }
                if (!all) hub_dirty[u] = 0;
            }
        }
        __syncthreads();
    }
    int32_t* val = ph_lds + (size_t)wv * tw;
    for (int32_t r = blockIdx.x * nwv + wv; r < nmid; r += (int32_t)gridDim.x * nwv) {
        const vid_t u = mid[r];
        if (!all && !hub_dirty[u]) continue;
        const eoff_t rs = g.rowptr[u], re = g.rowptr[u + 1];
        const eoff_t co = conn_off[u];
        const int32_t cap = (int32_t)(conn_off[u + 1] - co);
        const int32_t vsz = conn_size[u];
        const part_t pu = part[u], du = dest[u];
        const part_t nu = moved(u) ? du : pu;
        const bool any = scan(rs, re, lane, WAVE, pu, nu, val, [&] {
            if (!rebuild) {
                ph_load(conn + co, cap, k, val, lane, WAVE);
                wave_sync();
            }
        });
        int32_t sz = vsz;
        if (any && !rebuild) {
            wave_sync();
            sz = ph_store(conn + co, cap, vsz, k, val, lane, err);
        }
        if (lane == 0) {
            if (any) {
                if (rebuild) {
                    mark[u] = 1;
                } else {
                    conn_size[u] = sz;
                    dest_cache[u] = NULL_PART;
                }
            }
            if (!all) hub_dirty[u] = 0;
        }
        wave_sync();  // the dense table is zero before the next row
    }
    cc = wave_reduce_sum(cc);
    if (lane == 0 && cc)
        atomicAdd((unsigned long long*)&partials[(int64_t)(blockIdx.x % PUB_GROUPS) * PUB_STRIDE],
                  (unsigned long long)cc);
}

// ---------------------------------------------------------------- rebalancing
// Rebalancer minibuckets (jet_refiner.hpp:359-412, :449-481, :632-643).
// Bucket sums are order-free, so they are accumulated with atomics and
// scanned. A vertex is evicted when pos + off[b] - off[begin_p] < limit_p,
// where pos is the weight of same-bucket candidates with smaller id. Whole
// buckets below a part's limit are decided without pos; only the members of
// buckets that straddle a limit (or, for the strong rebalancer, every bucket
// below it, whose scores feed the destination chunks) are ranked by id.

// Zeroes the bucket arrays and the next iteration's counters; workgroup 0
// also builds the undersized-part list (weak, jet_refiner.hpp:578-591) or
// the largest receiver capacity (strong, :440-448) and clears the eviction
// adjustments.
__global__ void __launch_bounds__(256)
    k_reset_buckets(int64_t* buckets, int64_t nb, int32_t* next_counters, const int64_t* sizes,
                    int32_t k, int64_t max_dest, int strong, part_t* undersized, int32_t* misc, int64_t* acc,
                    int64_t* evict_adjust) {
    FOR_THREAD(i, nb) buckets[i] = 0;
    if (blockIdx.x != 0) return;
    if (threadIdx.x < 8) next_counters[threadIdx.x] = 0;
    __shared__ int32_t ws[256 / WAVE + 1];
    __shared__ int64_t red[256 / WAVE];
    rebalance_prep_block(sizes, k, max_dest, strong != 0, undersized, misc, acc, evict_adjust, red, ws);
}

// Per-workgroup LDS map of bucket sums (a workgroup takes a contiguous range
// of vertices, and consecutive vertices share few buckets); overflow goes
// straight to global atomics.
constexpr int BH_SLOTS = 1024;

struct BucketMap {
    int32_t* key;
    unsigned long long* val;
    __device__ void init() {
        for (int t = threadIdx.x; t < BH_SLOTS; t += blockDim.x) {
            key[t] = -1;
            val[t] = 0;
        }
        __syncthreads();
    }
    __device__ void add(int32_t b, unsigned long long w, unsigned long long* global) {
        uint32_t h = ((uint32_t)b * 0x9E3779B1u) >> 22;
        int32_t slot = -1;
        for (int probe = 0; probe < 16; probe++) {
            int32_t k = key[h];
            if (k == -1) {
                int32_t old = atomicCAS(&key[h], -1, b);
                if (old == -1 || old == b) {
                    slot = (int32_t)h;
                    break;
                }
            } else if (k == b) {
                slot = (int32_t)h;
                break;
            }
            h = (h + 1) & (BH_SLOTS - 1);
        }
        // distinct scopes keep the LDS add and the global fallback apart (one
        // flat atomic for both would serve the common LDS case slowly)
        if (slot >= 0) __hip_atomic_fetch_add(&val[slot], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else atomicAdd(&global[b], w);
    }
    __device__ void flush(unsigned long long* global) {
        __syncthreads();
        for (int t = threadIdx.x; t < BH_SLOTS; t += blockDim.x)
            if (key[t] != -1) atomicAdd(&global[key[t]], val[t]);
    }
};

// The select kernels' workgroups flush their bucket maps into `copies`
// copies of the bucket array (workgroup b into copy b mod copies), so that
// fewer workgroups' atomics meet on one line of it; k_sum_bucket_copies folds
// copies 1.. into copy 0 (the bucket array itself) and clears them.
constexpr int BUCKET_COPIES_MAX = 16;
constexpr int64_t BUCKET_COPIES_BYTES = 64ll << 20;

__device__ inline unsigned long long* bucket_copy(unsigned long long* buckets, unsigned long long* extra,
                                                  int32_t copies, int64_t stride) {
    const int32_t c = (int32_t)(blockIdx.x % (uint32_t)copies);
    return c == 0 ? buckets : extra + (int64_t)(c - 1) * stride;
}

__global__ void k_sum_bucket_copies(int64_t* buckets, int64_t* extra, int32_t copies, int64_t nb, int64_t stride) {
    FOR_THREAD(j, nb) {
        int64_t sum = buckets[j];
        for (int32_t c0 = 0; c0 < copies - 1; c0 += 8) {
            int64_t v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = c0 + u < copies - 1 ? extra[(int64_t)(c0 + u) * stride + j] : 0;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                sum += v[u];
                if (v[u]) extra[(int64_t)(c0 + u) * stride + j] = 0;
            }
        }
        buckets[j] = sum;
    }
}

// Part sizes of the select kernels: staged in LDS when k <= SEL_LDS_K (each
// table slot's destination check is then an LDS read, not a dependent global
// load), read from global memory otherwise.
constexpr int SEL_LDS_K = 1024;

constexpr int SEL_BLOCK_MAX = 512;  // select kernels: 128 threads, 512 on large levels

template <bool LDS>
struct PartSizes {
    const int64_t* global;
    int64_t* lds;
    __device__ void stage(int32_t k) {
        if (LDS)
            for (int32_t t = threadIdx.x; t < k; t += blockDim.x) lds[t] = global[t];
    }
    __device__ int64_t operator[](int32_t p) const { return LDS ? lds[p] : global[p]; }
};

// jet_refiner.hpp:592-643: destination and bucket of each vertex of an
// oversized part.
template <bool LDS>
__global__ void __launch_bounds__(SEL_BLOCK_MAX)
    k_weak_select(DGraph g, const part_t* part, const int64_t* sizes, int32_t k, int64_t size_max, int32_t opt,
                  int64_t max_dest, const part_t* undersized, const int32_t* misc, const eoff_t* conn_off,
                  const int2* conn, const int32_t* conn_size, int32_t sections, part_t* dest, int32_t* bid,
                  unsigned long long* buckets_base, unsigned long long* extra, int32_t copies, int64_t stride,
                  unsigned long long* pc, int32_t* next_counters, BestCopy bc) {
    if (blockIdx.x == 0 && threadIdx.x < 8) next_counters[threadIdx.x] = 0;
    bc.sizes_block0();
    unsigned long long* buckets = bucket_copy(buckets_base, extra, copies, stride);
    __shared__ int32_t bk[BH_SLOTS];
    __shared__ unsigned long long bv[BH_SLOTS];
    __shared__ int64_t ssz[LDS ? SEL_LDS_K : 1];
    PartSizes<LDS> ps{sizes, ssz};
    ps.stage(k);
    BucketMap bm{bk, bv};
    bm.init();
    const int32_t tu = misc[0];
    int64_t n_eval = 0, n_slot = 0;
    // one contiguous range per workgroup (as FOR_BLOCK_RANGE), WS_V of a
    // thread's vertices per pass with their part and table-header loads
    // issued together: the dependent chain part -> header -> slots is paid
    // once per pass, not once per vertex
    constexpr int WS_V = 4;
    const int64_t per_block = ((g.n + gridDim.x - 1) / gridDim.x + blockDim.x - 1) / blockDim.x * blockDim.x;
    const int64_t lo = (int64_t)blockIdx.x * per_block;
    const int64_t hi = min((int64_t)g.n, lo + per_block);
    for (int64_t i0 = lo + threadIdx.x; i0 < hi; i0 += (int64_t)WS_V * blockDim.x) {
        part_t p[WS_V], spare[WS_V];
        wgt_t w[WS_V];
        eoff_t off[WS_V];
        int32_t sz[WS_V];
        int64_t sp[WS_V];
        bool ev[WS_V];
#pragma unroll
        for (int u = 0; u < WS_V; u++) {
            const int64_t i = i0 + (int64_t)u * blockDim.x;
            p[u] = i < hi ? part[i] : 0;
            if (bc.part_out && i < hi) bc.part_out[i] = p[u];
        }
#pragma unroll
        for (int u = 0; u < WS_V; u++) {
            const int64_t i = i0 + (int64_t)u * blockDim.x;
            sp[u] = ps[p[u]];
            const bool over = i < hi && sp[u] > size_max;
            w[u] = over ? g.vw[i] : 0;
            off[u] = over ? conn_off[i] : 0;
            sz[u] = over ? conn_size[i] : 0;
            spare[u] = over && tu > 0 ? undersized[(uint32_t)i % (uint32_t)tu] : p[u];
            ev[u] = over && (double)w[u] < 1.5 * (double)(sp[u] - opt);
        }
#pragma unroll
        for (int u = 0; u < WS_V; u++) {
            const int64_t i = i0 + (int64_t)u * blockDim.x;
            if (i >= hi) continue;
            part_t d = p[u];
            int32_t b = -1;
            if (ev[u]) {
                n_eval++;
                n_slot += sz[u];
                part_t best = p[u];
                int32_t gain = 0, p_gain = 0;
                for_slots(conn + off[u], sz[u], [&](int2 e) {
                    if (e.x > NULL_PART && ps[e.x] < max_dest) {
                        if (e.y > gain) {
                            best = e.x;
                            gain = e.y;
                        } else if (e.y == gain && gain > 0 && e.x < best) {
                            best = e.x;
                        }
                    }
                    if (e.x == p[u]) p_gain = e.y;
                });
                int64_t sv = 0;
                if (gain > 0) {
                    d = best;
                    sv = (int64_t)gain - p_gain;
                } else if (tu > 0) {
                    d = spare[u];
                    sv = -(int64_t)p_gain;
                }
                if (d != p[u]) {
                    int32_t gt = gain_bucket_fast(sv, w[u]);
                    b = (MAX_BUCKETS * p[u] + gt) * sections + (int32_t)((uint32_t)i % (uint32_t)sections);
                    bm.add(b, (unsigned long long)w[u], buckets);
                }
            }
            dest[i] = d;
            bid[i] = b;
        }
    }
    bm.flush(buckets);
    if (pc) {  // counting runs only: evaluated vertices and table slots read
        __shared__ int64_t red[SEL_BLOCK_MAX / WAVE];
        int64_t v2[2] = {n_eval, n_slot};
        for (int q = 0; q < 2; q++) {
            const int64_t v = blockDim.x == SEL_BLOCK_MAX ? block_reduce_sum<int64_t, SEL_BLOCK_MAX>(v2[q], red)
                                                          : block_reduce_sum<int64_t, 128>(v2[q], red);
            if (threadIdx.x == 0 && v) atomicAdd(&pc[q], (unsigned long long)v);
        }
    }
}

// jet_refiner.hpp:449-481.
template <bool LDS, bool LONG>
__global__ void __launch_bounds__(SEL_BLOCK_MAX)
    k_strong_select(DGraph g, const part_t* part, const int64_t* sizes, int32_t k, int64_t size_max, int32_t opt,
                    int64_t max_dest, const int64_t* acc, const eoff_t* conn_off, const int2* conn,
                    const int32_t* conn_size, int32_t sections, int32_t* bid, unsigned long long* buckets_base,
                    unsigned long long* extra, int32_t copies, int64_t stride, int32_t* next_counters,
                    BestCopy bc) {
    if (blockIdx.x == 0 && threadIdx.x < 8) next_counters[threadIdx.x] = 0;
    bc.sizes_block0();
    unsigned long long* buckets = bucket_copy(buckets_base, extra, copies, stride);
    __shared__ int32_t bk[BH_SLOTS];
    __shared__ unsigned long long bv[BH_SLOTS];
    __shared__ int64_t ssz[LDS ? SEL_LDS_K : 1];
    PartSizes<LDS> ps{sizes, ssz};
    ps.stage(k);
    BucketMap bm{bk, bv};
    bm.init();
    const int64_t max_vwgt = acc[3];
    // every lane of a wave takes part in each pass (long tables are shared)
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t per_block = ((g.n + gridDim.x - 1) / gridDim.x + blockDim.x - 1) / blockDim.x * blockDim.x;
    const int64_t lo = (int64_t)blockIdx.x * per_block;
    const int64_t hi = min((int64_t)g.n, lo + per_block);
    for (int64_t b0 = lo; b0 < hi; b0 += blockDim.x) {
        const int64_t i = b0 + threadIdx.x;
        const bool in = i < hi;
        const part_t p = in ? part[i] : 0;
        if (bc.part_out && in) bc.part_out[i] = p;
        int32_t b = -1;
        const int64_t sp = ps[p];
        const bool over = in && sp > size_max;
        const int64_t w = over ? g.vw[i] : 0;
        const eoff_t off = over ? conn_off[i] : 0;
        const int32_t sz = over ? conn_size[i] : 0;
        bool vw_ok = max_vwgt > 0 && w <= 2 * max_vwgt;
        const bool ev = over && vw_ok && w < 2 * (sp - opt);
        const bool lng = LONG && ev && sz > SEL_LONG;
        uint64_t tk = 0, tg = 0;
        int64_t p_gain = 0;
        for_long_rows(lng, [&](int q) {
            const part_t qp = __shfl(p, q, WAVE);
            const int2* tab = conn + (eoff_t)__shfl((int64_t)off, q, WAVE);
            const int32_t qs = __shfl(sz, q, WAVE);
            int64_t x = 0, c = 0, px = 0;
            for (int32_t s = lane; s < qs; s += WAVE) {
                const int2 e = tab[s];
                if (e.x == qp) {
                    px = e.y;
                } else if (e.x > NULL_PART && ps[e.x] < max_dest) {
                    x += e.y;
                    c++;
                }
            }
            x = wave_reduce_sum(x);
            c = wave_reduce_sum(c);
            px = wave_reduce_sum(px);
            if (lane == q) {
                tg = (uint64_t)x;
                tk = (uint64_t)c;
                p_gain = px;
            }
        });
        if (ev) {
            if (!lng) for_slots(conn + off, sz, [&](int2 e) {
                if (e.x == p) {
                    p_gain = e.y;
                } else if (e.x > NULL_PART && ps[e.x] < max_dest) {
                    tg += (uint64_t)e.y;
                    tk += 1;
                }
            });
            if (tk == 0) tk = 1;
            int64_t gain = (int64_t)(tg / tk) - p_gain;
            int64_t vwgt = w < sp - size_max ? w : sp - size_max;
            int32_t gt = gain_bucket_fast(gain, vwgt);
            if (gt < MAX_BUCKETS) {
                b = (MAX_BUCKETS * p + gt) * sections + (int32_t)((uint32_t)i % (uint32_t)sections) + 1;
                bm.add(b, (unsigned long long)w, buckets);
            }
        }
        if (in) bid[i] = b;
    }
    bm.flush(buckets);
}

// off = exclusive scan of the bucket sums. WEAK: evicts whole buckets below the
// limit and sends the members of straddling ones to the ranking list; STRONG:
// sends the members of every bucket below the limit there. All members of a
// bucket share its part and offsets, so each decides for itself. One vertex
// per lane: a lane's loads form one dependent chain (measured 0.4 ms less
// per 128^3 stencil partition than four vertices per lane).
// FUSED (nbk <= FUSE_SCAN_MAX): `off` holds the bucket sums, not their scan;
// every workgroup scans them in LDS (one load round trip instead of a scan
// launch) and workgroup 0 writes the scan to off_out for the ranking and
// destination kernels.
// Whether weak bucket b straddles the eviction limit of a part it holds
// members of: its owner q = b / width (gain buckets 0..49), and part q - 1 when
// b is among q's first `sections` minibuckets (the uncapped gain bucket 50 of
// part q - 1 lands there, jet_refiner.hpp:349-351; for q = k, past the last
// part, only part k - 1 holds it).
__device__ inline bool weak_straddle_of(int32_t b, int32_t q, const int64_t* off, const int64_t* sizes,
                                        int64_t size_max, int64_t width) {
    const int64_t base = off[b] - off[(int64_t)q * width];
    const int64_t limit = sizes[q] - size_max;
    return base < limit && base + (off[b + 1] - off[b]) > limit;
}
__device__ inline bool weak_bucket_straddles(int32_t b, int32_t k, int32_t sections, const int64_t* off,
                                             const int64_t* sizes, int64_t size_max, int64_t width) {
    const int32_t q = (int32_t)(b / width);
    if (q < k && weak_straddle_of(b, q, off, sizes, size_max, width)) return true;
    return q >= 1 && (int64_t)b - (int64_t)q * width < sections &&
           weak_straddle_of(b, q - 1, off, sizes, size_max, width);
}

constexpr int CL_CHW = WAVE;
constexpr int CL_WAVES = 16;  // fewer workgroups appending to the list counters (0.2 ms less than 4)
constexpr int64_t FUSE_SCAN_MAX = 4096;
template <bool STRONG, bool FUSED>
__global__ void __launch_bounds__(CL_WAVES* WAVE)
    k_classify(DGraph g, const part_t* part, const int32_t* bid, const int64_t* off_in, int64_t nbk,
               int64_t* off_out, const int64_t* sizes, int64_t size_max, int64_t width, int32_t k, int32_t sections,
               vid_t* moves, int32_t* counters, vid_t nmax, vid_t* rlist, int32_t* stamp, int32_t gen) {
    constexpr int BLOCK = CL_WAVES * WAVE;
    __shared__ int64_t soff[FUSED ? FUSE_SCAN_MAX : 1];
    __shared__ int64_t sws[BLOCK / WAVE + 1];
    const int64_t* off = off_in;
    if (FUSED) {
        constexpr int PER = (int)(FUSE_SCAN_MAX / BLOCK);
        int64_t loc[PER];
        int64_t sum = 0;
        const int64_t t0 = (int64_t)threadIdx.x * PER;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int64_t v = t0 + j < nbk ? off_in[t0 + j] : 0;
            loc[j] = sum;
            sum += v;
        }
        int64_t tot;
        const int64_t ex = block_excl_scan<int64_t, BLOCK>(sum, tot, sws);
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (t0 + j < nbk) soff[t0 + j] = ex + loc[j];
        __syncthreads();
        if (blockIdx.x == 0)
            for (int64_t t = threadIdx.x; t < nbk; t += BLOCK) off_out[t] = soff[t];
        off = soff;
    }
    __shared__ vid_t sbuf[CL_WAVES * CL_CHW];
    __shared__ vid_t rbuf[CL_WAVES * CL_CHW];
    __shared__ int32_t sh[2 * CL_WAVES + 2];
    __shared__ int32_t rsh[2 * CL_WAVES + 2];
    StagedLists<CL_WAVES, CL_CHW> st(sbuf);
    StagedLists<CL_WAVES, CL_CHW> rt(rbuf);
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t wbase = ((int64_t)blockIdx.x * CL_WAVES + threadIdx.x / WAVE) * CL_CHW;
    for (int32_t o = 0; o < CL_CHW; o += WAVE) {
        int64_t i = wbase + o + lane;
        bool ev = false, rank = false;
        eoff_t deg = 0;
        if (i < g.n) {
            int32_t b = bid[i];
            if (b >= 0) {
                part_t p = part[i];
                int64_t base = off[b] - off[(int64_t)p * width];
                int64_t limit = sizes[p] - size_max;
                int64_t bs = off[b + 1] - off[b];
                if (STRONG) {
                    rank = base < limit;
                } else if (base + bs <= limit) {
                    ev = true;
                    deg = g.rowptr[i + 1] - g.rowptr[i];
                }
                // a weak bucket that straddles its part's limit is ranked
                // with all of its members: bucket 50 of part q shares its
                // index with part q + 1's first gain bucket, and a member's
                // position counts every member of lower id (:363-384)
                if (!STRONG) rank = weak_bucket_straddles(b, k, sections, off, sizes, size_max, width);
            }
        }
        st.push(ev && deg <= BIG_DEG, ev && deg > BIG_DEG, (vid_t)i);
        rt.push(rank, false, (vid_t)i);
    }
    st.flush_stamped(moves, &counters[2], &counters[3], nmax, sh, stamp, gen);
    rt.flush(rlist, &counters[5], &counters[7], g.n, rsh);
}

// Decision for one ranked vertex: pos = weight of same-bucket members with a
// smaller id (of any part). Returns 0 (kept), 1 (evicted, degree <= BIG_DEG) or 2 (evicted,
// larger); the caller appends evicted members to the move list.
template <bool STRONG>
__device__ inline int rank_decide_with(vid_t v, int32_t b, int64_t pos, part_t p, int64_t w, bool big,
                                       const int64_t* off, const int64_t* sizes, int64_t size_max, int64_t width,
                                       int64_t* evict_adjust, int64_t* score, int32_t* stamp, int32_t gen) {
    int64_t base = off[b] - off[(int64_t)p * width];
    int64_t limit = sizes[p] - size_max;
    int64_t bs = off[b + 1] - off[b];
    bool ev = false;
    if (STRONG) {
        if (base < limit && base + pos < limit) {
            ev = true;
            if (base + pos + w >= limit) evict_adjust[p] = base + pos + w;
            score[v] = off[b] + pos;
        }
    } else if (base < limit && base + bs > limit) {
        ev = base + pos < limit;
    }
    if (!ev) return 0;
    stamp[v] = gen;
    return big ? 2 : 1;
}

template <bool STRONG>
__device__ inline int rank_decide(vid_t v, int32_t b, int64_t pos, const part_t* part, const int64_t* off,
                                  const int64_t* sizes, int64_t size_max, int64_t width, const wgt_t* vw,
                                  const eoff_t* rowptr, int64_t* evict_adjust, int64_t* score, int32_t* stamp,
                                  int32_t gen) {
    // the member's part, weight and row are loaded together
    const part_t p = part[v];
    const int64_t w = vw[v];
    const eoff_t deg = rowptr[v + 1] - rowptr[v];
    return rank_decide_with<STRONG>(v, b, pos, p, w, deg > BIG_DEG, off, sizes, size_max, width, evict_adjust, score,
                                    stamp, gen);
}


// The cookie cutter (jet_refiner.hpp:491-518) by one workgroup of BLOCK
// threads: two scans over the parts give each part's eviction adjustment and
// the destination chunk starts; the re-draw counter starts after every
// eviction.
template <int BLOCK>
__device__ inline void cookie_block(int32_t k, int64_t width, const int64_t* off, const int64_t* sizes,
                                    int64_t max_dest, int64_t* evict_adjust, int64_t* evict_start, int64_t* acc,
                                    int64_t* ws) {
    int64_t run = 0, run2 = 0;
    for (int32_t p0 = 0; p0 < k; p0 += BLOCK) {
        int32_t p = p0 + threadIdx.x;
        int64_t add = 0, cap = 0, beg = 0;
        if (p < k) {
            int64_t begin = (int64_t)p * width;
            beg = off[begin];
            add = evict_adjust[p];
            if (add == 0) add = off[begin + width] - beg;
            if (max_dest > sizes[p]) cap = max_dest - sizes[p];
        }
        int64_t t1, t2;
        int64_t e1 = block_excl_scan<int64_t, BLOCK>(add, t1, ws);
        int64_t e2 = block_excl_scan<int64_t, BLOCK>(cap, t2, ws);
        if (p < k) {
            evict_adjust[p] = beg - (run + e1);
            evict_start[p + 1] = run2 + e2 + cap;
        }
        run += t1;
        run2 += t2;
    }
    if (threadIdx.x == 0) {
        acc[3] = run;
        evict_start[0] = 0;
    }
}

// What a strong ranking workgroup also does when it ranks every member
// itself: the cookie cutter (so the step needs no cookie launch).
struct CookieArgs {
    int32_t k;  // 0: not here
    int64_t max_dest;
    int64_t* evict_start;
    int64_t* acc;
};

constexpr int RS_CAP = 8192;
constexpr int RS_BLOCK = 1024;

// Ranks up to RS_CAP members in one workgroup: bitonic sort of
// (bucket << 32 | id) in LDS, prefix of weights, decisions.
template <bool STRONG>
__global__ void __launch_bounds__(RS_BLOCK)
    k_rank_small(const vid_t* rlist, const int32_t* counters, const int32_t* bid, const part_t* part,
                 const int64_t* off, const int64_t* sizes, int64_t size_max, int64_t width, const wgt_t* vw,
                 const eoff_t* rowptr, int64_t* evict_adjust, int64_t* score, vid_t* moves, int32_t* mcounters,
                 vid_t nmax, int32_t* deferred, int32_t* stamp, int32_t gen, CookieArgs ck) {
    __shared__ uint64_t keys[RS_CAP];
    __shared__ int64_t pre[RS_CAP];
    __shared__ int64_t ws[RS_BLOCK / WAVE + 1];
    __shared__ uint32_t pay_w[RS_BLOCK];
    __shared__ uint32_t pay_p[RS_BLOCK];
    // each thread's first member is loaded together with the count
    const vid_t m0 = (vid_t)threadIdx.x < nmax ? rlist[threadIdx.x] : 0;
    const int32_t R = counters[5];
    if (R > RS_CAP) {
        // too many members for one workgroup: the host ranks them with the
        // radix path after the iteration's sync; until then the iteration's
        // remaining kernels see the flag and do nothing
        if (threadIdx.x == 0) *deferred = 1;
        return;
    }
    uint32_t cap = 1;
    while ((int32_t)cap < R) cap <<= 1;
    if (cap <= RS_BLOCK) {
        // one member per thread, its weight, part and degree class loaded
        // with its bucket and carried through the sort: exchanges within a
        // wave are shuffles, only strides of a wave or more go through LDS
        // (10 barriers instead of 55 for 1024 keys)
        const uint32_t t = threadIdx.x;
        uint64_t key = ~0ull;
        uint32_t pw = 0, pp = 0;  // weight; part | big << 31
        if ((int32_t)t < R) {
            const int32_t bb = bid[m0];
            const wgt_t w0 = vw[m0];
            const part_t p0 = part[m0];
            const eoff_t d0 = rowptr[m0 + 1] - rowptr[m0];
            key = ((uint64_t)(uint32_t)bb << 32) | (uint32_t)m0;
            pw = (uint32_t)w0;
            pp = (uint32_t)p0 | (d0 > BIG_DEG ? 0x80000000u : 0u);
        }
        for (uint32_t size = 2; size <= cap; size <<= 1) {
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                uint64_t other;
                uint32_t opw, opp;
                if (stride >= WAVE) {
                    keys[t] = key;
                    pay_w[t] = pw;
                    pay_p[t] = pp;
                    __syncthreads();
                    other = keys[t ^ stride];
                    opw = pay_w[t ^ stride];
                    opp = pay_p[t ^ stride];
                    __syncthreads();
                } else {
                    const uint32_t lo = __shfl_xor((uint32_t)key, (int)stride, WAVE);
                    const uint32_t hi = __shfl_xor((uint32_t)(key >> 32), (int)stride, WAVE);
                    other = ((uint64_t)hi << 32) | lo;
                    opw = __shfl_xor(pw, (int)stride, WAVE);
                    opp = __shfl_xor(pp, (int)stride, WAVE);
                }
                // ascending blocks keep the smaller key at the lower index
                const bool lower = (t & stride) == 0, up = (t & size) == 0;
                const bool take = (lower == up) ? (other < key) : (other > key);
                if (take) {
                    key = other;
                    pw = opw;
                    pp = opp;
                }
            }
        }
        keys[t] = key;
        int64_t tot;
        const int64_t ex = block_excl_scan<int64_t, RS_BLOCK>((int32_t)t < R ? (int64_t)(int32_t)pw : 0, tot, ws);
        pre[t] = ex;
        __syncthreads();
        if ((int32_t)t < R) {
            const int32_t b = (int32_t)(key >> 32);
            const uint64_t lo_key = (uint64_t)(uint32_t)b << 32;
            int32_t lo = 0, hi = (int32_t)t;
            while (lo < hi) {
                int32_t mid = (lo + hi) >> 1;
                if (keys[mid] < lo_key) lo = mid + 1;
                else hi = mid;
            }
            const vid_t v = (vid_t)(key & 0xffffffffull);
            const int code = rank_decide_with<STRONG>(v, b, pre[t] - pre[lo], (part_t)(pp & 0x7fffffffu),
                                                      (int64_t)(int32_t)pw, (pp >> 31) != 0, off, sizes, size_max,
                                                      width, evict_adjust, score, stamp, gen);
            if (code == 2) moves[nmax - 1 - atomicAdd(&mcounters[3], 1)] = v;
            else if (code == 1) moves[atomicAdd(&mcounters[2], 1)] = v;
        }
        if (STRONG && ck.k > 0) {
            __syncthreads();  // every member's eviction adjustment written
            cookie_block<RS_BLOCK>(ck.k, width, off, sizes, ck.max_dest, evict_adjust, ck.evict_start, ck.acc, ws);
        }
        return;
    } else {
        for (uint32_t t = threadIdx.x; t < cap; t += RS_BLOCK) {
            if ((int32_t)t < R) {
                const vid_t v = t == threadIdx.x ? m0 : rlist[t];
                keys[t] = ((uint64_t)(uint32_t)bid[v] << 32) | (uint32_t)v;
            } else {
                keys[t] = ~0ull;
            }
        }
        for (uint32_t size = 2; size <= cap; size <<= 1) {
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                __syncthreads();
                for (uint32_t t = threadIdx.x; t < cap / 2; t += RS_BLOCK) {
                    uint32_t lo = 2 * t - (t & (stride - 1));
                    uint32_t hi = lo + stride;
                    bool up = (lo & size) == 0;
                    uint64_t x = keys[lo], y = keys[hi];
                    if ((x > y) == up) {
                        keys[lo] = y;
                        keys[hi] = x;
                    }
                }
            }
        }
    }
    __syncthreads();
    // exclusive prefix of weights in sorted order (RS_CAP / RS_BLOCK items per thread)
    constexpr int PER = RS_CAP / RS_BLOCK;
    int64_t loc[PER];
    int64_t sum = 0;
    for (int j = 0; j < PER; j++) {
        int32_t t = threadIdx.x * PER + j;
        int64_t w = t < R ? (int64_t)vw[(vid_t)(keys[t] & 0xffffffffull)] : 0;
        loc[j] = sum;
        sum += w;
    }
    int64_t tot;
    int64_t ex = block_excl_scan<int64_t, RS_BLOCK>(sum, tot, ws);
    for (int j = 0; j < PER; j++) pre[threadIdx.x * PER + j] = ex + loc[j];
    __syncthreads();
    for (int32_t t = threadIdx.x; t < R; t += RS_BLOCK) {
        const uint64_t key = keys[t];
        const int32_t b = (int32_t)(key >> 32);
        const uint64_t lo_key = (uint64_t)(uint32_t)b << 32;
        int32_t lo = 0, hi = t;
        while (lo < hi) {
            int32_t mid = (lo + hi) >> 1;
            if (keys[mid] < lo_key) lo = mid + 1;
            else hi = mid;
        }
        const vid_t v = (vid_t)(key & 0xffffffffull);
        const int code = rank_decide<STRONG>(v, b, pre[t] - pre[lo], part, off, sizes, size_max, width, vw, rowptr,
                                             evict_adjust, score, stamp, gen);
        if (code == 2) moves[nmax - 1 - atomicAdd(&mcounters[3], 1)] = v;
        else if (code == 1) moves[atomicAdd(&mcounters[2], 1)] = v;
    }
    if (STRONG && ck.k > 0) {
        __syncthreads();  // every member's eviction adjustment written
        cookie_block<RS_BLOCK>(ck.k, width, off, sizes, ck.max_dest, evict_adjust, ck.evict_start, ck.acc, ws);
    }
}

__global__ void k_rank_keys(const vid_t* rlist, int32_t R, const int32_t* bid, uint64_t* keys, uint32_t* vals) {
    FOR_THREAD(t, R) {
        vid_t v = rlist[t];
        keys[t] = ((uint64_t)(uint32_t)bid[v] << 32) | (uint32_t)v;
        vals[t] = (uint32_t)v;
    }
}

__global__ void k_rank_weights(int32_t R, const uint32_t* vals, const wgt_t* vw, int64_t* w) {
    FOR_THREAD(t, R) w[t] = vw[vals[t]];
}

template <bool STRONG>
__global__ void k_rank_apply(int32_t R, const uint64_t* keys, const int64_t* pre, const part_t* part,
                             const int64_t* off, const int64_t* sizes, int64_t size_max, int64_t width,
                             const wgt_t* vw, const eoff_t* rowptr, int64_t* evict_adjust, int64_t* score,
                             vid_t* moves, int32_t* mcounters, vid_t nmax, int32_t* stamp, int32_t gen) {
    FOR_THREAD(t, R) {
        uint64_t key = keys[t];
        int32_t b = (int32_t)(key >> 32);
        uint64_t lo_key = (uint64_t)(uint32_t)b << 32;
        int64_t lo = 0, hi = t;
        while (lo < hi) {
            int64_t mid = (lo + hi) >> 1;
            if (keys[mid] < lo_key) lo = mid + 1;
            else hi = mid;
        }
        const vid_t v = (vid_t)(key & 0xffffffffull);
        const int code = rank_decide<STRONG>(v, b, pre[t] - pre[lo], part, off, sizes, size_max, width, vw, rowptr,
                                             evict_adjust, score, stamp, gen);
        if (code == 2) moves[nmax - 1 - atomicAdd(&mcounters[3], 1)] = v;
        else if (code == 1) moves[atomicAdd(&mcounters[2], 1)] = v;
    }
}

// Cookie cutter (jet_refiner.hpp:491-518): per-part eviction totals become a
// global eviction order; receivers get consecutive chunks of capacity. Two
// workgroup scans over the parts.
constexpr int CK_BLOCK = 1024;
__global__ void __launch_bounds__(CK_BLOCK)
    k_cookie(int32_t k, int64_t width, const int64_t* off, const int64_t* sizes, int64_t max_dest,
             int64_t* evict_adjust, int64_t* evict_start, int64_t* acc, const int32_t* deferred) {
    if (*deferred) return;
    __shared__ int64_t ws[CK_BLOCK / WAVE + 1];
    cookie_block<CK_BLOCK>(k, width, off, sizes, max_dest, evict_adjust, evict_start, acc, ws);
}

// Last index q in [lo, k] with evict_start[q] <= s (evict_start is non-decreasing).
__device__ inline int32_t chunk_of(const int64_t* es, int32_t lo, int32_t k, int64_t s) {
    int32_t a = lo, b = k + 1;  // first index with es > s lies in [a, b]
    while (a < b) {
        int32_t mid = (a + b) >> 1;
        if (es[mid] <= s) a = mid + 1;
        else b = mid;
    }
    return a - 1;
}

// jet_refiner.hpp:519-544 without the re-draws, which are queued.
__global__ void k_strong_dest(const vid_t* moves, const int32_t* mc, vid_t nmax, const part_t* part, const wgt_t* vw,
                              const int64_t* evict_adjust, const int64_t* evict_start, int32_t k, int64_t* score,
                              part_t* dest, vid_t* redraw, int32_t* rcount, int32_t rmax,
                              const int32_t* deferred) {
    if (*deferred) return;
    const int32_t ns = mc[2], total = mc[2] + mc[3];
    FOR_THREAD(x, total) {
        vid_t v = list_at(moves, ns, nmax, x);
        part_t pv = part[v];
        int64_t s = score[v] - evict_adjust[pv];
        score[v] = s;
        int32_t q = chunk_of(evict_start, 0, k, s);
        if (q < k && vw[v] / 2 <= evict_start[q + 1] - s) {
            dest[v] = q;
        } else if (q < k) {
            int32_t r = atomicAdd(rcount, 1);
            if (r < rmax) redraw[r] = v;
            dest[v] = pv;
        } else {
            dest[v] = pv;
        }
    }
}

// Re-draws in increasing vertex id, one after another (the counter starts at
// the total eviction weight). The serial walk reads only LDS: the chunk
// starts (k + 1 <= RD_ES_MAX) and, a batch of 256 at a time, the re-drawn
// vertices' scores and weights are staged there first. Up to lds_max (at
// most RD_MAX) re-drawn vertices are sorted by id in LDS; a longer list is
// put in id order in place
// by marking its vertices in `mark` (n entries, all zero between launches)
// and compacting the marks over all vertex ids, clearing them as it goes.
constexpr int RD_MAX = 8192;
constexpr int RD_ES_MAX = 2049;
constexpr int RD_SCAN = 16;  // marks per thread per compaction pass
__global__ void __launch_bounds__(256) k_strong_redraw(vid_t* redraw, const int32_t* rcount, const part_t* part,
                                                       const wgt_t* vw, const int64_t* evict_start, int32_t k,
                                                       const int64_t* score, part_t* dest, int64_t* acc,
                                                       int32_t* mark, vid_t n, int32_t lds_max,
                                                       const int32_t* deferred) {
    __shared__ vid_t ids[RD_MAX];
    __shared__ int64_t es_lds[RD_ES_MAX];
    __shared__ int64_t bscore[256];
    __shared__ wgt_t bw[256];
    __shared__ int64_t red[256 / WAVE + 1];
    if (*deferred) return;
    const int32_t r = rcount[0];
    if (r == 0) return;
    const bool es_in_lds = k + 1 <= RD_ES_MAX;
    if (es_in_lds)
        for (int32_t t = threadIdx.x; t <= k; t += blockDim.x) es_lds[t] = evict_start[t];
    const int64_t* es = es_in_lds ? es_lds : evict_start;
    const vid_t* idp = ids;
    if (r <= lds_max) {
        uint32_t cap = 1;
        while ((int32_t)cap < r) cap <<= 1;
        for (uint32_t t = threadIdx.x; t < cap; t += blockDim.x) ids[t] = (int32_t)t < r ? redraw[t] : ORD_MAX;
        for (uint32_t size = 2; size <= cap; size <<= 1) {
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                __syncthreads();
                for (uint32_t t = threadIdx.x; t < cap / 2; t += blockDim.x) {
                    uint32_t lo = 2 * t - (t & (stride - 1));
                    uint32_t hi = lo + stride;
                    bool up = (lo & size) == 0;
                    vid_t a = ids[lo], b = ids[hi];
                    if ((a > b) == up) {
                        ids[lo] = b;
                        ids[hi] = a;
                    }
                }
            }
        }
    } else {
        // the list's vertices marked, then written back in increasing id
        for (int32_t x = threadIdx.x; x < r; x += blockDim.x) mark[redraw[x]] = 1;
        __threadfence_block();
        __syncthreads();
        int64_t out = 0;
        for (int64_t v0 = 0; v0 < n; v0 += 256 * RD_SCAN) {
            const int64_t t0 = v0 + (int64_t)threadIdx.x * RD_SCAN;
            int32_t f[RD_SCAN];
            int64_t c = 0;
#pragma unroll
            for (int j = 0; j < RD_SCAN; j++) {
                f[j] = t0 + j < n ? mark[t0 + j] : 0;
                c += f[j];
            }
            int64_t tot;
            int64_t at = out + block_excl_scan<int64_t, 256>(c, tot, red);
#pragma unroll
            for (int j = 0; j < RD_SCAN; j++)
                if (f[j]) {
                    redraw[at++] = (vid_t)(t0 + j);
                    mark[t0 + j] = 0;
                }
            out += tot;
        }
        __threadfence_block();
        idp = redraw;
    }
    __syncthreads();
    int64_t counter = acc[3];  // carried by thread 0
    for (int32_t base = 0; base < r; base += 256) {
        const int32_t nb = r - base < 256 ? r - base : 256;
        if ((int32_t)threadIdx.x < nb) {
            const vid_t v = idp[base + threadIdx.x];
            bscore[threadIdx.x] = score[v];
            bw[threadIdx.x] = vw[v];
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int32_t x = 0; x < nb; x++) {
                const vid_t v = idp[base + x];
                const wgt_t wv = bw[x];
                int64_t sc = bscore[x];
                int32_t p = 0;
                bool done = false;
                while (p < k) {
                    p = chunk_of(es, p, k, sc);
                    if (p < k && wv / 2 <= es[p + 1] - sc) {
                        dest[v] = p;
                        done = true;
                        break;
                    } else if (p < k) {
                        sc = counter;
                        counter += wv;
                    }
                }
                if (!done) dest[v] = part[v];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) acc[3] = counter;
}

__global__ void k_collect_moves(const vid_t* moves, const int32_t* mc, vid_t nmax, const part_t* dest, vid_t* out_v,
                                part_t* out_d) {
    const int32_t total = mc[2] + mc[3];
    FOR_THREAD(x, total) {
        vid_t v = list_at(moves, mc[2], nmax, x);
        out_v[x] = v;
        out_d[x] = dest[v];
    }
}

// ---------------------------------------------------------------- host side
static inline int32_t sections_for(vid_t n, int32_t k) {
    int32_t sections = MAX_SECTIONS;
    int32_t section_size = (n + sections * k) / (sections * k);
    if (section_size < 4096) {
        section_size = 4096;
        sections = (n + section_size * k) / (section_size * k);
    }
    return sections;
}

// Lanes per vertex of a list: the average degree rounded up to a power of
// two.
static int lanes_for(double avg) {
    return avg <= 4 ? 4 : avg <= 8 ? 8 : avg <= 16 ? 16 : avg <= 32 ? 32 : 64;
}

// Lanes per candidate in the afterburner: doubled on levels of up to
// SMALL_LEVEL_N vertices, whose few candidates leave the GPU idle otherwise.
// On levels with rows above BIG_DEG edges the average is that of the short
// rows, which these kernels take (R-MAT 22, 4,194,304 vertices: first update
// pass 0.18 -> 0.14 ms, second 0.13 -> 0.09).
// Lanes per move in the update passes: doubled on every level, so that a
// lane's chain of table updates is shorter (each measured 0.5 ms less per
// 128^3 stencil partition; doubling the afterburner's on large levels was
// slower).
static int group_for_avg(const DGraph& g) { return lanes_for(g.n > 0 ? (double)g.m / g.n : 0.0); }
static int group_for_afterburner(const DGraph& g, double avg) {
    const int m = g.n <= tuning().small_level_n ? (int)tuning().ab_lanes_small : 1;
    return std::min(64, m * lanes_for(avg));
}
static int group_for_update(double avg) { return std::min(64, (int)tuning().upd_lanes * lanes_for(avg)); }

// out: the largest degree; small[0], small[1]: the rows of 1 to BIG_DEG edges,
// and a sixteenth of their edges. Few workgroups: atomics on one address take
// some 12 ns each.
constexpr int MD_BLOCK = 1024;
__global__ void __launch_bounds__(MD_BLOCK) k_max_degree(DGraph g, int32_t* out, int32_t* small) {
    __shared__ int32_t red[MD_BLOCK / WAVE];
    int32_t mx = 0, rows = 0, edges = 0;
    FOR_THREAD(i, g.n) {
        int64_t d = g.rowptr[i + 1] - g.rowptr[i];
        if (d > mx) mx = (int32_t)(d > ORD_MAX ? ORD_MAX : d);
        if (d > 0 && d <= BIG_DEG) {
            rows++;
            edges += (int32_t)d;
        }
    }
    mx = block_reduce_max<int32_t, MD_BLOCK>(mx, red);
    if (threadIdx.x == 0 && mx) atomicMax(out, mx);
    rows = block_reduce_sum<int32_t, MD_BLOCK>(rows, red);
    edges = block_reduce_sum<int32_t, MD_BLOCK>(edges, red);
    if (threadIdx.x == 0) {
        atomicAdd(&small[0], rows);
        atomicAdd(&small[1], (edges + 8) / 16);
    }
}

// The refiner's state that starts at a fixed value, filled in one launch (ten
// launches of some 3 us each were a tenth of a small quality call).
struct InitWords {
    struct Seg {
        int32_t* p;
        int32_t v;
        int64_t words;
    } seg[10];
    int count;
};
__global__ void __launch_bounds__(256) k_init_words(InitWords w) {
    for (int q = 0; q < w.count; q++) FOR_THREAD(i, w.seg[q].words) w.seg[q].p[i] = w.seg[q].v;
}

// Dynamic LDS above 64 KB is allowed per kernel and device, once.
static void allow_pull_lds() {
    static std::once_flag once[64];
    static hipError_t rc[64];
    int dev = 0;
    JET_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) throw DeviceError("device index beyond 64");
    std::call_once(once[dev], [&] {
        for (const void* f : {reinterpret_cast<const void*>(&k_pull_hubs<true>),
                              reinterpret_cast<const void*>(&k_pull_hubs<false>)}) {
            rc[dev] = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)PH_LDS_MAX);
            if (rc[dev] != hipSuccess) return;
        }
    });
    JET_HIP(rc[dev]);
}

Refiner::Refiner(Arena& a, hipStream_t s, vid_t n, int64_t m, int64_t cap, const RefineParams& p)
    : a_(a), s_(s), p_(p), nmax_(n) {
    if (p.k < 1 || p.k > MAX_K) throw std::invalid_argument("k out of range");
    if (2 * sizeof(int2) * (size_t)p.k > 65536) {
        // dynamic LDS above 64 KB must be allowed per kernel (gfx950 has 160 KB)
        JET_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_conn_build_block),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)(2 * sizeof(int2) * MAX_K)));
    }
    allow_pull_lds();
    int64_t N = std::max<int64_t>(n, 1);
    conn_off_ = a.alloc<eoff_t>(N + 1);
    conn_size_ = a.alloc<int32_t>(N);
    dest_cache_ = a.alloc<part_t>(N);
    lock_ = a.alloc<int32_t>(N);
    gain_p_ = a.alloc<int32_t>(N);
    pregain_ = a.alloc<int32_t>(N);
    dest_ = a.alloc<part_t>(N);
    bid_ = a.alloc<int32_t>(N);
    cand_ = a.alloc<vid_t>(N);
    moves_ = a.alloc<vid_t>(N);
    mrec_ = a.alloc<MoveRec>(N);
    swap_bit_ = a.alloc<int32_t>(N);
    sval_ = a.alloc<uint32_t>(N);
    vtmp_ = a.alloc<uint32_t>(N);
    prefix_ = a.alloc<int64_t>(N + 1);
    score_ = a.alloc<int64_t>(N);
    cur_part_ = a.alloc<part_t>(N);
    tier_mid_ = a.alloc<vid_t>(N);
    tier_big_ = a.alloc<vid_t>(N);
    hub_ = a.alloc<uint8_t>(N);
    hub_dirty_ = a.alloc<uint8_t>(N);
    pull_mid_ = a.alloc<vid_t>(N);
    stamp_ = a.alloc<int32_t>(N);
    counters_ = a.alloc<int32_t>(32);
    acc_ = a.alloc<int64_t>(8);
    curr_sizes_ = a.alloc<int64_t>(p.k);
    best_sizes_ = a.alloc<int64_t>(p.k);
    evict_adjust_ = a.alloc<int64_t>(p.k);
    evict_start_ = a.alloc<int64_t>(p.k + 1);
    undersized_ = a.alloc<part_t>(p.k);
    misc_ = a.alloc<int32_t>(8);
    redraw_ = a.alloc<vid_t>(N);
    rd_mark_ = a.alloc<int32_t>(N);
    nbuckets_ = (int64_t)MAX_BUCKETS * p.k * sections_for(n, p.k) + MAX_SECTIONS + 4;
    buckets_ = a.alloc<int64_t>(nbuckets_);
    boff_ = a.alloc<int64_t>(std::max<int64_t>(FUSE_SCAN_MAX, nbuckets_));
    ncopies_ = (int32_t)std::max<int64_t>(
        1, std::min<int64_t>(BUCKET_COPIES_MAX, BUCKET_COPIES_BYTES / ((int64_t)sizeof(int64_t) * nbuckets_)));
    bcopies_ = a.alloc<int64_t>(std::max<int64_t>(1, nbuckets_ * (ncopies_ - 1)));
    moved_bits_ = a.alloc<uint32_t>((N + 31) / 32);
    cand_bits_ = a.alloc<uint64_t>((N + WAVE - 1) / WAVE);
    // tables of a level on the kernels (cap slots on the finest) or on a team,
    // whose rows start at their adjacency's offset: at most m slots either way
    conn_ = a.alloc<int2>(std::max<int64_t>({cap, std::min<int64_t>(m, TEAM_MAX_M), 1}));
    team_ctl_ = a.alloc<RefineCtl>(1);
    team_buckets_ = a.alloc<int32_t>(TEAM_MAX_NBK + 1);
    team_rkey_ = a.alloc<uint64_t>(std::min<int64_t>(N, TEAM_MAX_N));
    team_rweight_ = a.alloc<int32_t>(std::min<int64_t>(N, TEAM_MAX_N));
    pub_ = a.alloc<int64_t>((int64_t)PUB_GROUPS * PUB_STRIDE);
    szc_ = a.alloc<int64_t>((int64_t)SIZE_COPIES_MAX * p.k);
    InitWords iw{};
    auto set = [&](void* p, int32_t v, int64_t bytes) { iw.seg[iw.count++] = {static_cast<int32_t*>(p), v, (bytes + 3) / 4}; };
    set(bcopies_, 0, 8 * nbuckets_ * (ncopies_ - 1));
    set(swap_bit_, 0, 4 * N);
    set(rd_mark_, 0, 4 * N);
    set(hub_dirty_, 0, N);
    set(stamp_, -1, 4 * N);
    set(moved_bits_, 0, 4 * ((N + 31) / 32));
    set(counters_, 0, 4 * 32);
    set(acc_, 0, 8 * 8);
    set(pub_, 0, 8 * (int64_t)PUB_GROUPS * PUB_STRIDE);
    set(szc_, 0, 8 * (int64_t)SIZE_COPIES_MAX * p.k);
    int64_t words = 0;
    for (int q = 0; q < iw.count; q++) words = std::max(words, iw.seg[q].words);
    k_init_words<<<grid_for(words, 256, 8192), 256, 0, s>>>(iw);
    JET_LAUNCH_CHECK();
    // (cut change, largest part) of each iteration land in mailbox slots 8, 9
    Mailbox& mb = thread_mailbox();
    mailbox_ = &mb;
    res_host_ = mb.host + 8;
    res_dev_ = mb.dev + 8;
}

void Refiner::build_tiers(const Level& L) {
    DGraph g = L.view();
    fill_i32(counters_ + 16, 0, 8, s_);
    // on small levels every row with edges takes the wave tier: a thread per
    // row walks its edges one after another, a wave inserts them all at once
    small_max_ = g.n <= tuning().small_level_n ? 0 : SMALL_DEG;
    long_deg_ = (int32_t)(tuning().upd_big_slices * 2 * WAVE);
    k_conn_tiers<<<grid_for(g.n, 256, 8192), 256, 0, s_>>>(g, p_.k, tier_mid_, tier_big_, pull_mid_,
                                                            counters_ + 16, hub_, small_max_, long_deg_);
    k_max_degree<<<grid_for(g.n, MD_BLOCK, 256), MD_BLOCK, 0, s_>>>(g, counters_ + 18, counters_ + 22);
    JET_LAUNCH_CHECK();
    int32_t c[8];
    read_i32_words(counters_ + 16, 8, c, s_);
    ntier_mid_ = c[0];
    ntier_big_ = c[1];
    has_big_ = c[2] > BIG_DEG;
    has_long_ = c[2] > SEL_LONG && p_.k > SEL_LONG && g.n > SEL_LONG_N;
    npull_mid_ = c[3];
    nslices_ = c[4];
    // with long rows apart, the short ones' average says how many lanes they
    // keep busy
    avg_ = has_big_ ? 16.0 * (uint32_t)c[7] / std::max(1, c[6]) : (double)g.m / std::max<vid_t>(1, g.n);
}

// The level's row slices, in the caller's scope of the arena.
void Refiner::build_slices(const Level& L) {
    slices_ = nullptr;
    if (nslices_ == 0) return;
    DGraph g = L.view();
    slices_ = a_.alloc<int2>(nslices_);
    k_row_slices<<<grid_for(g.n, 256, 8192), 256, 0, s_>>>(g, long_deg_, slices_, counters_ + 21);
    JET_LAUNCH_CHECK();
}

void Refiner::init_conn(const Level& L, const part_t* part, const int32_t* mark) {
    DGraph g = L.view();
    int32_t* mk = const_cast<int32_t*>(mark);
    if (!mark) {
        ArenaScope sc(a_);
        int32_t* caps = a_.alloc<int32_t>((int64_t)g.n + 1);
        k_conn_caps<<<grid_for(g.n, 256, 8192), 256, 0, s_>>>(g, p_.k, caps);
        JET_LAUNCH_CHECK();
        excl_scan_i32_i64(caps, conn_off_, g.n, a_, s_);
        fill2_i32(dest_cache_, NULL_PART, g.n, lock_, 0, g.n, s_);
    }
    k_conn_build_small<<<grid_for(g.n, SB_BLOCK, 8192), SB_BLOCK, 0, s_>>>(g, part, p_.k, conn_off_, conn_,
                                                                          conn_size_, mk, dest_cache_, nullptr,
                                                                          small_max_);
    JET_LAUNCH_CHECK();
    if (ntier_mid_ > 0) {
        const size_t lds = 2 * sizeof(int2) * (size_t)WB_WAVES * std::min(p_.k, WAVE_TABLE_MAX);
        k_conn_build_wave<<<grid_for(ntier_mid_, WB_WAVES, 8192), WB_WAVES * WAVE, lds, s_>>>(
            g, part, p_.k, conn_off_, conn_, conn_size_, mk, dest_cache_, tier_mid_, ntier_mid_, nullptr);
        JET_LAUNCH_CHECK();
    }
    if (ntier_big_ > 0) {
        // a row's capacity is min(deg, k) <= k: two tables of k slots suffice
        const size_t lds = 2 * sizeof(int2) * (size_t)p_.k;
        k_conn_build_block<<<std::min(ntier_big_, 2048), BB_BLOCK, lds, s_>>>(
            g, part, p_.k, conn_off_, conn_, conn_size_, mk, dest_cache_, tier_big_, ntier_big_, nullptr);
        JET_LAUNCH_CHECK();
    }
}

// The best-state copy due from the previous step, for the next selection
// kernel to make (none when not due); the due flag is cleared.
BestCopy Refiner::take_best_copy() {
    BestCopy b{nullptr, nullptr, nullptr, 0};
    if (best_due_) b = BestCopy{best_out_, best_sizes_, curr_sizes_, p_.k};
    best_due_ = false;
    return b;
}

void Refiner::jet_lp(const Level& L, const part_t* part, double fr) {
    DGraph g = L.view();
    int32_t* c = cnt();
    gen_++;  // this step's moves are stamped with a new generation
    const BestCopy bcp = take_best_copy();
    // on levels with long rows the candidates' records, in the moves' array,
    // which the update passes fill later
    uint64_t* cbits = has_big_ ? cand_bits_ : nullptr;
    const uint32_t* cb = reinterpret_cast<const uint32_t*>(cbits);
    int4* crec = has_big_ ? reinterpret_cast<int4*>(mrec_) : nullptr;
    // a pass per wave on levels that fill the GPU with single-pass waves, two
    // passes per wave in 16-wave workgroups above that (see LS_MULTI_CHW)
    if (g.n <= tuning().lp_one_pass_n) {
        int nb = (int)std::max<int64_t>(1, ceil_div(g.n, (int64_t)LS_WAVES * WAVE));
        family_launch(PF_LP_SELECT, k_lp_select<WAVE, LS_WAVES, false>, dim3(nb), dim3(LS_WAVES * WAVE), 0, s_, g, part,
                      conn_off_, conn_, conn_size_, dest_cache_, gain_p_, lock_, fr, dest_, pregain_, cand_, c, nmax_,
                      cnt_next(), cbits, crec, prof_counters(PF_LP_SELECT), bcp);
    } else {
        int nb = (int)std::max<int64_t>(1, ceil_div(g.n, (int64_t)LS_MULTI_WAVES * LS_MULTI_CHW));
        family_launch(PF_LP_SELECT,
                      has_long_ ? k_lp_select<LS_MULTI_CHW, LS_MULTI_WAVES, true>
                                : k_lp_select<LS_MULTI_CHW, LS_MULTI_WAVES, false>,
                      dim3(nb), dim3(LS_MULTI_WAVES * WAVE), 0, s_, g, part, conn_off_, conn_, conn_size_, dest_cache_, gain_p_, lock_, fr, dest_, pregain_,
                      cand_, c, nmax_, cnt_next(), cbits, crec, prof_counters(PF_LP_SELECT), bcp);
    }
    JET_LAUNCH_CHECK();
    // per vertex: cached destination 4, lock 4 (and part 4, best copy 4 when
    // the previous step's best state rides along)
    prof_bytes(PF_LP_SELECT, (bcp.part_out ? 16.0 : 8.0) * g.n);
    if (unsigned long long* pc = prof_counters(PF_AFTERBURNER)) {
        // counting runs only: candidate degrees (the list is complete here)
        k_prof_degsum<<<grid_for(g.n, 256, 1024), 256, 0, s_>>>(g, cand_, c, 0, 1, nmax_, nullptr, pc);
    }
    unsigned ab = (unsigned)std::max<int64_t>(256, ceil_div((int64_t)g.n, (int64_t)AB_WAVES * AB_CHW));
#define JET_AB(GG)                                                                                                    \
    family_launch(PF_AFTERBURNER, has_big_ ? k_afterburner_small<GG, true> : k_afterburner_small<GG, false>, dim3(ab),  \
                  dim3(AB_WAVES * WAVE), 0, s_, g, cand_, c, part, dest_, pregain_, lock_, moves_, c, nmax_, stamp_, gen_, \
                  cb, crec)
    switch (group_for_afterburner(g, avg_)) {
        case 4: JET_AB(4); break;
        case 8: JET_AB(8); break;
        case 16: JET_AB(16); break;
        case 32: JET_AB(32); break;
        default: JET_AB(64); break;
    }
#undef JET_AB
    if (has_big_)
        family_launch(PF_AFTERBURNER, k_afterburner_big, dim3(grid_for((int64_t)g.n * WAVE, AB_WAVES * WAVE, 512)),
                      dim3(AB_WAVES * WAVE), 0, s_, g, cand_, c, part, dest_, pregain_, lock_, moves_, c, nmax_, stamp_,
                      gen_, long_deg_, cb, crec);
    JET_LAUNCH_CHECK();
}

// Ranks the members of flagged buckets (counter 5 of them) and applies the
// eviction decisions. The single-workgroup ranker is launched without reading
// the count on the host; when the count exceeds its capacity it raises the
// deferral flag (misc_[2]), the iteration's remaining kernels do nothing, and
// rank_deferred() finishes the step with the radix path after the sync.
void Refiner::rank_flagged(const Level& L, const part_t* part, const int64_t* sizes, int64_t width, bool strong) {
    DGraph g = L.view();
    int32_t* c = cnt();
    int64_t smax = size_max_;
    if (strong) {
        // the ranking workgroup also runs the cookie cutter (unless it defers)
        const CookieArgs ck{p_.k, rebalance_shape(g.n, true).max_dest, evict_start_, acc_};
        k_rank_small<true><<<1, RS_BLOCK, 0, s_>>>(cand_, c, bid_, part, off_, sizes, smax, width, g.vw, g.rowptr,
                                                  evict_adjust_, score_, moves_, c, nmax_, misc_ + 2, stamp_, gen_,
                                                  ck);
    } else {
        k_rank_small<false><<<1, RS_BLOCK, 0, s_>>>(cand_, c, bid_, part, off_, sizes, smax, width, g.vw,
                                                   g.rowptr, evict_adjust_, score_, moves_, c, nmax_, misc_ + 2, stamp_,
                                                   gen_, CookieArgs{});
    }
    JET_LAUNCH_CHECK();
}

void Refiner::rank_radix(const Level& L, const part_t* part, const int64_t* sizes, int64_t width, int key_bits,
                         bool strong) {
    DGraph g = L.view();
    int32_t* c = cnt();
    int64_t smax = size_max_;
    int32_t R = read_scalar(c + 5, s_);
    if (R == 0) return;
    ArenaScope sc(a_);
    uint64_t* keys = a_.alloc<uint64_t>(R);
    uint64_t* ktmp = a_.alloc<uint64_t>(R);
    int rb = grid_for(R, 256, 8192);
    k_rank_keys<<<rb, 256, 0, s_>>>(cand_, R, bid_, keys, sval_);
    JET_LAUNCH_CHECK();
    radix_sort_u64(keys, sval_, R, 32 + key_bits, ktmp, vtmp_, a_, s_);
    k_rank_weights<<<rb, 256, 0, s_>>>(R, sval_, g.vw, prefix_);
    JET_LAUNCH_CHECK();
    excl_scan_i64_i64(prefix_, prefix_, R, a_, s_);
    if (strong)
        k_rank_apply<true><<<rb, 256, 0, s_>>>(R, keys, prefix_, part, off_, sizes, smax, width, g.vw, g.rowptr,
                                              evict_adjust_, score_, moves_, c, nmax_, stamp_, gen_);
    else
        k_rank_apply<false><<<rb, 256, 0, s_>>>(R, keys, prefix_, part, off_, sizes, smax, width, g.vw, g.rowptr,
                                               evict_adjust_, score_, moves_, c, nmax_, stamp_, gen_);
    JET_LAUNCH_CHECK();
}

Refiner::RebalanceShape Refiner::rebalance_shape(vid_t n, bool strong) const {
    RebalanceShape r;
    const int32_t k = p_.k;
    r.sections = sections_for(n, k);
    r.width = (int64_t)MAX_BUCKETS * r.sections;
    // weak: gain bucket 50 is not capped (jet_refiner.hpp:349-351) and spills
    // past the last part's minibuckets, so `sections` more are kept and scanned
    r.nbk = strong ? (int64_t)k * r.width + 1 : (int64_t)k * r.width + r.sections + 1;
    const int64_t smax = size_max_;
    if (strong) {
        r.max_dest = std::max<int64_t>((int64_t)opt_ + 1, (int64_t)(smax * 0.99));
    } else {
        r.max_dest = (int64_t)(smax * 0.99);
        if (r.max_dest < smax - 100) r.max_dest = smax - 100;
    }
    r.key_bits = 1;
    while ((int64_t(1) << r.key_bits) <= r.nbk) r.key_bits++;
    return r;
}

// rebalance_strong's destination step (jet_refiner.hpp:480-544), after ranking.
void Refiner::strong_tail(const Level& L, const part_t* part, const int64_t* sizes, const RebalanceShape& r,
                          bool cookie_done) {
    DGraph g = L.view();
    int32_t* c = cnt();
    const int32_t k = p_.k;
    int nb = grid_for(g.n, 256, 8192);
    if (!cookie_done)
        k_cookie<<<1, CK_BLOCK, 0, s_>>>(k, r.width, off_, sizes, r.max_dest, evict_adjust_, evict_start_, acc_,
                                         misc_ + 2);
    k_strong_dest<<<nb, 256, 0, s_>>>(moves_, c, nmax_, part, g.vw, evict_adjust_, evict_start_, k, score_, dest_,
                                      redraw_, c + 4, nmax_, misc_ + 2);
    const int32_t lds_max = (int32_t)std::min<int64_t>(RD_MAX, tuning().redraw_lds_max);
    k_strong_redraw<<<1, 256, 0, s_>>>(redraw_, c + 4, part, g.vw, evict_start_, k, score_, dest_, acc_, rd_mark_,
                                       g.n, lds_max, misc_ + 2);
    JET_LAUNCH_CHECK();
}

// Finishes a step whose ranking was deferred: clears the flag, ranks with the
// radix path and runs the strong destination step.
void Refiner::rank_deferred(const Level& L, const part_t* part, const int64_t* sizes, bool strong) {
    fill_i32(misc_ + 2, 0, 1, s_);
    RebalanceShape r = rebalance_shape(L.n, strong);
    rank_radix(L, part, sizes, r.width, r.key_bits, strong);
    if (strong) strong_tail(L, part, sizes, r, false);
}

void Refiner::rebalance(const Level& L, const part_t* part, const int64_t* sizes, bool strong) {
    DGraph g = L.view();
    const int32_t k = p_.k;
    int32_t* c = cnt();
    const RebalanceShape r = rebalance_shape(g.n, strong);
    const int32_t sections = r.sections;
    const int64_t width = r.width, nbk = r.nbk, max_dest = r.max_dest;
    const int64_t smax = size_max_;
    gen_++;  // this step's moves are stamped with a new generation
    // the previous step's second update pass prepared this kind of step (bucket
    // sums zeroed, undersized parts or capacity), else a reset launch does
    if (!(prep_ready_ && prep_strong_ == strong))
        k_reset_buckets<<<grid_for(nbk + 1, 256, 2048), 256, 0, s_>>>(buckets_, nbk + 1, cnt_next(), sizes, k,
                                                                        max_dest, strong ? 1 : 0, undersized_, misc_,
                                                                        acc_, evict_adjust_);
    prep_ready_ = false;
    const BestCopy bcp = take_best_copy();
    // contiguous ranges of at least 512 vertices per workgroup (128 on small
    // levels, one per thread of a 128-thread workgroup): vertices of one
    // oversized part share few buckets, and the serial per-vertex chain of a
    // heavy range stays short
    int nsel = grid_for(g.n, g.n <= tuning().small_level_n ? 128 : 512, (int)tuning().sel_max_blocks);
    unsigned long long* bk = reinterpret_cast<unsigned long long*>(buckets_);
    unsigned long long* bc = reinterpret_cast<unsigned long long*>(bcopies_);
    // one copy per sel_copy_wgs workgroups (256 by default): fewer
    // workgroups meet on a line, and a copy costs a pass of the fold
    // With few parts every workgroup adds to every bucket, and the atomics of
    // all workgroups meet on each line (10 ns each): up to 64 parts a copy per
    // 32 to 64 workgroups. Stencil levels of 136,971 and 254,104 vertices with a
    // copy per 256 and now: k = 2 42 and 34, 36 and 34 us an iteration, k = 4
    // 47 and 40, 67 and 45, k = 30 43 and 42, 52 and 49; 2,097,152 vertices with
    // k = 32 77 and 75, k = 64 79 and 76, but k = 256 94 and 97.
    const int64_t copy_wgs =
        std::min<int64_t>(tuning().sel_copy_wgs, k > 64 ? INT64_MAX : std::min<int64_t>(64, std::max<int64_t>(32, 16 * (int64_t)k)));
    const int32_t copies = std::max(1, std::min<int32_t>(ncopies_, (int32_t)(nsel / copy_wgs)));
    const bool lds = k <= SEL_LDS_K;
    // 512 threads on large levels (half the serial vertices per thread), 128
    // on small ones (more workgroups over few vertices; 0.3 ms less per 128^3
    // stencil partition than 256)
    const int selb = g.n > tuning().small_level_n ? SEL_BLOCK_MAX : 128;
    if (strong) {
        if (lds)
            (has_long_ ? k_strong_select<true, true> : k_strong_select<true, false>)<<<nsel, selb, 0, s_>>>(g, part, sizes, k, smax, opt_, max_dest, acc_, conn_off_,
                                                         conn_, conn_size_, sections, bid_, bk, bc, copies, nbuckets_,
                                                         cnt_next(), bcp);
        else
            (has_long_ ? k_strong_select<false, true> : k_strong_select<false, false>)<<<nsel, selb, 0, s_>>>(g, part, sizes, k, smax, opt_, max_dest, acc_, conn_off_,
                                                          conn_, conn_size_, sections, bid_, bk, bc, copies, nbuckets_,
                                                          cnt_next(), bcp);
    } else {
        family_launch(PF_WEAK_SELECT, lds ? k_weak_select<true> : k_weak_select<false>, dim3(nsel), dim3(selb), 0,
                      s_, g, part, sizes, k, smax, opt_, max_dest, undersized_, misc_, conn_off_, conn_, conn_size_,
                      sections, dest_, bid_, bk, bc, copies, nbuckets_, prof_counters(PF_WEAK_SELECT), cnt_next(), bcp);
        // per vertex: part 4, destination 4, bucket id 4
        prof_bytes(PF_WEAK_SELECT, (bcp.part_out ? 16.0 : 12.0) * g.n);
    }
    if (copies > 1)
        k_sum_bucket_copies<<<grid_for(nbk + 1, 256, 2048), 256, 0, s_>>>(buckets_, bcopies_, copies, nbk + 1,
                                                                          nbuckets_);
    JET_LAUNCH_CHECK();
    // the scanned buckets go to boff_: a bucket array of up to FUSE_SCAN_MAX
    // sums is scanned by the classification kernel itself, a longer one by a
    // scan launch (out of place, so its workgroups need not wait on each other)
    const bool fused = nbk <= FUSE_SCAN_MAX;
    off_ = boff_;
    if (!fused) excl_scan_i64_i64(buckets_, boff_, nbk, a_, s_);
    int cb = (int)std::max<int64_t>(1, ceil_div(g.n, (int64_t)CL_WAVES * CL_CHW));
#define JET_CLASSIFY(ST, FU)                                                                                 \
    k_classify<ST, FU><<<cb, CL_WAVES * WAVE, 0, s_>>>(g, part, bid_, FU ? buckets_ : boff_, nbk, boff_, sizes,    \
                                                       smax, width, k, sections, moves_, c, nmax_, cand_, stamp_,  \
                                                       gen_)
    if (strong) {
        if (fused) JET_CLASSIFY(true, true);
        else JET_CLASSIFY(true, false);
    } else {
        if (fused) JET_CLASSIFY(false, true);
        else JET_CLASSIFY(false, false);
    }
#undef JET_CLASSIFY
    JET_LAUNCH_CHECK();
    rank_flagged(L, part, sizes, width, strong);
    // the ranking workgroup ran the cookie cutter (when it deferred, every
    // later kernel of the step does nothing and rank_deferred runs it)
    if (strong) strong_tail(L, part, sizes, r, true);
}

// Waits for the step's results in the mapped mailbox.
void Refiner::wait_published(volatile int64_t* res, int64_t seq) {
    if (!wait_mailbox(&res[5], seq, s_)) throw DeviceError("refinement step finished without publishing its results");
}

bool Refiner::perform_moves(const Level& L, part_t* part, int64_t* sizes, int64_t& cut_change, int64_t& max_size,
                             int next_strong) {
    DGraph g = L.view();
    const int32_t k = p_.k;
    int32_t* c = cnt();
    unsigned long long* usz = reinterpret_cast<unsigned long long*>(sizes);
    int G = group_for_update(avg_);
    int nbs = grid_for((int64_t)g.n * G, 256, 1024);
    const int64_t seq = ++mailbox_->seq;
    // size-delta copies for the LDS-aggregated deltas (k <= LDS_K): about
    // 4096 entries in all
    const int32_t nsc = k <= LDS_K ? std::max(1, std::min(SIZE_COPIES_MAX, 4096 / k)) : 0;
    const Publish pb{pub_, sizes, k, res_dev_, c, seq, reinterpret_cast<unsigned long long*>(szc_), nsc};
    // the next step's start in case it is a rebalancing step of kind
    // next_strong (the controller knows the kind before this step's result)
    RebalPrep prep{};
    if (next_strong >= 0) {
        const RebalanceShape nr = rebalance_shape(g.n, next_strong != 0);
        prep = RebalPrep{buckets_, nr.nbk + 1, nr.max_dest, next_strong, undersized_, misc_, acc_, evict_adjust_};
    }
    const RebalPrep no_prep{};
    prep_ready_ = false;
    int nbb = grid_for((int64_t)g.n * WAVE, UB_BLOCK, 512);
    // k_pull_hubs: a dense table of k parts per wave (about 32 KB of them) and
    // the moved bits, 2^ph_shift vertices each
    const bool hubs = ntier_big_ > 0 || npull_mid_ > 0;
    const int ph_waves = std::max(1, std::min<int>(PH_WAVES_MAX, 8192 / k));
    const size_t ph_tables = sizeof(int32_t) * (size_t)ph_table_words(k) * ph_waves;
    int32_t ph_shift = 0;
    auto bits_bytes = [&] { return 4 * (size_t)(((int64_t)g.n + (32ll << ph_shift) - 1) >> (5 + ph_shift)); };
    while (bits_bytes() > PH_BITS_MAX) ph_shift++;
    uint32_t* bits = hubs ? moved_bits_ : nullptr;
    int2* mv = reinterpret_cast<int2*>(score_);  // the scores of a strong step are done with
    const uint8_t* hub = hubs ? hub_ : nullptr;
    for (int add = 0; add < 2; add++) {
        if (unsigned long long* pc = prof_counters(PF_UPDATE)) {
            // counting runs only: move degrees, once per pass (nothing when
            // the step's ranking was deferred: its kernels then do nothing)
            k_prof_degsum<<<grid_for(g.n, 256, 1024), 256, 0, s_>>>(g, moves_, c, 2, 3, nmax_, misc_ + 2, pc);
        }
#define JET_UPD(GG)                                                                                                   \
    if (add) family_launch(PF_UPDATE, k_update_small<true, GG>, dim3(nbs + 1), dim3(256), 0, s_, g, moves_, mrec_, c, \
                           nmax_, part, dest_, conn_off_, conn_, conn_size_, dest_cache_, k, misc_ + 1, swap_bit_,    \
                           hub, hub_dirty_, misc_ + 2, stamp_, gen_, usz, pub_, bits, mv, pb, prep);                  \
    else family_launch(PF_UPDATE, k_update_small<false, GG>, dim3(nbs), dim3(256), 0, s_, g, moves_, mrec_, c, nmax_, \
                       part, dest_, conn_off_, conn_, conn_size_, dest_cache_, k, misc_ + 1, swap_bit_, hub,          \
                       hub_dirty_, misc_ + 2, stamp_, gen_, usz, pub_, bits, mv, pb, no_prep);
        switch (G) {
            case 4: JET_UPD(4) break;
            case 8: JET_UPD(8) break;
            case 16: JET_UPD(16) break;
            case 32: JET_UPD(32) break;
            default: JET_UPD(64) break;
        }
#undef JET_UPD
        if (has_big_) {
            family_launch(PF_UPDATE, add ? k_update_big<true> : k_update_big<false>, dim3(nbb), dim3(UB_BLOCK), 0, s_, g,
                          moves_, mrec_, c, nmax_, part, dest_, conn_off_, conn_, conn_size_, dest_cache_, k,
                          misc_ + 1, swap_bit_, hub, hub_dirty_, misc_ + 2, stamp_, gen_, usz, pub_, bits, mv, long_deg_,
                          slices_, nslices_, pb.copies, pb.ncopies);
        }
        if (!add && hubs) {
            const int want = std::max(ntier_big_, (int)ceil_div(npull_mid_, ph_waves));
            const int pb = std::max(1, std::min(want, 512));
            family_launch(PF_UPDATE, ph_shift == 0 ? k_pull_hubs<true> : k_pull_hubs<false>, dim3(pb),
                          dim3(ph_waves * WAVE), (uint32_t)(ph_tables + bits_bytes()), s_, g, tier_big_, ntier_big_,
                          pull_mid_, npull_mid_, c, moved_bits_, ph_shift, mv, hub_dirty_, part, dest_, conn_off_, conn_,
                          conn_size_, dest_cache_, k, misc_ + 1, swap_bit_, misc_ + 2, pub_);
        }
        JET_LAUNCH_CHECK();
    }
    volatile int64_t* res = res_host_;
    wait_published(res, seq);
    if (res[2]) return true;  // ranking deferred: nothing applied, counters kept
    cut_change = res[0];
    max_size = res[1];
    if (next_strong >= 0) {
        prep_ready_ = true;
        prep_strong_ = next_strong != 0;
    }
    // update_large: the marked rows are rebuilt before the tables are next
    // read (rebuild_pending), so a step that pushed its updates launches no
    // rebuild kernels
    rebuild_pending_ = res[3] != 0;
    par_ ^= 1;
    return false;
}

// The refinement kernels' error bits, as text.
static std::string refine_error_text(int32_t err) {
    std::string m = "refinement invariant violated:";
    if (err & 1) m += " a moved vertex's old part was missing from a neighbour's connectivity row;";
    if (err & 2) m += " a connectivity row ran out of slots;";
    if (err & 8) m += " a strong re-draw walked past its bound;";
    if (err & ~11) m += " error bits " + std::to_string(err) + ";";
    return m;
}

void Refiner::flush_rebuild(const Level& L) {
    if (!rebuild_pending_) return;
    init_conn(L, cur_part_, swap_bit_);
    rebuild_pending_ = false;
}

LevelRecord Refiner::refine(const Level& L, part_t* best_part) {
    auto t0 = std::chrono::steady_clock::now();
    changed_ = false;
    prep_ready_ = false;
    best_due_ = false;
    DGraph g = L.view();
    const int32_t k = p_.k;
    int64_t first_max = 0;
    if (!init_) {
        cut_ = total_cut2(g, best_part, a_, s_);
        part_sizes(g, best_part, k, best_sizes_, s_);
        std::vector<int64_t> hs(k);
        JET_HIP(hipMemcpyAsync(hs.data(), best_sizes_, sizeof(int64_t) * k, hipMemcpyDeviceToHost, s_));
        JET_HIP(hipStreamSynchronize(s_));
        total_size_ = 0;
        for (int64_t v : hs) {
            total_size_ += v;
            first_max = std::max(first_max, v);
        }
    }
    opt_ = (int32_t)(((int32_t)total_size_ + k - 1) / k);
    size_max_ = (int32_t)(opt_ * p_.imb);
    if (!init_) {
        init_ = true;
        total_imb_ = first_max > opt_ ? first_max - opt_ : 0;
    }
    std::vector<double> temps;
    if (p_.ultra) {
        for (double t = 0.85; t > 0; t -= 0.05) temps.push_back(t);
    } else if (L.uniform) {
        temps.push_back(0.25);
    } else {
        temps.push_back(0.75);
    }
    const RebalanceShape wr = rebalance_shape(g.n, false);
    // the kernel families are measured, and iterations traced, on the
    // multi-kernel path
    if (!trace && !prof_active() && team_fits(g.n, g.m, k, wr.nbk, team_max_n()) &&
        (int)temps.size() <= TEAM_MAX_TEMPS && !(team_irregular_ && g.m > TEAM_REGULAR_M)) {
        LevelRecord rec;
        if (refine_team(L, best_part, temps, rec)) {
            rec.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            return rec;
        }
    }
    fill2_i32(misc_, 0, 8, counters_, 0, 16, s_);
    par_ = 0;
    int64_t curr_cut = cut_, curr_imb = total_imb_;
    copy_i64(curr_sizes_, best_sizes_, k, s_);
    const int64_t imb_max = (int64_t)size_max_ - opt_;
    copy_i32(cur_part_, best_part, g.n, s_);
    ArenaScope level_scope(a_);
    build_tiers(L);
    build_slices(L);
    init_conn(L, cur_part_, nullptr);
    LevelRecord rec;
    int balance_counter = 0;
    for (double fr : temps) {
        int count = 0;
        while (count++ <= 11) {
            rec.iterations++;
            bool strong = false;
            flush_rebuild(L);
            if (curr_imb <= imb_max) {
                jet_lp(L, cur_part_, fr);
                balance_counter = 0;
                rec.lp_iterations++;
            } else {
                strong = balance_counter >= 2;
                rebalance(L, cur_part_, curr_sizes_, strong);
                balance_counter++;
            }
            int64_t cc = 0, mx = 0;
            // a rebalancing step after this one is strong iff two rebalancing
            // steps precede it (balance_counter as updated for this step)
            const int next_strong = balance_counter >= 2 ? 1 : 0;
            if (perform_moves(L, cur_part_, curr_sizes_, cc, mx, next_strong)) {
                rank_deferred(L, cur_part_, curr_sizes_, strong);
                if (perform_moves(L, cur_part_, curr_sizes_, cc, mx, next_strong))
                    throw DeviceError("rebalancing step deferred twice");
            }
            curr_imb = mx > opt_ ? mx - opt_ : 0;
            curr_cut -= cc;
            int take = 0;  // 1: better balance, 2: better cut
            if (total_imb_ > imb_max && curr_imb < total_imb_) {
                take = 1;
                count = 0;
            } else if (curr_cut < cut_ && (curr_imb <= imb_max || curr_imb <= total_imb_)) {
                if ((double)curr_cut < p_.tol * (double)cut_) count = 0;
                take = 2;
            }
            if (take) {
                changed_ = true;
                cut_ = curr_cut;
                total_imb_ = curr_imb;
                // the best state (partition and part sizes) is copied by the
                // next step's selection kernel, or at the end of the level
                best_due_ = true;
                best_out_ = best_part;
            }
            if (trace) {
                const int64_t kind = balance_counter == 0 ? 0 : (strong ? 2 : 1);
                trace->push_back({kind, -1, curr_cut, curr_imb, take, count});
            }
        }
    }
    prep_ready_ = false;
    if (best_due_) {
        k_copy_best<<<grid_for(g.n, 256, 8192), 256, 0, s_>>>(best_part, cur_part_, g.n, best_sizes_, curr_sizes_, k);
        JET_LAUNCH_CHECK();
        best_due_ = false;
    }
    flush_rebuild(L);
    int32_t err = read_scalar(misc_ + 1, s_);
    if (err) throw DeviceError(refine_error_text(err));
    rec.cut2 = cut_;
    rec.total_imb = total_imb_;
    rec.n = g.n;
    rec.m = g.m;
    rec.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return rec;
}

// The whole level in one launch (csrc/refine_team.hip).
bool Refiner::refine_team(const Level& L, part_t* best_part, const std::vector<double>& temps, LevelRecord& rec) {
    DGraph g = L.view();
    const int32_t k = p_.k;
    const RebalanceShape weak = rebalance_shape(g.n, false), strong = rebalance_shape(g.n, true);
    TeamParams P{};
    P.g = g;
    P.k = k;
    P.sections = weak.sections;
    P.nbk = (int32_t)weak.nbk;
    P.big_deg = (int32_t)tuning().wg_big_deg;
    P.lanes = group_for_avg(g);
    P.opt = opt_;
    P.size_max = size_max_;
    P.imb_max = (int64_t)size_max_ - opt_;
    P.max_dest_weak = weak.max_dest;
    P.max_dest_strong = strong.max_dest;
    P.tol = p_.tol;
    P.ntemps = (int32_t)temps.size();
    for (size_t i = 0; i < temps.size(); i++) P.temps[i] = temps[i];
    P.start.curr_cut = P.start.best_cut = cut_;
    P.start.curr_imb = P.start.best_imb = total_imb_;
    P.part = cur_part_;
    P.best_part = best_part;
    P.conn = conn_;
    P.conn_size = conn_size_;
    P.dest_cache = dest_cache_;
    P.lock = lock_;
    P.gain_p = gain_p_;
    P.pregain = pregain_;
    P.dest = dest_;
    P.bid = bid_;
    P.stamp = stamp_;
    P.gen0 = gen_;
    P.mark = swap_bit_;
    P.score = score_;
    P.rkey = team_rkey_;
    P.rweight = team_rweight_;
    P.redraw = redraw_;
    P.buckets = team_buckets_;
    P.sizes = curr_sizes_;
    P.best_sizes = best_sizes_;
    P.evict_adjust = evict_adjust_;
    P.ctl = team_ctl_;
    P.host_out = mailbox_->dev + TEAM_MAILBOX;
    volatile int64_t* out = mailbox_->host + TEAM_MAILBOX;
    P.team = team_size(g.n, g.m);
    P.start_spins = (int32_t)tuning().team_start_spins;
    // A launch ends after team_launch_iters iterations (about a second by
    // default, which no level measured here reaches); the next one goes on from
    // the state it left.
    for (int tries = 0;;) {
        P.seq = ++mailbox_->seq;
        P.iter_cap = P.start.iterations + (int32_t)tuning().team_launch_iters;
        TeamSlot slot(P.team);
        P.xcd = slot.xcd();
        launch_refine_team(P, s_);
        // without a result: no workgroup ran on the wanted XCD
        const bool ran = wait_mailbox(&out[TEAM_OUT_WORDS], P.seq, s_);
        const int64_t bits = ran ? out[6] : LEVEL_ABANDONED;
        const int32_t status = (int32_t)(bits & 0xffff), err = ran ? (int32_t)out[5] : 0;
        if (err) throw DeviceError(refine_error_text(err));
        if (status == LEVEL_DONE || status == LEVEL_MORE)
            P.start = LevelState{out[2],
                                 out[3],
                                 out[0],
                                 out[1],
                                 (int32_t)(bits >> 32 & 0xffff),
                                 (int32_t)(bits >> 48 & 0xffff),
                                 (int32_t)(out[5] >> 32),
                                 (int32_t)out[4],
                                 (int32_t)(out[4] >> 32),
                                 (int32_t)(bits >> 16 & 0xffff),
                                 status};
        if (status == LEVEL_DONE) break;
        if (status == LEVEL_MORE) {
            P.resume = 1;
            tries = 0;
            continue;
        }
        if (status == LEVEL_IRREGULAR) team_irregular_ = true;
        if (status == LEVEL_ABANDONED) team_abandoned();
        // a level that has begun can only go on where it was
        if (P.resume && status == LEVEL_ABANDONED && ++tries < 100) continue;
        if (!P.resume && (status == LEVEL_ABANDONED || status == LEVEL_IRREGULAR)) return false;
        throw DeviceError("team refinement made no progress");
    }
    const LevelState& S = P.start;
    cut_ = S.best_cut;
    total_imb_ = S.best_imb;
    rec.iterations = S.iterations;
    rec.lp_iterations = S.lp_iterations;
    gen_ += rec.iterations;
    if (S.changed) changed_ = true;
    rec.cut2 = cut_;
    rec.total_imb = total_imb_;
    rec.n = g.n;
    rec.m = g.m;
    return true;
}

void Refiner::single_step(const Level& L, const part_t* part, int kind, double fr, std::vector<int32_t>& moves,
                          std::vector<int32_t>& dest) {
    DGraph g = L.view();
    const int32_t k = p_.k;
    best_due_ = false;
    fill_i32(misc_, 0, 8, s_);
    fill_i32(counters_, 0, 16, s_);
    par_ = 0;
    copy_i32(cur_part_, part, g.n, s_);
    part_sizes(g, cur_part_, k, curr_sizes_, s_);
    std::vector<int64_t> hs(k);
    JET_HIP(hipMemcpyAsync(hs.data(), curr_sizes_, sizeof(int64_t) * k, hipMemcpyDeviceToHost, s_));
    JET_HIP(hipStreamSynchronize(s_));
    int64_t tot = 0;
    for (int64_t v : hs) tot += v;
    opt_ = (int32_t)(((int32_t)tot + k - 1) / k);
    size_max_ = (int32_t)(opt_ * p_.imb);
    build_tiers(L);
    init_conn(L, cur_part_, nullptr);
    if (kind == 0) jet_lp(L, cur_part_, fr);
    else {
        rebalance(L, cur_part_, curr_sizes_, kind == 2);
        if (read_scalar(misc_ + 2, s_)) rank_deferred(L, cur_part_, curr_sizes_, kind == 2);
    }
    int32_t c4[4];
    JET_HIP(hipMemcpyAsync(c4, cnt(), sizeof(c4), hipMemcpyDeviceToHost, s_));
    JET_HIP(hipStreamSynchronize(s_));
    int32_t total = c4[2] + c4[3];
    ArenaScope sc(a_);
    vid_t* ov = a_.alloc<vid_t>(std::max(total, 1));
    part_t* od = a_.alloc<part_t>(std::max(total, 1));
    if (total > 0) {
        k_collect_moves<<<grid_for(total, 256, 8192), 256, 0, s_>>>(moves_, cnt(), nmax_, dest_, ov, od);
        JET_LAUNCH_CHECK();
    }
    std::vector<int32_t> v(total), d(total);
    if (total > 0) {
        JET_HIP(hipMemcpyAsync(v.data(), ov, sizeof(int32_t) * total, hipMemcpyDeviceToHost, s_));
        JET_HIP(hipMemcpyAsync(d.data(), od, sizeof(int32_t) * total, hipMemcpyDeviceToHost, s_));
    }
    JET_HIP(hipStreamSynchronize(s_));
    int32_t err = read_scalar(misc_ + 1, s_);
    if (err) throw DeviceError(refine_error_text(err));
    std::vector<int32_t> idx(total);
    for (int32_t t = 0; t < total; t++) idx[t] = t;
    std::sort(idx.begin(), idx.end(), [&](int32_t x, int32_t y) { return v[x] < v[y]; });
    moves.resize(total);
    dest.resize(total);
    for (int32_t t = 0; t < total; t++) {
        moves[t] = v[idx[t]];
        dest[t] = d[idx[t]];
    }
}

// part_stat.hpp:131-144, 186-239 from the connectivity tables: the
// communication volume (per vertex, the parts other than its own that its
// neighbours are in) and the cut weight incident to each part.
// Each workgroup sums the parts' cut weights in LDS (k <= LDS_K): an atomic per
// vertex on k addresses took 296 us on a 64^3 stencil with k = 256.
constexpr int QU_BLOCK = 1024;
__global__ void __launch_bounds__(QU_BLOCK)
    k_quality(DGraph g, const part_t* part, int32_t k, const eoff_t* conn_off, const int2* conn,
              const int32_t* conn_size, unsigned long long* comm, unsigned long long* cut_per_part) {
    __shared__ int64_t red[QU_BLOCK / WAVE];
    __shared__ unsigned long long ls[LDS_K];
    const bool lds = k <= LDS_K;
    if (lds) {
        for (int t = threadIdx.x; t < k; t += QU_BLOCK) ls[t] = 0;
        __syncthreads();
    }
    int64_t c = 0;
    FOR_THREAD(i, g.n) {
        const part_t p = part[i];
        int64_t ext = 0;
        for_slots(conn + conn_off[i], conn_size[i], [&](int2 e) {
            if (e.x > NULL_PART && e.x != p && e.y > 0) {
                c++;
                ext += e.y;
            }
        });
        if (ext) atomicAdd(lds ? &ls[p] : &cut_per_part[p], (unsigned long long)ext);
    }
    c = block_reduce_sum<int64_t, QU_BLOCK>(c, red);
    if (threadIdx.x == 0 && c) atomicAdd(comm, (unsigned long long)c);
    if (lds) {
        __syncthreads();
        for (int t = threadIdx.x; t < k; t += QU_BLOCK)
            if (ls[t]) atomicAdd(&cut_per_part[t], ls[t]);
    }
}

void Refiner::quality(const Level& L, const part_t* part, int64_t& comm_size, std::vector<int64_t>& cut_per_part) {
    DGraph g = L.view();
    copy_i32(cur_part_, part, g.n, s_);
    build_tiers(L);
    init_conn(L, cur_part_, nullptr);
    ArenaScope sc(a_);
    unsigned long long* d = a_.alloc<unsigned long long>(1 + p_.k);
    fill_i64(reinterpret_cast<int64_t*>(d), 0, 1 + p_.k, s_);
    k_quality<<<grid_for(g.n, QU_BLOCK, 512), QU_BLOCK, 0, s_>>>(g, cur_part_, p_.k, conn_off_, conn_, conn_size_, d,
                                                                 d + 1);
    JET_LAUNCH_CHECK();
    std::vector<int64_t> h(1 + p_.k);
    JET_HIP(hipMemcpyAsync(h.data(), d, sizeof(int64_t) * h.size(), hipMemcpyDeviceToHost, s_));
    JET_HIP(hipStreamSynchronize(s_));
    comm_size = h[0];
    cut_per_part.assign(h.begin() + 1, h.end());
}

// part_stat.hpp:116-129 from the connectivity tables: heat[p * k + q] = cut
// weight from vertices of part p to part q (q != p). With k * k <= HEAT_LDS
// each workgroup sums into LDS first.
constexpr int HEAT_LDS = 4096;

template <bool LDS>
__global__ void __launch_bounds__(256)
    k_heatmap(DGraph g, const part_t* part, const eoff_t* conn_off, const int2* conn, const int32_t* conn_size,
              int32_t k, unsigned long long* heat) {
    __shared__ unsigned long long lh[LDS ? HEAT_LDS : 1];
    if (LDS) {
        for (int t = threadIdx.x; t < k * k; t += blockDim.x) lh[t] = 0;
        __syncthreads();
    }
    FOR_BLOCK_RANGE(i, g.n) {
        const part_t p = part[i];
        for_slots(conn + conn_off[i], conn_size[i], [&](int2 e) {
            if (e.x > NULL_PART && e.x != p && e.y > 0) {
                const int64_t at = (int64_t)p * k + e.x;
                if (LDS) atomicAdd(&lh[at], (unsigned long long)e.y);
                else atomicAdd(&heat[at], (unsigned long long)e.y);
            }
        });
    }
    if (LDS) {
        __syncthreads();
        for (int t = threadIdx.x; t < k * k; t += blockDim.x)
            if (lh[t]) atomicAdd(&heat[t], lh[t]);
    }
}

void Refiner::heatmap(const Level& L, const part_t* part, int64_t* heat) {
    DGraph g = L.view();
    copy_i32(cur_part_, part, g.n, s_);
    build_tiers(L);
    init_conn(L, cur_part_, nullptr);
    const int64_t kk = (int64_t)p_.k * p_.k;
    fill_i64(heat, 0, kk, s_);
    unsigned long long* h = reinterpret_cast<unsigned long long*>(heat);
    if (kk <= HEAT_LDS)
        k_heatmap<true><<<grid_for(g.n, 2048, 1024), 256, 0, s_>>>(g, cur_part_, conn_off_, conn_, conn_size_, p_.k, h);
    else
        k_heatmap<false><<<grid_for(g.n, 256, 8192), 256, 0, s_>>>(g, cur_part_, conn_off_, conn_, conn_size_, p_.k,
                                                                   h);
    JET_LAUNCH_CHECK();
}

void Refiner::conn_tables(const Level& L, const part_t* part, std::vector<int64_t>& off,
                          std::vector<int32_t>& slot_part, std::vector<int32_t>& slot_val, std::vector<int32_t>& size) {
    DGraph g = L.view();
    copy_i32(cur_part_, part, g.n, s_);
    build_tiers(L);
    init_conn(L, cur_part_, nullptr);
    off.resize(g.n + 1);
    size.resize(g.n);
    JET_HIP(hipMemcpyAsync(off.data(), conn_off_, sizeof(int64_t) * (g.n + 1), hipMemcpyDeviceToHost, s_));
    JET_HIP(hipMemcpyAsync(size.data(), conn_size_, sizeof(int32_t) * g.n, hipMemcpyDeviceToHost, s_));
    JET_HIP(hipStreamSynchronize(s_));
    int64_t C = off[g.n];
    std::vector<int2> slots(std::max<int64_t>(C, 1));
    if (C > 0) JET_HIP(hipMemcpyAsync(slots.data(), conn_, sizeof(int2) * C, hipMemcpyDeviceToHost, s_));
    JET_HIP(hipStreamSynchronize(s_));
    slot_part.resize(C);
    slot_val.resize(C);
    for (int64_t c = 0; c < C; c++) {
        slot_part[c] = slots[c].x;
        slot_val[c] = slots[c].y;
    }
}

}  // namespace jet
