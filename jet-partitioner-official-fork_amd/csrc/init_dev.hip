// Coarsening of large graphs for the initial partition, on the device (the
// host's coarsen_once, csrc/initpart.cpp, for graphs of at least
// PAR_MATCH_EDGES entries; the level below is the same entry for entry).
//
// On the host a level of R-MAT 22's coarsest graph (362,220 vertices, 70.4 M
// entries) is bound by random reads of the neighbours' state and of the
// position tables, after the graph has been copied there through pageable
// memory. Here the six handshake rounds stream the rows (a wave per vertex,
// four edges per lane in flight, the longest rows by a workgroup), and a
// coarse row is one pass over its two members' rows with a hash table in LDS:
// an entry is the first of its neighbour when its position is the table's
// minimum, and a prefix count over those puts the row in first-seen order
// without a sort. Only the vertex-sized arrays (mates, first neighbours) go to
// the host, which pairs the leftovers and numbers the coarse vertices.
#include "init_dev.h"

#include <algorithm>

#include "conn_table.h"
#include "initpart.h"
#include "prims.h"
#include "wave.h"

namespace jet {

namespace {

constexpr int HS_BLOCK = 1024;
constexpr int HS_WAVES = HS_BLOCK / WAVE;
constexpr int HS_UNROLL = 4;
constexpr int HS_QUEUE = 1024;
constexpr int32_t HS_LONG = 2048;

// Better proposal: heavier edge, then larger seeded key, then the earlier edge.
__device__ inline bool hs_better(int32_t w, uint32_t k, eoff_t j, int32_t bw, uint32_t bk, eoff_t bj) {
    return w > bw || (w == bw && (k > bk || (k == bk && j < bj)));
}

__global__ void __launch_bounds__(HS_BLOCK)
    k_propose(DGraph g, uint64_t seed, int64_t cap, const int32_t* mate, int32_t* prop) {
    __shared__ vid_t queue[HS_QUEUE];
    __shared__ int32_t nqueue;
    __shared__ int32_t sw[HS_WAVES];
    __shared__ uint32_t sk[HS_WAVES];
    __shared__ eoff_t sj[HS_WAVES];
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = threadIdx.x / WAVE;
    if (threadIdx.x == 0) nqueue = 0;
    __syncthreads();
    // the best proposal among edges rs + sub, rs + sub + stride, ... in every lane of the wave
    auto best = [&](vid_t v, eoff_t rs, eoff_t re, int sub, int stride, int32_t& bw, uint32_t& bk, eoff_t& bj) {
        const int64_t room = cap - (int64_t)g.vw[v];
        bw = -1;
        bk = 0;
        bj = re;
        for (eoff_t b0 = rs; b0 < re; b0 += (eoff_t)HS_UNROLL * stride) {
            vid_t u[HS_UNROLL];
            int32_t w[HS_UNROLL], m[HS_UNROLL], uw[HS_UNROLL];
#pragma unroll
            for (int q = 0; q < HS_UNROLL; q++) {
                const eoff_t j = b0 + (eoff_t)q * stride + sub;
                u[q] = j < re ? g.col[j] : v;
                w[q] = j < re ? g.ew[j] : -1;
            }
#pragma unroll
            for (int q = 0; q < HS_UNROLL; q++) {
                m[q] = mate[u[q]];
                uw[q] = g.vw[u[q]];
            }
#pragma unroll
            for (int q = 0; q < HS_UNROLL; q++) {
                if (u[q] == v || m[q] >= 0 || (int64_t)uw[q] > room || w[q] < bw) continue;
                const uint32_t k = (uint32_t)mix64(seed + (uint64_t)u[q]);
                const eoff_t j = b0 + (eoff_t)q * stride + sub;
                if (hs_better(w[q], k, j, bw, bk, bj)) {
                    bw = w[q];
                    bk = k;
                    bj = j;
                }
            }
        }
#pragma unroll
        for (int d = 1; d < WAVE; d <<= 1) {
            const int32_t ow = __shfl_xor(bw, d, WAVE);
            const uint32_t ok = __shfl_xor(bk, d, WAVE);
            const eoff_t oj = (eoff_t)__shfl_xor((int64_t)bj, d, WAVE);
            if (hs_better(ow, ok, oj, bw, bk, bj)) {
                bw = ow;
                bk = ok;
                bj = oj;
            }
        }
    };
    for (int64_t v = (int64_t)wv * gridDim.x + blockIdx.x; v < g.n; v += (int64_t)gridDim.x * HS_WAVES) {
        if (mate[v] >= 0) {
            if (lane == 0) prop[v] = -1;
            continue;
        }
        const eoff_t rs = g.rowptr[v], re = g.rowptr[v + 1];
        if (re - rs > HS_LONG) {
            int32_t slot = 0;
            if (lane == 0) slot = atomicAdd(&nqueue, 1);
            slot = __shfl(slot, 0, WAVE);
            if (slot < HS_QUEUE) {
                if (lane == 0) queue[slot] = (vid_t)v;
                continue;
            }
        }
        int32_t bw;
        uint32_t bk;
        eoff_t bj;
        best((vid_t)v, rs, re, lane, WAVE, bw, bk, bj);
        if (lane == 0) prop[v] = bw >= 0 ? g.col[bj] : -1;
    }
    __syncthreads();
    const int32_t nq = min(nqueue, HS_QUEUE);
    for (int32_t q = 0; q < nq; q++) {
        const vid_t v = queue[q];
        int32_t bw;
        uint32_t bk;
        eoff_t bj;
        best(v, g.rowptr[v], g.rowptr[v + 1], threadIdx.x, HS_BLOCK, bw, bk, bj);
        if (lane == 0) {
            sw[wv] = bw;
            sk[wv] = bk;
            sj[wv] = bj;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < HS_WAVES; w++)
                if (hs_better(sw[w], sk[w], sj[w], bw, bk, bj)) {
                    bw = sw[w];
                    bk = sk[w];
                    bj = sj[w];
                }
            prop[v] = bw >= 0 ? g.col[bj] : -1;
        }
        __syncthreads();
    }
}

__global__ void k_mutual(vid_t n, const int32_t* prop, int32_t* mate) {
    FOR_THREAD(v, n) {
        const int32_t u = prop[v];
        if (u >= 0 && prop[u] == (vid_t)v) mate[v] = u;
    }
}

// The first neighbour of every vertex (-1: none).
__global__ void k_first_adj(DGraph g, int32_t* first) {
    FOR_THREAD(v, g.n) {
        const eoff_t rs = g.rowptr[v];
        first[v] = g.rowptr[v + 1] > rs ? g.col[rs] : -1;
    }
}

// Entries of each coarse row (those of its members, self-edges included), and
// the row's tier list.
constexpr int32_t FS_WAVE_MAX = 256;
constexpr int32_t FS_SMALL_MAX = 1024;
constexpr int32_t FS_BLOCK_MAX = 4096;

__global__ void __launch_bounds__(256)
    k_fs_sizes(DGraph g, vid_t nc, const vid_t* m1, const vid_t* m2, eoff_t* size, vid_t* lists, int32_t* cnt) {
    __shared__ int32_t sh[256 / WAVE + 1];
    FOR_BLOCK_UNIFORM(c, nc) {
        eoff_t sz = 0;
        if (c < nc) {
            const vid_t a = m1[c], b = m2[c];
            sz = g.rowptr[a + 1] - g.rowptr[a];
            if (b >= 0) sz += g.rowptr[b + 1] - g.rowptr[b];
            size[c] = sz;
        }
        const int tier = c >= nc ? -1 : sz <= FS_WAVE_MAX ? 0 : sz <= FS_SMALL_MAX ? 1 : sz <= FS_BLOCK_MAX ? 2 : 3;
        for (int q = 0; q < 4; q++) {
            const int32_t at = block_append<256>(&cnt[q], tier == q, sh);
            if (at >= 0) lists[(int64_t)q * nc + at] = (vid_t)c;
        }
    }
}

// Edge of the row's e-th entry: its first member's row, then its second's.
struct FsRow {
    eoff_t rs1, rs2;
    int32_t len1;
    int64_t len;
    __device__ FsRow(const DGraph& g, vid_t a, vid_t b) {
        rs1 = g.rowptr[a];
        len1 = (int32_t)(g.rowptr[a + 1] - rs1);
        rs2 = b >= 0 ? g.rowptr[b] : 0;
        len = len1 + (b >= 0 ? g.rowptr[b + 1] - rs2 : 0);
    }
    __device__ eoff_t edge(int64_t e) const { return e < len1 ? rs1 + e : rs2 + (e - len1); }
};

// Adds an entry to a table of mask + 1 slots (at most half full): the
// neighbour's weight and its first position. Returns the slot.
__device__ inline int32_t fs_insert(int32_t* key, int32_t* pos, int32_t* val, uint32_t mask, vid_t u, int32_t e,
                                    int32_t w) {
    uint32_t h = ((uint32_t)u * 0x9E3779B1u) & mask;
    for (;;) {
        const int32_t k = key[h];
        if (k == u) break;
        if (k < 0) {
            const int32_t old = atomicCAS(&key[h], -1, u);
            if (old < 0 || old == u) break;
        }
        h = (h + 1) & mask;
    }
    atomicMin(&pos[h], e);
    atomicAdd(&val[h], w);
    return (int32_t)h;
}

// A wave per row of up to FS_WAVE_MAX entries, four per lane.
constexpr int FS_WAVES = 4;
__global__ void __launch_bounds__(FS_WAVES* WAVE)
    k_fs_wave(DGraph g, const vid_t* map, const vid_t* m1, const vid_t* m2, const vid_t* list, int32_t nlist,
              const eoff_t* off, vid_t* tkey, wgt_t* tval, int32_t* ucount) {
    constexpr int CAP = 2 * FS_WAVE_MAX;
    constexpr int PER = FS_WAVE_MAX / WAVE;
    __shared__ int32_t key[FS_WAVES][CAP], pos[FS_WAVES][CAP], val[FS_WAVES][CAP];
    const int lane = threadIdx.x & (WAVE - 1);
    const int w = threadIdx.x / WAVE;
    int32_t *K = key[w], *O = pos[w], *V = val[w];
    for (int32_t r = blockIdx.x * FS_WAVES + w; r < nlist; r += gridDim.x * FS_WAVES) {
        const vid_t c = list[r];
        const FsRow row(g, m1[c], m2[c]);
        uint32_t cap = 64;
        while ((int64_t)cap < 2 * row.len) cap <<= 1;
        for (uint32_t t = lane; t < cap; t += WAVE) {
            K[t] = -1;
            O[t] = ORD_MAX;
            V[t] = 0;
        }
        wave_sync();
        vid_t u[PER];
        int32_t ew[PER], slot[PER];
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int64_t e = q * WAVE + lane;
            u[q] = -1;
            ew[q] = 0;
            if (e < row.len) {
                const eoff_t j = row.edge(e);
                u[q] = g.col[j];
                ew[q] = g.ew[j];
            }
        }
#pragma unroll
        for (int q = 0; q < PER; q++) u[q] = u[q] >= 0 ? map[u[q]] : c;
#pragma unroll
        for (int q = 0; q < PER; q++)
            slot[q] = u[q] != c ? fs_insert(K, O, V, cap - 1, u[q], q * WAVE + lane, ew[q]) : -1;
        wave_sync();
        const eoff_t o = off[c];
        int32_t base = 0;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const bool first = slot[q] >= 0 && O[slot[q]] == q * WAVE + lane;
            const uint64_t mk = __ballot(first);
            if (first) {
                const int32_t at = base + (int32_t)__popcll(mk & ((1ull << lane) - 1ull));
                tkey[o + at] = u[q];
                tval[o + at] = V[slot[q]];
            }
            base += (int32_t)__popcll(mk);
        }
        if (lane == 0) ucount[c] = base;
        wave_sync();
    }
}

// A workgroup per row of up to 4 * BLOCK entries, four per thread.
template <int BLOCK>
__global__ void __launch_bounds__(BLOCK)
    k_fs_block(DGraph g, const vid_t* map, const vid_t* m1, const vid_t* m2, const vid_t* list, int32_t nlist,
               const eoff_t* off, vid_t* tkey, wgt_t* tval, int32_t* ucount) {
    constexpr int CAP = 8 * BLOCK;
    extern __shared__ int32_t fs_lds[];
    __shared__ int32_t ws[BLOCK / WAVE + 1];
    int32_t *K = fs_lds, *O = fs_lds + CAP, *V = fs_lds + 2 * CAP;
    for (int32_t r = blockIdx.x; r < nlist; r += gridDim.x) {
        const vid_t c = list[r];
        const FsRow row(g, m1[c], m2[c]);
        uint32_t cap = BLOCK;
        while ((int64_t)cap < 2 * row.len) cap <<= 1;
        for (uint32_t t = threadIdx.x; t < cap; t += BLOCK) {
            K[t] = -1;
            O[t] = ORD_MAX;
            V[t] = 0;
        }
        __syncthreads();
        vid_t u[4];
        int32_t ew[4], slot[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int64_t e = q * BLOCK + threadIdx.x;
            u[q] = -1;
            ew[q] = 0;
            if (e < row.len) {
                const eoff_t j = row.edge(e);
                u[q] = g.col[j];
                ew[q] = g.ew[j];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; q++) u[q] = u[q] >= 0 ? map[u[q]] : c;
#pragma unroll
        for (int q = 0; q < 4; q++)
            slot[q] = u[q] != c ? fs_insert(K, O, V, cap - 1, u[q], q * BLOCK + threadIdx.x, ew[q]) : -1;
        __syncthreads();
        const eoff_t o = off[c];
        int32_t base = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const bool first = slot[q] >= 0 && O[slot[q]] == q * BLOCK + (int32_t)threadIdx.x;
            int32_t tot;
            const int32_t at = base + block_excl_scan<int32_t, BLOCK>(first ? 1 : 0, tot, ws);
            if (first) {
                tkey[o + at] = u[q];
                tval[o + at] = V[slot[q]];
            }
            base += tot;
        }
        if (threadIdx.x == 0) ucount[c] = base;
        __syncthreads();
    }
}

// Longer rows: a workgroup per row with position and weight arrays over all
// coarse vertices in memory, one of each per workgroup (ORD_MAX and 0 between
// rows).
__global__ void __launch_bounds__(1024)
    k_fs_dense(DGraph g, const vid_t* map, const vid_t* m1, const vid_t* m2, const vid_t* list, int32_t nlist,
               const eoff_t* off, vid_t nc, int32_t* dense, vid_t* tkey, wgt_t* tval, int32_t* ucount) {
    constexpr int BLOCK = 1024;
    __shared__ int32_t ws[BLOCK / WAVE + 1];
    int32_t* O = dense + (int64_t)blockIdx.x * nc;
    int32_t* V = dense + ((int64_t)gridDim.x + blockIdx.x) * nc;
    for (int32_t r = blockIdx.x; r < nlist; r += gridDim.x) {
        const vid_t c = list[r];
        const FsRow row(g, m1[c], m2[c]);
        for (int64_t e = threadIdx.x; e < row.len; e += BLOCK) {
            const eoff_t j = row.edge(e);
            const vid_t u = map[g.col[j]];
            if (u == c) continue;
            atomicMin(&O[u], (int32_t)e);
            atomicAdd(&V[u], g.ew[j]);
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
        const eoff_t o = off[c];
        int32_t base = 0;
        for (int64_t e0 = 0; e0 < row.len; e0 += 4 * BLOCK) {
            vid_t u[4];
            bool first[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int64_t e = e0 + q * BLOCK + threadIdx.x;
                u[q] = e < row.len ? map[g.col[row.edge(e)]] : c;
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                first[q] = u[q] != c && ld_rx(&O[u[q]]) == (int32_t)(e0 + q * BLOCK + threadIdx.x);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                int32_t tot;
                const int32_t at = base + block_excl_scan<int32_t, BLOCK>(first[q] ? 1 : 0, tot, ws);
                if (first[q]) {
                    tkey[o + at] = u[q];
                    tval[o + at] = ld_rx(&V[u[q]]);
                }
                base += tot;
            }
        }
        if (threadIdx.x == 0) ucount[c] = base;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
        // the row's neighbours (just written) back to the empty state
        for (int32_t e = threadIdx.x; e < base; e += BLOCK) {
            const vid_t u = ld_rx(&tkey[o + e]);
            O[u] = ORD_MAX;
            V[u] = 0;
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
    }
}

// Rows moved from their reserved stretches to their final offsets, a wave per
// row (a workgroup's waves share the long ones).
__global__ void __launch_bounds__(256)
    k_fs_pack(vid_t nc, const eoff_t* rowptr, const eoff_t* off, const vid_t* tkey, const wgt_t* tval, vid_t* col,
              wgt_t* ew) {
    __shared__ EdgeWalkLds walk;
    block_edges<256>(rowptr, nc, rowptr[nc], walk, [&](vid_t r, eoff_t j) {
        const eoff_t src = off[r] + (j - rowptr[r]);
        col[j] = tkey[src];
        ew[j] = tval[src];
    });
}

template <class T>
std::vector<T> fetch(const T* d, int64_t count, hipStream_t s) {
    std::vector<T> h((size_t)count);
    if (count > 0) JET_HIP(hipMemcpyAsync(h.data(), d, sizeof(T) * count, hipMemcpyDeviceToHost, s));
    JET_HIP(hipStreamSynchronize(s));
    return h;
}

}  // namespace

bool init_coarsen_device(const DGraph& g, std::vector<int32_t>& vw, uint64_t seed, int lvl, Arena& persist, Arena& a,
                         hipStream_t s, Level& out) {
    const vid_t n = g.n;
    ArenaScope sc(a);
    const uint64_t lseed = jet_init::level_seed(seed, lvl);
    int64_t total = 0;
    for (int32_t w : vw) total += w;
    const int64_t cap = jet_init::match_weight_cap(total);
    int32_t* mate = a.alloc<int32_t>(n);
    int32_t* prop = a.alloc<int32_t>(n);
    fill_i32(mate, -1, n, s);
    const int nb = grid_for(n, 256, 8192);
    for (int round = 0; round < jet_init::HANDSHAKE_ROUNDS; round++) {
        k_propose<<<512, HS_BLOCK, 0, s>>>(g, lseed, cap, mate, prop);
        k_mutual<<<nb, 256, 0, s>>>(n, prop, mate);
    }
    k_first_adj<<<nb, 256, 0, s>>>(g, prop);
    JET_LAUNCH_CHECK();
    std::vector<int32_t> h_mate = fetch(mate, n, s);
    const std::vector<int32_t> h_first = fetch(prop, n, s);
    jet_init::CoarseMap cm = jet_init::finish_matching(n, h_mate, h_first.data(), vw.data(), cap);
    const vid_t nc = cm.n;
    if (!jet_init::shrinks_enough(nc, n)) return false;
    // the coarse level's vertex arrays
    out.n = nc;
    out.uniform = false;
    out.map = persist.alloc<vid_t>(n);
    out.vw = persist.alloc<wgt_t>(nc);
    out.rowptr = persist.alloc<eoff_t>((int64_t)nc + 1);
    vid_t* m1 = a.alloc<vid_t>(nc);
    vid_t* m2 = a.alloc<vid_t>(nc);
    JET_HIP(hipMemcpyAsync(out.map, cm.map.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
    JET_HIP(hipMemcpyAsync(out.vw, cm.vw.data(), sizeof(int32_t) * nc, hipMemcpyHostToDevice, s));
    JET_HIP(hipMemcpyAsync(m1, cm.first.data(), sizeof(int32_t) * nc, hipMemcpyHostToDevice, s));
    JET_HIP(hipMemcpyAsync(m2, cm.second.data(), sizeof(int32_t) * nc, hipMemcpyHostToDevice, s));
    // its rows, at stretches of the members' lengths first
    eoff_t* off = a.alloc<eoff_t>((int64_t)nc + 1);
    vid_t* lists = a.alloc<vid_t>(4 * (int64_t)nc);
    int32_t* cnt = a.alloc<int32_t>(4);
    int32_t* ucount = a.alloc<int32_t>((int64_t)nc + 1);
    fill2_i32(cnt, 0, 4, ucount, 0, (int64_t)nc + 1, s);
    k_fs_sizes<<<grid_for(nc, 256, 8192), 256, 0, s>>>(g, nc, m1, m2, off, lists, cnt);
    JET_LAUNCH_CHECK();
    excl_scan_i64_i64(off, off, nc, a, s);
    int32_t h[4];
    read_i32_words(cnt, 4, h, s);
    vid_t* tkey = a.alloc<vid_t>(g.m);
    wgt_t* tval = a.alloc<wgt_t>(g.m);
    if (h[3] > 0) {
        // at most 1 GB of position and weight arrays, and no more than the
        // level's columns and weights take
        const int64_t fit = std::max<int64_t>(1, std::min<int64_t>(int64_t(1) << 30, 8 * (int64_t)g.m) / (8 * (int64_t)nc));
        const int G = (int)std::min<int64_t>({(int64_t)h[3], 512, fit});
        ArenaScope sd(a);
        int32_t* dense = a.alloc<int32_t>((int64_t)G * 2 * nc);
        fill2_i32(dense, ORD_MAX, (int64_t)G * nc, dense + (int64_t)G * nc, 0, (int64_t)G * nc, s);
        k_fs_dense<<<G, 1024, 0, s>>>(g, out.map, m1, m2, lists + 3 * (int64_t)nc, h[3], off, nc, dense, tkey, tval,
                                     ucount);
        JET_LAUNCH_CHECK();
    }
    if (h[2] > 0) {
        const size_t lds = 3 * sizeof(int32_t) * 8 * 1024;
        JET_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_fs_block<1024>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        k_fs_block<1024><<<std::min(h[2], 2048), 1024, lds, s>>>(g, out.map, m1, m2, lists + 2 * (int64_t)nc, h[2], off,
                                                                 tkey, tval, ucount);
        JET_LAUNCH_CHECK();
    }
    if (h[1] > 0) {
        k_fs_block<256><<<std::min(h[1], 8192), 256, 3 * sizeof(int32_t) * 8 * 256, s>>>(
            g, out.map, m1, m2, lists + (int64_t)nc, h[1], off, tkey, tval, ucount);
        JET_LAUNCH_CHECK();
    }
    if (h[0] > 0) {
        k_fs_wave<<<grid_for(h[0], FS_WAVES, 16384), FS_WAVES * WAVE, 0, s>>>(g, out.map, m1, m2, lists, h[0], off, tkey,
                                                                            tval, ucount);
        JET_LAUNCH_CHECK();
    }
    excl_scan_i32_i64(ucount, out.rowptr, nc, a, s);
    out.m = read_scalar(out.rowptr + nc, s);  // also: the copies from cm have been made
    out.col = persist.alloc<vid_t>(std::max<int64_t>(out.m, 1));
    out.ew = persist.alloc<wgt_t>(std::max<int64_t>(out.m, 1));
    if (out.m > 0) {
        k_fs_pack<<<grid_for(out.m, EB_TILE, 16384), 256, 0, s>>>(nc, out.rowptr, off, tkey, tval, out.col, out.ew);
        JET_LAUNCH_CHECK();
    }
    vw = std::move(cm.vw);
    return true;
}

}  // namespace jet
