// Contraction of one level (contract.hpp of the reference) in one launch, by a
// team of workgroups on one XCD (team_dev.h).
//
// The kernels of contract.hip are sixteen launches and two host reads, some
// 100 us on a level of a few thousand vertices, whatever its size: a
// hierarchy of small levels spends more time on launching its contractions
// than on its matchings. Here a level is counted, scanned, gathered,
// deduplicated and written with the team's barriers between the steps.
// Workgroups own chunks of 64 fine vertices in turn for the counts, and one
// block of consecutive coarse rows each. A coarse row of up to CT_GROUP_EDGES
// fine edges and four members is summed in an LDS hash table by 16 lanes (four
// rows at a time in a wave), up to CT_WAVE_EDGES by a wave, up to
// CT_BLOCK_EDGES by the workgroup. The rows are those of contract.hip: unique
// neighbours in increasing id, weights summed.
//
// Measured with its launch and the wait for the result, against the kernels of
// contract.hip: 24 against 72 us a level on the eight levels of a mesh of 4096
// vertices, 43 against 86 over the 74 small levels of a mesh of 166,833 whose
// matching stalls on a hub.
#include "contract_team.h"

#include <algorithm>
#include <mutex>

#include "contract_dev.h"
#include "prims.h"
#include "team_dev.h"
#include "tuning.h"
#include "wave.h"

namespace jet {

namespace {

constexpr int CT_BLOCK = 1024;
constexpr int CT_WAVES = CT_BLOCK / WAVE;
constexpr int CT_LANES = 16;
constexpr int CT_GROUPS = WAVE / CT_LANES;
constexpr int32_t CT_GROUP_EDGES = 32;
constexpr int32_t CT_GROUP_MEMBERS = 4;
constexpr int32_t CT_WAVE_EDGES = 128;
constexpr int32_t CT_BLOCK_EDGES = 2048;
// LDS words of a wave: group tables of 64 slots and their unique entries, or
// one table of 256, its unique entries and a chunk of 64 members
constexpr int32_t CT_WAVE_WORDS = 1024;
constexpr int32_t CT_ROWS_WG = 64;  // while the team is not at its largest (32 to 256: the same within 2%)
// Levels of more edges, or of more per coarse row, need the whole device: the
// levels of more than 16,384 vertices of a mesh of 65,536 (391,170 edges) take
// 0.14 ms less by the team, a stencil level of 46,131 (685,786 edges) 0.15 ms
// more.
constexpr int64_t CT_TEAM_M = 400000;
constexpr int64_t CT_TEAM_AVG = 64;
constexpr int CT_MAILBOX = 40;
constexpr int32_t CT_ROWS = TEAM_OWN;  // coarse rows of a workgroup at most
static_assert(CT_WAVES * CT_WAVE_WORDS >= 6 * CT_BLOCK_EDGES, "the workgroup's table and unique entries");

struct ContractCtl {
    TeamCtl team;
    int32_t too_long, pad1[31];
    int64_t sums[TEAM_MAX];    // a workgroup's rows: fine edges (high word) and members (low word)
    int64_t unique[TEAM_MAX];  // and coarse edges
};

struct ContractParams {
    DGraph g;
    const vid_t* map;
    int32_t nc, rows;  // rows of a workgroup
    int32_t team, xcd, start_spins;
    uint64_t* count;  // nc: fine edges (high word) and members (low word), zero at the launch
    int32_t* moff;    // nc
    vid_t* members;   // n
    vid_t* tkey;      // m
    wgt_t* tval;      // m
    eoff_t* rowptr;
    wgt_t* vw;  // zero at the launch
    char* out;  // columns, then at a multiple of 256 bytes the weights
    ContractCtl* ctl;
    int64_t* host_out;  // coarse edges (-1 not built, -2 failed, -3 abandoned), then the sequence word
    int64_t seq;
};

struct ContractShared {
    int64_t red[CT_WAVES + 1];
    int64_t base, total;
    int32_t h[CT_ROWS + 1];   // first fine edge of an own row
    int32_t m[CT_ROWS + 1];   // first member
    int32_t u[CT_ROWS + 1];   // unique neighbours, then the first coarse edge; before: places of own fine vertices
    uint16_t big[CT_ROWS];    // rows for the whole workgroup
    int32_t nbig, nu;
    int32_t go, size, me;
};

__device__ inline void ct_publish(const ContractParams& P, int64_t mc) {
    P.host_out[0] = mc;
    __threadfence_system();
    P.host_out[1] = P.seq;  // the host waits for this word
    __threadfence_system();
}

// Sum of x[0 .. c) and of x[0 .. T), T <= 64, by one wave.
__device__ inline void ct_prefix(const int64_t* x, int32_t T, int32_t c, int64_t& pre, int64_t& all) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t v = lane < T ? ldr64(&x[lane]) : 0;
    all = wave_reduce_sum(v);
    pre = wave_reduce_sum(lane < c ? v : 0);
}

// Row r of the workgroup by a wave: a table of up to 256 slots.
__device__ inline void ct_wave_row(const ContractParams& P, ContractShared& L, int32_t* lds, int32_t r, vid_t c) {
    const int lane = threadIdx.x & (WAVE - 1);
    int32_t* K = lds;
    int32_t* V = lds + 256;
    int32_t* UK = lds + 512;
    int32_t* UV = lds + 512 + CT_WAVE_EDGES;
    eoff_t* s_ex = reinterpret_cast<eoff_t*>(lds + 768);
    eoff_t* s_rs = s_ex + WAVE;
    const int32_t h0 = L.h[r], hsz = L.h[r + 1] - h0;
    int32_t cap = 64;
    while (cap < 2 * hsz) cap <<= 1;
    for (int32_t t = lane; t < cap; t += WAVE) {
        K[t] = EMPTY;
        V[t] = 0;
    }
    wave_sync();
    wave_row_edges(P.g, [&](int32_t x) { return ld_rx(&P.members[x]); }, L.m[r], L.m[r + 1], s_ex, s_rs, [&](eoff_t j) {
        const vid_t u = P.map[P.g.col[j]];
        if (u != c) lds_insert(K, V, cap - 1, u, P.g.ew[j]);
    });
    wave_sync();
    int32_t U = 0;
    for (int32_t t0 = 0; t0 < cap; t0 += WAVE) {
        const int32_t k = K[t0 + lane];
        const uint64_t bal = __ballot(k != EMPTY);
        const int32_t pos = U + (int32_t)__popcll(bal & ((1ull << lane) - 1ull));
        if (k != EMPTY) {
            UK[pos] = k;
            UV[pos] = V[t0 + lane];
        }
        U += (int32_t)__popcll(bal);
    }
    wave_sync();
    for (int32_t e = lane; e < U; e += WAVE) {
        const int32_t k = UK[e];
        int32_t rank = 0;
        for (int32_t q = 0; q < U; q++) rank += UK[q] < k ? 1 : 0;
        P.tkey[h0 + rank] = k;
        P.tval[h0 + rank] = UV[e];
    }
    if (lane == 0) L.u[r] = U;
    wave_sync();
}

}  // namespace

__global__ void k_contract_prep(ContractCtl* ctl, uint64_t* count, wgt_t* vw, int32_t nc) {
    FOR_THREAD(x, nc) {
        count[x] = 0;
        vw[x] = 0;
    }
    if (blockIdx.x == 0)
        for (int32_t x = threadIdx.x; x < (int32_t)(sizeof(ContractCtl) / 4); x += blockDim.x)
            reinterpret_cast<int32_t*>(ctl)[x] = 0;
}

__global__ void __launch_bounds__(CT_BLOCK) k_contract_team(ContractParams P) {
    extern __shared__ __align__(16) int32_t dyn[];
    __shared__ ContractShared L;
    const DGraph g = P.g;
    const vid_t n = g.n;
    const int32_t nc = P.nc;
    const int t = threadIdx.x;
    const int lane = t & (WAVE - 1);
    const int wv = t / WAVE;
    ContractCtl* C = P.ctl;
    if (t == 0) {
        const int32_t st = team_start(C->team, P.xcd, P.team, P.team, P.start_spins, L.go, L.size, L.me);
        if (st == TEAM_ABANDON) ct_publish(P, -3);
        L.nbig = 0;
    }
    __syncthreads();
    if (!L.go) return;
    const int32_t T = L.size, me = L.me;
    Team team{&C->team, T, me, 0, &L.go};
    auto for_own = [&](auto&& f) {  // fine vertices: f(x, i)
        for (int32_t x0 = WAVE * wv;; x0 += WAVE * CT_WAVES) {
            if (own_vertex(x0, WAVE, T, me) >= n) break;
            const int64_t i = own_vertex(x0 + lane, WAVE, T, me);
            if (i < n) f(x0 + lane, (vid_t)i);
        }
    };
    // ---- the rows' fine edges, members and weights; a member's place
    for_own([&](int32_t x, vid_t i) {
        const vid_t c = P.map[i];
        const uint64_t d = (uint64_t)(g.rowptr[i + 1] - g.rowptr[i]);
        L.u[x] = (int32_t)(uint32_t)atomicAdd((unsigned long long*)&P.count[c], (unsigned long long)((d << 32) | 1));
        atomicAdd(&P.vw[c], g.vw[i]);
    });
    bool alive = team.sync();
    // ---- their offsets: two consecutive rows a thread
    const int32_t c0 = min(nc, me * P.rows), nrows = min(nc, c0 + P.rows) - c0;
    int64_t pre = 0, v0 = 0, v1 = 0, tot = 0;
    if (alive) {
        v0 = 2 * t < nrows ? (int64_t)ldr64(&P.count[c0 + 2 * t]) : 0;
        v1 = 2 * t + 1 < nrows ? (int64_t)ldr64(&P.count[c0 + 2 * t + 1]) : 0;
        if ((v0 >> 32) > CT_BLOCK_EDGES || (v1 >> 32) > CT_BLOCK_EDGES) atomicOr(&C->too_long, 1);
        pre = block_excl_scan<int64_t, CT_BLOCK>(v0 + v1, tot, L.red);
        if (t == 0) C->sums[me] = tot;
        alive = team.sync();
    }
    if (alive && ld_rx(&C->too_long)) {
        if (me == 0 && t == 0) ct_publish(P, -1);
        return;
    }
    if (alive) {
        if (wv == 0) {
            int64_t b, all;
            ct_prefix(C->sums, T, me, b, all);
            if (lane == 0) L.base = b;
        }
        __syncthreads();
        const int64_t b = L.base + pre;
        if (2 * t <= nrows) {
            L.h[2 * t] = (int32_t)(b >> 32);
            L.m[2 * t] = (int32_t)(uint32_t)b;
        }
        if (2 * t + 1 <= nrows) {
            L.h[2 * t + 1] = (int32_t)((b + v0) >> 32);
            L.m[2 * t + 1] = (int32_t)(uint32_t)(b + v0);
        }
        if (nrows == 2 * CT_BLOCK && t == CT_BLOCK - 1) {
            L.h[nrows] = (int32_t)((b + v0 + v1) >> 32);
            L.m[nrows] = (int32_t)(uint32_t)(b + v0 + v1);
        }
        if (2 * t < nrows) P.moff[c0 + 2 * t] = (int32_t)(uint32_t)b;
        if (2 * t + 1 < nrows) P.moff[c0 + 2 * t + 1] = (int32_t)(uint32_t)(b + v0);
        alive = team.sync();
    }
    // ---- the rows' members
    if (alive) {
        for_own([&](int32_t x, vid_t i) { P.members[ld_rx(&P.moff[P.map[i]]) + L.u[x]] = i; });
        alive = team.sync();
    }
    // ---- unique neighbours
    if (alive) {
        int32_t* lds = dyn + wv * CT_WAVE_WORDS;
        const int grp = lane / CT_LANES, sub = lane & (CT_LANES - 1);
        int32_t* K = lds + grp * 64;
        int32_t* V = lds + 256 + grp * 64;
        int32_t* UK = lds + 512 + grp * CT_GROUP_EDGES;
        int32_t* UV = lds + 512 + CT_GROUPS * CT_GROUP_EDGES + grp * CT_GROUP_EDGES;
        for (int32_t x0 = CT_GROUPS * wv; x0 < nrows; x0 += CT_GROUPS * CT_WAVES) {
            const int32_t r = x0 + grp;
            const bool in = r < nrows;
            const int32_t h0 = in ? L.h[r] : 0, hsz = in ? L.h[r + 1] - h0 : 0;
            const int32_t m0 = in ? L.m[r] : 0, mn = in ? L.m[r + 1] - m0 : 0;
            const vid_t c = c0 + r;
            const bool small = in && hsz <= CT_GROUP_EDGES && mn <= CT_GROUP_MEMBERS;
            for (int s = sub; s < 64; s += CT_LANES) {
                K[s] = EMPTY;
                V[s] = 0;
            }
            // lane q < 4 of the group holds the q-th member's row
            eoff_t rs = 0;
            int32_t d = 0;
            if (small && sub < mn) {
                const vid_t i = ld_rx(&P.members[m0 + sub]);
                rs = g.rowptr[i];
                d = (int32_t)(g.rowptr[i + 1] - rs);
            }
            wave_sync();
            for (int32_t q0 = 0; q0 < CT_GROUP_EDGES; q0 += CT_LANES) {
                // edge q0 + sub of the members' concatenated rows
                int32_t e = q0 + sub;
                eoff_t j = -1;
#pragma unroll
                for (int q = 0; q < CT_GROUP_MEMBERS; q++) {
                    const int32_t dq = __shfl(d, grp * CT_LANES + q, WAVE);
                    const eoff_t rq = (eoff_t)__shfl((int64_t)rs, grp * CT_LANES + q, WAVE);
                    if (j < 0 && e < dq) j = rq + e;
                    e -= dq;
                }
                if (small && j >= 0) {
                    const vid_t u = P.map[g.col[j]];
                    if (u != c) lds_insert(K, V, 63, u, g.ew[j]);
                }
            }
            wave_sync();
            int32_t U = 0;
            for (int s0 = 0; s0 < 64; s0 += CT_LANES) {
                const int32_t k = K[s0 + sub];
                const bool has = small && k != EMPTY;
                const uint32_t bal = (uint32_t)(__ballot(has) >> (grp * CT_LANES)) & ((1u << CT_LANES) - 1u);
                if (has) {
                    const int32_t pos = U + __popc(bal & ((1u << sub) - 1u));
                    UK[pos] = k;
                    UV[pos] = V[s0 + sub];
                }
                U += __popc(bal);
            }
            wave_sync();
            for (int32_t e = sub; e < U; e += CT_LANES) {
                const int32_t k = UK[e];
                int32_t rank = 0;
                for (int32_t q = 0; q < U; q++) rank += UK[q] < k ? 1 : 0;
                P.tkey[h0 + rank] = k;
                P.tval[h0 + rank] = UV[e];
            }
            if (small && sub == 0) L.u[r] = U;
            if (in && hsz > CT_WAVE_EDGES && sub == 0) L.big[atomicAdd(&L.nbig, 1)] = (uint16_t)r;
            wave_sync();
            uint64_t mid = __ballot(in && !small && hsz <= CT_WAVE_EDGES && sub == 0);
            while (mid) {
                const int b = (__ffsll((unsigned long long)mid) - 1) / CT_LANES;
                mid &= mid - 1;
                ct_wave_row(P, L, lds, x0 + b, c0 + x0 + b);
            }
        }
        __syncthreads();
        // rows for the whole workgroup: tables of 2 * CT_BLOCK_EDGES slots
        const int32_t nbig = L.nbig;
        for (int32_t x = 0; x < nbig; x++) {
            const int32_t r = L.big[x];
            const vid_t c = c0 + r;
            const int32_t h0 = L.h[r], hsz = L.h[r + 1] - h0;
            int32_t cap = 2 * CT_WAVE_EDGES;
            while (cap < 2 * hsz) cap <<= 1;
            int32_t* BK = dyn;
            int32_t* BV = dyn + 2 * CT_BLOCK_EDGES;
            int32_t* BU = dyn + 4 * CT_BLOCK_EDGES;
            int32_t* BW = dyn + 5 * CT_BLOCK_EDGES;
            for (int32_t s = t; s < cap; s += CT_BLOCK) {
                BK[s] = EMPTY;
                BV[s] = 0;
            }
            if (t == 0) L.nu = 0;
            __syncthreads();
            // a wave per member: members of a long row are many, or long themselves
            for (int32_t q = L.m[r] + wv; q < L.m[r + 1]; q += CT_WAVES) {
                const vid_t i = ld_rx(&P.members[q]);
                const eoff_t re = g.rowptr[i + 1];
                for (eoff_t j = g.rowptr[i] + lane; j < re; j += WAVE) {
                    const vid_t u = P.map[g.col[j]];
                    if (u != c) lds_insert(BK, BV, cap - 1, u, g.ew[j]);
                }
            }
            __syncthreads();
            for (int32_t s = t; s < cap; s += CT_BLOCK) {
                const int32_t pos = wave_append(&L.nu, BK[s] != EMPTY);
                if (pos >= 0) {
                    BU[pos] = BK[s];
                    BW[pos] = BV[s];
                }
            }
            __syncthreads();
            const int32_t U = L.nu;
            for (int32_t e = t; e < U; e += CT_BLOCK) {
                const int32_t k = BU[e];
                int32_t rank = 0;
                for (int32_t q = 0; q < U; q++) rank += BU[q] < k ? 1 : 0;
                P.tkey[h0 + rank] = k;
                P.tval[h0 + rank] = BW[e];
            }
            if (t == 0) L.u[r] = U;
            __syncthreads();
        }
        // ---- the coarse rows' offsets
        const int32_t u0 = 2 * t < nrows ? L.u[2 * t] : 0, u1 = 2 * t + 1 < nrows ? L.u[2 * t + 1] : 0;
        pre = block_excl_scan<int64_t, CT_BLOCK>((int64_t)u0 + u1, tot, L.red);
        if (t == 0) C->unique[me] = tot;
        alive = team.sync();
        if (alive) {
            if (wv == 0) {
                int64_t b, all;
                ct_prefix(C->unique, T, me, b, all);
                if (lane == 0) {
                    L.base = b;
                    L.total = all;
                }
            }
            __syncthreads();
            const int64_t mc = L.total, b = L.base + pre;
            if (me == 0 && t == 0) {
                ct_publish(P, mc);
                P.rowptr[nc] = mc;
            }
            if (2 * t < nrows) {
                P.rowptr[c0 + 2 * t] = b;
                L.u[2 * t] = (int32_t)b;
            }
            if (2 * t + 1 < nrows) {
                P.rowptr[c0 + 2 * t + 1] = b + u0;
                L.u[2 * t + 1] = (int32_t)b + u0;
            }
            if (t == 0) L.u[nrows] = (int32_t)(L.base + tot);
            __syncthreads();
            vid_t* col = reinterpret_cast<vid_t*>(P.out);
            wgt_t* ew = reinterpret_cast<wgt_t*>(P.out + ((4 * mc + 255) & ~int64_t(255)));
            for (int32_t r = t / CT_LANES; r < nrows; r += CT_BLOCK / CT_LANES) {
                const int32_t d0 = L.u[r], d1 = L.u[r + 1], src = L.h[r];
                for (int32_t q = sub; q < d1 - d0; q += CT_LANES) {
                    col[d0 + q] = ld_rx(&P.tkey[src + q]);
                    ew[d0 + q] = ld_rx(&P.tval[src + q]);
                }
            }
        }
    }
    if (!alive && me == 0 && t == 0) ct_publish(P, -2);
}

// ---------------------------------------------------------------- host side
bool team_contract_fits(int64_t n, int64_t m, int64_t nc) {
    return n >= 1 && nc >= 1 && m >= 1 && n <= team_max_n() && nc <= n && m <= CT_TEAM_M &&
           m <= CT_TEAM_AVG * nc;
}

bool contract_team(const DGraph& g, const vid_t* map, vid_t nc, Arena& persist, Arena& a, hipStream_t s, Level& out) {
    static std::once_flag once[64];
    static hipError_t rc[64];
    constexpr size_t lds = sizeof(int32_t) * CT_WAVES * CT_WAVE_WORDS;
    int dev = 0;
    JET_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) throw DeviceError("device index beyond 64");
    std::call_once(once[dev], [&] {
        rc[dev] = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_contract_team),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    JET_HIP(rc[dev]);
    const Arena::Mark start = persist.mark();
    ArenaScope sc(a);
    ContractParams P{};
    P.g = g;
    P.map = map;
    P.nc = nc;
    // at most CT_ROWS fine vertices each, too
    P.team = (int32_t)std::max<int64_t>(ceil_div((int64_t)g.n, (int64_t)CT_ROWS),
                                        std::min<int64_t>(TEAM_MAX, ceil_div((int64_t)nc, CT_ROWS_WG)));
    P.rows = (int32_t)ceil_div((int64_t)nc, (int64_t)P.team);
    if (P.rows > CT_ROWS || ceil_div((int64_t)g.n, (int64_t)P.team * WAVE) * WAVE > CT_ROWS)
        throw DeviceError("team contraction: level outside the kernel's limits");
    P.rowptr = persist.alloc<eoff_t>((int64_t)nc + 1);
    P.vw = persist.alloc<wgt_t>(nc);
    // columns and weights for as many edges as the fine level has; cut to
    // the coarse level's below
    const size_t upper = 2 * (((size_t)g.m * 4 + 255) & ~size_t(255));
    P.out = static_cast<char*>(persist.alloc_bytes(upper));
    const Arena::Mark end = persist.mark();
    P.count = a.alloc<uint64_t>(nc);
    P.moff = a.alloc<int32_t>(nc);
    P.members = a.alloc<vid_t>(g.n);
    P.tkey = a.alloc<vid_t>(g.m);
    P.tval = a.alloc<wgt_t>(g.m);
    P.ctl = a.alloc<ContractCtl>(1);
    Mailbox& mb = thread_mailbox();
    P.host_out = mb.dev + CT_MAILBOX;
    volatile int64_t* res = mb.host + CT_MAILBOX;
    P.seq = ++mb.seq;
    TeamSlot slot(P.team);
    P.xcd = slot.xcd();
    P.start_spins = (int32_t)tuning().team_start_spins;
    k_contract_prep<<<grid_for(nc, 256, 256), 256, 0, s>>>(P.ctl, P.count, P.vw, nc);
    k_contract_team<<<P.team == 1 ? 1 : 8 * P.team, CT_BLOCK, lds, s>>>(P);
    JET_LAUNCH_CHECK();
    const bool ran = wait_mailbox(&res[1], P.seq, s);
    const int64_t mc = ran ? res[0] : -3;
    if (mc == -2) throw DeviceError("team contraction made no progress");
    if (mc < 0) {
        if (mc == -3) team_abandoned();
        JET_HIP(hipStreamSynchronize(s));  // the kernel's last stores to what is released here
        persist.release(start);
        return false;
    }
    persist.release({end.ci, end.off - upper});
    out.n = nc;
    out.m = mc;
    out.rowptr = P.rowptr;
    out.vw = P.vw;
    out.col = persist.alloc<vid_t>(mc);
    out.ew = persist.alloc<wgt_t>(mc);
    return true;
}

}  // namespace jet
