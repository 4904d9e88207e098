// Evaluators: edge cut and J(C,D,Pi), block weights, and graph metadata.
//
// edge cut  = sum over directed (u,v) of w * [P(u) != P(v)], halved
//             (src/utility/edge_cut.h:71-90)
// J         = sum over directed (u,v) of w * D[P(u)][P(v)], not halved
//             (src/utility/comm_cost.h:36-56)
// Both accumulate in 64 bits (the reference's s32 sums overflow on large
// weighted graphs).  One streaming pass over the CSR; the reference's COO
// source array edges_u is not needed: a workgroup takes a contiguous share of
// the edges, whatever the degrees, and finds an edge's source by a search in
// the offsets it holds in LDS.  D lives in LDS when k*k <= 16384.  The input
// checks run in one launch before it and the evaluator tests their result on
// the device, so a call waits for the device once.
//
// Algorithmic bytes per launch: 4(n+1) + 4m(1+w) + 4n.
#include "eval.hpp"

namespace heipa {

namespace {

// out[0] the largest degree, out[1] the number of hubs: one update each per
// workgroup over a small grid (per-wave updates of one address serialise)
__global__ __launch_bounds__(256) void degrees_kernel(const u32 *xadj, u32 n, u32 hub_deg, u32 *out) {
    __shared__ u32 s_deg, s_hubs;
    if (threadIdx.x == 0) s_deg = s_hubs = 0;
    __syncthreads();
    u32 mx = 0, hubs = 0;
    for (u64 u = (u64) blockIdx.x * blockDim.x + threadIdx.x; u < n; u += (u64) gridDim.x * blockDim.x) {
        const u32 d = xadj[u + 1] - xadj[u];
        mx = d > mx ? d : mx;
        hubs += d > hub_deg ? 1u : 0u;
    }
    mx = wave_max(mx);
    hubs = wave_sum(hubs);
    if (lane_id() == 0) {
        atomicMax(&s_deg, mx);
        if (hubs) atomicAdd(&s_hubs, hubs);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicMax(&out[0], s_deg);
        if (s_hubs) atomicAdd(&out[1], s_hubs);
    }
}

__global__ void hub_list_kernel(const u32 *xadj, u32 n, u32 hub_deg, u32 *count, u32 *list) {
    for (u64 u = (u64) blockIdx.x * blockDim.x + threadIdx.x; u < n; u += (u64) gridDim.x * blockDim.x)
        if (xadj[u + 1] - xadj[u] > hub_deg) list[atomicAdd(count, 1u)] = (u32) u;
}

constexpr int EVAL_BLOCK = 512;
constexpr u32 D_LDS_MAX = 16384;  // k*k entries kept in LDS
constexpr u32 EVAL_ROWS = 2048;   // source vertices whose offsets a workgroup holds at a time
constexpr u32 EVAL_SHARE = 1024;  // edges per workgroup, at least ...
constexpr u32 EVAL_PER_CU = 2;    // ... of a grid of at most this many per CU

// The number of entries <= key among the non-decreasing x[0, n), by one wave:
// 64 probes per step instead of one (n = 2^18: three dependent loads, not 18).
// Stays inside x for any contents.
__device__ __forceinline__ u32 wave_upper_bound(const u32 *x, u32 n, u32 key) {
    u32 lo = 0, end = n;
    while (lo < end) {
        const u32 stride = (end - lo + WAVE - 1) / WAVE;
        const u64 i = (u64) lo + (u64) (lane_id() + 1) * stride - 1;
        const u32 c = (u32) __popcll(__ballot(i < end && x[i] <= key));
        const u64 next = (u64) lo + (u64) c * stride;
        if (stride == 1) return next < end ? (u32) next : end;
        lo = next < end ? (u32) next : end;
        end = end - lo < stride ? end : lo + stride;
    }
    return lo;
}

// What the checks found.  `flags` is zero before the launch and updated only
// by workgroups that found something: bit 0 bad offsets, 1 bad id, 2 bad edge
// weight, 3 bad vertex weight, 4 self loop, 5 block id >= k.  The degrees come
// as one partial per workgroup, reduced by the host (a thousand updates of one
// address took longer than the reads: about 15 ns each).
struct CheckPart {
    u32 max_deg, n_hubs;
};

// Input checks, one launch: xadj monotone within [0, m], neighbour ids < n,
// edge weights > 0, vertex weights >= 0, no self loops; the largest degree,
// the hubs and the largest block id beside them.  Vertices and edges are
// shared out evenly whatever the degrees; edge j is a self loop iff it lies in
// its neighbour's row, and only a neighbour among the share's own source
// vertices can own it, so almost no edge reads an offset.  A row scan per
// vertex took 809 us on R-MAT 2^18 (7.6 M edges) where the reads need 15.
__global__ __launch_bounds__(EVAL_BLOCK) void check_kernel(DGraph g, const u32 *__restrict__ part, u32 k, u32 hub_deg,
                                                           u32 *flags, CheckPart *parts) {
    __shared__ u32 s_lo[2];
    __shared__ u32 s_flags, s_hubs, s_deg;
    if (threadIdx.x == 0) s_flags = s_hubs = s_deg = 0;
    const u32 share = (u32) (((u64) g.m + gridDim.x - 1) / gridDim.x);
    const u64 b0 = (u64) blockIdx.x * share;
    const u32 c0 = b0 < g.m ? (u32) b0 : g.m;
    const u32 c1 = g.m - c0 < share ? g.m : c0 + share;
    if (c0 < c1 && g.xadj && threadIdx.x < 2 * WAVE) {  // the vertices whose rows hold edges c0 .. c1 - 1
        const u32 q = threadIdx.x / WAVE;
        const u32 ub = wave_upper_bound(g.xadj, g.n + 1, q ? c1 - 1 : c0);
        if (lane_id() == 0) s_lo[q] = ub;
    }
    __syncthreads();
    u32 f = 0, deg = 0, hubs = 0;
    for (u64 u = (u64) blockIdx.x * EVAL_BLOCK + threadIdx.x; u < g.n; u += (u64) gridDim.x * EVAL_BLOCK) {
        const u32 b = g.xadj[u], e = g.xadj[u + 1];
        if (b > e || e > g.m) {
            f |= 1u;
        } else {
            deg = e - b > deg ? e - b : deg;
            hubs += e - b > hub_deg ? 1u : 0u;
        }
        if (g.vw && g.vw[u] < 0) f |= 8u;
        if (part && part[u] >= k) f |= 32u;
    }
    if (c0 < c1 && g.xadj) {
        const u32 lo = s_lo[0] ? s_lo[0] - 1 : 0, hi = s_lo[1];  // source vertices [lo, hi)
        for (u64 j0 = (u64) c0 + threadIdx.x; j0 < c1; j0 += EVAL_BLOCK * 4) {
            u32 v[4];
            s32 w[4];
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                const u64 j = j0 + q * EVAL_BLOCK;
                v[q] = j < c1 ? g.adj[j] : 0u;
                w[q] = j < c1 && g.ew ? g.ew[j] : 1;
            }
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                const u64 j = j0 + q * EVAL_BLOCK;
                if (j >= c1) continue;
                f |= w[q] <= 0 ? 4u : 0u;
                if (v[q] >= g.n) f |= 2u;
                else if (v[q] >= lo && v[q] < hi && g.xadj[v[q]] <= j && j < g.xadj[v[q] + 1]) f |= 16u;
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && g.xadj && (g.xadj[0] != 0 || g.xadj[g.n] != g.m)) f |= 1u;
    if (f) atomicOr(&s_flags, f);
    deg = wave_max(deg);
    hubs = wave_sum(hubs);
    if (lane_id() == 0) {
        atomicMax(&s_deg, deg);
        if (hubs) atomicAdd(&s_hubs, hubs);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_flags) atomicOr(flags, s_flags);
        parts[blockIdx.x] = CheckPart{s_deg, s_hubs};
    }
}

// MODE 0: edge cut, MODE 1: J with D; one partial sum per workgroup, added up
// by the host.  `bad`: the checks' flags (null: the graph is known to be
// sound); nothing is read through the graph if they are set.
template<bool UEW, int MODE, bool D_LDS>
__global__ __launch_bounds__(EVAL_BLOCK) void eval_kernel(DGraph g, const u32 *__restrict__ part,
                                                          const s32 *__restrict__ D, u32 k, const u32 *bad,
                                                          s64 *out) {
    extern __shared__ s32 sD[];
    __shared__ u32 sx[EVAL_ROWS + 1], sp[EVAL_ROWS];
    __shared__ u32 s_lo[2];
    __shared__ s64 red[EVAL_BLOCK / WAVE];
    const u32 share = (u32) (((u64) g.m + gridDim.x - 1) / gridDim.x);
    const u64 b0 = (u64) blockIdx.x * share;
    if (b0 >= g.m || (bad && *bad)) {
        if (threadIdx.x == 0) out[blockIdx.x] = 0;
        return;
    }
    const u32 c0 = (u32) b0;
    const u32 c1 = g.m - c0 < share ? g.m : c0 + share;
    const s32 *Dp = D;
    if constexpr (MODE == 1 && D_LDS) {
        for (u32 i = threadIdx.x; i < k * k; i += EVAL_BLOCK) sD[i] = D[i];
        Dp = sD;
    }
    if (threadIdx.x < 2 * WAVE) {  // the source vertices of edges c0 .. c1 - 1
        const u32 q = threadIdx.x / WAVE;
        const u32 ub = wave_upper_bound(g.xadj, g.n + 1, q ? c1 - 1 : c0);
        if (lane_id() == 0) s_lo[q] = ub;
    }
    __syncthreads();
    s64 acc = 0;
    u32 c = c0;
    const u32 hi = s_lo[1];
    for (u32 lo = s_lo[0] - 1; c < c1; lo += EVAL_ROWS) {  // xadj[0] = 0 <= c0
        const u32 rows = hi - lo < EVAL_ROWS ? hi - lo : EVAL_ROWS;
        for (u32 i = threadIdx.x; i <= rows; i += EVAL_BLOCK) {
            sx[i] = g.xadj[lo + i];
            if (i < rows) sp[i] = part[lo + i];
        }
        __syncthreads();
        const u32 end = sx[rows] < c1 ? sx[rows] : c1;
        const u32 cnt = end - c;  // counted from c: offsets up to 2^32 - 1 never wrap
        const u32 *adj = g.adj + c;
        const s32 *ew = UEW ? nullptr : g.ew + c;
        for (u32 x0 = threadIdx.x; x0 < cnt; x0 += EVAL_BLOCK * 4) {
            u32 v[4];
            s32 w[4];
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                const u32 x = x0 + q * EVAL_BLOCK;
                v[q] = x < cnt ? adj[x] : 0u;
                w[q] = UEW ? 1 : x < cnt ? ew[x] : 0;
            }
#pragma unroll
            for (u32 q = 0; q < 4; ++q) v[q] = x0 + q * EVAL_BLOCK < cnt ? part[v[q]] : 0u;
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                const u32 x = x0 + q * EVAL_BLOCK, j = c + x;
                if (x >= cnt) continue;
                u32 a = 0, b = rows;  // the last row that starts at or before j
                while (b - a > 1) {
                    const u32 mid = (a + b) >> 1;
                    if (sx[mid] <= j) a = mid;
                    else b = mid;
                }
                const u32 pu = sp[a];
                if constexpr (MODE == 0) acc += v[q] != pu ? (s64) w[q] : 0;
                else acc += (s64) w[q] * (s64) Dp[(u64) pu * k + v[q]];
            }
        }
        c = end;
        __syncthreads();
    }
    acc = block_sum<EVAL_BLOCK>(acc, red);
    if (threadIdx.x == 0) out[blockIdx.x] = acc;
}

// at most as many workgroups as their partial results (8 bytes each of the
// checks and of the evaluator) fit the free scratch
u32 eval_grid(const Ctx &c, u64 items) {
    const u64 room = (c.arena.free_bytes() & ~(size_t) 255) / 16;
    return (u32) std::min<u64>(grid_for(c, items, EVAL_SHARE, EVAL_PER_CU), room > 1 ? room - 1 : 1);
}

void eval_launch(Ctx &c, const DGraph &g, const u32 *part, const s32 *D, u32 k, int mode, const u32 *bad, u32 groups,
                 s64 *out) {
    const bool uew = g.ew == nullptr;
    const double bytes = 4.0 * (g.n + 1) + 4.0 * g.m * (uew ? 1 : 2) + 4.0 * g.n;
    const dim3 grid(groups), block(EVAL_BLOCK);
    const bool dl = mode == 1 && (u64) k * k <= D_LDS_MAX;
    const size_t shmem = dl ? sizeof(s32) * k * k : 0;
    const char *name = mode == 0 ? "edge_cut" : "comm_cost";
#define EV(UEWv, MODEv, DLv) launch(c, name, bytes, grid, block, shmem, eval_kernel<UEWv, MODEv, DLv>, g, part, D, k, bad, out)
    if (mode == 0) {
        if (uew) EV(true, 0, false);
        else EV(false, 0, false);
    } else if (dl) {
        if (uew) EV(true, 1, true);
        else EV(false, 1, true);
    } else {
        if (uew) EV(true, 1, false);
        else EV(false, 1, false);
    }
#undef EV
}

// block weights: LDS histogram per workgroup, then global 64-bit atomics
template<bool UVW>
__global__ __launch_bounds__(256) void block_weights_kernel(u32 n, const u32 *__restrict__ part,
                                                            const s32 *__restrict__ vw, u32 k,
                                                            unsigned long long *bw, const u32 *bad) {
    extern __shared__ unsigned long long hist[];
    if (bad && *bad) return;
    for (u32 i = threadIdx.x; i < k; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    for (u64 u = (u64) blockIdx.x * blockDim.x + threadIdx.x; u < n; u += (u64) gridDim.x * blockDim.x)
        atomicAdd(&hist[part[u]], (unsigned long long) (UVW ? 1 : vw[u]));
    __syncthreads();
    for (u32 i = threadIdx.x; i < k; i += blockDim.x)
        if (hist[i]) atomicAdd(&bw[i], hist[i]);
}

// block weights for k beyond the LDS histogram: global 64-bit atomics
template<bool UVW>
__global__ __launch_bounds__(256) void block_weights_global_kernel(u32 n, const u32 *__restrict__ part,
                                                                   const s32 *__restrict__ vw, u32 k,
                                                                   unsigned long long *bw, const u32 *bad) {
    if (bad && *bad) return;
    for (u64 u = (u64) blockIdx.x * blockDim.x + threadIdx.x; u < n; u += (u64) gridDim.x * blockDim.x) {
        const s64 w = UVW ? 1 : vw[u];
        if (w) atomicAdd(&bw[part[u]], (unsigned long long) w);
    }
}

} // namespace

namespace {

// one device buffer for a call's results, copied back at once: the flags, the
// checks' partials, then the evaluator's
struct Checks {
    u32 grid_c, grid_e;
    char *dev;
    size_t bytes;
    u32 *flags() const { return (u32 *) dev; }
    CheckPart *parts() const { return (CheckPart *) (dev + 8); }
    s64 *sums() const { return (s64 *) (dev + 8 + sizeof(CheckPart) * grid_c); }
};
Checks check_launch(Ctx &c, BackScope &bs, const DGraph &g, const u32 *part, u32 k, u32 hub_deg, bool eval) {
    Checks r;
    r.grid_c = eval_grid(c, std::max<u64>(g.m, g.n + 1));
    r.grid_e = eval ? eval_grid(c, g.m) : 0;
    r.bytes = 8 + sizeof(CheckPart) * r.grid_c + 8ull * r.grid_e;
    r.dev = bs.get<char>(r.bytes);
    fill<u32>(c, r.flags(), 1, 0u);
    launch(c, "validate", 4.0 * (g.n + 1) + 4.0 * g.m * (g.ew ? 2 : 1), dim3(r.grid_c), dim3(EVAL_BLOCK), 0, check_kernel,
           g, part, k, hub_deg, r.flags(), r.parts());
    return r;
}
void check_throw(u32 f) {
    if (f & 1u) throw Error(HEIPA_ERR_INVALID, "invalid graph: xadj is not a monotone offset array ending at m");
    if (f & 2u) throw Error(HEIPA_ERR_INVALID, "invalid graph: neighbour id >= n");
    if (f & 4u) throw Error(HEIPA_ERR_INVALID, "invalid graph: edge weights must be positive");
    if (f & 8u) throw Error(HEIPA_ERR_INVALID, "invalid graph: vertex weights must be non-negative");
    if (f & 16u) throw Error(HEIPA_ERR_INVALID, "invalid graph: self loops are not allowed");
    if (f & 32u) throw Error(HEIPA_ERR_INVALID, "partition holds a block id >= k");
}
} // namespace

GraphMeta meta_of(const DGraph &g) {
    GraphMeta meta;
    meta.G = group_for_avg(g.n ? (double) g.m / (double) g.n : 0.0);
    meta.hub_deg = std::max<u32>(512, 32 * meta.G);
    return meta;
}
void hub_list(Ctx &c, const DGraph &g, GraphMeta &meta, bool back) {
    if (!meta.n_hubs) return;
    meta.hubs = (u32 *) (back ? c.arena.push_back(4ull * (meta.n_hubs + 1)) : c.arena.push_front(4ull * (meta.n_hubs + 1)));
    u32 *cnt = meta.hubs + meta.n_hubs;
    fill<u32>(c, cnt, 1, 0u);
    launch(c, "graph_meta", 4.0 * (g.n + 1), dim3(grid_for(c, g.n, 256)), dim3(256), 0, hub_list_kernel, g.xadj, g.n,
           meta.hub_deg, cnt, meta.hubs);
}
void meta_launch(Ctx &c, const DGraph &g, const GraphMeta &meta, u32 *out) {
    launch(c, "graph_meta", 4.0 * (g.n + 1), dim3(grid_for(c, g.n, 256 * 4, 2)), dim3(256), 0, degrees_kernel, g.xadj, g.n,
           meta.hub_deg, out);
}

// the checks alone, and their wait; adds up the degrees in meta
static void check(Ctx &c, const DGraph &g, const u32 *part, u32 k, GraphMeta &meta) {
    BackScope bs(c.arena);
    const Checks r = check_launch(c, bs, g, part, k, meta.hub_deg, false);
    std::vector<char> h(r.bytes);
    readback(c, h.data(), (const char *) r.dev, r.bytes);
    u32 f;
    std::memcpy(&f, h.data(), 4);
    check_throw(f);
    for (u32 i = 0; i < r.grid_c; ++i) {
        CheckPart p;
        std::memcpy(&p, h.data() + 8 + sizeof(p) * i, sizeof(p));
        meta.max_deg = std::max(meta.max_deg, p.max_deg);
        meta.n_hubs += p.n_hubs;
    }
}

GraphMeta validate(Ctx &c, const DGraph &g, const u32 *part, u32 k) {
    GraphMeta meta = meta_of(g);
    check(c, g, part, k, meta);
    hub_list(c, g, meta, true);
    return meta;
}

GraphMeta make_meta(Ctx &c, const DGraph &g, bool back) {
    GraphMeta meta = meta_of(g);
    if (g.n == 0) return meta;
    {
        BackScope bs(c.arena);
        u32 *scr = bs.get<u32>(2);
        fill<u32>(c, scr, 2, 0u);
        meta_launch(c, g, meta, scr);
        u32 h[2];
        readback(c, h, scr, 2);
        meta.max_deg = h[0];
        meta.n_hubs = h[1];
    }
    hub_list(c, g, meta, back);
    return meta;
}

// the checked entry points' form: checks and evaluation queued together, one
// wait for both results
static s64 evaluate_checked(Ctx &c, const DGraph &g, const u32 *part, const s32 *D, u32 k) {
    BackScope bs(c.arena);
    const Checks r = check_launch(c, bs, g, D ? part : nullptr, k, ~0u, true);
    eval_launch(c, g, part, D, k, D ? 1 : 0, r.flags(), r.grid_e, r.sums());
    std::vector<char> h(r.bytes);
    readback(c, h.data(), (const char *) r.dev, r.bytes);
    u32 f;
    std::memcpy(&f, h.data(), 4);
    check_throw(f);
    s64 sum = 0;
    for (u32 i = 0; i < r.grid_e; ++i) {
        s64 x;
        std::memcpy(&x, h.data() + ((char *) (r.sums() + i) - r.dev), 8);
        sum += x;
    }
    return sum;
}
s64 edge_cut_checked(Ctx &c, const DGraph &g, const u32 *part) {
    return evaluate_checked(c, g, part, nullptr, 0) / 2;
}
s64 comm_cost_checked(Ctx &c, const DGraph &g, const u32 *part, const s32 *D, u32 k) {
    return evaluate_checked(c, g, part, D, k);
}
void block_weights_checked(Ctx &c, const DGraph &g, const u32 *part, u32 k, s64 *bw_host) {
    BackScope bs(c.arena);
    if (!c.arena.spare(8ull * k, 0)) {  // one after the other in the same scratch, a wait each
        GraphMeta meta = meta_of(g);
        check(c, g, part, k, meta);
        s64 *bw = bs.get<s64>(k);
        block_weights_dev(c, g, part, k, bw);
        readback(c, bw_host, bw, k);
        return;
    }
    s64 *bw = bs.get<s64>(k);
    const Checks r = check_launch(c, bs, g, part, k, ~0u, false);
    block_weights_dev(c, g, part, k, bw, r.flags());
    // the caller's array is written only once the checks are known to have passed
    std::vector<s64> h;
    s64 *got = (s64 *) ((char *) c.pinned + 64);
    if (8ull * k + 64 > c.pinned_bytes) {
        h.resize(k);
        got = h.data();
    }
    copy_d2h(c, c.pinned, r.flags(), 4);
    copy_d2h(c, got, bw, 8ull * k);
    c.sync();
    u32 f;
    std::memcpy(&f, c.pinned, 4);
    check_throw(f);
    std::memcpy(bw_host, got, 8ull * k);
}

static s64 evaluate(Ctx &c, const DGraph &g, const u32 *part, const s32 *D, u32 k) {
    BackScope bs(c.arena);
    std::vector<s64> h(eval_grid(c, g.m));
    s64 *sums = bs.get<s64>(h.size());
    eval_launch(c, g, part, D, k, D ? 1 : 0, nullptr, (u32) h.size(), sums);
    readback(c, h.data(), (const s64 *) sums, h.size());
    s64 sum = 0;
    for (s64 x: h) sum += x;
    return sum;
}
s64 edge_cut(Ctx &c, const DGraph &g, const u32 *part) { return evaluate(c, g, part, nullptr, 0) / 2; }
s64 comm_cost(Ctx &c, const DGraph &g, const u32 *part, const s32 *D, u32 k) { return evaluate(c, g, part, D, k); }

void block_weights_dev(Ctx &c, const DGraph &g, const u32 *part, u32 k, s64 *bw_dev, const u32 *bad) {
    fill<s64>(c, bw_dev, k, 0);
    block_weights_add(c, g, part, k, bw_dev, bad);
}
void block_weights_add(Ctx &c, const DGraph &g, const u32 *part, u32 k, s64 *bw_dev, const u32 *bad) {
    const double bytes = 4.0 * g.n * (g.vw ? 2 : 1);
    const size_t shmem = sizeof(unsigned long long) * k;
    if (shmem > 64 * 1024) {  // no LDS histogram: one global atomic per vertex
        launch(c, "block_weights", bytes, dim3(grid_for(c, g.n, 256)), dim3(256), 0,
               g.vw ? block_weights_global_kernel<false> : block_weights_global_kernel<true>, g.n, part, g.vw, k,
               (unsigned long long *) bw_dev, bad);
        return;
    }
    launch(c, "block_weights", bytes, dim3(grid_for(c, g.n, 256 * 8)), dim3(256), shmem,
           g.vw ? block_weights_kernel<false> : block_weights_kernel<true>, g.n, part, g.vw, k,
           (unsigned long long *) bw_dev, bad);
}

} // namespace heipa
