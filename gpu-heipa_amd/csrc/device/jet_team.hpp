// Team form of the Jet loop: one launch in which up to TEAM_MAX workgroups of
// ONE accelerator die (XCD), or one or two per compute unit of all of them
// (WIDE), run whole iterations together.  Included by jet.hip inside its
// anonymous namespace (it uses that file's device functions).
//
// What it replaces: the multi-launch form pays, per iteration, six to twelve
// launches at 3.6 us each from the last wave of one to the first of the next,
// and a cold L2 in each of them (a launch boundary writes back and invalidates
// the L2s), so every dependent load of its chains is a trip past L2 (220-370 ns
// measured).  The workgroups of one XCD share an L2: a barrier among them costs
// 0.6 us whether 8 or 32 take part, and the level's state stays in that L2 (88
// ns); over all XCDs a barrier takes 2.0 us.  What bounds both is the chain of
// dependent loads and instructions of each phase, plus three barriers (LP) or
// five (rebalancing) per iteration.  us per iteration, set-up of the level
// included: 17 against 36 at 3000 vertices, 30 against 45 at 60000, 47 against
// 58 at 500000 (RGG, k = 64), 79 against 129 at 16000 vertices of R-MAT.
//
// The team itself (formation, barrier, hand-offs) is team.hpp.
#pragma once

constexpr u32 TEAM_ITERS = 128;               // iterations per launch
constexpr u32 TEAM_RCAP = 4096;               // resolve entries sorted in LDS
constexpr u32 TEAM_U = 2;                     // sweep tiles a wave has in flight
constexpr u32 TILE = WAVE * TEAM_U;           // vertices of one sweep step of a wave
constexpr u32 TEAM_BUF = 2048;                // list entries a workgroup collects (edge-balanced form)
constexpr u32 ROW_DEG = 2 * ROW;              // largest degree of the register form of a rebuild
constexpr u32 LONG_DEG = 128;                 // degree from which a rebuild takes a whole wave
constexpr u32 ROW_FEW = 16;                   // wide vertices of a wave up to which 16 lanes update each one's row
constexpr size_t TEAM_CONN_LDS = 64 * 1024;   // block counters of the others, per workgroup
constexpr u32 TEAM_BW = 1024;                 // blocks whose weight changes a workgroup sums in LDS

struct TeamAcc {  // totals of the iteration in flight
    unsigned long long delta, mhash, ghash, miss, miss_deg, cand_deg, move_deg;
    u32 ncand, nmoves, nrl, stall, nextra;
    u32 pad[13];
};
static_assert(sizeof(TeamAcc) == 128, "one line each");
struct TeamCtl {  // zero before the launch
    TeamHead head;
    TeamAcc acc[2];      // iteration i uses acc[i & 1] and clears the other
};
constexpr u32 TEAM_SLOTS = 16;  // launches between two clears
struct WideCtl {  // zero before the launch
    WideHead head;
    TeamAcc acc[2][XCC_MAX];  // a copy per XCD; the resolve list's and its moves' lengths are in the first
};
constexpr u32 WIDE_SLOTS = 4;
constexpr u32 WIDE_SHORT = 8;  // iterations of a launch whose team formed at less than half its size

struct TeamArgs {
    TeamCtl *tc;
    WideCtl *wc;
    const u32 *hubs, *chunk_hub, *chunk_idx;
    u32 n_hubs, n_chunks, xcc, want, max_iters;
    u32 wgroups;  // lane groups with block counters per wave
    u32 rcap;     // resolve entries that fit the LDS
};

// the same for a workgroup (edge-balanced form; uniform over the workgroup)
__device__ __forceinline__ void team_flush(const u32 *buf, u32 *s_cnt, u32 *s_base, u32 *list, u32 *counter) {
    __syncthreads();
    const u32 cnt = *s_cnt;
    if (cnt) {
        if (threadIdx.x == 0) *s_base = atomicAdd(counter, cnt);
        __syncthreads();
        const u32 base = *s_base;
        for (u32 i = threadIdx.x; i < cnt; i += TM) list[base + i] = buf[i];
        __syncthreads();
        if (threadIdx.x == 0) *s_cnt = 0;
    }
    __syncthreads();
}

// the phases' LDS areas share one union behind the k block weights and the
// rebalance prologue's result
__host__ __device__ inline size_t team_union_off(u32 k) { return (8ull * k + 16 + 4ull * k + 15) & ~(size_t) 15; }
constexpr size_t TEAM_WAVE_SWEEP = 12ull * TILE + 4ull * WBUF;
__host__ inline size_t team_lds_bytes(u32 k, u32 wgroups, u32 rcap) {
    size_t u = std::max<size_t>(conn_group_bytes(k) * wgroups * TW + TEAM_WAVE_SWEEP * TW, resolve_lds_bytes(rcap));
    u = std::max<size_t>(u, 12ull * WBUF * TW);
    u = std::max<size_t>(u, 16ull * k + 8);
    u = std::max<size_t>(u, 8ull * TEAM_BW + sizeof(FlatLds<TM>) + 4ull * TEAM_BUF);
    return team_union_off(k) + u;
}

// ---- lp_eval / reb_eval of one vertex of degree <= ROW_DEG per DPP row (same
// decisions, same writes).  Each lane holds up to two neighbours' blocks and
// edge weights; the row takes the distinct blocks in ascending order (the
// smallest not taken yet, then the sum of its weights), the own block first:
// most vertices have one to three.  The LDS counters cost a chain of about
// eight LDS round trips and limited the lane groups to what k left room for.
// Under the mapping objective the vertex has no row (degree < k).  Returns,
// on the row's lane 0, whether u is a candidate.
template<typename JD>
__device__ __forceinline__ bool row_eval(const JD &d, u32 mode, s64 mbw, const RebShared *rs, double ratio, u32 u,
                                         u32 beg, u32 deg, u32 own, bool locked, u32 lane, bool active) {
    const bool a0 = active && lane < deg, a1 = active && lane + ROW < deg;
    u32 v0 = 0, v1 = 0;
    s64 w0 = 0, w1 = 0;
    if (a0) {
        v0 = d.adj[beg + lane];
        w0 = ewt(d, beg + lane);
    }
    if (a1) {
        v1 = d.adj[beg + ROW + lane];
        w1 = ewt(d, beg + ROW + lane);
    }
    const s64 wu = active && mode ? vwt(d, u) : 1;
    u32 r = 0;
    const bool full = mode == 2 && active && row_full(d, u, r);
    u32 b0 = NO_MOVE, b1 = NO_MOVE;  // larger than any block
    if (a0) b0 = d.work[v0];
    if (a1) b1 = d.work[v1];
    const bool in0 = b0 == own, in1 = b1 == own;
    const s64 own_c = row_sum((in0 ? w0 : 0) + (in1 ? w1 : 0));
    s64 jo = 0;
    if (JD::map && mode == 0) {
        const s32 *Do = d.D + (u64) own * d.k;
        jo = row_sum((b0 != NO_MOVE ? w0 * (s64) Do[b0] : 0) + (b1 != NO_MOVE ? w1 * (s64) Do[b1] : 0));
    }
    u32 l0 = in0 ? NO_MOVE : b0, l1 = in1 ? NO_MOVE : b1;  // not taken yet
    Best best{0, NO_MOVE};
    s64 sum = 0;
    u32 count = 0;
    u32 b = row_min(l0 < l1 ? l0 : l1);
    const s64 ic = b == NO_MOVE ? own_c : -1;  // no neighbour outside the own block
    while (__any(b != NO_MOVE)) {
        const bool t0 = l0 == b, t1 = l1 == b;
        s64 c;
        if (JD::map && mode == 0) {
            const s32 *Db = d.D + (u64) (b == NO_MOVE ? own : b) * d.k;
            c = jo - row_sum((b0 != NO_MOVE ? w0 * (s64) Db[b0] : 0) + (b1 != NO_MOVE ? w1 * (s64) Db[b1] : 0));
        } else {
            c = row_sum((t0 ? w0 : 0) + (t1 ? w1 : 0));
        }
        if (b != NO_MOVE && (mode == 0 || d.bw[b] < mbw)) {
            if (best.b == NO_MOVE || c > best.c) best = Best{c, b};  // ascending blocks: ties keep the smaller
            sum += c;
            count += 1;
        }
        if (t0) l0 = NO_MOVE;
        if (t1) l1 = NO_MOVE;
        b = row_min(l0 < l1 ? l0 : l1);
    }
    bool cand = false;
    if (mode == 0) {
        if (active && lane == 0) {
            u32 best_id = best.b;
            s64 gain = 0;
            if (best_id != NO_MOVE) {
                const s64 bc = best.c;
                if (JD::map) {
                    if (bc >= 0) gain = bc;
                    else best_id = NO_MOVE;
                } else if (bc >= own_c || ((double) own_c - (double) bc) < floor(ratio * (double) own_c)) {
                    gain = bc - own_c;
                } else {
                    best_id = NO_MOVE;
                }
            }
            d.icache[u] = ic;
            d.gcache[u] = gain;
            d.dcache[u] = best_id;
            stale_of(d)[u] = 0;
            d.dest[u] = best_id;
            cand = best_id != NO_MOVE && !locked;
            d.gain1[u] = cand ? gain : GAIN_MIN;
            if (!cand) d.lock[u] = 0;
        }
        return cand;
    }
    if (mode == 2) {
        // entries of weight 0 in a full row count too (jet:418-428)
        if (full && lane == 0) {
            for (u32 i = 0; i < d.W; ++i) {
                u32 z = d.wV[(u64) r * d.W + i] & ~(u32) d.wP[(u64) r * d.W + i];
                if (own >> 5 == i) z &= ~(1u << (own & 31));
                while (z) {
                    const u32 x = i * 32 + (u32) __builtin_ctz(z);
                    z &= z - 1;
                    count += d.bw[x] < mbw;
                }
            }
        }
    }
    if (active && lane == 0) {
        d.icache[u] = ic;
        stale_of(d)[u] = stale_of(d)[u] & 1u;
        u32 dst = NO_MOVE, off = 0;
        s64 gain, wb = wu;
        if (mode == 1) {
            if (best.b != NO_MOVE && best.c > 0) {
                dst = best.b;
                gain = best.c - own_c;
            } else {
                const u32 nu = rs->n_under;
                dst = nu ? rs->under[u % nu] : own;
                gain = -own_c;
            }
            d.dest[u] = dst;
        } else {
            gain = (count ? sum / (s64) count : sum) - own_c;
            const s64 lim = d.bw[own] - d.lmax;
            wb = wu < lim ? wu : lim;
            off = 1;
        }
        if (dst != own) {
            const u32 g = (MAX_BUCKETS * own + gain_bucket(gain, wb)) * d.sections + (u % d.sections) + off;
            d.gid[u] = g;
            btot_add(d, u, g, wu);
            cand = true;
        }
    }
    return cand;
}

// the afterburner change of candidate u / the objective change of moved
// vertex u (invalidating its neighbours' caches), one vertex per row; every
// lane of the row returns the sum
template<typename JD>
__device__ __forceinline__ s64 row_burn(const JD &d, u32 u, s64 ug, u32 o, u32 nn, u32 beg, u32 end, u32 lane) {
    s64 change = 0;
    const u32 deg = end - beg;
    for (u32 x0 = lane; __any(x0 < deg); x0 += 2 * ROW) {
        const u32 j0 = beg + x0, j1 = j0 + ROW;
        const bool a0 = x0 < deg, a1 = x0 + ROW < deg;
        u32 v[2] = {0, 0};
        s64 w[2] = {0, 0}, vg[2] = {GAIN_MIN, GAIN_MIN};
        u32 vn[2] = {0, 0}, vo[2] = {0, 0};
        if (a0) v[0] = d.adj[j0], w[0] = ewt(d, j0);
        if (a1) v[1] = d.adj[j1], w[1] = ewt(d, j1);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (q ? a1 : a0) {
                vg[q] = d.gain1[v[q]];
                vn[q] = d.dest[v[q]];
                vo[q] = d.work[v[q]];
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (!((q ? a1 : a0) && (vg[q] > ug || (vg[q] == ug && v[q] < u)))) continue;
            if (JD::map) {  // promap:297-314
                const s32 *Do = d.D + (u64) o * d.k, *Dn = d.D + (u64) nn * d.k;
                change += w[q] * (((s64) Do[vn[q]] - (s64) Dn[vn[q]]) - ((s64) Do[vo[q]] - (s64) Dn[vo[q]]));
            } else {
                change += w[q] * (s64) ((s32) (vn[q] == nn) - (s32) (vn[q] == o) + (s32) (vo[q] == o) - (s32) (vo[q] == nn));
            }
        }
    }
    return row_sum(change);
}

// the blocks (k <= 64) of the neighbours over edges [b, e), by the G = ROW or
// WAVE lanes of a group
template<u32 G, typename JD>
__device__ __forceinline__ u64 row_blocks(const JD &d, u32 b, u32 e, u32 lane) {
    u64 m = 0;
    const u32 deg = e - b;
    for (u32 x = lane; x < deg; x += 8 * G) {
        u32 v[8];
#pragma unroll
        for (u32 q = 0; q < 8; ++q) v[q] = x + q * G < deg ? d.adj[b + x + q * G] : 0u;
#pragma unroll
        for (u32 q = 0; q < 8; ++q)
            if (x + q * G < deg) m |= 1ull << (u32) d.work[v[q]];
    }
    u32 lo = (u32) m, hi = (u32) (m >> 32);
    lo |= ror16<8>(lo);
    lo |= ror16<4>(lo);
    lo |= ror16<2>(lo);
    lo |= ror16<1>(lo);
    if (d.k > 32) {
        hi |= ror16<8>(hi);
        hi |= ror16<4>(hi);
        hi |= ror16<2>(hi);
        hi |= ror16<1>(hi);
    }
    if (G == WAVE) {
        lo = lane_value(lo, 0) | lane_value(lo, 16) | lane_value(lo, 32) | lane_value(lo, 48);
        hi = lane_value(hi, 0) | lane_value(hi, 16) | lane_value(hi, 32) | lane_value(hi, 48);
    }
    return (u64) hi << 32 | lo;
}

// resolve_body for a list of L <= 64 entries (most lists) by one wave, entry i
// in lane i: offsets inside a minibucket by comparing all pairs instead of a
// sort, block tables in LDS (2k + 1 words at `lds`), no barrier.  Returns the
// new length of the move list.
template<typename JD>
__device__ __forceinline__ u32 resolve_wave(const JD &d, bool strong, u32 stamp, u32 L, s64 *lds, u32 nmoves) {
    const u32 i = lane_id();
    const bool in = i < L;
    u32 u = 0xFFFFFFFFu, g = 0xFFFFFFFFu, ub = 0;
    s64 w = 0, score = 0, limit = 0;
    if (in) {
        const u64 key = d.rlist[i];
        u = (u32) key;
        g = (u32) (key >> 32);
        ub = d.work[u];
        w = vwt(d, u);
        score = bucket_prefix(d, g, ub);
        limit = d.bw[ub] - d.lmax;
    }
    for (u32 j = 0; j < L; ++j) {  // vertex weights are s32
        const u32 gj = lane_value(g, (int) j), uj = lane_value(u, (int) j), wj = lane_value((u32) w, (int) j);
        if (gj == g && uj < u) score += (s64) wj;
    }
    const bool take = in && score < limit;
    if (strong) {
        s64 *adj = lds, *es = lds + d.k;
        for (u32 b = i; b < d.k; b += WAVE) adj[b] = 0;
        wave_sync();
        if (take && score + w >= limit) adj[ub] = score + w;  // one entry per block ends beyond the limit
        wave_sync();
        // cookie cutter (jet:508-552)
        const s64 mbw = max_block_weight(d, true);
        s64 carry = 0, carry2 = 0;
        for (u32 b0 = 0; b0 < d.k; b0 += WAVE) {
            const u32 p = b0 + i;
            s64 add = 0, cap = 0;
            if (p < d.k) {
                add = adj[p];
                if (add == 0) add = d.Tseg[p];
                cap = mbw > d.bw[p] ? mbw - d.bw[p] : 0;
            }
            const s64 inc = wave_inclusive_scan(add), inc2 = wave_inclusive_scan(cap);
            if (p < d.k) {
                adj[p] = carry + inc - add;
                es[p + 1] = carry2 + inc2;
            }
            carry += lane_value(inc, WAVE - 1);
            carry2 += lane_value(inc2, WAVE - 1);
        }
        if (i == 0) es[0] = 0;
        wave_sync();
        u32 dst = ub;
        bool over = false;
        if (take) {  // adjust_scores, first pass
            const s64 pos = score + adj[ub];
            const s64 id = chunk_index(les_of(es), d.k, pos);
            if (id >= 0 && id < (s64) d.k && w / 2 <= es[id + 1] - pos) dst = (u32) id;
            else over = id < (s64) d.k;
        }
        // overflowing vertices in id order: each takes the counter's position
        // and adds its weight until it lands in a chunk with room
        s64 counter = carry, cid = -1;
        for (u64 left = __ballot(over); left;) {
            u32 best = over && (left >> i & 1ull) ? u : 0xFFFFFFFFu;
            best = row_min(best);
            const u32 m0 = lane_value(best, 0), m1 = lane_value(best, 16), m2 = lane_value(best, 32),
                      m3 = lane_value(best, 48);
            const u32 ma = m0 < m1 ? m0 : m1, mb = m2 < m3 ? m2 : m3, um = ma < mb ? ma : mb;
            const int l = __builtin_ctzll(__ballot(over && u == um));
            left &= ~(1ull << l);
            const s64 wu = lane_value(w, l);
            s64 pos = counter;
            u32 got = ~0u;
            while (got == ~0u) {
                while (cid < (s64) d.k && les_of(es)[cid + 1] <= pos) ++cid;
                if (cid >= (s64) d.k) got = d.k;
                else if (cid >= 0 && wu / 2 <= les_of(es)[cid + 1] - pos) got = (u32) cid;
                else if (wu <= 0) got = d.k;  // a weightless vertex never leaves a position before the first chunk
                else pos += round_up_to(les_of(es)[cid + 1] - pos, wu);
            }
            if ((int) i == l && got < d.k) dst = got;
            counter = pos + wu;
        }
        if (take) d.dest[u] = dst;
    }
    if (take) {
        d.mark[u] = stamp;
        d.oldp[u] = ub;
    }
    const u64 bal = __ballot(take);
    if (take) raw(d.moves_x)[nmoves + (u32) __popcll(bal & lanemask_lt())] = u;
    return nmoves + (u32) __popcll(bal);
}

// entries a wide team's member has room for in its list regions
__host__ __device__ inline u32 wide_cap(u32 n, u32 members, u32 n_hubs) {
    const u64 step = (u64) members * TW * WAVE * TEAM_U;
    return (u32) ((((u64) n + step - 1) / step) * TW * WAVE * TEAM_U + (n_hubs + members - 1) / members);
}

// WIDE: a team over all XCDs, for levels that outgrow one.  Its lists stay with
// the member that made them (regions of cand and moves, counted in LDS): one
// list for all would cost an update of one address per wave (15 ns each, 2048
// waves).  Totals have a copy per XCD.  PER_CU 2: two members per compute unit,
// 128 registers each (28 spilled), for levels whose sweep takes one member per
// unit several steps: us per iteration with one / two, balanced RGG, k = 64, set-up
// included: degree 12, 140000 vertices 33.5 / 31.8, 1000000 67.4 / 63.9; degree 6,
// 300000 31.9 / 31.6, 1500000 63.1 / 57.7, 3000000 110 / 90.
template<bool FLAT, bool MAP, bool WIDE, int PER_CU = 1>
__global__ __launch_bounds__(TM, PER_CU == 2 ? 4 : 1) void jet_team_kernel(JetDevT<true, MAP> dg, TeamArgs ta) {
    extern __shared__ __align__(16) char smem[];
    constexpr u32 CW = (sizeof(JetCtl) + 7) / 8;
    static_assert(CW <= TM && sizeof(JetCtl) % 8 == 0, "control block copy");
    __shared__ u64 s_ctl[CW];
    __shared__ u64 s_red[TM / WAVE];
    __shared__ Best s_best[TM / WAVE];
    __shared__ u32 s_join[3], s_ok, s_nmv, s_base, s_cc, s_mc, s_rc, s_nm;
    __shared__ unsigned long long s_delta;
    if (!WIDE && xcc_id() != ta.xcc) return;
    u32 tid = threadIdx.x;
    TeamCtl *tc = ta.tc;
    WideCtl *wc = ta.wc;
    if (tid < CW) s_ctl[tid] = ((const u64 *) dg.ctl)[tid];
    JetCtl *ctl = (JetCtl *) s_ctl;
    __syncthreads();
    if (!live(ctl)) return;
    u32 rank, T;
    std::conditional_t<WIDE, WideBar, TeamBar> bar;
    bool failed = false;
    if constexpr (WIDE) {
        if (!team_join<WIDE_MAX>(&wc->head, ta.want, s_join, rank, T)) return;
        bar.h = &wc->head;
        bar.ok = &s_ok;
        __syncthreads();
        failed = !wide_place(bar, T, s_join);
        if (2 * T < ta.want && ta.max_iters > WIDE_SHORT) ta.max_iters = WIDE_SHORT;
    } else {
        if (!team_join(&tc->head, ta.want, s_join, rank, T)) return;
        bar = TeamBar{tc->head.flag, rank, T, 0, &s_ok};
    }
    JetDevT<true, MAP> d = dg;
    const bool do_hash = dg.trace != nullptr;
    if (rank) d.trace = nullptr;  // one member writes the trace
    d.ctl = ctl;
    u32 xcd = 0;
    if constexpr (WIDE) xcd = bar.x;
    d.shard = (WIDE ? xcd : rank) % dg.nshard;
    // this member's list regions
    const u32 rcap = WIDE ? wide_cap(dg.n, T, ta.n_hubs) : 0u;
    u32 *const cand_l = raw(dg.cand) + (u64) rank * rcap;
    u32 *const move_l = WIDE ? dg.moves + (u64) rank * rcap : raw(dg.moves_x);
    s64 *s_bw = (s64 *) smem;
    d.bw = s_bw;
    RebShared *rs = (RebShared *) (smem + 8ull * d.k);
    char *um = smem + team_union_off(d.k);
    for (u32 b = tid; b < d.k; b += TM) s_bw[b] = dev_load(&dg.bw[b]);
    __syncthreads();
    if (tid < WAVE && ctl->mode) reb_prologue_wave(d, ctl->mode == 2, max_block_weight(d, ctl->mode == 2), rs);
    const size_t cgb = conn_group_bytes(d.k);
    const u32 NWV = T * TW;  // waves of the team
    // vertices per sweep tile: a whole wave's, fewer on levels that do not fill the team
    const u32 tile = d.n >= NWV * WAVE ? WAVE : WIDE ? (d.n + NWV - 1) / NWV : ((d.n + NWV - 1) / NWV + 3u) & ~3u;
#define TEAM_SYNC()             \
    if (!team_barrier(bar)) {   \
        failed = true;          \
        break;                  \
    }
    for (u32 iter = 0; iter < ta.max_iters && !failed; ++iter) {
        __syncthreads();  // the control step's block is complete
        if (WIDE && tid == 0) s_cc = s_mc = s_rc = 0, s_delta = 0;
        const CtlHead hd = ctl_head(ctl);
        if (!live(hd)) break;
        // opaque per iteration: hoisting every per-thread address out of this
        // loop held over a hundred registers across all phases
        asm volatile("" : "+v"(tid));
        const u32 wl = tid % WAVE;
        const u32 wid = (u32) __builtin_amdgcn_readfirstlane((int) (tid / WAVE));
        const u32 gw = rank * TW + wid;  // this wave among the team's
        const u32 mode = (u32) __builtin_amdgcn_readfirstlane((int) hd.mode);
        const u32 stamp = (u32) __builtin_amdgcn_readfirstlane((int) hd.stamp);
        const bool save = __builtin_amdgcn_readfirstlane((int) hd.save) != 0, strong = mode == 2;
        const double ratio = hd.ratio;
        const s64 mbw = mode ? max_block_weight(d, strong) : 0;
        TeamAcc *acc = WIDE ? &wc->acc[iter & 1][xcd] : &tc->acc[iter & 1];
        TeamAcc *acc0 = WIDE ? &wc->acc[iter & 1][0] : acc;
        u32 *const ncand = WIDE ? &s_cc : &acc->ncand, *const nmoves = WIDE ? &s_mc : &acc->nmoves;
        if (WIDE) __syncthreads();
        const u32 rl = wl % ROW, rg = wl / ROW;
        // ---- sweep, each wave on its own
        {
            char *wm = um + cgb * ta.wgroups * TW + TEAM_WAVE_SWEEP * wid;
            u32 *list = (u32 *) wm, *lbeg = list + TILE, *linfo = lbeg + TILE;
            WaveList<u32> wl_c{linfo + TILE, 0};
            u64 nev = 0, degs = 0;
            // skewed levels keep their heavy vertices together (low numbers, and
            // numbers with few bits set): there a wave's vertices lie far apart
            u32 off = gw * tile + wl;
            if (FLAT && WIDE) off = wl * NWV + (gw + wl * 37) % NWV;
            for (u64 t0 = 0; t0 < d.n; t0 += (u64) NWV * tile * TEAM_U) {
                // phase A, one vertex per lane, TEAM_U tiles in flight: cached
                // decisions are taken (LP) or eligibility is tested
                // (rebalancing); the vertices to rebuild go to the list, from
                // its front (degree <= ROW_DEG) or from its back
                u32 nl = 0, nw = 0;
                bool heavy[TEAM_U], cand[TEAM_U], in[TEAM_U];
                u32 hb[TEAM_U], he[TEAM_U], own[TEAM_U], vv[TEAM_U];
                u8 lk[TEAM_U];
#pragma unroll
                for (u32 q = 0; q < TEAM_U; ++q) {
                    const u64 v = t0 + (u64) q * NWV * tile + off;
                    in[q] = wl < tile && v < d.n;
                    vv[q] = (u32) v;
                    own[q] = in[q] ? (u32) d.work[v] : 0u;
                    lk[q] = 0;
                    hb[q] = he[q] = 0;
                }
                if (mode == 0) {
                    u32 dc[TEAM_U];
                    u8 sv[TEAM_U];
#pragma unroll
                    for (u32 q = 0; q < TEAM_U; ++q) {
                        dc[q] = in[q] ? (u32) d.dcache[vv[q]] : 0u;
                        lk[q] = in[q] ? (u8) d.lock[vv[q]] : (u8) 0;
                        sv[q] = in[q] ? (u8) stale_of(d)[vv[q]] : (u8) 0;
                    }
                    s64 gc0[TEAM_U];
#pragma unroll
                    for (u32 q = 0; q < TEAM_U; ++q) {
                        if (sv[q] & 1u) dc[q] = NULL_PART;
                        heavy[q] = in[q] && dc[q] == NULL_PART;
                        cand[q] = in[q] && !heavy[q] && dc[q] != NO_MOVE && lk[q] == 0;
                        gc0[q] = GAIN_MIN;
                        if (heavy[q]) {
                            hb[q] = d.xadj[vv[q]];
                            he[q] = d.xadj[vv[q] + 1];
                        } else if (cand[q]) {
                            gc0[q] = d.gcache[vv[q]];
                        }
                    }
#pragma unroll
                    for (u32 q = 0; q < TEAM_U; ++q) {
                        if (in[q] && !heavy[q]) {
                            d.dest[vv[q]] = dc[q];
                            d.gain1[vv[q]] = gc0[q];
                            if (!cand[q] && lk[q]) d.lock[vv[q]] = 0;
                        }
                    }
                } else {
                    s64 ic[TEAM_U];
#pragma unroll
                    for (u32 q = 0; q < TEAM_U; ++q) {
                        heavy[q] = in[q] && reb_eligible(d, strong, rs, vv[q], own[q]);
                        ic[q] = -1;
                        cand[q] = false;
                        if (heavy[q]) {
                            hb[q] = d.xadj[vv[q]];
                            he[q] = d.xadj[vv[q] + 1];
                            const s64 ic0 = d.icache[vv[q]];
                            ic[q] = (stale_of(d)[vv[q]] & 2u) ? -1 : ic0;
                        }
                    }
#pragma unroll
                    for (u32 q = 0; q < TEAM_U; ++q) {
                        if (heavy[q] && he[q] - hb[q] <= d.hub_deg && ic[q] >= 0) {
                            cand[q] = reb_interior(d, strong, rs, vv[q], ic[q]);
                            heavy[q] = false;
                        }
                    }
                }
#pragma unroll
                for (u32 q = 0; q < TEAM_U; ++q) {
                    if (save && in[q]) d.part[vv[q]] = own[q];
                    wl_c.add(cand[q], vv[q]);
                    const u32 deg = he[q] - hb[q];
                    const bool small = deg <= ROW_DEG && !(MAP && deg >= d.k);
                    const u32 info = own[q] << 16 | (lk[q] ? 1u << 15 : 0u) | deg;
                    const bool hs = heavy[q] && small, hl = heavy[q] && !small && deg <= d.hub_deg;
                    const u64 bs = __ballot(hs), bl = __ballot(hl);
                    if (hs || hl) {
                        const u32 i = hs ? nl + (u32) __popcll(bs & lanemask_lt())
                                         : TILE - 1 - (nw + (u32) __popcll(bl & lanemask_lt()));
                        list[i] = vv[q];
                        lbeg[i] = hb[q];
                        linfo[i] = info;
                    }
                    nl += (u32) __popcll(bs);
                    nw += (u32) __popcll(bl);
                }
                wave_sync();
                // phase B: a row per listed vertex of small degree
                for (u32 r0 = 0; r0 < nl; r0 += WAVE / ROW) {
                    const u32 idx = r0 + rg;
                    const bool active = idx < nl;
                    const u32 u = active ? list[idx] : 0, ub = active ? lbeg[idx] : 0;
                    const u32 info = active ? linfo[idx] : 0;
                    if (active && rl == 0) {
                        nev++;
                        degs += info & 0x7FFFu;
                    }
                    const bool listed = row_eval(d, mode, mbw, rs, ratio, u, ub, info & 0x7FFFu, info >> 16,
                                                 (info >> 15) & 1u, rl, active);
                    wl_c.add(listed, u);
                }
                // the others through LDS block counters, a row each, then a wave
                // each for the longest
                if (nw) {
                    const u32 gi = rg;
                    const bool ingroup = gi < ta.wgroups;
                    const GroupConn gc = group_conn(um, d.k, wid * ta.wgroups + (ingroup ? gi : 0));
                    if (ingroup) {
                        for (u32 i = rl; i < d.k; i += ROW) gc.cnt[i] = 0;
                        if (rl == 0) *gc.tcount = 0;
                    }
                    wave_sync();
                    bool longer = false;
                    for (u32 r0 = 0; r0 < nw; r0 += ta.wgroups) {
                        const bool here = ingroup && r0 + gi < nw;
                        const u32 idx = TILE - 1 - (r0 + gi);
                        const u32 u = here ? list[idx] : 0;
                        const u32 ub = here ? lbeg[idx] : 0, info = here ? linfo[idx] : 0;
                        const u32 ow = info >> 16, deg = info & 0x7FFFu;
                        const bool active = here && deg <= LONG_DEG;
                        longer |= here && deg > LONG_DEG;
                        if (!__any(active)) continue;
                        if (active) {
                            if (rl == 0) {
                                nev++;
                                degs += deg;
                            }
                            conn_accumulate_range<4>(d, gc, ub, (u64) ub + deg, rl, ROW);
                        }
                        wave_sync();
                        const bool listed =
                            mode == 0 ? lp_eval<(int) ROW>(d, gc, u, ow, (info >> 15) & 1u, rl, ratio, nullptr, nullptr, active)
                                      : reb_eval<(int) ROW>(d, strong, mbw, rs, gc, u, ow, rl, nullptr, nullptr, active);
                        wave_sync();
                        if (active) conn_reset(gc, *gc.tcount, rl, ROW);
                        wave_sync();
                        if (active && rl == 0) *gc.tcount = 0;
                        wave_sync();
                        wl_c.add(listed, u);
                    }
                    const GroupConn g0 = group_conn(um, d.k, wid * ta.wgroups);
                    for (u32 r0 = 0; __any(longer) && r0 < nw; ++r0) {
                        const u32 idx = TILE - 1 - r0, info = linfo[idx], deg = info & 0x7FFFu;
                        if (deg <= LONG_DEG) continue;
                        const u32 u = list[idx], ub = lbeg[idx], ow = info >> 16;
                        if (wl == 0) {
                            nev++;
                            degs += deg;
                        }
                        conn_accumulate_range<8>(d, g0, ub, (u64) ub + deg, wl, WAVE);
                        wave_sync();
                        const bool listed =
                            mode == 0 ? lp_eval<(int) WAVE>(d, g0, u, ow, (info >> 15) & 1u, wl, ratio, nullptr, nullptr, true)
                                      : reb_eval<(int) WAVE>(d, strong, mbw, rs, g0, u, ow, wl, nullptr, nullptr, true);
                        wave_sync();
                        conn_reset(g0, *g0.tcount, wl, WAVE);
                        wave_sync();
                        if (wl == 0) *g0.tcount = 0;
                        wave_sync();
                        wl_c.add(listed, u);
                    }
                }
                wl_c.reserve(TILE, cand_l, ncand);  // this step added at most TILE
                wave_sync();
            }
            wl_c.flush(cand_l, ncand);
            if (FLAT && ta.n_hubs) {  // hubs come with skewed degrees only
                // the members' sweeps have read the hubs' caches: one member
                // per hub now rebuilds or scores it
                TEAM_SYNC();
                GroupConn hc = group_conn(um, d.k, 0);
                for (u32 h = rank; h < ta.n_hubs; h += T) {
                    const u32 u = ta.hubs[h];
                    if (mode == 0) {
                        const u32 dc0 = d.dcache[u];
                        if (!(stale_of(d)[u] & 1u) && dc0 != NULL_PART) continue;
                    } else if (!reb_eligible(d, strong, rs, u, (u32) d.work[u])) {
                        continue;
                    }
                    __syncthreads();
                    for (u32 i = tid; i < d.k; i += TM) hc.cnt[i] = 0;
                    if (tid == 0) *hc.tcount = 0;
                    __syncthreads();
                    const u32 own = d.work[u];
                    const bool locked = d.lock[u] != 0;
                    conn_accumulate<ADJ_UNROLL>(d, hc, u, tid, TM);
                    __syncthreads();
                    const bool listed =
                        mode == 0
                            ? lp_eval<TM>(d, hc, u, own, locked, tid, ratio, s_best, (s64 *) s_red, true)
                            : reb_eval<TM>(d, strong, mbw, rs, hc, u, own, tid, s_best, (s64 *) s_red, true);
                    if (listed) cand_l[atomicAdd(ncand, 1u)] = u;
                    if (tid == 0) {
                        nev++;
                        degs += degree(d, u);
                    }
                }
            }
            if (d.count_bytes) {
                wave_add(&acc->miss, nev);
                wave_add(&acc->miss_deg, degs);
            }
        }
        TEAM_SYNC();
        if constexpr (WIDE) {
            if (rank == 0 && tid < XCC_MAX * sizeof(TeamAcc) / 8) ((u64 *) &wc->acc[(iter + 1) & 1][0])[tid] = 0;
            static_assert(XCC_MAX * sizeof(TeamAcc) / 8 <= TM, "one word per thread");
        } else {
            if (rank == 0 && tid < sizeof(TeamAcc) / 8) ((u64 *) &tc->acc[(iter + 1) & 1])[tid] = 0;
        }
        // ---- minibucket prefixes, one wave per block range
        if (mode) {
            const u64 stride = (u64) d.t + 1;
            for (u32 p = gw; p < d.k; p += NWV) {
                const u64 base = (u64) p * d.width;
                s64 carry = 0;
                for (u32 c0 = 0; c0 < d.width; c0 += WAVE) {
                    const u32 i = c0 + wl;
                    s64 v = 0;
                    if (i < d.width) {
#pragma unroll 1
                        for (u32 c = 0; c < d.nshard; c += 4) {
                            s64 x[4];
#pragma unroll
                            for (u32 q = 0; q < 4; ++q)
                                x[q] = c + q < d.nshard ? (s64) d.btot[(c + q) * stride + base + i] : 0;
#pragma unroll
                            for (u32 q = 0; q < 4; ++q)
                                if (x[q]) {
                                    v += x[q];
                                    d.btot[(c + q) * stride + base + i] = 0;
                                }
                        }
                    }
                    const s64 inc = wave_inclusive_scan(v);
                    if (i < d.width) {
                        d.Q[base + i] = carry + inc - v;
                        d.R[base + i] = carry + inc;
                    }
                    carry += lane_value(inc, WAVE - 1);
                }
                if (wl == 0) {
                    d.Tseg[p] = carry;
                    if (p == d.k - 1)
                        for (u32 c = 0; c < d.nshard; ++c) d.btot[c * stride + (u64) d.k * d.width] = 0;
                }
            }
            TEAM_SYNC();
        }
        // ---- afterburner / classify
        // (the candidates of all members, or of this one)
        u32 nc = (u32) __builtin_amdgcn_readfirstlane((int) (WIDE ? s_cc : dev_load(&acc->ncand)));
        const DevPtr<u32> cl{cand_l};
        if (WIDE && tid == 0 && nc) atomicAdd(&acc->ncand, nc);
        // list i of the members' (one-XCD form) or of this member's own
        const u32 lrank = WIDE ? 0u : rank, lsize = WIDE ? 1u : T;
        const u32 lw = WIDE ? wid : gw, lwaves = WIDE ? TW : NWV;
        if (mode == 0) {
            u64 cdeg = 0, gh = 0;
            if constexpr (FLAT) {
                FlatLds<TM> &L = *(FlatLds<TM> *) (um + 8ull * TEAM_BW);
                u32 *s_mv = (u32 *) (um + 8ull * TEAM_BW + sizeof(FlatLds<TM>));
                if (tid == 0) s_nmv = 0;
                __syncthreads();
                u32 cs = (nc + lsize - 1) / lsize;
                cs = cs < TM ? (cs ? cs : 1u) : (u32) TM;
                for (u32 c0 = lrank * cs; c0 < nc; c0 += lsize * cs) {
                    const u32 cnt = nc - c0 < cs ? nc - c0 : cs;
                    if constexpr (WIDE) {
                        afterburner_flat<TM>(d, stamp, cl, c0, cnt, move_l, &s_mc, L, do_hash, cdeg, gh);
                    } else {
                        afterburner_flat<TM>(d, stamp, cl, c0, cnt, s_mv, &s_nmv, L, do_hash, cdeg, gh);
                        if (s_nmv + TM > TEAM_BUF) team_flush(s_mv, &s_nmv, &s_base, move_l, nmoves);
                    }
                }
                if constexpr (!WIDE) team_flush(s_mv, &s_nmv, &s_base, move_l, nmoves);
            } else {
                WaveList<u32> wv{(u32 *) um + wid * WBUF, 0};
                const u32 step = lwaves * (WAVE / ROW);
                u32 i = lw * (WAVE / ROW) + rg;
                u32 nxu = 0, nxb = 0, nxe = 0;
                if (i < nc) {
                    nxu = cl[i];
                    nxb = d.xadj[nxu];
                    nxe = d.xadj[nxu + 1];
                }
                for (u32 i0 = lw * (WAVE / ROW); i0 < nc; i0 += step, i += step) {
                    const bool active = i < nc && nxe - nxb <= d.hub_deg;
                    const u32 u = nxu, ub = nxb, ue = active ? nxe : nxb;
                    s64 ug = 0;
                    u32 o = 0, nn = 0;
                    if (active) {
                        ug = d.gain1[u];
                        o = d.work[u];
                        nn = d.dest[u];
                    }
                    if (i + step < nc) {
                        nxu = cl[i + step];
                        nxb = d.xadj[nxu];
                        nxe = d.xadj[nxu + 1];
                    }
                    const s64 ch = row_burn(d, u, ug, o, nn, ub, ue, rl);
                    bool sel = false;
                    if (active && rl == 0) {
                        cdeg += ue - ub;
                        if (do_hash) gh += mix64d(mix64d(u) + (u64) ug);
                        if (ug + ch >= 0) {
                            d.lock[u] = 1;
                            d.mark[u] = stamp;
                            d.oldp[u] = o;
                            sel = true;
                        }
                    }
                    wv.add(sel, u);
                    wv.reserve(TILE, move_l, nmoves);
                }
                wv.flush(move_l, nmoves);
            }
            for (u32 h = rank; FLAT && h < ta.n_hubs; h += T) {
                const u32 u = ta.hubs[h];
                const s64 ug = d.gain1[u];
                if (ug == GAIN_MIN) continue;  // not a candidate
                s64 ch = afterburner_change<ADJ_UNROLL>(d, u, tid, TM);
                ch = group_sum<TM>(ch, (s64 *) s_red);
                if (tid == 0) {
                    cdeg += degree(d, u);
                    if (do_hash) gh += mix64d(mix64d(u) + (u64) ug);
                    if (ug + ch >= 0) {
                        d.lock[u] = 1;
                        d.mark[u] = stamp;
                        d.oldp[u] = d.work[u];
                        move_l[atomicAdd(nmoves, 1u)] = u;
                    }
                }
            }
            if (d.count_bytes) wave_add(&acc->cand_deg, cdeg);
            if (do_hash) wave_add(&acc->ghash, gh);
        } else {
            WaveList<u64> wr{(u64 *) um + wid * WBUF, 0};
            WaveList<u32> wv{(u32 *) (um + 8ull * WBUF * TW) + wid * WBUF, 0};
            for (u32 i0 = lw * WAVE; i0 < nc; i0 += lwaves * WAVE) {
                const u32 i = i0 + wl;
                const u32 u = i < nc ? (u32) cl[i] : 0u;
                u64 key = 0;
                const Take take = i < nc ? classify_take(d, strong, stamp, u, key) : TAKE_NO;
                wv.add(take == TAKE_SURE, u);
                wr.add(take == TAKE_BOUNDARY, key);
                wv.reserve(TILE, move_l, nmoves);
                wr.reserve(TILE, raw(d.rlist), &acc0->nrl);
            }
            wv.flush(move_l, nmoves);
            if constexpr (WIDE) {  // one update of the shared counter per member
                u32 base = 0;
                if (wl == 0 && wr.cnt) base = atomicAdd(&s_rc, wr.cnt);
                base = (u32) __builtin_amdgcn_readfirstlane((int) base);
                __syncthreads();
                if (tid == 0 && s_rc) s_base = atomicAdd(&acc0->nrl, s_rc);
                __syncthreads();
                if (s_rc)
                    for (u32 i = wl; i < wr.cnt; i += WAVE) raw(d.rlist)[s_base + base + i] = wr.buf[i];
            } else {
                wr.flush(raw(d.rlist), &acc->nrl);
            }
        }
        if constexpr (WIDE) {
            __syncthreads();
            if (tid == 0 && s_mc) atomicAdd(&acc->nmoves, s_mc);
        }
        TEAM_SYNC();
        // ---- resolve, by one member
        u32 L = 0;
        if (mode) {
            L = (u32) __builtin_amdgcn_readfirstlane((int) dev_load(&acc0->nrl));
            if (L) {
                if (rank == 0 && L <= WAVE && L <= d.rcap) {
                    if (wid == 0) {
                        const u32 n2 = resolve_wave(d, strong, stamp, L, (s64 *) um, WIDE ? 0u : dev_load(&acc->nmoves));
                        if (tid == 0) (WIDE ? acc0->nextra : acc->nmoves) = n2;
                    }
                } else if (rank == 0) {
                    if (tid == 0) s_nmv = WIDE ? 0u : dev_load(&acc->nmoves);
                    __syncthreads();
                    const bool ok = resolve_body<WIDE ? RESOLVE_CAP : TEAM_RCAP, TM>(d, strong, stamp, L, resolve_lds(um, ta.rcap), &s_nmv);
                    __syncthreads();
                    if (tid == 0) {
                        if (ok) (WIDE ? acc0->nextra : acc->nmoves) = s_nmv;
                        else acc0->stall = 1;
                    }
                }
                TEAM_SYNC();
                if (dev_load(&acc0->stall)) {
                    // the list does not fit: the host's global path and the
                    // multi-launch apply finish this iteration (the region
                    // lists are empty, the moves so far in the extra list)
                    if constexpr (WIDE) {
                        if (tid == 0 && s_mc) s_base = atomicAdd(&acc0->nextra, s_mc);
                        __syncthreads();
                        if (s_mc)
                            for (u32 i = tid; i < s_mc; i += TM) raw(d.moves_x)[s_base + i] = dev_load(&move_l[i]);
                        TEAM_SYNC();
                        nc = 0;
                        for (u32 x = 0; x < XCC_MAX; ++x) nc += dev_load(&wc->acc[iter & 1][x].ncand);
                    }
                    if (rank == 0) {
                        for (u32 r = tid; r < d.nreg; r += TM) {
                            d.cand_n[r] = 0;
                            d.moves_n[r] = 0;
                        }
                        for (u64 j = tid; j < (u64) d.nreg * PT_COUNT; j += TM) d.pstat[j] = 0;
                        if (tid == 0) {
                            u64 miss = 0, miss_deg = 0;
                            for (u32 x = 0; x < (WIDE ? XCC_MAX : 1u); ++x) {
                                miss += dev_load(&acc0[x].miss);
                                miss_deg += dev_load(&acc0[x].miss_deg);
                            }
                            ctl->st[ST_MISS] = miss;
                            ctl->st[ST_MISS_DEG] = miss_deg;
                            ctl->st[ST_CAND] = nc;
                            ctl->st[ST_MOVES] = dev_load(WIDE ? &acc0->nextra : &acc->nmoves);
                            ctl->st[ST_RLIST] = L;
                            ctl->stalled = 1;
                        }
                    }
                    break;
                }
            }
        }
        // ---- apply
        // (the moves of all members, or of this one and then the resolve step's)
        u32 nm = (u32) __builtin_amdgcn_readfirstlane((int) (WIDE ? s_mc : dev_load(&acc->nmoves)));
        const u32 nx = WIDE && L ? (u32) __builtin_amdgcn_readfirstlane((int) dev_load(&acc0->nextra)) : 0u;
        const DevPtr<u32> ml{move_l};
        {
            s64 delta = 0;
            u64 mdeg = 0, mh = 0;
            // block weight changes: summed per workgroup in LDS where a
            // workgroup has many moves, else added directly
            const bool lds_bw = d.k <= TEAM_BW && (FLAT || nm >= 8 * lsize * TW);
            s64 *s_bwa = (s64 *) um;
            if (lds_bw)
                for (u32 b = tid; b < d.k; b += TM) s_bwa[b] = 0;
            if (FLAT || lds_bw) __syncthreads();
            s64 *bwt = lds_bw ? s_bwa : dg.bw;
            if constexpr (FLAT) {
                FlatLds<TM> &L2 = *(FlatLds<TM> *) (um + 8ull * TEAM_BW);
                if constexpr (WIDE) {  // the own moves and a share of the others in one list
                    const u32 xc = (nx + T - 1) / T, x0 = rank * xc < nx ? rank * xc : nx;
                    const u32 all = nm + (x0 + xc < nx ? xc : nx - x0);
                    for (u32 c0 = 0; c0 < all; c0 += TM)
                        apply_flat<TM>(
                            d, stamp,
                            [&](u32 t) { return c0 + t < nm ? (u32) ml[c0 + t] : (u32) d.moves_x[x0 + (c0 + t - nm)]; },
                            all - c0 < TM ? all - c0 : (u32) TM, L2, do_hash, delta, mdeg, mh, bwt);
                } else {
                    u32 cs = (nm + T - 1) / T;
                    cs = cs < TM ? (cs ? cs : 1u) : (u32) TM;
                    for (u32 c0 = rank * cs; c0 < nm; c0 += T * cs)
                        apply_flat<TM>(d, stamp, [&](u32 t) { return (u32) ml[c0 + t]; }, nm - c0 < cs ? nm - c0 : cs, L2,
                                       do_hash, delta, mdeg, mh, bwt);
                }
            } else {
                // own moves first, then the others' by waves of the whole team
                const u32 o4 = ((nm + 3) / 4 + lwaves - 1) / lwaves * lwaves;  // rounds of four, whole passes
                const u32 x4 = WIDE ? (nx + 3) / 4 : 0u;
                for (u32 r = lw;; r += lwaves) {
                    if (!WIDE && r * (WAVE / ROW) >= nm) break;
                    u32 i = r * (WAVE / ROW) + rg;
                    bool has = i < nm;
                    if (r >= o4) {
                        const u32 xr = ((r - o4) / TW) * NWV + gw;
                        if (xr >= x4) break;
                        i = xr * (WAVE / ROW) + rg;
                        has = i < nx;
                    }
                    u32 u = 0, xb = 0, xe = 0, ou = 0, nu = 0;
                    s64 wu = 0;
                    if (has) {
                        u = WIDE && r >= o4 ? (u32) d.moves_x[i] : (u32) ml[i];
                        xb = d.xadj[u];
                        xe = d.xadj[u + 1];
                        ou = d.oldp[u];
                        nu = d.dest[u];
                        wu = vwt(d, u);
                    }
                    const bool mine = has && xe - xb <= d.hub_deg;
                    if (mine) delta += move_delta_pre<1>(d, ou, nu, xb, xe, rl, ROW, stamp);
                    if (mine && rl == 0) {
                        mdeg += xe - xb;
                        stale_of(d)[u] = 3;
                        d.work[u] = nu;
                        atomicAdd((unsigned long long *) &bwt[ou], (unsigned long long) (-wu));
                        atomicAdd((unsigned long long *) &bwt[nu], (unsigned long long) wu);
                        if (do_hash) mh += mix64d(((u64) u << 32) | nu);
                    }
                }
            }
            for (u32 c = rank; FLAT && c < ta.n_chunks; c += T) {
                const u32 u = ta.hubs[ta.chunk_hub[c]], ci = ta.chunk_idx[c];
                if (d.mark[u] != stamp) continue;
                const u64 b = (u64) d.xadj[u] + (u64) ci * HUB_CHUNK, end = d.xadj[u + 1];
                const u64 e = b + HUB_CHUNK < end ? b + HUB_CHUNK : end;
                delta += move_delta_range<ADJ_UNROLL>(d, u, b, e, tid, TM, stamp);
                if (ci == 0 && tid == 0) {
                    mdeg += degree(d, u);
                    move_commit(d, u, bwt);
                    if (do_hash) mh += mix64d(((u64) u << 32) | (u32) d.dest[u]);
                }
            }
            delta = wave_sum(delta);
            if (wl == 0 && delta) atomicAdd(WIDE ? &s_delta : &acc->delta, (unsigned long long) delta);
            if (d.count_bytes) wave_add(&acc->move_deg, mdeg);
            if (do_hash) wave_add(&acc->mhash, mh);
            if (lds_bw) {
                __syncthreads();
                for (u32 b = tid; b < d.k; b += TM)
                    if (s_bwa[b]) atomicAdd((unsigned long long *) &dg.bw[b], (unsigned long long) s_bwa[b]);
            }
            if constexpr (WIDE) {
                __syncthreads();
                if (tid == 0 && s_delta) atomicAdd(&acc->delta, s_delta);
            }
        }
        // ---- control, the same step in every member, and the next
        // iteration's rebalance prologue, by the wave that saw the barrier end
        const bool ok = team_barrier(bar, [&] {
            s64 delta;
            if constexpr (WIDE) {  // the XCDs' totals, one per lane
                const bool in = wl < XCC_MAX;
                const TeamAcc *a = &wc->acc[iter & 1][in ? wl : 0];
                delta = wave_sum(in ? (s64) dev_load(&a->delta) : 0);
                nc = wave_sum(in ? dev_load(&a->ncand) : 0u);
                nm = wave_sum(in ? dev_load(&a->nmoves) : 0u) + nx;
                if (wl == 0) s_nm = nm;
            } else {
                delta = (s64) dev_load(&acc->delta);
            }
            s64 mx = INT64_MIN;
            for (u32 b = wl; b < d.k; b += WAVE) {
                const s64 w = dev_load(&dg.bw[b]);
                s_bw[b] = w;
                mx = w > mx ? w : mx;
            }
            mx = wave_max(mx);
            if (wl == 0) {
                u64 t[PT_COUNT + 2];
#pragma unroll
                for (u32 j = 0; j < PT_COUNT; ++j) t[j] = 0;
                t[PT_DELTA] = (u64) delta;
                if (d.count_bytes || do_hash) {
#pragma unroll 1
                    for (u32 x = 0; x < (WIDE ? XCC_MAX : 1u); ++x) {
                        t[PT_MISS] += dev_load(&acc0[x].miss);
                        t[PT_MISS_DEG] += dev_load(&acc0[x].miss_deg);
                        t[PT_CAND_DEG] += dev_load(&acc0[x].cand_deg);
                        t[PT_GHASH] += dev_load(&acc0[x].ghash);
                        t[PT_MOVE_DEG] += dev_load(&acc0[x].move_deg);
                        t[PT_MHASH] += dev_load(&acc0[x].mhash);
                    }
                }
                t[PT_COUNT] = nc;
                t[PT_COUNT + 1] = nm;
                ctl->st[ST_RLIST] = L;
                control_step(d, mx, t, *ctl);
            }
            wave_sync();
            const u32 nmode = ctl->mode;
            if (nmode) reb_prologue_wave(d, nmode == 2, max_block_weight(d, nmode == 2), rs);
        });
        if (!ok) {
            failed = true;
            break;
        }
        if constexpr (WIDE) nm = (u32) __builtin_amdgcn_readfirstlane((int) s_nm);
        // ---- rows of the wide vertices next to the moves
        if (d.rflag && nm) {
            const u32 rmode = nm > d.n / 10 ? ROW_LARGE : ROW_SMALL;
            u32 off = gw * tile + wl;
            if (FLAT && WIDE) off = wl * NWV + (gw + wl * 37) % NWV;
            if (d.W <= 2) {
                // From the adjacencies, a lane, a row or a wave each by their
                // length; where a wave has few of them, a row takes also those
                // that a lane would walk alone, four neighbours at a time: with
                // lanes only, the rows took 12 of the 28 us of an iteration at 40
                // to 75 vertices of degree 24 (3 of 19 us now; a limit of 8 or 32
                // vertices: the same).  Counts kept by the moves (two updates of
                // shared memory per edge of a moved vertex) made the apply step of
                // a skewed level 50 us where most vertices move; walking the
                // touched rows again is a gather per edge.
                u32 *list = (u32 *) um + wid * TILE;
                for (u64 t0 = 0; t0 < d.n; t0 += (u64) NWV * tile) {
                    const u64 vv = t0 + off;
                    const u32 v = (u32) vv;
                    const bool flagged = wl < tile && vv < d.n && (d.rflag[v] & 3u) == 3u;
                    const u32 deg = flagged ? degree(d, v) : 0u;
                    const u32 lane_deg = (u32) __popcll(__ballot(deg > 4 && deg <= ROW_THREAD_DEG)) <= ROW_FEW ? 4u : ROW_THREAD_DEG;
                    const bool mid = deg > lane_deg && deg <= 2 * LONG_DEG;
                    const u64 bm = __ballot(mid);
                    if (mid) list[(u32) __popcll(bm & lanemask_lt())] = v;
                    if (flagged && deg <= lane_deg) row_thread(d, v, rmode);
                    wave_sync();
                    const u32 nl = (u32) __popcll(bm);
                    for (u32 r0 = 0; r0 < nl; r0 += WAVE / ROW) {
                        const bool act = r0 + rg < nl;
                        const u32 u = act ? list[r0 + rg] : 0u;
                        const u32 xb = act ? d.xadj[u] : 0u, xe = act ? d.xadj[u + 1] : 0u;
                        const u64 mask = row_blocks<ROW>(d, xb, xe, rl);
                        if (act && rl == 0) row_finish(d, u, (u8) 3u, mask, rmode);
                    }
                    for (u64 left = __ballot(deg > 2 * LONG_DEG && deg <= d.hub_deg); left; left &= left - 1) {
                        const u32 u = lane_value(v, __builtin_ctzll(left));
                        const u64 mask = row_blocks<WAVE>(d, d.xadj[u], d.xadj[u + 1], wl);
                        if (wl == 0) row_finish(d, u, (u8) 3u, mask, rmode);
                    }
                    wave_sync();
                }
            } else {
                // The same with the block masks in LDS, W words each: the
                // vertices have degree >= k > 64, so a row or a wave each.  The
                // vertices are spread as in the sweep: with 64 consecutive ones
                // per wave, one after another, the first waves of a skewed level
                // took 64 long adjacencies in turn while most had none (R-MAT of
                // 16384 vertices, k = 128: 9.9 ms per refine, 4.5 now).
                u32 *list = (u32 *) um + wid * (WAVE + WAVE / ROW * d.W), *wm = list + WAVE;
                for (u64 t0 = 0; t0 < d.n; t0 += (u64) NWV * tile) {
                    const u64 vv = t0 + off;
                    const u32 v = (u32) vv;
                    const bool flagged = wl < tile && vv < d.n && (d.rflag[v] & 3u) == 3u;
                    const u32 deg = flagged ? degree(d, v) : 0u;
                    const bool mid = flagged && deg <= 2 * LONG_DEG;
                    const u64 bm = __ballot(mid);
                    if (mid) list[(u32) __popcll(bm & lanemask_lt())] = v;
                    wave_sync();
                    const u32 nl = (u32) __popcll(bm);
                    for (u32 r0 = 0; r0 < nl; r0 += WAVE / ROW) {
                        const bool act = r0 + rg < nl;
                        row_update<(int) ROW>(d, wm + rg * d.W, act ? list[r0 + rg] : 0u, rl, rmode, act, nullptr);
                    }
                    for (u64 left = __ballot(deg > 2 * LONG_DEG && deg <= d.hub_deg); left; left &= left - 1)
                        row_update<(int) WAVE>(d, wm, lane_value(v, __builtin_ctzll(left)), wl, rmode, true, nullptr);
                    wave_sync();
                }
            }
            for (u32 h = rank; FLAT && h < ta.n_hubs; h += T) {
                const u32 u = ta.hubs[h];
                if ((d.rflag[u] & 3u) != 3u) continue;
                __syncthreads();
                row_update<TM>(d, (u32 *) um, u, tid, rmode, true, (u32 *) s_red);
            }
            // strong rebalancing and the mapping objective read rows of other
            // members' vertices
            if (MAP || ctl->mode == 2) TEAM_SYNC();
        }
    }
#undef TEAM_SYNC
    __syncthreads();
    if (failed && tid == 0) dg.ctl->failed = 1;
    if (rank == 0 && !failed) {
        // all but `failed`, the last word's other half: a member that gave up
        // on the last barrier has set it
        static_assert(offsetof(JetCtl, launches) == 8 * (CW - 1) && offsetof(JetCtl, failed) == 8 * (CW - 1) + 4, "last word");
        if (tid == 0) dg.ctl->launches = ctl->launches + 1;
        if (tid < CW - 1) ((u64 *) dg.ctl)[tid] = s_ctl[tid];
    }
}
