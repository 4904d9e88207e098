// Teams: kernels in which up to TEAM_MAX workgroups of ONE accelerator die (XCD)
// work through many phases in one launch.  The workgroups of one XCD share an
// L2: a barrier among them costs 0.6 us whether 8 or 32 take part (a launch
// boundary 1.6 us, and a cold L2 after it), and what one writes the others read
// from that L2 at 88 ns (past L2: 220-370 ns).
//
// Hand-offs between workgroups: stores write through L1 to the shared L2 and
// are complete there after s_waitcnt vmcnt(0); readers use device-scope loads
// (DevPtr), which do not read L1.  No L2 write-back or invalidate is needed
// inside one XCD (each costs 50-60 ns and they serialise: with one
// invalidate per workgroup the barrier of 32 took 2.1 us).
//
// A team over all XCDs (WideHead) meets XCD by XCD; see its barrier below.
//
// No assumption on co-residency: the workgroups that have started on the XCD
// register, the first one closes the registration after a bounded wait, and
// the team is whoever has registered: every member is running, so every
// barrier ends.  A launch runs max_iters iterations, so a team that formed
// small on a busy chip does not last a whole level.
#pragma once

#include "eval.hpp"

namespace heipa {

constexpr int TM = 512;                       // threads of a team workgroup
constexpr u32 TW = TM / WAVE;                 // its waves
constexpr u32 TEAM_MAX = 64;                  // members: one wave polls all flags
constexpr u32 TEAM_WANT = 32;                 // workgroups wanted: the compute units of an XCD
constexpr u32 WIDE_MAX = 512;                 // members of a team over all XCDs
constexpr u32 XCC_MAX = 16;
constexpr u32 ROW = 16;                       // lanes of a DPP row
constexpr u32 WBUF = 256;                     // list entries a wave collects before it appends them
constexpr u32 TEAM_FROZEN = 0x80000000u;
constexpr u64 TEAM_FORM_TICKS = 1000;         // 10 us of the 100 MHz counter
constexpr u64 TEAM_WAIT_TICKS = 1000000000;   // 10 s: a wait that long is a fault (reported, not hung)

struct TeamHead {  // zero before the launch
    u32 reg, pad0[31];   // registrations, then TEAM_FROZEN
    u32 size, pad1[31];  // members, set once
    u32 flag[TEAM_MAX];  // barrier round of each member
};

struct WideHead {  // of a team over all XCDs; zero before the launch
    u32 reg, pad0[31];
    u32 size, pad1[31];
    u32 here, pad2[31];          // members that know their place on their XCD
    u32 xreg[XCC_MAX][32];       // members of each XCD
    u32 xdone[XCC_MAX][32];      // barrier round that all members of the XCD have reached
    u32 xgo[XCC_MAX][32];        // barrier round that the XCD's members may leave
    u32 flag[XCC_MAX][WIDE_MAX]; // barrier round of each member
};

// A pointer to device memory that other workgroups of the same launch write:
// every load is a device-scope one, which reads the L2 and not this compute
// unit's L1 (88 ns against 52 ns from L1 on an idle chip; the same rate under
// load).  Stores are plain: L1 writes through.
template<typename T>
struct DevRef {
    T *p;
    __device__ __forceinline__ operator T() const { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ __forceinline__ void operator=(T v) const { *p = v; }
    __device__ __forceinline__ void operator=(const DevRef &o) const { *p = (T) o; }
    __device__ __forceinline__ void operator&=(T v) const { *p = (T) ((T) *this & v); }
};
template<typename T>
struct DevPtr {
    T *p;
    __device__ __forceinline__ DevRef<T> operator[](u64 i) const { return {p + i}; }
    __device__ __forceinline__ DevPtr operator+(u64 i) const { return {p + i}; }
    __device__ __forceinline__ explicit operator bool() const { return p != nullptr; }
};
template<typename T>
__device__ __forceinline__ T *raw(T *p) { return p; }
template<typename T>
__device__ __forceinline__ T *raw(const DevPtr<T> &p) { return p.p; }

template<typename T>
__device__ __forceinline__ T dev_load(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the XCD this wave runs on (hardware register 20, bits 0-3)
__device__ __forceinline__ u32 xcc_id() { return __builtin_amdgcn_s_getreg((3 << 11) | 20) & 15u; }

// orders the LDS traffic of one wave (lane groups never span waves)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Registers this workgroup (all threads call it); false: it is not a member
// (another XCD's turn is the caller's test).  The first to register closes the
// list once `want` are there or 10 us have passed.  s: two LDS words.
template<u32 MAX = TEAM_MAX, typename Head>
__device__ __forceinline__ bool team_join(Head *h, u32 want, u32 *s, u32 &rank, u32 &size) {
    if (threadIdx.x == 0) {
        u32 sz = 0;
        const u32 r = __hip_atomic_fetch_add(&h->reg, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (r == 0) {
            const u64 t0 = wall_clock64();
            while (dev_load(&h->reg) < want && wall_clock64() - t0 < TEAM_FORM_TICKS) __builtin_amdgcn_s_sleep(1);
            sz = __hip_atomic_fetch_or(&h->reg, TEAM_FROZEN, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sz = sz < MAX ? sz : MAX;
            __hip_atomic_store(&h->size, sz, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else if (r < MAX) {  // not closed yet; the first member closes in bounded time
            const u64 t0 = wall_clock64();
            while ((sz = dev_load(&h->size)) == 0 && wall_clock64() - t0 < TEAM_WAIT_TICKS) __builtin_amdgcn_s_sleep(1);
        }
        s[0] = r;
        s[1] = sz;
    }
    __syncthreads();
    rank = (u32) __builtin_amdgcn_readfirstlane((int) s[0]);
    size = (u32) __builtin_amdgcn_readfirstlane((int) s[1]);
    return rank < size;
}

struct TeamBar {
    u32 *flag;
    u32 rank, size, round;
    u32 *ok;  // LDS
};

// every member has stored everything before it and sees what the others
// stored; false: a member never arrived (10 s).  The first wave runs `then`
// between the last arrival and the workgroup's release.
template<typename F>
__device__ __forceinline__ bool team_barrier(TeamBar &b, F &&then) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this wave's stores are in the L2
    __syncthreads();
    ++b.round;
    if (threadIdx.x < WAVE) {
        if (threadIdx.x == 0)
            __hip_atomic_store(&b.flag[b.rank], b.round, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const u32 *p = &b.flag[threadIdx.x < b.size ? threadIdx.x : b.rank];
        bool ok = true;
        u64 t0 = 0;
        for (u32 spin = 1; !__all((s32) (dev_load(p) - b.round) >= 0); ++spin) {
            if ((spin & 1023u) == 0) {
                if (t0 == 0) t0 = wall_clock64();
                if (wall_clock64() - t0 > TEAM_WAIT_TICKS) {
                    ok = false;
                    break;
                }
            }
        }
        if (threadIdx.x == 0) *b.ok = ok;
        if (ok) then();
    }
    __syncthreads();
    return *b.ok != 0;
}
__device__ __forceinline__ bool team_barrier(TeamBar &b) {
    return team_barrier(b, [] {});
}

// The barrier of a team over all XCDs.  Each XCD has an L2 of its own, so what
// crosses XCDs goes past L2: the members of an XCD meet there first, its
// leader (local rank 0) writes the L2 back (one fence for all of them: their
// stores are in it), the leaders meet, each invalidates its L2, and the members
// go on.  2.0 us for 256 workgroups on 8 XCDs, of which a launch boundary
// (3.6 us from the last wave to the first of the next kernel) also pays the
// write-back and the invalidate.  The loads that follow are device-scope ones
// (DevPtr), as in the one-XCD form.
struct WideBar {
    WideHead *h;
    u32 x, lr, xs;  // XCD, rank and members there
    u32 xmask;      // XCDs with members
    u32 round;
    u32 *ok;  // LDS
};

template<typename P>
__device__ __forceinline__ bool team_poll(P &&arrived) {
    u64 t0 = 0;
    for (u32 spin = 1; !__all(arrived()); ++spin) {
        if ((spin & 1023u) == 0) {
            if (t0 == 0) t0 = wall_clock64();
            if (wall_clock64() - t0 > TEAM_WAIT_TICKS) return false;
        }
    }
    return true;
}

// the member's place on its XCD, once the team is closed (all threads call it)
__device__ __forceinline__ bool wide_place(WideBar &b, u32 size, u32 *s) {
    b.x = xcc_id() % XCC_MAX;
    b.round = 0;
    if (threadIdx.x < WAVE) {
        u32 lr = 0;
        if (threadIdx.x == 0) {
            lr = __hip_atomic_fetch_add(&b.h->xreg[b.x][0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(lr)::"memory");
            __hip_atomic_fetch_add(&b.h->here, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const bool ok = team_poll([&] { return dev_load(&b.h->here) >= size; });
        const u32 cnt = threadIdx.x < XCC_MAX ? dev_load(&b.h->xreg[threadIdx.x][0]) : 0u;
        const u64 mask = __ballot(cnt != 0);
        if (threadIdx.x == b.x) s[1] = cnt;
        if (threadIdx.x == 0) {
            s[0] = lr;
            s[2] = (u32) mask;
            *b.ok = ok;
        }
    }
    __syncthreads();
    b.lr = (u32) __builtin_amdgcn_readfirstlane((int) s[0]);
    b.xs = (u32) __builtin_amdgcn_readfirstlane((int) s[1]);
    b.xmask = (u32) __builtin_amdgcn_readfirstlane((int) s[2]);
    return *b.ok != 0;
}

template<typename F>
__device__ __forceinline__ bool team_barrier(WideBar &b, F &&then) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this wave's stores are in its XCD's L2
    __syncthreads();
    ++b.round;
    if (threadIdx.x < WAVE) {
        const u32 l = threadIdx.x;
        bool ok = true;
        if (l == 0)
            __hip_atomic_store(&b.h->flag[b.x][b.lr], b.round, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (b.lr == 0) {
            for (u32 m0 = 0; m0 < b.xs && ok; m0 += WAVE) {
                const u32 *p = &b.h->flag[b.x][m0 + l < b.xs ? m0 + l : 0];
                ok = team_poll([&] { return (s32) (dev_load(p) - b.round) >= 0; });
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            if (l == 0) __hip_atomic_store(&b.h->xdone[b.x][0], b.round, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const u32 *q = &b.h->xdone[l < XCC_MAX && (b.xmask >> l & 1u) ? l : b.x][0];
            ok = ok && team_poll([&] { return (s32) (dev_load(q) - b.round) >= 0; });
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (l == 0 && ok)
                __hip_atomic_store(&b.h->xgo[b.x][0], b.round, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else {
            const u32 *q = &b.h->xgo[b.x][0];
            ok = team_poll([&] { return (s32) (dev_load(q) - b.round) >= 0; });
        }
        if (l == 0) *b.ok = ok;
        if (ok) then();
    }
    __syncthreads();
    return *b.ok != 0;
}
__device__ __forceinline__ bool team_barrier(WideBar &b) {
    return team_barrier(b, [] {});
}

// a list that one wave collects in LDS; the count is a wave-uniform register
template<typename T>
struct WaveList {
    T *buf;
    u32 cnt;
    __device__ __forceinline__ void add(bool pred, T val) {
        const u64 bal = __ballot(pred);
        if (pred) buf[cnt + (u32) __popcll(bal & lanemask_lt())] = val;
        cnt += (u32) __popcll(bal);
    }
    // appends the entries to a shared list with one counter update
    __device__ __forceinline__ void flush(T *list, u32 *counter) {
        if (cnt == 0) return;
        u32 base = 0;
        if (lane_id() == 0) base = atomicAdd(counter, cnt);
        base = (u32) __builtin_amdgcn_readfirstlane((int) base);
        wave_sync();
        for (u32 i = lane_id(); i < cnt; i += WAVE) list[base + i] = buf[i];
        wave_sync();
        cnt = 0;
    }
    // room for `step` more entries
    __device__ __forceinline__ void reserve(u32 step, T *list, u32 *counter) {
        if (cnt + step > WBUF) flush(list, counter);
    }
};

} // namespace heipa
