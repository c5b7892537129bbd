// paths.hip -- SGM path costs by independent chains, and the winner from their
// sum (sgm.cpp:26-455; WTALeft on S, convert and crop: hpp:283,111-118).
//
// S is the sum of eight path costs.  Each path is a family of independent
// chains of cells (rows, columns, diagonals, anti-diagonals; two directions
// each), and along every chain the same recurrence runs:
//   L(d) = M(d) + min(L'(d), min(L'(d-1), L'(d+1)) + P1, minL' + P2) - minL'
// with L'(-1) = L'(D) = guard.  (L - M) lies in [0, P2] and M <= 252, so the
// reference's saturating u16 arithmetic never saturates and u16 lanes hold it.
// The pass structure of the reference (sgm.cpp:89-440) is in the chains' starts:
//   - a row restarts from L' = 0, minL' = 0 at each border: its first L is M;
//   - a vertical chain starting on the first line of its pass (row 0 going
//     down, row H'-1 going up) takes the state c~ = M there (M never reaches
//     255, the entry c~ would clear) and adds nothing to S: again L' = 0;
//   - one entering from beyond the left or right border sees L' = guard and
//     minL' = 0: its first L is M + P2.
// On the first line of a pass the row path runs truncated to 8 bits; S is read
// at the crop only, which holds no such line, so only the debug variant (KEEP,
// every cell of the padded frame) reproduces it.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "rig.h"
#include "kernels.h"
#include "lanes.h"

namespace sister {

constexpr int kPathLanes = 16;              // lanes per chain: one DPP row
constexpr int kPathChains = 64 / kPathLanes;   // chains per wave

// 2 NP bytes of a lane (NP pairs, 2 NP disparities) as one or two vector
// accesses: NW dwords, the first W0 = min(NW, 4) of them in the first
template <int NP> struct Span {
    static constexpr int NW = NP / 2, W0 = NW < 4 ? NW : 4, W1 = NW - W0;
    uint32_t w[NW];
};
// N dwords at a uniform base plus a 32-bit lane offset
template <int N> __device__ __forceinline__ void load_dw(const uint8_t* base, uint32_t off, uint32_t* w)
{
    typedef typename Vec<N>::T T;
    typedef T TA __attribute__((aligned(4)));
    const T v = *(gptr<const TA>)((gptr<const uint8_t>)base + off);
    if constexpr (N == 1) w[0] = v;
    else
#pragma unroll
        for (int i = 0; i < N; i++) w[i] = v[i];
}
// uniform 64-bit value of lane l
__device__ __forceinline__ long lane64(long v, int l)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), l);
    return (long)(((uint64_t)hi << 32) | lo);
}

// DPP within a chain's 16 lanes: the neighbour's value, the guard past the ends
__device__ __forceinline__ uint32_t from_left(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)kGuard2, (int)v, 0x111, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t from_right(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)kGuard2, (int)v, 0x101, 0xF, 0xF, false);
}

// cells the chains cover: the crop, or the whole padded frame (KEEP)
struct PathArea { int x0, x1, y0, y1; };
template <bool KEEP>
__device__ __forceinline__ PathArea path_area(const RigDesc& g)
{
    return KEEP ? PathArea{0, g.Wp - 1, 0, g.Hp - 1} : PathArea{g.D, g.D + g.W - 1, g.D, g.D + g.H - 1};
}
__host__ __device__ inline int path_chains(int w, int h, int f) { return f == 0 ? h : f == 1 ? w : w + h - 1; }

// cells of a segment of the joined form
__host__ __device__ constexpr int path_seg(int np) { return np <= 8 ? 16 : 8; }
// bytes of a wave's forward states in the joined form: one per segment of the
// crop part but the last, of at most that family's longest chain and 3 cells
__host__ __device__ inline size_t path_state_bytes(int w, int h, int f, int np)
{
    const int longest = f == 0 ? w : f == 1 ? h : (w < h ? w : h), seg = path_seg(np);
    return (size_t)((longest + 3 + seg - 1) / seg) * 64 * (np + 1) * 4;
}

// ---------------------------------------------------------------------------
// The path kernel.  A wave carries four chains, 16 lanes each; a lane holds
// 2 NP consecutive disparities as NP packed u16 pairs, so d-1 / d+1 are a byte
// shift of neighbouring pairs (across lanes one DPP move) and min over d is a
// packed running minimum and four DPP steps.  All directions of all families
// run in one launch: they read M alone, and each writes its (L - M) bytes to a
// volume of its own (part[2f + dir]); k_winner adds them.  Only what S needs
// runs: chains that meet the crop, from their border to their last crop cell.
// A family whose part[2f + 1] is null (a workspace too small for eight
// volumes) runs both directions in one wave, the second adding to the first's
// bytes (each <= 100).
//
// Cells of a chain lie a fixed stride apart, so an access is a scalar base
// that advances by the stride plus a lane offset that never changes.  Loads
// are issued PF - 1 cells ahead and carry no condition, and stores outside the
// chain's crop range take an out-of-range buffer offset instead of a branch:
// a branch around either would make every wait for a load drain the whole
// queue (s_waitcnt vmcnt(0), one memory latency per cell).
// What bounds it: one rig has fewer waves than the chip has SIMDs, so the
// step's own instructions (about 9 per pair and 40 for the exchange, the
// minimum and the addresses) set its time; a batch is bound by memory.
// Against one kernel per family with conditional accesses, the two directions
// one after the other and every padded cell: a 640x480 D=64 call 3.07 -> 0.56
// ms, 1920x1080 D=192 10.0 -> 4.26 ms, 4096x3000 D=384 57.9 -> 42.3 ms; 64
// batched 1920x1080 rigs (rows family alone) 172 -> 167 ms.
// ---------------------------------------------------------------------------
template <int NP>
constexpr int path_pf() { return NP <= 2 ? 16 : NP <= 4 ? 12 : NP <= 8 ? 8 : 4; }

template <int NP>
struct PathLane {
    uint32_t L[NP], mp;       // path state and its minimum over the chain
    uint32_t pad[NP];         // guard on the lane's pairs at or past D, else 0
    uint32_t moff, moff1;     // lane offset from the wave's cost base: first and second access
    uint32_t poff, poff1;     // from the wave's volume base; kDropped where the lane holds no cell bytes
    int n, t0, t1;            // the chain's cells, and the range of them stored
};

// One step of the recurrence on a cell's cost bytes w: the state takes L, d the
// pairs L - M.  tmask: 8-bit first-line path (KEEP).
template <int NP, bool FULL, bool KEEP>
__device__ __forceinline__ void path_step(uint32_t (&L)[NP], uint32_t& mp, const uint32_t (&pad)[NP], const uint32_t* w,
                                          uint32_t (&d)[NP], uint32_t tmask)
{
    const uint32_t mpp = dup16(mp);
    const us2 p2t = U2(mpp) + (us2){(unsigned short)kP2, (unsigned short)kP2};
    uint32_t a[NP + 1];      // pair j: entries 2j - 1 and 2j
    a[0] = __builtin_amdgcn_alignbit(L[0], from_left(L[NP - 1]), 16);
    a[NP] = __builtin_amdgcn_alignbit(from_right(L[0]), L[NP - 1], 16);
#pragma unroll
    for (int j = 1; j < NP; j++) a[j] = __builtin_amdgcn_alignbit(L[j], L[j - 1], 16);
    us2 rmin;
#pragma unroll
    for (int j = 0; j < NP; j++) {
        const uint32_t m = (j & 1) ? bytes23(w[j / 2]) : bytes01(w[j / 2]);
        const us2 nb = umin2(U2(a[j]), U2(a[j + 1])) + (us2){(unsigned short)kP1, (unsigned short)kP1};
        const us2 v = umin3(nb, U2(L[j]), p2t) - U2(mpp);
        uint32_t l = W2(v + U2(m));
        if constexpr (KEEP) l &= tmask;
        // every value is below 0x4000 (at most P2 + 255, or the guard), so
        // or-ing the guard 0x3FFF into a pair past D yields the guard
        if constexpr (!FULL) l |= pad[j];
        d[j] = W2(v);
        L[j] = l;
        if (j & 1) rmin = j == 1 ? umin2(U2(L[0]), U2(l)) : umin3(rmin, U2(L[j - 1]), U2(l));   // NP is even
    }
    mp = group_min<kPathLanes>(min((uint32_t)rmin.x, (uint32_t)rmin.y));
}

// one direction of the wave's chains.  mb / pb: address of the wave's first
// cell in M and in the volume, ms / ps: byte strides per cell
template <int NP, bool FULL, bool KEEP, bool ADD>
__device__ __forceinline__ void path_sweep(PathLane<NP>& st, const uint8_t* mb, long ms, uint8_t* pb, long ps, int nmax,
                                           int tmin, uint32_t mlast, uint32_t tmask)
{
    typedef Span<NP> S;
    constexpr int PF = path_pf<NP>();
    S ring[PF], old[ADD ? PF : 1];
    const uint8_t* fp = mb;      // next cell to request
    uint8_t* fo = pb;            // its place in the volume (ADD)
    int ft = 0;
    auto fetch = [&](S& b, S& o) __attribute__((always_inline)) {
        // the debug variant's chains end at the frame's border: a lane whose
        // chain is over reads along the wave's longest one (mlast) instead
        const auto rm = buf((uint8_t*)fp);
        buf_load<S::W0>(b.w, rm, !KEEP || ft < st.n ? st.moff : mlast);
        if constexpr (S::W1 > 0) buf_load<S::W1>(b.w + 4, rm, !KEEP || ft < st.n ? st.moff1 : mlast);
        if constexpr (ADD) {
            const bool in = ft >= st.t0 && ft < st.t1;
            const auto r = buf(fo);
            buf_load<S::W0>(o.w, r, in ? st.poff : kDropped);
            if constexpr (S::W1 > 0) buf_load<S::W1>(o.w + 4, r, in ? st.poff1 : kDropped);
        }
        // past the wave's last cell the request repeats it
        const bool more = ft < nmax - 1;
        fp += more ? ms : 0;
        if constexpr (ADD) fo += more ? ps : 0;
        ft = min(ft + 1, nmax - 1);
        // steps stay apart: the scheduler would gather the unpacking of several
        // cells behind one wait
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](const S& b, const S& o, int t, uint8_t* out, auto store) __attribute__((always_inline)) {
        uint32_t d[NP];
        path_step<NP, FULL, KEEP>(st.L, st.mp, st.pad, b.w, d, tmask);
        if constexpr (decltype(store)::value) {
            uint32_t w[S::NW];
#pragma unroll
            for (int k = 0; k < S::NW; k++) {
                w[k] = pack4(d[2 * k], d[2 * k + 1]);
                if constexpr (ADD) w[k] += o.w[k];   // bytes <= 100 each
            }
            const bool in = t >= st.t0 && t < st.t1;
            const auto r = buf(out);
            buf_store<S::W0>(w, r, in ? st.poff : kDropped);
            if constexpr (S::W1 > 0) buf_store<S::W1>(w + 4, r, in ? st.poff1 : kDropped);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    static_for<0, PF - 1>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        fetch(ring[i], old[ADD ? i : 0]);
    });
    int t = 0;
    uint8_t* out = pb;
    // cells before any chain of the wave reaches the crop: nothing to store
    for (; t + PF <= tmin; t += PF, out += PF * ps)
        static_for<0, PF>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, j = (i + PF - 1) % PF;
            fetch(ring[j], old[ADD ? j : 0]);
            step(ring[i], old[ADD ? i : 0], 0, nullptr, IC<0>{});
        });
    for (; t < nmax; t += PF)
        static_for<0, PF>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, j = (i + PF - 1) % PF;
            fetch(ring[j], old[ADD ? j : 0]);
            // steps past the wave's last cell store nothing (t >= every t1)
            step(ring[i], old[ADD ? i : 0], t + i, out, IC<1>{});
            out += ps;
        });
}

// ---------------------------------------------------------------------------
// Both directions of the wave's chains with one byte per cell and disparity
// (their (L - M) summed, at most 200) instead of one each.  The crop part of
// the chains is cut into segments of path_seg cells.
//   1. forward from the chains' first border: at each segment's start the
//      state goes to memory (pairs and minimum, 2 bytes per disparity and
//      segment); nothing else is stored;
//   2. backward from the last border to the crop;
//   3. segment by segment, last first: the costs of its cells (requested one
//      segment ahead) and its forward state are read, the forward steps run
//      again with their bytes kept in registers, then the backward steps, and
//      the sums are stored.
// The costs are read as often as by two separate waves, 1 / 2 of the bytes are
// written (and read by k_winner or the fused sweep), for half as many steps
// again: the form for plans bound by memory (4096x3000 D=384 39.5 -> 33.3 ms a
// call, 1920x1080 D=192 3.84 -> 3.39, pair modes of eight 1000x620 D=136 rigs
// 11.1 -> 9.3, the rows family ahead of the fused sweep of 64 1920x1080 rigs
// 21.6 -> 16.7 and the sweep reading one byte less 61.7 -> 59.1).  Chains of a wave run aligned:
// position s is a chain's own cell, and the crop part of the wave is
// [aw, bw), the union of its chains' (which differ by at most 3 cells: all
// inside the frame, which reaches D >= 16 cells beyond the crop).
// ---------------------------------------------------------------------------
template <int NP>
constexpr int join_pf() { return NP <= 8 ? 8 : 4; }
constexpr int kJoinMinD = 16;   // a segment's cells below the crop stay in the frame

// the wave's chains in the joined form (lane values marked *)
struct JoinGeo {
    const uint8_t* mb;    // cost bytes of position 0 of the wave's lowest chain
    uint8_t* pb;          // its place in the volume
    uint32_t ms, ps;      // byte strides per position (forward, positive)
    uint8_t* ck;          // the wave's states, one per segment after the last
    int len, lmax;        // cells of the chain *, of the wave's longest
    int a, b, aw, bw;     // crop part of the chain *, of the wave
    uint32_t mlast;       // offset of the longest chain
    uint32_t f0, b0;      // the states before the first cell *: 0, or guards (from beyond a side)
};

template <int NP, bool FULL>
__device__ __forceinline__ void path_joined(PathLane<NP>& st, const JoinGeo& g, int lane)
{
    typedef Span<NP> S;
    constexpr int PF = join_pf<NP>(), G = path_seg(NP);
    static_assert(G % PF == 0, "states are stored between rounds of the ring");
    const int nseg = (g.bw - g.aw + G - 1) / G, s0 = g.bw - nseg * G;   // first segment's start, above aw - G
    auto load_cell = [&](S& c, const uint8_t* p, uint32_t o, uint32_t o1) __attribute__((always_inline)) {
        const auto r = buf((uint8_t*)p);
        buf_load<S::W0>(c.w, r, o);
        if constexpr (S::W1 > 0) buf_load<S::W1>(c.w + 4, r, o1);
    };
    // states: planes of up to 4 dwords per lane, then the minima
    constexpr uint32_t CK = 64 * (NP + 1) * 4;
    auto ck_store = [&](int k, const uint32_t (&L)[NP], uint32_t mp) __attribute__((always_inline)) {
        const auto r = buf(g.ck + (size_t)(k - 1) * CK);
        static_for<0, NP / 4>([&](auto ic) { buf_store<4>(L + 4 * decltype(ic)::value, r, 1024u * decltype(ic)::value + 16u * lane); });
        if constexpr (NP % 4 == 2) buf_store<2>(L + NP - 2, r, 256u * (NP - 2) + 8u * lane);
        buf_store<1>(&mp, r, 256u * NP + 4u * lane);
    };
    auto ck_load = [&](int k, uint32_t (&L)[NP], uint32_t& mp) __attribute__((always_inline)) {
        const auto r = buf(g.ck + (size_t)(k - 1) * CK);
        static_for<0, NP / 4>([&](auto ic) { buf_load<4>(L + 4 * decltype(ic)::value, r, 1024u * decltype(ic)::value + 16u * lane); });
        if constexpr (NP % 4 == 2) buf_load<2>(L + NP - 2, r, 256u * (NP - 2) + 8u * lane);
        buf_load<1>(&mp, r, 256u * NP + 4u * lane);
    };
    // `rounds` rounds of PF steps from the wave's position p0 by step dir; the
    // first `hold` steps stay at p0 (and, lane by lane, a chain's first `wait`
    // steps change nothing: its state keeps init).  Requests past the last
    // step repeat its cell.
    auto lead = [&](uint32_t (&L)[NP], uint32_t& mp, uint32_t init, int p0, int dir, int hold, int wait, int waitmax,
                    int rounds, auto each) __attribute__((always_inline)) {
        const int n = rounds * PF;
        S ring[PF];
        const uint8_t* fp = g.mb + (long)p0 * g.ms;
        const long ms = dir > 0 ? (long)g.ms : -(long)g.ms;
        int fu = 0;
        auto fetch = [&](S& c) __attribute__((always_inline)) {
            load_cell(c, fp, fu >= wait ? st.moff : g.mlast, fu >= wait ? st.moff1 : g.mlast);
            const bool more = fu >= hold && fu < n - 1;
            fp += more ? ms : 0;
            fu = min(fu + 1, n - 1);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int j = 0; j < NP; j++) L[j] = FULL ? init : (init | st.pad[j]);
        mp = 0;
        if (rounds == 0) return;
        static_for<0, PF - 1>([&](auto ic) __attribute__((always_inline)) { fetch(ring[decltype(ic)::value]); });
        int r = 0;
        for (; r * PF < waitmax; r++) {
            static_for<0, PF>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                fetch(ring[(i + PF - 1) % PF]);
                uint32_t d[NP];
                path_step<NP, FULL, false>(L, mp, st.pad, ring[i].w, d, 0);
                const bool live = r * PF + i >= wait;
#pragma unroll
                for (int j = 0; j < NP; j++) L[j] = live ? L[j] : FULL ? init : (init | st.pad[j]);
                mp = live ? mp : 0;
                __builtin_amdgcn_sched_barrier(0);
            });
            each(r + 1);
        }
        for (; r < rounds; r++) {
            static_for<0, PF>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                fetch(ring[(i + PF - 1) % PF]);
                uint32_t d[NP];
                path_step<NP, FULL, false>(L, mp, st.pad, ring[i].w, d, 0);
                __builtin_amdgcn_sched_barrier(0);
            });
            each(r + 1);
        }
    };
    uint32_t F[NP], B[NP], fm, bm;
    // 1. forward to the last segment's start
    const int r0 = (s0 + PF - 1) / PF, pad0 = r0 * PF - s0;
    lead(F, fm, g.f0, 0, 1, pad0, pad0, pad0, r0 + (nseg - 1) * (G / PF), [&](int r) __attribute__((always_inline)) {
        const int k = r - r0;   // rounds past the first segment's start
        if (k >= 0 && k % (G / PF) == 0 && k / (G / PF) < nseg - 1) ck_store(nseg - 1 - k / (G / PF), F, fm);
    });
    // 2. backward to the crop
    const int n1 = g.lmax - g.bw, r1 = (n1 + PF - 1) / PF, pad1 = r1 * PF - n1;
    lead(B, bm, g.b0, g.lmax - 1, -1, pad1, pad1 + g.lmax - g.len, pad1 + 3, r1, [](int) {});
    // 3. the segments (segment k ends at bw - k G)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's states, read back below
    S cur[G], nxt[G];
    uint32_t Fn[NP], fmn = 0;
    auto request = [&](int k, S (&c)[G]) __attribute__((always_inline)) {
        const uint8_t* p = g.mb + (long)(g.bw - (k + 1) * G) * g.ms;
        static_for<0, G>([&](auto ic) __attribute__((always_inline)) {
            load_cell(c[decltype(ic)::value], p, st.moff, st.moff1);
            p += g.ms;
        });
    };
    request(0, nxt);
    for (int k = 0; k < nseg; k++) {
#pragma unroll
        for (int i = 0; i < G; i++) cur[i] = nxt[i];
        if (k > 0) {
#pragma unroll
            for (int j = 0; j < NP; j++) F[j] = Fn[j];
            fm = fmn;
        }
        const int kn = min(k + 1, nseg - 1);   // past the last segment: requested again
        request(kn, nxt);
        ck_load(max(kn, 1), Fn, fmn);
        __builtin_amdgcn_sched_barrier(0);
        uint32_t fw[G][S::NW];
        static_for<0, G>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            uint32_t d[NP];
            path_step<NP, FULL, false>(F, fm, st.pad, cur[i].w, d, 0);
#pragma unroll
            for (int q = 0; q < S::NW; q++) fw[i][q] = pack4(d[2 * q], d[2 * q + 1]);
            __builtin_amdgcn_sched_barrier(0);
        });
        const int sk = g.bw - (k + 1) * G;
        uint8_t* out = g.pb + (long)(sk + G - 1) * g.ps;
        static_for<0, G>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = G - 1 - decltype(ic)::value;
            uint32_t d[NP], w[S::NW];
            path_step<NP, FULL, false>(B, bm, st.pad, cur[i].w, d, 0);
#pragma unroll
            for (int q = 0; q < S::NW; q++) w[q] = fw[i][q] + pack4(d[2 * q], d[2 * q + 1]);   // bytes <= 100 each
            const bool in = sk + i >= g.a && sk + i < g.b;
            const auto r = buf(out);
            buf_store<S::W0>(w, r, in ? st.poff : kDropped);
            if constexpr (S::W1 > 0) buf_store<S::W1>(w + 4, r, in ? st.poff1 : kDropped);
            out -= g.ps;
            __builtin_amdgcn_sched_barrier(0);
        });
    }
}

template <int NP, bool FULL, bool KEEP, bool JOIN>
__global__ __launch_bounds__(64) void k_paths(const RigDesc* __restrict__ rigs, int nrig, const int* __restrict__ bs,
                                              int nfam, int frame)
{
    // frame: the volumes hold every cell of the padded frame (debug, and the
    // rows family ahead of the fused vertical sweep), else the crop
    const int ri = find_rig(bs, nrig, blockIdx.x);
    const RigDesc& g = rigs[ri];
    const PathArea ar = path_area<KEEP>(g);
    const int aw = ar.x1 - ar.x0 + 1, ah = ar.y1 - ar.y0 + 1;
    int lb = blockIdx.x - bs[ri], f = 0, dir = 0;
    bool both = false;
    for (;; dir ^= 1, f += dir ^ 1) {
        if (f >= nfam) return;
        if (dir == 1 && !g.part[2 * f + 1]) continue;
        const int nb = (path_chains(aw, ah, f) + kPathChains - 1) / kPathChains;
        if (lb < nb) break;
        lb -= nb;
    }
    both = dir == 0 && !g.part[2 * f + 1];
    const int nch = path_chains(aw, ah, f);
    const int lane = threadIdx.x, lid = lane % kPathLanes;
    const int ci = lb * kPathChains + lane / kPathLanes, c = min(ci, nch - 1);
    const int Wp = g.Wp, Hp = g.Hp, Dp = g.Dp;
    const int pw = frame ? Wp : g.W, pox = frame ? 0 : g.D, poy = pox;   // volume rows and origin

    PathLane<NP> st;
    // lanes past the cell's Dp bytes repeat lane 0's loads and store nothing
    const int b0 = lid * 2 * NP;
    const bool has = b0 < Dp, has1 = b0 + 16 < Dp;
#pragma unroll
    for (int j = 0; j < NP; j++) st.pad[j] = b0 + 2 * j < g.D ? 0u : kGuard2;
    auto sweep = [&](int dr, auto add) __attribute__((always_inline)) {
        int x, y, dx, dy;      // first cell and step of the chain
        bool enter = false;    // it enters from beyond a side border
        if (f == 0) {
            y = ar.y0 + c; x = dr ? Wp - 1 : 0;
            dx = dr ? -1 : 1; dy = 0;
            st.t0 = dr ? Wp - 1 - ar.x1 : ar.x0;
            st.n = st.t0 + aw;
        } else {
            dy = dr ? -1 : 1;
            const int ys = dr ? Hp - 1 : 0;        // first line of the pass
            int ya = ar.y0, yb = ar.y1;            // rows of the chain inside the area
            if (f == 1) {
                x = ar.x0 + c; y = ys; dx = 0;
            } else if (f == 2) {
                const int k = c + ar.x0 - ar.y1;   // x - y
                y = dr ? min(Hp - 1, Wp - 1 - k) : max(0, -k);
                x = y + k; dx = dy;
                ya = max(ya, ar.x0 - k); yb = min(yb, ar.x1 - k);
            } else {
                const int s = c + ar.x0 + ar.y0;   // x + y
                y = dr ? min(Hp - 1, s) : max(0, s - (Wp - 1));
                x = s - y; dx = -dy;
                ya = max(ya, s - ar.x1); yb = min(yb, s - ar.x0);
            }
            enter = y != ys;
            st.t0 = dr ? y - yb : ya - y;
            st.n = (dr ? y - ya : yb - y) + 1;
        }
        st.t1 = st.n;
        if (ci >= nch) st.t1 = st.t0;              // a repeated chain: not stored
        // first cell of each chain, as offsets from the wave's lowest
        const long mo = ((long)y * Wp + x) * Dp, po = ((long)(y - poy) * pw + (x - pox)) * Dp;
        long mlo = lane64(mo, 0), plo = lane64(po, 0), mlong = mlo;
        int nmax = __builtin_amdgcn_readlane(st.n, 0), tmin = __builtin_amdgcn_readlane(st.t0, 0);
#pragma unroll
        for (int k = 1; k < kPathChains; k++) {
            const long m1 = lane64(mo, k * kPathLanes), p1 = lane64(po, k * kPathLanes);
            const int n1 = __builtin_amdgcn_readlane(st.n, k * kPathLanes);
            mlo = min(mlo, m1);
            plo = min(plo, p1);
            if (n1 > nmax) { nmax = n1; mlong = m1; }
            tmin = min(tmin, __builtin_amdgcn_readlane(st.t0, k * kPathLanes));
        }
        st.moff = (uint32_t)(mo - mlo) + (has ? b0 : 0);
        st.moff1 = (uint32_t)(mo - mlo) + (has1 ? b0 + 16 : 0);
        st.poff = has ? (uint32_t)(po - plo) + b0 : kDropped;
        st.poff1 = has1 ? (uint32_t)(po - plo) + b0 + 16 : kDropped;
#pragma unroll
        for (int j = 0; j < NP; j++) st.L[j] = FULL ? (enter ? kGuard2 : 0u) : ((enter ? kGuard2 : 0u) | st.pad[j]);
        st.mp = 0;
        const bool first_line = KEEP && f == 0 && y == (dr ? Hp - 1 : 0);
        path_sweep<NP, FULL, KEEP, decltype(add)::value != 0>(
            st, g.msum + mlo, (long)(dy * Wp + dx) * Dp, g.part[2 * f + (both ? 0 : dr)] + plo, (long)(dy * pw + dx) * Dp,
            nmax, tmin, (uint32_t)(mlong - mlo), first_line ? 0x00FF00FFu : 0xFFFFFFFFu);
    };
    if (JOIN && g.ck[f]) {
        // chain c from its forward border: position 0 .. len - 1, crop part [a, b)
        JoinGeo J;
        int x, y, dx = 1, dy = 1, ya = ar.y0, yb = ar.y1, ye = Hp - 1;
        J.f0 = J.b0 = 0;
        if (f == 0) {
            y = ar.y0 + c; x = 0; dy = 0;
            J.a = ar.x0; J.b = ar.x1 + 1; J.len = Wp;
        } else {
            if (f == 1) {
                x = ar.x0 + c; y = 0; dx = 0;
            } else if (f == 2) {
                const int k = c + ar.x0 - ar.y1;   // x - y
                y = max(0, -k); ye = min(Hp - 1, Wp - 1 - k);
                x = y + k;
                ya = max(ya, ar.x0 - k); yb = min(yb, ar.x1 - k);
            } else {
                const int s = c + ar.x0 + ar.y0;   // x + y
                y = max(0, s - (Wp - 1)); ye = min(Hp - 1, s);
                x = s - y; dx = -1;
                ya = max(ya, s - ar.x1); yb = min(yb, s - ar.x0);
            }
            J.a = ya - y; J.b = yb - y + 1; J.len = ye - y + 1;
            J.f0 = y > 0 ? kGuard2 : 0u;
            J.b0 = ye < Hp - 1 ? kGuard2 : 0u;
        }
        const long mo = ((long)y * Wp + x) * Dp, po = ((long)(y - poy) * pw + (x - pox)) * Dp;
        long mlo = lane64(mo, 0), plo = lane64(po, 0), mlong = mlo;
        J.lmax = __builtin_amdgcn_readlane(J.len, 0);
        J.aw = __builtin_amdgcn_readlane(J.a, 0);
        J.bw = __builtin_amdgcn_readlane(J.b, 0);
#pragma unroll
        for (int k = 1; k < kPathChains; k++) {
            const long m1 = lane64(mo, k * kPathLanes);
            const int n1 = __builtin_amdgcn_readlane(J.len, k * kPathLanes);
            mlo = min(mlo, m1);
            plo = min(plo, lane64(po, k * kPathLanes));
            if (n1 > J.lmax) { J.lmax = n1; mlong = m1; }
            J.aw = min(J.aw, __builtin_amdgcn_readlane(J.a, k * kPathLanes));
            J.bw = max(J.bw, __builtin_amdgcn_readlane(J.b, k * kPathLanes));
        }
        if (ci >= nch) J.b = J.a;                  // a repeated chain: not stored
        st.moff = (uint32_t)(mo - mlo) + (has ? b0 : 0);
        st.moff1 = (uint32_t)(mo - mlo) + (has1 ? b0 + 16 : 0);
        st.poff = has ? (uint32_t)(po - plo) + b0 : kDropped;
        st.poff1 = has1 ? (uint32_t)(po - plo) + b0 + 16 : kDropped;
        J.mlast = (uint32_t)(mlong - mlo);
        J.mb = g.msum + mlo;
        J.pb = g.part[2 * f] + plo;
        J.ms = (uint32_t)((dy * Wp + dx) * Dp);
        J.ps = (uint32_t)((dy * pw + dx) * Dp);
        J.ck = g.ck[f] + (size_t)lb * path_state_bytes(aw, ah, f, NP);
        path_joined<NP, FULL>(st, J, lane);
        return;
    }
    sweep(dir, IC<0>{});
    if (both) {
        // the second direction reads the bytes this wave has just stored
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        sweep(1, IC<1>{});
    }
}

// ---------------------------------------------------------------------------
// S and the winner (hpp:283; convert, crop and x255: hpp:111-118; sub-pixel:
// the vertex of the parabola through S at d* - 1, d*, d* + 1).  16 lanes per
// cell as above, S = 8 M + the directions' bytes; each byte of two directions
// is at most 200, so pairs of volumes add as words before they are unpacked.
// Bound by memory: 9 bytes per cell and disparity (8 volumes and M).
// ---------------------------------------------------------------------------
constexpr int kWinCells = 64;   // cells per block of 4 waves

template <int NP, bool FULL, bool KEEP>
__global__ __launch_bounds__(256) void k_winner(const RigDesc* __restrict__ rigs, int nrig, const int* __restrict__ bs,
                                                int mode)
{
    typedef Span<NP> Sp;
    __shared__ uint32_t sh[4 * 64 * NP];      // S pairs of each wave's four cells
    const int ri = find_rig(bs, nrig, blockIdx.x);
    const RigDesc& g = rigs[ri];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lid = lane % kPathLanes, grp = lane / kPathLanes;
    uint32_t* const mine = sh + (wave * 4 + grp) * kPathLanes * NP;
    const int Wp = g.Wp, Dp = g.Dp, D = g.D;
    const int aw = KEEP ? Wp : g.W, ncell = aw * (KEEP ? g.Hp : g.H);
    const int p0 = (blockIdx.x - bs[ri]) * kWinCells + wave * (kWinCells / 4);
    const int b0 = lid * 2 * NP;
    const int o0 = b0 < Dp ? b0 : 0, o1 = b0 + 16 < Dp ? b0 + 16 : 0;
    const bool sub = mode == 0 && g.subpix != nullptr;
    uint16_t* const outm = g.out[mode];
#pragma unroll 2
    for (int i = 0; i < kWinCells / 4 / kPathChains; i++) {
        const int pi = p0 + i * kPathChains + grp, p = min(pi, ncell - 1);
        if (p0 + i * kPathChains >= ncell) break;
        const int ay = p / aw, ax = p - ay * aw;
        const int y = KEEP ? ay : ay + D, x = KEEP ? ax : ax + D;
        const size_t mc = ((size_t)y * Wp + x) * Dp, pc = (size_t)p * Dp;
        auto load = [&](const uint8_t* v, size_t cell, uint32_t (&w)[Sp::NW]) __attribute__((always_inline)) {
            load_dw<Sp::W0>(v + cell, o0, w);
            if constexpr (Sp::W1 > 0) load_dw<Sp::W1>(v + cell, o1, w + 4);
        };
        uint32_t m[Sp::NW], v[4][Sp::NW], u[4][Sp::NW];
        load(g.msum, mc, m);
        static_for<0, 4>([&](auto fc) __attribute__((always_inline)) {
            constexpr int f = decltype(fc)::value;
            load(g.part[2 * f], pc, v[f]);
#pragma unroll
            for (int k = 0; k < Sp::NW; k++) u[f][k] = 0;
            if (g.part[2 * f + 1]) load(g.part[2 * f + 1], pc, u[f]);
        });
        uint32_t S[NP];
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int k = j / 2;
            auto pr = [&](uint32_t w) __attribute__((always_inline)) { return U2((j & 1) ? bytes23(w) : bytes01(w)); };
            const us2 mm = pr(m[k]);
            us2 s = (mm << (us2){3, 3}) + pr(v[0][k] + u[0][k]) + pr(v[1][k] + u[1][k]) + pr(v[2][k] + u[2][k]) +
                    pr(v[3][k] + u[3][k]);
            if constexpr (KEEP) {
                // first lines of the passes: only that pass's row path, cut to
                // 8 bits, and the other pass's four paths add to S
                if (y == 0 || y == g.Hp - 1) {
                    const us2 cut = pr(y == 0 ? v[0][k] : u[0][k]), std = pr(y == 0 ? u[0][k] : v[0][k]);
                    s = U2(W2(mm + cut) & 0x00FF00FFu) + mm + std + mm * (us2){3, 3} + pr(v[1][k] + u[1][k]) +
                        pr(v[2][k] + u[2][k]) + pr(v[3][k] + u[3][k]);
                }
            }
            S[j] = W2(s);
        }
        if constexpr (KEEP) {
            if (pi < ncell && b0 < Dp) {
#pragma unroll
                for (int j = 0; j < NP; j++)
                    if (b0 + 2 * j < Dp) *(uint32_t*)(g.sum + mc + b0 + 2 * j) = S[j];
            }
        }
        const int oy = y - D, ox = x - D;
        const bool crop = pi < ncell && (!KEEP || (oy >= 0 && oy < g.H && ox >= 0 && ox < g.W));
        // keys (S << 9) | d, lowest d on ties; pairs past D exceed every key.
        // The lane's first d is added after its minimum (d < 512: no carry).
        uint32_t key = 0xFFFFFFFFu;
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const uint32_t s = FULL || b0 + 2 * j < D ? S[j] : 0xFFFFFFFFu;
            key = min(key, min(((s & 0xFFFFu) << 9) | (2 * j), ((s >> 16) << 9) | (2 * j + 1)));
        }
        key = group_min<kPathLanes>(key + b0);
        const uint32_t best = key & 511u;
        float delta = 0.0f;
        if (sub) {
#pragma unroll
            for (int j = 0; j < NP; j++) mine[lid * NP + j] = S[j];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // one wave's own LDS, in order
            __builtin_amdgcn_wave_barrier();
            if (best > 0 && (int)best < D - 1) {
                const uint16_t* sv = (const uint16_t*)mine;
                const int sm = sv[best - 1], s0 = (int)(key >> 9), sp = sv[best + 1];
                const int den = sm - 2 * s0 + sp;
                if (den > 0) delta = (float)(sm - sp) / (2.0f * (float)den);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        if (crop && lid == 0) {
            const size_t o = (size_t)oy * g.W + ox;
            if (outm) G(outm)[o] = (uint16_t)min(best * 255u, 65535u);
            if (mode == 0 && g.disp) G(g.disp)[o] = (uint16_t)best;
            if (sub) G(g.subpix)[o] = (float)best + delta;
        }
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// pairs per lane: the fewest with which 16 lanes hold Dp disparities and a
// cell ends at a lane's end (a lane's store never reaches the next cell); 16
// pairs are two accesses of 16 bytes, each whole or absent.  Fewer pairs are
// fewer instructions per step.
int path_pairs(int Dp)
{
    for (int np : {2, 4, 6, 8, 12})
        if (32 * np >= Dp && Dp % (2 * np) == 0) return np;
    return 16;
}

// blocks of one rig: nfam families, one set of waves per volume; whole: chains
// over the padded frame
int path_blocks(const RigDesc& g, int nfam, bool whole)
{
    const int w = whole ? g.Wp : g.W, h = whole ? g.Hp : g.H;
    int n = 0;
    for (int f = 0; f < nfam; f++) {
        const int nb = (path_chains(w, h, f) + kPathChains - 1) / kPathChains;
        n += nb * (g.part[2 * f + 1] ? 2 : 1);
    }
    return n;
}

int path_waves(int W, int H, int f) { return (path_chains(W, H, f) + kPathChains - 1) / kPathChains; }

int winner_blocks(const RigDesc& g, bool whole)
{
    const long n = whole ? (long)g.Wp * g.Hp : (long)g.W * g.H;
    return (int)((n + kWinCells - 1) / kWinCells);
}

#define SISTER_PATHS(NPV, FULLV, KEEPV)                                                                           \
    do {                                                                                                          \
        if (!KEEPV && G.joined)                                                                                   \
            hipLaunchKernelGGL((k_paths<NPV, FULLV, KEEPV, !KEEPV>), dim3(G.blocks[kGPaths]), dim3(64), 0, st,    \
                               G.rigs, G.nrig, G.bs[kGPaths], nfam, frame);                                       \
        else                                                                                                      \
            hipLaunchKernelGGL((k_paths<NPV, FULLV, KEEPV, false>), dim3(G.blocks[kGPaths]), dim3(64), 0, st,     \
                               G.rigs, G.nrig, G.bs[kGPaths], nfam, frame);                                       \
    } while (0)
#define SISTER_WINNER(NPV, FULLV, KEEPV)                                                                          \
    hipLaunchKernelGGL((k_winner<NPV, FULLV, KEEPV>), dim3(G.blocks[kGWinner]), dim3(256), 0, st, G.rigs, G.nrig, \
                       G.bs[kGWinner], mode)
// FULL where every pair of every lane is a real disparity
#define SISTER_BY_PAIRS(K)                                                                                        \
    do {                                                                                                          \
        const int np = path_pairs(G.Dp);                                                                          \
        const bool full = G.D == 32 * np && !keep_sum;                                                            \
        switch (np) {                                                                                             \
        case 2: if (keep_sum) K(2, false, true); else if (full) K(2, true, false); else K(2, false, false); break;      \
        case 4: if (keep_sum) K(4, false, true); else if (full) K(4, true, false); else K(4, false, false); break;      \
        case 6: if (keep_sum) K(6, false, true); else if (full) K(6, true, false); else K(6, false, false); break;      \
        case 8: if (keep_sum) K(8, false, true); else if (full) K(8, true, false); else K(8, false, false); break;      \
        case 12: if (keep_sum) K(12, false, true); else if (full) K(12, true, false); else K(12, false, false); break;  \
        default: if (keep_sum) K(16, false, true); else if (full) K(16, true, false); else K(16, false, false); break;  \
        }                                                                                                         \
    } while (0)

// bytes of the forward states of family f of a rig in the joined form (0: D
// too small for it)
size_t path_state_total(int W, int H, int D, int f)
{
    if (D < kJoinMinD) return 0;
    const size_t waves = (size_t)(path_chains(W, H, f) + kPathChains - 1) / kPathChains;
    return waves * path_state_bytes(W, H, f, path_pairs((D + 15) & ~15));
}

// every path of a group (its rows family alone ahead of the fused vertical sweep)
void launch_paths(const DGroup& G, int keep_sum, hipStream_t st)
{
    const int nfam = G.vcols > 0 ? 1 : 4, frame = G.vcols > 0 || keep_sum ? 1 : 0;
    SISTER_BY_PAIRS(SISTER_PATHS);
}

void launch_winner(const DGroup& G, int mode, int keep_sum, hipStream_t st)
{
    SISTER_BY_PAIRS(SISTER_WINNER);
}

}  // namespace sister
