// median.hip -- the in-place 3x3 median of the WTA maps (postprocess.cpp:15-71
// called with source == dest).
//
// Over flat index q of an R x C map, processed in increasing q:
//   out[q] = in[q]                       q < C  or  q >= RC-C-4
//   out[C] = 0                           (first store is the zero lastMedian)
//   out[q] = med9(out[q-C-1], out[q-C], out[q-C+1],
//                 in[q-1],  in[q],  in[q+1],  in[q+C-1], in[q+C], in[q+C+1])
//                                        C+1 <= q <= RC-C-5
// A row depends on the row above alone, so rows run in sequence and columns in
// parallel.  With the six fixed values sorted (s0 <= ... <= s5) and the three
// recursive ones (u0 <= u1 <= u2), the 5th smallest of the nine is
//   min(s4, max(s3, u0), max(s2, u1), max(s1, u2))
// (k-th smallest of the union of two sorted lists; s0 and s5 can never be the
// median).
#include <hip/hip_runtime.h>
#include <algorithm>
#include "rig.h"
#include "kernels.h"
#include "lanes.h"

namespace sister {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// three values sorted, two columns at a time
struct Tri { us2 lo, mid, hi; };
__device__ __forceinline__ Tri sort3(us2 a, us2 b, us2 c)
{
    return {umin3(a, b, c), umax2(umin2(a, b), umin2(umax2(a, b), c)), umax3(a, b, c)};
}
// the 2nd to 5th smallest of two sorted triples
struct Mid4 { us2 s1, s2, s3, s4; };
__device__ __forceinline__ Mid4 merge(const Tri& x, const Tri& y)
{
    return {umin3(x.mid, y.mid, umax2(x.lo, y.lo)),
            umin2(umin3(x.hi, y.hi, umax2(x.lo, y.mid)), umax2(x.mid, y.lo)),
            umin3(umax2(x.lo, y.hi), umax2(x.mid, y.mid), umax2(x.hi, y.lo)),
            umin2(umax2(x.mid, y.hi), umax2(x.hi, y.mid))};
}
__device__ __forceinline__ us2 med9(const Mid4& s, const Tri& u)
{
    return umin2(umin3(s.s4, umax2(s.s3, u.lo), umax2(s.s2, u.mid)), umax2(s.s1, u.hi));
}
// pairs (a.hi, b.lo): one column to the left of b's pair, right of a's
__device__ __forceinline__ us2 between(uint32_t a, uint32_t b) { return U2(__builtin_amdgcn_alignbit(b, a, 16)); }

// The order statistics s1..s4 of every position as bytes (D <= 256), a dword a
// position.
__global__ __launch_bounds__(256) void k_median_prep(const RigDesc* __restrict__ rigs, int nrig,
                                                     const int* __restrict__ bs, uint64_t* const* __restrict__ scratch)
{
    const int ri = find_rig(bs, nrig, blockIdx.x);
    const RigDesc& g = rigs[ri];
    const long npair = (long)g.Wp * g.Hp / 2;
    const long perMap = (npair + 255) / 256;
    const long lb = blockIdx.x - bs[ri];
    const int m = (int)(lb / perMap);
    const long i = (lb % perMap) * 256 + threadIdx.x;
    if (i >= npair) return;
    const long C2 = frame_cols(g, m >> 1) / 2;   // C and R C are multiples of 4
    const uint32_t* in = (const uint32_t*)g.wta[m];
    uint2* out = (uint2*)(scratch[ri] + (size_t)m * 2 * npair) + i;
    if (i < C2 || i > npair - C2 - 3) { *out = make_uint2(0, 0); return; }
    const uint32_t a0 = in[i - 1], a1 = in[i], a2 = in[i + 1];
    const uint32_t b0 = in[i + C2 - 1], b1 = in[i + C2], b2 = in[i + C2 + 1];
    const Mid4 s = merge(sort3(between(a0, a1), U2(a1), between(a1, a2)), sort3(between(b0, b1), U2(b1), between(b1, b2)));
    const uint32_t a = W2(s.s1) | (W2(s.s2) << 8), b = W2(s.s3) | (W2(s.s4) << 8);   // (s1, s2), (s3, s4) by column
    *out = make_uint2(__builtin_amdgcn_perm(b, a, 0x05040100u), __builtin_amdgcn_perm(b, a, 0x07060302u));
}

// ---------------------------------------------------------------------------
// The recursion: one block per (rig, map), a wave per strip of columns.  A
// lane holds K pairs of neighbouring columns, so the three upper neighbours of
// a pair are a byte shift of neighbouring registers (across lanes one DPP
// move) and everything is packed 16-bit arithmetic.  A strip also carries
// kMedGhost columns on each side, copies of its neighbours' columns: a wrong
// value entering at a strip's edge moves inwards one column per row, so the
// columns it owns stay right for kMedGhost rows with no exchange.  The waves
// meet once per kMedSeg rows, publish their columns in LDS and read their
// ghosts anew.
// Columns are flat: column C of row r is column 0 of row r + 1, column -1 is
// column C - 1 of row r - 1, which is the recursion's own raster neighbourhood.
// The first strip's left ghosts are therefore the last columns of the row
// before, and the last strip's right ghosts the first columns of the next row,
// which the first wave computes one row ahead when they are published.
// RAW: a row of the map is read once and kept as sorted triples (the six fixed
// values of row r are the triples of rows r and r + 1); otherwise s1..s4 come
// from the prepass.
// What bounds it: a map's rows run on one compute unit, so the instructions of
// a row over its four SIMDs (15 per pair and 14 from the prepass, 33 and 14
// raw) set the time, if the row's bytes do not: one CU moves 35-55 GB/s, which
// is why the prepass keeps bytes (statistics of 16 bits: 768 us where bytes
// take 500). Loads run NB - 1 rows ahead (none in k_median_wide: no registers
// left).  Per map set of one rig, against a block of 1024 threads with one
// barrier per row: 640x480 D=64 225 -> 102 us, 1920x1080 D=192 920 -> 500 us;
// 64 rigs of 1920x1080 (raw) 5.0 -> 1.4 ms.
// ---------------------------------------------------------------------------
constexpr int kMedGhost = 16, kMedSeg = 12;

template <int K> struct MedStrip {
    static constexpr int LC = 2 * K;                               // columns per lane
    static constexpr int GL = (kMedGhost + LC - 1) / LC;           // ghost lanes per side
    static constexpr int OW = (64 - 2 * GL) * LC;                  // columns a wave owns
};

// row r's step needs row 0 .. row 13 (1 + kMedSeg) from the first ghosts, one
// more where the first wave runs ahead
static_assert(1 + kMedSeg + 1 <= kMedGhost, "ghost columns cover a segment and the row ahead");

size_t median_lds(int C) { return 2 * ((size_t)C / 2 + kMedGhost) * sizeof(uint32_t); }

template <int K, bool RAW, int NB>
__device__ __forceinline__ void median_strip(int R, int C, uint16_t* in, uint16_t* out, uint64_t* pre, uint32_t* lds)
{
    typedef MedStrip<K> S;
    static_assert(kMedSeg % NB == 0, "ring slots are compile-time");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nfull = (R - 4) / kMedSeg;
    if (wave * S::OW >= C) {   // no columns: only the barriers
        for (int s = 0; s < nfull; s++) __syncthreads();
        return;
    }
    const int c0 = wave * S::OW + (lane - S::GL) * S::LC;   // the lane's first column
    const bool olane = lane >= S::GL && lane < 64 - S::GL;
    // raw buffers: an offset past the map (or before it) reads 0 and stores nothing
    const auto rin = buf((uint8_t*)in, (uint32_t)(R * C) * 2u), rout = buf((uint8_t*)out, (uint32_t)(R * C) * 2u);
    const auto rpre = buf((uint8_t*)pre, (uint32_t)(R * C) * 4u);
    const uint32_t rb = (uint32_t)C * 2u;                   // bytes per row
    // store offset of the lane's columns, all of them inside the row, or (sp, at
    // most one lane of the block) of those inside it, by groups of 4 (C % 4 == 0)
    const int room = olane ? min(max(C - c0, 0), S::LC) : 0;
    uint32_t so = room == S::LC ? (uint32_t)c0 * 2u : kDropped;
    uint32_t sp = room > 0 && room < S::LC ? (uint32_t)c0 * 2u : kDropped;
    const bool part = __builtin_amdgcn_ballot_w64(sp != kDropped) != 0;

    struct Row { uint32_t w[RAW ? K : 2 * K]; };
    uint32_t L[K];            // the row above's results
    Tri T[K];                 // RAW: sorted triples of the current row
    auto load_in = [&](uint32_t off, uint32_t (&w)[K]) __attribute__((always_inline)) {
        static_for<0, K / 4>([&](auto kc) { buf_load<4>(w + 4 * decltype(kc)::value, rin, off + 16u * decltype(kc)::value); });
        if constexpr (K % 4 == 2) buf_load<2>(w + K - 2, rin, off + 4u * (K - 2));
    };
    auto triples = [&](const uint32_t (&w)[K], Tri (&t)[K]) __attribute__((always_inline)) {
        const uint32_t pl = wave_from_left(w[K - 1]), pr = wave_from_right(w[0]);
#pragma unroll
        for (int j = 0; j < K; j++)
            t[j] = sort3(between(j ? w[j - 1] : pl, w[j]), U2(w[j]), between(w[j], j + 1 < K ? w[j + 1] : pr));
    };
    // what row r needs: its order statistics, or the input row below it
    uint32_t fo = (uint32_t)((RAW ? 2 : 1) * C + c0) * (RAW ? 2u : 4u);   // of row 1
    auto fetch = [&](Row& b) __attribute__((always_inline)) {
        if constexpr (RAW) load_in(fo, b.w);
        else static_for<0, K / 2>([&](auto kc) { buf_load<4>(b.w + 4 * decltype(kc)::value, rpre, fo + 16u * decltype(kc)::value); });
        fo += RAW ? rb : 2u * rb;
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](const Row& b, uint32_t (&l)[K], Tri (&t)[K]) __attribute__((always_inline)) {
        const uint32_t pl = wave_from_left(l[K - 1]), pr = wave_from_right(l[0]);
        Tri n[RAW ? K : 1];
        if constexpr (RAW) triples(b.w, n);
        uint32_t prev = pl;
#pragma unroll
        for (int j = 0; j < K; j++) {
            const uint32_t nx = j + 1 < K ? l[j + 1] : pr, cur = l[j];
            const Tri u = sort3(between(prev, cur), U2(cur), between(cur, nx));
            Mid4 s;
            if constexpr (RAW) {
                s = merge(t[j], n[j]);
                t[j] = n[j];
            } else {
                // byte k of both columns as a pair
                auto byte = [&](uint32_t sel) __attribute__((always_inline)) {
                    return U2(__builtin_amdgcn_perm(b.w[2 * j + 1], b.w[2 * j], sel));
                };
                s = {byte(0x0c040c00u), byte(0x0c050c01u), byte(0x0c060c02u), byte(0x0c070c03u)};
            }
            prev = cur;
            l[j] = W2(med9(s, u));
        }
    };
    auto put = [&](const uint32_t (&w)[K], uint32_t row) __attribute__((always_inline)) {
        static_for<0, K / 4>([&](auto kc) { buf_store<4>(w + 4 * decltype(kc)::value, rout, so + row + 16u * decltype(kc)::value); });
        if constexpr (K % 4 == 2) buf_store<2>(w + K - 2, rout, so + row + 4u * (K - 2));
        if (part)
            static_for<0, K / 2>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                buf_store<2>(w + 2 * k, rout, 4 * k < room ? sp + row + 8u * k : kDropped);
            });
    };
    auto store = [&]() __attribute__((always_inline)) {
        so += rb;
        sp += rb;
        put(L, 0);
        __builtin_amdgcn_sched_barrier(0);
    };

    // rows 0 and R - 1 are copied; L = row 0
    load_in((uint32_t)c0 * 2u, L);
    {
        uint32_t w[K];
        load_in((uint32_t)((R - 1) * C + c0) * 2u, w);
        put(L, 0);
        put(w, (uint32_t)(R - 1) * rb);
    }
    // columns C .. of row 0 are the first of row 1: position C is 0, the others
    // have row 0's inputs above them
    if (c0 + S::LC > C) {
        static_for<0, 2 * K>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int j = c0 + i - C, q = c0 + i;
            if (j < 0 || j >= kMedGhost) return;
            uint32_t v = 0;
            if (j > 0) {
                auto at = [&](int k) { return (us2){G(in)[k], 0}; };
                v = W2(med9(merge(sort3(at(q - 1), at(q), at(q + 1)), sort3(at(q + C - 1), at(q + C), at(q + C + 1))),
                            sort3(at(j - 1), at(j), at(j + 1))));
            }
            L[i / 2] = (i & 1) ? (L[i / 2] & 0xFFFFu) | (v << 16) : (L[i / 2] & 0xFFFF0000u) | (v & 0xFFFFu);
        });
    }
    Row ring[NB];
    if constexpr (RAW) {
        uint32_t w[K];
        load_in((uint32_t)(C + c0) * 2u, w);
        triples(w, T);
    }
    // row 1: position C is 0, positions below C (columns < 0) are row 0's inputs
    fetch(ring[0]);
    step(ring[0], L, T);
    {
        uint32_t w[K];
        load_in((uint32_t)(C + c0) * 2u, w);
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int c = c0 + 2 * j;
            L[j] = c < 0 ? w[j] : c == 0 ? L[j] & 0xFFFF0000u : L[j];
        }
    }
    store();
    static_for<0, NB - 1>([&](auto ic) __attribute__((always_inline)) { fetch(ring[decltype(ic)::value]); });
    int p = 0;
    uint32_t Lp[K];
    for (int s = 0; s < nfull; s++) {
        static_for<0, kMedSeg>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            fetch(ring[(i + NB - 1) % NB]);
            if constexpr (i == kMedSeg - 1) {
#pragma unroll
                for (int j = 0; j < K; j++) Lp[j] = L[j];
            }
            step(ring[i % NB], L, T);
            store();
        });
        // publish: the row's columns, the row before's last ones, the next
        // row's first ones (two buffers: a wave is at most one segment ahead)
        uint32_t* const cur = lds + p * (C / 2 + kMedGhost);
        uint32_t* const tail = cur + C / 2;
        uint32_t* const head = tail + kMedGhost / 2;
        p ^= 1;
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int c = c0 + 2 * j;
            if (olane && c < C) {
                cur[c / 2] = L[j];
                if (c >= C - kMedGhost) tail[(c - (C - kMedGhost)) / 2] = Lp[j];
            }
        }
        if (wave == 0) {
            uint32_t l[K];
            Tri t[K];
#pragma unroll
            for (int j = 0; j < K; j++) {
                l[j] = L[j];
                if constexpr (RAW) t[j] = T[j];
            }
            if constexpr (NB == 1) {   // not requested yet
                fetch(ring[0]);
                fo -= RAW ? rb : 2u * rb;
            }
            step(ring[0], l, t);
#pragma unroll
            for (int j = 0; j < K; j++) {
                const int c = c0 + 2 * j;
                if (c >= 0 && c < kMedGhost) head[c / 2] = l[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int c = c0 + 2 * j;
            if (olane && c < C) continue;
            if (c < 0) {
                if (c >= -kMedGhost) L[j] = tail[(c + kMedGhost) / 2];
            } else if (c < C) {
                L[j] = cur[c / 2];
            } else if (c < C + kMedGhost) {
                L[j] = head[(c - C) / 2];
            }
        }
    }
    // the rows left before R - 2
    const int left = R - 4 - nfull * kMedSeg;
    static_for<0, kMedSeg - 1>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if (i < left) {
            fetch(ring[(i + NB - 1) % NB]);
            step(ring[i % NB], L, T);
            store();
        }
    });
    // row R - 2: its last four positions (and all beyond) are copied
    fo = RAW ? (uint32_t)((R - 1) * C + c0) * 2u : (uint32_t)((R - 2) * C + c0) * 4u;
    fetch(ring[0]);
    step(ring[0], L, T);
    {
        uint32_t w[K];
        load_in((uint32_t)((R - 2) * C + c0) * 2u, w);
#pragma unroll
        for (int j = 0; j < K; j++) L[j] = c0 + 2 * j >= C - 4 ? w[j] : L[j];
    }
    store();
}

// K by frame width: with up to four waves (one per SIMD) a row costs one
// wave's instructions, 14 K + 14 (prepass) or 33 K + 14 (raw), so the smallest
// K that needs no more than four; beyond 2880 columns two waves per SIMD.
// Wider than kMedNarrow: more than eight waves, k_median_wide.
constexpr int kMedNarrow = 8 * MedStrip<10>::OW;
__host__ __device__ inline int med_pairs(int C)
{
    return C <= 4 * MedStrip<2>::OW ? 2 : C <= 4 * MedStrip<4>::OW ? 4 : C <= 4 * MedStrip<6>::OW ? 6
         : C <= 8 * MedStrip<4>::OW ? 4 : C <= 8 * MedStrip<6>::OW ? 6 : 10;
}
static int med_waves(int C)
{
    auto n = [&](int ow) { return (C + ow - 1) / ow; };
    switch (med_pairs(C)) {
    case 2: return n(MedStrip<2>::OW);
    case 4: return n(MedStrip<4>::OW);
    case 6: return n(MedStrip<6>::OW);
    default: return n(MedStrip<10>::OW);
    }
}

// Blocks are dispatched long maps first: block b takes map slot b / nrig of rig
// b % nrig, slots 0-3 being the rig's four maps of the frames with more rows
// (the chain is one row per step) and slots 4-7 the other four.  When the
// blocks take more than one round of the CUs, the short maps then fill the CUs
// the long ones leave, instead of long maps starting last.
__device__ __forceinline__ int median_map(const RigDesc& g, int slot)
{
    // frames 1/3 have W' rows, frames 0/2 H' rows; map m = 2 F + side
    const int long_odd = g.Wp > g.Hp ? 1 : 0;
    const int fr = (slot >> 1) & 1, side = slot & 1;             // frame pair index, side
    const int F = ((slot < 4) == (long_odd == 1)) ? 2 * fr + 1 : 2 * fr;
    return 2 * F + side;
}

// NW: most waves of a block.  Four waves leave each its SIMD's 512 registers,
// eight half: the rings of prefetched rows are sized for that.
template <bool RAW, int NW>
__global__ __launch_bounds__(64 * NW) void k_median(const RigDesc* __restrict__ rigs, int nrig,
                                                    uint64_t* const* __restrict__ scratch)
{
    extern __shared__ uint32_t lds32[];
    const int ri = blockIdx.x % nrig;
    const RigDesc& g = rigs[ri];
    const int m = median_map(g, blockIdx.x / nrig);
    const int R = frame_rows(g, m >> 1), C = frame_cols(g, m >> 1);
    if (C > kMedNarrow) return;
    uint64_t* pre = scratch[ri] + (size_t)m * R * C;
    constexpr bool deep = RAW || NW == 4;
    switch (med_pairs(C)) {
    case 2: median_strip<2, RAW, 12>(R, C, g.wta[m], g.med[m], pre, lds32); break;
    case 4: median_strip<4, RAW, deep ? 12 : 6>(R, C, g.wta[m], g.med[m], pre, lds32); break;
    case 6: median_strip<6, RAW, deep ? 12 : 6>(R, C, g.wta[m], g.med[m], pre, lds32); break;
    default: median_strip<10, RAW, RAW ? 6 : 4>(R, C, g.wta[m], g.med[m], pre, lds32); break;
    }
}

// frames wider than kMedNarrow, up to 16 waves
template <bool RAW>
__global__ __launch_bounds__(1024) void k_median_wide(const RigDesc* __restrict__ rigs, int nrig,
                                                      uint64_t* const* __restrict__ scratch)
{
    extern __shared__ uint32_t lds32[];
    const int ri = blockIdx.x % nrig;
    const RigDesc& g = rigs[ri];
    const int m = median_map(g, blockIdx.x / nrig);
    const int R = frame_rows(g, m >> 1), C = frame_cols(g, m >> 1);
    if (C <= kMedNarrow) return;
    median_strip<10, RAW, 1>(R, C, g.wta[m], g.med[m], scratch[ri] + (size_t)m * R * C, lds32);
}

int median_setup(int lds_limit)
{
    // frames past 16 k columns of LDS rows take more than the default 64 KB
    for (const void* f : {(const void*)k_median_wide<false>, (const void*)k_median_wide<true>})
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_limit) != hipSuccess) return -1;
    return 0;
}

#define TB(id) do { if (t) t->begin(id, st); } while (0)
#define TE(id) do { if (t) t->end(id, st); } while (0)
#define TD(id, n) do { if (t) t->dispatched[id] += (n); } while (0)

void launch_median(const LaunchSet& ls, hipStream_t st, KernelTimer* t)
{
    // With enough (rig, map) blocks to spread over the chip the recursion sorts
    // each position's six fixed values itself; with few, each block's row chain
    // is the critical path and the parallel prepass takes the sorting off it.
    // Between: eight 1920x1080 rigs take 815 us raw, 500 us and 60 us a rig for
    // the prepass otherwise.  Disparities past 255 do not fit the prepass's bytes.
    const bool raw = ls.nrig * 8 >= std::max(g_num_cu / 4, 1) || ls.maxD > 256;
    if (!raw) {
        TB(kKMedianPrep);
        hipLaunchKernelGGL(k_median_prep, dim3(ls.blocks[kStageMedianPrep]), dim3(256), 0, st, ls.rigs, ls.nrig,
                           ls.bs[kStageMedianPrep], ls.scratch);
        TD(kKMedianPrep, 1);
        TE(kKMedianPrep);
    }
    TB(kKMedianSerial);
    if (ls.med_waves > 0) {
        const dim3 grid(ls.nrig * 8), block(64 * ls.med_waves);
        const size_t lds = median_lds(std::min(ls.maxCols, kMedNarrow));
        const bool four = ls.med_waves <= 4;
#define SISTER_MEDIAN(RAWV, NWV) \
    hipLaunchKernelGGL((k_median<RAWV, NWV>), grid, block, lds, st, ls.rigs, ls.nrig, ls.scratch)
        if (raw) SISTER_MEDIAN(true, 8);
        else if (four) SISTER_MEDIAN(false, 4);
        else SISTER_MEDIAN(false, 8);
#undef SISTER_MEDIAN
        TD(kKMedianSerial, 1);
    }
    if (ls.maxCols > kMedNarrow) {
        const dim3 grid(ls.nrig * 8), block(64 * med_waves(ls.maxCols));
        const size_t lds = median_lds(ls.maxCols);
        if (raw) hipLaunchKernelGGL(k_median_wide<true>, grid, block, lds, st, ls.rigs, ls.nrig, ls.scratch);
        else hipLaunchKernelGGL(k_median_wide<false>, grid, block, lds, st, ls.rigs, ls.nrig, ls.scratch);
        TD(kKMedianSerial, 1);
    }
    TE(kKMedianSerial);
}

// waves of the rig's widest map that k_median takes (0: it takes none of them)
int median_waves(const RigDesc& g)
{
    int n = 0;
    for (int C : {g.Wp, g.Hp})
        if (C <= kMedNarrow) n = std::max(n, med_waves(C));
    return n;
}

}  // namespace sister
