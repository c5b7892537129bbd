// kernels.hip -- gfx950 kernels of the 5-view disparity path.
//
// Stage map (reference file:line -> kernel):
//   censusTransform        census.cpp:38-51             k_census
//   WTALeft/WTARight on    postprocess.cpp:74-315       k_wta (wta.hip; cost recomputed from
//     the raw frame DSIs     (hpp:196-197,...)                   census, never stored)
//   median3x3_SSE in place postprocess.cpp:15-71        k_median (median.hip)
//   doLRCheck + mask loops postprocess.cpp:318-341,     k_mask
//                          hpp:201-251
//   realign + weighted sum hpp:255-277                  k_cost (cost.hip)
//   accumulateCostsSSE     sgm.cpp:26-455               k_paths (paths.hip); batches: rows
//                                                       in k_paths, the rest in k_vsweep
//   WTALeft on S, convert  hpp:283,111-118              k_winner (paths.hip), or in k_vsweep
//
// Every kernel takes the rig table plus a block-start table so one launch can
// cover many rigs of different sizes: block b belongs to rig i when
// bs[i] <= b < bs[i+1].
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdlib>
#include "rig.h"
#include "kernels.h"
#include "lanes.h"

namespace sister {

// padded original (y, x) of frame pixel (r, c)
__device__ __forceinline__ void frame_to_orig(const RigDesc& g, int F, int r, int c, int& y, int& x)
{
    switch (F) {
    case 0: y = r; x = c; break;
    case 1: y = g.Hp - 1 - c; x = g.Wp - 1 - r; break;
    case 2: y = r; x = g.Wp - 1 - c; break;
    default: y = c; x = g.Wp - 1 - r; break;
    }
}

// frame pixel (r, c) of padded original (y, x)
__device__ __forceinline__ void orig_to_frame(const RigDesc& g, int F, int y, int x, int& r, int& c)
{
    switch (F) {
    case 0: r = y; c = x; break;
    case 1: r = g.Wp - 1 - x; c = g.Hp - 1 - y; break;
    case 2: r = y; c = g.Wp - 1 - x; break;
    default: r = g.Wp - 1 - x; c = y; break;
    }
}

// pixel of the replicate-padded view (copyMakeBorder REPLICATE, hpp:35-39)
__device__ __forceinline__ int padded_px(const RigDesc& g, const uint8_t* v, int y, int x)
{
    y = min(max(y - g.D, 0), g.H - 1);
    x = min(max(x - g.D, 0), g.W - 1);
    return v[(size_t)y * g.stride + x];
}

__device__ __forceinline__ int frame_px(const RigDesc& g, const uint8_t* v, int F, int r, int c)
{
    int y, x;
    frame_to_orig(g, F, r, c, y, x);
    return padded_px(g, v, y, x);
}

// ---------------------------------------------------------------------------
// K1 census (census.cpp:38-51), one 32x32 tile of frame pixels per block.
// Test bit for offset (y,x), y=-3..3 outer, x=-4..4 inner, is
// I(r+y, c+x) > I(r-y, c-x), shifted in MSB-first; bit 63 carries bit 0 of
// the previous domain pixel in frame raster order (the accumulator is never
// reset, census.cpp:42), i.e. the (3,4) test of that pixel.
// The tile (frame rows r0-3 .., columns c0-8 ..) is staged in LDS as bytes,
// rows 40 dwords apart (40 = 8 mod 32 banks: the 32 lanes of a half-wave,
// 4 rows x 8 runs, read 32 different banks).  A thread takes a run of 4
// frame pixels of one row and reads each of its 7 window rows once as 3 or 4
// aligned dwords; one alignbyte gathers a test's 4 left-hand bytes (one per
// pixel), another the 4 right-hand bytes, and each pixel's two bits come from
// two byte-select subtractions.
// ---------------------------------------------------------------------------
constexpr int kCT = 32;   // tile side (frame pixels)

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_census(const RigDesc* __restrict__ rigs, int nrig,
                                                const int* __restrict__ bs)
{
    constexpr int TR = kCT + 6;       // frame rows r0-3 .. r0+kCT+2
    constexpr int TB = kCT + 12;      // bytes used per row: columns c0-8 .. c0+kCT+3
    constexpr int TW = 40;            // dwords per tile row
    __shared__ uint32_t tile[TR * TW];
    uint8_t* const tb = (uint8_t*)tile;
    const int ri = find_rig(bs, nrig, blockIdx.x);
    const RigDesc& g = rigs[ri];
    const int lb = blockIdx.x - bs[ri];
    const int T = ((g.Wp + kCT - 1) / kCT) * ((g.Hp + kCT - 1) / kCT);
    const int unit = lb / T, t = lb % T;
    const int F = unit >> 1;
    const int R = frame_rows(g, F), C = frame_cols(g, F);
    const int tilesC = (C + kCT - 1) / kCT;
    const int r0 = (t / tilesC) * kCT, c0 = (t % tilesC) * kCT;
    const uint8_t* v = g.view[(unit & 1) ? 1 + F : 0];
    // rows of the deep padding bands other than their first rows are never
    // stored (readers take the first row, band_row): a tile of such rows only
    // has nothing to do
    if (r0 + kCT - 1 < R && band_row(r0, R, g.D) != r0 && band_row(r0 + kCT - 1, R, g.D) != r0 + kCT - 1 &&
        band_row(r0, R, g.D) == band_row(r0 + kCT - 1, R, g.D))
        return;

    // frames 90/270 are transposes: step along frame rows there, so that
    // consecutive lanes read along an image row
    const bool odd = F & 1;
    for (int i = threadIdx.x; i < TR * TB; i += 256) {
        const int rr = odd ? i % TR : i / TB, cc = odd ? i / TR : i % TB;
        const int r = r0 - 3 + rr, c = c0 - 8 + cc;
        tb[rr * TW * 4 + cc] = (r >= 0 && r < R && c >= 0 && c < C) ? (uint8_t)frame_px(g, v, F, r, c) : 0;
    }
    __syncthreads();
    // codes of the run of pixels (r0 + rl, c0 + 4 run .. + 3), from the tile
    auto run_codes = [&](int rl, int run, uint64_t (&code)[4]) __attribute__((always_inline)) {
        const int r = r0 + rl, cb = c0 + 4 * run;
        // w[i][k]: dword run + k of tile row rl + i (frame row r - 3 + i); byte b of
        // the run's window is frame column cb - 8 + b
        uint32_t w[7][4];
#pragma unroll
        for (int i = 0; i < 7; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) w[i][k] = tile[(rl + i) * TW + run + k];
        // bytes s .. s+3 of row i: byte p is pixel p's entry at window byte s + p
        auto quad = [&](int i, int sb) __attribute__((always_inline)) {
            return (sb & 3) == 0 ? w[i][sb >> 2] : __builtin_amdgcn_alignbyte(w[i][(sb >> 2) + 1], w[i][sb >> 2], sb & 3);
        };
        // test u (offset (u/9 - 3, u%9 - 4)) and its mirror 62 - u compare the same
        // two pixels in opposite order: bit 62 - u = (a > b) is the sign of b - a,
        // bit u = (b > a) the sign of a - b.  hi collects bits 62..32 MSB-first;
        // lf collects bits 0..30 in the same order and is bit-reversed at the end.
        uint32_t hi[4] = {0, 0, 0, 0}, lf[4] = {0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < 31; u++) {
            const int y = u / 9 - 3, x = u % 9 - 4;
            const uint32_t qa = quad(3 + y, 8 + x), qb = quad(3 - y, 8 - x);
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const uint32_t a = (qa >> (8 * p)) & 0xFFu, b = (qb >> (8 * p)) & 0xFFu;
                hi[p] = __builtin_amdgcn_alignbit(hi[p], b - a, 31);
                lf[p] = __builtin_amdgcn_alignbit(lf[p], a - b, 31);
            }
        }
        // carry of pixel c: the (3,4) test of pixel c-1, I(r+3, c+3) > I(r-3, c-5)
        const uint32_t ca = quad(6, 11 + 0), cbq = quad(0, 3);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int c = cb + p;
            code[p] = 0;
            if (r >= 3 && r < R - 3 && c >= 4 && c < C - 4) {
                const uint32_t lo = __builtin_bitreverse32(lf[p]) >> 1;
                unsigned carry;
                if (c > 4)
                    carry = ((ca >> (8 * p)) & 0xFFu) > ((cbq >> (8 * p)) & 0xFFu);
                else if (r > 3)
                    carry = frame_px(g, v, F, r + 2, C - 1) > frame_px(g, v, F, r - 4, C - 9);  // (r-1, C-5)
                else
                    carry = 0;
                code[p] = ((uint64_t)(hi[p] | (carry << 31)) << 32) | lo;
            }
        }
    };
    auto store_run = [&](int r, int cb, const uint64_t (&code)[4]) __attribute__((always_inline)) {
        if (band_row(r, R, g.D) != r) return;                // a band's copy row: not stored
        uint64_t* out = g.code[unit] + (size_t)r * C + cb;   // 32-byte aligned: cb % 4 == 0
        ST16(out, make_uint4((uint32_t)code[0], (uint32_t)(code[0] >> 32), (uint32_t)code[1], (uint32_t)(code[1] >> 32)));
        ST16(out + 2, make_uint4((uint32_t)code[2], (uint32_t)(code[2] >> 32), (uint32_t)code[3], (uint32_t)(code[3] >> 32)));
    };
    const int run = threadIdx.x & 7, rl = threadIdx.x >> 3;
    // Tiles in the deep padding.  With replicate padding the window of a pixel
    // at frame rows [3, D-4] holds the image's first row only (rows
    // [R-D+3, R-4]: its last row), so its code does not depend on the row; the
    // carry of column 4 compares two copies of one pixel there (0, as at row
    // 3).  Likewise a pixel at columns [5, D-5] or [C-D+4, C-5] sees one image
    // column and its carry compares two copies of the same column, so within a
    // row its code does not depend on the column.  A tile wholly inside such a
    // band computes its distinct codes in one wave (one run of 4 per tile row
    // band, one pixel per row for a column band, one code for both) and copies.
    const int D = g.D;
    const bool rows_deep = (r0 >= 3 && r0 + kCT - 1 <= D - 4) || (r0 >= R - D + 3 && r0 + kCT - 1 <= R - 4);
    const bool cols_deep = (c0 >= 5 && c0 + kCT - 1 <= D - 5) || (c0 >= C - D + 4 && c0 + kCT - 1 <= C - 5);
    const bool deep = rows_deep || cols_deep;   // uniform over the block
    const int nrep = rows_deep ? (cols_deep ? 1 : kCT / 4) : kCT;
    const bool work = deep ? (int)threadIdx.x < nrep : r0 + rl < R && c0 + 4 * run < C;
    uint64_t code[4] = {0, 0, 0, 0};
    if (work)
        run_codes(deep ? (rows_deep ? 0 : (int)threadIdx.x) : rl,
                  deep ? (rows_deep && !cols_deep ? (int)threadIdx.x : 0) : run, code);
    if (deep) {
        __shared__ uint64_t rep[kCT * 4];
        if (work) {
#pragma unroll
            for (int p = 0; p < 4; p++) rep[threadIdx.x * 4 + p] = code[p];
        }
        __syncthreads();
        // a row band's tile may end past column C, a column band's past row R
        if (r0 + rl >= R || c0 + 4 * run >= C) return;
#pragma unroll
        for (int p = 0; p < 4; p++)
            code[p] = rows_deep ? (cols_deep ? rep[0] : rep[run * 4 + p]) : rep[rl * 4];
    } else if (!work) {
        return;   // C is a multiple of 4, so a run is all in or all out
    }
    store_run(r0 + rl, c0 + 4 * run, code);
}

// ---------------------------------------------------------------------------
// K4 LR check + mask (postprocess.cpp:318-341, hpp:201-206 etc.): frame pixel
// (r,c) keeps L when 0 <= L <= c and |L - R[c-L]| <= 5; mask = kept && L > 0
// && c >= D, written at the padded original coordinates (hpp:216,235-236,250-251).
// ---------------------------------------------------------------------------
// One block per 32x32 tile of frame pixels (4 per thread), read along frame
// rows.  Frames 0/180 store along image rows directly; frames 90/270, whose
// frame rows are image columns, pass the tile through LDS so that their
// stores also run along image rows.
constexpr int kMT32 = 32;

__global__ __launch_bounds__(256) void k_mask(const RigDesc* __restrict__ rigs, int nrig,
                                              const int* __restrict__ bs, int fmask)
{
    __shared__ uint8_t tile[kMT32][kMT32 + 1];
    const int ri = find_rig(bs, nrig, blockIdx.x);
    const RigDesc& g = rigs[ri];
    const int T = ((g.Wp + kMT32 - 1) / kMT32) * ((g.Hp + kMT32 - 1) / kMT32);
    const int lb = blockIdx.x - bs[ri];
    const int F = lb / T, t = lb % T;
    if (!(fmask & (1 << F))) return;
    const int R = frame_rows(g, F), C = frame_cols(g, F);
    const int tilesC = (C + kMT32 - 1) / kMT32;
    const int r0 = (t / tilesC) * kMT32, c0 = (t % tilesC) * kMT32;
    const int tc = threadIdx.x % kMT32, tr = threadIdx.x / kMT32;
    const uint16_t* ml = g.med[2 * F];
    const uint16_t* mr = g.med[2 * F + 1];
    uint8_t* const mk = g.mask[F];
    const bool odd = F & 1;
#pragma unroll
    for (int k = 0; k < kMT32 / 8; k++) {
        const int r = r0 + tr + 8 * k, c = c0 + tc;
        if (r >= R || c >= C) continue;
        const size_t q = (size_t)r * C + c;
        const int L = G(ml)[q];
        unsigned ok = 0;
        if (c >= g.D && L >= 1 && L <= c) {
            const int Rv = G(mr)[q - L];
            ok = abs(L - Rv) <= kLrThreshold;
        }
        if (odd) {
            tile[tr + 8 * k][tc] = (uint8_t)ok;
        } else {
            int y, x;
            frame_to_orig(g, F, r, c, y, x);
            G(mk)[(size_t)y * g.Wp + x] = (uint8_t)ok;
        }
    }
    if (!odd) return;
    __syncthreads();
    // frame (r, c) -> image (y, x): x = W'-1-r for both frames, y = H'-1-c
    // (90) or c (270); a thread takes frame row r0 + tc (image column) and
    // columns c0 + tr + 8 k (image rows), so lanes store along image rows
#pragma unroll
    for (int k = 0; k < kMT32 / 8; k++) {
        const int r = r0 + tc, c = c0 + tr + 8 * k;
        if (r >= R || c >= C) continue;
        int y, x;
        frame_to_orig(g, F, r, c, y, x);
        G(mk)[(size_t)y * g.Wp + x] = tile[tc][tr + 8 * k];
    }
}

// One chain is held by KL consecutive lanes; lane `lid` of the group owns
// chunks [lid*CH, lid*CH + CH) of the chain's Dp/16 chunks (16 disparities,
// 8 packed pairs each).  Chunks at or beyond nq are padding and stay guards.
template <int CH>
struct LaneState {
    uint32_t L[8 * CH];
    uint32_t mp;
};

struct ChainGeo {
    int lid;        // lane within the chain group
    int nq;         // valid chunks of the chain
    bool half_tail; // D % 16 == 8: the last valid chunk holds 4 real pairs
};

// One standard step (paths.hip) over the lane's chunks, the cost pairs taken
// from packed bytes (4 per word, 16 per chunk).  DEFER: the state is kept raw
// (minL' not subtracted): the new raw values are the normalized ones plus the
// previous raw minimum, which the caller tracks.
template <int CH, int KL, bool DEFER>
__device__ __forceinline__ void lane_step(LaneState<CH>& st, const ChainGeo& cg, const uint4 (&mb)[CH])
{
    // left lane's last pair and right lane's first pair (old); KL divides the
    // 16-lane DPP row, so the lanes at a row's ends are group ends, which take
    // the guard instead
    const uint32_t nbl = row_shr1(st.L[8 * CH - 1]);
    const uint32_t nbr = row_shl1(st.L[0]);
    uint32_t prv = (cg.lid == 0) ? kGuard2 : nbl;
    const uint32_t rfill = (cg.lid == KL - 1) ? kGuard2 : nbr;
    const uint32_t mpp = dup16(st.mp);
    const us2 p2t = U2(mpp) + (us2){(unsigned short)kP2, (unsigned short)kP2};
    us2 rmin;
    static_for<0, CH>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int qg = cg.lid * CH + q;
        const bool valid = qg < cg.nq;
        const bool ht = cg.half_tail && qg == cg.nq - 1;
        // every new value is below 0x4000 (at most P2 + 255 normalised, raw
        // values stay below the guard), so or-ing the guard 0x3FFF into a
        // padding pair yields the guard itself
        const uint32_t pad_lo = valid ? 0u : kGuard2;           // pairs 0..3 of the chunk
        const uint32_t pad_hi = valid && !ht ? 0u : kGuard2;    // pairs 4..7
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int j = 8 * q + i;
            const uint32_t w = i < 2 ? mb[q].x : i < 4 ? mb[q].y : i < 6 ? mb[q].z : mb[q].w;
            const uint32_t m = (i & 1) ? bytes23(w) : bytes01(w);
            const uint32_t cur = st.L[j];
            const uint32_t nxt = (j + 1 < 8 * CH) ? st.L[j + 1] : rfill;
            const us2 left = U2(__builtin_amdgcn_alignbit(cur, prv, 16));
            const us2 right = U2(__builtin_amdgcn_alignbit(nxt, cur, 16));
            const us2 nb = umin2(left, right) + (us2){(unsigned short)kP1, (unsigned short)kP1};
            const us2 t = umin3(nb, U2(cur), p2t);   // below 0x7C00: at most the guard + 255 + P2
            const us2 d = DEFER ? t : t - U2(mpp);
            const us2 l = U2(W2(d + U2(m)) | (i < 4 ? pad_lo : pad_hi));
            if (i & 1) rmin = j == 1 ? umin2(U2(st.L[0]), l) : umin3(rmin, U2(st.L[j - 1]), l);
            st.L[j] = W2(l);
            prv = cur;
        }
    });
    st.mp = group_min<KL>(min((uint32_t)rmin.x, (uint32_t)rmin.y));
}

// state <- given pairs (first-line c~ or a restart), padding as guards
template <int CH, int KL>
__device__ __forceinline__ void lane_set(LaneState<CH>& st, const ChainGeo& cg, const uint32_t (&m)[CH][8], bool on)
{
    us2 rmin = U2(0xFFFFFFFFu);
    static_for<0, CH>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int qg = cg.lid * CH + q;
        const bool valid = on && qg < cg.nq;
        const bool ht = cg.half_tail && qg == cg.nq - 1;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t l = (!valid || (ht && i >= 4)) ? kGuard2 : m[q][i];
            st.L[8 * q + i] = l;
            rmin = umin2(rmin, U2(l));
        }
    });
    st.mp = group_min<KL>(min((uint32_t)rmin.x, (uint32_t)rmin.y));
    st.mp = st.mp == 0x3FFFu ? 0u : st.mp;   // a chain with no state yet: minL' = 0
}

template <int CH>
__device__ __forceinline__ void lane_guard(LaneState<CH>& st, bool keep)
{
    static_for<0, 8 * CH>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        st.L[j] = keep ? st.L[j] : kGuard2;
    });
    st.mp = keep ? st.mp : 0u;
}

__device__ __forceinline__ uint4 add_u16x8(uint4 a, uint4 b)
{
    return make_uint4(W2(U2(a.x) + U2(b.x)), W2(U2(a.y) + U2(b.y)), W2(U2(a.z) + U2(b.z)), W2(U2(a.w) + U2(b.w)));
}

// ---------------------------------------------------------------------------
// K6b fused vertical families: the column, diagonal and anti-diagonal chains
// of a pass in one sweep (same recurrence and pass rules as
// k_paths).  Lanes own
// columns (kVKL = 4 lanes per column, CH chunks of 16 disparities each), so
// every cell of a row sees its three vertical paths in one lane group:
//   downward pass:  P = rows_fwd + rows_bwd + sum_f (L_f,down - M)  (u16, rows 1..H'-2)
//   upward pass:    S = 8 M + P + sum_f (L_f,up - M), winner and sub-pixel
// -- 8 bytes per cell over both passes, against 17 for the three separate
// families (5 + 5 + 7).  Along a pass the diagonal-family state moves one
// column per row (down-right, up-left) and the anti-diagonal state the other
// way; both live in LDS, one slot per column, updated in place between
// barriers.  Call FL the family whose state moves to higher columns (diagonal
// going down, anti-diagonal going up) and FR the other.
// A block owns ncol columns and also computes kVGhost ghost columns on each
// side (one wave each; what matters there is the family that flows inwards,
// FL on the left and FR on the right).  A wrong state entering at the ghost
// edge moves inwards one column per row, so the owned columns stay exact for
// kVGhost rows without any exchange with neighbouring blocks: one launch runs
// one segment of kVGhost rows, and the states cross segments through memory
// (owned columns stored at the end, owned + ghost columns loaded at the start).
// No block ever waits for another.
// Buffers: the rows family's two directions in part[0] and part[1] (bytes,
// added as words: each sum is at most 200), P (u16) in psum, or over
// the rows bytes once the down pass has read them in plans short of memory
// (pd_at below), the segment states in vstate
// ([parity][cols, diag, anti][W'][Dp + 16] bytes: the normalised (L - M)
// bytes, then minL').
// ---------------------------------------------------------------------------
#ifndef SISTER_VS_XCD
#define SISTER_VS_XCD 1
#endif
constexpr int kVGhost = 16;        // ghost columns per side = rows per launch
constexpr int kVMaxThreads = 768;  // 12 waves: up to 168 VGPRs per lane
// Lanes per column: 4 up to D = 192 (3 chunks of 16 per lane), 8 up to D =
// 384.  Owned columns per block: 144 with 4 lanes (176 computed, 11 waves;
// 16 blocks per 2304-wide rig), 64 with 8 (96 computed, 12 waves).
__host__ __device__ constexpr int vs_cols(int KL) { return KL == 4 ? 144 : 64; }
// 8-byte granules per pair slot of the family state slots: nt computed
// columns plus the two border columns, KL lanes each, rounded up to 64
__host__ __device__ constexpr int vs_gs(int nt, int KL) { return ((nt + 2) * KL + 63) / 64 * 64; }

template <int CH>
__device__ __forceinline__ void vs_guard_all(LaneState<CH>& st)
{
    static_for<0, 8 * CH>([&](auto jc) { st.L[decltype(jc)::value] = kGuard2; });
    st.mp = 0;
}

// S pair j (0 <= j < 8 CH) of the lane, by a select tree
template <int CH>
__device__ __forceinline__ uint32_t vs_pick(const uint32_t (&S)[CH][8], int j)
{
    uint32_t r = 0;
    static_for<0, CH>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int i = j - 8 * q;
        const uint32_t a0 = (i & 1) ? S[q][1] : S[q][0], a1 = (i & 1) ? S[q][3] : S[q][2];
        const uint32_t a2 = (i & 1) ? S[q][5] : S[q][4], a3 = (i & 1) ? S[q][7] : S[q][6];
        const uint32_t b0 = (i & 2) ? a1 : a0, b1 = (i & 2) ? a3 : a2;
        const uint32_t v = (i & 4) ? b1 : b0;
        r = (i >= 0 && i < 8) ? v : r;
    });
    return r;
}

template <int KL>
__device__ __forceinline__ uint32_t group_max(uint32_t v)
{
    return ~group_min<KL>(~v);
}

// winner key (S << 9) | D of the low (HI = false) or high u16 half S of a pair,
// in one v_mad_u32_u16 (op_sel picks the half; D <= 64 is an inline constant,
// 512 comes in a register: one scalar operand at most on this VOP3)
template <int D, bool HI>
__device__ __forceinline__ uint32_t vs_key(uint32_t pair, uint32_t m512)
{
    static_assert(D >= 0 && D <= 64, "inline constant");
    uint32_t r;
    if (HI) asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(r) : "v"(pair), "v"(m512), "i"(D));
    else asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(r) : "v"(pair), "v"(m512), "i"(D));
    return r;
}

template <int CH, int DIR, bool KEEP, bool FULL, int VKL>
__global__ __launch_bounds__(kVMaxThreads) void k_vsweep(const RigDesc* __restrict__ rigs, int nrig,
                                                        const int* __restrict__ bs, int ncol, int seg, int mode)
{
    // KEEP: also the debug sums S (all rows) and the edge rows they need.
    // FULL: D == Dp == 16 VKL CH, every chunk of every lane is real (no padding
    // chunk, no half chunk), so no per-chunk lane conditions are needed.
    constexpr bool keep_sum = KEEP;
    // deferred normalisation: within a segment the states stay raw (the step
    // does not subtract minL'); the row's output subtracts the three
    // families' pre-step minima once, and the segment-end store normalises.
    // Raw values grow by at most 255 per row, so 16 rows stay far below the
    // guard 0x3FFF.  The debug variant keeps exact states for its edge rows.
    constexpr bool DEFER = !KEEP;
    constexpr int KL = VKL, NP = 8 * CH;
    constexpr int VC = vs_cols(KL);                // owned columns per block
    extern __shared__ uint32_t xs[];               // FL slots, then FR slots
    // neighbouring column blocks on one XCD: a block's ghost columns are its
    // neighbours' owned ones, whose cost bytes and states then come from the
    // same L2
#if SISTER_VS_XCD
    const int bid = xcd_order(blockIdx.x, gridDim.x);
#else
    const int bid = blockIdx.x;
#endif
    const int ri = find_rig(bs, nrig, bid);
    const RigDesc& g = rigs[ri];
    const int Wp = g.Wp, Hp = g.Hp, D = g.D, Dp = g.Dp;
    const int t0 = seg * kVGhost;
    // a pass ends with its last crop row: the D rows beyond it reach no S (the
    // debug sums cover every row).  1920x1080 D=192: 1272 of 1464 rows, 160
    // launches of 184, 64 rigs 68.3 -> 61.7 ms
    const int tend = KEEP ? Hp : Hp - D;
    if (t0 >= tend) return;                        // the rig has no such segment: whole block
    const int nrows = min(kVGhost, tend - t0);
    (void)ncol;                                    // VC (compile-time LDS strides)
    constexpr int nt = VC + 2 * kVGhost;
    const int tid = threadIdx.x, c = tid / KL;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = (int)(blockDim.x >> 6);
    const int x = (bid - bs[ri]) * VC - kVGhost + c;
    const bool act = x >= 0 && x < Wp;
    // every column of the wave inside the image: no border guards to apply
    const bool wave_act = __builtin_amdgcn_ballot_w64(!act) == 0;
    // ghost waves step all three families too (their outward-flowing chains
    // and columns are never read by an owned column), so no wave branches
    // around a step; the busiest SIMD still carries three owned waves.  The
    // kVGhost ghost columns of a side fill kVGhost KL / 64 waves.
    constexpr int GW = kVGhost * KL / 64;
    static_assert(GW * 64 == kVGhost * KL, "ghost columns fill whole waves");
    const bool own = wave >= GW && wave < nwaves - GW;
    ChainGeo cg;
    cg.lid = tid % KL;
    cg.nq = FULL ? KL * CH : Dp >> 4;
    cg.half_tail = FULL ? false : (D & 15) != 0;
    const int boff = cg.lid * CH * 16;
    // LDS slots of a family, lane-interleaved so that a wave's accesses are
    // contiguous: pairs 2m, 2m+1 of lane (column cc, lid) in the 8-byte granule
    // m * GS + (cc + 1) * KL + lid, then minL' of column cc at word
    // NP * GS + cc + 1.  Columns -1 and nt hold a border state (guards,
    // minL' = 0), written once and never overwritten, so reads need no test.
    // GS is a multiple of 64 granules, so that the compiler pairs the slot
    // accesses (ds_read2st64 / ds_write2st64).
    constexpr int GS = vs_gs(nt, KL);
    uint32_t* XL = xs;
    uint32_t* XR = xs + NP * GS + nt + 2;
    constexpr int famL = DIR == 0 ? 2 : 3, famR = DIR == 0 ? 3 : 2;   // family ids of FL, FR
    // segment states as bytes: at the segment's last row r a chain's
    // t = L - M(r) lies in [m, m + P2] (m = its row r-1 minimum, reached at that
    // row's argmin), so t - min_d t is the normalised (L - M) in [0, 100].  A
    // column's state is those Dp bytes and the u32 min_d L - min_d t, SB bytes
    // in all; the next segment rebuilds the normalised L = M(r) + byte.
    const int SB = Dp + 16;
    uint8_t* const Sg = (uint8_t*)g.vstate;
    const uint8_t* const msum = g.msum;
    auto sg_col = [&](int par, int f) { return Sg + ((size_t)(par * 3 + f - 1) * Wp + x) * SB; };
    // FULL: loads of a column outside the image read the nearest inside one
    // (in bounds, no exec-masked loads or zero fills in the row loop); such a
    // column's states are reset to guards and nothing of it is stored
    const int xc = min(max(x, 0), Wp - 1);
    // P is this kernel's own intermediate (rows 1..H'-2).  When the plan gives
    // it volumes of its own (psum): FULL, planes per (row, chunk slot
    // q, half h) in which lane (x, lid) holds 8 u16 at byte (x KL + lid) * 16,
    // so a wave's 64 lanes move 1 KB contiguous per access (3 ms faster than
    // the cell layout at 16 rigs); otherwise cell layout (chunk qg of cell
    // (y, x) at (y W' + x) Dp + 16 qg).
    // Plans short of memory give it none (psum null, FULL only): P then
    // takes the place of the rows family's bytes of the same row and columns,
    // which the down pass reads just before it stores P.  The 2 Dp bytes of
    // column x occupy its Dp part[0] bytes and its Dp part[1] bytes, and only
    // the wave that owns column x reads or writes them; its loads of the row's
    // bytes complete before its P stores (P depends on them).  A lane's
    // 16-byte piece k = 2 q + h lies in part[0] for k < CH, in part[1] above.
    // Waves whose columns all lie inside the row keep whole-wave planes:
    // plane k of the wave's 64 / KL columns is 1 KB with wave lane l at byte
    // 16 l, planes 0..CH-1 over the wave's part[0] bytes of the row and
    // CH..2CH-1 over its part[1] bytes.  The others (the last wave of a row)
    // keep a column's pieces together: piece k of lane lid at 16 (lid CH +
    // k mod CH) in the column's bytes of its half.  (1.3 ms slower per
    // 64-rig step than volumes of its own.)  Either way the address is a
    // uniform base plus a loop-invariant lane offset.
    uint16_t* const Pd = g.psum;
    const bool rows2 = g.part[1] != nullptr;   // the rows family's directions in volumes of their own
    const bool p_own = Pd != nullptr;
    constexpr int CPW = 64 / KL;                       // columns per wave
    const int lw = tid & 63;
    const int x0w = __builtin_amdgcn_readfirstlane(x - lw / KL);   // the wave's first column
    // S, and so P and the rows family's bytes it is formed from, is read only
    // at the crop (D <= y < D + H, D <= x < D + W) outside the debug variant:
    // rows outside it, and waves whose columns all lie outside it, neither
    // load nor store them (the family steps run everywhere)
    const bool wave_crop = KEEP || (x0w + CPW > D && x0w < D + g.W);
    const bool wave_planes = FULL && x0w >= 0 && x0w + CPW <= Wp;
    const uint32_t pd_lane = p_own ? (uint32_t)(xc * KL + cg.lid) * 16u
                           : wave_planes ? (uint32_t)lw * 16u : (uint32_t)(xc * Dp + cg.lid * CH * 16);
    auto pd_at = [&](int y, int q, int h) __attribute__((always_inline)) {
        if (FULL) {
            if (p_own) {
                const uint16_t* plane = Pd + (((size_t)y * CH + q) * 2 + h) * ((size_t)Wp * KL * 8);   // uniform
                return (uint16_t*)((const char*)plane + pd_lane);
            }
            const int k = 2 * q + h, r = k >= CH ? 1 : 0, kk = k - r * CH;
            const size_t s = (size_t)y * Wp * Dp + (wave_planes ? (size_t)x0w * Dp + kk * 1024 : (size_t)kk * 16);
            return (uint16_t*)(g.part[r] + s + pd_lane);
        }
        return Pd + ((size_t)y * Wp + x) * Dp + boff + 16 * q + 8 * h;
    };

    // lane state <-> a column's segment state (bytes, then minL' at byte Dp)
    // mr: the cost bytes M(r) of the segment's last row r (the previous
    // segment's, when loading); padding pairs come back as guards
    auto st_load = [&](LaneState<CH>& st, const uint8_t* v, const uint4 (&mr)[CH]) __attribute__((always_inline)) {
        static_for<0, CH>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const int qg = cg.lid * CH + q;
            const bool ok = act && (FULL || qg < cg.nq);
            const bool tail = !FULL && cg.half_tail && qg == cg.nq - 1;
            uint32_t m[8], bt[8];
            unpack16(mr[q], m);
            unpack16(ok ? LD16(v + qg * 16) : make_uint4(0, 0, 0, 0), bt);
#pragma unroll
            for (int k = 0; k < 8; k++)
                st.L[8 * q + k] = (!ok || (tail && k >= 4)) ? kGuard2 : W2(U2(m[k]) + U2(bt[k]));
        });
        st.mp = act ? G((const uint32_t*)(v + Dp))[0] : 0u;
    };
    auto st_store = [&](const LaneState<CH>& st, uint8_t* v, const uint4 (&mr)[CH]) __attribute__((always_inline)) {
        uint32_t tq[CH][8];
        us2 tm = U2(0xFFFFFFFFu);
        static_for<0, CH>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            uint32_t m[8];
            unpack16(mr[q], m);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                tq[q][k] = W2(U2(st.L[8 * q + k]) - U2(m[k]));   // padding pairs: guard-sized
                tm = umin2(tm, U2(tq[q][k]));
            }
        });
        const uint32_t tmin = group_min<KL>(min((uint32_t)tm.x, (uint32_t)tm.y));
        const us2 n = U2(dup16(tmin));
        static_for<0, CH>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const int qg = cg.lid * CH + q;
            if (!(FULL || qg < cg.nq)) return;
            uint32_t b[8];
#pragma unroll
            for (int k = 0; k < 8; k++) b[k] = W2(U2(tq[q][k]) - n);
            ST16(v + qg * 16, pack16(b));
        });
        if (cg.lid == 0) G((uint32_t*)(v + Dp))[0] = st.mp - tmin;
    };
    auto slot_write = [&](uint32_t* X, const LaneState<CH>& st) __attribute__((always_inline)) {
        uint2* w = (uint2*)X + (c + 1) * KL + cg.lid;
        static_for<0, NP / 2>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            w[k * GS] = make_uint2(st.L[2 * k], st.L[2 * k + 1]);
        });
        if (cg.lid == 0) X[NP * GS + c + 1] = st.mp;
    };
    auto slot_read = [&](const uint32_t* X, int cc, LaneState<CH>& st) __attribute__((always_inline)) {
        const uint2* w = (const uint2*)X + (cc + 1) * KL + cg.lid;   // -1 <= cc <= nt
        static_for<0, NP / 2>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            const uint2 v = w[k * GS];
            st.L[2 * k] = v.x;
            st.L[2 * k + 1] = v.y;
        });
        st.mp = X[NP * GS + cc + 1];
    };
    auto row_of = [&](int t) { return DIR == 0 ? t : Hp - 1 - t; };
    auto load_m = [&](int t, uint4 (&b)[CH]) __attribute__((always_inline)) {
        const size_t cell = ((size_t)row_of(t) * Wp + (FULL ? xc : x)) * Dp + boff;
        static_for<0, CH>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const bool ok = act && (FULL || cg.lid * CH + q < cg.nq);
            b[q] = FULL ? LD16(msum + cell + 16 * q) : ok ? LD16(msum + cell + 16 * q) : make_uint4(0, 0, 0, 0);
        });
    };
    // exact L of a family on an edge row (debug sums only)
    auto edge_out = [&](int f, int y, const LaneState<CH>& st) __attribute__((always_inline)) {
        static_for<0, CH>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const int qg = cg.lid * CH + q;
            if (qg >= cg.nq) return;
            uint16_t* e = g.edge + ((size_t)((f - 1) * 2 + (y == 0 ? 0 : 1)) * Wp + x) * Dp + qg * 16;
            const uint4 a = make_uint4(st.L[8 * q + 0], st.L[8 * q + 1], st.L[8 * q + 2], st.L[8 * q + 3]);
            uint4 bb = make_uint4(st.L[8 * q + 4], st.L[8 * q + 5], st.L[8 * q + 6], st.L[8 * q + 7]);
            if (cg.half_tail && qg == cg.nq - 1) bb = make_uint4(0, 0, 0, 0);
            ST16(e, a);
            ST16(e + 8, bb);
        });
    };
    // S of an edge row (debug): the three vertical families' exact rows and the
    // rows family's two directions, of which the one of this line's own pass is
    // the 8-bit first-line path
    auto edge_sum = [&](int y) __attribute__((always_inline)) {
        const int e = y == 0 ? 0 : 1;
        static_for<0, CH>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const int qg = cg.lid * CH + q;
            if (qg >= cg.nq) return;
            const size_t eo = (size_t)x * Dp + qg * 16;
            const size_t ro = ((size_t)y * Wp + x) * Dp + qg * 16;
            uint32_t m[8], b8[8], bs8[8];
            unpack16(LD16(g.msum + ro), m);
            unpack16(LD16(g.part[e] + ro), b8);
            unpack16(LD16(g.part[e ^ 1] + ro), bs8);
#pragma unroll
            for (int i = 0; i < 8; i++)
                m[i] = (W2(U2(m[i]) + U2(b8[i])) & 0x00FF00FFu) + W2(U2(m[i]) + U2(bs8[i]));
#pragma unroll
            for (int h = 0; h < 2; h++) {
                uint4 acc = make_uint4(m[4 * h], m[4 * h + 1], m[4 * h + 2], m[4 * h + 3]);
#pragma unroll
                for (int fm = 0; fm < 3; fm++)
                    acc = add_u16x8(acc, LD16(g.edge + (size_t)(fm * 2 + e) * Wp * Dp + eo + 8 * h));
                ST16(g.sum + (size_t)y * Wp * Dp + eo + 8 * h, acc);
            }
        });
    };

    const bool want_sub = DIR == 1 && mode == 0 && g.subpix != nullptr;
    uint16_t* const outm = g.out[mode];
    LaneState<CH> sc, sx;
    uint4 mb[CH];
    // the border slots (columns -1 and nt) of both families
    for (int i = tid; i < 2 * (NP / 2) * KL; i += blockDim.x) {
        const int side = i / ((NP / 2) * KL), rem = i % ((NP / 2) * KL);
        const int pos = side ? nt + 1 : 0, k = rem / KL, lid = rem % KL;
        ((uint2*)XL)[k * GS + pos * KL + lid] = make_uint2(kGuard2, kGuard2);
        ((uint2*)XR)[k * GS + pos * KL + lid] = make_uint2(kGuard2, kGuard2);
        if (k == 0 && lid == 0) {
            XL[NP * GS + pos] = 0;
            XR[NP * GS + pos] = 0;
        }
    }
    if (t0 > 0) {
        const int pin = (seg - 1) & 1;
        uint4 mr[CH];
        load_m(t0 - 1, mr);
        st_load(sc, sg_col(pin, 1), mr);
        st_load(sx, sg_col(pin, famL), mr);
        slot_write(XL, sx);
        st_load(sx, sg_col(pin, famR), mr);
        slot_write(XR, sx);
    } else {
        vs_guard_all<CH>(sc);
    }
    load_m(t0, mb);
    __syncthreads();
#pragma unroll 1
    for (int i = 0; i < nrows; i++) {
        const int t = t0 + i, y = row_of(t);
        uint32_t acc[CH][8];
        uint4 mc[CH];
        static_for<0, CH>([&](auto qc) { mc[decltype(qc)::value] = mb[decltype(qc)::value]; });
        if (i + 1 < nrows) load_m(t + 1, mb);
        if (t == 0) {
            // first line of the pass: every chain takes c~ and adds nothing (sgm.cpp:103-207)
            uint32_t m[CH][8];
            static_for<0, CH>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                unpack16(mc[q], m[q]);
#pragma unroll
                for (int k = 0; k < 8; k++) m[q][k] = tilde2(m[q][k]);
            });
            lane_set<CH, KL>(sc, cg, m, act);
            lane_set<CH, KL>(sx, cg, m, act);
            slot_write(XL, sx);
            slot_write(XR, sx);
            if (DIR == 1 && keep_sum && g.sum && own && act) edge_sum(y);
            __syncthreads();
            continue;
        }
        const bool interior = y >= 1 && y <= Hp - 2;
        const bool edge_row = !interior;
        const bool pc = wave_crop && (KEEP || (y >= D && y < D + g.H));   // P and rows bytes needed
        const size_t cell = ((size_t)y * Wp + x) * Dp + boff;
        // addends of the row's output, loaded now and used after the three steps
        uint4 ob[2 * CH];
        static_for<0, 2 * CH>([&](auto kc) { ob[decltype(kc)::value] = make_uint4(0, 0, 0, 0); });
        if (own && act && interior && pc) {
            static_for<0, CH>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if (!FULL && cg.lid * CH + q >= cg.nq) return;
                if (DIR == 0) {
                    ob[q] = LD16(g.part[0] + cell + 16 * q);
                    if (KEEP || rows2) ob[CH + q] = LD16(g.part[1] + cell + 16 * q);
                } else {
                    ob[2 * q] = LD16(pd_at(y, q, 0));
                    ob[2 * q + 1] = LD16(pd_at(y, q, 1));
                }
            });
        }
        // (the steps' L - M outputs are not kept: their sum is formed after the
        // three steps from the new states, sum_f (L_f - M) = sum_f L_f - 3 M,
        // which keeps 24 registers free while the states are stepped)
        // Two barriers per row: FL slots are read (old) before the first and
        // written after it; FR slots read between the two and written after
        // the second.  The next row's FL reads follow this row's second
        // barrier, its FR reads its own first one, which orders them after
        // this row's writes.
        slot_read(XL, c - 1, sx);
        __syncthreads();
        uint32_t off;   // DEFER: sum of the three pre-step minima
        {
            off = sx.mp;
            lane_step<CH, KL, DEFER>(sx, cg, mc);
            if (!wave_act) lane_guard<CH>(sx, act);
            slot_write(XL, sx);
            if (own && edge_row && keep_sum && g.sum && act) edge_out(famL, y, sx);
        }
        __builtin_amdgcn_sched_barrier(0);
        {
            off += sc.mp;
            lane_step<CH, KL, DEFER>(sc, cg, mc);
            if (own && edge_row && keep_sum && g.sum && act) edge_out(1, y, sc);
        }
        __builtin_amdgcn_sched_barrier(0);
        slot_read(XR, c + 1, sx);
        __syncthreads();
        {
            off += sx.mp;
            lane_step<CH, KL, DEFER>(sx, cg, mc);
            if (!wave_act) lane_guard<CH>(sx, act);
            slot_write(XR, sx);
            if (own && edge_row && keep_sum && g.sum && act) edge_out(famR, y, sx);
        }
        if (!own || !act) continue;
        if (edge_row) {
            if (DIR == 1 && keep_sum && g.sum) edge_sum(y);   // y == 0
            continue;
        }
        if (!pc) continue;
        // acc = (L_cols + L_FL + L_FR) - 3 M (- the pre-step minima) from the new states of this column,
        // one chunk at a time (scheduling barriers keep the compiler from
        // hoisting every chunk's LDS reads at once)
        auto chunk_sum = [&](auto qc) __attribute__((always_inline)) {
            constexpr int q = decltype(qc)::value;
            const uint2* wl = (const uint2*)XL + (c + 1) * KL + cg.lid + 4 * q * GS;
            const uint2* wr = (const uint2*)XR + (c + 1) * KL + cg.lid + 4 * q * GS;
            uint32_t lv[8], rv[8];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint2 a = wl[k * GS], b = wr[k * GS];
                lv[2 * k] = a.x; lv[2 * k + 1] = a.y;
                rv[2 * k] = b.x; rv[2 * k + 1] = b.y;
            }
            uint32_t mq[8];
            unpack16(mc[q], mq);
            const us2 o2 = DEFER ? U2(dup16(off)) : (us2){0, 0};
            // going down: sum - 3 M - off; going up S's 8 M is folded in: sum + 5 M - off
            // (u16 arithmetic modulo 2^16; the true results are below 2^16)
#pragma unroll
            for (int k = 0; k < 8; k++) {
                if (DIR == 0) {
                    const us2 m3 = U2(mq[k]) * (us2){3, 3} + o2;
                    acc[q][k] = W2(U2(sc.L[8 * q + k]) + U2(lv[k]) + U2(rv[k]) - m3);
                } else {
                    const us2 m5 = U2(mq[k]) * (us2){5, 5} - o2;
                    acc[q][k] = W2(U2(sc.L[8 * q + k]) + U2(lv[k]) + U2(rv[k]) + m5);
                }
            }
        };
        if (DIR == 0) {
            static_for<0, CH>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if (!FULL && cg.lid * CH + q >= cg.nq) return;
                chunk_sum(qc);
                uint32_t pr[8];
                const uint4 rw = make_uint4(ob[q].x + ob[CH + q].x, ob[q].y + ob[CH + q].y, ob[q].z + ob[CH + q].z,
                                            ob[q].w + ob[CH + q].w);   // rows fwd + bwd, bytes <= 200
                unpack16(rw, pr);
#pragma unroll
                for (int k = 0; k < 8; k++) acc[q][k] = W2(U2(acc[q][k]) + U2(pr[k]));
                ST16(pd_at(y, q, 0), make_uint4(acc[q][0], acc[q][1], acc[q][2], acc[q][3]));
                ST16(pd_at(y, q, 1), make_uint4(acc[q][4], acc[q][5], acc[q][6], acc[q][7]));
                __builtin_amdgcn_sched_barrier(0);
            });
            continue;
        }
        // upward pass: S and the winner (hpp:283)
        const int oy = y - D, ox = x - D;
        const bool crop = oy >= 0 && oy < g.H && ox >= 0 && ox < g.W;
        if (!(crop || keep_sum)) continue;
        uint32_t key = 0xFFFFFFFFu;
        const uint32_t m512 = 512u;
        static_for<0, CH>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const int qg = cg.lid * CH + q;
            chunk_sum(qc);
            const uint32_t pw[8] = {ob[2 * q].x, ob[2 * q].y, ob[2 * q].z, ob[2 * q].w,
                                    ob[2 * q + 1].x, ob[2 * q + 1].y, ob[2 * q + 1].z, ob[2 * q + 1].w};
#pragma unroll
            for (int k = 0; k < 8; k++) acc[q][k] = W2(U2(pw[k]) + U2(acc[q][k]));   // S pairs
            if (!FULL && qg >= cg.nq) return;
            if (keep_sum && g.sum) {
                uint16_t* sp = g.sum + cell + 16 * q;
                ST16(sp, make_uint4(acc[q][0], acc[q][1], acc[q][2], acc[q][3]));
                ST16(sp + 8, make_uint4(acc[q][4], acc[q][5], acc[q][6], acc[q][7]));
            }
            // keys (S << 9) | (d - the lane's first d): compile-time low bits, so
            // no per-pair lane constants are kept across rows; the lane's base
            // is added after the minimum (d < 512, no carry into S).  In the
            // half-filled last chunk (D % 16 == 8) pairs 4..7 are padding.
            const bool tail = cg.half_tail && qg == cg.nq - 1;
            static_for<0, 8>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const uint32_t k0 = vs_key<16 * q + 2 * k, false>(acc[q][k], m512);
                const uint32_t k1 = vs_key<16 * q + 2 * k + 1, true>(acc[q][k], m512);
                const uint32_t kk = min(k0, k1);
                key = (k < 4 || !tail) ? min(key, kk) : key;
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        if (!crop) continue;
        if (key != 0xFFFFFFFFu) key += (uint32_t)(cg.lid * CH * 16);   // lanes of padding only keep ~0
        key = group_min<KL>(key);   // the four lanes of a column share crop
        const uint32_t best = key & 511u;
        float delta = 0.0f;
        if (want_sub) {
            // S at best - 1 and best + 1 from the lanes holding them
            auto held = [&](int d) __attribute__((always_inline)) {
                const int j = (d >> 1) - cg.lid * NP;
                const uint32_t w = vs_pick<CH>(acc, j);
                const uint32_t v = (d & 1) ? (w >> 16) : (w & 0xFFFFu);
                return (d >= 0 && j >= 0 && j < NP) ? v : 0u;
            };
            const int sm = (int)group_max<KL>(held((int)best - 1));
            const int sp = (int)group_max<KL>(held((int)best + 1));
            if (best > 0 && (int)best < D - 1) {
                const int s0 = (int)(key >> 9);
                const int den = sm - 2 * s0 + sp;
                if (den > 0) delta = (float)(sm - sp) / (2.0f * (float)den);
            }
        }
        if (cg.lid == 0) {
            const size_t o = (size_t)oy * g.W + ox;
            if (outm) G(outm)[o] = (uint16_t)min(best * 255u, 65535u);
            if (mode == 0 && g.disp) G(g.disp)[o] = (uint16_t)best;
            if (want_sub) G(g.subpix)[o] = (float)best + delta;
        }
    }
    // states at the end of the segment, for the next launch
    if (t0 + nrows < tend && own && act) {
        const int pout = seg & 1;
        uint4 mr[CH];
        load_m(t0 + nrows - 1, mr);
        st_store(sc, sg_col(pout, 1), mr);
        slot_read(XL, c, sx);
        st_store(sx, sg_col(pout, famL), mr);
        slot_read(XR, c, sx);
        st_store(sx, sg_col(pout, famR), mr);
    }
}

// ---------------------------------------------------------------------------
// host-side launchers
// ---------------------------------------------------------------------------
const char* const kKernelNames[kNumKernels] = {
    "census", "wta", "median_prep", "median_serial", "mask", "msum",
    "sgm_rows", "sgm_paths", "winner", "sgm_vsweep",
};

#define TB(id) do { if (t) t->begin(id, st); } while (0)
#define TE(id) do { if (t) t->end(id, st); } while (0)
#define TD(id, n) do { if (t) t->dispatched[id] += (n); } while (0)

void launch_census(const LaunchSet& ls, hipStream_t st, KernelTimer* t)
{
    TB(kKCensus);
    hipLaunchKernelGGL(k_census, dim3(ls.blocks[kStageCensus]), dim3(256), 0, st, ls.rigs, ls.nrig, ls.bs[kStageCensus]);
    TD(kKCensus, 1);
    TE(kKCensus);
}

static size_t g_lds_per_block = 0;   // set by kernels_setup
int g_num_cu = 0;

void launch_mask(const LaunchSet& ls, int fmask, hipStream_t st, KernelTimer* t)
{
    TB(kKMask);
    hipLaunchKernelGGL(k_mask, dim3(ls.blocks[kStageMask]), dim3(256), 0, st, ls.rigs, ls.nrig, ls.bs[kStageMask], fmask);
    TD(kKMask, 1);
    TE(kKMask);
}

int kernels_setup(int device)
{
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess) return -1;
    const int lim = v;
    if (hipDeviceGetAttribute(&g_num_cu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return -1;
    g_lds_per_block = (size_t)lim;
    if (wta_setup(lim) != 0 || median_setup(lim) != 0) {
        (void)hipGetLastError();
        return -1;
    }
#define SISTER_VS_FNS(K, F)                                                         \
    (const void*)k_vsweep<1, 0, K, F, 4>, (const void*)k_vsweep<2, 0, K, F, 4>,     \
        (const void*)k_vsweep<3, 0, K, F, 4>, (const void*)k_vsweep<1, 1, K, F, 4>, \
        (const void*)k_vsweep<2, 1, K, F, 4>, (const void*)k_vsweep<3, 1, K, F, 4>, \
        (const void*)k_vsweep<2, 0, K, F, 8>, (const void*)k_vsweep<3, 0, K, F, 8>, \
        (const void*)k_vsweep<2, 1, K, F, 8>, (const void*)k_vsweep<3, 1, K, F, 8>
    const void* vfns[30] = {SISTER_VS_FNS(false, false), SISTER_VS_FNS(false, true), SISTER_VS_FNS(true, false)};
#undef SISTER_VS_FNS
    for (const void* f : vfns)
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lim) != hipSuccess) {
            (void)hipGetLastError();
            g_lds_per_block = 0;
            return 0;
        }
    return 0;
}

// lanes per column of the fused sweep for D (0: beyond its reach, D > 384)
static int vs_kl(int D)
{
    const int k16 = (D + 15) / 16;
    return (k16 + 3) / 4 <= 3 ? 4 : (k16 + 7) / 8 <= 3 ? 8 : 0;
}
static int vs_ch(int D) { const int kl = vs_kl(D); return kl ? ((D + 15) / 16 + kl - 1) / kl : 0; }

// the fused sweep can keep P over the rows family's bytes (no volumes of its own)
bool vsweep_in_place(int D)
{
    const int kl = vs_kl(D);
    return kl && D == 16 * kl * vs_ch(D);
}

static size_t vs_lds(int D, int vcols)
{
    const int kl = vs_kl(D);
    const size_t nt = vcols + 2 * kVGhost;
    return 2 * ((size_t)8 * vs_ch(D) * vs_gs((int)nt, kl) + nt + 2) * sizeof(uint32_t);
}

int vsweep_pick_cols(long cols, int D, int choice)
{
    // choice: 0 separate families, 1 fused sweep where D allows, -1 automatic;
    // SISTER_VSWEEP=0/1 in the environment overrides the automatic choice
    static const int env = [] {
        const char* e = getenv("SISTER_VSWEEP");
        return e ? atoi(e) : -1;
    }();
    const int forced = choice >= 0 ? choice : env;
    // up to 3 chunks of 16 per lane (beyond, the state spills): 4 lanes per
    // column up to D = 192, 8 up to D = 384
    if (forced == 0 || vs_kl(D) == 0) return 0;
    const int vcols = vs_cols(vs_kl(D));
    if (vs_lds(D, vcols) > g_lds_per_block) return 0;
    // enough blocks to fill the chip (few rigs keep the per-chain families,
    // which spread a single rig over every CU)
    if (forced != 1 && (cols + vcols - 1) / vcols < std::max(g_num_cu / 2, 1)) return 0;
    return vcols;
}

int vsweep_blocks(const RigDesc& g, int vcols)
{
    return vcols > 0 ? (g.Wp + vcols - 1) / vcols : 0;
}

static int launch_vsweep(const DGroup& G, int mode, int keep_sum, hipStream_t st)
{
    const int kl = vs_kl(G.D);
    const int nt = G.vcols + 2 * kVGhost;
    const size_t lds = vs_lds(G.D, G.vcols);
    const dim3 grid(G.blocks[kGVSweep]), block(kl * nt);
    const int* bs = G.bs[kGVSweep];
    const int nseg = (G.maxHp - (keep_sum ? 0 : G.D) + kVGhost - 1) / kVGhost;
    // 1..3 chunks with 4 lanes per column, 2..3 with 8 (vsweep_pick_cols
    // gives no columns beyond)
    const int ch = vs_ch(G.D);
    const bool full = G.D == G.Dp && G.Dp == 16 * kl * ch;
    for (int dir = 0; dir < 2; dir++)
        for (int seg = 0; seg < nseg; seg++) {
#define SISTER_VS(CHV, DIRV, KLV)                                                                              \
    do {                                                                                                       \
        if (keep_sum)                                                                                          \
            hipLaunchKernelGGL((k_vsweep<CHV, DIRV, true, false, KLV>), grid, block, lds, st, G.rigs, G.nrig,  \
                               bs, G.vcols, seg, mode);                                                        \
        else if (full)                                                                                         \
            hipLaunchKernelGGL((k_vsweep<CHV, DIRV, false, true, KLV>), grid, block, lds, st, G.rigs, G.nrig,  \
                               bs, G.vcols, seg, mode);                                                        \
        else                                                                                                   \
            hipLaunchKernelGGL((k_vsweep<CHV, DIRV, false, false, KLV>), grid, block, lds, st, G.rigs, G.nrig, \
                               bs, G.vcols, seg, mode);                                                        \
    } while (0)
            if (kl == 4) {
                if (dir == 0) {
                    switch (ch) {
                    case 1: SISTER_VS(1, 0, 4); break;
                    case 2: SISTER_VS(2, 0, 4); break;
                    default: SISTER_VS(3, 0, 4); break;
                    }
                } else {
                    switch (ch) {
                    case 1: SISTER_VS(1, 1, 4); break;
                    case 2: SISTER_VS(2, 1, 4); break;
                    default: SISTER_VS(3, 1, 4); break;
                    }
                }
            } else {
                if (dir == 0) {
                    if (ch == 2) SISTER_VS(2, 0, 8);
                    else SISTER_VS(3, 0, 8);
                } else {
                    if (ch == 2) SISTER_VS(2, 1, 8);
                    else SISTER_VS(3, 1, 8);
                }
            }
#undef SISTER_VS
        }
    return 2 * nseg;
}

void launch_sgm(const LaunchSet& ls, int mode, int keep_sum, hipStream_t st, KernelTimer* t)
{
    for (int gi = 0; gi < ls.ngroups; gi++) {
        const DGroup& G = ls.groups[gi];
        const bool fused = G.vcols > 0;
        // every path and then the winner, or the rows family and then the
        // fused vertical sweep (which reads its bytes)
        const int k1 = fused ? kKRows : kKPaths, k2 = fused ? kKVSweep : kKWinner;
        TB(k1);
        launch_paths(G, keep_sum, st);
        TD(k1, 1);
        TE(k1);
        TB(k2);
        int nl = 1;
        if (fused) nl = launch_vsweep(G, mode, keep_sum, st);
        else launch_winner(G, mode, keep_sum, st);
        TD(k2, nl);
        TE(k2);
    }
}

// per-rig block counts of each stage (the host builds the block-start tables)
void stage_blocks(const RigDesc& g, int out[kNumStages])
{
    const long npx = (long)g.Wp * g.Hp;
    out[kStageCensus] = 8 * ((g.Wp + kCT - 1) / kCT) * ((g.Hp + kCT - 1) / kCT);
    out[kStageWta] = 2 * g.Hp;     // rows of frames 0 and 2
    out[kStageWtaV] = 2 * g.Wp;    // rows of frames 1 and 3
    out[kStageWtaFill] = wta_fill_blocks(g);
    out[kStageMedianPrep] = (int)(8 * ((npx / 2 + 255) / 256));
    out[kStageMask] = 4 * ((g.Wp + kMT32 - 1) / kMT32) * ((g.Hp + kMT32 - 1) / kMT32);
}

}  // namespace sister
