// wta.hip -- both disparity maps of every frame row (postprocess.cpp:74-315).
//
//   L(r,c) = argmin_{d <= min(c,D-1)} pop(CC[r][c] ^ CN[r][c-d])    (postprocess.cpp:74-185)
//   R(r,p) = argmin_{d <= min(D-1,C-1-p)} pop(CC[r][p+d] ^ CN[r][p]) (postprocess.cpp:187-315)
// on raw costs recomputed from the census codes (census.cpp:81-82; pairs with
// d > c are the 255 entries and are never the minimum).  The lowest index wins
// ties: keys are 8192 pop + d, reduced with min.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "rig.h"
#include "kernels.h"
#include "lanes.h"

namespace sister {

// Rows of the deep padding bands other than a band's first row (band_row):
// the kernel computes the first row of each band and k_wta_fill copies it.
__device__ __forceinline__ bool wta_band_copy(int r, int R, int D) { return band_row(r, R, D) != r; }

// ---------------------------------------------------------------------------
// The costs of 16 pixels against 16 partners are a 16 x 16 x 64 product of
// bytes: with code bits as 64 or -64 (the centre's negated) the sum over the 64
// bits is 8192 pop - 262144, and the matrix unit's addend brings 262144 + d, so
// its result is the key itself, exact in 32 bits.
// What is left to the VALU is the two minima, half an instruction per cost each
// (three-input minimum), where popcounts took seven in all.
//
// One block per frame row, one wave per 64 pixels (four A tiles of 16), J over
// the tiles of 16 partners whose disparities reach them.  The block steps along
// the row, 64 * waves pixels at a time; each partner tile is expanded to bytes
// once, into a ring of LDS that keeps what later pixels still reach, and a lane
// reads its 16 bytes of a tile in one conflict-free load, for four products.  It
// holds column j = lane & 15 of a product and rows 4 (lane >> 4) + r:
//   left map: rows' minima stay in registers over J, the 16 columns meet once
//     per 64 pixels
//   right map: a column's rows meet in the lane, then in LDS (atomic min)
// The addend of pixels 16 b .. 16 b + 15 (tile b) lacks 16 b, the same for the
// whole tile: the left minima need no more, the right ones add it per tile.
// What bounds it: VALU, about 650 a wave's 64 pixels at D = 192 (3.4 per cost and
// lane, a third of it the minima, the rest the tiles at the band's edges, the
// expansion and the columns' meeting), against 7.2 per cost with popcounts and
// both accumulators in registers: 640x480 D=64 52 -> 43 us, 1920x1080 D=192 0.48 ->
// 0.30 ms, 4096x3000 D=384 4.63 -> 2.17 ms, 64 rigs 1920x1080 D=192 23.1 -> 14.8 ms.
// Tiles that hold pairs outside 0 <= d < D (at d = 0 and at d = D) have kFar as
// their addend there.
// ---------------------------------------------------------------------------
constexpr int kWtaWaves = 8, kLds = 160 << 10;
constexpr int kFar = 1 << 28, kBase = 64 * 64 * 64;
typedef int i32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline int wta_tmax(int D) { return (D + 14) / 16; }   // tiles t hold 16 t - 15 .. 16 t + 15
static size_t wta_lds(int C, int D, int waves)
{
    return (size_t)(4 * waves + wta_tmax(D)) * 1024 + (size_t)((C + 63) / 64) * 64 * sizeof(int);
}
// Waves per block: 4 where four such blocks fit a CU's LDS, whose loads and steps
// then overlap, else 8 (two blocks); the row in even steps.  1920x1080 D=192: 4
// waves 0.30 ms, 8 0.33, 2 0.39, 3 0.34, 5 0.39; 64 such rigs 14.8 ms, 8 waves 17.2;
// eight 1000x620 D=136 rigs 0.60, 8 waves 0.82.  4096x3000 D=384 has 8: 2.17 ms.
static int wta_waves(int C, int D)
{
    const int cap = 4 * wta_lds(C, D, kWtaWaves / 2) <= kLds ? kWtaWaves / 2 : kWtaWaves;
    const int n = (C + 63) / 64, steps = (n + cap - 1) / cap;
    return (n + steps - 1) / steps;
}

// A lane's 16 code bits as bytes: 64, and -64 where the bit is set (the sign bit
// alone tells them apart).  `word` is half a code, shifted left by 4 in the
// lanes of odd 16-groups; register k takes its bits 7 - k, 15 - k, 23 - k, 31 - k.
__device__ __forceinline__ i32x4 wta_bytes(uint32_t word)
{
    i32x4 v;
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = (int)(((word << k) & 0x80808080u) | 0x40404040u);
    return v;
}

template <bool V>
__global__ __launch_bounds__(64 * kWtaWaves) __attribute__((amdgpu_waves_per_eu(4))) void k_wta(const RigDesc* __restrict__ rigs, int nrig,
                                                        const int* __restrict__ bs)
{
    extern __shared__ i32x4 tilesB[];
    const int ri = find_rig(bs, nrig, blockIdx.x);
    const RigDesc& g = rigs[ri];
    const int lb = blockIdx.x - bs[ri];
    const int D = g.D;
    // V: frames 1 and 3 (W' rows of H' pixels), else frames 0 and 2 (H' rows of W')
    const int nrow = V ? g.Wp : g.Hp, C = V ? g.Hp : g.Wp;
    const int F = (V ? 1 : 0) + (lb >= nrow ? 2 : 0);
    const int row = lb >= nrow ? lb - nrow : lb;
    if (wta_band_copy(row, nrow, D)) return;   // copied from the band's first row
    const auto cc = G((const uint32_t*)(g.code[2 * F] + (size_t)row * C));
    const auto cn = G((const uint32_t*)(g.code[2 * F + 1] + (size_t)row * C));
    const int nw = blockDim.x >> 6, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int j = lane & 15, grp = lane >> 4, sh = 4 * (grp & 1);
    const int tmax = wta_tmax(D), tl = D / 16;   // tl: the first tile that reaches d = D (D a multiple of 8)
    const int nchunk = (C + 63) >> 6;
    int* const RP = (int*)(tilesB + 64 * (4 * nw + tmax));   // right-map minima
    for (int i = threadIdx.x; i < nchunk * 64; i += blockDim.x) RP[i] = 0x7FFFFFFF;

    i32x4 ci;   // addend of tile t = 0
    bool in0[4], inT[4], inT1[4];   // pairs of tiles 0, tmax and tmax - 1 with 0 <= d < D
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int d = 4 * grp + r - j;
        ci[r] = kBase + d;
        in0[r] = d >= 0;
        inT[r] = d + 16 * tmax < D;
        inT1[r] = d + 16 * (tmax - 1) < D;
    }
    uint16_t* const outL = g.wta[2 * F] + (size_t)row * C;

    const int S = 4 * nw + tmax;                       // tiles of LDS, a ring
    int base = 0;                                      // place of tile 4 s0
    for (int s0 = 0; s0 < nchunk; s0 += nw) {
        const int c0 = 64 * (s0 + wave), I0 = c0 >> 4;
        uint32_t ab[4], nb[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int at = 2 * min(c0 + 16 * b + j, C - 1) + (grp >> 1);
            ab[b] = cc[at] << sh;
            nb[b] = cn[at] << sh;
        }
        if (s0 > 0) {
            __syncthreads();                           // the last step's tiles are read
            base = base + 4 * nw >= S ? base + 4 * nw - S : base + 4 * nw;
        }
        auto slot = [&](int J) __attribute__((always_inline)) {   // LDS place of partner tile J
            int k = base + J - 4 * s0;
            k = k < 0 ? k + S : k;
            return 64 * (k >= S ? k - S : k) + lane;
        };
#pragma unroll
        for (int b = 0; b < 4; b++) tilesB[slot(I0 + b)] = wta_bytes(nb[b]);
        __syncthreads();
        if (c0 >= C) continue;
        i32x4 A[4], L[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            A[b] = wta_bytes(~ab[b]);
            L[b] = i32x4{0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF};
        }
        auto partner = [&](int J) __attribute__((always_inline)) { return tilesB[slot(J)]; };
        // the keys of partner tile J with pixel tiles LO .. HI: KIND 1 the tile at
        // d = 0 is LO, 2 the tiles at d = D are HI and HI - 1, 3 only HI, as HI - 1
        auto keys = [&](int J, auto lo, auto hi, auto kind, i32x4 (&k)[4]) __attribute__((always_inline)) {
            constexpr int LO = decltype(lo)::value, HI = decltype(hi)::value, KIND = decltype(kind)::value;
            const i32x4 B = partner(J);
            int at = 16 * (I0 - J);
            asm volatile("" : "+s"(at));   // or the addends of every step leave the loop, 64 registers
#pragma unroll
            for (int b = LO; b <= HI; b++) {
                i32x4 c;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    c[r] = ci[r] + at;
                    if (KIND == 1 && b == LO) c[r] = in0[r] ? c[r] : kFar;
                    if (KIND == 2 && b == HI) c[r] = inT[r] ? c[r] : kFar;
                    if ((KIND == 2 && b == HI - 1) || (KIND == 3 && b == HI)) c[r] = inT1[r] ? c[r] : kFar;
                }
                k[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[b], B, c, 0, 0, 0);
            }
        };
        // a lane's minimum of its column, with the tiles' 16 b
        auto column = [&](auto lo, auto hi, const i32x4 (&k)[4]) __attribute__((always_inline)) {
            constexpr int LO = decltype(lo)::value, HI = decltype(hi)::value;
            int x = min(min(min(k[HI][0], k[HI][1]), k[HI][2]), k[HI][3]);
#pragma unroll
            for (int b = HI - 1; b >= LO; b--) {
                x += 16;
                x = min(min(x, k[b][0]), k[b][1]);
                x = min(min(x, k[b][2]), k[b][3]);
            }
            return x + 16 * LO;
        };
        auto one = [&](int J, auto lo, auto hi, auto kind) __attribute__((always_inline)) {
            constexpr int LO = decltype(lo)::value, HI = decltype(hi)::value;
            i32x4 k[4];
            keys(J, lo, hi, kind, k);
#pragma unroll
            for (int b = LO; b <= HI; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) L[b][r] = min(L[b][r], k[b][r]);
            atomicMin(&RP[16 * J + j], column(lo, hi, k));
            __builtin_amdgcn_sched_barrier(0);   // one tile's keys at a time: registers
        };
        if (tl >= 4 && c0 + 64 <= C) {
            int J = I0 - tmax;
            static_for<0, 4>([&](auto h) __attribute__((always_inline)) {
                if (J >= 0) one(J, IC<0>{}, h, IC<2>{});
                J++;
            });
            if (tmax > tl) {
                if (J >= 0) one(J, IC<0>{}, IC<3>{}, IC<3>{});
                J++;
            }
            J = max(J, 0);
            if ((I0 - J) & 1) {
                one(J, IC<0>{}, IC<3>{}, IC<0>{});
                J++;
            }
            for (; J < I0; J += 2) {
                i32x4 k[4], q[4];
                keys(J, IC<0>{}, IC<3>{}, IC<0>{}, k);
                keys(J + 1, IC<0>{}, IC<3>{}, IC<0>{}, q);
#pragma unroll
                for (int b = 0; b < 4; b++)
#pragma unroll
                    for (int r = 0; r < 4; r++) L[b][r] = min(min(L[b][r], k[b][r]), q[b][r]);
                // lanes 0..31 keep J's column, the others J + 1's
                const auto x = __builtin_amdgcn_permlane32_swap((unsigned)column(IC<0>{}, IC<3>{}, k),
                                                                (unsigned)column(IC<0>{}, IC<3>{}, q), false, false);
                atomicMin(&RP[16 * (J + (lane >> 5)) + j], min((int)x[0], (int)x[1]));
                __builtin_amdgcn_sched_barrier(0);
            }
            static_for<0, 4>([&](auto h) __attribute__((always_inline)) {
                one(I0 + decltype(h)::value, h, IC<3>{}, IC<1>{});
            });
        } else {
            // few disparities, or the row's end inside the 64 pixels: any tile may
            // hold pairs out of range
            for (int J = max(0, I0 - tmax); J < I0 + 4 && 16 * J < C; J++) {
                const i32x4 B = partner(J);
                static_for<0, 4>([&](auto bc) __attribute__((always_inline)) {
                    constexpr int b = decltype(bc)::value;
                    const int t = I0 + b - J;
                    if (t < 0 || t > tmax) return;
                    i32x4 c;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int d = 16 * t + 4 * grp + r - j;
                        const bool in = (unsigned)d < (unsigned)D && c0 + 16 * b + 4 * grp + r < C;
                        c[r] = in ? kBase + d - 16 * b : kFar;
                    }
                    const i32x4 k = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[b], B, c, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) L[b][r] = min(L[b][r], k[r]);
                    atomicMin(&RP[16 * J + j], min(min(min(k[0], k[1]), k[2]), k[3]) + 16 * b);
                });
            }
        }
        // the 16 columns meet: each exchange halves the rows a lane still holds,
        // j's bits 0, 1, 3, 2 choosing r's bits 0, 1 and b's bits 0, 1
        auto other = [&](int v, auto ctrl) __attribute__((always_inline)) {
            return __builtin_amdgcn_update_dpp(0, v, decltype(ctrl)::value, 0xF, 0xF, true);
        };
        auto half = [&](int lo, int hi, bool up, auto ctrl) __attribute__((always_inline)) {
            return min(up ? hi : lo, other(up ? lo : hi, ctrl));
        };
        int w[4];
#pragma unroll
        for (int b = 0; b < 4; b++)
            w[b] = half(half(L[b][0], L[b][1], j & 1, IC<0xB1>{}), half(L[b][2], L[b][3], j & 1, IC<0xB1>{}), j & 2,
                        IC<0x4E>{});
        const int v0 = half(w[0], w[1], j & 8, IC<0x128>{}), v1 = half(w[2], w[3], j & 8, IC<0x128>{});   // row_ror:8
        const bool up = j & 4;
        const int mine = up ? v1 : v0, give = up ? v0 : v1;
        const int a = __builtin_amdgcn_update_dpp(0, give, 0x104, 0xF, 0x5, true);      // lanes 0-3, 8-11: from lane + 4
        const int got = __builtin_amdgcn_update_dpp(a, give, 0x114, 0xF, 0xA, false);   // the others: from lane - 4
        const int b = ((j >> 3) & 1) + 2 * ((j >> 2) & 1), best = min(mine, got) + 16 * b;
        const int c = c0 + 16 * b + 4 * grp + (j & 3);
        if (c < C) G(outL)[c] = (uint16_t)(best & 511);
    }
    __syncthreads();
    uint16_t* const outR = g.wta[2 * F + 1] + (size_t)row * C;
    for (int p = threadIdx.x; p < C; p += blockDim.x) G(outR)[p] = (uint16_t)(RP[p] & 511);
}

// The WTA maps of the deep padding bands' rows from each band's first row:
// one block per (map, band, 1024 columns), 4 columns per thread.
constexpr int kWtaFillCols = 1024;
__global__ __launch_bounds__(256) void k_wta_fill(const RigDesc* __restrict__ rigs, int nrig,
                                                  const int* __restrict__ bs)
{
    const int ri = find_rig(bs, nrig, blockIdx.x);
    const RigDesc& g = rigs[ri];
    const int lb = blockIdx.x - bs[ri];
    const int nch = (max(g.Wp, g.Hp) + kWtaFillCols - 1) / kWtaFillCols;
    const int m = lb / (2 * nch), band = (lb / nch) & 1;
    const int F = m >> 1;
    const int R = frame_rows(g, F), C = frame_cols(g, F), D = g.D;
    const int c = (lb % nch) * kWtaFillCols + 4 * (int)threadIdx.x;   // C % 4 == 0
    if (c >= C) return;
    const int lo = band ? R - D + 3 : 3, hi = band ? R - 4 : D - 4;
    uint16_t* const map = g.wta[m];
    const uint2 v = *(const uint2*)(map + (size_t)lo * C + c);
    for (int r = lo + 1; r <= hi; r++) *(uint2*)(map + (size_t)r * C + c) = v;
}

void launch_wta(const LaunchSet& ls, hipStream_t st, KernelTimer* t)
{
    if (t) t->begin(kKWta, st);
    // frames 0/2 (rows of W' pixels), then frames 1/3 (rows of H')
    const int w02 = wta_waves(ls.maxWp, ls.maxD), w13 = wta_waves(ls.maxHp, ls.maxD);
    hipLaunchKernelGGL(k_wta<false>, dim3(ls.blocks[kStageWta]), dim3(64 * w02), wta_lds(ls.maxWp, ls.maxD, w02), st,
                       ls.rigs, ls.nrig, ls.bs[kStageWta]);
    hipLaunchKernelGGL(k_wta<true>, dim3(ls.blocks[kStageWtaV]), dim3(64 * w13), wta_lds(ls.maxHp, ls.maxD, w13), st,
                       ls.rigs, ls.nrig, ls.bs[kStageWtaV]);
    // the deep padding bands' rows, copied from each band's first row
    hipLaunchKernelGGL(k_wta_fill, dim3(ls.blocks[kStageWtaFill]), dim3(256), 0, st, ls.rigs, ls.nrig,
                       ls.bs[kStageWtaFill]);
    if (t) t->dispatched[kKWta] += 3;
    if (t) t->end(kKWta, st);
}

// blocks of 1024 columns of the fill, per rig
int wta_fill_blocks(const RigDesc& g)
{
    return 8 * 2 * ((std::max(g.Wp, g.Hp) + kWtaFillCols - 1) / kWtaFillCols);
}

// the kernels take up to the chip's LDS (a row of 16376 pixels with D = 512: 129 KB)
int wta_setup(int lds_limit)
{
    for (const void* f : {(const void*)k_wta<false>, (const void*)k_wta<true>})
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_limit) != hipSuccess) return -1;
    return 0;
}

}  // namespace sister
