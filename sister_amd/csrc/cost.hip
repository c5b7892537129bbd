// cost.hip -- the mask-weighted cost sum (hpp:255-277).
//
// M(y,x,d) = sum over the used frames F with mask_F(y,x) = 1 of
// pop(CC_F[r][c] ^ CN_F[r][c-d]), (r,c) the frame pixel of (y,x).  A set mask
// implies c >= D > d, so every term is a plain popcount (<= 63) and M <= 252
// fits a byte.  A pixel's partners lie along its frame row: an image row for
// frames 0 and 180, an image column for frames 90 and 270.
#include <hip/hip_runtime.h>
#include "rig.h"
#include "kernels.h"
#include "lanes.h"

namespace sister {

// ---------------------------------------------------------------------------
// A block takes a T x T tile of pixels, a group of 16 lanes ("walker") a line
// of it: the rows for frames 0/180, then the columns for frames 90/270, whose
// sums meet the first ones in LDS, so M is written once.  A lane holds 2 NP
// consecutive disparities, as in the path kernels.  Along a line the frame
// column moves by one per pixel, and with it the window of partner codes: lane
// l keeps CN[c - 2 NP l - j], j < 2 NP, in registers, and a step drops one code
// and takes in the one its neighbour lane drops (DPP), so the only codes read
// after the window itself are those of the lane at the end, one a pixel.  Centre
// codes and masks are loaded one pixel per lane and broadcast (row_newbcast).
// What bounds it: VALU, 4 per disparity, frame and pixel group (two halves,
// xor and popcount with addend), about 20 more per step.  Against 16 x 16 tiles
// with every window in LDS, one block of 16 waves per CU and a pixel per wave:
// 640x480 D=64 48 -> 32 us, 1920x1080 D=192 528 -> 470 us, 64 rigs of it 33.0 ->
// 25.8 ms, pair modes of eight 1000x620 D=136 rigs 1.28 -> 1.20 ms.
// ---------------------------------------------------------------------------
// Pairs per lane, by the disparities a tile pass has to cover: 64, 128 or 192 (no
// lane's disparities straddle Dp), and past that as many blocks to a tile, of
// 128 each, as Dp needs.  Wider lanes spend fewer steps on the same cells, but
// their windows' registers leave fewer waves, and they lose wherever 128 serve
// (1920x1080 rigs: D=160 0.53 ms against 0.68 with 16 disparities a lane, D=256
// 0.66 / 0.88, D=264 0.97 / 1.58; D=192 is 0.48 with 12 a lane and would be
// 0.57 as two blocks).  A block per row or column run with a pixel per wave and
// its windows in LDS took 1.12 ms at D=264, 1.54 against 1.21 (1.28 with 12 a
// lane) at D=384, 2.35 against 1.95 at D=512.
constexpr int kCostTile = 16;
static int cost_pairs(int Dp) { return Dp <= 64 ? 2 : Dp > 128 && Dp <= 192 && Dp % 12 == 0 ? 6 : 4; }
static int cost_parts(int Dp) { return (Dp + 32 * cost_pairs(Dp) - 1) / (32 * cost_pairs(Dp)); }

// lane s of each 16 to all of them
template <int S> __device__ __forceinline__ uint32_t bcast16(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + S, 0xF, 0xF, true);
}
// lane l takes lane l-1's value, lane 0 lane S's `fresh`
template <int S> __device__ __forceinline__ uint32_t take_left(uint32_t v, uint32_t fresh)
{
    const int f = S == 0 ? (int)fresh : __builtin_amdgcn_update_dpp(0, (int)fresh, 0x100 + (S == 0 ? 1 : S), 0xF, 0xF, true);
    return (uint32_t)__builtin_amdgcn_update_dpp(f, (int)v, 0x111, 0xF, 0xF, false);
}
// lane l takes lane l+1's value, lane 15 lane S's `fresh`
template <int S> __device__ __forceinline__ uint32_t take_right(uint32_t v, uint32_t fresh)
{
    const int f = S == 15 ? (int)fresh : __builtin_amdgcn_update_dpp(0, (int)fresh, 0x110 + (S == 15 ? 1 : 15 - S), 0xF, 0xF, true);
    return (uint32_t)__builtin_amdgcn_update_dpp(f, (int)v, 0x101, 0xF, 0xF, false);
}
__device__ __forceinline__ unsigned count_add(uint32_t x, unsigned acc)
{
    unsigned r;   // v_bcnt adds its second operand (written out: the compiler splits the sum)
    asm("v_bcnt_u32_b32 %0, %1, %2" : "=v"(r) : "v"(x), "v"(acc));
    return r;
}

__host__ __device__ inline size_t cost_row(int T, int width) { return (size_t)T * width + 64; }   // LDS bytes of a tile row

template <int NP>
__global__ __launch_bounds__(16 * kCostTile) void k_cost(const RigDesc* __restrict__ rigs, int nrig, const int* __restrict__ bs,
                                              int fuse)
{
    constexpr int T = kCostTile, N = 2 * NP, NW = NP / 2;
    extern __shared__ uint32_t lds32[];
    const int bid = xcd_order(blockIdx.x, gridDim.x);   // neighbouring tiles share windows: one L2
    const int ri = find_rig(bs, nrig, bid);
    const RigDesc& g = rigs[ri];
    const int Wp = g.Wp, Hp = g.Hp, D = g.D, Dp = g.Dp;
    const int parts = (Dp + 32 * NP - 1) / (32 * NP), PW = parts > 1 ? 32 * NP : Dp;   // a part's disparities
    const int ntx = (Wp + T - 1) / T, lb = bid - bs[ri], tile = lb / parts;
    const int x0 = (tile % ntx) * T, y0 = (tile / ntx) * T;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lid = lane & 15, line = 4 * wave + (lane >> 4);
    const int l0 = lid * N, c0 = (lb - tile * parts) * PW, b0 = c0 + l0;   // the lane's first disparity
    uint8_t* const tile0 = g.msum + ((size_t)y0 * Wp + x0) * Dp;   // M of the tile's first pixel
    const bool two = (fuse & 5) && (fuse & 10);
    const int rs = (int)cost_row(T, PW) / 4;               // LDS dwords per tile row

    // ROWS: the tile's rows (frames 0 and 2), else its columns (3 and 1); the
    // first frame's column grows along the line, the second's falls
    auto pass = [&](auto rowsc) __attribute__((always_inline)) {
        constexpr bool ROWS = decltype(rowsc)::value != 0;
        constexpr int FI = ROWS ? 0 : 3, FD = ROWS ? 2 : 1;
        const int at = (ROWS ? y0 : x0) + line;          // the line: image row or column
        const int along = ROWS ? x0 : y0;                // its first pixel
        const int nline = ROWS ? Hp : Wp, C = ROWS ? Wp : Hp;
        const bool on = at < nline;
        // stored rows: the line's, counted from the tile's first (band_row never falls)
        const int row0 = band_row(ROWS ? y0 : Wp - 1 - min(x0 + T - 1, Wp - 1), nline, D);
        const int frow = band_row(ROWS ? min(at, Hp - 1) : Wp - 1 - min(at, Wp - 1), nline, D) - row0;
        const size_t left = (size_t)(nline - row0) * C * 8;
        const uint32_t plane = left < 0x7FFFFFFF ? (uint32_t)left : 0x7FFFFFFFu;
        const int ci = along, cd = C - 1 - along;        // frame columns of the first pixel
        // codes at frame column c of the line (outside the plane: 0; a set mask
        // never reaches outside the line)
        auto off = [&](int c) __attribute__((always_inline)) { return (uint32_t)(frow * C + c) * 8u; };
        auto rows = [&](const uint64_t* p) __attribute__((always_inline)) { return buf((uint8_t*)(p + (size_t)row0 * C), plane); };
        const auto ni = rows(g.code[2 * FI + 1]), nd = rows(g.code[2 * FD + 1]);
        const auto cci = rows(g.code[2 * FI]), ccd = rows(g.code[2 * FD]);
        uint32_t wi[2 * N], wd[2 * N];                   // [2 j]: low, [2 j + 1]: high half of window entry j
        static_for<0, NP>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;       // entries N - 1 - 2 i and N - 2 - 2 i, ascending columns
            uint32_t v[4];
            buf_load<4>(v, ni, off(ci - b0 - (N - 1) + 2 * i));
            wi[2 * (N - 1 - 2 * i)] = v[0]; wi[2 * (N - 1 - 2 * i) + 1] = v[1];
            wi[2 * (N - 2 - 2 * i)] = v[2]; wi[2 * (N - 2 - 2 * i) + 1] = v[3];
            buf_load<4>(v, nd, off(cd - b0 - (N - 1) + 2 * i));
            wd[2 * (N - 1 - 2 * i)] = v[0]; wd[2 * (N - 1 - 2 * i) + 1] = v[1];
            wd[2 * (N - 2 - 2 * i)] = v[2]; wd[2 * (N - 2 - 2 * i) + 1] = v[3];
        });
        uint32_t fi[2], fd[2], ei[2], ed[2];             // the end lane's codes to come; centres
        buf_load<2>(fi, ni, off(ci - c0 + 1 + lid));
        buf_load<2>(fd, nd, off(cd - c0 - 16 * N - lid));
        buf_load<2>(ei, cci, off(ci + lid));
        buf_load<2>(ed, ccd, off(cd - lid));
        uint32_t mk = 0;
        if (on && along + lid < C) {
            const size_t q = ROWS ? (size_t)at * Wp + along + lid : (size_t)(along + lid) * Wp + at;
            // a set mask implies frame column >= D; the check keeps partners in the line
            if (ci + lid >= D && G(g.mask[FI])[q]) mk |= 1;
            if (cd - lid >= D && G(g.mask[FD])[q]) mk |= 2;
        }
        uint32_t* const cell = lds32 + (ROWS ? line * rs : line * (PW / 4)) + l0 / 4;
        const uint32_t so = on ? (uint32_t)((ROWS ? (long)line * Wp : line) * Dp) + b0 : kDropped;
        static_for<0, T>([&](auto sc) __attribute__((always_inline)) {
            constexpr int s = decltype(sc)::value;
            const uint32_t m = bcast16<s>(mk);
            const uint32_t i0 = bcast16<s>(ei[0]), i1 = bcast16<s>(ei[1]), d0 = bcast16<s>(ed[0]), d1 = bcast16<s>(ed[1]);
            unsigned cnt[N];
#pragma unroll
            for (int j = 0; j < N; j++) cnt[j] = 0;
            // window entry j sits in slot (j - s) mod N of the growing frame,
            // (j + s) mod N of the falling one
            if (m & 1) {
                static_for<0, N>([&](auto jc) __attribute__((always_inline)) {
                    constexpr int j = decltype(jc)::value, p = (j - s % N + N) % N;
                    cnt[j] = count_add(i1 ^ wi[2 * p + 1], count_add(i0 ^ wi[2 * p], cnt[j]));
                });
            }
            if (m & 2) {
                static_for<0, N>([&](auto jc) __attribute__((always_inline)) {
                    constexpr int j = decltype(jc)::value, p = (j + s) % N;
                    cnt[j] = count_add(d1 ^ wd[2 * p + 1], count_add(d0 ^ wd[2 * p], cnt[j]));
                });
            }
            uint32_t w[NW];
#pragma unroll
            for (int k = 0; k < NW; k++) {
                w[k] = cnt[4 * k] | (cnt[4 * k + 1] << 8) | (cnt[4 * k + 2] << 16) | (cnt[4 * k + 3] << 24);
                w[k] = b0 + 4 * k < D ? w[k] : 0u;       // D is a multiple of 8
            }
            if constexpr (s + 1 < T) {
                constexpr int pi = (N - 1 - s % N + N) % N, pd = s % N;   // the entries dropped
                wi[2 * pi] = take_left<s>(wi[2 * pi], fi[0]);
                wi[2 * pi + 1] = take_left<s>(wi[2 * pi + 1], fi[1]);
                wd[2 * pd] = take_right<s>(wd[2 * pd], fd[0]);
                wd[2 * pd + 1] = take_right<s>(wd[2 * pd + 1], fd[1]);
            }
            uint32_t* const o = cell + s * (ROWS ? PW / 4 : rs);
            if (ROWS && two) {
#pragma unroll
                for (int k = 0; k < NW; k++)
                    if (b0 + 4 * k < Dp) o[k] = w[k];
                return;
            }
            if (two) {
#pragma unroll
                for (int k = 0; k < NW; k++)
                    if (b0 + 4 * k < Dp) w[k] += o[k];   // bytes: at most 252
            }
            const bool in = along + s < C;
            const uint32_t st = so + (uint32_t)((ROWS ? s : (long)s * Wp) * Dp);
            const auto rm = buf(tile0);
            buf_store<NW>(w, rm, in && b0 < Dp && on ? st : kDropped);
        });
    };
    if (fuse & 5) pass(IC<1>{});
    if (two) __syncthreads();
    if (fuse & 10) pass(IC<0>{});
}

int cost_blocks(const RigDesc& g)
{
    const int T = kCostTile;
    return cost_parts(g.Dp) * ((g.Wp + T - 1) / T) * ((g.Hp + T - 1) / T);
}

void launch_msum(const LaunchSet& ls, int fuse, hipStream_t st, KernelTimer* t)
{
    if (t) t->begin(kKMsum, st);
    for (int gi = 0; gi < ls.ngroups; gi++) {
        const DGroup& G = ls.groups[gi];
        const int np = cost_pairs(G.Dp), T = kCostTile;
        const size_t lds = (fuse & 5) && (fuse & 10) ? T * cost_row(T, cost_parts(G.Dp) > 1 ? 32 * np : G.Dp) : 0;
        const dim3 grid(G.blocks[kGCost]), block(16 * T);
#define SISTER_COST(NPV) \
    hipLaunchKernelGGL(k_cost<NPV>, grid, block, lds, st, G.rigs, G.nrig, G.bs[kGCost], fuse)
        switch (np) {
        case 2: SISTER_COST(2); break;
        case 4: SISTER_COST(4); break;
        default: SISTER_COST(6); break;
        }
#undef SISTER_COST
        if (t) t->dispatched[kKMsum] += 1;
    }
    if (t) t->end(kKMsum, st);
}

}  // namespace sister
