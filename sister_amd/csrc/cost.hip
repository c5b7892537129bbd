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
constexpr int kCostMaxDp = 256;
// tile side by pairs per lane: a 16 x 16 tile of 256 disparities takes 66 KB of
// LDS, two blocks (eight waves) per CU; 8 x 8 tiles leave the registers' 16
// waves (mixed 16-rig graph 26.2 -> 25.7 ms).  Up to 192 disparities 8 x 8 tiles
// only load twice the windows (64 rigs 1920x1080 D=192 25.8 -> 29.8 ms).
__host__ __device__ constexpr int cost_tile(int np) { return np >= 8 ? 8 : 16; }

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

__host__ __device__ inline size_t cost_row(int T, int Dp) { return (size_t)T * Dp + 64; }   // LDS bytes of a tile row

template <int NP>
__global__ __launch_bounds__(16 * cost_tile(NP)) void k_cost(const RigDesc* __restrict__ rigs, int nrig, const int* __restrict__ bs,
                                              int fuse)
{
    constexpr int T = cost_tile(NP), N = 2 * NP, NW = NP / 2, W0 = NW < 4 ? NW : 4, W1 = NW - W0;
    extern __shared__ uint32_t lds32[];
    const int bid = xcd_order(blockIdx.x, gridDim.x);   // neighbouring tiles share windows: one L2
    const int ri = find_rig(bs, nrig, bid);
    const RigDesc& g = rigs[ri];
    const int Wp = g.Wp, Hp = g.Hp, D = g.D, Dp = g.Dp;
    const int ntx = (Wp + T - 1) / T, lb = bid - bs[ri];
    const int x0 = (lb % ntx) * T, y0 = (lb / ntx) * T;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lid = lane & 15, line = 4 * wave + (lane >> 4);
    const int b0 = lid * N;
    uint8_t* const tile0 = g.msum + ((size_t)y0 * Wp + x0) * Dp;   // M of the tile's first pixel
    const bool two = (fuse & 5) && (fuse & 10);
    const int rs = (int)cost_row(T, Dp) / 4;               // LDS dwords per tile row

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
        buf_load<2>(fi, ni, off(ci + 1 + lid));
        buf_load<2>(fd, nd, off(cd - 16 * N - lid));
        buf_load<2>(ei, cci, off(ci + lid));
        buf_load<2>(ed, ccd, off(cd - lid));
        uint32_t mk = 0;
        if (on && along + lid < C) {
            const size_t q = ROWS ? (size_t)at * Wp + along + lid : (size_t)(along + lid) * Wp + at;
            // a set mask implies frame column >= D; the check keeps partners in the line
            if (ci + lid >= D && G(g.mask[FI])[q]) mk |= 1;
            if (cd - lid >= D && G(g.mask[FD])[q]) mk |= 2;
        }
        uint32_t* const cell = lds32 + (ROWS ? line * rs : line * (Dp / 4)) + b0 / 4;
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
            uint32_t* const o = cell + s * (ROWS ? Dp / 4 : rs);
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
            buf_store<W0>(w, rm, in && b0 < Dp && on ? st : kDropped);
            if constexpr (W1 > 0) buf_store<W1>(w + 4, rm, in && b0 + 16 < Dp && on ? st + 16 : kDropped);
        });
    };
    if (fuse & 5) pass(IC<1>{});
    if (two) __syncthreads();
    if (fuse & 10) pass(IC<0>{});
}

// ---------------------------------------------------------------------------
// Disparity counts past 256: two launches, k_msum_run<0> (frames 0 and 180, one
// block = a run of kRun pixels of one row) writes M, k_msum_run<1> (frames 90
// and 270, one block = a run of one column) adds to it.  Each block stages the
// partner window of its run (kRun + D - 1 codes per frame) in LDS once.  A wave
// takes one pixel at a time, lane q the disparities q + 64 j: conflict-free
// 8-byte LDS reads at immediate offsets, with no per-disparity branches, and
// stores four pixels together (quad_bytes).  The tile form above loses there:
// its windows of 24 or 32 codes per lane are loads of 64 separate lines, and a
// 16-pixel tile leaves one block per CU (4096x3000 D=384: 7.6 ms, and 9.7 ms
// with T = 16, against 5.7).
// ---------------------------------------------------------------------------
constexpr int kRun = 256;   // pixels per block
constexpr int kWinPad = 8;  // window entries before each partner window

// acc[j] += pop(cc ^ window[base - d]) for lane q's disparities d = q + 64 j.
// In the last group, lanes at or past Dp read as lane qlast = Dp - 1 - 64 (J-1)
// (their sums are not stored) and lanes at or past D are zeroed by the caller.
template <int J>
__device__ __forceinline__ void msum_add_frame(const uint64_t* L, uint64_t cc, int base, int q, int qlast,
                                               unsigned (&acc)[J])
{
    uint64_t tv[J];
    const uint64_t* w = L + base - q;       // w[-64 j] = window[base - d]
#pragma unroll
    for (int j = 0; j < J - 1; j++) tv[j] = w[-64 * j];
    tv[J - 1] = L[base - qlast - 64 * (J - 1)];
#pragma unroll
    for (int j = 0; j < J; j++) {
        const uint64_t x = cc ^ tv[j];
        acc[j] = count_add((uint32_t)(x >> 32), count_add((uint32_t)x, acc[j]));
    }
}

// Stores of M.  A wave's lane q holds one disparity of a pixel, so one pixel's
// bytes would leave as byte stores (16 or more address cycles for 64 bytes).
// Four pixels go together instead: a lane packs its disparity's four sums and
// a 4 x 4 byte transpose over each four lanes (two DPP exchanges, two byte
// permutes) leaves lane l the disparities (l & ~3) .. + 3 of pixel l & 3, one
// dword store for four pixels (4096x3000 D=384 6.2 -> 5.7 ms).
__device__ __forceinline__ uint32_t quad_bytes(const unsigned (&a)[4], int lane)
{
    const uint32_t own = a[0] | (a[1] << 8) | (a[2] << 16) | (a[3] << 24);
    const uint32_t n1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)own, 0xB1, 0xF, 0xF, true);   // lane ^ 1
    const uint32_t h = __builtin_amdgcn_perm(n1, own, (lane & 1) ? 0x03070105u : 0x06020400u);
    const uint32_t n2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h, 0x4E, 0xF, 0xF, true);     // lane ^ 2
    return __builtin_amdgcn_perm(n2, h, (lane & 2) ? 0x03020706u : 0x05040100u);
}

// SIDE = 0: frames 0/180 along row y; SIDE = 1: frames 90/270 along column x.
// J = ceil(Dp / 64) groups of 64 disparities; every rig of the launch has this Dp.
template <int SIDE, int J>
__global__ __launch_bounds__(256) void k_msum_run(const RigDesc* __restrict__ rigs, int nrig,
                                                  const int* __restrict__ bs, int fuse)
{
    extern __shared__ uint64_t lds64[];
    const int ri = find_rig(bs, nrig, blockIdx.x);
    const RigDesc& g = rigs[ri];
    const int lb = blockIdx.x - bs[ri];
    const int Wp = g.Wp, Hp = g.Hp, D = g.D, Dp = g.Dp;
    const int FA = SIDE == 0 ? 0 : 1, FB = SIDE == 0 ? 2 : 3;   // frame pair
    const bool useA = (fuse >> FA) & 1, useB = (fuse >> FB) & 1;
    // the run: SIDE 0 -> row y, x in [p0, p0+kRun); SIDE 1 -> column x, y in [p0, p0+kRun)
    const int runs = SIDE == 0 ? (Wp + kRun - 1) / kRun : (Hp + kRun - 1) / kRun;
    const int line = lb / runs, p0 = (lb % runs) * kRun;
    const int len = SIDE == 0 ? Wp : Hp;        // pixels along the line
    const int SPAN = kRun + D - 1;
    // lanes of the last group past D read up to Dp - D <= 8 entries before
    // their window; those terms are masked
    uint64_t* LA = lds64 + kWinPad;             // partners of frame FA
    uint64_t* LB = LA + SPAN + kWinPad;         // partners of frame FB
    uint64_t* LCa = LB + SPAN;                  // centers
    uint64_t* LCb = LCa + kRun;
    uint8_t* LM = (uint8_t*)(LCb + kRun);
    const int tid = threadIdx.x;
    // frame row holding the line and the frame column of run pixel i:
    //  SIDE 0: F0 row y col x;  F2 row y col W'-1-x
    //  SIDE 1: F1 row W'-1-x col H'-1-y;  F3 row W'-1-x col y
    const int frow = band_row(SIDE == 0 ? line : Wp - 1 - line, SIDE == 0 ? Hp : Wp, D);   // stored row
    const int fcols = SIDE == 0 ? Wp : Hp;
    const uint64_t* NA = g.code[2 * FA + 1] + (size_t)frow * fcols;
    const uint64_t* NB = g.code[2 * FB + 1] + (size_t)frow * fcols;
    const uint64_t* CA = g.code[2 * FA] + (size_t)frow * fcols;
    const uint64_t* CB = g.code[2 * FB] + (size_t)frow * fcols;
    // window of frame X: the frame columns [lo, lo + SPAN) covering every
    // partner col - d of the run (frame A columns run with the line
    // coordinate for F0 and F3, against it for F1 and F2)
    int loA, loB;
    if (SIDE == 0) { loA = p0 - (D - 1); loB = Wp - p0 - kRun - (D - 1); }
    else { loA = Hp - p0 - kRun - (D - 1); loB = p0 - (D - 1); }
    for (int k = tid - kWinPad; k < SPAN; k += 256) {
        const int ca = loA + k, cb = loB + k;
        LA[k] = (useA && k >= 0 && ca >= 0 && ca < fcols) ? G(NA)[ca] : 0;
        LB[k] = (useB && k >= 0 && cb >= 0 && cb < fcols) ? G(NB)[cb] : 0;
    }
    for (int i = tid; i < kRun; i += 256) {
        const int pos = p0 + i;                 // x (SIDE 0) or y (SIDE 1)
        uint64_t a = 0, b = 0;
        uint8_t mb = 0;
        if (pos < len) {
            const int colA = SIDE == 0 ? pos : Hp - 1 - pos;
            const int colB = SIDE == 0 ? Wp - 1 - pos : pos;
            const int y = SIDE == 0 ? line : pos, x = SIDE == 0 ? pos : line;
            const size_t q = (size_t)y * Wp + x;
            if (useA) a = G(CA)[colA];
            if (useB) b = G(CB)[colB];
            // a set mask implies frame column >= D; the check keeps indices in range
            if (useA && G(g.mask[FA])[q] && colA >= D) mb |= 1;
            if (useB && G(g.mask[FB])[q] && colB >= D) mb |= 2;
        }
        LCa[i] = a;
        LCb[i] = b;
        LM[i] = mb;
    }
    __syncthreads();
    // one wave per pixel, four pixels of the run at a time (the line's length is
    // a multiple of 4); lane q owns d = q + 64 j.  In the last group, lanes at
    // or past Dp read as lane Dp - 1 - 64 (J - 1) (and store nothing), lanes at
    // or past D add nothing.
    const int wave = tid >> 6, q = tid & 63;
    const int qlast = min(q, Dp - 1 - 64 * (J - 1));
    const bool store_last = (q & ~3) + 64 * (J - 1) < Dp;
    const bool live_last = q + 64 * (J - 1) < D;
    const size_t pstep = (size_t)(SIDE == 0 ? 1 : Wp) * Dp;     // to the line's next pixel
    for (int i = 4 * wave; i < kRun; i += 16) {
        const int pos = p0 + i;
        if (pos >= len) break;
        const int y = SIDE == 0 ? line : pos, x = SIDE == 0 ? pos : line;
        gptr<uint32_t> o = (gptr<uint32_t>)(G(g.msum) + ((size_t)y * Wp + x) * Dp + (q & 3) * pstep + (q & ~3));
        uint32_t old[J];
        if (SIDE == 1 && (fuse & 5)) {
#pragma unroll
            for (int j = 0; j < J; j++)
                if (j < J - 1 || store_last) old[j] = o[16 * j];
        }
        unsigned acc[J][4];
        static_for<0, 4>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            unsigned a[J];
#pragma unroll
            for (int j = 0; j < J; j++) a[j] = 0;
            const int mb = __builtin_amdgcn_readfirstlane(LM[i + k]);   // one pixel per wave
            const int pk = pos + k;
            if (mb & 1) msum_add_frame<J>(LA, LCa[i + k], (SIDE == 0 ? pk : Hp - 1 - pk) - loA, q, qlast, a);
            if (mb & 2) msum_add_frame<J>(LB, LCb[i + k], (SIDE == 0 ? Wp - 1 - pk : pk) - loB, q, qlast, a);
            a[J - 1] = live_last ? a[J - 1] : 0u;
#pragma unroll
            for (int j = 0; j < J; j++) acc[j][k] = a[j];
        });
#pragma unroll
        for (int j = 0; j < J; j++) {
            uint32_t w = quad_bytes(acc[j], q);
            if (SIDE == 1 && (fuse & 5)) w += old[j];   // bytes <= 126 each
            if (j < J - 1 || store_last) o[16 * j] = w;
        }
    }
}

int cost_blocks(const RigDesc& g)
{
    const int T = cost_tile(path_pairs(g.Dp));
    return ((g.Wp + T - 1) / T) * ((g.Hp + T - 1) / T);
}

static size_t msum_lds(int D) { return (size_t)(2 * kWinPad + 2 * (kRun + D - 1) + 2 * kRun) * 8 + kRun; }

int msum_blocks(const RigDesc& g, int side)
{
    return side == 0 ? g.Hp * ((g.Wp + kRun - 1) / kRun) : g.Wp * ((g.Hp + kRun - 1) / kRun);
}

template <int SIDE>
static void launch_msum_side(const DGroup& G, int fuse, hipStream_t st)
{
    const size_t lds = msum_lds(G.D);
    const int k = kGMsumRows + SIDE;
    const dim3 grid(G.blocks[k]), block(256);
    switch ((G.Dp + 63) / 64) {
    case 5: hipLaunchKernelGGL((k_msum_run<SIDE, 5>), grid, block, lds, st, G.rigs, G.nrig, G.bs[k], fuse); break;
    case 6: hipLaunchKernelGGL((k_msum_run<SIDE, 6>), grid, block, lds, st, G.rigs, G.nrig, G.bs[k], fuse); break;
    case 7: hipLaunchKernelGGL((k_msum_run<SIDE, 7>), grid, block, lds, st, G.rigs, G.nrig, G.bs[k], fuse); break;
    default: hipLaunchKernelGGL((k_msum_run<SIDE, 8>), grid, block, lds, st, G.rigs, G.nrig, G.bs[k], fuse); break;
    }
}

void launch_msum(const LaunchSet& ls, int fuse, hipStream_t st, KernelTimer* t)
{
    if (t) t->begin(kKMsum, st);
    for (int gi = 0; gi < ls.ngroups; gi++) {
        const DGroup& G = ls.groups[gi];
        if (G.Dp > kCostMaxDp) {
            if (fuse & 5) launch_msum_side<0>(G, fuse, st);    // frames 0/180 write M
            if (fuse & 10) launch_msum_side<1>(G, fuse, st);   // frames 90/270 add (or write when alone)
            if (t) t->dispatched[kKMsum] += ((fuse & 5) ? 1 : 0) + ((fuse & 10) ? 1 : 0);
            continue;
        }
        const int T = cost_tile(path_pairs(G.Dp));
        const size_t lds = (fuse & 5) && (fuse & 10) ? T * cost_row(T, G.Dp) : 0;
        const dim3 grid(G.blocks[kGCost]), block(16 * T);
#define SISTER_COST(NPV) \
    hipLaunchKernelGGL(k_cost<NPV>, grid, block, lds, st, G.rigs, G.nrig, G.bs[kGCost], fuse)
        switch (path_pairs(G.Dp)) {
        case 2: SISTER_COST(2); break;
        case 4: SISTER_COST(4); break;
        case 6: SISTER_COST(6); break;
        default: SISTER_COST(8); break;
        }
#undef SISTER_COST
        if (t) t->dispatched[kKMsum] += 1;
    }
    if (t) t->end(kKMsum, st);
}

}  // namespace sister
