// k_xdrop_wave.hip -- gapped X-drop seed extension with one 16-lane row of a
// wave per work item (four items per wave), for bands wider than the other
// kernels hold.  Same algorithm, step for step, as k_xdrop_pl and the oracle's
// or_xdrop_one (SeqAn's one-direction GappedXDrop as called at
// src/align/SeqanXdropAligner.cpp:281-283), so extents and evaluated-cell
// counts are bit-identical.
//
// The cells of one anti-diagonal depend only on the two before it, so all of
// them are evaluated at once.  A lane holds a block of BL neighbouring columns,
// two 16-bit values a register, and the 16 lanes a window of W = 16 BL
// columns; column c sits at place c mod W, and a lane whose block the band has
// left behind takes the block W columns further.  So nothing is moved when the
// band moves, and column c - 1 is a register shift, or one DPP rotation at a
// block's first column.
//   - Values are kept as v + X - base in int16, the undefined cell as -32768: a
//     cell kept on anti-diagonal d is at least best - X, so a defined value is
//     not negative, "undefined" is its sign, saturating sums of an undefined
//     cell stay undefined, and the limit in these units is best - base.  base
//     is 0 until the best score nears the type's range, and then moves up to
//     it: the values of the last three anti-diagonals lie no more than 93 below
//     the limit (31 a step, the largest matrix score).  Long homologs need it:
//     300 pairs of 8,000 nearly equal residues were handed on from window to
//     window to the last kernel below, 181 ms, now 8.5.
//     An item whose band nears the window (W - 3 BL columns: 104, 208 and
//     416), or for whose X the type has no room, is handed on through
//     the overflow list: from the 128-column to the 256-column and to the
//     512-column kernel, then to the rings in global memory, where a lane has
//     the item alone: 10,000 pairs of homologs of 800 residues took 56 ms
//     there for two items of 40,000, and 300 of 2,500 residues 139 ms for
//     eight of 1,200.
//   - Outside the range [minCol, maxCol) of an anti-diagonal the recurrence
//     gives undefined cells by itself: the columns that the update of minCol
//     passes are undefined on both anti-diagonals it reads, and so are those
//     from two past the last defined one.  Only where minCol or maxCol was set
//     by the ends of the segments, and in the first steps, where column 0 and
//     row 0 hold gap scores, are the columns masked.
//   - A lane's database residues move up one column a step (a byte shift); the
//     one that enters comes from a ring in LDS, and so do the query residues
//     of a new block.  The rings are filled every kSteps steps with what was
//     loaded kSteps steps before.  A lane takes its new block at least BL + 2
//     steps before the band gets there, when its residues are in place.
// Bound by instructions, about 190 per step of four items; a column per lane
// in 32-bit values (up to eight chunks of 16 columns) took over 450.  60,001
// pairs, log-normal lengths to 3,000, X = 49, gap -2: the two windows 9.2 + 4.2
// -> 4.7 + 1.3 ms.
#include <limits.h>

#include "pa_internal.h"

namespace pa {
namespace {

constexpr uint32_t kClaim = 4;        // items claimed per queue atomic
constexpr int kSteps = 16;            // anti-diagonals between ring refills
// largest best - base + X; base follows the best score at this distance from
// what the steps to the next refill may add, and needs room to do so
constexpr int kTop = 32000, kStepTop = kTop - 31 * kSteps, kBelow = 128;
// registers per lane and anti-diagonal: windows of 128, 256 and 512 columns
constexpr int kBandRegs[3] = {4, 8, 16};
constexpr uint32_t kUndef2 = 0x80008000u;
constexpr int kUndef = -32768;

struct WaveArgs {
    const XdTask *tasks;
    const uint32_t *list;   // work items (k = 2 * task + dir), NULL = 0..count
    const uint32_t *count;
    uint32_t *queue;
    const int8_t *mat;
    int gap, X, seed_len;
    XdOut *out;
    uint32_t *ovf_list, *ovf_count;
};

typedef short s2v __attribute__((ext_vector_type(2)));
typedef unsigned short u2v __attribute__((ext_vector_type(2)));
// a register's two values stored over int16 places
typedef uint32_t __attribute__((may_alias)) u32a;

__device__ inline s2v sv(uint32_t x) { return __builtin_bit_cast(s2v, x); }
__device__ inline uint32_t uv(s2v x) { return __builtin_bit_cast(uint32_t, x); }
__device__ inline uint32_t pk_add(uint32_t a, uint32_t b)
{
    return uv(__builtin_elementwise_add_sat(sv(a), sv(b)));
}
__device__ inline uint32_t pk_sub(uint32_t a, uint32_t b)
{
    return uv(__builtin_elementwise_sub_sat(sv(a), sv(b)));
}
__device__ inline uint32_t pk_max(uint32_t a, uint32_t b)
{
    return uv(__builtin_elementwise_max(sv(a), sv(b)));
}
__device__ inline uint32_t pk_minu(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(
        uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u2v, a),
                                            __builtin_bit_cast(u2v, b)));
}
// all ones where negative
__device__ inline uint32_t pk_neg(uint32_t a) { return uv(sv(a) >> (short)15); }
__device__ inline uint32_t splat(int x)
{
    return __builtin_amdgcn_perm((uint32_t)x, (uint32_t)x, 0x01000100u);
}

// lane j of each 16-lane row reads lane j - K (mod 16) of its row (every
// lane has a source, so no "old" operand: the compiler can fold the move
// into the instruction that uses it)
template <int K> __device__ inline int32_t ror(int32_t v)
{
    return __builtin_amdgcn_mov_dpp(v, 0x120 + K, 0xf, 0xf, true);
}

__device__ inline int row_max(int v)
{
    v = max(v, ror<1>(v));
    v = max(v, ror<2>(v));
    v = max(v, ror<4>(v));
    v = max(v, ror<8>(v));
    return v;
}

__device__ inline int row_min(int v)
{
    v = min(v, ror<1>(v));
    v = min(v, ror<2>(v));
    v = min(v, ror<4>(v));
    v = min(v, ror<8>(v));
    return v;
}

// kEmpty: nothing to extend; kOut: handed on
enum : int { kNeed = 0, kRun = 1, kDone = 2, kEmpty = 3, kOut = 4 };

// The longest items are chains of thousands of steps, and the caller waits for
// them: these waves issue ahead of those of another batch's DP that they share
// a SIMD with.
__device__ inline void band_first_issue()
{
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_s_setprio(3);
#endif
}

template <int NR>
__global__ __launch_bounds__(64) void k_xdrop_band(WaveArgs a)
{
    band_first_issue();
    constexpr int BL = 2 * NR;         // columns per lane
    constexpr int W = 16 * BL;         // columns of the window
    constexpr int QR = 4 * W, DR = 2 * W;   // residues per ring
    constexpr int WL = W - 3 * BL;     // widest written range
    __shared__ int8_t mat[32 * 32];
    __shared__ uint8_t rings[4 * (QR + DR)];
    __shared__ int16_t dump[4 * 3 * W];   // three anti-diagonals at an end
    const int lane = threadIdx.x, j = lane & 15, row = lane >> 4;
    for (int i = lane; i < 32 * 32; i += 64)
        mat[i] = a.mat[i];
    // (residue codes are below 32: a slot not yet stored must be, too)
    for (int i = lane; i < 4 * (QR + DR); i += 64)
        rings[i] = 0;
    __syncthreads();
    const uint32_t n = *a.count;
    if (n == 0)
        return;
    const int gap = max(a.gap, -32000);
    const uint32_t GAP = splat(gap);
    uint8_t *const qring = rings + row * (QR + DR);
    uint8_t *const dring = qring + QR;
    int16_t *const dmp = dump + row * 3 * W;

    // row-uniform state of the current item
    int state = kNeed;
    uint32_t k = 0;
    int X = 0, best_max = 0, base = 0;
    int cols = 0, rows = 0, d = 0, minCol = 0, maxCol = 0, best = 0;
    int off1 = 0, off2 = 0, off3 = 0, l1 = 0, l2 = 0, l3 = 0;
    bool right = false, invalid = false;
    uint32_t nc = 0;
    int64_t dgap = 0;       // d * gap, while a border cell is kept
    bool edge = false;      // one may be
    int masked = 0;         // steps that still need masks (INT_MAX: all)
    const uint8_t PA_GLOBAL *qb = nullptr, *db = nullptr;
    int qstep = 1;          // column c at qb[qstep * c], row r at db[qstep * r]
    // rings: columns below qfill and rows below dfill are stored, the next W
    // columns (BL a lane) and 16 rows are on their way
    int qfill = 0, dfill = 0, dpre = 0;
    uint64_t qpre[NR / 4];
    // this lane's block: columns c0 + 2 r + h in half h of register r, values
    // of anti-diagonals d (P), d-1 (O), d-2 (Z) and column - 1 of d-1 (LD)
    int c0 = 0;
    uint32_t P[NR], O[NR], Z[NR], LD[NR];
    uint32_t Q[NR];         // query residues * 32
    uint32_t R[NR / 2];     // database residues of anti-diagonal d + 1
    int S0[NR], S1[NR];     // and its scores (joined where they are used, so
                            // that no step waits for its own lookups)
    int nb = 0;             // residue that enters for d + 2
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        P[r] = O[r] = Z[r] = LD[r] = kUndef2;
        Q[r] = 0;
        S0[r] = S1[r] = 0;
        R[r / 2] = 0;
        qpre[r / 4] = 0;
    }
    uint32_t cbase = 0, cend = 0;   // claimed, not yet handed out

    // residues of columns c .. c + 7 (0 past the end: up to seven bytes beside
    // the segment are read, which the store's margins hold)
    auto q_load8 = [&](int c) -> uint64_t {
        typedef uint64_t __attribute__((aligned(1))) u64u;
        if (c >= cols)
            return 0;
        if (qstep > 0)
            return *(const u64u PA_GLOBAL *)(qb + c) & 0x1f1f1f1f1f1f1f1full;
        return __builtin_bswap64(*(const u64u PA_GLOBAL *)(qb - c - 7)) &
               0x1f1f1f1f1f1f1f1full;
    };
    auto d_load = [&](int r) {
        return r >= 1 && r < rows ? (int)db[qstep > 0 ? r : -r] : 0;
    };
    // query residues of the block as pairs, times 32
    auto set_q = [&](const uint64_t *w) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const uint32_t x = (uint32_t)(w[r / 4] >> (16 * (r % 4)));
            Q[r] = ((x & 0xffu) | ((x & 0xff00u) << 8)) << 5;
        }
    };
    auto scores = [&]() {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            // bytes 2r, 2r+1 as two halves
            const uint32_t sel = r % 2 ? 0x0c030c02u : 0x0c010c00u;
            const uint32_t ad =
                Q[r] | __builtin_amdgcn_perm(0u, R[r / 2], sel);
            S0[r] = mat[ad & 0xffffu];
            S1[r] = mat[ad >> 16];
        }
    };

    for (;;) {
        // ---- hand out items to rows that need one (wave-uniform)
        uint64_t need = __ballot(state == kNeed && j == 0);
        while (need) {
            if (cbase >= cend) {
                uint32_t b = atomicAdd(a.queue, lane == 0 ? kClaim : 0u);
                b = __builtin_amdgcn_readfirstlane(b);
                cbase = b;
                cend = b + kClaim;
            }
            const uint32_t cnt = (uint32_t)__popcll(need);
            const uint32_t take = min(cnt, cend - cbase);
            const uint32_t rank =
                (uint32_t)__popcll(need & ((1ull << (16 * row)) - 1ull));
            const bool mine =
                ((need >> (16 * row)) & 1ull) != 0 && rank < take;
            if (mine) {
                const uint32_t idx = cbase + rank;
                if (idx >= n) {
                    state = kDone;
                    cols = rows = 0;   // nothing more to load
                } else {
                    k = a.list ? glb(a.list)[idx] : idx;
                    const XdTask T = a.tasks[k >> 1];
                    const uint8_t PA_GLOBAL *h = glb_addr<const uint8_t>(T.h_off);
                    const uint8_t PA_GLOBAL *v = glb_addr<const uint8_t>(T.v_off);
                    const int beg_h = (int)T.beg_h, beg_v = (int)T.beg_v;
                    right = (k & 1) != 0;
                    if (!right) {   // query V[0, beg_v), database H[0, beg_h)
                        cols = beg_v + 1;
                        rows = beg_h + 1;
                        qb = v + beg_v;
                        db = h + beg_h;
                        qstep = -1;
                    } else {        // suffixes after the seed
                        cols = (int)T.nv - beg_v - a.seed_len + 1;
                        rows = (int)T.nh - beg_h - a.seed_len + 1;
                        qb = v + beg_v + a.seed_len - 1;
                        db = h + beg_h + a.seed_len - 1;
                        qstep = 1;
                    }
                    // the rings load up to cols and rows whatever the item's
                    // state, and the seed of an invalid task may lie anywhere
                    invalid = (T.pad & kXdInvalid) != 0;
                    if (invalid)
                        cols = rows = 0;
                    // No cell lies more below the best score than the gaps of
                    // its anti-diagonal and 31 (the largest matrix score) per
                    // row or column: a larger X drops nothing either.
                    X = (int)min((int64_t)a.X,
                                 31ll * min(cols, rows) + 1 -
                                     (int64_t)(cols + rows) * gap);
                    best_max = a.gap < -32000 ? -1 : kTop - X;
                    base = 0;
                    d = 1;
                    minCol = 1;
                    maxCol = 2;
                    off1 = off2 = off3 = 0;
                    l1 = 0;
                    l2 = 1;
                    l3 = 2;
                    best = 0;
                    nc = 0;
                    dgap = gap;
                    edge = -gap <= X;
                    masked = 3;
                    state = kRun;
                    if (rows <= 1 || cols <= 1) {
                        state = kEmpty;
                    } else {
                        // anti-diagonal 0: column 0 = 0; anti-diagonal 1:
                        // columns 0 and 1 = gap (undefined when -gap > X)
                        const uint32_t z = (uint32_t)X;
                        const uint32_t g1 = -gap > X ? kUndef2 : splat(gap + X);
#pragma unroll
                        for (int r = 0; r < NR; ++r)
                            P[r] = O[r] = LD[r] = Z[r] = kUndef2;
                        if (j == 0) {
                            O[0] = 0x80000000u | z;
                            P[0] = g1;
                            LD[0] = (z << 16) | 0x8000u;
                        }
                        c0 = j * BL;
                        uint64_t w[NR / 4];
#pragma unroll
                        for (int q = 0; q < NR / 4; ++q) {
                            w[q] = q_load8(c0 + 8 * q);
                            qpre[q] = q_load8(W + c0 + 8 * q);
                        }
                        set_q(w);
                        qfill = W;
                        dring[1 + j] = (uint8_t)d_load(1 + j);
                        dring[17 + j] = (uint8_t)d_load(17 + j);
                        dfill = 33;
                        dpre = d_load(33 + j);
                        // anti-diagonal 2: column 1, row 1 only
#pragma unroll
                        for (int q = 0; q < NR / 2; ++q)
                            R[q] = 0;
                        if (j == 0)
                            R[0] = (uint32_t)d_load(2) |
                                   ((uint32_t)d_load(1) << 8);
                        nb = j == 0 ? d_load(3) : 0;
                        scores();
                    }
                }
            }
            cbase += take;
            for (uint32_t t = 0; t < take; ++t)
                need &= need - 1;   // the rows served
        }
        if (!__ballot(state != kDone))
            break;

        // ---- rings for the next kSteps anti-diagonals.  Blocks are taken up
        // to W - 1 columns above minCol - 1, which passes maxCol by no more
        // than kSteps; rows enter at most BL columns below minCol, two
        // anti-diagonals ahead.
        if (qfill < minCol + kSteps + WL + W) {
#pragma unroll
            for (int q = 0; q < NR / 4; ++q) {
                *(uint64_t *)(qring + ((qfill + j * BL + 8 * q) & (QR - 1))) =
                    qpre[q];
                qpre[q] = q_load8(qfill + W + j * BL + 8 * q);
            }
            qfill += W;
        }
        if (dfill < d - minCol + kSteps + BL + 4) {
            dring[(dfill + j) & (DR - 1)] = (uint8_t)dpre;
            dfill += 16;
            dpre = d_load(dfill + j);
        }
        // ---- the base of the values, where they near the type's range
        const bool rise = state == kRun && best_max > 0 &&
                          best - base > max(kStepTop - X, 2 * kBelow);
        if (__ballot(rise)) {
            const int up = rise ? best - base - kBelow : 0;
            const uint32_t UP = splat(up);
            base += up;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                P[r] = pk_sub(P[r], UP);
                O[r] = pk_sub(O[r], UP);
                Z[r] = pk_sub(Z[r], UP);
                LD[r] = pk_sub(LD[r], UP);
            }
        }
        // ---- kSteps anti-diagonals, or until a row's item ends.  Rows
        // without an item compute on (their results go nowhere).
        bool fin = state != kDone && !(state == kRun && minCol < maxCol);
        uint64_t any = __ballot(fin);
        for (int st = 0; st < kSteps && !any; ++st) {
            const bool ovf =
                maxCol - minCol + 2 > WL || best - base > best_max;
            const int noff3 = minCol - 1;
            const int nl3 = maxCol + 1 - noff3;
            ++d;
            // column - 1
            uint32_t L[NR], V[NR], m[NR];
            L[0] = __builtin_amdgcn_alignbit(P[0], (uint32_t)ror<1>((int)P[NR - 1]), 16);
#pragma unroll
            for (int r = 1; r < NR; ++r)
                L[r] = __builtin_amdgcn_alignbit(P[r], P[r - 1], 16);
            const uint32_t BEST = splat(best - base);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const uint32_t sc = __builtin_amdgcn_perm(
                    (uint32_t)S1[r], (uint32_t)S0[r], 0x05040100u);
                V[r] = pk_max(pk_add(pk_max(P[r], L[r]), GAP),
                              pk_add(LD[r], sc));
                m[r] = pk_neg(pk_sub(V[r], BEST));
            }
            if (__ballot(masked > 0 && state == kRun)) {
                const uint32_t lo = splat(c0 - minCol);
                const uint32_t w1 = splat(maxCol - minCol - 1);
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const uint32_t x =
                        pk_add(lo, (uint32_t)(2 * r) | ((2 * r + 1) << 16));
                    m[r] |= pk_neg(x) | pk_neg(pk_sub(w1, x));
                }
            }
#pragma unroll
            for (int r = 0; r < NR; ++r)
                V[r] = (m[r] & kUndef2) | (V[r] & ~m[r]);
            uint32_t ab = V[0];
#pragma unroll
            for (int r = 1; r < NR; ++r)
                ab = pk_max(ab, V[r]);
            // cells of column 0 and row 0, while the gap to them is kept: d *
            // gap falls and the limit does not, so once it is not, never again
            if (__ballot(edge && state == kRun)) {
                dgap += gap;
                edge = edge && dgap > (int64_t)best - X;
                if (edge) {
                    const uint32_t e =
                        (uint32_t)((int)dgap + X - base) & 0xffffu;
                    masked = 3;
                    if (c0 == 0 && noff3 == 0)
                        V[0] = (V[0] & 0xffff0000u) | e;
                    const int x = d - c0;
                    if (d == maxCol && x >= 0 && x < BL) {
#pragma unroll
                        for (int r = 0; r < NR; ++r) {
                            if (x == 2 * r)
                                V[r] = (V[r] & 0xffff0000u) | e;
                            if (x == 2 * r + 1)
                                V[r] = (V[r] & 0xffffu) | (e << 16);
                        }
                    }
                }
            }
            // minCol: the first column defined here or, at column - 1, on the
            // anti-diagonal before; maxCol: two past the last column below it
            // that is defined on either
            uint32_t f = ~0u, g = ~0u;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const uint32_t at = (uint32_t)(2 * r) | ((2 * r + 1) << 16);
                f = pk_minu(f, pk_neg(pk_max(V[r], L[r])) | at);
                g = pk_max(g, pk_neg(pk_max(V[r], P[r])) | at);
            }
            const int fl = min((int)(f & 0xffffu), (int)(f >> 16));
            const int gl = max((int)(int16_t)g, (int)g >> 16);
            const int lo = row_min(c0 + fl);
            const int hi = row_max(gl < 0 ? -1 : c0 + gl);
            const int adb =
                row_max(max((int)(int16_t)ab, (int)ab >> 16)) - X + base;
            nc += (uint32_t)(maxCol - minCol);
            best = max(best, adb);
            // scores of the next anti-diagonal
#pragma unroll
            for (int q = NR / 2 - 1; q > 0; --q)
                R[q] = __builtin_amdgcn_alignbit(R[q], R[q - 1], 24);
            R[0] = (R[0] << 8) | (uint32_t)nb;
            nb = dring[(d + 2 - c0) & (DR - 1)];
            scores();
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                Z[r] = O[r];
                O[r] = P[r];
                P[r] = V[r];
                LD[r] = L[r];
            }
            off1 = off2;
            off2 = off3;
            off3 = noff3;
            l1 = l2;
            l2 = l3;
            l3 = nl3;
            const int nmin = min(max(lo, minCol), maxCol + 1);
            const int nmax = max(min(hi, maxCol - 1) + 1, noff3) + 1;
            if (masked < INT_MAX)
                masked = nmin < d + 2 - rows || nmax > cols
                             ? INT_MAX
                             : max(masked - 1, 0);
            minCol = max(nmin, d + 2 - rows);
            maxCol = min(nmax, cols);
            const bool up = state == kRun && c0 + BL < minCol;
            if (__ballot(up)) {
                if (up) {
                    c0 += W;
                    uint64_t w[NR / 4];
#pragma unroll
                    for (int q = 0; q < NR / 4; ++q)
                        w[q] = *(const uint64_t *)(qring + ((c0 + 8 * q) &
                                                            (QR - 1)));
                    set_q(w);
                }
            }
            state = ovf && state == kRun ? kOut : state;
            fin = state != kDone && (state != kRun || minCol >= maxCol);
            any = __ballot(fin);
        }
        if (!any)
            continue;

        // ---- finish rows whose band emptied (or that never started): the
        // "longest extension" end point, from the last computed column of the
        // last anti-diagonal, then the end of d-1, else the best of d-2
        {
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                *(u32a *)(dmp + j * BL + 2 * r) = P[r];
                *(u32a *)(dmp + W + j * BL + 2 * r) = O[r];
                *(u32a *)(dmp + 2 * W + j * BL + 2 * r) = Z[r];
            }
            any = __ballot(fin);
            int lcol = l3 + off3 - 2;
            int lrow = d - lcol;
            int ls = dmp[lcol & (W - 1)];
            const int c2a = l2 + off2 - 2, c2b = l2 + off2 - 3;
            const int v2a = dmp[W + (c2a & (W - 1))];
            const int v2b = dmp[W + (c2b & (W - 1))];
            if (ls == kUndef) {
                if (v2a != kUndef) {
                    lcol = c2a;
                    lrow = d - 1 - lcol;
                    ls = v2a;
                } else if (l2 > 2 && v2b != kUndef) {
                    lcol = c2b;
                    lrow = d - 1 - lcol;
                    ls = v2b;
                }
            }
            // first maximum of anti-diagonal d-2 over columns [off1, off1+l1)
            int m1 = INT_MIN, cm = INT_MAX;
            for (int x = j; x < W; x += 16) {
                const int col = off1 + x;
                const int v = x < l1 ? (int)dmp[2 * W + (col & (W - 1))] : INT_MIN;
                if (v > m1) {
                    m1 = v;
                    cm = col;
                }
            }
            const int mm = row_max(m1);
            cm = row_min(m1 == mm ? cm : INT_MAX);
            if (ls == kUndef && l1 > 0 && mm > kUndef) {
                ls = mm;
                lcol = cm;
                lrow = d - 2 - lcol;
            }
            if (fin && j == 0) {
                const XdTask T = a.tasks[k >> 1];
                XdOut PA_GLOBAL &o = glb(a.out)[T.id];
                const bool upd = state != kEmpty && ls != kUndef;
                const int beg_h = (int)T.beg_h, beg_v = (int)T.beg_v;
                const uint16_t fg = state == kOut ? 1 : 0;
                // (score kUndef of the other kernels where nothing is defined)
                const int score = state == kEmpty || state == kOut ? 0
                                  : ls == kUndef ? INT_MIN / 4
                                                 : ls - X + base;
                if (state == kOut) {
                    const uint32_t pos = atomicAdd(a.ovf_count, 1u);
                    a.ovf_list[pos] = k;
                }
                if (!right) {
                    o.beg_h = invalid ? 0 : (upd ? beg_h - lrow : beg_h);
                    o.beg_v = invalid ? 0 : (upd ? beg_v - lcol : beg_v);
                    o.score_left = score;
                    o.cells_left = nc;
                    o.flags_left = fg;
                } else {
                    const int end_h = beg_h + a.seed_len;
                    const int end_v = beg_v + a.seed_len;
                    o.end_h = invalid ? 0 : (upd ? end_h + lrow : end_h);
                    o.end_v = invalid ? 0 : (upd ? end_v + lcol : end_v);
                    o.score_right = score;
                    o.cells_right = nc;
                    o.flags_right = fg;
                }
            }
            state = fin ? kNeed : state;
        }
    }
}

}  // namespace

hipError_t launch_xdrop_wave(const XdTask *tasks, const uint32_t *list,
                             const uint32_t *count, uint32_t *queue,
                             const int8_t *mat, int gap, int xdrop,
                             int seed_len, XdOut *out, uint32_t *ovf_list,
                             uint32_t *ovf_count, int grid, int wide,
                             hipStream_t s)
{
    WaveArgs a{tasks, list, count, queue, mat, gap, xdrop, seed_len,
               out, ovf_list, ovf_count};
    if (wide == 0)
        hipLaunchKernelGGL(k_xdrop_band<kBandRegs[0]>, dim3(grid), dim3(64), 0,
                           s, a);
    else if (wide == 1)
        hipLaunchKernelGGL(k_xdrop_band<kBandRegs[1]>, dim3(grid), dim3(64), 0,
                           s, a);
    else
        hipLaunchKernelGGL(k_xdrop_band<kBandRegs[2]>, dim3(grid), dim3(64), 0,
                           s, a);
    return hipGetLastError();
}

int xdrop_wave_occupancy(int wide)
{
    static int cache[3] = {0, 0, 0};
    if (!cache[wide]) {
        int n = 0;
        if (wide == 0)
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &n, k_xdrop_band<kBandRegs[0]>, 64, 0);
        else if (wide == 1)
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &n, k_xdrop_band<kBandRegs[1]>, 64, 0);
        else
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &n, k_xdrop_band<kBandRegs[2]>, 64, 0);
        cache[wide] = n > 0 ? n : 1;
    }
    return cache[wide];
}

}  // namespace pa
