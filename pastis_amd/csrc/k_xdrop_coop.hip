// k_xdrop_coop.hip -- gapped X-drop extension, one work item per 16-lane row
// of a wavefront (four items per wave).
//
// Same algorithm and results as xd_dir in k_xdrop.hip (the restatement of
// SeqAn's GappedXDrop one-direction extension used at
// src/align/SeqanXdropAligner.cpp:281-283), mapped onto lanes instead of
// loops:
//   - the cells written on anti-diagonal d are the columns [off, maxCol]
//     (off = minCol - 1); column c lives in lane c mod 16 of the item's row,
//     so as long as that range is at most 16 columns wide every column has
//     its own lane and the three live anti-diagonals are three registers;
//   - the left neighbour (column c-1) is lane c-1 mod 16: one DPP row_ror:1
//     move; the anti-diagonal maximum is four DPP rotations;
//   - the new band limits (leading / trailing undefined columns) are a row
//     minimum and a row maximum over the columns that meet the conditions.
//   - residues come from rings in LDS (the item's next columns and rows, 16
//     at a time, loaded 16 steps before they are needed), and the score of
//     the next anti-diagonal is looked up while this one is computed: for the
//     lane's column and for the one 16 further, which it holds if the band
//     leaves its column behind.
// What bounds it is the chain of one anti-diagonal (neighbour, maximum, band
// limits): about 0.2 us for four items a wave, a quarter of what the per-lane
// kernel of k_xdrop.hip takes for its 64.  So it runs where the per-lane
// kernel would leave the chip waiting for single lanes: all items of a small
// batch, and the items of a larger one that may go on for long (xd_route).
// An item whose written range would exceed 16 columns stops and goes to the
// overflow list; the band kernels recompute it from scratch.  A row whose
// item ends takes the next item of the queue at once, so the four rows of a
// wave stay busy whatever the item lengths.
#include <limits.h>

#include "pa_internal.h"

namespace pa {
namespace {

constexpr int32_t kUndef = INT_MIN / 4;
constexpr int G = 16;   // lanes per item
constexpr uint32_t kChunk = 4;    // items claimed per queue atomic
constexpr int kRing = 128;        // residues per LDS ring (a power of two)
constexpr int kItems = 16;        // items per workgroup (four waves)
constexpr int kSteps = 16;        // anti-diagonals between ring refills

// lane (j - k) mod 16 of the same row
template <int K> __device__ inline int ror(int v)
{
    // every lane has a source: no old operand, so that the move folds into
    // the instruction that uses it
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

struct CoopArgs {
    const XdTask *tasks;
    const uint32_t *list;   // work items k = 2 * task + dir, NULL = 0..count
    const uint32_t *count;
    uint32_t *queue;
    const int8_t *mat;
    int gap, X, seed_len;
    XdOut *out;
    uint32_t *ovf_list, *ovf_count;
};

enum : int { kNeed = 0, kRun = 1, kDone = 2 };

// These waves hold the batch's longest chains: they issue ahead of the waves
// they share a SIMD with (beside the per-lane kernel's six, a step took three
// times as long).
__device__ inline void xd_first_issue()
{
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_s_setprio(3);
#endif
}

__global__ __launch_bounds__(256) void k_xdrop_coop(CoopArgs a)
{
    xd_first_issue();
    __shared__ int8_t mat[32 * 32];
    // residues of columns (q) and rows (d) of each item
    __shared__ uint8_t rings[2 * kItems * kRing];
    for (int i = threadIdx.x; i < 32 * 32; i += blockDim.x)
        mat[i] = a.mat[i];
    // (residue codes are below 32: a slot not yet stored must be, too)
    for (int i = threadIdx.x; i < 2 * kItems * kRing; i += blockDim.x)
        rings[i] = 0;
    __syncthreads();
    const uint32_t n = *a.count;
    const int lane = threadIdx.x & 63;
    const int j = lane & 15;
    const int row = lane >> 4;
    const int gap = a.gap, X = a.X;
    uint8_t *const qring = rings + (threadIdx.x >> 4) * (2 * kRing);
    uint8_t *const dring = qring + kRing;

    // row-uniform state of the current item
    int state = kNeed;
    uint32_t k = 0;
    int cols = 0, rows = 0, d = 0, minCol = 0, maxCol = 0, best = 0;
    int off1 = 0, off2 = 0, off3 = 0, l1 = 0, l2 = 0, l3 = 0;
    bool right = false;
    bool invalid = false;   // kXdInvalid task: empty extents
    uint32_t nc = 0;
    int64_t dgap = 0;       // d * gap, while a border cell is kept
    bool edge = false;      // one may be
    // rings: columns 1 .. qfill and rows 1 .. dfill have been stored, the
    // next 32 columns and 16 rows are on their way (one each per lane)
    int qfill = 0, dfill = 0, qpre0 = 0, qpre1 = 0, dpre = 0;
    // residue addresses: column c at qb[qstep * c], row r at db[qstep * r]
    const uint8_t PA_GLOBAL *qb = nullptr, *db = nullptr;
    int qstep = 1;
    int c = 0;              // this lane's column on anti-diagonal d + 1
    int qv = 0, sc = 0;     // its residue * 32, its score on anti-diagonal d+1
    auto q_load = [&](int col) {
        return col < cols ? (int)qb[qstep > 0 ? col : -col] : 0;
    };
    auto d_load = [&](int r) {
        return r < rows ? (int)db[qstep > 0 ? r : -r] : 0;
    };
    // this lane's values on anti-diagonals d-2, d-1, d
    int A1 = kUndef, A2 = kUndef, A3 = kUndef;
    // items claimed by this wave and not yet handed out: [cbase, cend)
    uint32_t cbase = 0, cend = 0;

    for (;;) {
        // ---- hand out items to rows that need one.  The wave claims
        // kChunk items per atomic and hands them out in row order; all
        // lanes run this block together (wave-uniform control flow).
        {
            uint64_t need = __ballot(state == kNeed && j == 0);
            while (need) {
                if (cbase >= cend) {
                    uint32_t b = atomicAdd(a.queue, lane == 0 ? kChunk : 0u);
                    b = __builtin_amdgcn_readfirstlane(b);
                    cbase = b;
                    cend = b + kChunk;
                }
                const uint32_t cnt = (uint32_t)__popcll(need);
                const uint32_t take = min(cnt, cend - cbase);
                const uint32_t rank = (uint32_t)__popcll(
                    need & ((1ull << (16 * row)) - 1ull));
                const bool mine = ((need >> (16 * row)) & 1ull) != 0 &&
                                  rank < take;
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
                        // the rings load up to cols and rows whatever the
                        // item's state, and the seed of an invalid task may
                        // lie anywhere
                        invalid = (T.pad & kXdInvalid) != 0;
                        if (invalid)
                            cols = rows = 0;
                        // anti-diagonal 0: column 0 = 0; anti-diagonal 1:
                        // columns 0 and 1 = gap (undefined when -gap > X)
                        const int g1 = -gap > X ? kUndef : gap;
                        A2 = j == 0 ? 0 : kUndef;
                        A3 = j <= 1 ? g1 : kUndef;
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
                        state = kRun;
                        if (rows <= 1 || cols <= 1) {
                            state = 3;   // finished without an update
                        } else {
                            const int f = 1 + j;
                            qring[f] = (uint8_t)q_load(f);
                            qring[f + 16] = (uint8_t)q_load(f + 16);
                            dring[f] = (uint8_t)d_load(f);
                            qpre0 = q_load(f + 32);
                            qpre1 = q_load(f + 48);
                            dpre = d_load(f + 16);
                            qfill = 32;
                            dfill = 16;
                            // anti-diagonal 2: column 1, row 1 only
                            c = j;
                            qv = q_load(max(j, 1)) << 5;
                            sc = mat[qv | d_load(1)];
                        }
                    }
                }
                cbase += take;
                for (uint32_t t = 0; t < take; ++t)
                    need &= need - 1;   // the rows served
            }
        }
        if (!__ballot(state != kDone))
            break;

        // ---- residues of the next kSteps anti-diagonals: they read columns
        // up to minCol + 61 (a band moves up by a column a step and at most
        // its own width more) and rows up to d + 19 - minCol
        if (qfill < minCol + 62) {
            qring[(qfill + 1 + j) & (kRing - 1)] = (uint8_t)qpre0;
            qring[(qfill + 17 + j) & (kRing - 1)] = (uint8_t)qpre1;
            qfill += 32;
            qpre0 = q_load(qfill + 1 + j);
            qpre1 = q_load(qfill + 17 + j);
        }
        if (dfill < d + 20 - minCol) {
            dring[(dfill + 1 + j) & (kRing - 1)] = (uint8_t)dpre;
            dfill += 16;
            dpre = d_load(dfill + 1 + j);
        }
        // ---- kSteps anti-diagonals, or until a row's band is empty or too
        // wide.  Rows without an item compute on (their results go nowhere):
        // with the updates under a condition the compiler copies the whole
        // state twice a step.
        bool fin = state != kDone && !(state == kRun && minCol < maxCol);
        uint64_t any = __ballot(fin);
        for (int st = 0; st < kSteps && !any; ++st) {
            // the written range of the new anti-diagonal is [minCol-1, maxCol]
            const bool ovf = maxCol - minCol + 2 > G;
            const int noff3 = minCol - 1;
            const int nl3 = maxCol + 1 - noff3;
            ++d;
            // residues of the anti-diagonal after the new one, for this
            // lane's column (A) and the one 16 further (B)
            const int ra = d + 1 - c;
            const int dA = dring[ra & (kRing - 1)];
            const int dB = dring[(ra - 16) & (kRing - 1)];
            const int qB = qring[(c + 16) & (kRing - 1)] << 5;
            const bool ge = c >= minCol, comp = ge && c < maxCol;
            // left neighbours: column c-1 on anti-diagonal d (A3) and d-1
            // (A2); column c on d is this lane's A3 (the written ranges nest,
            // so these registers hold exactly those columns wherever they are
            // read)
            const int lA3 = ror<1>(A3);
            const int lA2 = ror<1>(A2);
            const int tmp = max(max(lA3, A3) + gap, lA2 + sc);
            int v = comp && tmp >= best - X ? tmp : kUndef;
            const int scA = mat[qv | dA], scB = mat[qB | dB];
            // cells of column 0 and row 0, while the gap to them is kept: d *
            // gap falls and the limit does not, so once it is not, never again
            if (__ballot(edge)) {
                dgap += gap;
                edge = edge && dgap > (int64_t)best - X;
                if (edge && !comp && (c == 0 || (c == maxCol && d == maxCol)))
                    v = (int)dgap;
            }
            // anti-diagonal best (best >= 0 > any border cell)
            const int adb = row_max(v);
            // minCol: first column c >= minCol where the run of cells
            // undefined on the new anti-diagonal and (column c-1) on d stops;
            // column c-1 lies on d's written range [off3, off3+l3) or the run
            // stops there
            const bool stop =
                max(v, lA3) != kUndef || c - 1 - off3 >= l3;
            const int lo =
                row_min(ge && c <= maxCol && stop ? c : INT_MAX);
            // maxCol: last c in [off, maxCol-1] defined on the new
            // anti-diagonal or on d
            const int hi =
                row_max(c < maxCol && max(v, A3) != kUndef ? c : -1);
            nc += (uint32_t)(maxCol - minCol);
            best = max(best, adb);
            A1 = A2;
            A2 = A3;
            A3 = v;
            off1 = off2;
            off2 = off3;
            off3 = noff3;
            l1 = l2;
            l2 = l3;
            l3 = nl3;
            minCol = max(min(lo, maxCol + 1), d + 2 - rows);
            maxCol = min(max(hi + 1, noff3) + 1, cols);
            // the column of the next anti-diagonal, [minCol - 1, + 16): the
            // same or the one 16 further
            const bool up = c < minCol - 1;
            c += up ? 16 : 0;
            qv = up ? qB : qv;
            sc = up ? scB : scA;
            state = ovf && state == kRun ? 4 : state;
            fin = state != kDone && (state != kRun || minCol >= maxCol);
            any = __ballot(fin);
        }
        if (!any)
            continue;

        // ---- finish rows whose band emptied (or that never started)
        {
            // longest extension: the last computed column of the last
            // anti-diagonal, then the end of d-1, else the best of d-2
            const int rb = row * 16;
            int lcol = l3 + off3 - 2;
            int lrow = d - lcol;
            int ls = __shfl(A3, rb + (lcol & 15));
            const int c2a = l2 + off2 - 2, c2b = l2 + off2 - 3;
            const int v2a = __shfl(A2, rb + (c2a & 15));
            const int v2b = __shfl(A2, rb + (c2b & 15));
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
            const int c1 = off1 + ((j - off1) & 15);
            const bool in1 = c1 < off1 + l1;
            const int m1 = row_max(in1 ? A1 : INT_MIN);
            const int cm = row_min(in1 && A1 == m1 ? c1 : INT_MAX);
            if (ls == kUndef && l1 > 0 && m1 > ls) {
                ls = m1;
                lcol = cm;
                lrow = d - 2 - lcol;
            }
            if (fin && j == 0) {
                const XdTask T = a.tasks[k >> 1];
                XdOut PA_GLOBAL &o = glb(a.out)[T.id];
                const bool upd = state != 3 && ls != kUndef;
                const int beg_h = (int)T.beg_h, beg_v = (int)T.beg_v;
                const uint16_t fl = state == 4 ? 1 : 0;
                if (state == 4) {
                    const uint32_t pos = atomicAdd(a.ovf_count, 1u);
                    a.ovf_list[pos] = k;
                }
                if (!right) {
                    o.beg_h = invalid ? 0 : (upd ? beg_h - lrow : beg_h);
                    o.beg_v = invalid ? 0 : (upd ? beg_v - lcol : beg_v);
                    o.score_left = state == 3 ? 0 : ls;
                    o.cells_left = nc;
                    o.flags_left = fl;
                } else {
                    o.end_h = invalid ? 0
                              : (upd ? beg_h + a.seed_len + lrow
                                     : beg_h + a.seed_len);
                    o.end_v = invalid ? 0
                              : (upd ? beg_v + a.seed_len + lcol
                                     : beg_v + a.seed_len);
                    o.score_right = state == 3 ? 0 : ls;
                    o.cells_right = nc;
                    o.flags_right = fl;
                }
            }
            state = fin ? kNeed : state;
        }
    }
}

}  // namespace

hipError_t launch_xdrop_coop(const XdTask *tasks, const uint32_t *list,
                             const uint32_t *count, uint32_t *queue,
                             const int8_t *mat, int gap, int xdrop,
                             int seed_len, XdOut *out, uint32_t *ovf_list,
                             uint32_t *ovf_count, int grid, hipStream_t s)
{
    CoopArgs a{tasks, list, count, queue, mat, gap, xdrop, seed_len,
               out, ovf_list, ovf_count};
    hipLaunchKernelGGL(k_xdrop_coop, dim3(grid), dim3(256), 0, s, a);
    return hipGetLastError();
}

int xdrop_coop_occupancy()
{
    static int cache = 0;
    if (!cache) {
        int n = 0;
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_xdrop_coop, 256, 0);
        cache = n > 0 ? n : 1;
    }
    return cache;
}

}  // namespace pa
