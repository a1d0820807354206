// k_dp_linear.h -- alignment under a linear gap cost: traced global, score-only
// local and traced local.  Included by k_dp.hip.
//
// With open > ext a gap is never extended: H >= E gives H + open > E + ext,
// so every gap residue costs `open` (= g) and the three-state recurrence is
//   H(i,j) = max(H(i-1,j-1) + s, H(i-1,j) + g, H(i,j-1) + g [, 0 local]).
// Ties: restart (local) > diagonal > up > left, as in k_dp; a walk never
// continues a gap by an extension bit.
//
// Two cells share a register (lo and hi strip of a lane's rows, the hi strip
// one column behind) as non-negative int16 below 0x7c00.  There int16 order is
// half-float order, so one v_pk_maximum3_f16 takes the maximum of three cells
// of both strips (half denormals are kept: the kernels run with the default
// mode).  Traced values are 4 * value + tag (3 restart, 2 diagonal, 1 up, 0
// left); the tag of the maximum is the cell's 2-bit trace code.
//
// Global (LinGlobal): in the frame H'(i,j) = H(i,j) - g (i + j) gap steps cost
// nothing and a diagonal step scores s' = s - 2g, 0 .. 15 here (lin_global).
// H' grows along rows and columns by 0 .. 15 per step, so only differences
// are kept:
//   u(i,j) = H'(i,j) - H'(i-1,j),   v(i,j) = H'(i,j) - H'(i,j-1)
//   z = max(s', u(i,j-1), v(i-1,j)),  u(i,j) = z - v(i-1,j),
//   v(i,j) = z - u(i,j-1),            score = sum of u(i,n) + g (m + n).
// No value leaves 0 .. 15, whatever the lengths, so no task needs int32; one
// register per row holds the state and the borders are zeros.  A cell pair is
//   z = max3(s, v, u); z1 = (z & ~3) | 1; u = z1 - v; v = z1 - u
// (no half borrows, so plain 32-bit subtractions).  Alignment by differences
// is published (Suzuki and Kasahara, BMC Bioinformatics 19, 2018, for affine
// gaps in SIMD lanes).
//
// Local (LinLocal): H and H + g (saturated at 0) per row; saturating
// subtraction takes the place of the maximum with 0.  Scores that come near
// 0x7c00 run again in int32.
//
// Lanes ahead of their first column or behind their last one compute on
// without a test: there the profile holds the lowest score, which leaves the
// global state zero before the first column and unchanged after the last, and
// keeps local cells below the best one.
//
// What bounds it: VALU instructions.  A step of 16 row pairs takes 125 in
// global mode, 7.8 per pair (4 recurrence, 2 score unpack, 1.25 code packing),
// 165-185 in traced local mode and 105-125 in score-only mode, against 22-28
// per pair in the affine kernels, which carry E, F and H.  By the counters the
// global kernel issues VALU in 81 % of the cycles with 96 % of the lanes on,
// the traced local one in 76 % (90 %) and the score-only one in 75 % (87 %):
// 26,624 bytes of LDS a wave hold it to six waves per CU, two SIMDs with one.
// Measured, affine kernels -> these:
//   400,000 pairs of the log-normal X-drop workload (30 % homologs), traced
//     global DP 16.6 -> 5.0 ms (eight launches -> one);
//   100,000 pairs U[50,500], traced local DP 6.9 -> 2.6 ms, score only
//     4.9 -> 1.7 ms;
//   100,000 pairs with a tail to 35,000 residues, score only, a pass alone
//     180-470 -> 14 ms (one pass among others 5-12, by the longest pair).
#pragma once

namespace pa {

// maximum of three packed pairs of non-negative int16 below 0x7c00
__device__ inline uint32_t lin_max3(uint32_t a, uint32_t b, uint32_t c)
{
#ifdef __HIP_DEVICE_COMPILE__
    uint32_t d;
    asm("v_pk_maximum3_f16 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
#else
    const uint32_t h[3] = {a, b, c};
    uint32_t lo = 0, hi = 0;
    for (uint32_t x : h) {
        lo = (x & 0xffffu) > lo ? (x & 0xffffu) : lo;
        hi = (x >> 16) > hi ? (x >> 16) : hi;
    }
    return lo | (hi << 16);
#endif
}

// Constants the optimiser cannot see through, one in a scalar and one in a
// vector register: (x & mask) | tag is then one v_and_or_b32 and a bit select
// one v_bfi_b32 (with literals each is two instructions).
struct LinConst {
    uint32_t zmask = 0xfffcfffcu, smask = 0x003c003cu, m2 = 0x03030303u,
             m4 = 0x0f0f0f0fu;
    uint32_t tag1 = 0x00010001u, tag2 = 0x00020002u;
    __device__ inline LinConst()
    {
#ifdef __HIP_DEVICE_COMPILE__
        asm volatile("" : "+s"(zmask));
        asm volatile("" : "+s"(smask));
        asm volatile("" : "+s"(m2));
        asm volatile("" : "+s"(m4));
        asm volatile("" : "+v"(tag1));
        asm volatile("" : "+v"(tag2));
#endif
    }
};

__device__ inline void lin_opaque(uint32_t &x)
{
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(x));
#endif
}

// Value of the lane before; the first lane of a task (fl) takes `first`
// (lane 0 as the DPP "old" operand, other first lanes by a select).
template <bool ONE> __device__ inline int lin_lane_up(int first, int src,
                                                      bool fl)
{
    const int v = __builtin_amdgcn_update_dpp(first, src, 0x138, 0xf, 0xf,
                                              false);
    return ONE ? v : fl ? first : v;
}

// Eight bytes at any address (gfx950 global loads need no alignment).
__device__ inline uint64_t lin_load8(const uint8_t PA_GLOBAL *p)
{
    typedef uint64_t __attribute__((aligned(1))) u64u;
    return *(const u64u PA_GLOBAL *)p;
}

// Bytes k of an 8-byte window whose index i0 + k lies in [0, n), `fill`
// elsewhere.
__device__ inline uint64_t lin_window(uint64_t raw, int i0, int n,
                                      uint64_t fill)
{
    uint64_t m = ~0ull;
    if (i0 < 0)
        m = i0 > -8 ? m << (8 * -i0) : 0ull;
    const int nh = n - i0;
    if (nh < 8)
        m &= nh > 0 ? (1ull << (8 * nh)) - 1ull : 0ull;
    return (raw & m) | (fill & ~m);
}

// Words that waves on different XCDs exchange: stores that go through to
// memory and loads that bypass the caches of their XCD.
__device__ inline uint64_t lin_get(const uint64_t PA_GLOBAL *p)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#else
    return __atomic_load_n(p, __ATOMIC_RELAXED);
#endif
}
__device__ inline void lin_put(uint64_t PA_GLOBAL *p, uint64_t v)
{
#ifdef __HIP_DEVICE_COMPILE__
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#else
    __atomic_store_n(p, v, __ATOMIC_RELAXED);
#endif
}
// Every store of this wave has reached memory.
__device__ inline void lin_flush()
{
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}
__device__ inline void lin_pause()
{
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_s_sleep(8);
#endif
}

// Profile: kProfChars codes x two strips x 64 lanes x 16 nibbles (two
// words).  Each lane holds the scores of its own 32 rows whatever the lanes
// per task, so the layout is the same for all classes; lanes of a wave read
// consecutive 8-byte words (no bank conflict).  Byte k of word w holds rows
// 8w + k and 8w + 4 + k as the two tables of the mode give them: in bits 2-5
// and in bits 6, 7, 0, 1 (traced), or in the low and the high nibble.
constexpr int kLinProfWords = kProfChars * 2 * 64 * 2;

// ---- cell arithmetic of the modes -------------------------------------------
// A mode keeps a lane's rows and provides
//   V            a pair of values (lo, hi strip) handed down the rows
//   reset()      before a pass
//   step(...)    one step of the lane's rows from profile words and the row
//                above; returns the last row's pair, and the trace record
//   pass_value() what the pass adds to the task's result, the same on all
//                lanes of the task; merge() combines passes; write() stores

typedef unsigned short lin_u2 __attribute__((ext_vector_type(2)));

// max(a - b, 0) in both halves
__device__ inline uint32_t lin_subsat(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(
        uint32_t,
        __builtin_elementwise_sub_sat(__builtin_bit_cast(lin_u2, a),
                                      __builtin_bit_cast(lin_u2, b)));
}
__device__ inline uint32_t lin_max(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(
        uint32_t, __builtin_elementwise_max(__builtin_bit_cast(lin_u2, a),
                                            __builtin_bit_cast(lin_u2, b)));
}

// Bytes q of both words: in both bytes of each half (traced profiles), or
// in the low byte.
__device__ inline uint32_t lin_bytes2(uint32_t hi, uint32_t lo, int q)
{
    return __builtin_amdgcn_perm(hi, lo, (uint32_t)q * 0x0101u |
                                             (uint32_t)(4 + q) * 0x01010000u);
}
__device__ inline uint32_t lin_bytes1(uint32_t hi, uint32_t lo, int q)
{
    return __builtin_amdgcn_perm(hi, lo, (uint32_t)q | 0x0c00u |
                                             ((uint32_t)(4 + q) << 16) |
                                             0x0c000000u);
}

// 2-bit codes (low bits of each half of z) of 16 rows: byte 2 (r % 2) + half
// of word r / 8, bits 2 ((r % 8) / 2).
__device__ inline void lin_pack(const uint32_t *z, const LinConst &C,
                                uint32_t *rec)
{
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        uint32_t y[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            y[q] = __builtin_amdgcn_perm(z[8 * w + 2 * q + 1],
                                         z[8 * w + 2 * q], 0x06040200u);
        const uint32_t x01 = (y[0] & C.m2) | ((y[1] << 2) & ~C.m2);
        const uint32_t x23 = (y[2] & C.m2) | ((y[3] << 2) & ~C.m2);
        rec[w] = (x01 & C.m4) | ((x23 << 4) & ~C.m4);
    }
}

// Sum over the lanes of a task (L lanes from its first lane): suffix sums
// within the task, then the first lane's value.
__device__ inline uint32_t lin_task_sum(uint32_t v, int lane, int gl, int L)
{
    for (int off = 1; off < L; off <<= 1) {
        const uint32_t x = __shfl(v, lane + off);
        v += gl + off < L ? x : 0u;
    }
    return __shfl(v, lane - gl);
}
__device__ inline uint64_t lin_shfl64(uint64_t v, int lane)
{
    return ((uint64_t)__shfl((uint32_t)(v >> 32), lane) << 32) |
           __shfl((uint32_t)v, lane);
}
__device__ inline uint64_t lin_task_max(uint64_t v, int lane, int gl, int L)
{
    for (int off = 1; off < L; off <<= 1) {
        const uint64_t x = lin_shfl64(v, lane + off);
        v = gl + off < L && x > v ? x : v;
    }
    return lin_shfl64(v, lane - gl);
}

// Packed pairs: V is two int16 in one register.
struct LinPacked {
    typedef uint32_t V;
    static constexpr bool I16 = true;
    __device__ static inline V mk(uint32_t lo, uint32_t hi)
    {
        return lo | (hi << 16);
    }
    __device__ static inline uint32_t hi(V v) { return v >> 16; }
    // row above of the next step: lo from the hi half of the lane before,
    // hi from the own lo half
    template <bool ONE>
    __device__ static inline V hand_up(V v, uint32_t first, bool fl)
    {
        const uint32_t sh =
            (uint32_t)lin_lane_up<ONE>((int)(first << 16), (int)v, fl);
        return __builtin_amdgcn_alignbit(v, sh, 16);
    }
};
struct LinPair {
    uint32_t x, y;
};
struct LinWide {
    typedef LinPair V;
    static constexpr bool I16 = false;
    __device__ static inline V mk(uint32_t lo, uint32_t hi)
    {
        return LinPair{lo, hi};
    }
    __device__ static inline uint32_t hi(V v) { return v.y; }
    template <bool ONE>
    __device__ static inline V hand_up(V v, uint32_t first, bool fl)
    {
        return LinPair{(uint32_t)lin_lane_up<ONE>((int)first, (int)v.y, fl),
                       v.x};
    }
};

// Global alignment by differences (top of file).  V: 4 v + 1.
struct LinGlobal : LinPacked {
    static constexpr bool TRACE = true, LOCAL = false;
    static constexpr uint32_t kBorder = 1;   // v = 0
    static constexpr int kTable = kPmatRot;
    uint32_t u[kLinR];
    __device__ inline LinGlobal(const LinArgs &) {}
    __device__ inline void reset(int)
    {
#pragma unroll
        for (int r = 0; r < kLinR; ++r)
            u[r] = 0;
    }
    __device__ inline V step(uint2 lw, uint2 hw, V vv, const LinConst &C,
                             uint32_t *rec)
    {
        uint32_t z[kLinR];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            uint32_t s[8];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t b =
                    lin_bytes2(w ? hw.y : hw.x, w ? lw.y : lw.x, q);
                s[q] = (b & C.smask) | C.tag2;
                s[q + 4] = ((b >> 4) & C.smask) | C.tag2;
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int r = 8 * w + q;
                z[r] = lin_max3(s[q], vv, u[r]);
                const uint32_t z1 = (z[r] & C.zmask) | C.tag1;
                const uint32_t un = z1 - vv;
                vv = z1 - u[r];
                u[r] = un;
            }
        }
        lin_pack(z, C, rec);
        return vv;
    }
    // 4 times the sum of u(i, tlen) over this pass's rows
    __device__ inline uint64_t pass_value(int qlen, int row0, int lane, int gl,
                                          int L)
    {
        const int nlo = qlen - row0, nhi = nlo - kLinR;
        uint32_t sum = 0;
#pragma unroll
        for (int r = 0; r < kLinR; ++r) {
            const uint32_t m = (r < nlo ? 0x0000ffffu : 0u) |
                               (r < nhi ? 0xffff0000u : 0u);
            sum += u[r] & m;
        }
        return lin_task_sum((sum & 0xffffu) + (sum >> 16), lane, gl, L);
    }
    __device__ static inline uint64_t merge(uint64_t a, uint64_t b)
    {
        return a + b;
    }
    __device__ static inline void write(const LinArgs &a, uint32_t tid,
                                        const DpTask &T, uint64_t v, bool)
    {
        DpOut o = {};
        o.score = (int)(v >> 2) + a.gap * (int)(T.qlen + T.tlen);
        o.q_beg = o.q_end = (int)T.qlen;
        o.t_beg = o.t_end = (int)T.tlen;
        a.out[tid] = o;
    }
};

// Local alignment: H(i,j) = max(0, H(i-1,j-1) + s, H(i-1,j) + g,
// H(i,j-1) + g), with saturating subtraction as the maximum with 0.  V: the
// row's H (times 4 when traced).  Rows past the query and columns past its
// end score the matrix minimum, so their cells lie below some cell before
// them and never become the best one.
template <bool TR, bool PACKED>
struct LinLocal : std::conditional_t<PACKED, LinPacked, LinWide> {
    typedef std::conditional_t<PACKED, LinPacked, LinWide> Base;
    typedef typename Base::V V;
    static constexpr bool TRACE = TR, LOCAL = true;
    static constexpr uint32_t kBorder = 0;
    static constexpr int kTable = TR ? kPmatRot : kPmatPair;
    static constexpr int SH = TR ? 2 : 0;
    V H[kLinR], Ho[kLinR], saved[kLinR];
    V dg, best, col, bcol, G, B;
    // g and -nib_min, times 4 when traced; in registers the optimiser cannot
    // see through, so that each is one operand
    __device__ inline LinLocal(const LinArgs &a)
    {
        const uint32_t g = (uint32_t)(-a.gap) << SH,
                       b = (uint32_t)(-a.nib_min) << SH;
        G = Base::mk(g, g);
        B = Base::mk(b, b);
    }
    // col: column of step 0 (this lane's lo strip)
    __device__ inline void reset(int c0)
    {
#pragma unroll
        for (int r = 0; r < kLinR; ++r)
            H[r] = Ho[r] = saved[r] = Base::mk(0, 0);
        dg = best = bcol = Base::mk(0, 0);
        if constexpr (PACKED)
            col = ((uint32_t)c0 & 0xffffu) | ((uint32_t)(c0 - 1) << 16);
        else
            col = LinPair{(uint32_t)c0, (uint32_t)(c0 - 1)};
    }
    __device__ inline V step(uint2 lw, uint2 hw, V up, const LinConst &C,
                             uint32_t *rec)
    {
        if constexpr (PACKED)
            return step16(lw, hw, up, C, rec);
        else
            return step32(lw, hw, up, rec);
    }
    __device__ inline V step16(uint2 lw, uint2 hw, V up, const LinConst &C,
                               uint32_t *rec)
    {
        uint32_t z[kLinR], hd = dg, ho = lin_subsat(up, G), cm = 0;
        dg = up;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            uint32_t s[8];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t hi = w ? hw.y : hw.x, lo = w ? lw.y : lw.x;
                if (TR) {
                    const uint32_t b = lin_bytes2(hi, lo, q);
                    s[q] = (b & C.smask) | C.tag2;
                    s[q + 4] = ((b >> 4) & C.smask) | C.tag2;
                } else {
                    const uint32_t b = lin_bytes1(hi, lo, q);
                    s[q] = b & 0x000f000fu;
                    s[q + 4] = __builtin_bit_cast(
                        uint32_t, __builtin_bit_cast(lin_u2, b) >>
                                      (unsigned short)4);
                }
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int r = 8 * w + q;
                // halves stay below 2^15: no carry between them
                const uint32_t t = lin_subsat(hd + s[q], B);
                hd = H[r];
                uint32_t h;
                if (TR) {
                    // tags: 3 restart (value 0), 2 diagonal, 1 up, 0 left
                    z[r] = lin_max(lin_max3(t, ho | 0x00010001u, Ho[r]),
                                   0x00030003u);
                    h = z[r] & C.zmask;
                } else {
                    h = lin_max3(t, ho, Ho[r]);
                }
                ho = lin_subsat(h, G);
                H[r] = h;
                Ho[r] = ho;
                if (r & 1)
                    cm = lin_max3(cm, H[r - 1], h);
            }
        }
        if (TR)
            lin_pack(z, C, rec);
        col = __builtin_bit_cast(uint32_t,
                                 __builtin_bit_cast(lin_u2, col) +
                                     (unsigned short)1);
        const uint32_t nb = lin_max(best, cm);
        const uint32_t chg = nb ^ best;
        if (chg) {
            // halves that rose: all ones
            const lin_u2 one = {1, 1}, zero = {0, 0};
            uint32_t m = __builtin_bit_cast(
                uint32_t,
                zero - __builtin_elementwise_min(
                           __builtin_bit_cast(lin_u2, chg), one));
            lin_opaque(m);   // one bit select a row, not two half selects
            bcol = (col & m) | (bcol & ~m);
#pragma unroll
            for (int r = 0; r < kLinR; ++r)
                saved[r] = (H[r] & m) | (saved[r] & ~m);
            best = nb;
        }
        return H[kLinR - 1];
    }
    __device__ inline V step32(uint2 lw, uint2 hw, V up, uint32_t *rec)
    {
        auto floor0 = [](uint32_t a, uint32_t b) { return a > b ? a - b : 0u; };
        auto mx = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
        LinPair hd = dg, ho{floor0(up.x, G.x), floor0(up.y, G.y)}, cm{0, 0};
        dg = up;
        uint32_t w0 = 0, w1 = 0;
#pragma unroll
        for (int r = 0; r < kLinR; ++r) {
            const uint32_t lo = r < 8 ? lw.x : lw.y, hi = r < 8 ? hw.x : hw.y;
            const int sh = 8 * (r & 3);
            const uint32_t bl = (lo >> sh) & 0xffu, bh = (hi >> sh) & 0xffu;
            LinPair n;
            if (TR) {   // rows 4 .. 7 of a word in bits 6, 7, 0, 1
                n.x = (r & 4 ? (bl >> 6) | ((bl & 3u) << 2) : (bl >> 2) & 15u)
                          << 2 | 2u;
                n.y = (r & 4 ? (bh >> 6) | ((bh & 3u) << 2) : (bh >> 2) & 15u)
                          << 2 | 2u;
            } else {
                n.x = r & 4 ? bl >> 4 : bl & 15u;
                n.y = r & 4 ? bh >> 4 : bh & 15u;
            }
            LinPair t{floor0(hd.x + n.x, B.x), floor0(hd.y + n.y, B.y)};
            hd = H[r];
            LinPair h;
            if (TR) {
                h.x = mx(mx(t.x, ho.x | 1u), mx(Ho[r].x, 3u));
                h.y = mx(mx(t.y, ho.y | 1u), mx(Ho[r].y, 3u));
                const uint32_t c = (h.x & 3u) | ((h.y & 3u) << 8);
                const uint32_t v = c << (16 * (r & 1) + 2 * ((r & 7) >> 1));
                (r < 8 ? w0 : w1) |= v;
                h.x &= ~3u;
                h.y &= ~3u;
            } else {
                h.x = mx(mx(t.x, ho.x), Ho[r].x);
                h.y = mx(mx(t.y, ho.y), Ho[r].y);
            }
            ho = LinPair{floor0(h.x, G.x), floor0(h.y, G.y)};
            H[r] = h;
            Ho[r] = ho;
            cm = LinPair{mx(cm.x, h.x), mx(cm.y, h.y)};
        }
        rec[0] = w0;
        rec[1] = w1;
        ++col.x;
        ++col.y;
        const bool cx = cm.x > best.x, cy = cm.y > best.y;
        if (cx || cy) {
            bcol = LinPair{cx ? col.x : bcol.x, cy ? col.y : bcol.y};
#pragma unroll
            for (int r = 0; r < kLinR; ++r)
                saved[r] = LinPair{cx ? H[r].x : saved[r].x,
                                   cy ? H[r].y : saved[r].y};
            best = LinPair{cx ? cm.x : best.x, cy ? cm.y : best.y};
        }
        return H[kLinR - 1];
    }
    // score << 40 | first column (complemented) | first row (complemented)
    // of the pass's best cell, 0 if none is positive
    __device__ inline uint64_t pass_value(int qlen, int row0, int lane, int gl,
                                          int L)
    {
        auto half = [](V v, int hf) -> uint32_t {
            if constexpr (PACKED)
                return hf ? v >> 16 : v & 0xffffu;
            else
                return hf ? v.y : v.x;
        };
        uint64_t key = 0;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const uint32_t sc = half(best, hf), c = half(bcol, hf);
            const int rbase = row0 + hf * kLinR;
            int row = -1;
#pragma unroll
            for (int r = kLinR - 1; r >= 0; --r)
                if (half(saved[r], hf) == sc && rbase + r < qlen)
                    row = rbase + r;
            const uint64_t ck = ((uint64_t)(sc >> SH) << 40) |
                                ((uint64_t)(0xffffu - c) << 24) |
                                (uint64_t)(0xffffff - row);
            key = sc && row >= 0 && ck > key ? ck : key;
        }
        return lin_task_max(key, lane, gl, L);
    }
    __device__ static inline uint64_t merge(uint64_t a, uint64_t b)
    {
        return a > b ? a : b;
    }
    // first: one lane of the task
    __device__ static inline void write(const LinArgs &a, uint32_t tid,
                                        const DpTask &, uint64_t v, bool first)
    {
        const int sc = (int)(v >> 40);
        DpOut o = {};
        if (sc > 0) {
            o.score = sc;
            o.t_beg = o.t_end = 0xffff - (int)((v >> 24) & 0xffff);
            o.q_beg = o.q_end = 0xffffff - (int)(v & 0xffffff) + 1;
        }
        if (PACKED) {
            // the score may have left the range of the int16 maximum: the
            // int32 kernel runs the task again
            if (sc >= (TR ? kLinSatTraced : kLinSat) && first)
                a.sat_list[atomicAdd(a.sat_count, 1u)] = tid;
        } else if (sc >= (TR ? kSatTraced : kSat) && first) {
            // reported as a re-run from the scores that do not fit int16
            a.tflags[tid] |= 1;
            atomicAdd(a.reruns, 1ull);
        }
        a.out[tid] = o;
    }
};

// ---- the wavefront ----------------------------------------------------------

// Progress word of a pipelined pass (item x): the number of the item after
// it, then the columns of its last row that are in memory.
__device__ inline uint64_t lin_progress(uint32_t x, uint32_t cols)
{
    return ((uint64_t)(x + 1u) << 32) | cols;
}
constexpr uint32_t kLinDone = 0xffffffffu;

// Runs the tasks of list[0, count): L lanes per task, 64 / L tasks side by
// side in a wave.  MULTI: 64 lanes, tasks of any row count, pass after pass.
// PIPE: every pass of a task is an item of its own, so that the passes of a
// long task run on as many waves, each a few hundred columns behind the one
// before: without it the longest task of a batch ran its passes on one wave
// (35,000 x 35,000 residues: 320 ms) while the chip was idle.  (The grid has
// no more workgroups than the batch tasks, so a single task gains nothing:
// 20,000 x 20,000 residues 66 ms.)  Items are
// claimed in order, a task's passes one after the other, and an item waits
// only for items claimed before it (its predecessor's columns, the last
// owner and reader of its boundary slot), so the first unfinished item always runs.
template <class P, bool MULTI, bool PIPE>
__device__ inline void lin_run(const LinArgs &a, uint32_t *prof,
                               const uint32_t PA_GLOBAL *list, uint32_t count,
                               uint32_t *queue, int L)
{
    typedef typename P::V V;
    constexpr int R = kLinR;        // rows per half
    const int G = MULTI ? 1 : 64 / L;
    constexpr uint64_t kFillRes = 0x1919191919191919ull;   // kSentinel
    static_assert(kSentinel == 0x19, "window fill");
    if (count == 0)
        return;
    if (MULTI)
        L = 64;
    const int lane = threadIdx.x & 63;
    const int gl = lane % L, grp = lane / L;   // grp G: lanes left over
    const bool fl = gl == 0;
    uint8_t *plds = (uint8_t *)prof;
    const uint32_t lane8 = (uint32_t)lane * 8u;
    const uint32_t *pmat = (const uint32_t *)(a.mat + P::kTable);
    uint64_t PA_GLOBAL *bnd_all = glb(a.bnd);
    uint64_t PA_GLOBAL *prog = glb(a.prog);
    const uint32_t items = PIPE ? *a.pipe_items : count;
    const LinConst C;
    P cells(a);
    for (;;) {
        // every lane takes part in the atomic (only lane 0 adds)
        uint32_t k0 = atomicAdd(queue, lane == 0 ? (uint32_t)G : 0u);
        k0 = __builtin_amdgcn_readfirstlane(k0);
        if (k0 >= items)
            break;
        uint32_t k = k0 + (uint32_t)grp;
        int p0 = 0;
        if (PIPE) {   // task whose passes hold item k0: last start <= k0
            uint32_t lo = 0, hi = count - 1;
            while (lo < hi) {
                const uint32_t mid = (lo + hi + 1) / 2;
                if (a.pipe_start[mid] <= k0)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            k = lo;
            p0 = (int)(k0 - a.pipe_start[lo]);
        }
        const bool valid = grp < G && k < count;
        const uint32_t tid = list[valid ? k : k0];
        DpTask T = a.tasks[tid];
        if (!valid)
            T.qlen = T.tlen = 0;
        const uint8_t PA_GLOBAL *qs = glb_addr<const uint8_t>(T.q_off);
        const uint8_t PA_GLOBAL *ts = glb_addr<const uint8_t>(T.t_off);
        const int qlen = (int)T.qlen, tlen = (int)T.tlen;
        uint8_t PA_GLOBAL *tr = nullptr;
        if (P::TRACE)
            tr = glb(a.trace) +
                 (glb(a.trace_off)[tid] -
                  (a.trace_base ? *glb(a.trace_base) : 0ull));
        const int npass =
            MULTI ? (int)__builtin_amdgcn_readfirstlane(
                        (qlen + kLinRows - 1) / kLinRows)
                  : 1;
        const int pend = PIPE ? p0 + 1 : npass;
        // boundary rows: the item's slot (PIPE: the item before wrote the
        // one to read), or this workgroup's own
        const uint32_t S = a.pipe_slots;
        const uint64_t PA_GLOBAL *bin =
            bnd_all + (size_t)(PIPE ? (k0 + S - 1) % S : S + blockIdx.x) *
                          a.bnd_words;
        uint64_t PA_GLOBAL *bout =
            bnd_all + (size_t)(PIPE ? k0 % S : S + blockIdx.x) * a.bnd_words;
        auto wait = [&](uint32_t item, uint32_t cols) -> uint32_t {
            const uint64_t want = lin_progress(item, cols);
            uint64_t got;
            while ((got = lin_get(prog + item % S)) < want)
                lin_pause();
            asm volatile("" ::: "memory");
            return got >= lin_progress(item, kLinDone) ? kLinDone
                                                       : (uint32_t)got;
        };
        auto publish = [&](uint32_t cols) {
            lin_flush();
            if (lane == 0)
                lin_put(prog + k0 % S, lin_progress(k0, cols));
        };
        if (PIPE && k0 >= S) {
            // The slot's last owner and its reader are done with it.  (The
            // reader may be the first pass of another task, which waits for
            // nobody, so its end does not imply the owner's: an owner still
            // running would set the progress word back under this item.)
            wait(k0 - S, kLinDone);
            wait(k0 - S + 1, kLinDone);
        }
        uint64_t value = 0;
        uint32_t avail = 0;    // columns the pass before has published

        for (int p = p0; p < pend; ++p) {
            const int i0 = p * kLinRows;
            const int row0 = i0 + 2 * R * gl;
            __syncthreads();
            // ---- query profile of this lane's 32 rows -------------------
            // word (strip, w): rows 8w .. 8w+3 from the mode's first table,
            // rows 8w+4 .. 8w+7 from its second
#pragma unroll 1
            for (int sw = 0; sw < 4; ++sw) {
                const int ra = row0 + 8 * sw;   // strip sw / 2, word sw % 2
                uint32_t *dst = prof + (sw >> 1) * 128 + 2 * lane + (sw & 1);
                if (!__ballot(ra < qlen)) {
                    // rows past every query: any scores do in global mode
                    // (no cell reads a row below it), the minimum in local
                    // mode (no such cell may be the best)
                    if (P::LOCAL) {
#pragma unroll
                        for (int c = 0; c < kProfChars; ++c)
                            dst[c * 256] = 0;
                    }
                    continue;
                }
                uint32_t xs[kProfChars];
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    uint32_t mr[4][8];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int row = ra + 4 * g + q;
                        const int qc = row < qlen ? (int)qs[row] : 31;
                        // generic pointer: vector-struct loads from the
                        // global address space do not compile
                        const uint4 *src =
                            (const uint4 *)(pmat + g * 256 + qc * 8);
                        const uint4 x0 = src[0], x1 = src[1];
                        mr[q][0] = x0.x; mr[q][1] = x0.y; mr[q][2] = x0.z;
                        mr[q][3] = x0.w; mr[q][4] = x1.x; mr[q][5] = x1.y;
                        mr[q][6] = x1.z; mr[q][7] = x1.w;
                    }
#pragma unroll
                    for (int c = 0; c < kProfChars; ++c) {
                        const int wd = c >> 2, sh = c & 3;
                        const uint32_t sel = (uint32_t)sh |
                                             ((uint32_t)(4 + sh) << 8) |
                                             0x0c0c0000u;
                        const uint32_t x01 =
                            __builtin_amdgcn_perm(mr[1][wd], mr[0][wd], sel);
                        const uint32_t x23 =
                            __builtin_amdgcn_perm(mr[3][wd], mr[2][wd], sel);
                        const uint32_t x =
                            __builtin_amdgcn_perm(x23, x01, 0x05040100u);
                        xs[c] = g == 0 ? x : xs[c] | x;
                    }
                }
#pragma unroll
                for (int c = 0; c < kProfChars; ++c)
                    dst[c * 256] = xs[c];
            }
            if (MULTI && !PIPE && p > 0)
                lin_flush();   // the boundary row this pass reads
            __syncthreads();

            const int qrem = qlen - i0;
            int nact = (qrem + 2 * R - 1) / (2 * R);
            nact = nact > L ? L : nact < 0 ? 0 : nact;
            const int own_blk =
                nact > 0 ? (tlen + 2 * (nact - 1) + 1 + 7) / 8 : 0;
            int nblk = own_blk;
            if (!MULTI) {
#pragma unroll
                for (int off = 1; off < 64; off <<= 1)
                    nblk = max(nblk, __shfl_xor(nblk, off));
            }
            nblk = __builtin_amdgcn_readfirstlane(nblk);
            const bool more_passes = MULTI && p + 1 < npass;
            // blocks of this lane whose records are stored
            const int st_blk = gl < nact ? own_blk : 0;
            const uint32_t seg_bytes =
                (uint32_t)(more_passes ? 64 : nact) * (kTraceSeg * kLinRec);
            uint8_t PA_GLOBAL *trp = nullptr;
            if (P::TRACE)
                trp = tr + (uint64_t)p * lin_pass_bytes((uint32_t)tlen) +
                      (uint32_t)gl * (kTraceSeg * kLinRec);

            cells.reset(-2 * gl);
            // residues: lane's columns of block b are 8b + 1 - 2 gl .. + 7
            auto res_raw = [&](int blk) -> uint64_t {
                const int i = 8 * blk - 2 * gl;
                return i > -8 && i < tlen ? lin_load8(ts + i) : 0ull;
            };
            auto res_win = [&](uint64_t raw, int blk) {
                return lin_window(raw, 8 * blk - 2 * gl, tlen, kFillRes);
            };
            // boundary row of the pass before, 4 bytes a column: columns
            // 8b + 1 .. 8b + 8 of block b, the border's value past the end
            auto bnd_load = [&](int blk, uint32_t *w) {
                const int c0 = 8 * blk;
                if (PIPE && c0 < tlen) {
                    const uint32_t need = (uint32_t)min(c0 + 8, tlen);
                    if (avail < need)
                        avail = wait(k0 - 1, need);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint64_t x =
                        c0 < tlen ? lin_get(bin + 64 + c0 / 2 + q) : 0ull;
                    w[2 * q] = c0 + 2 * q < tlen ? (uint32_t)x : P::kBorder;
                    w[2 * q + 1] = c0 + 2 * q + 1 < tlen ? (uint32_t)(x >> 32)
                                                         : P::kBorder;
                }
            };
            uint64_t wc = res_win(res_raw(0), 0), wraw = res_raw(1);
            uint32_t bc[8], bn[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                bc[q] = bn[q] = P::kBorder;
            if (MULTI && p > 0) {
                bnd_load(0, bc);
                bnd_load(1, bn);
            }
            // LDS address of the lo strip's words of the current column;
            // the hi strip reads the column before it
            auto paddr = [&](uint32_t code) { return code * 1024u + lane8; };
            uint32_t ac = paddr((uint32_t)wc & 0xffu);
            uint2 lw = *(const uint2 *)(plds + ac);
            uint2 hw = *(const uint2 *)(plds + paddr(kSentinel) + 512);
            V vin = P::mk(fl ? bc[0] : P::kBorder, P::kBorder);
            uint32_t carry = 0;   // last column of the last row's last block

            auto run_blocks = [&](auto first_pass) {
                constexpr bool FIRST = decltype(first_pass)::value;
                for (int blk = 0; blk < nblk; ++blk) {
                    const uint64_t wn = res_win(wraw, blk + 1);
                    wraw = res_raw(blk + 2);
                    uint32_t bnn[8];
                    if (!FIRST)
                        bnd_load(blk + 2, bnn);
                    const bool store = P::TRACE && blk < st_blk;
                    uint32_t rec[4], vout[8];
#pragma unroll
                    for (int st = 0; st < 8; ++st) {
                        // profile words of the next step
                        const uint32_t code =
                            st < 7 ? (uint32_t)(wc >> (8 * ((st + 1) & 7))) &
                                         0xffu
                                   : (uint32_t)wn & 0xffu;
                        const uint32_t an = paddr(code);
                        const uint2 lwn = *(const uint2 *)(plds + an);
                        const uint2 hwn = *(const uint2 *)(plds + ac + 512);
                        const V vv = cells.step(lw, hw, vin, C,
                                                rec + 2 * (st & 1));
                        if (P::TRACE && (st & 1)) {
                            if (store) {
                                typedef uint32_t v4u
                                    __attribute__((ext_vector_type(4)));
                                v4u x;
                                x.x = rec[0];
                                x.y = rec[1];
                                x.z = rec[2];
                                x.w = rec[3];
                                *(v4u PA_GLOBAL *)(trp + (st - 1) * kLinRec) =
                                    x;
                            }
                        }
                        if (MULTI)   // the pass's last row (lane 63)
                            vout[st] = P::hi(vv);
                        const uint32_t first =
                            FIRST ? P::kBorder
                                  : st < 7 ? bc[(st + 1) & 7] : bn[0];
                        vin = P::template hand_up<MULTI>(vv, first, fl);
                        lw = lwn;
                        hw = hwn;
                        ac = an;
                    }
                    if (MULTI && more_passes) {
                        // step t's column is t - 127; columns 2m + 1 and
                        // 2m + 2 share word 64 + m, so the last step's value
                        // waits for the next block
                        if (lane == 63) {
#pragma unroll
                            for (int q = 0; q < 4; ++q)
                                lin_put(bout + (size_t)blk * 4 + q,
                                        (q ? vout[2 * q - 1] : carry) |
                                            ((uint64_t)vout[2 * q] << 32));
                        }
                        carry = vout[7];
                        if (PIPE && (blk & 7) == 7) {
                            const int cols = 8 * blk + 8 - 128;
                            if (cols > 0)
                                publish((uint32_t)min(cols, tlen));
                        }
                    }
                    if (P::TRACE)
                        trp += seg_bytes;
                    wc = wn;
                    if (!FIRST) {
#pragma unroll
                        for (int q = 0; q < 8; ++q) {
                            bc[q] = bn[q];
                            bn[q] = bnn[q];
                        }
                    }
                }
            };
            if (!MULTI || p == 0)
                run_blocks(std::true_type{});
            else
                run_blocks(std::false_type{});
            if (MULTI && more_passes && lane == 63)
                lin_put(bout + (size_t)nblk * 4, carry);
            if (PIPE && more_passes)
                publish((uint32_t)tlen);
            const uint64_t pv = cells.pass_value(qlen, row0, lane, gl, L);
            value = p == p0 ? pv : P::merge(value, pv);
        }
        if (PIPE) {
            // the passes before this one: their merged value
            if (p0 > 0) {
                wait(k0 - 1, kLinDone);
                value = P::merge(lin_get(prog + S + (k0 - 1) % S), value);
            }
            if (p0 + 1 < npass) {
                if (lane == 0)
                    lin_put(prog + S + k0 % S, value);
            } else {
                P::write(a, tid, T, value, lane == 0);
            }
            publish(kLinDone);
        } else if (valid) {
            // every lane of a task stores the same result (no lane-0 branch
            // closes the loop)
            P::write(a, tid, T, value, fl);
        }
    }
}

// All classes in one launch, the pipelined ones and then the longest rows
// first: a workgroup that finds a class drained goes on with the next one, so
// no class waits for the last tasks of another.
template <class P>
__device__ inline void lin_all(const LinArgs &a, uint32_t *prof)
{
    auto list = [&](int cls) { return glb(a.list) + a.starts[cls]; };
    lin_run<P, true, true>(a, prof, list(kLinPipe), a.counts[kLinPipe],
                           a.queues + kLinPipe, 64);
    lin_run<P, true, false>(a, prof, list(kLinPipe - 1),
                            a.counts[kLinPipe - 1], a.queues + kLinPipe - 1,
                            64);
    for (int cls = kLinPipe - 2; cls >= 0; --cls)
        lin_run<P, false, false>(a, prof, list(cls), a.counts[cls],
                                 a.queues + cls, lin_lanes(cls));
}

__global__ __launch_bounds__(64) void k_nw_linear(LinArgs a)
{
    __shared__ uint32_t prof[kLinProfWords];
    lin_all<LinGlobal>(a, prof);
}

template <bool TRACE>
__global__ __launch_bounds__(64) void k_sw_linear(LinArgs a)
{
    __shared__ uint32_t prof[kLinProfWords];
    lin_all<LinLocal<TRACE, true>>(a, prof);
}

// The tasks whose int16 scores may have left their range, in int32.
template <bool TRACE>
__global__ __launch_bounds__(64) void k_sw_linear_rerun(LinArgs a)
{
    __shared__ uint32_t prof[kLinProfWords];
    lin_run<LinLocal<TRACE, false>, true, false>(
        a, prof, glb((const uint32_t *)a.sat_list), *a.sat_count, a.sat_queue,
        64);
}

// Items of the pipelined class: its tasks' passes, one after the other
// (exclusive sums of the pass counts).  One workgroup: the class is small.
__global__ __launch_bounds__(256) void k_lin_passes(LinArgs a)
{
    __shared__ uint32_t part[4], total;
    const uint32_t n = a.counts[kLinPipe];
    const uint32_t *list = a.list + a.starts[kLinPipe];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t base = 0;
    for (uint32_t k0 = 0; k0 < n; k0 += 256) {
        const uint32_t k = k0 + threadIdx.x;
        const uint32_t own =
            k < n ? (a.tasks[list[k]].qlen + kLinRows - 1) / kLinRows : 0u;
        uint32_t run = own;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t x = __shfl(run, lane - off);
            run += lane >= off ? x : 0u;
        }
        if (lane == 63)
            part[w] = run;
        __syncthreads();
        uint32_t before = 0;
        for (int q = 0; q < w; ++q)
            before += part[q];
        if (k < n)
            a.pipe_start[k] = base + before + run - own;
        if (threadIdx.x == 255)
            total = before + run;
        __syncthreads();
        base += total;
    }
    if (threadIdx.x == 0)
        *a.pipe_items = base;
}

// Traceback over the 2-bit codes, one walk per thread, the tasks of all
// classes (longest first).  A walk goes through windows: the records of one
// lane in the segment it stands in and in the one before (64 contiguous,
// 64-byte aligned bytes each), and the 16 residues of either sequence that end
// at its cell.  Every walk of a wave loads its window at the same time, then
// all walk until they have left theirs: bound by the latency of those loads,
// once in about 12 steps.  With one segment and 8 residues a window, loaded as
// each walk needed them, some walk of the wave waited in nearly every step:
// 400,000 walks of the log-normal X-drop workload 2.4 -> 1.0 ms, 100,000 local
// walks of up to 500 residues 0.64 -> 0.36 ms.
template <bool LOCAL>
__global__ __launch_bounds__(kTbThreads) void k_traceback_linear(LinArgs a)
{
    constexpr int R = kLinR;
    constexpr int RUNW = kTraceSeg * kLinRec / 4;
    __shared__ uint32_t stage[kTbThreads * (2 * RUNW + 1)];
    uint32_t *run = stage + threadIdx.x * (2 * RUNW + 1);
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.starts[0] + a.counts[0])   // class 0 ends the list
        return;
    const uint32_t tid = glb(a.list)[k];
    const DpTask T = a.tasks[tid];
    DpOut o = a.out[tid];
    const uint8_t PA_GLOBAL *qs = glb_addr<const uint8_t>(T.q_off);
    const uint8_t PA_GLOBAL *ts = glb_addr<const uint8_t>(T.t_off);
    const uint8_t *trg =
        a.trace + (glb(a.trace_off)[tid] -
                   (a.trace_base ? *glb(a.trace_base) : 0ull));
    // position of row i - 1: pass p, lane l, half h, row r of the half;
    // byte offsets within one task's trace fit in 32 bits
    const uint32_t qlen = T.qlen, tlen = T.tlen;
    const uint32_t last = (qlen - 1) / kLinRows;
    const uint32_t pass_bytes = (uint32_t)lin_pass_bytes(tlen);
    constexpr uint32_t RUN = kTraceSeg * kLinRec;
    int i = o.q_end, j = o.t_end;   // an empty local alignment: 0, 0
    const uint32_t i1 = i > 0 ? (uint32_t)i - 1u : 0u;
    const int rr = (int)(i1 % kLinRows);
    int l = rr / (2 * R), h = (rr / R) & 1, r = rr % R;
    uint32_t pbase = i1 / kLinRows * pass_bytes;
    uint32_t seg_bytes =
        (i1 / kLinRows < last ? 64u : lin_last_lanes(qlen)) * RUN;
    int matches = 0, cols = 0, runs = 0, prev = 0;   // prev: last gap's row
    bool more = i > 0 && j > 0;
    while (more) {
        const int seg = (j + 2 * l + h - 1) / (int)kTraceSeg;
        const uint32_t off =
            pbase + (uint32_t)seg * seg_bytes + (uint32_t)l * RUN;
        // generic pointers: vector-struct loads from the global address
        // space do not compile
        const uint4 *s1 = (const uint4 *)(trg + off);
        const uint4 *s0 = (const uint4 *)(trg + (seg ? off - seg_bytes : off));
        uint4 x[RUNW / 2];
#pragma unroll
        for (int q = 0; q < RUNW / 4; ++q) {
            x[q] = s0[q];
            x[RUNW / 4 + q] = s1[q];
        }
        // residues i - 16 .. i - 1 and j - 16 .. j - 1, the next one on top
        // (those before a sequence's start lie in the store and are not used)
        static_assert(kWalkRes == 16, "two words of residues");
        uint64_t q0 = lin_load8(qs + i - 16), q1 = lin_load8(qs + i - 8);
        uint64_t t0 = lin_load8(ts + j - 16), t1 = lin_load8(ts + j - 8);
#pragma unroll
        for (int q = 0; q < RUNW / 2; ++q) {
            run[4 * q + 0] = x[q].x;
            run[4 * q + 1] = x[q].y;
            run[4 * q + 2] = x[q].z;
            run[4 * q + 3] = x[q].w;
        }
        const int tb = (seg - 1) * (int)kTraceSeg;   // step of the first record
        const int lw = l, iw = i - 16 > 0 ? i - 16 : 0;
        const int jw = j - 16 > 0 ? j - 16 : 0;
        for (;;) {
            const int at = j + 2 * l + h - 1 - tb;
            if (at < 0)
                break;
            const uint32_t word = run[at * 2 + (r >> 3)];
            const int c =
                (int)(word >> (8 * (2 * (r & 1) + h) + 2 * ((r & 7) >> 1))) & 3;
            if (LOCAL && c == 3) {
                more = false;   // restart
                break;
            }
            ++cols;
            if (c >= 2) {
                matches += (q1 ^ t1) >> 56 == 0;
                prev = 0;
            } else {
                runs += prev != c + 1;
                prev = c + 1;   // 1 horizontal, 2 vertical
            }
            if (c != 1) {
                --j;
                t1 = (t1 << 8) | (t0 >> 56);
                t0 <<= 8;
            }
            if (c != 0) {
                --i;
                q1 = (q1 << 8) | (q0 >> 56);
                q0 <<= 8;
                if (--r < 0) {
                    r = R - 1;
                    h ^= 1;
                    if (h && --l < 0) {
                        l = 63;
                        pbase -= pass_bytes;
                        seg_bytes = 64 * RUN;
                    }
                }
            }
            if (i <= iw || j <= jw || l != lw)
                break;
        }
        more = more && i > 0 && j > 0;
    }
    // border: a single gap run to the origin
    if (LOCAL) {
        ;   // an alignment starts with a diagonal step
    } else if (i > 0) {
        cols += i;
        runs += prev != 2;
        i = 0;
    } else if (j > 0) {
        cols += j;
        runs += prev != 1;
        j = 0;
    }
    o.q_beg = i;
    o.t_beg = j;
    o.matches = matches;
    o.cols = cols;
    o.gap_opens = runs;
    a.out[tid] = o;
}

// Score-only and traced local modes, and the global one (traced).  The int32
// run has the same grid (its boundary rows are the workgroups' own): all tasks
// of a batch may need it, and where none does its workgroups end at once.
// 3,000 traced pairs of homologs of 3,000 residues: with a wave per CU 70 ms,
// now 26; 100,000 pairs without such a task 1.69 ms either way.
hipError_t launch_dp_linear(const LinArgs &a, bool local, bool trace, int grid,
                            hipStream_t s)
{
    if (a.pipe_slots)
        hipLaunchKernelGGL(k_lin_passes, dim3(1), dim3(256), 0, s, a);
    if (!local) {
        hipLaunchKernelGGL(k_nw_linear, dim3(grid), dim3(64), 0, s, a);
    } else if (trace) {
        hipLaunchKernelGGL(k_sw_linear<true>, dim3(grid), dim3(64), 0, s, a);
        hipLaunchKernelGGL(k_sw_linear_rerun<true>, dim3(grid), dim3(64), 0, s,
                           a);
    } else {
        hipLaunchKernelGGL(k_sw_linear<false>, dim3(grid), dim3(64), 0, s, a);
        hipLaunchKernelGGL(k_sw_linear_rerun<false>, dim3(grid), dim3(64), 0,
                           s, a);
    }
    return hipGetLastError();
}

// one-wave workgroups of a mode's kernel that fit a CU
int dp_linear_occupancy(bool local, bool trace)
{
    static int n[3] = {0, 0, 0};
    const int i = !local ? 0 : trace ? 1 : 2;
    if (!n[i]) {
        int k = 0;
        if (i == 0)
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&k, k_nw_linear, 64,
                                                         0);
        else if (i == 1)
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &k, k_sw_linear<true>, 64, 0);
        else
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &k, k_sw_linear<false>, 64, 0);
        n[i] = k > 0 ? k : 1;
    }
    return n[i];
}

hipError_t launch_traceback_linear(const LinArgs &a, bool local,
                                   uint32_t ntasks, hipStream_t s)
{
    if (!ntasks)
        return hipSuccess;
    const dim3 g((ntasks + kTbThreads - 1) / kTbThreads), b(kTbThreads);
    if (local)
        hipLaunchKernelGGL(k_traceback_linear<true>, g, b, 0, s, a);
    else
        hipLaunchKernelGGL(k_traceback_linear<false>, g, b, 0, s, a);
    return hipGetLastError();
}

}  // namespace pa
