// k_dp_linear.h -- traced global alignment under a linear gap cost, included
// by k_dp.hip (namespace pa).
//
// With open > ext a gap is never extended: H >= E gives H + open > E + ext,
// so every gap residue costs `open` (= g) and the three-state recurrence is
//   H(i,j) = max(H(i-1,j-1) + s, H(i-1,j) + g, H(i,j-1) + g).
// In the frame H'(i,j) = H(i,j) - g (i + j) gap steps cost nothing and a
// diagonal step scores s' = s - 2g, which for this path's matrices is 0 ..
// 15 (lin_ok).  H' grows along rows and columns by 0 .. 15 per step, so the
// kernel keeps differences only:
//   u(i,j) = H'(i,j) - H'(i-1,j),   v(i,j) = H'(i,j) - H'(i,j-1)
//   z = max(s', u(i,j-1), v(i-1,j)),  u(i,j) = z - v(i-1,j),
//   v(i,j) = z - u(i,j-1),            score = sum of u(i,n) + g (m + n).
// No value leaves 0 .. 15, whatever the lengths, so no task needs int32; one
// register per row holds the state (three in the affine kernel) and the
// borders are zeros, so lanes ahead of their first column or behind their
// last one compute on without a test: with s' = 0 outside the columns the
// state stays zero before the first and stays u(i,n) after the last.
//
// Values are held as 4 * value + tag (tag 2 diagonal, 1 up, 0 left; v
// carries tag 1, u tag 0), two cells per register as in k_dp.  All are
// non-negative int16 below 0x7c00, where int16 order is half-float order, so
// one v_pk_maximum3_f16 takes the maximum of three cells (half denormals are
// kept: the kernels run with the default mode).  A cell pair then is
//   z = max3(s, v, u); z1 = (z & ~3) | 1; u = z1 - v; v = z1 - u
// (no half borrows, so plain 32-bit subtractions), the tag of z is its
// 2-bit trace code.
//
// What bounds it: VALU issue.  A step of 16 row pairs takes 125 instructions,
// 7.8 per pair (4 recurrence, 2 score unpack, 1.25 code packing), against
// about 22 for the affine kernel, which carries E, F and H.  400,000 pairs
// of the log-normal X-drop workload (30 % homologs): 16.6 ms of traced DP in
// the affine kernels' eight launches (2.9 of them int32, for spans whose
// all-gap path leaves int16), 5.0 ms here; the walks 2.8 ms beside each
// other on two streams, 2.4 ms here.
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

// Profile: kProfChars codes x two strips x 64 lanes x 16 nibbles (two
// words).  Each lane holds the scores of its own 32 rows whatever the lanes
// per task, so the layout is the same for all classes; lanes of a wave read
// consecutive 8-byte words (no bank conflict).  Byte k of word w: row 8w + k
// in bits 2-5, row 8w + 4 + k in bits 6, 7, 0, 1.
constexpr int kLinProfWords = kProfChars * 2 * 64 * 2;

// One class: L lanes per task, 64 / L tasks side by side in a wave.  MULTI:
// the class of 64 lanes, whose tasks may take several passes.
template <bool MULTI>
__device__ inline void lin_class_run(const LinArgs &a, uint32_t *prof,
                                     int cls)
{
    constexpr int R = kLinR;        // rows per half
    const int L = MULTI ? 64 : lin_lanes(cls);
    const int G = MULTI ? 1 : 64 / L;
    constexpr uint64_t kFillRes = 0x1919191919191919ull;   // kSentinel
    constexpr uint64_t kFillBnd = 0x0101010101010101ull;   // v = 0
    static_assert(kSentinel == 0x19, "window fill");
    const int lane = threadIdx.x & 63;
    const int gl = lane % L, grp = lane / L;   // grp G: lanes left over
    const bool fl = gl == 0;
    const uint32_t count = a.counts[cls];
    if (count == 0)
        return;
    const uint32_t PA_GLOBAL *list = glb(a.list) + a.starts[cls];
    uint8_t PA_GLOBAL *bnd =
        glb(a.bnd) + (size_t)blockIdx.x * a.bnd_stride;
    uint8_t *plds = (uint8_t *)prof;
    const uint32_t lane8 = (uint32_t)lane * 8u;
    const LinConst C;
    for (;;) {
        // every lane takes part in the atomic (only lane 0 adds)
        uint32_t k0 = atomicAdd(a.queues + cls, lane == 0 ? (uint32_t)G : 0u);
        k0 = __builtin_amdgcn_readfirstlane(k0);
        if (k0 >= count)
            break;
        const uint32_t k = k0 + (uint32_t)grp;
        const bool valid = grp < G && k < count;
        const uint32_t tid = list[valid ? k : k0];
        DpTask T = a.tasks[tid];
        if (!valid)
            T.qlen = T.tlen = 0;
        const uint8_t PA_GLOBAL *qs = glb_addr<const uint8_t>(T.q_off);
        const uint8_t PA_GLOBAL *ts = glb_addr<const uint8_t>(T.t_off);
        const int qlen = (int)T.qlen, tlen = (int)T.tlen;
        uint8_t PA_GLOBAL *tr =
            glb(a.trace) + (glb(a.trace_off)[tid] -
                            (a.trace_base ? *glb(a.trace_base) : 0ull));
        const int npass =
            MULTI ? (int)__builtin_amdgcn_readfirstlane(
                        (qlen + kLinRows - 1) / kLinRows)
                  : 1;
        uint32_t total = 0;   // this lane's rows of sum u(i, tlen), times 4

        for (int p = 0; p < npass; ++p) {
            const int i0 = p * kLinRows;
            const int row0 = i0 + 2 * R * gl;
            __syncthreads();
            // ---- query profile of this lane's 32 rows -------------------
            // word (strip, w): rows of group A (8w .. 8w+3) from the
            // shifted table, of group B (8w+4 .. 8w+7) from the rotated one
#pragma unroll 1
            for (int sw = 0; sw < 4; ++sw) {
                const int ra = row0 + 8 * sw;   // strip sw / 2, word sw % 2
                if (!__ballot(ra < qlen))
                    continue;
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
                        const uint4 *src = (const uint4 *)(a.pmat +
                                                           g * 256 + qc * 8);
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
                uint32_t *dst = prof + (sw >> 1) * 128 + 2 * lane + (sw & 1);
#pragma unroll
                for (int c = 0; c < kProfChars; ++c)
                    dst[c * 256] = xs[c];
            }
            if (MULTI && p > 0)
                __threadfence();
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
            uint8_t PA_GLOBAL *trp =
                tr + (uint64_t)p * lin_pass_bytes((uint32_t)tlen) +
                (uint32_t)gl * (kTraceSeg * kLinRec);

            uint32_t u[R];
#pragma unroll
            for (int r = 0; r < R; ++r)
                u[r] = 0;
            // residues: lane's columns of block b are 8b + 1 - 2 gl .. + 7
            auto res_raw = [&](int blk) -> uint64_t {
                const int i = 8 * blk - 2 * gl;
                return i > -8 && i < tlen ? lin_load8(ts + i) : 0ull;
            };
            auto res_win = [&](uint64_t raw, int blk) {
                return lin_window(raw, 8 * blk - 2 * gl, tlen, kFillRes);
            };
            // boundary row of the previous pass: byte 126 + column
            auto bnd_raw = [&](int blk) -> uint64_t {
                return 8 * blk < tlen ? lin_load8(bnd + 127 + 8 * blk) : 0ull;
            };
            auto bnd_win = [&](uint64_t raw, int blk) {
                return lin_window(raw, 8 * blk, tlen, kFillBnd);
            };
            uint64_t wc = res_win(res_raw(0), 0), wraw = res_raw(1);
            uint64_t bc = kFillBnd, braw = 0;
            if (MULTI && p > 0) {
                bc = bnd_win(bnd_raw(0), 0);
                braw = bnd_raw(1);
            }
            // LDS address of the lo strip's words of the current column;
            // the hi strip reads the column before it
            auto paddr = [&](uint32_t code) { return code * 1024u + lane8; };
            uint32_t ac = paddr((uint32_t)wc & 0xffu);
            uint2 lw = *(const uint2 *)(plds + ac);
            uint2 hw = *(const uint2 *)(plds + paddr(kSentinel) + 512);
            uint32_t vin = 0x00010001u;
            if (MULTI && p > 0 && fl)
                vin = 0x00010000u | ((uint32_t)bc & 0xffu);

            auto run_blocks = [&](auto first_pass) {
                constexpr bool FIRST = decltype(first_pass)::value;
                for (int blk = 0; blk < nblk; ++blk) {
                    const uint64_t wn = res_win(wraw, blk + 1);
                    wraw = res_raw(blk + 2);
                    uint64_t bn = 0;
                    if (!FIRST) {
                        bn = bnd_win(braw, blk + 1);
                        braw = bnd_raw(blk + 2);
                    }
                    const bool store = blk < st_blk;
                    uint64_t bout = 0;
                    uint32_t rec[4];
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
                        uint32_t z[R], vv = vin;
#pragma unroll
                        for (int w = 0; w < 2; ++w) {
                            const uint32_t lo = w ? lw.y : lw.x;
                            const uint32_t hi = w ? hw.y : hw.x;
                            uint32_t s[8];
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                // byte q of both words, twice in each half
                                const uint32_t sel =
                                    (uint32_t)q * 0x0101u |
                                    (uint32_t)(4 + q) * 0x01010000u;
                                const uint32_t b =
                                    __builtin_amdgcn_perm(hi, lo, sel);
                                s[q] = (b & C.smask) | C.tag2;
                                s[q + 4] = ((b >> 4) & C.smask) | C.tag2;
                            }
#pragma unroll
                            for (int q = 0; q < 8; ++q) {
                                const int r = 8 * w + q;
                                z[r] = lin_max3(s[q], vv, u[r]);
                                const uint32_t z1 =
                                    (z[r] & C.zmask) | C.tag1;
                                const uint32_t un = z1 - vv;
                                vv = z1 - u[r];
                                u[r] = un;
                            }
                        }
                        // codes: byte 2 (r % 2) + half of word r / 8, bits
                        // 2 ((r % 8) / 2)
#pragma unroll
                        for (int w = 0; w < 2; ++w) {
                            uint32_t y[4];
#pragma unroll
                            for (int q = 0; q < 4; ++q)
                                y[q] = __builtin_amdgcn_perm(
                                    z[8 * w + 2 * q + 1], z[8 * w + 2 * q],
                                    0x06040200u);
                            const uint32_t x01 =
                                (y[0] & C.m2) | ((y[1] << 2) & ~C.m2);
                            const uint32_t x23 =
                                (y[2] & C.m2) | ((y[3] << 2) & ~C.m2);
                            rec[2 * (st & 1) + w] =
                                (x01 & C.m4) | ((x23 << 4) & ~C.m4);
                        }
                        if (st & 1) {
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
                        if (MULTI)   // v of the pass's last row (lane 63)
                            bout |= (uint64_t)((vv >> 16) & 0xffu)
                                    << (8 * st);
                        // row above of the next step: lo from the hi half
                        // of the lane before, hi from the own lo half; the
                        // first lane of a task takes the border
                        uint32_t first = 0x00010000u;
                        if (!FIRST)
                            first = ((st < 7
                                          ? (uint32_t)(bc >>
                                                       (8 * ((st + 1) & 7)))
                                          : (uint32_t)bn) &
                                     0xffu)
                                    << 16;
                        const uint32_t sh = (uint32_t)lin_lane_up<MULTI>(
                            (int)first, (int)vv, fl);
                        vin = __builtin_amdgcn_alignbit(vv, sh, 16);
                        lw = lwn;
                        hw = hwn;
                        ac = an;
                    }
                    if (MULTI && more_passes && lane == 63)
                        *(uint64_t PA_GLOBAL *)(bnd + 8 * (size_t)blk) = bout;
                    trp += seg_bytes;
                    wc = wn;
                    bc = bn;
                }
            };
            if (!MULTI || p == 0)
                run_blocks(std::true_type{});
            else
                run_blocks(std::false_type{});

            // this pass's rows of the last column
            const int nlo = qlen - row0, nhi = nlo - R;
            uint32_t sum = 0;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t m = (r < nlo ? 0x0000ffffu : 0u) |
                                   (r < nhi ? 0xffff0000u : 0u);
                sum += u[r] & m;
            }
            total += (sum & 0xffffu) + (sum >> 16);
        }
        // suffix sums within the task: its first lane ends with the total
        for (int off = 1; off < L; off <<= 1) {
            const uint32_t x = __shfl(total, lane + off);
            total += gl + off < L ? x : 0u;
        }
        total = __shfl(total, lane - gl);
        DpOut o = {};
        o.score = (int)(total >> 2) + a.gap * (qlen + tlen);
        o.q_beg = o.q_end = qlen;
        o.t_beg = o.t_end = tlen;
        // every lane of a task stores the same result (no lane-0 branch
        // closes the loop)
        if (valid)
            a.out[tid] = o;
    }
}

// All classes in one launch, the longest rows first: a workgroup that finds
// a class drained goes on with the next one, so no class waits for the last
// tasks of another, and a batch takes one launch.
__global__ __launch_bounds__(64) void k_nw_linear(LinArgs a)
{
    __shared__ uint32_t prof[kLinProfWords];
    lin_class_run<true>(a, prof, kLinClasses - 1);
    for (int cls = kLinClasses - 2; cls >= 0; --cls)
        lin_class_run<false>(a, prof, cls);
}

// Traceback over the 2-bit codes, one walk per thread, the tasks of all
// classes (longest first).  The records of one lane in one segment (64
// contiguous, 64-byte aligned bytes) are copied into LDS when the walk
// enters them.
__global__ __launch_bounds__(kTbThreads) void k_traceback_linear(LinArgs a)
{
    constexpr int R = kLinR;
    constexpr int RUNW = kTraceSeg * kLinRec / 4;
    __shared__ uint32_t stage[kTbThreads * (RUNW + 1)];
    uint32_t *run = stage + threadIdx.x * (RUNW + 1);
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
    int i = (int)qlen, j = (int)tlen;
    const int rr = (int)((qlen - 1) % kLinRows);
    int l = rr / (2 * R), h = (rr / R) & 1, r = rr % R;
    uint32_t pbase = last * pass_bytes;
    uint32_t seg_bytes = lin_last_lanes(qlen) * RUN;
    uint32_t cur = 0xffffffffu;
    ResWin qwin{qs}, twin{ts};
    int matches = 0, cols = 0, runs = 0, prev = 0;   // prev: last gap's row
    while (i > 0 && j > 0) {
        const uint32_t t1 = (uint32_t)(j + 2 * l + h) - 1u;
        const uint32_t off =
            pbase + (t1 / kTraceSeg) * seg_bytes + (uint32_t)l * RUN;
        if (off != cur) {
            cur = off;
            // generic pointer: vector-struct loads from the global address
            // space do not compile
            const uint4 *src = (const uint4 *)(trg + off);
#pragma unroll
            for (int q = 0; q < RUNW / 4; ++q) {
                const uint4 x = src[q];
                run[4 * q + 0] = x.x;
                run[4 * q + 1] = x.y;
                run[4 * q + 2] = x.z;
                run[4 * q + 3] = x.w;
            }
        }
        const uint32_t word = run[(t1 % kTraceSeg) * 2 + (uint32_t)(r >> 3)];
        const int c =
            (int)(word >> (8 * (2 * (r & 1) + h) + 2 * ((r & 7) >> 1))) & 3;
        ++cols;
        if (c >= 2) {
            matches += qwin.at(i - 1) == twin.at(j - 1);
            prev = 0;
        } else {
            runs += prev != c + 1;
            prev = c + 1;   // 1 horizontal, 2 vertical
        }
        j -= c != 1;
        if (c != 0) {
            --i;
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
    }
    // border: a single gap run to the origin
    if (i > 0) {
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

hipError_t launch_nw_linear(const LinArgs &a, int grid, hipStream_t s)
{
    hipLaunchKernelGGL(k_nw_linear, dim3(grid), dim3(64), 0, s, a);
    return hipGetLastError();
}

int nw_linear_occupancy()
{
    static int n = 0;
    if (!n) {
        int k = 0;
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&k, k_nw_linear, 64, 0);
        n = k > 0 ? k : 1;
    }
    return n;
}

hipError_t launch_traceback_linear(const LinArgs &a, uint32_t ntasks,
                                   hipStream_t s)
{
    if (!ntasks)
        return hipSuccess;
    hipLaunchKernelGGL(k_traceback_linear,
                       dim3((ntasks + kTbThreads - 1) / kTbThreads),
                       dim3(kTbThreads), 0, s, a);
    return hipGetLastError();
}

}  // namespace pa
