// pa_internal.h -- structures shared by the HIP kernels and the host side of
// libpastis_hip.so.  Not part of the public ABI (include/pastis_hip.h).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/pastis_hip.h"

namespace pa {

// Pointers into global memory.  Pointers that reach a kernel inside an
// argument struct or as a stored address are generic, and generic accesses
// compile to flat instructions, which also count against the LDS wait
// counter; casting them to the global address space gives global_load /
// global_store instead.
#ifndef PA_GLOBAL   // the CPU emulation build of the tests defines it empty
#define PA_GLOBAL __attribute__((address_space(1)))
#endif
// Waves per SIMD a kernel's register allocation must allow.
#ifndef PA_WAVES_PER_EU   // the CPU emulation build of the tests: empty
#define PA_WAVES_PER_EU(n) __attribute__((amdgpu_waves_per_eu(n)))
#endif
// Makes a wave-uniform integer opaque to the optimiser (no instruction): it
// is then kept in a scalar register and not folded into the code using it.
#ifndef PA_OPAQUE   // the CPU emulation build: a general register
#define PA_OPAQUE(x) asm volatile("" : "+s"(x))
#endif
template <class T> __device__ inline T PA_GLOBAL *glb(T *p)
{
    return (T PA_GLOBAL *)p;
}
template <class T> __device__ inline T PA_GLOBAL *glb_addr(uint64_t a)
{
    return (T PA_GLOBAL *)(uintptr_t)a;
}

// Residue codes 0..24 are real letters; code 25 is the sentinel used for the
// DP's column 0 and for columns past the end of the streamed sequence.  Its
// profile entries are -128, strictly below any real score.
constexpr int kAlpha = 25;
constexpr int kSentinel = 25;
constexpr int kProfChars = 26;
// Sentinels ahead of the first sequence of a store: the walks' window of
// kWalkRes residues that end at a cell starts up to kWalkRes - 1 bytes before
// a sequence, the other kernels' windows up to 7.
constexpr int kWalkRes = 16;
constexpr size_t kSeqPad = 64;
static_assert(kSeqPad >= kWalkRes, "walk windows stay in the store");

// One DP task: the row (V, lanes) and column (H, streamed) sequence spans.
struct DpTask {
    uint64_t q_off;   // first residue of the row span in the sequence store
    uint64_t t_off;   // first residue of the column span
    uint32_t qlen;    // rows
    uint32_t tlen;    // columns
    uint32_t id;      // output slot
    uint32_t flags;
};
static_assert(sizeof(DpTask) == 32, "DpTask layout");

// Output of a DP task: score and end cell (1-based DP coordinates, i.e. the
// exclusive 0-based end), plus traceback statistics when traced.
struct DpOut {
    int32_t score;
    int32_t q_end, t_end;     // rows / columns consumed at the end cell
    int32_t q_beg, t_beg;     // traceback start (filled by the traceback)
    int32_t matches, cols, gap_opens;
};
static_assert(sizeof(DpOut) == 32, "DpOut layout");

// Task flags
constexpr uint32_t kTaskSat = 1u;  // int16 saturated, needs the int32 re-run

// Profile matrices: 32x32 int8, row = row-sequence code, column = column
// code, -128 outside the 25x25 alphabet.  The DP kernels build their query
// profiles from the one of their mode: the score (untraced), 4*score+2
// (traced local) or 4*score+2, +1 on the diagonal (traced global: a
// diagonal step between equal residues carries tag 3).  Byte offsets inside
// the device copy of the scoring matrix, after the plain 32x32 table.
//
// The kernels with 8 rows per lane (rows_nib) hold 4-bit query profiles:
// kPmatNib gives score - nib_min in 0..15 (0 outside the alphabet), and
// the kernel adds nib_min (untraced) or 4*nib_min + 2 (traced) back; their
// global traces tag every diagonal step 2 and the traceback compares the
// residues for identities.  They need a matrix whose scores over the 25x25
// alphabet span at most 16 values with a negative minimum (BLOSUM62: -4 ..
// 11); with any other matrix the context runs their 4-row counterparts.
constexpr size_t kPmatUntraced = 1024, kPmatLocal = 2048, kPmatGlobal = 3072,
                 kPmatNib = 4096;
// Profiles of the linear-gap kernels (k_dp_linear.h), two tables each, for
// the two rows of a profile byte.  Traced: the same nibble n as n << 2, and n
// rotated to bits 6, 7, 0, 1; score only: n and n << 4.
constexpr int kPmatRot = 5120, kPmatPair = 7168;
// After them: the best score of each code (32 uint32, ResBound), then for
// ASCII and for code input the residue code and the k-mer letter of each byte
// (k_encode).
constexpr int kTabBest = 9216, kTabEnc = kTabBest + 128;
constexpr size_t kPmatBytes = kTabEnc + 4 * 256;
// Global task whose scores are bounded by the residue bound below (no cell
// exceeds min over the two spans of the sum of each residue's best score),
// small enough for the traced int16 kernels.
constexpr uint32_t kTaskBounded = 2u;

// Residue bound of a sequence store: pre[k] = sum over the residues of the
// sequence that holds residue k, up to and with k, of max(0, best score of
// that code against any code).  Only the affine kernels ask for it (null
// otherwise).
struct ResBound {
    uint64_t base;          // device address of the store's first residue
    const uint32_t *pre;
};

// Arguments of the wavefront DP kernels.
struct DpArgs {
    const uint8_t *codes;      // sequence store
    const DpTask *tasks;
    const uint32_t *list;      // task indices of this launch
    const uint32_t *count;     // device: number of entries in list
    uint32_t *queue;           // device: work-queue head (zeroed before launch)
    const int8_t *mat;         // 32x32 scores
    const uint32_t *pmat;      // profile matrix of the mode (kPmat* below)
    DpOut *out;
    uint8_t *trace;            // trace store (traced kernels)
    const uint64_t *trace_off; // per task byte offset into trace
    const uint64_t *trace_base;// device: offset of the chunk's first task
                               // (chunks sized on the GPU), or null
    int32_t *bnd;              // per-workgroup boundary rows (multi-pass)
    uint32_t bnd_stride;       // int32 entries per workgroup
    uint32_t *sat_list;        // tasks that saturated (int16 kernels)
    uint32_t *sat_count;
    uint8_t *tflags;           // and their flag, 1
    unsigned long long *reruns;// and their number (pa_stats.rerun_pairs)
    int32_t gap_open, gap_ext;
    uint32_t chunk;            // most tasks claimed per queue atomic (>= 1)
    int32_t nib_min;           // 4-bit profiles: the score of nibble 0
};

// Arguments of the traceback kernel.
struct TbArgs {
    const uint8_t *codes;
    const DpTask *tasks;
    const uint32_t *list;
    const uint32_t *count;
    const uint8_t *trace;
    const uint64_t *trace_off;
    const uint64_t *trace_base;   // as DpArgs::trace_base
    DpOut *out;
    int local;
};

// The four row classes in one launch (dp_one_launch).
struct DpAllArgs {
    DpArgs cls[4];
};
struct TbAllArgs {
    TbArgs tb;                 // without list and count
    const uint32_t *list[8];   // bins, the longest class first
    const uint32_t *count[8];
    int bins;                  // 4 (no int32 bins) or 8
};

// DP kernel shapes: L lanes per task (G = 64 / L tasks per wave, one per
// L-lane group) and R rows per lane per half, so a pass covers 2RL rows and
// longer tasks take several passes linked by a boundary row.  Every shape
// runs any row count; the kernels are compiled for these six.
constexpr int kShapes = 6;
constexpr int kShapeL16R4 = 0, kShapeL16R8 = 1, kShapeL64R4 = 2,
              kShapeL64R8 = 3, kShapeL32R8 = 4, kShapeL8R8 = 5;
__host__ __device__ constexpr int shape_rows(int sh)
{
    return sh == kShapeL16R4 || sh == kShapeL64R4 ? 4 : 8;
}
__host__ __device__ constexpr int shape_lanes(int sh)
{
    return sh == kShapeL64R4 || sh == kShapeL64R8 ? 64
           : sh == kShapeL32R8                    ? 32
           : sh == kShapeL8R8                     ? 8
                                                  : 16;
}
// task slots (boundary rows) of a one-wave DP workgroup
__host__ __device__ constexpr int shape_slots(int sh)
{
    return 64 / shape_lanes(sh);
}
// 4-bit query profiles: the shapes with 8 rows per lane
__host__ __device__ constexpr bool rows_nib(int R) { return R == 8; }
// the shape that replaces a 4-bit-profile shape when the matrix does not
// fit 4 bits (same rows per pass where one exists)
__host__ __device__ constexpr int shape_byte_fallback(int sh)
{
    return sh == kShapeL16R8   ? kShapeL16R4
           : sh == kShapeL64R8 ? kShapeL64R4
           : sh == kShapeL32R8 ? kShapeL64R4
           : sh == kShapeL8R8  ? kShapeL16R4
                               : sh;
}

// DP row classes: a task's class is the first c with qlen <= edge[c] (class
// 3 takes the rest), and each class has its kernel shape.  Narrow groups
// keep more of a wave busy on short tasks (the wavefront's fill and drain
// take 2L steps per pass and the last pass rounds the rows up to 2RL); wide
// ones cost fewer boundary rows, profile builds and loop overhead per cell
// on long tasks.  The defaults (kDefaultShapes) are
//   0: qlen <= 128:  8 lanes x 8 rows, 128 rows per pass (one pass);
//   1: qlen <= 256: 16 lanes x 8 rows, 256 rows per pass (one pass);
//   2: qlen <= 512: 32 lanes x 8 rows, 512 rows per pass (one pass);
//   3: longer:      64 lanes x 8 rows, 1024 rows per pass.
struct DpShapes {
    uint32_t edge[3];
    uint8_t shape[4];
};
constexpr DpShapes kDefaultShapes = {{128, 256, 512},
                                     {kShapeL8R8, kShapeL16R8, kShapeL32R8,
                                      kShapeL64R8}};

// The classes may share a launch (DpAllArgs): the default shapes, with one
// pass for every task below the last class.  A task of several passes keeps
// its boundary row at workgroup * slots + slot, and the slots per workgroup
// differ between classes: were there such tasks in two classes, workgroups
// that are in different classes at the same time would share rows.
inline bool dp_one_launch(const DpShapes &sh)
{
    for (int c = 0; c < 4; ++c)
        if (sh.shape[c] != kDefaultShapes.shape[c] ||
            (c < 3 && sh.edge[c] > 2u * (uint32_t)shape_rows(sh.shape[c]) *
                                       (uint32_t)shape_lanes(sh.shape[c])))
            return false;
    return true;
}

__host__ __device__ inline int dp_class(uint32_t qlen, const DpShapes &sh)
{
    return qlen <= sh.edge[0] ? 0
           : qlen <= sh.edge[1] ? 1
           : qlen <= sh.edge[2] ? 2
                                : 3;
}
__host__ __device__ inline int rows_per_lane(uint32_t qlen, const DpShapes &sh)
{
    return shape_rows(sh.shape[dp_class(qlen, sh)]);
}
__host__ __device__ inline int lanes_per_task(uint32_t qlen, const DpShapes &sh)
{
    return shape_lanes(sh.shape[dp_class(qlen, sh)]);
}

// Trace layout of a task traced with R rows per lane and L lanes: pass after
// pass; a pass holds one record of R bytes (2R 4-bit codes) per (step,
// active lane).  Full passes have L active lanes and tlen + 2L - 1 steps;
// the last pass has nact lanes and tlen + 2*(nact-1) + 1 steps.  Steps are
// grouped in segments of kTraceSeg: a segment holds, lane after lane, the
// kTraceSeg consecutive records of each lane, so a traceback that walks
// back along a lane reads neighbouring bytes (8R contiguous bytes per lane
// and segment) while one step of the DP still writes L records in a few
// cache lines.  A pass is padded to whole segments.
constexpr uint32_t kTraceSeg = 8;

// Threads (one traceback walk each) per workgroup of the traceback kernels.
constexpr int kTbThreads = 256;

__host__ __device__ inline uint32_t trace_last_lanes(uint32_t qlen, int R,
                                                     int L)
{
    const uint32_t rows = 2u * (uint32_t)R * (uint32_t)L;
    const uint32_t rem = qlen - ((qlen - 1) / rows) * rows;
    return (rem + 2u * R - 1u) / (2u * R);
}

// steps of a pass rounded up to whole segments
__host__ __device__ inline uint32_t trace_seg_steps(uint32_t steps)
{
    return (steps + kTraceSeg - 1u) / kTraceSeg * kTraceSeg;
}

__host__ __device__ inline uint64_t trace_bytes(uint32_t qlen, uint32_t tlen,
                                                int R, int L)
{
    const uint32_t rows = 2u * (uint32_t)R * (uint32_t)L;
    const uint32_t full = (qlen - 1) / rows;
    const uint32_t nl = trace_last_lanes(qlen, R, L);
    return ((uint64_t)full * trace_seg_steps(tlen + 2u * L - 1u) * L +
            (uint64_t)trace_seg_steps(tlen + 2u * (nl - 1u) + 1u) * nl) *
           (uint64_t)R;
}

// Record index (in units of R bytes) of (pass p, step t >= 1, lane).
__host__ __device__ inline uint64_t trace_rec(uint32_t qlen, uint32_t tlen,
                                              int R, int L, uint32_t p,
                                              uint32_t t, uint32_t lane)
{
    const uint32_t rows = 2u * (uint32_t)R * (uint32_t)L;
    const uint32_t full = (qlen - 1) / rows;
    const uint32_t nact = p < full ? (uint32_t)L : trace_last_lanes(qlen, R, L);
    const uint32_t seg = (t - 1u) / kTraceSeg, off = (t - 1u) % kTraceSeg;
    return (uint64_t)p * trace_seg_steps(tlen + 2u * L - 1u) * L +
           (uint64_t)seg * nact * kTraceSeg + lane * kTraceSeg + off;
}

// Linear-gap global alignment (k_dp_linear.h).  A lane holds 2 * kLinR rows.
// A class has a lane count per task (lin_lanes); as many tasks as fit sit
// side by side in a wave.  Tasks take the narrowest class that holds their
// rows, those of more than kLinRows rows the last class in several passes.
// The counts are those where the tasks of a wave change (64 / L), so few
// lanes stay idle: rows are rounded up to 32, lanes to 60 .. 64 per wave.
constexpr int kLinR = 16;
constexpr int kLinClasses = 16;
// class whose tasks' passes run on a wave each, one behind the other: more
// than one pass, and columns enough to hide the 200 or so by which a pass
// follows the one before.  It pays where a few long tasks outlast the rest; a
// batch of nothing but such tasks fills the chip without it and loses by its
// waits, the more the fewer columns.  Score only, one wave a task / pipelined:
// 2,000 tasks of 20,000 rows x 512 columns 4.9 / 9.4 ms, x 1,024 8.8 / 13.3,
// x 2,048 16.4 / 20.8, x 4,096 31.3 / 35.5; of 5,000 rows x 2,048 4.8 / 4.9,
// of 2,200 x 20,000 25.2 / 24.4.
constexpr int kLinPipe = kLinClasses - 1;
constexpr uint32_t kLinPipeCols = 2048;
constexpr int kLinRows = 2 * kLinR * 64;
// bytes of one trace record: the 2-bit codes of a lane's rows at one step
constexpr int kLinRec = kLinR / 2;
// 8-byte words of a boundary row besides its columns (two a word)
constexpr uint32_t kLinBndPad = 80;
// Scores from which a result counts as re-run in int32 (what 16 bits hold),
// and the lower ones from which the linear-gap kernels run a task again: their
// maximum is taken in half-float order, below 0x7c00, and a step adds at most
// 14 to a score.
constexpr int kSat = 32766, kSatTraced = 8190;
constexpr int kLinSat = 0x7c00 - 16, kLinSatTraced = 0x7c00 / 4 - 16;

__host__ __device__ inline int lin_lanes(int cls)
{
    return cls < 10 ? cls + 1
           : cls == 10 ? 12
           : cls == 11 ? 16
           : cls == 12 ? 21
           : cls == 13 ? 32
                       : 64;
}
// pipe: the pipelined class may be used
__host__ __device__ inline int lin_class(uint32_t qlen, uint32_t tlen,
                                         bool pipe)
{
    if (pipe && qlen > kLinRows && tlen >= kLinPipeCols)
        return kLinPipe;
    const uint32_t need = (qlen + 2u * kLinR - 1u) / (2u * kLinR);
    return need <= 10   ? (int)need - 1
           : need <= 12 ? 10
           : need <= 16 ? 11
           : need <= 21 ? 12
           : need <= 32 ? 13
                        : 14;
}
// lanes of the last pass
__host__ __device__ inline uint32_t lin_last_lanes(uint32_t qlen)
{
    const uint32_t rem = qlen - (qlen - 1) / kLinRows * kLinRows;
    return (rem + 2u * kLinR - 1u) / (2u * kLinR);
}
// Trace layout as above with R = kLinR, L = 64 (a class's lane count does not
// enter: a task with fewer rows than a pass has one pass of its own lanes),
// and records of kLinRec bytes.  Offsets are multiples of 64.
__host__ __device__ inline uint64_t lin_pass_bytes(uint32_t tlen)
{
    return (uint64_t)trace_seg_steps(tlen + 127u) * 64u * kLinRec;
}
__host__ __device__ inline uint64_t lin_trace_bytes(uint32_t qlen,
                                                    uint32_t tlen)
{
    const uint32_t nl = lin_last_lanes(qlen);
    return (uint64_t)((qlen - 1) / kLinRows) * lin_pass_bytes(tlen) +
           (uint64_t)trace_seg_steps(tlen + 2u * (nl - 1u) + 1u) * nl *
               kLinRec;
}
// Arguments of the linear-gap kernels: the task list, class after class (the
// last class first), and per class its start, length and work-queue head.
struct LinArgs {
    const DpTask *tasks;
    const uint32_t *list;
    const uint32_t *starts;
    const uint32_t *counts;
    uint32_t *queues;
    const int8_t *mat;          // scoring matrix and profile tables (kPmat*)
    DpOut *out;
    uint8_t *trace;
    const uint64_t *trace_off;
    const uint64_t *trace_base; // as DpArgs::trace_base
    // boundary rows of bnd_words words: pipe_slots for pipelined passes (0:
    // no task is in their class), then one per workgroup
    uint64_t *bnd;
    uint32_t bnd_words;
    uint32_t pipe_slots;
    uint64_t *prog;             // per slot: progress (zeroed), then values
    uint32_t *pipe_start;       // first item of each pipelined task
    uint32_t *pipe_items;
    uint32_t *sat_list, *sat_count, *sat_queue;   // int32 re-runs (local)
    uint8_t *tflags;
    unsigned long long *reruns;
    int32_t gap, nib_min;
};
hipError_t launch_dp_linear(const LinArgs &a, bool local, bool trace, int grid,
                            hipStream_t s);
int dp_linear_occupancy(bool local, bool trace);
hipError_t launch_traceback_linear(const LinArgs &a, bool local,
                                   uint32_t ntasks, hipStream_t s);

// X-drop extension task: one seed of one pair.
struct XdTask {
    uint64_t h_off, v_off;     // column (H) and row (V) sequence starts
    uint32_t nh, nv;           // lengths
    uint32_t beg_h, beg_v;     // seed start
    uint32_t id;               // output slot
    uint32_t pad;              // kXdInvalid: no extension, empty extents
};
static_assert(sizeof(XdTask) == 40, "XdTask layout");
// The pair names a sequence that is not loaded or its seed does not fit.
constexpr uint32_t kXdInvalid = 1u;

// Residues an item (direction dir of a task: 0 left, 1 right) can extend over
// at most, the shorter of its two segments; 0 for an invalid task.
__host__ __device__ inline uint32_t xd_reach(const XdTask &t, int dir,
                                             int seed_len)
{
    if (t.pad & kXdInvalid)
        return 0;
    const uint32_t h = dir ? t.nh - t.beg_h - (uint32_t)seed_len : t.beg_h;
    const uint32_t v = dir ? t.nv - t.beg_v - (uint32_t)seed_len : t.beg_v;
    return h < v ? h : v;
}

// X-drop work items of a batch small enough for 16 lanes per item, the reach
// (xd_reach) from which an item of a larger batch gets 16 lanes, and the items
// up to which a batch is split that way.
constexpr uint64_t kXdSmall = 65536, kXdSplit = (uint64_t)4 << 20;
constexpr uint32_t kXdLong = 512;
constexpr int64_t kXdBandItems = 120000;

// Which kernel takes an item first.  Sixteen lanes per item take a fifth of the
// time per anti-diagonal that one lane takes (0.2 us; a lane 0.7 in an idle
// chip, 3 beside five other waves), at four times the instructions.
//   small16: all items of a small batch.
//   split: the items of a larger one that may extend far, on the second stream
//     beside the others.  Not in a full chip, where the instructions count and
//     the longest item ends before the rest does.
//   sorted: the one-lane kernel's items (with all_band: the band kernel's) in
//     falling order of their reach, so that the grid does not end on long ones.
//   all_band: 16 lanes and wide bands for all items.
// 16 lanes hold 14 columns.  A gap costs -xdrop_gap and an extension ends X below
// its best, so a band spans up to 2 X / -xdrop_gap columns (9 as called, 49 as
// documented).  Bands of 10 fit in nearly every item.  Wider ones outgrow 16
// columns in the more items the smaller the gap for the same ratio (bands end
// on mismatches too): from 2 X = g (12 + g) on, g = -xdrop_gap, the band kernels
// are faster whatever the batch, and up to 120,000 items, divided by what is
// missing to that line, they are faster since the chip is not full.  The stage
// in ms, one lane unsorted / split / all_band:
//   X, gap      line    60,000 pairs        150,000             400,000
//    66, -11    0.52    6.27  3.53  3.42     7.63  3.77  8.22    9.47  5.49 20.47
//   100, -11    0.79    8.48  5.49  3.90    11.25  6.51  9.25   16.53 11.23 23.95
//    40, -5     0.94   10.65  7.06  4.13    16.35 12.53  9.71   29.94 25.36 24.98
//   130, -11    1.03   11.57  8.66  4.12    18.76 15.76  9.93   37.52 33.73 25.71
//    20, -2     1.43   11.21  8.94  4.46    18.72 16.19 10.82   39.24 35.06 27.90
// (log-normal workload, 30 % homologs, four items a pair).  As called:
//   pairs          one lane, unsorted   sorted   split   16 lanes
//       16,384                   4.42     5.11    2.30      1.43
//       65,536                   5.73     6.03    2.42      2.27
//      262,144                   7.14     7.02    4.07      5.41
//      800,000                  10.99     9.75    9.25
//    1,200,000                  13.67    12.28   12.94
//    5,000,000                  42.70    40.08   45.22
struct XdRoute {
    bool small16, split, sorted, all_band;
};
inline XdRoute xd_route(uint64_t ni, int xdrop, int xdrop_gap, int xd_coop,
                        int xd_wave)
{
    XdRoute r{};
    if (xd_coop)
        return r;
    const int64_t g = -(int64_t)xdrop_gap;
    const bool thin = xdrop / g <= 5;
    if (!thin && (xd_wave != 1 || xdrop > 30000))
        return r;
    const int64_t line = g * (12 + g), missing = line - 2 * (int64_t)xdrop;
    r.small16 = thin && ni <= kXdSmall;
    r.all_band = !thin && (missing <= 0 ||
                           (int64_t)ni * missing <= kXdBandItems * line);
    r.split = !r.small16 && !r.all_band && ni <= kXdSplit;
    r.sorted = !r.small16;
    return r;
}

// Seed extension result; the left direction writes beg_*, score_left,
// cells_left, flags_left and the right direction the other half.
struct XdOut {
    int32_t beg_h, beg_v, end_h, end_v;
    int32_t score_left, score_right;
    uint32_t cells_left, cells_right;
    uint16_t flags_left, flags_right;  // 1 band too wide, 2 budget exhausted
    uint32_t pad;
};
static_assert(sizeof(XdOut) == 40, "XdOut layout");

// Launchers (k_dp.hip, k_xdrop.hip, k_misc.hip).
hipError_t launch_dp(int shape, bool local, bool trace, bool i16,
                     const DpArgs &a, int grid, hipStream_t s);
// Traceback of tasks traced by the DP kernels of one shape; stage: copy each
// lane run (8R bytes) the walk enters into LDS with wide loads instead of
// loading one byte per step.
hipError_t launch_dp_all(const DpAllArgs &a, bool local, bool trace, bool i16,
                         int grid, hipStream_t s);
hipError_t launch_traceback_all(const TbAllArgs &a, bool stage, uint32_t ntasks,
                                hipStream_t s);
hipError_t launch_traceback(const TbArgs &a, int shape, bool stage, int grid,
                            hipStream_t s);
// X-drop with one 16-lane row of a wave per work item (k_xdrop_coop.hip);
// items whose band outgrows 16 columns are appended to ovf_list.
hipError_t launch_xdrop_coop(const XdTask *tasks, const uint32_t *list,
                             const uint32_t *count, uint32_t *queue,
                             const int8_t *mat, int gap, int xdrop,
                             int seed_len, XdOut *out, uint32_t *ovf_list,
                             uint32_t *ovf_count, int grid, hipStream_t s);
int xdrop_coop_occupancy();
// X-drop with 16 lanes per work item (k_xdrop_wave.hip), for the items whose
// band outgrew the per-lane kernel's LDS rings: a window of 128 columns, 256
// (wide 1) or 512 (wide 2); items whose band outgrows the window are appended
// to ovf_list.
hipError_t launch_xdrop_wave(const XdTask *tasks, const uint32_t *list,
                             const uint32_t *count, uint32_t *queue,
                             const int8_t *mat, int gap, int xdrop,
                             int seed_len, XdOut *out, uint32_t *ovf_list,
                             uint32_t *ovf_count, int grid, int wide,
                             hipStream_t s);
int xdrop_wave_occupancy(int wide);

// Workgroups of one DP kernel variant (of a kernel shape) that fit on one
// CU (occupancy).
int dp_occupancy(int shape, bool local, bool trace, bool i16);
// Same for the LDS-ring X-drop kernel with `ring` slots per lane (the
// variant launch_xdrop picks for these X-drop and gap values).
int xdrop_occupancy(int ring, int xdrop, int gap);

hipError_t launch_xdrop(const XdTask *tasks, const uint32_t *list,
                        const uint32_t *count, uint32_t *queue,
                        const int8_t *mat, int gap, int xdrop, int seed_len,
                        int32_t *scratch, int cap, XdOut *out,
                        uint32_t *ovf_list, uint32_t *ovf_count, int grid,
                        int ring, hipStream_t s);

}  // namespace pa
