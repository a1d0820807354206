// k_kmer.hip -- k-mer candidate generation on the GPU (pa_kmer_candidates).
//
// The reference builds the candidate pairs as the sparse product C = A * A^T
// of the sequence-by-k-mer matrix A (generate_A, src/kmer/KmerOps.cpp:92-245)
// under the KmerIntersectLoc semiring (inc/sr.hpp:30-117) with CombBLAS.
// Here the same overlap matrix is a sort-based join:
//   1. every k-mer occurrence of a sequence set becomes (code, seq << 16 |
//      offset); codes of k-mers with a letter outside the alphabet are
//      marked invalid (add_kmers, KmerOps.cpp:31-87);
//   2. a stable radix sort by code groups equal k-mers, occurrences in
//      (sequence, offset) order inside a group; the sorted occurrences and
//      the group table of a set are kept for later calls;
//   3. for each k-mer group, the products are the (column occurrence, row
//      occurrence) pairs, column occurrences outer: the order in which a
//      column-by-column SpGEMM adds them;
//   4. a stable radix sort of the products by (column, row) lines up the
//      products of each pair in that order, and one pass over each run
//      folds them: count = products (ushort), score = max self score,
//      first = the first product's offsets, second = the last one's (the
//      default (0, 0) for a single product).
// The symmetric pruning of the similarity search (src/sim_search.cpp:
// 173-187, 403-412, 569-578) is applied to the products, the k-mer
// threshold prune of DistPWRunner.cpp:48-54 to the folded pairs.  Output:
// pa_pair in column-major order (column, then row).
//
// All of this is integer sort / scan / gather work bound by HBM traffic.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "pa_ctx.h"

using namespace pa;

namespace pa {

// The k-mer alphabets of inc/Alphabet.hpp:66-254: each letter of the
// 25-letter protein order maps to a representative; codes are given to
// representatives in the order they first appear while scanning that order
// (Alphabet::init, src/Alphabet.cpp:31-51).
struct KmerAlphabet {
    uint8_t code[kAlpha];    // alphabet code of each residue code
    int16_t self[kAlpha];    // BLOSUM62 self score of each code's representative
    int size;
};

struct KmerGroups {         // occurrences [start, end) of each code
    Buf start, end, code, cost;
    uint64_t n = 0;
    bool built = false;
};

struct KmerSet {            // sorted occurrences of one sequence set
    Buf keys, vals;
    uint64_t nocc = 0;      // valid occurrences
    KmerGroups groups[2];   // all codes; those of more than one occurrence
    uint64_t gen = ~0ull;   // sequence generation they were built for
    int k = 0, stride = 0, alph = -1;
};

struct KmerState {
    KmerSet rows, cols;
    Buf slots, keys_a, vals_a, pcount, poff, gscr, pkey, pval, pkey2, pval2,
        heads, runid, rstart, keep, kpos, tmp, cnt, cand;
    // the last call's result, reused by an identical call (the count / copy
    // protocol of pa_kmer_candidates)
    pa_kmer_config last{};
    uint64_t last_cb = 0, last_ce = 0, last_gen = ~0ull, last_n = 0;
    bool have_last = false;
    uint64_t *host = nullptr;   // pinned words for values read back
};

void kmer_free(KmerState *k)
{
    if (!k)
        return;
    for (KmerSet *s : {&k->rows, &k->cols}) {
        release(s->keys);
        release(s->vals);
        for (KmerGroups &g : s->groups)
            for (Buf *b : {&g.start, &g.end, &g.code, &g.cost})
                release(*b);
    }
    for (Buf *b : {&k->slots, &k->keys_a, &k->vals_a, &k->pcount, &k->poff,
                   &k->gscr, &k->pkey, &k->pval, &k->pkey2, &k->pval2, &k->heads,
                   &k->runid, &k->rstart, &k->keep, &k->kpos, &k->tmp,
                   &k->cnt, &k->cand})
        release(*b);
    if (k->host)
        hipHostFree(k->host);
    delete k;
}

}  // namespace pa

namespace {

const char kProtein[] = "ARNDCQEGHILKMFPSTWYVBZX*J";
const int8_t kSelfB62[kAlpha] = {4, 5, 6, 6, 9, 5, 5, 6, 8, 4, 4, 5, 5,
                                 6, 7, 4, 5, 11, 7, 4, 4, 4, -1, 1, 4};
// letter groups of the reduced alphabets; the first letter represents them
const char *const kGroups[6][8] = {
    {nullptr},
    {"DENQ", "FWY", "ILMV", "KR", "ST", nullptr},               // murphy10
    {"EKQR", "IV", "LY", "AM", "HT", "DNS", "GP", nullptr},     // dssp10
    {"AEFIKLMQRVW", nullptr},                                   // gbmr10
    {"EKRQ", "DSN", "HC", "IV", "WYF", "LM", nullptr},          // td10
    {"KREDQN", "ILV", "STA", nullptr},                          // diamond
};

bool make_alphabet(int id, KmerAlphabet &a)
{
    if (id < 0 || id > 5)
        return false;
    auto idx = [](char ch) { return (int)(std::strchr(kProtein, ch) - kProtein); };
    int rep[kAlpha];
    for (int i = 0; i < kAlpha; ++i)
        rep[i] = i;
    for (int g = 0; kGroups[id][g]; ++g)
        for (const char *p = kGroups[id][g]; *p; ++p)
            rep[idx(*p)] = idx(kGroups[id][g][0]);
    int code_of_rep[kAlpha];
    std::fill(code_of_rep, code_of_rep + kAlpha, -1);
    int next = 0;
    for (int i = 0; i < kAlpha; ++i) {
        if (code_of_rep[rep[i]] < 0)
            code_of_rep[rep[i]] = next++;
        a.code[i] = (uint8_t)code_of_rep[rep[i]];
        a.self[a.code[i]] = kSelfB62[rep[i]];
    }
    a.size = next;
    return true;
}

// smallest b with 2^b - 1 >= v (v > 0)
int bits_for(uint64_t v)
{
    int b = 1;
    while (b < 64 && ((1ull << b) - 1ull) < v)
        ++b;
    return b;
}

constexpr int kTB = 256;

inline unsigned nblocks(uint64_t n, unsigned per = kTB)
{
    uint64_t b = (n + per - 1) / per;
    return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(b, 1u << 20));
}

// Occurrence slot t -> (code or invalid, seq << 16 | offset).  slots[i] is
// the first slot of sequence i (exclusive scan of its k-mer positions).
__global__ void k_kmer_extract(const uint8_t *__restrict__ kc,
                               const uint64_t *__restrict__ seq_addr,
                               uint64_t base_addr,
                               const uint64_t *__restrict__ slots,
                               uint64_t nseq, uint64_t nslots, int k,
                               int stride, KmerAlphabet alph,
                               uint32_t invalid, uint32_t *__restrict__ keys,
                               uint64_t *__restrict__ vals,
                               unsigned long long *nbad)
{
    uint64_t bad = 0;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
         t < nslots; t += (uint64_t)gridDim.x * blockDim.x) {
        // sequence of the slot: last i with slots[i] <= t
        uint64_t lo = 0, hi = nseq - 1;
        while (lo < hi) {
            const uint64_t mid = (lo + hi + 1) / 2;
            if (slots[mid] <= t)
                lo = mid;
            else
                hi = mid - 1;
        }
        const uint64_t off = (t - slots[lo]) * (uint64_t)stride;
        const uint8_t *p = kc + (seq_addr[lo] - base_addr) + off;
        uint32_t code = 0;
        bool ok = true;
        for (int j = 0; j < k; ++j) {
            const int x = p[j];
            if (x >= kAlpha) {
                ok = false;
                break;
            }
            code = code * (uint32_t)alph.size + alph.code[x];
        }
        keys[t] = ok ? code : invalid;
        vals[t] = (lo << 16) | off;
        bad += ok ? 0 : 1;
    }
    if (bad)
        atomicAdd(nbad, (unsigned long long)bad);
}

// heads[i] = 1 where a new code group (multi: of more than one occurrence)
// starts (i < n)
__global__ void k_group_heads(const uint32_t *__restrict__ keys, uint64_t n,
                              bool multi, uint32_t *__restrict__ heads)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        heads[i] = (i == 0 || keys[i] != keys[i - 1]) &&
                           (!multi || (i + 1 < n && keys[i + 1] == keys[i]))
                       ? 1u
                       : 0u;
}

// self score of a k-mer code (sum over its letters' representatives)
__device__ inline int code_cost(uint32_t code, const KmerAlphabet &al, int k)
{
    int cost = 0;
    for (int j = 0; j < k; ++j) {
        cost += al.self[code % (uint32_t)al.size];
        code /= (uint32_t)al.size;
    }
    return cost;
}

// group g (inclusive scan value - 1 from its head on) -> start, end, code,
// self score
__global__ void k_group_table(const uint32_t *__restrict__ keys,
                              const uint32_t *__restrict__ heads,
                              const uint64_t *__restrict__ incl, uint64_t n,
                              bool multi, KmerAlphabet alph, int k,
                              uint64_t *__restrict__ gstart,
                              uint64_t *__restrict__ gend,
                              uint32_t *__restrict__ gcode,
                              int16_t *__restrict__ gcost)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t key = keys[i];
        const bool first = i == 0 || keys[i - 1] != key;
        const bool last = i + 1 == n || keys[i + 1] != key;
        if (multi && first && last)
            continue;
        const uint64_t g = incl[i] - 1;
        if (first) {
            gstart[g] = i;
            gcode[g] = key;
            gcost[g] = (int16_t)code_cost(key, alph, k);
        }
        if (last)
            gend[g] = i + 1;
    }
}

__device__ inline uint64_t lower_bound_u32(const uint32_t *a, uint64_t n,
                                           uint32_t v)
{
    uint64_t lo = 0, hi = n;
    while (lo < hi) {
        const uint64_t mid = (lo + hi) / 2;
        if (a[mid] < v)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// first index in vals[lo, hi) whose sequence is >= s
__device__ inline uint64_t lower_bound_seq(const uint64_t *vals, uint64_t lo,
                                           uint64_t hi, uint64_t s)
{
    while (hi - lo > 4) {
        const uint64_t mid = (lo + hi) / 2;
        if ((vals[mid] >> 16) < s)
            lo = mid + 1;
        else
            hi = mid;
    }
    if (lo == hi)
        return lo;
    // the last four (most groups hold no more) in loads that do not wait for
    // one another
    uint64_t v[4];
    for (int i = 0; i < 4; ++i)
        v[i] = vals[lo + i < hi ? lo + i : hi - 1] >> 16;
    uint64_t n = 0;
    for (int i = 0; i < 4; ++i)
        n += lo + i < hi && v[i] < s ? 1 : 0;
    return lo + n;
}

// Groups by the number of their products: one thread emits the products of a
// small group, a block those of a large one, all blocks together those of a
// huge one.
constexpr uint64_t kSmallGroup = 64, kLargeGroup = 1u << 16;
// Under PA_SYM_UPPER a group of few column occurrences counts only the
// products that are kept: for a column sequence the row occurrences of lower
// (global) sequences, a prefix of the row group.  Most groups hold a single
// occurrence, whose only product is with itself: 60,000 sequences give 35
// million products of which 7.9 million are kept, and all of them were sorted.  Larger groups count all products and drop some.
constexpr uint32_t kTriCols = 32;

// symmetric pruning of the product of (global) row R and column C
__device__ inline bool keep_product(int sym, uint64_t R, uint64_t C)
{
    if (sym == PA_SYM_UPPER)
        return C > R;
    const bool ro = R & 1, co = C & 1;
    return sym != PA_SYM_EVEN_ODD ||
           !(R == C || (R > C ? (ro ^ co) : !(ro ^ co)));
}

// A short group of a set that is both rows and columns under one base: its
// occurrences are read at once, and only the products that are kept count.  All
// but one in forty groups of more than one occurrence are short (60,000
// sequences); the searches of the general path are chains of dependent loads.
// 32-bit compares, since these kernels are bound by their instructions: joining
// and emitting 3.7 million groups took 112 and 219 us with 64-bit ones (and a
// division per letter of the code) and every wave waiting for its groups that
// are not short; now 88 and 136 us.
constexpr uint32_t kShort = 4;

struct ShortGroup {
    uint64_t v[kShort];
    uint32_t seq[kShort];
    bool col[kShort], row[kShort];
    int sym;

    template <class A>
    __device__ ShortGroup(const A &a, uint64_t gs, uint64_t ge) : sym(a.sym)
    {
        const uint32_t n = (uint32_t)(ge - gs);
        for (uint32_t i = 0; i < kShort; ++i)
            v[i] = a.cvals[i < n ? gs + i : gs];
        for (uint32_t i = 0; i < kShort; ++i) {
            seq[i] = (uint32_t)(v[i] >> 16);
            row[i] = i < n;
            col[i] = i < n && seq[i] >= a.c_begin && seq[i] < a.c_end;
        }
    }

    // column occurrence x and row occurrence y make a product
    __device__ bool product(uint32_t x, uint32_t y) const
    {
        const uint32_t c = seq[x], r = seq[y];
        const bool odd = (r ^ c) & 1;
        const bool keep = sym == PA_SYM_UPPER ? c > r
                          : sym == PA_SYM_NONE
                              ? true
                              : r != c && !(r > c ? odd : !odd);
        return col[x] && row[y] && keep;
    }
};

struct JoinGroup {
    uint64_t ca, ra;           // first column / row occurrence
    uint32_t cn, rn;           // and their numbers
};

// Per column group g: the column occurrences in [c_begin, c_end) and the
// row group with the same code; products = both counts multiplied, or the
// kept ones (kTriCols).
struct JoinArgs {
    const uint64_t *cgstart, *cgend;   // column groups
    const uint32_t *cgcode;
    const uint64_t *cvals;
    uint64_t cngroups;
    const uint32_t *rkeys;     // row occurrences (sorted keys)
    uint64_t rnocc;
    bool shared;               // rows and columns are one set
    bool one_set;              // and of one base
    uint64_t c_begin, c_end;
    JoinGroup *grp;            // written where emit_group reads it
    uint64_t *pcount;
    const uint64_t *rvals;
    int sym;                   // pa_symmetric
    uint64_t up_off;           // row sequences kept: below c + up_off
    uint32_t *large, *huge;    // group lists and their lengths
    uint32_t *nlarge, *nhuge;
    uint32_t tile;             // groups a block takes (group_tile)
};

// Row occurrences of rvals[ra, ra + rn) whose sequence lies below the column
// sequence c in global indices (up_off = col_base - row_base, wrapping).
__device__ inline uint64_t rows_below(const uint64_t *rvals, uint64_t ra,
                                      uint64_t rn, uint64_t c, uint64_t up_off)
{
    const int64_t lim = (int64_t)(c + up_off);
    if (lim <= 0)
        return 0;
    if (rn == 1)
        return (rvals[ra] >> 16) < (uint64_t)lim ? 1 : 0;
    return lower_bound_seq(rvals, ra, ra + rn, (uint64_t)lim) - ra;
}

// products of group g = occurrences [gs, ge) of the column set
__device__ inline uint64_t join_group(const JoinArgs &a, uint64_t g,
                                      uint64_t gs, uint64_t ge)
{
    const uint64_t c0 = lower_bound_seq(a.cvals, gs, ge, a.c_begin);
    const uint64_t c1 = lower_bound_seq(a.cvals, c0, ge, a.c_end);
    uint64_t r0 = gs, r1 = ge;
    if (!a.shared) {
        const uint32_t code = a.cgcode[g];
        r0 = lower_bound_u32(a.rkeys, a.rnocc, code);
        r1 = lower_bound_u32(a.rkeys, a.rnocc, code + 1);
    }
    uint64_t np = (c1 - c0) * (r1 - r0);
    if (np && a.sym == PA_SYM_UPPER && c1 - c0 <= kTriCols) {
        np = 0;
        for (uint64_t x = c0; x < c1; ++x)
            np += rows_below(a.rvals, r0, r1 - r0, a.cvals[x] >> 16, a.up_off);
    }
    if (np)
        a.grp[g] = {c0, r0, (uint32_t)(c1 - c0), (uint32_t)(r1 - r0)};
    if (np > kLargeGroup)
        a.huge[atomicAdd(a.nhuge, 1u)] = (uint32_t)g;
    else if (np > kSmallGroup)
        a.large[atomicAdd(a.nlarge, 1u)] = (uint32_t)g;
    return np;
}

// A block takes a tile of groups, a thread each; the few that are not short
// are listed and counted at the end, so that their searches fill waves of
// their own instead of holding up every wave.  Tiles of kGroupTile groups, or
// fewer where those would leave CUs idle (group_tile): 300 sequences in 11
// letters, unlike bases, two column blocks 1.25 ms, 0.88 before, now 0.74.
constexpr uint32_t kGroupTile = 2048;

uint32_t group_tile(const pa_ctx *c, uint64_t groups)
{
    const uint64_t rounds = groups / ((uint64_t)c->ncu * 4u * kTB);
    return (uint32_t)std::min<uint64_t>(kGroupTile,
                                        kTB * std::max<uint64_t>(1, rounds));
}

__global__ void __launch_bounds__(kTB) k_join_count(JoinArgs a)
{
    __shared__ uint16_t list[kGroupTile];
    __shared__ uint32_t nlist;
    for (uint64_t g0 = (uint64_t)blockIdx.x * a.tile; g0 < a.cngroups;
         g0 += (uint64_t)gridDim.x * a.tile) {
        if (threadIdx.x == 0)
            nlist = 0;
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < a.tile; i += kTB) {
            const uint64_t g = g0 + i;
            if (g >= a.cngroups)
                break;
            const uint64_t gs = a.cgstart[g], ge = a.cgend[g];
            if (a.one_set && ge - gs <= kShort) {
                const ShortGroup sg(a, gs, ge);
                uint32_t np = 0;
                for (uint32_t x = 0; x < kShort; ++x)
                    for (uint32_t y = 0; y < kShort; ++y)
                        np += sg.product(x, y) ? 1 : 0;
                a.pcount[g] = np;
            } else {
                list[atomicAdd(&nlist, 1u)] = (uint16_t)i;
            }
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < nlist; i += kTB) {
            const uint64_t g = g0 + list[i];
            a.pcount[g] = join_group(a, g, a.cgstart[g], a.cgend[g]);
        }
        __syncthreads();
    }
}

struct EmitArgs {
    const uint64_t *poff;     // exclusive scan of products per group
    uint64_t ngroups;
    const JoinGroup *grp;
    const int16_t *gcost;
    const uint64_t *cvals, *rvals;
    const uint64_t *cgstart, *cgend;
    bool one_set;
    int sym;                  // pa_symmetric
    uint64_t row_base, col_base, c_begin, c_end;
    int rbits;
    uint64_t keymax;
    uint64_t *pkey, *pval;
    unsigned long long *ndrop;
    const uint64_t *pcount;
    uint64_t up_off;
    const uint32_t *large, *huge, *nlarge, *nhuge;
    uint32_t tile;
};

// Products [t0, t1) of group g (column occurrence outer), every step-th: each
// to put(its place from poff[g] on, key, value); returns the number dropped.
template <class Put>
__device__ inline uint64_t emit_group(const EmitArgs &a, uint64_t g, uint64_t t0,
                                      uint64_t t1, uint64_t step, Put put)
{
    const JoinGroup j = a.grp[g];
    const uint64_t ca = j.ca, ra = j.ra, rn = j.rn, off = a.poff[g];
    const uint32_t cn = j.cn;
    const uint64_t cost = (uint16_t)a.gcost[g];
    const bool tri = a.sym == PA_SYM_UPPER && cn <= kTriCols;
    uint64_t drop = 0, bi = 0, first = 0, width = 0;
    if (tri)
        width = rows_below(a.rvals, ra, rn, a.cvals[ca] >> 16, a.up_off);
    for (uint64_t t = t0; t < t1; t += step) {
        uint64_t ai;
        if (tri) {   // products first .. first + width of column bi
            while (t - first >= width) {
                first += width;
                ++bi;
                width = rows_below(a.rvals, ra, rn, a.cvals[ca + bi] >> 16,
                                   a.up_off);
            }
            ai = t - first;
        } else {
            bi = t / rn;
            ai = t % rn;
        }
        const uint64_t cv = a.cvals[ca + bi], rv = a.rvals[ra + ai];
        const uint64_t c = cv >> 16, r = rv >> 16;
        const bool keep = keep_product(a.sym, r + a.row_base, c + a.col_base);
        put(off + t, keep ? ((c - a.c_begin) << a.rbits) | r : a.keymax,
            ((rv & 0xffffull) << 48) | ((cv & 0xffffull) << 32) | cost);
        drop += keep ? 0 : 1;
    }
    return drop;
}

template <class Put>
__device__ inline void emit_short(const EmitArgs &a, uint64_t g, uint64_t gs,
                                  uint64_t ge, Put put)
{
    uint64_t at = a.poff[g];
    const uint64_t cost = (uint16_t)a.gcost[g];
    const ShortGroup sg(a, gs, ge);
    for (uint32_t x = 0; x < kShort; ++x)
        for (uint32_t y = 0; y < kShort; ++y)
            if (sg.product(x, y)) {
                const uint64_t cv = sg.v[x], rv = sg.v[y];
                put(at++, (((cv >> 16) - a.c_begin) << a.rbits) | rv >> 16,
                    ((rv & 0xffffull) << 48) | ((cv & 0xffffull) << 32) | cost);
            }
}

// Groups of up to kSmallGroup products, a thread each, as in k_join_count.
// The short ones of kTB neighbouring groups fill neighbouring places, which
// are gathered in LDS and written in order; places of other groups are left
// out there.  Before, the group of every eighth product was searched among all
// groups: 1.06 ms per block of 17 million products, most of them dropped; now
// 136 us for the 3.9 million that are kept.
constexpr uint32_t kStage = 1024;

__global__ void __launch_bounds__(kTB) k_emit_small(EmitArgs a)
{
    __shared__ uint64_t key[kStage], val[kStage];
    __shared__ uint16_t list[kGroupTile];
    __shared__ uint32_t nlist;
    uint64_t drop = 0;
    for (uint64_t t0 = (uint64_t)blockIdx.x * a.tile; t0 < a.ngroups;
         t0 += (uint64_t)gridDim.x * a.tile) {
        if (threadIdx.x == 0)
            nlist = 0;
        for (uint32_t i0 = 0; i0 < a.tile && t0 + i0 < a.ngroups;
             i0 += kTB) {
            const uint64_t g0 = t0 + i0, g = g0 + threadIdx.x;
            const uint64_t g1 = g0 + kTB < a.ngroups ? g0 + kTB : a.ngroups;
            const uint64_t base = a.poff[g0], n = a.poff[g1] - base;
            const bool stage = n <= kStage;
            if (stage)
                for (uint32_t i = threadIdx.x; i < n; i += kTB)
                    key[i] = ~0ull;
            __syncthreads();
            const uint64_t np = g < a.ngroups ? a.pcount[g] : 0;
            if (np > 0 && np <= kSmallGroup) {
                const uint64_t gs = a.cgstart[g], ge = a.cgend[g];
                if (a.one_set && ge - gs <= kShort)
                    emit_short(a, g, gs, ge,
                               [&](uint64_t at, uint64_t k, uint64_t v) {
                                   if (stage) {
                                       key[at - base] = k;
                                       val[at - base] = v;
                                   } else {
                                       a.pkey[at] = k;
                                       a.pval[at] = v;
                                   }
                               });
                else
                    list[atomicAdd(&nlist, 1u)] = (uint16_t)(i0 + threadIdx.x);
            }
            __syncthreads();
            if (stage)
                for (uint32_t i = threadIdx.x; i < n; i += kTB)
                    if (key[i] != ~0ull) {
                        a.pkey[base + i] = key[i];
                        a.pval[base + i] = val[i];
                    }
            __syncthreads();
        }
        for (uint32_t i = threadIdx.x; i < nlist; i += kTB) {
            const uint64_t g = t0 + list[i];
            drop += emit_group(a, g, 0, a.pcount[g], 1,
                               [&](uint64_t at, uint64_t k, uint64_t v) {
                                   a.pkey[at] = k;
                                   a.pval[at] = v;
                               });
        }
        __syncthreads();
    }
    if (drop)
        atomicAdd(a.ndrop, (unsigned long long)drop);
}

__global__ void __launch_bounds__(kTB) k_emit_large(EmitArgs a)
{
    auto put = [&](uint64_t at, uint64_t k, uint64_t v) {
        a.pkey[at] = k;
        a.pval[at] = v;
    };
    uint64_t drop = 0;
    for (uint32_t k = blockIdx.x; k < *a.nlarge; k += gridDim.x) {
        const uint64_t g = a.large[k];
        drop += emit_group(a, g, threadIdx.x, a.pcount[g], kTB, put);
    }
    for (uint32_t k = 0; k < *a.nhuge; ++k) {
        const uint64_t g = a.huge[k];
        drop += emit_group(a, g,
                           (uint64_t)blockIdx.x * kTB + threadIdx.x,
                           a.pcount[g], (uint64_t)gridDim.x * kTB, put);
    }
    if (drop)
        atomicAdd(a.ndrop, (unsigned long long)drop);
}

__global__ void k_run_heads(const uint64_t *__restrict__ keys, uint64_t n,
                            uint32_t *__restrict__ heads)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        heads[i] = (i == 0 || keys[i] != keys[i - 1]) ? 1u : 0u;
}

__global__ void k_run_starts(const uint32_t *__restrict__ heads,
                             const uint64_t *__restrict__ incl, uint64_t n,
                             uint64_t *__restrict__ rstart)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        if (heads[i])
            rstart[incl[i] - 1] = i;
}

// Fold of one run (one candidate pair) and the k-mer threshold prune.
struct FoldArgs {
    const uint64_t *rstart;
    uint64_t nruns, nprod;
    const uint64_t *pkey, *pval;
    int rbits;
    uint64_t c_begin;
    int ckthr;
    float mosthr;
    pa_pair *cand;
    uint32_t *keep;
};

__global__ void k_fold_runs(FoldArgs a)
{
    for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
         g < a.nruns; g += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t s = a.rstart[g];
        const uint64_t e = g + 1 < a.nruns ? a.rstart[g + 1] : a.nprod;
        const uint64_t key = a.pkey[s];
        const uint64_t v0 = a.pval[s], vl = a.pval[e - 1];
        int score = (int16_t)(uint16_t)(v0 & 0xffffu);
        for (uint64_t i = s + 1; i < e; ++i) {
            const int x = (int16_t)(uint16_t)(a.pval[i] & 0xffffu);
            score = x > score ? x : score;
        }
        pa_pair p;
        p.r = (uint32_t)(key & ((1ull << a.rbits) - 1ull));
        p.c = (uint32_t)((key >> a.rbits) + a.c_begin);
        p.count = (uint16_t)(e - s);
        p.kscore = (int16_t)score;
        p.seed[0] = (uint16_t)(v0 >> 48);
        p.seed[1] = (uint16_t)(v0 >> 32);
        p.seed[2] = e - s > 1 ? (uint16_t)(vl >> 48) : 0;
        p.seed[3] = e - s > 1 ? (uint16_t)(vl >> 32) : 0;
        a.cand[g] = p;
        // DistPWRunner.cpp:48-54: count <= ckthr || score <= mosthr
        const bool prune = (int)p.count <= a.ckthr ||
                           (float)p.kscore <= a.mosthr;
        a.keep[g] = prune ? 0u : 1u;
    }
}

__global__ void k_compact(const pa_pair *__restrict__ cand,
                          const uint32_t *__restrict__ keep,
                          const uint64_t *__restrict__ pos, uint64_t n,
                          pa_pair *__restrict__ out)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        if (keep[i])
            out[pos[i]] = cand[i];
}

#define KCHK(ctx, x)                                                         \
    do {                                                                     \
        hipError_t e_ = (x);                                                 \
        if (e_ != hipSuccess)                                                \
            return fail((ctx), PA_ERR_HIP,                                   \
                        std::string(#x) + ": " + hipGetErrorString(e_));     \
    } while (0)

// inclusive scan of u32 flags into u64
int scan_flags(pa_ctx *c, KmerState *K, const uint32_t *in, uint64_t *out,
               uint64_t n, bool inclusive, hipStream_t s)
{
    size_t tmp = 0;
    if (inclusive)
        KCHK(c, hipcub::DeviceScan::InclusiveSum(nullptr, tmp, in, out, n, s));
    else
        KCHK(c, hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, in, out, n, s));
    int rc;
    if ((rc = grow(c, K->tmp, tmp)))
        return rc;
    if (inclusive)
        KCHK(c, hipcub::DeviceScan::InclusiveSum(K->tmp.p, tmp, in, out, n, s));
    else
        KCHK(c, hipcub::DeviceScan::ExclusiveSum(K->tmp.p, tmp, in, out, n, s));
    return PA_OK;
}

// Value i of src to the host's pinned words, ready after the next wait for
// the stream (a copy to pageable memory costs 20 us more).
template <class T> int d2h_start(pa_ctx *c, KmerState *K, int i, const T *src,
                                 hipStream_t s)
{
    KCHK(c, hipMemcpyAsync(&K->host[i], src, sizeof(T), hipMemcpyDeviceToHost,
                           s));
    return PA_OK;
}

template <class T> int d2h_value(pa_ctx *c, KmerState *K, T *dst, const T *src,
                                 hipStream_t s)
{
    int rc;
    if ((rc = d2h_start(c, K, 0, src, s)))
        return rc;
    KCHK(c, hipStreamSynchronize(s));
    std::memcpy(dst, &K->host[0], sizeof(T));
    return PA_OK;
}

// Sorted k-mer occurrences and group table of one loaded set.
int build_set(pa_ctx *c, KmerState *K, KmerSet &S, bool rows,
              const pa_kmer_config &kc, const KmerAlphabet &al, int kbits,
              hipStream_t s)
{
    if (S.gen == c->seq_gen && S.k == kc.k && S.stride == kc.stride &&
        S.alph == kc.alphabet)
        return PA_OK;
    int rc;
    const std::vector<uint32_t> &len = rows ? c->rlen : c->clen;
    const uint64_t nseq = len.size();
    std::vector<uint64_t> slots(nseq + 1, 0);
    for (uint64_t i = 0; i < nseq; ++i) {
        const uint64_t L = len[i];
        const uint64_t np =
            L >= (uint64_t)kc.k ? (L - kc.k) / (uint64_t)kc.stride + 1 : 0;
        slots[i + 1] = slots[i] + np;
    }
    const uint64_t nslots = slots[nseq];
    S.k = kc.k;
    S.stride = kc.stride;
    S.alph = kc.alphabet;
    S.gen = c->seq_gen;
    S.nocc = 0;
    S.groups[0].built = S.groups[1].built = false;
    if (nslots == 0)
        return PA_OK;
    if ((rc = grow(c, K->slots, (nseq + 1) * 8)) ||
        (rc = grow(c, K->keys_a, nslots * 4)) ||
        (rc = grow(c, K->vals_a, nslots * 8)) ||
        (rc = grow(c, S.keys, nslots * 4)) ||
        (rc = grow(c, S.vals, nslots * 8)) ||
        (rc = grow(c, K->cnt, 64)))
        return rc;
    KCHK(c, hipMemcpyAsync(K->slots.p, slots.data(), (nseq + 1) * 8,
                           hipMemcpyHostToDevice, s));
    KCHK(c, hipMemsetAsync(K->cnt.p, 0, 64, s));
    const uint32_t invalid = (uint32_t)((1ull << kbits) - 1ull);
    const Buf &kcb = rows ? c->rkc : c->ckc;
    const Buf &cb = rows ? c->rcodes : c->ccodes;
    hipLaunchKernelGGL(k_kmer_extract, dim3(nblocks(nslots)), dim3(kTB), 0, s,
                       P<uint8_t>(const_cast<Buf &>(kcb)),
                       P<uint64_t>(rows ? c->roffs : c->coffs),
                       (uint64_t)(uintptr_t)seq_base(cb), P<uint64_t>(K->slots), nseq,
                       nslots, kc.k, kc.stride, al, invalid,
                       P<uint32_t>(K->keys_a), P<uint64_t>(K->vals_a),
                       (unsigned long long *)K->cnt.p);
    KCHK(c, hipGetLastError());
    size_t tmp = 0;
    KCHK(c, hipcub::DeviceRadixSort::SortPairs(
                 nullptr, tmp, P<uint32_t>(K->keys_a), P<uint32_t>(S.keys),
                 P<uint64_t>(K->vals_a), P<uint64_t>(S.vals), nslots, 0, kbits,
                 s));
    if ((rc = grow(c, K->tmp, tmp)))
        return rc;
    KCHK(c, hipcub::DeviceRadixSort::SortPairs(
                 K->tmp.p, tmp, P<uint32_t>(K->keys_a), P<uint32_t>(S.keys),
                 P<uint64_t>(K->vals_a), P<uint64_t>(S.vals), nslots, 0, kbits,
                 s));
    uint64_t nbad = 0;
    if ((rc = d2h_value(c, K, &nbad, P<uint64_t>(K->cnt), s)))
        return rc;
    S.nocc = nslots - nbad;
    return PA_OK;
}

// Group table over the valid occurrences of a set; multi leaves out the codes
// that occur once.
int build_groups(pa_ctx *c, KmerState *K, KmerSet &S, bool multi,
                 const KmerAlphabet &al, hipStream_t s)
{
    KmerGroups &T = S.groups[multi];
    if (T.built)
        return PA_OK;
    T.n = 0;
    int rc;
    if (S.nocc) {
        if ((rc = grow(c, K->heads, S.nocc * 4)) ||
            (rc = grow(c, K->runid, S.nocc * 8)))
            return rc;
        hipLaunchKernelGGL(k_group_heads, dim3(nblocks(S.nocc)), dim3(kTB), 0,
                           s, P<uint32_t>(S.keys), S.nocc, multi,
                           P<uint32_t>(K->heads));
        if ((rc = scan_flags(c, K, P<uint32_t>(K->heads), P<uint64_t>(K->runid),
                             S.nocc, true, s)) ||
            (rc = d2h_value(c, K, &T.n, P<uint64_t>(K->runid) + S.nocc - 1, s)))
            return rc;
    }
    if (T.n) {
        if ((rc = grow(c, T.start, T.n * 8)) ||
            (rc = grow(c, T.end, T.n * 8)) ||
            (rc = grow(c, T.code, T.n * 4)) || (rc = grow(c, T.cost, T.n * 2)))
            return rc;
        hipLaunchKernelGGL(k_group_table, dim3(nblocks(S.nocc)), dim3(kTB), 0,
                           s, P<uint32_t>(S.keys), P<uint32_t>(K->heads),
                           P<uint64_t>(K->runid), S.nocc, multi, al, S.k,
                           P<uint64_t>(T.start), P<uint64_t>(T.end),
                           P<uint32_t>(T.code), P<int16_t>(T.cost));
        KCHK(c, hipGetLastError());
    }
    T.built = true;
    return PA_OK;
}

bool same_cfg(const pa_kmer_config &a, const pa_kmer_config &b)
{
    return a.k == b.k && a.stride == b.stride && a.alphabet == b.alphabet &&
           a.symmetric == b.symmetric && a.ckthr == b.ckthr &&
           a.mosthr == b.mosthr && a.row_base == b.row_base &&
           a.col_base == b.col_base;
}

// Runs the join for columns [cb, ce) and leaves the candidates in K->cand
// (compacted), their number in *n.
int generate(pa_ctx *c, KmerState *K, const pa_kmer_config &kc, uint64_t cb,
             uint64_t ce, uint64_t *n, hipStream_t s)
{
    int rc;
    KmerAlphabet al{};
    if (!make_alphabet(kc.alphabet, al))
        return fail(c, PA_ERR_ARG, "unknown k-mer alphabet");
    uint64_t universe = 1;
    for (int j = 0; j < kc.k; ++j)
        universe *= (uint64_t)al.size;
    if (universe >= (1ull << 31))
        return fail(c, PA_ERR_ARG, "alphabet size ^ k must stay below 2^31");
    const int kbits = bits_for(universe);   // 2^kbits - 1 >= universe
    if ((rc = build_set(c, K, K->rows, true, kc, al, kbits, s)))
        return rc;
    const bool shared = c->shared_cols;
    KmerSet &C = shared ? K->rows : K->cols;
    if (!shared && (rc = build_set(c, K, K->cols, false, kc, al, kbits, s)))
        return rc;
    KmerSet &R = K->rows;
    *n = 0;
    const uint64_t up_off = kc.col_base - kc.row_base;
    // a lone occurrence of a code meets only itself, and the symmetric rules
    // drop that: 14 million groups of 60,000 sequences become 3.7 million
    const bool multi = shared && kc.symmetric != PA_SYM_NONE && up_off == 0;
    if ((rc = build_groups(c, K, C, multi, al, s)))
        return rc;
    KmerGroups &T = C.groups[multi];
    if (T.n == 0 || R.nocc == 0 || cb >= ce)
        return PA_OK;
    const uint64_t G = T.n;
    const uint32_t tile = group_tile(c, G);
    if ((rc = grow(c, K->pcount, (G + 1) * 8)) ||
        (rc = grow(c, K->poff, (G + 1) * 8)) ||
        (rc = grow(c, K->gscr, G * 32)) || (rc = grow(c, K->cnt, 64)))
        return rc;
    uint64_t *pcount = P<uint64_t>(K->pcount);
    JoinGroup *grp = P<JoinGroup>(K->gscr);
    uint32_t *large = (uint32_t *)(grp + G), *huge = large + G;
    // counters: dropped products (u64), large and huge groups
    uint32_t *ngr = P<uint32_t>(K->cnt) + 2;
    KCHK(c, hipMemsetAsync(K->cnt.p, 0, 64, s));
    JoinArgs ja{P<uint64_t>(T.start), P<uint64_t>(T.end), P<uint32_t>(T.code),
                P<uint64_t>(C.vals), G, P<uint32_t>(R.keys), R.nocc, shared,
                shared && up_off == 0, cb, ce, grp, pcount, P<uint64_t>(R.vals),
                kc.symmetric, up_off, large, huge, ngr, ngr + 1, tile};
    hipLaunchKernelGGL(k_join_count, dim3(nblocks(G, tile)), dim3(kTB), 0, s,
                       ja);
    KCHK(c, hipGetLastError());
    {
        size_t tmp = 0;
        KCHK(c, hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, pcount,
                                                 P<uint64_t>(K->poff), G + 1,
                                                 s));
        if ((rc = grow(c, K->tmp, tmp)))
            return rc;
        // pcount[G] = 0 so that poff[G] is the total
        KCHK(c, hipMemsetAsync(pcount + G, 0, 8, s));
        KCHK(c, hipcub::DeviceScan::ExclusiveSum(K->tmp.p, tmp, pcount,
                                                 P<uint64_t>(K->poff), G + 1,
                                                 s));
    }
    if ((rc = d2h_start(c, K, 0, P<uint64_t>(K->poff) + G, s)) ||
        (rc = d2h_start(c, K, 1, (uint64_t *)ngr, s)))
        return rc;
    KCHK(c, hipStreamSynchronize(s));
    const uint64_t nprod = K->host[0];
    const uint32_t nlarge = (uint32_t)K->host[1];
    const uint32_t nhuge = (uint32_t)(K->host[1] >> 32);
    if (nprod == 0)
        return PA_OK;
    const uint64_t ncols_blk = ce - cb;
    const uint64_t nrows = c->rlen.size();
    const int rbits = bits_for(nrows);
    const int cbits = bits_for(ncols_blk);
    if (rbits + cbits > 63)
        return fail(c, PA_ERR_LIMIT, "row x column block too large");
    const uint64_t keymax = (1ull << (rbits + cbits)) - 1ull;   // unused key
    if ((rc = grow(c, K->pkey, nprod * 8)) || (rc = grow(c, K->pval, nprod * 8)) ||
        (rc = grow(c, K->pkey2, nprod * 8)) ||
        (rc = grow(c, K->pval2, nprod * 8)))
        return rc;
    EmitArgs ea{P<uint64_t>(K->poff), G, grp,
                P<int16_t>(T.cost), P<uint64_t>(C.vals), P<uint64_t>(R.vals),
                P<uint64_t>(T.start), P<uint64_t>(T.end),
                shared && up_off == 0, kc.symmetric, kc.row_base,
                kc.col_base, cb, ce, rbits,
                keymax, P<uint64_t>(K->pkey), P<uint64_t>(K->pval),
                (unsigned long long *)K->cnt.p, pcount, up_off, large, huge,
                ngr, ngr + 1, tile};
    hipLaunchKernelGGL(k_emit_small, dim3(nblocks(G, tile)), dim3(kTB), 0, s,
                       ea);
    if (nlarge || nhuge)
        hipLaunchKernelGGL(k_emit_large,
                           dim3(nhuge ? 1024u : std::min(nlarge, 1024u)),
                           dim3(kTB), 0, s, ea);
    KCHK(c, hipGetLastError());
    // the number of dropped products arrives while they are sorted
    if ((rc = d2h_start(c, K, 0, P<uint64_t>(K->cnt), s)))
        return rc;
    KCHK(c, hipEventRecord(c->ev_fork[0], s));
    {
        size_t tmp = 0;
        KCHK(c, hipcub::DeviceRadixSort::SortPairs(
                     nullptr, tmp, P<uint64_t>(K->pkey), P<uint64_t>(K->pkey2),
                     P<uint64_t>(K->pval), P<uint64_t>(K->pval2), nprod, 0,
                     rbits + cbits, s));
        if ((rc = grow(c, K->tmp, tmp)))
            return rc;
        KCHK(c, hipcub::DeviceRadixSort::SortPairs(
                     K->tmp.p, tmp, P<uint64_t>(K->pkey), P<uint64_t>(K->pkey2),
                     P<uint64_t>(K->pval), P<uint64_t>(K->pval2), nprod, 0,
                     rbits + cbits, s));
    }
    KCHK(c, hipEventSynchronize(c->ev_fork[0]));
    const uint64_t ndrop = K->host[0];
    const uint64_t np = nprod - ndrop;   // dropped products sort last
    if (np == 0)
        return PA_OK;
    if ((rc = grow(c, K->heads, np * 4)) || (rc = grow(c, K->runid, np * 8)))
        return rc;
    hipLaunchKernelGGL(k_run_heads, dim3(nblocks(np)), dim3(kTB), 0, s,
                       P<uint64_t>(K->pkey2), np, P<uint32_t>(K->heads));
    if ((rc = scan_flags(c, K, P<uint32_t>(K->heads), P<uint64_t>(K->runid),
                         np, true, s)))
        return rc;
    uint64_t nruns = 0;
    if ((rc = d2h_value(c, K, &nruns, P<uint64_t>(K->runid) + np - 1, s)))
        return rc;
    if ((rc = grow(c, K->rstart, nruns * 8)) ||
        (rc = grow(c, K->keep, nruns * 4 + 8)) ||
        (rc = grow(c, K->kpos, (nruns + 1) * 8)) ||
        (rc = grow(c, K->cand, nruns * sizeof(pa_pair))))
        return rc;
    hipLaunchKernelGGL(k_run_starts, dim3(nblocks(np)), dim3(kTB), 0, s,
                       P<uint32_t>(K->heads), P<uint64_t>(K->runid), np,
                       P<uint64_t>(K->rstart));
    // folded pairs go to pkey (free now) before the compaction
    if ((rc = grow(c, K->pkey, nruns * sizeof(pa_pair))))
        return rc;
    FoldArgs fa{P<uint64_t>(K->rstart), nruns, np, P<uint64_t>(K->pkey2),
                P<uint64_t>(K->pval2), rbits, cb, kc.ckthr, kc.mosthr,
                P<pa_pair>(K->pkey), P<uint32_t>(K->keep)};
    hipLaunchKernelGGL(k_fold_runs, dim3(nblocks(nruns)), dim3(kTB), 0, s, fa);
    KCHK(c, hipGetLastError());
    if ((rc = scan_flags(c, K, P<uint32_t>(K->keep), P<uint64_t>(K->kpos),
                         nruns, false, s)))
        return rc;
    if ((rc = d2h_start(c, K, 0, P<uint64_t>(K->kpos) + nruns - 1, s)) ||
        (rc = d2h_start(c, K, 1, P<uint32_t>(K->keep) + nruns - 1, s)))
        return rc;
    KCHK(c, hipStreamSynchronize(s));
    const uint64_t last = K->host[0], lastkeep = (uint32_t)K->host[1];
    const uint64_t nout = last + lastkeep;
    hipLaunchKernelGGL(k_compact, dim3(nblocks(nruns)), dim3(kTB), 0, s,
                       P<pa_pair>(K->pkey), P<uint32_t>(K->keep),
                       P<uint64_t>(K->kpos), nruns, P<pa_pair>(K->cand));
    KCHK(c, hipGetLastError());
    KCHK(c, hipStreamSynchronize(s));
    *n = nout;
    return PA_OK;
}

}  // namespace

extern "C" int pa_kmer_candidates(pa_ctx *c, const pa_kmer_config *kc,
                                  uint64_t c_begin, uint64_t c_end,
                                  pa_pair *d_out, uint64_t cap,
                                  uint64_t *n_out)
{
    if (!c || !kc || !n_out)
        return PA_ERR_ARG;
    *n_out = 0;
    if (!c->have_rows || !c->have_cols)
        return fail(c, PA_ERR_NOSEQ, "load row and column sequences first");
    if (kc->k < 1 || kc->stride < 1 || kc->symmetric < PA_SYM_NONE ||
        kc->symmetric > PA_SYM_EVEN_ODD)
        return fail(c, PA_ERR_ARG, "bad k-mer configuration");
    if (c_end > c->clen.size())
        c_end = c->clen.size();
    if (c_begin > c_end)
        c_begin = c_end;
    if (c->rlen.size() > 0xffffffffull || c->clen.size() > 0xffffffffull)
        return fail(c, PA_ERR_LIMIT, "more than 2^32 sequences");
    hipSetDevice(c->device);
    if (!c->kmer)
        c->kmer = new KmerState();
    KmerState *K = c->kmer;
    if (!K->host)
        KCHK(c, hipHostMalloc((void **)&K->host, 64, hipHostMallocDefault));
    hipStream_t s = c->st;
    int rc;
    if (!(K->have_last && same_cfg(K->last, *kc) && K->last_cb == c_begin &&
          K->last_ce == c_end && K->last_gen == c->seq_gen)) {
        K->have_last = false;
        uint64_t n = 0;
        if ((rc = generate(c, K, *kc, c_begin, c_end, &n, s)))
            return rc;
        K->last = *kc;
        K->last_cb = c_begin;
        K->last_ce = c_end;
        K->last_n = n;
        K->last_gen = c->seq_gen;
        K->have_last = true;
    }
    *n_out = K->last_n;
    if (!d_out)
        return PA_OK;
    if (K->last_n > cap)
        return fail(c, PA_ERR_LIMIT,
                    std::to_string(K->last_n) + " candidates exceed the "
                    "output capacity " + std::to_string(cap));
    if (K->last_n)
        KCHK(c, hipMemcpyAsync(d_out, K->cand.p, K->last_n * sizeof(pa_pair),
                               hipMemcpyDeviceToDevice, s));
    KCHK(c, hipStreamSynchronize(s));
    return PA_OK;
}
