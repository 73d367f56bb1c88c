// dp.hip -- batched NWSmall-exact affine-gap DP for gfx950.
//
// One wavefront per job (or four narrow jobs a wavefront, one a 16-lane row).
// The B axis is cut into stripes of 64 * COLS columns; lane k owns COLS
// consecutive columns of the stripe and walks down the rows of A one step
// behind lane k-1 (anti-diagonal skew), so at step t lane k is on row i = t -
// k + 1.  The right-edge values of each lane's last column move to lane k+1
// with a DPP wave_shr:1 each step; lane 0 reads the stripe's left boundary
// column from a per-job buffer written by lane 63 of the previous stripe, 64
// rows at a time.
//
// Scores are int32.  On this path every operand of the reference's float DP
// is an integer (NUC_SP, -200 open/close halves, extend 0, MU/nucmx.cpp:8-25,
// MU/profilefrommsa.cpp:291-292), and MINUS_INFINITY (-1e37, MU/intmath.h:46)
// only ever meets finite values or itself, so a large negative sentinel
// reproduces every comparison.  Cell rules follow MU/nwsmall.cpp:
//   D(i,j) = max(D(i-1,j), M(i-1,j) + open_A[i-1])       tie -> M   (68-86)
//   I(i,j) = max(I(i,j-1), M(i,j-1) + open_B[j-1])       tie -> M   (91-106)
//   M(i,j) = s(i,j) + max(M(i-1,j-1), D(i-1,j-1) + close, I(i-1,j-1) + close)
//            tie order M, D, I                                      (111-142)
// with the boundary rows/columns of 546-569, 579-595, 616-637 expressed as
// virtual row/column 0 values, and the one-row case (LA == 1) where M(1,1)
// carries close_A[0] (616-626; SetTermGaps leaves close[0] alone for a length-1
// profile, MU/termgaps.cpp:24).
//
// Each cell leaves a 4-bit record for the trace-back, which the same wavefront
// runs right after its forward pass.
#include "mh_internal.hpp"
#include "dp_tune_table.h"
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <numeric>
#include <cstdlib>
#include <utility>
#include <type_traits>
#include <cstring>
#include <thread>
#include <mutex>

namespace mh {
namespace {

constexpr int NEG = -(1 << 29);
constexpr int SBIAS = 65;           // smallest NUC_SP entry is -125 + 60 = -65

struct DevJob {
    uint64_t a_off, b_off;
    uint32_t la, lb;
    uint64_t tb_off;    // bytes
    uint64_t bnd_off;   // int32 elements
    uint64_t path_off;  // bytes (slot start)
    uint32_t user;      // index in the caller's job array
    uint32_t cols;      // columns per lane (4, 8 or 16): stripe width 64*cols
    uint32_t band;      // 0: the whole matrix; W > 0: the stripes' rows that meet |j - i*lb/la| <= W
    uint32_t pad_;
};

struct DpOut {
    int32_t score;
    int32_t edge;       // 'M', 'D' or 'I'
};

}  // namespace

// Rows [r0, r1] (1-based) that stripe s (columns s*sw+1 .. min((s+1)*sw, lb))
// computes.  Full DP: every row.  Band W: the rows where some column of the
// stripe lies within W of the corner-to-corner line j = i*lb/la, i.e.
// la*(c0-W)/lb <= i <= la*(c1+W)/lb; empty when r1 < r0.
__host__ __device__ inline void stripe_rows(uint32_t la, uint32_t lb, uint32_t band, uint32_t sw, uint32_t s,
                                            int &r0, int &r1)
{
    if (band == 0) {
        r0 = 1;
        r1 = (int)la;
        return;
    }
    const int64_t c0 = (int64_t)s * sw + 1;
    const int64_t c1e = (int64_t)(s + 1) * sw;
    const int64_t c1 = c1e < (int64_t)lb ? c1e : (int64_t)lb;
    const int64_t lo = c0 - (int64_t)band;
    int64_t a0 = lo <= 0 ? 1 : ((int64_t)la * lo + lb - 1) / lb;
    if (a0 < 1) a0 = 1;
    int64_t a1 = ((int64_t)la * (c1 + (int64_t)band)) / lb;
    if (a1 > (int64_t)la) a1 = la;
    r0 = (int)a0;
    r1 = (int)a1;
}

// Steps of one job run by g lanes of cols columns: rows + g - 1 per non-empty
// stripe.  A step evaluates g * cols cells.
static uint64_t dp_steps(uint32_t la, uint32_t lb, uint32_t band, uint32_t cols, uint32_t g)
{
    const uint32_t sw = g * cols;
    const uint32_t ns = (lb + sw - 1) / sw;
    uint64_t steps = 0;
    for (uint32_t s = 0; s < ns; ++s) {
        int r0, r1;
        stripe_rows(la, lb, band, sw, s, r0, r1);
        if (r1 >= r0) steps += (uint64_t)(r1 - r0 + 1) + (g - 1);
    }
    return steps;
}

namespace {

__device__ __forceinline__ int shr1_old(int v, int old)
{
    // wave_shr:1 -- lane k receives lane k-1's value, lane 0 receives `old`
    return __builtin_amdgcn_update_dpp(old, v, 0x138, 0xF, 0xF, false);
}

// The same shift within the job's lanes: the whole wavefront (G = 64) or each
// 16-lane DPP row (G = 16, row_shr:1; the row's first lane receives `old`).
template <int G> __device__ __forceinline__ int shr1_group(int v, int old)
{
    if constexpr (G == 64) return shr1_old(v, old);
    else return __builtin_amdgcn_update_dpp(old, v, 0x111, 0xF, 0xF, false);
}

template <int... Cs, class F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, Cs...>, F &&f)
{
    (f(std::integral_constant<int, Cs>{}), ...);
}

// ---- the cell ---------------------------------------------------------------
//
// NWSmall's recurrences (see above) are evaluated in a form that keeps two
// values a column instead of three and adds once a cell instead of three times.
// With o the gap open (goh) and c the close (goh), both constant inside the
// matrix, and
//   E(i,j) = D(i,j) - o,   F(i,j) = I(i,j) - o,   N(i,j) = M(i,j) - (o + c),
// the rules become
//   H(i,j)   = max(N, E, F)(i,j)        the best source of M(i+1,j+1)
//   N(i,j)   = s(i,j) + H(i-1,j-1),     M = N + (o + c)
//   E(i+1,j) = max(E(i,j), M(i,j)),     F(i,j+1) = max(F(i,j), M(i,j)).
// Each is the reference's comparison with both sides shifted alike, and all
// values are integers, so scores and ties are the same.  The terminal gaps
// (open 0 at the first position, no close at the last) only touch column 0, row
// 0 and the final pick.
//
// A cell's trace record holds, for a walk that arrives at (i, j), the state it
// continues in: bits 0-1 the source of H(i, j) for one that arrives by an M edge
// from (i+1, j+1) (TAG_M, TAG_D, TAG_I), bit 2 set when D(i+1, j) opens from M(i, j),
// bit 3 set when I(i, j+1) does.  The int32 cell keeps values times four with
// the state in the two low bits (M 3, D 2, I 0): a maximum then breaks ties as
// the reference does (M before D before I) and its low bits are the record's,
// shifted into the trace word by one v_alignbit each, instead of compares and
// selects.
//
// The forward pass is bound by VALU issue.  Per cell this takes 11.5 VALU
// instructions: two adds (one an SDWA add that also picks the cell's 16-bit
// score), one max3, two max, three v_alignbit, three that restore the tags, and
// half a v_perm (the scores of two columns by A's letter).  Measured on MI355X:
// the 16-column row step went from 348 instructions (compares, selects and s_nops
// for the trace bits) to 199; 20,000 jobs of 5-500 columns from 1,697 to 992 us,
// 4,000 of 10-20,000 from 113.8 to 75.9 ms (both with the walks below).
enum : uint32_t { TAG_M = 3, TAG_D = 2, TAG_I = 0 };

__device__ __forceinline__ uint32_t walk_next(uint32_t nib, int t)
{
    if (t == 'M') return (nib & 3u) == TAG_M ? 'M' : ((nib & 3u) == TAG_D ? 'D' : 'I');
    if (t == 'D') return (nib & 4u) ? 'M' : 'D';
    return (nib & 8u) ? 'M' : 'I';
}

// does a walk in state t stay in it at a position with this record
__device__ __forceinline__ bool walk_stays(uint32_t nib, int t)
{
    return t == 'M' ? (nib & 3u) == TAG_M : (t == 'D' ? (nib & 4u) == 0u : (nib & 8u) == 0u);
}

// bytes of a lane's records of one step: a nibble a column, in whole words a
// lane can store at once
__host__ __device__ constexpr uint32_t lane_bytes_of(uint32_t cols)
{
    return cols <= 2 ? 1u : (cols <= 4 ? 2u : (cols <= 8 ? 4u : 8u));
}

template <int COLS> __device__ __forceinline__ void store_records(uint8_t *dst, const uint32_t *word)
{
    if constexpr (COLS <= 2) *dst = (uint8_t)word[0];
    else if constexpr (COLS <= 4) *reinterpret_cast<uint16_t *>(dst) = (uint16_t)word[0];
    else if constexpr (COLS <= 8) *reinterpret_cast<uint32_t *>(dst) = word[0];
    else *reinterpret_cast<uint2 *>(dst) = make_uint2(word[0], word[1]);
}

// Match scores: int32, NUC_SP (MU/nucmx.cpp:8-25) as packed_rows gives it, or
// the 6 x 6 float table of operands with wildcard letters.
struct ScoreArgs {
    uint32_t lo[4], hi[4];     // int32: row a's scores times 4, 16 bits each (columns 0, 1 | 2, 3)
    uint32_t sr[4];            // int32: row a's scores plus SBIAS, 8 bits each (sliding-window jobs)
};

constexpr int GOH = -200;      // half of the gap open (MU/profilefrommsa.cpp:291-292)

// int32 cells: values times 4 plus the state's tag
struct IntCell {
    static constexpr int OC = 4 * (2 * GOH);
    static constexpr int NEGV = -(1 << 30);
    __device__ static int neg_h() { return NEGV | 3; }
    __device__ static int neg_e() { return NEGV | 2; }
    __device__ static int neg_f() { return NEGV; }
    // H(0,0): the source of M(1,1) is M(0,0) = 0; with LA == 1 the reference
    // gives M(1,1) the close of the one position (MU/nwsmall.cpp:616-626)
    __device__ static int corner(int la) { return 4 * (la == 1 ? GOH : 0) - OC + 3; }
    // H(i,0) and H(0,j): D(i,0) = I(0,j) = 0, closed
    __device__ static int edge() { return 4 * GOH - OC + 3; }

    template <int COLS> struct Lane {
        int H[COLS], E[COLS], F[COLS];   // row i: H(i,j), E(i+1,j), F(i,j+1)
        uint32_t sel[(COLS + 1) / 2];    // byte selectors of two columns' scores
        uint32_t word[COLS > 8 ? 2 : 1];
    };
    template <int COLS, class Code> __device__ static void init(Lane<COLS> &s, Code &&code, bool top, bool first)
    {
#pragma unroll
        for (int c = 0; c < COLS; c += 2) {
            const uint32_t b0 = code(c) & 3u, b1 = c + 1 < COLS ? code(c + 1) & 3u : 0u;
            s.sel[c / 2] = (2u * b0) | ((2u * b0 + 1u) << 8) | ((2u * b1) << 16) | ((2u * b1 + 1u) << 24);
        }
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            s.H[c] = top ? edge() : neg_h();
            s.E[c] = neg_e();
            s.F[c] = neg_f();
        }
        (void)first;
        for (uint32_t &w : s.word) w = 0;
    }
    // the row operand of A's letter
    __device__ static void operand(const ScoreArgs &sc, uint32_t code, int &lo, int &hi)
    {
        lo = (int)((code & 2) ? ((code & 1) ? sc.lo[3] : sc.lo[2]) : ((code & 1) ? sc.lo[1] : sc.lo[0]));
        hi = (int)((code & 2) ? ((code & 1) ? sc.hi[3] : sc.hi[2]) : ((code & 1) ? sc.hi[1] : sc.hi[0]));
    }
    // one row: diagH = H(i-1, first column - 1), f = F(i, first column)
    template <int COLS>
    __device__ static __forceinline__ void row(Lane<COLS> &s, const float *, int lo, int hi, int diagH, int f)
    {
        // (N of column c + 1 is taken before H of column c changes, so that no
        // register is copied)
        uint32_t p = __builtin_amdgcn_perm((uint32_t)hi, (uint32_t)lo, s.sel[0]);
        int n = diagH + (int)(int16_t)(p & 0xFFFFu);
        static_for(std::make_integer_sequence<int, COLS>{}, [&](auto ic) {
            constexpr int c = decltype(ic)::value;
            constexpr int w = c >> 3;
            const int m = n + OC;
            const int h = max(max(n, s.E[c]), f);
            s.word[w] = __builtin_amdgcn_alignbit((uint32_t)h, s.word[w], 2);
            if constexpr (c + 1 < COLS) {
                if constexpr ((c & 1) == 1) p = __builtin_amdgcn_perm((uint32_t)hi, (uint32_t)lo, s.sel[(c + 1) / 2]);
                n = s.H[c] + ((c & 1) ? (int)(int16_t)(p & 0xFFFFu) : (int)p >> 16);
            }
            s.H[c] = h | 3;
            const int x = max(s.E[c], m);
            s.word[w] = __builtin_amdgcn_alignbit((uint32_t)x, s.word[w], 1);
            s.E[c] = x & ~1;
            const int y = max(f, m);
            s.word[w] = __builtin_amdgcn_alignbit((uint32_t)y, s.word[w], 1);
            f = y & ~3;
            s.F[c] = f;
        });
        if constexpr ((COLS & 7) != 0) s.word[COLS >> 3] >>= 32 - 4 * (COLS & 7);
    }
    // the final pick (MU/nwsmall.cpp:641-656) of the cell with values h, e, f
    // and record nib: M(LA,LB), D and I without their close.  e and f hold
    // max(E, M) and max(F, M); the record's bits say which, and an M that
    // neither shows and that is not H's source is below D or I.
    __device__ static void pick(int h, int e, int f, uint32_t nib, int, int, int, int &score, int &edge_out)
    {
        constexpr int NONE = -(1 << 30);
        const int hv = h >> 2, ev = e >> 2, fv = f >> 2;
        const int M = (nib & 4u) ? ev : ((nib & 8u) ? fv : ((nib & 3u) == TAG_M ? hv + 2 * GOH : NONE));
        const int D = (nib & 4u) ? NONE : ev + GOH, I = (nib & 8u) ? NONE : fv + GOH;
        score = M;
        edge_out = 'M';
        if (D > score) { score = D; edge_out = 'D'; }
        if (I > score) { score = I; edge_out = 'I'; }
    }
};

// Cells whose values carry no tag: float for operands with wildcard letters
// (fractional scores, added in the reference's order: M = s + best, D and I
// closed before the comparison, so every value and tie is its float), and
// int32 for jobs whose scores times four could leave 32 bits.  H(i,j) =
// max(M, D + c, I + c), E(i+1,j) = max(D, M + o), F(i,j+1) = max(I, M + o).
// Bound by latency: such jobs are few.  2,000 jobs of 10-1,000 columns, one in
// twenty with wildcard letters: 943 ms with a thread a wildcard job (rows and a
// byte a cell in device memory, one dependent access after another), 1.65 ms
// with these cells in dp_job's wavefronts.
template <class T> struct CmpCell {
    static constexpr bool FLT = std::is_same<T, float>::value;
    static constexpr T G = (T)GOH;
    __device__ static T neg() { return FLT ? (T)-1e37f : (T)-(1 << 29); }     // MINUS_INFINITY, MU/intmath.h:46
    __device__ static int bits(T v)
    {
        if constexpr (FLT) return __float_as_int(v);
        else return v;
    }
    __device__ static T val(int b)
    {
        if constexpr (FLT) return __int_as_float(b);
        else return b;
    }
    __device__ static int neg_h() { return bits(neg()); }
    __device__ static int neg_e() { return bits(neg()); }
    __device__ static int neg_f() { return bits(neg()); }
    __device__ static int corner(int la) { return bits(la == 1 ? G : (T)0); }
    __device__ static int edge() { return bits(G); }

    template <int COLS> struct Lane {
        int H[COLS], E[COLS], F[COLS];   // row i: H(i,j), D(i+1,j), I(i,j+1)
        T M[COLS], D[COLS], I[COLS];     // row i
        uint8_t code[COLS];
        uint32_t word[COLS > 8 ? 2 : 1];
    };
    template <int COLS, class Code> __device__ static void init(Lane<COLS> &s, Code &&code, bool top, bool)
    {
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            s.code[c] = (uint8_t)code(c);
            s.H[c] = top ? edge() : neg_h();
            s.E[c] = neg_e();
            s.F[c] = neg_f();
            s.M[c] = s.D[c] = s.I[c] = neg();
        }
        for (uint32_t &w : s.word) w = 0;
    }
    __device__ static void operand(const ScoreArgs &, uint32_t code, int &lo, int &hi)
    {
        lo = 6 * (int)code;
        hi = 0;
    }
    template <int COLS>
    __device__ static __forceinline__ void row(Lane<COLS> &s, const float *table, int lo, int, int diagH, int f)
    {
#pragma clang fp contract(off)
        T dh = val(diagH), fi = val(f);
        static_for(std::make_integer_sequence<int, COLS>{}, [&](auto ic) {
            constexpr int c = decltype(ic)::value;
            constexpr int w = c >> 3, sh = 4 * (c & 7);
            const T sc = (T)table[lo + s.code[c]];
            const T m = sc + dh, d = val(s.E[c]), i = fi;
            const T a = m + G, dc = d + G, ic2 = i + G;
            const T h = max(max(m, dc), ic2);
            uint32_t nib = m == h ? (uint32_t)TAG_M : (dc == h ? (uint32_t)TAG_D : (uint32_t)TAG_I);
            dh = val(s.H[c]);
            s.H[c] = bits(h);
            if (a >= d) nib |= 4u;
            s.E[c] = bits(a >= d ? a : d);
            if (a >= i) nib |= 8u;
            fi = a >= i ? a : i;
            s.F[c] = bits(fi);
            s.M[c] = m;
            s.D[c] = d;
            s.I[c] = i;
            s.word[w] = (sh == 0 ? 0u : s.word[w]) | (nib << sh);
        });
    }
    // M, D, I of the final cell
    __device__ static void pick(int, int, int, uint32_t, int M, int D, int I, int &score, int &edge_out)
    {
        T s = val(M);
        edge_out = 'M';
        if (val(D) > s) { s = val(D); edge_out = 'D'; }
        if (val(I) > s) { s = val(I); edge_out = 'I'; }
        if constexpr (FLT) score = (int)rintf(s);
        else score = s;
    }
};

// One job per G lanes: a wavefront (G = 64), or each 16-lane DPP row of a
// wavefront (G = 16: four jobs at once, for jobs at most 16*COLS columns wide,
// whose skew and column padding would leave most of a wavefront idle).  In
// what follows "64" is G.  Stripe s computes rows [r0, r1] (stripe_rows); at
// step t lane k is on row r0 + t - k.  Cells outside those rows are outside
// the computed region and read as minus infinity, so a banded job is the exact
// DP restricted to that region; with band 0 every stripe runs all rows.  Lanes
// outside their row range sit out the step (exec mask).  Two values a row move
// to the next lane: H of the lane's last column (the diagonal source of the
// next lane's first column on the row below) and F past it.  Each lane stores
// lane_bytes_of(COLS) bytes of records per step, so a wavefront stores 512
// contiguous bytes (16 columns a lane).  Cell (i, j) of lane k, column c is at
// byte  stripe_base + ((i - r0 + k)*64 + k)*lane_bytes + c/2, nibble c%2.
//
// PIPE: the job's stripes are shared by P wavefronts, wavefront p0 taking
// stripes p0, p0 + P, ...: stripe s reads the boundary column that stripe
// s - 1 (another wavefront) writes.  Each boundary value travels as one
// 64-bit word, the value and a tag (the writing stripe's index + 1), in one
// of two buffers by stripe parity (zeroed by the host before the round):
// written with atomic stores and read with atomic loads at device scope, a
// word is either the one stripe s - 1 wrote or visibly not, so no fence is
// needed.  A reader fetches a chunk of rows one chunk ahead and checks the
// tags when it is about to use them, fetching again the rows not yet
// written.  A wait is bounded (DP_SPIN_MAX polls), past which it sets *err
// and goes on, and the wavefront waits no more (so a stuck job ends within a
// few bounds, its result flagged by the host as an error).  A buffer is
// rewritten by stripe s + 1 only at rows stripe s has used: it computes a row
// after stripe s published it, and stripe s publishes it after reading it.
// Deadlock-free: parts take tickets from their bin in the order they start
// running, so a part waits only on parts that run or have run, except the
// parts of the one job a bin whose parts are not all taken; those are far
// fewer than the resident wavefronts.
// The result is the same as one wavefront's.  The boundary moves CH rows at a
// time, each chunk's rows as soon as its steps are done.
//
// Returns whether this wavefront (this row of it) computed the final cell;
// score and edge are then the final pick in every lane of the group.
constexpr uint32_t DP_SPIN_MAX = 1u << 22;

// Between one lane's write to LDS and another lane's access to the same slot
// (the lanes of a wavefront): its LDS operations complete in order, and the
// compiler moves none across this.
__device__ __forceinline__ void lanes_ordered()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of one wavefront: the rows a group's first lane takes in, and the
// boundary column its last lane hands on
struct DpLds {
    int4 in[64];        // H(i, j0 - 1), F(i, j0), A's row operand (two words)
    int2 out[64];
    int2 idle[64];
    int fin[6][64];
};

template <class CELL, int COLS, int G, bool PIPE = false>
__device__ __forceinline__ bool dp_job(const DevJob &jb, const uint8_t *__restrict__ A, const uint8_t *__restrict__ B,
                                       uint8_t *__restrict__ tb, int *__restrict__ bnd, const ScoreArgs &sc,
                                       const float *table, DpLds &lds, int &score, int &edge, int p0 = 0, int P = 1,
                                       uint32_t *__restrict__ err = nullptr)
{
    constexpr int STRIPE_W = G * COLS;
    constexpr int LANE_BYTES = (int)lane_bytes_of(COLS);
    constexpr int CH = G == 64 && COLS >= 8 ? 32 : 16;   // steps of a chunk
    const int lane = (int)threadIdx.x & (G - 1);
    const int gb = (int)threadIdx.x & ~(G - 1);    // the job's slots in the LDS rows
    const int la = (int)jb.la, lb = (int)jb.lb;
    const uint8_t *a = A + jb.a_off;
    const uint8_t *b = B + jb.b_off;
    const int nr = (la + 63) & ~63;
    int *bH = bnd + jb.bnd_off;
    int *bF = bH + nr;
    uint8_t *tbj = tb + jb.tb_off;
    const int nstripes = (lb + STRIPE_W - 1) / STRIPE_W;
    const int fin_lane = ((lb - 1) % STRIPE_W) / COLS;
    const int fin_col = (lb - 1) % COLS;
    bool fin = false;
    int prev_r0 = 1, prev_r1 = 0;     // rows of the previous stripe's last column held in bnd
    uint64_t tbs = 0;                 // byte offset of the stripe's trace block
    int counted = 0;                  // PIPE: the stripes whose blocks it counts
    bool gave_up = false;             // PIPE: a wait ran past its bound

    for (int s = PIPE ? p0 : 0; s < nstripes; s += PIPE ? P : 1) {
        int r0, r1;
        stripe_rows(jb.la, jb.lb, jb.band, STRIPE_W, s, r0, r1);
        // PIPE: the tagged boundary words read (written by stripe s - 1, tag s) and written (tag s + 1)
        unsigned long long *pin = nullptr, *pout = nullptr;
        if constexpr (PIPE) {
            // stripe s - 1 runs on another wavefront: its rows, and this
            // stripe's trace block after the blocks of the stripes before it
            prev_r0 = 1;
            prev_r1 = 0;
            if (s > 0) stripe_rows(jb.la, jb.lb, jb.band, STRIPE_W, s - 1, prev_r0, prev_r1);
            for (; counted < s; ++counted) {
                int a0, a1;
                stripe_rows(jb.la, jb.lb, jb.band, STRIPE_W, counted, a0, a1);
                if (a1 >= a0) tbs += (uint64_t)(a1 - a0 + G) * G * LANE_BYTES;
            }
            unsigned long long *pb = reinterpret_cast<unsigned long long *>(bnd + jb.bnd_off);
            pin = pb + (size_t)((s + 1) & 1) * 2 * nr;
            pout = pb + (size_t)(s & 1) * 2 * nr;
        }
        if (r1 < r0) {
            prev_r0 = 1;
            prev_r1 = 0;
            continue;
        }
        // PIPE: until every lane with want set holds the words stripe s - 1
        // wrote for row i (tag s), fetch them again
        auto settle = [&](bool want, int i, unsigned long long &wH, unsigned long long &wF) {
            if constexpr (PIPE) {
                uint32_t spins = 0;
                for (;;) {
                    const bool bad = want && ((uint32_t)(wH >> 32) != (uint32_t)s || (uint32_t)(wF >> 32) != (uint32_t)s);
                    if (__ballot(bad) == 0 || gave_up) break;
                    if (++spins > DP_SPIN_MAX) {
                        if (lane == 0) atomicOr(err, 1u);
                        gave_up = true;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(2);
                    if (bad) {
                        wH = __hip_atomic_load(pin + i - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        wF = __hip_atomic_load(pin + nr + i - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            }
        };
        const int nrows = r1 - r0 + 1;
        const int j0 = s * STRIPE_W + 1;
        const int jl = j0 + lane * COLS;
        const int rem = lb - (jl - 1);
        const int ncols = rem < 0 ? 0 : (rem > COLS ? COLS : rem);
        const int span = lb - s * STRIPE_W;
        const int nl = span >= STRIPE_W ? G : (span + COLS - 1) / COLS;
        const bool last_stripe = (s == nstripes - 1);
        const bool top0 = (r0 == 1);

        // the row above the stripe: row 0 when the stripe starts at row 1, else outside
        typename CELL::template Lane<COLS> st;
        CELL::template init<COLS>(st, [&](int c) { return c < ncols ? (uint32_t)b[jl - 1 + c] : 0u; }, top0, s == 0);
        // H above-left of the lane's first column: the corner for column 1,
        // row 0 for other columns of row 1, the previous stripe's last column
        // (row r0-1) for lane 0 when it holds that row, else outside
        int lpH = CELL::neg_h();
        if (top0) {
            lpH = jl == 1 ? CELL::corner(la) : CELL::edge();
        } else if constexpr (PIPE) {
            const int i = r0 - 1;
            const bool want = lane == 0 && s > 0 && i >= prev_r0 && i <= prev_r1;
            unsigned long long wH = 0, wF = 0;
            if (want) {
                wH = __hip_atomic_load(pin + i - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                wF = __hip_atomic_load(pin + nr + i - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            settle(want, i, wH, wF);
            if (want) lpH = (int)(uint32_t)wH;
        } else if (lane == 0 && s > 0 && r0 - 1 >= prev_r0 && r0 - 1 <= prev_r1) {
            lpH = bH[r0 - 2];
        }
        int outH = CELL::neg_h(), outF = CELL::neg_f(), rlo = 0, rhi = 0;

        // lane 0's inputs, CH rows per chunk (a lane a row): column jl-1 of the
        // previous stripe where it computed that row, column 0, or outside;
        // and A's letters.  The next chunk is loaded one chunk ahead.  (PIPE: the
        // words are fetched here, for rows this stripe computes, and settled
        // before use)
        unsigned long long wH = 0, wF = 0;
        bool want = false;
        int wrow = 0;
        auto left_in = [&](int x, int &h, int &f, uint32_t &ac) {
            const int i = r0 + x;
            h = s == 0 ? CELL::edge() : CELL::neg_h();
            f = CELL::neg_f();
            ac = 0;
            if constexpr (PIPE) want = false;
            if (CH < G && lane >= CH) return;
            if (s > 0 && i >= prev_r0 && i <= prev_r1) {
                if constexpr (PIPE) {
                    want = i <= r1;
                    wrow = i;
                    if (want) {
                        wH = __hip_atomic_load(pin + i - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        wF = __hip_atomic_load(pin + nr + i - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                } else {
                    h = bH[i - 1];
                    f = bF[i - 1];
                }
            }
            if (i <= r1) ac = a[i - 1];
        };
        int nH, nF;
        uint32_t nA;
        left_in(lane, nH, nF, nA);

        const int nsteps = nrows + nl - 1;
        const uint32_t my_rows = lane < nl ? (uint32_t)nrows : 0u;
        uint8_t *dst = tbj + tbs;
        const uint32_t dst_lane = (uint32_t)lane * LANE_BYTES;
        // The last lane's values go to the step's slot of the chunk (the other
        // lanes' to a slot no one reads).
        int2 *const out_slot = lane == G - 1 ? &lds.out[gb] : &lds.idle[threadIdx.x & 63];
        const int out_next = lane == G - 1 ? 1 : 0;
        // (nothing loaded above is waited for inside the step loop, where the
        // wait would be for the last step's store too)
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
        int4 ahead = make_int4(0, 0, 0, 0);
        for (int t = 0; t < nsteps; ++t) {
            const int q = t & (CH - 1);
            if (q == 0) {
                if constexpr (PIPE) {
                    settle(want, wrow, wH, wF);
                    if (want) {
                        nH = (int)(uint32_t)wH;
                        nF = (int)(uint32_t)wF;
                    }
                    // A SIMD gives its oldest wavefront every slot it can use, and
                    // the parts of a job wait for the slowest of them: each
                    // wavefront's priority falls with its progress, modulo four
                    // chunks, so that those that fell behind go first.
                    switch ((t / CH) & 3) {
                    case 0: __builtin_amdgcn_s_setprio(3); break;
                    case 1: __builtin_amdgcn_s_setprio(2); break;
                    case 2: __builtin_amdgcn_s_setprio(1); break;
                    default: __builtin_amdgcn_s_setprio(0); break;
                    }
                }
                int lo, hi;
                CELL::operand(sc, nA, lo, hi);
                lanes_ordered();     // (the chunk before has been read)
                if (CH == G || lane < CH) lds.in[gb + lane] = make_int4(nH, nF, lo, hi);
                lanes_ordered();
                left_in(t + CH + lane, nH, nF, nA);
                ahead = lds.in[gb];
            }
            // row r0 + t - lane of every lane that has one
            const int4 in = ahead;
            ahead = lds.in[gb + ((q + 1) & (CH - 1))];   // the next step's
            const int rH = shr1_group<G>(outH, in.x);
            const int rF = shr1_group<G>(outF, in.y);
            rlo = shr1_group<G>(rlo, in.z);
            rhi = shr1_group<G>(rhi, in.w);
            if ((uint32_t)(t - lane) < my_rows) {
                CELL::template row<COLS>(st, table, rlo, rhi, lpH, rF);
                lpH = rH;
                outH = st.H[COLS - 1];
                outF = st.F[COLS - 1];
                store_records<COLS>(dst + dst_lane, st.word);
            }
            dst += G * LANE_BYTES;
            out_slot[q * out_next] = make_int2(outH, outF);
            if ((q == CH - 1 || t == nsteps - 1) && !last_stripe && (CH == G || lane < CH)) {
                // the rows of the stripe's last column that this chunk finished
                lanes_ordered();
                const int x = t - q - (G - 1) + lane;
                if (x >= 0 && x < nrows) {
                    const int r = r0 - 1 + x;
                    const int2 v = lds.out[gb + lane];
                    if constexpr (PIPE) {
                        const unsigned long long tag = (unsigned long long)(uint32_t)(s + 1) << 32;
                        __hip_atomic_store(pout + r, tag | (uint32_t)v.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_store(pout + nr + r, tag | (uint32_t)v.y, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                    } else {
                        bH[r] = v.x;
                        bF[r] = v.y;
                    }
                }
                lanes_ordered();     // (before the next chunk's writes)
            }
        }
        if constexpr (PIPE) __builtin_amdgcn_s_setprio(0);
        if (last_stripe) {
            // the lane's registers hold row LA, the last it computed: the
            // final cell's values, picked by way of LDS, so that no
            // per-column select on fin_col is held through the step loop
            fin = true;
            int sco = CELL::neg_e(), ed = 'M';
            if (lane == fin_lane && r1 == la) {
                static_assert(COLS <= G, "a column a slot");
#pragma unroll
                for (int c = 0; c < COLS; ++c) {
                    lds.fin[0][gb + c] = st.H[c];
                    lds.fin[1][gb + c] = st.E[c];
                    lds.fin[2][gb + c] = st.F[c];
                    if constexpr (!std::is_same<CELL, IntCell>::value) {
                        lds.fin[3][gb + c] = CELL::bits(st.M[c]);
                        lds.fin[4][gb + c] = CELL::bits(st.D[c]);
                        lds.fin[5][gb + c] = CELL::bits(st.I[c]);
                    }
                }
                const uint32_t w = COLS > 8 && fin_col >= 8 ? st.word[COLS > 8 ? 1 : 0] : st.word[0];
                const int k = gb + fin_col;
                CELL::pick(lds.fin[0][k], lds.fin[1][k], lds.fin[2][k], (w >> (4 * (fin_col & 7))) & 15u,
                           lds.fin[3][k], lds.fin[4][k], lds.fin[5][k], sco, ed);
            }
            score = __shfl(sco, gb + fin_lane, 64);
            edge = __shfl(ed, gb + fin_lane, 64);
        }
        prev_r0 = r0;
        prev_r1 = r1;
        if constexpr (!PIPE) tbs += (uint64_t)(nrows + G - 1) * G * LANE_BYTES;
        // the next stripe reads the boundary column, and the walk the records,
        // that other lanes of this wavefront wrote
        if constexpr (!PIPE) __threadfence_block();
    }
    return fin;
}


// Row-packed jobs: four jobs of one shape per wavefront, one per 16-lane row
// (DevJob::cols = GROUP_TAG + COLS, COLS even from 4 to 16: the narrowest
// stripe that holds the job).
constexpr uint32_t GROUP_TAG = 32;
constexpr uint32_t ROWS_MAX_LB = 256;     // widest job run four to a wavefront
constexpr uint32_t ROWS_MAX_WALK = 1024;  // a + b from which a job takes a wavefront to itself

// ---- one round of jobs: a length-binned work queue ----------------------
//
// A round's jobs sit in one table in queue order: the 64-lane stripe jobs
// (those with long trace-back walks first, each part largest first), the
// row-packed jobs by shape (16, 14, ..., 4 columns a lane), the sliding-window
// jobs, the one-lane jobs.  The queue cuts that table into bins: stripe jobs
// by trace size (a new bin where it falls below the next power of 4), one bin
// per row shape, one of window jobs, one of one-lane jobs.  A bin hands out
// items (1 stripe or window job, 4 row-packed jobs, 64 one-lane jobs) through
// its own atomic cursor.  One launch drains the bins in order: a wavefront
// takes the next item of the first bin that is not empty (a persistent
// wavefront keeps taking items until the last bin is empty).  Everything a
// launch needs is in the round's descriptor in device memory, so the
// launches of a round take one pointer and are captured in a graph once per
// context; a round only sets the grid sizes of the graph's nodes.
constexpr int ROW_SHAPES = 7;
// QK_PIPE + P - 1 (P = 1 .. DP_PIPE_MAX): 64-lane stripe jobs whose stripes P
// wavefronts share (an item is one wavefront's part: job first + item / P,
// part item % P)
enum : uint32_t { QK_STRIPE = 0, QK_ROWS = 1, QK_WINDOW = QK_ROWS + ROW_SHAPES, QK_TINY = QK_WINDOW + 1,
                  QK_PIPE = QK_TINY + 1 };
constexpr uint32_t DP_PIPE_MAX = 32;
constexpr int DPQ_MAXB = 72;
constexpr int DPQ_CURSORS = DPQ_MAXB;

struct alignas(16) DpBin {
    uint32_t kind, first, count;
    uint32_t item0;     // the bin's first item in queue order (prefix sums)
};

// (Behind its bins in device memory: DPQ_CURSORS cursors, zeroed at the start of
// every round, the last of them the round's wait-bound error flag.)
struct DpRound {
    uint32_t nbins;
    float table[DP_NCLASS * DP_NCLASS];   // match scores of cells without a tag
    DpBin bin[DPQ_MAXB + 1];              // the last one's item0: the items
};

__device__ __forceinline__ uint32_t qk_per_item(uint32_t kind)
{
    return kind == QK_STRIPE || kind == QK_WINDOW || kind >= QK_PIPE ? 1u : (kind == QK_TINY ? 64u : 4u);
}

// ---- sliding-window banded DP ---------------------------------------------
//
// A banded job whose band fits 64*C columns (C = 1, 2, 4, 8) runs as a window
// that slides along the corner-to-corner line: all 64 lanes work on one row,
// lane k holding window columns base(i)+1+kC .. +C, with
//   base(i) = clamp(ceil((i*lb - h*la)/la) - 1, 0, lb - 64C),  h = (64C-1)/2
// so the window is centred on the line and holds every cell within h of it.
// Cells outside the window are -infinity: the result is the exact DP over the
// window region.  Per row: the previous row's M, D', I' shift left by
// s = base(i) - base(i-1) columns (DPP wave_shl:1 per column step), M and D'
// follow from the previous row (a right-to-left register pass), and
// I' -- a running maximum along the row since the gap extension is 0 -- is a
// lane-local prefix maximum joined by a cross-lane exclusive prefix maximum
// (DPP row_shr within 16-lane rows, readlane across rows).  Trace: C*4 bits
// per lane per row, 8/C rows per 32-bit word; the word of row i, lane k is
// at ((i-1) / (8/C)) * 64 + k.
constexpr uint32_t WINDOW_TAG = 64;   // DevJob::cols = WINDOW_TAG + C

__host__ __device__ inline int window_base(int la, int lb, int width, int i)
{
    const int64_t num = (int64_t)i * lb - (int64_t)((width - 1) / 2) * la;
    const int64_t q = num >= 0 ? (num + la - 1) / la : -((-num) / la);
    int64_t b = q - 1;
    const int64_t top = lb > width ? (int64_t)lb - width : 0;
    if (b > top) b = top;
    if (b < 0) b = 0;
    return (int)b;
}

__device__ __forceinline__ int shl1_old(int v, int old)
{
    // wave_shl:1 -- lane k receives lane k+1's value, lane 63 receives `old`
    return __builtin_amdgcn_update_dpp(old, v, 0x130, 0xF, 0xF, false);
}

__device__ __forceinline__ int row_shr_old(int v, int old, int n)
{
    switch (n) {
    case 1: return __builtin_amdgcn_update_dpp(old, v, 0x111, 0xF, 0xF, false);
    case 2: return __builtin_amdgcn_update_dpp(old, v, 0x112, 0xF, 0xF, false);
    case 4: return __builtin_amdgcn_update_dpp(old, v, 0x114, 0xF, 0xF, false);
    default: return __builtin_amdgcn_update_dpp(old, v, 0x118, 0xF, 0xF, false);
    }
}

template <int C>
__device__ __forceinline__ void dp_window_job(const DevJob &jb, const uint8_t *__restrict__ A,
                                              const uint8_t *__restrict__ B, uint8_t *__restrict__ tb,
                                              const ScoreArgs &sa, int &score, int &edge)
{
    constexpr int WD = 64 * C;
    constexpr int goh = GOH;
    constexpr int RPD = 8 / C;   // rows per trace word
    const int lane = threadIdx.x;
    const int la = (int)jb.la, lb = (int)jb.lb;
    const uint8_t *a = A + jb.a_off;
    const uint8_t *b = B + jb.b_off;
    uint32_t *tbj = reinterpret_cast<uint32_t *>(tb + jb.tb_off);
    const int go2 = 2 * goh;
    // base(i) without a division per row: q = ceil((i*lb - h*la)/la) kept with
    // its remainder rem = q*la - (i*lb - h*la) in [0, la)
    const int top = lb > WD ? lb - WD : 0;
    const int dq = lb / la, dr = lb % la;
    int q, rem;
    {
        const int64_t num = (int64_t)lb - (int64_t)((WD - 1) / 2) * la;
        const int64_t qq = num >= 0 ? (num + la - 1) / la : -((-num) / la);
        q = (int)qq;
        rem = (int)(qq * la - num);
    }
    auto clampb = [&](int v) { return v - 1 > top ? top : (v - 1 < 0 ? 0 : v - 1); };
    int bprev = clampb(q);
    int Mp[C], Dp[C], Ip[C];
    uint32_t bsh[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {   // row 0 in the frame of base(1)
        Mp[c] = NEG;
        Dp[c] = NEG + goh;
        Ip[c] = goh;
        const int j0 = bprev + lane * C + c;
        bsh[c] = j0 < lb ? 8u * (uint32_t)b[j0] : 0u;
    }
    // A codes 64 rows at a time, the next chunk loaded one chunk ahead
    int achunk = lane < la ? a[lane] : 0;
    int anext = 64 + lane < la ? a[64 + lane] : 0;
    uint32_t bnx[C];   // B codes of the next row's window, loaded a row ahead
#pragma unroll
    for (int c = 0; c < C; ++c) bnx[c] = bsh[c];
    uint32_t tbw = 0;
    int finM = NEG, finD = NEG, finI = NEG;
    for (int i = 1; i <= la; ++i) {
        if (i > 1) {
            q += dq;
            rem -= dr;
            if (rem < 0) {
                ++q;
                rem += la;
            }
        }
        const int bi = clampb(q);
        const int s = bi - bprev;
        if (s) {
            // this row's window codes, loaded during the previous row
#pragma unroll
            for (int c = 0; c < C; ++c) bsh[c] = bnx[c];
        }
        {   // issue the next row's B codes if its window moves
            int qn = q + dq;
            if (rem - dr < 0) ++qn;
            const int bn = clampb(qn);
            if (bn != bi && i < la) {
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const int j0 = bn + lane * C + c;
                    bnx[c] = j0 < lb ? 8u * (uint32_t)b[j0] : 0u;
                }
            }
        }
        // (i-1, bi): the cell left of the window on the previous row
        int ldM, ldD, ldI;
        if (i == 1) {
            ldM = bi == 0 ? 0 : NEG;
            ldD = NEG + goh;
            ldI = bi == 0 ? NEG + goh : goh;
        } else if (bi == 0) {
            ldM = NEG;
            ldD = goh;
            ldI = NEG + goh;
        } else {
            ldM = NEG;
            ldD = NEG;
            ldI = NEG;
            for (int st = 0; st < s; ++st) {
                if (st == s - 1) {
                    ldM = __builtin_amdgcn_readlane(Mp[0], 0);
                    ldD = __builtin_amdgcn_readlane(Dp[0], 0);
                    ldI = __builtin_amdgcn_readlane(Ip[0], 0);
                }
                const int eM = shl1_old(Mp[0], NEG), eD = shl1_old(Dp[0], NEG), eI = shl1_old(Ip[0], NEG);
#pragma unroll
                for (int c = 0; c + 1 < C; ++c) {
                    Mp[c] = Mp[c + 1];
                    Dp[c] = Dp[c + 1];
                    Ip[c] = Ip[c + 1];
                }
                Mp[C - 1] = eM;
                Dp[C - 1] = eD;
                Ip[C - 1] = eI;
            }
        }
        if (i > 1 && ((i - 1) & 63) == 0) {
            achunk = anext;
            anext = (i + 63 + lane < la) ? a[i + 63 + lane] : 0;
        }
        const int ra = __builtin_amdgcn_readlane(achunk, (i - 1) & 63);
        const uint32_t srow = (ra & 2) ? ((ra & 1) ? sa.sr[3] : sa.sr[2]) : ((ra & 1) ? sa.sr[1] : sa.sr[0]);
        const int oa2 = (i == 1) ? goh : go2;   // open_A[i-1] + goh
        // diagonal inputs of the lane's first column: lane k-1's last column
        // of the previous row, or the cell left of the window for lane 0
        const int dM0 = shr1_old(Mp[C - 1], ldM), dD0 = shr1_old(Dp[C - 1], ldD), dI0 = shr1_old(Ip[C - 1], ldI);
        uint32_t bits = 0;
        // pass 1, right to left: D'(i,j) and M(i,j) from row i-1
        static_for(std::make_integer_sequence<int, C>{}, [&](auto ic) {
            constexpr int c = C - 1 - decltype(ic)::value;
            constexpr uint32_t K = 1u << (4 * c);
            const int md = Mp[c] + oa2;
            const bool tD = md >= Dp[c];
            const int Dn = max(md, Dp[c]);
            const int dM = c ? Mp[c > 0 ? c - 1 : 0] : dM0;
            const int dD = c ? Dp[c > 0 ? c - 1 : 0] : dD0;
            const int dI = c ? Ip[c > 0 ? c - 1 : 0] : dI0;
            const int best = max(max(dM, dD), dI);
            uint32_t srcK = (dM != best) ? ((dD == best) ? K : 2u * K) : 0u;
            const int sc = (int)__builtin_amdgcn_ubfe(srow, bsh[c], 8) - SBIAS;
            int Mn = sc + best;
            if (c == 0 && la == 1 && i == 1 && bi == 0 && lane == 0) {
                // one-row quirk: with LA == 1, M(1,1) carries close_A[0] and a 'D' bit
                Mn = sc + goh;
                srcK = K;
            }
            Mp[c] = Mn;
            Dp[c] = Dn;
            bits |= srcK | (tD ? 4u * K : 0u);
        });
        // pass 2: I'(i,j) = max(I'(i,j-1), M(i,j-1) + open_B[j-1] + goh) along the row
        const int mleft = shr1_old(Mp[C - 1], NEG);   // M(i, first column - 1); left of the window: NEG
        const int j1 = bi + lane * C + 1;                // the lane's first column
        int cand[C], pre[C];
        int run = NEG;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int mprev = c ? Mp[c > 0 ? c - 1 : 0] : mleft;
            cand[c] = mprev + ((j1 + c == 1) ? goh : go2);
            run = max(run, cand[c]);
            pre[c] = run;
        }
        // exclusive prefix maximum of the lane totals across the wave
        int v = run;
        v = max(v, row_shr_old(v, NEG, 1));
        v = max(v, row_shr_old(v, NEG, 2));
        v = max(v, row_shr_old(v, NEG, 4));
        v = max(v, row_shr_old(v, NEG, 8));
        const int t15 = __builtin_amdgcn_readlane(v, 15), t31 = __builtin_amdgcn_readlane(v, 31);
        const int t47 = __builtin_amdgcn_readlane(v, 47);
        const int r1 = t15, r2 = max(t15, t31), r3 = max(r2, t47);
        v = max(v, lane >= 48 ? r3 : (lane >= 32 ? r2 : (lane >= 16 ? r1 : NEG)));
        const int leftI = bi == 0 ? NEG + goh : NEG;    // I'(i, window start - 1)
        const int excl = shr1_old(v, leftI);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int iprev = c ? max(excl, pre[c > 0 ? c - 1 : 0]) : excl;
            const bool tI = cand[c] >= iprev;
            Ip[c] = max(iprev, cand[c]);
            bits |= tI ? (8u << (4 * c)) : 0u;
        }
        const int sub = (i - 1) % RPD;
        tbw |= bits << (4 * C * sub);
        if (sub == RPD - 1 || i == la) {
            tbj[(size_t)((i - 1) / RPD) * 64 + lane] = tbw;
            tbw = 0;
        }
        if (i == la && lane == 63) {
            finM = Mp[C - 1];
            finD = Dp[C - 1];
            finI = Ip[C - 1];
        }
        bprev = bi;
    }
    // the final pick, in lane 63
    finD -= goh;
    finI -= goh;
    score = finM;
    edge = 'M';
    if (finD > score) { score = finD; edge = 'D'; }
    if (finI > score) { score = finI; edge = 'I'; }
}

// Narrow jobs (lb <= 16): one lane per job.  The lane keeps a whole row in
// registers and walks the rows of A with dp_job's row step; columns past lb are
// computed and ignored (nothing flows leftwards).  The left boundary is column
// 0 and the top row 0, as for the first stripe of dp_job.  Trace: 8 bytes per
// row, cell (i, j) at byte (i-1)*8 + (j-1)/2, nibble (j-1)%2.
constexpr int TINY_LB = 16;
constexpr uint32_t TINY_COLS_TAG = 128;   // DevJob::cols of a one-lane job

__device__ __forceinline__ void tiny_job(const DevJob &jb, const uint8_t *__restrict__ A,
                                         const uint8_t *__restrict__ B, uint8_t *__restrict__ tb,
                                         const ScoreArgs &sc, int &score, int &edge)
{
    const int la = (int)jb.la, lb = (int)jb.lb;
    const uint8_t *a = A + jb.a_off;
    const uint8_t *b = B + jb.b_off;
    uint8_t *tbj = tb + jb.tb_off;
    IntCell::Lane<TINY_LB> st;
    IntCell::init<TINY_LB>(st, [&](int c) { return c < lb ? (uint32_t)b[c] : 0u; }, true, true);
    int diag = IntCell::corner(la);
    for (int i = 1; i <= la; ++i) {
        int lo, hi;
        IntCell::operand(sc, a[i - 1], lo, hi);
        IntCell::row<TINY_LB>(st, nullptr, lo, hi, diag, IntCell::neg_f());
        diag = IntCell::edge();
        store_records<TINY_LB>(tbj + (size_t)(i - 1) * 8, st.word);
    }
    int h = 0, e = 0, f = 0;
#pragma unroll
    for (int c = 0; c < TINY_LB; ++c)
        if (c == lb - 1) { h = st.H[c]; e = st.E[c]; f = st.F[c]; }
    const uint32_t w = lb > 8 ? st.word[1] : st.word[0];
    IntCell::pick(h, e, f, (w >> (4 * ((lb - 1) & 7))) & 15u, 0, 0, 0, score, edge);
}

__device__ __forceinline__ void put_result(const DevJob &jb, bool ok, int score, int pos, int64_t maxdev,
                                           mh_dp_result *__restrict__ res, uint32_t *__restrict__ dev)
{
    mh_dp_result r;
    r.score = score;
    r.path_len = ok ? jb.la + jb.lb - (uint32_t)pos : 0u;
    r.path_start = jb.path_off + (uint64_t)pos;
    res[jb.user] = r;
    if (dev) dev[jb.user] = ok ? (uint32_t)((maxdev + jb.la - 1) / jb.la) : 0xFFFFFFFFu;
}

// BitTraceBack (MU/bittraceback.cpp:138-209) by the G lanes that computed the
// job (64 lanes for a job whose stripes other wavefronts computed): the walk
// from (LA, LB) writes the edges backwards into the job's path slot and records
// the path's largest distance from the corner-to-corner line, ceil(max |i*LB -
// j*LA| / LA) over the visited positions, which is the band label and the edge
// test of a banded job.
//
// A step reads the records of the next G positions in the walk's direction (M
// along the diagonal, D up the column, I along the row) at once, a lane each;
// a ballot finds the first whose record leaves the state, and the walk moves
// there.  So it costs one round of loads per run of one state (or per G
// positions, or stripe), and runs are long: substitutions do not end one, only
// indels do.  It follows the forward pass on the same wavefront, whose records
// are still in the L2, while other wavefronts compute.  (20,000 jobs of 5 to 500
// columns walked by a thread each in a kernel of its own: 424 us after a forward
// pass of 648 us; together now 407 us.)
template <int G>
__device__ __forceinline__ void walk_group(const DevJob &jb, const uint8_t *tb, uint8_t *__restrict__ paths,
                                           mh_dp_result *__restrict__ res, uint32_t *__restrict__ dev, int score,
                                           int edge)
{
    const int lane = (int)threadIdx.x & (G - 1), gb = (int)threadIdx.x & 63 & ~(G - 1);
    const int la = (int)jb.la, lb = (int)jb.lb;
    const int cols = G == 16 ? (int)(jb.cols - GROUP_TAG) : (int)jb.cols, sw = G * cols;
    const int lane_bytes = (int)lane_bytes_of((uint32_t)cols);
    const uint32_t inv = (65536u + (uint32_t)cols - 1u) / (uint32_t)cols;   // x / cols = x * inv >> 16 below 4096
    const uint8_t *tj = tb + jb.tb_off;
    uint8_t *slot = paths + jb.path_off;
    // the trace block of the last stripe: the sum over the stripes before it
    int cur = (lb - 1) / sw, r0 = 1, r1 = 0;
    uint64_t base = 0;
    for (int s = 0; s < cur; ++s) {
        int a0, a1;
        stripe_rows(jb.la, jb.lb, jb.band, sw, s, a0, a1);
        if (a1 >= a0) base += (uint64_t)(a1 - a0 + G) * G * lane_bytes;
    }
    stripe_rows(jb.la, jb.lb, jb.band, sw, cur, r0, r1);
    int i = la, j = lb, pos = la + lb, type = edge;
    int co = (lb - 1) - cur * sw;        // j's column in its stripe, from 0
    int64_t dnum = 0, maxdev = 0;        // i*lb - j*la
    bool ok = true;
    while (i > 0 && j > 0) {
        const int up = type != 'I', left = type != 'D';
        if (left && co == 0 && cur > 0) {
            // the next position lies in the previous stripe: back over its trace block
            --cur;
            stripe_rows(jb.la, jb.lb, jb.band, sw, cur, r0, r1);
            if (r1 >= r0) base -= (uint64_t)(r1 - r0 + G) * G * lane_bytes;
            co = sw;
        }
        const int ci = i - (up ? 1 + lane : 0), o = co - (left ? 1 + lane : 0);
        const bool in = ci >= 1 && ci >= r0 && ci <= r1 && o >= 0;
        uint32_t nib = 0;
        if (in) {
            const int kl = (int)(((uint32_t)o * inv) >> 16), c = o - kl * cols;
            const uint32_t byte = tj[base + ((uint64_t)(ci - r0 + kl) * G + kl) * lane_bytes + (c >> 1)];
            nib = (byte >> (4 * (c & 1))) & 15u;
        }
        uint64_t vm = __ballot(in), sm = __ballot(in && walk_stays(nib, type));
        if constexpr (G < 64) {
            vm = (vm >> gb) & ((1ull << (G & 63)) - 1);
            sm = (sm >> gb) & ((1ull << (G & 63)) - 1);
        }
        const int cnt = ~vm ? __builtin_ctzll(~vm) : 64, n = ~sm ? __builtin_ctzll(~sm) : 64;
        const uint32_t nn = (uint32_t)__shfl((int)nib, gb + (n < G ? n : 0), 64);
        int e, next;
        if (n < cnt) {
            e = n + 1;
            next = (int)walk_next(nn, type);
        } else if (cnt > 0) {
            e = cnt;
            next = type;
        } else {
            // onto row 0 or column 0 (by an M edge, or along the edge itself), or out of the region
            e = 1;
            const int i1 = i - up, j1 = j - left;
            if ((i1 > 0 && j1 > 0) || (type == 'D' && j1 > 0) || (type == 'I' && i1 > 0)) {
                ok = false;
                break;
            }
            next = type;
        }
        if (lane < e) slot[pos - 1 - lane] = (uint8_t)type;
        pos -= e;
        const int64_t dd = (up ? -(int64_t)lb : 0) + (left ? (int64_t)la : 0);
        const int64_t d1 = dnum + dd, d2 = dnum + (int64_t)e * dd;
        maxdev = max(maxdev, max(d1 < 0 ? -d1 : d1, d2 < 0 ? -d2 : d2));
        dnum = d2;
        if (up) i -= e;
        if (left) {
            j -= e;
            co -= e;
        }
        type = next;
    }
    if (ok) {
        // along the edge to the corner
        const int rest = i + j;
        const uint8_t t = i > 0 ? 'D' : 'I';
        for (int x = lane; x < rest; x += G) slot[pos - 1 - x] = t;
        pos -= rest;
    }
    if (lane == 0) put_result(jb, ok, score, pos, maxdev, res, dev);
}

// The walk of a one-lane job by its lane, eight positions looked at at once.
__device__ __forceinline__ void walk_tiny(const DevJob &jb, const uint8_t *tb, uint8_t *__restrict__ paths,
                                          mh_dp_result *__restrict__ res, uint32_t *__restrict__ dev, int score,
                                          int edge)
{
    constexpr int AHEAD = 8;
    const int la = (int)jb.la, lb = (int)jb.lb;
    const uint8_t *tj = tb + jb.tb_off;
    uint8_t *slot = paths + jb.path_off;
    int i = la, j = lb, pos = la + lb, type = edge;
    int64_t dnum = 0, maxdev = 0;
    bool ok = true;
    while (i > 0 && j > 0) {
        const int up = type != 'I', left = type != 'D';
        uint32_t nib[AHEAD];
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) {
            const int ci = i - up * (1 + d), cj = j - left * (1 + d);
            nib[d] = 16;
            if (ci >= 1 && cj >= 1) nib[d] = ((uint32_t)tj[(uint64_t)(ci - 1) * 8 + ((cj - 1) >> 1)] >> (4 * ((cj - 1) & 1))) & 15u;
        }
        int e = 0, next = type;
        bool stay = true;
#pragma unroll
        for (int d = 0; d < AHEAD; ++d)
            if (stay && nib[d] < 16) {
                ++e;
                stay = walk_stays(nib[d], type);
                if (!stay) next = (int)walk_next(nib[d], type);
            } else {
                stay = false;
            }
        if (e == 0) {
            e = 1;
            const int i1 = i - up, j1 = j - left;
            if ((type == 'D' && j1 > 0) || (type == 'I' && i1 > 0)) {
                ok = false;
                break;
            }
        }
        for (int d = 0; d < e; ++d) slot[pos - 1 - d] = (uint8_t)type;
        pos -= e;
        const int64_t dd = (up ? -(int64_t)lb : 0) + (left ? (int64_t)la : 0);
        const int64_t d1 = dnum + dd, d2 = dnum + (int64_t)e * dd;
        maxdev = max(maxdev, max(d1 < 0 ? -d1 : d1, d2 < 0 ? -d2 : d2));
        dnum = d2;
        i -= up * e;
        j -= left * e;
        type = next;
    }
    if (ok) {
        const uint8_t t = i > 0 ? 'D' : 'I';
        for (int rest = i + j; rest > 0; --rest) slot[--pos] = t;
    }
    put_result(jb, ok, score, pos, maxdev, res, dev);
}

// The walk of a sliding-window job by one lane; its records are the
// reference's code at the cell the walk leaves (dp_window_job).
__device__ __forceinline__ void walk_window(const DevJob &jb, const uint8_t *tb, uint8_t *__restrict__ paths,
                                            mh_dp_result *__restrict__ res, uint32_t *__restrict__ dev, int score,
                                            int edge)
{
    const int la = (int)jb.la, lb = (int)jb.lb;
    const uint32_t *tj = reinterpret_cast<const uint32_t *>(tb + jb.tb_off);
    uint8_t *slot = paths + jb.path_off;
    const int C = (int)jb.cols - (int)WINDOW_TAG, rpd = 8 / C;
    int pos = la + lb, i = la, j = lb, type = edge;
    int64_t dnum = 0, maxdev = 0;
    bool ok = true;
    for (;;) {
        slot[--pos] = (uint8_t)type;
        uint32_t nib = 0;
        if (i > 0 && j > 0) {
            const int xw = j - window_base(la, lb, 64 * C, i) - 1;
            if (xw < 0 || xw >= 64 * C) { ok = false; break; }
            const uint32_t w = tj[(uint64_t)((i - 1) / rpd) * 64 + xw / C];
            nib = (w >> (4 * (C * ((i - 1) % rpd) + xw % C))) & 15u;
        }
        int nx;
        if (type == 'M') {
            const uint32_t v = nib & 3u;
            nx = v == 0 ? 'M' : (v == 1 ? 'D' : (v == 2 ? 'I' : '?'));
            if (i == 0 || j == 0) { ok = false; break; }
            --i;
            --j;
            dnum += (int64_t)la - lb;
        } else if (type == 'D') {
            nx = (nib & 4u) ? 'M' : 'D';
            if (i == 0) { ok = false; break; }
            --i;
            dnum -= lb;
        } else {
            nx = (nib & 8u) ? 'M' : 'I';
            if (j == 0) { ok = false; break; }
            --j;
            dnum += la;
        }
        maxdev = max(maxdev, dnum < 0 ? -dnum : dnum);
        if (i == 0 && j == 0) break;
        if (pos == 0 || nx == '?') { ok = false; break; }
        type = nx;
    }
    put_result(jb, ok, score, pos, maxdev, res, dev);
}

// ---- the round's launches ------------------------------------------------

__global__ __launch_bounds__(64) void dp_queue_reset(uint32_t *__restrict__ cursor)
{
    for (int k = threadIdx.x; k < DPQ_CURSORS; k += 64) cursor[k] = 0u;
}

// The forward kernels' arguments: every pointer restrict-qualified (so that
// job records and the bin table are read with scalar loads; the walk reads the
// trace the same wavefront wrote, through tb itself), the bin table in the
// round's descriptor.
#define DP_FWD_PARAMS                                                                                            \
    const DevJob *__restrict__ jobs, DpOut *__restrict__ outs, const uint8_t *__restrict__ A,                      \
        const uint8_t *__restrict__ B, uint8_t *tb, int *__restrict__ bnd, const DpRound *__restrict__ rd,       \
        uint32_t *__restrict__ cursor, uint8_t *__restrict__ paths, mh_dp_result *__restrict__ res,              \
        uint32_t *__restrict__ dev, ScoreArgs sc
#define DP_FWD_ARGS jobs, outs, A, B, tb, bnd, rd, cursor, paths, res, dev, sc

// one work item: the forward pass of its jobs and their walks (a pipelined
// part only its stripes; the job's walk waits for the others, dp_tb_wave)
template <class CELL, int MAXC>
__device__ __forceinline__ void run_item(DP_FWD_PARAMS, const float *table, uint32_t kind, uint32_t first,
                                         uint32_t count, uint32_t item, DpLds &lds)
{
    int score = 0, edge = 'M';
    if (kind >= QK_PIPE) {
        const uint32_t P = kind - QK_PIPE + 1;
        const uint32_t x = first + item / P;
        const int p0 = (int)(item % P);
        const DevJob jb = jobs[x];
        uint32_t *err = cursor + (DPQ_CURSORS - 1);
        bool fin = false;
        if (MAXC >= 16 && jb.cols == 16) {
            if constexpr (MAXC >= 16)
                fin = dp_job<CELL, 16, 64, true>(jb, A, B, tb, bnd, sc, table, lds, score, edge, p0, (int)P, err);
        } else if (jb.cols == 8) {
            fin = dp_job<CELL, 8, 64, true>(jb, A, B, tb, bnd, sc, table, lds, score, edge, p0, (int)P, err);
        } else if (std::is_same<CELL, IntCell>::value && jb.cols <= 2) {
            if constexpr (std::is_same<CELL, IntCell>::value) {
                if (jb.cols == 2) fin = dp_job<CELL, 2, 64, true>(jb, A, B, tb, bnd, sc, table, lds, score, edge, p0, (int)P, err);
                else fin = dp_job<CELL, 1, 64, true>(jb, A, B, tb, bnd, sc, table, lds, score, edge, p0, (int)P, err);
            }
        } else {
            fin = dp_job<CELL, 4, 64, true>(jb, A, B, tb, bnd, sc, table, lds, score, edge, p0, (int)P, err);
        }
        if (fin && threadIdx.x == 0) {
            outs[x].score = score;
            outs[x].edge = edge;
        }
    } else if (kind == QK_STRIPE) {
        const DevJob jb = jobs[first + item];
        if (MAXC >= 16 && jb.cols == 16) {
            if constexpr (MAXC >= 16) dp_job<CELL, 16, 64>(jb, A, B, tb, bnd, sc, table, lds, score, edge);
        } else if (jb.cols == 8) {
            dp_job<CELL, 8, 64>(jb, A, B, tb, bnd, sc, table, lds, score, edge);
        } else {
            dp_job<CELL, 4, 64>(jb, A, B, tb, bnd, sc, table, lds, score, edge);
        }
        walk_group<64>(jb, tb, paths, res, dev, score, edge);
    } else if (kind == QK_WINDOW) {
        if constexpr (std::is_same<CELL, IntCell>::value) {
            const DevJob jb = jobs[first + item];
            switch (jb.cols - WINDOW_TAG) {
            case 1: dp_window_job<1>(jb, A, B, tb, sc, score, edge); break;
            case 2: dp_window_job<2>(jb, A, B, tb, sc, score, edge); break;
            case 4: dp_window_job<4>(jb, A, B, tb, sc, score, edge); break;
            default: dp_window_job<8>(jb, A, B, tb, sc, score, edge); break;
            }
            __threadfence_block();
            if (threadIdx.x == 63) walk_window(jb, tb, paths, res, dev, score, edge);
        }
    } else if (kind == QK_TINY) {
        if constexpr (std::is_same<CELL, IntCell>::value) {
            const uint32_t x = first + item * 64 + threadIdx.x;
            if (x < first + count) {
                const DevJob jb = jobs[x];
                tiny_job(jb, A, B, tb, sc, score, edge);
                __threadfence_block();
                walk_tiny(jb, tb, paths, res, dev, score, edge);
            }
        }
    } else {
        // four jobs of one shape, one per 16-lane row; a row past the bin's end sits out
        const uint32_t x = first + item * 4 + (threadIdx.x >> 4);
        if (x >= first + count) return;
        const DevJob jb = jobs[x];
        switch (kind - QK_ROWS) {
        case 0: if constexpr (MAXC >= 16) dp_job<CELL, 16, 16>(jb, A, B, tb, bnd, sc, table, lds, score, edge); break;
        case 1: if constexpr (MAXC >= 14) dp_job<CELL, 14, 16>(jb, A, B, tb, bnd, sc, table, lds, score, edge); break;
        case 2: if constexpr (MAXC >= 12) dp_job<CELL, 12, 16>(jb, A, B, tb, bnd, sc, table, lds, score, edge); break;
        case 3: if constexpr (MAXC >= 10) dp_job<CELL, 10, 16>(jb, A, B, tb, bnd, sc, table, lds, score, edge); break;
        case 4: dp_job<CELL, 8, 16>(jb, A, B, tb, bnd, sc, table, lds, score, edge); break;
        case 5: dp_job<CELL, 6, 16>(jb, A, B, tb, bnd, sc, table, lds, score, edge); break;
        default: dp_job<CELL, 4, 16>(jb, A, B, tb, bnd, sc, table, lds, score, edge); break;
        }
        walk_group<16>(jb, tb, paths, res, dev, score, edge);
    }
}

// The forward launch.  MAXC is the widest shape it holds (16: every shape;
// 8: stripes and row shapes of at most 8 columns a lane, which need fewer
// registers and so fit more wavefronts a SIMD).  PERSIST: a grid of resident
// wavefronts, each taking the next item from the bins' atomic cursors until
// the last bin is empty.  Otherwise one workgroup per item in queue order
// (workgroup w takes item w; workgroups start in that order), which needs no
// cursor.  The host picks the variant a round's shapes allow, by the tuning
// table.
template <class CELL, int MAXC, int WPE, bool PERSIST>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE))) void dp_fwd(DP_FWD_PARAMS)
{
    __shared__ DpLds lds;
    __shared__ float table_s[DP_NCLASS * DP_NCLASS];
    const float *table = nullptr;
    if constexpr (!std::is_same<CELL, IntCell>::value) {
        if (threadIdx.x < DP_NCLASS * DP_NCLASS) table_s[threadIdx.x] = rd->table[threadIdx.x];
        __syncthreads();
        table = table_s;
    }
    const uint32_t nb = rd->nbins;
    if constexpr (!PERSIST) {
        const uint32_t w = blockIdx.x;
        if (nb == 0 || w >= rd->bin[nb].item0) return;
        uint32_t b = 0;    // the last bin that starts at or before item w
        for (uint32_t len = nb; len > 1;) {
            const uint32_t half = len >> 1;
            if (rd->bin[b + half].item0 <= w) { b += half; len -= half; }
            else len = half;
        }
        uint32_t item = w - rd->bin[b].item0;
        if (rd->bin[b].kind >= QK_PIPE) {
            // a ticket, so that the parts of a job are taken in order by
            // running wavefronts (a part waits only on parts taken before it)
            uint32_t v = 0;
            if (threadIdx.x == 0) v = atomicAdd(&cursor[b], 1u);
            item = (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
        }
        run_item<CELL, MAXC>(DP_FWD_ARGS, table, rd->bin[b].kind, rd->bin[b].first, rd->bin[b].count, item, lds);
    } else {
        uint32_t b = 0;
        for (;;) {
            // the next item: the first bin whose cursor is still inside it
            uint32_t item = 0;
            for (; b < nb; ++b) {
                uint32_t v = 0;
                if (threadIdx.x == 0) v = atomicAdd(&cursor[b], 1u);
                item = (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
                if ((uint64_t)item * qk_per_item(rd->bin[b].kind) < rd->bin[b].count) break;
            }
            if (b >= nb) return;
            run_item<CELL, MAXC>(DP_FWD_ARGS, table, rd->bin[b].kind, rd->bin[b].first, rd->bin[b].count, item, lds);
        }
    }
}

// The walks of the pipelined jobs (the first npipe of the table), a wavefront
// each, once the forward launch has ended.
__global__ __launch_bounds__(64) void dp_tb_wave(const DevJob *__restrict__ jobs, const DpOut *__restrict__ outs,
                                                 const uint8_t *__restrict__ tb, uint8_t *__restrict__ paths,
                                                 mh_dp_result *__restrict__ res, uint32_t *__restrict__ dev,
                                                 uint32_t npipe)
{
    if (blockIdx.x >= npipe) return;
    const DevJob jb = jobs[blockIdx.x];
    walk_group<64>(jb, tb, paths, res, dev, outs[blockIdx.x].score, outs[blockIdx.x].edge);
}

// NUC_SP (MU/nucmx.cpp:8-25) as the kernels take it (ScoreArgs)
void packed_rows(ScoreArgs &sc)
{
    static const int hoxd[4][4] = {{91, -114, -31, -123},
                                   {-114, 100, -125, -31},
                                   {-31, -125, 100, -114},
                                   {-123, -31, -114, 91}};
    for (int a = 0; a < 4; ++a) {
        uint32_t h[4];
        sc.sr[a] = 0;
        for (int b = 0; b < 4; ++b) {
            const int v = hoxd[a][b] + 60;
            sc.sr[a] |= (uint32_t)(v + SBIAS) << (8 * b);
            h[b] = (uint32_t)(uint16_t)(int16_t)(4 * v);
        }
        sc.lo[a] = h[0] | (h[1] << 16);
        sc.hi[a] = h[2] | (h[3] << 16);
    }
}

}  // namespace

namespace {

struct DpItem {
    uint32_t job;     // index in the caller's job array
    uint32_t band;    // 0 = full matrix
    uint32_t cols;
    uint64_t tb_bytes;
    uint64_t cells;   // of the region evaluated, padding included
    uint32_t parts;   // wavefronts that share its stripes (0: not pipelined)
};

// Relative cost per computed cell of the stripe shapes, used to pick a banded
// job's shape (which decides how much of each stripe lies outside the band).
// Per shape alone (one class of B's width at a time, MI355X) 64-lane stripes
// of 16 columns evaluate cells fastest and 16-lane stripes slowest (2-4x),
// but a round's shapes share one forward kernel, and weights taken from those
// runs pick more 16-column stripes, whose wide kernel then slows the round's
// other jobs.  These weights were chosen by timing whole banded runs (learned
// and constant bands, edge fallback included) over 100k training gaps: the
// fastest learned-band run of the sets tried, on cells of 348 instructions a
// 16-column step.  They decide the regions, and so the results of bands without
// the fallback, and were not measured again on the present cells.
constexpr double COST_PER_CELL[3] = {1.34, 1.00, 1.30};   // 64-lane stripes of cols 4, 8, 16
constexpr double COST_PER_CELL_G16[2] = {2.40, 1.50};      // 16-lane stripes of cols 4, 8


}  // namespace

// Scratch of the no-allocation entry point (mh_dp_align_device_noalloc): the
// round's job table, stripe boundary columns and trace arena, in one array
// that every GPU the library runs on holds until the process ends.  Host code
// never uses the array's name: each device's address comes from
// hipGetSymbolAddress, resolved once per device by dp_scratch_init.
constexpr uint64_t DP_SCRATCH_BYTES = 64ull << 20;
static __device__ __align__(256) uint8_t scratch[DP_SCRATCH_BYTES];

namespace {
constexpr int DP_SCRATCH_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
uint8_t *g_scratch_ptr[DP_SCRATCH_MAX_DEVICES] = {};
}  // namespace

int dp_scratch_init(int device)
{
    MH_CHECK(device >= 0 && device < DP_SCRATCH_MAX_DEVICES, MH_ERR_UNSUPPORTED, "device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return MH_OK;
    int cur = -1;
    MH_HIP(hipGetDevice(&cur));
    MH_CHECK(cur == device, MH_ERR_INVALID, "dp_scratch_init: device is not current");
    void *ptr = nullptr;
    MH_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    MH_CHECK(ptr != nullptr, MH_ERR_DEVICE, "hipGetSymbolAddress gave a null address for the DP scratch");
    g_scratch_ptr[device] = static_cast<uint8_t *>(ptr);
    return MH_OK;
}

uint64_t dp_scratch_bytes() { return DP_SCRATCH_BYTES; }

// The banded shapes' weights: COST_PER_CELL, COST_PER_CELL_G16, or five
// comma-separated values in MH_DP_BAND_COST (read once per process, for sweeps)
static const double *band_cost_weights()
{
    static double w[5];
    static std::once_flag once;
    std::call_once(once, [] {
        for (int q = 0; q < 5; ++q) w[q] = q < 3 ? COST_PER_CELL[q] : COST_PER_CELL_G16[q - 3];
        const char *e = getenv("MH_DP_BAND_COST");
        if (!e) return;
        double v[5];
        int n = 0;
        for (const char *p = e; *p && n < 5;) {
            char *end = nullptr;
            const double x = strtod(p, &end);
            if (end == p || !(x > 0.0)) return;
            v[n++] = x;
            p = *end == ',' ? end + 1 : end;
        }
        if (n == 5) std::memcpy(w, v, sizeof(v));
    });
    return w;
}

// MH_DP_COLS forces one shape: 4, 8 or 16 (64-lane stripes of that many
// columns a lane) or 36, 40 (16-lane stripes of 4, 8 columns, four jobs a
// wavefront)
int dp_force_cols()
{
    if (const char *e = getenv("MH_DP_COLS")) {
        const int c = atoi(e);
        if (c == 4 || c == 8 || c == 16 || c == (int)GROUP_TAG + 4 || c == (int)GROUP_TAG + 8) return c;
    }
    return 0;
}

// class of B's width in the tuning table
static int dp_tune_class(uint32_t lb)
{
    int c = 0;
    while (c < DP_TUNE_NCLASS - 1 && lb > DP_TUNE_LB_CLASS[c]) ++c;
    return c;
}

// The full DP's shape per class: the tuning table, or MH_DP_SHAPES (a comma
// list of DP_TUNE_NCLASS values, each 0, 4, 8 or 16; read once per process,
// for the tuner's sweeps)
static const uint8_t *shape_table()
{
    static uint8_t t[DP_TUNE_NCLASS];
    static std::once_flag once;
    std::call_once(once, [] {
        for (int c = 0; c < DP_TUNE_NCLASS; ++c) t[c] = DP_TUNE_SHAPE[c];
        const char *e = getenv("MH_DP_SHAPES");
        if (!e) return;
        uint8_t v[DP_TUNE_NCLASS];
        int c = 0;
        for (const char *p = e; *p && c < DP_TUNE_NCLASS;) {
            char *end = nullptr;
            const long x = strtol(p, &end, 10);
            if (end == p || !(x == 0 || x == 4 || x == 8 || x == 16)) return;
            v[c++] = (uint8_t)x;
            p = *end == ',' ? end + 1 : end;
        }
        if (c == DP_TUNE_NCLASS) std::memcpy(t, v, sizeof(v));
    });
    return t;
}

// Stripe shape of a job: the full DP takes the shape the tuning table names
// for B's width (stripes of 8 columns a lane where it names the row-packed
// shape and the job cannot take it); a banded job takes the shape with the
// lowest estimated cost: ceil(lb/w) stripes of min(la, la*(w+2W)/lb + 1) +
// g - 1 steps of w cells (g lanes), times the shape's cost per cell.  force
// (any MH_DP_COLS shape) overrides.  A rerun pass holds few jobs, whose time
// is the longest job's: its banded jobs take 64-lane stripes only
// (wide_only), since a 16-lane stripe runs one job on a quarter of a
// wavefront.
uint32_t dp_cols_for(uint32_t la, uint32_t lb, uint32_t band, int force, bool wide_only)
{
    if (force) return (uint32_t)force;
    if (band == 0) {
        const uint32_t t = shape_table()[dp_tune_class(lb)];
        return t ? t : 8u;
    }
    // 64-lane stripes of 4, 8 or 16 columns a lane, and (unless
    // MH_DP_BAND_G16=0) 16-lane stripes of 4 or 8 columns a lane, four jobs a
    // wavefront: narrower stripes, whose rows follow a narrow band closer
    uint32_t best = 16;
    double best_cost = 0;
    const char *g16e = getenv("MH_DP_BAND_G16");
    const int nshape = wide_only || (g16e && g16e[0] == '0') ? 3 : 5;
    const double *wt = band_cost_weights();
    for (int q = 0; q < nshape; ++q) {
        const uint32_t g = q < 3 ? 64u : 16u;
        const uint32_t c = q < 3 ? 4u << q : 4u << (q - 3), sw = g * c;
        const double ns = (double)((lb + sw - 1) / sw);
        double rows = (double)la * (sw + 2.0 * band) / lb + 1.0;
        if (rows > la) rows = la;
        const double cost = ns * (rows + (g - 1.0)) * sw * wt[q];
        if (q == 0 || cost < best_cost) {
            best = g == 64 ? c : GROUP_TAG + c;
            best_cost = cost;
        }
    }
    return best;
}

// The sliding window spends much of each row on the shift and the cross-lane
// scan: measured on MI355X over 100k learned bands it evaluates its cells
// about 1.45x slower than the stripes evaluate theirs and saves fewer cells
// than that, so the scheduler uses it only when MH_DP_BAND_KIND=window asks.
int dp_force_kind()
{
    if (const char *e = getenv("MH_DP_BAND_KIND")) {
        if (!strcmp(e, "stripes")) return 1;
        if (!strcmp(e, "window")) return 2;
    }
    return 0;
}

// Columns per lane of the sliding window for a banded region (0: use
// stripes): when the window is asked for (kind 2), the narrowest window
// reaching the region band on each side of the line (64C >= 2R+2), if it is
// narrower than B and the slope lb/la is at most 4.
uint32_t dp_window_cols(uint32_t la, uint32_t lb, uint32_t band, int kind)
{
    if (band == 0 || kind != 2 || (uint64_t)lb > 4ull * la) return 0;
    int q = 0;
    while (q < 4 && 64u * (1u << q) < 2u * band + 2u) ++q;
    if (q == 4) return 0;
    const uint32_t c = 1u << q;
    if (64u * c >= lb) return 0;
    return c;
}

uint32_t dp_stripe_width(uint32_t cols) { return cols > GROUP_TAG ? 16 * (cols - GROUP_TAG) : 64 * cols; }

// A band whose region is the whole matrix is the full DP.
uint32_t dp_effective_band(uint32_t la, uint32_t lb, uint32_t band, uint32_t cols)
{
    if (band == 0) return 0;
    const uint32_t sw = cols > GROUP_TAG ? 16 * (cols - GROUP_TAG) : 64 * cols;
    const uint32_t ns = (lb + sw - 1) / sw;
    int f0, f1, l0, l1;
    stripe_rows(la, lb, band, sw, 0, f0, f1);
    stripe_rows(la, lb, band, sw, ns - 1, l0, l1);
    return (l0 == 1 && f1 == (int)la) ? 0u : band;
}

static inline uint64_t align256(uint64_t v) { return (v + 255) & ~255ull; }

// device bytes of a round's descriptor with room for `bins` bins, and its queue cursors
static constexpr uint64_t dp_cursor_at(uint32_t bins) { return offsetof(DpRound, bin) + (bins + 1) * sizeof(DpBin); }
static constexpr uint64_t dp_round_bytes(uint32_t bins) { return (dp_cursor_at(bins) + DPQ_CURSORS * 4 + 255) & ~255ull; }

// The fixed scratch's rounds hold no pipelined jobs, so fewer bins.  A job there
// is refused by its trace, its boundary at 12 bytes a row and 1,792 bytes, which
// the layout must not exceed.
constexpr uint32_t DPQ_FIXED_MAXB = 48;
static_assert(dp_round_bytes(DPQ_FIXED_MAXB) <= 1280, "the fixed scratch's limit");

// The forward kernel's variants: the widest shape each holds, its
// wavefronts a SIMD, and whether its wavefronts persist.  Rounds with a shape
// wider than 8 columns a lane run the tuning table's wide variant, the others
// its narrow one; MH_DP_VARIANT forces one (for sweeps), where the round's
// shapes allow it.
struct FwdVariant {
    const void *fn;
    int maxc, wpe;
    bool persist;
};
#define MH_FWD(CELL, MAXC, WPE, PERSIST) \
    {reinterpret_cast<const void *>(&dp_fwd<CELL, MAXC, WPE, PERSIST>), MAXC, WPE, PERSIST}
const FwdVariant FWD_VARIANTS[] = {
    MH_FWD(IntCell, 16, 3, false), MH_FWD(IntCell, 8, 4, false), MH_FWD(IntCell, 16, 2, false),
    MH_FWD(IntCell, 16, 3, true),  MH_FWD(IntCell, 16, 2, true), MH_FWD(IntCell, 8, 4, true),
    MH_FWD(IntCell, 16, 4, false),
    // jobs whose scores times four could leave 32 bits; jobs with wildcard letters
    MH_FWD(CmpCell<int>, 16, 2, false), MH_FWD(CmpCell<float>, 16, 2, false),
};
#undef MH_FWD
constexpr int N_ALL_VARIANTS = (int)(sizeof(FWD_VARIANTS) / sizeof(FWD_VARIANTS[0]));
constexpr int N_FWD_VARIANTS = N_ALL_VARIANTS - 2;   // of the tagged int32 cells
constexpr int VARIANT_LONG = N_FWD_VARIANTS, VARIANT_FLOAT = N_FWD_VARIANTS + 1;
static_assert(N_ALL_VARIANTS <= MH_DP_MAX_VARIANTS, "context graph slots");

// The cells a run of jobs takes: tagged int32 (values times four), int32
// without a tag, float.  The tagged form holds |score| < 2^28: a score is at
// most 160 a position of the shorter operand, and a reachable cell of a band at
// least -65 a position, so 225 * 2^20 < 2^28 keeps both apart from minus
// infinity.  Longer jobs (only banded ones can be) keep untagged values.
enum class DpCells { TAGGED, LONG, FLOAT };
constexpr uint32_t TAGGED_MAX = 1u << 20;
static_assert(DP_TUNE_WIDE_VARIANT < N_FWD_VARIANTS && DP_TUNE_NARROW_VARIANT < N_FWD_VARIANTS, "tuning table");

static int dp_variant_for(bool wide)
{
    for (const char *name : {"MH_DP_VARIANT", wide ? "MH_DP_VARIANT_WIDE" : "MH_DP_VARIANT_NARROW"})
        if (const char *e = getenv(name)) {
            const int v = atoi(e);
            if (v >= 0 && v < N_FWD_VARIANTS && (!wide || FWD_VARIANTS[v].maxc >= 16)) return v;
        }
    return wide ? DP_TUNE_WIDE_VARIANT : DP_TUNE_NARROW_VARIANT;
}

// Graph replay of the round's launches (MH_DP_GRAPH=0 launches them directly)
static bool dp_use_graph()
{
    const char *e = getenv("MH_DP_GRAPH");
    return !(e && e[0] == '0');
}

static int dp_round_staging(mh_context *ctx)
{
    if (ctx->dp_round_host) return MH_OK;
    if (hipHostMalloc(&ctx->dp_round_host, sizeof(DpRound), hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        ctx->dp_round_host = nullptr;
        set_error("pinned host allocation failed");
        return MH_ERR_NOMEM;
    }
    return MH_OK;
}

// resident workgroups of a 64-thread kernel over the whole device
static int resident_grid(mh_context *ctx, const void *fn, unsigned *grid)
{
    int cus = 0, per = 0;
    MH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
    MH_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, 64, 0));
    *grid = (unsigned)std::max(1, cus * std::max(1, per));
    return MH_OK;
}

// forward grid of a round: its items, or the resident grid of a persistent variant
static int fwd_grid(mh_context *ctx, int v, uint64_t items, unsigned *g)
{
    if (FWD_VARIANTS[v].persist) {
        if (!ctx->dp_fwd_grid[v]) {
            unsigned r = 0;
            int rc;
            if ((rc = resident_grid(ctx, FWD_VARIANTS[v].fn, &r)) != MH_OK) return rc;
            ctx->dp_fwd_grid[v] = r;
        }
        *g = ctx->dp_fwd_grid[v];
    } else {
        MH_CHECK(items < (1ull << 31), MH_ERR_INVALID, "too many DP work items in one round");
        *g = (unsigned)std::max<uint64_t>(1, items);
    }
    return MH_OK;
}

// the kernels' arguments of a round (DP_FWD_PARAMS; dp_tb_wave)
struct RoundArgs {
    const DevJob *jobs;
    DpOut *outs;
    const uint8_t *A, *B;
    uint8_t *tb;
    int *bnd;
    const DpRound *rd;
    uint32_t *cursor;
    uint8_t *paths;
    mh_dp_result *res;
    uint32_t *dev;
    ScoreArgs sc;
    uint32_t npipe;
    void *fwd[12], *walk[7];
    void set()
    {
        void *a[12] = {&jobs, &outs, &A, &B, &tb, &bnd, &rd, &cursor, &paths, &res, &dev, &sc};
        void *w[7] = {&jobs, &outs, &tb, &paths, &res, &dev, &npipe};
        std::memcpy(fwd, a, sizeof(a));
        std::memcpy(walk, w, sizeof(w));
    }
};

static int launch_fwd(mh_context *ctx, RoundArgs &a, int v, unsigned grid)
{
    a.set();
    hipLaunchKernelGGL(dp_queue_reset, dim3(1), dim3(64), 0, ctx->stream, a.cursor);
    MH_HIP(hipLaunchKernel(FWD_VARIANTS[v].fn, dim3(grid), dim3(64), a.fwd, 0, ctx->stream));
    MH_HIP(hipGetLastError());
    return MH_OK;
}

static int launch_walks(mh_context *ctx, RoundArgs &a)
{
    a.set();
    MH_HIP(hipLaunchKernel(reinterpret_cast<const void *>(&dp_tb_wave), dim3(a.npipe), dim3(64), a.walk, 0,
                           ctx->stream));
    MH_HIP(hipGetLastError());
    return MH_OK;
}

// Captures f's launches on the context stream: the graph (kept, for its
// nodes), its executable form, and the kernel nodes of the given functions.
template <class F>
static int capture(mh_context *ctx, hipGraph_t *graph, hipGraphExec_t *exec, const void *const *fns,
                   hipGraphNode_t *nodes, int nfns, F f)
{
    MH_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    const int rc = f();
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(ctx->stream, &g);
    if (rc != MH_OK) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    MH_HIP(e);
    size_t nn = 0;
    MH_HIP(hipGraphGetNodes(g, nullptr, &nn));
    std::vector<hipGraphNode_t> all(nn);
    MH_HIP(hipGraphGetNodes(g, all.data(), &nn));
    for (int k = 0; k < nfns; ++k) nodes[k] = nullptr;
    for (hipGraphNode_t nd : all) {
        hipGraphNodeType t;
        MH_HIP(hipGraphNodeGetType(nd, &t));
        if (t != hipGraphNodeTypeKernel) continue;
        hipKernelNodeParams kp;
        MH_HIP(hipGraphKernelNodeGetParams(nd, &kp));
        for (int k = 0; k < nfns; ++k)
            if (kp.func == fns[k]) nodes[k] = nd;
    }
    for (int k = 0; k < nfns; ++k)
        if (!nodes[k]) {
            (void)hipGraphDestroy(g);
            MH_CHECK(false, MH_ERR_DEVICE, "a captured DP launch has no kernel node");
        }
    const hipError_t ei = hipGraphInstantiate(exec, g, nullptr, nullptr, 0);
    if (ei != hipSuccess) {
        (void)hipGraphDestroy(g);
        MH_HIP(ei);
    }
    *graph = g;
    return MH_OK;
}

// sets a captured kernel node's grid and arguments in the executable graph
static int set_node(hipGraphExec_t exec, hipGraphNode_t node, unsigned grid, void **args)
{
    hipKernelNodeParams kp;
    MH_HIP(hipGraphKernelNodeGetParams(node, &kp));
    kp.gridDim = dim3(grid);
    kp.kernelParams = args;
    kp.extra = nullptr;
    MH_HIP(hipGraphExecKernelNodeSetParams(exec, node, &kp));
    return MH_OK;
}

// The round's forward launch (queue reset + forward kernel) and the walks of
// its pipelined jobs, timed apart; from graphs captured once per context (the
// descriptor's address is fixed; a round sets the nodes' grids) or launched
// directly.
static int dp_launch_round(mh_context *ctx, int v, bool graph, unsigned grid, RoundArgs &a)
{
    int rc;
    if (graph && a.rd != ctx->dp_round.as<DpRound>()) graph = false;
    if (graph && !ctx->dp_graph_fwd[v]) {
        const void *fns[1] = {FWD_VARIANTS[v].fn};
        if ((rc = capture(ctx, &ctx->dp_graph_fwd_src[v], &ctx->dp_graph_fwd[v], fns, &ctx->dp_graph_fwd_node[v], 1,
                          [&] { return launch_fwd(ctx, a, v, grid); })) != MH_OK)
            return rc;
    }
    if (graph) {
        a.set();
        if ((rc = set_node(ctx->dp_graph_fwd[v], ctx->dp_graph_fwd_node[v], grid, a.fwd)) != MH_OK) return rc;
    }
    {
        TimedLaunch tl(ctx, "dp_forward");
        if (graph) {
            MH_HIP(hipGraphLaunch(ctx->dp_graph_fwd[v], ctx->stream));
        } else if ((rc = launch_fwd(ctx, a, v, grid)) != MH_OK) {
            return rc;
        }
    }
    if (a.npipe) {
        TimedLaunch tl(ctx, "dp_traceback");
        if ((rc = launch_walks(ctx, a)) != MH_OK) return rc;
    }
    return MH_OK;
}

// ints of the boundary columns of an item's job: two values a row, for a
// pipelined job two 64-bit words in each of two buffers
static uint64_t item_bnd_ints(const DpItem &it, const mh_dp_job *jobs)
{
    // one-lane and window jobs hand no column over; a job of 16-lane
    // stripes does when it has more than one (banded jobs)
    if (it.cols == TINY_COLS_TAG || it.cols >= WINDOW_TAG) return 0ull;
    const uint64_t sw = it.cols > GROUP_TAG ? 16ull * (it.cols - GROUP_TAG) : 64ull * it.cols;
    const uint64_t ns = (jobs[it.job].b_len + sw - 1) / sw;
    return ns > 1 ? (it.parts ? 8ull : 2ull) * ((jobs[it.job].a_len + 63) & ~63ull) : 0ull;
}

// bytes of the arena of a round with tbb bytes of trace and bi boundary ints
static uint64_t arena_bytes(uint64_t tbb, uint64_t bi) { return align256(bi * 4) + tbb; }

// an item's part of them (boundary columns are whole multiples of 256 bytes)
static uint64_t item_bytes(const DpItem &it, const mh_dp_job *jobs)
{
    return arena_bytes((it.tb_bytes + 15) & ~15ull, item_bnd_ints(it, jobs));
}

// footprint in a fixed scratch of a round of `cnt` jobs with trace bytes
// tbb (each rounded up to 16) and bi boundary ints
static uint64_t fixed_need(uint64_t cnt, uint64_t tbb, uint64_t bi)
{
    return dp_round_bytes(DPQ_FIXED_MAXB) + align256(cnt * (sizeof(DevJob) + sizeof(DpOut) + 4)) + align256(bi * 4) +
           tbb + 256;
}

// does the fixed scratch take the job (see DPQ_FIXED_MAXB)
static bool fixed_takes(const DpItem &it, const mh_dp_job *jobs, const FixedScratch *fx)
{
    return fixed_need(1, (it.tb_bytes + 15) & ~15ull, item_bnd_ints(it, jobs) / 2 * 3) <= fx->bytes;
}

// Pipelined stripe jobs.  Where the longest job takes longer on its own wavefront
// than the round's work shared evenly by the forward launch's wavefront slots,
// SIMDs would be idle at the end.  Then the jobs above a quarter of a slot's share
// spread their stripes over several wavefronts, and a long banded job of 16-lane
// stripes (a quarter of a wavefront, its stripes one after the other) takes all 64
// lanes, with a quarter of the columns a lane: the same stripes, so the same
// region.  A job's time is its steps times the instructions of a step; with P
// wavefronts it is that of ceil(stripes / P) stripes.  A quarter, since an even end
// is worth more than the lags between parts (46.4 ms on the 4,000 jobs below;
// spreading the jobs above 0.4, 0.6, 0.8 and 1.05 shares 47.9, 50.0, 53.6 and 58.6;
// parts of a whole share 52.3, of two 58.4); equal jobs are left alone (3,072 of
// 2,048 columns 4.9 ms, spread 5.3).  A banded job's stripe starts when the one
// before it has sent the row the stripe starts at, its row shift and the lanes'
// skew later, so more parts than a stripe's steps over that lag would only wait.
// Jobs over all 64 lanes leave fewer SIMDs idle but take two to three times the
// steps, so a round with enough of them is better off without (10,000 banded
// jobs of 1,000 columns, 4 to 100 wide: 0.8 to 2.6 ms without, 2.8 to 6.0 with;
// 50 of 4,000, 100 wide: 5.8 and 1.9).  Where there are such jobs, the round's
// time is estimated with all its long jobs spread, with those of 64 lanes
// alone, and with none, in cycles as measured: a step of a job alone on its SIMD 630
// with one or two columns a lane, 760 or 6.5 an instruction with 16 lanes, 6 an
// instruction in a part; of several on a SIMD 4.2 (4.6 with 16 lanes) an
// instruction, 4 for each of 60 + 14 a column with one or two columns.  The
// estimates fit 60 rounds (equal jobs of 300 to 4,000 columns, log-uniform ones
// up to 1,000, 5,000 and 20,000) to about a quarter; the plan that spreads all
// has to be 7% ahead, since rounds at 6% lost by it.
// Pipelined jobs start first.  items[0, n): the round's stripe jobs (every lane
// shape), longest first; other: its remaining wavefronts.  MH_DP_PIPE = P (p_env)
// instead gives P wavefronts to the first 64-lane jobs with at least P stripes,
// as many as the idle slots hold.
// A pipelined job's boundary takes four times the memory, and a byte a column
// holds half a byte where a lane has one: spare is what the round's bytes may
// still grow by (item_bytes), and the jobs that would pass it, the longest
// first, keep one wavefront.  Returns the bytes it grew by.
//
// Measured, with the parts' priorities (dp_job): 4,000 jobs of 10-20,000 columns
// (at most 8 parts a job, all the round's wavefronts fitting the slots together,
// before) 75.9 -> 46.4 ms, a learned band's run over 6,000 such jobs 55.8 -> 20
// ms.  Left: a part alone on its SIMD issues an instruction every six cycles
// instead of four, and a banded job's stripes wait for each other (9 ms for 20,000
// columns).
static int64_t plan_parts(const mh_dp_job *jobs, DpItem *items, uint64_t n, uint64_t other, uint64_t simds, int wpe,
                          int p_env, uint64_t spare)
{
    int64_t grown = 0;
    auto group = [](const DpItem &it) { return it.cols > GROUP_TAG; };
    auto cols_of = [&](const DpItem &it) { return group(it) ? it.cols - GROUP_TAG : it.cols; };
    double est = 0;     // wavefronts of the round as it stands
    bool wide = false;
    for (uint64_t x = 0; x < n; ++x) {
        est += group(items[x]) ? 0.25 : 1.0;
        if (cols_of(items[x]) > 8) wide = true;
    }
    const bool tagged = wpe < 0;     // (only these cells have the one- and two-column lanes)
    if (tagged) wpe = FWD_VARIANTS[dp_variant_for(wide)].wpe;
    const double slots = std::max(1.0, (double)(simds * (uint64_t)wpe) - (double)other);
    // p wavefronts for it (over all lanes, if it is of 16-lane stripes), while the memory lasts
    auto give = [&](DpItem &it, uint32_t p) {
        DpItem w = it;
        w.parts = p;
        if (group(it)) {
            w.cols = cols_of(it) / 4;
            w.tb_bytes = dp_steps(jobs[it.job].a_len, jobs[it.job].b_len, it.band, w.cols, 64) * 64 * lane_bytes_of(w.cols);
        }
        const int64_t more = (int64_t)item_bytes(w, jobs) - (int64_t)item_bytes(it, jobs);
        if (more > 0 && grown + more > (int64_t)spare) return false;
        grown += more;
        it = w;
        return true;
    };
    if (p_env > 1) {
        if (est >= slots) return 0;
        double used = est;
        for (uint64_t x = 0; x < n; ++x) {
            DpItem &it = items[x];
            const uint64_t ns = (jobs[it.job].b_len + 64ull * it.cols - 1) / (64ull * it.cols);
            if (group(it) || ns < (uint64_t)p_env || used + p_env - 1 > slots) continue;
            if (give(it, (uint32_t)p_env)) used += p_env - 1;
        }
        return grown;
    }
    // instructions of a step: about 24 around the cells, 12.4 a cell
    auto step_cost = [](uint32_t cols) { return 24.0 + 12.4 * cols; };
    struct Opt {
        double own, stripe;    // time on its own; of one stripe when pipelined
        double steps, lead;    // steps on its own; between stripes' starts at least, when pipelined
        uint32_t ns, pmax, c2; // c2: columns a lane when pipelined
        float weight;
        bool widen;
    };
    std::vector<Opt> opt(n);
    double total = 0, longest = 0;
    for (uint64_t x = 0; x < n; ++x) {
        const DpItem &it = items[x];
        const mh_dp_job &jb = jobs[it.job];
        const uint32_t c = cols_of(it), g = group(it) ? 16 : 64, sw = g * c;
        Opt &o = opt[x];
        const double steps = (double)(it.cells / ((uint64_t)g * c));
        o.own = steps * step_cost(c);
        o.ns = (jb.b_len + sw - 1) / sw;
        o.weight = group(it) ? 0.25f : 1.0f;
        o.steps = steps;
        o.pmax = 0;
        o.widen = tagged && group(it) && it.band != 0 && (c == 4 || c == 8);
        if (o.ns > 1 && (g == 64 || o.widen)) {
            o.c2 = o.widen ? c / 4 : c;
            const double rows = steps / o.ns - (g - 1);
            o.stripe = (rows + 63) * step_cost(o.c2);
            o.pmax = std::min(DP_PIPE_MAX, o.ns);
            o.lead = 0;
            if (it.band) {
                o.lead = (double)jb.a_len * sw / jb.b_len + 63 + (o.c2 <= 2 ? 16 : 64);
                o.pmax = std::min<uint32_t>(o.pmax, (uint32_t)std::max(1.0, std::ceil((rows + 63) / o.lead)));
            }
        }
        total += o.own * o.weight;
        longest = std::max(longest, o.own);
    }
    const double share = total / slots, T = 0.25 * share;
    if (longest <= 1.1 * share) return 0;
    int spread = 2;     // 0: no job, 1: those of 64 lanes, 2: all
    bool up = false;
    auto parts_of = [&](const Opt &o, bool up) -> uint32_t {
        if (o.own <= T || !o.pmax || spread < (o.widen ? 2 : 1)) return 0;
        const double m = std::max(1.0, up ? std::ceil(T / o.stripe) : std::floor(T / o.stripe));   // stripes a part
        return std::min<uint32_t>(o.pmax, (uint32_t)std::ceil(o.ns / m));
    };
    // parts past the slots would run after the others: fewer, longer ones then
    auto plan = [&] {
        double all = 0;
        for (const Opt &o : opt) all += parts_of(o, false);
        up = all > slots;
    };
    plan();
    if (std::any_of(opt.begin(), opt.end(), [&](const Opt &o) { return o.widen && parts_of(o, up); })) {
        // cycles of the round: the SIMDs' issue shared evenly, or the longest
        // job's own steps, after the pipelined ones' issue where it is not one
        double cycles[3];
        for (spread = 2; spread >= 0; --spread) {
            plan();
            double issue = 0, issue_piped = 0, longest_piped = 0, longest_own = 0;
            for (const Opt &o : opt) {
                const uint32_t p = parts_of(o, up);
                if (!p || (p == 1 && !o.widen)) {
                    const bool g16 = o.weight < 1.0f;
                    issue += (g16 ? 4.6 : 4.2) * o.own * o.weight;
                    longest_own = std::max(longest_own, g16 ? std::max(6.5 * o.own, 760.0 * o.steps) : 7.5 * o.own);
                } else {
                    const double st = o.stripe / step_cost(o.c2);     // steps of a stripe
                    const double i = o.ns * st * 4.0 * (o.widen ? 60.0 + 14.0 * o.c2 : step_cost(o.c2));
                    issue += i;
                    issue_piped += i;
                    longest_piped = std::max(longest_piped, std::max(std::ceil((double)o.ns / p) * st, (o.ns - 1) * o.lead + st) *
                                                                (o.widen ? 630.0 : 6.0 * step_cost(o.c2)));
                }
            }
            cycles[spread] = std::max({issue / (double)simds, longest_piped, issue_piped / (double)simds + longest_own});
        }
        spread = cycles[0] <= cycles[1] ? 0 : 1;
        if (cycles[2] < 0.93 * cycles[spread]) spread = 2;
        plan();
    }
    for (uint64_t x = 0; x < n; ++x) {
        DpItem &it = items[x];
        const uint32_t p = parts_of(opt[x], up);
        if (p && (p > 1 || group(it))) give(it, p);
    }
    return grown;
}

static int dp_run_items(mh_context *ctx, const uint8_t *d_a, const uint8_t *d_b, const mh_dp_job *jobs,
                        const std::vector<uint64_t> &slot, std::vector<DpItem> &items, uint8_t *d_paths,
                        mh_dp_result *d_results, uint32_t *d_dev, uint64_t *cells,
                        const FixedScratch *fx = nullptr, DpCells form = DpCells::TAGGED)
{
    const uint64_t nitems = items.size();
    if (nitems == 0) return MH_OK;
    // largest first so the long tails start early: a stable counting sort on
    // the trace size quantised to 1/16 octave (the order only balances load)
    const double ts0 = now_ms();
    {
        auto q = [](uint64_t v) -> uint32_t {
            if (v < 16) return (uint32_t)v;
            const int e = 63 - __builtin_clzll(v);
            return (uint32_t)(e * 16 + ((v >> (e - 4)) & 15u));
        };
        constexpr uint32_t NQ = 64 * 16 + 16;
        std::vector<uint32_t> cnt(NQ + 1, 0);
        for (const DpItem &it : items) ++cnt[NQ - 1 - q(it.tb_bytes)];
        uint32_t acc = 0;
        for (uint32_t &c : cnt) {
            const uint32_t t = c;
            c = acc;
            acc += t;
        }
        std::vector<DpItem> sorted(nitems);
        for (const DpItem &it : items) sorted[cnt[NQ - 1 - q(it.tb_bytes)]++] = it;
        items.swap(sorted);
    }
    host_time(ctx, "host_dp_sort", now_ms() - ts0);
    auto bnd_ints = [&](const DpItem &it) { return item_bnd_ints(it, jobs); };
    if (fx) {
        for (const DpItem &it : items)
            MH_CHECK(fixed_takes(it, jobs, fx), MH_ERR_INVALID,
                     "DP job " + std::to_string(it.job) + " (" + std::to_string(jobs[it.job].a_len) + " x " +
                         std::to_string(jobs[it.job].b_len) + ") needs more than the " +
                         std::to_string(fx->bytes >> 20) + " MiB scratch of the no-allocation entry point");
    }
    // trace arena budget: 70% of the memory that is free or already held by
    // this context's arena (at most 192 GB); once grown the arena is kept
    uint64_t budget = 0;
    if (!fx) {
        size_t free_b = 0, total_b = 0;
        MH_HIP(hipMemGetInfo(&free_b, &total_b));
        budget = (uint64_t)((free_b + ctx->dp_tb.bytes) * 0.7);
        const uint64_t cap = 192ull << 30;
        if (budget > cap) budget = cap;
        if (const char *e = getenv("MH_DP_TB_BUDGET_GB")) budget = (uint64_t)(atof(e) * (1ull << 30));
    }
    RoundArgs ra;
    packed_rows(ra.sc);
    // pipelined stripe jobs: wavefronts a job by the round's size (up to
    // DP_PIPE_MAX), or MH_DP_PIPE (0 or 1 keeps one wavefront a job); the
    // no-allocation path keeps one
    int pipe_env = -1;
    if (const char *e = getenv("MH_DP_PIPE")) pipe_env = std::max(0, std::min((int)DP_PIPE_MAX, atoi(e)));
    int ncu = 0;
    if (!fx && pipe_env != 0 && pipe_env != 1)
        MH_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, ctx->device));

    // the rounds, and each one's pipelined jobs
    struct Round {
        uint64_t last, nbig, nstripe;   // end of the items; how many are not one-lane jobs; stripe jobs
    };
    std::vector<Round> rounds;
    uint64_t arena = 0;
    // several rounds leave a 32nd of the budget for what their pipelined jobs add
    // (a quarter of a percent for 20,000 columns, 2.4 for 2,000): with none, each
    // round ends on its longest job (100,000 jobs of 10-20,000 columns 1.33 s, 1.07
    // with it)
    uint64_t room = budget;
    for (uint64_t first = 0; first < nitems;) {
        // one round: as many jobs (in schedule order) as fit the trace budget
        uint64_t tbb = 0, bi = 0, last = first;
        while (last < nitems) {
            const uint64_t w = (items[last].tb_bytes + 15) & ~15ull, b = bnd_ints(items[last]);
            if (last > first && (fx ? fixed_need(last - first + 1, tbb + w, bi + b) > fx->bytes
                                    : arena_bytes(tbb + w, bi + b) > room))
                break;
            tbb += w;
            bi += b;
            ++last;
        }
        if (last < nitems && room == budget && budget >= 32) {
            room -= budget / 32;     // (and the first round again)
            continue;
        }
        const uint64_t n = last - first;
        // stripe jobs, then sliding-window jobs, then one-lane jobs, each in order
        std::stable_partition(items.begin() + (ptrdiff_t)first, items.begin() + (ptrdiff_t)last,
                              [](const DpItem &it) { return it.cols != TINY_COLS_TAG; });
        uint64_t nbig = 0;
        while (nbig < n && items[first + nbig].cols != TINY_COLS_TAG) ++nbig;
        std::stable_partition(items.begin() + (ptrdiff_t)first, items.begin() + (ptrdiff_t)(first + nbig),
                              [](const DpItem &it) { return it.cols < WINDOW_TAG; });
        uint64_t nstripe = 0;
        while (nstripe < nbig && items[first + nstripe].cols < WINDOW_TAG) ++nstripe;
        uint64_t bytes = arena_bytes(tbb, bi);
        if (!fx && ncu > 0)
            bytes += plan_parts(jobs, items.data() + first, nstripe, (nbig - nstripe) + (n - nbig + 63) / 64,
                                (uint64_t)ncu * 4, form == DpCells::TAGGED ? -1 : FWD_VARIANTS[VARIANT_FLOAT].wpe, pipe_env,
                                bytes < budget ? budget - bytes : 0);
        arena = std::max(arena, bytes);
        rounds.push_back({last, nbig, nstripe});
        first = last;
    }
    if (!fx) {
        // the arena, once for the whole call
        const int rc = ctx->dp_tb.ensure(arena + 256);
        if (rc != MH_OK) return rc;
        // (a count under the timers' names: its bytes)
        host_time(ctx, "dp_arena_bytes", (double)arena);
    }
    std::vector<DpItem> shaped;
    uint64_t first = 0;
    for (const Round &rd : rounds) {
        const uint64_t last = rd.last, n = last - first, nbig = rd.nbig, nstripe = rd.nstripe;
        // wavefront stripes (the pipelined ones first, most parts first), then
        // the row-packed jobs by shape (16, 14, ..., 4 columns a lane), each in
        // order: a stable bucket pass
        auto shape = [](const DpItem &it) {
            return it.cols < GROUP_TAG ? 0 : 1 + (int)(GROUP_TAG + 16 - it.cols) / 2;
        };
        uint64_t rows_at[ROW_SHAPES + 2] = {};
        for (uint64_t x = 0; x < nstripe; ++x) ++rows_at[shape(items[first + x]) + 1];
        for (int q = 0; q <= ROW_SHAPES; ++q) rows_at[q + 1] += rows_at[q];
        {
            uint64_t put[ROW_SHAPES + 1];
            for (int q = 0; q <= ROW_SHAPES; ++q) put[q] = rows_at[q];
            shaped.resize(nstripe);
            for (uint64_t x = 0; x < nstripe; ++x) shaped[put[shape(items[first + x])]++] = items[first + x];
            std::copy(shaped.begin(), shaped.end(), items.begin() + (ptrdiff_t)first);
        }
        // A wavefront of 16-lane stripes runs four jobs whose stripe loops
        // diverge: each stripe costs it the longest of the four, so banded
        // jobs of those shapes go in order of stripe count, then rows a
        // stripe (largest first), and the four of a wavefront step alike.
        // (Full jobs of these shapes hold one stripe of LA rows: their
        // largest-first order is that order already.)
        for (int q : {5, 7}) {   // 16-lane stripes of 8 and of 4 columns a lane
            const uint64_t b0 = first + rows_at[q], b1 = first + rows_at[q + 1];
            bool banded = false;
            for (uint64_t x = b0; x < b1 && !banded; ++x) banded = items[x].band != 0;
            if (!banded) continue;
            std::vector<std::pair<uint64_t, uint32_t>> keyed(b1 - b0);
            for (uint64_t x = b0; x < b1; ++x) {
                const DpItem &it = items[x];
                const mh_dp_job &jb = jobs[it.job];
                const uint64_t sw = 16ull * (it.cols - GROUP_TAG);
                const uint64_t ns = (jb.b_len + sw - 1) / sw;
                uint64_t rows = jb.a_len;
                if (it.band) rows = std::min<uint64_t>(jb.a_len, jb.a_len * (sw + 2ull * it.band) / jb.b_len + 1);
                keyed[x - b0] = {(ns << 32) | rows, (uint32_t)(x - b0)};
            }
            std::stable_sort(keyed.begin(), keyed.end(),
                             [](const std::pair<uint64_t, uint32_t> &a, const std::pair<uint64_t, uint32_t> &b) {
                                 return a.first > b.first;
                             });
            shaped.resize(b1 - b0);
            for (uint64_t x = 0; x < b1 - b0; ++x) shaped[x] = items[b0 + keyed[x].second];
            std::copy(shaped.begin(), shaped.end(), items.begin() + (ptrdiff_t)b0);
        }
        const uint64_t n64 = rows_at[1];   // rows_at[1..]: the row jobs, 16 columns a lane first
        std::stable_sort(items.begin() + (ptrdiff_t)first, items.begin() + (ptrdiff_t)(first + n64),
                         [](const DpItem &x, const DpItem &y) { return x.parts > y.parts; });
        // the forward variant: the wide one when a shape wider than 8 columns a lane is in the round
        bool wide = false;
        for (uint64_t z = 0; z < n64 && !wide; ++z) wide = items[first + z].cols == 16;
        for (int q = 0; q < 4; ++q)
            if (rows_at[q + 2] > rows_at[q + 1]) wide = true;
        const int variant = form == DpCells::TAGGED ? dp_variant_for(wide)
                                                    : (form == DpCells::FLOAT ? VARIANT_FLOAT : VARIANT_LONG);
        uint64_t npipe = 0;
        while (npipe < n64 && items[first + npipe].parts) ++npipe;
        // (a count under the timers' names: pipelined jobs a round)
        if (npipe) host_time(ctx, "dp_pipe_jobs", (double)npipe);
        DevJob *dj = nullptr;
        std::vector<DevJob> host_jobs;
        if (fx) {
            host_jobs.resize(n);
            dj = host_jobs.data();
        } else {
            const int rc0 = pinned_jobs(ctx, n * sizeof(DevJob) + 64, (void **)&dj);
            if (rc0 != MH_OK) return rc0;
        }
        uint64_t tw = 0, bo = 0, bo_pipe = 0;
        for (uint64_t x = 0; x < n; ++x) {
            const DpItem &it = items[first + x];
            const uint32_t j = it.job;
            DevJob &d = dj[x];
            d.a_off = jobs[j].a_off;
            d.b_off = jobs[j].b_off;
            d.la = jobs[j].a_len;
            d.lb = jobs[j].b_len;
            d.tb_off = tw;
            d.bnd_off = bo;
            d.path_off = slot[j];
            d.user = j;
            d.cols = it.cols;
            d.band = it.band;
            d.pad_ = 0;
            tw += (it.tb_bytes + 15) & ~15ull;
            bo += bnd_ints(it);
            if (x < npipe) bo_pipe = bo;
            if (cells) *cells += it.cells;
        }
        DevJob *d_jobs;
        DpOut *d_outs;
        uint8_t *d_tb;
        int *d_bnd;
        DpRound *d_round;
        if (fx) {
            // [round descriptor + cursors] [jobs | results] [boundary ints] [trace]
            uint8_t *q = fx->ptr;
            d_round = reinterpret_cast<DpRound *>(q);
            q += dp_round_bytes(DPQ_FIXED_MAXB);
            d_jobs = reinterpret_cast<DevJob *>(q);
            d_outs = reinterpret_cast<DpOut *>(d_jobs + n);
            q += align256(n * (sizeof(DevJob) + sizeof(DpOut) + 4));
            d_bnd = reinterpret_cast<int *>(q);
            q += align256(bo * 4);
            d_tb = q;
            MH_CHECK((uint64_t)(q - fx->ptr) + tw <= fx->bytes, MH_ERR_INVALID, "DP round exceeds the scratch");
        } else {
            int rc;
            if ((rc = ctx->dp_jobs.ensure(n * (sizeof(DevJob) + sizeof(DpOut) + 4) + 256)) != MH_OK) return rc;
            if ((rc = ctx->dp_round.ensure(dp_round_bytes(DPQ_MAXB))) != MH_OK) return rc;
            d_jobs = ctx->dp_jobs.as<DevJob>();
            d_outs = reinterpret_cast<DpOut *>(d_jobs + n);
            d_bnd = ctx->dp_tb.as<int>();
            d_tb = ctx->dp_tb.as<uint8_t>() + align256(bo * 4);
            d_round = ctx->dp_round.as<DpRound>();
        }
        MH_HIP(hipMemcpyAsync(d_jobs, dj, n * sizeof(DevJob), hipMemcpyHostToDevice, ctx->stream));
        // the pipelined jobs' boundary words (the first jobs') start untagged
        if (bo_pipe) MH_HIP(hipMemsetAsync(d_bnd, 0, bo_pipe * 4, ctx->stream));
        // the round's descriptor: the queue's bins
        DpRound hr;
        std::memset(&hr, 0, sizeof(hr));
        const uint32_t max_bins = fx ? DPQ_FIXED_MAXB : DPQ_MAXB;
        if (form != DpCells::TAGGED) dp_score6(hr.table);
        auto add_bin = [&](uint32_t kind, uint64_t b0, uint64_t cnt) {
            if (cnt == 0) return;
            hr.bin[hr.nbins++] = {kind, (uint32_t)b0, (uint32_t)cnt, 0};
        };
        {
            // stripe jobs: a new bin where the trace size falls below the next power of 4
            // the pipelined jobs first, a bin for each part count, an item a part
            for (uint64_t x = 0; x < npipe;) {
                uint64_t y = x + 1;
                while (y < npipe && items[first + y].parts == items[first + x].parts) ++y;
                add_bin(QK_PIPE + (items[first + x].parts - 1u), x, (y - x) * items[first + x].parts);
                x = y;
            }
            auto cls = [](uint64_t v) { return v ? (63 - __builtin_clzll(v)) / 2 : 0; };
            uint64_t x = npipe;
            while (x < n64) {
                const int c0 = cls(items[first + x].tb_bytes);
                uint64_t y = x + 1;
                while (y < n64 && cls(items[first + y].tb_bytes) == c0) ++y;
                // keep ROW_SHAPES + 2 bins for the row, window and one-lane
                // jobs, and the last cursor for the wait-bound error flag
                if (hr.nbins + 1 >= max_bins - ROW_SHAPES - 3) y = n64;
                add_bin(QK_STRIPE, x, y - x);
                x = y;
            }
            for (int q = 0; q < ROW_SHAPES; ++q) add_bin(QK_ROWS + q, rows_at[q + 1], rows_at[q + 2] - rows_at[q + 1]);
            add_bin(QK_WINDOW, nstripe, nbig - nstripe);
            add_bin(QK_TINY, nbig, n - nbig);
        }
        MH_CHECK(hr.nbins < max_bins, MH_ERR_INVALID, "DP round: too many queue bins");
        uint64_t nitems_q = 0;
        for (uint32_t q = 0; q < hr.nbins; ++q) {
            const uint32_t kind = hr.bin[q].kind;
            const uint32_t per =
                kind == QK_STRIPE || kind == QK_WINDOW || kind >= QK_PIPE ? 1u : (kind == QK_TINY ? 64u : 4u);
            hr.bin[q].item0 = (uint32_t)nitems_q;
            nitems_q += (hr.bin[q].count + per - 1) / per;
        }
        hr.bin[hr.nbins].item0 = (uint32_t)nitems_q;
        const uint64_t hr_bytes = offsetof(DpRound, bin) + (hr.nbins + 1) * sizeof(DpBin);
        unsigned grid = 0;
        {
            int rc;
            if ((rc = fwd_grid(ctx, variant, nitems_q, &grid)) != MH_OK) return rc;
        }
        ra.jobs = d_jobs;
        ra.outs = d_outs;
        ra.A = d_a;
        ra.B = d_b;
        ra.tb = d_tb;
        ra.bnd = d_bnd;
        ra.rd = d_round;
        ra.cursor = reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(d_round) + dp_cursor_at(max_bins));
        ra.paths = d_paths;
        ra.res = d_results;
        ra.dev = d_dev;
        ra.npipe = (uint32_t)npipe;
        if (fx) {
            MH_HIP(hipMemcpyAsync(d_round, &hr, hr_bytes, hipMemcpyHostToDevice, ctx->stream));
            int rc;
            if ((rc = dp_launch_round(ctx, variant, false, grid, ra)) != MH_OK) return rc;
        } else {
            int rc;
            if ((rc = dp_round_staging(ctx)) != MH_OK) return rc;
            std::memcpy(ctx->dp_round_host, &hr, hr_bytes);
            MH_HIP(hipMemcpyAsync(d_round, ctx->dp_round_host, hr_bytes, hipMemcpyHostToDevice, ctx->stream));
            if ((rc = dp_launch_round(ctx, variant, dp_use_graph(), grid, ra)) != MH_OK) return rc;
        }
        // the host job table is reused by the next round
        uint32_t err = 0;
        if (npipe) MH_HIP(hipMemcpyAsync(&err, ra.cursor + (DPQ_CURSORS - 1), 4, hipMemcpyDeviceToHost, ctx->stream));
        MH_HIP(hipStreamSynchronize(ctx->stream));
        MH_CHECK(err == 0, MH_ERR_DEVICE, "DP: a pipelined stripe's wait ran past its limit");
        first = last;
    }
    return MH_OK;
}

__global__ void pack_paths_kernel(const uint8_t *__restrict__ p, uint64_t n, uint8_t *__restrict__ out)
{
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k * 4 >= n) return;
    uint32_t v = 0;
    for (int x = 0; x < 4; ++x) {
        const uint64_t at = k * 4 + x;
        const uint8_t e = at < n ? p[at] : 0;
        const uint32_t c = e == 'M' ? 0u : (e == 'D' ? 1u : (e == 'I' ? 2u : 3u));
        v |= c << (2 * x);
    }
    out[k] = (uint8_t)v;
}

int dp_pack_paths(mh_context *ctx, const uint8_t *d_paths, uint64_t n, uint8_t *d_out)
{
    const uint64_t nb = (n + 3) / 4;
    if (!nb) return MH_OK;
    hipLaunchKernelGGL(pack_paths_kernel, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, ctx->stream, d_paths, n,
                       d_out);
    MH_HIP(hipGetLastError());
    return MH_OK;
}

static int dp_check_jobs(const mh_dp_job *jobs, uint64_t njobs, std::vector<uint64_t> &slot)
{
    MH_CHECK(njobs < (1ull << 31), MH_ERR_INVALID, "too many DP jobs in one call");
    slot.resize(njobs);
    uint64_t acc = 0;
    for (uint64_t j = 0; j < njobs; ++j) {
        MH_CHECK(jobs[j].a_len > 0 && jobs[j].b_len > 0, MH_ERR_ZERO_LENGTH,
                 "NWSmall: length=0 (job " + std::to_string(j) + ")");
        MH_CHECK(jobs[j].a_len < (1u << 24) && jobs[j].b_len < (1u << 24), MH_ERR_UNSUPPORTED,
                 "DP operand longer than 2^24");
        slot[j] = acc;
        acc += (uint64_t)jobs[j].a_len + jobs[j].b_len;
    }
    return MH_OK;
}

static DpItem make_item(const mh_dp_job &jb, uint32_t job, uint32_t band, int force, bool rerun = false,
                        bool tiny = true)
{
    DpItem it;
    it.job = job;
    it.parts = 0;
    it.cols = dp_cols_for(jb.a_len, jb.b_len, band, force, rerun);
    it.band = dp_effective_band(jb.a_len, jb.b_len, band, it.cols);
    if (it.band == 0 && band != 0) it.cols = dp_cols_for(jb.a_len, jb.b_len, 0, force);
    if (it.band == 0 && !force && tiny && jb.b_len <= (uint32_t)TINY_LB) {
        it.cols = TINY_COLS_TAG;
        it.tb_bytes = (uint64_t)jb.a_len * 8;
        it.cells = 2 * it.tb_bytes;
        return it;
    }
    if (it.band == 0 && !force && jb.b_len <= ROWS_MAX_LB && jb.a_len + jb.b_len < ROWS_MAX_WALK &&
        shape_table()[dp_tune_class(jb.b_len)] == 0) {
        // four jobs per wavefront, one stripe each of the fewest columns a lane
        // (an even number from 4 to 16) that holds the job
        it.cols = GROUP_TAG + std::max(4u, 2u * ((jb.b_len + 31) / 32));
    }
    const uint32_t g = it.cols > GROUP_TAG ? 16u : 64u, c = it.cols > GROUP_TAG ? it.cols - GROUP_TAG : it.cols;
    const uint64_t steps = dp_steps(jb.a_len, jb.b_len, it.band, c, g);
    it.tb_bytes = steps * g * lane_bytes_of(c);
    it.cells = steps * g * c;
    if (it.band) {
        const uint32_t wc = dp_window_cols(jb.a_len, jb.b_len, it.band, dp_force_kind());
        if (wc) {
            it.cols = WINDOW_TAG + wc;
            it.tb_bytes = (uint64_t)((jb.a_len + 8 / wc - 1) / (8 / wc)) * 256;
            it.cells = 2 * it.tb_bytes;
        }
    }
    return it;
}

// items[x] = make_item(jobs[x], x, bands[x]) for every job, in parallel host
// threads for large batches
static void make_items(const mh_dp_job *jobs, uint64_t njobs, const uint32_t *bands, std::vector<DpItem> &items)
{
    const int force = dp_force_cols();
    items.resize(njobs);
    auto fill = [&](uint64_t lo, uint64_t hi) {
        for (uint64_t j = lo; j < hi; ++j) items[j] = make_item(jobs[j], (uint32_t)j, bands ? bands[j] : 0u, force);
    };
    const uint64_t chunk = 8192;
    host_parallel((size_t)((njobs + chunk - 1) / chunk),
                  [&](size_t k) { fill(k * chunk, std::min<uint64_t>(njobs, (k + 1) * chunk)); });
}

uint64_t dp_item_cells(uint32_t la, uint32_t lb, uint32_t band)
{
    if (la == 0 || lb == 0) return 0;
    const DpItem it = make_item(mh_dp_job{0, 0, la, lb}, 0, band, dp_force_cols());
    if (it.cols == TINY_COLS_TAG) return (uint64_t)la * lb;
    if (it.cols > WINDOW_TAG) return (uint64_t)la * 64 * (it.cols - WINDOW_TAG);
    return it.cells;
}

// The jobs whose operands hold letters other than A, C, G, T (class > 3):
// from the caller's flags, or a device scan; codes above 5 are refused.
static int split_wild(mh_context *ctx, const uint8_t *d_a, const uint8_t *d_b, const mh_dp_job *jobs,
                      uint64_t njobs, const uint8_t *wild, const FixedScratch *fx, std::vector<uint32_t> &out)
{
    out.clear();
    if (wild) {
        for (uint64_t j = 0; j < njobs; ++j)
            if (wild[j]) out.push_back((uint32_t)j);
        return MH_OK;
    }
    std::vector<uint8_t> mx;
    const int rc = dp_code_max(ctx, d_a, d_b, jobs, njobs, fx, mx);
    if (rc != MH_OK) return rc;
    for (uint64_t j = 0; j < njobs; ++j) {
        MH_CHECK(mx[j] < DP_NCLASS, MH_ERR_INVALID,
                 "DP operand code above 5 in job " + std::to_string(j) + " (codes: 0-3 A,C,G,T, 4 X, 5 other)");
        if (mx[j] > 3) out.push_back((uint32_t)j);
    }
    return MH_OK;
}

// dp_run_items over the items' two forms of cells
static int dp_run_forms(mh_context *ctx, const uint8_t *d_a, const uint8_t *d_b, const mh_dp_job *jobs,
                        const std::vector<uint64_t> &slot, std::vector<DpItem> &items, uint8_t *d_paths,
                        mh_dp_result *d_results, uint32_t *d_dev, uint64_t *cells, const FixedScratch *fx = nullptr)
{
    auto tagged = [&](const DpItem &it) {
        return it.cols > WINDOW_TAG || std::min(jobs[it.job].a_len, jobs[it.job].b_len) <= TAGGED_MAX;
    };
    std::vector<DpItem> longs;
    for (const DpItem &it : items)
        if (!tagged(it)) longs.push_back(it);
    if (!longs.empty()) {
        items.erase(std::remove_if(items.begin(), items.end(), [&](const DpItem &it) { return !tagged(it); }),
                    items.end());
        const int rc = dp_run_items(ctx, d_a, d_b, jobs, slot, longs, d_paths, d_results, d_dev, cells, fx, DpCells::LONG);
        if (rc != MH_OK) return rc;
    }
    return dp_run_items(ctx, d_a, d_b, jobs, slot, items, d_paths, d_results, d_dev, cells, fx, DpCells::TAGGED);
}

// The jobs `which` (indices into jobs), whose operands hold wildcard letters:
// the full DP in float cells.  In the fixed scratch a job keeps the limit it has
// always had, that of a float row set and a byte a cell (dp_float.hip); a long
// thin job whose records would not fit there (a lane's share of a step is at
// least 2 bytes) takes that form still, a thread a job.
static int dp_run_wild(mh_context *ctx, const uint8_t *d_a, const uint8_t *d_b, const mh_dp_job *jobs,
                       const std::vector<uint64_t> &slot, const std::vector<uint32_t> &which, uint8_t *d_paths,
                       mh_dp_result *d_results, uint32_t *d_dev, uint64_t *cells, const FixedScratch *fx)
{
    if (which.empty()) return MH_OK;
    const int force = dp_force_cols();
    std::vector<DpItem> items;
    std::vector<uint32_t> thin;
    int rc;
    for (uint32_t j : which) {
        if (fx && (rc = dp_float_fits(jobs, j, fx)) != MH_OK) return rc;
        DpItem it = make_item(jobs[j], j, 0, force, false, false);
        it.cells = (uint64_t)jobs[j].a_len * jobs[j].b_len;
        if (fx && !fixed_takes(it, jobs, fx)) thin.push_back(j);
        else items.push_back(it);
    }
    if ((rc = dp_run_items(ctx, d_a, d_b, jobs, slot, items, d_paths, d_results, d_dev, cells, fx, DpCells::FLOAT)) !=
        MH_OK)
        return rc;
    return thin.empty() ? MH_OK : dp_run_float_threads(ctx, d_a, d_b, jobs, slot, thin, d_paths, d_results, fx);
}

// drops the items of the float-DP jobs (items[j] is job j's)
static void drop_wild(std::vector<DpItem> &items, const std::vector<uint32_t> &wild)
{
    if (wild.empty()) return;
    size_t w = 0, k = 0;
    for (size_t j = 0; j < items.size(); ++j) {
        if (k < wild.size() && wild[k] == j) {
            ++k;
            continue;
        }
        items[w++] = items[j];
    }
    items.resize(w);
}

int dp_run(mh_context *ctx, const uint8_t *d_a, const uint8_t *d_b, const mh_dp_job *jobs,
           uint64_t njobs, uint8_t *d_paths, mh_dp_result *d_results, const uint8_t *wild)
{
    if (njobs == 0) return MH_OK;
    std::vector<uint64_t> slot;
    int rc;
    if ((rc = dp_check_jobs(jobs, njobs, slot)) != MH_OK) return rc;
    std::vector<uint32_t> wj;
    if ((rc = split_wild(ctx, d_a, d_b, jobs, njobs, wild, nullptr, wj)) != MH_OK) return rc;
    std::vector<DpItem> items;
    const double tp0 = now_ms();
    make_items(jobs, njobs, nullptr, items);
    drop_wild(items, wj);
    host_time(ctx, "host_dp_plan", now_ms() - tp0);
    if ((rc = dp_run_forms(ctx, d_a, d_b, jobs, slot, items, d_paths, d_results, nullptr, nullptr)) != MH_OK)
        return rc;
    return dp_run_wild(ctx, d_a, d_b, jobs, slot, wj, d_paths, d_results, nullptr, nullptr, nullptr);
}

int dp_run_noalloc(mh_context *ctx, const uint8_t *d_a, const uint8_t *d_b, const mh_dp_job *jobs, uint64_t njobs,
                   uint8_t *d_paths, mh_dp_result *d_results)
{
    uint8_t *base = nullptr;
    if (ctx->device >= 0 && ctx->device < DP_SCRATCH_MAX_DEVICES) {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        base = g_scratch_ptr[ctx->device];
    }
    MH_CHECK(base, MH_ERR_INVALID, "the DP scratch of this device was not set up (mh_create does it)");
    if (njobs == 0) return MH_OK;
    std::vector<uint64_t> slot;
    int rc;
    if ((rc = dp_check_jobs(jobs, njobs, slot)) != MH_OK) return rc;
    FixedScratch fx;
    fx.ptr = base;
    fx.bytes = DP_SCRATCH_BYTES;
    std::vector<uint32_t> wj;
    if ((rc = split_wild(ctx, d_a, d_b, jobs, njobs, nullptr, &fx, wj)) != MH_OK) return rc;
    std::vector<DpItem> items;
    make_items(jobs, njobs, nullptr, items);
    drop_wild(items, wj);
    if ((rc = dp_run_forms(ctx, d_a, d_b, jobs, slot, items, d_paths, d_results, nullptr, nullptr, &fx)) != MH_OK)
        return rc;
    return dp_run_wild(ctx, d_a, d_b, jobs, slot, wj, d_paths, d_results, nullptr, nullptr, &fx);
}

int dp_run_banded(mh_context *ctx, const uint8_t *d_a, const uint8_t *d_b, const mh_dp_job *jobs, uint64_t njobs,
                  const uint32_t *bands, uint32_t flags, uint8_t *d_paths, mh_dp_result *d_results,
                  uint32_t *d_dev, mh_band_stats *stats)
{
    mh_band_stats st;
    std::memset(&st, 0, sizeof(st));
    if (stats) *stats = st;
    if (njobs == 0) return MH_OK;
    std::vector<uint64_t> slot;
    int rc;
    if ((rc = dp_check_jobs(jobs, njobs, slot)) != MH_OK) return rc;
    if (!d_dev) {
        if ((rc = ctx->dp_dev.ensure(njobs * 4 + 64)) != MH_OK) return rc;
        d_dev = ctx->dp_dev.as<uint32_t>();
    }
    const double tp0 = now_ms();
    // a job with band W evaluates the region of band 2W and accepts its path
    // when it stays within W of the line (the region reaches at least W past
    // the accepted band, where a path that wants to leave shows itself)
    std::vector<uint32_t> region(njobs, 0);
    for (uint64_t j = 0; j < njobs; ++j) {
        const uint64_t w = bands ? bands[j] : 0u;
        region[j] = 2 * w > 0xFFFFFFFFull ? 0u : (uint32_t)(2 * w);
    }
    // jobs with letters other than A,C,G,T run the full DP in float, unbanded
    std::vector<uint32_t> wj;
    if ((rc = split_wild(ctx, d_a, d_b, jobs, njobs, nullptr, nullptr, wj)) != MH_OK) return rc;
    std::vector<DpItem> items;
    make_items(jobs, njobs, region.data(), items);
    std::vector<uint32_t> accept1(njobs, 0);
    {
        size_t k = 0;
        for (uint64_t j = 0; j < njobs; ++j) {
            if (k < wj.size() && wj[k] == j) {
                ++k;
                continue;
            }
            if (items[j].band) {
                accept1[j] = bands[j];
                ++st.banded;
            }
        }
    }
    drop_wild(items, wj);
    host_time(ctx, "host_dp_plan", now_ms() - tp0);
    const int force = dp_force_cols();
    if ((rc = dp_run_forms(ctx, d_a, d_b, jobs, slot, items, d_paths, d_results, d_dev, &st.cells)) != MH_OK)
        return rc;
    if ((rc = dp_run_wild(ctx, d_a, d_b, jobs, slot, wj, d_paths, d_results, d_dev, &st.cells, nullptr)) != MH_OK)
        return rc;
    if (!(flags & MH_BAND_NO_FALLBACK) && st.banded) {
        // edge fallback: a banded path that reaches distance W is rerun with
        // the band doubled (region 4W, accepted within 2W), and one that
        // reaches 2W too with the full DP
        std::vector<uint32_t> dev(njobs);
        MH_HIP(hipMemcpyAsync(dev.data(), d_dev, njobs * 4, hipMemcpyDeviceToHost, ctx->stream));
        MH_HIP(hipStreamSynchronize(ctx->stream));
        double tq = now_ms();
        host_time(ctx, "band_pass1", tq - tp0);
        std::vector<DpItem> again;
        std::vector<uint32_t> accept2(njobs, 0);
        for (uint64_t j = 0; j < njobs; ++j)
            if (accept1[j] && dev[j] >= accept1[j]) {
                const uint64_t r2 = 4ull * accept1[j];
                again.push_back(make_item(jobs[j], (uint32_t)j, r2 > 0xFFFFFFFFull ? 0u : (uint32_t)r2, force, true));
                if (again.back().band) {
                    accept2[j] = 2 * accept1[j];
                    ++st.rerun_doubled;
                } else {
                    ++st.rerun_full;
                }
            }
        if (!again.empty()) {
            if ((rc = dp_run_forms(ctx, d_a, d_b, jobs, slot, again, d_paths, d_results, d_dev, &st.cells)) != MH_OK)
                return rc;
            MH_HIP(hipMemcpyAsync(dev.data(), d_dev, njobs * 4, hipMemcpyDeviceToHost, ctx->stream));
            MH_HIP(hipStreamSynchronize(ctx->stream));
            host_time(ctx, "band_pass2", now_ms() - tq);
            tq = now_ms();
            std::vector<DpItem> full;
            for (uint64_t j = 0; j < njobs; ++j)
                if (accept2[j] && dev[j] >= accept2[j]) {
                    full.push_back(make_item(jobs[j], (uint32_t)j, 0, force));
                    ++st.rerun_full;
                }
            if (!full.empty()) {
                if ((rc = dp_run_forms(ctx, d_a, d_b, jobs, slot, full, d_paths, d_results, d_dev, &st.cells)) != MH_OK)
                    return rc;
                MH_HIP(hipStreamSynchronize(ctx->stream));
                host_time(ctx, "band_pass3", now_ms() - tq);
            }
        }
    }
    if (stats) *stats = st;
    return MH_OK;
}

}  // namespace mh
