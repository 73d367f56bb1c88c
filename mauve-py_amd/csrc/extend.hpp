// extend.hpp -- ungapped seed extension over k genomes, on the device.
//
// ExtendMatch (LM/MatchFinder.h:218-374) moves a match's two ends through the
// genomes a seed holds.  A step matches when the masked windows of all of them
// agree.  Within one round each end takes seed-length jumps while the next
// window matches, then, step by step, moves to the furthest matching window
// within one seed length (or stays); rounds repeat while either end made a
// single step.  An end's moves depend only on its own position (the room to the
// sequence ends and the windows read are functions of it), and an end whose
// single-step phase found nothing finds nothing again.  So an end moves from
// matching window to matching window, never past a seed length without one,
// and stops where the next seed length of windows holds none: wherever it
// stepped in between, it stops at the last matching window before the first
// run of a seed length of windows that do not match or leave a sequence.  Two
// seeds of the same genomes on one diagonal (each start of the one the same
// distance from the other's) at most a seed length apart therefore extend to
// the same match, and one of them is walked for both.
//
// The reference compares GetDnaSeedMer values: the smaller of the masked window
// and its reverse complement, and which of the two it was.  Under a palindromic
// pattern (the seed families all are) that is a comparison of the windows
// themselves: for two genomes in one orientation, equal masked windows; in
// opposite orientations, the masked window equal to the other's reverse
// complement and not its own (a window that is its own reverse complement
// counts as forward in both).  So a walk reads the packed sequences (reversed
// genomes' from their packed reverse complement), 64 characters a genome, and
// has 32 windows' outcomes from shifting the differing characters' bits by the
// pattern.  Other patterns compare the values by position (PAL false).
//
// A thread's walk is bound by the latency of its scattered reads; a walk over a
// long stretch is a chain of them, which a block cuts to one for 32,000
// windows.  Measured, against walks step by step of eight bytes a position from
// seeds exactly a seed length apart (and, for two genomes, the long ones by
// pointer jumping over every window of their diagonals): eight genomes of 5 Mb
// 1.3 ms (34.3), two of 200 kb 63 us (a 105 us walk and 0.72 ms of jumping).
#pragma once
#if defined(__HIP__)
#include <hip/hip_runtime.h>
#endif
#include <cstdint>

#if defined(__HIPCC__)
#define MH_HD __host__ __device__
#define MH_PRAGMA_UNROLL _Pragma("unroll")
#else
#define MH_HD
#define MH_PRAGMA_UNROLL
#endif

namespace mh {

constexpr int EXT_MAXK = 16;

// Seeds of two genomes by genome-0 position: a word holds the partner's forward
// position in genome 1 (31 bits) with the strand relation in bit 31, or this.
// It is also what a reversed partner at position 2^31 - 1 would give, which is
// past the last window of the longest genomes (2^31 - 1 bases).
constexpr uint32_t NO_SEED = 0xFFFFFFFFu;

// The furthest seed of position p's diagonal within a seed length S before it,
// or p: word(x) is the table's word of position x, word(p) a seed's.
template <class W> MH_HD inline uint32_t spaced_link(uint32_t p, uint32_t S, W word)
{
    const uint32_t v = word(p), rev = v & 0x80000000u, q = v & 0x7FFFFFFFu;
    for (uint32_t t = p < S ? p : S; t > 0; --t) {
        if (!rev && q < t) continue;
        const uint32_t want = (rev ? q + t : q - t) | rev;
        if (want != NO_SEED && word(p - t) == want) return p - t;
    }
    return p;
}

#if defined(__HIP__)

// Per genome: the packed sequence and its reverse complement's, or (other
// patterns) GetDnaSeedMer by position, twice; the length.  mask: the values' top
// 2 * weight bits; pat: the pattern's characters, the first in bit 0.
struct WalkEnv {
    const void *fwd[EXT_MAXK], *rev[EXT_MAXK];
    uint32_t L[EXT_MAXK];
    int seed_len;
    uint32_t pat;
    uint64_t mask;
};

constexpr uint32_t WALK_CHUNKS = 16;    // chunks of 32 windows an end before a whole block takes the walk over
constexpr uint32_t WALK_BLOCK = 1024;

// 32 characters starting at pos (first character in the top two bits)
__device__ __forceinline__ uint64_t win32(const uint32_t *__restrict__ w, uint64_t pos)
{
    const uint64_t q = pos >> 4;
    const uint32_t bit = (uint32_t)(pos & 15) * 2;
    uint64_t m = ((uint64_t)w[q] << 32) | w[q + 1];
    if (bit) m = (m << bit) | (w[q + 2] >> (32 - bit));
    return m;
}

// 64 characters starting at pos; words past the last one (whose characters no
// caller uses) read as the last
__device__ __forceinline__ void win64(const uint32_t *__restrict__ w, uint32_t pos, uint32_t last, uint64_t *hi,
                                      uint64_t *lo)
{
    uint32_t v[5];
    MH_PRAGMA_UNROLL
    for (uint32_t u = 0; u < 5; ++u) {
        const uint32_t q = (pos >> 4) + u;
        v[u] = w[q < last ? q : last];
    }
    const uint32_t bit = (pos & 15) * 2;
    uint64_t a = (uint64_t)v[0] << 32 | v[1], b = (uint64_t)v[2] << 32 | v[3];
    if (bit) {
        a = (a << bit) | (v[2] >> (32 - bit));
        b = (b << bit) | (v[4] >> (32 - bit));
    }
    *hi = a;
    *lo = b;
}

// the even bits of hi and lo, the topmost (the first character's) in bit 0
__device__ __forceinline__ uint64_t char_bits(uint64_t hi, uint64_t lo)
{
    uint64_t r[2] = {hi, lo};
    MH_PRAGMA_UNROLL
    for (int u = 0; u < 2; ++u) {
        uint64_t x = r[u] & 0x5555555555555555ull;
        x = (x | x >> 1) & 0x3333333333333333ull;
        x = (x | x >> 2) & 0x0F0F0F0F0F0F0F0Full;
        x = (x | x >> 4) & 0x00FF00FF00FF00FFull;
        x = (x | x >> 8) & 0x0000FFFF0000FFFFull;
        r[u] = __brev((uint32_t)(x | x >> 16));
    }
    return r[0] | r[1] << 32;
}

// A seed of up to K genomes: each genome's sequence in its orientation, the
// window's start there (the first present genome forward); slots past the
// seed's genomes repeat the first, so that every slot's reads go out together.
template <int K, bool PAL> struct Walk {
    const void *b[K];
    uint32_t p[K], n[K];
    uint32_t rev;        // bit x: slot x reversed
    uint32_t S, pat;
    uint64_t mask;

    // pos: the window's start in genome g's forward coordinates
    __device__ __forceinline__ void set(int x, const WalkEnv &env, int g, uint32_t pos, bool reversed)
    {
        n[x] = env.L[g];
        b[x] = reversed ? env.rev[g] : env.fwd[g];
        p[x] = reversed ? n[x] - pos - (uint32_t)env.seed_len : pos;
        if (reversed) rev |= 1u << x;
    }
    __device__ __forceinline__ void fill(int used)
    {
        MH_PRAGMA_UNROLL
        for (int x = 1; x < K; ++x)
            if (x >= used) {
                b[x] = b[0];
                p[x] = p[0];
                n[x] = n[0];
            }
    }
    __device__ __forceinline__ uint32_t room_left() const
    {
        uint32_t r = p[0];
        MH_PRAGMA_UNROLL
        for (int x = 1; x < K; ++x) r = p[x] < r ? p[x] : r;
        return r;
    }
    __device__ __forceinline__ uint32_t room_right() const
    {
        uint32_t r = n[0] - p[0];
        MH_PRAGMA_UNROLL
        for (int x = 1; x < K; ++x) r = n[x] - p[x] < r ? n[x] - p[x] : r;
        return r - S;
    }
    // bit i: the windows c + i characters from the seed's (left or right of it)
    // match; 0 past the room
    template <bool RIGHT> __device__ __forceinline__ uint32_t chunk(uint32_t c, uint32_t room) const
    {
        if (c > room) return 0;
        const uint32_t cnt = room - c < 31 ? room - c + 1 : 32;      // windows inside
        const uint32_t d = RIGHT ? c : 0u - (c + cnt - 1);           // the first by position
        uint32_t m = 0;
        if (PAL) {
            uint64_t fh, fl, dh = 0, dl = 0;
            win64((const uint32_t *)b[0], p[0] + d, (n[0] + 15) / 16 + 1, &fh, &fl);
            MH_PRAGMA_UNROLL
            for (int x = 1; x < K; ++x) {
                uint64_t h, l;
                win64((const uint32_t *)b[x], p[x] + d, (n[x] + 15) / 16 + 1, &h, &l);
                dh |= fh ^ h;
                dl |= fl ^ l;
            }
            const uint64_t diff = char_bits(dh | dh >> 1, dl | dl >> 1);
            uint32_t bad = 0;
            for (uint32_t t = pat; t; t &= t - 1) bad |= (uint32_t)(diff >> __builtin_ctz(t));
            if (rev) {
                // windows that are their own reverse complement
                const uint64_t b1 = char_bits(fh >> 1, fl >> 1), b0 = char_bits(fh, fl);
                uint32_t own = ~0u;
                for (uint32_t t = pat; t; t &= t - 1) {
                    const uint32_t a = __builtin_ctz(t), z = S - 1 - a;
                    if (a > z) break;
                    own &= (uint32_t)((b1 >> a) ^ (b1 >> z)) & (uint32_t)((b0 >> a) ^ (b0 >> z));
                }
                bad |= own;
            }
            m = ~bad;
        } else {
            // eight positions' values at once
            for (uint32_t i0 = 0; i0 < cnt; i0 += 8) {
                uint64_t f[8];
                uint32_t ok = 0xFF;
                MH_PRAGMA_UNROLL
                for (uint32_t u = 0; u < 8; ++u) {
                    const uint32_t i = i0 + u < cnt ? i0 + u : cnt - 1;
                    f[u] = ((const uint64_t *)b[0])[p[0] + d + i];
                }
                MH_PRAGMA_UNROLL
                for (int x = 1; x < K; ++x) {
                    const uint32_t r = (rev >> x) & 1u;
                    uint64_t v[8];
                    MH_PRAGMA_UNROLL
                    for (uint32_t u = 0; u < 8; ++u) {
                        const uint32_t i = i0 + u < cnt ? i0 + u : cnt - 1, q = p[x] + d + i;
                        v[u] = ((const uint64_t *)b[x])[r ? n[x] - q - S : q];
                    }
                    MH_PRAGMA_UNROLL
                    for (uint32_t u = 0; u < 8; ++u)
                        if (((f[u] ^ v[u]) & mask) != 0 || (uint32_t)((f[u] ^ v[u]) & 1ull) != r) ok &= ~(1u << u);
                }
                m |= ok << i0;
            }
        }
        if (!RIGHT) m = __brev(m) >> (32 - cnt);
        return cnt < 32 ? m & ((1u << cnt) - 1) : m;
    }
};

// chunk() for a wavefront's 64 chunks in a row from c, a lane each.  Values by
// position are read a window a lane (a chunk a lane, a load's lanes are 256 bytes
// apart, and identical genomes of 2 million bases took 19.2 ms, 17.7 this way).
template <bool RIGHT, int K, bool PAL>
__device__ __forceinline__ uint32_t chunk_wave(const Walk<K, PAL> &w, uint64_t c, uint32_t room)
{
    const uint32_t lane = threadIdx.x & 63;
    if constexpr (PAL) {
        const uint64_t at = c + 32 * lane;
        return at <= room ? w.template chunk<RIGHT>((uint32_t)at, room) : 0;
    } else {
        uint32_t m = 0;
        MH_PRAGMA_UNROLL
        for (uint32_t j = 0; j < 32; j += 8) {
            uint64_t f[8];
            uint32_t ok = 0;
            MH_PRAGMA_UNROLL
            for (uint32_t u = 0; u < 8; ++u) {
                const uint64_t at = c + 64 * (j + u) + lane;
                const uint32_t d = at <= room ? (uint32_t)at : 0;
                ok |= (at <= room ? 1u : 0u) << u;
                f[u] = ((const uint64_t *)w.b[0])[RIGHT ? w.p[0] + d : w.p[0] - d];
            }
            MH_PRAGMA_UNROLL
            for (int x = 1; x < K; ++x) {
                const uint32_t r = (w.rev >> x) & 1u;
                uint64_t v[8];
                MH_PRAGMA_UNROLL
                for (uint32_t u = 0; u < 8; ++u) {
                    const uint64_t at = c + 64 * (j + u) + lane;
                    const uint32_t d = at <= room ? (uint32_t)at : 0, q = RIGHT ? w.p[x] + d : w.p[x] - d;
                    v[u] = ((const uint64_t *)w.b[x])[r ? w.n[x] - q - w.S : q];
                }
                MH_PRAGMA_UNROLL
                for (uint32_t u = 0; u < 8; ++u)
                    if (((f[u] ^ v[u]) & w.mask) != 0 || (uint32_t)((f[u] ^ v[u]) & 1ull) != r) ok &= ~(1u << u);
            }
            MH_PRAGMA_UNROLL
            for (uint32_t u = 0; u < 8; ++u) {
                const uint64_t b = __ballot((ok >> u) & 1u);
                if (lane >> 1 == j + u) m = (uint32_t)(lane & 1 ? b >> 32 : b);
            }
        }
        return m;
    }
}

// the matching windows of m with another within the next S bits of m
__device__ __forceinline__ uint32_t followed(uint32_t m, uint32_t S)
{
    uint32_t a = m >> 1;
    for (uint32_t have = 1; have < S && have < 31;) {
        const uint32_t step = have < S - have ? have : S - have;
        a |= step < 32 ? a >> step : 0;
        have += step;
    }
    return m & a;
}

constexpr uint32_t WALK_FAR = 0xFFFFFFFFu;

// One end by a thread: its distance from the seed's window, or one of at least
// lim once it is known to reach that far; false past WALK_CHUNKS chunks.
template <bool RIGHT, class W>
__device__ __forceinline__ bool walk_end(const W &w, uint32_t *end, uint32_t lim = WALK_FAR)
{
    const uint32_t room = RIGHT ? w.room_right() : w.room_left();
    uint32_t last = 0;
    for (uint32_t c = 0; c < 32 * WALK_CHUNKS; c += 32) {
        const uint32_t m = w.template chunk<RIGHT>(c, room);
        if (m) {
            if (c + __builtin_ctz(m) - last > w.S) {
                *end = last;
                return true;
            }
            // the first that none follows within S: the chunk's last, or the end
            const uint32_t lone = m & ~followed(m, w.S);
            last = c + __builtin_ctz(lone);
            if ((lone & (lone - 1)) || last >= lim) {
                *end = last;
                return true;
            }
        }
        if (c + 31 >= room || c + 31 - last >= w.S) {
            *end = last;
            return true;
        }
    }
    return false;
}

// The same by WALK_BLOCK threads, a chunk each; the last WALK_AHEAD only show
// the others whether a match follows within a seed length (of at most 64).
constexpr uint32_t WALK_AHEAD = 3;
constexpr uint32_t WALK_STEP = 32 * (WALK_BLOCK - WALK_AHEAD);      // windows a step
template <bool RIGHT, class W>
__device__ __forceinline__ uint32_t walk_end_block(const W &w, uint32_t *lds, uint32_t lim = WALK_FAR)
{
    const uint32_t room = RIGHT ? w.room_right() : w.room_left(), t = threadIdx.x;
    uint32_t *first = lds, *best = lds + WALK_BLOCK;
    for (uint64_t c0 = 0; c0 <= room; c0 += WALK_STEP) {
        if (lim != WALK_FAR && c0 > lim) return lim;      // every match before it is followed
        const uint64_t c = c0 + 32 * t;
        const uint32_t m = chunk_wave<RIGHT>(w, c - 32 * (t & 63), room);
        __syncthreads();
        first[t] = m ? (uint32_t)__builtin_ctz(m) : 0xFFFFFFFFu;     // in its chunk
        if (t == 0) *best = 0xFFFFFFFFu;
        __syncthreads();
        if (m && t < WALK_BLOCK - WALK_AHEAD) {
            const uint32_t lone = m & ~followed(m, w.S), at = __builtin_ctz(lone);
            bool stop = (lone & (lone - 1)) != 0;
            if (!stop) {
                uint32_t gap = 0xFFFFFFFFu;      // to the next match
                MH_PRAGMA_UNROLL
                for (uint32_t u = WALK_AHEAD; u > 0; --u)
                    if (first[t + u] != 0xFFFFFFFFu) gap = 32 * u + first[t + u] - at;
                stop = gap > w.S;
            }
            if (stop) atomicMin(best, (uint32_t)c + at);
        }
        __syncthreads();
        if (*best != 0xFFFFFFFFu) return *best;
    }
    return 0;      // (not reached: the last matching window stops it)
}

#endif

}  // namespace mh
