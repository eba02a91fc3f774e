// Synaptic currents of a few ticks for one range of posts, summed in LDS from the spikes (no
// global atomics).
//
// Layout: spike-major rows (Table::SpikeRows), range by range: for a range of `bin` posts, row
// q * n_pre + pre holds presynaptic neuron pre's synapses onto the range with delays
// kSpkDelays q + 1 .. kSpkDelays (q + 1), in ascending (delay, post, synapse id).
// Activity: spike words, and a digest per segment of neurons: how many spiked and, up to
// kDigIds, which (past that the words are read).
//
// A workgroup owns the posts of one range in one batch entry, a thread per post.  It lists the
// active presynaptic neurons of the ticks that reach its current ticks ("visits", from the
// digests), looks up where each one's synapses onto its range lie, loads those entries flat
// (a lane per entry), and links every entry that arrives in one of the ticks
// into a list per (tick, post) in LDS with an exchange.  The post's thread then adds its lists'
// terms in entry order.  Visits are made in descending spike tick (ascending delay for any one
// arrival tick), then ascending neuron, the recurrent ones before the inputs', so entry order is
// ascending (column, synapse id) in each population, the order in which TF's CPU
// UnsortedSegmentSum meets the events of a post (models.py:141-169).  SPLIT (deterministic mode):
// the two populations have lists, and sums, of their own, as the reference has; otherwise (event
// mode) one sum takes both.
//
// That work grows with the spikes.  Where the batch entry's last window had many, the recurrent currents are summed from the posts' rows instead (win_dense): every entry tested
// against a history of the last 8 ticks per neuron, the hits added in the same order, so the sums have
// the same bits.
#pragma once

#include "glif_internal.h"

namespace glif {

// memory the kernel's arguments lie in (scalar loads)
#define WIN_CONST __attribute__((address_space(4)))

constexpr int kWinMaxThreads = kSpkMaxBin;
constexpr int kWinTicks = 3;      // current ticks of one launch (see cell.hip)
constexpr int kWinK = 3;          // visits per thread listed at a time
constexpr int kWinJ = 4;          // entries per thread loaded at a time
constexpr int kWinSlots = 8;      // linked entries held, per thread
constexpr int kDigIds = 15, kDigHalfs = 16;   // a digest: u16 count, then up to kDigIds positions
constexpr int kDigInputs = 512;   // inputs per digest
constexpr uint32_t kNil16 = 0xFFFF;
static_assert(kWinTicks * (kWinMaxThreads / kWave) <= kWave);   // a lane per spike word of a workgroup
static_assert(kWinJ <= kWinSlots && kWinSlots * kWinMaxThreads < static_cast<int>(kNil16));

// Row length of the basis in LDS (vector reads).
constexpr int win_basis_stride(int nb) { return nb <= 1 ? 1 : nb <= 2 ? 2 : nb <= 4 ? 4 : 8; }

// One presynaptic population's activity and rows.  Neurons come in n_seg segments of seg.
struct WinSrc {
    const uint64_t *words;  // word w of (slot, b): words[(slot * B + b) * W + w]
    const uint16_t *dig;    // digest j of (slot, b): dig + ((slot * B + b) * n_seg + j) * kDigHalfs
    const int32_t *off;     // first entry of (range, row) at range * rows + row (ascending over the whole table)
    const uint2 *ent;       // {post & 0xFFFF | (delay - 1) % kSpkDelays << 16 | syn_id << 24, weight bits}
    int32_t W, n_pre;
    int32_t rows;           // 0: no synapses
    int32_t D;              // delay slots; 0: no delay (inputs), a spike arrives in its own tick
    int32_t slot0;          // slot of tick 0
    int32_t seg, n_seg;
};

// The recurrent population's rows and history (win_dense).
struct WinDense {
    const uint64_t *words;  // the spike words (WinSrc::words of the recurrent population)
    const uint8_t *hist;    // [B][Np], bit k: z of tick t0 - 1 - k; nullptr: made in LDS from the words
    const int32_t *row;     // post-grouped table: row pointers,
    const uint32_t *pd;     // pre | (delay - 1) << 24,
    const uint8_t *sid;
    const float *w;
    int32_t N, Np, D;
    int32_t cap;            // hits queued per wave
};
constexpr int kDenseMaxDelay = 6;   // a delay-d spike of the first current tick is bit d + 1
constexpr int kRateRanges = 8;      // ranges whose spikes are counted for the choice
constexpr int kDenseU = 4;          // entries per lane tested together,
constexpr int kDenseAhead = 3;      // and rounds of them loaded ahead (pd's padding holds that many)
static_assert(2 * kDenseU * kWave * kDenseAhead <= kPdPad);
constexpr int kDenseLoads = 4;      // hits per lane whose weights are loaded together
constexpr int kDenseAdd = 4;        // hits of a post read together

// Write the digest of n_words spike words; returns how many spiked.
__device__ inline uint32_t win_digest(const uint64_t *w, int n_words, uint16_t *dig) {
    uint32_t cnt = 0;
#pragma unroll 1
    for (int i = 0; i < n_words; ++i) {
        uint64_t x = w[i];
        while (x) {
            if (++cnt <= kDigIds) dig[cnt] = static_cast<uint16_t>(i * kWave + __builtin_ctzll(x));
            x &= x - 1ull;
        }
    }
    dig[0] = static_cast<uint16_t>(cnt);
    return cnt;
}

// LDS of a workgroup of `threads` threads and RP posts: the linked entries ({weight, next |
// syn_id << 16}), the visits' first entries (relative to their flat position) and arrival
// ticks, the marks of the entries being loaded, the lists' heads [list][post] and the padded basis.
struct WinLds {
    uint2 *rec;
    int32_t *vbase;
    uint16_t *vinfo;    // arrival tick of the row's first delay + 128, from the first current tick; bit 8: inputs
    uint16_t *mark;
    int32_t *heads;
    int32_t *part;
    float *basis;
    int threads;
    // bytes before the basis, and of the basis
    static size_t room(int threads, int lists, int RP) {
        return static_cast<size_t>(threads) * (kWinSlots * sizeof(uint2) + kWinK * 6 + kWinJ * 2) +
               sizeof(int32_t) * (lists * static_cast<size_t>(RP) + 16);
    }
    static size_t basis_bytes(int n_types, int nb) {
        return sizeof(float) * static_cast<size_t>(n_types) * win_basis_stride(nb);
    }
    __device__ static WinLds carve(char *p, int threads, int lists, int RP, int room) {
        // threads and RP are multiples of 64: every part starts on a multiple of 16 bytes
        WinLds l;
        l.threads = threads;
        l.basis = reinterpret_cast<float *>(p + room);
        l.rec = reinterpret_cast<uint2 *>(p);
        p += threads * kWinSlots * sizeof(uint2);
        l.vbase = reinterpret_cast<int32_t *>(p);
        p += threads * kWinK * sizeof(int32_t);
        l.vinfo = reinterpret_cast<uint16_t *>(p);
        p += threads * kWinK * sizeof(uint16_t);
        l.mark = reinterpret_cast<uint16_t *>(p);
        p += threads * kWinJ * sizeof(uint16_t);
        l.heads = reinterpret_cast<int32_t *>(p);
        p += lists * RP * sizeof(int32_t);
        l.part = reinterpret_cast<int32_t *>(p);
        return l;
    }
};

// Inclusive scan over the wave's lanes by DPP (row shifts within 16 lanes, then the rows'
// last lanes broadcast), identity 0.
template <bool MAX>
__device__ inline int win_wave_scan(int x) {
#define GLIF_WIN_DPP(ctrl, rows)                                                    \
    {                                                                               \
        const int y = __builtin_amdgcn_update_dpp(0, x, ctrl, rows, 0xF, false);    \
        x = MAX ? max(x, y) : x + y;                                                \
    }
    GLIF_WIN_DPP(0x111, 0xF) GLIF_WIN_DPP(0x112, 0xF) GLIF_WIN_DPP(0x114, 0xF) GLIF_WIN_DPP(0x118, 0xF)
    GLIF_WIN_DPP(0x142, 0xA) GLIF_WIN_DPP(0x143, 0xC)
#undef GLIF_WIN_DPP
    return x;
}

// Exclusive scan of v >= 0 over the workgroup's threads (sum, or running maximum); *total over
// all of them (at most 16 waves).  Every thread calls it; the first barrier inside orders what
// came before it.
template <bool MAX>
__device__ inline int win_scan(const WinLds &l, int v, int *total) {
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave, waves = l.threads / kWave;
    const int x = win_wave_scan<MAX>(v);
    if (lane == kWave - 1) l.part[wv] = x;
    __syncthreads();
    // every wave scans the waves' totals in its first 16 lanes
    const int y = win_wave_scan<MAX>(lane < waves ? l.part[lane] : 0);
    const int base = wv ? __shfl(y, wv - 1, kWave) : 0;
    *total = __builtin_amdgcn_readlane(y, waves - 1);
    __syncthreads();
    if (!MAX) return base + x - v;
    return max(base, __builtin_amdgcn_update_dpp(0, x, 0x138, 0xF, 0xF, false));   // wave_shr:1
}

// Put the list that starts at h and has more than one entry into ascending entry order, in place,
// and return its first entry: insertion with a finger at the last insertion (the links of one wave
// come out in descending entry order, so most insertions are next to the one before).
__device__ inline uint32_t win_sort_list(uint2 *rec, uint32_t h) {
    auto next = [&](uint32_t j) { return rec[j].y & kNil16; };
    auto link = [&](uint32_t j, uint32_t n) { rec[j].y = (rec[j].y & ~kNil16) | n; };
    uint32_t first = h, finger = h, cur = next(h);
    link(h, kNil16);
    while (cur != kNil16) {
        const uint32_t after = next(cur);
        if (cur < first) {
            link(cur, first);
            first = finger = cur;
        } else {
            uint32_t p = cur > finger ? finger : first;
            for (uint32_t nx = next(p); nx != kNil16 && nx < cur; nx = next(p)) p = nx;
            link(cur, next(p));
            link(p, cur);
            finger = p;
        }
        cur = after;
    }
    return first;
}

// x / d for x < 2^21 and a quotient below 2^20 (the half keeps the approximate reciprocal's error, under 2^-21
// of the quotient, from crossing a whole number)
__device__ inline int win_div(uint32_t x, uint32_t d) {
    if (x >= (1u << 21)) return static_cast<int>(x / d);
    return static_cast<int>((static_cast<float>(x) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(d)));
}

// Add the terms of post `local`'s lists to s and empty them.
template <int NB, bool SPLIT>
__device__ inline void win_sum_post(const WinLds &l, int RP, int local, float (&s)[(SPLIT ? 2 : 1) * kWinTicks][NB]) {
    constexpr int BS = win_basis_stride(NB), L = (SPLIT ? 2 : 1) * kWinTicks;
    // lists of more than one entry into entry order
#pragma unroll 1
    for (int i = 0; i < L; ++i) {
        const int h = l.heads[i * RP + local];
        if (h >= 0 && (l.rec[h].y & kNil16) != kNil16)
            l.heads[i * RP + local] = static_cast<int>(win_sort_list(l.rec, static_cast<uint32_t>(h)));
    }
    uint32_t h[L];
#pragma unroll
    for (int i = 0; i < L; ++i) h[i] = static_cast<uint32_t>(l.heads[i * RP + local]) & kNil16;
#pragma unroll
    for (int i = 0; i < L; ++i) l.heads[i * RP + local] = -1;
#pragma unroll
    for (int i = 0; i < L; ++i) {
#pragma unroll 1
        while (h[i] != kNil16) {
            const uint2 e = l.rec[h[i]];
            const float wv = __uint_as_float(e.x);
            const float *bs = l.basis + (e.y >> 16) * BS;
#pragma unroll
            for (int r = 0; r < NB; ++r) s[i][r] = s[i][r] + wv * bs[r];
            h[i] = e.y & kNil16;
        }
    }
}

// the element at a byte offset below 4 GiB of a uniform pointer (scalar-base addresses)
template <class T>
__device__ inline T win_ld(const T *p, uint32_t byte) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + byte);
}

// The 8 x 8 bit matrix x (row r in byte r) transposed: Hacker's Delight's three exchanges of blocks.
__device__ inline uint64_t win_transpose(uint64_t x) {
    uint64_t t = (x ^ (x >> 7)) & 0x00AA00AA00AA00AAull;
    x ^= t ^ (t << 7);
    t = (x ^ (x >> 14)) & 0x0000CCCC0000CCCCull;
    x ^= t ^ (t << 14);
    t = (x ^ (x >> 28)) & 0x00000000F0F0F0F0ull;
    return x ^ t ^ (t << 28);
}

// Whether a window takes win_dense, of the batch entry's row of the rates (n: lane j the j-th, loaded where there is
// other work to wait for, and not by a scalar load: every wait for one waits for all).
__device__ inline bool win_dense_due(uint32_t n, int limit, int n_ranges) {
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < kRateRanges; ++j) sum += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(n), j));
    return limit && static_cast<int64_t>(sum) * n_ranges >= static_cast<int64_t>(limit - 1) * kRateRanges;
}

// The spikes n of a window in range `range`, where that is one of those looked at.
__device__ inline void win_rate(uint32_t *rate, int range, int n_ranges, uint32_t n) {
#pragma unroll
    for (int j = 0; j < kRateRanges; ++j)
        if (j * n_ranges / kRateRanges == range) rate[j] = n;
}

// The recurrent currents of the ticks i_lo + [i0, i1) for the RP posts from n0 on in batch entry b, from
// their rows: a wave takes its 64 posts' rows as one run of entries, 256 at a time, and queues the hits
// ({entry, the ticks it arrives in << 16}) in LDS in row order; once a queue is nearly full their weights
// and types are loaded together, in place, and added post by post, a lane per tick and receptor.  Called by every thread; leaves the heads at -1.
template <int NB, int L>
__device__ inline void win_dense(const WIN_CONST WinDense &a, const WinLds &l, int t0, int B, int b, int i0, int i1, int n0,
                                 int RP, float (&s)[L][NB]) {
    constexpr int BS = win_basis_stride(NB), U = kDenseU;
    const int tid = threadIdx.x, threads = l.threads, lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave), wave0 = wv * kWave;
    // the history where it fits, then the waves' queues
    char *base = reinterpret_cast<char *>(l.rec);
    uint2 *queue = reinterpret_cast<uint2 *>(base + (a.hist ? 0 : a.Np)) + wv * a.cap;
    if (!a.hist) {
        // a thread per word: 8 neurons' bits of 8 ticks are an 8 x 8 bit matrix, transposed
        const int W = a.Np / kWave;
        for (int i = tid; i < W; i += threads) {
            uint64_t x[8];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                x[k] = k <= a.D + 1 ? a.words[(static_cast<int64_t>(t0 - 1 - k + a.D) * B + b) * W + i] : 0ull;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                uint64_t m = 0;
#pragma unroll
                for (int k = 0; k < 8; ++k) m |= (x[k] >> (8 * j) & 0xFFull) << (8 * k);
                reinterpret_cast<uint64_t *>(base)[i * 8 + j] = win_transpose(m);
            }
        }
    }
    __syncthreads();
    if (wave0 < RP && n0 + wave0 < a.N) {
        // bits of a history byte shifted by delay - 1: 2, 1, 0 for the current ticks 0, 1, 2
        uint32_t ticks = 0;
        for (int i = i0; i < i1; ++i) ticks |= 4u >> i;
        const int32_t rp = a.row[min(n0 + wave0 + lane, a.N)];
        const int32_t j0 = __builtin_amdgcn_readfirstlane(rp);
        const int32_t j1 = __builtin_amdgcn_readfirstlane(a.row[min(n0 + wave0 + kWave, a.N)]);
        constexpr int32_t kNone = 0x7FFFFFFF;
        int32_t first = kNone;   // this post's first hit, counted over the wave's
        int known = 0;           // posts whose rows have begun, and where the next one's does
        int32_t begin = 0;       // (from j0)
        int32_t hits = 0, q0 = 0;   // hits so far, the first one in the queue
        auto fence = [&]() {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        // LP lanes add a post's hits, one for each tick and receptor, G posts at a time
        constexpr int LP = 3 * NB <= 4 ? 4 : 3 * NB <= 8 ? 8 : 3 * NB <= 16 ? 16 : 32, G = kWave / LP;
        static_assert(kWinTicks == 3);
        const int g = lane / LP;
        const uint32_t r4 = lane % LP % NB * 4, bit = lane % LP < 3 * NB ? 0x40000u >> (lane % LP / NB) : 0u;
        int posts = 0;         // posts done
        float carry = 0.0f;    // the next one's sums so far (lanes 0 .. LP - 1, and their copies)
        auto add = [&](bool last) {
            // the queued hits' weights and types, all loads of kDenseLoads rounds together
            fence();
#pragma unroll 1
            for (int32_t i0 = 0; i0 < hits - q0; i0 += kDenseLoads * kWave) {
                uint2 e[kDenseLoads];
                float w[kDenseLoads];
                uint32_t sid[kDenseLoads];
#pragma unroll
                for (int u = 0; u < kDenseLoads; ++u) {
                    e[u] = queue[min(i0 + u * kWave + lane, hits - q0 - 1)];
                    w[u] = win_ld(a.w + j0, e[u].x * 4u);
                    sid[u] = win_ld(a.sid + j0, e[u].x);
                }
                fence();   // a clamped lane reads a slot that another lane writes
#pragma unroll
                for (int u = 0; u < kDenseLoads; ++u)
                    if (i0 + u * kWave + lane < hits - q0)
                        queue[i0 + u * kWave + lane] = make_uint2(__float_as_uint(w[u]), sid[u] * (BS * 4) | e[u].y);
            }
            fence();
            const int done_to = last ? known : known - 1;   // the last row begun is perhaps not at its end
#pragma unroll 1
            for (int p0 = posts; p0 < known; p0 += G) {
                const int p = p0 + g;
                int32_t i = __shfl(first, min(p, kWave - 1), kWave), end = __shfl(first, min(p + 1, kWave - 1), kWave);
                i = p < known ? max(i, q0) : q0;   // a row not begun has no hits, and no first one
                end = p < known ? (p + 1 < known ? end : hits) : q0;
                float acc = p == posts ? carry : 0.0f;
                const uint2 *q = queue + (i - q0);
                auto term = [&](const uint2 e) { return __uint_as_float(e.x) * win_ld(l.basis, (e.y & 0xFFFFu) + r4); };
#pragma unroll 1
                for (; i + kDenseAdd <= end; i += kDenseAdd, q += kDenseAdd) {
                    uint2 e[kDenseAdd];
                    float x[kDenseAdd];
#pragma unroll
                    for (int u = 0; u < kDenseAdd; ++u) e[u] = q[u];
#pragma unroll
                    for (int u = 0; u < kDenseAdd; ++u) x[u] = term(e[u]);
#pragma unroll
                    for (int u = 0; u < kDenseAdd; ++u) acc = e[u].y & bit ? acc + x[u] : acc;
                }
#pragma unroll 1
                for (; i < end; ++i, ++q) {
                    const uint2 e = *q;
                    const float x = term(e);
                    acc = e.y & bit ? acc + x : acc;
                }
                // to the posts' lanes
                const bool mine = lane >= p0 && lane < p0 + G && lane < done_to;
#pragma unroll
                for (int t = 0; t < kWinTicks; ++t)
#pragma unroll
                    for (int q = 0; q < NB; ++q) {
                        const float x = __shfl(acc, (lane - p0) * LP + t * NB + q, kWave);
                        s[t][q] = mine ? x : s[t][q];
                    }
                if (p0 + G >= known) carry = __shfl(acc, (known - 1 - p0) * LP + lane % LP, kWave);
            }
            posts = done_to;
            fence();
            q0 = hits;
        };
        const uint32_t n = static_cast<uint32_t>(j1 - j0);
        // hist(pre): the history byte; one loop for each place it is read from, so that each waits for its
        // own kind of load only
        auto walk = [&](auto hist) {
            uint32_t next[kDenseAhead][U];
            // the entries from `at` on: past the run's end the next rows', past the table's its padding
            auto load = [&](uint32_t (&x)[U], const uint32_t *at) {
#pragma unroll
                for (int u = 0; u < U; ++u) x[u] = win_ld(at, static_cast<uint32_t>(lane + u * kWave) * 4u);
            };
            const uint32_t *at = a.pd + j0;
            // the entries x of [j, j + U waves), and x loaded anew kDenseAhead rounds on (rounds past the run's
            // end find nothing: a round that may be left out makes the next wait for every load)
            auto round = [&](uint32_t (&x)[U], uint32_t j) {
                uint32_t m[U];
#pragma unroll
                for (int u = 0; u < U; ++u) m[u] = hist(x[u] & kLow24);
#pragma unroll
                for (int u = 0; u < U; ++u) m[u] = (m[u] >> (x[u] >> 24)) & ticks;
                at += U * kWave;
                load(x, at + (kDenseAhead - 1) * U * kWave);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint32_t ju = j + u * kWave, in = ju < n ? min(n - ju, 64u) : 0u;   // lanes before the run's end
                    const uint64_t on = __ballot(m[u] != 0u) & (in ? ~0ull >> (kWave - in) : 0ull);
                    while (begin < static_cast<int32_t>(ju) + kWave) {   // a row begins here
                        const int32_t h = hits + __popcll(on & ((1ull << (begin - ju)) - 1ull));
                        first = lane == known ? h : first;
                        begin = ++known < kWave ? __builtin_amdgcn_readlane(rp, known) - j0 : kNone;
                    }
                    if (on) {
                        if (__builtin_amdgcn_inverse_ballot_w64(on)) {
                            const int before = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(on >> 32),
                                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(on), 0));
                            queue[hits - q0 + before] = make_uint2(ju + lane, m[u] << 16);
                        }
                        hits += __popcll(on);
                    }
                }
                if (hits - q0 > a.cap - U * kWave) add(false);
            };
#pragma unroll
            for (int k = 0; k < kDenseAhead; ++k) load(next[k], at + k * U * kWave);
#pragma unroll 1
            for (uint32_t j = 0; j < n; j += kDenseAhead * U * kWave) {
#pragma unroll
                for (int k = 0; k < kDenseAhead; ++k) round(next[k], j + k * U * kWave);
            }
            first = lane >= known ? hits : first;   // rows that begin at the run's end
            known = kWave;
            add(true);
        };
        using lds_u8 = const __attribute__((address_space(3))) uint8_t;
        using global_u8 = const __attribute__((address_space(1))) uint8_t;
        if (n == 0) {
        } else if (!a.hist) {
            lds_u8 *h = (lds_u8 *)base;
            walk([&](uint32_t pre) -> uint32_t { return h[pre]; });
        } else {
            global_u8 *h = (global_u8 *)(a.hist + static_cast<int64_t>(b) * a.Np);
            walk([&](uint32_t pre) -> uint32_t { return h[pre]; });
        }
    }
    __syncthreads();
    for (int i = tid; i < L * RP; i += threads) l.heads[i] = -1;
    __syncthreads();
}

// Currents of the ticks i_lo + [i0, i1) (0 <= i0, i1 <= kWinTicks) for the RP posts of range `range`
// (the first one's number's low bits: post0) in batch entry b, from the recurrent population (rec; not with
// with_rec false) and the inputs (inp), added to s of the post's thread: [tick], or SPLIT [population][tick].
// Called by every thread; heads are all -1 on entry and on return.
template <int NB, bool SPLIT>
__device__ inline void win_currents(const WIN_CONST WinSrc &rec, const WIN_CONST WinSrc &inp, bool with_rec, const WinLds &l,
                                    int B, int b, int i_lo, int i0, int i1, int range, int RP,
                                    float (&s)[(SPLIT ? 2 : 1) * kWinTicks][NB]) {
    const int tid = threadIdx.x, threads = l.threads;
    const int n_load = kWinJ * threads, n_slots = kWinSlots * threads, n_list = kWinK * threads;
    const uint32_t post0 = static_cast<uint32_t>(range) * static_cast<uint32_t>(RP);
    // Segments in visit order: rows of n_seg, one per (delay group q, spike tick), the latest
    // tick first -- group q's spikes reach [i_lo + i0, i_lo + i1) from `per` ticks (the last group,
    // of fewer delays, from fewer) -- then one per input tick.
    const int per = i1 - i0 - 1 + kSpkDelays, groups = (rec.D + kSpkDelays - 1) / kSpkDelays;
    const uint32_t n_rec =
        with_rec && rec.rows ? static_cast<uint32_t>(groups * per - (groups * kSpkDelays - rec.D)) * static_cast<uint32_t>(rec.n_seg) : 0u;
    const uint32_t n_all = n_rec + (inp.rows ? static_cast<uint32_t>(i1 - i0) * static_cast<uint32_t>(inp.n_seg) : 0u);
    const int32_t *off_r = rec.off + static_cast<int64_t>(range) * rec.rows;
    const int32_t *off_i = inp.off + static_cast<int64_t>(range) * inp.rows;
    int used = 0;   // slots
    for (uint32_t d0 = 0; d0 < n_all; d0 += threads) {
        // this thread's segment
        const uint32_t x = d0 + tid;
        int mine = 0, first = 0, info = 0, n0 = 0, at = 0;
        uint32_t digest = 0;
        const bool pop = x >= n_rec;
        if (x < n_all) {
            const uint32_t rel = pop ? x - n_rec : x, ns = static_cast<uint32_t>(pop ? inp.n_seg : rec.n_seg);
            const int row = win_div(rel, ns), j = static_cast<int>(rel - static_cast<uint32_t>(row) * ns);
            int t = i1 - 1 - row, slot0 = inp.slot0;
            n0 = j * (pop ? inp.seg : rec.seg);
            first = n0;
            info = t + 128 + 256;
            if (!pop) {
                const int q = groups > 1 ? row / per : 0;
                t = i1 - 2 - kSpkDelays * q - (row - q * per);
                slot0 = rec.slot0;
                first = n0 + q * rec.n_pre;
                info = t + 128 + 1 + kSpkDelays * q;
            }
            at = (i_lo + t + slot0) * B + b;
            digest = static_cast<uint32_t>(at) * ns + static_cast<uint32_t>(j);
            mine = (pop ? inp.dig : rec.dig)[static_cast<size_t>(digest) * kDigHalfs];
        }
        int n_vis;
        const int rank0 = win_scan<false>(l, mine, &n_vis);
        for (int r0 = 0; r0 < n_vis; r0 += n_list) {
            // list the visits of ranks [r0, r0 + n_list): rows in vbase
            const int nv = min(n_list, n_vis - r0);
            int rank = rank0 - r0;
            auto visit = [&](int row) {
                if (rank >= 0 && rank < nv) {
                    l.vbase[rank] = row;
                    l.vinfo[rank] = static_cast<uint16_t>(info);
                }
                ++rank;
            };
            if (mine == 0) {
            } else if (mine <= kDigIds) {
                const uint4 *dig = reinterpret_cast<const uint4 *>((pop ? inp.dig : rec.dig) + static_cast<size_t>(digest) * kDigHalfs);
                const uint4 head = dig[0], rest = dig[1];
                uint64_t ids = static_cast<uint64_t>(head.x) | static_cast<uint64_t>(head.y) << 32;
#pragma unroll 1
                for (int u = 1; u <= mine; ++u) {
                    ids >>= 16;
                    if ((u & 3) == 0)
                        ids = u == 4   ? static_cast<uint64_t>(head.z) | static_cast<uint64_t>(head.w) << 32
                              : u == 8 ? static_cast<uint64_t>(rest.x) | static_cast<uint64_t>(rest.y) << 32
                                       : static_cast<uint64_t>(rest.z) | static_cast<uint64_t>(rest.w) << 32;
                    visit(first + static_cast<int>(ids & 0xFFFFull));
                }
            } else {
                const int W = pop ? inp.W : rec.W, n = min(pop ? inp.seg : rec.seg, W * kWave - n0);
                const uint64_t *w = (pop ? inp.words : rec.words) + static_cast<int64_t>(at) * W + n0 / kWave;
#pragma unroll 1
                for (int i = 0; i * kWave < n; ++i) {
                    uint64_t bits = w[i];
                    while (bits) {
                        visit(first + i * kWave + __builtin_ctzll(bits));
                        bits &= bits - 1ull;
                    }
                }
            }
            __syncthreads();
            // where each visit's entries lie: kWinK consecutive visits per thread, the lookups together
            int pre[kWinK], cnt[kWinK], sum = 0;
#pragma unroll
            for (int u = 0; u < kWinK; ++u) {
                const int v = tid * kWinK + u;
                pre[u] = cnt[u] = 0;
                if (v < nv) {
                    const int32_t *o = (l.vinfo[v] & 256 ? off_i : off_r) + l.vbase[v];
                    pre[u] = o[0];
                    cnt[u] = o[1];
                }
            }
#pragma unroll
            for (int u = 0; u < kWinK; ++u) {
                cnt[u] -= pre[u];
                sum += cnt[u];
            }
            int M;
            int at_e = win_scan<false>(l, sum, &M);
#pragma unroll
            for (int u = 0; u < kWinK; ++u) {
                l.vbase[tid * kWinK + u] = pre[u] - at_e;
                pre[u] = at_e;
                at_e += cnt[u];
            }
            if (M == 0) __syncthreads();   // before the next listing writes vbase
            for (int m0 = 0; m0 < M; m0 += n_load) {
                // the visit of every entry: visits mark their first entry, a running maximum fills in
                for (int i = tid; i < n_load / 2; i += threads) reinterpret_cast<uint32_t *>(l.mark)[i] = 0u;
                __syncthreads();
#pragma unroll
                for (int u = 0; u < kWinK; ++u) {
                    if (cnt[u] > 0 && pre[u] < m0 + n_load && pre[u] + cnt[u] > m0)
                        l.mark[max(pre[u] - m0, 0)] = static_cast<uint16_t>(tid * kWinK + u + 1);
                }
                __syncthreads();
                {
                    uint16_t *mk = l.mark + tid * kWinJ;
                    int vis[kWinJ], run = 0, all;
#pragma unroll
                    for (int j = 0; j < kWinJ; ++j) vis[j] = run = max(run, static_cast<int>(mk[j]));
                    const int before = win_scan<true>(l, run, &all);
#pragma unroll
                    for (int j = 0; j < kWinJ; ++j) mk[j] = static_cast<uint16_t>(max(vis[j], before));
                }
                __syncthreads();
                // the entries, a wave's 64 lanes on consecutive ones (a visit's share a line)
                uint2 e[kWinJ];
                int list[kWinJ];   // the entry's list, -1: arrives in no tick
#pragma unroll
                for (int j = 0; j < kWinJ; ++j) {
                    const int i = j * threads + tid;
                    e[j] = make_uint2(0u, 0u);
                    list[j] = 0;
                    if (m0 + i < M) {
                        const int v = l.mark[i] - 1;
                        list[j] = l.vinfo[v];
                        e[j] = (list[j] & 256 ? inp.ent : rec.ent)[l.vbase[v] + m0 + i];
                    }
                }
#pragma unroll
                for (int j = 0; j < kWinJ; ++j) {
                    const int i = (list[j] & 255) - 128 + static_cast<int>((e[j].x >> 16) & (kSpkDelays - 1));
                    list[j] = i >= i0 && i < i1 ? (SPLIT && (list[j] & 256) ? kWinTicks : 0) + i : -1;
                }
                // slots in entry order
                const int loaded = min(n_load, M - m0);
                if (used + loaded > n_slots) {
                    if (tid < RP) win_sum_post<NB, SPLIT>(l, RP, tid, s);
                    used = 0;
                    __syncthreads();
                }
                int slot = used + tid;
                used += loaded;
#pragma unroll
                for (int j = 0; j < kWinJ; ++j) {
                    if (list[j] >= 0) {
                        const uint32_t local = (e[j].x - post0) & 0xFFFFu;
                        const uint32_t old = static_cast<uint32_t>(atomicExch(&l.heads[list[j] * RP + local], slot));
                        l.rec[slot] = make_uint2(e[j].y, (old & kNil16) | (e[j].x >> 24) << 16);
                    }
                    slot += threads;
                }
                __syncthreads();
            }
        }
    }
    if (tid < RP) win_sum_post<NB, SPLIT>(l, RP, tid, s);
    __syncthreads();
}

}  // namespace glif
