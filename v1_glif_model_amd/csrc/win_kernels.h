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

// Write the digest of n_words spike words.
__device__ inline void win_digest(const uint64_t *w, int n_words, uint16_t *dig) {
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
    __host__ __device__ static size_t bytes(int threads, int lists, int RP, int n_types, int nb) {
        return static_cast<size_t>(threads) * (kWinSlots * sizeof(uint2) + kWinK * 6 + kWinJ * 2) +
               sizeof(int32_t) * (lists * static_cast<size_t>(RP) + 16) +
               sizeof(float) * static_cast<size_t>(n_types) * win_basis_stride(nb);
    }
    __device__ static WinLds carve(char *p, int threads, int lists, int RP) {
        // threads and RP are multiples of 64: every part starts on a multiple of 16 bytes
        WinLds l;
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
        p += 16 * sizeof(int32_t);
        l.basis = reinterpret_cast<float *>(p);
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
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave, waves = blockDim.x / kWave;
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

// Currents of the ticks i_lo + [i0, i1) (0 <= i0, i1 <= kWinTicks) for the RP posts of range `range`
// (the first one's number's low bits: post0) in batch entry b, from the recurrent population (rec)
// and the inputs (inp), added to s of the post's thread: [tick], or SPLIT [population][tick].
// Called by every thread; heads are all -1 on entry and on return.
template <int NB, bool SPLIT>
__device__ inline void win_currents(const WIN_CONST WinSrc &rec, const WIN_CONST WinSrc &inp, const WinLds &l, int B, int b, int i_lo,
                                    int i0, int i1, int range, int RP, float (&s)[(SPLIT ? 2 : 1) * kWinTicks][NB]) {
    const int tid = threadIdx.x, threads = blockDim.x;
    const int n_load = kWinJ * threads, n_slots = kWinSlots * threads, n_list = kWinK * threads;
    const uint32_t post0 = static_cast<uint32_t>(range) * static_cast<uint32_t>(RP);
    // Segments in visit order: rows of n_seg, one per (delay group q, spike tick), the latest
    // tick first -- group q's spikes reach [i_lo + i0, i_lo + i1) from `per` ticks (the last group,
    // of fewer delays, from fewer) -- then one per input tick.
    const int per = i1 - i0 - 1 + kSpkDelays, groups = (rec.D + kSpkDelays - 1) / kSpkDelays;
    const uint32_t n_rec =
        rec.rows ? static_cast<uint32_t>(groups * per - (groups * kSpkDelays - rec.D)) * static_cast<uint32_t>(rec.n_seg) : 0u;
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
