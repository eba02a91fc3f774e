// Op-level entry points of calculate_synaptic_currents (models.py:103-263):
// forward (event push or deterministic pull) and the custom gradient.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "compact.h"
#include "glif_internal.h"
#include "prof.h"
#include "pull_kernels.h"
#include "syn_kernels.h"

namespace glif {

// Tables with a column longer than this take dz over work units and pull in event mode too (the
// background table's shape).  The dz walk sums a column on one lane per 4 batch entries and the
// column scan pushes it on one wave, so their time is the longest column's serial chain (a
// 6600-synapse column: ~4 ms for dz, ~5 ms for the push); the units split long columns over many
// waves and cost at most ~1.5x the walk on short ones (runs of short columns use few lanes).
constexpr int32_t kUnitDzMinColLen = 2048;
// The event push takes the units when the column scan (a wave per 64 columns) would run on fewer
// waves than this (the LGN table's 17,400 columns: 272 waves) or a column has more synapses than
// one unit (its chunks then go to waves of their own).
constexpr int64_t kPushUnitsMaxScanWaves = 2048;
constexpr int32_t kPushUnitsMinColLen = 1024;
constexpr int64_t kPushWideMinSyn = int64_t(4) << 20;   // and the wide units from here: enough waves of them
// The backward takes the units too when the walk would run on fewer lanes than this -- unless G's rows
// are a cache line or more (Bp >= 16) and the columns short: a lane group then waits for few rows, while
// the split walk streams them (whole calls, units against walk, batch 20: 25 synapses a column 42 against
// 25 us, 50: 37 against 26, 62: 53 against 47, 132: 37 against 46; batch 1 at 25: 10 against 16).
constexpr int64_t kUnitDzMaxWalkLanes = 1024 * kWave;
constexpr int64_t kUnitDzMinAvgLen = 96;
// dz alone over long columns takes the wide units once they are enough waves (2.6M synapses in 17,400 columns, batch 1 / 5 /
// 32: 34 / 54 / 86 us by small units, 29 / 41 / 83 by wide ones; with dW beside it 36 / 58 / 104 against 34 / 55 / 145; 1.8M
// in 8,000, batch 32: 52 against 71).
constexpr int64_t kWideDzMinAvgLen = 128, kWideDzMinSyn = int64_t(2) << 20;

// ---------------------------------------------------------------- forward ----
// Deterministic pull of Poisson-count inputs (the background form, models.py:917-931): thread
// per (b, post) walks the post's row in ascending (column, synapse id) -- the order in which
// TF's CPU UnsortedSegmentSum meets the events of this (b, post) -- scaling each weight by its
// input's count, and writes I[b][post][:] (models.py:141-169).  Spike inputs take the row
// pulls over batch masks (pull_kernels.h), which read each entry once for all batch entries.
__global__ void __launch_bounds__(kBlock)
    k_syn_pull_dense(const float *__restrict__ z, int32_t B, int64_t n_cols, int32_t n_post,
                     int32_t n_pre, const int32_t *__restrict__ row_ptr,
                     const uint32_t *__restrict__ pd, const uint8_t *__restrict__ sid,
                     const float *__restrict__ w, const float *__restrict__ basis, int n_types,
                     int nb, float *__restrict__ I) {
    extern __shared__ float basis_lds[];
    load_basis_lds(basis_lds, basis, n_types * nb);
    const int64_t gt = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gt >= static_cast<int64_t>(B) * n_post) return;
    const int b = static_cast<int>(gt / n_post);
    const int32_t n = static_cast<int32_t>(gt % n_post);
    float acc[kMaxBasis];
    for (int r = 0; r < nb; ++r) acc[r] = 0.0f;
    const float *zb = z + static_cast<int64_t>(b) * n_cols;
    for (int32_t j = row_ptr[n]; j < row_ptr[n + 1]; ++j) {
        const uint32_t q = pd[j];
        const int64_t c = static_cast<int64_t>(q & kLow24) + static_cast<int64_t>(q >> 24) * n_pre;
        const float a = zb[c];
        if (!(a > 0.0f)) continue;
        const float wv = w[j] * a;
        const float *bs = basis_lds + sid[j] * nb;
        for (int r = 0; r < nb; ++r) acc[r] = acc[r] + wv * bs[r];
    }
    float *dst = I + gt * nb;
    for (int r = 0; r < nb; ++r) dst[r] = acc[r];
}

// The same over an input table's ELL copy: a thread per post and BB batch entries, so an entry
// (one coalesced load) is read once for all of them; the inputs' counts [input][batch entry] in LDS.
// Each (post, batch entry) adds its row's active entries in row order, as k_syn_pull_dense does.
// Bound by instruction issue, BB batch entries a synapse: background table (66,000 posts, 10 synapses each, 100
// inputs), batch 32: 98 -> 28 us with BB = 8; 3,000 posts with 150 each, batch 1, BB = 8 59 us, 1 16.
constexpr int64_t kEllMaxInputs = 1024;
constexpr int64_t kEllMaxStage = 2048;    // counts that a workgroup stages for its 256 posts
constexpr int32_t kEllEventMaxRow = 48;   // the longest rows pulled in event mode
constexpr int64_t kEllMinLanes = 32768;   // posts x groups of BB batch entries: fewer leave CUs idle

template <int BB>
__global__ void __launch_bounds__(kBlock)
    k_syn_pull_ell(const float *__restrict__ z, int32_t B, int32_t n_cols, int32_t n_post,
                   const int32_t *__restrict__ row_ptr, const uint2 *__restrict__ ell,
                   const float *__restrict__ basis, int n_types, int nb, float *__restrict__ I) {
    extern __shared__ __align__(16) float ell_lds[];   // [n_cols][BB]
    float *basis_lds = ell_lds + static_cast<size_t>(n_cols) * BB;
    const int b0 = static_cast<int>(blockIdx.y) * BB;
    for (int i = threadIdx.x; i < n_cols * BB; i += blockDim.x) {
        const int bb = i / n_cols, c = i - bb * n_cols;
        const float x = b0 + bb < B ? z[static_cast<int64_t>(b0 + bb) * n_cols + c] : 0.0f;
        ell_lds[c * BB + bb] = x > 0.0f ? x : 0.0f;
    }
    load_basis_lds(basis_lds, basis, n_types * nb);
    const int64_t n = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (n >= n_post) return;
    const int32_t len = row_ptr[n + 1] - row_ptr[n];   // without the padding, which an infinite count would turn to NaN
    float acc[BB][kMaxBasis];
#pragma unroll
    for (int bb = 0; bb < BB; ++bb)
#pragma unroll
        for (int r = 0; r < kMaxBasis; ++r) acc[bb][r] = 0.0f;
    for (int32_t j0 = 0; j0 < len; j0 += 4) {
        uint2 e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = ell[static_cast<int64_t>(min(j0 + u, len - 1)) * n_post + n];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (j0 + u >= len) break;
            const float w = __uint_as_float(e[u].y);
            const float *bs = basis_lds + (e[u].x >> 24) * nb;
            float x[BB];
#pragma unroll
            for (int bb = 0; bb < BB; ++bb) x[bb] = ell_lds[(e[u].x & kLow24) * BB + bb];
#pragma unroll
            for (int r = 0; r < kMaxBasis; ++r) {
                if (r >= nb) break;
                const float s = bs[r];
#pragma unroll
                for (int bb = 0; bb < BB; ++bb)
                    acc[bb][r] = x[bb] > 0.0f ? acc[bb][r] + (w * x[bb]) * s : acc[bb][r];
            }
        }
    }
#pragma unroll
    for (int bb = 0; bb < BB; ++bb) {
        if (b0 + bb >= B) break;
        float *dst = I + (static_cast<int64_t>(b0 + bb) * n_post + n) * nb;
#pragma unroll
        for (int r = 0; r < kMaxBasis; ++r)
            if (r < nb) dst[r] = acc[bb][r];
    }
}

// One active column, by a wave; Q = 1: a lane per synapse, else Q lanes (push_column_wide).
template <int Q, class Mult>
__device__ inline void push_spiking(int lane, int32_t lo, int32_t hi, uint32_t m, Mult mult,
                                    const uint32_t *__restrict__ ps, const float *__restrict__ w,
                                    const float *basis_lds, int nb, int32_t n_post, float *__restrict__ I) {
    const int64_t bstride = static_cast<int64_t>(n_post) * nb;
    if (Q == 1) push_column<kWave>(lane, lo, hi, m, mult, ps, w, basis_lds, nb, bstride, nb, 1, I);
    else push_column_wide<kWave, Q>(lane, lo, hi, m, mult, ps, w, basis_lds, nb, bstride, I);
}

// Event push straight from z [B][n_cols]: a wave per 64 consecutive columns builds each
// column's batch mask (z > 0, the test of tf.where at models.py:128-130), and all 64 lanes
// push the wave's active columns one after another.  No column list, no count pass.
// The event push over the table's work units (a run of up to 64 short columns, or a chunk of
// at most kUnitEntries synapses of a long column), a wave per unit: the lanes hold the
// run's columns' batch masks, and all 64 lanes push each active column's share of the unit.
// For tables whose column scan would run on few waves (few columns, or long ones).
template <bool COUNTS, int Q>
__global__ void __launch_bounds__(kBlock)
    k_syn_push_units(const float *__restrict__ z, int32_t B, int64_t n_cols, const int4 *__restrict__ units,
                     int32_t n_units, const int32_t *__restrict__ col_ptr, const uint32_t *__restrict__ ps,
                     const float *__restrict__ w, const float *__restrict__ basis, int n_types, int nb,
                     int32_t n_post, float *__restrict__ I) {
    extern __shared__ float basis_lds[];
    load_basis_lds(basis_lds, basis, n_types * nb);
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t ui = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWave) +
                       __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
    if (ui >= n_units) return;  // the whole wave leaves together
    const int4 un = units[ui];
    uint32_t m = 0u;
    if (lane < un.y)
        for (int b = 0; b < B; ++b) m |= (z[b * n_cols + un.x + lane] > 0.0f ? 1u : 0u) << b;
    uint64_t act = __ballot(m != 0u);
    while (act) {
        const int l = __builtin_ctzll(act);
        act &= act - 1ull;
        const uint32_t ml = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m), l));
        const int64_t cl = un.x + l;
        const int32_t lo = un.y == 1 ? un.z : col_ptr[cl];
        const int32_t hi = un.y == 1 ? un.w : col_ptr[cl + 1];
        if (COUNTS) push_spiking<Q>(lane, lo, hi, ml, MultF32{z + cl, n_cols}, ps, w, basis_lds, nb, n_post, I);
        else push_spiking<Q>(lane, lo, hi, ml, MultOne{}, ps, w, basis_lds, nb, n_post, I);
    }
}

template <bool COUNTS, int Q>
__global__ void __launch_bounds__(kBlock)
    k_syn_push_scan(const float *__restrict__ z, int32_t B, int64_t n_cols, const int32_t *__restrict__ col_ptr,
                    const uint32_t *__restrict__ ps, const float *__restrict__ w, const float *__restrict__ basis,
                    int n_types, int nb, int32_t n_post, float *__restrict__ I) {
    extern __shared__ float basis_lds[];
    load_basis_lds(basis_lds, basis, n_types * nb);
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t n_words = (n_cols + kWave - 1) / kWave;
    const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x / kWave);
    const int64_t u0 = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWave) +
                       __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
    for (int64_t u = u0; u < n_words; u += waves) {
        const int64_t c = u * kWave + lane;
        uint32_t m = 0u;
        if (c < n_cols)
            for (int b = 0; b < B; ++b) m |= (z[b * n_cols + c] > 0.0f ? 1u : 0u) << b;
        uint64_t act = __ballot(m != 0u);
        while (act) {
            const int l = __builtin_ctzll(act);
            act &= act - 1ull;
            const uint32_t ml = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m), l));
            const int64_t cl = u * kWave + l;
            const int32_t lo = col_ptr[cl], hi = col_ptr[cl + 1];
            if (COUNTS) push_spiking<Q>(lane, lo, hi, ml, MultF32{z + cl, n_cols}, ps, w, basis_lds, nb, n_post, I);
            else push_spiking<Q>(lane, lo, hi, ml, MultOne{}, ps, w, basis_lds, nb, n_post, I);
        }
    }
}

// ---------------------------------------------------------------- backward ----
// G rows from dy [B][n_post][nb].  A workgroup takes P consecutive posts: it copies their dy
// into LDS (coalesced), then each thread writes row quarters (four batch entries of one G row,
// one 16-byte store; consecutive threads write consecutive quarters), padding entries b >= B
// written +0 (no separate fill).  Type-major rows: G[s * n_post + post][b] =
// sum_r dy[b][post][r] * basis[s][r]; a table's own compact rows (COMPACT): G[post * rows + q][b]
// with s = gtype[post][q], +0 past the post's types.  Each element sums r ascending from
// dy[0] * bs[0], one rounding per product and per add.
// The workgroups from g_blocks on zero the dense dW instead (grid-stride), which the
// weight-gradient pass after this launch writes for the active synapses.
template <bool COMPACT>
__global__ void __launch_bounds__(kBlock)
    k_make_G(const float *__restrict__ dy, int32_t B, int32_t n_post, int Bp, const float *__restrict__ basis,
             int n_types, int nb, const uint8_t *__restrict__ gtype, int rows, int P, float *__restrict__ G,
             int g_blocks, float *__restrict__ fill, int64_t n_fill) {
    if (static_cast<int>(blockIdx.x) >= g_blocks) {
        const int64_t stride = static_cast<int64_t>(gridDim.x - g_blocks) * blockDim.x;
        for (int64_t i = static_cast<int64_t>(blockIdx.x - g_blocks) * blockDim.x + threadIdx.x; i < n_fill;
             i += stride)
            fill[i] = 0.0f;
        return;
    }
    extern __shared__ float lds_f[];
    float *basis_lds = lds_f;
    float *tile = lds_f + ((n_types * nb + 3) & ~3);   // [B][P][nb]
    for (int i = threadIdx.x; i < n_types * nb; i += blockDim.x) basis_lds[i] = basis[i];
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * P;
    const int np = static_cast<int>(min(static_cast<int64_t>(P), n_post - n0));
    const int span = np * nb, total = B * span;
    for (int base = 0; base < total; base += 8 * static_cast<int>(blockDim.x)) {
        float v[8];   // the loads of a round go out together
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int i = base + k * static_cast<int>(blockDim.x) + static_cast<int>(threadIdx.x);
            const int b = i / span;
            v[k] = i < total ? dy[(static_cast<int64_t>(b) * n_post + n0) * nb + (i - b * span)] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int i = base + k * static_cast<int>(blockDim.x) + static_cast<int>(threadIdx.x);
            const int b = i / span;
            if (i < total) tile[b * P * nb + (i - b * span)] = v[k];
        }
    }
    __syncthreads();
    const int nrow = COMPACT ? rows : n_types;
    const int nq = Bp / 4;
    const int items = nrow * np * nq;
    for (int it = threadIdx.x; it < items; it += blockDim.x) {
        const int b0 = (it % nq) * 4;
        int p, s;
        int64_t row;
        if (COMPACT) {   // memory order: post, then rank, then quarter
            const int pq = it / nq;
            p = pq / rows;
            row = (n0 + p) * rows + (pq - p * rows);
            s = gtype[row];
        } else {         // type, then post, then quarter
            const int sp = it / nq;
            s = sp / np;
            p = sp - s * np;
            row = static_cast<int64_t>(s) * n_post + n0 + p;
        }
        float e[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (!COMPACT || s != 0xFF) {
            const float *bs = basis_lds + s * nb;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (b0 + j >= B) break;
                const float *d = tile + ((b0 + j) * P + p) * nb;
                float x = d[0] * bs[0];
#pragma unroll
                for (int r = 1; r < kMaxBasis; ++r)
                    if (r < nb) x = x + d[r] * bs[r];
                e[j] = x;
            }
        }
        *reinterpret_cast<float4 *>(G + row * Bp + b0) = make_float4(e[0], e[1], e[2], e[3]);
    }
}

// Posts per workgroup of k_make_G: the dy tile holds at most 2048 floats.
static int make_G_posts(int B, int nb) {
    int P = 64;
    while (P > 1 && B * P * nb > 2048) P >>= 1;
    return P;
}

// Batch masks and "active in some batch entry" bitmaps of a dense z [B][n_cols] in the
// row pull's layout: slot plane n_slots - d holds column pre + n_pre * (d - 1) at bit
// pre (planes of pre_pad = round64(n_pre) bits); one thread per (plane, pre), one wave per
// 64-bit word.
__global__ void __launch_bounds__(kBlock)
    k_op_colmask(const float *__restrict__ z, int32_t B, int64_t n_cols, int32_t n_pre, int32_t n_slots,
                 int32_t pre_pad, uint32_t *__restrict__ cm, uint64_t *__restrict__ bits) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<int64_t>(n_slots) * pre_pad) return;  // whole waves (pre_pad % 64 == 0)
    const int32_t plane = static_cast<int32_t>(i / pre_pad);
    const int32_t pre = static_cast<int32_t>(i - static_cast<int64_t>(plane) * pre_pad);
    uint32_t m = 0u;
    if (pre < n_pre) {
        const int64_t c = pre + static_cast<int64_t>(n_pre) * (n_slots - 1 - plane);
        for (int b = 0; b < B; ++b)
            if (z[static_cast<int64_t>(b) * n_cols + c] > 0.0f) m |= 1u << b;
    }
    cm[i] = m;
    const uint64_t bal = __ballot(m != 0u);
    if ((threadIdx.x & (kWave - 1)) == 0) bits[i >> 6] = bal;
}

template <int LG>
__global__ void __launch_bounds__(kBlock) k_syn_bwd_cols(ColArgs a, ActDense act) {
    bwd_cols<LG, 2>(a, act);
}

// dW of the active columns (z[b][c] > 0) next to the grouped dz walk: a wave per 64
// consecutive columns finds each column's batch mask, then 16-lane sub-groups walk the
// column-grouped synapses of four active columns at a time and write each synapse's dW
// once, straight to reference order: the sum over the set batch entries b, ascending, of
// G[sid][post][b] times the input value (counts) or 1 (spikes).
struct SynDwArgs {
    int64_t n_cols;
    int32_t B, hm, lm, R, counts;  // G row of entry p: (p >> 24) * hm + (p & kLow24) * lm
    const float *z;  // [B][n_cols]
    const int4 *units;  // the table's work units (Table::wide), one wave each
    int32_t n_units;
    const int32_t *col_ptr;
    const uint32_t *ps;
    const int32_t *order;
    const float *G;
    float *dw;  // reference order, zero-filled by the caller
};

// Workgroup bid of the pass: a wave per work unit -- up to 64 consecutive short columns (lane l
// tests column first + l), or one chunk of a long column, which the wave's four 16-lane
// sub-groups split in quarters, so a table of few long columns (the background's) still spreads
// over many waves.
__device__ inline void syn_dw_body(const SynDwArgs &a, int64_t bid) {
    const int lane = threadIdx.x % kWave;
    const int64_t ui = bid * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (ui >= a.n_units) return;  // the whole wave leaves together
    const int4 un = a.units[ui];
    const int64_t c0 = un.x;
    const bool chunk = un.y == 1;  // one column: its [un.z, un.w) in four quarters
    const int64_t c = c0 + (chunk ? 0 : lane);
    // a chunk's quarters are held by lanes 0, 16, 32, 48, so the loop below gives one to
    // each sub-group; otherwise lane l holds column c0 + l
    const bool mine = chunk ? (lane % 16) == 0 : lane < un.y;
    uint32_t m = 0;
    if (mine)
        for (int b = 0; b < a.B; ++b) m |= (a.z[b * a.n_cols + c] > 0.0f ? 1u : 0u) << b;
    int32_t lo = 0, hi = 0;
    if (m) {
        lo = chunk ? un.z : a.col_ptr[c];
        hi = chunk ? un.w : a.col_ptr[c + 1];
        if (chunk) {   // quarter lane / 16 of the chunk
            const int32_t q = (hi - lo + 3) / 4, s4 = lane / 16;
            lo = min(hi, lo + s4 * q);
            hi = min(hi, lo + q);
        }
    }
    const int sub = lane / 16, sl = lane % 16;
    uint64_t live = __ballot(m != 0u);
    while (live) {
        uint64_t lv = live;
        int src = -1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int f = lv ? __ffsll(static_cast<unsigned long long>(lv)) - 1 : -1;
            if (i == sub) src = f;
            lv &= lv - 1;
        }
        live = lv;
        // every lane takes part in the shuffles; idle sub-groups are masked afterwards
        const int sl_src = src >= 0 ? src : 0;
        const uint32_t msrc = static_cast<uint32_t>(__shfl(static_cast<int>(m), sl_src, kWave));
        const int32_t clo = __shfl(lo, sl_src, kWave);
        const int32_t hsrc = __shfl(hi, sl_src, kWave);
        const uint32_t mm = src >= 0 ? msrc : 0u;
        const int32_t chi = src >= 0 ? hsrc : clo;
        const int64_t cc = chunk ? c0 : c0 + sl_src;
        for (int32_t k0 = clo; k0 < chi; k0 += 64) {
            float d[4];
            const float *gp[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int32_t k = min(k0 + 16 * u + sl, chi - 1);
                const uint32_t p = a.ps[k];
                gp[u] = a.G + (static_cast<int64_t>(p >> 24) * a.hm + static_cast<int64_t>(p & kLow24) * a.lm) * a.R;
                d[u] = 0.0f;
            }
            uint32_t mb = mm;
            while (mb) {
                const int b = __ffs(mb) - 1;
                mb &= mb - 1;
                const float mult = a.counts ? a.z[b * a.n_cols + cc] : 1.0f;
#pragma unroll
                for (int u = 0; u < 4; ++u) d[u] += a.counts ? gp[u][b] * mult : gp[u][b];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (k0 + 16 * u + sl < chi) a.dw[a.order[k0 + 16 * u + sl]] = d[u];
        }
    }
}


// dz and dW over the same work units, for tables whose walk runs on few lanes or whose time a long
// column sets (the input tables).  A wave per unit; LG lanes hold one synapse's G row (4 floats each), so a
// row is one request of LG lanes and is read once for both gradients.  The wave's 64 / LG lane
// groups take the synapses of a one-column unit in turn, or share the columns of a run, a power of
// two of groups per column, in passes where the run has more columns than groups.  dz: each group's
// sums are added in a fixed butterfly order; a one-column unit's go to partial[unit], and k_dz_chunks
// adds a column's units in order.  dW of a column with any input: its synapses' sum over the batch
// entries of G[row][b] times the input value (counts) or 1, written once, straight to reference
// order.  What bounds it is the gathers' latency (kUnitRows rows in flight per lane group, and
// kUnitEntries synapses a wave for enough waves).  Whole backward calls, against a lane per
// synapse for dz, which held whole rows, and dW by a pass of its own, both over 1024-synapse
// units: background table, 66,000 posts, batch 32, 174 -> 63 us; LGN table at batch 5, 94 -> 58.
struct UnitArgs {
    int64_t n_cols;
    int32_t B, hm, lm, counts;  // G row of entry p: (p >> 24) * hm + (p & kLow24) * lm, 4 LG floats
    const float *z;       // [B][n_cols]
    const int4 *units;
    int32_t n_units;
    const int32_t *col_ptr;
    const uint32_t *ps;
    const float *w;       // column-grouped weights
    const int32_t *order;
    const float *G;
    float *dz;            // [B][n_cols], or nullptr
    float *partial;       // [n_units][4 LG]
    float *dw;            // reference order, zero-filled by the caller, or nullptr
};

constexpr int kUnitRows = 4;

template <int LG>
__global__ void __launch_bounds__(kBlock) k_syn_units(UnitArgs a) {
    constexpr int SG = kWave / LG, U = kUnitRows;
    const int lane = threadIdx.x % kWave, q = lane % LG, sg = lane / LG;
    const int64_t ui = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWave) +
                       __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
    if (ui >= a.n_units) return;  // the whole wave leaves together
    const int4 un = a.units[ui];
    int cp = 1;                   // columns of a pass: a power of two of the run's, at most SG
    while (cp < un.y && cp < SG) cp *= 2;
    const int n = SG / cp;        // lane groups per column
    for (int j0 = 0; j0 < un.y; j0 += cp) {
        const int j = j0 + sg / n;
        const bool own = j < un.y;
        const int64_t c = un.x + (own ? j : 0);
        int32_t k = 0, k_end = 0;
        if (own) {
            k = (un.y == 1 ? un.z : a.col_ptr[c]) + sg % n;
            k_end = un.y == 1 ? un.w : a.col_ptr[c + 1];
        }
        float zv[4];
        bool on[4], any = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int b = 4 * q + i;
            const float x = a.dw && own && b < a.B ? a.z[b * a.n_cols + c] : 0.0f;
            on[i] = x > 0.0f;
            zv[i] = a.counts ? x : 1.0f;
            any |= on[i];
        }
        const uint64_t bal = __ballot(any);
        const bool live = ((bal >> (sg * LG)) & ((1ull << LG) - 1ull)) != 0ull;   // the same in the group's lanes
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        // without dz only the active columns' synapses are read
        if (!a.dz && !live) k = k_end;
        for (; k < k_end; k += U * n) {
            uint32_t p[U];
            float wk[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int32_t kk = min(k + u * n, k_end - 1);
                p[u] = a.ps[kk];
                wk[u] = a.dz ? a.w[kk] : 0.0f;
            }
            float4 g[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                g[u] = reinterpret_cast<const float4 *>(a.G)[(static_cast<int64_t>(p[u] >> 24) * a.hm +
                                                              static_cast<int64_t>(p[u] & kLow24) * a.lm) * LG + q];
            if (a.dz) {
                // the rows' terms in pairs, then onto the sums: a quarter of the roundings at their size
                float4 x[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool in = k + u * n < k_end;
                    x[u].x = in ? wk[u] * g[u].x : 0.0f;
                    x[u].y = in ? wk[u] * g[u].y : 0.0f;
                    x[u].z = in ? wk[u] * g[u].z : 0.0f;
                    x[u].w = in ? wk[u] * g[u].w : 0.0f;
                }
                static_assert(U == 4, "two pairs");
                acc[0] = acc[0] + ((x[0].x + x[1].x) + (x[2].x + x[3].x));
                acc[1] = acc[1] + ((x[0].y + x[1].y) + (x[2].y + x[3].y));
                acc[2] = acc[2] + ((x[0].z + x[1].z) + (x[2].z + x[3].z));
                acc[3] = acc[3] + ((x[0].w + x[1].w) + (x[2].w + x[3].w));
            }
            if (live) {
                float d[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    d[u] = on[0] ? g[u].x * zv[0] : 0.0f;
                    d[u] = on[1] ? d[u] + g[u].y * zv[1] : d[u];
                    d[u] = on[2] ? d[u] + g[u].z * zv[2] : d[u];
                    d[u] = on[3] ? d[u] + g[u].w * zv[3] : d[u];
                }
#pragma unroll
                for (int o = 1; o < LG; o <<= 1)
#pragma unroll
                    for (int u = 0; u < U; ++u) d[u] = d[u] + __shfl_xor(d[u], o, kWave);
                if (q == 0) {
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (k + u * n < k_end) a.dw[a.order[k + u * n]] = d[u];
                }
            }
        }
        if (!a.dz) continue;
        for (int o = LG; o < n * LG; o <<= 1)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = acc[i] + __shfl_xor(acc[i], o, kWave);
        if (!own || sg % n) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int b = 4 * q + i;
            if (b >= a.B) continue;
            if (un.y == 1) a.partial[ui * (4 * LG) + b] = acc[i];
            else a.dz[b * a.n_cols + c] = acc[i];
        }
    }
}

// dz of the one-column units' columns: 2^sh lanes per (column, b) take the column's units in turn, four at
// a time in pairs (their sums are the largest, and every rounding at that size counts), and add theirs in
// a fixed order.  One lane's chain of loads was the backward's longest part over long columns: 100 columns of
// 40,000 synapses, batch 1, 54 -> 41 us a call with 32.
constexpr int kChunkUnits = 8;   // units per lane

__global__ void __launch_bounds__(kBlock)
    k_dz_chunks(const int4 *__restrict__ chunked, int32_t n_chunked, const float *__restrict__ partial, int32_t B,
                int32_t R, int64_t n_cols, int sh, float *__restrict__ dz) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> sh;
    const int L = 1 << sh, l = threadIdx.x & (L - 1);
    const bool own = i < static_cast<int64_t>(n_chunked) * B;
    const int4 d = own ? chunked[i / B] : make_int4(0, 0, 0, 0);
    const int b = static_cast<int>(i % B);
    const int64_t step = static_cast<int64_t>(R) << sh;
    const float *p = partial + static_cast<int64_t>(d.y + l) * R + b;
    float s = 0.0f;
    int u = l;
    for (; u + 3 * L < d.z; u += 4 * L, p += 4 * step) s = s + ((p[0] + p[step]) + (p[2 * step] + p[3 * step]));
    for (; u < d.z; u += L, p += step) s = s + p[0];
    for (int o = 1; o < L; o <<= 1) s = s + __shfl_xor(s, o, kWave);
    if (own && l == 0) dz[static_cast<int64_t>(b) * n_cols + d.x] = s;
}

// The grouped dz walk (the first walk_blocks workgroups) beside the weight-gradient pass of
// the active columns (the rest): both read G only, the walk is bound by its gathers' latency,
// and one launch overlaps them.
template <int LG, bool SPLIT>
__global__ void __launch_bounds__(kBlock) k_syn_bwd_gs(GsArgs a, ActDense act, int walk_blocks, SynDwArgs da) {
    __shared__ float stage[kBlock / kWave * kGsStage];
    if (static_cast<int>(blockIdx.x) < walk_blocks) bwd_groups<LG, SPLIT>(a, act, stage, blockIdx.x);
    else syn_dw_body(da, blockIdx.x - walk_blocks);
}

int sub_wave_for(const Table *t) {  // lanes per column: ~ the mean column length
    double avg = t->n_cols ? static_cast<double>(t->n_syn) / t->n_cols : 0.0;
    return avg <= 24.0 ? 16 : (avg <= 48.0 ? 32 : 64);
}

int grid_subwaves(int64_t items, int L) {
    int64_t per_block = kBlock / L;
    int64_t g = (items + per_block - 1) / per_block;
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(g, 32768)));
}

int batch_pad(int B) { return B <= 4 ? 4 : (B <= 8 ? 8 : (B <= 16 ? 16 : 32)); }

struct SynWs {
    uint32_t *cm;      // [n_slots * pre_pad] batch masks (deterministic forward)
    uint64_t *cbits;   // [n_slots * pre_pad / 64] activity bitmaps
    float *G;          // the custom gradient's projection
    float *partial;    // [units][padded B] the unit dz pass's one-column sums
};

// with_G: the backward's projection G too (the forward does not use it)
static SynWs carve_syn(void *ws, const Table *t, int32_t B, size_t *bytes, bool with_G = true) {
    Carver cv(ws, SIZE_MAX);
    SynWs w{};
    const int64_t pre_pad = (static_cast<int64_t>(t->n_pre) + 63) / 64 * 64;
    w.cm = cv.take<uint32_t>(static_cast<size_t>(t->n_slots) * pre_pad);
    w.cbits = cv.take<uint64_t>(static_cast<size_t>(t->n_slots) * pre_pad / 64);
    // G: a row per (type, post), or per (post, own type) with the table's compact rows
    const int rows = t->og.rows ? t->og.rows : t->n_types;
    if (with_G) {
        w.G = cv.take<float>(static_cast<size_t>(t->n_post) * rows * batch_pad(B));
        w.partial = cv.take<float>(std::max<size_t>(static_cast<size_t>(t->units.n) * batch_pad(B), 1));
    }
    if (bytes) *bytes = cv.off;
    return w;
}

// Whether the op forward pulls (deterministic mode, or event mode on a table with long
// columns: each active input would cost an atomic per synapse of its column and batch entry,
// and with the background's Poisson counts ~2.4 of them land on each (b, post, receptor) per
// call, 67 against 24 us pulled at B = 5), and whether that pull uses the workspace (batch
// masks and activity bits built from z; Poisson counts take the dense-row pull, which needs
// none).  glif_syn_fwd validates the workspace with the same predicate syn_fwd dispatches on.
// Poisson counts of a few inputs onto short rows pull in event mode whatever the columns' length: as background a fifth of
// them is active in every batch entry (12,007 posts, 100 inputs, batch 32: 157 us pushed, 12 pulled), and with next to none
// a short row costs no more than the push (3,000 posts, batch 5, 40 synapses each: 15 us, pushed 14 with 0.2 % active, 42 with
// 10 %; 150 each: 38 us, pushed 18 and 95).
static bool ell_counts(const Table *t) { return t->ell_len > 0 && t->n_cols <= kEllMaxInputs; }
static bool fwd_pulls(const Table *t, int32_t counts, int32_t mode) {
    return mode == GLIF_MODE_DETERMINISTIC || t->max_col_len > kUnitDzMinColLen || 
           (counts && ell_counts(t) && t->ell_len <= kEllEventMaxRow);
}
static bool fwd_uses_ws(const Table *t, int32_t counts, int32_t mode) { return fwd_pulls(t, counts, mode) && !counts; }

// The op forward on a carved workspace (every buffer it reads is written first by this call,
// so nothing in it has to start at zero).  Launches only; no allocation, no synchronisation.
static int syn_fwd(const Table *t, const float *z, int32_t B, int32_t counts, int32_t mode, float *I,
                   const SynWs &w, hipStream_t s) {
    const size_t lds = sizeof(float) * t->n_types * t->n_basis;
    const int64_t nI = static_cast<int64_t>(B) * t->n_post;
    // the pull's sums are the reference's, well within the event mode's bar
    if (fwd_pulls(t, counts, mode)) {
        if (fwd_uses_ws(t, counts, mode)) {
            // the row pulls over batch masks and activity bitmaps built from z (one step, t = 0):
            // the resident chunk form where it fits, else the half-wave row pull (B * nb > 64,
            // or bitmaps beyond LDS), which reads each entry once for all batch entries
            const int32_t pre_pad = static_cast<int32_t>((static_cast<int64_t>(t->n_pre) + 63) / 64 * 64);
            PullArgs pa{};
            pa.t = 0;
            pa.T = 1;
            pa.N = t->n_post;
            pa.Np = pre_pad;
            pa.B = B;
            pa.D = t->n_slots;
            pa.nb = t->n_basis;
            pa.n_types = t->n_types;
            pa.os_r = 1;
            pa.os_b = static_cast<int64_t>(t->n_post) * t->n_basis;
            pa.os_n = t->n_basis;
            pa.W = pre_pad / 64;
            pa.Wl = 0;
            pa.rec_chunks = t->chunk_desc ? t->n_chunks : 0;
            pa.rec_cdesc = t->chunk_desc;
            pa.rec_row = t->row_ptr;
            pa.rec_pd = t->pd;
            pa.rec_pidx = t->chunk_desc ? t->pidx : nullptr;   // no chunk form without both
            pa.rec_sid = t->sid_row;
            pa.rec_w = t->w_row;
            pa.zmask = w.cm;
            pa.abits = w.cbits;
            pa.lbits = w.cbits;
            pa.basis = t->basis;
            pa.I = I;
            const int64_t n_mask = static_cast<int64_t>(t->n_slots) * pre_pad;
            hipLaunchKernelGGL(k_op_colmask, dim3(ceil_div(n_mask, kBlock)), dim3(kBlock), 0, s, z, B, t->n_cols,
                               t->n_pre, t->n_slots, pre_pad, w.cm, w.cbits);
            GLIF_HIP(hipGetLastError());
            // a wave per row on tables whose rows average 64 entries or more (the op's output is
            // post-major)
            launch_pull(pa, lds, s, t->n_syn >= static_cast<int64_t>(kWave) * t->n_post);
            GLIF_HIP(hipGetLastError());
            return GLIF_OK;
        }
        if (ell_counts(t)) {
            int bb = 8;
            while (bb > 1 && (bb >= 2 * B || bb * t->n_cols > kEllMaxStage || t->n_post * static_cast<int64_t>(ceil_div(B, bb)) < kEllMinLanes)) bb /= 2;
            const size_t l = sizeof(float) * static_cast<size_t>(t->n_cols) * bb + lds;
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(ceil_div(t->n_post, kBlock), ceil_div(B, bb)), dim3(kBlock), l, s, z, B,
                                   static_cast<int32_t>(t->n_cols), t->n_post, t->row_ptr, t->ell_pw, t->basis, t->n_types,
                                   t->n_basis, I);
            };
            if (bb == 8) launch(k_syn_pull_ell<8>);
            else if (bb == 4) launch(k_syn_pull_ell<4>);
            else if (bb == 2) launch(k_syn_pull_ell<2>);
            else launch(k_syn_pull_ell<1>);
            GLIF_HIP(hipGetLastError());
            return GLIF_OK;
        }
        // Poisson counts scale the weights: a thread per (b, post) over the post's row
        dim3 grid(ceil_div(nI, kBlock));
        hipLaunchKernelGGL(k_syn_pull_dense, grid, dim3(kBlock), lds, s, z, B, t->n_cols, t->n_post,
                           t->n_pre, t->row_ptr, t->pd, t->sid_row, t->w_row, t->basis, t->n_types, t->n_basis, I);
        GLIF_HIP(hipGetLastError());
        return GLIF_OK;
    }
    int rc = launch_fill_u32(I, 0u, static_cast<size_t>(nI) * t->n_basis, s);
    if (rc) return rc;
    const int Q = t->basis_nnz < 2 * t->n_types ? 1 : t->n_basis <= 4 ? 4 : 8;   // lanes per synapse
    const Units &un = t->n_syn < kPushWideMinSyn ? t->units : t->wide;
    if (un.n > 0 && (ceil_div(t->n_cols, kWave) < kPushUnitsMaxScanWaves || t->max_col_len > kPushUnitsMinColLen)) {
        const dim3 grid(static_cast<unsigned>(ceil_div(un.n, kBlock / kWave)));
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(kBlock), lds, s, z, B, t->n_cols, un.unit, un.n, t->col_ptr,
                               t->ps, t->w_col, t->basis, t->n_types, t->n_basis, t->n_post, I);
        };
        if (Q == 1) counts ? launch(k_syn_push_units<true, 1>) : launch(k_syn_push_units<false, 1>);
        else if (Q == 4) counts ? launch(k_syn_push_units<true, 4>) : launch(k_syn_push_units<false, 4>);
        else counts ? launch(k_syn_push_units<true, 8>) : launch(k_syn_push_units<false, 8>);
        GLIF_HIP(hipGetLastError());
        return GLIF_OK;
    }
    const dim3 grid(static_cast<unsigned>(std::max<int64_t>(
        1, std::min<int64_t>(ceil_div(ceil_div(t->n_cols, kWave), kBlock / kWave), 32768))));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kBlock), lds, s, z, B, t->n_cols, t->col_ptr, t->ps, t->w_col, t->basis,
                           t->n_types, t->n_basis, t->n_post, I);
    };
    if (Q == 1) counts ? launch(k_syn_push_scan<true, 1>) : launch(k_syn_push_scan<false, 1>);
    else if (Q == 4) counts ? launch(k_syn_push_scan<true, 4>) : launch(k_syn_push_scan<false, 4>);
    else counts ? launch(k_syn_push_scan<true, 8>) : launch(k_syn_push_scan<false, 8>);
    GLIF_HIP(hipGetLastError());
    return GLIF_OK;
}

constexpr int kMaxDevices = 64;

}  // namespace glif

// Scratch of glif_syn_fwd_noalloc: a file-scope device array, so the entry point needs no
// allocation.  Every GPU the library runs on holds its own copy until the process ends.  In host
// code this name is only a handle for hipGetSymbolAddress, never a device address.
static __device__ __align__(256) char scratch[GLIF_NOALLOC_SCRATCH_BYTES];

namespace glif {

static std::mutex g_scratch_mu;
static void *g_scratch_dev[kMaxDevices];

// The device address of `scratch` on the current device, looked up once per device.
static int scratch_on_current_device(void **out) {
    int dev = -1;
    GLIF_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(GLIF_EINVAL, "device index beyond the library's table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (!p) return fail(GLIF_EHIP, "hipGetSymbolAddress(scratch) returned NULL");
        g_scratch_dev[dev] = p;
    }
    *out = g_scratch_dev[dev];
    return GLIF_OK;
}

}  // namespace glif

using namespace glif;

extern "C" {

size_t glif_syn_workspace(const glif_table *tt, int32_t B) {
    if (!tt || B <= 0) return 0;
    size_t bytes = 0;
    carve_syn(nullptr, reinterpret_cast<const Table *>(tt), B, &bytes);
    return bytes;
}

int glif_syn_fwd(const glif_table *tt, const float *z, int32_t B, int32_t counts, int32_t mode,
                 float *I, void *ws, size_t ws_bytes, void *stream) {
    if (!tt || !z || !I) return fail(GLIF_EINVAL, "NULL argument");
    if (B <= 0 || B > kMaxBatch) return fail(GLIF_EINVAL, "B must be in [1, 32]");
    if (mode != GLIF_MODE_EVENT && mode != GLIF_MODE_DETERMINISTIC) return fail(GLIF_EINVAL, "unknown mode");
    const Table *t = reinterpret_cast<const Table *>(tt);
    hipStream_t s = static_cast<hipStream_t>(stream);
    // the row pulls of spikes use the workspace (batch masks and activity bits); the event
    // push and the dense-row pull of counts need none
    if (fwd_uses_ws(t, counts, mode) && (!ws || ws_bytes < glif_syn_workspace(tt, B)))
        return fail(GLIF_ENOMEM, "workspace too small");
    ProfScope prof(kProfSynFwd, s);
    return syn_fwd(t, z, B, counts, mode, I, carve_syn(ws, t, B, nullptr), s);
}

int glif_syn_fwd_noalloc(const glif_table *tt, const float *z, int32_t B, int32_t counts, int32_t mode, float *I,
                         void *stream) {
    if (!tt || !z || !I) return fail(GLIF_EINVAL, "NULL argument");
    if (B <= 0 || B > kMaxBatch) return fail(GLIF_EINVAL, "B must be in [1, 32]");
    if (mode != GLIF_MODE_EVENT && mode != GLIF_MODE_DETERMINISTIC) return fail(GLIF_EINVAL, "unknown mode");
    const Table *t = reinterpret_cast<const Table *>(tt);
    size_t need = 0;
    carve_syn(nullptr, t, B, &need, false);
    if (need > GLIF_NOALLOC_SCRATCH_BYTES)
        return fail(GLIF_ENOMEM, "glif_syn_fwd_noalloc: this table's forward at batch " + std::to_string(B) +
                                     " needs " + std::to_string(need) + " bytes of scratch, above the " +
                                     std::to_string(GLIF_NOALLOC_SCRATCH_BYTES) +
                                     "-byte static array; call glif_syn_fwd with a workspace instead");
    void *p = nullptr;
    const int rc = scratch_on_current_device(&p);
    if (rc) return rc;
    return syn_fwd(t, z, B, counts, mode, I, carve_syn(p, t, B, nullptr, false), static_cast<hipStream_t>(stream));
}

int glif_syn_bwd(const glif_table *tt, const float *z, const float *dy, int32_t B, int32_t counts,
                 float *dz, float *dw, void *ws, size_t ws_bytes, void *stream) {
    if (!tt || !z || !dy) return fail(GLIF_EINVAL, "NULL argument");
    if (B <= 0 || B > kMaxBatch) return fail(GLIF_EINVAL, "B must be in [1, 32]");
    if (!dz && !dw) return GLIF_OK;
    const Table *t = reinterpret_cast<const Table *>(tt);
    size_t need = glif_syn_workspace(tt, B);
    if (!ws || ws_bytes < need) return fail(GLIF_ENOMEM, "workspace too small");
    const SynWs w = carve_syn(ws, t, B, nullptr);
    return syn_bwd_run(t, z, dy, B, counts, dz, dw, w.G, false, w.partial, static_cast<hipStream_t>(stream));
}

}  // extern "C"

namespace glif {

size_t syn_g_floats(const Table *t, int32_t B) {
    const int rows = t->og.rows ? t->og.rows : t->n_types;
    return static_cast<size_t>(t->n_post) * rows * batch_pad(B);
}

bool same_g_layout(const Table *a, const Table *b) {
    return a->og.rows == 0 && b->og.rows == 0 && a->n_post == b->n_post && a->n_types == b->n_types &&
           a->n_basis == b->n_basis &&
           std::memcmp(a->basis_host, b->basis_host, sizeof(float) * a->n_types * a->n_basis) == 0;
}

static void launch_syn_units(const UnitArgs &a, int Bp, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(ceil_div(a.n_units, kBlock / kWave)));
    switch (Bp / 4) {
        case 1: hipLaunchKernelGGL(k_syn_units<1>, grid, dim3(kBlock), 0, s, a); break;
        case 2: hipLaunchKernelGGL(k_syn_units<2>, grid, dim3(kBlock), 0, s, a); break;
        case 4: hipLaunchKernelGGL(k_syn_units<4>, grid, dim3(kBlock), 0, s, a); break;
        default: hipLaunchKernelGGL(k_syn_units<8>, grid, dim3(kBlock), 0, s, a); break;
    }
}

int syn_bwd_run(const Table *t, const float *z, const float *dy, int32_t B, int32_t counts, float *dz, float *dw,
                float *G, bool g_ready, float *partial, hipStream_t s) {
    if (!dz && !dw) return GLIF_OK;
    const int Bp = batch_pad(B);
    // the table's own compact rows (post * rows + rank) when it has them, else type-major rows
    const CompactRows &oc = t->og;
    const bool cmp = oc.rows > 0;
    const int rows = cmp ? oc.rows : t->n_types;
    if (static_cast<int64_t>(rows) * t->n_post * Bp * 4 >= (int64_t(1) << 32))
        return fail(GLIF_ERANGE, "G rows per post * n_post * padded batch * 4 bytes must be < 4 GiB");
    ProfScope prof(kProfSynBwd, s);
    int rc;
    const bool grouped = (cmp ? oc.n_gs : t->n_gs) > 0;
    // the work units instead of a walk whose time the longest column sets (the background
    // table's few, long columns) or that runs on few lanes (the LGN table's 17,400 columns):
    // for dz when the caller gives their partial sums room, and for dW, whose grouped-path
    // pass always runs over them
    const int64_t walk_lanes = (grouped ? t->n_groups : t->n_cols) * (Bp / 4);
    const bool prefer_units =
        t->units.n > 0 && (t->max_col_len > kUnitDzMinColLen ||
                         (walk_lanes < kUnitDzMaxWalkLanes && (Bp <= 8 || t->n_syn >= kUnitDzMinAvgLen * t->n_cols)));
    const bool dz_units = dz && partial && prefer_units;
    const bool dw_units = dw && (grouped || prefer_units);
    // G, with the zero fill of dW beside it when the units' weight-gradient pass writes only
    // the active synapses
    const int gP = make_G_posts(B, t->n_basis);
    const int g_blocks = g_ready ? 0 : static_cast<int>(ceil_div(static_cast<int64_t>(t->n_post), gP));
    const int fill_blocks = dw_units && t->n_syn ? 256 : 0;
    const int64_t n_fill = fill_blocks ? t->n_syn : 0;
    const dim3 g_grid(g_blocks + fill_blocks);
    const size_t g_lds = sizeof(float) * (((t->n_types * t->n_basis + 3) & ~3) + static_cast<size_t>(B) * gP * t->n_basis);
    if (g_grid.x == 0) {
        // no posts and nothing to fill
    } else if (cmp) {
        hipLaunchKernelGGL(k_make_G<true>, g_grid, dim3(kBlock), g_lds, s, dy, B, t->n_post, Bp, t->basis,
                           t->n_types, t->n_basis, oc.gtype, rows, gP, G, g_blocks, dw, n_fill);
    } else {
        hipLaunchKernelGGL(k_make_G<false>, g_grid, dim3(kBlock), g_lds, s, dy, B, t->n_post, Bp, t->basis,
                           t->n_types, t->n_basis, nullptr, rows, gP, G, g_blocks, dw, n_fill);
    }
    GLIF_HIP(hipGetLastError());
    // (dW alone by the same kernel as beside dz: the same bits)
    if (dz_units || (dw && prefer_units)) {
        const bool wide = dz_units && !dw && t->n_syn >= std::max(kWideDzMinSyn, kWideDzMinAvgLen * t->n_cols);
        const Units &un = wide ? t->wide : t->units;
        const UnitArgs ua{t->n_cols, B, cmp ? 1 : t->n_post, cmp ? rows : 1, counts, z, un.unit, un.n, t->col_ptr,
                          cmp ? oc.ps : t->ps, t->w_col, t->order, G, dz_units ? dz : nullptr, partial, dw};
        launch_syn_units(ua, Bp, s);
        GLIF_HIP(hipGetLastError());
        if (dz_units && un.n_chunked > 0) {
            int sh = 0;
            while (sh < 6 && kChunkUnits << sh < un.most) ++sh;
            hipLaunchKernelGGL(k_dz_chunks, dim3(static_cast<unsigned>(ceil_div(static_cast<int64_t>(un.n_chunked) * B << sh, kBlock))),
                               dim3(kBlock), 0, s, un.chunked, un.n_chunked, partial, B, Bp, t->n_cols, sh, dz);
            GLIF_HIP(hipGetLastError());
        }
        // done; what is left is a dz that found no room for the partial sums
        dw = nullptr;
        if (dz_units || !dz) return GLIF_OK;
    }
    if (grouped) {
        // the grouped row-sliced walk for dz (when grouped and dz is still wanted) beside the
        // active columns' dW over the units (every active synapse's written once, in reference
        // order)
        ActDense act{z, dz, t->n_cols, counts};
        GsArgs ga{t->n_cols, (t->n_cols + kGsCols - 1) / kGsCols, B, cmp ? oc.gs_seg : t->gs_seg,
                  cmp ? oc.gs_pw : t->gs_pw, G};
        ga.split = gs_split(ga.n_groups, Bp / 4);
        SynDwArgs da{t->n_cols, B, cmp ? 1 : t->n_post, cmp ? rows : 1, Bp, counts, z, t->wide.unit, t->wide.n,
                     t->col_ptr, cmp ? oc.ps : t->ps, t->order, G, dw};
        const int LG = Bp / 4;
        const int walk_blocks = dz ? static_cast<int>(ceil_div(t->n_groups * LG << ga.split, kBlock)) : 0;
        const int dw_blocks = dw ? static_cast<int>(ceil_div(t->wide.n, kBlock / kWave)) : 0;
        const dim3 grid(walk_blocks + dw_blocks);
        if (grid.x == 0) return GLIF_OK;   // no columns
        auto launch = [&](auto whole, auto split) {
            if (ga.split) hipLaunchKernelGGL(split, grid, dim3(kBlock), 0, s, ga, act, walk_blocks, da);
            else hipLaunchKernelGGL(whole, grid, dim3(kBlock), 0, s, ga, act, walk_blocks, da);
        };
        switch (LG) {
            case 1: launch(k_syn_bwd_gs<1, false>, k_syn_bwd_gs<1, true>); break;
            case 2: launch(k_syn_bwd_gs<2, false>, k_syn_bwd_gs<2, true>); break;
            case 4: launch(k_syn_bwd_gs<4, false>, k_syn_bwd_gs<4, true>); break;
            default: launch(k_syn_bwd_gs<8, false>, k_syn_bwd_gs<8, true>); break;
        }
        GLIF_HIP(hipGetLastError());
        return GLIF_OK;
    }
    // the type-phased column walk writes the active columns' synapses; the rest stay 0
    if (dw && (rc = launch_fill_u32(dw, 0u, static_cast<size_t>(t->n_syn), s))) return rc;
    ColArgs ca{t->n_cols, t->n_post, t->n_types, B, t->ph_ptr, cmp ? oc.ph_pw : t->ph_pw, G, dz ? 1 : 0, dw,
               t->ph_order, cmp ? 1 : 0};
    ActDense act{z, dz, t->n_cols, counts};
    const dim3 grid(ceil_div(t->n_cols * (Bp / 4), kBlock));
    switch (Bp / 4) {
        case 1: hipLaunchKernelGGL(k_syn_bwd_cols<1>, grid, dim3(kBlock), 0, s, ca, act); break;
        case 2: hipLaunchKernelGGL(k_syn_bwd_cols<2>, grid, dim3(kBlock), 0, s, ca, act); break;
        case 4: hipLaunchKernelGGL(k_syn_bwd_cols<4>, grid, dim3(kBlock), 0, s, ca, act); break;
        default: hipLaunchKernelGGL(k_syn_bwd_cols<8>, grid, dim3(kBlock), 0, s, ca, act); break;
    }
    GLIF_HIP(hipGetLastError());
    return GLIF_OK;
}

}  // namespace glif
