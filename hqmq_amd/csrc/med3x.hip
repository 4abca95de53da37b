// Med3x outlier statistics and sideband compaction.
//
// hqmq_med3x_threshold follows the torch.quantile half of
// OutlierAwareHQMQQuantizer._qdq (src/quantizers/outlier_aware.py:60-69 of the
// reference): per head, the median over every chunk norm of the call (fp32
// interpolation between the two middle order statistics), times the
// multiplier, rounded to D.  The order statistics are exact: chunk norms are
// non-negative, so their bit patterns sort like the values.  Calls of a 16-bit
// type with 65 to 16384 chunks per head take one block per head and a histogram of
// its whole key in LDS (one launch); at most 64 chunks, and fp32 up to 8192, keep the
// keys in registers and search the key bit by bit (one launch); larger 16-bit calls
// take such a histogram per block, which the selection adds up where it looks (two
// launches); larger fp32, calls too large for 16-bit counters and workspaces too small for that take
// one histogram per head of the top 16 bits, and fp32 a second pass over the low 16
// bits of the bin(s) holding the two ranks.  K and V of one append share the launches.
//
// hqmq_outlier_compact has no counterpart in the reference: it copies the
// flagged chunks into the fp16/bf16/fp32 sideband in (token, chunk) order.
//
// Compiled with -ffp-contract=off.
#include "med_select.h"

namespace hqmq {

constexpr int kBins2 = 65536;
constexpr int kState = 16;  // ints per head
// workspace (uint32 units): hist1[H][kBins1] | state[H][kState] | (fp32 only) hist2[H][2][kBins2], or, of a 16-bit type, a part per
// block (med_select.h)
// state: 0 nan count, 1 key_lo, 2 key_hi, 3 rank_lo within bin, 4 rank_hi within bin
__host__ __device__ inline int64_t ws_words(int H, bool f32) {
    return (int64_t)H * (kBins1 + kState) + (f32 ? (int64_t)H * 2 * kBins2 : 0);
}
inline int64_t ws_words_parts(int H) { return (int64_t)(H > kPartBlocks ? H : kPartBlocks) * kPartWords; }

// One tensor of a call, as the kernels see it; a launch takes one or two of equal shape (blockIdx.z).
struct MedTensor {
    const void *x;
    int64_t xsb, xsh, xst;
    int vec;                    // chunks may be read with one vector load
    float mult;
    uint32_t *ws;
    float *median;
    void *thr;
    int32_t *n_out;
};
struct MedPair {
    MedTensor t[2];
    int B, H, T, n;
};
__device__ __forceinline__ uint32_t *med_hist(const MedTensor &m, int h) { return m.ws + (size_t)h * kBins1; }
__device__ __forceinline__ uint32_t *med_state(const MedTensor &m, int H, int h) { return m.ws + (size_t)H * kBins1 + (size_t)h * kState; }
__device__ __forceinline__ uint32_t *med_hist2(const MedTensor &m, int H, int h) { return m.ws + (size_t)H * (kBins1 + kState) + (size_t)h * 2 * kBins2; }

__global__ void fill_zero_kernel(uint32_t *p, uint32_t *q, int64_t n) {
    uint32_t *w = blockIdx.y ? q : p;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) w[i] = 0;
}

template <class D>
__device__ __forceinline__ float chunk_norm(const typename D::storage *xp) {
    return chunk_norm_d<D>(D::load(xp), D::load(xp + 1), D::load(xp + 2), D::load(xp + 3));
}

// f(norm) for the chunks of rows [r0, r1) of head h (row = b * T + t), one chunk per lane of a block of NT threads and
// step, U loads in flight per lane.  The rows of a lane lie NT / n apart: no division per chunk.
// meanwhile(): what every thread does, once, while the first chunks travel (it may wait for the block).
template <class D, int NT, int U, class F, class M>
__device__ __forceinline__ void for_each_norm(const MedTensor &m, const MedPair &a, int h, int64_t r0, int64_t r1, F f, M meanwhile) {
    using ST = typename D::storage;
    const int n = a.n, per = n <= NT ? NT / n : 1, rl = n <= NT ? (int)threadIdx.x / n : 0;
    const int dq = per / a.T, dt = per - dq * a.T;                   // `per` rows on: dq sequences and dt tokens
    const int64_t step = dq * m.xsb + dt * m.xst, wrap = m.xsb - a.T * m.xst, b0 = (r0 + rl) / a.T;
    const int t0 = (int)(r0 + rl - b0 * a.T);
    const ST *p0 = (const ST *)m.x + b0 * m.xsb + h * m.xsh + (int64_t)t0 * m.xst, *p;
    int c = (int)threadIdx.x - rl * n, t = t0, k;
    int64_t r = r0 + rl;
    bool more = rl < per && r < r1;
    RawChunk<D> raw[U];
    auto request = [&]() {
        k = 0;
#pragma unroll
        for (int i = 0; i < U; i++) {
            if (r < r1) {
                raw[i].load(p, m.vec);
                k = i + 1;
            }
            r += per;
            t += dt;
            p += step;
            if (t >= a.T) { t -= a.T; p += wrap; }
        }
    };
    p = p0 + c * 4;
    if (more) request();
    meanwhile();
    while (more) {
#pragma unroll
        for (int i = 0; i < U; i++)
            if (i < k) f(chunk_norm_d<D>(raw[i].get(0), raw[i].get(1), raw[i].get(2), raw[i].get(3)));
        if (r >= r1) {
            c += NT;                                                 // one round, unless a row has more chunks than the block lanes
            if (c >= n) break;
            r = r0;                                                  // (rl is 0 then)
            t = t0;
            p = p0 + c * 4;
        }
        request();
    }
}

// fp32, very large calls and small workspaces: a histogram of the top 16 bits per head.  The 32768 bins live in LDS, and a block adds only its
// non-zero bins (some 3000 of an ordinary tensor) to the global histogram.  Blocks of at most 65535 chunks pack two 16-bit
// counters in a word: 64 KB, two blocks per CU and half the bins to clear and to look through.  The groups' sums are collected in LDS first: all blocks of a head add to the same dozen words,
// and with an atomic per 64 bins those additions, one after the other, were most of the kernel (8 heads x 32768 tokens fp16:
// 54 us instead of 33).
template <class D, bool WIDE>
__global__ __launch_bounds__(1024) void med_hist_kernel(MedPair a, int64_t rows_per_block) {
    extern __shared__ uint32_t lh[];    // [words] | sums of the groups | NaN count
    constexpr int words = WIDE ? kBins1 : kBins1 / 2, sums = words, nans = words + kGroups;
    const MedTensor &m = a.t[blockIdx.z];
    const int h = blockIdx.y;
    for (int i = threadIdx.x; i < words / 4; i += 1024) reinterpret_cast<uint4 *>(lh)[i] = uint4{0, 0, 0, 0};
    if (threadIdx.x <= kGroups) lh[sums + threadIdx.x] = 0;
    __syncthreads();
    const int64_t rows = (int64_t)a.B * a.T, r0 = blockIdx.x * rows_per_block;
    for_each_norm<D, 1024, 4>(m, a, h, r0, min(rows, r0 + rows_per_block), [&](float nrm) {
        const uint32_t key = norm_bits<D>(nrm) >> 16;
        if (is_nan(nrm)) atomicAdd(&lh[nans], 1u);
        else if (WIDE) atomicAdd(&lh[key], 1u);
        else atomicAdd(&lh[key >> 1], 1u << (16 * (key & 1)));
    }, [] {});
    __syncthreads();
    uint32_t *hist1 = med_hist(m, h);
    for (int i = threadIdx.x; i < words; i += 1024) {                    // the 64 words of a wavefront lie in one group
        const uint32_t v = lh[i];
        uint32_t sum;
        if (WIDE) {
            if (v) atomicAdd(&hist1[i], v);
            sum = v;
        } else {
            if (v & 0xffffu) atomicAdd(&hist1[2 * i], v & 0xffffu);
            if (v >> 16) atomicAdd(&hist1[2 * i + 1], v >> 16);
            sum = (v & 0xffffu) + (v >> 16);
        }
        if (__builtin_amdgcn_ballot_w64(sum != 0u) == 0ull) continue;
        sum = wave_sum(sum);
        if ((threadIdx.x & 63) == 0) atomicAdd(&lh[sums + (WIDE ? i : 2 * i) / kGroupBins], sum);
    }
    __syncthreads();
    if (threadIdx.x < kGroups && lh[sums + threadIdx.x]) atomicAdd(&hist1[kGroupAt + threadIdx.x], lh[sums + threadIdx.x]);
    if (threadIdx.x == 0 && lh[nans]) atomicAdd(&med_state(m, a.H, h)[0], lh[nans]);
}

// fp32, second pass: low 16 bits of the norms whose top bits are a selected bin
__global__ __launch_bounds__(1024) void med_hist_low_kernel(MedPair a, int64_t rows_per_block) {
    const MedTensor &m = a.t[blockIdx.z];
    const int h = blockIdx.y;
    const uint32_t *state = med_state(m, a.H, h);
    const uint32_t key_lo = state[1], key_hi = state[2];
    uint32_t *hist2 = med_hist2(m, a.H, h);
    const int64_t rows = (int64_t)a.B * a.T, r0 = blockIdx.x * rows_per_block;
    for_each_norm<F32, 1024, 4>(m, a, h, r0, min(rows, r0 + rows_per_block), [&](float nrm) {
        const uint32_t bits = __float_as_uint(nrm);
        if ((bits >> 16) == key_lo) atomicAdd(&hist2[bits & 0xffffu], 1u);
        else if ((bits >> 16) == key_hi) atomicAdd(&hist2[kBins2 + (bits & 0xffffu)], 1u);
    }, [] {});
}

// Finds the bins holding 0-based ranks r[0] <= r[1] in a histogram of PER * 1024 counters (a block of 1024 threads).
// Wavefront w owns bins w * PER * 64 .., read as PER coalesced rows of 64 into registers; the wavefront whose range
// holds a rank walks its rows, then the lanes of the row.  (Every thread summing PER consecutive counters and walking
// them again one dependent load at a time took 20 us a launch.)  counts: the thread's counters, row by row.
template <int PER>
__device__ __forceinline__ void select_two(const uint32_t *hist, const int64_t (&r)[2], uint32_t (&counts)[PER], uint32_t (&key)[2], int64_t (&inner)[2]) {
    __shared__ unsigned long long tot[16];
    __shared__ uint32_t res[2];
    __shared__ long long resr[2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < PER; i++) counts[i] = hist[(wave * PER + i) * 64 + lane];
    unsigned long long s = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) s += counts[i];
    for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
    if (lane == 0) tot[wave] = s;
    if (threadIdx.x < 2) { res[threadIdx.x] = (uint32_t)(PER * 1024 - 1); resr[threadIdx.x] = 0; }
    __syncthreads();
    unsigned long long before = 0;
    for (int w = 0; w < wave; w++) before += tot[w];
    for (int which = 0; which < 2; which++) {
        const unsigned long long want = (unsigned long long)r[which];
        if (want < before || want >= before + s) continue;           // wave-uniform
        unsigned long long at = before;
        bool found = false;
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const uint32_t row = wave_sum(counts[i]);                // a row holds fewer than 2^32 chunks
            if (!found && want < at + row) {
                found = true;
                uint32_t incl = counts[i];
                for (int o = 1; o < 64; o <<= 1) {
                    const uint32_t v = __shfl_up(incl, o, 64);
                    if (lane >= o) incl += v;
                }
                const uint32_t rest = (uint32_t)(want - at), excl = incl - counts[i];
                if (rest >= excl && rest < incl) {
                    res[which] = (uint32_t)((wave * PER + i) * 64 + lane);
                    resr[which] = (long long)(rest - excl);
                }
            }
            at += row;
        }
    }
    __syncthreads();
    for (int which = 0; which < 2; which++) { key[which] = res[which]; inner[which] = resr[which]; }
}

// 16-bit types, first of two launches: every block counts the keys of its rows (at most 65535 chunks) in 32768 bins in LDS,
// two 16-bit counters a word, and stores the groups of bins that hold any, and the sums of all groups, in a part of the
// workspace that is its own: nothing to clear beforehand and no atomics behind.  A wavefront's 16-byte reads take one group
// at a time, so its sum is there when the words are, in registers, to be stored.  8 heads fp16, this launch and the selection:
// 2048 tokens 17.7 -> 12.0 us, 32768 tokens 60 -> 23.5 (18.0 for this launch: 3.7 TB/s); with bins added to one histogram per
// head by atomics, cleared by a launch of its own, the additions of the blocks to the same words took longer than the counting.
// The bins are cleared while the first chunks travel: cleared before they were requested, 4 x 4001 tokens bf16 s24_r3 appended took 99.1 us
// (98.0), K and V of 2048 tokens fake-quantized 40.2 (39.7), of 4 x 4000 with heads of 64 62.0 (61.1), of 3 x 2500 bf16 63.4 (62.1).
template <class D>
__global__ __launch_bounds__(1024) void med_hist16_kernel(MedPair a, int64_t rows_per_block) {
    extern __shared__ uint32_t lh[];    // [kBins1 / 2] | NaN count
    constexpr int words = kBins1 / 2;
    const MedTensor &m = a.t[blockIdx.z];
    const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t rows = (int64_t)a.B * a.T, r0 = blockIdx.x * rows_per_block;
    for_each_norm<D, 1024, 4>(m, a, h, r0, min(rows, r0 + rows_per_block), [&](float nrm) {
        const uint32_t key = norm_bits<D>(nrm) >> 16;
        if (is_nan(nrm)) atomicAdd(&lh[words], 1u);
        else atomicAdd(&lh[key >> 1], 1u << (16 * (key & 1)));
    }, [&] {
        for (int i = tid; i < words / 4; i += 1024) reinterpret_cast<uint4 *>(lh)[i] = uint4{0, 0, 0, 0};
        if (tid == 0) lh[words] = 0;
        __syncthreads();
    });
    __syncthreads();
    uint32_t *part = m.ws + (size_t)(h * gridDim.x + blockIdx.x) * kPartWords;
    static_assert(kGroupBins / 2 == 4 * 64, "a group is one 16-byte read of a wavefront");
#pragma unroll
    for (int group = wave; group < kGroups; group += 16) {
        const uint4 v = reinterpret_cast<const uint4 *>(lh)[group * 64 + lane];
        auto both = [](uint32_t w) { return (w & 0xffffu) + (w >> 16); };
        const uint32_t sum = wave_sum(both(v.x) + both(v.y) + both(v.z) + both(v.w));
        if (sum) reinterpret_cast<uint4 *>(part)[group * 64 + lane] = v;
        if (lane == 0) part[kPartSums + group] = sum;
    }
    if (tid == 0) part[kPartNan] = lh[words];
}

// Second launch, one block per head
template <class D>
__global__ __launch_bounds__(1024) void med_select16_kernel(MedPair a, int parts) {
    const MedTensor &m = a.t[blockIdx.z];
    __shared__ __align__(8) uint32_t sh[kSelectWords];
    select16<D>(MedSelect{m.ws, m.median, m.thr, m.n_out, m.mult, parts, (uint32_t)((int64_t)a.B * a.T * a.n)}, blockIdx.x, true, sh, [] {});
}

// One wavefront per rank: the group that holds it (64 sums), then the bin inside the group (8 bins per lane).
template <class D>
__global__ __launch_bounds__(128) void med_select_kernel(MedPair a) {
    const MedTensor &m = a.t[blockIdx.z];
    const int h = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t per_head = (uint32_t)((int64_t)a.B * a.T * a.n);
    uint32_t *state = med_state(m, a.H, h);
    const uint32_t *hist = med_hist(m, h);
    const uint32_t sum = hist[kGroupAt + lane];
    if (state[0] > 0) {
        if (threadIdx.x == 0) {
            nan_threshold<D>(m.median, m.thr, m.n_out, h);
            state[1] = 0xffffffffu; state[2] = 0xffffffffu;
        }
        return;
    }
    auto before = [&](uint32_t v) {                      // exclusive prefix sum over the wavefront
        uint32_t incl = v;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t u = __shfl_up(incl, o, 64);
            if (lane >= o) incl += u;
        }
        return incl - v;
    };
    auto bins = [&](int group, uint32_t (&v)[8]) {       // the lane's 8 bins of a group; the sums' own places count nothing
        const uint4 *p = reinterpret_cast<const uint4 *>(hist + group * kGroupBins + lane * 8);
        const uint4 x = p[0], y = p[1];
        const bool real = group * kGroupBins + lane * 8 < kGroupAt;
        const uint32_t w[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = real ? w[i] : 0u;
    };
    __shared__ uint32_t key_sh[2], in_sh[2];
    const uint32_t rank = wave == 0 ? (per_head - 1) / 2 : per_head / 2;
    {
        const uint32_t at = before(sum);
        const uint64_t mine = __builtin_amdgcn_ballot_w64(rank >= at && rank < at + sum);
        const int group = mine ? __builtin_ctzll(mine) : kGroups - 1;
        uint32_t v[8], tot = 0;
        bins(group, v);
        uint32_t rest = rank - __shfl(at, group);
#pragma unroll
        for (int i = 0; i < 8; i++) tot += v[i];
        const uint32_t first = before(tot);
        if (rest >= first && rest < first + tot) {
            rest -= first;
            int i = 0;
#pragma unroll
            for (int k = 0; k < 7; k++)
                if (i == k && rest >= v[k]) { rest -= v[k]; i = k + 1; }
            key_sh[wave] = (uint32_t)(group * kGroupBins + lane * 8 + i);
            in_sh[wave] = rest;
        }
    }
    __syncthreads();
    if (D::code == HQMQ_F32) {
        if (threadIdx.x == 0) { state[1] = key_sh[0]; state[2] = key_sh[1]; state[3] = in_sh[0]; state[4] = in_sh[1]; }
        return;
    }
    if (wave != 0) return;
    const bool same = (per_head - 1) / 2 == per_head / 2;
    const float lo = key_value<D>(key_sh[0]), hi = key_value<D>(key_sh[1]);
    const float tv = D::rnd((same ? lo : hi - (hi - lo) * 0.5f) * m.mult);
    if (lane == 0) finish_threshold<D>(lo, hi, same, m.mult, h, m.median, (typename D::storage *)m.thr);
    if (!m.n_out) return;
    // chunks with norm > thr: whole groups above the one that holds the threshold, and the bins above it in there.  (A
    // threshold below every norm or beyond infinity: group 0 or none.)
    const uint32_t thr_key = norm_bits<D>(fmaxf(tv, 0.f)) >> 16;
    const int group = (int)min(thr_key / kGroupBins, (uint32_t)kGroups - 1u);
    uint32_t v[8], n = lane > group ? sum : 0u;
    bins(group, v);
#pragma unroll
    for (int i = 0; i < 8; i++)
        if (key_value<D>((uint32_t)(group * kGroupBins + lane * 8 + i)) > tv) n += v[i];
    n = wave_sum(n);
    if (lane == 0) m.n_out[h] = (int32_t)n;
}

// fp32: the low halves of the two keys
__global__ __launch_bounds__(1024) void med_select_low_kernel(MedPair a) {
    const MedTensor &m = a.t[blockIdx.z];
    const int h = blockIdx.x;
    const int64_t per_head = (int64_t)a.B * a.T * a.n;
    uint32_t *state = med_state(m, a.H, h);
    const uint32_t *hist2 = med_hist2(m, a.H, h);
    if (state[0] > 0) return;
    const uint32_t klo = state[1], khi = state[2];
    constexpr int PER = kBins2 / 1024;
    uint32_t counts[PER], low[2], up[2];
    int64_t inner[2];
    const int64_t r[2] = {state[3], klo == khi ? state[4] : state[3]};
    select_two<PER>(hist2, r, counts, low, inner);
    if (klo != khi) {
        __syncthreads();
        const int64_t r2[2] = {state[4], state[4]};
        select_two<PER>(hist2 + kBins2, r2, counts, up, inner);
        low[1] = up[1];
    }
    if (threadIdx.x == 0) {
        const float x = __uint_as_float((klo << 16) | low[0]), y = __uint_as_float((khi << 16) | low[1]);
        finish_threshold<F32>(x, y, (per_head - 1) / 2 == per_head / 2, m.mult, h, m.median, (float *)m.thr);
        if (m.n_out) m.n_out[h] = 0;
    }
}

__global__ __launch_bounds__(1024) void count_gt_kernel(MedPair a, int64_t rows_per_block) {
    const MedTensor &m = a.t[blockIdx.z];
    const int h = blockIdx.y;
    if (!m.n_out) return;
    const float tv = ((const float *)m.thr)[h];
    uint32_t cnt = 0;
    const int64_t rows = (int64_t)a.B * a.T, r0 = blockIdx.x * rows_per_block;
    for_each_norm<F32, 1024, 4>(m, a, h, r0, min(rows, r0 + rows_per_block), [&](float nrm) { cnt += nrm > tv ? 1u : 0u; }, [] {});
    cnt = wave_sum(cnt);
    if ((threadIdx.x & 63) == 0 && cnt) atomicAdd(&m.n_out[h], (int)cnt);
}

// Small calls (a decode step appends B * n chunks per head), fp32, or of at most 64 chunks: norms, exact order statistics and count in one launch, one
// block per head, up to eight keys per lane in registers.  The key of rank r is the largest v with fewer than r + 1 keys below
// it, found bit by bit from the top: a compare and a scalar bit count per key, one barrier per round (none in a block of
// one wavefront); two bits, three thresholds a round.  The second rank is the next one: the same key again, or the smallest key above it.
// (256-bin histograms of keys in LDS, two passes per rank, took 9.5 us for 2048 chunks per head.)
template <class D, int NT, int KEYS>
__global__ __launch_bounds__(NT) void med_small_kernel(MedPair a) {
    constexpr int W = NT / 64, BITS = D::code == HQMQ_F32 ? 31 : 15;
    __shared__ uint4 sums[W > 1 ? BITS / 2 + 4 : 1];
    const MedTensor &m = a.t[blockIdx.z];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int per_head = a.B * a.T * a.n, rows = a.B * a.T;
    using ST = typename D::storage;
    if (W > 1) {
        if (tid < BITS / 2 + 4) sums[tid] = uint4{0, 0, 0, 0};
        __syncthreads();
    }
    // lane (rl, c) holds chunk c of rows rl, rl + per, ..: one division per lane, not one per key
    const int per = NT / a.n, rl = tid / a.n, c = tid - rl * a.n;
    uint32_t key[KEYS];
    bool nan = false, have[KEYS];
    {
        RawChunk<D> raw[KEYS] = {};
        const int b0 = rl / a.T;
        int r = rl < per ? rl : rows, t = rl - b0 * a.T;
        const ST *p = (const ST *)m.x + b0 * m.xsb + h * m.xsh + (int64_t)t * m.xst + c * 4;
        const int dq = per / a.T, dt = per - dq * a.T;               // `per` rows on: dq sequences and dt tokens
        const int64_t step = dq * m.xsb + dt * m.xst, wrap = m.xsb - a.T * m.xst;
#pragma unroll
        for (int i = 0; i < KEYS; i++) {
            have[i] = r < rows;
            if (have[i]) raw[i].load(p, m.vec);
            r += per;
            t += dt;
            p += step;
            if (t >= a.T) { t -= a.T; p += wrap; }
        }
#pragma unroll
        for (int i = 0; i < KEYS; i++) {
            const float nrm = chunk_norm_d<D>(raw[i].get(0), raw[i].get(1), raw[i].get(2), raw[i].get(3));
            nan |= have[i] && is_nan(nrm);
            key[i] = have[i] ? (D::code == HQMQ_F32 ? __float_as_uint(nrm) : norm_bits<D>(nrm) >> 16) : 0x7fffffffu;    // absent: above every key
        }
    }
    // Sums over the block of up to three wave-uniform numbers: one LDS atomic each per wavefront into the round's own
    // counters, one broadcast read back (sixteen wavefronts reading sixteen partial sums each took 1.7 us a round).
    int round = 0;
    auto total3 = [&](uint32_t &x, uint32_t &y, uint32_t &z) {
        if (W == 1) return;
        if (lane == 0) {
            atomicAdd(&sums[round].x, x);
            atomicAdd(&sums[round].y, y);
            atomicAdd(&sums[round].z, z);
        }
        __syncthreads();
        const uint4 s = sums[round++];
        x = s.x; y = s.y; z = s.z;
    };
    const uint32_t r_lo = (uint32_t)((per_head - 1) / 2), r_hi = (uint32_t)(per_head / 2);
    uint32_t k_lo = 0, any_nan = __builtin_amdgcn_ballot_w64(nan) != 0ull ? 1u : 0u;
#pragma unroll 1
    for (int bit = BITS - 1; bit >= 0; bit -= 2) {       // two bits a round (the last has one: its three thresholds coincide)
        const uint32_t v1 = k_lo | 1u << (bit - (bit ? 1 : 0)), v2 = k_lo | 1u << bit, v3 = v2 | v1;
        uint32_t c1 = 0, c2 = 0, c3 = 0;
#pragma unroll
        for (int i = 0; i < KEYS; i++) {
            c1 += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(key[i] < v1));
            c2 += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(key[i] < v2));
            c3 += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(key[i] < v3));
        }
        total3(c1, c2, c3);
        k_lo = c3 <= r_lo ? v3 : c2 <= r_lo ? v2 : c1 <= r_lo ? v1 : k_lo;
    }
    // how many keys are at most k_lo, and the smallest one above it (complemented: a sum's place serves a maximum as well)
    uint32_t upto = 0, above = 0;
#pragma unroll
    for (int i = 0; i < KEYS; i++) {
        upto += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(key[i] <= k_lo));
        above = max(above, key[i] > k_lo ? ~key[i] : 0u);
    }
    above = group_max(above, 64, [](uint32_t p, uint32_t q) { return max(p, q); });
    if (W > 1) {
        if (lane == 0) {
            atomicAdd(&sums[round].x, upto);
            atomicMax(&sums[round].y, above);
            atomicAdd(&sums[round].z, any_nan);
        }
        __syncthreads();
        upto = sums[round].x; above = sums[round].y; any_nan = sums[round].z;
        round++;
    }
    if (any_nan) {
        if (tid == 0) nan_threshold<D>(m.median, m.thr, m.n_out, h);
        return;
    }
    const uint32_t k_hi = upto > r_hi ? k_lo : ~above;
    auto value = [](uint32_t k) { return D::code == HQMQ_F32 ? __uint_as_float(k) : key_value<D>(k); };
    const float x = value(k_lo), y = value(k_hi);
    const float med = r_lo == r_hi ? x : y - (y - x) * 0.5f;
    const float tv = D::rnd(med * m.mult);
    if (m.n_out) {
        uint32_t c = 0;
#pragma unroll
        for (int i = 0; i < KEYS; i++)
            c += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(have[i] && value(key[i]) > tv));
        uint32_t y = 0, z = 0;
        total3(c, y, z);
        if (tid == 0) m.n_out[h] = (int32_t)c;
    }
    if (tid == 0) finish_threshold<D>(x, y, r_lo == r_hi, m.mult, h, m.median, (ST *)m.thr);
}

// 16-bit calls of 65 to 16384 chunks per head: one block per head and a histogram of the 15-bit keys in LDS, 16-bit counters two to a
// word, instead of a search bit by bit (a barrier, 24 compares and three LDS atomics per wavefront for every two bits).  A wavefront
// owns 2048 neighbouring keys, a lane four words of each quarter of them (reads of 16 bytes side by side): a sum per quarter, the
// wavefronts' sums through LDS, then the wavefront that holds a rank finds its quarter, lane and key.  Ranks, NaN rule and count as in
// med_small_kernel.  Clearing, four barriers and code that arrives cold bound it, so the code is no longer than its keys per lane ask
// for; us replayed in a graph, 8 heads fp16, against the search: 512 chunks 5.3 -> 4.8, 1024 7.2 -> 4.9, 2048 7.6 -> 5.5, 4096 7.3 -> 6.1, 8192
// 7.4; against two launches over histograms of blocks: 16384 10.4 -> 10.0, one launch saved.  Up to 64 chunks the search is one wavefront
// without a barrier: 2.7 against 4.7.
constexpr int kLdsBins = 32768;
template <class D, int KEYS>
__global__ __launch_bounds__(1024) void med_lds_kernel(MedPair a) {
    constexpr int NT = 1024;
    extern __shared__ uint4 bins[];                 // kLdsBins / 8 of them, then the wavefronts' sums and the results
    uint32_t *const words = reinterpret_cast<uint32_t *>(bins), *const sums = words + kLdsBins / 2, *const res = sums + 16;
    const MedTensor &m = a.t[blockIdx.z];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per_head = a.B * a.T * a.n, rows = a.B * a.T;
    using ST = typename D::storage;
    const int per = NT / a.n, rl = tid / a.n, c = tid - rl * a.n;
    RawChunk<D> raw[KEYS] = {};
    bool have[KEYS];
    {
        const int b0 = rl / a.T;
        int r = rl < per ? rl : rows, t = rl - b0 * a.T;
        const ST *p = (const ST *)m.x + b0 * m.xsb + h * m.xsh + (int64_t)t * m.xst + c * 4;
        const int dq = per / a.T, dt = per - dq * a.T;
        const int64_t step = dq * m.xsb + dt * m.xst, wrap = m.xsb - a.T * m.xst;
#pragma unroll
        for (int i = 0; i < KEYS; i++) {
            have[i] = r < rows;
            if (have[i]) raw[i].load(p, m.vec);
            r += per;
            t += dt;
            p += step;
            if (t >= a.T) { t -= a.T; p += wrap; }
        }
    }
#pragma unroll
    for (int i = 0; i < kLdsBins / 8 / NT; i++) bins[tid + i * NT] = uint4{0, 0, 0, 0};
    if (tid < 4) res[tid] = 0;                      // low key, high key, NaN seen, count
    __syncthreads();
    uint32_t key[KEYS];
    bool nan = false;
#pragma unroll
    for (int i = 0; i < KEYS; i++) {
        const float nrm = chunk_norm_d<D>(raw[i].get(0), raw[i].get(1), raw[i].get(2), raw[i].get(3));
        nan |= have[i] && is_nan(nrm);
        key[i] = (norm_bits<D>(nrm) >> 16) & 0x7fffu;
        if (have[i]) atomicAdd(&words[key[i] >> 1], 1u << (16 * (key[i] & 1)));
    }
    if (__builtin_amdgcn_ballot_w64(nan) != 0ull && lane == 0) res[2] = 1;
    __syncthreads();
    if (res[2]) {
        if (tid == 0) nan_threshold<D>(m.median, m.thr, m.n_out, h);
        return;
    }
    uint4 own[4];
    uint32_t quarter[4], mine = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        own[i] = bins[wave * 256 + i * 64 + lane];
        const uint32_t s = own[i].x + own[i].y, t = own[i].z + own[i].w;      // at most 8192 in each half: no carry between them
        quarter[i] = (s & 0xffffu) + (s >> 16) + (t & 0xffffu) + (t >> 16);
        mine += quarter[i];
    }
    const uint32_t total = wave_sum(mine);
    if (lane == 0) sums[wave] = total;
    __syncthreads();
    uint32_t before = 0;
    for (int w = 0; w < 16; w++) {
        const uint32_t s = sums[w];
        before += w < wave ? s : 0u;
    }
    const uint32_t ranks[2] = {(uint32_t)((per_head - 1) / 2), (uint32_t)(per_head / 2)};
#pragma unroll
    for (int k = 0; k < 2; k++) {
        if (ranks[k] < before || ranks[k] >= before + total) continue;        // wave-uniform
        uint32_t left = ranks[k] - before;
        bool found = false;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t sum = wave_sum(quarter[i]);
            if (!found && left < sum) {
                found = true;
                const uint32_t lo = lanes_before(quarter[i]), up = lo + quarter[i];
                if (left >= lo && left < up) {
                    const uint32_t w4[4] = {own[i].x, own[i].y, own[i].z, own[i].w};
                    uint32_t at = left - lo, key16 = 0;
                    bool hit = false;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const uint32_t n = (w4[j >> 1] >> (16 * (j & 1))) & 0xffffu;
                        if (!hit && at < n) { hit = true; key16 = (uint32_t)j; }
                        if (!hit) at -= n;
                    }
                    res[k] = (uint32_t)((wave * 256 + i * 64 + lane) * 8) + key16;
                }
            } else if (!found) {
                left -= sum;
            }
        }
    }
    __syncthreads();
    const float x = key_value<D>(res[0]), y = key_value<D>(res[1]);
    const bool same = ranks[0] == ranks[1];
    if (m.n_out) {
        const float med = same ? x : y - (y - x) * 0.5f, tv = D::rnd(med * m.mult);
        uint32_t above = 0;
#pragma unroll
        for (int i = 0; i < KEYS; i++) above += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(have[i] && key_value<D>(key[i]) > tv));
        if (lane == 0) atomicAdd(&res[3], above);
        __syncthreads();
        if (tid == 0) m.n_out[h] = (int32_t)res[3];
    }
    if (tid == 0) finish_threshold<D>(x, y, same, m.mult, h, m.median, (ST *)m.thr);
}

// The flag bits of a row (up to 256 chunks) in registers; dwords where the row's address allows it.
__device__ __forceinline__ int row_flags(const uint8_t *fr, int frb, bool words, uint64_t (&own)[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) own[i] = 0;
    if (words && frb == 4) own[0] = *reinterpret_cast<const uint32_t *>(fr);
    else if (words && frb == 8) own[0] = *reinterpret_cast<const uint32_t *>(fr) | (uint64_t)reinterpret_cast<const uint32_t *>(fr)[1] << 32;
    else if (words && frb == 2) own[0] = *reinterpret_cast<const uint16_t *>(fr);
    else {
#pragma unroll
        for (int by = 0; by < 32; by++)
            if (by < frb) own[by >> 3] |= (uint64_t)fr[by] << (8 * (by & 7));
    }
    return __popcll(own[0]) + __popcll(own[1]) + __popcll(own[2]) + __popcll(own[3]);
}
// rows of `frb` flag bytes start at multiples of their width (2) or of 4
__host__ __device__ inline bool flag_words(const uint8_t *plane, int frb) { return !((uintptr_t)plane & 3) && (frb == 2 || !(frb & 3)); }

// Copies the flagged chunks of one row to sideband slots k, k + 1, ...
template <class D>
__device__ __forceinline__ void copy_row(const CompactCall &a, size_t bh, int64_t row, const typename D::storage *xr, const uint64_t (&own)[4], int k,
                                         bool vec) {
    using ST = typename D::storage;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        for (uint64_t bits = own[q]; bits; bits &= bits - 1) {
            const int c = 64 * q + __builtin_ctzll(bits);
            if (c >= a.n) break;
            if (k < a.sb_cap) {
                RawChunk<D> raw;
                raw.load(xr + c * 4, vec);
                raw.store((ST *)a.sideband + (bh * a.sb_cap + k) * 4, vec);
                if (a.sb_coord) a.sb_coord[bh * a.sb_cap + k] = (uint16_t)(((row & (kTile - 1)) << 8) | c);
            } else {
                *a.overflow = 1;
                degrade_to_plain<D>(a, bh * a.t_cap + row, c, xr + c * 4);
            }
            k++;
        }
    }
}
struct CompactPair {
    CompactCall c[2];           // blockIdx.z picks one; equal shapes
    int vec[2];                 // chunks of x and of the sideband may be moved by one vector access
};

// Exclusive prefix sum over the block (NT threads), and its total.
template <int NT>
__device__ __forceinline__ int block_scan(int v, int *part, int &total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int incl = (int)lanes_before((uint32_t)v) + v;
    if (NT == 64) {
        total = __shfl(incl, 63);
        return incl - v;
    }
    __syncthreads();
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    int before = 0;
    total = 0;
    for (int w = 0; w < NT / 64; w++) {
        if (w < wave) before += part[w];
        total += part[w];
    }
    return before + incl - v;
}

// One block of NT threads per (b, h): walks the T new rows in order, NT rows per step (one wavefront for short
// appends: its barriers cost nothing).
template <class D, int NT>
__global__ __launch_bounds__(NT) void compact_kernel(CompactPair pair) {
    using ST = typename D::storage;
    const CompactCall &a = pair.c[blockIdx.z];
    __shared__ int part[NT / 64];
    const int bh = blockIdx.x, b = bh / a.H, h = bh - b * a.H;
    const int frb = (a.n + 7) >> 3;
    const bool words = flag_words(a.flag_plane, frb);
    const int64_t row0 = (a.pos ? a.pos[b] : 0) + a.t_off;
    const int64_t tiles = (a.t_cap + kTile - 1) / kTile;
    int base = a.sb_count[bh];
    for (int t0 = 0; t0 < a.T; t0 += NT) {
        const int t = t0 + threadIdx.x;
        const int64_t row = row0 + t;
        const bool live = t < a.T && row >= 0 && row < a.t_cap;
        uint64_t own[4] = {0, 0, 0, 0};          // the row's flags as they are now (bits may be cleared below)
        const int cnt = live ? row_flags(a.flag_plane + ((size_t)bh * a.t_cap + row) * frb, frb, words, own) : 0;
        int total;
        const int before = base + block_scan<NT>(cnt, part, total);
        if (live) {
            if ((row & (kTile - 1)) == 0) a.sb_tile_off[(size_t)bh * tiles + (row >> 4)] = before;
            copy_row<D>(a, bh, row, (const ST *)a.x + b * a.xsb + h * a.xsh + (int64_t)t * a.xst, own, before, pair.vec[blockIdx.z]);
        }
        base += total;
    }
    __syncthreads();                             // every wavefront has read the count
    if (threadIdx.x == 0) a.sb_count[bh] = base;
}

// ---- bulk appends (whole 16-row tiles from an aligned first row): two passes with one thread per tile / row ----
// Pass 1, one block per (b, h): flagged chunks of every new tile, exclusive scan behind the chunks already stored.
__global__ __launch_bounds__(1024) void tile_scan_kernel(CompactPair pair) {
    const CompactCall &a = pair.c[blockIdx.z];
    __shared__ int part[16];
    const int bh = blockIdx.x, frb = (a.n + 7) >> 3, row0 = a.t_off;
    const int64_t tiles = (a.t_cap + kTile - 1) / kTile;
    const int n_tiles = (a.T + kTile - 1) / kTile;
    int32_t *to = a.sb_tile_off + (size_t)bh * tiles + (row0 >> 4);
    const uint8_t *fr = a.flag_plane + ((size_t)bh * a.t_cap + row0) * frb;
    const bool vec = !((uintptr_t)fr & 15);      // a tile is 16 frb bytes: whole 16-byte words, then, at 16-byte addresses
    int base = a.sb_count[bh];
    for (int i0 = 0; i0 < n_tiles; i0 += 1024) {
        const int i = i0 + threadIdx.x;
        int cnt = 0;
        if (i < n_tiles) {
            const int rows = min(a.T - i * kTile, kTile);
            const uint8_t *f = fr + (size_t)i * kTile * frb;
            if (vec && rows == kTile) {
                for (int w = 0; w < frb; w++) {
                    const uint4 v = reinterpret_cast<const uint4 *>(f)[w];
                    cnt += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
                }
            } else {
                for (int k = 0; k < rows * frb; k++) cnt += __popc((uint32_t)f[k]);
            }
        }
        int total;
        const int before = block_scan<1024>(cnt, part, total);
        if (i < n_tiles) to[i] = base + before;
        base += total;
    }
    __syncthreads();                             // every wavefront has read the count
    if (threadIdx.x == 0) a.sb_count[bh] = base;
}
// Pass 2: one thread per new row (the 16 rows of a tile are 16 neighbouring lanes) copies the row's flagged chunks behind
// those of the tile's earlier rows.  (4 x 8 x 4001 rows, one tensor: 8.5 + 4.8 us for counting and scanning apart, and
// 10 us for the copy with every row reading the flags of the tile's earlier rows again.)
template <class D>
__global__ __launch_bounds__(256) void tile_copy_kernel(CompactPair pair) {
    using ST = typename D::storage;
    const CompactCall &a = pair.c[blockIdx.z];
    const int bh = blockIdx.y, b = bh / a.H, h = bh - b * a.H;
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int frb = (a.n + 7) >> 3, row = a.t_off + t;
    const int64_t tiles = (a.t_cap + kTile - 1) / kTile;
    uint64_t own[4] = {0, 0, 0, 0};              // the row's flags, read before any row of the tile clears bits
    const int cnt = t < a.T ? row_flags(a.flag_plane + ((size_t)bh * a.t_cap + row) * frb, frb, flag_words(a.flag_plane, frb), own) : 0;
    int before = cnt;
    for (int o = 1; o < kTile; o <<= 1) {
        const int v = __shfl_up(before, o, kTile);
        if ((threadIdx.x & (kTile - 1)) >= o) before += v;
    }
    before -= cnt;
    if (!cnt) return;
    copy_row<D>(a, bh, row, (const ST *)a.x + b * a.xsb + h * a.xsh + (int64_t)t * a.xst, own, a.sb_tile_off[(size_t)bh * tiles + (row >> 4)] + before,
                pair.vec[blockIdx.z]);
}

// ---- cropping: rows from `len` on are forgotten ----
// A thread per tile resets the offsets of the tiles that hold no kept row, the block clears their flags in 16-byte words.
// The block that holds the tile of the cut works the new entry count out first: the tile's offset plus the flags of its
// kept rows (the count as it was, where the tile was never written or the offsets disagree).
constexpr int kCropTiles = 256;
__global__ __launch_bounds__(kCropTiles) void crop_kernel(hqmq_crop_args a) {
    const int z = blockIdx.z, bh = blockIdx.y, b = bh / a.H, frb = (a.n_chunks + 7) >> 3;
    const int64_t tiles = (a.t_cap + kTile - 1) / kTile, first = (int64_t)blockIdx.x * kCropTiles;
    const int64_t len = max(a.lengths ? a.lengths[b] : a.length, 0);
    const int64_t cut = len / kTile, free_tile = (len + kTile - 1) / kTile;
    if (first + kCropTiles <= cut || len >= a.t_cap) return;           // every row of the block is kept
    int32_t *off = a.sb_tile_off[z] + bh * tiles;
    uint8_t *flags = a.flag_plane[z] + (size_t)bh * a.t_cap * frb;
    if (cut >= first && threadIdx.x == 0) {
        const int at = off[cut], count = a.sb_count[z][bh];
        if (at <= count) {
            int kept = 0;
            for (int i = 0; i < (int)(len - cut * kTile) * frb; i++) kept += __popc((uint32_t)flags[cut * kTile * frb + i]);
            a.sb_count[z][bh] = min(at + kept, count);
        }
    }
    __syncthreads();
    const int64_t tile = first + threadIdx.x;
    if (tile >= free_tile && tile < tiles) off[tile] = 0x7fffffff;
    const int64_t lo = max(len, first * kTile) * frb, hi = min(a.t_cap, (first + kCropTiles) * kTile) * frb;      // bytes to clear
    uint8_t *p = flags + lo;
    const int64_t bytes = hi - lo, head = min(bytes, (int64_t)((16 - ((uintptr_t)p & 15)) & 15)), words = (bytes - head) / 16;
    for (int64_t i = threadIdx.x; i < head; i += kCropTiles) p[i] = 0;
    for (int64_t i = threadIdx.x; i < words; i += kCropTiles) reinterpret_cast<uint4 *>(p + head)[i] = uint4{0, 0, 0, 0};
    for (int64_t i = head + words * 16 + threadIdx.x; i < bytes; i += kCropTiles) p[i] = 0;
}

}  // namespace hqmq

using namespace hqmq;

extern "C" int64_t hqmq_med3x_workspace_bytes(int H, int dtype) {
    if (H < 1) return 0;
    return ws_words(H, dtype == HQMQ_F32) * 4;
}

extern "C" int64_t hqmq_med3x_workspace_best_bytes(int H, int dtype) {
    if (H < 1) return 0;
    const int64_t least = ws_words(H, dtype == HQMQ_F32) * 4, parts = dtype == HQMQ_F32 ? 0 : ws_words_parts(H) * 4;
    return parts > least ? parts : least;
}

template <class D>
static int run_med3x(const MedPair &a, int count, bool parts, MedSelect *later, hipStream_t st) {
    const bool f32 = D::code == HQMQ_F32;
    const int64_t per_head = (int64_t)a.B * a.T * a.n, rows = (int64_t)a.B * a.T;
    // Few keys per lane: such a call lasts about as long as its code takes to arrive (every launch starts
    // with cold instruction caches), and the code is written out once per key.
    auto fits = [&](int nt, int keys) { return a.n <= nt && rows <= (int64_t)(nt / a.n) * keys; };
    const dim3 heads(a.H, 1, count);
    if (fits(64, 1)) {
        hipLaunchKernelGGL((med_small_kernel<D, 64, 1>), heads, dim3(64), 0, st, a);
        return hip_status(hipGetLastError());
    }
    if constexpr (D::code == HQMQ_F32) {
        if (fits(1024, 8)) {
            auto kern = fits(256, 2) ? med_small_kernel<D, 256, 2> : fits(1024, 2) ? med_small_kernel<D, 1024, 2> : med_small_kernel<D, 1024, 8>;
            hipLaunchKernelGGL(kern, heads, dim3(fits(256, 2) ? 256 : 1024), 0, st, a);
            return hip_status(hipGetLastError());
        }
    } else if (fits(1024, 16)) {        // beyond, a block per head is slower than two launches (19200 chunks 15.3 against 10.5 us)
        auto kern = fits(1024, 1) ? med_lds_kernel<D, 1> : fits(1024, 2) ? med_lds_kernel<D, 2> : fits(1024, 4) ? med_lds_kernel<D, 4>
                  : fits(1024, 8) ? med_lds_kernel<D, 8> : med_lds_kernel<D, 16>;
        const size_t lds = (kLdsBins / 2 + 20) * sizeof(uint32_t);
        const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        hipLaunchKernelGGL(kern, heads, dim3(1024), lds, st, a);
        return hip_status(hipGetLastError());
    }
    // Blocks of about 4096 chunks (of 2048 / 4096 / 8192, us, whole calls with the quantize launch selecting: 2 x 1501 tokens, 28 / 4 heads, bf16
    // s192_r6 appended 51.5 / 48.9 / 49.4, 700 of bf16 s24_r3 fake-quantized 30.2 / 30.8 / 33.4) while that leaves at most two per CU; larger calls get larger blocks, beyond 65535 chunks
    // with 32-bit counters, one block per CU and tensor.
    const int rps = a.n <= 1024 ? 1024 / a.n : 1;        // rows a block takes per step
    auto blocks_of = [&](int64_t most, int64_t &rpb) {
        int64_t blocks = (per_head + 4095) / 4096;
        most = most > 0 ? most : 1;
        if (blocks > most) blocks = most;
        rpb = (rows + blocks - 1) / blocks;
        rpb = (rpb + rps - 1) / rps * rps;
        return (rows + rpb - 1) / rpb;
    };
    int64_t rpb, blocks;
    if constexpr (D::code != HQMQ_F32) {
        blocks = blocks_of(kPartBlocks / a.H, rpb);
        if (parts && rpb * a.n <= 65535) {
            const size_t lds = ((size_t)kBins1 / 2 + 1) * sizeof(uint32_t);
            const hipError_t e = hipFuncSetAttribute((const void *)med_hist16_kernel<D>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return (int)e;
            hipLaunchKernelGGL(med_hist16_kernel<D>, dim3((unsigned)blocks, a.H, count), dim3(1024), lds, st, a, rpb);
            if (later && blocks <= kSelectParts)
                for (int i = 0; i < count; i++)
                    later[i] = MedSelect{a.t[i].ws, a.t[i].median, a.t[i].thr, a.t[i].n_out, a.t[i].mult, (int)blocks, (uint32_t)per_head};
            else hipLaunchKernelGGL(med_select16_kernel<D>, dim3(a.H, 1, count), dim3(1024), 0, st, a, (int)blocks);
            return hip_status(hipGetLastError());
        }
    }
    const int64_t words = ws_words(a.H, f32);
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)(words / 1024 < 1024 ? (words + 1023) / 1024 : 1024), count), dim3(256), 0, st, a.t[0].ws,
                       a.t[count - 1].ws, words);
    blocks = blocks_of(512 / ((int64_t)a.H * count), rpb);
    bool wide = rpb * a.n > 60000;
    if (wide) {
        blocks = 256 / ((int64_t)a.H * count) > 0 ? 256 / ((int64_t)a.H * count) : 1;
        if (blocks < 16) blocks = 16;
        rpb = (rows + blocks - 1) / blocks;
        rpb = (rpb + rps - 1) / rps * rps;
        blocks = (rows + rpb - 1) / rpb;
        wide = rpb * a.n > 65535;
    }
    const dim3 grid((unsigned)blocks, a.H, count);
    auto kern = wide ? med_hist_kernel<D, true> : med_hist_kernel<D, false>;
    const size_t lds = ((size_t)(wide ? kBins1 : kBins1 / 2) + kGroups + 1) * sizeof(uint32_t);
    const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(kern, grid, dim3(1024), lds, st, a, rpb);
    hipLaunchKernelGGL(med_select_kernel<D>, dim3(a.H, 1, count), dim3(128), 0, st, a);
    if (f32) {
        hipLaunchKernelGGL(med_hist_low_kernel, grid, dim3(1024), 0, st, a, rpb);
        hipLaunchKernelGGL(med_select_low_kernel, dim3(a.H, 1, count), dim3(1024), 0, st, a);
        hipLaunchKernelGGL(count_gt_kernel, grid, dim3(1024), 0, st, a, rpb);
    }
    return hip_status(hipGetLastError());
}

static int check_med3x(const Med3xCall &c) {
    if (!c.x || !c.ws || !c.median || !c.thr) return HQMQ_ERR_NULL;
    if (c.B < 1 || c.H < 1 || c.H > 65535 || c.T < 1 || c.n < 1) return HQMQ_ERR_SHAPE;
    if (c.dtype != HQMQ_F32 && c.dtype != HQMQ_F16 && c.dtype != HQMQ_BF16) return HQMQ_ERR_DTYPE;
    if (c.ws_bytes < hqmq_med3x_workspace_bytes(c.H, c.dtype)) return HQMQ_ERR_WORKSPACE;
    if ((int64_t)c.B * c.T * c.n > 0xffffffffll) return HQMQ_ERR_SHAPE;      // counters are 32-bit
    if (((uintptr_t)c.ws & 3) != 0) return HQMQ_ERR_ALIGN;
    return HQMQ_OK;
}

// parts: the workspaces hold a part per block
static int med3x_launch(const MedPair &a, int dtype, int count, bool parts, MedSelect *later, hipStream_t st) {
    switch (dtype) {
        case HQMQ_F32: return run_med3x<F32>(a, count, false, later, st);
        case HQMQ_F16: return run_med3x<F16>(a, count, parts, later, st);
        default: return run_med3x<BF16>(a, count, parts, later, st);
    }
}

int hqmq::med3x_calls(const Med3xCall *c, int count, MedSelect *later, hipStream_t st) {
    MedTensor t[2];
    for (int i = 0; i < count; i++) {
        const int rc = check_med3x(c[i]);
        if (rc) return rc;
        const int elt = c[i].dtype == HQMQ_F32 ? 4 : 2;
        const int vec = !(((uintptr_t)c[i].x | (uintptr_t)(c[i].xsb * elt) | (uintptr_t)(c[i].xsh * elt) | (uintptr_t)(c[i].xst * elt)) & (4 * elt - 1));
        t[i] = MedTensor{c[i].x, c[i].xsb, c[i].xsh, c[i].xst, vec, c[i].mult, (uint32_t *)c[i].ws, c[i].median, c[i].thr, c[i].n_out};
    }
    // What a call's launches touch of its workspace.  Two calls may share one, or a part: then they go one after the other, each with its
    // selection, which cannot wait for the quantize launch: the second call's histograms come over the first one's.
    auto used = [&](int i, bool best) { return best ? hqmq_med3x_workspace_best_bytes(c[i].H, c[i].dtype) : hqmq_med3x_workspace_bytes(c[i].H, c[i].dtype); };
    auto has_best = [&](int i) { return c[i].ws_bytes >= used(i, true); };
    auto apart = [&](bool best0, bool best1) {
        const uintptr_t w0 = (uintptr_t)c[0].ws, w1 = (uintptr_t)c[1].ws;
        return w0 + used(0, best0) <= w1 || w1 + used(1, best1) <= w0;
    };
    // one set of launches for both tensors where their shapes agree and their workspaces are apart
    if (count == 2 && c[0].dtype == c[1].dtype && c[0].B == c[1].B && c[0].H == c[1].H && c[0].T == c[1].T && c[0].n == c[1].n) {
        const bool parts = has_best(0) && has_best(1) && apart(true, true);
        if (parts || apart(false, false))
            return med3x_launch(MedPair{{t[0], t[1]}, c[0].B, c[0].H, c[0].T, c[0].n}, c[0].dtype, 2, parts, later, st);
    }
    if (count == 2 && later && !apart(has_best(0), has_best(1))) later = nullptr;
    for (int i = 0; i < count; i++) {
        const int rc = med3x_launch(MedPair{{t[i], t[i]}, c[i].B, c[i].H, c[i].T, c[i].n}, c[i].dtype, 1, has_best(i), later ? later + i : nullptr, st);
        if (rc) return rc;
    }
    return HQMQ_OK;
}

extern "C" int hqmq_med3x_threshold(const void *x, int64_t x_stride_b, int64_t x_stride_h, int64_t x_stride_t, int dtype, int B,
                                    int H, int T, int n_chunks, float mult, void *workspace, int64_t workspace_bytes,
                                    float *median, void *thr, int32_t *n_out, void *stream) {
    const Med3xCall c{x, x_stride_b, x_stride_h, x_stride_t, dtype, B, H, T, n_chunks, mult, workspace, workspace_bytes,
                      median, thr, n_out};
    return med3x_calls(&c, 1, nullptr, (hipStream_t)stream);
}

int hqmq::check_compact(const CompactCall &c) {
    if (!c.x || !c.flag_plane || !c.sideband || !c.sb_tile_off || !c.sb_count || !c.overflow) return HQMQ_ERR_NULL;
    if (c.B < 1 || c.H < 1 || c.T < 0 || c.n < 1 || c.t_cap < 1 || c.sb_cap < 1 || c.t_off < 0) return HQMQ_ERR_SHAPE;
    if (c.dtype != HQMQ_F32 && c.dtype != HQMQ_F16 && c.dtype != HQMQ_BF16) return HQMQ_ERR_DTYPE;
    return HQMQ_OK;
}

// whole 16-row tiles from an aligned first row: the two tile-parallel passes
static bool bulk_compact(const CompactCall &c) {
    return !c.pos && (c.t_off % kTile) == 0 && c.T >= 512 && (int64_t)c.t_off + c.T <= c.t_cap && c.B * c.H <= 65535;
}

static int launch_compact(const CompactPair &p, int count, hipStream_t st) {
    const CompactCall &c = p.c[0];
    if (c.T == 0) return HQMQ_OK;
    if (bulk_compact(c)) {
        hipLaunchKernelGGL(tile_scan_kernel, dim3(c.B * c.H, 1, count), dim3(1024), 0, st, p);
        const dim3 grid((c.T + 255) / 256, c.B * c.H, count);
        switch (c.dtype) {
            case HQMQ_F32: hipLaunchKernelGGL(tile_copy_kernel<F32>, grid, dim3(256), 0, st, p); break;
            case HQMQ_F16: hipLaunchKernelGGL(tile_copy_kernel<F16>, grid, dim3(256), 0, st, p); break;
            default: hipLaunchKernelGGL(tile_copy_kernel<BF16>, grid, dim3(256), 0, st, p); break;
        }
        return hip_status(hipGetLastError());
    }
    const dim3 grid(c.B * c.H, 1, count);
#define LAUNCH(NT)                                                                                              \
    switch (c.dtype) {                                                                                          \
        case HQMQ_F32: hipLaunchKernelGGL((compact_kernel<F32, NT>), grid, dim3(NT), 0, st, p); break;          \
        case HQMQ_F16: hipLaunchKernelGGL((compact_kernel<F16, NT>), grid, dim3(NT), 0, st, p); break;          \
        default: hipLaunchKernelGGL((compact_kernel<BF16, NT>), grid, dim3(NT), 0, st, p); break;               \
    }
    if (c.T <= 64) { LAUNCH(64) } else { LAUNCH(1024) }
#undef LAUNCH
    return hip_status(hipGetLastError());
}

int hqmq::compact_calls(const CompactCall *c, int count, hipStream_t st) {
    int vec[2] = {0, 0};
    for (int i = 0; i < count; i++) {
        const int rc = check_compact(c[i]);
        if (rc) return rc;
        const int elt = c[i].dtype == HQMQ_F32 ? 4 : 2;
        vec[i] = !(((uintptr_t)c[i].x | (uintptr_t)c[i].sideband | (uintptr_t)(c[i].xsb * elt) | (uintptr_t)(c[i].xsh * elt) | (uintptr_t)(c[i].xst * elt)) &
                   (4 * elt - 1));
    }
    if (count == 2 && c[0].dtype == c[1].dtype && c[0].B == c[1].B && c[0].H == c[1].H && c[0].T == c[1].T && c[0].n == c[1].n &&
        bulk_compact(c[0]) == bulk_compact(c[1]))
        return launch_compact(CompactPair{{c[0], c[1]}, {vec[0], vec[1]}}, 2, st);
    for (int i = 0; i < count; i++) {
        const int rc = launch_compact(CompactPair{{c[i], c[i]}, {vec[i], vec[i]}}, 1, st);
        if (rc) return rc;
    }
    return HQMQ_OK;
}

extern "C" int hqmq_crop(const hqmq_crop_args *a, void *stream) {
    if (!a) return HQMQ_ERR_NULL;
    if (a->count < 1 || a->count > 2 || a->B < 1 || a->H < 1 || (int64_t)a->B * a->H > 65535 || a->t_cap < 1 || a->n_chunks < 1) return HQMQ_ERR_SHAPE;
    for (int i = 0; i < a->count; i++)
        if (!a->flag_plane[i] || !a->sb_tile_off[i] || !a->sb_count[i]) return HQMQ_ERR_NULL;
    const int64_t tiles = (a->t_cap + kTile - 1) / kTile;
    hipLaunchKernelGGL(crop_kernel, dim3((unsigned)((tiles + kCropTiles - 1) / kCropTiles), a->B * a->H, a->count), dim3(kCropTiles), 0,
                       (hipStream_t)stream, *a);
    return hip_status(hipGetLastError());
}

extern "C" int hqmq_outlier_compact(const void *x, int64_t x_stride_b, int64_t x_stride_h, int64_t x_stride_t, int dtype, int B,
                                    int H, int T, int n_chunks, uint8_t *flag_plane, int64_t t_cap, int t_off,
                                    const int32_t *pos, void *sideband, int64_t sb_cap, int32_t *sb_tile_off,
                                    int32_t *sb_count, int32_t *overflow, uint16_t *sb_coord, const hqmq_packed_rows *planes,
                                    void *stream) {
    CompactCall c{x, x_stride_b, x_stride_h, x_stride_t, dtype, B, H, T, n_chunks, flag_plane, t_cap, t_off, pos,
                  sideband, sb_cap, sb_tile_off, sb_count, overflow, sb_coord, nullptr, nullptr, nullptr, 0, 0, 0, 0};
    if (planes) {
        if (!planes->main_plane || !planes->scale_plane || (planes->aux_bits > 0 && !planes->aux_plane)) return HQMQ_ERR_NULL;
        if (planes->idx_bits < 1 || planes->main_bits < planes->idx_bits - 8 || planes->main_bits > 16 || planes->aux_bits < 0 ||
            planes->aux_bits > 8 || planes->qmax < 1)
            return HQMQ_ERR_LAYOUT;
        c.main_plane = planes->main_plane; c.aux_plane = planes->aux_plane; c.scale_plane = planes->scale_plane;
        c.idx_bits = planes->idx_bits; c.main_bits = planes->main_bits; c.aux_bits = planes->aux_bits; c.qmax = planes->qmax;
    }
    return compact_calls(&c, 1, (hipStream_t)stream);
}

namespace hqmq {
template <class D>
__global__ void outlier_mask_kernel(const typename D::storage *x, int64_t xsb, int64_t xsh, int64_t xst, int B, int H, int T, int n,
                                    const typename D::storage *thr, uint8_t *mask) {
    const int64_t total = (int64_t)B * H * T * n;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(g % n);
        const int64_t row = g / n;
        const int t = (int)(row % T), h = (int)((row / T) % H), b = (int)(row / ((int64_t)T * H));
        mask[g] = chunk_norm<D>(x + b * xsb + h * xsh + (int64_t)t * xst + c * 4) > D::load(thr + h) ? 1 : 0;
    }
}
}  // namespace hqmq

extern "C" int hqmq_outlier_mask(const void *x, int64_t x_stride_b, int64_t x_stride_h, int64_t x_stride_t, int dtype, int B,
                                 int H, int T, int n_chunks, const void *thr, uint8_t *mask, void *stream) {
    if (!x || !thr || !mask) return HQMQ_ERR_NULL;
    if (B < 1 || H < 1 || T < 0 || n_chunks < 1) return HQMQ_ERR_SHAPE;
    if (T == 0) return HQMQ_OK;
    const int64_t total = (int64_t)B * H * T * n_chunks;
    int64_t g = (total + 255) / 256;
    if (g > (1 << 20)) g = 1 << 20;
    hipStream_t st = (hipStream_t)stream;
#define LAUNCH(DT, ST)                                                                                                      \
    hipLaunchKernelGGL(outlier_mask_kernel<DT>, dim3((unsigned)g), dim3(256), 0, st, (const ST *)x, x_stride_b, x_stride_h, \
                       x_stride_t, B, H, T, n_chunks, (const ST *)thr, mask)
    switch (dtype) {
        case HQMQ_F32: LAUNCH(F32, float); break;
        case HQMQ_F16: LAUNCH(F16, uint16_t); break;
        case HQMQ_BF16: LAUNCH(BF16, uint16_t); break;
        default: return HQMQ_ERR_DTYPE;
    }
#undef LAUNCH
    return hip_status(hipGetLastError());
}
