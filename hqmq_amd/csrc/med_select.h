// The order statistics of Med3x over histograms of blocks, 16-bit types: what the selection's own launch (med3x.hip) and the
// quantizer's long-call kernel, which selects for itself (quantize_grid.hip), share.
// Compiled with -ffp-contract=off.
#pragma once
#include "quantize_common.h"

namespace hqmq {

constexpr int kBins1 = 32768;
// The last 64 bins would count NaN patterns, which are counted apart: they hold the sums of 64 groups of 512 bins instead,
// which spare the selection all but the two groups it needs.
constexpr int kGroups = 64, kGroupBins = kBins1 / kGroups, kGroupAt = kBins1 - kGroups;

// A block's part of the workspace: bins[kBins1 / 2] (two 16-bit counters a word; only those of groups whose
// sum is not zero are written) | sums[kGroups] | NaN count | padding
constexpr int kPartWords = kBins1 / 2 + kGroups + 64, kPartSums = kBins1 / 2, kPartNan = kPartSums + kGroups;
constexpr int kPartBlocks = 256;        // at most, and one per head where there are more heads

// fp32 bit pattern whose order is the norm's; of a 16-bit type only the upper 16 bits can be set
template <class D>
__device__ __forceinline__ uint32_t norm_bits(float nrm) {
    if (D::code == HQMQ_F32) return __float_as_uint(nrm);
    if (D::code == HQMQ_F16) return (uint32_t)__half_as_ushort(__float2half_rn(nrm)) << 16;
    return __float_as_uint(nrm);  // bf16 value: low 16 bits are zero
}
// the norm whose 16-bit key this is (16-bit types)
template <class D>
__device__ __forceinline__ float key_value(uint32_t key16) {
    return D::code == HQMQ_F16 ? __half2float(__ushort_as_half((uint16_t)key16)) : __uint_as_float(key16 << 16);
}

// Sum over the wavefront, in every lane (lane permutations inside the vector unit).
__device__ __forceinline__ uint32_t wave_sum(uint32_t x) {
    x += dpp_u32<0xB1>(x);
    x += dpp_u32<0x4E>(x);
    x += dpp_u32<0x141>(x);
    x += dpp_u32<0x140>(x);
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    x = r[0] + r[1];
    const auto q = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return q[0] + q[1];
}

template <class D>
__device__ __forceinline__ void finish_threshold(float a, float b, bool same, float mult, int h, float *median,
                                                 typename D::storage *thr) {
    float med;
    if (same) med = a;
    else {
        const float d = b - a;
        const float e = d * 0.5f;
        med = b - e;
    }
    median[h] = med;
    const float t32 = med * mult;
    D::store(thr + h, D::rnd(t32));
}
// a NaN norm makes the quantile NaN, the mask empty
template <class D>
__device__ __forceinline__ void nan_threshold(float *median, void *thr, int32_t *n_out, int h) {
    median[h] = NAN;
    D::store((typename D::storage *)thr + h, NAN);
    if (n_out) n_out[h] = 0;
}

__device__ __forceinline__ uint32_t lanes_before(uint32_t v) {          // exclusive prefix sum over the wavefront, inside the vector unit
    uint32_t incl = v;
    incl += dpp_u32<0x111>(incl);       // row_shr 1, 2, 4, 8: over rows of 16
    incl += dpp_u32<0x112>(incl);
    incl += dpp_u32<0x114>(incl);
    incl += dpp_u32<0x118>(incl);
    incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x142, 0xa, 0xf, false);        // row_bcast 15: rows 1 and 3 behind 0 and 2
    incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x143, 0xc, 0xf, false);        // row_bcast 31: rows 2 and 3 behind 1
    return incl - v;
}
// The bin with rank `rank` among the 512 counters of a group, 8 per lane: its number, in the lane that holds it (-1 elsewhere).
__device__ __forceinline__ int bin_of_rank(const uint32_t (&v)[8], uint32_t rank) {
    uint32_t tot = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) tot += v[i];
    const uint32_t first = lanes_before(tot);
    if (rank < first || rank >= first + tot) return -1;
    rank -= first;
    int i = 0;
#pragma unroll
    for (int k = 0; k < 7; k++)
        if (i == k && rank >= v[k]) { rank -= v[k]; i = k + 1; }
    return (int)(threadIdx.x & 63) * 8 + i;
}

// By a block of 1024 threads: sums of the groups over the head's parts, the group of each rank, that group's bins over
// the parts (a wavefront per part, 1 KB a time), the bin inside it.  The count wants the bins of the threshold's group as
// well; the median's group leaves two for it nearly always.  Up to kAheadParts parts these are asked for along with the median's (a third
// round trip otherwise: 8 heads, 32 parts, 6.9 -> 5.5 us; with every loop unrolled, 7.5: a launch this short waits for its code).  Of more
// parts four wavefronts a group take more trips one after the other than all sixteen do for the median's group and then for the threshold's,
// and the block with the outputs came last of the whole quantize launch: 32768 tokens of one head, fp16 s96_r4 (256 parts), appended 64.8 -> 54.5 us,
// with a launch of its own 56.4 -> 51.4; 16384 tokens of two heads fake-quantized (128 parts) 32.4 -> 28.3.
// outputs: median, threshold and count are wanted; otherwise just the threshold, which is returned to every thread, and the wavefronts
// share the one or two groups of the median.  sh: kSelectWords words of LDS, which the last wavefront reads until the block's next barrier.
constexpr int kAheadParts = 32;
// The quantize launch selects for itself up to this many parts.  Every one of its blocks reads all of them, so what it saves shrinks with their
// number: over 480 appended and fake-quantized calls of one to six heads 5 % on average up to 64 parts, 2 % at 128 (6 % lost at worst), and
// beyond, single heads of more than 16384 tokens, 1.4 % with 6 % lost where the blocks fill the chip (54.5 us above, 51.4 with the launch).
constexpr int kSelectParts = 128;
constexpr int kSelectWords = 16 * kGroups + 4 * kGroupBins + 2 * kPartBlocks + 4;
// meanwhile(): what the block does while the first words travel.
template <class D, class F>
__device__ __forceinline__ float select16(const MedSelect &m, int h, bool outputs, uint32_t *sh, F meanwhile) {
    const int parts = m.parts, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint64_t *some_sh = reinterpret_cast<uint64_t *>(sh);                       // the groups a part has any of
    uint32_t *sums_sh = sh + 2 * kPartBlocks, *bins_sh = sums_sh + 16 * kGroups, *key_sh = bins_sh + 4 * kGroupBins, *nan_sh = key_sh + 2;
    const uint32_t per_head = m.per_head;
    const uint32_t *ws = m.ws + (size_t)h * parts * kPartWords;
    for (int i = tid; i < 4 * kGroupBins; i += 1024) bins_sh[i] = 0;
    if (tid == 0) *nan_sh = 0;
    uint32_t s = 0, nan = 0;
    auto sums_of = [&](int p) { return ws[(size_t)min(p, parts - 1) * kPartWords + kPartSums + lane]; };
    uint32_t v0 = sums_of(wave), v1 = sums_of(wave + 16);
    if (tid < parts) nan = ws[(size_t)tid * kPartWords + kPartNan];
    meanwhile();
    for (int p0 = wave; p0 < parts; p0 += 32) {         // (two requested at a time)
        const int p1 = p0 + 16;
        if (p0 != wave) { v0 = sums_of(p0); v1 = sums_of(p1); }
        s += v0 + (p1 < parts ? v1 : 0u);
        const uint64_t some0 = __builtin_amdgcn_ballot_w64(v0 != 0u), some1 = __builtin_amdgcn_ballot_w64(v1 != 0u);
        if (lane == 0) {
            some_sh[p0] = some0;
            if (p1 < parts) some_sh[p1] = some1;
        }
    }
    sums_sh[wave * kGroups + lane] = s;
    __syncthreads();
    if (nan) *nan_sh = 1;
    uint32_t sum = 0;                                   // of group `lane`, in every wavefront
#pragma unroll
    for (int w = 0; w < 16; w++) sum += sums_sh[w * kGroups + lane];
    const uint32_t at = lanes_before(sum), rank[2] = {(per_head - 1) / 2, per_head / 2};
    int group[2];
    uint32_t rest[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint64_t here = __builtin_amdgcn_ballot_w64(rank[i] >= at && rank[i] < at + sum);
        group[i] = here ? (int)__builtin_ctzll(here) : kGroups - 1;
        rest[i] = rank[i] - (uint32_t)__builtin_amdgcn_readlane((int)at, group[i]);
    }
    // the bins of group g, added up over the parts first, first + step, .. by this wavefront
    auto gather = [&](int g, uint32_t *to, int first, int step) {
        uint32_t v[8] = {};
        for (int p0 = first; p0 < parts; p0 += 4 * step) {
            uint4 x[4];                                 // (all four requested, also where the group was not written: not used then)
#pragma unroll
            for (int i = 0; i < 4; i++) x[i] = reinterpret_cast<const uint4 *>(ws + (size_t)min(p0 + i * step, parts - 1) * kPartWords)[g * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const bool some = p0 + i * step < parts && (some_sh[min(p0 + i * step, parts - 1)] >> g & 1ull);
                const uint32_t w[4] = {x[i].x, x[i].y, x[i].z, x[i].w};
#pragma unroll
                for (int k = 0; k < 4; k++) { v[2 * k] += some ? w[k] & 0xffffu : 0u; v[2 * k + 1] += some ? w[k] >> 16 : 0u; }
            }
        }
#pragma unroll
        for (int i = 0; i < 8; i++)
            if (v[i]) atomicAdd(&to[lane * 8 + i], v[i]);
    };
    auto bins = [&](const uint32_t *from, uint32_t (&v)[8]) {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = from[lane * 8 + i];
    };
    // the group of the threshold that a median of this key has (a threshold below every norm or beyond infinity: 0, or the last)
    auto group_above = [&](float tv) { return (int)min((norm_bits<D>(fmaxf(tv, 0.f)) >> 16) / kGroupBins, (uint32_t)kGroups - 1u); };
    const bool ahead = outputs && parts <= kAheadParts;
    const int top_lo = group_above(D::rnd(key_value<D>((uint32_t)(group[0] * kGroupBins)) * m.mult));
    {
        const int q = wave >> 2, g = q == 0 ? group[0] : q == 1 ? group[1] : min(top_lo + q - 2, kGroups - 1);
        if (ahead) {
            if (q < 2 || m.n_out) gather(g, bins_sh + q * kGroupBins, wave & 3, 4);
        } else if (group[0] == group[1]) gather(group[0], bins_sh, wave, 16);
        else gather(group[wave >> 3], bins_sh + (wave >> 3) * kGroupBins, wave & 7, 8);
    }
    __syncthreads();
    if (*nan_sh) {
        if (outputs && tid == 0) nan_threshold<D>(m.median, m.thr, m.n_out, h);
        return NAN;
    }
    if (wave < 2) {
        const int side = wave;
        uint32_t v[8];
        bins(bins_sh + (!ahead && group[0] == group[1] ? 0 : side) * kGroupBins, v);
        const int bin = bin_of_rank(v, rest[side]);
        if (bin >= 0) key_sh[side] = (uint32_t)(group[side] * kGroupBins + bin);
    }
    __syncthreads();
    const bool same = rank[0] == rank[1];
    const float lo = key_value<D>(key_sh[0]), hi = key_value<D>(key_sh[1]);
    const float tv = D::rnd((same ? lo : hi - (hi - lo) * 0.5f) * m.mult);
    if (!outputs) return tv;
    if (tid == 0) finish_threshold<D>(lo, hi, same, m.mult, h, m.median, (typename D::storage *)m.thr);
    if (!m.n_out) return tv;
    // chunks with norm > thr: whole groups above the one that holds the threshold, and the bins above it in there
    const int top = group_above(tv);
    uint32_t *there = bins_sh + (!ahead || top == top_lo ? 2 : 3) * kGroupBins;
    if (!ahead || (top != top_lo && top != top_lo + 1)) {
        if (ahead) {                                    // the median's bin is far from its group's first
            for (int i = tid; i < kGroupBins; i += 1024) there[i] = 0;
            __syncthreads();
        }
        gather(top, there, wave, 16);
        __syncthreads();
    }
    if (wave != 0) return tv;
    uint32_t v[8], n = lane > top ? sum : 0u;
    bins(there, v);
#pragma unroll
    for (int i = 0; i < 8; i++)
        if (key_value<D>((uint32_t)(top * kGroupBins + lane * 8 + i)) > tv) n += v[i];
    n = wave_sum(n);
    if (lane == 0) m.n_out[h] = (int32_t)n;
    return tv;
}

}  // namespace hqmq
