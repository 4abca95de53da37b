// What the two codeword searches of the quantizer share (quantize.hip: scan over the secondaries, quantize_grid.hip:
// cell lists): the kernel parameters and everything that happens to a chunk once its codeword is known - per-token
// scale, radius code, Med3x mask, unpacked outputs, packed rows and the sideband compaction of short appends.
// Compiled with -ffp-contract=off.
#pragma once
#include "common.h"

#include <type_traits>

namespace hqmq {

constexpr int kQThreads = 256;   // short appends: all new rows of a (b, h) in one block of this many lanes

// Maximum over groups of `n` neighbouring lanes (n a power of two up to 64), every lane of a group receiving it:
// lane permutations inside the vector unit (quad, half-row and row mirrors, then the 16- and 32-lane row swaps).
// The operands are ordinary numbers or -inf (no NaN), as unsigned bit patterns of non-negative floats order like the
// values, the same routine serves both.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, false);
}
template <class T, class MAX>
__device__ __forceinline__ T group_max(T x, int n, MAX mx) {
    auto step = [&](uint32_t other) { x = mx(x, __builtin_bit_cast(T, other)); };
    if (n >= 2) step(dpp_u32<0xB1>(__builtin_bit_cast(uint32_t, x)));       // quad_perm [1,0,3,2]
    if (n >= 4) step(dpp_u32<0x4E>(__builtin_bit_cast(uint32_t, x)));       // quad_perm [2,3,0,1]
    if (n >= 8) step(dpp_u32<0x141>(__builtin_bit_cast(uint32_t, x)));      // row_half_mirror
    if (n >= 16) step(dpp_u32<0x140>(__builtin_bit_cast(uint32_t, x)));     // row_mirror
    if (n >= 32) {
        const uint32_t b = __builtin_bit_cast(uint32_t, x);
        const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
        x = mx(__builtin_bit_cast(T, (uint32_t)r[0]), __builtin_bit_cast(T, (uint32_t)r[1]));
    }
    if (n >= 64) {
        const uint32_t b = __builtin_bit_cast(uint32_t, x);
        const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
        x = mx(__builtin_bit_cast(T, (uint32_t)r[0]), __builtin_bit_cast(T, (uint32_t)r[1]));
    }
    return x;
}

struct QParams {
    const void *x;
    int64_t xsb, xsh, xst;
    int B, H, T, n;
    const void *joint;
    const float *slack;
    int S, qmax;
    int32_t *idx_out, *rq_out;
    void *rmax_out, *dense_out;
    const void *thr;
    uint8_t *mask_out;
    uint8_t *main_plane, *aux_plane, *flag_plane;
    void *scale_plane;
    int64_t t_cap;
    int t_off;
    const int32_t *pos;
    int idx_bits, main_bits, aux_bits;
    int tokens_per_block;       // of the scan kernels and of appends that compact in the quantize launch: kQThreads / n
    int32_t *stats;
    uint32_t *scale_max;
    // sideband compaction in the same launch (compact != 0): see ChunkSink
    int compact;
    void *sideband;
    int64_t sb_cap;
    int32_t *sb_tile_off, *sb_count, *overflow;
    uint16_t *sb_coord;
    // chunks of x and of dense_out may be moved by one vector access (bases and strides allow it)
    int vec_in, vec_out;
    int vec_rows;               // rows of the code planes are whole dwords at dword addresses
    // cell lists (quantize_grid.hip); NULL: scan
    const uint4 *grid;
    int64_t grid_stride;        // uint4 per head
    int iters;                  // rounds of tokens a block of the cell-list kernel takes
    MedSelect med;              // parts != 0: blocks of the long-call kernel work the threshold out first (med_select.h)
};
struct QPair {
    QParams p[2];               // K, V: blockIdx.z picks one
    int per_head;               // cell-list kernel, long calls: blocks per tensor, b and h
    int med_at;                 // and where in LDS a threshold is selected (-1: where the table comes afterwards)
};

// The four stored elements of a chunk, as they are in memory.
template <class D>
struct RawChunk {
    uint32_t w[sizeof(typename D::storage)];     // 2 words of two 16-bit elements, or 4 fp32 words
    __device__ __forceinline__ void load(const typename D::storage *p, bool vec) {
        if constexpr (sizeof(typename D::storage) == 2) {
            if (vec) {
                const uint2 v = *reinterpret_cast<const uint2 *>(p);
                w[0] = v.x; w[1] = v.y;
            } else {
                w[0] = (uint32_t)p[0] | (uint32_t)p[1] << 16;
                w[1] = (uint32_t)p[2] | (uint32_t)p[3] << 16;
            }
        } else {
            if (vec) {
                const uint4 v = *reinterpret_cast<const uint4 *>(p);
                w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
            } else {
                for (int j = 0; j < 4; j++) w[j] = __float_as_uint(p[j]);
            }
        }
    }
    __device__ __forceinline__ void store(typename D::storage *p, bool vec) const {
        if constexpr (sizeof(typename D::storage) == 2) {
            if (vec) *reinterpret_cast<uint2 *>(p) = uint2{w[0], w[1]};
            else { p[0] = (uint16_t)w[0]; p[1] = (uint16_t)(w[0] >> 16); p[2] = (uint16_t)w[1]; p[3] = (uint16_t)(w[1] >> 16); }
        } else {
            if (vec) *reinterpret_cast<uint4 *>(p) = uint4{w[0], w[1], w[2], w[3]};
            else for (int j = 0; j < 4; j++) p[j] = __uint_as_float(w[j]);
        }
    }
    __device__ __forceinline__ float get(int j) const {
        if constexpr (D::code == HQMQ_F32) return __uint_as_float(w[j]);
        else if constexpr (D::code == HQMQ_F16) return __half2float(__ushort_as_half((uint16_t)(w[j >> 1] >> (16 * (j & 1)))));
        else return __uint_as_float((j & 1) ? (w[j >> 1] & 0xffff0000u) : (w[j >> 1] << 16));
    }
    __device__ __forceinline__ void set(int j, float f) {
        if constexpr (D::code == HQMQ_F32) w[j] = __float_as_uint(f);
        else {
            typename D::storage h;
            D::store(&h, f);
            w[j >> 1] = (j & 1) ? (w[j >> 1] & 0xffffu) | (uint32_t)h << 16 : (w[j >> 1] & 0xffff0000u) | h;
        }
    }
};

// Byte `byte` of the little-endian bit stream of W-bit fields vals[0 .. count) >> shift (W = 0: width w at run time).
// A byte meets at most (7 + W - 1) / W + 1 fields.
template <int W>
__device__ __forceinline__ uint8_t gather_byte_w(const uint32_t *vals, int count, int w, int shift, int byte) {
    const int ww = W ? W : w;
    const int i0 = byte * 8 / ww, o = byte * 8 - i0 * ww;
    const uint32_t fmask = (1u << ww) - 1u;
    const int most = W ? (7 + W - 1) / W + 1 : (7 + ww - 1) / ww + 1;
    uint32_t out = 0;
#pragma unroll
    for (int k = 0; k < most; k++)
        if (i0 + k < count) out |= (uint32_t)((((uint64_t)((vals[i0 + k] >> shift) & fmask) << (k * ww)) >> o) & 0xffu);
    return (uint8_t)out;
}
__device__ __forceinline__ uint8_t gather_byte(const uint32_t *vals, int count, int w, int shift, int byte) {
    switch (w) {        // the widths the layout rule produces (main 8 / 12, aux 1..3, flags 1)
        case 1: return gather_byte_w<1>(vals, count, w, shift, byte);
        case 2: return gather_byte_w<2>(vals, count, w, shift, byte);
        case 3: return gather_byte_w<3>(vals, count, w, shift, byte);
        case 8: return gather_byte_w<8>(vals, count, w, shift, byte);
        case 12: return gather_byte_w<12>(vals, count, w, shift, byte);
        default: return gather_byte_w<0>(vals, count, w, shift, byte);
    }
}

// n one-bit fields (n = 8, 16, 32 or 64: whole bytes) as one store, or byte by byte where the row's address may be odd
__device__ __forceinline__ void store_bits(uint8_t *dst, uint64_t bits, int n, bool vec) {
    if (vec && n == 32) *reinterpret_cast<uint32_t *>(dst) = (uint32_t)bits;
    else if (vec && n == 64) { reinterpret_cast<uint32_t *>(dst)[0] = (uint32_t)bits; reinterpret_cast<uint32_t *>(dst)[1] = (uint32_t)(bits >> 32); }
    else for (int i = 0; i < (n >> 3); i++) dst[i] = (uint8_t)(bits >> (8 * i));
}

template <class D>
__device__ __forceinline__ float ref_score(const float u[4], const typename D::storage *row) {
    float j0 = D::load(row), j1 = D::load(row + 1), j2 = D::load(row + 2), j3 = D::load(row + 3);
    float acc = u[0] * j0;
    acc = fmaf(u[1], j1, acc);
    acc = fmaf(u[2], j2, acc);
    acc = fmaf(u[3], j3, acc);
    return D::rnd(acc);
}

// argmax over all K rows with torch's rule: first maximum, NaN counts as maximum.
template <class D>
__device__ int brute_argmax(const float u[4], const typename D::storage *jh, int K) {
    int best = 0;
    float bs = 0.f;
    for (int k = 0; k < K; k++) {
        float s = ref_score<D>(u, jh + (size_t)k * 4);
        if (is_nan(s)) return k;
        if (k == 0 || s > bs) { bs = s; best = k; }
    }
    return best;
}

// Everything after the search, for one chunk per lane: lane tid = tok_local * n + c of a block of NT lanes holds chunk c of
// token t0 + tok_local of one (b, h), in one or more rounds of tokens (t0).
//   ROWS     the n lanes of a token sit side by side inside one wavefront (n a power of two up to 64); otherwise the
//            block's lanes meet at barriers, so every lane of the block has to take every round
//   WHAT     what the call can ask for: kUnpacked (codes, scales, masks, dense tensor), kPlanes (packed rows), kCompact
//            (sideband entries in the same launch); a launch that is known to ask for less carries less
//   MB       main_bits where known at compile time, else 0
//   FAST     packed rows of the usual forms (fast_rows): neighbouring lanes put the rows together among themselves (DPP) and
//            everything that does not change from round to round is worked out once.  Through LDS, with its addresses and the
//            parameters fetched again in every round, packing took a fifth of the cell-list kernel's time at 16-bit codes and a third at
//            12 + 1 bits
// Addresses are a wave-uniform base (scalar arithmetic, once per round) plus a 32-bit lane offset that does not change.
constexpr int kUnpacked = 1, kPlanes = 2, kCompact = 4;
// Rows of 16 or 32 codes of MB + at most three bits, whole chunks of x as vectors, planes at dword addresses.
inline bool fast_rows(const QParams &p, int mb) {
    return (p.n == 16 || p.n == 32) && p.vec_in && p.vec_rows && p.main_plane && p.scale_plane && p.main_bits == mb && p.aux_bits <= 3 &&
           (!p.aux_bits || p.aux_plane) && !p.compact;
}
template <class D, int NT, bool ROWS, int WHAT, int MB, bool FAST = false>
struct ChunkSink {
    using ST = typename D::storage;
    const QParams &a;
    int b, h, tok_local, c;
    uint32_t *code_sh, *aux_sh;     // NT words of LDS each (aux_sh: without ROWS, with compaction, or n = 4)
    int64_t bh, row0;               // row0: the plane row of token 0
    int t_lo, t_hi;                 // this lane's rows of the planes are those of rounds t_lo <= t0 < t_hi
    float thr, qmaxf, inv_qmax;
    uint32_t seen = 0;              // the largest finite scale this lane has written so far, as bits
    // FAST: row 0 of the call in every plane
    uint8_t *main0, *aux0, *flag0;
    ST *scale0;
    int idx_bits, aux_bits;

    __device__ __forceinline__ ChunkSink(const QParams &a_, int b_, int h_, int tok_local_, int c_, uint32_t *code_sh_, uint32_t *aux_sh_)
        : a(a_), b(b_), h(h_), tok_local(tok_local_), c(c_), code_sh(code_sh_), aux_sh(aux_sh_) {
        bh = (int64_t)b * a.H + h;
        row0 = (WHAT & kPlanes) ? (int64_t)(a.pos ? a.pos[b] : 0) + a.t_off : 0;
        if (WHAT & kPlanes) {       // (a bad pos[] must not write outside the plane)
            const int64_t lo = -(row0 + tok_local), hi = a.t_cap + lo;
            t_lo = (int)(lo < 0 ? 0 : lo > INT32_MAX ? INT32_MAX : lo);
            t_hi = (int)(hi < 0 ? 0 : hi > INT32_MAX ? INT32_MAX : hi);
        }
        thr = a.thr ? D::load((const ST *)a.thr + h) : INFINITY;
        qmaxf = (float)a.qmax;
        inv_qmax = __builtin_amdgcn_rcpf(qmaxf);
        if constexpr (FAST) {
            const int n = a.n;
            const int64_t first = bh * a.t_cap + row0;
            idx_bits = a.idx_bits;
            aux_bits = a.aux_bits;
            main0 = a.main_plane + first * (n * MB >> 3);
            aux0 = aux_bits ? a.aux_plane + first * (n * aux_bits >> 3) : nullptr;
            flag0 = a.flag_plane ? a.flag_plane + first * (n >> 3) : nullptr;
            scale0 = (ST *)a.scale_plane + first;
            t_hi = t_hi < a.T - tok_local ? t_hi : a.T - tok_local;
        }
    }

    // The packed rows of one round (FAST).  keep: stays an outlier.
    __device__ __forceinline__ void put_rows(int t0, float rm, uint32_t idx, uint32_t rq, bool keep) {
        const int n = a.n;
        const bool row_ok = t0 >= t_lo && t0 < t_hi;
        // the lane's place in a round's rows, worked out anew each time: the search has no registers to spare
        uint32_t tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const uint32_t lg = n == 32 ? 5 : 4, c = tid & (uint32_t)(n - 1), tok = tid >> lg, eighth = tid >> 3;
        const uint32_t code = (keep ? 0u : rq) << idx_bits | idx;
        const uint32_t lane_base = tid & 63u & ~(uint32_t)(n - 1);
        auto store_ballot = [&](uint8_t *row, uint64_t votes) {                // n bits per token, in its first lane
            const uint64_t mine = votes >> lane_base;
            if (row_ok && c == 0) {
                if (n == 32) *reinterpret_cast<uint32_t *>(row + 4u * tok) = (uint32_t)mine;
                else *reinterpret_cast<uint16_t *>(row + 2u * tok) = (uint16_t)mine;
            }
        };
        uint8_t *main = main0 + (int64_t)t0 * (n * MB >> 3);
        if constexpr (MB == 16) {
            if (row_ok) *reinterpret_cast<uint16_t *>(main + 2u * tid) = (uint16_t)code;
        } else {
            // pairs of codes (24 bits) in even lanes; dword k of eight lanes is the pairs k and k + 1 from bit 8 k on
            const uint32_t low = code & 0xfffu, pair = dpp_u32<0xB1>(low) << 12 | low;             // quad_perm [1,0,3,2]
            const uint32_t next = dpp_u32<0x102>(pair);                                            // row_shl:2
            const uint32_t v = __builtin_amdgcn_alignbit(next >> 8, next << 24 | pair, 4u * tid & 24u);
            if (row_ok && !(tid & 1u) && (tid & 7u) < 6u) *reinterpret_cast<uint32_t *>(main + 4u * (3u * eighth + (tid >> 1 & 3u))) = v;
        }
        if (aux_bits == 1) store_ballot(aux0 + (int64_t)t0 * (n >> 3), __builtin_amdgcn_ballot_w64((code & (1u << MB)) != 0u));
        else if (aux_bits) {
            // the fields of eight lanes, 16 or 24 bits, or'ed together in all of them, then a byte from each of the first
            uint32_t v = (code >> MB) << ((uint32_t)aux_bits * (tid & 7u));
            v |= dpp_u32<0xB1>(v);
            v |= dpp_u32<0x4E>(v);
            v |= dpp_u32<0x141>(v);
            if (row_ok && (tid & 7u) < (uint32_t)aux_bits) (aux0 + (int64_t)t0 * (n * aux_bits >> 3))[(uint32_t)aux_bits * eighth + (tid & 7u)] = (uint8_t)(v >> 8u * (tid & 7u));
        }
        if (flag0) store_ballot(flag0 + (int64_t)t0 * (n >> 3), __builtin_amdgcn_ballot_w64(keep));
        if (row_ok && c == 0) {
            D::store(scale0 + t0 + tok, rm);
            if (rm < INFINITY) seen = max(seen, __float_as_uint(rm));       // scales are positive: bits order like values
        }
    }

    // jrow(g): the chunk's row of the joint table.  QUICK (std::true_type): every norm of the wavefront is an ordinary number of
    // a 16-bit type (quick_divisor), at or above the clamp.
    template <class ROW, class QUICK>
    __device__ __forceinline__ void put(int t0, bool active, const RawChunk<D> &raw, float nrm, float r, int idx, ROW jrow, QUICK) {
        constexpr bool quick = QUICK::value;
        const int tid = threadIdx.x, n = a.n, lane = tid & 63;
        const int lane_base = ROWS ? (lane & ~(n - 1)) : 0;
        const uint64_t tok_lanes = n >= 64 ? ~0ull : ((1ull << n) - 1ull) << lane_base;      // ROWS only
        // ---- per-token scale and radius code ----
        float rm = -INFINITY;
        if (ROWS) {
            // norms are not negative, so their bits order like the values, with NaN (made the positive one) above all others
            uint32_t bits = __float_as_uint(r);
            if (!quick) bits = is_nan(r) ? 0x7fc00000u : bits;
            rm = __uint_as_float(group_max(bits, n, [](uint32_t p, uint32_t q) { return max(p, q); }));
        } else {
            bool rm_nan = false;
            float *radius_sh = reinterpret_cast<float *>(aux_sh);
            __syncthreads();
            radius_sh[tid] = r;
            __syncthreads();
            const int base = tok_local * n;
            for (int i = 0; i < n; i++) {
                const float o = (base + i < NT) ? radius_sh[base + i] : 0.f;
                if (is_nan(o)) rm_nan = true;
                else if (o > rm) rm = o;
            }
            __syncthreads();
            if (rm_nan) rm = NAN;
        }
        if (!quick) rm = clamp_min_d<D>(rm, 1e-8f);
        float scale, qf;
        if (D::code != HQMQ_F32 && (quick || __builtin_amdgcn_ballot_w64(!quick_divisor<D>(rm)) == 0ull)) scale = quick_div<D>(rm, qmaxf, inv_qmax);      // qmax: at most 255
        else scale = D::rnd(rm / qmaxf);
        if constexpr (FAST && quick) {
            // rounded to a whole number by adding 2^23, whose low bits the sum then holds
            const float sum = div_d<D>(r, scale) + 8388608.f;
            put_rows(t0, rm, (uint32_t)idx, min(__float_as_uint(sum) & 0xffffu, (uint32_t)a.qmax), nrm > thr);
            return;
        }
        qf = rintf(div_d<D>(r, scale));
        if (quick) qf = fminf(qf, qmaxf);
        else if (!is_nan(qf)) qf = fminf(fmaxf(qf, 0.f), qmaxf);
        const int rq = !quick && is_nan(qf) ? 0 : (int)qf;
        const bool flagged = nrm > thr;
        if constexpr (FAST) {
            put_rows(t0, rm, (uint32_t)idx, (uint32_t)rq, flagged);
            return;
        }

        if ((WHAT & kUnpacked) && active) {
            const int64_t tok = bh * a.T + t0;                           // wave-uniform; the lanes of a round are neighbours
            if (a.idx_out) a.idx_out[tok * n + tid] = idx;
            if (a.rq_out) a.rq_out[tok * n + tid] = rq;
            if (a.mask_out) a.mask_out[tok * n + tid] = flagged ? 1 : 0;
            if (a.rmax_out && c == 0) D::store((ST *)a.rmax_out + tok + tok_local, rm);
            if (a.dense_out) {
                RawChunk<D> dst = raw;                   // a flagged chunk comes out as it went in
                if (!flagged) {
                    const float rqs = D::rnd(qf * scale);
                    float g[4];
                    jrow(g);
#pragma unroll
                    for (int j = 0; j < 4; j++) dst.set(j, D::rnd(rqs * g[j]));
                }
                dst.store((ST *)a.dense_out + tok * n * 4 + tid * 4, a.vec_out);
            }
        }
        if constexpr ((WHAT & kPlanes) == 0) return;
        if ((WHAT & kUnpacked) && !(a.main_plane || a.flag_plane || a.scale_plane)) return;

        // ---- packed rows ----
        const int64_t row = row0 + t0 + tok_local;
        const bool row_ok = active && t0 >= t_lo && t0 < t_hi;
        // Sideband compaction in the same launch, for appends whose new rows of a (b, h) all sit in this block
        // (T <= tokens_per_block; n a power of two, so the lanes of a token share a wavefront).  Entries, tile
        // offsets and counters come out as the in-order compaction kernel leaves them: flagged chunks in
        // (row, chunk) order behind the entries already there, the offset of a tile = the count before its
        // first row.  The entry slots are worked out before the rows are packed: a flagged chunk that finds the
        // sideband full is packed as a plain chunk (its radius code, no flag) instead of decoding to zero.
        bool keep = flagged;            // stays an outlier in the packed planes
        bool entry = false;             // this lane writes a sideband entry
        int ent_slot = 0, tile_first = 0, ent_total = 0;
        if ((WHAT & kCompact) && ROWS && a.compact) {
            const bool f = row_ok && flagged;
            const uint64_t m = __builtin_amdgcn_ballot_w64(f);
            const int before_c = __popcll(m & tok_lanes & ((1ull << lane) - 1ull));
            int *cnt_sh = reinterpret_cast<int *>(aux_sh);
            if (NT > 64) __syncthreads();
            if (c == 0 && tok_local < a.T) cnt_sh[tok_local] = __popcll(m & tok_lanes);
            const int base = a.sb_count[bh];                            // read by every thread before the barrier,
            __syncthreads();                                            // rewritten by one thread at the end
            int mine = base, total = base;
            for (int i = 0; i < a.T; i++) {
                const int ci = cnt_sh[i];
                if (i < tok_local) mine += ci;
                total += ci;
            }
            tile_first = mine;
            ent_total = total;
            ent_slot = mine + before_c;
            entry = f && ent_slot < a.sb_cap;
            if (f && !entry) {
                keep = false;
                *a.overflow = 1;
            }
        }
        // a flagged chunk is read from the sideband; its packed code keeps idx with radius code 0, which decodes to zero
        const uint32_t code = (uint32_t)idx | ((uint32_t)(keep ? 0 : rq) << a.idx_bits);
        const int main_bits = MB ? MB : a.main_bits;
        // one-bit planes (flags, a one-bit aux field) of tokens whose lanes sit side by side in a wavefront come
        // straight from a ballot: the token's n bits are n / 8 whole bytes of it
        const bool bits_by_ballot = ROWS && n >= 8;
        const uint64_t flag_bits1 = __builtin_amdgcn_ballot_w64(keep) >> lane_base;
        // widths other than 16 and 1 are gathered from the codes of the token's other lanes
        const bool through_lds = (a.main_plane && main_bits != 16) || (a.aux_plane && a.aux_bits && !(a.aux_bits == 1 && bits_by_ballot)) ||
                                 (a.flag_plane && !bits_by_ballot);
        const uint32_t *codes = code_sh + tok_local * n;
        if (through_lds) {
            code_sh[tid] = code;
            if (ROWS) __builtin_amdgcn_wave_barrier();          // the lanes of a token run in step; their LDS accesses stay in order
            else {
                aux_sh[tid] = keep ? 1u : 0u;
                __syncthreads();
            }
            if (ROWS && !bits_by_ballot && a.flag_plane) {      // n = 4: flags through LDS as well
                aux_sh[tid] = keep ? 1u : 0u;
                __builtin_amdgcn_wave_barrier();
            }
        }
        const int64_t prow0 = bh * a.t_cap + row0 + t0;         // wave-uniform: the plane row of the round's first token
        if (a.main_plane) {
            const int rb = (n * main_bits + 7) >> 3;
            uint8_t *base = a.main_plane + prow0 * rb;
            if (main_bits == 16) {
                if (row_ok) reinterpret_cast<uint16_t *>(base)[tid] = (uint16_t)code;       // one code per lane
            } else if (main_bits == 12 && a.vec_rows && !(n & 7)) {
                const int nd = 3 * n >> 3;                                      // 8 codes = 3 dwords
                if (row_ok && c < nd) {
                    const int i0 = 32 * c / 12, o = 32 * c - 12 * i0;           // o = 0, 8 or 4: fields i0 .. i0 + 2 (and i0 + 3 for o = 8)
                    uint32_t v = (codes[i0] & 0xfffu) >> o | (codes[i0 + 1] & 0xfffu) << (12 - o) | (codes[i0 + 2] & 0xfffu) << (24 - o);
                    if (o == 8) v |= (codes[i0 + 3] & 0xfffu) << 28;
                    reinterpret_cast<uint32_t *>(base)[tok_local * nd + c] = v;
                }
            } else if (row_ok) {
                for (int byte = c; byte < rb; byte += n) base[tok_local * rb + byte] = gather_byte(codes, n, main_bits, 0, byte);
            }
        }
        if (a.aux_plane && a.aux_bits) {
            const int rb = (n * a.aux_bits + 7) >> 3;
            uint8_t *base = a.aux_plane + prow0 * rb + tok_local * rb;
            if (a.aux_bits == 1 && bits_by_ballot) {
                const uint64_t aux_bits1 = __builtin_amdgcn_ballot_w64(((code >> main_bits) & 1u) != 0u) >> lane_base;
                if (row_ok && c == 0) store_bits(base, aux_bits1, n, a.vec_rows);
            } else if (row_ok) {
                for (int byte = c; byte < rb; byte += n) base[byte] = gather_byte(codes, n, a.aux_bits, main_bits, byte);
            }
        }
        if (a.flag_plane && row_ok) {
            const int rb = (n + 7) >> 3;
            uint8_t *base = a.flag_plane + prow0 * rb + tok_local * rb;
            if (bits_by_ballot) {
                if (c == 0) store_bits(base, flag_bits1, n, a.vec_rows);
            } else {
                for (int byte = c; byte < rb; byte += n) base[byte] = gather_byte(aux_sh + tok_local * n, n, 1, 0, byte);
            }
        }
        if (a.scale_plane && row_ok && c == 0) {
            D::store((ST *)a.scale_plane + prow0 + tok_local, rm);
            if (rm < INFINITY) seen = max(seen, __float_as_uint(rm));       // scales are positive: bits order like values
        }
        if ((WHAT & kCompact) && ROWS && a.compact) {
            if (row_ok) {
                const int64_t tiles = (a.t_cap + kTile - 1) / kTile;
                if (c == 0 && (row & (kTile - 1)) == 0) a.sb_tile_off[bh * tiles + (row >> 4)] = tile_first;
                if (entry) {
                    raw.store((ST *)a.sideband + (bh * a.sb_cap + ent_slot) * 4, false);
                    if (a.sb_coord) a.sb_coord[bh * a.sb_cap + ent_slot] = (uint16_t)(((row & (kTile - 1)) << 8) | c);
                }
            }
            if (tid == 0) a.sb_count[bh] = ent_total;
        }
    }

    // The largest finite scale written so far, for the attention kernels' range guard: the wavefront's maximum, and an
    // atomic only when it raises the value (after the first blocks it hardly ever does).
    __device__ __forceinline__ void done() {
        if constexpr ((WHAT & kPlanes) == 0) return;
        if (!a.scale_max || !a.scale_plane) return;
        const uint32_t most = group_max(seen, 64, [](uint32_t p, uint32_t q) { return max(p, q); });
        if ((threadIdx.x & 63) == 0 && most > __hip_atomic_load(a.scale_max, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(a.scale_max, most);
    }
};

// quantize_grid.hip: launches the cell-list kernel for one tensor (count = 1) or K and V of equal shape (count = 2)
int launch_quantize_grid(QPair kv, int count, int dtype, hipStream_t st);

}  // namespace hqmq
