// Attention with many query columns per KV head (chunked and whole prefill) over plain 16-bit caches and fp16 caches with verbatim
// outliers, d_h 64 / 128.
//
// The decode kernels give a wavefront 16 or 32 columns and let it decode every KV tile for itself; with hundreds of
// columns the same tile is decoded again and again.  Here a block of eight wavefronts decodes each tile of 64 tokens once
// into LDS (K and V as fp16 codeword * radius code, [token][d]) and all its columns use it:
//   * a wavefront owns 32 columns (a column is a query token and a query head of the group), 256 per block with KVG = 1;
//     with KVG = 2 four wavefronts take the first half of every tile and four the second half for the same 128 columns, and the
//     halves merge through LDS at the end: twice the blocks, for launches that would leave compute units idle otherwise;
//   * S^T = K . Q^T and O^T += V^T . P^T on v_mfma_f32_32x32x16_f16.  The accumulators of S^T (lane = column + 32 * half,
//     rows 8 i + 4 half + j) are the B operand of the second product if the 16 tokens of a step are numbered
//     {4 half + j, 8 + 4 half + j}: P never leaves the registers, and V^T comes from LDS in that order by two transposing
//     reads (ds_read_b64_tr_b16) per 32 x 16 operand;
//   * LDS rows are stored with their 16-byte parts permuted by the token, so that the writes (16 tokens at the same part),
//     the K reads (16 tokens) and the transposing V reads (4 tokens by 64 bytes) all meet 64 different banks;
//   * K and V in LDS are codeword * radius code; K's scale of the token is applied to the score and V's to P, in fp32, as the decode
//     kernels do (V times radius * scale / qmax in LDS saves 16 multiplications per 32 tokens, but rounds once more: 4 to 8 % further
//     from 64-bit results at fp16);
//   * fp16 outlier caches (FL): the wavefront that decoded a tile writes the tile's verbatim chunks over the zeros that flagged
//     chunks decode to, and marks K's in a flag word per token.  K is codeword * radius code elsewhere, as above: the operand of
//     a score step is split by the flags into codes and verbatim values (a mask per chunk), which are multiplied one after
//     the other; the two sums meet when the token's scale is applied, so that K has the decode kernels' precision at every magnitude.
//     V is held as values, multiplied out in fp32 and rounded once, in which the verbatim chunks have their place, and P is not
//     multiplied with scales, one rounding less.  bf16 caches keep the decode kernels: a verbatim bf16 chunk need not fit fp16;
//   * one basic block per 32 tokens, written out one matrix instruction at a time: the scores of the next 32 tokens run with
//     the exponentials of these, their products with V with the decoding of a later tile.  A matrix instruction takes 32
//     cycles of its own pipe, a vector instruction about 4.3 of the shared issue slot (8.3 for an exponential), so that the
//     two kinds have to be interleaved, and every vector instruction saved counts;
//   * two tile buffers, one barrier per tile (two with KVG = 1).  The codes of a tile are requested two tiles ahead into
//     registers that nothing copies (a copy would wait for them).
// Measured, B = 1, 32 / 8 heads of 128, s96_r4, 1024 queries on 32768 tokens (541 GFLOP, 0.43 ms at the rate of a large matrix
// product): 0.61 ms against 0.96 with the decode kernels' two-column-group variants; 4096 on 4096 tokens causal, s24_r3:
// 0.185 against 0.41; four sequences of 300 on 300: 0.023 against 0.048.  With 2 % of the K and V chunks verbatim: 1024 queries on
// 32768 tokens 0.76 ms against 2.88, 300 on 8000 (28 / 4 heads, s192_r6) 0.087 against 0.318.  (K held as values like V, without the
// second product, with the launch plans of a time when this took 0.93 and 0.122: 0.70 and 0.101, but up to 1.55 times as far from
// 64-bit results at K of 3e-5 and 1.34 times at K of order one; values only in tokens with verbatim chunks, in units of a power of two: 0.80 and 0.107, still up to 1.11.)  Error against 64-bit
// results relative to the decode kernels', 162 calls: K from 3e-5 to 30 at V of order one 0.96 on average, 1.03 at most; V of 1e-4
// 0.96 and 1.00, V of 3e-5, where outputs are fp16 subnormals, 1.02 and 1.08; plain fp16 caches 1.00 to 1.01, bf16 1.00 to 1.02
// (s24_r3, where the codes are exact in fp16 and little but P is rounded, 1.30 to 1.45).
// What bounds it: overlap, no pipe is full.  By the counters (profiles/attn_prefill_kernel_instruction_counters.txt) a compute unit
// spends 44 % of its busy cycles in the matrix pipe, 49 % issuing vector instructions and 54 % in LDS, a quarter of that bank
// conflicts (plain, 1024 on 32768), at 2.0 to 2.1 GHz; with verbatim chunks 45, 63 and 34 %; 2048 on 2048 causal 23, 55 and 42 %.
#include "attention_mfma.h"
#include <algorithm>

namespace hqmq {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
typedef short short4v __attribute__((ext_vector_type(4)));

constexpr uint32_t kPfV = 16384, kPfBuf = 32768, kPfScale = 2 * kPfBuf, kPfScaleV = 1024, kPfFlag = kPfScale + 2048;   // LDS: K | V, twice; scales; flags (FL); tables
constexpr uint32_t pf_tab(bool fl) { return kPfFlag + (fl ? 1024u : 0u); }
// The codeword tables' places, and whether fp16 tables land in LDS, in whole KB, without passing through registers (not where a KB more each
// would not fit).  us, through registers and landing: unpacked 8 x 141 tokens, 28 / 4 heads, s192_r4, 20.1 / 19.0, 2 x 1024 heads of 64 s96_r4
// 46.8 / 45.8, 4 x 300 queries on 300 tokens s192_r4 24.6 / 23.3.
struct PfTables {
    uint32_t unit, end;         // V's table begins a whole number of units behind K's; the end of LDS
    bool land;
};
// (Worked out from K's size wherever it is needed, not kept: held as one number chosen between both units, the outlier variants of d_h 128 put nine
// registers more into scratch: 8 x 335 queries on 793 tokens s192_r6 107.2 us, worked out again 103.5; 8 x 214 on 298 s192_r4 36.7, 33.6.)
__host__ __device__ __forceinline__ uint32_t pf_behind(int kk, uint32_t unit) { return (8u * (uint32_t)kk + unit - 1u) & ~(unit - 1u); }
__host__ __device__ __forceinline__ PfTables pf_tables(int kk, int vk, bool fl, bool fp16) {
    const uint32_t tab = pf_tab(fl), whole = tab + pf_behind(kk, 1024u) + pf_behind(vk, 1024u);
    if (fp16 && whole <= 160u * 1024u) return PfTables{1024u, whole, true};
    return PfTables{128u, tab + pf_behind(kk, 128u) + 8u * (uint32_t)vk, false};
}

// permutation of a row's 16-byte parts
template <int DH>
__device__ __forceinline__ uint32_t pf_part(uint32_t t, uint32_t q) {
    if (DH == 128) return q ^ ((t & 3u) << 2 | ((t >> 2) & 3u));
    return q ^ (((t >> 1) & 1u) << 2 | ((t >> 2) & 3u));
}

#define PF_INLINE __attribute__((always_inline))

template <int DH, int MB, bool AUX, int DT, int KVG, bool FL>
__global__ __launch_bounds__(512, 2) void attn_prefill_kernel(AttnParams p, int gx, int rows) {
    constexpr int n = DH / 4, ROWB = DH * 2, CW = 8 / KVG, KS = DH / 16, DB = DH / 32;
    constexpr int TILE = 8192 / DH, NSUB = TILE / 32 / KVG;              // tokens per tile; units of 32 of them per wavefront
    constexpr int TOK = DH == 128 ? 16 : 32;                             // tokens a wavefront decodes: 8 chunks per lane
    constexpr uint32_t kPfTab = pf_tab(FL);
    extern __shared__ uint2 lds_tab[];
    touch_kernargs();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31;
    const int G = p.G, nz = p.B * p.Hkv;
    // block numbers: (sequence, KV head) fastest, then splits, then `rows` rows; row r takes the column blocks r, 2 rows - 1 - r,
    // 2 rows + r, ... counted from the last (the longest of a causal launch), so that all rows get about the same work
    const int r0 = (int)blockIdx.x / nz, bz = (int)blockIdx.x - r0 * nz;
    const int row0 = r0 / p.n_splits, sp = r0 % p.n_splits;
    const int slot = bz / p.Hkv, hkv = bz - slot * p.Hkv;
    const int b = p.batch_order ? min(max(uniform_word(p.batch_order, slot), 0), p.B - 1) : slot;
    const size_t plane_row0 = (size_t)(b * p.Hkv + hkv) * p.t_cap;
    const int cw = wave % CW, kvg = wave / CW;

    // ---- codeword tables as fp16: K, then V; every load is on its way before the first one is stored ----
    const uint2 *kj = (const uint2 *)p.Kc.joint + hkv * (p.Kc.jsh / 4), *vj = (const uint2 *)p.Vc.joint + hkv * (p.Vc.jsh / 4);
    const PfTables place = pf_tables(p.Kc.K, p.Vc.K, FL, DT == HQMQ_F16);
    const bool pairs = ((((uintptr_t)kj) | ((uintptr_t)vj)) & 15) == 0 && ((p.Kc.K | p.Vc.K) & 1) == 0, land = DT == HQMQ_F16 && place.land && pairs;
    // (requested first of all; the wait for them is behind the first tiles' requests)
    if (land) land_tables<8>(uniform_ptr((const uint8_t *)kj), 8u * (uint32_t)p.Kc.K, uniform_ptr((const uint8_t *)vj), 8u * (uint32_t)p.Vc.K, kPfTab, kPfTab + pf_behind(p.Kc.K, 1024u), wave, lane);
    auto tables = [&]() PF_INLINE {
        const int kk = p.Kc.K, vk = p.Vc.K;
        const uint32_t vt = kPfTab + pf_behind(kk, place.unit);
        if (land) {
            wait_vm<0>();
            return;
        }
        if (pairs) {
            // two codewords a load, all of 2 x 5120 of them in one round: in rounds of 5 x 512 codewords the tables of s192 took four trips
            // to memory (8 x 141 tokens, unpacked, s192_r4 25.4 -> 24.1 us; a chunk of 8 x 353 on 451 tokens, bf16, 55.5 -> 54.2)
            constexpr int U = 10;
            const int k2 = kk / 2, all = k2 + vk / 2;
            for (int k0 = tid; k0 < all; k0 += 512 * U) {
                uint4v w[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int k = min(k0 + 512 * u, all - 1);
                    w[u] = k < k2 ? reinterpret_cast<const uint4v *>(kj)[k] : reinterpret_cast<const uint4v *>(vj)[k - k2];
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int k = k0 + 512 * u;
                    if (k < all) *(uint4v __attribute__((address_space(3))) *)(uintptr_t)(k < k2 ? kPfTab + 16u * k : vt + 16u * (k - k2)) = pair_to_half<DT>(w[u]);
                }
            }
            return;
        }
        constexpr int U = 5;
        for (int k0 = tid; k0 < kk + vk; k0 += 512 * U) {
            uint2 w[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = min(k0 + 512 * u, kk + vk - 1);
                w[u] = k < kk ? kj[k] : vj[k - kk];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = k0 + 512 * u;
                if (k < kk + vk)
                    *(uint2v __attribute__((address_space(3))) *)(uintptr_t)(k < kk ? kPfTab + 8u * k : vt + 8u * (k - kk)) = __builtin_bit_cast(uint2v, chunk_to_half<DT>(w[u]));
            }
        }
    };
    for (int it = 0; it * rows < gx; it++) {
    const int pos = (it & 1) ? (it + 1) * rows - 1 - row0 : it * rows + row0;
    if (pos >= gx) continue;
    const int cb = gx - 1 - pos;
    // ---- this wavefront's columns and the block's KV range ----
    int kv_end = p.kv_len ? uniform_word(p.kv_len, b) : p.Tkv;
    kv_end = min(max(kv_end, 0), p.Tkv);
    const int cols = p.Tq * G, cidx = (cb * CW + cw) * 32 + col;
    const bool col_ok = cidx < cols;
    const int tq = col_ok ? cidx / G : 0, hq = hkv * G + (col_ok ? cidx - tq * G : 0);
    auto limit = [&](int q) PF_INLINE { return p.causal ? (int)max((int64_t)0, min((int64_t)kv_end, (int64_t)q + p.causal_offset + 1)) : kv_end; };
    const int col_lim = col_ok ? limit(tq) : 0;
    // columns are ordered by query token: the last real column of a range sees most, the first least
    const int first_c = (cb * CW + cw) * 32;
    const int wave_min = first_c + 31 < cols ? limit(first_c / G) : 0;
    const int blk_lim = limit((min((cb + 1) * CW * 32, cols) - 1) / G);
    const int col_start = p.kv_start ? min(max(uniform_word(p.kv_start, b), 0), blk_lim) : 0;
    const int blk_lo = col_start / TILE * TILE;
    int per_split = (blk_lim - blk_lo + p.n_splits - 1) / p.n_splits;
    per_split = (per_split + TILE - 1) / TILE * TILE;
    const int b_begin = min(blk_lo + sp * per_split, blk_lim), b_end = min(blk_lim, b_begin + per_split);
    const bool work = b_begin < b_end;

    // ---- decoding: wavefronts 0..3 take K, 4..7 take V; lane = token + TOK * (group of 8 chunks) ----
    const bool dec_v = wave >= 4;
    const int d_tok = (wave & 3) * TOK + lane % TOK, d_grp = lane / TOK;
    const PackedDev &dc = dec_v ? p.Vc : p.Kc;
    constexpr int NW = MB / 4;
    constexpr uint32_t mrb = n * MB / 8;
    const uint32_t ab = AUX ? p.aux_bits : 0, arb = n * ab / 8;
    const uint8_t *d_main = dc.main_plane + plane_row0 * mrb;
    const uint32_t *d_aux = AUX ? (const uint32_t *)(dc.aux_plane + plane_row0 * arb) : nullptr;
    const uint16_t *d_scale = (const uint16_t *)dc.scale_plane + b * dc.ssb + hkv * dc.ssh;
    const uint32_t idx_mask = (1u << p.idx_bits) - 1u;
    const int idx_bits = p.idx_bits;
    const uint32_t tab = kPfTab + (dec_v ? pf_behind(p.Kc.K, place.unit) : 0u);
    // Outlier caches (FL): a wavefront decodes whole 16-token tiles of the sideband (one at d_h 128, two at 64), so it also writes
    // their verbatim chunks, over the zeros that flagged chunks decode to.  Lane e takes entry e of the contiguous range that the tile
    // offsets name; the offsets (scalar loads) travel
    // a tile ahead of the entries, the entries from the start of a tile's products to the end of its decoding.
    constexpr int SBT = TOK / 16;
    const int bh = b * p.Hkv + hkv, sb_tiles = (int)(p.t_cap >> 4);
    const int32_t *sb_off = FL ? dc.sb_tile_off + (size_t)bh * sb_tiles : nullptr;
    const uint2 *sb_val = FL ? (const uint2 *)dc.sideband + (size_t)bh * dc.sb_cap : nullptr;
    const uint16_t *sb_xy = FL ? dc.sb_coord + (size_t)bh * dc.sb_cap : nullptr;
    const int sb_count = FL ? min(max(uniform_word(dc.sb_count, bh), 0), (int)dc.sb_cap) : 0;
    // LEAN: no registers are left over, and a spilled one that is read back in the loop waits for every request in flight
    constexpr bool LEAN = FL && AUX;
    auto lane_id = [&]() PF_INLINE {
        if (!LEAN) return lane;
        int id = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(id));
        return id;
    };
    int rg[SBT + 1];                                                      // of the tile whose entries are requested next
    auto offsets = [&](int t0) PF_INLINE {
        const int first = (t0 >> 4) + (wave & 3) * SBT;
#pragma unroll
        for (int i = 0; i <= SBT; i++) {
            const int o = uniform_word(sb_off, min(first + i, sb_tiles - 1));
            rg[i] = first + i < sb_tiles ? o : 0x7fffffff;              // tiles never written hold that, too: up to the count
        }
    };
    struct { uint2 val; uint32_t xy; int t0, from, mid, to; } ent;
    auto entries = [&](int t0) PF_INLINE {
        ent.t0 = t0;
        ent.from = min(max(rg[0], 0), sb_count);
        ent.to = max(ent.from, min(rg[SBT], sb_count));
        ent.mid = rg[SBT - 1];
        const int e = min(ent.from + lane_id(), (int)dc.sb_cap - 1);
        ent.val = sb_val[e];
        ent.xy = sb_xy[e];
        offsets(t0 + TILE);
    };
    // Entry e into LDS; those of rows past the range are dropped (their scores are masked, but 0 * inf is not 0).  K's are marked in
    // their token's flag word.
    auto patch = [&](int e, uint2 val, uint32_t xy, uint32_t buf) PF_INLINE {
        const uint32_t t = (uint32_t)(wave & 3) * TOK + ((xy >> 8) & 15u) + (SBT > 1 && e >= ent.mid ? 16u : 0u), ch = xy & (uint32_t)(n - 1);
        if (e < ent.to && ent.t0 + (int)t < b_end) {
            if (!dec_v) __hip_atomic_fetch_or((uint32_t __attribute__((address_space(3))) *)(uintptr_t)(kPfFlag + buf * 512u + 4u * t), 1u << ch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            *(uint2v __attribute__((address_space(3))) *)(uintptr_t)(buf * kPfBuf + (dec_v ? kPfV : 0u) + t * ROWB + (pf_part<DH>(t, ch >> 1) << 4) + (ch & 1u) * 8u) = __builtin_bit_cast(uint2v, val);
        }
    };
    struct Codes { uint32_t w[NW], aux, aux2, sh, scale; };
    auto request = [&](int t0, Codes &c) PF_INLINE {
        const uint32_t row = (uint32_t)min(t0 + d_tok, b_end - 1);        // rows past the range were perhaps never written
        const uint8_t *m = d_main + (row * mrb + (uint32_t)d_grp * MB);
        if (MB == 16) {
            const uint4 v = *reinterpret_cast<const uint4 *>(m);
            c.w[0] = v.x; c.w[1] = v.y; c.w[2] = v.z; c.w[NW - 1] = v.w;
        } else {
#pragma unroll
            for (int i = 0; i < NW; i++) c.w[i] = reinterpret_cast<const uint32_t *>(m)[i];
        }
        if (AUX) {                                                        // the dwords of the plane that hold the lane's bytes
            const uint32_t o = row * arb + (uint32_t)d_grp * ab;
            c.aux = d_aux[o >> 2];
            c.aux2 = d_aux[(o + ab - 1) >> 2];
            c.sh = o;
        }
        c.scale = d_scale[row];
    };
    // decoding goes in eight pieces, so that it can be spread between the matrix instructions: codewords requested (0, 1),
    // radii unpacked (2, 3), products stored (4 .. 7); in registers between them:
    half4 wg[8];
    half2v wr[4];
    float w_scale = 0.f, w_mul = 1.f;
    uint32_t w_at = (dec_v ? kPfV : 0u) + (uint32_t)d_tok * ROWB + (pf_part<DH>((uint32_t)d_tok, (uint32_t)(d_grp * 4)) << 4);
    uint32_t ws_at = kPfScale + (dec_v ? kPfScaleV : 0u) + 4u * (uint32_t)d_tok;
    const bool w_lane = d_grp == 0;
    auto piece = [&](int j, Codes &c) PF_INLINE {
        if (j == 0) {
#pragma unroll
            for (int i = 0; i < NW; i++) asm volatile("" : "+v"(c.w[i]));     // nothing of this moves up
        }
        if (j < 2) {
            const uint32_t aux = AUX ? __builtin_amdgcn_alignbyte(c.aux2, c.aux, c.sh) : 0u;
#pragma unroll
            for (int i = 4 * j; i < 4 * j + 4; i++) {
                if constexpr (MB == 16 && !AUX) {
                    wg[i] = __builtin_bit_cast(half4, *(lds_u2_ptr)(uintptr_t)(((i & 1 ? c.w[i / 2] >> 16 : c.w[i / 2]) & idx_mask) * 8u + tab));
                } else {
                    uint32_t code = code_at<MB, NW>(c.w, i);
                    if (AUX) code |= ((aux >> (i * ab)) & ((1u << ab) - 1u)) << MB;
                    wg[i] = __builtin_bit_cast(half4, *(lds_u2_ptr)(uintptr_t)((code & idx_mask) * 8u + tab));
                    wr[i >> 1][i & 1] = (_Float16)(uint16_t)(code >> idx_bits);
                }
            }
        } else if (j < 4) {
            if constexpr (MB == 16 && !AUX) {
                uint32_t rq2 = (0xffffu >> idx_bits) * 0x00010001u, magic = 0x64006400u;
                asm("" : "+s"(rq2));
                asm("" : "+v"(magic));
#pragma unroll
                for (int i = 2 * j - 4; i < 2 * j - 2; i++) {
                    const uint32_t t = ((c.w[i] >> idx_bits) & rq2) | magic;             // 0x6400 | rq = the fp16 number 1024 + rq
                    wr[i] = __builtin_bit_cast(half2v, t) - half2v{(_Float16)1024.0f, (_Float16)1024.0f};
                }
            }
            // K and V keep their radius codes; the token's scales are applied to the score and to P, in fp32.  (FL: V rows hold the
            // values themselves, rounded once, as its verbatim chunks are)
            if (j == 3) {
                w_scale = DT == HQMQ_F16 ? __half2float(__ushort_as_half((uint16_t)c.scale)) : __uint_as_float(c.scale << 16);
                if (FL) w_mul = dec_v ? w_scale * p.inv_qmax : 1.f;
            }
        } else {
            const int i = j - 4;
            if (FL) {                                                     // rounded once (K: codeword * radius code, as below)
                half8 v;
#pragma unroll
                for (int x = 0; x < 2; x++) {
                    const float r = (float)wr[i][x] * w_mul;
#pragma unroll
                    for (int y = 0; y < 4; y++) v[4 * x + y] = (_Float16)__builtin_fmaf((float)wg[2 * i + x][y], r, 0.f);
                }
                *(uint4v __attribute__((address_space(3))) *)(uintptr_t)(w_at ^ ((uint32_t)i << 4)) = __builtin_bit_cast(uint4v, v);
            } else *(uint4v __attribute__((address_space(3))) *)(uintptr_t)(w_at ^ ((uint32_t)i << 4)) =
                __builtin_bit_cast(uint4v, cat8(wg[2 * i] * wr[i][0], wg[2 * i + 1] * wr[i][1]));
            if (j == 7) {
                if (w_lane) *(float __attribute__((address_space(3))) *)(uintptr_t)ws_at = dec_v ? w_scale : w_scale * p.c_log2;
                if (FL) {
                    if (w_lane && !dec_v) *(uint32_t __attribute__((address_space(3))) *)(uintptr_t)(ws_at + (kPfFlag - kPfScale)) = 0u;
                    asm volatile("" ::: "memory");                        // the wavefront's LDS accesses keep their order
                    const uint32_t buf = w_at / kPfBuf;
                    const int first = ent.from + lane_id();
                    patch(first, ent.val, ent.xy, buf);
                    for (int e = first + 64; e < ent.to; e += 64) patch(e, sb_val[e], sb_xy[e], buf);
                }
                w_at ^= kPfBuf;
                ws_at ^= 512u;
            }
        }
    };
    // K runs one tile ahead of V: while tile i is multiplied, K of tile i + 2 and V of tile i + 1 are decoded
    // (in even steps from cc[0], in odd ones from cc[1], then the codes of the tile two further on are requested)
    Codes cc[2];
    if (work) {
        if (FL) {
            offsets(b_begin);
            entries(b_begin);
        }
        request(b_begin, cc[1]);
        request(b_begin + TILE, cc[0]);
    }
    int d_t = b_begin + (dec_v ? 3 : 4) * TILE;                           // the tile requested next

    // ---- query columns: the B operand of S^T, lane (col, half) holds d = 16 kk + 8 half .. + 7 ----
    half8 qf[KS];
    {
        const uint16_t *qp = (const uint16_t *)p.Q + b * p.qsb + hq * p.qsh + (int64_t)tq * p.qst + 8 * half;
        const bool wide_q = ((((uintptr_t)p.Q) | (uintptr_t)(p.qsb * 2) | (uintptr_t)(p.qsh * 2) | (uintptr_t)(p.qst * 2)) & 15) == 0;
#pragma unroll
        for (int kk = 0; kk < KS; kk++) {
            uint4v w;
            if (wide_q) w = *reinterpret_cast<const uint4v *>(qp + 16 * kk);
            else {
                const uint2 lo = *reinterpret_cast<const uint2 *>(qp + 16 * kk), hi = *reinterpret_cast<const uint2 *>(qp + 16 * kk + 4);
                w = uint4v{lo.x, lo.y, hi.x, hi.y};
            }
            qf[kk] = __builtin_bit_cast(half8, col_ok ? pair_to_half<DT>(w) : uint4v{0, 0, 0, 0});
        }
    }
    if (it == 0) tables();
    __syncthreads();
    if (work) {
#pragma unroll
        for (int j = 0; j < 8; j++) piece(j, cc[1]);
        request(b_begin + 2 * TILE, cc[1]);
        if (!dec_v) {
            if (FL) entries(b_begin + TILE);
#pragma unroll
            for (int j = 0; j < 8; j++) piece(j, cc[0]);
            cc[0] = cc[1];
            request(b_begin + 3 * TILE, cc[1]);
        }
    }
    __syncthreads();

    // ---- LDS addresses of the operands (tile buffer 0) ----
    uint32_t ka[KS], va[2][DB], ka0;
    const uint32_t wo = (uint32_t)kvg * (32u * NSUB * ROWB);              // this wavefront's share of a tile
#pragma unroll
    for (int kk = 0; kk < KS; kk++) ka[kk] = wo + (uint32_t)col * ROWB + (pf_part<DH>((uint32_t)col, (uint32_t)(2 * kk + half)) << 4);
#pragma unroll
    for (int hf = 0; hf < 2; hf++)
#pragma unroll
        for (int db = 0; db < DB; db++) {
            // lane i of a group of 16 reads token row i / 4, d part i % 4; afterwards it holds d = i of the four rows
            const uint32_t i = lane & 15, t = (uint32_t)(8 * hf + 4 * half) + (i >> 2);
            const uint32_t q = (uint32_t)(4 * db + 2 * ((lane >> 4) & 1)) + ((i & 3) >> 1);
            va[hf][db] = wo + kPfV + t * ROWB + (pf_part<DH>(t, q) << 4) + (i & 1) * 8u;
        }
    ka0 = ka[0];                                                          // the parts of a row differ by an exclusive-or
    const uint32_t sa = kPfScale + 16u * (uint32_t)half + 128u * NSUB * (uint32_t)kvg;
    const uint32_t fa = kPfFlag + 4u * (uint32_t)col + 128u * NSUB * (uint32_t)kvg;

    // exponents are in base 2: s becomes score * scale - (running maximum); seen is -inf until a column has met a token, then 0
    float neg_m = 0.f, seen = -INFINITY, l_run = 0.f;
    float16v acc[DB], s;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[db][e] = 0.f;

    // sub-unit u of the tile in buffer buf, u == NSUB: the first one of the next tile
    constexpr int AHEAD = FL ? 2 : 4;                                     // (FL: a step takes twice as long, and registers are short)
    auto k_load = [&](uint32_t buf, int u, int kk) PF_INLINE {
        const uint32_t at = ((u == NSUB ? buf ^ 1u : buf) * kPfBuf + (uint32_t)(u % NSUB) * (32u * ROWB)) / 16;
        return __builtin_bit_cast(half8, ((lds_u4_ptr)(uintptr_t)(LEAN ? ka0 ^ ((uint32_t)kk << 5) : ka[kk]))[at]);
    };
    auto v_load = [&](uint32_t buf, int u, int i) PF_INLINE {             // operand i: tokens 16 (i / DB) .. + 15, d block i % DB
        typedef short4v __attribute__((address_space(3))) *lds_s4;
        const uint32_t at = (buf * kPfBuf + (uint32_t)u * (32u * ROWB) + 16u * ROWB * (uint32_t)(i / DB)) / 8;
        const half4 v0 = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(uintptr_t)va[0][i % DB] + at));
        const half4 v1 = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(uintptr_t)va[1][i % DB] + at));
        return cat8(v0, v1);
    };
    auto s_load = [&](uint32_t buf, int u, int i) PF_INLINE {             // K scales of tokens 8 i + 4 half .. + 3
        const uint32_t at = ((u == NSUB ? buf ^ 1u : buf) * 512u + 128u * (uint32_t)(u % NSUB) + 32u * i) / 16;
        return __builtin_bit_cast(float4v, ((lds_u4_ptr)(uintptr_t)sa)[at]);
    };
    auto vs_load = [&](uint32_t buf, int u, int i) PF_INLINE {            // V scales of the same tokens
        const uint32_t at = (kPfScaleV + buf * 512u + 128u * (uint32_t)u + 32u * i) / 16;
        return __builtin_bit_cast(float4v, ((lds_u4_ptr)(uintptr_t)sa)[at]);
    };
    // FL: the flags of the lane's K row, shifted to the chunks the lane holds
    auto f_load = [&](uint32_t buf, int u) PF_INLINE {
        const uint32_t at = ((u == NSUB ? buf ^ 1u : buf) * 512u + 128u * (uint32_t)(u % NSUB)) / 4;
        return ((const uint32_t __attribute__((address_space(3))) *)(uintptr_t)fa)[at] >> (2 * half);
    };
    // One step of the scores.  FL: flagged chunks hold their verbatim values, the others codeword * radius code; the operand is
    // split by chunk, and the two sums meet in maxima, the token's scale on the second.
    auto score_step = [&](half8 k8, int kk, uint32_t flags, float16v &sn, float16v &svn) PF_INLINE {
        if (FL) {
            const uint4v w = __builtin_bit_cast(uint4v, k8);
            const uint32_t m0 = (uint32_t)__builtin_amdgcn_sbfe((int)flags, 4 * kk, 1), m1 = (uint32_t)__builtin_amdgcn_sbfe((int)flags, 4 * kk + 1, 1);
            const uint4v verb = uint4v{w[0] & m0, w[1] & m0, w[2] & m1, w[3] & m1};
            const uint4v code = uint4v{w[0] & ~m0, w[1] & ~m0, w[2] & ~m1, w[3] & ~m1};
            sn = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, code), qf[kk], sn, 0, 0, 0);
            svn = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, verb), qf[kk], svn, 0, 0, 0);
        } else sn = __builtin_amdgcn_mfma_f32_32x32x16_f16(k8, qf[kk], sn, 0, 0, 0);
    };
    // FL: rows 8 x + 4 half .. + 3 of a unit's scores, relative to the running maximum: the codes' part times the token's scale
    auto join = [&](int x, float16v &sn, const float16v &svn, float4v ks) PF_INLINE {
#pragma unroll
        for (int e = 4 * x; e < 4 * x + 4; e++) sn[e] = __builtin_fmaf(sn[e], ks[e & 3], __builtin_fmaf(svn[e], p.c_plain, neg_m));
    };
    // scores of a unit (first token tw): times their K scale, relative to the running maximum, which moves if it has to
    auto maxima = [&](int tw, const float4v (&ks)[4]) PF_INLINE {
        const bool edge = !(tw + 32 <= wave_min && tw + 32 <= b_end && tw >= col_start);
        float tmax = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16 && !FL; e++) s[e] = __builtin_fmaf(s[e], ks[e >> 2][e & 3], neg_m);
        if (edge) {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int t = tw + 8 * (e >> 2) + 4 * half + (e & 3);
                if (!(t < col_lim && t < b_end && t >= col_start)) s[e] = -INFINITY;
            }
        }
#pragma unroll
        for (int e = 0; e < 16; e++) tmax = fmaxf(tmax, s[e]);
        // The halves of a column meet only where one of them exceeds it (they hold the same `seen`): most units move no maximum.  Met in every
        // unit, us: 1024 on 32768 615 (611), on 16384 with heads of 64 383.7 (379.5), 512 on 16384 with verbatim chunks 266.6 (263.9).
        if (__builtin_amdgcn_ballot_w64(tmax > seen) != 0) {
            const uint32_t x = __float_as_uint(tmax);
            const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
            tmax = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
            const float d = tmax > seen ? tmax : 0.f;
            const float alpha = seen == 0.f ? __builtin_amdgcn_exp2f(-d) : 0.f;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[db][e] *= alpha;
#pragma unroll
            for (int e = 0; e < 16; e++) s[e] -= d;
            neg_m -= d;
            seen = tmax > seen ? 0.f : seen;
        }
    };
    // One unit of 32 tokens.  In program order, one matrix instruction at a time with vector work behind it:
    //   S^T of the next unit, with the exponentials of this one; O^T += V^T . P^T of this one, with the decoding.
    half8 kf[AHEAD];                                                      // operands of the next unit's first products
    uint32_t kfl = 0u;                                                    // and its flags
    auto unit = [&](int tw, uint32_t buf, int u) PF_INLINE {
        if (LEAN) asm volatile("" : "+v"(ka0));                         // (or all eight addresses would be kept)
        constexpr int NV = 2 * DB, PER = 8 / KS;               // pairs of exponentials per matrix instruction
        const bool dec = u == NSUB - 1;
        half8 vf[AHEAD];
        float4v ks[4], vs[4];
        float16v sn, svn;
        float pe[2 * PER];
        uint32_t pp[8];
        if (FL && u == 0) entries(d_t - 2 * TILE);                        // of the tile decoded next
#pragma unroll
        for (int e = 0; e < 16; e++) sn[e] = svn[e] = 0.f;
        if (!FL) vs[0] = vs_load(buf, u, 0);
        auto finish = [&](int k) PF_INLINE {                              // the exponentials of step k: summed, times V's scale, packed
#pragma unroll
            for (int x = 0; x < PER; x++) {
                const int i = k * PER + x;
                l_run += pe[2 * x] + pe[2 * x + 1];
                const float v0 = FL ? 1.f : vs[i >> 1][2 * i & 3], v1 = FL ? 1.f : vs[i >> 1][(2 * i & 3) + 1];
                pp[i] = __builtin_bit_cast(uint32_t, half2v{(_Float16)(FL ? pe[2 * x] : pe[2 * x] * v0), (_Float16)(FL ? pe[2 * x + 1] : pe[2 * x + 1] * v1)});
            }
        };
#pragma unroll
        for (int k = 0; k < KS; k++) {
            __builtin_amdgcn_sched_barrier(0);
            score_step(kf[k % AHEAD], k, kfl, sn, svn);
            if (k + AHEAD < KS) kf[k % AHEAD] = k_load(buf, u + 1, k + AHEAD);
            else vf[k + AHEAD - KS] = v_load(buf, u, k + AHEAD - KS);
            if (k > 0) finish(k - 1);
            if (!FL && (2 * PER * (k + 1)) % 4 == 0 && k + 1 < KS) vs[PER * (k + 1) / 2] = vs_load(buf, u, PER * (k + 1) / 2);
#pragma unroll
            for (int x = 0; x < 2 * PER; x++) pe[x] = __builtin_amdgcn_exp2f(s[2 * PER * k + x]);
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            if (FL && i == 0 && NV / 2 - 2 == 0) ks[0] = s_load(buf, u + 1, 0);
            if (i == 0) finish(KS - 1);
            if (i > 0) __builtin_amdgcn_sched_barrier(0);
            const int st = i / DB, db = i % DB;
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i % AHEAD], __builtin_bit_cast(half8, uint4v{pp[4 * st], pp[4 * st + 1], pp[4 * st + 2], pp[4 * st + 3]}), acc[db], 0, 0, 0);
            if (i + AHEAD < NV) vf[i % AHEAD] = v_load(buf, u, i + AHEAD);
            if (dec) {
#pragma unroll
                for (int j = i * 8 / NV; j < (i + 1) * 8 / NV; j++) piece(j, cc[buf]);
                if (i * 8 / NV <= 3 && (i + 1) * 8 / NV > 3) {
                    request(d_t, cc[buf]);
                    d_t += TILE;
                }
            }
            if (FL) {                                                     // in registers no longer than needed
                constexpr int J0 = NV / 2 - 2;
                if (i >= J0 && i < J0 + 4) join(i - J0, sn, svn, ks[i - J0]);
                if (i + 1 >= J0 && i + 1 < J0 + 4) ks[i + 1 - J0] = s_load(buf, u + 1, i + 1 - J0);
            } else if (i == NV / 2) {
#pragma unroll
                for (int x = 0; x < 4; x++) ks[x] = s_load(buf, u + 1, x);
            }
        }
        s = sn;
        if (dec) __syncthreads();
        const bool over = u + 1 == NSUB;                                  // the next unit is the first one of the next tile
#pragma unroll
        for (int i = 0; i < AHEAD; i++) kf[i] = k_load(over ? buf ^ 1u : buf, over ? 1 : u + 2, i);
        if (FL) kfl = f_load(over ? buf ^ 1u : buf, over ? 1 : u + 2);
        maxima(over ? tw + 32 + TILE - 32 * NSUB : tw + 32, ks);
    };
    auto tile = [&](int t0, uint32_t buf) PF_INLINE {
#pragma unroll
        for (int u = 0; u < NSUB; u++) {
            if (NSUB > 1 && u == NSUB - 1) __syncthreads();               // K of this tile is read no more: its buffer is next
            unit(t0 + 32 * (NSUB * kvg + u), buf, u);
        }
    };
    if (work) {
        float4v ks[4];
#pragma unroll
        for (int x = 0; x < 4; x++) ks[x] = s_load(0u, 0, x);
        float16v sv0;
        const uint32_t fl0 = FL ? f_load(0u, 0) : 0u;
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] = sv0[e] = 0.f;
#pragma unroll
        for (int kk = 0; kk < KS; kk++) score_step(k_load(0u, 0, kk), kk, fl0, s, sv0);
#pragma unroll
        for (int x = 0; x < 4 && FL; x++) join(x, s, sv0, ks[x]);
#pragma unroll
        for (int i = 0; i < AHEAD; i++) kf[i] = k_load(0u, 1, i);
        if (FL) kfl = f_load(0u, 1);
        maxima(b_begin + 32 * NSUB * kvg, ks);
    }
    // (a wavefront whose columns end before the block's goes on with masked scores: it has to decode anyway)
    for (int t0 = b_begin; t0 < b_end;) {
        tile(t0, 0u);
        t0 += TILE;
        if (t0 >= b_end) break;
        tile(t0, 1u);
        t0 += TILE;
    }

    // ---- epilogue: lane (col, half) holds d = 32 db + 8 i + 4 half + j of its column ----
    {
        const uint32_t x = __float_as_uint(l_run);
        const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        l_run = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    float m_run = seen == 0.f ? -neg_m : -INFINITY;
    if (KVG == 2) {
        // the wavefronts of tokens 32..63 hand their part over: [wave][element][lane], then m and l
        float *red = reinterpret_cast<float *>(lds_tab) + cw * (DB * 16 * 64);
        float *ml = reinterpret_cast<float *>((unsigned char *)lds_tab + kPfScale) + cw * 128;
        if (kvg == 1) {
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int e = 0; e < 16; e++) red[(db * 16 + e) * 64 + lane] = acc[db][e];
            ml[lane] = m_run;
            ml[64 + lane] = l_run;
        }
        __syncthreads();
        if (kvg == 0) {
        const float m1 = ml[lane], l1 = ml[64 + lane], m = fmaxf(m_run, m1);
        const float f0 = m > -INFINITY ? __builtin_amdgcn_exp2f(m_run - m) : 0.f, f1 = m > -INFINITY ? __builtin_amdgcn_exp2f(m1 - m) : 0.f;
        l_run = fmaf(l1, f1, l_run * f0);
        m_run = m;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[db][e] = fmaf(red[(db * 16 + e) * 64 + lane], f1, acc[db][e] * f0);
        }
    }
    if (!col_ok || (KVG == 2 && kvg == 1)) {
    } else if (p.n_splits == 1) {
        const float f = l_run > 0.f ? (FL ? 1.f : p.inv_qmax) / l_run : 0.f;
        const bool wide_out = ((((uintptr_t)p.O) | (uintptr_t)(p.osb * 2) | (uintptr_t)(p.osh * 2) | (uintptr_t)(p.ost * 2)) & 15) == 0;
        uint16_t *o = (uint16_t *)p.O + b * p.osb + hq * p.osh + (int64_t)tq * p.ost;
        // Two quarters at a time: the halves of a column exchange four dims, so that each lane stores eight in a row, in one piece
        // where the rows are aligned to it (as the queries are loaded).  With 8-byte accesses both ways a block started and ended
        // slower: unpacked 8 x 118 tokens s192_r6 20.9 -> 18.0 us, 2048 x 2048 87.5 -> 81.6 (kernel and packing, replayed in a
        // graph), a chunk of 8 x 353 queries on 451 tokens 55.6 -> 49.3.
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                uint32_t w[2][2];
#pragma unroll
                for (int k = 0; k < 2; k++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const float v0 = acc[db][4 * (i + k) + 2 * j] * f, v1 = acc[db][4 * (i + k) + 2 * j + 1] * f;
                        w[k][j] = DT == HQMQ_F16 ? (uint32_t)__half_as_ushort(__float2half_rn(v0)) | (uint32_t)__half_as_ushort(__float2half_rn(v1)) << 16
                                                 : (uint32_t)f32_to_bf16_bits(v0) | (uint32_t)f32_to_bf16_bits(v1) << 16;
                    }
                const auto x = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false), y = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
                if (wide_out) *reinterpret_cast<uint4 *>(o + 32 * db + 8 * (i + half)) = uint4{x[0], y[0], x[1], y[1]};
                else {
                    *reinterpret_cast<uint2 *>(o + 32 * db + 8 * (i + half)) = uint2{x[0], y[0]};
                    *reinterpret_cast<uint2 *>(o + 32 * db + 8 * (i + half) + 4) = uint2{x[1], y[1]};
                }
            }
    } else {
        float *wp = p.ws + ((((size_t)b * p.Hq + hq) * p.Tq + tq) * p.n_splits + sp) * (size_t)(DH + kPartialHead);
        if (half == 0) { wp[0] = m_run; wp[1] = l_run; }
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float4v v;
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = FL ? acc[db][4 * i + j] : acc[db][4 * i + j] * p.inv_qmax;
                *reinterpret_cast<float4v *>(wp + kPartialHead + 32 * db + 8 * i + 4 * half) = v;
            }
    }
    __syncthreads();
    }
}

// Launch plan, from times in us fitted to 100 chunks of 64 and more columns, every number of splits and both widths of block: a tile takes
// a block of 128 columns / of 256 columns, starting (tables, first tiles) and finishing take a block; a compute unit holds one block;
// partials are written and merged at 3.2 TB/s.  The plan takes 0.8 % longer than the best one (14 % at worst).  With one set for both
// head sizes (1.37 / 2.7, over outlier caches 1.75 / 3.5, 12 and 2 TB/s) blocks of 256 columns were taken too seldom and splits too: 3.4 %
// (37 %); 1024 queries on 16384 tokens, 32 / 8 heads of 128, fp16 s96_r4 369 us in blocks of 128 columns, 342 in two splits of 256;
// heads of 64 448 / 390; with 2 % of the K chunks verbatim 483 / 415.
struct PfTimes {
    double narrow, wide, start, merge, rate;
};
static PfTimes pf_times(int d_h, bool flags) {
    if (flags) return d_h == 64 ? PfTimes{2.75, 4.7, 11.0, 2.0, 3.2e6} : PfTimes{2.4, 3.1, 13.0, 2.0, 3.2e6};
    return d_h == 64 ? PfTimes{2.25, 3.5, 9.0, 2.0, 3.2e6} : PfTimes{1.5, 2.65, 11.0, 2.0, 3.2e6};
}
struct PfPlan {
    bool wide;
    int splits;
    double us;
};
static PfPlan pf_plan(int64_t cols, int64_t nz, int Tq, int Tkv, int d_h, int causal, int64_t off, int fixed_splits, const PfTimes &times) {
    const double last = causal ? std::max(1.0, std::min((double)Tkv, (double)off + Tq)) : std::max(Tkv, 1);      // tokens the last query sees
    const double mean = causal ? std::min(1.0, std::max(0.5, ((double)off + 0.5 * Tq) / last)) : 1.0;            // all, relative to it
    const int tiles = (int)((last * d_h + 8191) / 8192);
    PfPlan best{false, 1, 1e30};
    static const int kSplits[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 16, 20, 24, 32};
    for (int i = 0; i < (fixed_splits > 0 ? 1 : (int)(sizeof(kSplits) / sizeof(int))); i++) {
        const int s = fixed_splits > 0 ? fixed_splits : kSplits[i];
        if (i > 0 && s > tiles / 2) break;
        for (int wide = 0; wide < 2; wide++) {
            const double rounds = (double)(((cols + (wide ? 255 : 127)) / (wide ? 256 : 128) * nz * s + 255) / 256);
            // the longest block or a compute unit's share of all of them, whichever is more
            const double us = std::max(1.0, mean * rounds) * ((tiles + s - 1) / s) * (wide ? times.wide : times.narrow) + times.start * rounds +
                              (s > 1 ? times.merge + (double)(cols * nz) * s * (d_h + 4) * 8 / times.rate : 0.0);
            if (us < best.us) best = PfPlan{wide != 0, s, us};
        }
    }
    return best;
}
// Whether these kernels can take the call at all.
static bool attn_prefill_takes(const hqmq_attn_args *a) {
    if ((a->dtype != HQMQ_F16 && a->dtype != HQMQ_BF16) || a->wide_range || (a->n_chunks != 16 && a->n_chunks != 32) ||
        a->fp8_table_storage || (a->force_generic && a->force_generic != 3) || a->softmax_scale <= 0.f)
        return false;
    if (a->main_bits != 16 && (a->main_bits != 12 || a->aux_bits < 1)) return false;
    if (a->idx_bits < 6 || a->aux_bits > 4) return false;                          // the 16-bit decode needs radius codes below 1024
    if (a->t_cap % 64 || a->t_cap >= (1 << 25)) return false;                      // rows are addressed by 32-bit offsets
    if (pf_tab(a->K.flag_plane || a->V.flag_plane) + ((size_t)a->K.K + a->V.K) * 8 + 128 > 160 * 1024) return false;
    if (a->K.flag_plane || a->V.flag_plane) {
        if (a->dtype != HQMQ_F16) return false;                                   // verbatim bf16 chunks need not fit fp16
        const hqmq_packed *kv[2] = {&a->K, &a->V};
        for (const hqmq_packed *t : kv)
            if (!t->flag_plane || !t->sideband || !t->sb_coord || !t->sb_count || !t->sb_tile_off || t->sb_cap < 1 || t->sb_cap >= (1 << 28) || ((uintptr_t)t->sideband & 7))
                return false;
    }
    if (a->aux_bits && (((uintptr_t)a->K.aux_plane | (uintptr_t)a->V.aux_plane) & 3)) return false;
    if ((((uintptr_t)a->O) | (uintptr_t)(a->o_sb * 2) | (uintptr_t)(a->o_sh * 2) | (uintptr_t)(a->o_st * 2)) & 7) return false;
    return true;
}
// The same for the kernels of attention_fast.hip: blocks of 16 columns or of 32 (attn_two_groups; over outlier caches always of 16), fitted
// to the same and 100 more chunks: 4 to 11 % off on average.
struct FastTimes {
    double base, start, two, one, merge, rate;
};
static FastTimes fast_times(int d_h, bool flags) {
    if (d_h == 64) return FastTimes{2.1, flags ? 4.3 : 4.7, 0.68, flags ? 0.6 : 0.41, 1.5, 1.95e6};
    return FastTimes{2.1, flags ? 5.3 : 6.4, 0.5, flags ? 0.5 : 0.27, 1.5, 1.95e6};
}
static double fast_us(const hqmq_attn_args *a, int64_t cols, int splits, const FastTimes &times) {
    const int64_t nz = (int64_t)a->B * a->H_kv, cg = (cols + 15) / 16, pairs = (cg + 1) / 2 * nz * splits;
    const int d_h = 4 * a->n_chunks;
    const bool flags = a->K.flag_plane != nullptr, two = attn_two_groups((int)cg, flags, cg * nz * splits, a->T_kv / splits, a->n_chunks, a->aux_bits);
    const double tiles = ((double)a->T_kv * d_h + 8191) / 8192;
    return times.base + (double)(((two ? pairs : cg * nz * splits) + 255) / 256) * (times.start + tiles / splits * (two ? times.two : times.one)) +
           (splits > 1 ? times.merge + (double)(cols * nz) * splits * (d_h + 4) * 8 / times.rate : 0.0);
}
// The number of splits of a call that leaves it open, 0 if it is better off with the other kernels; splits > 0: the same decision for
// a given number.  Both estimates are of the plan that would run, the other kernels' with the splits of attn_decode_splits.  us, and with the
// kernel chosen by numbers of splits that would not run: 1 x 33 queries on 19403 tokens, 32 / 8 heads of 128, s24_r3, 37.8 (prefill
// kernel 47.2); 3 x 70 on 5811, 28 / 4, s192_r4, 50.8 (decode kernels 62.9).
// fp16 caches have a line of their own, from times of an earlier state of both kernels: the kernels differ in their error, and a line that
// follows the times moves calls to the less precise one.  Prefill kernel against decode kernels, error against 64 bits, 420 chunks near the line:
// over outlier caches 0.82 to 0.84 where K's verbatim chunks are large (heads of 128, 2 % of them 50 to 200 times the others), 1.01 to 1.03 on
// normal and lognormal channels, so a call changes kernel in neither direction; over plain fp16 caches 1.00 to 1.02, so it comes here
// only where both lines say so; bf16 at most 1.002.  What that costs against the present times for all of them: 10 % of the fp16 chunks over outlier
// caches take 1.09 of the time (0.86 to 1.52; 8 x 33 queries on 437 tokens, 28 / 4 heads, s192_r4, 30.6 us for 22.4), 2 % of those over
// plain caches 1.06.
int attn_prefill_splits(const hqmq_attn_args *a, int splits) {
    const int64_t cols = (int64_t)a->T_q * (a->H_q / a->H_kv), nz = (int64_t)a->B * a->H_kv;
    if (cols < 64 || !attn_prefill_takes(a)) return 0;
    const int d_h = 4 * a->n_chunks;
    const bool flags = a->K.flag_plane != nullptr;
    auto plan_of = [&](const PfTimes &times) { return pf_plan(cols, nz, a->T_q, a->T_kv, d_h, a->causal, a->causal_offset, splits, times); };
    const PfPlan plan = plan_of(pf_times(d_h, flags));
    if (a->force_generic == 3) return plan.splits;
    // Outlier caches of three radius bits keep the decode kernels: most radius codes are 1, 2 or 4, with which those kernels' V is
    // exact, and V rounded as a value left lognormal channels 0.5 % further from 64-bit results (s24_r3; 6 % nearer on average).  Plain
    // bf16 caches of three radius bits may come here: rounding the output to bf16 leaves 0.05 % of that on average, 0.16 % at most (72 chunks).
    if (flags && a->qmax < 15) return 0;
    const int other = splits > 0 ? splits : attn_decode_splits(a);
    if (a->dtype == HQMQ_F16) {
        const PfTimes then{flags ? 1.75 : 1.37, flags ? 3.5 : 2.7, 12.0, 5.0, 2e6};
        const FastTimes fast_then{3.0, 6.0, 0.6, flags ? 0.7 : 0.47, 3.0, 2e6};
        if (plan_of(then).us >= 0.95 * fast_us(a, cols, other, fast_then)) return 0;
        if (flags) return plan.splits;
    }
    return plan.us < fast_us(a, cols, other, fast_times(d_h, flags)) ? plan.splits : 0;
}

template <int DH, int MB, bool AUX, int DT, bool FL>
static int launch_pf(const AttnParams &p, hipStream_t st, const LaunchTiming &tm) {
    const int64_t cols = (int64_t)p.Tq * p.G, nz = (int64_t)p.B * p.Hkv * p.n_splits;
    const bool wide = pf_plan(cols, (int64_t)p.B * p.Hkv, p.Tq, p.Tkv, DH, p.causal, p.causal_offset, p.n_splits, pf_times(DH, FL)).wide;
    const int64_t gx = (cols + (wide ? 255 : 127)) / (wide ? 256 : 128);
    // Column blocks per block, one after the other (the tables stay in LDS): as few rounds of 256 blocks as possible.  Ragged
    // batches leave the choice of the next block to the hardware.
    int64_t rows = gx;
    if (!p.kv_len && !p.kv_start) {
        int64_t best = (gx * nz + 255) / 256;
        for (int64_t per = 2; per <= gx && per <= 64; per++) {
            const int64_t r = (gx + per - 1) / per, rounds = (r * nz + 255) / 256 * per;
            if (rounds <= best) { best = rounds; rows = r; }
        }
    }
    if (rows * nz > 0x7fffffff) return HQMQ_ERR_SHAPE;
    const size_t shmem = pf_tables(p.Kc.K, p.Vc.K, FL, DT == HQMQ_F16).end;
    auto kern = wide ? attn_prefill_kernel<DH, MB, AUX, DT, 1, FL> : attn_prefill_kernel<DH, MB, AUX, DT, 2, FL>;
    const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
    if (e != hipSuccess) return (int)e;
    const dim3 grid((unsigned)(rows * nz));
    if (tm.start || tm.stop) hipExtLaunchKernelGGL(kern, grid, dim3(512), shmem, st, tm.start, tm.stop, 0, p, (int)gx, (int)rows);
    else hipLaunchKernelGGL(kern, grid, dim3(512), shmem, st, p, (int)gx, (int)rows);
    return hip_status(hipGetLastError());
}

template <int DH, int DT, bool FL>
static int launch_pf_layout(const AttnParams &p, int mb, hipStream_t st, const LaunchTiming &tm) {
    if (mb == 16 && p.aux_bits == 0) return launch_pf<DH, 16, false, DT, FL>(p, st, tm);
    return mb == 16 ? launch_pf<DH, 16, true, DT, FL>(p, st, tm) : launch_pf<DH, 12, true, DT, FL>(p, st, tm);
}
template <int DH>
static int launch_pf_type(const AttnParams &p, int mb, bool flags, hipStream_t st, const LaunchTiming &tm) {
    if (flags) return launch_pf_layout<DH, HQMQ_F16, true>(p, mb, st, tm);
    return p.dtype == HQMQ_F16 ? launch_pf_layout<DH, HQMQ_F16, false>(p, mb, st, tm) : launch_pf_layout<DH, HQMQ_BF16, false>(p, mb, st, tm);
}

int launch_attn_prefill(const AttnParams &p, int mb, bool flags, hipStream_t st, const LaunchTiming &tm) {
    return p.n == 32 ? launch_pf_type<128>(p, mb, flags, st, tm) : launch_pf_type<64>(p, mb, flags, st, tm);
}

}  // namespace hqmq
