// Attention kernels specialised at compile time for the layouts of the benchmark shapes:
// d_h = 64 / 128, fp16 or bf16 caches, codes of 16+0 (s96_r4), 12+1 (s24_r3) or 16+3 (s192_r6) bits, and with a generic field decode
// of 16+1, 16+2, 12+2 or 12+3.
//
// Lane mapping (one wavefront, one 16-token tile): lane = 16 * grp + col decodes the CPL = d_h / 16 chunks
// grp * CPL ... of token `col` of K.
//   S^T = K . Q^T     v_mfma_f32_16x16x32_f16: A = two decoded K chunks of the lane, B = the matching Q chunks.
//   V^T               the A operand of O^T = V^T . P^T needs 4 tokens of one d per lane, a codeword is 4 d of one token: the
//                     codewords and radius codes are gathered from LDS by transposing reads (gather_tokens), for which lane
//                     4 * token + part holds the codes of a quarter of its token's chunks.  Float8 tables: lanes as for K,
//                     transposed by one v_mfma_f32_16x16x16_f16 against the identity (exact: every output is one fp16 input
//                     times 1.0) and two packed conversions per chunk.
//   O^T += V^T . P^T  v_mfma_f32_16x16x32_f16 over two tiles (32 tokens) at a time.
// P times the token's V scale is an fp32 product rounded to fp16 once, as in the other attention kernels; so is qmax P, the weight of
// verbatim chunks.  Row j of the V-side product is d = (grp * CPL + j) * 4 + e, the order the epilogue writes back.
// Scores are kept as S^T * rs; 1/qmax is folded into the softmax scale and the epilogue.  Outlier chunks
// carry radius code 0 in the planes, so they decode to zero; their verbatim values, found through the sideband entry list (values +
// coordinates, never the flag plane), enter through products of their own.
#include "attention_mfma.h"
#include <cstdlib>

namespace hqmq {

// Time stamps inside the kernels: measurement builds only (-DHQMQ_STAMPS, libhqmq_amd_stamps.so)
#ifdef HQMQ_STAMPS
__device__ unsigned long long *g_stamps;
#define STAMP(i) do { st_[i] = __builtin_amdgcn_s_memrealtime(); } while (0)
#else
#define STAMP(i) do { } while (0)
#endif
#if defined(HQMQ_STAMPS) && HQMQ_STAMPS + 0 >= 2     // -DHQMQ_STAMPS=2: time per phase of the outlier variants' half-steps (the stamps cost time themselves)
#define PHASE(i) do { if constexpr (FLAGS) { const unsigned long long t_ = __builtin_amdgcn_s_memrealtime(); ph_[i] += t_ - tl_; tl_ = t_; } } while (0)
#else
#define PHASE(i) do { } while (0)
#endif

// One codeword (four fp16 in two dwords) of e4m3 numbers -> four float8 bytes (exact)
__device__ __forceinline__ uint32_t codeword_to_f8(uint32_t w0, uint32_t w1) {
    const half2v a = __builtin_bit_cast(half2v, w0), b = __builtin_bit_cast(half2v, w1);
    int v = __builtin_amdgcn_cvt_pk_fp8_f32((float)a[0], (float)a[1], 0, false);
    v = __builtin_amdgcn_cvt_pk_fp8_f32((float)b[0], (float)b[1], v, true);
    return (uint32_t)v;
}
// Two codewords of a table whose entries are e4m3 numbers -> the same two as eight float8 bytes
template <int DT>
__device__ __forceinline__ uint2 pair_to_f8(uint4v w) {
    const uint4v h = pair_to_half<DT>(w);
    const uint32_t h0 = h[0], h1 = h[1], h2 = h[2], h3 = h[3];
    return uint2{codeword_to_f8(h0, h1), codeword_to_f8(h2, h3)};
}
template <int DT, bool F8>
__device__ __forceinline__ void store_pair(void *tab, int k, uint4v w) {
    if constexpr (F8) reinterpret_cast<uint2 *>(tab)[k] = pair_to_f8<DT>(w);
    else reinterpret_cast<uint4v *>(tab)[k] = pair_to_half<DT>(w);
}

// The same wave-uniform address, known to be one: added to a lane's offset the compiler would otherwise keep row + offset of every plane, six
// 64-bit addresses per lane.  As scalar base + 32-bit offset the plain variants take fewer registers: at twelve wavefronts s24_r3 in fp16
// reloaded V's address from scratch once a round, behind a wait for every load in flight (32 x 8000 tokens, 32 / 8 heads of 128, whole call
// 53.8 -> 49.9 us; 4500 tokens 34.1 -> 32.0).
template <bool ON, class T>
__device__ __forceinline__ const T *scalar_base(const T *p) {
    auto g = (const __attribute__((address_space(1))) T *)p;       // (a generic address out of an asm block would be read by flat loads)
    if constexpr (ON) asm("" : "+s"(g));
    return (const T *)g;
}

constexpr int kFastWaves = 8;     // wavefronts per block; 12 (three per SIMD) with long ranges per block, see launch_layout

// codes, aux bits and raw 16-bit scales of 32 tokens (two 16-token tiles) for one lane
template <int NW, int AB, bool FLAGS>
struct HalfTile {
    uint32_t kw[2][NW], vw[2][NW];
    uint32_t kaux[AB ? 2 : 1], vaux[AB ? 2 : 1];
    uint2 ks[2], vs[2];
};
// outlier bookkeeping of the same 32 tokens; it travels one half-step ahead of the codes, so that the sideband
// chunks it points to can be requested a whole half-step before use
struct FlagTile {
    int koff[3];               // K: sideband entries [koff[u], koff[u + 1]) belong to tile u (wave-uniform)
    int voff[3];               // V: the same
};
// verbatim chunks of one half-step and tensor, requested ahead: lane i holds the i-th of its first 64 sideband entries
struct Entries {
    int off[3];
    uint2 x;                   // the chunk (raw bits of the cache dtype) and its coordinates, (token & 15) << 8 | chunk, as loaded
    uint32_t cc;
};
// the unit of prefetch: NH half-tiles of 32 tokens
template <int NW, int AB, bool FLAGS, int NH>
struct FastTile {
    HalfTile<NW, AB, FLAGS> h[NH];
};

template <int NBYTES>
__device__ __forceinline__ uint32_t load_small(const uint8_t *p) {
    if constexpr (NBYTES == 4) return *reinterpret_cast<const uint32_t *>(p);
    else if constexpr (NBYTES == 2) return *reinterpret_cast<const uint16_t *>(p);
    else {
        uint32_t v = 0;
#pragma unroll
        for (int i = 0; i < NBYTES; i++) v |= (uint32_t)p[i] << (8 * i);
        return v;
    }
}

// The dynamic LDS block is the kernel's only LDS, so it starts at LDS address 0: the K table sits at byte 0,
// the V table at kVTabOffset, and a gather addresses them with idx * 8 (+ the instruction's immediate offset).
constexpr int kTabMax = 5120;               // codewords the K slot has room for
constexpr int kRadiusTabOffset = kTabMax * 8;           // 8 bytes a code: rq as four fp16, see gather_tokens
constexpr int kVTabOffset = kRadiusTabOffset + 8 * kRadiusCodes;
constexpr int kStageOffset = kVTabOffset + 36864;       // outlier variants: staging rows of the wavefronts, after the V table
constexpr int kFlagsTabMax = (kStageOffset - kVTabOffset) / 8;  // codewords the V slot of the outlier variants holds
static_assert(kFlagsTabMax == 4608, "V table slot of the outlier variants");
constexpr int kAuxTabOffset = 36864;        // s192_r6: 64 dwords with the high radius bits of a pair of chunks, see gather_chunks
// s24_r3 (13-bit codes, K <= 1022, qmax = 7): the tables are kept multiplied out, entry [rq][idx] = codeword * rq at byte
// (rq << 10 | idx) * 8, so that the 13-bit code is the table index and a decode is one gather (no radius arithmetic).
constexpr int kPsTabBytes = 8 * 1024 * 8;   // 64 KB per tensor
// The V table starts two entries before the K table's end (K <= 1022: they are free): an LDS instruction's immediate offset ends at 65535,
// beyond which every address takes an addition of its own (16 + 16 of some 330 vector instructions per half-step at d_h 128).
constexpr int kPsVTabOffset = kPsTabBytes - 16;
constexpr int kPsKMax = 1022;
constexpr bool is_prescaled(int MB, int AB, int IB) { return MB == 12 && AB == 1 && IB == 10; }
constexpr int vtab_offset(bool ps) { return ps ? kPsVTabOffset : kVTabOffset; }
// Outlier variants: a wavefront's staging rows hold this many 16-token tiles (beside the multiplied tables there is room for one)
constexpr int stage_offset(bool ps) { return ps ? 2 * kPsTabBytes : kStageOffset; }
constexpr int stage_tiles(bool ps) { return ps ? 1 : 2; }
constexpr int stage_bytes(bool ps, int CPL) { return stage_tiles(ps) * 16 * 32 * CPL; }
// The wavefronts' progress slots: behind the staging rows, or in the last eight entries of the multiplied V table (Vc.K <= 1016)
constexpr int flags_prog_offset(bool ps, int CPL, int WV) { return ps ? 2 * kPsTabBytes - 64 : stage_offset(ps) + WV * stage_bytes(ps, CPL); }
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint2v_t __attribute__((ext_vector_type(2)));
template <int TAB_OFF>
__device__ __forceinline__ half4 gather8(uint32_t byte_addr) {
    return __builtin_bit_cast(half4, *(lds_u2_ptr)(uintptr_t)(byte_addr + TAB_OFF));
}

// Table byte address of the low (HI = 0) or high (HI = 1) 16-bit index of a masked pair: one shift that reads
// a half of the register (the compiler's own lowering is a shift and an and).
template <int HI>
__device__ __forceinline__ uint32_t half_addr8(uint32_t pair) {
    uint32_t r;
    if constexpr (HI)
        asm("v_lshlrev_b32_sdwa %0, 3, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(r) : "v"(pair));
    else
        asm("v_lshlrev_b32_sdwa %0, 3, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(r) : "v"(pair));
    return r;
}

// The same for a table kept as float8 e4m3 (F8 variants: four bytes per codeword, for tables whose entries are e4m3
// numbers): one 32-bit LDS read and two conversions that widen two bytes each to packed fp16 (exact).
template <int TAB_OFF>
__device__ __forceinline__ half4 gather4_f8(uint32_t byte_addr) {
    const uint32_t w = *(lds_u1_ptr)(uintptr_t)(byte_addr + TAB_OFF);
    const half2v lo = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false);
    const half2v hi = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true);
    return half4{lo[0], lo[1], hi[0], hi[1]};
}
template <int HI>
__device__ __forceinline__ uint32_t half_addr4(uint32_t pair) {
    uint32_t r;
    if constexpr (HI)
        asm("v_lshlrev_b32_sdwa %0, 2, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(r) : "v"(pair));
    else
        asm("v_lshlrev_b32_sdwa %0, 2, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(r) : "v"(pair));
    return r;
}
template <int TAB_OFF, bool F8, int HI>
__device__ __forceinline__ half4 gather_pair_half(uint32_t ix) {
    if constexpr (F8) return gather4_f8<TAB_OFF>(half_addr4<HI>(ix));
    else return gather8<TAB_OFF>(half_addr8<HI>(ix));
}

// Decode of the CPL chunks of one lane in two steps, so that a caller can put all gathers of a half-step in flight
// before the first multiply: gather_chunks requests the codewords from the LDS table (g) and prepares the radius
// codes as packed fp16 pairs (r, chunk j in r[j / 2][j & 1]); scale_chunks multiplies.
// 16+0 layout: the two radius codes of a dword become an fp16 pair with one shift, one and-or
// (0x6400 | rq is the fp16 number 1024 + rq) and one packed subtract.  IB = idx_bits when known at compile
// time (12 for s96), else 0.
template <int OFF>
__device__ __forceinline__ half4 gather8_tr(uint32_t byte_addr);
template <int CPL, int MB, int AB, int IB, int NW, int TAB_OFF, bool F8 = false, bool TR = false>
__device__ __forceinline__ void gather_chunks(const uint32_t (&w)[NW], uint32_t aux, int idx_bits_rt, half4 (&g)[CPL], half2v (&r)[CPL / 2]) {
    const int idx_bits = IB ? IB : idx_bits_rt;
    const uint32_t idx_mask = (1u << idx_bits) - 1u;
    const half2v k1024 = half2v{(_Float16)1024.0f, (_Float16)1024.0f};
    if constexpr (MB == 16 && AB == 0) {
        // mask in a scalar register and magic in a vector register, so that (x & mask) | magic is one v_and_or_b32
        uint32_t rq2 = (0xffffu >> idx_bits) * 0x00010001u, magic = 0x64006400u;
        asm("" : "+s"(rq2));
        asm("" : "+v"(magic));
        const uint32_t im2 = idx_mask * 0x00010001u;
#pragma unroll
        for (int i = 0; i < CPL / 2; i++) {
            const uint32_t ix = w[i] & im2;
            g[2 * i] = gather_pair_half<TAB_OFF, F8, 0>(ix);
            g[2 * i + 1] = gather_pair_half<TAB_OFF, F8, 1>(ix);
            const uint32_t t = ((w[i] >> idx_bits) & rq2) | magic;
            r[i] = __builtin_bit_cast(half2v, t) - k1024;
        }
    } else if constexpr (MB == 16 && AB == 3 && IB == 13) {
        // s192_r6: idx (13 bits) and the low three radius bits in the 16-bit main field, the high three in the aux
        // row.  Six aux bits (two chunks) index a 64-entry LDS table holding them at bits 3..5 and 19..21 together
        // with the 0x6400 fp16 magic.
        constexpr uint32_t im2 = 0x1fff1fffu;
#pragma unroll
        for (int i = 0; i < CPL / 2; i++) {
            const uint32_t ix = w[i] & im2;
            g[2 * i] = gather_pair_half<TAB_OFF, F8, 0>(ix);
            g[2 * i + 1] = gather_pair_half<TAB_OFF, F8, 1>(ix);
            const uint32_t hi = *(lds_u1_ptr)(uintptr_t)(kAuxTabOffset + ((aux >> (6 * i)) & 63u) * 4u);
            const uint32_t t = ((w[i] >> 13) & 0x00070007u) | hi;
            r[i] = __builtin_bit_cast(half2v, t) - k1024;
        }
    } else if constexpr (MB == 12 && AB == 1 && IB == 10) {
        static_assert(!F8, "the float8 table variants exist for 16-bit main fields");
        // s24_r3, tables multiplied out (see kPsTabBytes): eight (d_h 64: four) 12-bit fields (idx in the low 10 bits, the
        // low two radius bits above) in three dwords (one and a half) and the high radius bits in the low bits of aux;
        // field | aux bit << 12 is the table index.  No radius arithmetic: r stays unused.
        const uint32_t w0 = w[0], w1 = w[1], w2 = w[NW - 1];
        constexpr uint32_t M = 0x7ff8u;
        const uint32_t ad[8] = {(w0 << 3) & M, (w0 >> 9) & M, __builtin_amdgcn_alignbit(w1, w0, 21) & M, (w1 >> 1) & M,
                                (w1 >> 13) & M, __builtin_amdgcn_alignbit(w2, w1, 25) & M, (w2 >> 5) & M, (w2 >> 17) & M};
#pragma unroll
        for (int j = 0; j < CPL; j++) {
            const uint32_t at = ((aux << (15 - j)) & 0x8000u) | ad[j];
            if constexpr (TR) g[j] = gather8_tr<TAB_OFF>(at);
            else g[j] = gather8<TAB_OFF>(at);
        }
    } else {
        static_assert(!F8, "the float8 table variants exist for the layouts with compile-time index widths");
#pragma unroll
        for (int j = 0; j < CPL; j++) {
            uint32_t code = code_at<MB, NW>(w, j);
            if (AB) code |= ((aux >> (j * AB)) & ((1u << AB) - 1u)) << MB;
            g[j] = gather8<TAB_OFF>((code & idx_mask) << 3);
            r[j >> 1][j & 1] = (_Float16)(uint16_t)(code >> idx_bits);
        }
    }
}
template <int CPL, bool PS = false>
__device__ __forceinline__ void scale_chunks(const half4 (&g)[CPL], const half2v (&r)[CPL / 2], half4 (&a)[CPL]) {
#pragma unroll
    for (int j = 0; j < CPL; j++) a[j] = PS ? g[j] : g[j] * r[j >> 1][j & 1];
}

// V: the codewords arrive transposed.  ds_read_b64_tr_b16 takes an address per lane like any gather and then transposes 4 x 4 blocks of
// 16-bit elements among 16 lanes: with lane i of a group of 16 asking for a codeword of token i / 4 it holds element i % 4 of that
// lane group's chunk (of lane 4 t + i / 4) for the tokens t = 0..3 afterwards, which is the A operand of O^T = V^T . P^T.  The
// radius codes have to be transposed too: a second gather, of a table whose entry rq is four times fp16(rq), hands them over in the
// same places.  The products are the ones scale_chunks forms, rounded alike, and so are the outputs.  This replaced a product with the
// identity (one matrix instruction and two packs of its fp32 results per chunk position and tile, 16 and 32 per half-step at d_h 128)
// by as many LDS reads; what it took from the vector and matrix units is worth more than what it adds to LDS, which was busy 60 %.
// Whole calls over one cache, without -> with: 64 sequences of 1k to 16k, bf16 s24_r3 with outliers (multiplied tables: no second gather),
// decode step 191 -> 175 us; 4 x 131072, heads of 64, bf16 s96_r4 with outliers 89.7 -> 84.8; 8 x 32768, s192_r6 with outliers
// 48.8 -> 47.6; 32768, s96_r4 13.3 -> 13.0.
template <int OFF>
__device__ __forceinline__ half4 gather8_tr(uint32_t byte_addr) {
    typedef short short4v __attribute__((ext_vector_type(4)));
    typedef short4v __attribute__((address_space(3))) *lds_s4;
    return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(uintptr_t)(byte_addr + OFF)));
}
// (x's low / high 16 bits) >> SH in one instruction
template <int HI>
__device__ __forceinline__ uint32_t half_shr(uint32_t pair, int sh) {
    uint32_t r;
    if constexpr (HI)
        asm("v_lshrrev_b32_sdwa %0, %2, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(r) : "v"(pair), "s"(sh));
    else
        asm("v_lshrrev_b32_sdwa %0, %2, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(r) : "v"(pair), "s"(sh));
    return r;
}
template <int CPL, int MB, int AB, int IB, int NW, int TAB_OFF, int RAD_OFF>
__device__ __forceinline__ void gather_tokens(const uint32_t (&w)[NW], uint32_t aux, int idx_bits_rt, half4 (&a)[CPL]) {
    const int idx_bits = IB ? IB : idx_bits_rt;
    const uint32_t idx_mask = (1u << idx_bits) - 1u;
    if constexpr (is_prescaled(MB, AB, IB)) {
        half2v unused[CPL / 2];
        gather_chunks<CPL, MB, AB, IB, NW, TAB_OFF, false, true>(w, aux, idx_bits, a, unused);
    } else if constexpr (MB == 16 && AB == 0) {
        const uint32_t im2 = idx_mask * 0x00010001u, rm2 = ~im2;
        const int sh = idx_bits - 3;                    // (at least 5, see attn_radius_in_table)
#pragma unroll
        for (int i = 0; i < CPL / 2; i++) {
            const uint32_t ix = w[i] & im2, rx = w[i] & rm2;
            a[2 * i] = gather8_tr<TAB_OFF>(half_addr8<0>(ix)) * gather8_tr<RAD_OFF>(half_shr<0>(rx, sh));
            a[2 * i + 1] = gather8_tr<TAB_OFF>(half_addr8<1>(ix)) * gather8_tr<RAD_OFF>(half_shr<1>(rx, sh));
        }
    } else if constexpr (MB == 16 && AB == 3 && IB == 13) {
        constexpr uint32_t im2 = 0x1fff1fffu;
#pragma unroll
        for (int j = 0; j < CPL; j++) {
            const uint32_t ix = w[j / 2] & im2, lo = j & 1 ? w[j / 2] >> 26 : w[j / 2] >> 10, hi = 3 * j < 6 ? aux << (6 - 3 * j) : aux >> (3 * j - 6);
            a[j] = gather8_tr<TAB_OFF>(j & 1 ? half_addr8<1>(ix) : half_addr8<0>(ix)) * gather8_tr<RAD_OFF>(((lo & 0x38u) | (hi & ~0x38u)) & 0x1f8u);
        }
    } else {
#pragma unroll
        for (int j = 0; j < CPL; j++) {
            uint32_t code = code_at<MB, NW>(w, j);
            if (AB) code |= ((aux >> (j * AB)) & ((1u << AB) - 1u)) << MB;
            a[j] = gather8_tr<TAB_OFF>((code & idx_mask) << 3) * gather8_tr<RAD_OFF>((code >> idx_bits) << 3);
        }
    }
}

// max over the four 16-lane rows (lanes l, l^16, l^32, l^48) without going through LDS
__device__ __forceinline__ float row_max4(float x) {
    const uint32_t b = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const float y = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    const uint32_t c = __float_as_uint(y);
    const auto q = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float row_sum4(float x) {
    const uint32_t b = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const float y = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const uint32_t c = __float_as_uint(y);
    const auto q = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

// fp32 4-vector (exact fp16 values) -> packed fp16
__device__ __forceinline__ half4 pack4(float4v t) {
    const auto lo = __builtin_amdgcn_cvt_pkrtz(t[0], t[1]);
    const auto hi = __builtin_amdgcn_cvt_pkrtz(t[2], t[3]);
    return __builtin_bit_cast(half4, uint2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)});
}

// The merge at the end of a block: rows [wavefront][16 columns][DH accumulators, m, l, pad] in LDS -> the columns' outputs, or their
// partials, E elements a thread.  Four where the columns are more than the threads: their weights are worked out once for them, rows
// are read 16 bytes at a time and leave in pieces of 8 or 16 (one by one, 16 columns took four rounds of 24 LDS reads).  us before ->
// now, with the queries in 16-byte loads: 2 x 21 queries on 204 tokens 7.5 -> 6.4, 8 x 23 on 467 fp16 s24_r3 with verbatim chunks 23.4 -> 20.9,
// 8 x 31 on 584 (d_h 64) 20.5 -> 18.6, 8 x 74 on 2405 bf16 with verbatim chunks 162 -> 157; decode steps alike.
template <int DT, int WV, int DH, int E>
__device__ __forceinline__ void merge_elements(const AttnParams &p, const float *red, int cg, int ncols, int b, int hkv, int sp) {
    typedef float floats __attribute__((ext_vector_type(E)));
    constexpr int RS = DH + 4, PIECES = DH / E;
    const bool wide_o = ((((uintptr_t)p.O) | (uintptr_t)(p.osb * 2) | (uintptr_t)(p.osh * 2) | (uintptr_t)(p.ost * 2)) & 7) == 0;
    for (int o = threadIdx.x; o < ncols * PIECES; o += WV * 64) {
        const int cc = o / PIECES, e = E * (o - cc * PIECES);
        const int ci = cg * 16 + cc;
        float m = -INFINITY;
#pragma unroll
        for (int w = 0; w < WV; w++) m = fmaxf(m, red[((size_t)w * 16 + cc) * RS + DH]);
        float l = 0.f, a[E] = {};
        if (m > -INFINITY) {
#pragma unroll
            for (int w = 0; w < WV; w++) {
                const float *q = red + ((size_t)w * 16 + cc) * RS;
                const float f = __builtin_amdgcn_exp2f((q[DH] - m) * p.c_log2);
                l = fmaf(q[DH + 1], f, l);
                const floats v = *reinterpret_cast<const floats *>(q + e);
#pragma unroll
                for (int i = 0; i < E; i++) a[i] = fmaf(v[i], f, a[i]);
            }
        }
        const int tq2 = (int)fast_div((unsigned)ci, (unsigned)p.G, p.m_G), hq2 = hkv * p.G + (ci - tq2 * p.G);
        if (p.n_splits == 1) {
            uint16_t *op = (uint16_t *)p.O + b * p.osb + hq2 * p.osh + (int64_t)tq2 * p.ost + e;
            uint16_t h[E];
#pragma unroll
            for (int i = 0; i < E; i++) {
                const float v = l > 0.f ? a[i] * p.inv_qmax / l : 0.f;
                h[i] = DT == HQMQ_F16 ? __half_as_ushort(__float2half_rn(v)) : f32_to_bf16_bits(v);
            }
            if (E == 4 && wide_o) *reinterpret_cast<uint2 *>(op) = uint2{(uint32_t)h[0] | (uint32_t)h[E > 1 ? 1 : 0] << 16, (uint32_t)h[E > 2 ? 2 : 0] | (uint32_t)h[E - 1] << 16};
            else {
#pragma unroll
                for (int i = 0; i < E; i++) op[i] = h[i];
            }
        } else {
            // partials carry the maximum in softmax units (base-2 exponent) and acc already divided by qmax
            float *wp = p.ws + ((((size_t)b * p.Hq + hq2) * p.Tq + tq2) * p.n_splits + sp) * (size_t)(DH + kPartialHead);
            if (e == 0) { wp[0] = m * p.c_log2; wp[1] = l; }
            floats v;
#pragma unroll
            for (int i = 0; i < E; i++) v[i] = a[i] * p.inv_qmax;
            *reinterpret_cast<floats *>(wp + kPartialHead + e) = v;
        }
    }
}
template <int DT, int WV, int DH>
__device__ __forceinline__ void merge_waves(const AttnParams &p, const float *red, int cg, int ncols, int b, int hkv, int sp) {
    if (ncols * DH <= WV * 64) merge_elements<DT, WV, DH, 1>(p, red, cg, ncols, b, hkv, sp);      // few columns: more threads, one division each
    else merge_elements<DT, WV, DH, 4>(p, red, cg, ncols, b, hkv, sp);
}

// NCG: column groups (of 16 columns) per wavefront.  Two for chunked prefill with more than 16 columns per KV head:
// a decoded tile and its V transposition then serve 32 columns.
// F8: the codeword tables are kept as float8 e4m3 in LDS (callers that rounded their tables to e4m3)
// Plain caches at d_h 64, tables not multiplied out: two blocks of eight wavefronts share a compute unit (LDS has room for both), which the host
// plans with; four wavefronts per SIMD leave a form 128 registers.  With 130 to 136 (whole calls of 64 / 8 heads, 512 blocks, one block ->
// two): bf16 s192_r4 2000 / 4000 tokens 31.2 -> 27.6 / 47.5 -> 43.5 us, s192_r6 32.7 -> 30.1 / 50.5 -> 48.4, 48 x 1500 s96_r6 23.5 -> 19.5.
constexpr bool two_blocks(int CPL, int MB, int AB, int IB, bool flags, int WV, int NCG) {
    return CPL == 4 && !flags && WV == 8 && NCG == 1 && !is_prescaled(MB, AB, IB);
}
template <int CPL, int MB, int AB, int IB, int DT, bool FLAGS, int WV = kFastWaves, int NCG = 1, bool F8 = false>
__global__ __launch_bounds__(WV * 64, WV == 12 ? 3 : two_blocks(CPL, MB, AB, IB, FLAGS, WV, NCG) ? 4 : 2) void attn_fast_kernel(AttnParams p) {
    static_assert(NCG == 1 || !FLAGS, "outlier variants take one column group");
    constexpr int NB = CPL * MB / 8;
    constexpr int NW = (NB + 3) / 4;
    constexpr int ABYTES = CPL * AB / 8;     // aux bytes per lane where its bits are whole bytes, see load_aux_word
    static_assert((CPL * AB) % 8 == 0 || (CPL == 4 && (AB == 1 || AB == 3)), "aux bits of one lane");
    static_assert(NB % 4 == 0 || NB == 6, "main bytes of one lane");
    static_assert(CPL % 2 == 0, "two chunks per 16x16x32 operand");
    constexpr int NT = WV * 64;
    // Outlier variants gather V before the softmax, whose exponentials then cover the LDS reads (caches read from HBM: 64 sequences of 1k to 16k,
    // bf16 s24_r3, 157.2 -> 153.9 us, 8 x 32768, s192_r6 46.4 -> 45.0; calls over one cache, with the tile offsets by vector loads that came
    // with it, decode step 174 -> 165, s192_r6 47.6 -> 48.3); the plain ones, at three wavefronts per SIMD, would spill (111 -> 195 us), and
    // bf16 ones of 16 + 2 and 16 + 3 bits with the generic field decode.
    constexpr bool kEarlyV = FLAGS && !F8 && !(CPL == 8 && DT == HQMQ_BF16 && MB == 16 && AB >= 2 && IB == 0);
    constexpr int NH = 1;       // half-steps per prefetched tile: one measures faster than two on every shape
    extern __shared__ uint2 lds_tab[];
#ifdef HQMQ_STAMPS
    unsigned long long ph_[8] = {}, tl_ = 0;         // outlier variants: time per phase of the half-steps, summed per wavefront
    int n_steps_ = 0;
    const unsigned long long t_in_ = __builtin_amdgcn_s_memrealtime();
    unsigned long long t_loop_ = 0;
#endif
    constexpr bool PS = is_prescaled(MB, AB, IB);
    constexpr int VTAB = vtab_offset(PS);
    // fp16 tables that stay as they are land in LDS where that is the better form, kernel in us through registers -> landing: outlier caches
    // at d_h 128, s96_r4, 27 sequences of 222 tokens 9.1 -> 8.5, 8 of 2000 10.7 -> 9.8, s192_r6, 8 x 32768 48.4 -> 47.4 (4 x 1000 10.1 -> 10.3).
    // Not so plain s192_r6 (1 x 2000 8.4 -> 8.7), heads of 64 (6 x 900, s192_r4 8.6 -> 9.2), bf16, which is converted in place behind a
    // barrier of its own (64 / 8 heads of 64, 300 tokens, whole call 7.8 -> 9.1).
    constexpr bool kLand = FLAGS && CPL == 8 && MB == 16 && IB != 0 && !F8 && DT == HQMQ_F16;
    uint2 *ktab = lds_tab, *vtab = lds_tab + VTAB / 8;
    touch_kernargs();

    // blocks are dispatched in grid order: batch_order lists the sequences in the order they should start
    // (longest first for ragged batches, so that no long sequence is left for the end)
    int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    if (p.xcd_remap) {
        // the hardware hands workgroups to the XCDs round-robin in linear order (x fastest): renumber so that the
        // (sequence, KV head) index runs fastest and, with a multiple of eight of them, stays on one XCD
        const unsigned lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        const unsigned r = fast_div(lin, gridDim.z, p.m_gz);
        bz = (int)(lin - r * gridDim.z);
        by = (int)fast_div(r, gridDim.x, p.m_gx);
        bx = (int)(r - (unsigned)by * gridDim.x);
    }
    const int slot = (int)fast_div((unsigned)bz, (unsigned)p.Hkv, p.m_hkv);
    // Consecutive sequences start with different KV heads: with eight heads (or a multiple) block index modulo 8, and
    // so the XCD, would otherwise always be the same head, and heads differ in cost (config 4: 20 to 45 sideband
    // entries per half-step and head, 2.8 to 3.4 us per half-step: the XCD of the densest head finished 20 % after
    // the others).
    // (With fewer than eight heads, 8 / Hkv consecutive sequences fill one round of the XCDs and share a rotation.)
    const int turn = slot >> (p.Hkv == 4 ? 1 : p.Hkv == 2 ? 2 : p.Hkv == 1 ? 3 : 0);
    int hkv = bz - slot * p.Hkv + (turn - (int)fast_div((unsigned)turn, (unsigned)p.Hkv, p.m_hkv) * p.Hkv);
    if (hkv >= p.Hkv) hkv -= p.Hkv;
    // The codeword-table loads are the longest dependency chain of the prologue (load, convert, LDS store, barrier)
    // and need nothing but the KV head: they are requested before anything else is worked out.  16-byte loads of two
    // codewords, all unconditional (clamped): straight-line code, exact wait counts.
    // (every pair of the largest table the LDS slots hold, 2560 pairs, in one round of requests: a second round would
    // be a loop of loads, and the wait at its head covers every request in flight, the first tile's included)
    constexpr int FU = is_prescaled(MB, AB, IB) ? (512 + NT - 1) / NT : (kTabMax / 2 + NT - 1) / NT;
    const uint4v *ksrc = (const uint4v *)((const uint2 *)p.Kc.joint + hkv * (p.Kc.jsh / 4));
    const uint4v *vsrc = (const uint4v *)((const uint2 *)p.Vc.joint + hkv * (p.Vc.jsh / 4));
    const int Kk2 = p.Kc.K >> 1, Kv2 = p.Vc.K >> 1;        // tables of an even number of codewords (checked at launch)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint4v tk[kLand ? 1 : FU], tv[kLand ? 1 : FU];
    if constexpr (kLand) land_tables<WV>(uniform_ptr((const uint8_t *)ksrc), 16u * (uint32_t)Kk2, uniform_ptr((const uint8_t *)vsrc), 16u * (uint32_t)Kv2, 0u, VTAB, wave, lane);
    else {
#pragma unroll
        for (int u = 0; u < FU; u++) {
            const int k = threadIdx.x + u * NT;
            tk[u] = ksrc[min(k, Kk2 - 1)];
            tv[u] = vsrc[min(k, Kv2 - 1)];
        }
    }
#ifdef HQMQ_STAMPS
    ph_[0] = __builtin_amdgcn_s_memrealtime();      // table loads requested
#endif
    const int b = p.batch_order ? min(max(uniform_word(p.batch_order, slot), 0), p.B - 1) : slot;
    const int bh = b * p.Hkv + hkv;
    const int cg0 = by * NCG, sp = bx;
    const int G = p.G;
    constexpr int n = 4 * CPL, d_h = 16 * CPL;
    const int col = lane & 15, grp = lane >> 4;
    // The four per-sequence words go out together, without a branch on the optional pointers (an absent array reads
    // a word of the kernel arguments instead): one scalar round trip instead of one per word.
    const int32_t *const spare_word = (const int32_t *)(uintptr_t)__builtin_amdgcn_kernarg_segment_ptr();
    const int32_t w_len = uniform_word(p.kv_len ? p.kv_len + b : spare_word, 0);
    const int32_t w_start = uniform_word(p.kv_start ? p.kv_start + b : spare_word, 0);
    const int32_t w_kcount = uniform_word(FLAGS ? p.Kc.sb_count + bh : spare_word, 0);
    const int32_t w_vcount = uniform_word(FLAGS ? p.Vc.sb_count + bh : spare_word, 0);
    int kv_end = p.kv_len ? w_len : p.Tkv;
    kv_end = min(max(kv_end, 0), p.Tkv);
    bool col_ok[NCG];
    int tq[NCG], hq[NCG], col_lim[NCG];
    int blk_lim = 0, lim_min = 0x7fffffff;
#pragma unroll
    for (int cgi = 0; cgi < NCG; cgi++) {
        const int cidx = (cg0 + cgi) * 16 + col;
        col_ok[cgi] = cidx < p.Tq * G;
        tq[cgi] = col_ok[cgi] ? (int)fast_div((unsigned)cidx, (unsigned)G, p.m_G) : 0;
        hq[cgi] = hkv * G + (col_ok[cgi] ? cidx - tq[cgi] * G : 0);
        int64_t lim64 = kv_end;
        if (p.causal) lim64 = min(lim64, (int64_t)tq[cgi] + p.causal_offset + 1);
        if (!col_ok[cgi] || lim64 < 0) lim64 = 0;
        col_lim[cgi] = (int)lim64;
        blk_lim = max(blk_lim, col_lim[cgi]);
        if (col_ok[cgi]) lim_min = min(lim_min, col_lim[cgi]);
    }
    if (p.causal) {
        for (int o = 1; o < 16; o <<= 1) {
            blk_lim = max(blk_lim, __shfl_xor(blk_lim, o));
            lim_min = min(lim_min, __shfl_xor(lim_min, o));
        }
        blk_lim = __builtin_amdgcn_readfirstlane(blk_lim);      // the same in every lane: all rows hold all 16 columns
        lim_min = __builtin_amdgcn_readfirstlane(lim_min);
    } else {
        blk_lim = lim_min = kv_end;         // every column in range sees the whole sequence (a launched block has one)
    }
    // tokens before kv_start[b] are invisible (left padding): the walk starts at the super-tile that holds it
    const int col_start = p.kv_start ? min(max(w_start, 0), blk_lim) : 0;
    const int blk_lo = col_start / kSuper * kSuper;
    int per_split = (int)fast_div((unsigned)(blk_lim - blk_lo + p.n_splits - 1), (unsigned)p.n_splits, p.m_splits);
    per_split = (per_split + kSuper - 1) / kSuper * kSuper;
    const int b_begin = min(blk_lo + sp * per_split, blk_lim), b_end = min(blk_lim, b_begin + per_split);
    // The block's half-steps go to its wavefronts round-robin: wavefront w takes the 32 tokens at b_begin + 32 (w + i WV),
    // i = 0, 1, ...  What the wavefronts of a block request at any one time is then one contiguous stretch of the
    // planes (batch 8: 3.5 % faster than a contiguous range per wavefront, ragged config 4: 2 %).
    // Every half-step starts at a multiple of 32 below T_kv <= t_cap (a multiple of 64): whole tiles are readable.
    constexpr int TS = 32 * WV;
    const int t_begin = min(b_begin + wave * 32, b_end), t_end = b_end;
    const size_t plane_row0 = (size_t)bh * p.t_cap;
    constexpr int mrb = n * MB / 8, arb = (n * AB + 7) / 8;
    const int64_t tiles_cap = p.t_cap / kTile;
    const int tiles_cap1 = (int)tiles_cap - 1;
    const int idx_bits = p.idx_bits;
    const uint16_t *ks_plane = (const uint16_t *)p.Kc.scale_plane + b * p.Kc.ssb + hkv * p.Kc.ssh;
    const uint16_t *vs_plane = (const uint16_t *)p.Vc.scale_plane + b * p.Vc.ssb + hkv * p.Vc.ssh;
    const uint8_t *k_rows = p.Kc.main_plane + plane_row0 * mrb;
    const uint8_t *v_rows = p.Vc.main_plane + plane_row0 * mrb;
    const uint8_t *ka_rows = AB ? p.Kc.aux_plane + plane_row0 * arb : nullptr;
    const uint8_t *va_rows = AB ? p.Vc.aux_plane + plane_row0 * arb : nullptr;
    const int32_t *k_toff = FLAGS ? p.Kc.sb_tile_off + (size_t)bh * tiles_cap : nullptr;
    const int32_t *v_toff = FLAGS ? p.Vc.sb_tile_off + (size_t)bh * tiles_cap : nullptr;
    // The lane's CPL * AB aux bits start at bit aux_sh of the word at aux_off.  At d_h 64 they are 4 or 12 bits of a row of 2 or
    // 6 bytes: the whole row, or the dword (2-byte aligned) at its byte 0 or 2, is loaded and shifted where it is used.
    constexpr bool kAuxRow2 = CPL == 4 && AB == 1, kAuxRow6 = CPL == 4 && AB == 3;
    const uint32_t main_off = (uint32_t)(col * mrb + grp * NB), aux_off = (uint32_t)(col * arb + (kAuxRow2 ? 0 : kAuxRow6 ? (grp & 2) : grp * ABYTES));
    const uint32_t aux_sh = kAuxRow2 ? 4u * (uint32_t)grp : kAuxRow6 ? 12u * (uint32_t)grp - 8u * (uint32_t)(grp & 2) : 0u;
    // V: lane 4 * token + chunk group, as gather_tokens has it (the float8 variants decode V like K and transpose it by matrix products)
    const int vcol = F8 ? col : lane >> 2, vgrp = F8 ? grp : lane & 3;
    const uint32_t vmain_off = (uint32_t)(vcol * mrb + vgrp * NB), vaux_off = (uint32_t)(vcol * arb + (kAuxRow2 ? 0 : kAuxRow6 ? (vgrp & 2) : vgrp * ABYTES));
    const uint32_t vaux_sh = kAuxRow2 ? 4u * (uint32_t)vgrp : kAuxRow6 ? 12u * (uint32_t)vgrp - 8u * (uint32_t)(vgrp & 2) : 0u;
    auto load_aux_word = [&](const uint8_t *q) -> uint32_t {
        if constexpr (kAuxRow2) return *reinterpret_cast<const uint16_t *>(q);
        else if constexpr (kAuxRow6) return *reinterpret_cast<const uint32_a2 *>(q);
        else return load_small<ABYTES>(q);
    };
    auto load_main = [&](const uint8_t *q, uint32_t (&w)[NW]) {
        if constexpr (NB == 6) {        // 2-byte aligned; as loaded, like everything here: put together at once they would be waited for
            w[0] = *reinterpret_cast<const uint32_a2 *>(q);
            w[1] = *reinterpret_cast<const uint16_t *>(q + 4);
        } else load_bytes<NB>(q, w);
    };
    const uint32_t scale_off = (uint32_t)(4 * grp);
    const int k_count = FLAGS ? (int)min((int64_t)max(w_kcount, 0), p.Kc.sb_cap) : 0;
    const int v_count = FLAGS ? (int)min((int64_t)max(w_vcount, 0), p.Vc.sb_cap) : 0;
    const char *k_side = FLAGS ? (const char *)p.Kc.sideband + (size_t)bh * p.Kc.sb_cap * 8 : nullptr;
    const char *v_side = FLAGS ? (const char *)p.Vc.sideband + (size_t)bh * p.Vc.sb_cap * 8 : nullptr;
    const char *k_coord = FLAGS ? (const char *)p.Kc.sb_coord + (size_t)bh * p.Kc.sb_cap * 2 : nullptr;
    const char *v_coord = FLAGS ? (const char *)p.Vc.sb_coord + (size_t)bh * p.Vc.sb_cap * 2 : nullptr;

    constexpr bool kScalarRows = !FLAGS && NCG == 1 && !F8;        // (with two column groups 12 + 2 bits took 39.5 us where it takes 38.6)
    // At d_h 64 two planes stay with lane addresses, or the 128 registers that a second block leaves (see the launch bounds) do not hold
    // the form: 64 x 3000 tokens, bf16, 12 + 2 bits 42.9 us with all scalar, 40.9 so; 12 + 3 bits 44.9, 43.8 so.
    constexpr bool kScalarAux = kScalarRows && !(CPL == 4 && MB == 12 && AB == 2), kScalarScales = kScalarRows && !(CPL == 4 && MB == 12 && AB == 3);
    auto load_k = [&](int th, HalfTile<NW, AB, FLAGS> &h) {
        const uint8_t *kb = scalar_base<kScalarRows>(k_rows + (size_t)th * mrb), *ka = scalar_base<kScalarAux>(AB ? ka_rows + (size_t)th * arb : nullptr);
        const uint16_t *kp = scalar_base<kScalarScales>(ks_plane + th);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            load_main(kb + main_off + u * 16 * mrb, h.kw[u]);
            if constexpr (AB > 0) h.kaux[u] = load_aux_word(ka + aux_off + u * 16 * arb);
            h.ks[u] = *reinterpret_cast<const uint2 *>(kp + scale_off + 16 * u);
        }
    };
    auto load_v = [&](int th, HalfTile<NW, AB, FLAGS> &h) {
        const uint8_t *vb = scalar_base<kScalarRows>(v_rows + (size_t)th * mrb), *va = scalar_base<kScalarAux>(AB ? va_rows + (size_t)th * arb : nullptr);
        const uint16_t *vp = scalar_base<kScalarScales>(vs_plane + th);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            load_main(vb + vmain_off + u * 16 * mrb, h.vw[u]);
            if constexpr (AB > 0) h.vaux[u] = load_aux_word(va + vaux_off + u * 16 * arb);
            h.vs[u] = *reinterpret_cast<const uint2 *>(vp + scale_off + 16 * u);
        }
    };
    auto load_super = [&](int t0, FastTile<NW, AB, FLAGS, NH> &s) {
        // in the order the half-steps consume them: K, then V, of tokens 0..31, then the same of tokens 32..63
#pragma unroll
        for (int hh = 0; hh < NH; hh++) {
            load_k(t0 + 32 * hh, s.h[hh]);
            load_v(t0 + 32 * hh, s.h[hh]);
        }
    };

    // Tile offsets of the first two half-steps, in two parts: the loads (scalar ones, through the constant address space: nothing writes the
    // offsets while this kernel runs), and their clamping once flags_ready has let them through.
    typedef const int32_t __attribute__((address_space(4))) *const_i32_ptr;
    const const_i32_ptr k_toff_c = (const_i32_ptr)(uintptr_t)k_toff, v_toff_c = (const_i32_ptr)(uintptr_t)v_toff;
    auto load_flags = [&](int th, FlagTile &f) {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int tc = min((th >> 4) + i, tiles_cap1);
            f.koff[i] = k_toff_c[tc];
            f.voff[i] = v_toff_c[tc];
        }
    };
    auto flags_ready = [&](int th, FlagTile &f) {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            asm volatile("" : "+s"(f.koff[i]), "+s"(f.voff[i]));        // this is where the scalar loads are waited for
        }
        // tiles not written yet hold INT32_MAX, and so does the slot after the last tile: the count bounds them
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const bool in = (th >> 4) + i <= tiles_cap1;
            f.koff[i] = min(in ? f.koff[i] : 0x7fffffff, k_count);
            f.voff[i] = min(in ? f.voff[i] : 0x7fffffff, v_count);
        }
        // a tile has at most 16 n entries: bounds the walk if the caller's offsets are inconsistent
#pragma unroll
        for (int i = 1; i < 3; i++) {
            f.koff[i] = min(f.koff[i], f.koff[i - 1] + 16 * n);
            f.voff[i] = min(f.voff[i], f.voff[i - 1] + 16 * n);
        }
    };

    // The same in the loop, as one vector load: lane i holds K's offset i (V's: lane 32 + i), read lane by lane when it has arrived.  Scalar
    // loads share their counter with LDS and return out of order: with one outstanding every wait for LDS is a wait for everything.
    const int lane_tile = min(lane & 31, 2), lane_count = lane & 32 ? v_count : k_count;
    const int32_t *const lane_toff = lane & 32 ? v_toff : k_toff;
    auto load_offsets = [&](int th) { return lane_toff[min((th >> 4) + lane_tile, tiles_cap1)]; };
    auto offsets_ready = [&](int th, int w, FlagTile &f) {
        w = min((th >> 4) + lane_tile <= tiles_cap1 ? w : 0x7fffffff, lane_count);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            f.koff[i] = __builtin_amdgcn_readlane(w, i);
            f.voff[i] = __builtin_amdgcn_readlane(w, 32 + i);
        }
#pragma unroll
        for (int i = 1; i < 3; i++) {
            f.koff[i] = min(f.koff[i], f.koff[i - 1] + 16 * n);
            f.voff[i] = min(f.voff[i], f.voff[i - 1] + 16 * n);
        }
    };
    // Every load of the loop is issued unconditionally (clamped addresses): a load inside a branch would make the
    // compiler's wait counts assume it was not issued, and the waits would then cover the next tile's prefetch.
    // The sideband entries of a half-step are a contiguous range known from three tile offsets, so no flag is read.  Lane i takes
    // entry i of the range (the last one again behind its end), at 32-bit byte offsets from wave-uniform bases (sb_cap < 2^28 is
    // checked at launch).
    auto entry_load = [&](const char *side, const char *coord, const int (&off)[3], int e, uint2 &x, uint32_t &cc) {
        const uint32_t at = min((uint32_t)e, (uint32_t)max(off[2] - 1, 0));       // (inconsistent offsets of a caller may be negative)
        x = *reinterpret_cast<const uint2 *>(side + at * 8u);
        cc = *reinterpret_cast<const uint16_t *>(coord + at * 2u);
    };
    auto issue_one = [&](const char *side, const char *coord, const int (&off)[3], Entries &q) {
#pragma unroll
        for (int i = 0; i < 3; i++) q.off[i] = off[i];
        entry_load(side, coord, q.off, q.off[0] + lane, q.x, q.cc);
    };
    // sideband requests of one half-step
    auto issue_all = [&](const FlagTile &f, Entries &k, Entries &v) {
        issue_one(k_side, k_coord, f.koff, k);
        issue_one(v_side, v_coord, f.voff, v);
    };
    Entries kc = {}, vc = {};
    FastTile<NW, AB, FLAGS, NH> cur;
    FlagTile f0 = {}, f1 = {};
    uint2 q_raw[NCG][CPL];      // the query rows as stored
    const bool wide_q = ((((uintptr_t)p.Q) | (uintptr_t)(p.qsb * 2) | (uintptr_t)(p.qsh * 2) | (uintptr_t)(p.qst * 2)) & 15) == 0;
    {
        // unconditional (a wavefront without a range reads a valid tile it never uses): no branch, so the waits for the
        // table loads below count these loads as issued
        const int t_first = min(t_begin, (int)p.t_cap - 32);
        if (FLAGS) load_flags(t_first, f0);
        // Requests go out in the order their data is used, since they come back in that order and a wait for one is a
        // wait for all before it: tables (requested at the very start), query rows, first tile, its sideband entries.
        // All 16 lanes of a row load (columns past the end read column 0 again and are cleared below): unconditional,
        // so that the waits count them.
#pragma unroll
        for (int cgi = 0; cgi < NCG; cgi++) {
            const uint16_t *qp = (const uint16_t *)p.Q + b * p.qsb + hq[cgi] * p.qsh + (int64_t)tq[cgi] * p.qst + grp * CPL * 4;
            if (wide_q) {
#pragma unroll
                for (int j = 0; j < CPL; j += 2) {
                    const uint4v w = *reinterpret_cast<const uint4v *>(qp + 4 * j);
                    q_raw[cgi][j] = uint2{w[0], w[1]};
                    q_raw[cgi][j + 1] = uint2{w[2], w[3]};
                }
            } else {
#pragma unroll
                for (int j = 0; j < CPL; j++) q_raw[cgi][j] = *reinterpret_cast<const uint2 *>(qp + 4 * j);
            }
        }
        load_super(t_first, cur);
#ifdef HQMQ_STAMPS
        ph_[2] = __builtin_amdgcn_s_memrealtime();      // first tile requested
#endif
        if constexpr (FLAGS) {
            // the first half-step's sideband entries are requested here, behind its tile: they travel while the tables
            // are filled (requested behind the barrier, they were the last thing the first half-step waited for)
            flags_ready(t_first, f0);
            issue_all(f0, kc, vc);          // unconditional (clamped addresses): a wavefront without a range reads entries it never uses
            load_flags(t_begin + TS < t_end ? t_begin + TS : t_first, f1);        // made ready behind the barrier
        }
    }
#ifdef HQMQ_STAMPS
    ph_[1] = __builtin_amdgcn_s_memrealtime();      // the first half-step's entries requested
#endif
    // Plain variants keep two half-steps in flight; the second is requested right behind the first (both queue
    // behind the table loads, which were requested at the very start).
    auto readable = [&](int t) { return min(t, (int)p.t_cap - 32); };
    FastTile<NW, AB, FLAGS, NH> tb;
    if constexpr (!FLAGS) load_super(readable(t_begin + TS < t_end ? t_begin + TS : t_begin), tb);
    half4 ident;                        // float8 variants, B operand of the transposing MFMA: the 16x16 identity
#pragma unroll
    for (int e = 0; e < 4; e++) ident[e] = (_Float16)((4 * grp + e) == col ? 1.f : 0.f);
    // bf16 caches: K's verbatim chunks (and the Q they meet) go into bf16 MFMAs as they are stored; the products are exact
    constexpr bool kBfEntries = FLAGS && DT == HQMQ_BF16;

    {
        if constexpr (PS) {
            // tables multiplied out: codeword * rq for rq = 0..7 at (rq << 10 | idx) * 8 (K <= 1022: FU * NT pairs cover it)
#pragma unroll
            for (int u = 0; u < FU; u++) {
                const int k = threadIdx.x + u * NT;
                const uint4v hk = pair_to_half<DT>(tk[u]), hv = pair_to_half<DT>(tv[u]);
#pragma unroll
                for (int rq = 0; rq < 8; rq++) {
                    const half2v f = half2v{(_Float16)(float)rq, (_Float16)(float)rq};
                    auto mul = [&](uint32_t w) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, w) * f); };
                    if (k < Kk2) reinterpret_cast<uint4v *>(ktab)[rq * 512 + k] = uint4v{mul(hk[0]), mul(hk[1]), mul(hk[2]), mul(hk[3])};
                    if (k < Kv2) reinterpret_cast<uint4v *>(vtab)[rq * 512 + k] = uint4v{mul(hv[0]), mul(hv[1]), mul(hv[2]), mul(hv[3])};
                }
            }
        } else if constexpr (!kLand) {
#pragma unroll
            for (int u = 0; u < FU; u++) {
                const int k = threadIdx.x + u * NT;
                if (k < Kk2) store_pair<DT, F8>(ktab, k, tk[u]);
                if (k < Kv2) store_pair<DT, F8>(vtab, k, tv[u]);
            }
        }
    }
    half8 qf[NCG][CPL / 2];
#pragma unroll
    for (int cgi = 0; cgi < NCG; cgi++) {
#pragma unroll
        for (int j = 0; j < CPL / 2; j++) {
            const half4 z = half4{0, 0, 0, 0};
            qf[cgi][j] = cat8(col_ok[cgi] ? chunk_to_half<DT>(q_raw[cgi][2 * j]) : z, col_ok[cgi] ? chunk_to_half<DT>(q_raw[cgi][2 * j + 1]) : z);
        }
    }
    bf16x8 qb[kBfEntries ? CPL / 2 : 1];            // the stored bf16 values
    if constexpr (kBfEntries) {
#pragma unroll
        for (int j = 0; j < CPL / 2; j++) {
            const uint2 lo = col_ok[0] ? q_raw[0][2 * j] : uint2{0, 0}, hi = col_ok[0] ? q_raw[0][2 * j + 1] : uint2{0, 0};
            qb[j] = __builtin_bit_cast(bf16x8, uint4v{lo.x, lo.y, hi.x, hi.y});
        }
    }
    // staging rows for verbatim chunks, cleared here and after every use
    constexpr int ST = stage_tiles(PS), ROWB = 32 * CPL, STB = 16 * ROWB;
    const uint32_t stage = (uint32_t)(stage_offset(PS) + wave * stage_bytes(PS, CPL));
    auto wipe = [&]() {
#pragma unroll
        for (int i = 0; i < ST * STB / 1024; i++) *(uint4v __attribute__((address_space(3))) *)(uintptr_t)(stage + 1024u * i + 16u * (uint32_t)lane) = uint4v{0, 0, 0, 0};
    };
    if constexpr (FLAGS) wipe();
    // Progress slots of the wavefronts (see `publish` below), behind everything else the loop keeps in LDS
    const uint32_t prog_base = FLAGS ? (uint32_t)flags_prog_offset(PS, CPL, WV) : PS ? 2u * (uint32_t)kPsTabBytes : (uint32_t)kVTabOffset + (uint32_t)p.Vc.K * 8u;
    typedef int __attribute__((address_space(3))) *lds_i32_ptr;
    if (threadIdx.x < 16) *(lds_i32_ptr)(uintptr_t)(prog_base + 4u * threadIdx.x) = 0;
    if constexpr (!PS && !F8) {
        if (threadIdx.x < kRadiusCodes) {
            const half4 r = half4{1, 1, 1, 1} * (_Float16)(uint16_t)threadIdx.x;
            lds_tab[kRadiusTabOffset / 8 + threadIdx.x] = __builtin_bit_cast(uint2, r);
        }
    }
    if constexpr (MB == 16 && AB == 3 && IB == 13) {
        if (threadIdx.x < 64) {
            const uint32_t b6 = threadIdx.x;
            reinterpret_cast<uint32_t *>(lds_tab)[kAuxTabOffset / 4 + b6] = ((b6 & 7u) << 3) | ((b6 >> 3) << 19) | 0x64006400u;
        }
    }
    // Tables in: a query chunk, requested behind them, is used here, so the compiler waits for it and with it for them.  (Not by a count of the
    // loads behind the tables: how many those are is the compiler's choice.)
    if constexpr (kLand) asm volatile("" ::"v"(q_raw[0][CPL - 1].y) : "memory");
#ifdef HQMQ_STAMPS
    const unsigned long long t_fill_ = __builtin_amdgcn_s_memrealtime();
#endif
    __syncthreads();
#ifdef HQMQ_STAMPS
    const unsigned long long t_bar_ = __builtin_amdgcn_s_memrealtime();
#endif

    // Scores are kept as v = S^T * rs (+ qmax * unscaled outlier part); the softmax argument is c_log2 * v.
    const float c = p.c_log2, qmaxf = (float)p.qmax;
    float m_run[NCG], l_run[NCG];
    float4v acc[NCG][CPL];
#pragma unroll
    for (int cgi = 0; cgi < NCG; cgi++) {
        m_run[cgi] = -INFINITY;
        l_run[cgi] = 0.f;
#pragma unroll
        for (int j = 0; j < CPL; j++) acc[cgi][j] = float4v{0.f, 0.f, 0.f, 0.f};
    }
    const float4v zero4 = float4v{0.f, 0.f, 0.f, 0.f};
    // Verbatim chunks.  The wavefront writes a half-step's entries (K's, then V's) over zeros into rows of its own in LDS,
    // [token][chunk], reads them as whole matrix operands and clears what it wrote: its LDS accesses keep their order, so nothing
    // has to be waited for but the data itself.  The walk over the list in batches that this replaced (eight entries of K, sixteen of
    // V the reduction dimension of a product, with masks, look-ups and a transposition per chunk position) was 173 of 567 vector
    // instructions per half-step at d_h 128 and a chain of 40 matrix instructions; this is 60 and 16.  Whole calls over
    // one cache, before -> now: 64 sequences of 1k to 16k, bf16 s24_r3, 1.7 % of the chunks verbatim, decode step 249 -> 197 us; 8 x 32768,
    // 28 / 4 heads, s192_r6, 2 % of K's 59.3 -> 48.8; 4 x 131072, heads of 64, bf16, 1 % 95.1 -> 89.7.  Without the test in front of V's part
    // calls whose values have no outliers take 5 % longer (48.8 -> 51.4) and calls with both 1 to 2 % less (196 -> 193).  The chunks of a
    // row are permuted by the token (16-byte parts, exclusive-or), so that K's reads (16 tokens at the same part) and V's transposing ones
    // (4 tokens at 4 parts) meet 64 different banks.
    typedef uint2v_t __attribute__((address_space(3))) *lds_w2_ptr;
    auto swizzled = [&](uint32_t row, uint32_t byte) {          // byte: 8 * chunk
        return CPL == 8 ? byte ^ row * 0x110u : byte ^ (row * 0x88u & ~8u);
    };
    auto entry_at = [&](const int (&off)[3], int e, uint32_t cc) {
        const uint32_t at = swizzled((cc >> 8) & 15u, (cc & (uint32_t)(n - 1)) << 3) + stage;
        return ST == 2 && e >= off[1] ? at + (uint32_t)STB : at;
    };
    auto mine = [&](const int (&off)[3], int u0, int e) { return (ST == 2 || e >= off[u0]) && e < off[u0 + ST]; };
    auto verbatim = [&](uint2 x, bool v) {                      // V meets fp16 weights
        if (!kBfEntries || !v) return x;
        return __builtin_bit_cast(uint2, pack4(float4v{__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xffff0000u), __uint_as_float(x.y << 16), __uint_as_float(x.y & 0xffff0000u)}));
    };
    auto stage_entries = [&](const Entries &q, int u0, bool v) {
        const int e = q.off[0] + lane;
        const uint32_t at = entry_at(q.off, e, q.cc);
        if (mine(q.off, u0, e)) *(lds_w2_ptr)(uintptr_t)at = __builtin_bit_cast(uint2v_t, verbatim(q.x, v));
        for (int bs = q.off[0] + 64; bs < q.off[2]; bs += 64) {             // more than 64: rare
            uint2 x;
            uint32_t cc;
            entry_load(v ? v_side : k_side, v ? v_coord : k_coord, q.off, bs + lane, x, cc);
            if (mine(q.off, u0, bs + lane)) *(lds_w2_ptr)(uintptr_t)entry_at(q.off, bs + lane, cc) = __builtin_bit_cast(uint2v_t, verbatim(x, v));
        }
        asm volatile("" ::: "memory");
        return at;
    };
    auto unstage = [&](const Entries &q, int u0, uint32_t at) {
        asm volatile("" ::: "memory");
        if (mine(q.off, u0, q.off[0] + lane)) *(lds_w2_ptr)(uintptr_t)at = uint2v_t{0u, 0u};
        if (q.off[2] - q.off[0] > 64) wipe();
        asm volatile("" ::: "memory");
    };
    // K: A operands of S^T, as the main product has them
    const uint32_t k_at = stage + swizzled((uint32_t)col, (uint32_t)(grp * CPL * 8));
    auto k_operands = [&](int u, uint4v (&a)[CPL / 2]) {
#pragma unroll
        for (int jj = 0; jj < CPL / 2; jj++) a[jj] = *(lds_u4_ptr)(uintptr_t)((k_at ^ (uint32_t)(16 * jj)) + (uint32_t)(u % ST * STB));
    };
    auto k_products = [&](const uint4v (&a)[CPL / 2], float4v &so) {
#pragma unroll
        for (int jj = 0; jj < CPL / 2; jj++) {
            if constexpr (kBfEntries) so = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[jj]), qb[jj], so, 0, 0, 0);
            else so = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a[jj]), qf[0][jj], so, 0, 0, 0);
        }
    };
    // V: lane i of a group of 16 reads chunk (i % 4) CPL + j of token 4 grp + i / 4; the transposing read leaves it element i % 4 of
    // chunk (i / 4) CPL + j of the four tokens: the rows of the main V product, tokens as P has them
    const uint32_t v_at = stage + swizzled((uint32_t)(4 * grp + (col >> 2)), (uint32_t)((col & 3) * CPL * 8));
    auto v_operands = [&](int u, half4 (&a)[CPL]) {
        typedef short4v __attribute__((address_space(3))) *lds_s4;
#pragma unroll
        for (int j = 0; j < CPL; j++)
            a[j] = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(uintptr_t)((v_at ^ (uint32_t)(16 * (j >> 1))) + (uint32_t)(8 * (j & 1) + u % ST * STB))));
    };

    // One half-step: 32 tokens (two tiles) through scores, online softmax and the V product.  A flagged chunk
    // carries radius code 0 in the main plane, so its decoded value is exactly zero and only the verbatim
    // value from the sideband contributes.
    // next_*: the requests for the next half-step that take the place of what has just been used (outlier variants at d_h 64)
    auto half_step = [&](const HalfTile<NW, AB, FLAGS> &h, int th, const Entries &kc, const Entries &vc, auto next_k_entries, auto next_k, auto next_v, auto next_v_entries) {
        float4v sT[NCG][2], so[2] = {zero4, zero4};
        // the operands of the verbatim chunks are requested first and used after the main product
        uint4v kv[2][CPL / 2];
        if constexpr (FLAGS) {
#pragma unroll
            for (int u0 = 0; u0 < 2; u0 += ST) {
                const uint32_t at = stage_entries(kc, u0, false);
#pragma unroll
                for (int u = u0; u < u0 + ST; u++) k_operands(u, kv[u]);
                unstage(kc, u0, at);
            }
            next_k_entries();
        }
        // (gathers and multiplies interleaved by the compiler: every gather of the 32 K tokens requested before the first one is used was no faster
        // on any shape, at 178 registers against 157)
        half4 gk[2][CPL];
        half2v rk[2][CPL / 2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            half4 a[CPL];
            gather_chunks<CPL, MB, AB, IB, NW, 0, F8>(h.kw[u], AB ? h.kaux[u] >> aux_sh : 0u, idx_bits, gk[u], rk[u]);
            scale_chunks<CPL, PS>(gk[u], rk[u], a);
#pragma unroll
            for (int cgi = 0; cgi < NCG; cgi++) {
                float4v s = zero4;
#pragma unroll
                for (int jj = 0; jj < CPL / 2; jj++)
                    s = __builtin_amdgcn_mfma_f32_16x16x32_f16(cat8(a[2 * jj], a[2 * jj + 1]), qf[cgi][jj], s, 0, 0, 0);
                if constexpr (!FLAGS) {
#pragma unroll
                    for (int e = 0; e < 4; e++) s[e] = scaled<DT>(s[e], e < 2 ? h.ks[u].x : h.ks[u].y, e & 1, 0.f);
                }
                sT[cgi][u] = s;
            }
        }
#ifdef HQMQ_STAMPS
        asm volatile("" ::"v"(sT[0][0]), "v"(sT[0][1]));
        PHASE(1);
#endif
        if constexpr (FLAGS) {
#pragma unroll
            for (int u = 0; u < 2; u++) k_products(kv[u], so[u]);
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    sT[0][u][e] = scaled<DT>(sT[0][u][e], e < 2 ? h.ks[u].x : h.ks[u].y, e & 1, so[u][e] * qmaxf);
            next_k();
        }
#ifdef HQMQ_STAMPS
        asm volatile("" ::"v"(sT[0][0]), "v"(sT[0][1]));
        PHASE(2);
#endif
        half4 early[kEarlyV ? 2 : 1][CPL];
        if constexpr (kEarlyV) {
#pragma unroll
            for (int u = 0; u < 2; u++) gather_tokens<CPL, MB, AB, IB, NW, VTAB, kRadiusTabOffset>(h.vw[u], AB ? h.vaux[u] >> vaux_sh : 0u, idx_bits, early[u]);
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- mask (boundary half-steps only), online softmax, per column group ----
        const bool edge = !(th + 32 <= lim_min && th + 32 <= t_end && th >= col_start);
        half8 pp[NCG];
        half4 pTo[2];
#pragma unroll
        for (int cgi = 0; cgi < NCG; cgi++) {
            if (edge) {
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int t = th + 16 * u + 4 * grp + e;
                        if (!(t < col_lim[cgi] && t < t_end && t >= col_start)) sT[cgi][u][e] = -INFINITY;
                    }
            }
            float tmax = fmaxf(fmaxf(fmaxf(sT[cgi][0][0], sT[cgi][0][1]), fmaxf(sT[cgi][0][2], sT[cgi][0][3])),
                               fmaxf(fmaxf(sT[cgi][1][0], sT[cgi][1][1]), fmaxf(sT[cgi][1][2], sT[cgi][1][3])));
            tmax = row_max4(tmax);
            const float m_new = fmaxf(m_run[cgi], tmax);
            const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
            if (__builtin_amdgcn_ballot_w64(m_new != m_run[cgi]) != 0) {     // rescale only when some column's maximum moved
                const float alpha = __builtin_amdgcn_exp2f((m_run[cgi] - m_use) * c);
                l_run[cgi] *= alpha;
#pragma unroll
                for (int j = 0; j < CPL; j++) acc[cgi][j] = acc[cgi][j] * alpha;
                m_run[cgi] = m_new;
            }
            const float mc = -m_use * c;
            half4 pT[2];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                float pe[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    pe[e] = __builtin_amdgcn_exp2f(fmaf(sT[cgi][u][e], c, mc));
                    l_run[cgi] += pe[e];
                }
                pT[u] = weigh<DT>(pe, h.vs[u]);
                if constexpr (FLAGS) {          // for the verbatim chunks; qmax P is rounded to fp16 here and nowhere else
#pragma unroll
                    for (int e = 0; e < 4; e++) pTo[u][e] = (_Float16)(pe[e] * qmaxf);
                }
            }
            pp[cgi] = cat8(pT[0], pT[1]);
        }
        if constexpr (kEarlyV) next_v();
#ifdef HQMQ_STAMPS
        asm volatile("" ::"v"(pp[0]));
        PHASE(3);
#endif
        // ---- O^T += V^T . P^T, both tiles in one MFMA (the 1/qmax of the radius is applied once, in the epilogue) ----
        half8 vt[CPL];
        if constexpr (F8) {
            half4 g[CPL], av[2][CPL];
            half2v r[CPL / 2];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                gather_chunks<CPL, MB, AB, IB, NW, VTAB, F8>(h.vw[u], AB ? h.vaux[u] >> vaux_sh : 0u, idx_bits, g, r);
                scale_chunks<CPL, PS>(g, r, av[u]);
            }
#pragma unroll
            for (int j = 0; j < CPL; j++)
                vt[j] = cat8(pack4(__builtin_amdgcn_mfma_f32_16x16x16f16(av[0][j], ident, zero4, 0, 0, 0)), pack4(__builtin_amdgcn_mfma_f32_16x16x16f16(av[1][j], ident, zero4, 0, 0, 0)));
        } else if constexpr (kEarlyV) {
#pragma unroll
            for (int j = 0; j < CPL; j++) vt[j] = cat8(early[0][j], early[1][j]);
        } else {
            half4 av[2][CPL];
#pragma unroll
            for (int u = 0; u < 2; u++) gather_tokens<CPL, MB, AB, IB, NW, VTAB, kRadiusTabOffset>(h.vw[u], AB ? h.vaux[u] >> vaux_sh : 0u, idx_bits, av[u]);
#pragma unroll
            for (int j = 0; j < CPL; j++) vt[j] = cat8(av[0][j], av[1][j]);
        }
        if constexpr (!kEarlyV) next_v();
#pragma unroll
        for (int j = 0; j < CPL; j++)
#pragma unroll
            for (int cgi = 0; cgi < NCG; cgi++) acc[cgi][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vt[j], pp[cgi], acc[cgi][j], 0, 0, 0);
#ifdef HQMQ_STAMPS
        asm volatile("" ::"v"(acc[0][0]), "v"(acc[0][CPL - 1]));
        PHASE(4);
#endif
        if (FLAGS && vc.off[0] < vc.off[2]) {   // (tested for V only: keys have outliers far more often than values)
            half4 vv[2][CPL];
#pragma unroll
            for (int u0 = 0; u0 < 2; u0 += ST) {
                const uint32_t at = stage_entries(vc, u0, true);
#pragma unroll
                for (int u = u0; u < u0 + ST; u++) v_operands(u, vv[u]);
                unstage(vc, u0, at);
            }
#pragma unroll
            for (int j = 0; j < CPL; j++) acc[0][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cat8(vv[0][j], vv[1][j]), cat8(pTo[0], pTo[1]), acc[0][j], 0, 0, 0);
        }
        next_v_entries();
#ifdef HQMQ_STAMPS
        asm volatile("" ::"v"(acc[0][0]), "v"(acc[0][CPL - 1]));
        PHASE(5);
#endif
    };

    // The wavefronts that share a SIMD drift apart: the older one wins every tie for an issue slot, ends up several
    // half-steps ahead (config 4: 15 us at the end of a block) and leaves the younger to finish alone, with nothing
    // to overlap its waits.  Every wavefront publishes its position in LDS at the top of a half-step and reads its
    // SIMD neighbours' (wavefronts w, w + 4, w + 8 share a SIMD); at the end of the half-step it raises its priority
    // if one of them is ahead and drops it otherwise.
    int peer_pos = 0;
    auto publish = [&](int t0) {
        const int mine = t0 - 32 * wave;        // the same for all wavefronts at the same distance from the block's start
        *(lds_i32_ptr)(uintptr_t)(prog_base + 4u * (uint32_t)wave) = mine;
        peer_pos = *(lds_i32_ptr)(uintptr_t)(prog_base + 4u * (uint32_t)((wave + 4) % WV));
        if constexpr (WV > 8) peer_pos = max(peer_pos, *(lds_i32_ptr)(uintptr_t)(prog_base + 4u * (uint32_t)((wave + 8) % WV)));
    };
    // (A tie goes to the younger wavefront, w >= 4: at equal priority the hardware would give it to the older one.)
    auto rebalance = [&](int t0) {
        if (__builtin_amdgcn_readfirstlane(peer_pos) + (wave >= 4 ? 1 : 0) > t0 - 32 * wave) __builtin_amdgcn_s_setprio(3);
        else __builtin_amdgcn_s_setprio(0);
    };
    if constexpr (FLAGS) flags_ready(t_begin + TS < t_end ? t_begin + TS : min(t_begin, (int)p.t_cap - 32), f1);

    if constexpr (!FLAGS) {
        // ring of three tile buffers, every load unconditional (past the end the current tile is requested again)
        auto nothing = [] {};
        FastTile<NW, AB, FLAGS, NH> tc;
        int t0 = t_begin;
        if (t0 < t_end) {
            while (true) {
                load_super(readable(t0 + 2 * TS < t_end ? t0 + 2 * TS : t0), tc);
                publish(t0);
                half_step(cur.h[0], t0, kc, vc, nothing, nothing, nothing, nothing);
                rebalance(t0);
                t0 += TS;
                if (t0 >= t_end) break;
                load_super(readable(t0 + 2 * TS < t_end ? t0 + 2 * TS : t0), cur);
                publish(t0);
                half_step(tb.h[0], t0, kc, vc, nothing, nothing, nothing, nothing);
                rebalance(t0);
                t0 += TS;
                if (t0 >= t_end) break;
                load_super(readable(t0 + 2 * TS < t_end ? t0 + 2 * TS : t0), tb);
                publish(t0);
                half_step(tc.h[0], t0, kc, vc, nothing, nothing, nothing, nothing);
                rebalance(t0);
                t0 += TS;
                if (t0 >= t_end) break;
            }
        }
    }
    if constexpr (FLAGS) {
        // Outlier variants, tile offsets two half-steps ahead; past the end the current tile is requested again.  d_h 128: two sets of buffers
        // (tile, entries) take turns, requested one half-step ahead and written out as two half-steps per round of the loop: with one set
        // handed on (cur = nxt) the compiler copied some fifty registers per half-step.  d_h 64: one set, refilled piece by piece as a
        // half-step uses it up (K's entries, K, V, V's entries: the order of their use).  Each form where it is the better one, caches read
        // from HBM: 16 x 5000 tokens, heads of 64, bf16 s24_r3 24.5 us with two sets, 22.4 with one; 8 x 32768 tokens, 28 / 4 heads of 128,
        // s96_r4 41.6 and 43.1; 64 sequences of 1k to 16k, 4 x 131072 tokens, heads of 64, alike.  (Twelve wavefronts of 168 registers
        // at d_h 128, staging rows in the gaps of the multiplied tables, nothing spilled in the loop, s24_r3: 154.4 where eight take 152.3, and
        // 175 against 163 with bf16 s96_r4: with eight LDS is busy 57 to 70 % of a CU's cycles already, and the vector units issue in 58 to 61 %.)
        FastTile<NW, AB, FLAGS, NH> tile_b;
        Entries k_b = {}, v_b = {};
        auto nothing = [] {};
        constexpr bool kRefill = CPL == 4;
        auto one = [&](int t0, const FastTile<NW, AB, FLAGS, NH> &tile_use, const Entries &k_use, const Entries &v_use,
                       FastTile<NW, AB, FLAGS, NH> &tile_load, Entries &k_load_to, Entries &v_load_to) {
            const bool more = t0 + TS < t_end, more2 = t0 + 2 * TS < t_end;
            const int t1 = more ? t0 + TS : t0, t2 = more2 ? t0 + 2 * TS : t0;
#ifdef HQMQ_STAMPS
            if (tl_ == 0) tl_ = t_loop_ = __builtin_amdgcn_s_memrealtime();
            n_steps_++;
#endif
            auto next_ke = [&] { issue_one(k_side, k_coord, f1.koff, k_load_to); };
            auto next_ve = [&] { issue_one(v_side, v_coord, f1.voff, v_load_to); };
            if constexpr (!kRefill) load_super(t1, tile_load);
            const int w = load_offsets(t2);
            if constexpr (!kRefill) { next_ke(); next_ve(); }
            publish(t0);
            PHASE(0);
            if constexpr (kRefill) half_step(tile_use.h[0], t0, k_use, v_use, next_ke, [&] { load_k(t1, tile_load.h[0]); }, [&] { load_v(t1, tile_load.h[0]); }, next_ve);
            else half_step(tile_use.h[0], t0, k_use, v_use, nothing, nothing, nothing, nothing);
            rebalance(t0);
            offsets_ready(t2, w, f1);
            PHASE(6);
            return more;
        };
        if (t_begin < t_end) {
            int t0 = t_begin;
            while (true) {
                if constexpr (kRefill) {
                    if (!one(t0, cur, kc, vc, cur, kc, vc)) break;
                } else {
                    if (!one(t0, cur, kc, vc, tile_b, k_b, v_b)) break;
                    t0 += TS;
                    if (!one(t0, tile_b, k_b, v_b, cur, kc, vc)) break;
                }
                t0 += TS;
            }
        }
    }
#ifdef HQMQ_STAMPS
    if constexpr (FLAGS) {
        if (lane == 0 && g_stamps) {
            unsigned long long *o = g_stamps + ((size_t)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)) * WV + wave) * 16;
#pragma unroll
            for (int i = 0; i < 7; i++) o[i] = ph_[i];
            o[7] = (unsigned long long)n_steps_;
            o[8] = t_in_;                   // entry, first half-step, last half-step done (the block's merge follows)
            o[9] = t_loop_;
            o[10] = __builtin_amdgcn_s_memrealtime();
            // where the block ran: HW_ID (bits 8-11 CU, 12 SH, 13-15 SE) and XCC_ID (bits 0-3)
            o[11] = (unsigned long long)__builtin_amdgcn_s_getreg(((32 - 1) << 11) | 4) |
                    ((unsigned long long)__builtin_amdgcn_s_getreg(((4 - 1) << 11) | 20) << 32);
            o[12] = (unsigned long long)b;
            o[14] = t_fill_;                // own share of the tables stored, barrier passed
            o[15] = t_bar_;
        }
    }
#endif

    // ---- merge the block's waves through LDS: rows of [d_h accumulators, m, l, pad], one column group at a time ----
    constexpr int RS = d_h + 4;
    float *red = reinterpret_cast<float *>(lds_tab);            // [wave][16 cols][RS]
#pragma unroll
    for (int cgi = 0; cgi < NCG; cgi++) {
        const int cg = cg0 + cgi;
        const float l_tot = row_sum4(l_run[cgi]);
        __syncthreads();
        const int ncols = min(16, p.Tq * G - cg * 16);          // <= 0 for a column group past the end
        if (col < ncols) {                                      // padding columns are never read back
            float *wp = red + ((size_t)wave * 16 + col) * RS;
            if (grp == 0) { wp[d_h] = m_run[cgi]; wp[d_h + 1] = l_tot; }
#pragma unroll
            for (int j = 0; j < CPL; j++) *reinterpret_cast<float4v *>(wp + grp * CPL * 4 + 4 * j) = acc[cgi][j];
        }
        __syncthreads();
        merge_waves<DT, WV, d_h>(p, red, cg, ncols, b, hkv, sp);
    }
#ifdef HQMQ_STAMPS
    if constexpr (FLAGS) {
        if (lane == 0 && g_stamps)
            g_stamps[((size_t)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)) * WV + wave) * 16 + 13] = __builtin_amdgcn_s_memrealtime();
    }
#endif
}

// ---------------------------------------------------------------------------------------------------------------
// Plain 16+0 caches at d_h 128 with tables of at most 2304 codewords (s96_r4 and smaller): the variant whose loads
// all land in LDS (global_load_lds: the data goes from memory to LDS without passing through registers).  Tables,
// the query rows and the first half-step of every wavefront are requested in the prologue; from then on a wavefront
// asks for its next half-step when the current one has arrived and its words have been read out of the slot, so one
// half-step per wavefront is in flight while one is being worked on.  Measured on config 2 at 32k, planes read cold
// from HBM: asking for more ahead (two or three half-steps, before or behind the barrier) floods the memory system,
// and the half-steps that are needed first then arrive behind later ones (first half-step in at 4.4 us median and
// 8.2 us at worst with three ahead, 3.2 / 4.4 us with one); kernel 15.0 - 15.9 us with two or three ahead, 13.2 us
// with one (the register-tile kernel, which keeps two ahead in 40 registers: 15.0 us).
// No tile lives in registers while in flight (111 registers against 145 - 256).  The compiler neither sees these
// loads nor counts them: every wait is written by hand (s_waitcnt vmcnt(n) lets the n youngest requests stay
// outstanding; requests complete in order), and the kernel has no other vector loads before its epilogue.
// LDS: K table at 0, V table at 18432, 4 KB of query rows, 2 KB of radius codes, then per wavefront two slots of
// [256 B scales: K tokens 0..31, V tokens 0..31, the same again][K rows of 32 tokens, 2 KB][V rows, 2 KB].
constexpr int kLdVTab = 2304 * 8;
constexpr int kLdQ = 2 * kLdVTab;
constexpr int kLdRad = kLdQ + 4096;        // the radius codes, see gather_tokens
constexpr int kLdSlot0 = kLdRad + 8 * kRadiusCodes;
constexpr int kLdSlotBytes = 256 + 4096;

// wait until at most `groups` (0..3) groups of five requests are outstanding
__device__ __forceinline__ void wait_groups(int groups) {
    if (groups >= 3) wait_vm<15>();
    else if (groups == 2) wait_vm<10>();
    else if (groups == 1) wait_vm<5>();
    else wait_vm<0>();
}
__device__ __forceinline__ void lds_load16_addr(uint32_t lds_base, const uint8_t *addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(addr) : "memory");
}
__device__ __forceinline__ uint4v lds_read16(uint32_t a) { return *(lds_u4_ptr)(uintptr_t)a; }
__device__ __forceinline__ uint2 lds_read8(uint32_t a) { return __builtin_bit_cast(uint2, *(lds_u2_ptr)(uintptr_t)a); }


constexpr int kLdDepth = 2;

template <int DT, int IB, int WV>
__global__ __launch_bounds__(WV * 64) void attn_lds_kernel(AttnParams p) {
    constexpr int CPL = 8, NW = 4, d_h = 128, mrb = 64;
    extern __shared__ uint2 lds_tab[];
#ifdef HQMQ_STAMPS
    unsigned long long st_[16] = {};
#endif
    STAMP(0);
    // Everything the first requests need is read from the argument block in one go (the empty asm below is where
    // all of it has to be there): read where it is used, every group of arguments costs its own round trip.
    // The grid is (n_splits, column groups, B * Hkv): taken from the arguments, which spares the dispatch packet.
    const unsigned gx = (unsigned)p.n_splits, gy = (unsigned)p.n_cg, gz = (unsigned)(p.B * p.Hkv);
    const int Hkv = p.Hkv, remap = p.xcd_remap;
    const unsigned m_gz = p.m_gz, m_gx = p.m_gx, m_hkv = p.m_hkv;
    const int32_t *order_p = p.batch_order, *len_p = p.kv_len, *start_p = p.kv_start;
    const uint8_t *kj = (const uint8_t *)p.Kc.joint, *vj = (const uint8_t *)p.Vc.joint;
    const int64_t kjsh = p.Kc.jsh, vjsh = p.Vc.jsh;
    const int KK = p.Kc.K, KV = p.Vc.K, Tkv = p.Tkv, Bn = p.B;
    asm volatile("" ::"s"(gx), "s"(gy), "s"(gz), "s"(Hkv), "s"(remap), "s"(m_gz), "s"(m_gx), "s"(m_hkv), "s"(order_p), "s"(len_p), "s"(start_p),
                 "s"(kj), "s"(vj), "s"(kjsh), "s"(vjsh), "s"(KK), "s"(KV), "s"(Tkv), "s"(Bn));
    int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    if (remap) {
        const unsigned lin = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
        const unsigned r = fast_div(lin, gz, m_gz);
        bz = (int)(lin - r * gz);
        by = (int)fast_div(r, gx, m_gx);
        bx = (int)(r - (unsigned)by * gx);
    }
    const int slot = (int)fast_div((unsigned)bz, (unsigned)Hkv, m_hkv), hkv = bz - slot * Hkv;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#ifdef HQMQ_STAMPS
    asm volatile("" ::"s"(hkv));
    STAMP(15);
#endif
    // the per-sequence words of ragged batches are read before the first request goes out: behind one, the wait for
    // such a word would also wait for every request in flight
    const int b = order_p ? min(max(uniform_word(order_p, slot), 0), Bn - 1) : slot;
    int kv_end = len_p ? uniform_word(len_p, b) : Tkv;
    kv_end = min(max(kv_end, 0), Tkv);
    const int kv_first = start_p ? max(uniform_word(start_p, b), 0) : 0;
    // ---- tables ----
    {
        const uint8_t *ksrc = uniform_ptr(kj + (size_t)hkv * kjsh * 2);
        const uint8_t *vsrc = uniform_ptr(vj + (size_t)hkv * vjsh * 2);
        land_tables<WV>(ksrc, (uint32_t)KK * 8u, vsrc, (uint32_t)KV * 8u, 0u, kLdVTab, wave, lane);
    }
    STAMP(1);
    const int bh = b * p.Hkv + hkv;
    const int cg = by, sp = bx;
    const int G = p.G;
    const int col = lane & 15, grp = lane >> 4;
    const int ncols = min(16, p.Tq * G - cg * 16);
    const int cidx = cg * 16 + col;
    const bool col_ok = col < ncols;
    const int tq = col_ok ? (int)fast_div((unsigned)cidx, (unsigned)G, p.m_G) : 0;
    int col_lim, blk_lim, lim_min;
    {
        int64_t lim64 = kv_end;
        if (p.causal) lim64 = min(lim64, (int64_t)tq + p.causal_offset + 1);
        if (!col_ok || lim64 < 0) lim64 = 0;
        col_lim = (int)lim64;
        blk_lim = col_lim;
        lim_min = col_ok ? col_lim : 0x7fffffff;
    }
    if (p.causal) {
        for (int o = 1; o < 16; o <<= 1) {
            blk_lim = max(blk_lim, __shfl_xor(blk_lim, o));
            lim_min = min(lim_min, __shfl_xor(lim_min, o));
        }
        blk_lim = __builtin_amdgcn_readfirstlane(blk_lim);
        lim_min = __builtin_amdgcn_readfirstlane(lim_min);
    } else {
        blk_lim = lim_min = kv_end;
    }
    const int col_start = min(kv_first, blk_lim);
    const int blk_lo = col_start / kSuper * kSuper;
    int per_split = (int)fast_div((unsigned)(blk_lim - blk_lo + p.n_splits - 1), (unsigned)p.n_splits, p.m_splits);
    per_split = (per_split + kSuper - 1) / kSuper * kSuper;
    const int b_begin = min(blk_lo + sp * per_split, blk_lim), b_end = min(blk_lim, b_begin + per_split);
    constexpr int TS = 32 * WV;
    const int t_begin = min(b_begin + wave * 32, b_end), t_end = b_end;
    const int n_hs = __builtin_amdgcn_readfirstlane(t_begin < t_end ? (t_end - t_begin + TS - 1) / TS : 0);
    const size_t plane_row0 = (size_t)bh * p.t_cap;
    const int idx_bits = p.idx_bits;
    // instruction offsets count for the memory and the LDS side alike: the bases are moved back by the slot offsets
    const uint8_t *k_rows = p.Kc.main_plane + plane_row0 * mrb - 256;
    const uint8_t *v_rows = p.Vc.main_plane + plane_row0 * mrb - 2304;
    const uint32_t main_off = (uint32_t)(col * mrb + grp * 16), vmain_off = 16u * (uint32_t)lane;    // V: see gather_tokens
    // scales: lanes 0..15 fetch the K scales of tokens 2 lane, 2 lane + 1, lanes 16..31 the V scales; the upper half repeats
    const uint8_t *sc_lane = (lane & 16) ? (const uint8_t *)((const uint16_t *)p.Vc.scale_plane + b * p.Vc.ssb + hkv * p.Vc.ssh)
                                         : (const uint8_t *)((const uint16_t *)p.Kc.scale_plane + b * p.Kc.ssb + hkv * p.Kc.ssh);
    sc_lane += 4 * (lane & 15);
    const uint32_t slot_base = (uint32_t)(kLdSlot0 + wave * kLdDepth * kLdSlotBytes);
    auto request = [&](int th, uint32_t slot_lds) {
        const uint8_t *kb = uniform_ptr(k_rows + (size_t)th * mrb), *vb = uniform_ptr(v_rows + (size_t)th * mrb);
        const uint8_t *sa = sc_lane + 2 * (size_t)th;
        asm volatile("s_mov_b32 m0, %0\n\t"
                     "s_nop 0\n\t"
                     "global_load_lds_dwordx4 %2, %3 offset:256\n\t"
                     "global_load_lds_dwordx4 %2, %3 offset:1280\n\t"
                     "global_load_lds_dword %1, off\n\t"
                     "global_load_lds_dwordx4 %5, %4 offset:2304\n\t"
                     "global_load_lds_dwordx4 %5, %4 offset:3328"
                     ::"s"(slot_lds), "v"(sa), "v"(main_off), "s"(kb), "s"(vb), "v"(vmain_off) : "memory");
    };
    // ---- query rows (first wavefront): column c of the block at kLdQ + 256 c, raw 16-bit values ----
    if (wave == 0) {
        for (int i = 0; 4 * i < ncols; i++) {       // four columns per request; a decode step of G <= 4 heads takes one
            const int c = min(4 * i + (lane >> 4), ncols - 1);              // lanes past the last real column repeat it (never read)
            const int ci = cg * 16 + c;
            const int tqc = (int)fast_div((unsigned)ci, (unsigned)G, p.m_G), hqc = hkv * G + (ci - tqc * G);
            const uint8_t *qa = (const uint8_t *)((const uint16_t *)p.Q + b * p.qsb + hqc * p.qsh + (int64_t)tqc * p.qst) + 16 * (lane & 15);
            lds_load16_addr((uint32_t)(kLdQ + 1024 * i), qa);
        }
    }
    // the first half-step; the later ones are requested from inside the loop, one ahead
    if (n_hs > 0) request(t_begin, slot_base);
    STAMP(2);
    if (threadIdx.x < kRadiusCodes) {
        const half4 r = half4{1, 1, 1, 1} * (_Float16)(uint16_t)threadIdx.x;
        lds_tab[kLdRad / 8 + threadIdx.x] = __builtin_bit_cast(uint2, r);
    }
    wait_groups(n_hs > 0 ? 1 : 0);            // tables (and query rows) in: only the tile request may still be outstanding
    __builtin_amdgcn_s_waitcnt(0xc07f);         // lgkmcnt(0): the radius codes are in LDS
    STAMP(3);
    asm volatile("s_barrier" ::: "memory");
    if constexpr (DT != HQMQ_F16) {
        // the tables landed in the cache dtype: converted to fp16 in place, two codewords per thread and round
        for (int k = threadIdx.x; k < (2 * kLdVTab) / 16; k += WV * 64) {
            const uint4v w = pair_to_half<DT>(lds_read16((uint32_t)k * 16u));
            *(uint4v __attribute__((address_space(3))) *)(uintptr_t)((uint32_t)k * 16u) = w;
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);         // lgkmcnt(0): the stores are in LDS
        asm volatile("s_barrier" ::: "memory");
    }
    STAMP(4);
    half8 qf[CPL / 2];
#pragma unroll
    for (int j = 0; j < CPL / 2; j++) {
        const uint4v w = lds_read16((uint32_t)(kLdQ + col * 256 + grp * 64 + 16 * j));
        const half4 lo = chunk_to_half<DT>(uint2{w[0], w[1]}), hi = chunk_to_half<DT>(uint2{w[2], w[3]});
        const half4 z = half4{0, 0, 0, 0};
        qf[j] = cat8(col_ok ? lo : z, col_ok ? hi : z);
    }

    const float c = p.c_log2;
    float m_run = -INFINITY, l_run = 0.f;
    float4v acc[CPL];
#pragma unroll
    for (int j = 0; j < CPL; j++) acc[j] = float4v{0.f, 0.f, 0.f, 0.f};
    const float4v zero4 = float4v{0.f, 0.f, 0.f, 0.f};
    int ring = 0;
    for (int i = 0, th = t_begin; i < n_hs; i++, th += TS) {
        const uint32_t sl = slot_base + (uint32_t)ring * kLdSlotBytes, sl_next = slot_base + (uint32_t)(ring ^ 1) * kLdSlotBytes;
        ring ^= 1;
        // The hardware prefers the older of the two wavefronts of a SIMD, which then ends 1.7 us before the younger and
        // leaves it to finish alone.  Priority by work left (finer towards the end) lets the one that is behind go first,
        // so that the two finish together (kernel -0.3 us).
        const int left = n_hs - i;
        if (left >= 3) __builtin_amdgcn_s_setprio(3);
        else if (left == 2) __builtin_amdgcn_s_setprio(3);
        else __builtin_amdgcn_s_setprio(1);
        wait_groups(0);
#ifdef HQMQ_STAMPS
        { const unsigned long long t_ = __builtin_amdgcn_s_memrealtime();
          if (i == 0) st_[5] = t_; else if (i == 1) st_[7] = t_; else if (i == 2) st_[9] = t_; else if (i == 3) st_[11] = t_; }
#endif
        uint4v kw[2], vw[2];
        uint2 ks[2], vs[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            kw[u] = lds_read16(sl + 256u + 1024u * u + 16u * (uint32_t)lane);
            ks[u] = lds_read8(sl + 32u * u + 8u * (uint32_t)grp);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            vw[u] = lds_read16(sl + 2304u + 1024u * u + 16u * (uint32_t)lane);
            vs[u] = lds_read8(sl + 64u + 32u * u + 8u * (uint32_t)grp);
        }
        // the words of this half-step are in registers: ask for the next one (into the other slot)
        asm volatile("" : "+v"(kw[0]), "+v"(kw[1]), "+v"(vw[0]), "+v"(vw[1]), "+v"(ks[0]), "+v"(ks[1]), "+v"(vs[0]), "+v"(vs[1]));
        if (i + 1 < n_hs) request(th + TS, sl_next);

        float4v sT[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            half4 g[CPL], a[CPL];
            half2v r[CPL / 2];
            const uint32_t w[NW] = {kw[u][0], kw[u][1], kw[u][2], kw[u][3]};
            gather_chunks<CPL, 16, 0, IB, NW, 0, false>(w, 0u, idx_bits, g, r);
            scale_chunks<CPL, false>(g, r, a);
            float4v s = zero4;
#pragma unroll
            for (int jj = 0; jj < CPL / 2; jj++) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(cat8(a[2 * jj], a[2 * jj + 1]), qf[jj], s, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; e++) s[e] = scaled<DT>(s[e], e < 2 ? ks[u].x : ks[u].y, e & 1, 0.f);
            sT[u] = s;
        }
        const bool edge = !(th + 32 <= lim_min && th + 32 <= t_end && th >= col_start);
        if (edge) {
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int t = th + 16 * u + 4 * grp + e;
                    if (!(t < col_lim && t < t_end && t >= col_start)) sT[u][e] = -INFINITY;
                }
        }
        float tmax = fmaxf(fmaxf(fmaxf(sT[0][0], sT[0][1]), fmaxf(sT[0][2], sT[0][3])), fmaxf(fmaxf(sT[1][0], sT[1][1]), fmaxf(sT[1][2], sT[1][3])));
        tmax = row_max4(tmax);
        const float m_new = fmaxf(m_run, tmax);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        if (__builtin_amdgcn_ballot_w64(m_new != m_run) != 0) {
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * c);
            l_run *= alpha;
#pragma unroll
            for (int j = 0; j < CPL; j++) acc[j] = acc[j] * alpha;
            m_run = m_new;
        }
        const float mc = -m_use * c;
        half4 pT[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            float pe[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                pe[e] = __builtin_amdgcn_exp2f(fmaf(sT[u][e], c, mc));
                l_run += pe[e];
            }
            pT[u] = weigh<DT>(pe, vs[u]);
        }
        const half8 pp = cat8(pT[0], pT[1]);
        if (left == 2) __builtin_amdgcn_s_setprio(2);
        else if (left == 1) __builtin_amdgcn_s_setprio(0);
        half4 av[2][CPL];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const uint32_t w[NW] = {vw[u][0], vw[u][1], vw[u][2], vw[u][3]};
            gather_tokens<CPL, 16, 0, IB, NW, kLdVTab, kLdRad>(w, 0u, idx_bits, av[u]);
        }
#pragma unroll
        for (int j = 0; j < CPL; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cat8(av[0][j], av[1][j]), pp, acc[j], 0, 0, 0);
#ifdef HQMQ_STAMPS
        asm volatile("" ::"v"(acc[0]), "v"(acc[7]));
        { const unsigned long long t_ = __builtin_amdgcn_s_memrealtime();
          if (i == 0) st_[6] = t_; else if (i == 1) st_[8] = t_; else if (i == 2) st_[10] = t_; else if (i == 3) st_[12] = t_; }
#endif
    }

    // ---- merge the block's wavefronts through LDS: rows of [d_h accumulators, m, l, pad] ----
    constexpr int RS = d_h + 4;
    float *red = reinterpret_cast<float *>(lds_tab);
    const float l_tot = row_sum4(l_run);
    __syncthreads();
    if (col < ncols) {
        float *wp = red + ((size_t)wave * 16 + col) * RS;
        if (grp == 0) { wp[d_h] = m_run; wp[d_h + 1] = l_tot; }
#pragma unroll
        for (int j = 0; j < CPL; j++) *reinterpret_cast<float4v *>(wp + grp * CPL * 4 + 4 * j) = acc[j];
    }
    __syncthreads();
    STAMP(13);
    merge_waves<DT, WV, d_h>(p, red, cg, ncols, b, hkv, sp);
#ifdef HQMQ_STAMPS
    STAMP(14);
    if (lane == 0 && g_stamps) {
        unsigned long long *o = g_stamps + ((size_t)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)) * WV + wave) * 16;
#pragma unroll
        for (int i = 0; i < 16; i++) o[i] = st_[i];
    }
#endif
}

template <int DT, int IB, int WV>
static int launch_lds_waves(const AttnParams &p, dim3 grid, hipStream_t st, const LaunchTiming &tm) {
    constexpr size_t kTiles = (size_t)kLdSlot0 + (size_t)WV * kLdDepth * kLdSlotBytes;
    constexpr size_t kMerge = (size_t)WV * 16 * (128 + 4) * sizeof(float);
    constexpr size_t shmem = kTiles > kMerge ? kTiles : kMerge;
    static_assert(shmem <= 160 * 1024, "LDS of one CU");
    auto kern = attn_lds_kernel<DT, IB, WV>;
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
    if (e != hipSuccess) return (int)e;
    launch_timed(kern, grid, dim3(WV * 64), shmem, st, tm, p);
    return hip_status(hipGetLastError());
}
template <int DT, int IB>
static int launch_lds(const AttnParams &p, dim3 grid, hipStream_t st, const LaunchTiming &tm) {
    // (four-wavefront blocks for short ranges measured no faster: 8.9 against 8.7 us per step at 4k tokens)
    return launch_lds_waves<DT, IB, kFastWaves>(p, grid, st, tm);
}

template <int CPL, int MB, int AB, int IB, int DT, int WV = kFastWaves, int NCG = 1, bool F8 = false>
static int launch_one(const AttnParams &p, bool flags, dim3 grid, hipStream_t st, const LaunchTiming &tm) {
    if (NCG > 1) grid.y = (grid.y + NCG - 1) / NCG;
    // LDS: K table at 0, V table at kVTabOffset; reused afterwards for the cross-wave merge [wave][16][d_h + 4] floats
    constexpr bool PS = is_prescaled(MB, AB, IB);
    size_t shmem = flags ? (size_t)stage_offset(PS) + (size_t)(CPL == 4 ? WV : kFastWaves) * stage_bytes(PS, CPL) : PS ? (size_t)2 * kPsTabBytes : (size_t)kVTabOffset + (size_t)p.Vc.K * 8;
    if (!flags || !PS) shmem += 64;        // the wavefronts' progress slots
    const size_t merge = (size_t)WV * 16 * (16 * CPL + 4) * sizeof(float);     // WV >= the wavefronts actually launched
    if (shmem < merge) shmem = merge;
    // Long sequences of different lengths, whole and started longest first, one or two for every compute unit: the longest bounds the call and is
    // slowed by a block beside it, so each gets a unit of its own, by asking for more than half the LDS.  Two blocks -> one, 44 / 52 /
    // 64 sequences of up to 8000 tokens, 64 / 8 heads of 64, bf16, uniform lengths: s192_r6 50.6 -> 41.5 / 56.0 -> 45.5 / 61.9 -> 55.1 us,
    // s192_r4 44.6 -> 40.6 / 47.7 -> 43.3 / 53.8 -> 53.2; exponential ones 41.2 -> 38.3 and 41.4 -> 40.1 (44 sequences), the upper half of a
    // uniform distribution 66.4 -> 60.2 and 58.5 -> 58.9.  At 4000 tokens both measure alike (64 sequences, uniform: 32.6 -> 31.2, 30.8 -> 31.2),
    // at 3000 two are faster (24.4 against 27.0), as with 576 blocks (72 of 5000 44.8 against 49.6) and over equal lengths (3 to 16 %).
    if (two_blocks(CPL, MB, AB, IB, flags, WV, NCG) && AB && p.kv_len && p.batch_order && p.n_splits == 1 && p.Tkv >= 4000) {
        const int64_t blocks = (int64_t)grid.x * grid.y * grid.z;
        if (blocks > 256 && blocks <= 512 && shmem < 84 * 1024) shmem = 84 * 1024;
    }
    constexpr int WF = CPL == 4 ? WV : kFastWaves;      // outlier variants fit three wavefronts per SIMD only at d_h 64
    auto kern = flags ? attn_fast_kernel<CPL, MB, AB, IB, DT, true, WF, 1, F8> : attn_fast_kernel<CPL, MB, AB, IB, DT, false, WV, NCG, F8>;
    if (shmem > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
        if (e != hipSuccess) return (int)e;
    }
    launch_timed(kern, grid, dim3((flags ? WF : WV) * 64), shmem, st, tm, p);
    return hip_status(hipGetLastError());
}

template <int CPL, int DT>
static int launch_layout(const AttnParams &p, int mb, bool flags, dim3 grid, hipStream_t st, const LaunchTiming &tm, bool *handled) {
    if (p.Kc.K > kTabMax || p.Vc.K > kTabMax) return HQMQ_OK;     // tables beyond the fixed LDS slots
    if (!attn_radius_in_table(mb, p.aux_bits, p.idx_bits)) return HQMQ_OK;
    // the kernels divide by multiplication only (fast_div): sizes for which a multiplier cannot be promised (index times
    // divisor beyond 2^32: millions of tokens times thousands of splits) stay with the layout-generic kernel
    if ((p.Hkv > 1 && !p.m_hkv) || (p.G > 1 && !p.m_G) || (p.n_splits > 1 && !p.m_splits)) return HQMQ_OK;
    // the outlier variants keep their staging rows behind a smaller V slot
    if (flags && (p.Kc.K > kFlagsTabMax || p.Vc.K > kFlagsTabMax)) return HQMQ_OK;
    // tables are read two codewords (16 bytes) at a time
    if ((p.Kc.K & 1) || (p.Vc.K & 1) || (p.Kc.jsh & 7) || (p.Vc.jsh & 7) || (((uintptr_t)p.Kc.joint | (uintptr_t)p.Vc.joint) & 15))
        return HQMQ_OK;
    *handled = true;
    // Long ranges per block run with twelve wavefronts, three per SIMD, which hide more of each other's waits than the extra partials
    // of the block's merge cost; the variants that need more than 168 registers stay at eight: from 4096 tokens on over plain caches, from 1536 on
    // over outlier caches at d_h 64.  (The lines lie a little above where both measured alike in the kernels' first twelve-wavefront form, with 224
    // blocks: d_h 128 plain 3000 tokens, 4000 / 5500 tokens of s96_r4 30.1 -> 29.1 / 38.3 -> 36.3 us; d_h 64 over outlier caches 1200, 3000 / 5500 tokens
    // 26.1 -> 23.3 / 42.3 -> 36.3 us; d_h 64 plain 4000, 8000 tokens 34.4 -> 32.3 us.)  d_h 64 plain only while no compute unit holds two blocks of
    // eight (480 blocks of 4000 tokens 33.3 against 38.2 us).
    const int range = p.Tkv / p.n_splits;
    const int64_t blocks = (int64_t)grid.x * grid.y * grid.z;
    // Where the kernel whose loads land in LDS can take the call it keeps it up to 5000 tokens a block if there is a block for every compute unit;
    // with fewer, loads come back sooner and twelve wavefronts are ahead.  us landing / twelve wavefronts, 4100, 4600 and 4900 tokens, codebooks of 288
    // (bf16), 576 (fp16) and 2304 codewords (fp16, bf16): 256 blocks 31.5..33.0 / 32.8..33.1, 34.2..35.2 / 35.6..35.7, 38.1..38.3 / 37.6..39.0; 384 blocks 54.9..56.6 /
    // 57.1..57.6, 60.3..62.8 / 61.4..62.1, 63.8..66.1 / 64.9..65.6; 224 blocks, alike, 29.5..29.9 / 29.7..30.5, 32.2..32.6 / 31.7..32.2, 33.3..35.0 / 33.6..34.0; 160 blocks
    // 27.7..28.9 / 26.9..27.9, 30.4..31.9 / 29.1..30.3, 32.2..33.6 / 30.7..31.9.
    const bool lands = CPL == 8 && mb == 16 && p.aux_bits == 0 && !flags && !p.no_lds_landing && p.Kc.K <= 2304 && p.Vc.K <= 2304 && p.Kc.K >= 2 && p.Vc.K >= 2 &&
                       ((((uintptr_t)p.Q) | (uintptr_t)(p.qsb * 2) | (uintptr_t)(p.qsh * 2) | (uintptr_t)(p.qst * 2)) & 15) == 0;
    const bool wide = CPL == 8 ? !flags && range >= (lands && blocks >= 256 ? 5000 : 4096) : flags ? range >= 1536 : range >= 4096 && blocks <= 256;
    const bool two = attn_two_groups(p.n_cg, flags, (int64_t)p.n_splits * p.n_cg * p.B * p.Hkv, range, p.n, p.aux_bits);
    // tables of e4m3 numbers kept as float8 in LDS, on request (decode shapes of the 16-bit layouts at d_h 128)
    if (p.tab_fp8 && CPL == 8 && !two) {
        if (mb == 16 && p.aux_bits == 0 && p.idx_bits == 12) return launch_one<8, 16, 0, 12, DT, kFastWaves, 1, true>(p, flags, grid, st, tm);
        if (mb == 16 && p.aux_bits == 3 && p.idx_bits == 13 && p.Kc.K <= 4608) return launch_one<8, 16, 3, 13, DT, kFastWaves, 1, true>(p, flags, grid, st, tm);
    }
    // plain 16+0 caches with small tables at d_h 128, one column group, eight wavefronts: every load lands in LDS
    if constexpr (CPL == 8) {
        if (lands && !two && !wide)
            return p.idx_bits == 12 ? launch_lds<DT, 12>(p, grid, st, tm) : launch_lds<DT, 0>(p, grid, st, tm);
    }
    if (mb == 16 && p.aux_bits == 0 && p.idx_bits == 12) {
        if (two) return launch_one<CPL, 16, 0, 12, DT, kFastWaves, 2>(p, flags, grid, st, tm);
        return wide ? launch_one<CPL, 16, 0, 12, DT, 12>(p, flags, grid, st, tm) : launch_one<CPL, 16, 0, 12, DT>(p, flags, grid, st, tm);
    }
    if (mb == 16 && p.aux_bits == 0) {
        if (two) return launch_one<CPL, 16, 0, 0, DT, kFastWaves, 2>(p, flags, grid, st, tm);
        return wide ? launch_one<CPL, 16, 0, 0, DT, 12>(p, flags, grid, st, tm) : launch_one<CPL, 16, 0, 0, DT>(p, flags, grid, st, tm);
    }
    // Heads of 64 take these layouts here as well.  Before, the layout-generic kernel had them: 8 sequences x 3000 tokens, 64 / 8 heads,
    // 28.8 (s24_r3 fp16) to 47.3 us (s192_r6 bf16), with verbatim chunks 52 to 83, 40 queries each then 940 to 1350; now 14.3 to
    // 14.8, 16.7 to 17.3 and 133 to 142 us.  Tables multiplied out pay there too (4 x 32000 tokens 32.7 without them, 28.8 with).
    if (mb == 12 && p.aux_bits == 1 && p.idx_bits == 10 && p.Kc.K <= kPsKMax && p.Vc.K <= (flags ? 1016 : kPsKMax)) {
        if (two) return launch_one<CPL, 12, 1, 10, DT, kFastWaves, 2>(p, flags, grid, st, tm);
        return wide ? launch_one<CPL, 12, 1, 10, DT, 12>(p, flags, grid, st, tm) : launch_one<CPL, 12, 1, 10, DT>(p, flags, grid, st, tm);
    }
    if (mb == 12 && p.aux_bits == 1) return launch_one<CPL, 12, 1, 0, DT>(p, flags, grid, st, tm);
    // (the 16+3 decode needs 182 registers at d_h 128: at three wavefronts per SIMD it spills and runs 40 % slower)
    if constexpr (CPL == 4) {
        if (wide && mb == 16 && p.aux_bits == 3 && p.idx_bits == 13 && p.Kc.K <= 4608) return launch_one<CPL, 16, 3, 13, DT, 12>(p, flags, grid, st, tm);
        if (wide && mb == 16 && p.aux_bits == 1) return launch_one<CPL, 16, 1, 0, DT, 12>(p, flags, grid, st, tm);
    }
    if (mb == 16 && p.aux_bits == 3 && p.idx_bits == 13 && p.Kc.K <= 4608)
        return two ? launch_one<CPL, 16, 3, 13, DT, kFastWaves, 2>(p, flags, grid, st, tm) : launch_one<CPL, 16, 3, 13, DT>(p, flags, grid, st, tm);
    if (mb == 16 && p.aux_bits == 3) return launch_one<CPL, 16, 3, 0, DT>(p, flags, grid, st, tm);
    // 16 + 1 bits (s192 with four radius bits, the shape of the reference's published prefill figure): generic field decode
    if (mb == 16 && p.aux_bits == 1)
        return two ? launch_one<CPL, 16, 1, 0, DT, kFastWaves, 2>(p, flags, grid, st, tm) : launch_one<CPL, 16, 1, 0, DT>(p, flags, grid, st, tm);
    // the remaining widths the layout rule produces (16 + 2: s96_r6, s192_r5; 12 + 2: s24_r4; 12 + 3: s96_r3, s24_r5), generic
    // field decode: five times faster than the layout-generic kernel at batch 8
    if (mb == 16 && p.aux_bits == 2)
        return two ? launch_one<CPL, 16, 2, 0, DT, kFastWaves, 2>(p, flags, grid, st, tm) : launch_one<CPL, 16, 2, 0, DT>(p, flags, grid, st, tm);
    if (mb == 12 && p.aux_bits == 2)
        return two ? launch_one<CPL, 12, 2, 0, DT, kFastWaves, 2>(p, flags, grid, st, tm) : launch_one<CPL, 12, 2, 0, DT>(p, flags, grid, st, tm);
    if (mb == 12 && p.aux_bits == 3)
        return two ? launch_one<CPL, 12, 3, 0, DT, kFastWaves, 2>(p, flags, grid, st, tm) : launch_one<CPL, 12, 3, 0, DT>(p, flags, grid, st, tm);
    *handled = false;
    return HQMQ_OK;
}

#ifdef HQMQ_STAMPS
extern "C" int hqmq_debug_set_stamps(void *ptr) { return (int)hipMemcpyToSymbol(HIP_SYMBOL(g_stamps), &ptr, sizeof(ptr)); }
#endif

int launch_attn_fast(const AttnParams &p, int main_bits, bool flags, dim3 grid, size_t table_bytes, hipStream_t st,
                     const LaunchTiming &tm, bool *handled) {
    (void)table_bytes;
    *handled = false;
    if (p.dtype != HQMQ_F16 && p.dtype != HQMQ_BF16) return HQMQ_OK;
    // The kernels of this file round P * (V scale) and verbatim chunks to fp16: a bf16 cache whose scales reach 2^15 (the caller says so: wide_range) takes the layout-generic kernel, which carries the range guard.
    if (p.wide_range) return HQMQ_OK;
    if (p.n != 16 && p.n != 32) return HQMQ_OK;
    if (p.t_cap % kSuper) return HQMQ_OK;
    // vector loads of plane rows: main rows 16-byte aligned (checked by the caller), aux and flag rows to their width
    if (p.aux_bits && (((uintptr_t)p.Kc.aux_plane | (uintptr_t)p.Vc.aux_plane) & 3)) return HQMQ_OK;
    if (flags && (!p.Kc.sb_coord || !p.Kc.sb_count || !p.Vc.sb_coord || !p.Vc.sb_count || p.Kc.sb_cap < 2 || p.Vc.sb_cap < 2 || p.Kc.sb_cap >= (1 << 28) || p.Vc.sb_cap >= (1 << 28)))
        return HQMQ_OK;     // the K side walks the entry list
    // 8-byte vector loads of Q rows, table rows and sideband chunks; strides were checked by the caller
    if (p.n == 32) {
        if (p.dtype == HQMQ_F16) return launch_layout<8, HQMQ_F16>(p, main_bits, flags, grid, st, tm, handled);
        return launch_layout<8, HQMQ_BF16>(p, main_bits, flags, grid, st, tm, handled);
    }
    if (p.dtype == HQMQ_F16) return launch_layout<4, HQMQ_F16>(p, main_bits, flags, grid, st, tm, handled);
    return launch_layout<4, HQMQ_BF16>(p, main_bits, flags, grid, st, tm, handled);
}

}  // namespace hqmq
