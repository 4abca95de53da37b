// Dense decode kernels and the code packer.
//   hqmq_dequant         unpacked codes -> dense, rounding of _decode_kv_torch
//                        (src/quantizers/hqmq_attention.py:39-65 of the reference);
//                        replaces hqmq_decode_triton (src/quantizers/hqmq_kernel.py:102-132)
//   hqmq_pack_codes      unpacked int32 codes -> packed main/aux rows
//   hqmq_pack_kv         unpacked int32 codes and scales of K and V -> all planes, in one launch
//   hqmq_dequant_packed  packed cache (+ outlier sideband) -> dense
// Compiled with -ffp-contract=off: every product rounds to D on its own.
#include "common.h"
#include <algorithm>

namespace hqmq {

// bits [bitpos, bitpos+nbits) of a little-endian bit stream held in `row` (row_bytes long)
__device__ __forceinline__ uint32_t read_bits(const uint8_t *row, int row_bytes, int bitpos, int nbits) {
    uint32_t v = 0;
    int byte = bitpos >> 3, sh = bitpos & 7, got = 0;
    while (got < nbits && byte < row_bytes) {
        v |= ((uint32_t)row[byte] >> sh) << got;
        got += 8 - sh;
        sh = 0;
        byte++;
    }
    return nbits >= 32 ? v : (v & ((1u << nbits) - 1u));
}

// PER chunks per thread (2: 16-bit types, even rows, aligned operands: 8-byte loads of the codes, 16-byte stores of the
// values); a row of the grid is one (b, h).  Bound by memory: 16 bytes in, 8 out and a gathered codeword per chunk of a
// 16-bit type.  fp16, B = 1, 8 heads, 4096 tokens of 128: 6.7 us against 13.9 with a chunk per thread and 64-bit index
// divisions.
template <class D, int PER>
__global__ __launch_bounds__(256) void dequant_kernel(const int32_t *idx, int64_t isb, int64_t ish, int64_t ist, const int32_t *rq, int64_t rsb_,
                               int64_t rsh_, int64_t rst_, const typename D::storage *rs, int64_t ssb, int64_t ssh,
                               int64_t sst, const typename D::storage *joint, int64_t jsh, int K, int BH, int H, int T, int n,
                               int qmax, typename D::storage *out) {
    using ST = typename D::storage;
    const uint32_t per_row = (uint32_t)n / PER;
    for (int bh = blockIdx.y; bh < BH; bh += gridDim.y) {
        const int b = bh / H, h = bh - b * H;
        const int32_t *ib = idx + b * isb + h * ish, *rb = rq + b * rsb_ + h * rsh_;
        const ST *sb = rs + b * ssb + h * ssh, *jb = joint + h * jsh;
        ST *ob = out + (int64_t)bh * T * n * 4;
        for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g < (int64_t)T * per_row; g += (int64_t)gridDim.x * 256) {
            const uint32_t t = g <= 0xffffffffll ? (uint32_t)g / per_row : (uint32_t)(g / per_row);
            const int c = (int)(g - (int64_t)t * per_row) * PER;
            int k[PER], q[PER];
            if constexpr (PER == 2) {
                const int2 kv = *reinterpret_cast<const int2 *>(ib + t * ist + c), qv = *reinterpret_cast<const int2 *>(rb + t * rst_ + c);
                k[0] = kv.x; k[1] = kv.y; q[0] = qv.x; q[1] = qv.y;
            } else {
                k[0] = ib[t * ist + c];
                q[0] = rb[t * rst_ + c];
            }
            const float s = D::load(sb + t * sst);
            ST v[4 * PER];
#pragma unroll
            for (int i = 0; i < PER; i++) {
                const int ki = k[i] < 0 ? 0 : (k[i] >= K ? K - 1 : k[i]);
                const float r = D::rnd(D::rnd(D::rnd((float)q[i]) * s) / (float)qmax);
                const ST *cw = jb + (int64_t)ki * 4;
                if constexpr (PER == 2) {
                    const uint2 w = *reinterpret_cast<const uint2 *>(cw);
                    const ST e[4] = {(ST)w.x, (ST)(w.x >> 16), (ST)w.y, (ST)(w.y >> 16)};
#pragma unroll
                    for (int j = 0; j < 4; j++) D::store(v + 4 * i + j, D::rnd(D::load(e + j) * r));
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++) D::store(v + 4 * i + j, D::rnd(D::load(cw + j) * r));
                }
            }
            ST *dst = ob + ((int64_t)t * n + c) * 4;
            if constexpr (PER == 2) {
                uint4 w;
                w.x = (uint32_t)v[0] | (uint32_t)v[1] << 16; w.y = (uint32_t)v[2] | (uint32_t)v[3] << 16;
                w.z = (uint32_t)v[4] | (uint32_t)v[5] << 16; w.w = (uint32_t)v[6] | (uint32_t)v[7] << 16;
                *reinterpret_cast<uint4 *>(dst) = w;
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) dst[j] = v[j];
            }
        }
    }
}

// The unpacked codes of K and V -> the planes that attention reads, one launch: a thread packs eight chunks of a row (of
// the last group of a row perhaps four), rows T .. t_cap - 1 are written as zeros, so that the planes need no clearing, and
// the largest finite scale goes to *scale_max.  Bound by reading the 8 bytes of a chunk: 2048 tokens of 8 heads of 128,
// 16.8 MB: 5.1 us for both tensors; packed a byte per thread they took 15 us each, and 8 launches for clearing and copying.
struct PackSide {
    const int32_t *idx, *rq;
    int64_t isb, ish, ist, rsb, rsh, rst;
    const void *scale_in;
    int64_t ssb, ssh, sst;
    uint8_t *main_plane, *aux_plane;
    void *scale_plane;
    uint32_t *scale_max;
    int T, vec;             // vec: the rows of idx and rq can be read 16 bytes at a time
};
struct PackPair { PackSide s[2]; };

template <class D, int MB>
__global__ __launch_bounds__(256) void pack_kv_kernel(PackPair pair, int BH, int H, int n, int idx_bits, int ab, int t_cap) {
    using ST = typename D::storage;
    const PackSide &p = pair.s[blockIdx.z];
    const int groups = (n + 7) >> 3, mrb = n * MB / 8, arb = (n * ab + 7) >> 3;
    const uint32_t g = blockIdx.x * 256u + threadIdx.x, t = g / (uint32_t)groups, grp = g - t * (uint32_t)groups;
    const uint32_t idx_mask = (1u << idx_bits) - 1u;
    uint32_t most = 0;
    if (t < (uint32_t)t_cap)
        for (int bh = blockIdx.y; bh < BH; bh += gridDim.y) {
            const int b = bh / H, h = bh - b * H;
            const int left = n - (int)grp * 8;                           // chunks in this group: 8, or 4 at the end of a row
            uint32_t code[8];
#pragma unroll
            for (int i = 0; i < 8; i++) code[i] = 0;
            ST scale = 0;
            if ((int)t < p.T) {
                const int32_t *ip = p.idx + b * p.isb + h * p.ish + t * p.ist + grp * 8;
                const int32_t *rp = p.rq + b * p.rsb + h * p.rsh + t * p.rst + grp * 8;
                if (p.vec && left >= 8) {
                    const int4 i0 = reinterpret_cast<const int4 *>(ip)[0], i1 = reinterpret_cast<const int4 *>(ip)[1];
                    const int4 r0 = reinterpret_cast<const int4 *>(rp)[0], r1 = reinterpret_cast<const int4 *>(rp)[1];
                    const int32_t ii[8] = {i0.x, i0.y, i0.z, i0.w, i1.x, i1.y, i1.z, i1.w}, rr[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
                    for (int i = 0; i < 8; i++) code[i] = ((uint32_t)ii[i] & idx_mask) | ((uint32_t)rr[i] << idx_bits);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        if (i < left) code[i] = ((uint32_t)ip[i] & idx_mask) | ((uint32_t)rp[i] << idx_bits);
                }
                if (grp == 0) scale = ((const ST *)p.scale_in)[b * p.ssb + h * p.ssh + t * p.sst];
            }
            uint32_t w[MB / 4];
#pragma unroll
            for (int i = 0; i < MB / 4; i++) w[i] = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t m = code[i] & ((1u << MB) - 1u);
                w[i * MB >> 5] |= m << (i * MB & 31);
                if ((i * MB & 31) + MB > 32) w[(i * MB >> 5) + 1] |= m >> (32 - (i * MB & 31));
            }
            const size_t row = (size_t)bh * t_cap + t;
            uint8_t *mp = p.main_plane + row * mrb + grp * MB;
            if ((n & 7) == 0) {
                if constexpr (MB == 16) *reinterpret_cast<uint4 *>(mp) = uint4{w[0], w[1], w[2], w[3]};
                else if constexpr (MB == 12) {
                    for (int i = 0; i < 3; i++) reinterpret_cast<uint32_t *>(mp)[i] = w[i];
                } else *reinterpret_cast<uint2 *>(mp) = uint2{w[0], w[1]};
            } else {
#pragma unroll
                for (int i = 0; i < MB; i++)
                    if (left >= 8 || i < MB / 2) mp[i] = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
            }
            if (ab) {
                uint64_t a = 0;
#pragma unroll
                for (int i = 0; i < 8; i++) a |= (uint64_t)((code[i] >> MB) & ((1u << ab) - 1u)) << (i * ab);
                uint8_t *ap = p.aux_plane + row * arb + grp * ab;
                const int bytes = left >= 8 ? ab : (4 * ab + 7) >> 3;
                for (int i = 0; i < bytes; i++) ap[i] = (uint8_t)(a >> (8 * i));
            }
            if (grp == 0) {
                ((ST *)p.scale_plane)[row] = scale;
                const float f = fabsf(D::load(&scale));
                if (f < __builtin_inff()) most = max(most, __float_as_uint(f));
            }
        }
    if (D::code == HQMQ_F16 || !p.scale_max) return;
    for (int o = 32; o; o >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, o));
    if ((threadIdx.x & 63) == 0 && most > __hip_atomic_load(p.scale_max, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p.scale_max, most);
}

// one thread per output byte of the main plane, then of the aux plane
__global__ void pack_codes_kernel(const int32_t *idx, int64_t isb, int64_t ish, int64_t ist, const int32_t *rq, int64_t rsb_,
                                  int64_t rsh_, int64_t rst_, int B, int H, int T, int n, int idx_bits, int main_bits,
                                  int aux_bits, uint8_t *main_plane, uint8_t *aux_plane, int64_t t_cap) {
    const int mrb = (n * main_bits + 7) >> 3, arb = (n * aux_bits + 7) >> 3;
    const int per_row = mrb + arb;
    const int64_t total = (int64_t)B * H * T * per_row;
    const uint32_t idx_mask = (1u << idx_bits) - 1u;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
        int byte = (int)(g % per_row);
        const int64_t row = g / per_row;
        const int t = (int)(row % T);
        const int h = (int)((row / T) % H);
        const int b = (int)(row / ((int64_t)T * H));
        const bool is_aux = byte >= mrb;
        if (is_aux) byte -= mrb;
        const int w = is_aux ? aux_bits : main_bits, shift = is_aux ? main_bits : 0;
        const int32_t *ip = idx + b * isb + h * ish + t * ist;
        const int32_t *rp = rq + b * rsb_ + h * rsh_ + t * rst_;
        uint32_t outv = 0;
        for (int bit = 0; bit < 8; bit++) {
            const int pos = byte * 8 + bit, i = pos / w, o = pos - i * w;
            if (i < n) {
                const uint32_t code = ((uint32_t)ip[i] & idx_mask) | ((uint32_t)rp[i] << idx_bits);
                outv |= ((((code >> shift) & ((1u << w) - 1u)) >> o) & 1u) << bit;
            }
        }
        const size_t prow = ((size_t)b * H + h) * t_cap + t;
        if (is_aux) aux_plane[prow * arb + byte] = (uint8_t)outv;
        else main_plane[prow * mrb + byte] = (uint8_t)outv;
    }
}

struct PackedView {
    const uint8_t *main_plane, *aux_plane, *flag_plane;
    const void *scale_plane;
    int64_t ssb, ssh, sst;
    const void *sideband;
    const int32_t *sb_tile_off;
    int64_t sb_cap;
    const void *joint;
    int64_t jsh;
    int K;
};

// mode 0: value = cw * ((rq * rs) / qmax)   (the attention kernels' convention)
// mode 1: value = (rq * (rs / qmax)) * cw   (the quantizer's fake-quant output)
template <class D>
__global__ void dequant_packed_kernel(PackedView p, int B, int H, int T, int n, int64_t t_cap, int idx_bits, int main_bits,
                                      int aux_bits, int qmax, int mode, typename D::storage *out) {
    using ST = typename D::storage;
    const int mrb = (n * main_bits + 7) >> 3, arb = (n * aux_bits + 7) >> 3, frb = (n + 7) >> 3;
    const int64_t total = (int64_t)B * H * T * n;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(g % n);
        const int64_t row = g / n;
        const int t = (int)(row % T);
        const int h = (int)((row / T) % H);
        const int b = (int)(row / ((int64_t)T * H));
        const size_t bh = (size_t)b * H + h;
        const size_t prow = bh * t_cap + t;
        ST *dst = out + g * 4;
        if (p.flag_plane && ((p.flag_plane[prow * frb + (c >> 3)] >> (c & 7)) & 1)) {
            const int tile = t >> 4;
            // 64-bit and clamped on both sides: a tile that was never written (or was cropped) holds INT32_MAX
            int64_t rank = p.sb_tile_off[bh * ((t_cap + kTile - 1) / kTile) + tile];
            for (int tt = tile * kTile; tt < t; tt++)
                for (int by = 0; by < frb; by++) rank += __popc((uint32_t)p.flag_plane[(bh * t_cap + tt) * frb + by]);
            for (int cc = 0; cc < c; cc++) rank += (p.flag_plane[prow * frb + (cc >> 3)] >> (cc & 7)) & 1;
            rank = rank < 0 ? 0 : (rank < p.sb_cap ? rank : p.sb_cap - 1);
            const ST *src = (const ST *)p.sideband + (bh * p.sb_cap + rank) * 4;
            for (int j = 0; j < 4; j++) dst[j] = src[j];
            continue;
        }
        uint32_t code = read_bits(p.main_plane + prow * mrb, mrb, c * main_bits, main_bits);
        if (aux_bits) code |= read_bits(p.aux_plane + prow * arb, arb, c * aux_bits, aux_bits) << main_bits;
        int k = (int)(code & ((1u << idx_bits) - 1u));
        k = k >= p.K ? p.K - 1 : k;
        const float q = (float)(code >> idx_bits);
        const float s = D::load((const ST *)p.scale_plane + b * p.ssb + h * p.ssh + t * p.sst);
        const ST *cw = (const ST *)p.joint + h * p.jsh + (int64_t)k * 4;
        if (mode == 0) {
            const float r = D::rnd(D::rnd(D::rnd(q) * s) / (float)qmax);
            for (int j = 0; j < 4; j++) D::store(dst + j, D::rnd(D::load(cw + j) * r));
        } else {
            const float r = D::rnd(q * D::rnd(s / (float)qmax));
            for (int j = 0; j < 4; j++) D::store(dst + j, D::rnd(r * D::load(cw + j)));
        }
    }
}

static inline int grid_for(int64_t total, int block) {
    int64_t g = (total + block - 1) / block;
    return (int)(g < 1 ? 1 : (g > 65535 * 16 ? 65535 * 16 : g));
}

}  // namespace hqmq

using namespace hqmq;

extern "C" int hqmq_dequant(const int32_t *idx, int64_t idx_sb, int64_t idx_sh, int64_t idx_st, const int32_t *rq,
                            int64_t rq_sb, int64_t rq_sh, int64_t rq_st, const void *rs, int64_t rs_sb, int64_t rs_sh,
                            int64_t rs_st, const void *joint, int64_t joint_sh, int K, int dtype, int B, int H, int T,
                            int n_chunks, int qmax, void *out, void *stream) {
    if (!idx || !rq || !rs || !joint || !out) return HQMQ_ERR_NULL;
    if (B < 1 || H < 1 || T < 0 || n_chunks < 1 || K < 1 || qmax < 1) return HQMQ_ERR_SHAPE;
    if (T == 0) return HQMQ_OK;
    if ((int64_t)B * H > 0x7fffffff) return HQMQ_ERR_SHAPE;
    // two chunks per thread where every row can be read and written that way
    const bool pairs = dtype != HQMQ_F32 && (n_chunks & 1) == 0 && !((idx_sb | idx_sh | idx_st | rq_sb | rq_sh | rq_st) & 1) && !(joint_sh & 3) &&
                       !(((uintptr_t)idx | (uintptr_t)rq | (uintptr_t)joint) & 7) && !((uintptr_t)out & 15);
    const int64_t per_bh = ((int64_t)T * (n_chunks / (pairs ? 2 : 1)) + 255) / 256;
    const dim3 grid((unsigned)std::min<int64_t>(per_bh, 1 << 20), (unsigned)std::min<int64_t>((int64_t)B * H, 65535)), block(256);
    hipStream_t st = (hipStream_t)stream;
#define LAUNCH(DT, ST, PER)                                                                                              \
    hipLaunchKernelGGL((dequant_kernel<DT, PER>), grid, block, 0, st, idx, idx_sb, idx_sh, idx_st, rq, rq_sb, rq_sh, rq_st, \
                       (const ST *)rs, rs_sb, rs_sh, rs_st, (const ST *)joint, joint_sh, K, B * H, H, T, n_chunks, qmax, (ST *)out)
    switch (dtype) {
        case HQMQ_F32: LAUNCH(F32, float, 1); break;
        case HQMQ_F16: if (pairs) LAUNCH(F16, uint16_t, 2); else LAUNCH(F16, uint16_t, 1); break;
        case HQMQ_BF16: if (pairs) LAUNCH(BF16, uint16_t, 2); else LAUNCH(BF16, uint16_t, 1); break;
        default: return HQMQ_ERR_DTYPE;
    }
#undef LAUNCH
    return hip_status(hipGetLastError());
}

template <class D>
static int launch_pack(const PackPair &p, const hqmq_pack_args *a, int mb, hipStream_t st) {
    const int64_t items = (int64_t)a->t_cap * ((a->n_chunks + 7) / 8);
    const dim3 grid((unsigned)((items + 255) / 256), (unsigned)std::min<int64_t>((int64_t)a->B * a->H, 65535), 2), block(256);
    auto kern = mb == 16 ? pack_kv_kernel<D, 16> : mb == 12 ? pack_kv_kernel<D, 12> : pack_kv_kernel<D, 8>;
    hipLaunchKernelGGL(kern, grid, block, 0, st, p, a->B * a->H, a->H, a->n_chunks, a->idx_bits, a->aux_bits, (int)a->t_cap);
    return hip_status(hipGetLastError());
}

extern "C" int hqmq_pack_kv(const hqmq_pack_args *a, void *stream) {
    if (!a) return HQMQ_ERR_NULL;
    if (a->B < 1 || a->H < 1 || a->n_chunks < 4 || (a->n_chunks & 3) || a->t_cap < 1 || (int64_t)a->B * a->H > 0x7fffffff) return HQMQ_ERR_SHAPE;
    if (a->t_cap * ((a->n_chunks + 7) / 8) > 0x7fffffff) return HQMQ_ERR_SHAPE;
    if (a->idx_bits < 1 || a->idx_bits > 16 || a->aux_bits < 0 || a->aux_bits > 8) return HQMQ_ERR_LAYOUT;
    if (a->main_bits != 8 && a->main_bits != 12 && a->main_bits != 16) return HQMQ_ERR_LAYOUT;
    PackPair p;
    for (int i = 0; i < 2; i++) {
        const hqmq_pack_side &k = a->side[i];
        if (k.T < 0 || k.T > a->t_cap) return HQMQ_ERR_SHAPE;
        if ((k.T && (!k.idx || !k.rq || !k.scale_in)) || !k.main_plane || !k.scale_plane || (a->aux_bits && !k.aux_plane)) return HQMQ_ERR_NULL;
        if ((uintptr_t)k.main_plane & 15) return HQMQ_ERR_ALIGN;
        const int vec = !((k.idx_sb | k.idx_sh | k.idx_st | k.rq_sb | k.rq_sh | k.rq_st) & 3) && !(((uintptr_t)k.idx | (uintptr_t)k.rq) & 15);
        p.s[i] = PackSide{k.idx, k.rq, k.idx_sb, k.idx_sh, k.idx_st, k.rq_sb, k.rq_sh, k.rq_st, k.scale_in, k.scale_sb, k.scale_sh, k.scale_st,
                          k.main_plane, k.aux_plane, k.scale_plane, k.scale_max_bits, k.T, vec};
    }
    switch (a->dtype) {
        case HQMQ_F32: return launch_pack<F32>(p, a, a->main_bits, (hipStream_t)stream);
        case HQMQ_F16: return launch_pack<F16>(p, a, a->main_bits, (hipStream_t)stream);
        case HQMQ_BF16: return launch_pack<BF16>(p, a, a->main_bits, (hipStream_t)stream);
        default: return HQMQ_ERR_DTYPE;
    }
}

extern "C" int hqmq_pack_codes(const int32_t *idx, int64_t idx_sb, int64_t idx_sh, int64_t idx_st, const int32_t *rq,
                               int64_t rq_sb, int64_t rq_sh, int64_t rq_st, int B, int H, int T, int n_chunks, int idx_bits,
                               int main_bits, int aux_bits, uint8_t *main_plane, uint8_t *aux_plane, int64_t t_cap,
                               void *stream) {
    if (!idx || !rq || !main_plane || (aux_bits && !aux_plane)) return HQMQ_ERR_NULL;
    if (B < 1 || H < 1 || T < 0 || n_chunks < 1 || t_cap < T) return HQMQ_ERR_SHAPE;
    if (idx_bits < 1 || idx_bits > 16 || main_bits < 1 || main_bits > 16 || aux_bits < 0 || aux_bits > 8) return HQMQ_ERR_LAYOUT;
    if (T == 0) return HQMQ_OK;
    const int per_row = ((n_chunks * main_bits + 7) >> 3) + ((n_chunks * aux_bits + 7) >> 3);
    dim3 grid(grid_for((int64_t)B * H * T * per_row, 256)), block(256);
    hipLaunchKernelGGL(pack_codes_kernel, grid, block, 0, (hipStream_t)stream, idx, idx_sb, idx_sh, idx_st, rq, rq_sb, rq_sh,
                       rq_st, B, H, T, n_chunks, idx_bits, main_bits, aux_bits, main_plane, aux_plane, t_cap);
    return hip_status(hipGetLastError());
}

extern "C" int hqmq_dequant_packed(const hqmq_packed *p, int dtype, int B, int H, int T, int n_chunks, int64_t t_cap,
                                   int idx_bits, int main_bits, int aux_bits, int qmax, int mode, void *out, void *stream) {
    if (!p || !p->main_plane || !p->scale_plane || !p->joint || !out) return HQMQ_ERR_NULL;
    if (aux_bits && !p->aux_plane) return HQMQ_ERR_NULL;
    if (p->flag_plane && (!p->sideband || !p->sb_tile_off || p->sb_cap < 1)) return HQMQ_ERR_NULL;
    if (B < 1 || H < 1 || T < 0 || n_chunks < 1 || t_cap < T || qmax < 1) return HQMQ_ERR_SHAPE;
    if (mode != 0 && mode != 1) return HQMQ_ERR_SHAPE;
    if (T == 0) return HQMQ_OK;
    PackedView v{p->main_plane, p->aux_plane, p->flag_plane, p->scale_plane, p->scale_sb, p->scale_sh, p->scale_st,
                 p->sideband, p->sb_tile_off, p->sb_cap, p->joint, p->joint_sh, p->K};
    dim3 grid(grid_for((int64_t)B * H * T * n_chunks, 256)), block(256);
    hipStream_t st = (hipStream_t)stream;
#define LAUNCH(DT, ST)                                                                                                  \
    hipLaunchKernelGGL(dequant_packed_kernel<DT>, grid, block, 0, st, v, B, H, T, n_chunks, t_cap, idx_bits, main_bits, \
                       aux_bits, qmax, mode, (ST *)out)
    switch (dtype) {
        case HQMQ_F32: LAUNCH(F32, float); break;
        case HQMQ_F16: LAUNCH(F16, uint16_t); break;
        case HQMQ_BF16: LAUNCH(BF16, uint16_t); break;
        default: return HQMQ_ERR_DTYPE;
    }
#undef LAUNCH
    return hip_status(hipGetLastError());
}
