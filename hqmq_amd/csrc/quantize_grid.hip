// Codeword search through cell lists.
//
// The codebook {q_p * q_s} is closed under left multiplication by the 24 Hurwitz units, and so is the score:
// <u, q_p * q_s> = <conj(q_g) * u, (conj(q_g) * q_p) * q_s> for every unit q_g.  Multiplying a direction u by the
// conjugate of its nearest unit q_g brings it into the cell of S^3 around 1, where w0 is the largest scalar part:
// w = conj(q_g) * u has |w1| + |w2| + |w3| <= w0, i.e. y = (w1, w2, w3) / w0 lies in the octahedron |y|_1 <= 1.  Only
// 1 / 24 of the directions are left to be searched, and every codebook of S secondaries has about S codewords there.
// A grid of kGrid^3 boxes over [-1, 1]^3 (those that meet the octahedron) carries, per box, the list of all codewords
// (p', s) that can win the reference's rounded comparison for some direction inside it; the lists are worked out once
// per codebook (hqmq_build_search_grid).  A search is then: nearest unit, one quaternion product, one list look-up,
// and the reference's own rounded score (bit for bit) for the few codewords of the list; the largest score wins, the
// smallest index k = p * S + s among equals.
//
// The reference scores with the stored table J, whose rows are rounded products: conj(q_g) * J[k] depends on g.  A
// codeword (p', s) therefore stands for 24 points, taken as a centre and the radius rho of the ball around it.
// A codeword g is left out of a box when some codeword g* beats it by more than any rounding can turn, everywhere in
// the box: <(1, y), g* - g> > (rho_g + rho_g* + m) |(1, y)|.  The left side is linear in y, so its minimum over the box
// is the value at the centre less half the box's width times |g*_i - g_i| summed over the three coordinates; |(1, y)| is
// largest in the corner farthest from 0.  m covers the roundings of the two scores to D: half a unit in the last place
// each, 2^-12 (fp16) and 2^-9 (bf16) for scores in [0.5, 1), twice that where a score can reach 1 (directions are
// vectors of length 1 within 1.5 %; others are scored against all rows).
//
// Lists, per head, in blocks of 16 bytes: seven 16-bit entries p' << 2 | s' << 7 (s' = S - 1 - s; p' = 31: no entry) and
// the number of the block that goes on (0: none, 0xffff: no list, score all rows).  The first kCells blocks are the
// boxes', the others a pool that the build hands out; block 0 of the pool holds no entry.  That is 185 KB per head (fp16,
// fp32) or 371 KB (bf16) at every S.  Behind the lists of all heads lies what only the build reads and a caller may drop
// afterwards (hqmq_search_grid_kept_bytes): the pools' counters, the centres and radii of the codewords.
//
// What it costs: per 64 chunks 342 vector-ALU instructions at fp16 s96_r4, 450 at bf16 s24_r3 with flags (180 for norm,
// division, nearest unit and box, 11 per list entry, 60 - 80 for scale, radius code and packing) where the scan over 96
// secondaries takes 1,885.  Bound by vector-ALU issue: 0.89 and 0.90 of the cycles a compute unit is busy, its LDS pipe 24
// and 19 % (profiles/quantize_grid_kernel_instruction_counters.txt).  K and V of 8 x 32768 tokens, fp16, s96_r4, packed:
// 792 -> 189 us; 8 x 4 x 4001 tokens bf16 s24_r3 with flags 371 -> 128 us; one tensor of 8 x 2048 tokens s192_r6,
// fake-quant output: 51 -> 11 us.  40 boxes per axis instead of 32 shorten the lists by a fifth and bought 3 %.
//
// Compiled with -ffp-contract=off; fused multiply-adds are written explicitly.
#include "quantize_common.h"

namespace hqmq {

constexpr int kCoarse = 8;                      // boxes per axis of the build's first level
constexpr int kFine = 4;                        // boxes per axis inside one of those
constexpr int kGrid = kCoarse * kFine;
constexpr int kGridSMax = 341;                  // 24 * 341 rows of 8 bytes: row offsets fit 16 bits, s' fits 9
constexpr uint32_t kNone = 31u << 2;            // an empty entry

// Does box (i, j, k) of a grid of `g` boxes per axis meet the octahedron (a hair dilated: w is computed in fp32)?
constexpr bool box_meets(int i, int j, int k, int g) {
    auto dist = [g](int x) {                    // smallest |y| of the box, in units of 1 / g
        const int lo = 2 * x - g, hi = lo + 2;
        return lo > 0 ? lo : hi < 0 ? -hi : 0;
    };
    return 1000 * (dist(i) + dist(j) + dist(k)) <= 1001 * g;
}
struct GridMap {
    int cells;
    int16_t off[kGrid * kGrid];                 // box (i, j, k) has number off[i * kGrid + j] + k
};
constexpr GridMap make_map() {
    GridMap m{};
    int n = 0;
    for (int i = 0; i < kGrid; i++)
        for (int j = 0; j < kGrid; j++) {
            int first = -1;
            for (int k = 0; k < kGrid; k++)
                if (box_meets(i, j, k, kGrid)) {
                    if (first < 0) { first = k; m.off[i * kGrid + j] = (int16_t)(n - k); }
                    n++;
                }
        }
    m.cells = n;
    return m;
}
constexpr GridMap kMap = make_map();
constexpr int kCells = kMap.cells;
static_assert(kCells < 32768, "box numbers are 16-bit");

constexpr float unit_part(int p, int j) {       // component j of Hurwitz unit p, in the order of the joint table
    return p < 8 ? (j == (p >> 1) ? ((p & 1) ? -1.f : 1.f) : 0.f) : (((p - 8) >> (3 - j)) & 1 ? -0.5f : 0.5f);
}
struct Units {
    float q[24][4];
    uint8_t mul[24][24];                        // unit number of q_a * q_b
};
constexpr Units make_units() {
    Units t{};
    for (int p = 0; p < 24; p++)
        for (int j = 0; j < 4; j++) t.q[p][j] = unit_part(p, j);
    for (int a = 0; a < 24; a++)
        for (int b = 0; b < 24; b++) {
            const float *x = t.q[a], *y = t.q[b];
            const float r[4] = {x[0] * y[0] - x[1] * y[1] - x[2] * y[2] - x[3] * y[3], x[0] * y[1] + x[1] * y[0] + x[2] * y[3] - x[3] * y[2],
                                x[0] * y[2] - x[1] * y[3] + x[2] * y[0] + x[3] * y[1], x[0] * y[3] + x[1] * y[2] - x[2] * y[1] + x[3] * y[0]};
            for (int p = 0; p < 24; p++)
                if (t.q[p][0] == r[0] && t.q[p][1] == r[1] && t.q[p][2] == r[2] && t.q[p][3] == r[3]) t.mul[a][b] = (uint8_t)p;
        }
    return t;
}
__device__ const GridMap d_map = make_map();
__device__ const Units d_units = make_units();

// Blocks of the pool: random codebooks take 1.05 blocks per box at most (bf16, S = 192; fp16 0.1).  A box that finds
// the pool empty scores all rows.
constexpr int64_t pool_blocks(int dtype) { return dtype == HQMQ_BF16 ? 2 * kCells : kCells / 2; }
static_assert(2 * kCells < 65535, "block numbers are 16-bit");

int64_t search_grid_blocks(int S, int dtype) {
    if (S < 1 || S > kGridSMax) return 0;
    return kCells + pool_blocks(dtype);
}

// ---------------------------------------------------------------- build
struct Codewords {              // where the build keeps the codewords' geometry
    float4 *centre;             // [H][24 S]
    float *rho;                 // [H][24 S]
};
__host__ __device__ inline uint32_t *grid_counters(uint4 *grid, int64_t stride, int H) { return reinterpret_cast<uint32_t *>(grid + stride * H); }
__host__ __device__ inline Codewords grid_codewords(uint4 *grid, int64_t stride, int H, int S) {
    float4 *c = reinterpret_cast<float4 *>(grid + stride * H + (H + 3) / 4);
    return Codewords{c, reinterpret_cast<float *>(c + (int64_t)H * 24 * S)};
}

__device__ __forceinline__ float4 quat_mul(float4 a, float4 b) {
    return float4{a.x * b.x - a.y * b.y - a.z * b.z - a.w * b.w, a.x * b.y + a.y * b.x + a.z * b.w - a.w * b.z,
                  a.x * b.z - a.y * b.w + a.z * b.x + a.w * b.y, a.x * b.w + a.y * b.z - a.z * b.y + a.w * b.x};
}

// Centre and radius of the 24 points conj(q_g) * J[q_g * q_p', s] for every (p', s), 32 lanes per codeword (lane = g; the
// last eight repeat g = 23); the head's counter and empty block.
template <class D>
__global__ __launch_bounds__(256) void grid_codewords_kernel(const typename D::storage *joint, int S, uint4 *grid, int64_t stride, int H) {
    const int h = blockIdx.y, k = blockIdx.x * 8 + (threadIdx.x >> 5), g = min((int)threadIdx.x & 31, 23);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        grid_counters(grid, stride, H)[h] = 1;
        grid[stride * h + kCells] = uint4{kNone | kNone << 16, kNone | kNone << 16, kNone | kNone << 16, kNone};
    }
    if (k >= 24 * S) return;            // (24 S is a multiple of 8: whole blocks)
    const int p = k / S, s = k - p * S;
    const typename D::storage *r = joint + ((size_t)h * 24 * S + (size_t)d_units.mul[g][p] * S + s) * 4;
    const float *q = d_units.q[g];
    const float4 v = quat_mul(float4{q[0], -q[1], -q[2], -q[3]}, float4{D::load(r), D::load(r + 1), D::load(r + 2), D::load(r + 3)});
    auto most = [](float x, auto op) {
        for (int o = 16; o; o >>= 1) x = op(x, __shfl_xor(x, o, 32));
        return x;
    };
    auto mid = [&](float x) {
        return 0.5f * (most(x, [](float i, float j) { return fminf(i, j); }) + most(x, [](float i, float j) { return fmaxf(i, j); }));
    };
    const float4 c = float4{mid(v.x), mid(v.y), mid(v.z), mid(v.w)};
    const float d0 = v.x - c.x, d1 = v.y - c.y, d2 = v.z - c.z, d3 = v.w - c.w;
    // (a NaN row makes the radius NaN: nothing is left out because of it, and it is left out nowhere)
    const float far = most(sqrtf(d0 * d0 + d1 * d1 + d2 * d2 + d3 * d3), [](float i, float j) { return i > j || is_nan(i) ? i : j; });
    const Codewords cw = grid_codewords(grid, stride, H, S);
    if ((threadIdx.x & 31) == 0) {
        cw.centre[(size_t)h * 24 * S + k] = c;
        cw.rho[(size_t)h * 24 * S + k] = far * 1.00001f + 1e-6f;
    }
}

// One block per coarse box and head.  First the codewords that matter anywhere in the coarse box are listed in LDS
// (lanes over codewords), then the kFine^3 boxes inside it are worked out from that list, kLanes lanes per box: 248 x 4608
// tests per head instead of 7728 x 4608.  kListCap bounds the coarse list (random codebooks: 30 - 250), kBoxCap a box's
// (random codebooks: 48 at most); beyond either the box scores all rows.
constexpr int kListCap = 1024;
constexpr int kBoxCap = 126;
constexpr int kBuildThreads = 256;
constexpr int kLanes = kBuildThreads / (kFine * kFine * kFine);
static_assert(kLanes == 4, "lanes per box");
template <class D>
__global__ __launch_bounds__(kBuildThreads) void grid_build_kernel(int S, uint4 *grid, int64_t stride, int pool, int H) {
    const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int ci = blockIdx.x / (kCoarse * kCoarse), cj = blockIdx.x / kCoarse % kCoarse, ck = blockIdx.x % kCoarse;
    if (!box_meets(ci, cj, ck, kCoarse)) return;
    __shared__ float4 geo[kListCap];
    __shared__ float rad[kListCap];
    __shared__ uint16_t id[kListCap];
    __shared__ uint16_t entries[kFine * kFine * kFine][kBoxCap + 1];
    __shared__ int count[kFine * kFine * kFine];
    __shared__ float best_sh[kBuildThreads / 64];
    __shared__ int arg_sh[kBuildThreads / 64], n_sh;
    const int K = 24 * S;
    const Codewords all = grid_codewords(grid, stride, H, S);
    const float4 *centre = all.centre + (size_t)h * K;
    const float *rho = all.rho + (size_t)h * K;
    struct Box { float y0, y1, y2, hw, longest, shortest; };             // centre, half width, |(1, y)| over the box
    auto box_at = [](int i, int j, int k, int g) {
        const float w = 2.f / (float)g, hw = 1.f / (float)g + 2e-5f;
        Box b{((float)i + 0.5f) * w - 1.f, ((float)j + 0.5f) * w - 1.f, ((float)k + 0.5f) * w - 1.f, hw, 0.f, 0.f};
        auto sq = [](float v) { return v * v; };
        b.longest = sqrtf(1.f + sq(fabsf(b.y0) + hw) + sq(fabsf(b.y1) + hw) + sq(fabsf(b.y2) + hw)) * 1.00001f;
        b.shortest = sqrtf(1.f + sq(fmaxf(fabsf(b.y0) - hw, 0.f)) + sq(fmaxf(fabsf(b.y1) - hw, 0.f)) + sq(fmaxf(fabsf(b.y2) - hw, 0.f))) * 0.99999f;
        return b;
    };
    auto dot = [](float4 g, const Box &b) { return g.x + b.y0 * g.y + b.y1 * g.z + b.y2 * g.w; };
    // what g* has to lead by, less the radii: the roundings of both scores, and of this kernel
    auto rounding = [&](float4 star, float r, const Box &b) {
        const float most = (dot(star, b) + b.hw * (fabsf(star.y) + fabsf(star.z) + fabsf(star.w))) / b.shortest + r;
        return 1.016f * (most * 1.016f < 1.f ? 1.f : 2.f) * D::eps() + 1.2e-5f;
    };
    auto beaten = [&](float4 s, float need, float4 g, float r, const Box &b) {
        const float d0 = s.x - g.x, d1 = s.y - g.y, d2 = s.z - g.z, d3 = s.w - g.w;
        const float lead = d0 + b.y0 * d1 + b.y1 * d2 + b.y2 * d3 - b.hw * (fabsf(d1) + fabsf(d2) + fabsf(d3));
        return lead > (need + r) * b.longest;
    };
    if (tid == 0) n_sh = 0;
    if (tid < kFine * kFine * kFine) count[tid] = 0;
    {
        const Box b = box_at(ci, cj, ck, kCoarse);
        float best = -INFINITY;
        int arg = 0;
#pragma unroll 4
        for (int k = tid; k < K; k += kBuildThreads) {
            const float v = dot(centre[k], b) - rho[k] * b.longest;
            if (v > best) { best = v; arg = k; }
        }
        for (int o = 32; o; o >>= 1) {
            const float v = __shfl_xor(best, o);
            const int g = __shfl_xor(arg, o);
            if (v > best || (v == best && g < arg)) { best = v; arg = g; }
        }
        if (lane == 0) { best_sh[tid >> 6] = best; arg_sh[tid >> 6] = arg; }
        __syncthreads();
        for (int w = 0; w < kBuildThreads / 64; w++)
            if (best_sh[w] > best || (best_sh[w] == best && arg_sh[w] < arg)) { best = best_sh[w]; arg = arg_sh[w]; }
        const float4 star = centre[arg];
        const float need = rounding(star, rho[arg], b) + rho[arg];
        for (int k0 = 0; k0 < K; k0 += kBuildThreads) {
            const int k = k0 + tid;
            const float4 g = centre[min(k, K - 1)];
            const float r = rho[min(k, K - 1)];
            const bool take = k < K && !beaten(star, need, g, r, b);
            const uint64_t mask = __builtin_amdgcn_ballot_w64(take);
            int at = 0;
            if (lane == 0 && mask) at = atomicAdd(&n_sh, (int)__popcll(mask));
            at = __shfl(at, 0) + __popcll(mask & ((1ull << lane) - 1ull));
            if (take && at < kListCap) { geo[at] = g; rad[at] = r; id[at] = (uint16_t)k; }
        }
        __syncthreads();
    }
    const int n_list = n_sh;
    uint4 *lists = grid + stride * h;
    uint32_t *used = grid_counters(grid, stride, H) + h;
    const int f = tid / kLanes, part = tid % kLanes;
    const int i = ci * kFine + f / (kFine * kFine), j = cj * kFine + f / kFine % kFine, k = ck * kFine + f % kFine;
    const bool wanted = box_meets(i, j, k, kGrid), listed = n_list <= kListCap;
    if (wanted && listed) {
        const Box b = box_at(i, j, k, kGrid);
        float best = -INFINITY;
        int arg = 0;
        for (int e = part; e < n_list; e += kLanes) {
            const float v = dot(geo[e], b) - rad[e] * b.longest;
            if (v > best) { best = v; arg = e; }
        }
        for (int o = 1; o < kLanes; o <<= 1) {
            const float v = __shfl_xor(best, o);
            const int g = __shfl_xor(arg, o);
            if (v > best || (v == best && g < arg)) { best = v; arg = g; }
        }
        const float4 star = geo[arg];
        const float need = rounding(star, rad[arg], b) + rad[arg];
        for (int e = part; e < n_list; e += kLanes) {
            if (beaten(star, need, geo[e], rad[e], b)) continue;
            const int at = atomicAdd(&count[f], 1);
            if (at < kBoxCap) entries[f][at] = id[e];
        }
    }
    __syncthreads();
    if (tid >= kFine * kFine * kFine) return;
    {
        const int f2 = tid, i2 = ci * kFine + f2 / (kFine * kFine), j2 = cj * kFine + f2 / kFine % kFine, k2 = ck * kFine + f2 % kFine;
        if (!box_meets(i2, j2, k2, kGrid)) return;
        const int cell = d_map.off[i2 * kGrid + j2] + k2, n = count[f2], more = n > 7 ? (n - 1) / 7 : 0;      // blocks from the pool
        uint32_t next = 0;
        bool full = !listed || n > kBoxCap;
        if (!full && more) {
            next = atomicAdd(used, (uint32_t)more);
            full = next + more > (uint32_t)pool;
        }
        int at = cell;
        for (int e0 = 0;; e0 += 7) {
            uint32_t w[8];
#pragma unroll
            for (int e = 0; e < 7; e++) {
                w[e] = kNone;
                if (!full && e0 + e < n) {
                    const int kk = entries[f2][e0 + e], p = kk / S;
                    w[e] = (uint32_t)p << 2 | (uint32_t)(S - 1 - (kk - p * S)) << 7;
                }
            }
            const bool last = full || e0 + 7 >= n;
            w[7] = full ? 0xffffu : last ? 0u : next;
            lists[at] = uint4{w[0] | w[1] << 16, w[2] | w[3] << 16, w[4] | w[5] << 16, w[6] | w[7] << 16};
            if (last) break;
            at = kCells + (int)next++;
        }
    }
}

// ---------------------------------------------------------------- search
// LDS: [K rows of the joint table, last row first (JLDS)] | 24 x 32 row offsets by (unit of the direction, p') | box
// numbers | two words per lane.  The dynamic block is the kernel's only LDS, so it starts at LDS address 0 and the row
// offset of a codeword is its address.
constexpr int lds_rows_at(int table_bytes) { return (table_bytes + 127) & ~127; }
constexpr int kBoxesAt = 24 * 32 * 4, kLanesAt = (kBoxesAt + kGrid * kGrid * 2 + 15) & ~15;       // behind the row offsets

template <class D, int NT, bool ROWS, bool JLDS, int WHAT, int MB>
__device__ __forceinline__ void grid_body(const QParams &a) {
    using ST = typename D::storage;
    typedef const uint32_t __attribute__((address_space(3))) *lds_u32;
    typedef const int16_t __attribute__((address_space(3))) *lds_i16;
    typedef uint32_t __attribute__((ext_vector_type(2))) u32x2;
    typedef uint32_t __attribute__((ext_vector_type(4))) u32x4;
    typedef const u32x2 __attribute__((address_space(3))) *lds_u64;
    typedef const u32x4 __attribute__((address_space(3))) *lds_u128;
    constexpr int RB = 4 * sizeof(ST), RSH = RB == 8 ? 3 : 4;            // bytes of a row
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, n = a.n, S = a.S, K = 24 * S;
    const int bh = blockIdx.y, b = bh / a.H, h = bh - b * a.H;
    const ST *jh = (const ST *)a.joint + (size_t)h * K * 4;
    const uint32_t rows_at = JLDS ? (uint32_t)lds_rows_at(K * RB) : 0u;
    uint32_t *code_sh = reinterpret_cast<uint32_t *>(lds + rows_at + kLanesAt), *aux_sh = code_sh + NT;
    const int tpb = NT / n, tok_local = tid / n, c = tid - tok_local * n;
    const int t_first = blockIdx.x * a.iters * tpb;
    const ST *xl = (const ST *)a.x + b * a.xsb + h * a.xsh + (int64_t)(t_first + tok_local) * a.xst + c * 4;
    const int64_t x_step = tpb * a.xst;
    const int t_left = tok_local < tpb ? a.T - t_first - tok_local : 0;     // this lane has a token while t0 - t_first < t_left
    RawChunk<D> raw = {};
    if (t_left > 0) raw.load(xl, a.vec_in);
    {
        // every load of the set-up is requested before the first one is used: one round trip
        constexpr int NP = (24 * 32 + NT - 1) / NT, NB = (kGrid * kGrid / 2 + NT - 1) / NT;
        uint32_t unit_mul[NP], boxes[NB];
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int k = min(tid + i * NT, 24 * 32 - 1);
            unit_mul[i] = d_units.mul[k >> 5][min(k & 31, 23)];
        }
#pragma unroll
        for (int i = 0; i < NB; i++) boxes[i] = reinterpret_cast<const uint32_t *>(d_map.off)[min(tid + i * NT, kGrid * kGrid / 2 - 1)];
        if (JLDS) {
            for (int k = tid; k < K; k += NT) {
                RawChunk<D> g;
                g.load(jh + (size_t)k * 4, true);
                g.store(reinterpret_cast<ST *>(lds) + (size_t)(K - 1 - k) * 4, true);
            }
        }
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int k = tid + i * NT;
            // Most entries have p' = 0, so the offsets of one p' would share a bank: the units are spread over the banks by an
            // exclusive-or (14.8 -> 4.5 cycles per LDS access over the kernel).  No entry: a row like any other.
            if (k < 24 * 32) reinterpret_cast<uint32_t *>(lds + rows_at)[k ^ (k >> 5)] = (k & 31) < 24 ? (23u - unit_mul[i]) * (uint32_t)(S * RB) : 0u;
        }
#pragma unroll
        for (int i = 0; i < NB; i++)
            if (tid + i * NT < kGrid * kGrid / 2) reinterpret_cast<uint32_t *>(lds + rows_at + kBoxesAt)[tid + i * NT] = boxes[i];
    }
    __syncthreads();

    const uint4 *lists = a.grid + a.grid_stride * h;
    ChunkSink<D, NT, ROWS, WHAT, MB> sink(a, b, h, tok_local, c, code_sh, aux_sh);
    const int t_end = JLDS ? a.iters * tpb : tpb;
    for (int t0 = 0; t0 < t_end; t0 += tpb) {
        const bool active = t0 < t_left;
        const RawChunk<D> cur = raw;
        raw = {};
        xl += x_step;
        if (t0 + tpb < t_end && t0 + tpb < t_left) raw.load(xl, a.vec_in);      // the next round's chunk
        const float nrm = chunk_norm_d<D>(cur.get(0), cur.get(1), cur.get(2), cur.get(3));
        const float r = clamp_min_d<D>(nrm, 1e-8f);
        float u[4] = {cur.get(0), cur.get(1), cur.get(2), cur.get(3)};
        div4_d<D>(u, r);

        // ---- the unit nearest to u, and w = conj(unit) * u (half units doubled: only the ratios are used) ----
        const float a0 = fabsf(u[0]), a1 = fabsf(u[1]), a2 = fabsf(u[2]), a3 = fabsf(u[3]);
        const float sum = (a0 + a1) + (a2 + a3), mx = fmaxf(fmaxf(a0, a1), fmaxf(a2, a3));
        // directions of length 1: the others (NaN, infinite, clamped or subnormal radius) follow the reference row by
        // row, an all-zero direction scores 0 everywhere and takes row 0
        const float len2 = fmaf(u[3], u[3], fmaf(u[2], u[2], fmaf(u[1], u[1], u[0] * u[0])));
        const bool ordinary = len2 > 0.97f && len2 < 1.03f;
        const bool zero = sum == 0.f;
        const bool half = sum > mx + mx;
        const bool i0 = a0 == mx, i1 = !i0 && a1 == mx, i2 = !i0 && !i1 && a2 == mx, i3 = !i0 && !i1 && !i2;
        const float q0 = (half || i0) ? copysignf(1.f, u[0]) : 0.f, q1 = (half || i1) ? copysignf(1.f, u[1]) : 0.f;
        const float q2 = (half || i2) ? copysignf(1.f, u[2]) : 0.f, q3 = (half || i3) ? copysignf(1.f, u[3]) : 0.f;
        const uint32_t n0 = __float_as_uint(u[0]) >> 31, n1 = __float_as_uint(u[1]) >> 31, n2 = __float_as_uint(u[2]) >> 31, n3 = __float_as_uint(u[3]) >> 31;
        const uint32_t p_axis = i0 ? n0 : i1 ? 2u + n1 : i2 ? 4u + n2 : 6u + n3;
        const uint32_t p_half = 8u + (((n0 * 2u + n1) * 2u + n2) * 2u + n3);
        const uint32_t unit = half ? p_half : p_axis;
        const float w0 = half ? sum : mx;
        const float w1 = fmaf(q3, u[2], fmaf(-q2, u[3], fmaf(q0, u[1], -q1 * u[0])));
        const float w2 = fmaf(-q3, u[1], fmaf(q1, u[3], fmaf(q0, u[2], -q2 * u[0])));
        const float w3 = fmaf(q2, u[1], fmaf(-q1, u[2], fmaf(q0, u[3], -q3 * u[0])));
        const float inv = __builtin_amdgcn_rcpf(w0) * (0.5f * kGrid);
        // (a NaN ends up in box 0: such a lane's result is not used)
        auto box = [&](float w) { return (uint32_t)fminf(fmaxf(fmaf(w, inv, 0.5f * kGrid), 0.f), kGrid - 0.5f); };
        const uint32_t bx = box(w1), by = box(w2), bz = box(w3);
        const int box_no = *(lds_i16)(uintptr_t)(rows_at + kBoxesAt + (bx * kGrid + by) * 2u) + (int)bz;
        uint4 e = lists[min(max(box_no, 0), kCells - 1)];

        // ---- the reference's score of every codeword of the list ----
        int key = 0;                                                    // 16-bit types: rounded score << 16 | row offset
        float best = -INFINITY;                                         // fp32
        uint32_t best_at = 0;
        bool brute = active && !ordinary && !zero;
        const uint32_t unit_row = rows_at + unit * 132u;
        auto score = [&](uint32_t entry) {
            // row offset from the end of the table: the larger of two offsets is the smaller index k
            const uint32_t at = *(lds_u32)(uintptr_t)(unit_row ^ (entry & 0x7cu)) + ((entry >> 7 & 0x1ffu) << RSH);
            RawChunk<D> g;
            if constexpr (!JLDS) g.load(reinterpret_cast<const ST *>((const unsigned char *)(jh + (size_t)(K - 1) * 4) - at), true);
            else if constexpr (RB == 8) { const u32x2 v = *(lds_u64)(uintptr_t)at; g.w[0] = v[0]; g.w[1] = v[1]; }
            else { const u32x4 v = *(lds_u128)(uintptr_t)at; g.w[0] = v[0]; g.w[1] = v[1]; g.w[2] = v[2]; g.w[3] = v[3]; }
            float s = fmaf(u[0], g.get(0), 0.f);                        // the product's own rounding (a sum with 0 keeps it)
            s = fmaf(u[1], g.get(1), s);
            s = fmaf(u[2], g.get(2), s);
            s = fmaf(u[3], g.get(3), s);
            if constexpr (D::code == HQMQ_F16) {
                asm("" : "+v"(s));                                      // rounded to fp32 first, then to fp16
                key = max(key, (int)((uint32_t)__half_as_ushort(__float2half_rn(s)) << 16 | at));
            } else if constexpr (D::code == HQMQ_BF16) {
                const uint32_t x = __float_as_uint(s);
                key = max(key, (int)(((x + 0x7fffu + ((x >> 16) & 1u)) & 0xffff0000u) | at));
            } else {
                const bool more = s > best || (s == best && at > best_at);
                best = more ? s : best;
                best_at = more ? at : best_at;
            }
        };
        while (true) {
            score(e.x);
            score(e.x >> 16);
            const uint32_t none2 = kNone | kNone << 16;
            if (__builtin_amdgcn_ballot_w64(e.y != none2)) {
                score(e.y);
                score(e.y >> 16);
                if (__builtin_amdgcn_ballot_w64(e.z != none2)) {
                    score(e.z);
                    score(e.z >> 16);
                    score(e.w);
                }
            }
            const uint32_t next = e.w >> 16;
            if (__builtin_amdgcn_ballot_w64(next != 0u) == 0ull) break;
            if (next == 0xffffu) brute |= active && ordinary;           // (a direction that is not ordinary keeps its own reason)
            e = lists[kCells + (next == 0xffffu ? 0u : next)];
        }
        const uint32_t at = D::code == HQMQ_F32 ? best_at : (uint32_t)key & 0xffffu;
        int idx = zero ? 0 : K - 1 - (int)(at >> RSH);
        if (brute) idx = brute_argmax<D>(u, jh, K);
        if ((WHAT & kUnpacked) && a.stats && active) {
            if (brute) atomicAdd(a.stats, 1);
            else if (!zero) atomicAdd(a.stats + 1, 1);
        }
        const ST *jrow = JLDS ? reinterpret_cast<const ST *>(lds) + (size_t)(K - 1 - idx) * 4 : jh + (size_t)idx * 4;
        sink.put(t_first + t0, active, cur, nrm, r, idx, jrow);
    }
    sink.done();
}

template <class D, int NT, bool ROWS, bool JLDS, int WHAT, int MB>
__global__ __launch_bounds__(NT) void quantize_grid_kernel(QPair kv) {
    grid_body<D, NT, ROWS, JLDS, WHAT, MB>(kv.p[blockIdx.z]);
}

template <class D, int NT, bool ROWS, bool JLDS, int WHAT, int MB>
static int launch_kernel(QPair &kv, int count, hipStream_t st) {
    const QParams &p = kv.p[0];
    const int tpb = NT / p.n, rounds = (p.T + tpb - 1) / tpb;
    // A block copies its head's table to LDS first: as many rounds of tokens per block as leave every CU two blocks or so
    const int64_t blocks = (int64_t)rounds * p.B * p.H * count;
    int iters = (int)(blocks / 1024);
    iters = iters < 1 ? 1 : iters > 8 ? 8 : iters;
    kv.p[0].iters = kv.p[1].iters = JLDS ? iters : 1;
    const dim3 grid((rounds + kv.p[0].iters - 1) / kv.p[0].iters, p.B * p.H, count);
    const size_t shmem = (JLDS ? (size_t)lds_rows_at(24 * p.S * 4 * (int)sizeof(typename D::storage)) : 0) + kLanesAt + (size_t)NT * 8;
    auto kern = quantize_grid_kernel<D, NT, ROWS, JLDS, WHAT, MB>;
    if (shmem > 48 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kern, grid, dim3(NT), shmem, st, kv);
    return hip_status(hipGetLastError());
}

// Short calls (a wavefront or a block of four per (b, h)) read the table where it is: its copy would cost more than the
// few rows they look at.  Long ones come in the kinds of calls there are: packed rows alone (an append) with 16- or
// 12-bit main fields, unpacked outputs alone (fake quantization, encode), and anything else.
template <class D>
static int launch_d(QPair &kv, int count, hipStream_t st) {
    const QParams &p = kv.p[0];
    const int64_t chunks = (int64_t)p.T * p.n;
    const bool rows = !(p.n & (p.n - 1)) && p.n <= 64;
    constexpr int kAll = kUnpacked | kPlanes | kCompact;
    if (chunks <= 64 && rows) return launch_kernel<D, 64, true, false, kAll, 0>(kv, count, st);
    if (chunks <= kQThreads)
        return rows ? launch_kernel<D, kQThreads, true, false, kAll, 0>(kv, count, st) : launch_kernel<D, kQThreads, false, false, kAll, 0>(kv, count, st);
    if (!rows) return launch_kernel<D, 1024, false, true, kUnpacked | kPlanes, 0>(kv, count, st);
    bool unpacked = false, planes = false;
    for (int i = 0; i < count; i++) {
        const QParams &q = kv.p[i];
        unpacked |= q.idx_out || q.rq_out || q.rmax_out || q.dense_out || q.mask_out || q.stats;
        planes |= q.main_plane || q.aux_plane || q.flag_plane || q.scale_plane;
    }
    if (!planes) return launch_kernel<D, 1024, true, true, kUnpacked, 0>(kv, count, st);
    if (!unpacked && p.main_bits == 16 && kv.p[1].main_bits == 16) return launch_kernel<D, 1024, true, true, kPlanes, 16>(kv, count, st);
    if (!unpacked && p.main_bits == 12 && kv.p[1].main_bits == 12) return launch_kernel<D, 1024, true, true, kPlanes, 12>(kv, count, st);
    return launch_kernel<D, 1024, true, true, kUnpacked | kPlanes, 0>(kv, count, st);
}

int launch_quantize_grid(QPair kv, int count, int dtype, hipStream_t st) {
    switch (dtype) {
        case HQMQ_F32: return launch_d<F32>(kv, count, st);
        case HQMQ_F16: return launch_d<F16>(kv, count, st);
        default: return launch_d<BF16>(kv, count, st);
    }
}

}  // namespace hqmq

using namespace hqmq;

extern "C" int64_t hqmq_search_grid_bytes(int H, int S, int dtype) {
    if (H < 1 || (dtype != HQMQ_F32 && dtype != HQMQ_F16 && dtype != HQMQ_BF16)) return 0;
    const int64_t blocks = search_grid_blocks(S, dtype);
    return blocks ? (blocks * H + (H + 3) / 4) * 16 + (int64_t)H * 24 * S * 20 : 0;
}

extern "C" int64_t hqmq_search_grid_kept_bytes(int H, int S, int dtype) {
    return hqmq_search_grid_bytes(H, S, dtype) > 0 ? search_grid_blocks(S, dtype) * H * 16 : 0;
}

extern "C" int hqmq_build_search_grid(const void *joint, int H, int S, int dtype, void *grid, int64_t grid_bytes, void *stream) {
    if (!joint || !grid) return HQMQ_ERR_NULL;
    if (dtype != HQMQ_F32 && dtype != HQMQ_F16 && dtype != HQMQ_BF16) return HQMQ_ERR_DTYPE;
    const int64_t need = hqmq_search_grid_bytes(H, S, dtype);
    if (H > 65535 || need == 0) return HQMQ_ERR_SHAPE;
    if (grid_bytes < need) return HQMQ_ERR_WORKSPACE;
    if ((uintptr_t)grid & 15) return HQMQ_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    const int64_t stride = search_grid_blocks(S, dtype);
    const int pool = (int)pool_blocks(dtype);
    const dim3 gc(3 * S, H), gb(kCoarse * kCoarse * kCoarse, H);
#define LAUNCH(DT, ST)                                                                                                              \
    do {                                                                                                                            \
        hipLaunchKernelGGL(grid_codewords_kernel<DT>, gc, dim3(256), 0, st, (const ST *)joint, S, (uint4 *)grid, stride, H);        \
        hipLaunchKernelGGL(grid_build_kernel<DT>, gb, dim3(kBuildThreads), 0, st, S, (uint4 *)grid, stride, pool, H);                          \
    } while (0)
    switch (dtype) {
        case HQMQ_F32: LAUNCH(F32, float); break;
        case HQMQ_F16: LAUNCH(F16, uint16_t); break;
        default: LAUNCH(BF16, uint16_t); break;
    }
#undef LAUNCH
    return hip_status(hipGetLastError());
}
