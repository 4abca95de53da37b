// Codeword search through cell lists.
//
// The codebook {q_p * q_s} is closed under left multiplication by the 24 Hurwitz units, and so is the score:
// <u, q_p * q_s> = <conj(e) * u, (conj(e) * q_p) * q_s> for every unit e.  Eight of the units are the axes {+-1, +-i, +-j,
// +-k}: multiplying a direction u by the conjugate of the axis nearest to it (its component of largest magnitude) permutes
// its components and changes signs, no more, and brings it into the cell of S^3 around 1, |w_i| <= w0.  Only 1 / 8 of the
// directions are left to be searched.  Seen in stereographic projection, z = (w1, w2, w3) / (w0 + 1), that cell almost
// fills the cube |z_i| <= sqrt(2) - 1, and equal boxes of the cube are nearly equal pieces of the sphere (the scale goes
// from 2 to 1.5).  A grid of kGrid^3 boxes over the cube carries, per box, the list of all codewords (p', s) that can win
// the reference's rounded comparison for some direction inside it; the lists are worked out once per codebook
// (hqmq_build_search_grid).  A search is then: the largest component, one reciprocal, one list look-up, and the
// reference's own rounded score (bit for bit) for the few codewords of the list; the largest score wins, the smallest index
// k = p * S + s among equals.
//
// The box is found without carrying out the multiplication: two packed multiply-adds put the positions t_j of u's four
// components into 16-bit halves, and since w is u with components exchanged and signs changed, the box number is a sum of
// +-1, +-kGrid, +-kGrid^2 times three of them - two dot products with constants that belong to the axis.  kGrid is odd, so
// rounding to the nearest box commutes with a change of sign.
//
// The reference scores with the stored table J, whose rows are rounded products: conj(e) * J[k] depends on e.  A
// codeword (p', s) therefore stands for 8 points, taken as a centre and the radius rho of the ball around it.
// A codeword g is left out of a box when some codeword g* beats it by more than any rounding can turn, everywhere in
// the box: <(1 - |z|^2, 2 z), g* - g> > (rho_g + rho_g* + m) (1 + |z|^2).  That is one parabola per coordinate, so its
// least value in the box is three least values on an interval.  g* is the best codeword at the box's centre, then every
// other one of the box's list.  m covers the roundings of the two scores to D: half a unit in the last place each, 2^-12
// (fp16) and 2^-9 (bf16) for scores in [0.5, 1), twice that where a score can reach 1 (directions are vectors of length 1
// within 1.5 %; others are scored against all rows).
//
// Lists, per head, in blocks of 16 bytes: seven 16-bit entries and the number of the block that goes on (0: none, 0xffff: no
// list, score all rows).  An entry holds p' << 2 and bit 8 of s' = S - 1 - s in its lower byte, the other bits of s' in its
// upper one (p' = 31: no entry): a byte is an operand of the vector unit, and the lower one, exclusive-or'ed with the axis,
// is the address of the number of row q_e * q_p', 0.  The first kCells blocks are the boxes', the others a pool that the
// build hands out; block 0 of the pool holds no entry.  That is 384 KB per head for fp16, fp32 and bf16 up to S = 32, for
// bf16 615 KB up to S = 96, 922 KB up to 192 and 1230 KB above.  Behind the lists of all heads lies what only the build
// reads and a caller may drop afterwards (hqmq_search_grid_kept_bytes): the pools' counters, the centres and radii of the
// codewords.
//
// What it costs: per 64 chunks 182 vector-ALU instructions at fp16 s96_r4, 254 at bf16 s24_r3 with flags (the selection of the
// threshold included), where the scan over 96 secondaries takes 1,885.  Bound by vector-ALU issue: 0.86 (fp16) and 0.90 (bf16) of the
// cycles a compute unit is busy, transcendental instructions counted once; its LDS pipe 36 and 39 %, half of it bank conflicts.  K and V of
// 8 x 32768 tokens, fp16, s96_r4, packed: 119.5 us; 8 x 4 x 4001 tokens bf16 s24_r3 with Med3x, whole call: 97 us.  With rows packed through LDS
// (180 and 249 vector instructions, but 99 and 192 scalar ones instead of 59 and 119): 123 and 117 us.  The form before that reduced directions to the
// cell of all 24 units (75 instructions for unit, quaternion product and box, where this takes 25), listed 3.35 codewords
// per box on average (S = 96, fp16; 8.7 is the longest of 64) where this lists 3.1 (7.5), and rounded every 16-bit number
// by itself: 342 and 450 instructions, 186 and 163 us.  33 boxes per axis instead of 27 take 5 % fewer instructions, 1 % less
// time and 1.8 times the memory; 27 without the comparison of all pairs: lists of 3.35 (9.3).
//
// Compiled with -ffp-contract=off; fused multiply-adds are written explicitly.
#include "med_select.h"

#include <type_traits>

namespace hqmq {

constexpr int kCoarse = 9;                      // boxes per axis of the build's first level
constexpr int kFine = 3;                        // boxes per axis inside one of those
constexpr int kGrid = kCoarse * kFine;          // odd: a box's mirror image is a box
constexpr int kMid = kGrid / 2;
constexpr int kCells = kGrid * kGrid * kGrid;
constexpr int kGridSMax = 341;                  // 24 * 341 rows of 8 bytes: row offsets fit 16 bits, s' fits 9
constexpr uint32_t kNone = 31u << 2;            // an empty entry
constexpr float kScale = (0.5f * kGrid - 0.1f) / 0.41422f;       // boxes per unit of z; the cell reaches |z_i| = sqrt(2) - 1
// How far, in boxes, the position that the search computes may lie from the direction's own: the reciprocal and (fp32) the
// components are rounded to fp16 (2^-11 of at most 13.4 each), w0 may be the unrounded quotient (fp16: half of 2^-11), and
// the search takes 1 for the length of a direction whose norm and components were rounded to D (2^-10 and 2^-7, two thirds
// of which reach z).
template <class D>
constexpr float slack_boxes() { return D::code == HQMQ_BF16 ? 0.085f : 0.022f; }
static_assert(0.5f * kGrid - 0.1f + 0.085f < kMid + 0.5f, "every direction's box is inside the grid");

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
__device__ const Units d_units = make_units();

// What the search needs to know of a unit e of {+-1, +-i, +-j, +-k}: the box number of w = conj(e) * u from the positions
// t_0 .. t_3 of u's components, 16 * (sum_j a_j t_j) + first, as two dot products of 16-bit numbers.  The positions come as
// the bits of fp16 numbers 1536 + t, which is 0x6600 + t.
struct AxisUnits {
    uint32_t a01[8], a23[8];
    int32_t first[8];
};
constexpr AxisUnits make_axis_units() {
    AxisUnits t{};
    const int stride[4] = {0, kGrid * kGrid, kGrid, 1};
    for (int e = 0; e < 8; e++) {
        int a[4] = {};
        const float q[4] = {unit_part(e, 0), -unit_part(e, 1), -unit_part(e, 2), -unit_part(e, 3)};
        for (int j = 0; j < 4; j++) {
            float u[4] = {};
            u[j] = 1.f;
            const float w[4] = {q[0] * u[0] - q[1] * u[1] - q[2] * u[2] - q[3] * u[3], q[0] * u[1] + q[1] * u[0] + q[2] * u[3] - q[3] * u[2],
                                q[0] * u[2] - q[1] * u[3] + q[2] * u[0] + q[3] * u[1], q[0] * u[3] + q[1] * u[2] - q[2] * u[1] + q[3] * u[0]};
            for (int c = 1; c < 4; c++) a[j] += 16 * stride[c] * (int)w[c];
        }
        t.a01[e] = ((uint32_t)a[0] & 0xffffu) | (uint32_t)a[1] << 16;
        t.a23[e] = ((uint32_t)a[2] & 0xffffu) | (uint32_t)a[3] << 16;
        t.first[e] = 16 * kMid * (kGrid * kGrid + kGrid + 1) - 0x6600 * (a[0] + a[1] + a[2] + a[3]);
    }
    return t;
}
__device__ const AxisUnits d_axis = make_axis_units();
static_assert(16 * kGrid * kGrid < 32768, "strides are 16-bit");

// Blocks of the pool.  Random codebooks (16 heads each) take at most 19 / 214 / 929 / 2903 at S = 24 / 96 / 192 / 341 with
// fp16, less with fp32, 190 / 7319 / 18733 / 33140 with bf16.  A box that finds the pool empty scores all rows.
constexpr int64_t pool_blocks(int S, int dtype) {
    return dtype != HQMQ_BF16 || S <= 32 ? kCells / 4 : S <= 96 ? kCells : S <= 192 ? 2 * kCells : 3 * kCells;
}
static_assert(3 * kCells < 65535, "block numbers are 16-bit");
// The first blocks of the pool, which long calls hold in LDS: as many as random codebooks take where that is few.  One list in 80
// (fp16, S = 96) goes on in the pool, so half the wavefronts' searches do, and from the L2 the block came last of all a round waits for.
// us, from the L2 and from LDS: K and V of 8 x 32768 tokens, fp16 s96_r4, 122.4 / 119.1; 8 x 4096 tokens encoded 24.2 / 23.3; 4 x 8 x 4001
// bf16 s24_r3 with Med3x 106.9 / 104.7.  bf16 codebooks above S = 32 take 7000 blocks and more, fp32 ones hardly any.
constexpr int pool_blocks_lds(int S, int dtype) {
    return dtype == HQMQ_F32 ? 0 : dtype == HQMQ_BF16 ? (S <= 32 ? 256 : 0) : S <= 96 ? 256 : S <= 192 ? 1024 : 0;
}
constexpr int kPoolRounds = 2;                  // and where a block takes that many rounds: one round of S = 192 lost 0.2 us to the copy

int64_t search_grid_blocks(int S, int dtype) {
    if (S < 1 || S > kGridSMax) return 0;
    return kCells + pool_blocks(S, dtype);
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

// Centre and radius of the 8 points conj(e) * J[e * q_p', s] for every (p', s), 8 lanes per codeword; the head's counter
// and empty block.
template <class D>
__global__ __launch_bounds__(256) void grid_codewords_kernel(const typename D::storage *joint, int S, uint4 *grid, int64_t stride, int H) {
    const int h = blockIdx.y, k = blockIdx.x * 32 + (threadIdx.x >> 3), g = threadIdx.x & 7;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        grid_counters(grid, stride, H)[h] = 1;
        grid[stride * h + kCells] = uint4{kNone | kNone << 16, kNone | kNone << 16, kNone | kNone << 16, kNone};
    }
    if (k >= 24 * S) return;            // (24 S is a multiple of 8: whole wavefronts)
    const int p = k / S, s = k - p * S;
    const typename D::storage *r = joint + ((size_t)h * 24 * S + (size_t)d_units.mul[g][p] * S + s) * 4;
    const float *q = d_units.q[g];
    const float4 v = quat_mul(float4{q[0], -q[1], -q[2], -q[3]}, float4{D::load(r), D::load(r + 1), D::load(r + 2), D::load(r + 3)});
    auto most = [](float x, auto op) {
        for (int o = 4; o; o >>= 1) x = op(x, __shfl_xor(x, o, 8));
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
    if (g == 0) {
        cw.centre[(size_t)h * 24 * S + k] = c;
        cw.rho[(size_t)h * 24 * S + k] = far * 1.00001f + 1e-6f;
    }
}

// One block per coarse box and head.  First the codewords that matter anywhere in the coarse box are listed in LDS
// (lanes over codewords), then the kFine^3 boxes inside it are worked out from that list, kLanes lanes per box, and every
// listed codeword is held against every other one.  kListCap bounds the coarse list, kBoxCap a box's (random codebooks stay
// far below both: no box of S = 24 ... 341 goes without a list); beyond either the box scores all rows.
constexpr int kListCap = 1024;
constexpr int kBoxCap = 126;
constexpr int kBuildThreads = 256;
constexpr int kBoxes = kFine * kFine * kFine;
constexpr int kLanes = 8;                       // per box
static_assert(kBoxes * kLanes <= kBuildThreads && kLanes == 8, "lanes per box");
template <class D>
__global__ __launch_bounds__(kBuildThreads) void grid_build_kernel(int S, uint4 *grid, int64_t stride, int pool, int H) {
    const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int ci = blockIdx.x / (kCoarse * kCoarse), cj = blockIdx.x / kCoarse % kCoarse, ck = blockIdx.x % kCoarse;
    __shared__ float4 geo[kListCap];
    __shared__ float rad[kListCap];
    __shared__ uint16_t id[kListCap];                          // as an entry
    __shared__ uint16_t entries[kBoxes][kBoxCap + 1];          // positions in the coarse list
    __shared__ uint16_t kept[kBoxes][kBoxCap + 1];             // what stays of them, as entries
    __shared__ float needs_sh[kBoxes][kBoxCap + 1];
    __shared__ int count[kBoxes];
    __shared__ float best_sh[kBuildThreads / 64];
    __shared__ int arg_sh[kBuildThreads / 64], n_sh, more_sh;
    __shared__ uint32_t first_sh;
    const int K = 24 * S;
    const Codewords all = grid_codewords(grid, stride, H, S);
    const float4 *centre = all.centre + (size_t)h * K;
    const float *rho = all.rho + (size_t)h * K;
    // c: centre, hw: half width, c2: |c|^2; mid: the direction at the centre; reach: the farthest one's angle
    struct Box { float c[3], hw, c2; float4 mid; float reach; bool met; };
    auto box_at = [](int i, int j, int k, int fine) {           // fine: fine boxes per axis of this one
        Box b;
        const int at[3] = {i, j, k};
        b.hw = (0.5f * (float)fine + slack_boxes<D>()) * (1.f / kScale) + 2e-6f;
        float near2 = 0.f, near[3];
        b.c2 = 0.f;
        for (int a = 0; a < 3; a++) {
            b.c[a] = ((float)(at[a] * fine - kMid) + 0.5f * (float)(fine - 1)) * (1.f / kScale);
            near[a] = fmaxf(fabsf(b.c[a]) - b.hw, 0.f);
            near2 += near[a] * near[a];
            b.c2 += b.c[a] * b.c[a];
        }
        // the cell: |w_i| <= w0, that is |z|^2 + 2 |z_i| <= 1
        b.met = near2 + 2.f * fmaxf(near[0], fmaxf(near[1], near[2])) <= 1.0005f;
        const float inv = 1.f / (1.f + b.c2);
        b.mid = float4{(1.f - b.c2) * inv, 2.f * b.c[0] * inv, 2.f * b.c[1] * inv, 2.f * b.c[2] * inv};
        b.reach = 2.f * 1.7321f * b.hw;
        return b;
    };
    auto dot = [](float4 g, float4 m) { return fmaf(g.w, m.w, fmaf(g.z, m.z, fmaf(g.y, m.y, g.x * m.x))); };
    // what g* has to lead by, less the radius of g: its own radius, the roundings of both scores, and of this kernel
    auto needs = [&](float4 star, float r, const Box &b) {
        // its largest score in the box: from the angle at the centre, less the box's reach
        const float len = sqrtf(star.x * star.x + star.y * star.y + star.z * star.z + star.w * star.w);
        const float c = fminf(dot(star, b.mid) / len, 1.f), s = sqrtf(fmaxf(1.f - c * c, 0.f));
        const float cr = 1.f - 0.5f * b.reach * b.reach, sr = b.reach;          // cos >= cr, sin <= sr
        const float most = (c > cr ? 1.f : fminf(c + s * sr, 1.f)) * len + r;
        return 1.016f * (most * 1.016f < 1.f ? 1.f : 2.f) * D::eps() + 1.2e-5f + r;
    };
    // Is <d, (1 - |z|^2, 2 z)> > m (1 + |z|^2) with d = g* - g all over the box?  A sum of one parabola 2 d_i z - a z^2 per
    // coordinate, a = d_0 + m: at least its value at the centre less the slope there times half the width, and less a hw^2
    // where it bends down.
    auto beaten = [](float4 s, float need, float4 g, float r, const Box &b) {
        const float d0 = s.x - g.x, d1 = s.y - g.y, d2 = s.z - g.z, d3 = s.w - g.w, m = (need + r) * 1.0001f, a = d0 + m;
        const float slopes = fabsf(fmaf(-a, b.c[0], d1)) + fabsf(fmaf(-a, b.c[1], d2)) + fabsf(fmaf(-a, b.c[2], d3));
        const float half = fmaf(d3, b.c[2], fmaf(d2, b.c[1], fmaf(d1, b.c[0], -b.hw * slopes)));
        return fmaf(2.f, half, d0 - m) - fmaf(a, b.c2, 3.f * b.hw * b.hw * fmaxf(a, 0.f)) > 2e-6f;
    };
    uint4 *lists = grid + stride * h;
    const int f = tid / kLanes, part = tid % kLanes;
    const int i = ci * kFine + f / (kFine * kFine), j = cj * kFine + f / kFine % kFine, k = ck * kFine + f % kFine;
    const bool mine = f < kBoxes;
    const uint4 empty = uint4{kNone | kNone << 16, kNone | kNone << 16, kNone | kNone << 16, kNone};
    const Box coarse = box_at(ci, cj, ck, kFine);
    if (!coarse.met) {                      // (no direction looks there; a block all the same, for lanes whose box is not used)
        if (mine && part == 0) lists[(i * kGrid + j) * kGrid + k] = empty;
        return;
    }
    if (tid == 0) n_sh = more_sh = 0;
    if (tid < kBoxes) count[tid] = 0;
    {
        float best = -INFINITY;
        int arg = 0;
#pragma unroll 8
        for (int k2 = tid; k2 < K; k2 += kBuildThreads) {
            const float v = dot(centre[k2], coarse.mid) - rho[k2];
            if (v > best) { best = v; arg = k2; }
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
        const float need = needs(star, rho[arg], coarse), inv_s = 1.f / (float)S;
        float4 ahead = centre[min(tid, K - 1)];
        float ahead_r = rho[min(tid, K - 1)];
        for (int k0 = 0; k0 < K; k0 += kBuildThreads) {
            const int k2 = k0 + tid;
            const float4 g = ahead;
            const float r = ahead_r;
            ahead = centre[min(k2 + kBuildThreads, K - 1)];
            ahead_r = rho[min(k2 + kBuildThreads, K - 1)];
            const bool take = k2 < K && !beaten(star, need, g, r, coarse);
            const uint64_t mask = __builtin_amdgcn_ballot_w64(take);
            int at = 0;
            if (lane == 0 && mask) at = atomicAdd(&n_sh, (int)__popcll(mask));
            at = __shfl(at, 0) + __popcll(mask & ((1ull << lane) - 1ull));
            if (take && at < kListCap) {
                const int p = (int)(((float)k2 + 0.5f) * inv_s), s = S - 1 - (k2 - p * S);       // (k2 < 8192: exact)
                geo[at] = g;
                rad[at] = r;
                id[at] = (uint16_t)(p << 2 | (s >> 8) << 7 | (s & 0xff) << 8);
            }
        }
        __syncthreads();
    }
    const int n_list = n_sh;
    uint32_t *used = grid_counters(grid, stride, H) + h;
    const Box b = box_at(i, j, k, 1);
    const bool listed = n_list <= kListCap, wanted = mine && b.met && listed;
    if (wanted) {
        float best = -INFINITY;
        int arg = 0;
#pragma unroll 4
        for (int e = part; e < n_list; e += kLanes) {
            const float v = dot(geo[e], b.mid) - rad[e];
            if (v > best) { best = v; arg = e; }
        }
        for (int o = 1; o < kLanes; o <<= 1) {
            const float v = __shfl_xor(best, o);
            const int g = __shfl_xor(arg, o);
            if (v > best || (v == best && g < arg)) { best = v; arg = g; }
        }
        const float4 star = geo[arg];
        const float need = needs(star, rad[arg], b);
        for (int e = part; e < n_list; e += kLanes) {
            if (beaten(star, need, geo[e], rad[e], b)) continue;
            const int at = atomicAdd(&count[f], 1);
            if (at < kBoxCap) entries[f][at] = (uint16_t)e;
        }
    }
    __syncthreads();
    // every codeword of the box against every other one (one that is beaten all over the box is beaten by one that stays: the
    // leads add up), then the blocks, a lane each
    if (wanted && count[f] <= kBoxCap)
        for (int x = part; x < count[f]; x += kLanes) needs_sh[f][x] = needs(geo[entries[f][x]], rad[entries[f][x]], b);
    __syncthreads();
    const int cell = (i * kGrid + j) * kGrid + k;
    const bool listed_here = wanted && count[f] <= kBoxCap;
    const int all_n = listed_here ? count[f] : 0;
    int n = 0;
    for (int x0 = 0; x0 < all_n; x0 += kLanes) {
        const int x = x0 + part;
        bool stays = x < all_n;
        int e = 0;
        if (stays) {
            e = entries[f][x];
            const float4 g = geo[e];
            const float r = rad[e];
#pragma unroll 4
            for (int y = 0; y < all_n; y++) stays &= y == x || !beaten(geo[entries[f][y]], needs_sh[f][y], g, r, b);
        }
        const uint32_t votes = (uint32_t)(__builtin_amdgcn_ballot_w64(stays) >> (lane & ~(kLanes - 1))) & ((1u << kLanes) - 1u);
        if (stays) kept[f][n + __popc(votes & ((1u << part) - 1u))] = id[e];
        n += __popc(votes);
    }
    // blocks from the pool, for all boxes together (every box asking for its own: the additions to the head's one counter took
    // most of the build at bf16)
    const int more = n > 7 ? (n - 1) / 7 : 0;
    uint32_t next = 0;
    if (more && part == 0) next = (uint32_t)atomicAdd(&more_sh, more);
    __syncthreads();
    if (tid == 0) first_sh = more_sh ? atomicAdd(used, (uint32_t)more_sh) : 0u;
    __syncthreads();
    if (!mine) return;
    if (!b.met) {
        if (part == 0) lists[cell] = empty;
        return;
    }
    next = __shfl(next, 0, kLanes) + first_sh;
    const bool full = !listed_here || next + more > (uint32_t)pool;
    for (int q = part; q <= (full ? 0 : more); q += kLanes) {
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 7; e++) w[e] = !full && 7 * q + e < n ? kept[f][7 * q + e] : kNone;
        w[7] = full ? 0xffffu : q == more ? 0u : next + q;
        lists[q == 0 ? cell : kCells + (int)next + q - 1] = uint4{w[0] | w[1] << 16, w[2] | w[3] << 16, w[4] | w[5] << 16, w[6] | w[7] << 16};
    }
}

// ---------------------------------------------------------------- search
// LDS: the axis units | row numbers by (unit of the direction, low byte of the entry) | K rows of the joint table, last row
// first (JLDS; bf16 widened to fp32) | the first blocks of the pool (JLDS) | one or two words per lane.  The dynamic block is the kernel's only LDS, so it starts
// at LDS address 0.
template <class D>
constexpr int lds_row_bytes() { return D::code == HQMQ_F16 ? 8 : 16; }
constexpr int kUnitsAt = 256, kRowsAt = kUnitsAt + 8 * 64 * 4;
// ChunkSink's second word per lane
template <bool ROWS, int WHAT>
constexpr bool needs_aux(int n) { return !ROWS || (WHAT & kCompact) || n < 8; }

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef short s2 __attribute__((ext_vector_type(2)));
// two fp32 numbers rounded to 16 bits each, in one instruction
__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
    return __builtin_bit_cast(uint32_t, h2{(_Float16)a, (_Float16)b});
}
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) { return __builtin_bit_cast(uint32_t, b2{(__bf16)a, (__bf16)b}); }
// a ^ one byte of b (the compiler shifts first)
__device__ __forceinline__ uint32_t xor_byte0(uint32_t a, uint32_t b) { return a ^ (b & 0xffu); }
__device__ __forceinline__ uint32_t xor_byte2(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_xor_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// k's upper half = s rounded to fp16 (from fp32: see F16::rnd); the s_nop lets the half written last arrive
__device__ __forceinline__ void round_over(uint32_t &k0, float s0, uint32_t &k1, float s1) {
    asm("v_cvt_f16_f32_sdwa %0, %2 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD\n\t"
        "v_cvt_f16_f32_sdwa %1, %3 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD\n\ts_nop 0" : "+v"(k0), "+v"(k1) : "v"(s0), "v"(s1));
}
__device__ __forceinline__ void round_over(uint32_t &k, float s) {
    asm("v_cvt_f16_f32_sdwa %0, %1 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD\n\ts_nop 0" : "+v"(k) : "v"(s));
}
// mixed multiply-adds on half j of w (the compiler converts the halves first): w_j * y, and w_j - r * q in one rounding
__device__ __forceinline__ float half_times(uint32_t w, int j, float y) {
    float o;
    if (j) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(o) : "v"(w), "v"(y));
    else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(o) : "v"(w), "v"(y));
    return o;
}
__device__ __forceinline__ float half_less(uint32_t w, int j, float r, float q) {
    float o;
    if (j) asm("v_fma_mix_f32 %0, -%2, %3, %1 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(o) : "v"(w), "v"(r), "v"(q));
    else asm("v_fma_mix_f32 %0, -%2, %3, %1 op_sel_hi:[0,0,1]" : "=v"(o) : "v"(w), "v"(r), "v"(q));
    return o;
}
__device__ __forceinline__ float half_at(uint32_t w, int j) { return (float)__builtin_bit_cast(h2, w)[j]; }

// A row of the joint table as the search holds it: as stored, or bf16 widened to fp32 (from LDS)
template <class D, bool JLDS>
struct RowWords {
    RawChunk<D> raw;
    uint32_t (&w)[sizeof(typename D::storage)] = raw.w;
    __device__ __forceinline__ float get(int j) const { return raw.get(j); }
};
template <>
struct RowWords<BF16, true> {
    uint32_t w[4];
    __device__ __forceinline__ float get(int j) const { return __uint_as_float(w[j]); }
};

// The best of all K rows for one direction, the same in all lanes, by the whole wavefront: torch's rule, first maximum, NaN counts as
// maximum.  (Each lane for its own direction held up the wavefront for K rows: 8 x 8192 tokens over codebooks of perturbed
// units, S = 192 bf16 with 0.2 % of the boxes without a list 3152 -> 120 us, 341 fp16 with 0.4 % 6422 -> 190, 341 bf16 with 3.2 %
// 13172 -> 721.)  A candidate is one word for 16-bit types, score in order and row number from the end, and two for fp32: the search has
// no registers to spare.
template <class D>
__device__ __forceinline__ int wave_argmax(const float (&u)[4], const typename D::storage *jh, int K) {
    constexpr bool W = D::code == HQMQ_F32;
    uint32_t key = 0, last = 0;                                         // last: fp32's row number
    uint32_t k;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(k));       // the lane; nothing of this is worked out ahead
    for (; k < (uint32_t)K; k += 64u) {
        const float s = ref_score<D>(u, jh + k * 4u) + 0.f;             // (-0 and 0 are equal)
        uint32_t x;
        if constexpr (D::code == HQMQ_F16) x = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)s) << 16;
        else x = __float_as_uint(s);
        x = is_nan(s) ? ~0u : x ^ ((uint32_t)((int32_t)x >> 31) | 0x80000000u);
        if constexpr (W) {
            last = x > key || last == 0u ? (uint32_t)K - k : last;      // (k grows: the first of equals stays)
            key = max(key, x);
        } else key = max(key, (x & 0xffff0000u) | (uint32_t)K - k);
    }
    auto join = [&](uint32_t x, uint32_t l) {
        if constexpr (W) last = x > key ? l : x == key ? max(last, l) : last;
        key = max(key, x);
    };
    // lanes 1, 2, 7 and 15 away from each other within rows of 16 (DPP), then the rows
#define ACROSS(CTRL) join((uint32_t)__builtin_amdgcn_update_dpp(0, (int)key, CTRL, 0xF, 0xF, false), W ? (uint32_t)__builtin_amdgcn_update_dpp(0, (int)last, CTRL, 0xF, 0xF, false) : 0u)
    ACROSS(0xB1);           // quad_perm [1,0,3,2]
    ACROSS(0x4E);           // quad_perm [2,3,0,1]
    ACROSS(0x141);          // row_half_mirror
    ACROSS(0x140);          // row_mirror
#undef ACROSS
    for (int row = 1; row < 4; row++)
        join((uint32_t)__builtin_amdgcn_readlane((int)key, 16 * row), W ? (uint32_t)__builtin_amdgcn_readlane((int)last, 16 * row) : 0u);
    key = (uint32_t)__builtin_amdgcn_readlane((int)key, 0);
    if constexpr (W) last = (uint32_t)__builtin_amdgcn_readlane((int)last, 0);
    return K - (int)(W ? last : key & 0xffffu);
}

template <class D, int NT, bool ROWS, bool JLDS, int WHAT, int MB, bool FAST, bool SEL>
__device__ __forceinline__ void grid_body(const QParams &a, int bh, int block, int med_at) {
    using ST = typename D::storage;
    typedef const uint32_t __attribute__((address_space(3))) *lds_u32;
    typedef uint32_t __attribute__((ext_vector_type(2))) u32x2;
    typedef uint32_t __attribute__((ext_vector_type(4))) u32x4;
    typedef const u32x2 __attribute__((address_space(3))) *lds_u64;
    typedef const u32x4 __attribute__((address_space(3))) *lds_u128;
    constexpr int RB = JLDS ? lds_row_bytes<D>() : 4 * (int)sizeof(ST);            // bytes of a row where it is read
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, n = a.n, S = a.S, K = 24 * S;
    const int b = bh / a.H, h = bh - b * a.H;
    const ST *jh = (const ST *)a.joint + (size_t)h * K * 4;
    const int pool_lds = JLDS && a.iters >= kPoolRounds ? pool_blocks_lds(S, D::code) : 0;
    const uint32_t pool_at = kRowsAt + (JLDS ? (uint32_t)(K * RB) : 0u);
    uint32_t *code_sh = reinterpret_cast<uint32_t *>(lds + pool_at + 16 * pool_lds), *aux_sh = code_sh + NT;
    const int tpb = NT / n, tok_local = tid / n, c = tid - tok_local * n;
    const int t_first = block * a.iters * tpb;
    const ST *xl = (const ST *)a.x + b * a.xsb + h * a.xsh + (int64_t)(t_first + tok_local) * a.xst + c * 4;
    const int64_t x_step = tpb * a.xst;
    const int t_left = tok_local < tpb ? a.T - t_first - tok_local : 0;     // this lane has a token while t0 - t_first < t_left
    RawChunk<D> none = {};                                                        // what lanes without a token work on: an ordinary direction
    for (int j = 0; j < 4; j++) none.set(j, 1.f);
    RawChunk<D> raw = none;
    if (t_left > 0) raw.load(xl, FAST || a.vec_in);
    auto set_up = [&]() {
        // every load of the set-up is requested before the first one is used: one round trip
        constexpr int NP = (8 * 32 + NT - 1) / NT;
        uint32_t unit_mul[NP];
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int k = min(tid + i * NT, 8 * 32 - 1);
            unit_mul[i] = d_units.mul[k >> 5][min(k & 31, 23)];
        }
        const int e = min(tid, 7);
        const uint32_t a01 = d_axis.a01[e], a23 = d_axis.a23[e], first = (uint32_t)d_axis.first[e];
        if (JLDS) {
            for (int k = tid; k < K; k += NT) {
                RawChunk<D> g;
                g.load(jh + (size_t)k * 4, true);
                unsigned char *row = lds + kRowsAt + (K - 1 - k) * RB;
                if constexpr (D::code == HQMQ_BF16)
                    *reinterpret_cast<float4 *>(row) = float4{g.get(0), g.get(1), g.get(2), g.get(3)};
                else g.store(reinterpret_cast<ST *>(row), true);
            }
        }
        for (int k = tid; k < pool_lds; k += NT)
            *reinterpret_cast<uint4 *>(lds + pool_at + k * 16) = a.grid[a.grid_stride * h + kCells + k];
        uint32_t *rows = reinterpret_cast<uint32_t *>(lds + kUnitsAt);
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int k = tid + i * NT, g = k >> 5, p = k & 31;
            // Most entries have p' = 0, so the words of one p' would share a bank: the units are spread over the banks by an
            // exclusive-or.  Bit 7 of an entry's low byte is bit 8 of s'.  No entry: a row like any other.
            if (k < 8 * 32) {
                const uint32_t row = p < 24 ? (23u - unit_mul[i]) * (uint32_t)S : 0u;
                rows[g * 64 + (p ^ g)] = row;
                rows[g * 64 + ((p + 32) ^ g)] = p < 24 ? row + 256u : 0u;
            }
        }
        if (tid < 8) *reinterpret_cast<uint4 *>(lds + tid * 16) = uint4{a01, a23, first, (uint32_t)(kUnitsAt + tid * 260)};
    };
    // Med3x: the histograms are there, and every block works the threshold out for itself while its table travels, the head's first one with
    // the outputs.  As a launch of its own, whole calls, us: K and V of 2048 tokens fake-quantized, fp16 s192_r6, 45.4 (here 43.0), 700 tokens bf16
    // s24_r3 38.3 (31.8), 4 x 4001 tokens appended 101.5 (98.1), 32768 fp16 s96_r4 171 (165).
    float thr = 0.f;
    const bool selected = SEL && a.med.parts;
    if constexpr (SEL) {
        uint32_t *sh = reinterpret_cast<uint32_t *>(lds + (med_at < 0 ? 0 : med_at));
        if (!selected) set_up();
        else if (med_at >= 0) thr = select16<D>(a.med, h, b == 0 && block == 0, sh, set_up);
        else {                          // (no room for both)
            thr = select16<D>(a.med, h, b == 0 && block == 0, sh, [] {});
            __syncthreads();
            set_up();
        }
    } else set_up();
    __syncthreads();

    const unsigned char *lists = reinterpret_cast<const unsigned char *>(a.grid + a.grid_stride * h);
    ChunkSink<D, NT, ROWS, WHAT, MB, FAST> sink(a, b, h, tok_local, c, code_sh, aux_sh);
    if (selected) sink.thr = thr;
    const int t_end = JLDS ? a.iters * tpb : tpb;
    // One round, once norm and direction are known: the search and everything after it.  QUICK: every lane of the wavefront has
    // an ordinary norm of a 16-bit type.  u: the direction; with QUICK fp16, the quotients before their rounding to fp16.
    auto rest = [&](auto QUICK, int t0, bool active, const RawChunk<D> &cur, float nrm, float r, const float (&u)[4], float len, bool brute, bool zero) {
        // the direction as fp16 (fp16: exactly; otherwise for its box only)
        uint32_t ud[2] = {pack_f16(u[0], u[1]), pack_f16(u[2], u[3])};
        if (D::code == HQMQ_F16) asm("" : "+v"(ud[0]), "+v"(ud[1]));          // (read as they are by mixed multiply-adds)
        // ---- the axis unit nearest to u: the component of largest magnitude.  Each competes as its bits, sign last, with
        // the number of its unit in place of the last three ----
        uint32_t best_axis = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t x = __float_as_uint(u[j]);
            const uint32_t v = (__builtin_amdgcn_alignbit(x, x, 31) & ~6u) | (uint32_t)(2 * j);
            best_axis = max(best_axis, v);
        }
        const float w0 = __uint_as_float(best_axis >> 1);
        const u32x4 axis = *(lds_u128)(uintptr_t)(best_axis << 4 & 0x70u);

        // ---- its box: z = w / (w0 + |u|), positions as fp16 numbers 1536 + t ----
        const float inv = __builtin_amdgcn_rcpf(fmaf(w0, 1.f / kScale, len * (1.f / kScale)));
        const h2 inv2 = __builtin_bit_cast(h2, pack_f16(inv, inv)), magic = {(_Float16)1536.f, (_Float16)1536.f};
        const h2 t01 = __builtin_elementwise_fma(__builtin_bit_cast(h2, ud[0]), inv2, magic), t23 = __builtin_elementwise_fma(__builtin_bit_cast(h2, ud[1]), inv2, magic);
        const uint32_t a01 = axis[0], a23 = axis[1];
        int at_box = __builtin_amdgcn_sdot2(__builtin_bit_cast(s2, t01), __builtin_bit_cast(s2, a01), (int)axis[2], false);
        at_box = __builtin_amdgcn_sdot2(__builtin_bit_cast(s2, t23), __builtin_bit_cast(s2, a23), at_box, false);
        // (a direction that is not of length 1 may end up anywhere: its list is not used)
        uint4 e = *reinterpret_cast<const uint4 *>(lists + min((uint32_t)at_box, (uint32_t)(kCells - 1) * 16u));

        // ---- the reference's score of every codeword of the list ----
        int key = 0;                                                    // 16-bit types: rounded score << 16 | row number
        float best = -INFINITY;                                         // fp32
        uint32_t best_at = 0;
        const uint32_t unit_row = axis[3];
        // The entries of `words` dwords (the upper half of the last one is none with ODD): row numbers, rows, scores, each
        // asked for together.  A row number counts from the end of the table: the larger of two is the smaller index k.
        auto score = [&](const uint32_t *e, auto WORDS, auto ODD) {
            constexpr int N = 2 * WORDS.value - ODD.value;
            uint32_t at[N];
            RowWords<D, JLDS> row[N];
            float s[N];
#pragma unroll
            for (int i = 0; i < N; i++) at[i] = *(lds_u32)(uintptr_t)(i & 1 ? xor_byte2(unit_row, e[i >> 1]) : xor_byte0(unit_row, e[i >> 1]));
#pragma unroll
            for (int i = 0; i < N; i++) at[i] += (i & 1 ? e[i >> 1] >> 24 : e[i >> 1] >> 8 & 0xffu);
#pragma unroll
            for (int i = 0; i < N; i++) {
                if constexpr (!JLDS) row[i].raw.load(reinterpret_cast<const ST *>(reinterpret_cast<const unsigned char *>(jh + (size_t)(K - 1) * 4) - at[i] * RB), true);
                else if constexpr (RB == 8) { const u32x2 v = *(lds_u64)(uintptr_t)(kRowsAt + at[i] * RB); row[i].w[0] = v[0]; row[i].w[1] = v[1]; }
                else { const u32x4 v = *(lds_u128)(uintptr_t)(kRowsAt + at[i] * RB); for (int j = 0; j < 4; j++) row[i].w[j] = v[j]; }
            }
#pragma unroll
            for (int i = 0; i < N; i++) {
                auto dir = [&](int j) { return D::code == HQMQ_F16 ? half_at(ud[j >> 1], j & 1) : u[j]; };
                s[i] = fmaf(dir(0), row[i].get(0), 0.f);                // the product's own rounding (a sum with 0 keeps it)
#pragma unroll
                for (int j = 1; j < 4; j++) s[i] = fmaf(dir(j), row[i].get(j), s[i]);
            }
            if constexpr (D::code == HQMQ_F32) {
#pragma unroll
                for (int i = 0; i < N; i++) {
                    const bool more = s[i] > best || (s[i] == best && at[i] > best_at);
                    best = more ? s[i] : best;
                    best_at = more ? at[i] : best_at;
                }
            } else {
#pragma unroll
                for (int i = 0; i < N; i += 2) {
                    if constexpr (D::code == HQMQ_F16) {
                        if (i + 1 < N) round_over(at[i], s[i], at[i + 1], s[i + 1]);
                        else round_over(at[i], s[i]);
                    } else {
                        const uint32_t v = pack_bf16(s[i], s[min(i + 1, N - 1)]);
                        at[i] |= v << 16;
                        if (i + 1 < N) at[i + 1] |= v & 0xffff0000u;
                    }
                    key = i + 1 < N ? max(max((int)at[i], (int)at[i + 1]), key) : max((int)at[i], key);
                }
            }
        };
        using std::integral_constant;
        typedef integral_constant<int, 0> Even;
        typedef integral_constant<int, 1> One;
        // (the first block whole: among 64 lists one has more than four entries nearly always)
        {
            const uint32_t w[4] = {e.x, e.y, e.z, e.w};
            if constexpr (RB == 8) score(w, integral_constant<int, 4>(), One());
            else {                  // (rows of 16 bytes: seven of them would not fit the registers)
                score(w, integral_constant<int, 2>(), Even());
                score(w + 2, integral_constant<int, 2>(), One());
            }
        }
        constexpr uint32_t none2 = kNone | kNone << 16;
        while (true) {
            const uint32_t next = e.w >> 16;
            if (__builtin_amdgcn_ballot_w64(next != 0u) == 0ull) break;
            if (next == 0xffffu) brute |= active && !zero;              // (a direction that is not ordinary keeps its own reason)
            const uint32_t block = next == 0xffffu ? 0u : next;
            if (JLDS && __builtin_amdgcn_ballot_w64((int)block >= pool_lds) == 0ull) {
                const u32x4 v = *(lds_u128)(uintptr_t)(pool_at + block * 16u);
                e = uint4{v[0], v[1], v[2], v[3]};
            } else e = *reinterpret_cast<const uint4 *>(lists + (kCells + block) * 16u);
            if (D::code == HQMQ_F16) asm volatile("" : "+v"(ud[0]), "+v"(ud[1]));      // (or the compiler converts them ahead of the loop)
            score(&e.x, One(), Even());
            if (__builtin_amdgcn_ballot_w64(e.y != none2)) {
                score(&e.y, One(), Even());
                if (__builtin_amdgcn_ballot_w64(e.z != none2)) {
                    const uint32_t w[2] = {e.z, e.w};
                    score(w, integral_constant<int, 2>(), One());
                }
            }
        }
        int idx = zero ? 0 : K - 1 - (int)(D::code == HQMQ_F32 ? best_at : (uint32_t)key & 0xffffu);
        for (uint64_t left = __builtin_amdgcn_ballot_w64(brute); __builtin_expect(left != 0ull, 0); left &= left - 1ull) {
            const int whose = __builtin_ctzll(left);
            float v[4];
            for (int j = 0; j < 4; j++) {
                const uint32_t w = __builtin_amdgcn_readlane(D::code == HQMQ_F16 ? ud[j >> 1] : __float_as_uint(u[j]), whose);
                v[j] = D::code == HQMQ_F16 ? __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(half_at(w, j & 1)))) : __uint_as_float(w);
            }
            const int k = wave_argmax<D>(v, jh, K);
            if ((tid & 63) == whose) idx = k;
        }
        if ((WHAT & kUnpacked) && a.stats && active) {
            if (brute) atomicAdd(a.stats, 1);
            else if (!zero) atomicAdd(a.stats + 1, 1);
        }
        auto row = [&](float (&g)[4]) {
            if constexpr (JLDS && D::code == HQMQ_BF16) {
                const float4 v = *reinterpret_cast<const float4 *>(lds + kRowsAt + (K - 1 - idx) * RB);
                g[0] = v.x; g[1] = v.y; g[2] = v.z; g[3] = v.w;
            } else {
                RawChunk<D> v;
                v.load(JLDS ? reinterpret_cast<const ST *>(lds + kRowsAt) + (K - 1 - idx) * 4 : jh + (size_t)idx * 4, true);
                for (int j = 0; j < 4; j++) g[j] = v.get(j);
            }
        };
        sink.put(t_first + t0, active, cur, nrm, r, idx, row, QUICK);
    };
    for (int t0 = 0; t0 < t_end; t0 += tpb) {
        const bool active = t0 < t_left;
        const RawChunk<D> cur = raw;
        raw = none;
        xl += x_step;
        if (t0 + tpb < t_end && t0 + tpb < t_left) raw.load(xl, FAST || a.vec_in);      // the next round's chunk

        // ---- norm and direction ----
        // 16-bit types: products of two numbers are exact in fp32, so fused multiply-adds round as products and sums do.
        // Norms of the quick range, far from D's ends, take the short forms of chunk_norm_d and div4_d; a wavefront with any
        // other (NaN, infinite, clamped, subnormal) takes the reference's operations one by one.
        if constexpr (D::code != HQMQ_F32) {
            float s = fmaf(cur.get(0), cur.get(0), 0.f);
#pragma unroll
            for (int j = 1; j < 4; j++) s = fmaf(cur.get(j), cur.get(j), s);
            const float ys = __builtin_amdgcn_rsqf(s);
            float g = s * ys;
            g = fmaf(fmaf(-g, g, s), 0.5f * ys, g);
            const float r = D::code == HQMQ_F16 ? D::rnd(g) : __uint_as_float(pack_bf16(0.f, g));
            const uint32_t lo = D::code == HQMQ_F16 ? 0x387bb000u : 0x32ac0000u, hi = D::code == HQMQ_F16 ? 0x47800000u : 0x71490000u;
            // (fp16: 6.0e-5 .. 65536, bf16: 2.0e-8 .. 9.9e29)
            if (__builtin_amdgcn_ballot_w64(__float_as_uint(r) - lo >= hi - lo) == 0ull) {
                float y = __builtin_amdgcn_rcpf(r);
                asm("s_nop 0" : "+v"(y));       // (one wait state between v_rcp and its use, which the compiler leaves to inline assembly)
                float u[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if constexpr (D::code == HQMQ_F16) {
                        u[j] = half_times(cur.w[j >> 1], j & 1, y);
                        u[j] = fmaf(half_less(cur.w[j >> 1], j & 1, r, u[j]), y, u[j]);
                        asm("" : "+v"(u[j]));                       // rounded to fp32 first, see F16::rnd
                    } else u[j] = cur.get(j) * y;
                }
                if constexpr (D::code == HQMQ_BF16) {
                    const uint32_t d01 = pack_bf16(u[0], u[1]), d23 = pack_bf16(u[2], u[3]);
                    u[0] = __uint_as_float(d01 << 16);
                    u[1] = __uint_as_float(d01 & 0xffff0000u);
                    u[2] = __uint_as_float(d23 << 16);
                    u[3] = __uint_as_float(d23 & 0xffff0000u);
                }
                rest(std::true_type(), t0, active, cur, r, r, u, 1.f, false, false);
                continue;
            }
        }
        // (a copy the compiler takes for another chunk: the quick path's multiply-adds then read the 16-bit values as they are)
        RawChunk<D> x = cur;
#pragma unroll
        for (uint32_t &w : x.w) asm("" : "+v"(w));
        float u[4];
#pragma unroll
        for (int j = 0; j < 4; j++) u[j] = x.get(j);
        const float nrm = chunk_norm_d<D>(u[0], u[1], u[2], u[3]);
        float r = clamp_min_d<D>(nrm, 1e-8f);
        if (is_nan(r)) r = NAN;
        div4_d<D>(u, r);
        // directions of length 1: the others follow the reference row by row, an all-zero direction scores 0 everywhere and
        // takes row 0
        const float len2 = fmaf(u[3], u[3], fmaf(u[2], u[2], fmaf(u[1], u[1], u[0] * u[0])));
        const bool ordinary = len2 > 0.97f && len2 < 1.03f, zero = u[0] == 0.f && u[1] == 0.f && u[2] == 0.f && u[3] == 0.f;
        rest(std::false_type(), t0, active, cur, nrm, r, u, __builtin_amdgcn_sqrtf(len2), active && !ordinary && !zero, zero);
    }
    sink.done();
}

template <class D, int NT, bool ROWS, bool JLDS, int WHAT, int MB, bool FAST, bool SEL>
__global__ __launch_bounds__(NT, NT == 1024 ? 8 : 1) void quantize_grid_kernel(QPair kv) {
    if constexpr (JLDS) {
        // blockIdx.x counts `per_head` blocks for each (tensor, b, h).  Workgroups go round-robin over the 8 XCDs; with a
        // multiple of 8 heads the blocks of one head stay on one, whose L2 then holds that head's lists and not everyone's
        // (8 heads of 32768 tokens, K and V, 512 blocks: 1.4 million cache lines from beyond the L2
        // instead of 4.3, half of which would be lists; 140 -> 123 us).
        auto same = [](int v) { return __builtin_amdgcn_readfirstlane(v); };        // (quotients come from the vector unit)
        const int per_head = kv.per_head, heads = same((int)gridDim.x / per_head), spread = heads % 8 == 0 ? 8 : 1;
        const int i = blockIdx.x / spread, q = same(i / per_head), which = q * spread + blockIdx.x % spread, bhs = kv.p[0].B * kv.p[0].H;
        const int z = same(which >= bhs ? 1 : 0);
        grid_body<D, NT, ROWS, JLDS, WHAT, MB, FAST, SEL>(kv.p[z], same(which - z * bhs), same(i - q * per_head), kv.med_at);
    } else grid_body<D, NT, ROWS, JLDS, WHAT, MB, FAST, SEL>(kv.p[blockIdx.z], blockIdx.y, blockIdx.x, -1);
}

template <class D, int NT, bool ROWS, bool JLDS, int WHAT, int MB, bool FAST = false>
static int launch_kernel(QPair &kv, int count, hipStream_t st) {
    const QParams &p = kv.p[0];
    const int tpb = NT / p.n, rounds = (p.T + tpb - 1) / tpb;
    size_t shmem = kRowsAt + (JLDS ? (size_t)(24 * p.S * lds_row_bytes<D>() + 16 * pool_blocks_lds(p.S, D::code)) : 0) + (size_t)NT * (needs_aux<ROWS, WHAT>(p.n) ? 8 : 4);
    kv.med_at = -1;
    if (JLDS && (p.med.parts || kv.p[1].med.parts)) {           // beside the table, if as many blocks share a compute unit as before
        const size_t both = (shmem + 15) / 16 * 16 + kSelectWords * 4;
        if (160 * 1024 / both == 160 * 1024 / shmem || both <= 80 * 1024) {
            kv.med_at = (int)(both - kSelectWords * 4);
            shmem = both;
        } else if (shmem < kSelectWords * 4) shmem = kSelectWords * 4;
    }
    // A block copies its head's table to LDS first, about as much work as one round.  Blocks come in waves of as many as the
    // CUs hold; the number of waves is chosen for the fewest rounds in a row, set-up included.
    int iters = 1;
    if (JLDS) {
        const int heads = p.B * p.H * count, slots = (160 * 1024 / shmem >= 2 ? 2 : 1) * 256;
        int least = INT32_MAX;
        for (int waves = 1; waves <= 8; waves++) {
            int per_head = waves * slots / heads;
            per_head = per_head < 1 ? 1 : per_head > rounds ? rounds : per_head;
            const int it = (rounds + per_head - 1) / per_head;
            const int blocks = (rounds + it - 1) / it * heads, cost = (blocks + slots - 1) / slots * (it + 1);
            if (cost < least) { least = cost; iters = it; }
        }
    }
    kv.p[0].iters = kv.p[1].iters = iters;
    kv.per_head = (rounds + iters - 1) / iters;
    const dim3 grid = JLDS ? dim3(kv.per_head * p.B * p.H * count) : dim3(rounds, p.B * p.H, count);
    auto kern = quantize_grid_kernel<D, NT, ROWS, JLDS, WHAT, MB, FAST, false>;
    if constexpr (JLDS && D::code != HQMQ_F32) {
        if (p.med.parts || kv.p[1].med.parts) kern = quantize_grid_kernel<D, NT, ROWS, JLDS, WHAT, MB, FAST, true>;
    }
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
    if constexpr (D::code != HQMQ_F32) {
        if (!unpacked && fast_rows(p, 16) && fast_rows(kv.p[1], 16)) return launch_kernel<D, 1024, true, true, kPlanes, 16, true>(kv, count, st);
        if (!unpacked && fast_rows(p, 12) && fast_rows(kv.p[1], 12)) return launch_kernel<D, 1024, true, true, kPlanes, 12, true>(kv, count, st);
    }
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
    const int pool = (int)pool_blocks(S, dtype);
    const dim3 gc((24 * S + 31) / 32, H), gb(kCoarse * kCoarse * kCoarse, H);
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
