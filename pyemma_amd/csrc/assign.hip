// Assignment of frames to their nearest cluster center.
//
// Reference semantics: label(x) = argmin_j sum_i (x_i - c_ji)^2 with the sum
// evaluated in FP32, in index order, without fused multiply-add, strict '<'
// (the first minimum wins) -- ClusterModel.transform as called from
// coordinates/clustering/interface.py:157-167.
//
// Two device paths produce exactly these labels:
//
//  * k_assign_plain: the sequential FP32 loop itself on the vector ALUs
//    (4 frames x 4 centers per thread, LDS-staged tiles).
//  * k_assign_tile in up to three passes, then exact loops on what they leave:
//    distances d~_j = |a|^2 + |b_j|^2 - 2 a.b_j on shifted data a = fl(x - mu),
//    b_j = fl(c_j - mu), from fp16 products (coarse pass, every frame) and from
//    bf16 hi/lo products (fine pass, the frames the coarse pass leaves).  With
//    E_j a rigorous bound on |d~_j - d_j| (see AsgCoef) and g = gamma_{d+2} the
//    relative rounding of the reference loop, a frame is decided when
//        (1 - g) min_{j != best} (d~_j - E_j)  >  (1 + g)(d~_best + E_best);
//    then no other center can reach the reference loop's minimum.  The other
//    frames are appended to a list and re-evaluated with the sequential FP32
//    loop, over recorded candidates or over every center (k_assign_plain).
#include <math.h>

#include <mutex>

#include "emma_common.hpp"

namespace emma {
namespace asg {

// ------------------------------------------------------------------
// exact sequential FP32 distance pieces (library built with -ffp-contract=off)
// ------------------------------------------------------------------
__device__ __forceinline__ float sq_step(float acc, float x, float c) {
    const float t = __fsub_rn(x, c);
    return __fadd_rn(acc, __fmul_rn(t, t));
}

// ------------------------------------------------------------------
// plain kernel: 64 frames x all centers per workgroup
// ------------------------------------------------------------------
constexpr int PF = 64;      // frames per workgroup
constexpr int PC = 64;      // centers per tile
constexpr int PD = 32;      // dims per staged chunk
constexpr int PPITCH = 68;  // floats per staged row (16-byte aligned)

__global__ __launch_bounds__(256) void k_assign_plain(const float *__restrict__ X, int64_t n, int d,
                                                      const float *__restrict__ C, int k,
                                                      int32_t *__restrict__ labels,
                                                      const int64_t *__restrict__ list,
                                                      const int64_t *__restrict__ list_count,
                                                      int64_t *__restrict__ n_rechecked,
                                                      const int64_t *__restrict__ n_listed,
                                                      int64_t *__restrict__ n_looped,
                                                      const int32_t *__restrict__ done) {
    if (done && *done) return;
    // the call's count of frames that this loop takes
    if (n_looped && blockIdx.x == 0 && threadIdx.x == 0) *n_looped = list ? *list_count : n;
    // the call's count of re-evaluated frames (0 for the loop over every frame)
    if (n_rechecked && blockIdx.x == 0 && threadIdx.x == 0) *n_rechecked = n_listed ? *n_listed : 0;
    __shared__ __align__(16) float xs[PD][PPITCH];
    __shared__ __align__(16) float cs[PD][PPITCH];
    __shared__ float s_best[16][PF];
    __shared__ int s_bidx[16][PF];
    __shared__ int64_t s_row[PF];
    __shared__ int s_nan0[PF];  // distance to center 0 is NaN

    const int tid = threadIdx.x;
    const int fg = tid >> 4;  // frames fg*4 .. +3
    const int cg = tid & 15;  // centers cg*4 .. +3 within the tile
    const int64_t nrows = list ? *list_count : n;
    // grid-stride over blocks of PF frames (a listed run sizes its grid for the
    // whole device and reads the list length on the device)
    for (int64_t f0 = (int64_t)blockIdx.x * PF; f0 < nrows; f0 += (int64_t)gridDim.x * PF) {
    __syncthreads();  // s_row / s_best of the previous block are consumed
    if (tid < PF) {
        const int64_t f = f0 + tid;
        s_row[tid] = f < nrows ? (list ? list[f] : f) : -1;
        s_nan0[tid] = 0;
    }
    __syncthreads();

    float best[4];
    int bidx[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        best[a] = INFINITY;
        bidx[a] = 0x7fffffff;
    }
    // loader mapping: row r = tid / 4 (0..63), dims (tid % 4) * 8 .. +7
    const int lr = tid >> 2, ld0 = (tid & 3) * 8;
    const int64_t xrow = s_row[lr];

    for (int c0 = 0; c0 < k; c0 += PC) {
        float acc[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] = 0.0f;
        const int crow = c0 + lr;
        for (int i0 = 0; i0 < d; i0 += PD) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int i = i0 + ld0 + q;
                xs[ld0 + q][lr] = (xrow >= 0 && i < d) ? X[xrow * d + i] : 0.0f;
                cs[ld0 + q][lr] = (crow < k && i < d) ? C[(int64_t)crow * d + i] : 0.0f;
            }
            __syncthreads();
            const int ni = d - i0 < PD ? d - i0 : PD;
            for (int ii = 0; ii < ni; ++ii) {
                const float4 xv = *reinterpret_cast<const float4 *>(&xs[ii][fg * 4]);
                const float4 cv = *reinterpret_cast<const float4 *>(&cs[ii][cg * 4]);
                const float xa[4] = {xv.x, xv.y, xv.z, xv.w};
                const float ca[4] = {cv.x, cv.y, cv.z, cv.w};
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b) acc[a][b] = sq_step(acc[a][b], xa[a], ca[b]);
            }
        }
        // the reference loop starts from best = d(x, c_0): a NaN there is
        // never replaced, so the label stays 0
        if (c0 == 0 && cg == 0) {
#pragma unroll
            for (int a = 0; a < 4; ++a)
                if (acc[a][0] != acc[a][0]) s_nan0[fg * 4 + a] = 1;
        }
        // centers of this thread in increasing index order: strict '<'
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int j = c0 + cg * 4 + b;
            if (j < k) {
#pragma unroll
                for (int a = 0; a < 4; ++a)
                    if (acc[a][b] < best[a]) {
                        best[a] = acc[a][b];
                        bidx[a] = j;
                    }
            }
        }
    }
    // reduce over the 16 center groups: smallest distance, then smallest index
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        s_best[cg][fg * 4 + a] = best[a];
        s_bidx[cg][fg * 4 + a] = bidx[a];
    }
    __syncthreads();
    if (tid < PF) {
        float bv = s_best[0][tid];
        int bi = s_bidx[0][tid];
        for (int g = 1; g < 16; ++g) {
            const float v = s_best[g][tid];
            const int vi = s_bidx[g][tid];
            if (v < bv || (v == bv && vi < bi)) {
                bv = v;
                bi = vi;
            }
        }
        // every distance +inf, or the distance to center 0 NaN: the
        // reference loop keeps center 0
        if (s_row[tid] >= 0) labels[s_row[tid]] = (bi == 0x7fffffff || s_nan0[tid]) ? 0 : bi;
    }
    }
}

constexpr int N_COUNTS = 8;  // counters and maxima at the head of the workspace, cleared by every call

__global__ void k_add_i64(int64_t *dst, const int64_t *src) { *dst += *src; }

// ------------------------------------------------------------------
// center preparation for the MFMA path
// ------------------------------------------------------------------
// Centers are packed once per call into "tile images", one contiguous block
// per tile of 32 centers.  An image holds the MFMA operand fragments in the
// order the lanes read them: for K-step s (16 dims) and plane p, 64 lanes x 16
// bytes, lane l the 8 dims 16 s + 8 (l / 32) .. of center l % 32, so that a
// wave loads a fragment with one contiguous 1 KB read from L2.
//   bf16 image: planes hi, lo of -2 b, b = fl(c - mu), d_pad / 16 K-steps; then
//               the constants of the 32 centers (FC_*)
//   fp16 image: one plane of -2 2^t b; then the constants HC_*
// (the factor -2 and the constant |b|^2 make d~ - |a|^2 = |b|^2 - 2 a.b the
// matrix core's own result when the accumulator starts from |b|^2).
struct CenterPack {
    uint8_t *img;    // k_pad / 32 bf16 tile images of tile_img_bytes each
    uint8_t *img16;  // k_pad / 32 fp16 tile images of tile_img16_bytes each (the coarse pass)
    float *mu;       // [d_pad] shift
    float *mx;       // [8] maxima over the centers (MX_*), zeroed before the packing, then atomic maxima
    float *sc16;     // [4] coarse pass: 2^t, 2^-2t, 2^-t
};
// constants of a bf16 image, 32 floats each: |b|^2, |b|^2 - c1b |b|^2 (the
// lower-bound start of the candidate pass), |b|, |lo part|, |what hi + lo leave|
constexpr int FC_NB = 0, FC_Q = 32, FC_BN = 64, FC_D1 = 96, FC_D2 = 128;
// constants of an fp16 image: 2^2t |b|^2, |b|, |what fp16 leaves of b|
constexpr int HC_NB = 0, HC_BN = 32, HC_D1 = 64;
constexpr int MX_BN = 0, MX_D1 = 1, MX_D2 = 2, MX_D16 = 3;

__host__ __device__ constexpr int tile_img_bytes(int d_pad) { return 128 * (d_pad + 8) + 3 * 32 * 4; }
__host__ __device__ constexpr int tile_img16_bytes(int d_pad) { return 64 * (d_pad + 8) + 3 * 32 * 4; }
static_assert(128 * 8 + 3 * 32 * 4 >= 5 * 32 * 4 && 64 * 8 + 3 * 32 * 4 >= 3 * 32 * 4, "constants fit behind the fragments");

// mu = FP64 mean (in a fixed order, rounded to FP32) of at most MU_SAMPLE
// centers spread over the set.  Any shift gives the same labels; one near the
// middle of the centers keeps |a| and |b|, and with them the error bound,
// small, and the mean of 128 centers is within a tenth of their spread of the
// mean of all.  64 dims per workgroup, wave w sums samples w, w + 16, ...: 8
// loads per lane, in flight together (one wave walking all of k = 1000 .. 4096
// centers took 92 .. 391 us, this 5).  The first workgroup clears the call's
// counters and maxima.
constexpr int MU_SAMPLE = 128, MU_WAVES = 16;
__global__ __launch_bounds__(64 * MU_WAVES) void k_center_mean(const float *__restrict__ C, int k, int d, int d_pad,
                                                               float *__restrict__ mu, int64_t *__restrict__ counts) {
    __shared__ double s_part[MU_WAVES][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (blockIdx.x == 0 && threadIdx.x < N_COUNTS) counts[threadIdx.x] = 0;
    const int i = blockIdx.x * 64 + lane;
    const int ns = k < MU_SAMPLE ? k : MU_SAMPLE;
    float v[MU_SAMPLE / MU_WAVES];
#pragma unroll
    for (int u = 0; u < MU_SAMPLE / MU_WAVES; ++u) {
        const int q = u * MU_WAVES + wave;
        v[u] = (i < d && q < ns) ? C[((int64_t)q * k / ns) * d + i] : 0.0f;
    }
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < MU_SAMPLE / MU_WAVES; ++u) acc += (double)v[u];
    s_part[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && i < d_pad) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < MU_WAVES; ++w) t += s_part[w][lane];
        mu[i] = i < d ? (float)(t / ns) : 0.0f;
    }
}

// upper bound of sqrt(v) as a float (v a nonnegative FP64 sum)
__device__ __forceinline__ float norm_up(double v) { return (float)(sqrt(v) * (1.0 + 1e-6)); }
__device__ __forceinline__ void atomic_max_pos(float *p, float v) {  // v >= 0 or NaN (which then stays)
    atomicMax(reinterpret_cast<unsigned int *>(p), __float_as_uint(v) & 0x7fffffffu);
}

// bf16 tile images; one wavefront per (padded) center, lane l owns dims 8 l .. 8 l + 7
__global__ __launch_bounds__(256) void k_center_pack(const float *__restrict__ C, int k, int d, int d_pad,
                                                     int k_pad, float c1b, CenterPack cp) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int j = blockIdx.x * 4 + wave;
    if (j >= k_pad) return;
    uint8_t *img = cp.img + (int64_t)(j >> 5) * tile_img_bytes(d_pad);
    double n2 = 0.0, e1 = 0.0, e2 = 0.0;
    if (lane * 8 < d_pad) {
        float b[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int i = lane * 8 + q;
            b[q] = (j < k && i < d) ? __fsub_rn(C[(int64_t)j * d + i], cp.mu[i]) : 0.0f;
        }
        uint32_t h[8], l[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            split_bf16(-2.0f * b[q], h[q], l[q]);
            const float lf = bf16_bits_to_f32(l[q]);
            const float r = (-2.0f * b[q] - bf16_bits_to_f32(h[q])) - lf;
            n2 += (double)b[q] * (double)b[q];
            e1 += (double)lf * (double)lf;
            e2 += (double)r * (double)r;
        }
        const int slot = (j & 31) + 32 * (lane & 1);
        uint8_t *dst = img + (lane >> 1) * 2048 + slot * 16;
        *reinterpret_cast<uint4 *>(dst) = make_uint4(pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7]));
        *reinterpret_cast<uint4 *>(dst + 1024) = make_uint4(pack2(l[0], l[1]), pack2(l[2], l[3]), pack2(l[4], l[5]), pack2(l[6], l[7]));
    }
    n2 = wave_butterfly_sum(n2);
    e1 = wave_butterfly_sum(e1);
    e2 = wave_butterfly_sum(e2);
    if (lane == 0) {
        float *cst = reinterpret_cast<float *>(img + 128 * d_pad) + (j & 31);
        // padding: a finite value beyond every real d~ (the epilogue's index
        // bits must not turn it into a NaN); never a candidate
        const bool in = j < k;
        const float nb = in ? (float)n2 : 3.0e38f, bn = in ? norm_up(n2) : 0.0f;
        const float d1 = in ? norm_up(0.25 * e1) : 0.0f, d2 = in ? norm_up(0.25 * e2) : 0.0f;
        cst[FC_NB] = nb;
        cst[FC_Q] = in ? nb - c1b * bn * bn : 3.0e38f;
        cst[FC_BN] = bn;
        cst[FC_D1] = d1;
        cst[FC_D2] = d2;
        if (in) {
            atomic_max_pos(cp.mx + MX_BN, bn);
            atomic_max_pos(cp.mx + MX_D1, d1);
            atomic_max_pos(cp.mx + MX_D2, d2);
        }
    }
}

// fp16 tile images, as above.  Scale of the coarse pass: 2^t with t = 9 - e,
// max|b| = m 2^e (m in [1/2, 1)), clamped to |t| <= 60, so that every
// |2 2^t b_ji| < 2^11 (fp16 holds up to 65504: frames with |a_i| < 128 max|b|
// stay finite; the residual of larger ones is not finite, which sends them to
// the fine pass).
__global__ __launch_bounds__(256) void k_center_pack16(const float *__restrict__ C, int k, int d, int d_pad,
                                                       int k_pad, CenterPack cp) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int j = blockIdx.x * 4 + wave;
    if (j >= k_pad) return;
    const float bm = cp.mx[MX_BN];
    int e = 0;
    frexpf(bm, &e);
    int t = bm > 0.0f && bm == bm && bm < INFINITY ? 9 - e : 0;
    t = t > 60 ? 60 : (t < -60 ? -60 : t);
    const float sc = ldexpf(1.0f, t);
    if (j == 0 && lane == 0) {
        cp.sc16[0] = sc;
        cp.sc16[1] = ldexpf(1.0f, -2 * t);
        cp.sc16[2] = ldexpf(1.0f, -t);
        cp.sc16[3] = 0.0f;
    }
    uint8_t *img = cp.img16 + (int64_t)(j >> 5) * tile_img16_bytes(d_pad);
    double e1 = 0.0;
    if (lane * 8 < d_pad) {
        half8 h;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int i = lane * 8 + q;
            const float b = (j < k && i < d) ? __fsub_rn(C[(int64_t)j * d + i], cp.mu[i]) : 0.0f;
            const float v = -2.0f * sc * b;
            h[q] = (_Float16)v;
            const float r = v - (float)h[q];
            e1 += (double)r * (double)r;
        }
        *reinterpret_cast<half8 *>(img + (lane >> 1) * 1024 + ((j & 31) + 32 * (lane & 1)) * 16) = h;
    }
    e1 = wave_butterfly_sum(e1);
    if (lane == 0) {
        const float *src = reinterpret_cast<const float *>(cp.img + (int64_t)(j >> 5) * tile_img_bytes(d_pad) +
                                                           128 * d_pad) + (j & 31);
        float *cst = reinterpret_cast<float *>(img + 64 * d_pad) + (j & 31);
        const float d1 = j < k ? (float)(sqrt(0.25 * e1) * ldexp(1.0, -t) * (1.0 + 1e-6)) : 0.0f;
        cst[HC_NB] = j < k ? src[FC_NB] * ldexpf(1.0f, 2 * t) : 3.0e38f;
        cst[HC_BN] = src[FC_BN];
        cst[HC_D1] = d1;
        if (j < k) atomic_max_pos(cp.mx + MX_D16, d1);
    }
}

__global__ void k_zero_i64n(int64_t *p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// ------------------------------------------------------------------
// the recheck of undecided frames
// ------------------------------------------------------------------
// Pass 1 (the MFMA kernel) appends every frame it cannot decide to `list`
// together with `upper`, a rigorous upper bound (rounded up to FP32) of the
// reference loop's distance to the frame's best candidate; NaN marks a
// frame whose distances are not finite.  Pass 2 (the MFMA kernel in
// candidate mode) recomputes the listed frames' distance bounds and records,
// per list position p < slots, every center j whose rigorous lower bound
// does not exceed upper[p] (at most CAND_MAX of them in cand[p][.], their
// number in ccnt[p]); those centers contain the reference loop's choice.
// Pass 3 runs the reference loop over the recorded candidates only; frames
// beyond the slots, with more than CAND_MAX candidates or without a finite
// bound go to `list2` and the full loop over every center.
constexpr int CAND_MAX = 8;

struct RecheckLists {
    int64_t *listA;  // [n] frames the coarse pass leaves undecided
    int64_t *list;   // [n] frames the fine pass leaves undecided
    int64_t *count;  // [N_COUNTS]: list length, unused, list2 length, listA length, the center maxima (CenterPack::mx)
    float *upper;    // [n] upper bound per list position
    int32_t *ccnt;   // [slots] candidates found per list position
    int32_t *cand;   // [slots][CAND_MAX]
    int64_t *list2;  // [n] frames for the full loop
    // consumed by k_compact before the candidate pass writes cand, whose memory they take
    uint32_t *mask;   // [n / 32] undecided positions of the pass
    float *upper_at;  // [n] their upper bounds
    int64_t slots;
};

// float >= v (v a finite double or NaN)
__device__ __forceinline__ float f32_round_up(double v) {
    float f = (float)v;
    if ((double)f < v) f = __uint_as_float(f >= 0.0f ? __float_as_uint(f) + 1u
                                                   : (__float_as_uint(f) == 0x80000000u ? 1u : __float_as_uint(f) - 1u));
    return f;
}

// ------------------------------------------------------------------
// MFMA kernel
// ------------------------------------------------------------------
// Error bounds, with u = 2^-24, gamma_n = n u / (1 - n u): a frame's and a
// center's contributions are norms of the parts their images leave out, which
// are computed exactly enough where the images are made, so the bound follows
// the data instead of the worst case of every rounding (about 2.4 times
// smaller for fp16, which lists that many fewer frames):
//   E_j = c1a |a|^2 + c1b |b_j|^2 + 2 c2 |a||b_j| + R_j,
//   coarse (a~ = fp16(2^t a) / 2^t, r = |a - a~|, the same for b):
//     R_j = 2.02 (r_a |b_j| + (|a| + r_a) r_b)
//   fine (a = hi + lo + rest; products hi hi, hi lo, lo hi):
//     R_j = 2.02 (|lo_a||lo_b| + rest_a |b_j| + (|a| + rest_a) rest_b)
//   c1a: shift rounding, combination and the element index in the 4 low
//        mantissa bits of d~ - |a|^2, (4.2 + 32) u (|a| + |b|)^2, and the FP32
//        sum of |a|^2
//   c1b: the same and the FP32 accumulation in the matrix core, which starts
//        from |b|^2
//   c2:  the same terms on 2 |a||b| and the accumulation of the products (each
//        addition rounded to nearest, as the device probe of the matrix core
//        shows)
// using (|a|+|b|)^2 = |a|^2 + |b|^2 + 2|a||b| and sum|a_i b_i| <= |a||b|.  A
// 25 % margin covers the rounding of the FP32 bound arithmetic itself.
// Below the normal numbers the roundings are absolute.  Each square, product and
// sum of the pass, the element index in a value's low bits and each term and sum
// of the reference loop is then off by at most 2^-126 (in the coarse pass of the
// scaled values), fewer than 8 d_pad of them together: E_j also has
//   e0 = 16 d_pad 2^-126 (1 + 2^-2t).
// The sums of squares behind |a|, r_a, lo_a and rest_a are FP32 too and off by at
// most 2 d_pad 2^-150 < SQ_FLOOR, which is added before each root.
constexpr double SQ_FLOOR = 0x1p-139;
struct AsgCoef {
    float c1a, c1b, c2, gref, e0;
};
static double gamma_n(double m) {
    const double u = ldexp(1.0, -24);
    return m * u / (1.0 - m * u);
}
static AsgCoef assign_coeffs(int d, int d_pad, int products) {
    const double c0 = (4.2 + 32.0) * ldexp(1.0, -24), chain = (double)products * d_pad + 2.0;
    AsgCoef c;
    c.c1a = (float)(1.25 * (c0 + gamma_n(d_pad / 8 + 8)));
    c.c1b = (float)(1.25 * (c0 + gamma_n(chain)));
    c.c2 = (float)(1.25 * (c0 + 1.02 * gamma_n(chain)));
    c.gref = (float)(1.25 * gamma_n(d + 2.0));
    c.e0 = (float)(16.0 * d_pad * ldexp(1.0, -126));
    return c;
}

// Running state of the epilogue per frame block and lane: the two smallest
// values v_j = d~_j - |a|^2 = |b_j|^2 - 2 a.b_j seen so far (m1 <= m2 as a
// multiset), each with the element e (0..15) of its 32 x 32 tile in the 4 low
// mantissa bits, and the tile of m1.  Per element: one and-or for the index,
// med3 and min for the pair (m2 = med3(m1, m2, v) is the new second smallest
// when m1 <= m2).
__device__ __forceinline__ float pack_elem(float v, int e) {
    return __uint_as_float((__float_as_uint(v) & 0xFFFFFFF0u) | (uint32_t)e);
}
// min(m1, vp) as the median of (m1, vp, -inf): v_min_f32 would first
// canonicalize the bit-built vp (one more instruction per element), and the
// compiler folds a median with a literal -inf back into that min, so the -inf
// comes from opaque_neg_inf() (an SGPR set once per kernel).
__device__ __forceinline__ float opaque_neg_inf() {
    float v = -INFINITY;
    asm volatile("" : "+s"(v));
    return v;
}
__device__ __forceinline__ void track2(float &m1, float &m2, float vp, float ninf) {
    m2 = __builtin_amdgcn_fmed3f(m1, m2, vp);
    m1 = __builtin_amdgcn_fmed3f(m1, vp, ninf);
}

// The MFMA distance kernel in its passes:
//   PASS_COARSE: every frame; one fp16 product per K-step; decides with the
//     coarse bound, lists the rest in listA.
//   PASS_FINE: the frames of listA; bf16 hi/lo of a and b, three products
//     per K-step; decides with the fine bound, lists the rest with their
//     upper bound.
//   PASS_CAND: the frames listed by PASS_FINE (positions below rl.slots);
//     the epilogue records the centers whose lower bound reaches the frame's
//     upper bound instead of tracking the minimum.
//   PASS_FULL: PASS_FINE over every frame (pass 1 without a coarse pass).
//
// A workgroup of NW waves holds the operand fragments of 32 FB frames in LDS
// (fragment order, so that an operand read is 1 KB contiguous and free of bank
// conflicts) and every wave runs all of those frames against its own center
// tiles: CT tiles at a time, tiles CT w, CT (w + NW), ...  A K-step of a wave
// is then FB LDS reads and CT fragment loads from L2 for FB CT MFMAs (three
// times as many in the fine passes), with no barrier until the frames are
// done.  The earlier form (frames in registers, every wave reading every
// center fragment from LDS for one MFMA) needed one LDS read per MFMA, the
// LDS's whole bandwidth at the matrix cores' peak, and a barrier per tile.
// The frames are read as 128 contiguous bytes of a row per 8 lanes, the rows of
// the next group in flight while one group is converted; the matrix work of
// the other workgroup on the CU covers that phase.  Measured, the first pass
// alone: 10^7 x 300, k = 1000 9.3 -> 6.6 ms (the whole call at k = 32, where the
// frames' 12 GB bound it, 7.6 -> 2.8 ms = 4.3 TB/s; 1.2 PFLOP/s per added
// center, where a large library product reaches 1.13); 10^7 x 32, k = 1000
// 8.2 -> 2.0 ms (1.6 with one wave per workgroup, see launch_pass); 2 10^6 x 512,
// k = 4096 12.6 -> 7.8 ms.
// v_mfma_f32_32x32x16: A = 32 centers x 16 dims, B = 16 dims x 32 frames; lane
// l holds frame l % 32 and centers 8(e>>2) + 4(l>>5) + (e&3).
constexpr int PASS_COARSE = 0, PASS_FINE = 1, PASS_CAND = 2, PASS_FULL = 3;

// smallest d that a kernel of KS K-steps sees (pick_ksteps takes the next size above d / 16)
constexpr int min_dim(int ks) { return (ks == 2 ? 0 : ks == 4 ? 2 : ks == 8 ? 4 : ks == 12 ? 8 : ks == 16 ? 12 : ks == 19 ? 16 : ks == 24 ? 19 : 24) * 16 + 1; }

// MASK: undecided frames as bits for k_compact, otherwise appended to the list here.
template <int KS, int FB, int CT, int NW, int PASS, bool MASK>
__global__ __launch_bounds__(NW * 64, 2) void k_assign_tile(const float *__restrict__ X, int64_t n, int d,
                                                            CenterPack cp, int k, int k_pad, AsgCoef ce,
                                                            int32_t *__restrict__ labels, RecheckLists rl,
                                                            const int32_t *__restrict__ done) {
    constexpr bool COARSE = PASS == PASS_COARSE, CAND = PASS == PASS_CAND, LISTED = CAND || PASS == PASS_FINE;
    if (done && *done) return;
    int64_t nf = n;  // frames: all, listA (fine), the candidate slots (cand)
    if constexpr (PASS == PASS_FINE) nf = rl.count[3];
    if constexpr (CAND) {
        const int64_t c = *rl.count;
        nf = c < rl.slots ? c : rl.slots;
    }
    constexpr int F = FB * 32, NT = NW * 64;
    constexpr int DP = KS * 16;
    constexpr int NPL = COARSE ? 1 : 2;  // operand planes
    constexpr int KB = NPL * 1024;       // fragment bytes of a (tile, K-step)
    constexpr int IMG = COARSE ? tile_img16_bytes(DP) : tile_img_bytes(DP);
    constexpr int MAT = KS * KB;         // fragment bytes of an image
    constexpr int FRAG = FB * KS * KB;
    constexpr int MERGE = NW * F * 12;
    __shared__ __align__(16) uint8_t s_buf[FRAG > MERGE ? FRAG : MERGE];
    __shared__ float s_na[F], s_e1[F], s_e2[COARSE ? 1 : F];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ntiles = k_pad / 32;
    const int npairs = (ntiles + CT - 1) / CT;
    const uint8_t *img = COARSE ? cp.img16 : cp.img;
    const float sc = COARSE ? cp.sc16[0] : 1.0f;
    const float ninf = opaque_neg_inf();

    // a listed pass walks its list with a resident grid, the others have a workgroup per block
    int64_t f0 = (int64_t)blockIdx.x * F;
    for (; f0 < nf; f0 = LISTED ? f0 + (int64_t)gridDim.x * F : nf) {
        // ---- frames: a = fl(x - mu) as operand fragments in LDS, |a|^2 and the norms of what they leave ----
        {
            constexpr int RPG = NT / 8, RG = F / RPG;  // rows per group of loads, groups
            constexpr int NCH = (DP + 31) / 32;                       // 16-byte chunks of a row per lane
            int sub = tid & 7;
            asm volatile("" : "+v"(sub));  // keeps the lane's offsets, masks and mu out of the matrix phase's registers
            // groups in flight: all of them where they are few and short, else the next one
            constexpr int NB = RG * NCH <= 8 ? RG : 2;
            float4_u x[NB][NCH], mu4[NCH];
            auto load_group = [&](int g, float4_u *xv) __attribute__((always_inline)) {
                int64_t pos = f0 + g * RPG + (tid >> 3);
                pos = pos < nf ? pos : nf - 1;
                int64_t fr = pos;
                if constexpr (PASS == PASS_FINE) fr = rl.listA[pos];
                if constexpr (CAND) fr = rl.list[pos];
                const float *row = X + fr * (int64_t)d;
                if (min_dim(KS) >= 4 || d >= 4) {
#pragma unroll
                    for (int i = 0; i < NCH; ++i) {
                        const int c = (i * 8 + sub) * 4;  // a chunk reaching past the row is read from the row's end
                        if (i * 32 + 32 <= min_dim(KS))
                            xv[i] = *reinterpret_cast<const float4_u *>(row + sub * 4 + i * 32);
                        else
                            xv[i] = *reinterpret_cast<const float4_u *>(row + (c + 4 <= d ? c : d - 4));
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < NCH; ++i) {
                        xv[i] = float4_u{0.0f, 0.0f, 0.0f, 0.0f};
                        xv[i].x = row[0];
                        xv[i].y = row[d > 1 ? 1 : 0];
                        xv[i].z = row[d > 2 ? 2 : 0];
                    }
                }
            };
            auto convert = [&](int g, const float4_u *xv) __attribute__((always_inline)) {
                const int r = g * RPG + (tid >> 3);
                float na = 0.0f, e1 = 0.0f, e2 = 0.0f;
                // fragment slot of row r, dims c .. c + 3, c = 32 i + 4 sub: K-step c / 16, half-wave (c / 8) & 1
                uint8_t *dst0 = s_buf + ((r >> 5) * KS + (sub >> 2)) * KB + ((sub >> 1) & 1) * 512 + (r & 31) * 16 + (sub & 1) * 8;
#pragma unroll
                for (int i = 0; i < NCH; ++i) {
                    const int c = (i * 8 + sub) * 4;
                    float v[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
                    const bool in_img = i * 32 + 32 <= DP || c < DP;
                    const float4_u m4 = mu4[i];
                    float a[4] = {__fsub_rn(v[0], m4.x), __fsub_rn(v[1], m4.y), __fsub_rn(v[2], m4.z), __fsub_rn(v[3], m4.w)};
                    if (i * 32 + 32 > min_dim(KS)) {  // the row may end inside these chunks
                        const int sh = (d >= 4 && c + 4 > d) ? c + 4 - d : 0;
                        if (sh) {
                            v[0] = sh == 1 ? v[1] : (sh == 2 ? v[2] : v[3]);
                            v[1] = sh == 1 ? v[2] : v[3];
                            v[2] = v[3];
                        }
                        const float mm[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
                        for (int q = 0; q < 4; ++q) a[q] = c + q < d ? __fsub_rn(v[q], mm[q]) : 0.0f;
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) na = fmaf(a[q], a[q], na);
                    uint8_t *dst = dst0 + i * 2 * KB;
                    if constexpr (COARSE) {
                        typedef _Float16 half4 __attribute__((ext_vector_type(4)));
                        half4 h;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const float s = __fmul_rn(a[q], sc);
                            h[q] = (_Float16)s;
                            const float rr = s - (float)h[q];
                            e1 = fmaf(rr, rr, e1);
                        }
                        if (in_img) *reinterpret_cast<half4 *>(dst) = h;
                    } else {
                        uint32_t h[2], l[2];
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            split_bf16x2(a[2 * q], a[2 * q + 1], h[q], l[q]);
                            const float l0 = __uint_as_float(l[q] << 16), l1 = __uint_as_float(l[q] & 0xffff0000u);
                            const float r0 = (a[2 * q] - __uint_as_float(h[q] << 16)) - l0;
                            const float r1 = (a[2 * q + 1] - __uint_as_float(h[q] & 0xffff0000u)) - l1;
                            e1 = fmaf(l0, l0, fmaf(l1, l1, e1));
                            e2 = fmaf(r0, r0, fmaf(r1, r1, e2));
                        }
                        if (in_img) {
                            *reinterpret_cast<uint2 *>(dst) = make_uint2(h[0], h[1]);
                            *reinterpret_cast<uint2 *>(dst + 1024) = make_uint2(l[0], l[1]);
                        }
                    }
                }
#pragma unroll
                for (int off = 1; off < 8; off <<= 1) {
                    na += __shfl_xor(na, off, 64);
                    e1 += __shfl_xor(e1, off, 64);
                    if constexpr (!COARSE) e2 += __shfl_xor(e2, off, 64);
                }
                if (sub == 0) {
                    s_na[r] = na;
                    s_e1[r] = e1;
                    if constexpr (!COARSE) s_e2[r] = e2;
                }
            };
            static_assert(F % RPG == 0 && F <= NT, "whole groups of rows; at the end a thread per frame");
            static_for<0, NB - 1>([&](auto gc) __attribute__((always_inline)) {
                load_group(decltype(gc)::value, x[decltype(gc)::value]);
            });
#pragma unroll
            for (int i = 0; i < NCH; ++i)
                mu4[i] = *reinterpret_cast<const float4_u *>(cp.mu + sub * 4 + (i * 32 + 32 <= DP || sub < 4 ? i * 32 : 0));
            static_for<0, RG>([&](auto gc) __attribute__((always_inline)) {
                constexpr int g = decltype(gc)::value;
                if constexpr (g + NB - 1 < RG) load_group(g + NB - 1, x[(g + NB - 1) % NB]);
                __builtin_amdgcn_sched_barrier(0);
                convert(g, x[g % NB]);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        __syncthreads();

        // ---- candidate pass: center j is recorded when its lower bound reaches
        // the frame's upper bound, (na + v_j - E_j)(1 - g) <= upper, as the
        // threshold v_j - c1b|b_j|^2 - ca |b_j| - cb |lo_j| - cc rest_j <= T, raised by
        // 16 u (|a| + max|b|)^2 so that rounding only ever adds candidates; no
        // threshold (NaN upper, norms near overflow, and the rows past the list, whose
        // ccnt is not set): NaN, which no value reaches (not even the -inf of an
        // overflowed product), so no candidate, and the frame goes to the full loop
        float thr[FB], ca[FB], cb[FB], cc[FB];
        if constexpr (CAND) {
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const int r = b * 32 + (lane & 31);
                thr[b] = __uint_as_float(0x7fc00000u);
                ca[b] = cb[b] = cc[b] = 0.0f;
                const float up = f0 + r < nf ? rl.upper[f0 + r] : __uint_as_float(0x7fc00000u);
                const double na = s_na[r], sa = sqrt(na + SQ_FLOOR) * (1.0 + 2e-5), mb = cp.mx[MX_BN];
                if (up == up && (sa + mb) * (sa + mb) < 1e38) {
                    const double e1 = sqrt((double)s_e1[r] + SQ_FLOOR) * (1.0 + 1e-4);
                    const double e2 = sqrt((double)s_e2[r] + SQ_FLOOR) * (1.0 + 1e-4);
                    const double T = (double)up / (1.0 - (double)ce.gref) - (na - (double)ce.c1a * sa * sa) +
                                     2.0 * (double)ce.e0 + 16.0 * 5.9604644775390625e-8 * (sa + mb) * (sa + mb);
                    thr[b] = f32_round_up(T);
                    ca[b] = (float)((2.0 * (double)ce.c2 * sa + 2.02 * e2) * 1.000001);
                    cb[b] = (float)(2.02 * e1 * 1.000001);
                    cc[b] = (float)(2.02 * (sa + e2) * 1.000001);
                }
            }
        }

        float m1[FB], m2[FB];
        int mt[FB];
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            m1[b] = m2[b] = INFINITY;
            mt[b] = -1;
        }

        // ---- the wave's center tiles ----
        constexpr int PF = KS < 4 ? KS : (COARSE ? 4 : 3);  // K-steps of center fragments in flight
        uint4 cf[PF][CT][NPL];
        float init[CT][16];
        const uint8_t *tp[CT];  // images of the wave's current tiles
        uint32_t vo = 0;        // the lane's offset of the next K-step to load
        auto load_cf = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int pl = 0; pl < NPL; ++pl)
                    cf[slot][ct][pl] = *reinterpret_cast<const uint4 *>(tp[ct] + vo + pl * 1024);
            vo += KB;
            asm volatile("" : "+v"(vo));  // one running offset, not an address per K-step
        };
        // start of a tile pair: its first fragments and the accumulators' start values
        auto start_pair = [&](int pr) __attribute__((always_inline)) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const int t = pr * CT + ct;
                tp[ct] = img + (int64_t)(t < ntiles ? t : ntiles - 1) * IMG;
                const float *cst = reinterpret_cast<const float *>(tp[ct] + MAT) + (CAND ? FC_Q : (COARSE ? HC_NB : FC_NB));
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float4 q4 = *reinterpret_cast<const float4 *>(cst + 8 * g + 4 * (lane >> 5));
                    init[ct][4 * g + 0] = q4.x;
                    init[ct][4 * g + 1] = q4.y;
                    init[ct][4 * g + 2] = q4.z;
                    init[ct][4 * g + 3] = q4.w;
                }
                if (CT > 1 && pr * CT + ct >= ntiles)  // no such tile: a repeat of the last one that never wins
#pragma unroll
                    for (int e = 0; e < 16; ++e) init[ct][e] = 3.0e38f;
            }
            vo = (uint32_t)lane * 16u;
            asm volatile("" : "+v"(vo));
#pragma unroll
            for (int s = 0; s < PF; ++s) load_cf(s);
        };
        const uint8_t *fb_base = s_buf + lane * 16;
        uint4 ff[2][FB][NPL];
        auto load_ff = [&](int s, int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < FB; ++b)
#pragma unroll
                for (int pl = 0; pl < NPL; ++pl)
                    ff[slot][b][pl] = *reinterpret_cast<const uint4 *>(fb_base + (b * KS + s) * KB + pl * 1024);
        };
        if (wave < npairs) start_pair(wave);
        for (int pr = wave; pr < npairs; pr += NW) {
            floatx16 acc[CT][FB];
            load_ff(0, 0);
            static_for<0, KS>([&](auto sc_) __attribute__((always_inline)) {
                constexpr int s = decltype(sc_)::value;
                if constexpr (s + 1 < KS) load_ff(s + 1, (s + 1) & 1);
                constexpr int sl = s % PF, fs = s & 1;
                // the product order of every accumulator: hi lo, lo hi, hi hi
#pragma unroll
                for (int pp = 0; pp < (COARSE ? 1 : 3); ++pp)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                        for (int b = 0; b < FB; ++b) {
                            floatx16 c0;
                            if constexpr (s == 0) {
                                if (pp == 0) {
#pragma unroll
                                    for (int e = 0; e < 16; ++e) c0[e] = init[ct][e];
                                } else {
                                    c0 = acc[ct][b];
                                }
                            } else {
                                c0 = acc[ct][b];
                            }
                            if constexpr (COARSE)
                                acc[ct][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                    __builtin_bit_cast(half8, cf[sl][ct][0]), __builtin_bit_cast(half8, ff[fs][b][0]), c0, 0, 0, 0);
                            else
                                acc[ct][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                    __builtin_bit_cast(bf16x8, cf[sl][ct][pp == 1 ? NPL - 1 : 0]),
                                    __builtin_bit_cast(bf16x8, ff[fs][b][pp == 0 ? NPL - 1 : 0]), c0, 0, 0, 0);
                        }
                if constexpr (s + PF < KS) load_cf(sl);
                // the next step's LDS reads first, then this step's MFMAs with the L2 loads behind them
                if constexpr (s + 1 < KS) __builtin_amdgcn_sched_group_barrier(0x100, FB * NPL, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, (COARSE ? 1 : 3) * CT * FB, 0);
                if constexpr (s + PF < KS) __builtin_amdgcn_sched_group_barrier(0x020, CT * NPL, 0);
                __builtin_amdgcn_sched_barrier(0);
            });
            if (pr + NW < npairs) start_pair(pr + NW);  // in flight during the epilogue below
            if constexpr (CAND) {
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    const int t = pr * CT + ct;
                    if (t >= ntiles) break;
                    const float *cst = reinterpret_cast<const float *>(img + (int64_t)t * IMG + MAT);
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int c0 = 8 * g + 4 * (lane >> 5);
                        const float4 bnv = *reinterpret_cast<const float4 *>(cst + FC_BN + c0);
                        const float4 d1v = *reinterpret_cast<const float4 *>(cst + FC_D1 + c0);
                        const float4 d2v = *reinterpret_cast<const float4 *>(cst + FC_D2 + c0);
                        const float bn[4] = {bnv.x, bnv.y, bnv.z, bnv.w}, d1[4] = {d1v.x, d1v.y, d1v.z, d1v.w};
                        const float d2[4] = {d2v.x, d2v.y, d2v.z, d2v.w};
#pragma unroll
                        for (int b = 0; b < FB; ++b)
#pragma unroll
                            for (int h = 0; h < 4; ++h) {
                                const float lb = fmaf(-cc[b], d2[h], fmaf(-cb[b], d1[h], fmaf(-ca[b], bn[h], acc[ct][b][4 * g + h])));
                                const int j = t * 32 + c0 + h;
                                if (lb <= thr[b] && j < k) {
                                    const int64_t pos = f0 + b * 32 + (lane & 31);
                                    const int q = atomicAdd(&rl.ccnt[pos], 1);
                                    if (q < CAND_MAX) rl.cand[pos * CAND_MAX + q] = j;
                                }
                            }
                    }
                }
            } else {
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    const int t = pr * CT + ct;
#pragma unroll
                    for (int b = 0; b < FB; ++b) {
                        const float prev = m1[b];
#pragma unroll
                        for (int e = 0; e < 16; ++e) track2(m1[b], m2[b], pack_elem(acc[ct][b][e], e), ninf);
                        mt[b] = m1[b] != prev ? t : mt[b];
                    }
                }
            }
        }
        __syncthreads();  // the fragments are consumed: their LDS takes the merge below (or the next frames)
        if constexpr (CAND) continue;

        // ---- merge the half-waves (the same frames, other centers) and the waves ----
        float *s_m1 = reinterpret_cast<float *>(s_buf), *s_m2 = s_m1 + NW * F;
        int *s_ix = reinterpret_cast<int *>(s_m2 + NW * F);
        auto merge = [&](float &a1, float &a2, int &ai, float o1, float o2, int oi) __attribute__((always_inline)) {
            a2 = fminf(fminf(a2, o2), fmaxf(a1, o1));
            if (o1 < a1 || (o1 == a1 && oi < ai)) {
                a1 = o1;
                ai = oi;
            }
        };
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            const int e = (int)(__float_as_uint(m1[b]) & 15u);
            int ix = mt[b] >= 0 ? mt[b] * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3) : 0x7fffffff;
            const float o1 = __shfl_xor(m1[b], 32, 64), o2 = __shfl_xor(m2[b], 32, 64);
            const int oi = __shfl_xor(ix, 32, 64);
            merge(m1[b], m2[b], ix, o1, o2, oi);
            if (lane < 32) {
                s_m1[wave * F + b * 32 + lane] = m1[b];
                s_m2[wave * F + b * 32 + lane] = m2[b];
                s_ix[wave * F + b * 32 + lane] = ix;
            }
        }
        __syncthreads();
        // ---- one thread per frame: its label, and whether it goes to the next
        // pass.  d_j >= |a|^2 + m2 - E_max for j != best, with E_max from the
        // largest norms of all centers, and d_best <= |a|^2 + m1 + E_best (both
        // through the reference loop's relative rounding g).  Anything not
        // finite (frames, centers, fp16 overflow) fails the comparison, except a
        // center whose |b|^2 overflows: its v is +inf, or no number once it holds an
        // element index, and from the latter m1 is -inf and m2 may be lost.  So a
        // frame is decided only where no v, partial sums included, can overflow:
        // all are below (|a| + max|b|)^2.
        if (tid < F) {
            float b1 = s_m1[tid], b2 = s_m2[tid];
            int ix = s_ix[tid];
#pragma unroll
            for (int w = 1; w < NW; ++w) merge(b1, b2, ix, s_m1[w * F + tid], s_m2[w * F + tid], s_ix[w * F + tid]);
            const int64_t pos = f0 + tid;
            const bool fvalid = pos < nf;
            bool undecided = false;
            float up = __uint_as_float(0x7fc00000u);
            int64_t fr = pos;
            if constexpr (PASS == PASS_FINE) fr = fvalid ? rl.listA[pos] : 0;
            if (fvalid) {
                undecided = true;
                int lab = 0;
                if (ix < k && fabsf(b1) < 1e38f) {
                    lab = ix;
                    const float *cst = reinterpret_cast<const float *>(img + (int64_t)(ix >> 5) * IMG + MAT) + (ix & 31);
                    const double un = COARSE ? (double)cp.sc16[1] : 1.0;  // the coarse pass's values carry 2^2t
                    const double na = s_na[tid], sa = sqrt(na + SQ_FLOOR) * (1.0 + 2e-5);
                    const double e1 = sqrt((double)s_e1[tid] + SQ_FLOOR) * (1.0 + 1e-4) * (COARSE ? (double)cp.sc16[2] : 1.0);
                    const double bb = cst[COARSE ? HC_BN : FC_BN], bd = cst[COARSE ? HC_D1 : FC_D1];
                    const double mb = cp.mx[MX_BN], md = cp.mx[COARSE ? MX_D16 : MX_D1];
                    double Rb, Rm;
                    if constexpr (COARSE) {
                        Rb = e1 * bb + (sa + e1) * bd;
                        Rm = e1 * mb + (sa + e1) * md;
                    } else {
                        const double e2 = sqrt((double)s_e2[tid] + SQ_FLOOR) * (1.0 + 1e-4);
                        Rb = e1 * bd + e2 * bb + (sa + e2) * (double)cst[FC_D2];
                        Rm = e1 * md + e2 * mb + (sa + e2) * (double)cp.mx[MX_D2];
                    }
                    const double aa = (double)ce.c1a * sa * sa + (double)ce.e0 * (1.0 + un);
                    const double Eb = aa + (double)ce.c1b * bb * bb + 2.0 * (double)ce.c2 * sa * bb + 2.02 * Rb;
                    const double Em = aa + (double)ce.c1b * mb * mb + 2.0 * (double)ce.c2 * sa * mb + 2.02 * Rm;
                    const double upper = (na + un * (double)b1 + Eb) * (1.0 + (double)ce.gref);
                    const double lower = (na + un * (double)b2 - Em) * (1.0 - (double)ce.gref);
                    undecided = !(lower > upper && (sa + mb) * (sa + mb) < 1e38);
                    if (fabs(upper) < 3e38) up = f32_round_up(upper);
                }
                labels[fr] = lab;
            }
            const unsigned long long um = __ballot(undecided);
            if constexpr (!MASK) {
                // few frames: appended here, one list reservation per wave
                if (um) {
                    const int leader = __builtin_ctzll(um);
                    unsigned long long base = 0;
                    if (lane == leader)
                        base = atomicAdd((unsigned long long *)(rl.count + (COARSE ? 3 : 0)), (unsigned long long)__popcll(um));
                    base = __shfl(base, leader, 64);
                    if (undecided) {
                        const int64_t q = (int64_t)base + __popcll(um & ((1ull << lane) - 1ull));
                        if constexpr (COARSE) {
                            rl.listA[q] = fr;
                        } else {
                            rl.list[q] = fr;
                            rl.upper[q] = up;
                            rl.ccnt[q] = 0;
                        }
                    }
                }
            } else {
                // otherwise one bit per position, made into the list by k_compact:
                // the waves' reservations would all go to one address, about 29 ns
                // each (10^7 frames x 32, k = 1000: 4.6 ms of reservations around
                // 1.6 ms of work)
                if (undecided && !COARSE) rl.upper_at[pos] = up;
                if (lane == 0) rl.mask[pos >> 5] = (uint32_t)um;
                if (lane == 32) rl.mask[pos >> 5] = (uint32_t)(um >> 32);
            }
        }
        __syncthreads();  // the merge buffers and norms are consumed before the next frames overwrite them
    }
}

static int pick_ksteps(int d) {
    const int ks = (int)cdiv(d, 16);
    static const int sizes[] = {2, 4, 8, 12, 16, 19, 24, 32};
    for (int s : sizes)
        if (ks <= s) return s;
    return -1;
}

struct AssignWs {
    CenterPack cp;
    RecheckLists rl;
    size_t bytes;
};

// candidate slots: one per frame that can be listed (near-tie-heavy center
// sets, such as the cluster means after a Lloyd update with many centers per
// mode of the data, list about half of the frames)
static int64_t cand_slots(int64_t n) { return n > 0 ? n : 1; }

static AssignWs carve_assign(void *ws, int64_t n, int d, int k, int mode) {
    AssignWs w{};
    Carver cv(ws);
    const size_t nl = n > 0 ? (size_t)n : 1;
    w.rl.count = cv.take<int64_t>(N_COUNTS);
    w.rl.list = cv.take<int64_t>(nl);
    w.cp.mx = w.rl.count ? reinterpret_cast<float *>(w.rl.count + 4) : nullptr;
    if (mode == EMMA_ASSIGN_BF16X3_RECHECK) {
        w.rl.slots = cand_slots(n);
        w.rl.upper = cv.take<float>(nl);
        w.rl.ccnt = cv.take<int32_t>((size_t)w.rl.slots);
        w.rl.cand = cv.take<int32_t>((size_t)w.rl.slots * CAND_MAX);
        w.rl.upper_at = reinterpret_cast<float *>(w.rl.cand);
        w.rl.mask = w.rl.cand ? reinterpret_cast<uint32_t *>(w.rl.cand) + nl : nullptr;
        // listA is consumed by the fine pass before the candidate recheck
        // writes list2: one buffer serves both
        w.rl.listA = cv.take<int64_t>(nl);
        w.rl.list2 = w.rl.listA;
        const int ks = pick_ksteps(d);
        const int d_pad = (ks > 0 ? ks : 1) * 16;
        const int k_pad = (int)cdiv(k, 32) * 32;
        w.cp.img = cv.take<uint8_t>((size_t)(k_pad / 32) * tile_img_bytes(d_pad));
        w.cp.img16 = cv.take<uint8_t>((size_t)(k_pad / 32) * tile_img16_bytes(d_pad));
        (void)cv.take<float>(k_pad);  // unused: keeps the sizes, and with them what emma_assign_noalloc accepts
        w.cp.mu = cv.take<float>(d_pad);
        w.cp.sc16 = cv.take<float>(4);
    }
    w.bytes = cv.bytes();
    return w;
}

// Pass 3 of the recheck: the reference loop over the recorded candidates.
// CAND_MAX consecutive threads serve one list position (thread c: candidate
// c); the smallest distance wins, the smallest center index among equal
// ones (the reference's first minimum: the candidates contain every center
// the loop could choose, see RecheckLists).  Positions without usable
// candidates go to list2.  VEC: rows read as 16-byte vectors (d % 4 == 0,
// aligned X and C).
template <bool VEC>
__global__ __launch_bounds__(256) void k_assign_cand_exact(const float *__restrict__ X, int d,
                                                           const float *__restrict__ C, int32_t *__restrict__ labels,
                                                           RecheckLists rl, const int32_t *__restrict__ done) {
    if (done && *done) return;
    const int64_t total = *rl.count * CAND_MAX;  // whole groups enter each iteration (the stride is a multiple)
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
        const int64_t pos = idx / CAND_MAX;
        const int c = (int)(idx % CAND_MAX);
        const int64_t fr = rl.list[pos];
        int nc = -1;  // -1: the full loop
        if (pos < rl.slots) {
            const int cc = rl.ccnt[pos];
            if (cc >= 1 && cc <= CAND_MAX) nc = cc;
        }
        float dist = INFINITY;
        int j = 0x7fffffff;
        if (c < nc) {
            j = rl.cand[pos * CAND_MAX + c];
            const float *x = X + fr * (int64_t)d;
            const float *cr = C + (int64_t)j * d;
            float acc = 0.0f;
            if (VEC) {
                for (int i = 0; i < d; i += 4) {
                    const float4 xv = *reinterpret_cast<const float4 *>(x + i);
                    const float4 cv = *reinterpret_cast<const float4 *>(cr + i);
                    acc = sq_step(acc, xv.x, cv.x);
                    acc = sq_step(acc, xv.y, cv.y);
                    acc = sq_step(acc, xv.z, cv.z);
                    acc = sq_step(acc, xv.w, cv.w);
                }
            } else {
                for (int i = 0; i < d; ++i) acc = sq_step(acc, x[i], cr[i]);
            }
            dist = acc;
        }
#pragma unroll
        for (int off = 1; off < CAND_MAX; off <<= 1) {
            const float od = __shfl_xor(dist, off, 64);
            const int oj = __shfl_xor(j, off, 64);
            if (od < dist || (od == dist && oj < j)) {
                dist = od;
                j = oj;
            }
        }
        if (c == 0) {
            if (nc < 0) {
                const unsigned long long p2 = atomicAdd((unsigned long long *)(rl.count + 2), 1ull);
                rl.list2[p2] = fr;
            } else {
                labels[fr] = j;
            }
        }
    }
}

// First-pass pipelines, timed by the autotuner (emma_assign_select may pick one
// per (K steps, k) bucket): the lower half of the variant numbers is the coarse
// pass over every frame with the fine pass on what it leaves; the upper half the
// fine pass over every frame.  Which is faster depends on d, k and the data: the
// coarse pass costs a third of the fine one's products, so on many frames it
// loses only where its bound leaves about two thirds of them or more.  Without a
// selection few_frames() decides.
// Each pipeline has one tile shape; the count of numbers per dimension is part of
// the C ABI, so that selections kept by a caller stay valid.
static int n_variants(int ks) { return ks <= 4 ? 12 : ks <= 8 ? 6 : ks <= 19 ? 4 : 2; }

// process-wide selection table: [K-step class][ceil(log2(k_pad / 32))]
static std::mutex g_sel_mu;
static int g_sel[8][16];
static bool g_sel_init = false;

static int ks_index(int ks) {
    static const int sizes[] = {2, 4, 8, 12, 16, 19, 24, 32};
    for (int i = 0; i < 8; ++i)
        if (sizes[i] == ks) return i;
    return -1;
}
static int k_bucket(int k_pad) {
    int b = 0;
    while ((32 << b) < k_pad && b < 15) ++b;
    return b;
}
// -1: none
static int selected_variant(int ks, int k_pad) {
    std::lock_guard<std::mutex> lk(g_sel_mu);
    if (!g_sel_init) return -1;
    const int v = g_sel[ks_index(ks)][k_bucket(k_pad)];
    return v < n_variants(ks) ? v : -1;
}
// Calls bound by their launches and by the latency of a workgroup rather than by
// products: the fine pass over every frame needs three launches less (the coarse
// images, pass and list).  Whole calls, us, coarse and fine first pass:
//   frames   d, k     coarse  fine      frames   d, k      coarse  fine
//   33,000   10, 64       54    44      200,000  32, 1000     152   149
//   66,000   32, 1000    129   116      200,000  100, 500     133   151
//   200,000  10, 10       59    49      400,000  100, 10      107   119
// Above 19 K-steps the fine pass has one workgroup per CU (200,000 x 350, k = 10: 227, 248).
static bool few_frames(int64_t n, int ks, int k_pad) {
    return ks < 24 && n * ks * 16 <= 30'000'000 && n * ks * 16 <= 5'000'000'000 / k_pad;
}

static int device_cus() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    return cus;
}

// List of a pass's undecided positions from its bit mask.  A workgroup takes
// 256 Q words (8192 Q positions) at a time, reserves their list range with one
// atomic, writes the positions of the set bits to LDS and copies the entries from
// there, a thread each: a thread that walked the bits of its words itself would
// wait for the loads of every entry in turn (one workgroup for 32,000 frames took
// 18 us).  FINE: the positions are those of listA (or frames, LISTED = false) and
// go to `list` with their upper bounds; otherwise frames to listA.
template <bool FINE, bool LISTED, int Q>
__global__ __launch_bounds__(256) void k_compact(int64_t n, RecheckLists rl, const int32_t *__restrict__ done) {
    if (done && *done) return;
    constexpr int WORDS = 256 * Q;
    static_assert(WORDS * 32 <= 65536, "a position in a chunk fits 16 bits");
    __shared__ uint16_t s_pos[WORDS * 32];
    __shared__ uint32_t s_wave[4];
    __shared__ unsigned long long s_base;
    const int64_t np = LISTED ? rl.count[3] : n;
    const int64_t words = (np + 31) >> 5;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int64_t w0 = (int64_t)blockIdx.x * WORDS; w0 < words; w0 += (int64_t)gridDim.x * WORDS) {
        uint32_t m[Q];
        uint32_t cnt = 0;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int64_t w = w0 + tid * Q + q;
            m[q] = w < words ? rl.mask[w] : 0u;
            cnt += __popc(m[q]);
        }
        uint32_t pre = cnt;  // inclusive scan over the wave
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = __shfl_up(pre, off, 64);
            if (lane >= off) pre += o;
        }
        if (lane == 63) s_wave[wave] = pre;
        __syncthreads();
        const uint32_t tot = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
        if (tid == 0)
            s_base = tot ? atomicAdd((unsigned long long *)(rl.count + (FINE ? 0 : 3)), (unsigned long long)tot) : 0ull;
        uint32_t at = pre - cnt;
        for (int w = 0; w < wave; ++w) at += s_wave[w];
#pragma unroll
        for (int q = 0; q < Q; ++q)
            for (uint32_t b = m[q]; b; b &= b - 1) s_pos[at++] = (uint16_t)((tid * Q + q) * 32 + __builtin_ctz(b));
        __syncthreads();
        const int64_t q0 = (int64_t)s_base;
        for (uint32_t e = tid; e < tot; e += 256) {
            const int64_t pos = w0 * 32 + s_pos[e];
            if constexpr (FINE) {
                rl.list[q0 + e] = LISTED ? rl.listA[pos] : pos;
                rl.upper[q0 + e] = rl.upper_at[pos];
                rl.ccnt[q0 + e] = 0;
            } else {
                rl.listA[q0 + e] = pos;
            }
        }
        __syncthreads();  // the shared values are consumed
    }
}

struct TileArgs {
    const float *X;
    int64_t n;
    int d, k, k_pad;
    int32_t *labels;
    const int32_t *done;
    int cus;
    bool coarse;
    hipStream_t s;
};

template <int KS, int FB, int CT, int NW, int PASS, bool MASK>
static void launch_tile(const TileArgs &a, const AssignWs &w, const AsgCoef &ce) {
    int64_t blocks = cdiv(PASS == PASS_CAND ? w.rl.slots : a.n, 32 * FB);
    // a listed pass does not know its list's length here: a resident grid walks it
    const int64_t cap = (int64_t)a.cus * (NW == 4 ? 2 : 1);
    if ((PASS == PASS_FINE || PASS == PASS_CAND) && blocks > cap) blocks = cap;
    k_assign_tile<KS, FB, CT, NW, PASS, MASK><<<(unsigned)blocks, NW * 64, 0, a.s>>>(a.X, a.n, a.d, w.cp, a.k, a.k_pad,
                                                                                     ce, a.labels, w.rl, a.done);
}

// Small chunks while there are few of them, so that more workgroups share the work (d = 32,
// k = 500, whole call: 33,000 frames 83 us in chunks of 32768, 81 of 8192; 10^7 frames, k = 200:
// 557 and 573 us, a reservation per chunk on one address)
template <int PASS>
static void launch_compact(const TileArgs &a, const AssignWs &w) {
    constexpr bool FINE = PASS != PASS_COARSE, LISTED = PASS == PASS_FINE;
    const int q = a.n < ((int64_t)1 << 20) ? 1 : 4;
    const int64_t chunks = cdiv(a.n, 8192 * q);
    const unsigned g = (unsigned)(chunks < 512 ? chunks : 512);
    if (q == 1)
        k_compact<FINE, LISTED, 1><<<g, 256, 0, a.s>>>(a.n, w.rl, a.done);
    else
        k_compact<FINE, LISTED, 4><<<g, 256, 0, a.s>>>(a.n, w.rl, a.done);
}

// Tile shape of a pass: 128 (coarse) or 64 frames per workgroup, two center
// tiles per wave step; two 4-wave workgroups per CU while the fragments of
// both fit in LDS (d <= 304), one of 8 waves beyond.  Few frames (less than
// one such workgroup per CU) are cut into workgroups of 32 (either side of that
// line, 4096 centers: d = 64 405 and 380 us, d = 512 728 and 754).
// d <= 64 and up to 1024 centers, passes over every frame: a workgroup is one
// wave with 64 frames.  Such a workgroup's time is a chain of latencies (rows,
// LDS, center fragments, the decision), in which the waves of a larger one
// wait for each other, and with fewer tiles than they take some have no
// centers.  Whole calls, 2 10^6 frames, us, coarse pass, four waves and one:
// d = 2, k = 10 205 and 91; d = 32, k = 64 237 and 126; d = 32, k = 1000 460 and 406;
// k = 2000 744 and 717; k = 4096 1343 and 1361; 200,000 x 10, k = 10, fine pass 49 and 40.
// d > 384 and up to 512 centers, coarse pass over every frame: four workgroups
// of 32 frames per CU instead of one of 128, so that frames are read while
// others are at their products.  1.9 10^6 x 512, whole call, us: k = 10 1883 and
// 1051, k = 256 1963 and 1408, k = 500 2246 and 2061, k = 1000 3036 and 3512.
template <int KS, int PASS>
static void launch_pass(const TileArgs &a, const AssignWs &w, const AsgCoef &ce) {
    constexpr int FB = PASS == PASS_COARSE ? 4 : 2, NW = KS <= 19 ? 4 : 8;
    constexpr bool EVERY = PASS == PASS_COARSE || PASS == PASS_FULL, MASK = PASS != PASS_CAND;
    if (cdiv(a.n, 32 * FB) < a.cus) {
        launch_tile<KS, 1, 1, 4, PASS, false>(a, w, ce);
        return;
    }
    bool small = false;
    if constexpr (EVERY && KS <= 4) {
        small = a.n >= (int64_t)256 * a.cus && a.k_pad <= 1024;
        if (small) launch_tile<KS, 2, 1, 1, PASS, true>(a, w, ce);
    }
    if constexpr (PASS == PASS_COARSE && KS == 32) {
        small = a.k_pad <= 512;
        if (small) launch_tile<KS, 1, 1, 4, PASS, true>(a, w, ce);
    }
    if (!small) launch_tile<KS, FB, 2, NW, PASS, MASK>(a, w, ce);
    if (MASK) launch_compact<PASS>(a, w);
}

template <int KS>
static void launch_mfma_ks(const TileArgs &a, const AssignWs &w, const AsgCoef &ce, const AsgCoef &ce16) {
    if (a.coarse) {
        launch_pass<KS, PASS_COARSE>(a, w, ce16);
        launch_pass<KS, PASS_FINE>(a, w, ce);
    } else {
        launch_pass<KS, PASS_FULL>(a, w, ce);
    }
    launch_pass<KS, PASS_CAND>(a, w, ce);
}

}  // namespace asg

// shared with kmeans.hip (Lloyd); n_call: frames of the whole call that these n belong to, so that
// every chunk of a call takes the same passes
size_t assign_workspace_bytes(int64_t n, int d, int k, int mode) { return asg::carve_assign(nullptr, n, d, k, mode).bytes; }

int assign_run(const float *X, int64_t n, int d, const float *C, int k, int32_t *labels, int mode,
               int64_t *n_rechecked, int64_t *n_looped, void *workspace, const int32_t *done, hipStream_t s,
               int64_t n_call) {
    using namespace asg;
    AssignWs w = carve_assign(workspace, n, d, k, mode);
    if (mode == EMMA_ASSIGN_FP32_PLAIN) {
        k_assign_plain<<<(unsigned)cdiv(n, PF), 256, 0, s>>>(X, n, d, C, k, labels, nullptr, nullptr, n_rechecked,
                                                             nullptr, n_looped, done);
        return check_launch("assign plain");
    }
    const int ks = pick_ksteps(d);
    EMMA_REQUIRE(ks > 0, "emma_assign: d=%d exceeds the MFMA path limit (512)", d);
    const int d_pad = ks * 16;
    const int k_pad = (int)cdiv(k, 32) * 32;
    const AsgCoef ce = assign_coeffs(d, d_pad, 3), ce16 = assign_coeffs(d, d_pad, 1);
    k_center_mean<<<(unsigned)cdiv(d_pad, 64), 64 * MU_WAVES, 0, s>>>(C, k, d, d_pad, w.cp.mu, w.rl.count);
    k_center_pack<<<(unsigned)cdiv(k_pad, 4), 256, 0, s>>>(C, k, d, d_pad, k_pad, ce.c1b, w.cp);
    const int v = selected_variant(ks, k_pad);
    const bool coarse = v < 0 ? !few_frames(n_call, ks, k_pad) : v < n_variants(ks) / 2;
    if (coarse) k_center_pack16<<<(unsigned)cdiv(k_pad, 4), 256, 0, s>>>(C, k, d, d_pad, k_pad, w.cp);
    EMMA_TRY(check_launch("assign center pack"));
    // the first pass over every frame, then the passes over what it leaves: the
    // fine pass, the candidates of the frames that one leaves, the reference
    // loop over them, the full loop over every center for the rest
    const TileArgs a = {X, n, d, k, k_pad, labels, done, device_cus(), coarse, s};
    switch (ks) {
        case 2: launch_mfma_ks<2>(a, w, ce, ce16); break;
        case 4: launch_mfma_ks<4>(a, w, ce, ce16); break;
        case 8: launch_mfma_ks<8>(a, w, ce, ce16); break;
        case 12: launch_mfma_ks<12>(a, w, ce, ce16); break;
        case 16: launch_mfma_ks<16>(a, w, ce, ce16); break;
        case 19: launch_mfma_ks<19>(a, w, ce, ce16); break;
        case 24: launch_mfma_ks<24>(a, w, ce, ce16); break;
        case 32: launch_mfma_ks<32>(a, w, ce, ce16); break;
    }
    EMMA_TRY(check_launch("assign candidates"));
    const int64_t eb = cdiv(n * CAND_MAX, 256) < 4096 ? cdiv(n * CAND_MAX, 256) : 4096;
    const bool vec = d % 4 == 0 && (((uintptr_t)X | (uintptr_t)C) & 15) == 0;
    if (vec)
        k_assign_cand_exact<true><<<(unsigned)eb, 256, 0, s>>>(X, d, C, labels, w.rl, done);
    else
        k_assign_cand_exact<false><<<(unsigned)eb, 256, 0, s>>>(X, d, C, labels, w.rl, done);
    EMMA_TRY(check_launch("assign candidate recheck"));
    const int64_t rb = cdiv(n, PF) < 1024 ? cdiv(n, PF) : 1024;
    k_assign_plain<<<(unsigned)rb, 256, 0, s>>>(X, n, d, C, k, labels, w.rl.list2, w.rl.count + 2, n_rechecked,
                                                w.rl.count, n_looped, done);
    return check_launch("assign recheck");
}

}  // namespace emma

using namespace emma;

extern "C" size_t emma_assign_workspace_size(int64_t n, int32_t d, int32_t k, int32_t mode) {
    if (n < 0 || d <= 0 || k <= 0) return 0;
    return assign_workspace_bytes(n, d, k, mode);
}

extern "C" int emma_assign(const float *X, int64_t n, int32_t d, const float *C, int32_t k, int32_t *labels,
                           int32_t mode, int64_t *n_rechecked, void *workspace, size_t workspace_bytes,
                           void *stream) {
    return emma_assign_counted(X, n, d, C, k, labels, mode, n_rechecked, nullptr, workspace, workspace_bytes, stream);
}

extern "C" int emma_assign_counted(const float *X, int64_t n, int32_t d, const float *C, int32_t k, int32_t *labels,
                                   int32_t mode, int64_t *n_rechecked, int64_t *n_looped, void *workspace,
                                   size_t workspace_bytes, void *stream) {
    EMMA_REQUIRE(n >= 0 && d > 0 && k > 0, "emma_assign: bad sizes n=%lld d=%d k=%d", (long long)n, d, k);
    EMMA_REQUIRE(mode == EMMA_ASSIGN_FP32_PLAIN || mode == EMMA_ASSIGN_BF16X3_RECHECK,
                 "emma_assign: unknown mode %d", mode);
    if (n == 0) {
        for (int64_t *p : {n_rechecked, n_looped})
            if (p) {
                asg::k_zero_i64n<<<1, 64, 0, (hipStream_t)stream>>>(p, 1);
                EMMA_TRY(check_launch("emma_assign"));
            }
        return EMMA_OK;
    }
    EMMA_REQUIRE(X && C && labels, "emma_assign: NULL pointer");
    const size_t need = assign_workspace_bytes(n, d, k, mode);
    EMMA_REQUIRE(workspace && workspace_bytes >= need, "emma_assign: workspace too small (%zu < %zu)",
                 workspace_bytes, need);
    return assign_run(X, n, d, C, k, labels, mode, n_rechecked, n_looped, workspace, nullptr, (hipStream_t)stream, n);
}

extern "C" int32_t emma_assign_variants(int32_t d) {
    const int ks = asg::pick_ksteps(d);
    return ks > 0 ? asg::n_variants(ks) : 0;
}

extern "C" int emma_assign_select(int32_t d, int32_t k, int32_t variant) {
    using namespace asg;
    EMMA_REQUIRE(d > 0 && k > 0, "emma_assign_select: bad sizes d=%d k=%d", d, k);
    const int ks = pick_ksteps(d);
    EMMA_REQUIRE(ks > 0, "emma_assign_select: d=%d exceeds the MFMA path limit (512)", d);
    EMMA_REQUIRE(variant < n_variants(ks), "emma_assign_select: variant %d of %d", variant, n_variants(ks));
    std::lock_guard<std::mutex> lk(g_sel_mu);
    if (!g_sel_init) {
        for (auto &row : g_sel)
            for (int &v : row) v = -1;
        g_sel_init = true;
    }
    g_sel[ks_index(ks)][k_bucket((int)cdiv(k, 32) * 32)] = variant < 0 ? -1 : variant;
    return EMMA_OK;
}

// ------------------------------------------------------------------
// allocation-free assignment: the workspace of emma_assign carved from a
// file-scope device array instead of a caller buffer
// ------------------------------------------------------------------
namespace emma {
namespace asg {

// Every GPU the library runs on holds its own copy of this array until the
// process ends; host code reaches it only through the address that
// hipGetSymbolAddress returns on that device (the array's name on the host
// is not a device address).
static __device__ __align__(256) uint8_t scratch[EMMA_ASSIGN_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device, resolved once per
// device (with that device current) and kept.
static int scratch_on_current_device(void **out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        set_error("emma_assign_noalloc: hipGetDevice: %s", hipGetErrorString(e));
        return EMMA_ERR_HIP;
    }
    EMMA_REQUIRE(dev >= 0 && dev < kMaxDevices, "emma_assign_noalloc: device %d beyond %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error("emma_assign_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", dev,
                      hipGetErrorString(e));
            return EMMA_ERR_HIP;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return EMMA_OK;
}

}  // namespace asg
}  // namespace emma

extern "C" int emma_assign_noalloc(const float *X, int64_t n, int32_t d, const float *C, int32_t k,
                                   int32_t *labels, int32_t mode, int64_t *n_rechecked, void *stream) {
    using namespace emma::asg;
    EMMA_REQUIRE(n >= 0 && d > 0 && k > 0, "emma_assign_noalloc: bad sizes n=%lld d=%d k=%d", (long long)n, d, k);
    EMMA_REQUIRE(mode == EMMA_ASSIGN_FP32_PLAIN || mode == EMMA_ASSIGN_BF16X3_RECHECK,
                 "emma_assign_noalloc: unknown mode %d", mode);
    hipStream_t s = (hipStream_t)stream;
    if (n == 0) {
        if (!n_rechecked) return EMMA_OK;
        k_zero_i64n<<<1, 64, 0, s>>>(n_rechecked, 1);
        return check_launch("emma_assign_noalloc");
    }
    EMMA_REQUIRE(X && C && labels, "emma_assign_noalloc: NULL pointer");
    if (mode == EMMA_ASSIGN_FP32_PLAIN)  // the plain loop needs no workspace
        return assign_run(X, n, d, C, k, labels, mode, n_rechecked, nullptr, nullptr, nullptr, s, n);
    // the center images and constants take a fixed part of the scratch; the
    // recheck arrays (56 bytes per frame) the rest, so the frames run
    // in chunks
    const size_t fixed = assign_workspace_bytes(0, d, k, mode);
    constexpr size_t cap = EMMA_ASSIGN_NOALLOC_SCRATCH_BYTES;
    // per frame: list (8 bytes), its upper bound (4), list2 (8), a candidate
    // slot (36), with room for the 256-byte alignments
    const int64_t chunk_max = fixed + 8192 < cap ? (int64_t)((cap - fixed - 8192) / 64) : 0;
    EMMA_REQUIRE(chunk_max >= EMMA_ASSIGN_NOALLOC_MIN_CHUNK,
                 "emma_assign_noalloc: k=%d centers of d=%d take %zu of the %zu scratch bytes; at most %lld bytes "
                 "leave room for %d frames per chunk (use emma_assign with a workspace)",
                 k, d, fixed, cap, (long long)(cap - 8192 - 64 * (size_t)EMMA_ASSIGN_NOALLOC_MIN_CHUNK),
                 EMMA_ASSIGN_NOALLOC_MIN_CHUNK);
    const int64_t chunk = chunk_max < ((int64_t)1 << 22) ? chunk_max : ((int64_t)1 << 22);
    EMMA_REQUIRE(assign_workspace_bytes(chunk, d, k, mode) <= cap, "emma_assign_noalloc: chunk of %lld frames "
                 "exceeds the scratch", (long long)chunk);
    void *ws = nullptr;
    EMMA_TRY(scratch_on_current_device(&ws));
    if (n_rechecked) k_zero_i64n<<<1, 64, 0, s>>>(n_rechecked, 1);
    // the list length of each chunk is the first int64 of the carved workspace
    const AssignWs w = carve_assign(ws, chunk, d, k, mode);
    for (int64_t f0 = 0; f0 < n; f0 += chunk) {
        const int64_t m = n - f0 < chunk ? n - f0 : chunk;
        EMMA_TRY(assign_run(X + f0 * (int64_t)d, m, d, C, k, labels + f0, mode, nullptr, nullptr, ws, nullptr, s, n));
        if (n_rechecked) k_add_i64<<<1, 1, 0, s>>>(n_rechecked, w.rl.count);
    }
    return check_launch("emma_assign_noalloc");
}
