// kmeans++ seeding and Lloyd iterations.
//
// The reference hands both to deeptime (coordinates/clustering/kmeans.py:211-212,
// 254-261), whose source is outside the reference tree.  This file implements
// the documented rules shared with the CPU oracle:
//
// kmeans++ (Arthur & Vassilvitskii 2007, D^2 sampling):
//   round 0 picks row floor(u_0 n); round r >= 1 picks a row with probability
//   proportional to D^2 = squared FP32 distance (sequential loop, no FMA) to the
//   nearest chosen center.  u_r is draw r of a SplitMix64 stream of the seed.
//   Sums are FP64 in a fixed order: blocks of 4096 frames are summed lane-
//   strided by a 64-lane wavefront and combined with a butterfly; superblocks
//   of 64 blocks and segments of 64 frames are summed sequentially.  The pick
//   walks superblock -> block -> segment -> frame with running FP64 prefixes.
//
// Lloyd: labels = assign(X, C); cost = blocked FP64 sum of each frame's FP32
//   distance to its center; new C_j = FP64 mean of its members taken in frame
//   order in chunks of 256 (empty centers unchanged); stop when
//   |cost - prev| / cost <= tol.  Every iteration's kernels read a device flag
//   and return immediately once converged, so the host enqueues max_iter
//   iterations without synchronizing.
#include <math.h>

#include "emma_common.hpp"

namespace emma {

size_t assign_workspace_bytes(int64_t n, int d, int k, int mode);
int assign_run(const float *X, int64_t n, int d, const float *C, int k, int32_t *labels, int mode,
               int64_t *n_rechecked, int64_t *n_looped, void *workspace, const int32_t *done, hipStream_t s,
               int64_t n_call);

namespace km {

constexpr int BLOCK = 4096;
static_assert(BLOCK % 64 == 0, "a wave's frames lie in one block");
constexpr int SUPER = 64;
constexpr int SEG = 64;
constexpr int CHUNK = 256;

__device__ __forceinline__ float dist_seq(const float *__restrict__ x, const float *__restrict__ c, int d) {
    float acc = 0.0f;
    for (int i = 0; i < d; ++i) {
        const float t = __fsub_rn(x[i], c[i]);
        acc = __fadd_rn(acc, __fmul_rn(t, t));
    }
    return acc;
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
__device__ __forceinline__ double uniform(uint64_t seed, uint64_t counter) {
    const uint64_t z = mix64(seed + (counter + 1ULL) * 0x9E3779B97F4A7C15ULL);
    return (double)(z >> 11) * 0x1.0p-53;
}

// ------------------------------------------------------------------
// kmeans++
// ------------------------------------------------------------------
// A round is three launches: the squared distances of the new center to the
// earlier ones (k_kmpp_cc), the D^2 update (k_kmpp_d2), and the block sums with the
// pick by the last workgroup to finish (k_kmpp_sum_pick).
//
// The D^2 update reads a frame only where the new center can be nearer than the
// frame's current one: with D2 the stored FP32 distance of x to its nearest center
// a, and cc the distance of a to the new center c, the triangle inequality gives
// D(x, c) >= D(a, c) - D(x, a), so c cannot win where cc >= 4 D2, with the factor
// raised by the relative rounding g = gamma_{d+2} of all three FP32 sums
// (kmpp_factor): the loop's own result for c is then >= D2, and the strict '<'
// leaves D2 alone.  Every D2, and so every pick, is the one of the full pass.  What
// that saves depends on the data: 200,000 frames x 300 distances, k = 1000, read 240
// MB per round without it (54 us of a 96 us round).

// round 0: first pick; the counters of the later rounds
__global__ void k_kmpp_first(const float *__restrict__ X, int64_t n, int d, uint64_t seed, float *__restrict__ C,
                             int64_t *__restrict__ idx, unsigned int *__restrict__ counters, int n_counters) {
    int64_t pick = (int64_t)(uniform(seed, 0) * (double)n);
    if (pick >= n) pick = n - 1;
    if (threadIdx.x == 0) idx[0] = pick;
    for (int i = threadIdx.x; i < d; i += blockDim.x) C[i] = X[pick * d + i];
    for (int i = threadIdx.x; i < n_counters; i += blockDim.x) counters[i] = 0;
}

// cc[j] = |C_j - C_new|^2 for j < new (any summation order: its rounding is inside
// kmpp_factor), one wavefront per center
__global__ __launch_bounds__(256) void k_kmpp_cc(const float *__restrict__ C, int d, int nw, float *__restrict__ cc) {
    const int lane = threadIdx.x & 63, j = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= nw) return;
    const float *a = C + (int64_t)j * d, *b = C + (int64_t)nw * d;
    float s = 0.0f;
#pragma unroll 4
    for (int i = lane; i < d; i += 64) {
        const float t = a[i] - b[i];
        s = fmaf(t, t, s);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) cc[j] = s;
}
static float kmpp_factor(int d) {
    const double u = ldexp(1.0, -24), g = (d + 2) * u / (1.0 - (d + 2) * u);
    return (float)(4.0 * (1.0 + 8.0 * g));
}

__device__ __forceinline__ float dist_step(float acc, float x, float c) {
    const float t = __fsub_rn(x, c);
    return __fadd_rn(acc, __fmul_rn(t, t));
}

// The sequential FP32 distance of row x to c (LDS), the loads of 16 dims in flight
// before their terms.  VEC: rows 16-byte aligned (d % 4 == 0 and X aligned).
template <bool VEC>
__device__ __forceinline__ float dist_row(const float *__restrict__ x, const float *c, int d) {
    float acc = 0.0f;
    int q = 0;
    for (; q + 16 <= d; q += 16) {
        float v[16];
        if constexpr (VEC) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float4 w = *reinterpret_cast<const float4 *>(x + q + 4 * u);
                v[4 * u] = w.x, v[4 * u + 1] = w.y, v[4 * u + 2] = w.z, v[4 * u + 3] = w.w;
            }
        } else {
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = x[q + u];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) acc = dist_step(acc, v[u], c[q + u]);
    }
    // the rest in the same way, four dims at a time: read one after the other, ten dims
    // were ten round trips (5 10^6 x 10: 80 us per round, 56 now)
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; u += 4) {
        if (q + u >= d) break;
        if constexpr (VEC) {
            const float4 w = *reinterpret_cast<const float4 *>(x + q + u);
            v[u] = w.x, v[u + 1] = w.y, v[u + 2] = w.z, v[u + 3] = w.w;
        } else {
#pragma unroll
            for (int e = u; e < u + 4; ++e)
                if (q + e < d) v[e] = x[q + e];
        }
    }
#pragma unroll
    for (int u = 0; u < 16; u += 4) {
        if (q + u >= d) break;
#pragma unroll
        for (int e = u; e < u + 4; ++e)
            if (VEC || q + e < d) acc = dist_step(acc, v[e], c[q + e]);
    }
    return acc;
}

// D^2 update against the new center C[r - 1]: the frames that the triangle
// inequality leaves are compacted over the workgroup, one thread each.  A thread that
// reads its row itself touches a cache line of its own with every load; where that is
// the time (kmpp_staged) a wave reads its 64 rows together instead, 64 dims at a time
// with 16 lanes to a row, and its threads add from LDS (the next 64 dims in flight
// meanwhile).  Rows of any alignment: the loads are 4-byte aligned, those across a
// row's end element by element.
// (200,000 distances x 300, k = 1000, per round: 54 us for all rows by their own threads, 30 with
// the triangle inequality, 26 staged.)
enum Rows { ROWS_ANY = 0, ROWS_VEC = 1, ROWS_STAGED = 2 };
constexpr int SDIM = 64, SPITCH = SDIM + 4;  // pitch: 16-byte rows on distinct banks
template <int ROWS>
__global__ __launch_bounds__(256) void k_kmpp_d2(const float *__restrict__ X, int64_t n, int d,
                                                 const float *__restrict__ c, int r, float factor,
                                                 const float *__restrict__ cc, float *__restrict__ d2,
                                                 int32_t *__restrict__ owner) {
    extern __shared__ float s_c[];
    __shared__ __align__(16) float s_x[ROWS == ROWS_STAGED ? 4 * 64 * SPITCH : 4];
    __shared__ int s_list[256];
    __shared__ float s_v[256];
    __shared__ int s_cnt;
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t i0 = (int64_t)blockIdx.x * 256, i = i0 + tid;
    if (tid == 0) s_cnt = 0;
    __syncthreads();
    bool act = false;
    float v = 0.0f;
    if (i < n) {
        act = true;
        if (r > 1) {
            v = d2[i];
            // v tiny, overflowed or NaN: no argument from it
            act = !(v > 1e-25f && v < 1e37f && cc[owner[i]] >= factor * v);
        }
    }
    const unsigned long long m = __ballot(act);
    if (m) {
        const int leader = __builtin_ctzll(m);
        int base = 0;
        if (lane == leader) base = atomicAdd(&s_cnt, __popcll(m));
        base = __shfl(base, leader, 64);
        if (act) {
            const int q = base + __popcll(m & ((1ull << lane) - 1ull));
            s_list[q] = tid;
            s_v[q] = v;
        }
    }
    __syncthreads();
    const int na = s_cnt;
    if (na == 0) return;
    float di = 0.0f;
    if constexpr (ROWS == ROWS_STAGED) {
        const int l0 = tid & ~63, cnt = na - l0 < 64 ? na - l0 : 64;
        if (cnt <= 0) return;  // no barrier below
        float *buf = s_x + (tid >> 6) * 64 * SPITCH;
        const int sub = lane >> 4, col = (lane & 15) * 4;
        int row[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) row[u] = u * 4 + sub < cnt ? s_list[l0 + u * 4 + sub] : -1;
        const float *base = X + i0 * d;
        float4 t[16];
        auto load = [&](int q0) __attribute__((always_inline)) {
            const int q = q0 + col;
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                if (row[u] < 0 || q >= d) continue;
                const float *x = base + (int64_t)row[u] * d + q;
                if (q + 4 <= d) {
                    const float4_u w = *reinterpret_cast<const float4_u *>(x);
                    t[u] = make_float4(w[0], w[1], w[2], w[3]);
                } else {
                    t[u].x = x[0];
                    if (q + 1 < d) t[u].y = x[1];
                    if (q + 2 < d) t[u].z = x[2];
                }
            }
        };
#pragma unroll
        for (int u = 0; u < 16; ++u) t[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        load(0);
        for (int q0 = 0; q0 < d; q0 += SDIM) {
#pragma unroll
            for (int u = 0; u < 16; ++u)
                *reinterpret_cast<float4 *>(buf + (u * 4 + sub) * SPITCH + col) = t[u];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (q0 + SDIM < d) load(q0 + SDIM);
            const float *mine = buf + lane * SPITCH;
            const int nq = d - q0 < SDIM ? d - q0 : SDIM;
            int q = 0;
            for (; q + 16 <= nq; q += 16) {
                float4 w[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) w[u] = *reinterpret_cast<const float4 *>(mine + q + 4 * u);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    di = dist_step(di, w[u].x, c[q0 + q + 4 * u]);
                    di = dist_step(di, w[u].y, c[q0 + q + 4 * u + 1]);
                    di = dist_step(di, w[u].z, c[q0 + q + 4 * u + 2]);
                    di = dist_step(di, w[u].w, c[q0 + q + 4 * u + 3]);
                }
            }
            for (; q < nq; ++q) di = dist_step(di, mine[q], c[q0 + q]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    } else {
        for (int q = tid; q < d; q += 256) s_c[q] = c[q];
        __syncthreads();
        if (tid < na) di = dist_row<ROWS == ROWS_VEC>(X + (i0 + s_list[tid]) * d, s_c, d);
    }
    if (tid < na && (r == 1 || di < s_v[tid])) {
        const int64_t f = i0 + s_list[tid];
        d2[f] = di;
        owner[f] = r - 1;
    }
}

// Lane l's value added after those of lanes 0 .. l - 1, in that order: inclusive
// running sums from `run`, as one thread walking the values would form them.  The
// values are >= 0 or NaN, and 0 from lane cnt on, so that adding those changes nothing
// and the lanes can be taken 16 at a time.
__device__ __forceinline__ double running_sum(double a, int cnt, double run, int lane) {
    double mine = run;
    const long long bits = __double_as_longlong(a);
    for (int l0 = 0; l0 < cnt; l0 += 16) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int lo = __builtin_amdgcn_readlane((int)(bits & 0xffffffffll), l0 + u);
            const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), l0 + u);
            run = run + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
            mine = lane == l0 + u ? run : mine;
        }
    }
    return mine;
}
__device__ __forceinline__ double lane_value(double a, int l) { return __shfl(a, l, 64); }

// One step of the oracle's walk over cnt <= 64 values a (lane l holds value l):
// the first whose running sum passes T, or else the last positive one (-1: none);
// `before` becomes the running sum in front of it.
__device__ __forceinline__ int walk_step(double a, int cnt, double T, double &before, int lane) {
    const double run = running_sum(a, cnt, before, lane);
    const unsigned long long over = __ballot(lane < cnt && run > T);
    const unsigned long long pos = __ballot(lane < cnt && a > 0.0);
    const int sel = over ? __builtin_ctzll(over) : (pos ? 63 - __builtin_clzll(pos) : -1);
    if (sel > 0) before = lane_value(run, sel - 1);
    return sel;
}

__device__ __forceinline__ void put_coherent(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get_coherent(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The counter's old value, after every earlier store of this thread has completed and
// before any later load: the wait orders the hardware, the signal fences (no instructions)
// keep the compiler from moving the relaxed accesses across it.
__device__ __forceinline__ unsigned int arrive(unsigned int *counter) {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    const unsigned int seen = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    return seen;
}

// Block sums (one workgroup per block of BLOCK frames), superblock sums by the last
// block of each, and the pick of round r by the last superblock's workgroup: exactly
// the oracle's oracle_kmpp_pick.  The sums travel between workgroups as coherent
// (device-scope) stores and loads, waited for before the arrival count: a release
// fence instead would write back the whole L2 from every workgroup.  The counters
// only grow: round r is complete at r times the number of arrivals.
// (Per round 41 us for block sums of one wave per block and a one-wave pick, 200,000
// frames; 13 here.  What is left is a chain of some eight dependent round trips to
// memory.)
__global__ __launch_bounds__(256) void k_kmpp_sum_pick(const float *__restrict__ X, int64_t n, int d, uint64_t seed,
                                                       int r, const float *__restrict__ d2,
                                                       double *__restrict__ bsum, double *__restrict__ sbsum,
                                                       unsigned int *__restrict__ counters,
                                                       float *__restrict__ C, int64_t *__restrict__ idx) {
    __shared__ float s_d[SEG * (SEG + 1)];  // a block's values, a segment per row (padded)
    __shared__ int s_last, s_blk;
    __shared__ int64_t s_pick;
    __shared__ double s_before, s_T;
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t nb = (n + BLOCK - 1) / BLOCK, nsb = (nb + SUPER - 1) / SUPER;
    // past the last frame: 0, which the sums below add without a change (values >= 0 or NaN)
    auto load_block = [&](int64_t blk) __attribute__((always_inline)) {
        const int64_t lo = blk * BLOCK;
        float v[BLOCK / 256];
#pragma unroll
        for (int u = 0; u < BLOCK / 256; ++u) {
            const int64_t i = lo + u * 256 + tid;
            v[u] = i < n ? d2[i] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < BLOCK / 256; ++u) {
            const int o = u * 256 + tid;
            s_d[(o / SEG) * (SEG + 1) + o % SEG] = v[u];
        }
    };
    const int64_t b = blockIdx.x, sb = b / SUPER;
    load_block(b);
    __syncthreads();
    double a_blk = 0.0, a_sb = 0.0;  // this superblock's block sums, its sum (the pick of a single one)
    if (tid < 64) {
        double s = 0.0;
#pragma unroll 16
        for (int m = 0; m < BLOCK / 64; ++m) s = s + (double)s_d[m * (SEG + 1) + lane];
        s = wave_butterfly_sum(s);
        const int in_sb = (int)(nb - sb * SUPER < SUPER ? nb - sb * SUPER : SUPER);
        unsigned int seen = 0;
        if (lane == 0) {
            put_coherent(bsum + b, s);
            seen = arrive(counters + 1 + sb);
        }
        seen = __shfl(seen, 0, 64);
        int last = 0;
        if (seen + 1 == (unsigned int)r * (unsigned int)in_sb) {
            a_blk = lane < in_sb ? get_coherent(bsum + sb * SUPER + lane) : 0.0;
            a_sb = lane_value(running_sum(a_blk, in_sb, 0.0, lane), in_sb - 1);
            unsigned int top = 0;
            if (nsb > 1 && lane == 0) {
                put_coherent(sbsum + sb, a_sb);
                top = arrive(counters);
            }
            last = nsb == 1 || __shfl(top, 0, 64) + 1 == (unsigned int)r * (unsigned int)nsb;
        }
        if (lane == 0) s_last = last;
    }
    __syncthreads();
    if (!s_last) return;

    const double u = uniform(seed, (uint64_t)r);
    if (tid < 64) {
        // superblocks 64 at a time: the total, then the walk
        auto superblocks = [&](int64_t s0, int cnt) __attribute__((always_inline)) {
            if (nsb == 1) return lane == 0 ? a_sb : 0.0;
            return lane < cnt ? get_coherent(sbsum + s0 + lane) : 0.0;
        };
        double total = 0.0;
        for (int64_t s0 = 0; s0 < nsb; s0 += 64) {
            const int cnt = (int)(nsb - s0 < 64 ? nsb - s0 : 64);
            const double a = superblocks(s0, cnt);
            total = lane_value(running_sum(a, cnt, total, lane), cnt - 1);
        }
        int64_t blk = -1;
        double before = 0.0;
        const double T = u * total;
        if (!(total > 0.0)) {
            const int64_t i = (int64_t)(u * (double)n);
            if (lane == 0) s_pick = i < n ? i : n - 1;
        } else {
            int64_t sel = -1, last_pos = -1;
            double run = 0.0, last_before = 0.0;
            for (int64_t s0 = 0; s0 < nsb && sel < 0; s0 += 64) {
                const int cnt = (int)(nsb - s0 < 64 ? nsb - s0 : 64);
                const double a = superblocks(s0, cnt);
                const double rs = running_sum(a, cnt, run, lane);
                const unsigned long long over = __ballot(lane < cnt && rs > T), pos = __ballot(lane < cnt && a > 0.0);
                if (over) {
                    const int q = __builtin_ctzll(over);
                    sel = s0 + q;
                    before = q > 0 ? lane_value(rs, q - 1) : run;
                } else if (pos) {
                    const int q = 63 - __builtin_clzll(pos);
                    last_pos = s0 + q;
                    last_before = q > 0 ? lane_value(rs, q - 1) : run;
                }
                run = lane_value(rs, cnt - 1);
            }
            if (sel < 0) {
                sel = last_pos;
                before = last_before;
            }
            const int cnt = (int)(nb - sel * SUPER < SUPER ? nb - sel * SUPER : SUPER);
            const double a = nsb == 1 ? a_blk : lane < cnt ? get_coherent(bsum + sel * SUPER + lane) : 0.0;
            blk = sel * SUPER + walk_step(a, cnt, T, before, lane);
        }
        if (lane == 0) {
            s_before = before;
            s_T = T;
            s_blk = (int)blk;
        }
    }
    __syncthreads();
    const int64_t blk = s_blk;
    if (blk >= 0) {
        load_block(blk);
        __syncthreads();
        if (tid < 64) {
            // segment sums (sequential inside a segment, one per lane), then the segment's frames
            const int64_t blo = blk * BLOCK, left = n - blo < BLOCK ? n - blo : BLOCK;
            const double T = s_T;
            double before = s_before;
            const int nseg = (int)((left + SEG - 1) / SEG);
            double a = 0.0;
#pragma unroll 16
            for (int q = 0; q < SEG; ++q) a = a + (double)s_d[lane * (SEG + 1) + q];
            const int seg = walk_step(a, nseg, T, before, lane);
            const int nf = (int)(left - seg * SEG < SEG ? left - seg * SEG : SEG);
            const int fr = walk_step((double)s_d[seg * (SEG + 1) + lane], nf, T, before, lane);
            if (lane == 0) s_pick = blo + (int64_t)seg * SEG + fr;
        }
        __syncthreads();
    }
    const int64_t pick = s_pick;
    if (tid == 0) idx[r] = pick;
    for (int i = tid; i < d; i += 256) C[(int64_t)r * d + i] = X[pick * d + i];
}

// Below 64 dims half of the lanes or more would have no dims to read.  With at most one
// workgroup per CU, and frames that the caches hold, the time is one row's chain of
// loads, which staging makes longer: k = 20, whole call, own rows and staged,
// 1000 x 300 367 and 482 us, 1000 x 1000 641 and 961, 64,000 x 300 510 and 562,
// 32,000 x 3001 3751 and 2412, 100,000 x 300 716 and 688.
static bool kmpp_staged(int64_t n, int d) {
    return d >= SDIM && (n > 65536 || n * d > 50'000'000 || d > 8192);  // own rows: the center in LDS
}

struct PpWs {
    float *d2;
    int32_t *owner;
    float *cc;
    double *bsum, *sbsum;
    unsigned int *counters;  // [1 + superblocks]
    size_t bytes;
};

static PpWs carve_pp(void *ws, int64_t n, int k) {
    PpWs w{};
    Carver cv(ws);
    const int64_t nb = cdiv(n, BLOCK), nsb = cdiv(nb, SUPER);
    w.d2 = cv.take<float>(n);
    w.owner = cv.take<int32_t>(n);
    w.cc = cv.take<float>(k);
    w.bsum = cv.take<double>(nb);
    w.sbsum = cv.take<double>(nsb);
    w.counters = cv.take<unsigned int>(1 + (size_t)nsb);
    w.bytes = cv.bytes();
    return w;
}

// Block sums of Lloyd's distances: one workgroup per block of BLOCK frames, whose
// values are loaded in one round trip; the first wave's lane l adds frames l, l +
// 64, ... in FP64 in that order, then a butterfly (the oracle's order; the zeros
// past the last frame change no sum).  done: skip
// once Lloyd has converged.
__global__ __launch_bounds__(256) void k_block_sums(int64_t n, const float *__restrict__ d2,
                                                    double *__restrict__ bsum, const int32_t *__restrict__ done) {
    if (*done) return;
    __shared__ float s_d[BLOCK];
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t lo = (int64_t)blockIdx.x * BLOCK, left = n - lo;
    float v[BLOCK / 256];
#pragma unroll
    for (int u = 0; u < BLOCK / 256; ++u) v[u] = u * 256 + tid < left ? d2[lo + u * 256 + tid] : 0.0f;
#pragma unroll
    for (int u = 0; u < BLOCK / 256; ++u) s_d[u * 256 + tid] = v[u];
    __syncthreads();
    if (tid >= 64) return;
    double s = 0.0;
#pragma unroll 16
    for (int m = 0; m < BLOCK / 64; ++m) s = s + (double)s_d[m * 64 + lane];
    s = wave_butterfly_sum(s);
    if (lane == 0) bsum[blockIdx.x] = s;
}

// ------------------------------------------------------------------
// Lloyd
// ------------------------------------------------------------------
struct LloydWs {
    int32_t *done;        // [1]
    double *prev_cost;    // [1]
    double *bcost;        // [nb]
    int64_t *cnt;         // [k]
    int64_t *off;         // [k + 1] member offsets
    int64_t *coff;        // [k + 1] chunk offsets
    int32_t *blk_cnt;     // [nb * k] per-block label counts -> block prefixes
    int64_t *order;       // [n] members sorted by (label, frame)
    float *dist;          // [n] distance of each frame to its center
    double *chunk_sums;   // [n / CHUNK + k][d]
    void *assign_ws;
    size_t bytes;
};

static LloydWs carve_lloyd(void *ws, int64_t n, int d, int k, int mode) {
    LloydWs w{};
    Carver cv(ws);
    const int64_t nb = cdiv(n, BLOCK);
    w.done = cv.take<int32_t>(1);
    w.prev_cost = cv.take<double>(1);
    w.bcost = cv.take<double>(nb);
    w.cnt = cv.take<int64_t>(k);
    w.off = cv.take<int64_t>((size_t)k + 1);
    w.coff = cv.take<int64_t>((size_t)k + 1);
    w.blk_cnt = cv.take<int32_t>((size_t)nb * k);
    w.order = cv.take<int64_t>(n);
    w.dist = cv.take<float>(n);
    w.chunk_sums = cv.take<double>((size_t)(n / CHUNK + k + 1) * d);
    w.assign_ws = cv.take<char>(assign_workspace_bytes(n, d, k, mode));
    w.bytes = cv.bytes();
    return w;
}

__global__ void k_lloyd_init(int32_t *done, double *prev_cost, int32_t *n_iter, int32_t *converged) {
    *done = 0;
    *prev_cost = 0.0;
    *n_iter = 0;
    *converged = 0;
}

// Counts of the labels of one block of frames, one workgroup per block, in LDS: one
// LDS atomic per run of equal labels in a wave (consecutive frames of a trajectory
// mostly share their label, and 64 lanes adding 1 to one counter serialize).  (Device
// atomics and clearing the counts beforehand: 21 us at 250,000 frames, k = 200; now
// 4.)
__global__ __launch_bounds__(1024) void k_lloyd_hist(int64_t n, int k, const int32_t *__restrict__ labels,
                                                     int32_t *__restrict__ blk_cnt,
                                                     const int32_t *__restrict__ done) {
    if (*done) return;
    extern __shared__ int32_t s_run[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t b = blockIdx.x, lo = b * BLOCK;
    int lab[BLOCK / 1024];
#pragma unroll
    for (int u = 0; u < BLOCK / 1024; ++u) lab[u] = lo + u * 1024 + tid < n ? labels[lo + u * 1024 + tid] : -1;
    for (int j = tid; j < k; j += 1024) s_run[j] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BLOCK / 1024; ++u) {
        const int prev = __shfl_up(lab[u], 1, 64);
        const bool start = lane == 0 || prev != lab[u];
        const unsigned long long starts = __ballot(start);
        const unsigned long long later = starts & ~((2ull << lane) - 1ull);  // starts after this lane
        if (start && lab[u] >= 0) atomicAdd(&s_run[lab[u]], (later ? __builtin_ctzll(later) : 64) - lane);
    }
    __syncthreads();
    for (int j = tid; j < k; j += 1024) blk_cnt[b * k + j] = s_run[j];
}

// The exact distance to the center of its label (the sequential FP32 loop; VEC: rows
// of X and C 16-byte aligned), one thread per frame, run after the update so that the
// cost is that of the new clusters against their means.  The block sums of the
// distances (the oracle's cost order) follow in k_block_sums.
template <bool VEC>
__global__ __launch_bounds__(256) void k_lloyd_dist(const float *__restrict__ X, int64_t n, int d,
                                                    const float *__restrict__ C, const int32_t *__restrict__ labels,
                                                    float *__restrict__ dist, const int32_t *__restrict__ done) {
    if (*done) return;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int lab = labels[i];
    const float *x = X + i * d;
    const float *c = C + (int64_t)lab * d;
    float di;
    if constexpr (VEC) {
        float acc = 0.0f;
        auto step4 = [&](const float4 xv, const float4 cv) __attribute__((always_inline)) {
            float t = __fsub_rn(xv.x, cv.x);
            acc = __fadd_rn(acc, __fmul_rn(t, t));
            t = __fsub_rn(xv.y, cv.y);
            acc = __fadd_rn(acc, __fmul_rn(t, t));
            t = __fsub_rn(xv.z, cv.z);
            acc = __fadd_rn(acc, __fmul_rn(t, t));
            t = __fsub_rn(xv.w, cv.w);
            acc = __fadd_rn(acc, __fmul_rn(t, t));
        };
        // dims in order; the loads of 16 dims are issued before their terms
        int q = 0;
        for (; q + 16 <= d; q += 16) {
            float4 xv[4], cv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                xv[u] = *reinterpret_cast<const float4 *>(x + q + 4 * u);
                cv[u] = *reinterpret_cast<const float4 *>(c + q + 4 * u);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) step4(xv[u], cv[u]);
        }
        for (; q < d; q += 4)
            step4(*reinterpret_cast<const float4 *>(x + q), *reinterpret_cast<const float4 *>(c + q));
        di = acc;
    } else {
        di = dist_seq(x, c, d);
    }
    dist[i] = di;
}

// Per label: turn the blk_cnt column into exclusive prefixes over blocks and
// total it (cnt); then member offsets off[j] and chunk offsets coff[j]
// (exclusive scans over k).  One workgroup.
__global__ __launch_bounds__(1024) void k_lloyd_scan(int k, int64_t nb, int64_t *__restrict__ cnt,
                                                     int64_t *__restrict__ off, int64_t *__restrict__ coff,
                                                     int32_t *__restrict__ blk_cnt, const int32_t *__restrict__ done) {
    if (*done) return;
    __shared__ int64_t s_a[16], s_c[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int64_t a0 = 0, c0 = 0;  // members and chunks of the labels before this pass of 1024
    for (int j0 = 0; j0 < k; j0 += 1024) {
        const int j = j0 + tid;
        int64_t m = 0;
        if (j < k) {
            int32_t run = 0, v[16];
            for (int64_t b = 0; b < nb; b += 16) {
                const int cnt16 = nb - b < 16 ? (int)(nb - b) : 16;
#pragma unroll
                for (int u = 0; u < 16; ++u) v[u] = u < cnt16 ? blk_cnt[(b + u) * k + j] : 0;
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    if (u < cnt16) blk_cnt[(b + u) * k + j] = run;
                    run += v[u];
                }
            }
            cnt[j] = m = run;
        }
        const int64_t ch = (m + CHUNK - 1) / CHUNK;
        int64_t a = m, c = ch;  // inclusive sums over the wave
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int64_t ta = __shfl_up(a, o, 64), tc = __shfl_up(c, o, 64);
            if (lane >= o) {
                a += ta;
                c += tc;
            }
        }
        __syncthreads();
        if (lane == 63) {
            s_a[wave] = a;
            s_c[wave] = c;
        }
        __syncthreads();
        int64_t ta = a0, tc = c0;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) {
                a += s_a[w];
                c += s_c[w];
            }
            ta += s_a[w];
            tc += s_c[w];
        }
        if (j < k) {
            off[j] = a0 + a - m;
            coff[j] = c0 + c - ch;
        }
        a0 = ta;
        c0 = tc;
    }
    if (tid == 0) {
        off[k] = a0;
        coff[k] = c0;
    }
}

// Stable scatter: position of frame i = off[label] + (members of label in earlier
// blocks) + (members in this block before i).  One workgroup per block: every wave
// ranks its four groups of 64 frames among the lanes of their label (a ballot per bit
// of the labels), then the waves take turns in frame order, the first lane of each
// label moving that label's running count on.  (One wave per block that compares each
// frame with the 63 others, a group after the other: 148 us at 250,000 frames; now
// 10.)
__global__ __launch_bounds__(1024) void k_lloyd_scatter(int64_t n, int k, const int32_t *__restrict__ labels,
                                                        const int64_t *__restrict__ off,
                                                        const int32_t *__restrict__ blk_cnt,
                                                        int64_t *__restrict__ order, const int32_t *__restrict__ done) {
    if (*done) return;
    constexpr int G = BLOCK / 1024;
    extern __shared__ int32_t s_run[];  // k running counters
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t b = blockIdx.x, lo = b * BLOCK + wave * (64 * G) + lane;
    int lab[G], rank[G], cnt[G], lead[G];
    int64_t start[G];
#pragma unroll
    for (int u = 0; u < G; ++u) lab[u] = lo + u * 64 < n ? labels[lo + u * 64] : -1;
    for (int j = tid; j < k; j += 1024) s_run[j] = blk_cnt[b * k + j];
    const int bits = k > 1 ? 32 - __builtin_clz((unsigned int)(k - 1)) : 0;
#pragma unroll
    for (int u = 0; u < G; ++u) {
        start[u] = lab[u] >= 0 ? off[lab[u]] : 0;
        unsigned long long same = __ballot(lab[u] >= 0);
        for (int q = 0; q < bits; ++q) {
            const bool bit = (lab[u] >> q) & 1;
            const unsigned long long m = __ballot(bit);
            same &= bit ? m : ~m;
        }
        rank[u] = __popcll(same & ((1ull << lane) - 1ull));
        cnt[u] = __popcll(same);
        lead[u] = same ? __builtin_ctzll(same) : 0;
    }
    __syncthreads();
    for (int w = 0; w < 16; ++w) {
        if (w == wave) {
#pragma unroll
            for (int u = 0; u < G; ++u) {
                int base = 0;
                if (lab[u] >= 0 && rank[u] == 0) {
                    base = s_run[lab[u]];
                    s_run[lab[u]] = base + cnt[u];
                }
                rank[u] += __shfl(base, lead[u], 64);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < G; ++u)
        if (lab[u] >= 0) order[start[u] + rank[u]] = lo + u * 64;
}

// Chunk sums: one wavefront per chunk, lanes over dimensions, members in order.
__global__ __launch_bounds__(256) void k_lloyd_chunks(const float *__restrict__ X, int d, int k,
                                                      const int64_t *__restrict__ off,
                                                      const int64_t *__restrict__ coff,
                                                      const int64_t *__restrict__ order,
                                                      double *__restrict__ chunk_sums,
                                                      const int32_t *__restrict__ done) {
    if (*done) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t ch = (int64_t)blockIdx.x * 4 + wave;
    if (ch >= coff[k]) return;
    // center owning this chunk: largest j with coff[j] <= ch
    int lo = 0, hi = k - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (coff[mid] <= ch) lo = mid; else hi = mid - 1;
    }
    const int j = lo;
    const int64_t m0 = off[j] + (ch - coff[j]) * CHUNK;
    const int64_t m1 = m0 + CHUNK < off[j + 1] ? m0 + CHUNK : off[j + 1];
    for (int i0 = 0; i0 < d; i0 += 64) {
        const int i = i0 + lane;
        double a = 0.0;
        if (i < d) {
            // members in order; the loads of 8 members are issued before
            // their adds (same sum, one memory round trip per 8)
            int64_t m = m0;
            for (; m + 8 <= m1; m += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = X[order[m + u] * d + i];
#pragma unroll
                for (int u = 0; u < 8; ++u) a = a + (double)v[u];
            }
            for (; m < m1; ++m) a = a + (double)X[order[m] * d + i];
        }
        if (i < d) chunk_sums[ch * d + i] = a;
    }
}

// New centers (one wavefront per center) and the convergence bookkeeping.
__global__ __launch_bounds__(256) void k_lloyd_update(int d, int k, const int64_t *__restrict__ cnt,
                                                      const int64_t *__restrict__ coff,
                                                      const double *__restrict__ chunk_sums, float *__restrict__ C,
                                                      const int32_t *__restrict__ done) {
    if (*done) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int j = blockIdx.x * 4 + wave;
    if (j >= k || cnt[j] == 0) return;
    const double cntd = (double)cnt[j];
    for (int i0 = 0; i0 < d; i0 += 64) {
        const int i = i0 + lane;
        if (i >= d) continue;
        double a = 0.0;
        for (int64_t ch = coff[j]; ch < coff[j + 1]; ++ch) a = a + chunk_sums[ch * d + i];
        C[(int64_t)j * d + i] = (float)(a / cntd);
    }
}

__global__ void k_lloyd_cost_final(int64_t nb, const double *__restrict__ bcost, double tol, int it,
                                   double *__restrict__ prev_cost, double *__restrict__ inertias,
                                   int32_t *__restrict__ n_iter, int32_t *__restrict__ converged,
                                   int32_t *__restrict__ done) {
    if (*done) return;
    double cost = 0.0;
    for (int64_t b = 0; b < nb; ++b) cost = cost + bcost[b];
    const double prev = *prev_cost;
    const double rel = cost != 0.0 ? fabs(cost - prev) / cost : 0.0;
    *prev_cost = cost;
    inertias[it] = cost;
    *n_iter = it + 1;
    if (rel <= tol) {
        *converged = 1;
        *done = 1;
    }
}

}  // namespace km
}  // namespace emma

using namespace emma;

extern "C" size_t emma_kmeanspp_workspace_size(int64_t n, int32_t d, int32_t k) {
    (void)d;
    if (n <= 0 || k <= 0) return 0;
    return km::carve_pp(nullptr, n, k).bytes;
}

extern "C" int emma_kmeanspp(const float *X, int64_t n, int32_t d, int32_t k, uint64_t seed, float *C_out,
                             int64_t *idx_out, void *workspace, size_t workspace_bytes, void *stream) {
    EMMA_REQUIRE(n > 0 && d > 0 && k > 0, "emma_kmeanspp: bad sizes n=%lld d=%d k=%d", (long long)n, d, k);
    EMMA_REQUIRE(X && C_out && idx_out, "emma_kmeanspp: NULL pointer");
    EMMA_REQUIRE(d <= 16384, "emma_kmeanspp: d=%d too large", d);
    const size_t need = km::carve_pp(nullptr, n, k).bytes;
    EMMA_REQUIRE(workspace && workspace_bytes >= need, "emma_kmeanspp: workspace too small (%zu < %zu)",
                 workspace_bytes, need);
    km::PpWs w = km::carve_pp(workspace, n, k);
    hipStream_t s = (hipStream_t)stream;
    const int64_t nb = cdiv(n, km::BLOCK);
    km::k_kmpp_first<<<1, 256, 0, s>>>(X, n, d, seed, C_out, idx_out, w.counters, (int)(1 + cdiv(nb, km::SUPER)));
    EMMA_TRY(check_launch("kmeans++ first"));
    const bool vec = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
    const size_t shm = sizeof(float) * (size_t)d;
    const float factor = km::kmpp_factor(d);
    const bool staged = km::kmpp_staged(n, d);
    for (int r = 1; r < k; ++r) {
        const float *c = C_out + (int64_t)(r - 1) * d;
        if (r > 1) km::k_kmpp_cc<<<(unsigned)cdiv(r - 1, 4), 256, 0, s>>>(C_out, d, r - 1, w.cc);
        const unsigned g = (unsigned)cdiv(n, 256);
        if (staged)
            km::k_kmpp_d2<km::ROWS_STAGED><<<g, 256, 0, s>>>(X, n, d, c, r, factor, w.cc, w.d2, w.owner);
        else if (vec)
            km::k_kmpp_d2<km::ROWS_VEC><<<g, 256, shm, s>>>(X, n, d, c, r, factor, w.cc, w.d2, w.owner);
        else
            km::k_kmpp_d2<km::ROWS_ANY><<<g, 256, shm, s>>>(X, n, d, c, r, factor, w.cc, w.d2, w.owner);
        km::k_kmpp_sum_pick<<<(unsigned)nb, 256, 0, s>>>(X, n, d, seed, r, w.d2, w.bsum, w.sbsum, w.counters, C_out, idx_out);
    }
    return check_launch("kmeans++ rounds");
}

extern "C" size_t emma_lloyd_workspace_size(int64_t n, int32_t d, int32_t k, int32_t assign_mode) {
    if (n <= 0 || d <= 0 || k <= 0) return 0;
    return km::carve_lloyd(nullptr, n, d, k, assign_mode).bytes;
}

extern "C" int emma_lloyd(const float *X, int64_t n, int32_t d, float *C, int32_t k, int32_t max_iter, double tol,
                          int32_t assign_mode, int32_t *labels, double *inertias, int32_t *n_iter,
                          int32_t *converged, void *workspace, size_t workspace_bytes, void *stream) {
    EMMA_REQUIRE(n > 0 && d > 0 && k > 0 && max_iter >= 0, "emma_lloyd: bad sizes n=%lld d=%d k=%d max_iter=%d",
                 (long long)n, d, k, max_iter);
    EMMA_REQUIRE(assign_mode == EMMA_ASSIGN_FP32_PLAIN || assign_mode == EMMA_ASSIGN_BF16X3_RECHECK,
                 "emma_lloyd: unknown assign mode %d", assign_mode);
    EMMA_REQUIRE(X && C && labels && n_iter && converged && (inertias || max_iter == 0), "emma_lloyd: NULL pointer");
    EMMA_REQUIRE(k <= 12288, "emma_lloyd: k=%d too large for the scatter kernel", k);
    const size_t need = km::carve_lloyd(nullptr, n, d, k, assign_mode).bytes;
    EMMA_REQUIRE(workspace && workspace_bytes >= need, "emma_lloyd: workspace too small (%zu < %zu)",
                 workspace_bytes, need);
    km::LloydWs w = km::carve_lloyd(workspace, n, d, k, assign_mode);
    hipStream_t s = (hipStream_t)stream;
    const int64_t nb = cdiv(n, km::BLOCK);
    km::k_lloyd_init<<<1, 1, 0, s>>>(w.done, w.prev_cost, n_iter, converged);
    const bool vec = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(C) & 15) == 0;
    for (int it = 0; it < max_iter; ++it) {
        EMMA_TRY(assign_run(X, n, d, C, k, labels, assign_mode, nullptr, nullptr, w.assign_ws, w.done, s, n));
        const size_t run_shm = sizeof(int32_t) * (size_t)k;
        km::k_lloyd_hist<<<(unsigned)nb, 1024, run_shm, s>>>(n, k, labels, w.blk_cnt, w.done);
        km::k_lloyd_scan<<<1, 1024, 0, s>>>(k, nb, w.cnt, w.off, w.coff, w.blk_cnt, w.done);
        km::k_lloyd_scatter<<<(unsigned)nb, 1024, run_shm, s>>>(n, k, labels, w.off, w.blk_cnt, w.order, w.done);
        const int64_t max_chunks = n / km::CHUNK + k + 1;
        km::k_lloyd_chunks<<<(unsigned)cdiv(max_chunks, 4), 256, 0, s>>>(X, d, k, w.off, w.coff, w.order,
                                                                         w.chunk_sums, w.done);
        // move the centers to the member means, then take the cost of the new
        // clusters against them and record it (which may raise the convergence flag)
        km::k_lloyd_update<<<(unsigned)cdiv(k, 4), 256, 0, s>>>(d, k, w.cnt, w.coff, w.chunk_sums, C, w.done);
        if (vec)
            km::k_lloyd_dist<true><<<(unsigned)cdiv(n, 256), 256, 0, s>>>(X, n, d, C, labels, w.dist, w.done);
        else
            km::k_lloyd_dist<false><<<(unsigned)cdiv(n, 256), 256, 0, s>>>(X, n, d, C, labels, w.dist, w.done);
        km::k_block_sums<<<(unsigned)nb, 256, 0, s>>>(n, w.dist, w.bcost, w.done);
        km::k_lloyd_cost_final<<<1, 1, 0, s>>>(nb, w.bcost, tol, it, w.prev_cost, inertias, n_iter, converged,
                                               w.done);
        EMMA_TRY(check_launch("lloyd iteration"));
    }
    return EMMA_OK;
}
