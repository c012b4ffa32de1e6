// The prompt gauge: a per-frame multiplicative correction exp(poly(u, v)) fitted robustly (IRLS) to
// log(prompt / prediction) on confident prompt pixels and applied at full resolution (prompt_gauge_poly,
// moge/model/v3.py:151-183; infer's default gauge_poly = 2, v3.py:841-853).
//
//   gauge_inputs_k  one thread per LiDAR pixel: the area-pooled valid depth z_lr (the window sums of
//                   where(ok, depth, 0) and of ok, each / height / width, as F.interpolate(mode='area')), the mask
//                   conf >= 2 & lidar > 0 & z_lr > 0, y = log(max(lidar, 1e-3)) - log(max(z_lr, 1e-3)), and the first
//                   round's sums: fp64 partials per block of the weighted normal equations (A w)^T (A w) c = (A w)^T (y w)
//   per IRLS round but the last
//     gauge_resid_k   solves the round's system (every block, from the same partials in the same order: Gaussian
//                     elimination with partial pivoting; the reference runs LAPACK least squares on the same fp32
//                     products), writes the fp32 residuals |y - A c| and counts them into bins of 1/128 octave (1/8
//                     octave below 2^-18 and from 2^-2 up)
//     gauge_pick_k    finds the bin holding the exact lower median and lists its residuals; more than 4096 of them also
//                     by sub-bins
//     gauge_third_k   (maps of more than 2^19 pixels) counts the median's sub-bin of more than 4096, value by value
//     gauge_sums_k    selects the median among the listed (more than 4096: counts the sub-bin's values itself, where
//                     gauge_third_k has not), forms the weights min(2 sc / max(|r|, 1e-6), 1),
//                     sc = 1.4826 median + 1e-4, and sums the next round's system
//   gauge_apply_k   solves the last system; per output pixel exp of the polynomial (a sequential fp32 sum over the basis)
//
// What bounds it: launches and the chain of small phases in them (the data is 0.4 MB at a 192x256 LiDAR map). Every step
// that one block or wave did for the whole frame in a launch of its own (the reduction of the partials, the solve, the
// median's bin) is done by all blocks of the next kernel instead, from the same data in the same order: 8 launches for
// three rounds where there were 22. Measured (depth 480x640, LiDAR 192x256, the whole call): 200 -> 56 us. By the
// residuals, us, the 22 launches (three radix passes each round whatever the values) / now: LiDAR 192x256, log noise of 1 (the
// median among the coarse bins) 205 / 77; 480x640, 2 % noise 370 / 86, log noise of 1 363 / 91, half the pixels off by 3x
// 365 / 189, all equal 341 / 184; 756x1008, 2 % noise 420 / 136; 1500x2000, 2 % noise 646 / 326, all equal 618 / 369.
//
// The basis is (1, u, v) or (1, u, v, u^2, uv, v^2) on torch.linspace(-1, 1, n) grids (the scalar rule: step
// 2 / (n - 1) in fp32, start + step i for the first half, end - step (n - 1 - i) for the second). A frame with
// fewer than 200 confident pixels, or a singular / non-finite system, gets the correction 1. The frame state (valid,
// count, median search) lives in device memory, so the whole sequence runs without a host round trip.
#include <climits>

#include "pmg_common.h"

namespace pmg {

constexpr int kGaugeMinPoints = 200;
constexpr int kGaugeMaxK = 6;

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

__device__ inline float linspace_at(int i, int n) {
    if (n == 1) return -1.0f;
    const float step = 2.0f / (float)(n - 1);
    return i < n / 2 ? -1.0f + step * (float)i : 1.0f - step * (float)(n - 1 - i);
}

__device__ inline void gauge_basis(float u, float v, float (&a)[kGaugeMaxK]) {
    a[0] = 1.0f;
    a[1] = u;
    a[2] = v;
    a[3] = u * u;
    a[4] = u * v;
    a[5] = v * v;
}

constexpr int kGaugeBlk = 256;        // threads of the grid kernels
constexpr int kGaugeMaxBlocks = 256;  // blocks per frame
constexpr int kGaugeVals = 28;        // 21 normal-matrix entries + 6 right-hand sides + count (K = 6; fewer for 3)
constexpr int kGaugeList = 4096;      // listed residuals a block keeps in LDS
// The bins, over the residuals' keys (fp32 bit patterns, a NaN's without its sign: below 2^31): 16 octaves, 2^-18 .. 2^-2, in
// 2^16 keys each, where the median of a noisy prompt lies; 2^20 keys each outside them (frames that fit exactly, or not
// at all).
constexpr uint32_t kGaugeLow = (127u - 18u) << 23, kGaugeHigh = kGaugeLow + (16u << 23);
constexpr int kGaugeFine = 16, kGaugeCoarse = 20;
constexpr int kGaugeBelow = (int)(kGaugeLow >> kGaugeCoarse);              // bins below the fine ones
constexpr int kGaugeAbove = kGaugeBelow + (int)((16u << 23) >> kGaugeFine);  // ... and those above them start here
constexpr int kGaugeBins = 4096;
static_assert(kGaugeAbove + (int)((0x7fffffffu - kGaugeHigh) >> kGaugeCoarse) < kGaugeBins, "every key has a bin");
// A bin of more than kGaugeList keys is counted again: 2048 sub-bins, and up to 512 values in one of those. On frames of
// at most kGaugeThird pixels every block of gauge_sums_k counts the values from the whole list (L2 holds it); above, that
// would read it 256 times from further away, and a launch of its own counts them once (3.5 us a call where the bin is small).
constexpr int kGaugeSub = 2048, kGaugeSubBits = 11, kGaugeValues = 1 << (kGaugeCoarse - kGaugeSubBits);
constexpr uint32_t kGaugeParts = 16;  // counters a value
constexpr int64_t kGaugeThird = (int64_t)1 << 19;
constexpr int kGaugeHist = kGaugeBins + kGaugeSub + kGaugeValues;

struct GaugeState {
    int32_t valid[2];  // by the round's parity: the frame has a finite solution so far
    uint32_t rank;     // rank of the lower median among the confident pixels' residuals
    uint32_t cursor;   // residuals listed so far by gauge_pick_k
    uint32_t listed;   // all of them: the median's bin
    uint32_t key_lo;   // its first key
    uint32_t bits;     // and its width: 2^bits keys
    uint32_t list_rank;  // rank of the median among the listed
};

__device__ inline int gauge_bin(uint32_t key) {
    const uint32_t d = key - kGaugeLow;
    const uint32_t coarse = key < kGaugeLow ? key >> kGaugeCoarse : kGaugeAbove + ((key - kGaugeHigh) >> kGaugeCoarse);
    return (int)(d < kGaugeHigh - kGaugeLow ? kGaugeBelow + (d >> kGaugeFine) : coarse);
}
// A bin's first key and the bits of its width.
__device__ inline uint32_t gauge_bin_keys(int bin, uint32_t& lo) {
    const bool fine = bin >= kGaugeBelow && bin < kGaugeAbove;
    lo = fine ? kGaugeLow + ((uint32_t)(bin - kGaugeBelow) << kGaugeFine)
              : (bin < kGaugeBelow ? (uint32_t)bin << kGaugeCoarse
                                   : kGaugeHigh + ((uint32_t)(bin - kGaugeAbove) << kGaugeCoarse));
    return fine ? kGaugeFine : kGaugeCoarse;
}

__device__ inline void gauge_range(int64_t N, int nblk, int blk, int64_t& n0, int64_t& n1) {
    n0 = N * blk / nblk;
    n1 = N * (blk + 1) / nblk;
}

// Adds one pixel's terms to a thread's sums: the upper triangle of (A w)^T (A w), then (A w)^T (y w) (products of
// two floats are exact in fp64, so the fused form rounds once, as the sum alone would).
template <int K>
__device__ inline void gauge_add(const float (&a)[kGaugeMaxK], float y, float wn, double* G) {
    constexpr int NG = K * (K + 1) / 2;
    float wa[K];
#pragma unroll
    for (int k = 0; k < K; ++k) wa[k] = a[k] * wn;
    const float wy = y * wn;
    int e = 0;
#pragma unroll
    for (int i = 0; i < K; ++i)
#pragma unroll
        for (int j = i; j < K; ++j, ++e) G[e] = __builtin_fma((double)wa[i], (double)wa[j], G[e]);
#pragma unroll
    for (int i = 0; i < K; ++i) G[NG + i] = __builtin_fma((double)wa[i], (double)wy, G[NG + i]);
    G[NG + K] += 1.0;
}

// A block's sums into its partials (DPP wave scans, then the waves in order).
template <int K>
__device__ inline void gauge_publish(const double* G, double* partials) {
    constexpr int NV = K * (K + 1) / 2 + K + 1;
    __shared__ double s_red[kGaugeBlk / 64][kGaugeVals];
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double v = wave_incl_scan_f64(G[k]);
        if (lane == 63) s_red[wv][k] = v;
    }
    __syncthreads();
    if (tid < NV) {
        double v = 0.0;
        for (int q = 0; q < kGaugeBlk / 64; ++q) v += s_red[q][tid];
        partials[tid] = v;
    }
}

// The frame's system from its nblk partials (eight runs of blocks, then the runs in order) and its solution, in every
// thread of every block alike. Returns whether the frame has a solution (v3.py:174-175: at least 200 confident pixels;
// a finite one) and the count of confident pixels.
template <int K>
__device__ inline bool gauge_solve(const double* partials, int nblk, float (&cf)[kGaugeMaxK], int& count) {
    constexpr int NG = K * (K + 1) / 2, NV = NG + K + 1;
    __shared__ double s_run[8][32];
    __shared__ double s_v[32];
    const int tid = threadIdx.x, val = tid & 31, run = tid >> 5;
    double acc = 0.0;
    if (val < NV) {
#pragma unroll 8
        for (int q = run; q < nblk; q += 8) acc += partials[(int64_t)q * kGaugeVals + val];
    }
    s_run[run][val] = acc;
    __syncthreads();
    if (tid < NV) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < 8; ++q) v += s_run[q][tid];
        s_v[tid] = v;
    }
    __syncthreads();
    count = (int)s_v[NG + K];
    double A[K][K + 1];
    {
        int e = 0;
#pragma unroll
        for (int i = 0; i < K; ++i) {
#pragma unroll
            for (int j = i; j < K; ++j, ++e) A[i][j] = A[j][i] = s_v[e];
            A[i][K] = s_v[NG + i];
        }
    }
    // Gaussian elimination on [G | g], the largest pivot brought up by conditional swaps (registers, no indexing)
    bool ok = count >= kGaugeMinPoints;
    double inv[K];
#pragma unroll
    for (int c = 0; c < K; ++c) {
#pragma unroll
        for (int r = c + 1; r < K; ++r) {
            const bool swap = fabs(A[r][c]) > fabs(A[c][c]);
#pragma unroll
            for (int k = c; k <= K; ++k) {
                const double x = A[c][k], y = A[r][k];
                A[c][k] = swap ? y : x;
                A[r][k] = swap ? x : y;
            }
        }
        ok = ok && fabs(A[c][c]) > 0.0;
        inv[c] = 1.0 / A[c][c];
#pragma unroll
        for (int r = c + 1; r < K; ++r) {
            const double f = A[r][c] * inv[c];
#pragma unroll
            for (int k = c + 1; k <= K; ++k) A[r][k] -= f * A[c][k];
        }
    }
    double x[K];
#pragma unroll
    for (int c = K - 1; c >= 0; --c) {
        double v = A[c][K];
#pragma unroll
        for (int k = c + 1; k < K; ++k) v -= A[c][k] * x[k];
        x[c] = v * inv[c];
    }
#pragma unroll
    for (int k = 0; k < kGaugeMaxK; ++k) {
        cf[k] = k < K ? (float)x[k < K ? k : 0] : 0.0f;
        ok = ok && __builtin_isfinite(cf[k]);
    }
    return ok;
}

template <int K>
__global__ __launch_bounds__(kGaugeBlk) void gauge_inputs_k(const float* __restrict__ depth,
                                                            const float* __restrict__ lidar,
                                                            const float* __restrict__ conf, int H, int W, int h, int w,
                                                            int nblk, float* __restrict__ y_out,
                                                            uint8_t* __restrict__ m_out, uint32_t* __restrict__ hist,
                                                            double* __restrict__ partials) {
    const int b = blockIdx.y, tid = threadIdx.x;
    const int64_t N = (int64_t)h * w, base = (int64_t)b * N;
    for (int i = blockIdx.x * kGaugeBlk + tid; i < kGaugeBins; i += nblk * kGaugeBlk) hist[(int64_t)b * kGaugeHist + i] = 0u;
    int64_t n0, n1;
    gauge_range(N, nblk, blockIdx.x, n0, n1);
    const float* db = depth + (int64_t)b * H * W;
    double G[K * (K + 1) / 2 + K + 1] = {};
    for (int64_t n = n0 + tid; n < n1; n += kGaugeBlk) {
        const int oh = (int)(n / w), ow = (int)(n - (int64_t)oh * w);
        const int r0 = (int)(((int64_t)oh * H) / h), r1 = (int)((((int64_t)oh + 1) * H + h - 1) / h);
        const int c0 = (int)(((int64_t)ow * W) / w), c1 = (int)((((int64_t)ow + 1) * W + w - 1) / w);
        const float ld = lidar[base + n];
        const float cfd = conf ? conf[base + n] : 2.0f;
        float num = 0.0f, den = 0.0f;
        for (int r = r0; r < r1; ++r)
            for (int c = c0; c < c1; ++c) {
                const float d = db[(int64_t)r * W + c];
                const bool ok = __builtin_isfinite(d) && d > 0.0f;
                num = num + (ok ? d : 0.0f);
                den = den + (ok ? 1.0f : 0.0f);
            }
        const float kh = (float)(r1 - r0), kw = (float)(c1 - c0);
        const float nump = num / kh / kw, denp = den / kh / kw;
        const float z = denp > 0.5f ? nump / fmax_(denp, 1e-6f) : 0.0f;
        const float y = log_f32(fmax_(ld, 1e-3f)) - log_f32(fmax_(z, 1e-3f));
        const bool m = cfd >= 2.0f && ld > 0.0f && z > 0.0f;
        y_out[base + n] = y;
        m_out[base + n] = m ? 1 : 0;
        if (m) {
            float a[kGaugeMaxK];
            gauge_basis(linspace_at(ow, w), linspace_at(oh, h), a);
            gauge_add<K>(a, y, 1.0f, G);
        }
    }
    gauge_publish<K>(G, partials + ((int64_t)b * nblk + blockIdx.x) * kGaugeVals);
}

template <int K>
__global__ __launch_bounds__(kGaugeBlk) void gauge_resid_k(int it, const float* __restrict__ y_all,
                                                           const uint8_t* __restrict__ m_all, int h, int w, int nblk,
                                                           const double* __restrict__ partials,
                                                           GaugeState* __restrict__ st, uint32_t* __restrict__ r_all,
                                                           uint32_t* __restrict__ hist) {
    __shared__ uint32_t s_h[kGaugeBins];
    const int b = blockIdx.y, tid = threadIdx.x;
    float c[kGaugeMaxK];
    int count;
    bool ok = gauge_solve<K>(partials + (int64_t)b * nblk * kGaugeVals, nblk, c, count);
    if (it > 0) ok = ok && st[b].valid[(it - 1) & 1] != 0;
    if (blockIdx.x == 0 && tid == 0) {
        st[b].valid[it & 1] = ok ? 1 : 0;
        st[b].rank = ok ? (uint32_t)((count - 1) / 2) : 0u;  // torch.median: the lower middle element
        st[b].cursor = 0u;
    }
    if (!ok) return;
    uint32_t* hg = hist + (int64_t)b * kGaugeHist;
    for (int i = tid; i < kGaugeBins; i += kGaugeBlk) s_h[i] = 0u;
    for (int i = blockIdx.x * kGaugeBlk + tid; i < kGaugeHist - kGaugeBins; i += nblk * kGaugeBlk) hg[kGaugeBins + i] = 0u;
    __syncthreads();
    const int64_t N = (int64_t)h * w, base = (int64_t)b * N;
    int64_t n0, n1;
    gauge_range(N, nblk, blockIdx.x, n0, n1);
    for (int64_t n = n0 + tid; n < n1; n += kGaugeBlk) {
        if (!m_all[base + n]) continue;
        float a[kGaugeMaxK];
        const int iy = (int)(n / w), ix = (int)(n - (int64_t)iy * w);
        gauge_basis(linspace_at(ix, w), linspace_at(iy, h), a);
        float p = 0.0f;
#pragma unroll
        for (int k = 0; k < K; ++k) p = p + a[k] * c[k];
        const uint32_t v = __float_as_uint(fabsf(y_all[base + n] - p));
        r_all[base + n] = v;
        atomicAdd(&s_h[gauge_bin(v)], 1u);
    }
    __syncthreads();
    uint32_t v[kGaugeBins / kGaugeBlk];
#pragma unroll
    for (int k = 0; k < kGaugeBins / kGaugeBlk; ++k) v[k] = s_h[k * kGaugeBlk + tid];
#pragma unroll
    for (int k = 0; k < kGaugeBins / kGaugeBlk; ++k)
        if (v[k]) atomicAdd(&hg[k * kGaugeBlk + tid], v[k]);
}

// The bin holding the rank-th (0-based) of the counted elements, in every thread of the block: its index, the count before
// it and its own (bin 0 of none when the rank lies past their total). `v`: the thread's PER consecutive bins.
template <int PER>
__device__ inline int gauge_find(const uint32_t (&v)[PER], uint32_t rank, uint32_t& before, uint32_t& own) {
    __shared__ uint32_t s_w[kGaugeBlk / 64];
    __shared__ int s_bin;
    __shared__ uint32_t s_before, s_own;
    const int tid = threadIdx.x;
    uint32_t sum = 0u;
#pragma unroll
    for (int k = 0; k < PER; ++k) sum += v[k];
    const uint32_t inc = wave_incl_scan_u32(sum);
    if ((tid & 63) == 63) s_w[tid >> 6] = inc;
    if (tid == 0) {
        s_bin = 0;
        s_before = 0u;
        s_own = 0u;
    }
    __syncthreads();
    uint32_t cum = inc - sum;
    for (int q = 0; q < (tid >> 6); ++q) cum += s_w[q];
    if (cum <= rank && rank < cum + sum) {
        int at = 0;
        uint32_t n = v[0];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const bool past = at == k && cum + v[k] <= rank;
            cum += past ? v[k] : 0u;
            at += past ? 1 : 0;
            n = past && k + 1 < PER ? v[k + 1 < PER ? k + 1 : k] : n;
        }
        s_bin = tid * PER + at;
        s_before = cum;
        s_own = n;
    }
    __syncthreads();
    before = s_before;
    own = s_own;
    const int bin = s_bin;
    __syncthreads();
    return bin;
}

// A frame's list starts at a multiple of 4 words (the counting loads 16 bytes).
__host__ __device__ inline int64_t gauge_list_stride(int64_t N) { return (N + 3) & ~(int64_t)3; }

// Every block: the median's bin. A bin of up to kGaugeList residuals is listed wave by wave; of a larger one (many equal
// residuals, or millions of pixels) a block counts its residuals by sub-bins and takes its part of the list at once.
__global__ __launch_bounds__(kGaugeBlk) void gauge_pick_k(int it, const uint8_t* __restrict__ m_all, int64_t N, int nblk,
                                                          GaugeState* __restrict__ st,
                                                          const uint32_t* __restrict__ r_all,
                                                          uint32_t* __restrict__ hist, uint32_t* __restrict__ list_all) {
    constexpr int PER = kGaugeBins / kGaugeBlk;
    __shared__ uint32_t s_sub[kGaugeSub];
    __shared__ uint32_t s_n, s_at;
    const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    if (!st[b].valid[it & 1]) return;
    uint32_t* hg = hist + (int64_t)b * kGaugeHist;
    const uint32_t rank = st[b].rank;
    uint32_t v[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) v[k] = hg[tid * PER + k];
    uint32_t before, own, lo;
    const int bin = gauge_find(v, rank, before, own);
    const uint32_t bits = gauge_bin_keys(bin, lo), keys = 1u << bits;
    if (blockIdx.x == 0 && tid == 0) {
        st[b].listed = own;
        st[b].key_lo = lo;
        st[b].bits = bits;
        st[b].list_rank = rank - before;
    }
    uint32_t* list = list_all + (int64_t)b * gauge_list_stride(N);
    const int64_t base = (int64_t)b * N;
    int64_t n0, n1;
    gauge_range(N, nblk, blockIdx.x, n0, n1);
    auto key_at = [&](int64_t n) {
        return n + tid < n1 && m_all[base + n + tid] != 0 ? r_all[base + n + tid] : 0xffffffffu;
    };
    const bool many = own > (uint32_t)kGaugeList;
    if (many) {
        for (int i = tid; i < kGaugeSub; i += kGaugeBlk) s_sub[i] = 0u;
        if (tid == 0) s_n = 0u;
        __syncthreads();
        uint32_t mine = 0u;
        for (int64_t n = n0; n < n1; n += kGaugeBlk) {
            const uint32_t d = key_at(n) - lo;
            if (d < keys) {
                atomicAdd(&s_sub[d >> (bits - kGaugeSubBits)], 1u);
                ++mine;
            }
        }
        mine = wave_incl_scan_u32(mine);
        if (lane == 63 && mine) atomicAdd(&s_n, mine);
        __syncthreads();
        if (tid == 0) s_at = s_n ? atomicAdd(&st[b].cursor, s_n) : 0u;
        for (int i = tid; i < kGaugeSub; i += kGaugeBlk)
            if (s_sub[i]) atomicAdd(&hg[kGaugeBins + i], s_sub[i]);
        __syncthreads();
    }
    for (int64_t n = n0; n < n1; n += kGaugeBlk) {  // whole waves: the listed of a wave take one atomic
        const uint32_t key = key_at(n);
        const bool hit = key - lo < keys;
        const uint64_t mask = __ballot(hit);
        if (mask == 0) continue;
        uint32_t at = 0u;
        if (many) {
            if (lane == 0) at = atomicAdd(&s_at, (uint32_t)__popcll(mask));
        } else {
            if (lane == 0) at = atomicAdd(&st[b].cursor, (uint32_t)__popcll(mask));
        }
        at = (uint32_t)__builtin_amdgcn_readlane((int)at, 0);
        if (hit)
            list[at + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] = key;
    }
}

// The median's sub-bin of a bin of many: its first key, the bits of its width, the median's rank in it.
__device__ inline void gauge_sub_bin(const GaugeState& st, const uint32_t* sub, uint32_t& lo, uint32_t& bits,
                                     uint32_t& rank) {
    constexpr int PER = kGaugeSub / kGaugeBlk;
    uint32_t v[PER], before, own;
#pragma unroll
    for (int k = 0; k < PER; ++k) v[k] = sub[threadIdx.x * PER + k];
    const int bin = gauge_find(v, st.list_rank, before, own);
    bits = st.bits - kGaugeSubBits;
    lo = st.key_lo + ((uint32_t)bin << bits);
    rank = st.list_rank - before;
}

// Counts the values key - lo < n among the listed [4 q0, 4 q1) of L, n at most kGaugeValues; the thread's consecutive values
// in v. 16 counters a value, by lane: a large bin's keys are mostly equal, and a wave's atomics to one address run one
// after the other (a round of 307k equal residuals, every block counting all: 160 us by ballots of equal values, 49 this way).
__device__ inline void gauge_count_values(const uint32_t* list, uint32_t q0, uint32_t q1, uint32_t L, uint32_t lo,
                                          uint32_t n, uint32_t* s_h, uint32_t (&v)[kGaugeValues / kGaugeBlk]) {
    constexpr int U = 16;
    const uint32_t tid = threadIdx.x, part = tid & (kGaugeParts - 1);
    const uint4* l4 = (const uint4*)list;
    for (uint32_t i = tid; i < kGaugeValues * kGaugeParts; i += kGaugeBlk) s_h[i] = 0u;
    __syncthreads();
    for (uint32_t q = q0; q < q1; q += kGaugeBlk * U) {
        uint4 x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = q + u * kGaugeBlk + tid;
            x[u] = l4[i < q1 ? i : q1 - 1];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = q + u * kGaugeBlk + tid, left = i < q1 ? L - 4 * i : 0u;  // listed from this word on
            const uint32_t k4[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
#pragma unroll
            for (uint32_t e = 0; e < 4; ++e)
                if (e < left && k4[e] - lo < n) atomicAdd(&s_h[(k4[e] - lo) * kGaugeParts + part], 1u);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kGaugeValues / kGaugeBlk; ++k) {
        v[k] = 0u;
#pragma unroll
        for (uint32_t e = 0; e < kGaugeParts; ++e)
            v[k] += s_h[(tid * (kGaugeValues / kGaugeBlk) + k) * kGaugeParts + ((e + tid) & (kGaugeParts - 1))];
    }
}

__global__ __launch_bounds__(kGaugeBlk) void gauge_third_k(int it, int64_t N, int nblk, const GaugeState* __restrict__ st,
                                                           const uint32_t* __restrict__ list_all,
                                                           uint32_t* __restrict__ hist) {
    constexpr int PV = kGaugeValues / kGaugeBlk;
    __shared__ uint32_t s_h[kGaugeValues * kGaugeParts];
    const int b = blockIdx.y, tid = threadIdx.x;
    const GaugeState s = st[b];
    if (!s.valid[it & 1] || s.listed <= (uint32_t)kGaugeList) return;
    uint32_t* hg = hist + (int64_t)b * kGaugeHist;
    uint32_t lo, bits, rank, v[PV];
    gauge_sub_bin(s, hg + kGaugeBins, lo, bits, rank);
    int64_t q0, q1;
    gauge_range((s.listed + 3) / 4, nblk, blockIdx.x, q0, q1);
    gauge_count_values(list_all + (int64_t)b * gauge_list_stride(N), (uint32_t)q0, (uint32_t)q1, s.listed, lo, 1u << bits,
                       s_h, v);
#pragma unroll
    for (int k = 0; k < PV; ++k)
        if (v[k]) atomicAdd(&hg[kGaugeBins + kGaugeSub + tid * PV + k], v[k]);
}

template <int K>
__global__ __launch_bounds__(kGaugeBlk) void gauge_sums_k(int it, const float* __restrict__ y_all,
                                                          const uint8_t* __restrict__ m_all, int h, int w, int nblk,
                                                          const GaugeState* __restrict__ st,
                                                          const uint32_t* __restrict__ r_all,
                                                          const uint32_t* __restrict__ list_all,
                                                          uint32_t* __restrict__ hist,
                                                          double* __restrict__ partials) {
    constexpr int PER = kGaugeSub / kGaugeBlk;
    __shared__ alignas(16) uint32_t s_mem[kGaugeValues * kGaugeParts];  // the listed keys and a histogram, or the values
    uint32_t* const s_keys = s_mem;
    uint32_t* const s_h = s_mem + kGaugeList;
    static_assert(kGaugeList + kGaugeSub <= kGaugeValues * kGaugeParts, "both fit");
    __shared__ uint32_t s_med;
    const int b = blockIdx.y, tid = threadIdx.x;
    if (!st[b].valid[it & 1]) return;
    uint32_t* hg = hist + (int64_t)b * kGaugeHist;
    for (int i = blockIdx.x * kGaugeBlk + tid; i < kGaugeBins; i += nblk * kGaugeBlk) hg[i] = 0u;
    const int64_t N = (int64_t)h * w, base = (int64_t)b * N;
    // ---- the median among the listed keys (their order in the list varies; the median does not)
    const uint32_t L = st[b].listed, lo = st[b].key_lo;
    uint32_t rank = st[b].list_rank;
    const uint32_t* list = list_all + (int64_t)b * gauge_list_stride(N);
    const bool many = L > (uint32_t)kGaugeList;
    if (!many)
        for (uint32_t i = tid; i < L; i += kGaugeBlk) s_keys[i] = list[i];
    uint32_t med = lo;
    if (L <= (uint32_t)kGaugeBlk) {  // each thread ranks one key against all
        if (tid == 0) s_med = lo;
        const uint32_t L4 = (L + 3u) & ~3u;
        if ((uint32_t)tid >= L && (uint32_t)tid < L4) s_keys[tid] = 0xffffffffu;
        __syncthreads();
        const uint32_t key = (uint32_t)tid < L ? s_keys[tid] : 0xffffffffu;
        uint32_t less = 0u, eq = 0u;
#pragma unroll 4
        for (uint32_t i = 0; i < L4; i += 4) {
            const uint4 q = *(const uint4*)&s_keys[i];
            less += (q.x < key ? 1u : 0u) + (q.y < key ? 1u : 0u) + (q.z < key ? 1u : 0u) + (q.w < key ? 1u : 0u);
            eq += (q.x == key ? 1u : 0u) + (q.y == key ? 1u : 0u) + (q.z == key ? 1u : 0u) + (q.w == key ? 1u : 0u);
        }
        if ((uint32_t)tid < L && less <= rank && rank < less + eq) s_med = key;  // equal keys write equal values
        __syncthreads();
        med = s_med;
    } else if (many) {  // the values of the median's sub-bin
        constexpr int PV = kGaugeValues / kGaugeBlk;
        uint32_t lo2, bits, before, own, v[PV];
        gauge_sub_bin(st[b], hg + kGaugeBins, lo2, bits, rank);
        if (N > kGaugeThird) {
#pragma unroll
            for (int k = 0; k < PV; ++k) v[k] = hg[kGaugeBins + kGaugeSub + tid * PV + k];
        } else {
            gauge_count_values(list, 0u, (L + 3u) / 4u, L, lo2, 1u << bits, s_mem, v);
        }
        med = lo2 + (uint32_t)gauge_find(v, rank, before, own);
    } else {  // radix select over key - lo, 11 bits a pass
        uint32_t prefix = 0u, pmask = 0u;
        for (int top = (int)st[b].bits; top > 0;) {
            const int width = top < 11 ? top : 11, sh = top - width;
            const uint32_t dmask = (1u << width) - 1u;
            __syncthreads();
            for (int i = tid; i < kGaugeSub; i += kGaugeBlk) s_h[i] = 0u;
            __syncthreads();
            for (uint32_t i = tid; i < L; i += kGaugeBlk) {
                const uint32_t k = s_keys[i] - lo;
                if ((k & pmask) == prefix) atomicAdd(&s_h[(k >> sh) & dmask], 1u);
            }
            __syncthreads();
            uint32_t v[PER], before, own;
#pragma unroll
            for (int k = 0; k < PER; ++k) v[k] = s_h[tid * PER + k];
            const int bin = gauge_find(v, rank, before, own);
            prefix |= (uint32_t)bin << sh;
            pmask |= dmask << sh;
            rank -= before;
            top = sh;
        }
        med = lo + prefix;
    }
    const float sc = 1.4826f * __uint_as_float(med) + 1e-4f;
    int64_t n0, n1;
    gauge_range(N, nblk, blockIdx.x, n0, n1);
    double G[K * (K + 1) / 2 + K + 1] = {};
    for (int64_t n = n0 + tid; n < n1; n += kGaugeBlk) {
        if (!m_all[base + n]) continue;
        float a[kGaugeMaxK];
        const int iy = (int)(n / w), ix = (int)(n - (int64_t)iy * w);
        gauge_basis(linspace_at(ix, w), linspace_at(iy, h), a);
        const float wn = fmin_((2.0f * sc) / fmax_(__uint_as_float(r_all[base + n]), 1e-6f), 1.0f);
        gauge_add<K>(a, y_all[base + n], wn, G);
    }
    gauge_publish<K>(G, partials + ((int64_t)b * nblk + blockIdx.x) * kGaugeVals);
}

// Solves the last round's system (each block) and applies it: grid.x blocks walk a frame's pixels.
template <int K>
__global__ __launch_bounds__(kGaugeBlk) void gauge_apply_k(int it, const double* __restrict__ partials, int nblk,
                                                           const GaugeState* __restrict__ st, int H, int W,
                                                           float* __restrict__ coef, float* __restrict__ out) {
    const int b = blockIdx.y, tid = threadIdx.x;
    float c[kGaugeMaxK];
    int count;
    bool ok = gauge_solve<K>(partials + (int64_t)b * nblk * kGaugeVals, nblk, c, count);
    if (it > 0) ok = ok && st[b].valid[(it - 1) & 1] != 0;
    if (blockIdx.x == 0 && tid < 8) coef[b * 8 + tid] = 0.0f;
    if (blockIdx.x == 0 && tid == 0 && ok) {
#pragma unroll
        for (int k = 0; k < K; ++k) coef[b * 8 + k] = c[k];
        coef[b * 8 + 7] = 1.0f;
    }
    const uint32_t plane = (uint32_t)(H * W);  // below 2^31
    float* const ob = out + (int64_t)b * plane;
    for (uint32_t q = blockIdx.x * kGaugeBlk + tid; q < plane; q += gridDim.x * kGaugeBlk) {
        const int i = (int)(q / (uint32_t)W), j = (int)(q - (uint32_t)i * (uint32_t)W);
        float a[kGaugeMaxK];
        gauge_basis(linspace_at(j, W), linspace_at(i, H), a);
        float p = 0.0f;
#pragma unroll
        for (int k = 0; k < K; ++k) p = p + a[k] * c[k];
        ob[q] = ok ? exp_f32(p) : 1.0f;
    }
}

}  // namespace pmg

using namespace pmg;

// Blocks per frame: two pixels a thread up to 256 blocks (every block of the next kernel reads all their partials).
static int gauge_blocks(int64_t N) {
    const int64_t nb = (N + 2 * kGaugeBlk - 1) / (2 * kGaugeBlk);
    return (int)(nb < 1 ? 1 : (nb > kGaugeMaxBlocks ? kGaugeMaxBlocks : nb));
}

template <int K>
static int gauge_run(const float* depth, const float* lidar, const float* conf, int B, int H, int W, int h, int w,
                     int iters, float* y, uint8_t* m, uint32_t* rb, uint32_t* list, double* partials, uint32_t* hist,
                     GaugeState* st, float* coef, float* corr, hipStream_t s) {
    const int nblk = gauge_blocks((int64_t)h * w);
    const dim3 grid((unsigned)nblk, (unsigned)B), blk(kGaugeBlk);
    hipLaunchKernelGGL(gauge_inputs_k<K>, grid, blk, 0, s, depth, lidar, conf, H, W, h, w, nblk, y, m, hist, partials);
    if (int e = check_launch("gauge_inputs_k")) return e;
    for (int it = 0; it + 1 < iters; ++it) {  // (the last round's weights are never used)
        hipLaunchKernelGGL(gauge_resid_k<K>, grid, blk, 0, s, it, y, m, h, w, nblk, partials, st, rb, hist);
        if (int e = check_launch("gauge_resid_k")) return e;
        hipLaunchKernelGGL(gauge_pick_k, grid, blk, 0, s, it, m, (int64_t)h * w, nblk, st, rb, hist, list);
        if (int e = check_launch("gauge_pick_k")) return e;
        if ((int64_t)h * w > kGaugeThird) {
            hipLaunchKernelGGL(gauge_third_k, grid, blk, 0, s, it, (int64_t)h * w, nblk, st, list, hist);
            if (int e = check_launch("gauge_third_k")) return e;
        }
        hipLaunchKernelGGL(gauge_sums_k<K>, grid, blk, 0, s, it, y, m, h, w, nblk, st, rb, list, hist, partials);
        if (int e = check_launch("gauge_sums_k")) return e;
    }
    // every block repeats the solve (2 us), so a frame gets at most 512 blocks, two per CU
    const int64_t na = ((int64_t)H * W + kGaugeBlk - 1) / kGaugeBlk;
    hipLaunchKernelGGL(gauge_apply_k<K>, dim3((unsigned)(na < 512 ? na : 512), (unsigned)B), blk, 0, s, iters - 1,
                       partials, nblk, st, H, W, coef, corr);
    return check_launch("gauge_apply_k");
}

extern "C" {

size_t pmg_gauge_poly_workspace_bytes(int B, int h, int w) {
    if (B < 1 || h < 1 || w < 1) return 0;
    const size_t n = (size_t)B * h * w;
    const int nblk = gauge_blocks((int64_t)h * w);
    const size_t list = (size_t)B * gauge_list_stride((int64_t)h * w);
    return align256(n * 4) + align256(n) + align256(list * 4) + align256(n * 4) +
           align256((size_t)B * nblk * kGaugeVals * sizeof(double)) + align256((size_t)B * kGaugeHist * 4) +
           align256((size_t)B * sizeof(GaugeState));
}

int pmg_gauge_poly(const float* depth, int B, int H, int W, const float* lidar, const float* conf, int h, int w,
                   int degree, int iters, float* corr, float* coef, void* workspace, size_t workspace_bytes,
                   void* stream) {
    PMG_REQUIRE(depth && lidar && corr && coef, "null buffer");
    PMG_REQUIRE(B >= 1 && H >= 1 && W >= 1 && h >= 1 && w >= 1, "bad shape");
    PMG_REQUIRE((int64_t)B * H * W < INT_MAX && (int64_t)B * h * w < INT_MAX && B <= 65535, "map too large");
    PMG_REQUIRE(degree >= 1, "degree must be >= 1");
    PMG_REQUIRE(iters >= 1 && iters <= 64, "iters must be in [1, 64]");
    PMG_REQUIRE(workspace && workspace_bytes >= pmg_gauge_poly_workspace_bytes(B, h, w), "workspace too small");
    hipStream_t s = (hipStream_t)stream;
    const int64_t n_lr = (int64_t)B * h * w;
    const int nblk = gauge_blocks((int64_t)h * w);
    uint8_t* p = (uint8_t*)workspace;
    float* y = (float*)p;
    p += align256((size_t)n_lr * 4);
    uint8_t* m = p;
    p += align256((size_t)n_lr);
    uint32_t* list = (uint32_t*)p;
    p += align256((size_t)B * gauge_list_stride((int64_t)h * w) * 4);
    uint32_t* rb = (uint32_t*)p;
    p += align256((size_t)n_lr * 4);
    double* partials = (double*)p;
    p += align256((size_t)B * nblk * kGaugeVals * sizeof(double));
    uint32_t* hist = (uint32_t*)p;
    p += align256((size_t)B * kGaugeHist * 4);
    GaugeState* st = (GaugeState*)p;
    return degree >= 2 ? gauge_run<6>(depth, lidar, conf, B, H, W, h, w, iters, y, m, rb, list, partials, hist, st, coef,
                                      corr, s)
                       : gauge_run<3>(depth, lidar, conf, B, H, W, h, w, iters, y, m, rb, list, partials, hist, st, coef,
                                      corr, s);
}

}  // extern "C"
