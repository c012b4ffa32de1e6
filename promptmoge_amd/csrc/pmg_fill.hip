// Nearest-valid fill of a LiDAR prompt: promptmoge/model.py:61-72 (nearest_fill).
//
// The reference takes the index map of scipy.ndimage.distance_transform_edt(~valid, return_indices=True): every
// pixel receives the coordinates of the valid pixel nearest in Euclidean distance. Where several valid pixels
// are equally near, that feature transform (a separable pass along axis 0, then along axis 1) keeps the one with
// the smallest column and, within that column, the smallest row. The same result in two passes:
//
//   fill_words_k  one 64-bit validity word per column and 64 rows (bit r = the chunk's row r);
//   fill_row_k    per image row: the nearest valid row F[c] of every column c from its words (ties: the upper row; two bit
//                 scans, further words only across holes of 64 rows and more), kept in LDS; then per pixel the nearest
//                 candidate over the columns of its row -- candidate c sits at (F[c], c) -- searched outward from its
//                 own column, stopping once the column distance alone exceeds the best squared distance. On equal
//                 distances the left candidate (visited first at each radius) wins and the right one loses, which is
//                 the smallest-column rule.
//
// Distances are exact integers, so the result is bit-identical to the reference's for any input. What bounds it: the
// outward search, proportional to the size of the hole around a pixel (a lane waits for the wave's deepest), and the
// latency of one row's chain in a block. With row-major words searched row by row in a pass of its own, which took
// 48-97 us by where the holes lay, a 756x1008 map with 20 % holes and four 64-pixel patches took 75 us; 17 us this way.
#include <climits>

#include "pmg_common.h"

namespace pmg {

constexpr int kFillMaxRows = 8192;
constexpr int kFillMaxCols = 8192;  // one int32 per column of a row in LDS (32 KB)
constexpr int kFillRowThreads = 512;

inline int fill_chunks(int n) { return (n + 63) >> 6; }
inline size_t fill_align(size_t x) { return (x + 255) & ~(size_t)255; }

// grid (ceil(w / 64), ceil(h / 64), B): lane = column, wave k takes rows 16k .. 16k+15 of the 64-row chunk. Bit r of
// words[b][chunk][j] = pixel (64 chunk + r, j) is valid (depth > 0; NaN is not).
__global__ __launch_bounds__(256) void fill_words_k(const float* __restrict__ depth, int h, int w,
                                                    uint64_t* __restrict__ words) {
    __shared__ uint32_t s_part[4][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + lane, jc = j < w ? j : w - 1;
    const int i0 = blockIdx.y * 64 + wv * 16;
    const float* src = depth + (int64_t)blockIdx.z * h * w + jc;
    float d[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) d[r] = src[(int64_t)(i0 + r < h ? i0 + r : h - 1) * w];  // all in flight
    uint32_t bits = 0u;
#pragma unroll
    for (int r = 0; r < 16; ++r) bits |= (i0 + r < h && d[r] > 0.0f) ? 1u << r : 0u;
    s_part[wv][lane] = bits;
    __syncthreads();
    if (wv == 0 && j < w) {
        const uint32_t lo = s_part[0][lane] | (s_part[1][lane] << 16), hi = s_part[2][lane] | (s_part[3][lane] << 16);
        words[((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * w + j] = ((uint64_t)hi << 32) | lo;
    }
}

// grid (h, B): one block per image row.
__global__ __launch_bounds__(kFillRowThreads) void fill_row_k(const float* depth, const float* conf, int h, int w,
                                                              int nchunk, const uint64_t* __restrict__ words,
                                                              float* depth_out, float* conf_out,
                                                              int32_t* __restrict__ src_out) {
    // depth_out / conf_out may alias depth / conf: a pixel writes only its own entries, and every source read is
    // a valid pixel, whose value the write leaves unchanged.
    __shared__ int32_t s_f[kFillMaxCols];
    const int i = blockIdx.x, b = blockIdx.y, nt = blockDim.x;
    const int64_t img = (int64_t)b * h * w;
    const int64_t row = img + (int64_t)i * w;
    const int q = i >> 6, r0 = i & 63;
    const uint64_t* wb = words + (int64_t)b * nchunk * w;
    for (int j = threadIdx.x; j < w; j += nt) {
        const uint64_t m = wb[(int64_t)q * w + j];
        uint64_t up = m & (~0ull >> (63 - r0)), dn = m & (~0ull << r0);  // both hold row i
        int qu = q, qd = q;
        while (up == 0 && qu > 0) up = wb[(int64_t)--qu * w + j];
        const int fu = up ? qu * 64 + 63 - __builtin_clzll(up) : -1;
        // a row below is nearer only within the distance found above
        while (dn == 0 && qd + 1 < nchunk && (fu < 0 || (qd + 1) * 64 - i < i - fu)) dn = wb[(int64_t)++qd * w + j];
        const int fd = dn ? qd * 64 + __builtin_ctzll(dn) : -1;
        s_f[j] = fu >= 0 && (fd < 0 || i - fu <= fd - i) ? fu : fd;
    }
    __syncthreads();
    for (int j = threadIdx.x; j < w; j += nt) {
        const int64_t p = row + j;
        const float own_d = depth[p], own_c = conf_out ? conf[p] : 0.0f;  // in flight during the search
        const int f0 = s_f[j];
        int bc = -1, bd = INT_MAX;
        if (f0 >= 0) {
            bc = j;
            bd = (f0 - i) * (f0 - i);
        }
        // Squared distances are below 2 * 8192^2, so int arithmetic is exact.
        for (int r = 1; bd > 0 && r * r <= bd; ++r) {
            const int cl = j - r, cr = j + r;
            if (cl < 0 && cr >= w) break;
            if (cl >= 0) {
                const int f = s_f[cl];
                if (f >= 0) {
                    const int d2 = (f - i) * (f - i) + r * r;
                    if (d2 <= bd) {  // a tie goes to the smaller column
                        bd = d2;
                        bc = cl;
                    }
                }
            }
            if (cr < w) {
                const int f = s_f[cr];
                if (f >= 0) {
                    const int d2 = (f - i) * (f - i) + r * r;
                    if (d2 < bd) {
                        bd = d2;
                        bc = cr;
                    }
                }
            }
        }
        const bool valid = f0 == i;
        const int src = bc >= 0 ? s_f[bc] * w + bc : -1;
        // A valid pixel is its own source (distance 0); a map with no valid pixel stays as it is.
        const float dv = bc >= 0 && !valid ? depth[img + src] : own_d;
        if (conf_out) conf_out[p] = (valid || bc < 0) ? own_c : 1.0f;
        depth_out[p] = dv;
        if (src_out) src_out[p] = src;
    }
}

}  // namespace pmg

using namespace pmg;

extern "C" {

size_t pmg_nearest_fill_workspace_bytes(int B, int h, int w) {
    if (B < 1 || h < 1 || w < 1) return 0;
    return fill_align((size_t)B * fill_chunks(h) * w * sizeof(uint64_t));
}

int pmg_nearest_fill(const float* depth, const float* conf, int B, int h, int w, float* depth_out, float* conf_out,
                     int32_t* src_index, void* workspace, size_t workspace_bytes, void* stream) {
    PMG_REQUIRE(depth && depth_out && workspace, "null buffer");
    PMG_REQUIRE((conf == nullptr) == (conf_out == nullptr), "conf and conf_out go together");
    PMG_REQUIRE(B >= 1 && B <= 65535 && h >= 1 && w >= 1, "bad shape");
    PMG_REQUIRE(h <= kFillMaxRows && w <= kFillMaxCols, "nearest_fill supports maps up to 8192 x 8192");
    PMG_REQUIRE((int64_t)B * h * w <= INT_MAX, "map too large");
    PMG_REQUIRE(workspace_bytes >= pmg_nearest_fill_workspace_bytes(B, h, w), "workspace too small");
    hipStream_t s = (hipStream_t)stream;
    const int nc = fill_chunks(h);
    uint64_t* words = (uint64_t*)workspace;
    fill_words_k<<<dim3(fill_chunks(w), nc, B), 256, 0, s>>>(depth, h, w, words);
    if (int e = check_launch("fill_words_k")) return e;
    // one pixel per thread up to 512 (a row's chain is latency, not work), then several
    const int nt = w >= kFillRowThreads ? kFillRowThreads : fill_chunks(w) * 64;
    fill_row_k<<<dim3(h, B), nt, 0, s>>>(depth, conf, h, w, nc, words, depth_out, conf_out, src_index);
    return check_launch("fill_row_k");
}

}  // extern "C"
