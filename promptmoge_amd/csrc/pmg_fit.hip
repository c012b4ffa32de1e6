// Robust scale/shift metric fit: fit_scale_shift (moge/model/modules/prompt_stem.py:211-240) on the GPU.
//
//   w = mask; ok = sum(w) >= min_points; k = max(long(fp32(1-trim) * fp32(count)), min_points)
//   repeat iters+1 times:  closed-form weighted LS (s, t) on w (kept only if ok); unless last:
//       r = |s*z + t - target| / max(target, 1e-3) on mask, +inf elsewhere
//       thr = kthvalue(r, min(k, N));  w = mask & (r <= thr)
//
// Design. One persistent kernel per batch item with few, fat blocks (256 threads x 16, 24 or 32 elements by the
// size, held in registers for the whole fit, so HBM is read once): a device-wide barrier costs more the more blocks
// arrive, and a trim round is latency-bound, not bandwidth-bound. Phases are separated by a device-wide barrier of
// per-block flags (fit_barrier). Sums are accumulated in fp64
// (n*sxx - sx^2 cancels badly in fp32) in a fixed order, and every block reduces the published per-block partials
// itself, so all blocks hold bit-identical (s, t) and take identical branches.
//
// The threshold is the exact k-th smallest residual; non-negative fp32 values order like their bit patterns ("keys").
// A trim round costs ONE barrier when the threshold stays inside a bracket [lo, hi] predicted from the previous
// rounds (along the last move's direction half of it, against it a quarter, plus a margin of ~32 expected
// candidates): each block publishes how many of its residuals fall below lo, its fp64 sums over those (they are in
// the new weight set whatever the exact threshold), and its residuals inside the bracket ("candidates", with z and
// target). After the barrier every block loads all candidates into LDS, selects the exact k-th among them (each
// thread ranks one candidate when there are at most 96, else an LDS radix select), and adds the candidates at or
// below it to the sums -- the next (s, t) without a second barrier. When the predicted bracket would hold more than
// ~1500 candidates (large moves), a histogram pass over a window of twice its range goes first (2048 bins of a
// power-of-two width, LDS histogram per block, merged by atomics), and the stage runs on the bin that holds the
// k-th; a bracket that misses is followed by such a window on the side that holds the k-th; round 0 (no threshold yet)
// takes a window over residuals 2^-15 .. 2, and round 1, where the first trim may have dropped the threshold by octaves, a
// window over 16 octaves around round 0's threshold (unless the trim moved little: plan_next). A window that misses is
// followed by radix passes over the whole key range (bins of 2^21 keys, then 2^10 within the first bin, then single
// keys, each only while the bin holds more than 2048 keys); when one key value holds the k-th and more than kCandCap
// elements, it is the threshold and the sums take one more barrier.
// The stage checks that its bracket holds the k-th, so a prediction can cost time but never change a result.
// Once the moves are small, the remaining rounds need no device-wide barrier at all: each block runs them by itself on the
// few elements whose side of the threshold may still change (run_local, in fit_k).
//
// Fixed point: once a round reproduces the previous round's (s, t) bit for bit, every later round would repeat
// it exactly, so the loop stops there with the bit-identical result (on the synthetic scenes after 3 rounds).
// This replaces the reference device engine's approximate two-level histogram (MetricFit.metal:141-189).
//
// Workspace: zero-filled once before its first use; the kernel leaves it reusable (the barrier flags and their
// epoch only grow, histograms are cleared at the start of every launch, everything else is overwritten before it is
// read). A bounded wait that expires (the grid was not co-resident, e.g. another stream held CUs) sets the launch's
// error flag; the launch then completes without waiting, the last block to finish reports the flag in info, writes
// (s, t) = NaN, counts the failure in a sticky word (read by pmg_refiner_check) and returns the barrier state to its
// initial zeros, so the next launch on the workspace starts clean.
#include <climits>
#include <mutex>

#include "pmg_common.h"
#include "pmg_internal.h"

namespace pmg {

constexpr int kFitThreads = 256;
constexpr int kFitWaves = kFitThreads / 64;
constexpr int kFitEPTMax = 32;                         // elements per thread, in registers (16, 24 or 32)
constexpr int kFitPerBlockMax = kFitThreads * kFitEPTMax;  // 8192
constexpr int kFitMaxBlocks = kFitThreads;             // N <= 2^21
constexpr int kFitBins = 2048;
constexpr int kFitHistWords = kFitBins + 64;           // one global histogram: the bins, then 16 below-window counts
constexpr int kFitHistSlots = 6;                       // histogram passes a round can take (window 3 + radix 3)
constexpr int kCandCap = 32768;                        // candidates every block holds in LDS (128 KiB)
constexpr unsigned kStageMax = 2048;                   // a pass bin with more elements is split by another pass
constexpr double kBracketMax = 1536.0;                 // expected candidates above which a window pass goes first
constexpr uint32_t kInvalid = 0xffffffffu;             // residual key of a padding slot (-1: every other key is >= 0)
constexpr int kLocalPer = 32;                          // elements per thread of a local round, in registers
constexpr float kLocalLow = 900.0f;                    // ... and the number below which fewer gain nothing
constexpr unsigned kLocalCap = (unsigned)(kFitThreads * kLocalPer);
constexpr int kFitTraceRounds = 64;
constexpr size_t kFitHeader = 4096;                    // barrier, error flag, trace, completion count
constexpr size_t kFitErrOffset = 64;                   // the launch's error flag
constexpr size_t kFitDoneOffset = 3904;                // finished blocks (after the trace, which ends below 3800)
static_assert(kFitErrSeenOffset == 3968, "pmg_internal.h names the sticky failure count's offset");

struct FitWs {
    unsigned* bar;        // [2]: the synchronisation epoch (the last flag value of the previous launch)
    unsigned* flags;      // [kFitMaxBlocks][16]: each block's arrival count, one 64-byte line per block
    int* err;
    uint32_t* trace;      // block 0's record: per round the selection path | candidates << 4 and the wall clock
                          // (100 MHz) at its end, per round the threshold bits; launch and first-solve times
    unsigned* done;       // blocks of the current launch that have finished (the last one resets it to 0)
    unsigned* err_seen;   // launches whose bounded wait expired since the owner last cleared it (sticky)
    uint64_t* partials;   // [2][kFitMaxBlocks][5] fp64 bit patterns
    unsigned* hist;       // [iters][kFitHistSlots][kFitHistWords]
    uint32_t* exch;       // elements exchanged by a stage, by its parity (FitExchange)
};

// Where the elements that a stage exchanges lie, in words from FitWs::exch, for launches of `cap` = nb x elements per
// block elements: key (residual bits | mask << 31), z and target of a bracket stage's candidates, [nb][elements per
// block] each, or the (z, target) pairs of a local stage's uncertain elements, [nb][elements per block][2]. A block may
// write stage n + 1's while a slower one still reads stage n's (fit_barrier), so the two parities share no word:
// a parity's z and targets, and its pairs, take the same 2 cap words.
struct FitExchange {
    int64_t key, z, t, pairs;
};
__host__ __device__ constexpr FitExchange fit_exchange(int64_t cap, int parity) {
    const int64_t zt = 2 * cap + parity * 2 * cap;
    return {parity * cap, zt, zt + cap, zt};
}

struct FitArgs {
    int mode;  // 0: (z, target, mask) arrays; 1: prompt map (logz, LiDAR, conf); 2: final fit, LiDAR at the map's size
    const float* z;
    const float* tg;
    const uint8_t* mask;
    const float* logz;
    int64_t stride;
    const float* lidar;
    const float* conf;
    int H, W, dh, dw;
    int64_t N;
    int iters;
    float keep;  // fp32(1 - trim)
    int min_points;
    int b;  // batch item
    float* st;
    int32_t* info;
    unsigned spin_limit;  // polls of one barrier wait before it gives up
    int plan_debug;       // test hook: 0, or a deliberately wrong round plan (see pmg_debug_fit_plan)
    FitWs ws;
};

// Device-wide barrier for a fully resident grid, by per-block flags: block b's thread 0 publishes (release, agent
// scope) the barrier's sequence number, with a 32-bit payload, in its own flag line; thread t < nb waits (bounded)
// until block t's flag has reached it, then acquires, and returns block t's payload (0 in other threads). Global
// writes before it are visible after it. Flag values only grow within a launch and across launches (the epoch in
// bar[2]), so a block that is already one barrier ahead still satisfies a late waiter; the flag of an even barrier
// and that of an odd one are separate 64-bit words of the line (sequence number low, payload high, one atomic
// store), and every data buffer exchanged across a barrier is double-buffered, so that block cannot overwrite what
// the late waiter is about to read (a block cannot get two barriers ahead). Half the cost of a central arrival
// counter (no serialised read-modify-write, and every waiter polls one line in parallel with the others); the
// payload carries a stage's candidate counts, which saves the read of them after the barrier.
__device__ inline unsigned fit_barrier(const FitWs& ws, unsigned nb, unsigned want, unsigned spin_limit,
                                       unsigned payload = 0u) {
    __syncthreads();
    uint64_t* const f64 = (uint64_t*)ws.flags;  // 8 words per block's 64-byte line: [0] even barriers, [1] odd
    if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __hip_atomic_store(&f64[blockIdx.x * 8 + (want & 1u)], ((uint64_t)payload << 32) | want, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    unsigned got = 0;
    if (threadIdx.x < nb && __hip_atomic_load(ws.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
        unsigned spins = 0;
        for (;;) {
            const uint64_t v =
                __hip_atomic_load(&f64[threadIdx.x * 8 + (want & 1u)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((int)((unsigned)v - want) >= 0) {
                got = (unsigned)(v >> 32);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            if (++spins > spin_limit) {
                __hip_atomic_store(ws.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    return got;
}

// Fixed-order block reduction of 5 doubles (DPP wave scans, then waves in order); result in every thread.
__device__ inline void block_sum5(double (&v)[5], double (*red)[kFitWaves]) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        v[k] = wave_incl_scan_f64(v[k]);
        if (lane == 63) red[k][w] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        double s = red[k][0];
        for (int q = 1; q < kFitWaves; ++q) s += red[k][q];
        v[k] = s;
    }
    __syncthreads();
}

// Exclusive scan of one unsigned per thread over the block; also returns the block total.
__device__ inline unsigned block_excl_scan(unsigned v, unsigned* tmp, unsigned& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned inc = wave_incl_scan_u32(v);
    if (lane == 63) tmp[w] = inc;
    __syncthreads();
    unsigned before = 0;
    total = 0;
    for (int k = 0; k < kFitWaves; ++k) {
        before += k < w ? tmp[k] : 0u;
        total += tmp[k];
    }
    __syncthreads();
    return before + inc - v;
}

// Two exclusive scans in one pass (returns a's exclusive prefix; totals of a and b).
__device__ inline unsigned block_excl_scan2(unsigned a, unsigned b, uint2* tmp, unsigned& ta, unsigned& tb) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned ia = wave_incl_scan_u32(a), ib = wave_incl_scan_u32(b);
    if (lane == 63) tmp[w] = make_uint2(ia, ib);
    __syncthreads();
    unsigned before = 0;
    ta = 0;
    tb = 0;
    for (int k = 0; k < kFitWaves; ++k) {
        const uint2 q = tmp[k];
        before += k < w ? q.x : 0u;
        ta += q.x;
        tb += q.y;
    }
    __syncthreads();
    return before + ia - a;
}

// Phase timestamps of block 0 (100 MHz wall clock) into the workspace header, for profiling the selection phases;
// compiled in with -DPMG_FIT_PHASE_TRACE.
#ifdef PMG_FIT_PHASE_TRACE
#define FIT_MARK(k)                                                                                      \
    do {                                                                                                 \
        if (b == 0 && tid == 0 && it < 32) ws.trace[256 + it * 8 + (k)] = (uint32_t)wall_clock64();     \
    } while (0)
#define FIT_MARK0(k)                                                                                     \
    do {                                                                                                 \
        if (b == 0 && tid == 0) ws.trace[900 + (k)] = (uint32_t)wall_clock64();                          \
    } while (0)
#else
#define FIT_MARK(k) \
    do {            \
    } while (0)
#define FIT_MARK0(k) \
    do {             \
    } while (0)
#endif
struct FitShared {
    unsigned hist[kFitBins];
    alignas(16) uint32_t cand[kCandCap];
    unsigned off[kFitMaxBlocks + 1];
    double red[5][kFitWaves];
    unsigned tmp[kFitWaves];
    uint2 tmp2[kFitWaves];
    alignas(16) unsigned cnt[2][2][kFitWaves];  // a local round's counts, alternating
    float s, t;
    long long kk;
    int ok;
    unsigned bin, below;
    unsigned bincnt, hbelow;  // elements in the found bin; this block's keys below a pass window
    int found;                // find_bin found the rank in the histogram
    unsigned total_below, total_cand;
    uint32_t blo_last, bhi_last;  // bracket of the last stage
    int last;                     // this block is the launch's last one to finish
};

// Finds, in a 2048-bin histogram whose bins follow `base` smaller elements, the bin holding the rank-th element
// (1-based); sets sh.bin, sh.below (the count before it, base included), sh.bincnt (the bin's count) and sh.found
// (0 when the rank-th element lies below the bins or above them). The bins are read through `load` and base
// through `load_base`, all in one round trip.
template <class Load, class LoadBase>
__device__ inline void find_bin(FitShared& sh, unsigned rank, Load load, LoadBase load_base) {
    constexpr int per = kFitBins / kFitThreads;  // 8 consecutive bins per thread
    unsigned cnt[per];
    unsigned local = 0;
    const unsigned base = load_base();
#pragma unroll
    for (int e = 0; e < per; ++e) {
        cnt[e] = load(threadIdx.x * per + e);
        local += cnt[e];
    }
    if (threadIdx.x == 0) {
        sh.bin = 0;
        sh.below = 0;
        sh.bincnt = 0;
        sh.found = 0;
    }
    unsigned total;
    const unsigned excl = block_excl_scan(local, sh.tmp, total) + base;
    if (excl < rank && rank <= excl + local) {
        unsigned cum = excl;
#pragma unroll
        for (int e = 0; e < per; ++e) {
            if (cum + cnt[e] >= rank) {
                sh.bin = (unsigned)(threadIdx.x * per + e);
                sh.below = cum;
                sh.bincnt = cnt[e];
                sh.found = 1;
                break;
            }
            cum += cnt[e];
        }
    }
    __syncthreads();
}

// A box of trim-round states around (s, t, thr): |s' - s| <= Ds, |u' - u| <= Du with u = s zc + t (the line's value at
// the mean z, which moves far less than t does), |thr' - thr| <= Dt.
struct FitBox {
    float s, t, thr, zc, Ds, Du, Dt;
    float sm, tm;  // the largest |s'| and |t'| of its states (fit_box_bounds)
};
__host__ __device__ inline void fit_box_bounds(FitBox& q) {
    q.sm = __builtin_fabsf(q.s) + q.Ds;
    q.tm = __builtin_fabsf(q.t) + q.Ds * __builtin_fabsf(q.zc) + q.Du;
}
// Whether an element's residual is below the threshold in every state of the box (`below` all ones), or above it
// (`above` all ones), or may be either (both 0; also for NaN). |s' z + t' - tg| moves by at most Ds |z - zc| + Du, the
// threshold by Dt; the residual's fp32 evaluation, here and in every later round, is off by at most
// 2^-24 (3 |s' z| + 2 |t'| + |tg|) before the division and 2^-24 relative after it, and 2e-6 of the magnitudes covers both
// evaluations four times over -- the magnitudes at the box's far end: few elements allow boxes of many times |s|, whose
// states round far more coarsely than the middle one (with the middle's magnitudes, boxes of 1000 |s| misplaced elements). The two tests are sign bits, not conditions: a condition combined with another goes
// through the scalar unit, and each such hop stalls a lone wave for ~25 cycles (measured: a ballot and its count 28
// cycles, a vector operation 5), which made these per-element loops three times longer.
__host__ __device__ inline void fit_class(const FitBox& q, float z, float tg, int& below, int& above) {
    const float e = (q.s * z + q.t) - tg;
    const float dm = __builtin_fmaxf(tg, 1e-3f);
    const float m = q.Ds * __builtin_fabsf(z - q.zc) + q.Du + q.Dt * dm +
                    (2e-6f * (q.sm * __builtin_fabsf(z) + q.tm + __builtin_fabsf(tg)) + 1e-30f);
    const float x = __builtin_fabsf(e) - q.thr * dm;
    below = (int)f2u(__builtin_fminf(x + m, 1e30f)) >> 31;  // (the minimum of a NaN and 1e30 is 1e30)
    above = (int)f2u(__builtin_fminf(m - x, 1e30f)) >> 31;
}
// A condition as a word (-1 or 0) that the compiler keeps in a vector register.
__device__ inline int word(bool c) {
    int m = c ? -1 : 0;
    asm("" : "+v"(m));
    return m;
}
__device__ inline float masked(float x, int mask) { return u2f(f2u(x) & (uint32_t)mask); }

// RN(1 / d) for the residuals' division, d >= 1e-3: the hardware reciprocal (1 ulp) and two Newton steps. Not exact for a
// significand of all ones (and for d so large that 1 / d is denormal): fit_keys divides there.
__device__ inline float fit_rcp(float d) {
    float y = __builtin_amdgcn_rcpf(d);
    y = __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
    return __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
}
// The keys of N elements: |((s z) + t) - tg| / max(tg, 1e-3) as ordered bits, the one operation order of every round. The
// quotient e / d is formed from y = RN(1 / d), kept per element: q0 = e y is within 2 ulp, one correction by the exact
// remainder makes it faithful, and a second gives the correctly rounded quotient (Markstein's theorem: y correctly
// rounded, q faithful, r = e - q d by fused multiply-add, then RN(q + r y) = RN(e / d)). The compiler's own division
// sequence is bit-identical, but passes a scale flag through VCC, so the N divisions ran one after the other: 16 elements
// took 1.9 us of a round, 1.5 us this way with their masks. Operands outside the theorem's range (under- or overflow, all-ones divisors)
// take the plain division, one branch for all N. Keys are below 2^31 (a NaN's sign is dropped): the loops compare them as
// signed numbers, and a NaN orders above every number.
template <int N>
__device__ inline void fit_keys(float s, float t, const float* z, const float* tg, const float* rc, bool odd_targets,
                                uint32_t* key) {
    uint32_t emin = 0xffffffffu, emax = 0u;  // of e's bits - 1 (0 stands aside), of e's bits
#pragma unroll
    for (int j = 0; j < N; ++j) {
        float e = s * z[j];
        e = e + t;
        e = __builtin_fabsf(e - tg[j]);
        const float d = fmax_(tg[j], 1e-3f), y = rc[j];
        float q = e * y;
        q = __builtin_fmaf(__builtin_fmaf(-q, d, e), y, q);
        q = __builtin_fmaf(__builtin_fmaf(-q, d, e), y, q);
        key[j] = f2u(q);
        const uint32_t eb = f2u(e);
        emin = eb - 1u < emin ? eb - 1u : emin;
        emax = eb > emax ? eb : emax;
    }
    if (__any(odd_targets || emin < f2u(0x1p-60f) || emax > f2u(0x1p60f))) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            float e = s * z[j];
            e = e + t;
            e = e - tg[j];
            key[j] = f2u(__builtin_fabsf(e) / fmax_(tg[j], 1e-3f)) & 0x7fffffffu;  // (inf / inf is -NaN)
        }
    }
}
// A target whose reciprocal fit_rcp may not round correctly, or whose quotients may leave the theorem's range.
__device__ inline bool fit_odd_target(float tg) {
    const float d = fmax_(tg, 1e-3f);
    return !(d < 0x1p60f) || (~f2u(d) & 0x7fffffu) == 0u;
}

__device__ inline uint32_t wave_max_u32(uint32_t v) {
    uint32_t o;
    o = dpp_u32<0x111, 0xf>(v);
    v = o > v ? o : v;
    o = dpp_u32<0x112, 0xf>(v);
    v = o > v ? o : v;
    o = dpp_u32<0x114, 0xf>(v);
    v = o > v ? o : v;
    o = dpp_u32<0x118, 0xf>(v);
    v = o > v ? o : v;
    o = dpp_u32<0x142, 0xa>(v);
    v = o > v ? o : v;
    o = dpp_u32<0x143, 0xc>(v);
    v = o > v ? o : v;
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

template <int kFitEPT>
__global__ __launch_bounds__(kFitThreads) void fit_k(FitArgs a) {
    constexpr int kFitPerBlock = kFitThreads * kFitEPT;
    static_assert(kFitEPT <= 32, "element masks are 32-bit");
    __shared__ FitShared sh;
    const int nb = (int)gridDim.x, b = (int)blockIdx.x, tid = (int)threadIdx.x;
    const FitWs& ws = a.ws;
    const int64_t cap_words = (int64_t)nb * kFitPerBlock;
    // barrier sequence numbers continue from the previous launch's last one (every block performs the same
    // barriers; block 0 advances the epoch when it is done, after every block has read it here)
    unsigned sync_seq = __hip_atomic_load(&ws.bar[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    if (b == 0 && tid == 0) ws.trace[2 * kFitTraceRounds + 1] = (uint32_t)wall_clock64();  // launch start
    // clear this launch's global histograms; the first barrier orders this before any use
    {
        const int64_t words = (int64_t)(a.iters > 0 ? a.iters : 1) * kFitHistSlots * kFitHistWords;
        for (int64_t q = (int64_t)b * kFitThreads + tid; q < words; q += (int64_t)nb * kFitThreads) ws.hist[q] = 0u;
    }

    // ---- elements into registers: every load of the thread is issued before any is used
    float zr[kFitEPT], tr[kFitEPT];
    uint32_t mbits = 0, vbits = 0;
    {
        const uint32_t i0 = (uint32_t)b * kFitPerBlock + tid;  // N <= 2^21
#pragma unroll
        for (int j = 0; j < kFitEPT; ++j)
            if ((int64_t)i0 + j * kFitThreads < a.N) vbits |= 1u << j;
        // Loads are unconditional (padding slots read the last element) so that none sits under a branch: a
        // branch would make the compiler wait for each element's load before the next one is issued.
        const int64_t last = a.N - 1;
        if (a.mode == 0) {
            uint8_t mk[kFitEPT];
            const int64_t o0 = (int64_t)a.b * a.N;
#pragma unroll
            for (int j = 0; j < kFitEPT; ++j) {
                int64_t i = (int64_t)i0 + j * kFitThreads;
                i = i < last ? i : last;
                zr[j] = a.z[o0 + i];
                tr[j] = a.tg[o0 + i];
                mk[j] = a.mask[o0 + i];
            }
#pragma unroll
            for (int j = 0; j < kFitEPT; ++j) mbits |= (uint32_t)word(mk[j] != 0) & vbits & (1u << j);
        } else if (a.mode == 2) {
            // the final fit on a LiDAR map of the depth map's own size (v3.py:768-775): every area window is one
            // pixel, so the pooled depth is exp(logz) itself (0 + z and z / 1 / 1 are exact) and the mask is
            // conf >= 2 & lidar > 0 & z > 0 (& mask_binary), as final_inputs_k forms them for larger windows
            const int64_t o0 = (int64_t)a.b * a.N;
            float lc[kFitEPT];
            uint8_t mb[kFitEPT];
#pragma unroll
            for (int j = 0; j < kFitEPT; ++j) {
                int64_t i = (int64_t)i0 + j * kFitThreads;
                i = i < last ? i : last;
                zr[j] = a.logz[(o0 + i) * a.stride];
                tr[j] = a.lidar[o0 + i];
                lc[j] = a.conf[o0 + i];
                mb[j] = a.mask ? a.mask[o0 + i] : (uint8_t)1;
            }
#pragma unroll
            for (int j = 0; j < kFitEPT; ++j) {
                zr[j] = exp_f32(zr[j]);
                mbits |= (uint32_t)(word(lc[j] >= 2.0f) & word(tr[j] > 0.0f) & word(zr[j] > 0.0f) & word(mb[j] != 0)) &
                         vbits & (1u << j);
            }
        } else {
            // v3.py:373-378: z = exp(logz); nearest LiDAR sample (F.interpolate's index rule); mask = valid & c >= 0.999
            const uint32_t W = (uint32_t)a.W;
            const float scy = (float)a.dh / (float)a.H, scx = (float)a.dw / (float)a.W;
            float lc[kFitEPT];
#pragma unroll
            for (int j = 0; j < kFitEPT; ++j) {
                int64_t i = (int64_t)i0 + j * kFitThreads;
                i = i < last ? i : last;
                const uint32_t ij = (uint32_t)i;
                const uint32_t row = ij / W, col = ij - row * W;  // branch-free 32-bit division
                int sy = (int)__builtin_floorf((float)row * scy);
                int sx = (int)__builtin_floorf((float)col * scx);
                sy = sy < a.dh - 1 ? sy : a.dh - 1;
                sx = sx < a.dw - 1 ? sx : a.dw - 1;
                const int64_t p = ((int64_t)a.b * a.dh + sy) * a.dw + sx;
                zr[j] = a.logz[((int64_t)a.b * a.N + i) * a.stride];
                tr[j] = a.lidar[p];
                lc[j] = a.conf[p];
            }
#pragma unroll
            for (int j = 0; j < kFitEPT; ++j) {
                // finite and positive: bits in [1, 0x7f7fffff]; clamp(conf / 2, 0, 1) >= 0.999: conf / 2 >= 0.999
                zr[j] = exp_f32(zr[j]);
                mbits |= (uint32_t)(word(f2u(tr[j]) - 1u < 0x7f7fffffu) & word(lc[j] * 0.5f >= 0.999f)) & vbits & (1u << j);
            }
        }
#pragma unroll
        for (int j = 0; j < kFitEPT; ++j) {  // padding slots hold zeros
            const int v = (int)(vbits << (31 - j)) >> 31;
            zr[j] = masked(zr[j], v);
            tr[j] = masked(tr[j], v);
        }
    }
    float ir[kFitEPT];  // 1 / max(target, 1e-3)
#pragma unroll
    for (int j = 0; j < kFitEPT; ++j) ir[j] = fit_rcp(fmax_(tr[j], 1e-3f));
    bool odd = false;
#pragma unroll
    for (int j = 0; j < kFitEPT; ++j) odd = odd || fit_odd_target(tr[j]);
    const int npad = kFitEPT - __popc(vbits);  // padding slots: their key is negative, so the loops count them below

    int stage = 0;  // publish buffers alternate between consecutive publishes
    // Publishes this block's fp64 sums into buffer `stage & 1` (a bracket stage's counts ride on its barrier).
    auto publish = [&](double (&v)[5]) {
        block_sum5(v, sh.red);
        if (tid == 0) {
            uint64_t* p = ws.partials + ((size_t)(stage & 1) * kFitMaxBlocks + b) * 5;
#pragma unroll
            for (int k = 0; k < 5; ++k) p[k] = __builtin_bit_cast(uint64_t, v[k]);
        }
    };
    // Sum of all blocks' published partials of buffer `stage & 1`, in block order, in every thread.
    auto gather_partials = [&](double (&g)[5]) {
#pragma unroll
        for (int k = 0; k < 5; ++k) g[k] = 0.0;
        if (tid < nb) {
            const uint64_t* p = ws.partials + ((size_t)(stage & 1) * kFitMaxBlocks + tid) * 5;
#pragma unroll
            for (int k = 0; k < 5; ++k)
                g[k] = __builtin_bit_cast(double, __hip_atomic_load(&p[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        }
        block_sum5(g, sh.red);
    };
    double pp[5];  // this thread's share of the published partials (threads < nb), loaded right after a barrier
    auto load_partials = [&]() {
#pragma unroll
        for (int k = 0; k < 5; ++k) pp[k] = 0.0;
        if (tid < nb) {
            const uint64_t* p = ws.partials + ((size_t)(stage & 1) * kFitMaxBlocks + tid) * 5;
#pragma unroll
            for (int k = 0; k < 5; ++k)
                pp[k] = __builtin_bit_cast(double, __hip_atomic_load(&p[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        }
    };
    float s = 1.0f, t = 0.0f;
    float s_last = 1.0f, t_last = 0.0f;  // (s, t) before the last solve
    bool same = false;  // the last solve reproduced the previous (s, t) bit for bit
    // Closed-form weighted LS on the global sums (prompt_stem.py:222-232). The first solve: thread 0 also decides
    // the fallback and k, all threads read. Later solves: every thread holds the same sums (fixed-order block
    // reductions), so each computes the same (s, t) with the same fp64 operations and no broadcast is needed.
    auto ls = [&](const double (&g)[5], bool ok, float& ns, float& nt) {
        const double n = g[0], sx = g[1], sy = g[2], sxx = g[3], sxy = g[4];
        const double nn = n > 1.0 ? n : 1.0;
        const double den = nn * sxx - sx * sx;
        const double sn = den > 1e-12 ? (nn * sxy - sx * sy) / (den > 1e-12 ? den : 1e-12) : 1.0;
        const double tn = (sy - sn * sx) / nn;
        ns = s;
        nt = t;
        if (ok) {
            ns = (float)sn;
            nt = (float)tn;
        }
    };
    auto solve = [&](const double (&g)[5], bool first) {
        if (!first) {
            float ns, nt;
            ls(g, sh.ok != 0, ns, nt);
            same = f2u(ns) == f2u(s) && f2u(nt) == f2u(t);
            s_last = s;
            t_last = t;
            s = ns;
            t = nt;
            return;
        }
        if (tid == 0) {
            const int64_t count = (int64_t)g[0];
            sh.ok = count >= a.min_points;
            int64_t k = (int64_t)(a.keep * (float)count);
            if (k < a.min_points) k = a.min_points;
            sh.kk = k < a.N ? k : a.N;
            if (a.info && b == 0) {
                a.info[5 * a.b + 0] = (int32_t)count;
                a.info[5 * a.b + 1] = (int32_t)k;
                a.info[5 * a.b + 2] = sh.ok;
            }
            float ns, nt;
            ls(g, sh.ok != 0, ns, nt);
            sh.s = ns;
            sh.t = nt;
        }
        __syncthreads();
        same = false;
        s = sh.s;
        t = sh.t;
        __syncthreads();
    };

    // ---- round 0 weights: the mask
    float zc = 0.0f, zsd = 0.0f, itg = 0.0f;  // mean z, its standard deviation, 1 / mean target (local rounds' plan)
    {
        double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < kFitEPT; ++j) {
            const int m = (int)(mbits << (31 - j)) >> 31;
            const double zd = masked(zr[j], m), td = masked(tr[j], m);
            v[1] += zd;
            v[2] += td;
            v[3] = __builtin_fma(zd, zd, v[3]);
            v[4] = __builtin_fma(zd, td, v[4]);
        }
        v[0] = (double)__popc(mbits);
        FIT_MARK0(0);
        publish(v);
        FIT_MARK0(1);
        fit_barrier(ws, nb, ++sync_seq, a.spin_limit);
        FIT_MARK0(2);
        double g[5];
        gather_partials(g);
        ++stage;
        const float rn = 1.0f / fmax_((float)g[0], 1.0f);
        zc = (float)g[1] * rn;
        zsd = __builtin_sqrtf(fmax_((float)g[3] * rn - zc * zc, 0.0f));
        itg = (float)g[0] / fmax_((float)g[2], 1e-30f);
        solve(g, true);
    }

    if (b == 0 && tid == 0) ws.trace[2 * kFitTraceRounds] = (uint32_t)wall_clock64();  // initial solve done
    if (tid == 0) {  // the last stage's record, read by the next round's plan before any stage has run
        sh.total_cand = 0;
        sh.blo_last = 0;
        sh.bhi_last = 0;
    }
    __syncthreads();
    uint32_t thr = 0, thr_prev = 0;
    bool have_prev = false;
    // the next round's plan (see its computation at the end of a round): mode, bracket, window. Round 0 has no
    // threshold to start from: a window over relative residuals 2^-15 .. 2 in bins of 1/128 octave, one pass where
    // the radix passes take two (round 0 at 480x640: 22.4 -> 17 us); a threshold outside it takes the radix passes.
    int plan_mode = 1, plan_wsh = 16;
    uint32_t lo = 0, hi = 0, plan_wlo = (127u - 15u) << 23;
    if (a.plan_debug == 2) {
        plan_wlo = 0x7f800001u;
        plan_wsh = 0;
    }
    float dens = 0.0f;  // candidates per key near the threshold, from the last stage with enough of them
    // local rounds: the last moves of (s, u, thr) and their decayed magnitudes, elements per unit of residual near the
    // threshold, and how often a plan of theirs has failed
    float ds = 0.0f, du = 0.0f, dt = 0.0f, mv_s = 0.0f, mv_u = 0.0f, mv_t = 0.0f, dens_r = 0.0f;
    int local_fails = (a.plan_debug == 2 || a.plan_debug == 3) ? 2 : 0;
    FitBox box{};
    // A mean displacement of the residuals over a box, relative to the target: what the number of uncertain elements is
    // proportional to.
    auto box_width = [&](float Ds, float Du, float Dt) { return 1.2f * (Ds * zsd + Du) * itg + Dt; };
    // Notes the moves of the round that gave the current (s, t) and thr.
    auto note_moves = [&](bool have) {
        const float fthr = u2f(thr);
        ds = s - s_last;
        du = ds * zc + (t - t_last);
        dt = have ? fthr - u2f(thr_prev) : 0.0f;
        mv_s = fmax_(__builtin_fabsf(ds), 0.5f * mv_s);
        mv_u = fmax_(__builtin_fabsf(du), 0.5f * mv_u);
        mv_t = fmax_(fmax_(__builtin_fabsf(dt), 0.5f * mv_t), 1e-4f * fthr);
    };
    // The box for the rounds ahead. The moves keep their direction while they are large and shrink to a jitter, so the
    // box reaches 0.8 c times the last move along it, and 0.3 c times the decayed magnitudes to either side; after round 0,
    // which has no move of the threshold to go by, +-0.8 % of it (only where plan_next expects it to stay within). c as large as
    // `target` uncertain elements allow, in [cmin, cmax] (above cmax while they are under kLocalLow: a wide box costs nothing
    // there); false if that is not to be had (or nothing finite can be said).
    auto plan_box = [&](bool have, float target, float cmin, float cmax) -> bool {
        const float fthr = u2f(thr);
        const float ws1 = 0.4f * __builtin_fabsf(ds) + 0.3f * mv_s, wu1 = 0.4f * __builtin_fabsf(du) + 0.3f * mv_u;
        const float wt1 = have ? 0.4f * __builtin_fabsf(dt) + 0.8f * mv_t : 0.0f, wt0 = have ? 0.0f : 8e-3f * fthr;
        const float u1 = 2.0f * box_width(ws1, wu1, wt1) * dens_r;
        float c = (target - 2.0f * wt0 * dens_r) * __builtin_amdgcn_rcpf(fmax_(u1, 1e-20f));
        const float cl = fmax_(cmax, kLocalLow * __builtin_amdgcn_rcpf(fmax_(u1, 1e-20f)));
        c = c < cl ? c : cl;
        if (!(c >= cmin && u1 < 1e30f && fthr < 1e12f && dens_r > 0.0f && __builtin_fabsf(s) < 1e12f &&
              __builtin_fabsf(t) < 1e12f))
            return false;
        box.s = s + 0.4f * c * ds;
        box.t = (s * zc + t + 0.4f * c * du) - box.s * zc;
        box.thr = have ? fthr + 0.4f * c * dt : fthr;
        box.zc = zc;
        box.Ds = c * ws1 + 1e-6f * __builtin_fabsf(s);
        box.Du = c * wu1 + 1e-6f * (__builtin_fabsf(s * zc) + __builtin_fabsf(t) + __builtin_fabsf(box.s * zc) +
                                    __builtin_fabsf(box.t));  // (the rounding of box.t: the current state is inside)
        box.Dt = c * wt1 + wt0;
        fit_box_bounds(box);
        return box.tm < 1e12f && box.thr + box.Dt < 1e15f;  // (below run_local's padding elements at every state)
    };
    // Whether the current (s, t) lies in the box (1e-4 of it is kept for the margins' own rounding): what a classification
    // over the box says of the current residuals holds only then. plan_box puts it there, its own rounding included, so
    // that a narrower box planned within a series is not tested (the fp64 test there spilled registers); a test hook may not.
    auto in_box = [&]() -> bool {
        const double du_now = ((double)s * zc + t) - ((double)box.s * zc + box.t);
        return fabs((double)s - box.s) <= 0.9999 * box.Ds && fabs(du_now) <= 0.9999 * box.Du;
    };
    bool use_local = false;  // the next round runs locally (box); the plan above is then its fallback
    auto plan_next = [&]() {
        // ---- the next round's plan. The threshold's move from round to round (in keys, which order like the
        // values) shrinks by 2-5x per round on the refined maps, keeps its sign while it is large, and jitters by
        // ~10^3 keys near the fixed point. The bracket reaches a quarter of the last move against it and half a move
        // along it, plus a margin of at least 2048 keys and ~32 expected candidates; when that bracket would hold
        // more than kBracketMax candidates at the density the stages saw (candidates per key, kept from the last
        // stage with at least 64), a window pass over twice that range goes first, its bins sized for 2048 over the
        // range. A move of more than an octave is the first trim dropping the outliers of an exact point map: the
        // next round usually repeats the threshold, so the bracket is ~256 expected candidates around it.
        // (heuristics only, in fp32 with the hardware reciprocal: the plan never changes a result)
        if (sh.total_cand >= 64u || dens <= 0.0f)
            dens = (float)sh.total_cand * __builtin_amdgcn_rcpf((float)(sh.bhi_last - sh.blo_last) + 1.0f);
        plan_mode = 2;
        // After round 0: whether the first trim leaves the threshold within 0.8 %, from the mean move of the residuals that it
        // caused. Seen (fits of synthetic rooms, 96x128 to 480x640): moves of up to 0.12 thresholds and under 0.016 go with
        // threshold moves of 0 to 0.8 % (5 mm noise) and 0.6 % (half the targets outliers), larger ones with 2.6 to 3.5 %
        // (20 % noise), 12 to 14 % (a bent map) and 33 % (unrelated targets); maps that one refiner step made: -1.5 % (A, passes
        // and misses), -2.4 % (T) and +10 % (H, both refused). A local series that fails at once costs 6 to 10 us, a missed
        // bracket 5: 192x256, four rounds, 20 % noise 92 us, unrelated targets 74; refused 75 and 62.
        const float first = box_width(mv_s, mv_u, 0.0f);
        const bool steady = have_prev || (first < 0.125f * u2f(thr) && first < 0.016f);
        if (!have_prev && steady && sh.total_cand >= 64u &&
            dens * 0.016f * (float)((thr & 0x7fffffu) | 0x800000u) < 4000.0f) {
            // a bracket of +-0.8 % (13 us at 480x640 against 20 by the window; 24 where it misses and the window follows)
            plan_mode = 0;
            lo = f2u(0.992f * u2f(thr));
            hi = f2u(1.008f * u2f(thr));
            plan_wsh = 16;
        } else if (!have_prev) {
            // after round 0: the first trim drops the outliers' pull, and the threshold falls by up to ~11 octaves
            // (exact point maps) or moves by under one (noisy ones); a window from 14 octaves below to 2 above it
            // in 2048 bins of 2^16 keys (1/128 octave) holds it
            plan_mode = 1;
            plan_wsh = 16;
            plan_wlo = thr > (14u << 23) ? thr - (14u << 23) : 0u;
        } else {
            // keys are below 2^31 (non-negative floats, NaN included), so every range here fits 32 bits
            const bool up = thr >= thr_prev;
            const uint32_t am = up ? thr - thr_prev : thr_prev - thr;
            const float rdens = dens > 0.0f ? __builtin_amdgcn_rcpf(dens) : 0.0f;
            auto keys_for = [&](float cands) {  // keys that hold about `cands` candidates, in [2048, 2^18]
                const float k = dens > 0.0f ? cands * rdens : 2048.0f;
                return (uint32_t)(k < 2048.0f ? 2048.0f : (k > 262144.0f ? 262144.0f : k));
            };
            const bool jump = am > (1u << 23);  // a jump of over an octave predicts no move
            uint32_t along = am / 2 + keys_for(32.0f), against = am / 4 + keys_for(32.0f);
            if (jump) along = against = keys_for(128.0f);
            const float expect = dens * ((float)(along + against) + 1.0f);
            const uint32_t dn = up ? against : along, dp = up ? along : against;
            if (expect <= kBracketMax || jump) {
                plan_mode = 0;
                lo = thr > dn ? thr - dn : 0u;
                hi = thr + dp < thr ? 0xffffffffu : thr + dp;
            } else {
                plan_mode = 1;
            }
            // window bins: the smallest power of two that spans twice the bracket's range in 2048 bins
            const uint32_t span = 2 * (along + against);
            const int lg = 32 - __builtin_clz(span - 1u);  // ceil(log2(span)), span >= 2^13
            plan_wsh = lg > 11 ? (lg - 11 < 21 ? lg - 11 : 21) : 0;
            plan_wlo = thr > 2 * dn ? thr - 2 * dn : 0u;
        }
        // ---- the rounds ahead run locally where a box of 1.2 to 2.5 times the last moves holds at most 7000 uncertain
        // elements at the density the stages saw (the stage and its first round then take 20 us at 480x640, 9 more than a
        // bracket round, and every later round 5 less); not where two such plans have failed within a round each
        use_local = false;
        if (local_fails < 2) {
            const float fthr = u2f(thr), h = fthr * 9.765625e-4f;
            dens_r = dens * (float)(f2u(fthr + h) - thr) * __builtin_amdgcn_rcpf(h);
            use_local = steady && plan_box(have_prev, 7000.0f, 1.2f, 2.5f);
            if (a.plan_debug == 1) {
                box.s = s;
                box.t = t;
                box.Ds *= 0.015625f;
                box.Du *= 0.015625f;
            } else if (a.plan_debug == 4) {
                box.s += 3.0f * box.Ds;
            }
        }
        // Test hook: plans that are wrong on purpose, to exercise the fallbacks (the results must not change).
        // 1: local rounds' boxes of a 64th of the moves around the current state (the next one leaves them), and a bracket
        // just above its predicted range (the k-th usually lies below: a window on that side follows);
        // 2: every plan a window above +inf (it misses: the radix passes follow); 3: windows of 2^21-key bins from
        // 2^24 keys below the threshold (split passes with a counted below-window part); 4: local rounds' boxes beside the
        // current state (no local round may run).
        if (a.plan_debug == 1 && plan_mode == 0) {
            const uint32_t w = hi - lo;
            lo = hi < 0xffffffffu ? hi + 1u : hi;
            hi = lo + w < lo ? 0xffffffffu : lo + w;
        } else if (a.plan_debug == 2) {
            plan_mode = 1;
            plan_wlo = 0x7f800001u;
            plan_wsh = 0;
        } else if (a.plan_debug == 3 && plan_mode == 1) {
            plan_wlo = thr > (1u << 24) ? thr - (1u << 24) : 0u;
            plan_wsh = 21;
        }
        thr_prev = thr;
        have_prev = true;
    };

    // Local rounds. From the second round on (s, t) and the threshold move little, so nearly every element keeps its
    // side of the threshold for all rounds to come. One stage classifies the elements over a box of states around the
    // current one (plan_box) and publishes the sums over those that stay below and the uncertain rest (z, target); after
    // its barrier every block holds the uncertain elements in its registers, and runs the remaining rounds by itself,
    // with no further grid barrier: exact residuals and the exact k-th among the uncertain ones, their sums added to the
    // published ones. Each round is checked: the k-th must lie in the box's threshold range (then it is the k-th of all
    // elements), and the new (s, t) in its (s, u) range before the next round may use the classification; a round that
    // leaves the box goes back to the grid's stages with the exact state of the rounds done. As the moves shrink the box
    // is narrowed once it pays, and elements that become certain are folded into the sums. Every block computes the
    // same. What bounds a local round is its chain of dependent steps in one block: residuals, two to four counting steps of one
    // block barrier each (0.45 us), sums, the solve: 4-5 us at 1000 elements, 7 at 6000, against a bracket round's 11 at
    // 75 blocks and 15 at 124 (publish, barrier, candidate loads). A fit of ten rounds on noisy maps, before and after:
    // 192x256 122 -> 74 us, 240x320 122 -> 89, 480x640 141 -> 98..121, 756x1008 206 -> 138..152.
    // Runs rounds it0, it0 + 1, ... and returns how many were completed: none where the current state is not in the box.
    auto run_local = [&](const int it0) -> int {
        if (!in_box()) return 0;
        fit_box_bounds(box);  // (a test hook may have moved the box)
        const unsigned kk = (unsigned)sh.kk;
        const int lane = tid & 63, wv = tid >> 6;
        int done = 0;
        asm volatile("" : "+v"(mbits));
        // ---- the stage: classify, publish, barrier
        double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        uint32_t unc = 0;
        int nm = 0;
#pragma unroll
        for (int j = 0; j < kFitEPT; ++j) {
            int below, above;
            fit_class(box, zr[j], tr[j], below, above);
            const int m = (int)(mbits << (31 - j)) >> 31, inc = below & m;
            unc |= (uint32_t)(m & ~below & ~above) & (1u << j);
            nm -= inc;
            const double zd = masked(zr[j], inc), td = masked(tr[j], inc);
            v[1] += zd;
            v[2] += td;
            v[3] = __builtin_fma(zd, zd, v[3]);
            v[4] = __builtin_fma(zd, td, v[4]);
        }
        v[0] = (double)nm;
        unsigned nub;
        unsigned slot = block_excl_scan((unsigned)__popc(unc), sh.tmp, nub);
        // pairs (z, target): one 8-byte load per element
        float2* const pairs = (float2*)(ws.exch + fit_exchange(cap_words, stage & 1).pairs);
        {
            const size_t base = (size_t)b * kFitPerBlock;
#pragma unroll
            for (int g = 0; g < kFitEPT; g += 4) {
                if (__any((unc >> g) & 15u)) {
#pragma unroll
                    for (int j = g; j < g + 4; ++j) {
                        if ((unc >> j) & 1u) {
                            pairs[base + slot] = make_float2(zr[j], tr[j]);
                            ++slot;
                        }
                    }
                }
            }
        }
        publish(v);
        const unsigned count = fit_barrier(ws, nb, ++sync_seq, a.spin_limit, nub);
        load_partials();
        unsigned cc = 0;
        if (tid < nb) cc = count < (unsigned)kFitPerBlock ? count : (unsigned)kFitPerBlock;  // (an expired wait's)
        unsigned u;
        const unsigned offc = block_excl_scan(cc, sh.tmp, u);
        if (tid < nb) sh.off[tid] = offc;
        if (tid == 0) sh.off[nb] = u;
        __syncthreads();
        ++stage;
        u = (unsigned)__builtin_amdgcn_readfirstlane((int)u);
        if (u > kLocalCap) return 0;
        // ---- the uncertain elements into LDS in block order (thread (r, j) = (tid % nb, tid / nb) takes pairs of
        // elements j, j + per, ... of block r's region, 16 bytes a load), then 32 to a thread
        float2* const lds = (float2*)sh.cand;
        static_assert(kLocalCap * 2 <= (unsigned)kCandCap, "the elements share the candidates' LDS");
        {
            constexpr int kHold = 16;
            const int per = kFitThreads / nb, rr = tid % nb, jj = tid / nb;
            const unsigned cr = jj < per ? sh.off[rr + 1] - sh.off[rr] : 0u;
            const unsigned obase = jj < per ? sh.off[rr] : 0u;
            const float4* const src = (const float4*)(pairs + (size_t)rr * kFitPerBlock);
            for (unsigned s0 = (unsigned)jj; 2 * s0 < cr; s0 += (unsigned)(kHold * per)) {
                float4 cz[kHold];
#pragma unroll
                for (int q = 0; q < kHold; ++q) {
                    const unsigned e = s0 + (unsigned)(q * per);
                    cz[q] = 2 * e < cr ? src[e] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                }
#pragma unroll
                for (int q = 0; q < kHold; ++q) {
                    const unsigned e = 2 * (s0 + (unsigned)(q * per));
                    if (e < cr) lds[obase + e] = make_float2(cz[q].x, cz[q].y);
                    if (e + 1 < cr) lds[obase + e + 1] = make_float2(cz[q].z, cz[q].w);
                }
            }
        }
        double base[5] = {pp[0], pp[1], pp[2], pp[3], pp[4]};
        block_sum5(base, sh.red);  // (its barriers order the LDS stores too)
        float ez[kLocalPer], et[kLocalPer], ei[kLocalPer];
        bool local_odd = false;
        auto load_elements = [&]() {
#pragma unroll
            for (int g = 0; g < kLocalPer; g += 4) {
                if ((unsigned)(g * kFitThreads) < u) {
#pragma unroll
                    for (int j = g; j < g + 4; ++j) {
                        // past the end: an element of residual 1e18, above every box (plan_box), in no sum
                        const unsigned f = (unsigned)(j * kFitThreads + tid);
                        const float2 e = f < u ? lds[f] : make_float2(0.0f, -1e15f);
                        ez[j] = e.x;
                        et[j] = e.y;
                        ei[j] = fit_rcp(fmax_(e.y, 1e-3f));
                        local_odd = local_odd || fit_odd_target(e.y);
                    }
                }
            }
        };
        load_elements();
        double s_lo = -1e300, s_hi = 1e300, u_lo = -1e300, u_hi = 1e300;
        uint32_t k_lo = 1u, k_hi = 0x7f7fffffu;
        // the states the current classification holds for (1e-4 of the box is kept for the margins' own rounding)
        auto enter_box = [&]() {
            const double us = (double)box.s * zc + box.t;
            const double Ds = 0.9999 * box.Ds, Du = 0.9999 * box.Du;
            s_lo = box.s - Ds > s_lo ? box.s - Ds : s_lo;
            s_hi = box.s + Ds < s_hi ? box.s + Ds : s_hi;
            u_lo = us - Du > u_lo ? us - Du : u_lo;
            u_hi = us + Du < u_hi ? us + Du : u_hi;
            const uint32_t a0 = f2u(fmax_(box.thr - 0.9999f * box.Dt, 0.0f)), a1 = f2u(box.thr + 0.9999f * box.Dt);
            k_lo = a0 > k_lo ? a0 : k_lo;
            k_hi = a1 < k_hi ? a1 : k_hi;
        };
        int par = 0;
        uint32_t key[kLocalPer];
        // Elements of the block with keys up to each of four pivots: one block barrier.
        auto counts = [&](auto& p, auto& c) {
            constexpr int P = sizeof(p) / sizeof(p[0]);
            unsigned n[P];
#pragma unroll
            for (int q = 0; q < P; ++q) n[q] = 0;
#pragma unroll
            for (int g = 0; g < kLocalPer; g += 4) {
                if ((unsigned)(g * kFitThreads) < u) {
#pragma unroll
                    for (int j = g; j < g + 4; ++j)
#pragma unroll
                        for (int q = 0; q < P; ++q) n[q] += key[j] <= p[q] ? 1u : 0u;
                }
            }
#pragma unroll
            for (int q = 0; q < P; q += 2) {
                const unsigned both = wave_incl_scan_u32(n[q] | (n[q + 1] << 16));  // at most 2048 each
                if (lane == 63) sh.cnt[par][q / 2][wv] = both;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < P; q += 2) {
                const uint4 v4 = *(const uint4*)sh.cnt[par][q / 2];
                const unsigned v = (unsigned)__builtin_amdgcn_readfirstlane((int)((v4.x + v4.y) + (v4.z + v4.w)));
                c[q] = v & 0xffffu;
                c[q + 1] = v >> 16;
            }
            par ^= 1;
        };
        enter_box();
        dens_r = 0.5f * (float)u * __builtin_amdgcn_rcpf(box_width(box.Ds, box.Du, box.Dt));

#pragma nounroll
        for (;;) {
#pragma unroll
            for (int g = 0; g < kLocalPer; g += 4) {
                if ((unsigned)(g * kFitThreads) < u) {
                    fit_keys<4>(s, t, ez + g, et + g, ei + g, local_odd, key + g);
                }
            }
            // ---- the k-th key: count(<= klo) = c_lo < rank <= c_hi = count(<= khi). The first step counts the range's ends
            // and two moves' reach around the last threshold; then four counts a step, around the rank's place among
            // evenly spread keys (a quarter and nine tenths of their number's square root to either side), then, should
            // that not end soon, quartering
            const unsigned n_in = (unsigned)base[0];
            const unsigned rank = kk - n_in;
            uint32_t klo = k_lo - 1u, khi = k_hi;
            unsigned c_lo, c_hi;
            if (khi <= klo || khi - klo < 4u) return done;
            {
                const float fthr = u2f(thr);
                uint32_t g0 = f2u(fmax_(fthr - 2.0f * mv_t, 0.0f)), g1 = f2u(fthr + 2.0f * mv_t);
                g0 = g0 > klo + 1u ? g0 : klo + 1u;
                g0 = g0 < khi - 2u ? g0 : khi - 2u;
                g1 = g1 > g0 + 1u ? g1 : g0 + 1u;
                g1 = g1 < khi - 1u ? g1 : khi - 1u;
                uint32_t p[4] = {klo, g0, g1, khi};
                unsigned c[4];
                counts(p, c);
                if (kk <= n_in || rank <= c[0] || rank > c[3]) return done;  // outside the box's range
                const int q = rank <= c[1] ? 0 : (rank <= c[2] ? 1 : 2);
                klo = q == 0 ? klo : (q == 1 ? g0 : g1);
                c_lo = c[q];
                khi = q == 0 ? g0 : (q == 1 ? g1 : khi);
                c_hi = c[q + 1];
            }
            int step = 0;
#pragma nounroll
            while (khi - klo > 1u && c_hi != rank && c_lo + 1u != rank) {
                const uint32_t w = khi - klo;
                const float fw = (float)(w - 1u);
                uint32_t p[4];
                float at = 0.5f * (float)w, o0 = 0.25f * (float)w, o1 = o0;
                if (++step <= 6) {
                    const float n = (float)(c_hi - c_lo), per = (float)w * __builtin_amdgcn_rcpf(n);
                    const float sd = __builtin_amdgcn_sqrtf(n);
                    at = ((float)(rank - c_lo) - 0.5f) * per;
                    o0 = fmax_(0.25f * sd, 0.5f) * per;
                    o1 = fmax_(0.9f * sd, 1.5f) * per;
                }
                const float off[4] = {at - o1, at - o0, at + o0, at + o1};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t d = (uint32_t)fmin_(fmax_(off[q], 1.0f), fw);
                    p[q] = klo + (uint32_t)__builtin_amdgcn_readfirstlane((int)(d < w - 1u ? d : w - 1u));
                }
                unsigned c[4];
                counts(p, c);
                // the gap of (klo, p0, .., p3, khi] that holds the rank
#pragma unroll
                for (int q = 3; q >= 0; --q)
                    if (c[q] >= rank) {
                        khi = p[q];
                        c_hi = c[q];
                    }
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (c[q] < rank) {
                        klo = p[q];
                        c_lo = c[q];
                    }
            }
            // the k-th is the largest key up to khi (count(<= khi) = rank, or khi = klo + 1), else the smallest above
            // klo (the complements' largest)
            const bool largest = c_hi == rank || khi - klo == 1u;
            uint32_t mx = 0u;
#pragma unroll
            for (int g = 0; g < kLocalPer; g += 4) {
                if ((unsigned)(g * kFitThreads) < u) {
#pragma unroll
                    for (int j = g; j < g + 4; ++j) {
                        // keys are below 2^31: sign bits of differences select
                        const int up = ((int)khi - (int)key[j]) >> 31, dn = ((int)klo - (int)key[j]) >> 31;
                        const uint32_t k = largest ? key[j] & ~(uint32_t)up : ~key[j] & (uint32_t)dn;
                        mx = k > mx ? k : mx;
                    }
                }
            }
            mx = wave_max_u32(mx);
            if (lane == 0) sh.cnt[par][0][wv] = mx;
            __syncthreads();
            {
                const uint4 o = *(const uint4*)sh.cnt[par][0];
                mx = o.x > o.y ? o.x : o.y;
                mx = o.z > mx ? o.z : mx;
                mx = o.w > mx ? o.w : mx;
            }
            par ^= 1;
            const uint32_t found = (uint32_t)__builtin_amdgcn_readfirstlane((int)(largest ? mx : ~mx));
            // ---- the sums and the next (s, t)
            double w[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            int nw = 0;
#pragma unroll
            for (int g = 0; g < kLocalPer; g += 4) {
                if ((unsigned)(g * kFitThreads) < u) {
#pragma unroll
                    for (int j = g; j < g + 4; ++j) {
                        const int inc = ((int)key[j] - (int)found - 1) >> 31;
                        nw -= inc;
                        const double zd = masked(ez[j], inc), td = masked(et[j], inc);
                        w[1] += zd;
                        w[2] += td;
                        w[3] = __builtin_fma(zd, zd, w[3]);
                        w[4] = __builtin_fma(zd, td, w[4]);
                    }
                }
            }
            w[0] = (double)nw;
            block_sum5(w, sh.red);
#pragma unroll
            for (int k = 0; k < 5; ++k) w[k] += base[k];
            solve(w, false);
            thr_prev = thr;
            thr = found;
            if (b == 0 && tid == 0 && it0 + done < kFitTraceRounds) {
                ws.trace[2 * (it0 + done)] = 3u | ((unsigned)(step < 15 ? step : 15) << 4) | (u << 8);
                ws.trace[768 + it0 + done] = thr;
                ws.trace[2 * (it0 + done) + 1] = (uint32_t)wall_clock64();
            }
            ++done;
            note_moves(true);
            const double us = (double)s * zc + t;
            if (same || it0 + done >= a.iters || !(s >= s_lo && s <= s_hi && us >= u_lo && us <= u_hi)) return done;
            // ---- narrow where it drops most of more than 1600 elements and two rounds are left to gain by it
            if (u <= 1600u || it0 + done + 2 > a.iters ||
                !plan_box(true, fmax_(0.4f * (float)u, kLocalLow), 1.2f, 16.0f))
                continue;
            double c5[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            uint32_t keep = 0;
            int nin = 0;
#pragma unroll
            for (int g = 0; g < kLocalPer; g += 4) {
                if ((unsigned)(g * kFitThreads) < u) {
#pragma unroll
                    for (int j = g; j < g + 4; ++j) {
                        int below, above;
                        fit_class(box, ez[j], et[j], below, above);
                        keep |= (uint32_t)(~below & ~above) & (1u << j);
                        nin -= below;
                        const double zd = masked(ez[j], below), td = masked(et[j], below);
                        c5[1] += zd;
                        c5[2] += td;
                        c5[3] = __builtin_fma(zd, zd, c5[3]);
                        c5[4] = __builtin_fma(zd, td, c5[4]);
                    }
                }
            }
            c5[0] = (double)nin;
            unsigned left;
            unsigned pos = block_excl_scan((unsigned)__popc(keep), sh.tmp, left);
#pragma unroll
            for (int g = 0; g < kLocalPer; g += 4) {
                if ((unsigned)(g * kFitThreads) < u) {
#pragma unroll
                    for (int j = g; j < g + 4; ++j) {
                        if ((keep >> j) & 1u) {
                            lds[pos] = make_float2(ez[j], et[j]);
                            ++pos;
                        }
                    }
                }
            }
            block_sum5(c5, sh.red);  // (and the stores are ordered)
#pragma unroll
            for (int k = 0; k < 5; ++k) base[k] += c5[k];
            u = (unsigned)__builtin_amdgcn_readfirstlane((int)left);
            load_elements();
            enter_box();
            dens_r = 0.5f * (float)u * __builtin_amdgcn_rcpf(box_width(box.Ds, box.Du, box.Dt));
        }
    };

    // A fit that falls back to (1, 0) never changes (s, t): its trim rounds cannot affect the result.
    int rounds = 0;  // trim rounds run (the loop stops early at a fixed point)
    for (int it = 0; it < (sh.ok ? a.iters : 0); ++it) {
        if (use_local) {
            const int done = run_local(it);
            it += done;
            rounds = it;
            if (same || it >= a.iters) break;
            if (done < 2) ++local_fails;
            use_local = false;
            if (done > 0) plan_next();
            if (use_local) {
                --it;
                continue;
            }
        }
        rounds = it + 1;
        // The element values and mask bits are loop-invariant; hiding that from the compiler keeps it from hoisting
        // their fp64 products and per-element lane masks out of the loop into hundreds of extra registers.
#pragma unroll
        for (int j = 0; j < kFitEPT; ++j) asm volatile("" : "+v"(zr[j]), "+v"(tr[j]), "+v"(ir[j]));
        asm volatile("" : "+v"(mbits), "+v"(vbits));
        // ---- relative residuals as ordered bit patterns (+inf off the mask, kInvalid on padding)
        uint32_t rb[kFitEPT];
        fit_keys<kFitEPT>(s, t, zr, tr, ir, odd, rb);
#pragma unroll
        for (int j = 0; j < kFitEPT; ++j) {
            // off the mask +inf, padding kInvalid (bit fields of mbits and vbits, no conditions)
            const uint32_t m = (uint32_t)((int)(mbits << (31 - j)) >> 31), v = (uint32_t)((int)(vbits << (31 - j)) >> 31);
            rb[j] = (rb[j] & m) | (0x7f800000u & ~m) | ~v;
        }
        const unsigned kk = (unsigned)sh.kk;

        // Publishes below-count, below-sums and the candidates in [blo, bhi]; then a barrier; then the totals.
        auto stage_bracket = [&](uint32_t blo, uint32_t bhi) {
            blo = blo < 0x7fffffffu ? blo : 0x7fffffffu;
            bhi = bhi < 0x7fffffffu ? bhi : 0x7fffffffu;
            FIT_MARK(0);
            asm volatile("" : "+v"(mbits), "+v"(vbits));  // no per-element lane masks kept across phases
            // branch-free: below-count, masked below-sums (fp64; z*z and z*t are exact in fp64, so the fused form rounds
            // once, as the sum alone would), candidate count. Keys are below 2^31 (padding is -1), so comparisons are
            // sign bits of differences
            double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            int below = -npad, nc = 0, nm = 0;
            uint32_t cm = 0;
#pragma unroll
            for (int j = 0; j < kFitEPT; ++j) {
                const int k = (int)rb[j];
                const int isb = (k - (int)blo) >> 31;
                const int isc = ~isb & ~(((int)bhi - k) >> 31);
                const int inc = isb & ((int)(mbits << (31 - j)) >> 31);
                below -= isb;
                nc -= isc;
                nm -= inc;
                cm |= (uint32_t)isc & (1u << j);
                const double zd = masked(zr[j], inc), td = masked(tr[j], inc);
                v[1] += zd;
                v[2] += td;
                v[3] = __builtin_fma(zd, zd, v[3]);
                v[4] = __builtin_fma(zd, td, v[4]);
            }
            v[0] = (double)nm;
            // one scan for both counts: below in the high half, candidates in the low half (each <= 8192 per block)
            unsigned packed_total;
            const unsigned packed = block_excl_scan(((unsigned)below << 16) | (unsigned)nc, sh.tmp, packed_total);
            unsigned slot = packed & 0xffffu;
            const unsigned ncb = packed_total & 0xffffu;
            const FitExchange ex = fit_exchange(cap_words, stage & 1);
            const size_t base = (size_t)b * kFitPerBlock;
            uint32_t* const c_key = ws.exch + ex.key;
            float* const c_z = (float*)(ws.exch + ex.z);
            float* const c_t = (float*)(ws.exch + ex.t);
#pragma unroll
            for (int g = 0; g < kFitEPT; g += 4) {
                if (__any((cm >> g) & 15u)) {  // few elements are candidates: most waves skip most groups
#pragma unroll
                    for (int j = g; j < g + 4; ++j) {
                        if ((cm >> j) & 1u) {
                            c_key[base + slot] = rb[j] | (((mbits >> j) & 1u) << 31);
                            c_z[base + slot] = zr[j];
                            c_t[base + slot] = tr[j];
                            ++slot;
                        }
                    }
                }
            }
            publish(v);
            FIT_MARK(1);
            // the block's counts (below in the high half, candidates in the low half) ride on the barrier's flag
            const unsigned counts = fit_barrier(ws, nb, ++sync_seq, a.spin_limit, packed_total);
            FIT_MARK(2);
            load_partials();  // needed only by the sums after the selection: in flight with the candidate loads
            // totals and region offsets, in block order
            unsigned cb = 0, cc = 0;
            if (tid < nb) {
                cb = counts >> 16;
                cc = counts & 0xffffu;
                // a block publishes at most its own element count; the clamp only matters after an expired wait,
                // when the counts may be another launch's, and keeps every candidate read inside this launch's
                // regions
                cb = cb < (unsigned)kFitPerBlock ? cb : (unsigned)kFitPerBlock;
                cc = cc < (unsigned)kFitPerBlock ? cc : (unsigned)kFitPerBlock;
            }
            unsigned tb, tc;
            const unsigned offc = block_excl_scan2(cc, cb, sh.tmp2, tc, tb);
            if (tid < nb) sh.off[tid] = offc;
            if (tid == 0) {
                sh.off[nb] = tc;
                sh.total_below = tb;
                sh.total_cand = tc;
                sh.blo_last = blo;
                sh.bhi_last = bhi;
            }
            __syncthreads();
            FIT_MARK(3);
        };

        // Exact k-th among the published candidates (all in [blo, bhi]) and the new (s, t); buffer `stage & 1`.
        auto select_and_solve = [&](uint32_t blo, uint32_t bhi) {
            const unsigned total = sh.total_cand;
            unsigned rank = kk - sh.total_below;
            const FitExchange ex = fit_exchange(cap_words, stage & 1);
            const uint32_t* const c_key = ws.exch + ex.key;
            const float* const c_z = (const float*)(ws.exch + ex.z);
            const float* const c_t = (const float*)(ws.exch + ex.t);
            // Thread (r, j) = (tid % nb, tid / nb) owns slots j, j + per, j + 2 per, ... of block r's region: no
            // search from a flat index to a region, and its loads are independent. Keys go to LDS in flat order
            // (region r at off[r]); the first kHold of the thread's candidates also keep z and target in registers
            // for the sums (loaded with the keys: usually no second round trip).
            constexpr int kHold = 12;
            const int per = kFitThreads / nb;  // threads per region (nb <= kFitThreads)
            const int rr = tid % nb, jj = tid / nb;
            const bool act = jj < per;
            const unsigned cr = act ? sh.off[rr + 1] - sh.off[rr] : 0u;
            const unsigned obase = act ? sh.off[rr] : 0u;
            const size_t rbase = (size_t)rr * kFitPerBlock;
            uint32_t hw[kHold];
            float hz[kHold], ht[kHold];
#pragma unroll
            for (int u = 0; u < kHold; ++u) {
                const unsigned slot = (unsigned)(jj + u * per);
                hw[u] = 0;
                hz[u] = 0.0f;
                ht[u] = 0.0f;
                if (slot < cr) {
                    hw[u] = c_key[rbase + slot];
                    hz[u] = c_z[rbase + slot];
                    ht[u] = c_t[rbase + slot];
                }
            }
#pragma unroll
            for (int u = 0; u < kHold; ++u) {
                const unsigned slot = (unsigned)(jj + u * per);
                if (slot < cr) sh.cand[obase + slot] = hw[u];
            }
            for (unsigned s0 = (unsigned)(jj + kHold * per); s0 < cr; s0 += (unsigned)(kHold * per)) {
                uint32_t w[kHold];
#pragma unroll
                for (int u = 0; u < kHold; ++u) {
                    const unsigned slot = s0 + (unsigned)(u * per);
                    w[u] = slot < cr ? c_key[rbase + slot] : 0u;
                }
#pragma unroll
                for (int u = 0; u < kHold; ++u) {
                    const unsigned slot = s0 + (unsigned)(u * per);
                    if (slot < cr) sh.cand[obase + slot] = w[u];
                }
            }
            __syncthreads();
            FIT_MARK(4);
            uint32_t prefix = 0, pmask = 0;
            int top = 0;
            if (total <= 96u) {
                // few candidates: each thread ranks its own against all of them (LDS broadcast reads; beyond ~100
                // candidates the radix select below is faster)
                if (tid == 0) sh.bin = 0;
                __syncthreads();
                if ((unsigned)tid < total) {
                    const uint32_t key = sh.cand[tid] & 0x7fffffffu;
                    unsigned less = 0, eq = 0;
                    // four keys per 16-byte LDS read and four reads in flight per trip: one 4-byte read per trip
                    // waited out its latency every time (107 candidates took 5.6 us)
                    const unsigned t4 = total & ~3u;
#pragma unroll 4
                    for (unsigned g = 0; g < t4; g += 4) {
                        const uint4 q = *(const uint4*)&sh.cand[g];
                        const uint32_t kq[4] = {q.x & 0x7fffffffu, q.y & 0x7fffffffu, q.z & 0x7fffffffu,
                                                q.w & 0x7fffffffu};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            less += kq[e] < key ? 1u : 0u;
                            eq += kq[e] == key ? 1u : 0u;
                        }
                    }
                    for (unsigned g = t4; g < total; ++g) {
                        const uint32_t kg = sh.cand[g] & 0x7fffffffu;
                        less += kg < key ? 1u : 0u;
                        eq += kg == key ? 1u : 0u;
                    }
                    if (less < rank && rank <= less + eq) sh.bin = key - blo;  // equal keys write equal values
                }
                __syncthreads();
                prefix = sh.bin;
            } else {
                // MSD radix select over key - blo in [0, bhi - blo], 11 bits per pass
                const uint32_t range = bhi - blo;
                top = range ? 32 - __builtin_clz(range) : 0;
            }
            while (top > 0) {
                const int width = top < 11 ? top : 11;
                const int shb = top - width;
                const uint32_t dmask = (1u << width) - 1u;
                for (int q = tid; q < kFitBins; q += kFitThreads) sh.hist[q] = 0;
                __syncthreads();
                for (unsigned f = tid; f < total; f += kFitThreads) {
                    const uint32_t key = (sh.cand[f] & 0x7fffffffu) - blo;
                    if ((key & pmask) == prefix) atomicAdd(&sh.hist[(key >> shb) & dmask], 1u);
                }
                __syncthreads();
                find_bin(sh, rank, [&](int q) { return sh.hist[q]; }, [] { return 0u; });
                prefix |= sh.bin << shb;
                pmask |= dmask << shb;
                rank -= sh.below;
                top = shb;
            }
            thr = blo + prefix;
            FIT_MARK(5);
            // sums: this thread's share of the published below-partials, then its candidates at or under thr in
            // flat order; then one fixed-order block reduction
            double v[5] = {pp[0], pp[1], pp[2], pp[3], pp[4]};
            int nsel = 0;
#pragma unroll
            for (int u = 0; u < kHold; ++u) {
                const int inc = ((int)hw[u] >> 31) & (((int)(hw[u] & 0x7fffffffu) - (int)thr - 1) >> 31);
                const double zd = masked(hz[u], inc), td = masked(ht[u], inc);
                nsel -= inc;
                v[1] += zd;
                v[2] += td;
                v[3] = __builtin_fma(zd, zd, v[3]);
                v[4] = __builtin_fma(zd, td, v[4]);
            }
            v[0] += (double)nsel;
            for (unsigned s0 = (unsigned)(jj + kHold * per); s0 < cr; s0 += (unsigned)(kHold * per)) {
                // kHold candidates per trip: all loads issued before any is used
                float cz[kHold], ct[kHold];
                bool use[kHold];
#pragma unroll
                for (int u = 0; u < kHold; ++u) {
                    const unsigned slot = s0 + (unsigned)(u * per);
                    const uint32_t w = slot < cr ? sh.cand[obase + slot] : 0u;
                    use[u] = (w >> 31) && (w & 0x7fffffffu) <= thr;
                    cz[u] = use[u] ? c_z[rbase + slot] : 0.0f;
                    ct[u] = use[u] ? c_t[rbase + slot] : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < kHold; ++u) {
                    if (use[u]) {
                        const double zd = cz[u], td = ct[u];
                        v[0] += 1.0;
                        v[1] += zd;
                        v[2] += td;
                        v[3] = __builtin_fma(zd, zd, v[3]);
                        v[4] = __builtin_fma(zd, td, v[4]);
                    }
                }
            }
            block_sum5(v, sh.red);
            ++stage;
            solve(v, false);
            FIT_MARK(6);
        };

        // Histogram pass over a window of keys: bin q counts the keys in [wlo + q 2^wsh, wlo + (q+1) 2^wsh), q < 2048,
        // and one more counter the keys below wlo; blocks merge their LDS histograms into this round's global slot
        // `hslot` by atomics, and after one barrier every block finds the bin holding the kk-th key. Returns false
        // when that key lies outside the window; else pbin_lo / pbin_cnt give the bin's first key and its count.
        // One call site serves the radix passes and the predicted windows (the unrolled element loop exists once).
        int hslot = 0;
        uint32_t pbin_lo = 0;
        unsigned pbin_cnt = 0, pbin_below = 0;
        // `below` is the count of keys below wlo when the caller knows it (the radix range starts at 0, and a pass
        // that splits a bin follows the keys before that bin), else kNoBelow: the pass counts them, into 16 words
        // (block b adds to word b % 16) so that the 75-94 blocks' atomics do not all queue on one address.
        constexpr unsigned kNoBelow = 0xffffffffu;
        auto hist_pass = [&](uint32_t wlo, int wsh, unsigned below) -> bool {
            asm volatile("" : "+v"(mbits), "+v"(vbits));
            for (int q = tid; q < kFitBins; q += kFitThreads) sh.hist[q] = 0;
            if (tid == 0) sh.hbelow = 0;
            __syncthreads();
            // one comparison per element (around its LDS atomic): the window's keys are [wlo, wlo + span), span at most
            // 2^31; a key below wlo and a padding slot's -1 give a difference of 2^31 or more
            const uint32_t span = wsh < 20 ? (uint32_t)kFitBins << wsh : 0x80000000u;
            int below_n = -npad;
#pragma unroll
            for (int j = 0; j < kFitEPT; ++j) {
                const uint32_t d = rb[j] - wlo;
                below_n -= ((int)rb[j] - (int)wlo) >> 31;
                if (d < span) atomicAdd(&sh.hist[d >> wsh], 1u);
            }
            unsigned nbelow = (unsigned)below_n;
            const bool count_below = below == kNoBelow;
            if (count_below) {
                nbelow = wave_incl_scan_u32(nbelow);
                if ((tid & 63) == 63 && nbelow) atomicAdd(&sh.hbelow, nbelow);
            }
            __syncthreads();
            unsigned* gh = ws.hist + ((int64_t)it * kFitHistSlots + hslot) * kFitHistWords;
            hslot = hslot + 1 < kFitHistSlots ? hslot + 1 : hslot;  // at most 6 passes a round (never reached)
            {
                unsigned h[kFitBins / kFitThreads];  // all read before any is merged
#pragma unroll
                for (int q = 0; q < kFitBins / kFitThreads; ++q) h[q] = sh.hist[q * kFitThreads + tid];
#pragma unroll
                for (int q = 0; q < kFitBins / kFitThreads; ++q)
                    if (h[q]) atomicAdd(&gh[q * kFitThreads + tid], h[q]);
            }
            if (count_below && tid == 0 && sh.hbelow) atomicAdd(&gh[kFitBins + (b & 15)], sh.hbelow);
            fit_barrier(ws, nb, ++sync_seq, a.spin_limit);
            find_bin(
                sh, kk, [&](int q) { return __hip_atomic_load(&gh[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); },
                [&] {
                    if (!count_below) return below;
                    unsigned v = 0;
#pragma unroll
                    for (int q = 0; q < 16; ++q)
                        v += __hip_atomic_load(&gh[kFitBins + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    return v;
                });
            if (!sh.found) return false;  // below or above the window (read from LDS: the block branches as one)
            pbin_lo = wlo + (sh.bin << wsh);
            pbin_cnt = sh.bincnt;
            pbin_below = sh.below;
            return true;
        };

        // The round's selection. mode 0: one bracket stage on the predicted bracket [lo, hi]; 1: a histogram pass on
        // the predicted window, then a stage on its bin; 2: radix passes over the whole key range (bits 31..21, then
        // 20..10 of the first bin, then single values, each only while the bin holds more than kStageMax keys),
        // then a stage on the bin. A bracket stage that misses the k-th is followed by a window on the side that
        // holds it; a window that misses it, by the radix passes. Trace codes: 0 bracket, 1 bracket missed -> radix
        // (no key above it), 2 radix, 4 window, 5 bracket missed -> window, 6 window missed -> radix, 7 bracket and
        // window missed -> radix; +8 when one
        // value holds the k-th and more than kCandCap keys (its sums take a barrier of their own).
        int mode = plan_mode;
        int path = mode == 0 ? 0 : (mode == 1 ? 4 : 2);
        int passes = 0;
        uint32_t blo = lo, bhi = hi, wlo = plan_wlo;
        int wsh = plan_wsh;
#pragma nounroll
        for (;;) {
            if (mode != 0) {
                if (mode == 2) {
                    wlo = 0;
                    wsh = 21;
                }
                bool hit;
                unsigned below = mode == 2 ? 0u : kNoBelow;
#pragma nounroll
                for (;;) {
                    hit = hist_pass(wlo, wsh, below);
                    ++passes;
                    if (!hit || pbin_cnt <= kStageMax || wsh == 0) break;
                    wlo = pbin_lo;  // split the bin: 2048 sub-bins of 2^(wsh - 11) keys
                    wsh = wsh > 11 ? wsh - 11 : 0;
                    below = pbin_below;
                }
                if (!hit) {
                    if (mode == 2) break;  // the whole range holds every key: only after an expired wait
                    mode = 2;
                    path = path == 5 ? 7 : 6;
                    continue;
                }
                blo = pbin_lo;
                const uint64_t e = (uint64_t)pbin_lo + ((1ull << wsh) - 1u);
                bhi = e > 0xffffffffull ? 0xffffffffu : (uint32_t)e;
                if (pbin_cnt > (unsigned)kCandCap) {
                    // one value (wsh == 0) holds the k-th and more keys than LDS holds: it is the threshold; the
                    // sums over the keys at or below it take one more barrier
                    path |= 8;
                    thr = blo;
                    double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int j = 0; j < kFitEPT; ++j) {
                        if (((mbits >> j) & 1u) && rb[j] <= thr) {
                            const double zd = zr[j], td = tr[j];
                            v[0] += 1.0;
                            v[1] += zd;
                            v[2] += td;
                            v[3] = __builtin_fma(zd, zd, v[3]);
                            v[4] = __builtin_fma(zd, td, v[4]);
                        }
                    }
                    publish(v);
                    fit_barrier(ws, nb, ++sync_seq, a.spin_limit);
                    double g[5];
                    gather_partials(g);
                    ++stage;
                    solve(g, false);
                    break;
                }
            }
            stage_bracket(blo, bhi);
            const unsigned tbl = sh.total_below, tcd = sh.total_cand;
            if (tbl < kk && kk <= tbl + tcd && tcd <= (unsigned)kCandCap) {
                select_and_solve(blo, bhi);
                break;
            }
            ++stage;
            if (mode != 0) break;  // a pass bin the stage does not confirm: only after an expired wait
            // the bracket missed: a window of 2^plan_wsh-key bins on the side that holds the k-th (or, when the
            // bracket held it among more candidates than LDS holds, a window over the bracket itself)
            mode = 1;
            path = 5;
            wsh = plan_wsh;
            const uint64_t span = (uint64_t)kFitBins << wsh;
            if (kk <= tbl) {
                wlo = (uint64_t)blo > span ? blo - (uint32_t)span : 0u;
            } else if (kk <= tbl + tcd) {
                wlo = blo;
                wsh = 0;
                while (((uint64_t)kFitBins << wsh) < (uint64_t)bhi - blo + 1u && wsh < 21) ++wsh;
            } else if (bhi >= 0x7fffffffu) {
                mode = 2;
                path = 1;
            } else {
                wlo = bhi + 1u;
            }
        }

        if (b == 0 && tid == 0 && it < kFitTraceRounds) {
            ws.trace[2 * it] = (uint32_t)path | ((uint32_t)(passes < 15 ? passes : 15) << 4) | (sh.total_cand << 8);
            ws.trace[768 + it] = thr;
            ws.trace[2 * it + 1] = (uint32_t)wall_clock64();
        }
        // Fixed point: when a round reproduces the previous (s, t) bit for bit, the next round sees the same
        // residuals, hence the same k-th value, weights and sums, so every remaining round -- and the final
        // solve -- returns exactly these (s, t). Stopping here gives the bit-identical result.
        if (same) break;
        note_moves(have_prev);
        plan_next();
    }

    if (b == 0 && tid == 0) {
        __hip_atomic_store(&ws.bar[2], sync_seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        a.st[2 * a.b] = s;
        a.st[2 * a.b + 1] = t;
        if (a.info) a.info[5 * a.b + 3] = (int32_t)thr;
        ws.trace[2 * kFitTraceRounds + 2] = (uint32_t)rounds;
    }

    // Completion. The last block to finish sees every block's writes; it reports the launch's error flag. After
    // an expired wait the blocks may have passed different numbers of barriers, so their flags and the epoch no
    // longer agree: it zeroes all of them (every flag line, not only this grid's, since the epoch restarts at 0),
    // clears the flag, counts the failure and replaces (s, t), which raced, by NaN.
    __syncthreads();
    if (tid == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const unsigned prev = __hip_atomic_fetch_add(ws.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sh.last = prev == (unsigned)nb - 1u;
        if (sh.last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    if (!sh.last) return;
    const int err = __hip_atomic_load(ws.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (err) {
        for (int q = tid; q < kFitMaxBlocks * 16; q += kFitThreads)
            __hip_atomic_store(&ws.flags[q], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (tid == 0) {
        if (err) {
            const float nan = __builtin_nanf("");
            a.st[2 * a.b] = nan;
            a.st[2 * a.b + 1] = nan;
            __hip_atomic_store(&ws.bar[2], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(ws.err, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(ws.err_seen, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (a.info) a.info[5 * a.b + 4] = err;
        __hip_atomic_store(ws.done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Elements per thread: 16 up to 2^19 elements (twice the blocks: faster loads and per-block passes, while the
// device-wide barrier still costs little), 24 up to 1.5 M (config H's 762,048: 124 blocks; measured against 20 and
// 28 per thread, 149 / 109 blocks, and the 32 used before: the fits on H's input / refined map took 85 / 210 us
// against 96 / 239, 86 / 212 and 91 / 220), else 32.
static int fit_ept(int64_t N) {
    return N <= (int64_t(1) << 19) ? 16 : N <= (int64_t)kFitThreads * 24 * kFitMaxBlocks ? 24 : 32;
}
static int fit_blocks(int64_t N) {
    const int64_t per = (int64_t)kFitThreads * fit_ept(N);
    return (int)((N + per - 1) / per);
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Bytes before the exchanged elements: the header, the barrier flags, the partial sums, the histograms.
static size_t fit_exchange_offset(int iters) {
    const size_t hist = (size_t)(iters > 0 ? iters : 1) * kFitHistSlots * kFitHistWords * sizeof(unsigned);
    return kFitHeader + align256(kFitMaxBlocks * 64) + align256(2 * kFitMaxBlocks * 5 * sizeof(uint64_t)) +
           align256(hist);
}

size_t fit_workspace_bytes(int64_t N, int iters) {
    const int64_t n = N > 0 ? N : 1;
    const size_t nb = (size_t)fit_blocks(n);
    const size_t cand = 6 * nb * (size_t)kFitThreads * fit_ept(n) * sizeof(uint32_t);
    return fit_exchange_offset(iters) + cand;
}

// Polls of one barrier wait before it expires (~0.1 s at the default); lowered only by the test hook
// pmg_debug_fit_spin_limit, so that tests can make waits expire with every kernel still exiting normally.
static unsigned g_fit_spin_limit = 1u << 23;
// Wrong-on-purpose round plans for tests (pmg_debug_fit_plan); 0 in normal use.
static int g_fit_plan_debug = 0;

int launch_fit(const FitLaunch& f, hipStream_t s) {
    PMG_REQUIRE(f.N > 0 && f.N <= (int64_t)kFitMaxBlocks * kFitPerBlockMax, "N must be in [1, 2^21]");
    PMG_REQUIRE(f.iters >= 0 && f.iters <= 64, "iters must be in [0, 64]");
    PMG_REQUIRE(f.min_points >= 1, "min_points must be >= 1");
    PMG_REQUIRE(f.trim >= 0.0f && f.trim < 1.0f, "trim must be in [0, 1)");
    PMG_REQUIRE(f.workspace && f.workspace_bytes >= fit_workspace_bytes(f.N, f.iters), "workspace too small");
    PMG_REQUIRE(aligned16(f.workspace), "workspace must be 16-byte aligned");
    const int nb = fit_blocks(f.N);
    const int ept = fit_ept(f.N);
    static int max_resident[3] = {-1, -1, -1};
    int& mr = max_resident[ept == 16 ? 0 : ept == 24 ? 1 : 2];
    if (mr < 0) {
        int per_cu = 0;
        if (ept == 16)
            PMG_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fit_k<16>, kFitThreads, 0));
        else if (ept == 24)
            PMG_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fit_k<24>, kFitThreads, 0));
        else
            PMG_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fit_k<32>, kFitThreads, 0));
        mr = per_cu * num_cus();
    }
    const int max_resident_n = mr;
    PMG_REQUIRE(nb <= max_resident_n && nb <= kFitMaxBlocks,
                "fit grid of " + std::to_string(nb) + " blocks cannot be resident (max " +
                    std::to_string(max_resident_n) + ")");
    uint8_t* p = (uint8_t*)f.workspace;
    FitWs ws;
    ws.bar = (unsigned*)p;
    ws.err = (int*)(p + kFitErrOffset);
    ws.trace = (uint32_t*)(p + 128);
    ws.done = (unsigned*)(p + kFitDoneOffset);
    ws.err_seen = (unsigned*)(p + kFitErrSeenOffset);
    p += kFitHeader;
    ws.flags = (unsigned*)p;
    p += align256(kFitMaxBlocks * 64);
    ws.partials = (uint64_t*)p;
    p += align256(2 * kFitMaxBlocks * 5 * sizeof(uint64_t));
    ws.hist = (unsigned*)p;
    ws.exch = (uint32_t*)((uint8_t*)f.workspace + fit_exchange_offset(f.iters));
    for (int b = 0; b < f.B; ++b) {
        FitArgs a{f.mode, f.z, f.tg, f.mask, f.logz, f.stride, f.lidar, f.conf, f.H, f.W, f.dh, f.dw,
                  f.N, f.iters, (float)(1.0 - (double)f.trim), f.min_points, b, f.st, f.info,
                  g_fit_spin_limit, g_fit_plan_debug, ws};
        if (ept == 16)
            hipLaunchKernelGGL(fit_k<16>, dim3(nb), dim3(kFitThreads), 0, s, a);
        else if (ept == 24)
            hipLaunchKernelGGL(fit_k<24>, dim3(nb), dim3(kFitThreads), 0, s, a);
        else
            hipLaunchKernelGGL(fit_k<32>, dim3(nb), dim3(kFitThreads), 0, s, a);
        if (int e = check_launch("fit_k")) return e;
    }
    return PMG_OK;
}

// ------------------------------------------------------------------------------------------------------------
// Final metric fit inputs (v3.py:768-775), one thread per LiDAR pixel: d_lr = F.interpolate(depth, (dh, dw),
// mode='area') of z = exp(logz) -- adaptive average pooling, the window [floor(o*H/dh), ceil((o+1)*H/dh)) summed
// in fp32 in row-major order and divided by its height, then by its width, as adaptive_avg_pool2d does -- and
// mask = conf >= 2 & lidar > 0 & d_lr > 0 (& the pooled mask_binary > 0.99).
__global__ __launch_bounds__(256) void final_inputs_k(const float* __restrict__ logz, int64_t stride,
                                                      const float* __restrict__ lidar, const float* __restrict__ conf,
                                                      const uint8_t* __restrict__ mask_binary, int H, int W, int dh,
                                                      int dw, int64_t n_out, float* __restrict__ z_out,
                                                      uint8_t* __restrict__ m_out) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= n_out) return;
    const int64_t plane = (int64_t)dh * dw;
    const int64_t b = q / plane;
    const int rem = (int)(q - b * plane);
    const int oh = rem / dw, ow = rem - oh * dw;
    const int r0 = (int)(((int64_t)oh * H) / dh), r1 = (int)((((int64_t)oh + 1) * H + dh - 1) / dh);
    const int c0 = (int)(((int64_t)ow * W) / dw), c1 = (int)((((int64_t)ow + 1) * W + dw - 1) / dw);
    const int64_t base = b * H * W;
    float sz = 0.0f, sm = 0.0f;
    for (int r = r0; r < r1; ++r)
        for (int c = c0; c < c1; ++c) {
            const int64_t p = base + (int64_t)r * W + c;
            sz = sz + exp_f32(logz[p * stride]);
            if (mask_binary) sm = sm + (mask_binary[p] ? 1.0f : 0.0f);
        }
    const float kh = (float)(r1 - r0), kw = (float)(c1 - c0);
    const float z = sz / kh / kw;
    const float d = lidar[q];
    bool m = conf[q] >= 2.0f && d > 0.0f && z > 0.0f;
    if (mask_binary) m = m && (sm / kh / kw > 0.99f);
    z_out[q] = z;
    m_out[q] = m ? 1 : 0;
}

// post_depth (MetricFit.metal:200-211; v3.py:776 depth = s * z + t): the metric depth of every pixel from the refined
// log depth and the final fit of its frame, d = s * exp(logz) + t in fp32; +inf where the mask is 0 or d <= 0.
__global__ __launch_bounds__(256) void post_depth_k(const float* __restrict__ logz, int64_t stride,
                                                    const uint8_t* __restrict__ mask, int64_t HW, int64_t n,
                                                    const float* __restrict__ st, float* __restrict__ depth) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    const int64_t b = p / HW;
    const float d = st[2 * b] * exp_f32(logz[p * stride]) + st[2 * b + 1];
    const bool ok = (mask == nullptr || mask[p] != 0) && d > 0.0f;
    depth[p] = ok ? d : __builtin_inff();
}

size_t final_fit_workspace_bytes(int B, int dh, int dw, int iters) {
    const size_t n = (size_t)B * dh * dw;
    return align256(fit_workspace_bytes((int64_t)dh * dw, iters)) + align256(n * sizeof(float)) + align256(n);
}

int launch_final_fit(const FinalFit& f, hipStream_t s) {
    PMG_REQUIRE(f.logz && f.lidar && f.conf && f.st, "null buffer");
    PMG_REQUIRE(f.B >= 1 && f.H >= 1 && f.W >= 1 && f.dh >= 1 && f.dw >= 1 && f.stride >= 1, "bad shape");
    PMG_REQUIRE((int64_t)f.dh * f.dw <= (int64_t)kFitMaxBlocks * kFitPerBlockMax, "LiDAR map larger than 2^21 pixels");
    PMG_REQUIRE(f.workspace && f.workspace_bytes >= final_fit_workspace_bytes(f.B, f.dh, f.dw, f.iters),
                "workspace too small");
    const int64_t N = (int64_t)f.dh * f.dw;
    const int64_t n_out = (int64_t)f.B * N;
    const size_t fit_bytes = align256(fit_workspace_bytes(N, f.iters));
    if (f.dh == f.H && f.dw == f.W) {
        // one-pixel area windows: the fit reads exp(logz), the LiDAR, conf and mask_binary itself (no
        // final_inputs_k launch; the same values)
        FitLaunch g{};
        g.mode = 2;
        g.logz = f.logz;
        g.stride = f.stride;
        g.lidar = f.lidar;
        g.conf = f.conf;
        g.mask = f.mask_binary;
        g.H = f.H;
        g.W = f.W;
        g.dh = f.dh;
        g.dw = f.dw;
        g.B = f.B;
        g.N = N;
        g.iters = f.iters;
        g.trim = f.trim;
        g.min_points = f.min_points;
        g.st = f.st;
        g.info = f.info;
        g.workspace = f.workspace;
        g.workspace_bytes = fit_bytes;
        return launch_fit(g, s);
    }
    float* z_lr = (float*)((uint8_t*)f.workspace + fit_bytes);
    uint8_t* m_lr = (uint8_t*)f.workspace + fit_bytes + align256((size_t)n_out * sizeof(float));
    hipLaunchKernelGGL(final_inputs_k, dim3((unsigned)((n_out + 255) / 256)), dim3(256), 0, s, f.logz, f.stride,
                       f.lidar, f.conf, f.mask_binary, f.H, f.W, f.dh, f.dw, n_out, z_lr, m_lr);
    if (int e = check_launch("final_inputs_k")) return e;
    FitLaunch g{};
    g.mode = 0;
    g.z = z_lr;
    g.tg = f.lidar;
    g.mask = m_lr;
    g.B = f.B;
    g.N = N;
    g.iters = f.iters;
    g.trim = f.trim;
    g.min_points = f.min_points;
    g.st = f.st;
    g.info = f.info;
    g.workspace = f.workspace;
    g.workspace_bytes = fit_bytes;
    return launch_fit(g, s);
}

// ------------------------------------------------------------------------------------------------------------
// Allocation-free fit: the workspace is a file-scope device array, one copy per GPU, instead of caller memory.
// 14 MiB holds the workspace of N <= 2^19 elements per batch item at iters <= 16 (13.4 MB). Host code never uses
// the array's name as an address: at a device's first call its address is looked up with hipGetSymbolAddress
// (the device current), kept per device, and only that pointer reaches kernels.
constexpr size_t kStaticFitBytes = (size_t)14 << 20;
constexpr int kStaticFitMaxDevices = 64;
static __device__ __align__(256) uint8_t scratch[kStaticFitBytes];

__global__ void zero_words_k(uint32_t* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

static std::mutex g_static_fit_mu;
static void* g_static_fit_ptr[kStaticFitMaxDevices];

// The current device's scratch address. At the device's first call it also enqueues, on `s`, the clearing of the
// part of the workspace the fit requires at zero before its first launch (the barrier epoch, error flag, completion
// count and per-block flags; the rest is cleared or overwritten by every launch).
static int static_fit_scratch(hipStream_t s, void** out) {
    int dev = -1;
    PMG_CHECK_HIP(hipGetDevice(&dev));
    PMG_REQUIRE(dev >= 0 && dev < kStaticFitMaxDevices, "device index out of range for the static fit scratch");
    std::lock_guard<std::mutex> lock(g_static_fit_mu);
    if (!g_static_fit_ptr[dev]) {
        void* p = nullptr;
        PMG_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        const int64_t words = (int64_t)(kFitHeader + align256((size_t)kFitMaxBlocks * 64)) / 4;
        hipLaunchKernelGGL(zero_words_k, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s, (uint32_t*)p, words);
        if (int e = check_launch("zero_words_k")) return e;
        g_static_fit_ptr[dev] = p;
    }
    *out = g_static_fit_ptr[dev];
    return PMG_OK;
}

}  // namespace pmg

using namespace pmg;

extern "C" {

size_t pmg_fit_workspace_bytes(int64_t N, int iters) { return fit_workspace_bytes(N, iters); }

int pmg_fit_scale_shift_static(const float* z, const float* target, const uint8_t* mask, int B, int64_t N, int iters,
                               float trim, int min_points, float* st, int32_t* info, void* stream) {
    PMG_REQUIRE(z && target && mask && st, "null buffer");
    PMG_REQUIRE(B >= 1, "bad batch");
    PMG_REQUIRE(N > 0 && N <= ((int64_t)1 << 19) && iters >= 0 && iters <= 16,
                "pmg_fit_scale_shift_static: N = " + std::to_string(N) + ", iters = " + std::to_string(iters) +
                    " exceed the static scratch (N <= 2^19 per batch item, iters <= 16); use pmg_fit_scale_shift "
                    "with a caller workspace");
    PMG_REQUIRE(fit_workspace_bytes(N, iters) <= kStaticFitBytes, "static fit scratch too small");
    hipStream_t s = (hipStream_t)stream;
    void* ws = nullptr;
    if (int e = static_fit_scratch(s, &ws)) return e;
    FitLaunch f{};
    f.mode = 0;
    f.z = z;
    f.tg = target;
    f.mask = mask;
    f.B = B;
    f.N = N;
    f.iters = iters;
    f.trim = trim;
    f.min_points = min_points;
    f.st = st;
    f.info = info;
    f.workspace = ws;
    f.workspace_bytes = kStaticFitBytes;
    return launch_fit(f, s);
}

unsigned pmg_debug_fit_spin_limit(unsigned polls) {
    const unsigned prev = g_fit_spin_limit;
    g_fit_spin_limit = polls ? polls : (1u << 23);
    return prev;
}

unsigned pmg_debug_fit_plan(unsigned mode) {
    const unsigned prev = (unsigned)g_fit_plan_debug;
    g_fit_plan_debug = mode <= 4 ? (int)mode : 0;
    return prev;
}

int pmg_debug_fit_exchange(int64_t N, int iters, int parity, int64_t* out) {
    PMG_REQUIRE(out && N > 0 && N <= (int64_t)kFitMaxBlocks * kFitPerBlockMax, "bad size");
    const int64_t per = (int64_t)kFitThreads * fit_ept(N), nb = fit_blocks(N);
    const FitExchange ex = fit_exchange(nb * per, parity & 1);
    const int64_t base = (int64_t)fit_exchange_offset(iters);
    out[0] = nb;
    out[1] = per;
    out[2] = base + 4 * ex.key;
    out[3] = base + 4 * ex.z;
    out[4] = base + 4 * ex.t;
    out[5] = base + 4 * ex.pairs;
    return PMG_OK;
}

int pmg_debug_fit_class(const float* box, const float* z, const float* target, int64_t n, int8_t* side) {
    PMG_REQUIRE(box && z && target && side && n >= 0, "bad arguments");
    FitBox q{box[0], box[1], box[2], box[3], box[4], box[5], box[6], 0.0f, 0.0f};
    fit_box_bounds(q);
    for (int64_t i = 0; i < n; ++i) {
        int below, above;
        fit_class(q, z[i], target[i], below, above);
        side[i] = (int8_t)(above ? 1 : below);
    }
    return PMG_OK;
}

size_t pmg_fit_final_workspace_bytes(int B, int dh, int dw, int iters) {
    if (B < 1 || dh < 1 || dw < 1) return 0;
    return final_fit_workspace_bytes(B, dh, dw, iters);
}

int pmg_fit_scale_shift(const float* z, const float* target, const uint8_t* mask, int B, int64_t N, int iters,
                        float trim, int min_points, float* st, int32_t* info, void* workspace,
                        size_t workspace_bytes, void* stream) {
    PMG_REQUIRE(z && target && mask && st, "null buffer");
    PMG_REQUIRE(B >= 1, "bad batch");
    FitLaunch f{};
    f.mode = 0;
    f.z = z;
    f.tg = target;
    f.mask = mask;
    f.B = B;
    f.N = N;
    f.iters = iters;
    f.trim = trim;
    f.min_points = min_points;
    f.st = st;
    f.info = info;
    f.workspace = workspace;
    f.workspace_bytes = workspace_bytes;
    return launch_fit(f, (hipStream_t)stream);
}

int pmg_fit_prompt(const float* logz, int64_t stride, const float* lidar, const float* conf, int B, int H, int W,
                   int dh, int dw, int iters, float trim, int min_points, float* st, int32_t* info,
                   void* workspace, size_t workspace_bytes, void* stream) {
    PMG_REQUIRE(logz && lidar && conf && st, "null buffer");
    PMG_REQUIRE(B >= 1 && H >= 1 && W >= 1 && dh >= 1 && dw >= 1 && stride >= 1, "bad shape");
    FitLaunch f{};
    f.mode = 1;
    f.logz = logz;
    f.stride = stride;
    f.lidar = lidar;
    f.conf = conf;
    f.B = B;
    f.H = H;
    f.W = W;
    f.dh = dh;
    f.dw = dw;
    f.N = (int64_t)H * W;
    f.iters = iters;
    f.trim = trim;
    f.min_points = min_points;
    f.st = st;
    f.info = info;
    f.workspace = workspace;
    f.workspace_bytes = workspace_bytes;
    return launch_fit(f, (hipStream_t)stream);
}

int pmg_post_depth(const float* logz, int64_t stride, const uint8_t* mask, int B, int H, int W, const float* st,
                   float* depth, void* stream) {
    PMG_REQUIRE(logz && st && depth, "null buffer");
    PMG_REQUIRE(B >= 1 && H >= 1 && W >= 1 && stride >= 1, "bad shape");
    const int64_t HW = (int64_t)H * W, n = (int64_t)B * HW;
    hipLaunchKernelGGL(post_depth_k, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, logz,
                       stride, mask, HW, n, st, depth);
    return check_launch("post_depth_k");
}

int pmg_fit_final(const float* logz, int64_t stride, const float* lidar, const float* conf, const uint8_t* mask_binary,
                  int B, int H, int W, int dh, int dw, int iters, float trim, int min_points, float* st, int32_t* info,
                  void* workspace, size_t workspace_bytes, void* stream) {
    FinalFit f{logz, stride, lidar, conf, mask_binary, B, H, W, dh, dw, iters, trim, min_points, st, info,
               workspace, workspace_bytes};
    return launch_final_fit(f, (hipStream_t)stream);
}

}  // extern "C"
