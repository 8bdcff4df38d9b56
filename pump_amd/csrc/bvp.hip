// bvp.hip -- kernel (a): 2pBVP optimal arrival time and cost for every
// ordered sample pair (reference: fillCoptsTopts, 2pBVP.cu:133-150), the
// cost-to-goal heuristic (mainPUMP.cu:351-355) and the FP64 Newton polish of
// arrival times.
//
// Pairs are enumerated in the output order idx = i*(num-1) + k (k skips the
// diagonal).  The reference's bisection (12.3 steps of two cost evaluations
// per pair on average for 16000 uniform samples) runs in two parts with the
// same decisions (pump_device.hpp): its leading steps from the sign of the
// derivative, 64 fresh pairs of a wave in lockstep, and the remaining ones
// (5.1 per pair and the final cost) by certified cost evaluations, as a
// per-lane state machine over persistent waves, since lanes need between 1
// and 32 of them.  The kernel is bound by VALU issue: 256 million pairs
// (16000 samples) in 7.9 ms, 3.2e10 pairs/s, against 17.3 ms with every step
// two full cost evaluations; a million pairs (1000 samples) 72 us against
// 590, 65 thousand 24 us against 45, where the longest lane's steps decide.
#include <algorithm>

#include "pump_device.hpp"
#include "pump_internal.hpp"

#pragma clang fp contract(off)

namespace pump {
namespace {

__device__ __forceinline__ void load_state(const float *__restrict__ s, int i, float *x)
{
    const float *p = s + (int64_t)i * kDim;
    for (int d = 0; d < kDim; ++d)
        x[d] = p[d];
}

__device__ __forceinline__ void pair_of(int64_t idx, int num, int &i, int &j)
{
    i = (int)(idx / (num - 1));
    int k = (int)(idx - (int64_t)i * (num - 1));
    j = k + (k >= i ? 1 : 0);
}

// A pair set up for the state machine, in the wave's LDS queue: its terms and
// bisection state, the states' indices, and the problem (batched launch).
struct alignas(16) PairEntry {
    PairTerms T;
    float tl, tu, x, w;
    int state_itr; // state in the low 3 bits
    int i, j, inst;
};
static_assert(sizeof(PairEntry) == 112, "28 dwords: seven 16-byte LDS accesses");

constexpr int kPairBlock = 256;
constexpr int kSet = 64;     // pairs set up together by a wave
// Idle lanes that are refilled together: 8, 16, 24, 32 give 8.25, 8.05, 8.27
// and 8.63 ms at 16000 samples.
constexpr int kRefill = 16;
constexpr int kMaxChunk = 2048; // pairs per claim of the work counter at most

// Pair sources: the states behind a global pair index, and where a finished
// pair's results go.  One instance, idx in the reference's output order.
// With fewer than 2^32 pairs the row i = g / (num - 1) is found by a
// multiply-high with the divisor's magic number (DivMagic).
struct OnePairSource {
    const float *samples;
    int num;
    float tmax;
    float *copts, *topts;
    DivMagic dm;
    __device__ void load(int64_t g, float *a, float *b, float &tm, int &i, int &j, int &) const
    {
        if (dm.m) {
            const uint32_t n = (uint32_t)g;
            const uint32_t q = div_magic_apply(n, dm);
            const int k = (int)(n - q * (uint32_t)(num - 1));
            i = (int)q;
            j = k + (k >= i ? 1 : 0);
        } else {
            pair_of(g, num, i, j);
        }
        load_state(samples, i, a);
        load_state(samples, j, b);
        tm = tmax;
    }
    __device__ void states(int i, int j, int, float *a, float *b) const
    {
        load_state(samples, i, a);
        load_state(samples, j, b);
    }
    __device__ void store(int i, int j, int, float tau, float cost) const
    {
        const int64_t o = (int64_t)i * (num - 1) + j - (j > i ? 1 : 0);
        topts[o] = tau;
        copts[o] = cost;
    }
};

// Every sample to the goal (mainPUMP.cu:351-355): the cost alone.
struct GoalSource {
    const float *samples;
    float goal[kDim];
    float tmax;
    float *h;
    __device__ void states(int i, int, int, float *a, float *b) const
    {
        load_state(samples, i, a);
        for (int d = 0; d < kDim; ++d)
            b[d] = goal[d];
    }
    __device__ void load(int64_t g, float *a, float *b, float &tm, int &i, int &, int &) const
    {
        i = (int)g;
        states(i, 0, 0, a, b);
        tm = tmax;
    }
    __device__ void store(int i, int, int, float, float cost) const { h[i] = cost; }
};

// Many instances: instance k owns global indices [prefix[k], prefix[k+1]).
// A lane keeps the range of the instance its last pair came from, so the
// search over the prefix table runs only when a lane crosses into another
// instance (a wave's chunks mostly lie inside one).
struct ManyPairSource {
    const PairJob *jobs;
    const int64_t *prefix;
    int n_inst;
    mutable int cur = 0;
    mutable int64_t cur_lo = 0, cur_hi = 0;
    __device__ void load(int64_t g, float *a, float *b, float &tm, int &i, int &j,
                         int &inst) const
    {
        if (!(g >= cur_lo && g < cur_hi)) {
            cur = instance_of(prefix, n_inst, g);
            cur_lo = prefix[cur];
            cur_hi = prefix[cur + 1];
        }
        const PairJob J = global_job(jobs[cur]);
        const int64_t idx = g - cur_lo;
        if (J.dm_m) {
            const uint32_t n = (uint32_t)idx;
            const uint32_t q = div_magic_apply(n, DivMagic{J.dm_m, J.dm_s1, J.dm_s2});
            const int k = (int)(n - q * (uint32_t)(J.num - 1));
            i = (int)q;
            j = k + (k >= i ? 1 : 0);
        } else {
            pair_of(idx, J.num, i, j);
        }
        inst = cur;
        load_state(J.samples, i, a);
        load_state(J.samples, j, b);
        tm = J.tmax;
    }
    __device__ void states(int i, int j, int inst, float *a, float *b) const
    {
        const float *s = gptr(jobs[inst].samples);
        load_state(s, i, a);
        load_state(s, j, b);
    }
    __device__ void store(int i, int j, int inst, float tau, float cost) const
    {
        const PairJob J = global_job(jobs[inst]);
        const int64_t o = (int64_t)i * (J.num - 1) + j - (j > i ? 1 : 0);
        J.topts[o] = tau;
        J.copts[o] = cost;
    }
};

// cost_eval from the states themselves, where cost_certified fails; out of
// line, so that its registers stay off the loop
__device__ __noinline__ float cost_of_states(float a0, float a1, float a2, float a3, float a4,
                                             float a5, float b0, float b1, float b2, float b3,
                                             float b4, float b5, float x)
{
    const float a[kDim] = {a0, a1, a2, a3, a4, a5}, b[kDim] = {b0, b1, b2, b3, b4, b5};
    CostTerms c;
    cost_terms(c, a, b);
    return cost_eval(c, x);
}

// A persistent wave.  It owns the first chunk with its own number and claims
// further ones from next_chunk (null: none).  Whenever kRefill lanes are
// idle, they store the results they finished with and take set-up pairs from
// the wave's queue; when that is empty the whole wave sets up the next kSet
// pairs (bisect_start) into it.  Every other lane then makes one step.
// steps_out (may be null) receives the number of toptBisection's steps over
// all pairs, the derivative's and the final cost's included.
template <class Src>
__device__ __forceinline__ void pairs_persistent(const Src &src, int64_t n_pairs, int chunk,
                                                 unsigned long long *__restrict__ next_chunk,
                                                 unsigned long long *__restrict__ steps_out)
{
    __shared__ PairEntry queue[kPairBlock / 64][kSet];
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    PairEntry *q = queue[wid];
    const int64_t n_waves = (int64_t)gridDim.x * (kPairBlock / 64);
    int64_t pool = ((int64_t)blockIdx.x * (kPairBlock / 64) + wid) * chunk;
    int64_t pool_end = pool + chunk < n_pairs ? pool + chunk : n_pairs;
    bool more = next_chunk != nullptr;
    int qh = 0, qn = 0; // the queue holds q[qh .. qn)

    PairTerms T;
    BisectState S;
    S.state = ST_IDLE;
    int i = 0, j = 0, inst = 0;
    float cost = 0.0f;
    int steps = 0;
    const auto cost_at = [&](float x) {
        float a[kDim], b[kDim];
        src.states(i, j, inst, a, b);
        return cost_of_states(a[0], a[1], a[2], a[3], a[4], a[5], b[0], b[1], b[2], b[3], b[4],
                              b[5], x);
    };

    while (true) {
        unsigned long long idle = __ballot(S.state >= ST_DONE);
        if (__popcll(idle) >= kRefill) {
            if (S.state == ST_DONE) {
                if (cost == 0.0f) // the sign of a zero
                    cost = cost_at(S.x);
                src.store(i, j, inst, S.x, cost);
                S.state = ST_IDLE;
            }
            while (idle) {
                if (qh == qn) {
                    if (pool >= pool_end) {
                        if (!more)
                            break;
                        unsigned long long claimed = 0;
                        if (lane == 0)
                            claimed = atomicAdd(next_chunk, (unsigned long long)chunk);
                        // every lane is active here, so the first active lane is lane 0
                        const uint32_t lo =
                            (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)claimed);
                        const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane(
                            (int)(uint32_t)(claimed >> 32));
                        pool = n_waves * chunk + (int64_t)(((uint64_t)hi << 32) | lo);
                        pool_end = pool + chunk < n_pairs ? pool + chunk : n_pairs;
                        if (pool >= n_pairs) {
                            more = false;
                            break;
                        }
                    }
                    const int n = pool_end - pool < kSet ? (int)(pool_end - pool) : kSet;
                    if (lane < n) {
                        PairEntry e;
                        DerivTerms D;
                        BisectState B;
                        float a[kDim], b[kDim], tmax;
                        e.i = e.j = e.inst = 0;
                        src.load(pool + lane, a, b, tmax, e.i, e.j, e.inst);
                        pair_terms(e.T, D, a, b);
                        bisect_start(D, tmax, B, steps);
                        e.tl = B.tl;
                        e.tu = B.tu;
                        e.x = B.x;
                        e.w = B.w;
                        e.state_itr = B.state | (B.itr << 3);
                        q[lane] = e;
                    }
                    pool += n;
                    qh = 0;
                    qn = n;
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                }
                const int rank = __popcll(idle & ((1ull << lane) - 1ull));
                const int n_idle = __popcll(idle);
                if (S.state == ST_IDLE && rank < qn - qh) {
                    const PairEntry e = q[qh + rank];
                    T = e.T;
                    S.tl = e.tl;
                    S.tu = e.tu;
                    S.x = e.x;
                    S.w = e.w;
                    S.state = e.state_itr & 7;
                    S.itr = e.state_itr >> 3;
                    i = e.i;
                    j = e.j;
                    inst = e.inst;
                }
                qh += n_idle < qn - qh ? n_idle : qn - qh;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                idle = __ballot(S.state == ST_IDLE);
            }
            if (idle == ~0ull)
                break; // nothing left to take
        }
        if (S.state < ST_DONE) {
            float xa, xb, ca, cb;
            int skipped;
            if (!bisect_costs(T, S, xa, xb, ca, cb)) {
                ca = cost_at(xa);
                cb = cost_at(xb);
            }
            cost = ca;
            bisect_update(S, ca, cb, skipped);
            steps += 1 + skipped;
        }
    }
    if (steps_out) {
        for (int off = 32; off > 0; off >>= 1)
            steps += __shfl_xor(steps, off, 64);
        if (lane == 0)
            atomicAdd(steps_out, (unsigned long long)steps);
    }
}

// A launch of one workgroup: each lane takes its pair to the end, without the
// queue and the refills.  10 samples to the goal take 6.6 us for 8.6, 64 take
// 11.4 for 15.3, all pairs of 16 samples 16-20 for 20; 300 samples to the goal
// 20.4 for 19.8 and 1000 26 for 22, so that it ends there.
template <class Src>
__device__ __forceinline__ void pairs_one_set(const Src &src, int64_t n_pairs)
{
    const int64_t g = (int64_t)blockIdx.x * kPairBlock + threadIdx.x;
    if (g >= n_pairs)
        return;
    PairTerms T;
    DerivTerms D;
    BisectState S;
    int i = 0, j = 0, inst = 0, steps = 0; // steps: not counted here
    float a[kDim], b[kDim], tmax, cost = 0.0f;
    src.load(g, a, b, tmax, i, j, inst);
    const auto cost_at = [&](float x) {
        float a[kDim], b[kDim];
        src.states(i, j, inst, a, b);
        return cost_of_states(a[0], a[1], a[2], a[3], a[4], a[5], b[0], b[1], b[2], b[3], b[4],
                              b[5], x);
    };
    pair_terms(T, D, a, b);
    bisect_start(D, tmax, S, steps);
    while (S.state < ST_DONE) {
        float xa, xb, ca, cb;
        if (!bisect_costs(T, S, xa, xb, ca, cb)) {
            ca = cost_at(xa);
            cb = cost_at(xb);
        }
        cost = ca;
        bisect_update(S, ca, cb, steps);
    }
    if (cost == 0.0f) // the sign of a zero
        cost = cost_at(S.x);
    src.store(i, j, inst, S.x, cost);
}

__global__ __launch_bounds__(kPairBlock) void k_fill_pairs_one_set(
    const float *__restrict__ samples, int num, float tmax, float *__restrict__ copts,
    float *__restrict__ topts, int64_t n_pairs, DivMagic dm)
{
    pairs_one_set(OnePairSource{samples, num, tmax, copts, topts, dm}, n_pairs);
}

__global__ __launch_bounds__(kPairBlock) void k_fill_pairs_persistent(
    const float *__restrict__ samples, int num, float tmax, float *__restrict__ copts,
    float *__restrict__ topts, int64_t n_pairs, DivMagic dm, int chunk,
    unsigned long long *__restrict__ next_chunk, unsigned long long *__restrict__ steps_out)
{
    const OnePairSource src{samples, num, tmax, copts, topts, dm};
    pairs_persistent(src, n_pairs, chunk, next_chunk, steps_out);
}

// all ordered pairs of many instances in one persistent launch
__global__ __launch_bounds__(kPairBlock) void k_fill_pairs_many(
    const PairJob *__restrict__ jobs, const int64_t *__restrict__ prefix, int n_inst,
    int64_t n_pairs, int chunk, unsigned long long *__restrict__ next_chunk)
{
    const ManyPairSource src{jobs, prefix, n_inst};
    pairs_persistent(src, n_pairs, chunk, next_chunk, nullptr);
}

// h[i] = cost(toptBisection(x_i, goal)) for i < num-1, h[num-1] = 0
template <bool kOneSet>
__global__ __launch_bounds__(kPairBlock) void k_heuristic(const GoalSource src, int num)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
        src.h[num - 1] = 0.0f;
    if constexpr (kOneSet)
        pairs_one_set(src, num - 1);
    else
        pairs_persistent(src, num - 1, kSet, nullptr, nullptr);
}

__global__ void k_zero_counter(unsigned long long *c)
{
    if (threadIdx.x == 0)
        *c = 0ull;
}

// FP64 polish of a bisected arrival time: the root of
//   q(t) = t^4 c'(t) = (1+g^2) t^4 - 4R t^2 + 24 S t - 36 D
// at the same local minimum.  A bracket [lo, hi] with q(lo) <= 0 <= q(hi) is
// grown geometrically around the bisection result (the float finite
// difference can stop anywhere within its noise, and at tmax it can read
// negative while c'(tmax) > 0), then safeguarded Newton steps converge to the
// last bit.  tmax is kept when c'(tmax) < 0 exactly.
__device__ __forceinline__ double q_of(double t, double k4, double D, double S, double R)
{
    return ((k4 * t * t - 4.0 * R) * t + 24.0 * S) * t - 36.0 * D;
}

__global__ __launch_bounds__(256) void k_polish(const float *__restrict__ samples, int num,
                                                float tmax, const float *__restrict__ topts,
                                                double *__restrict__ out, int64_t n_pairs)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const double k4 = 1.0 + (double)kGravity * (double)kGravity;
    const double tm = (double)tmax;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n_pairs;
         idx += stride) {
        int i, j;
        pair_of(idx, num, i, j);
        float a[kDim], b[kDim];
        load_state(samples, i, a);
        load_state(samples, j, b);
        double D = 0, S = 0, R = 0;
        for (int d = 0; d < 3; ++d) {
            double dp = (double)b[d] - (double)a[d];
            double v0 = a[d + 3], v1 = b[d + 3];
            D += dp * dp;
            S += dp * (v0 + v1);
            R += v0 * v0 + v0 * v1 + v1 * v1;
        }
        const double t0 = (double)topts[idx];
        double t = t0;
        if (t0 >= tm && q_of(tm, k4, D, S, R) < 0.0) {
            out[idx] = tm;
            continue;
        }
        double lo = t0, hi = t0;
        bool ok = false;
        for (int k = 0; k < 64; ++k) {
            double w = t0 * 1e-6 * (double)(1ull << (k < 60 ? k : 60));
            lo = fmax(t0 - w, 1e-9);
            hi = fmin(t0 + w, tm);
            if (q_of(lo, k4, D, S, R) <= 0.0 && q_of(hi, k4, D, S, R) >= 0.0) {
                ok = true;
                break;
            }
        }
        if (ok) {
            t = fmin(fmax(t0, lo), hi);
            for (int it = 0; it < 80; ++it) {
                double q = q_of(t, k4, D, S, R);
                if (q == 0.0)
                    break;
                if (q > 0.0)
                    hi = t;
                else
                    lo = t;
                double dq = (4.0 * k4 * t * t - 8.0 * R) * t + 24.0 * S;
                double tn = t - q / dq;
                if (!(tn > lo && tn < hi))
                    tn = 0.5 * (lo + hi);
                if (fabs(tn - t) <= 1e-16 * t) {
                    t = tn;
                    break;
                }
                t = tn;
            }
        }
        out[idx] = t;
    }
}

} // namespace
} // namespace pump

using namespace pump;

namespace pump {
// Launch shape of the persistent pair pass: the workgroups and the pairs per
// claim.  A launch with at most 16 sets of 64 pairs per resident wave is
// dealt out evenly (no claims, no counter): with so few, the claims
// themselves, which serialise on one address at about 12 ns each, would cost
// more than the unevenness.  Above that a wave's own first chunk is a
// quarter of its share, at least 8 sets (claims stay below the counter's
// rate) and at most kMaxChunk pairs.
struct PairShape {
    unsigned blocks;
    int chunk;
    bool claims;
};

static int pair_shape(int64_t n_pairs, int blocks_per_cu, PairShape &p)
{
    int dev = 0, cus = 256;
    PUMP_HIP(hipGetDevice(&dev));
    PUMP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t sets = (n_pairs + kSet - 1) / kSet;
    int64_t waves = (int64_t)cus * blocks_per_cu * (kPairBlock / 64);
    if (waves > sets)
        waves = sets;
    const int64_t per = (sets + waves - 1) / waves;
    p.claims = per > 16;
    const int64_t chunk = p.claims ? std::min<int64_t>(std::max<int64_t>(per / 4, 8) * kSet, kMaxChunk)
                                   : per * kSet;
    p.chunk = (int)chunk;
    if (!p.claims) // the waves that have a chunk
        waves = (n_pairs + chunk - 1) / chunk;
    p.blocks = (unsigned)((waves + kPairBlock / 64 - 1) / (kPairBlock / 64));
    return PUMP_OK;
}

constexpr int kPairBlocksPerCu = 4; // what 111 VGPRs keep resident

// All ordered pairs of one instance; *steps (may be null) receives the
// bisection steps of all pairs, 0 for a launch below 65,536 pairs (not
// counted there).
int fill_copts_topts(const float *d_samples, int num, float tmax, float *d_copts, float *d_topts,
                     hipStream_t s, int64_t *steps)
{
    PUMP_REQUIRE(d_samples && d_copts && d_topts && num >= 2);
    const int64_t n_pairs = (int64_t)num * (num - 1);
    if (steps)
        *steps = 0;
    if (n_pairs < (1 << 16))
        steps = nullptr;
    PairShape p;
    const int r = pair_shape(n_pairs, kPairBlocksPerCu, p);
    if (r != PUMP_OK)
        return r;
    const DivMagic dm = n_pairs < (1ll << 32) ? div_magic((uint32_t)(num - 1)) : DivMagic{0, 0, 0};
    if (n_pairs <= kPairBlock) {
        hipLaunchKernelGGL(k_fill_pairs_one_set, dim3(p.blocks), dim3(kPairBlock), 0, s, d_samples,
                           num, tmax, d_copts, d_topts, n_pairs, dm);
        PUMP_LAUNCHED();
        return PUMP_OK;
    }
    if (!p.claims && !steps) {
        hipLaunchKernelGGL(k_fill_pairs_persistent, dim3(p.blocks), dim3(kPairBlock), 0, s, d_samples, num,
                           tmax, d_copts, d_topts, n_pairs, dm, p.chunk,
                           (unsigned long long *)nullptr, (unsigned long long *)nullptr);
        PUMP_LAUNCHED();
        return PUMP_OK;
    }
    // [0]: work counter, [1]: step count
    unsigned long long *counter = nullptr;
    PUMP_HIP(hipMalloc((void **)&counter, 2 * sizeof(unsigned long long)));
    hipError_t me = hipMemsetAsync(counter, 0, 2 * sizeof(unsigned long long), s);
    if (me != hipSuccess) {
        hipFree(counter);
        PUMP_HIP(me);
    }
    hipLaunchKernelGGL(k_fill_pairs_persistent, dim3(p.blocks), dim3(kPairBlock), 0, s, d_samples,
                       num, tmax, d_copts, d_topts, n_pairs, dm, p.chunk,
                       p.claims ? counter : nullptr, steps ? counter + 1 : nullptr);
    hipError_t le = hipGetLastError();
    hipError_t se = hipStreamSynchronize(s);
    unsigned long long n_steps = 0;
    if (le == hipSuccess && se == hipSuccess && steps)
        se = hipMemcpy(&n_steps, counter + 1, sizeof(n_steps), hipMemcpyDeviceToHost);
    hipFree(counter);
    PUMP_HIP(le);
    PUMP_HIP(se);
    if (steps)
        *steps = (int64_t)n_steps;
    return PUMP_OK;
}
} // namespace pump

extern "C" int pump_fill_copts_topts(const float *d_samples, int num, float tmax, float *d_copts,
                                     float *d_topts, pump_stream_t stream)
{
    return pump::fill_copts_topts(d_samples, num, tmax, d_copts, d_topts, as_stream(stream),
                                  nullptr);
}

extern "C" int pump_polish_topts(const float *d_samples, int num, float tmax, const float *d_topts,
                                 double *d_topts64, pump_stream_t stream)
{
    PUMP_REQUIRE(d_samples && d_topts && d_topts64 && num >= 2);
    const int64_t n_pairs = (int64_t)num * (num - 1);
    hipLaunchKernelGGL(k_polish, dim3(grid_for(n_pairs, 256)), dim3(256), 0, as_stream(stream),
                       d_samples, num, tmax, d_topts, d_topts64, n_pairs);
    PUMP_LAUNCHED();
    return PUMP_OK;
}

extern "C" int pump_heuristic(const float *d_samples, int num, const float *goal_host, float tmax,
                              float *d_h, pump_stream_t stream)
{
    PUMP_REQUIRE(d_samples && goal_host && d_h && num >= 1);
    GoalSource src{d_samples, {}, tmax, d_h};
    for (int d = 0; d < kDim; ++d)
        src.goal[d] = goal_host[d];
    // a set of 64 samples per wave
    const unsigned blocks = (unsigned)((num + kPairBlock - 1) / kPairBlock);
    hipLaunchKernelGGL(blocks == 1 ? k_heuristic<true> : k_heuristic<false>, dim3(blocks),
                       dim3(kPairBlock), 0, as_stream(stream), src, num);
    PUMP_LAUNCHED();
    return PUMP_OK;
}

namespace pump {
// Many instances' pairs in one persistent launch (jobs and prefix in device
// memory; prefix[n_inst] = n_pairs).  The chunk counter is cleared by a
// kernel, so the sequence can be captured in a graph.
int fill_pairs_many(const PairJob *d_jobs, const int64_t *d_prefix, int n_inst, int64_t n_pairs,
                    int blocks_per_cu, unsigned long long *d_counter, hipStream_t s)
{
    PUMP_REQUIRE(d_jobs && d_prefix && d_counter && n_inst > 0 && n_pairs >= 0 &&
                 blocks_per_cu > 0);
    if (n_pairs == 0)
        return PUMP_OK;
    PairShape p;
    const int r = pair_shape(n_pairs, blocks_per_cu, p);
    if (r != PUMP_OK)
        return r;
    if (p.claims) {
        hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(64), 0, s, d_counter);
        PUMP_LAUNCHED();
    }
    hipLaunchKernelGGL(k_fill_pairs_many, dim3(p.blocks), dim3(kPairBlock), 0, s, d_jobs,
                       d_prefix, n_inst, n_pairs, p.chunk, p.claims ? d_counter : nullptr);
    PUMP_LAUNCHED();
    return PUMP_OK;
}
} // namespace pump

