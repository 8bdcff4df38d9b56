// mccp.hip -- full Monte Carlo collision probability (reference:
// collisionProbability + MCCP, collisionProbability.cu:4-92).
//
// The reference runs one thread per particle in 32 workgroups of 64 and walks
// the path's segments serially.  Here a workgroup owns 64 particles of one
// path, one per lane of each of its waves (small launches: 16, each on four
// lanes), and the waves share the path's segments.  At one segment the 64
// particles lie within the noise of one another, so few boxes meet the union
// of their segment boxes and only those are tested lane by lane; the boxes are
// tested against the union 64 at a time.  (Lanes over the segments of one
// particle had the whole path's extent as union, and idle lanes past its end:
// 64 paths of 4096 particles among 200 walls, 43 segments each, took 197 us,
// 5.7e10 segment-checks/s, and take 40 us, 2.8e11.)  Bound there: VALU issue
// (70% busy by four cycles an instruction; of 110 instructions per segment and
// wave 48 are the bounds' reductions) and the waves' chains of segments; 64
// paths of 2048 particles among 30 boxes, 28% busy, by the chains.  The noise
// rows are read a lane each, uncoalesced, from L2.  Paths of a batch are the grid's y dimension.
#include "pump_device.hpp"
#include "pump_internal.hpp"

#pragma clang fp contract(off)

namespace pump {
namespace {

constexpr int kMaxWaves = 16; // waves of a workgroup at most
// Waves of a launch, where the path count and particles leave fewer: 4096,
// 8192, 16384, 32768 give 46, 43, 40, 44 us for 64 paths of 4096 particles
// among 200 walls, 20, 18, 20, 23 for 32 paths among 64.
constexpr int kTargetWaves = 16384;
// A launch of few groups of 64 particles is one chain of a wave's segments
// long, on a few compute units: up to kSplitGroups of them a particle gets
// kSplit lanes with a run of segments each.  One path of 1024 particles, 64
// and 200 boxes: 4.6 and 4.7 us, 6.3 and 6.2 with one lane; 128 groups (8192
// particles) 6.2 and 5.0, 7.0 and 5.5; 192 groups 6.9 and 6.7, 6.4 and 6.3.
constexpr int kSplit = 4, kSplitGroups = 128;
// More than 64 boxes are held in registers where a wave has segments enough
// to use them on: from kRegisterWaves waves per workgroup down (11 segments of
// 43 each).  64 paths of 4096 particles, 128 and 256 boxes: 34 and 43 us, from
// memory 36 and 48; 32 paths (8 waves) 22 and 31, from memory 21 and 26; 16
// paths (16 waves) 18 and 30, from memory 14 and 17.
constexpr int kRegisterWaves = 4;

// kBoxes: boxes per lane held in registers (0: any count, from global memory).
// kSub: lanes per particle, each with segments of its own; 64 / kSub particles
// per workgroup.
template <int kBoxes, int kSub>
__global__ __launch_bounds__(64 * kMaxWaves) void k_mccp(
    const float *__restrict__ obstacles, int n_obs, const float *__restrict__ xcomb,
    int tmax_steps, int n_mc, float om, const float *__restrict__ paths, int64_t stride_rows,
    const int *__restrict__ Ts, int *__restrict__ hits)
{
    __shared__ unsigned long long hit_mask[kMaxWaves];
    const int k = blockIdx.y;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_waves = blockDim.x >> 6;
    const int mine = blockIdx.x * (64 / kSub) + lane / kSub;
    const int p = mine < n_mc ? mine : n_mc - 1; // idle lanes repeat the last
    const float *path = paths + (int64_t)k * stride_rows * kDim;
    // segments t < T-2 (the reference skips the final segment); bounded by
    // the noise table and the path buffer
    int nseg = Ts[k] - 2;
    if (nseg > tmax_steps - 1)
        nseg = tmax_steps - 1;
    if (nseg > (int)stride_rows - 1)
        nseg = (int)stride_rows - 1;
    // Segments in kSub runs per wave of chunk each: lane l % kSub = 0 goes from
    // u = t0 to t1, the others that many chunks ahead.  A lane past the last
    // segment waits there.
    const int chunk = (nseg + kSub * n_waves - 1) / (kSub * n_waves);
    const int t0 = wid * kSub * chunk, t1 = t0 + chunk < nseg ? t0 + chunk : nseg;
    const int ahead = kSub > 1 ? lane % kSub * chunk : 0;
    const auto seg = [&](int u) { return kSub > 1 ? min(u + ahead, nseg - 1) : u; };
    // this lane's boxes: lane, lane + 64, ...
    constexpr int kRegs = kBoxes > 0 ? kBoxes : 1;
    float blo[kRegs][3], bhi[kRegs][3];
    if (kBoxes > 0) {
#pragma unroll
        for (int c = 0; c < kRegs; ++c) {
            const int b = c * 64 + lane;
            for (int d = 0; d < 3; ++d) {
                blo[c][d] = b < n_obs ? obstacles[b * 12 + d] : INFINITY;
                bhi[c][d] = b < n_obs ? obstacles[b * 12 + 6 + d] : -INFINITY;
            }
        }
    }
    const float *xc = xcomb + (int64_t)p * 3 * tmax_steps;
    bool hit = false;
    if (t0 < t1) {
        // the first point, and the next point's noise loaded ahead
        float v[3], xn[3];
        int vmin[3], vmax[3]; // bounds over the wave, as ordered integers
        for (int d = 0; d < 3; ++d) {
            v[d] = path[seg(t0) * kDim + d] + xc[seg(t0) * 3 + d] * om;
            xn[d] = xc[(seg(t0) + 1) * 3 + d];
        }
        for (int d = 0; d < 3; ++d) {
            const int i = ordered_int(__float_as_int(v[d]));
            vmin[d] = wave_min_i(i);
            vmax[d] = wave_max_i(i);
        }
        for (int u = t0; u < t1; ++u) {
            const int t = seg(u);
            const bool done = kSub > 1 && u + ahead >= nseg;
            float w[3];
            int wmin[3], wmax[3];
            for (int d = 0; d < 3; ++d)
                w[d] = path[(t + 1) * kDim + d] + xn[d] * om;
            if (u + 1 < t1)
                for (int d = 0; d < 3; ++d)
                    xn[d] = xc[(seg(u + 1) + 1) * 3 + d];
            // The union of the particles' segment boxes: a box separated from
            // it (the broad phase's own <= test) is separated from each.
            float umin[3], umax[3];
            for (int d = 0; d < 3; ++d) {
                const int i = ordered_int(__float_as_int(w[d]));
                wmin[d] = wave_min_i(i);
                wmax[d] = wave_max_i(i);
                umin[d] = __int_as_float(ordered_int(min(vmin[d], wmin[d])));
                umax[d] = __int_as_float(ordered_int(max(vmax[d], wmax[d])));
            }
            float bmin[3], bmax[3];
            seg_bbox(v, w, bmin, bmax);
            const auto meets = [&](const float *lo, const float *hi) {
                return !((umax[0] <= lo[0]) | (hi[0] <= umin[0]) | (umax[1] <= lo[1]) |
                         (hi[1] <= umin[1]) | (umax[2] <= lo[2]) | (hi[2] <= umin[2]));
            };
            if (kBoxes > 0) {
#pragma unroll
                for (int c = 0; c < kRegs; ++c) {
                    unsigned long long cand = __ballot(meets(blo[c], bhi[c]));
                    while (cand) {
                        const int l = __builtin_ctzll(cand);
                        cand &= cand - 1;
                        float lo[3], hi[3];
                        for (int d = 0; d < 3; ++d) {
                            lo[d] = read_lane(blo[c][d], l);
                            hi[d] = read_lane(bhi[c][d], l);
                        }
                        if (!(hit || done))
                            hit = segment_hits_box(v, w, bmin, bmax, lo, hi);
                    }
                }
            } else {
                for (int b0 = 0; b0 < n_obs; b0 += 64) {
                    const int b = b0 + lane;
                    float lo[3] = {INFINITY, INFINITY, INFINITY};
                    float hi[3] = {-INFINITY, -INFINITY, -INFINITY};
                    if (b < n_obs)
                        for (int d = 0; d < 3; ++d) {
                            lo[d] = obstacles[(int64_t)b * 12 + d];
                            hi[d] = obstacles[(int64_t)b * 12 + 6 + d];
                        }
                    unsigned long long cand = __ballot(b < n_obs && meets(lo, hi));
                    while (cand) {
                        const int l = __builtin_ctzll(cand);
                        cand &= cand - 1;
                        float clo[3], chi[3];
                        for (int d = 0; d < 3; ++d) {
                            clo[d] = read_lane(lo[d], l);
                            chi[d] = read_lane(hi[d], l);
                        }
                        if (!(hit || done))
                            hit = segment_hits_box(v, w, bmin, bmax, clo, chi);
                    }
                }
            }
            if (__ballot(hit) == ~0ull)
                break;
            for (int d = 0; d < 3; ++d) {
                v[d] = w[d];
                vmin[d] = wmin[d];
                vmax[d] = wmax[d];
            }
        }
    }
    const unsigned long long m = __ballot(hit && mine < n_mc);
    if (lane == 0)
        hit_mask[wid] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long all = 0;
        for (int i = 0; i < n_waves; ++i)
            all |= hit_mask[i];
        for (int b = kSub / 2; b > 0; b /= 2) // a particle's lanes to its first
            all |= all >> b;
        if (kSub > 1)
            all &= ~0ull / ((1ull << (kSub % 64)) - 1ull);
        if (all)
            atomicAdd(&hits[k], __popcll(all));
    }
}

__global__ void k_zero_hits(int *h, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x)
        h[i] = 0;
}

} // namespace
} // namespace pump

using namespace pump;

extern "C" int pump_collision_probability_many(const float *d_obstacles, int n_obs,
                                               const float *d_xcomb, int tmax_steps, int n_mc,
                                               float offset_mult, const float *d_paths,
                                               int64_t path_stride_rows, const int *d_T,
                                               int n_paths, int *d_hits, int zero_hits,
                                               pump_stream_t stream)
{
    PUMP_REQUIRE(n_paths >= 0 && n_obs >= 0 && n_mc > 0 && tmax_steps > 0);
    if (n_paths == 0)
        return PUMP_OK;
    PUMP_REQUIRE(d_xcomb && d_paths && d_T && d_hits && path_stride_rows > 0);
    PUMP_REQUIRE(n_obs == 0 || d_obstacles);
    if (n_paths > 65535)
        return PUMP_E_RANGE;
    hipStream_t s = as_stream(stream);
    if (zero_hits) {
        hipLaunchKernelGGL(k_zero_hits, dim3(1), dim3(256), 0, s, d_hits, n_paths);
        PUMP_LAUNCHED();
    }
    // waves per workgroup: enough that the launch has kTargetWaves of them
    unsigned groups = (unsigned)((n_mc + 63) / 64);
    const bool split = (int64_t)groups * n_paths <= kSplitGroups;
    if (split)
        groups = (unsigned)((n_mc + 64 / kSplit - 1) / (64 / kSplit));
    int waves = 1;
    while (waves < kMaxWaves && (int64_t)groups * n_paths * waves < kTargetWaves)
        waves *= 2;
    const dim3 grid(groups, (unsigned)n_paths), block(64 * waves);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, d_obstacles, n_obs, d_xcomb, tmax_steps,
                           n_mc, offset_mult, d_paths, path_stride_rows, d_T, d_hits);
    };
    if (split)
        launch(k_mccp<0, kSplit>);
    else if (n_obs <= 64)
        launch(k_mccp<1, 1>);
    else if (n_obs <= 128 && waves <= kRegisterWaves)
        launch(k_mccp<2, 1>);
    else if (n_obs <= 256 && waves <= kRegisterWaves)
        launch(k_mccp<4, 1>);
    else
        launch(k_mccp<0, 1>);
    PUMP_LAUNCHED();
    return PUMP_OK;
}

extern "C" int pump_collision_probability(const float *d_obstacles, int n_obs,
                                          const float *d_xcomb, int tmax_steps, int n_mc,
                                          float offset_mult, const float *d_path, int T,
                                          float *cp_host, pump_stream_t stream)
{
    PUMP_REQUIRE(cp_host && d_path && T >= 0);
    if (T > tmax_steps + 1)
        return PUMP_E_RANGE;
    hipStream_t s = as_stream(stream);
    int *scratch = nullptr; // [0] = T, [1] = hits
    PUMP_HIP(hipMalloc((void **)&scratch, 2 * sizeof(int)));
    int hostT[2] = {T, 0};
    hipError_t ce = hipMemcpyAsync(scratch, hostT, 2 * sizeof(int), hipMemcpyHostToDevice, s);
    int r = PUMP_OK;
    if (ce == hipSuccess)
        r = pump_collision_probability_many(d_obstacles, n_obs, d_xcomb, tmax_steps, n_mc,
                                            offset_mult, d_path, T > 1 ? T : 1, scratch, 1,
                                            scratch + 1, 0, stream);
    int hits = 0;
    hipError_t de = hipMemcpyAsync(&hits, scratch + 1, sizeof(int), hipMemcpyDeviceToHost, s);
    hipError_t se = hipStreamSynchronize(s);
    hipFree(scratch);
    PUMP_HIP(ce);
    PUMP_HIP(de);
    PUMP_HIP(se);
    if (r != PUMP_OK)
        return r;
    *cp_host = ((float)hits) / ((float)n_mc);
    return PUMP_OK;
}
