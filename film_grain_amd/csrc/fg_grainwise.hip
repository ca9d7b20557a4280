// fg_grainwise.hip -- gfx950 grain-wise Boolean-model integrator.
//
// Computes exactly what render_grainwise computes (src/grainwise.rs:12-142):
// every input pixel (x, y) with lambda > 0 seeds pixel_rng(seed, x, y), draws
// q ~ Poisson(lambda) grains (centre (x + U, y + U), radius clamped to rm),
// and for every Monte-Carlo offset k each grain sets bit k of the output pixels
// whose centres (o + 0.5) lie in the disk of radius r*zoom around
// (cx*zoom + off_k.x, cy*zoom + off_k.y), using the reference's bounds()
// rounding.  The output is popcount(bits) * (1/N).
//
// Each workgroup owns an output tile and keeps the tile's N-bit sample sets in
// LDS, so the per-hit atomics are LDS atomics and the popcount epilogue writes
// each output pixel once.  It regenerates the grains of every input pixel whose
// grains can reach the tile (tile / zoom plus a halo of rm*zoom + max|offset|).
// Grain generation and grain testing alternate in rounds: each thread draws up
// to grains_per_thread grains of its input pixel into its LDS slots (keeping
// its Xoshiro state in registers between rounds), then all threads test all
// slotted grains with lanes over samples k, so the 64 lanes of a wave test one
// grain against 64 different offsets and the grain is a uniform (broadcast)
// LDS read.
#include <algorithm>

#include "fg_device.h"
#include "fg_pixelwise_hbm.h"

namespace fg {

// src/grainwise.rs:126-142, with the image limit; returns false for None.
__device__ __forceinline__ bool ref_bounds(float center, float radius, int limit, int &lo, int &hi)
{
    int mn = sat_i32(ceilf((center - radius) - 0.5f));
    int mx = sat_i32(floorf((center + radius) - 0.5f));
    if (mx < mn) return false;
    if (limit <= 0) return false;
    const int last = limit - 1;
    if (mn > last || mx < 0) return false;
    mn = min(max(mn, 0), last);
    mx = min(max(mx, 0), last);
    if (mn > mx) return false;
    lo = mn;
    hi = mx;
    return true;
}

template <int KIND, bool STATS>
__global__ __launch_bounds__(kBlock) void grainwise_tiles(GrainArgs a)
{
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ uint32_t s_slot_n[kBlock];

    const int tid = threadIdx.x;
    const int tile = blockIdx.x;
    if (tile >= a.n_tiles) return;
    const int tyi = tile / a.tiles_x, txi = tile - tyi * a.tiles_x;
    const int X0 = txi * a.tile_w, Y0 = tyi * a.tile_h;
    const int X1 = min(X0 + a.tile_w, a.out_w), Y1 = min(Y0 + a.tile_h, a.out_h);
    const int words = a.words;
    const int gpt = a.grains_per_thread;
    const int tile_px = a.tile_w * a.tile_h;

    uint32_t *bits = reinterpret_cast<uint32_t *>(lds);
    const size_t bits_bytes = (((size_t)tile_px * words * 4) + 15) & ~(size_t)15;
    float4 *slots = reinterpret_cast<float4 *>(lds + bits_bytes);

    for (int w = tid; w < tile_px * words; w += kBlock) bits[w] = 0u;

    // Input pixels whose grains can reach [X0, X1) x [Y0, Y1): centre in
    // [x, x+1], target t = cx*zoom + off, covered outputs within t +- R - 0.5.
    // The margins are generous; extra pixels only produce misses.
    const float z = a.zoom, R = a.r_out_max;
    const float4 orange = *a.off_range;
    const int xi0 = max(0, (int)floorf(((float)X0 + 0.5f - R - orange.y) / z) - 2);
    const int xi1 = min(a.in_w - 1, (int)ceilf(((float)X1 - 0.5f + R - orange.x) / z) + 2);
    const int yi0 = max(0, (int)floorf(((float)Y0 + 0.5f - R - orange.w) / z) - 2);
    const int yi1 = min(a.in_h - 1, (int)ceilf(((float)Y1 - 0.5f + R - orange.z) / z) + 2);
    const int rwi = xi1 - xi0 + 1;
    const int npx = (xi1 >= xi0 && yi1 >= yi0) ? rwi * (yi1 - yi0 + 1) : 0;

    // Test-phase mapping: lanes over samples, groups over grains.
    const int KL = a.n_samples >= kBlock ? kBlock : a.n_samples;
    const int GS = kBlock / KL;
    const int kl = tid % KL, gs = tid / KL;
    const bool tester = tid < KL * GS;

    const float uscale1 = 1.0f;  // Uniform::new(0.0f32, 1.0) keeps scale 1
    // instrumented twin: disk tests and hits of the tile's own pixels (each
    // output pixel lies in one tile, so the sums over tiles are the
    // reference's); grains and pairs are counted once per grain by
    // grain_count_kernel, since tiles regenerate their halo's grains
    unsigned long long st_tests = 0, st_hits = 0;
    __syncthreads();

    for (int pb = 0; pb < npx; pb += kBlock) {
        const int pix = pb + tid;
        Xoshiro rng;
        rng.s0 = rng.s1 = rng.s2 = rng.s3 = 0;
        uint32_t q = 0, done = 0;
        float fx = 0.0f, fy = 0.0f;
        if (pix < npx) {
            const int x = xi0 + pix % rwi, y = yi0 + pix / rwi;
            const float lam = a.lambda[(size_t)y * a.in_w + x];
            if (lambda_invalid(lam)) atomicOr(a.status, kStatusLambda);
            if (lam > 0.0f && lam <= kMaxLambda) {
                rng.seed(mix3(a.seed, kPixelStream, x, y));
                q = poisson_u32(rng, (double)lam);
            }
            fx = (float)x;
            fy = (float)y;
        }
        while (__syncthreads_or(done < q)) {
            int n = 0;
            while (n < gpt && done < q) {
                const float cx = fx + uniform_f32(rng, uscale1);
                const float cy = fy + uniform_f32(rng, uscale1);
                float rad = KIND == 0 ? a.r_const : lognormal_f32(rng, a.log_mu, a.log_sigma, d_zig_x, d_zig_f);
                ++done;
                if (rad > a.rm) rad = a.rm;
                if (rad <= 0.0f) continue;
                const float rout = rad * z;
                if (rout <= 0.0f) continue;
                slots[tid * gpt + n] = make_float4(cx * z, cy * z, rout, rout * rout);
                ++n;
            }
            s_slot_n[tid] = (uint32_t)n;
            __syncthreads();
            if (tester) {
                for (int b = 0; b < kBlock; ++b) {
                    const int nb = (int)s_slot_n[b];
                    for (int g = gs; g < nb; g += GS) {
                        const float4 G = slots[b * gpt + g];
                        for (int k = kl; k < a.n_samples; k += KL) {
                            const float2 o = a.offs[k];
                            const float txp = G.x + o.x, typ = G.y + o.y;
                            int xmn, xmx, ymn, ymx;
                            if (!ref_bounds(txp, G.z, a.out_w, xmn, xmx)) continue;
                            if (!ref_bounds(typ, G.z, a.out_h, ymn, ymx)) continue;
                            xmn = max(xmn, X0);
                            xmx = min(xmx, X1 - 1);
                            ymn = max(ymn, Y0);
                            ymx = min(ymx, Y1 - 1);
                            const uint32_t mask = 1u << (k & 31);
                            const int wk = k >> 5;
                            for (int oy = ymn; oy <= ymx; ++oy) {
                                const float dy = ((float)oy + 0.5f) - typ;
                                const float dy2 = dy * dy;
                                if (dy2 > G.w) continue;
                                for (int ox = xmn; ox <= xmx; ++ox) {
                                    const float dx = ((float)ox + 0.5f) - txp;
                                    if (STATS) ++st_tests;
                                    if (dx * dx + dy2 <= G.w) {
                                        atomicOr(&bits[((oy - Y0) * a.tile_w + (ox - X0)) * words + wk], mask);
                                        if (STATS) ++st_hits;
                                    }
                                }
                            }
                        }
                    }
                }
            }
            __syncthreads();
        }
    }

    // popcount epilogue: one store per output pixel of the tile
    const int tw = X1 - X0, th = Y1 - Y0;
    for (int p = tid; p < tw * th; p += kBlock) {
        const int ox = p % tw, oy = p / tw;
        const uint32_t *pw = bits + ((size_t)oy * a.tile_w + ox) * words;
        uint32_t count = 0;
        for (int w = 0; w < words; ++w) count += __popc(pw[w]);
        a.out[(size_t)(Y0 + oy) * a.out_w + (X0 + ox)] = (float)count * a.inv_samples;
    }
    if (STATS) {
        atomicAdd(&a.stats[2], st_tests);
        atomicAdd(&a.stats[3], st_hits);
    }
}

// ---------------------------------------------------------------------------
// Sorted-sample formulation (same result, far fewer (grain, sample) pairs)
// ---------------------------------------------------------------------------
// For grain centre t = cx*zoom and sample k, bounds() has a column iff some
// integer n lies in [(t + X_k - R) - 0.5, (t + X_k + R) - 0.5], i.e. iff
// frac(X_k) lies in the cyclic interval [A - 2R, A] with A = frac(R - (t -
// 0.5)).  With the samples ordered by frac(X_k) (SampleTable, built from the
// output-pixel offsets) those samples are one cyclic run, found through the
// bucket index; the interval is widened by the table's eps, so the run holds
// every such sample.  For narrow grains, candidate lists per radius class and
// cell of both fractions (grain_lists_kernel) replace the run.
// Each lane owns one input pixel of the tile's halo region: it draws that
// pixel's grains in the reference's order and, per grain, walks its list or
// run.  A listed grain, and a (grain, sample) pair whose bounds() box, clipped to
// the tile, is one pixel, takes the reference's disk test in the lane; larger boxes go to the
// wave's queue, one entry per pixel of the box inside the tile, drained
// through the same test.  Hits go to the tile's LDS bitset.
// Poisson pre-pass (src/grainwise.rs:37-45): per input pixel with lambda > 0,
// pixel_rng and the grain count; the count and the stream's state after the
// count draws are stored so that the splat kernel resumes each pixel's stream
// where the reference does (keeps the large Poisson sampler out of the splat
// kernel's registers).  Pixels with lambda <= 0 get q = 0.
//
// Bound by instruction issue (f64 logarithms, divisions and tangents).  A wave
// takes 64 pixels at a time through the setup and one attempt of the rejection
// sampler (lambda >= 12); the streams that were rejected, about half, wait in
// the wave's LDS queue and are tried again 64 at a time as soon as there are
// as many, the last ones at the wave's end.  (The wave's LDS accesses run in
// order, so no barrier is needed.)  A 4096x4096 plane with about 90 grains a
// pixel takes 1.05 ms; one pixel a lane until it was accepted took 1.83, with
// 24 of 64 lanes busy.
constexpr int kStateQueue = 128;  // entries: below 64 before a push of up to 64

struct StateQueue {
    uint64_t s[4][kStateQueue];
    double c[3][kStateQueue];  // PoissonReject's log_lambda, sqrt_2lambda, magic
    uint64_t pixel[kStateQueue];
    float lambda[kStateQueue];
};

__device__ __forceinline__ void put_pixel_state(const GrainArgs &a, long long p, uint32_t q, const Xoshiro &rng)
{
    a.pix_q[p] = q;
    a.pix_s01[p] = make_ulonglong2(rng.s0, rng.s1);
    a.pix_s23[p] = make_ulonglong2(rng.s2, rng.s3);
}

__global__ __launch_bounds__(kBlock) void pixel_state_kernel(GrainArgs a)
{
    __shared__ StateQueue s_queue[kBlock / 64];
    const int lane = threadIdx.x & 63;
    StateQueue &sq = s_queue[threadIdx.x >> 6];
    const long long n = (long long)a.in_w * a.in_h;
    const long long stride = (long long)gridDim.x * kBlock;
    long long base = (long long)blockIdx.x * kBlock + (threadIdx.x & ~63);
    int queued = 0;  // uniform
    while (base < n || queued > 0) {
        Xoshiro rng;
        rng.s0 = rng.s1 = rng.s2 = rng.s3 = 0;
        long long p;
        bool on;  // the lane takes an attempt
        PoissonReject pr(12.0, 0.0, 0.0, 0.0);
        if (queued < 64 && base < n) {  // 64 new pixels
            p = base + lane;
            base += stride;
            const bool in = p < n;
            const float lam = in ? a.lambda[p] : 0.0f;
            // values outside the accepted range are skipped and flagged (once per wave)
            if (__ballot(lambda_invalid(lam)) != 0ull && lane == 0) atomicOr(a.status, kStatusLambda);
            const bool drawn = lam > 0.0f && lam <= kMaxLambda;
            on = drawn && (double)lam >= 12.0;
            uint32_t q = 0;
            if (drawn) {
                const int y = (int)(p / a.in_w), x = (int)(p - (long long)y * a.in_w);
                rng.seed(mix3(a.seed, kPixelStream, x, y));
                if (!on) q = poisson_knuth(rng, (double)lam);
            }
            if (in && !on) put_pixel_state(a, p, q, rng);
            if (on) pr = PoissonReject((double)lam);
        } else {  // the queue's last ones again
            const int m = min(queued, 64);
            queued -= m;
            on = lane < m;
            const int slot = queued + (on ? lane : 0);
            rng.s0 = sq.s[0][slot];
            rng.s1 = sq.s[1][slot];
            rng.s2 = sq.s[2][slot];
            rng.s3 = sq.s[3][slot];
            pr = PoissonReject((double)sq.lambda[slot], sq.c[0][slot], sq.c[1][slot], sq.c[2][slot]);
            p = (long long)sq.pixel[slot];
            __builtin_amdgcn_wave_barrier();
        }
        bool again = false;
        if (on) {
            double r = 0.0;
            again = !pr.attempt(rng, &r);
            if (!again) put_pixel_state(a, p, poisson_count(r), rng);
        }
        const unsigned long long m = __ballot(again);
        const int slot = queued + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (again) {
            sq.s[0][slot] = rng.s0;
            sq.s[1][slot] = rng.s1;
            sq.s[2][slot] = rng.s2;
            sq.s[3][slot] = rng.s3;
            sq.c[0][slot] = pr.log_lambda;
            sq.c[1][slot] = pr.sqrt_2lambda;
            sq.c[2][slot] = pr.magic;
            sq.pixel[slot] = (uint64_t)p;
            sq.lambda[slot] = (float)pr.lambda;
        }
        queued += __popcll(m);
        __builtin_amdgcn_wave_barrier();
    }
}

// Instrumented twin, per input pixel: the grains the reference draws with a
// positive output radius (src/grainwise.rs:46-66), each of which it pairs with
// every sample.  stats[0] += grains, stats[1] += grains * N.
template <int KIND>
__global__ __launch_bounds__(kBlock) void grain_count_kernel(GrainArgs a)
{
    const long long n = (long long)a.in_w * a.in_h;
    unsigned long long cnt = 0;
    for (long long p = (long long)blockIdx.x * kBlock + threadIdx.x; p < n; p += (long long)gridDim.x * kBlock) {
        const int y = (int)(p / a.in_w), x = (int)(p - (long long)y * a.in_w);
        const float lam = a.lambda[p];
        if (!(lam > 0.0f && lam <= kMaxLambda)) continue;
        Xoshiro rng;
        rng.seed(mix3(a.seed, kPixelStream, x, y));
        const uint32_t q = poisson_u32(rng, (double)lam);
        for (uint32_t g = 0; g < q; ++g) {
            (void)uniform_f32(rng, 1.0f);
            (void)uniform_f32(rng, 1.0f);
            float rad = KIND == 0 ? a.r_const : lognormal_f32(rng, a.log_mu, a.log_sigma, d_zig_x, d_zig_f);
            if (rad > a.rm) rad = a.rm;
            if (rad <= 0.0f || rad * a.zoom <= 0.0f) continue;
            ++cnt;
        }
    }
    for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
    if ((threadIdx.x & 63) == 0 && cnt) {
        atomicAdd(&a.stats[0], cnt);
        atomicAdd(&a.stats[1], cnt * (unsigned long long)a.n_samples);
    }
}

hipError_t launch_grain_count(const GrainArgs &a, int dist_kind, hipStream_t s)
{
    const long long n = (long long)a.in_w * a.in_h;
    const unsigned blocks = (unsigned)std::max<long long>(1, std::min<long long>((n + kBlock - 1) / kBlock, 8192));
    if (dist_kind == 0)
        hipLaunchKernelGGL(grain_count_kernel<0>, dim3(blocks), dim3(kBlock), 0, s, a);
    else
        hipLaunchKernelGGL(grain_count_kernel<1>, dim3(blocks), dim3(kBlock), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_pixel_state(const GrainArgs &a, hipStream_t s)
{
    const long long n = (long long)a.in_w * a.in_h;
    // A wave's last attempts run nearly empty, so waves take 128 pixels or
    // more; 1024 workgroups are four a CU, as many as fit by LDS.  (64, 256 and
    // 512 pixels at least: the same at 4096x4096, 0.3, 0.4 and 1% more for a
    // 1280x720 RGB frame.)
    const long long per = 2 * kBlock, blocks = std::max<long long>(1, std::min<long long>((n + per - 1) / per, 1024));
    hipLaunchKernelGGL(pixel_state_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, a);
    return hipGetLastError();
}

// Input pixels whose grains can reach output rect [X0, X1) x [Y0, Y1): centre
// in [x, x+1], target cx*zoom + offset, covered outputs within target +- R -
// 0.5 (generous margins; extra pixels only produce grains that miss).  ext
// holds the offsets' (min x, max x, min y, max y).
struct PixRegion {
    int x0, y0, w, n;
};
__device__ __forceinline__ PixRegion grain_tile_region(const GrainArgs &a, const float4 &ext, int X0, int Y0, int X1,
                                                       int Y1)
{
    const float z = a.zoom, Rmax = a.r_out_max;
    const int xi0 = max(0, (int)floorf(((float)X0 + 0.5f - Rmax - ext.y) / z) - 2);
    const int xi1 = min(a.in_w - 1, (int)ceilf(((float)X1 - 0.5f + Rmax - ext.x) / z) + 2);
    const int yi0 = max(0, (int)floorf(((float)Y0 + 0.5f - Rmax - ext.w) / z) - 2);
    const int yi1 = min(a.in_h - 1, (int)ceilf(((float)Y1 - 0.5f + Rmax - ext.z) / z) + 2);
    PixRegion r;
    r.x0 = xi0;
    r.y0 = yi0;
    r.w = xi1 - xi0 + 1;
    r.n = (xi1 >= xi0 && yi1 >= yi0) ? r.w * (yi1 - yi0 + 1) : 0;
    return r;
}

// Work of each grain-wise tile (the grains of its input region, from the
// Poisson pre-pass), for a heaviest-first launch order; one workgroup per tile.
__global__ __launch_bounds__(kBlock) void grain_tile_weights_kernel(GrainArgs a, SampleTable st, uint32_t *w,
                                                                    int *ids)
{
    __shared__ uint32_t s_sum[kBlock / 64];
    const int tile = blockIdx.x;
    const int tyi = tile / a.tiles_x, txi = tile - tyi * a.tiles_x;
    const int X0 = txi * a.tile_w, Y0 = tyi * a.tile_h;
    const PixRegion r = grain_tile_region(a, *st.ext, X0, Y0, min(X0 + a.tile_w, a.out_w),
                                          min(Y0 + a.tile_h, a.out_h));
    uint32_t sum = 0;
    for (int p = threadIdx.x; p < r.n; p += kBlock) {
        const int y = r.y0 + p / r.w, x = r.x0 + p % r.w;
        sum += a.pix_q[(size_t)y * a.in_w + x];
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int i = 0; i < kBlock / 64; ++i) t += s_sum[i];
        w[tile] = t;
        ids[tile] = tile;
    }
}

hipError_t launch_grain_tile_weights(const GrainArgs &a, const SampleTable &st, uint32_t *w, int *ids,
                                     hipStream_t s)
{
    hipLaunchKernelGGL(grain_tile_weights_kernel, dim3((unsigned)a.n_tiles), dim3(kBlock), 0, s, a, st, w, ids);
    return hipGetLastError();
}

// How a plane's grains find their samples: constant radius through candidate
// lists, constant radius through runs of the sample order (grains too wide for
// lists), lognormal radii through lists where narrow and runs where not.
enum GrainMode { kConstLists, kConstRuns, kLognormal };

// Steps of the list walk in flight together: a round of 64 grains has about
// two entries a grain at the constant-radius workload (r = 0.05, N = 128) and
// five to twenty under lognormal laws.
constexpr int grain_stage(int mode) { return mode == kConstLists ? 4 : 8; }
constexpr int kGrainStageMax = 8;
// Words a wave keeps for its round: the listed grains' records (16 bytes
// each), then the candidate queue of the others.
constexpr int kGrainWaveWords = 256;
static_assert(kGrainWaveWords >= kQueueCap, "the queue shares the records' room");

// Waves per SIMD each mode's registers are held to (lognormal draws need f64
// transcendentals: at eight waves they spilled 25 registers; a CU holds two
// workgroups of 512 at four waves and at five, 1021x767 at zoom 2, r = 0.1 /
// 0.03, N = 128: 1.50 ms held to five, 1.40 to four).
constexpr int grain_waves(int mode) { return mode == kLognormal ? 4 : 8; }

// Per output tile: rounds of one grain per lane, each drawn from its input
// pixel's stream and its samples found through its list or run.
// Bounded by instruction issue: the draws (repeated for each tile whose halo
// holds the pixel) and about 28 VALU per list entry.  Before lognormal laws
// had lists their lanes walked runs in lockstep, every candidate by its box
// and the queue: 1021x767 at zoom 2, r = 0.1 / 0.03, N = 128 took 7.1 ms and
// takes 1.3; a 1280x720 plane, r = 0.1 / 0.05, N = 64, 2.69 and 0.71.  The
// constant-radius plane of 4096x4096 (r = 0.05, N = 128; owners from a byte
// map, boxes evaluated for every entry, 64x32 tiles): 16.7 and 14.6 ms.
template <int MODE, int BLOCK>
__global__ __launch_bounds__(BLOCK, grain_waves(MODE)) void grainwise_sorted(GrainArgs a, SampleTable st)
{
    constexpr int NW = BLOCK / 64, STAGE = grain_stage(MODE);
    constexpr bool LISTS = MODE != kConstRuns, RUNS = MODE != kConstLists;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ __align__(16) uint32_t s_wave[NW][kGrainWaveWords];
    __shared__ __align__(16) uint32_t s_ends[NW][2 * kGrainStageMax];
    // the region's next pixel that no lane has taken
    __shared__ int s_next;

    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    int tile = blockIdx.x;
    if (a.tile_list) tile = a.tile_list[tile];
    if (tile >= a.n_tiles) return;
    if (tile_cancelled(a.cancel, a.status)) return;
    const int tyi = tile / a.tiles_x, txi = tile - tyi * a.tiles_x;
    const int X0 = txi * a.tile_w, Y0 = tyi * a.tile_h;
    const int X1 = min(X0 + a.tile_w, a.out_w), Y1 = min(Y0 + a.tile_h, a.out_h);
    // per-tile floats held in SGPRs (this target has no scalar float ALU, so
    // they are computed in VGPRs; kept there all kernel long, they spilled)
    const float fx0 = uniform_f((float)X0), fx1 = uniform_f((float)(X1 - 1));
    const float fy0 = uniform_f((float)Y0), fy1 = uniform_f((float)(Y1 - 1));
    const int words = a.words, N = a.n_samples, Q = st.qbuckets;
    const int tile_words = a.tile_w * a.tile_h * words;
    const uint32_t w4 = (uint32_t)words * 4u, row_b = (uint32_t)a.tile_w * w4;

    // ---- LDS: (X, word, bit)[N] | qidx[Q + 1] | bitset ----
    // Per sorted position one 16-byte record: the sample's scaled offset, the
    // LDS address of its bitset word for pixel 0 and its bit's mask (as in the
    // splat); a list entry is its byte offset.
    size_t off = 0;
    float4 *srec = reinterpret_cast<float4 *>(lds);
    off += (size_t)N * 16;
    uint16_t *sq = reinterpret_cast<uint16_t *>(lds + off);
    if (RUNS) off += ((size_t)(Q + 1) * 2 + 15) & ~(size_t)15;
    uint32_t *bits = reinterpret_cast<uint32_t *>(lds + off);
    off += ((size_t)tile_words * 4 + 15) & ~(size_t)15;
    if (off > (size_t)a.lds_bytes) {
        if (tid == 0) atomicOr(a.status, kStatusRegion);
        return;
    }
    for (int w = tid; w < tile_words; w += BLOCK) bits[w] = 0u;
    for (int k = tid; k < N; k += BLOCK) {
        const float2 X = st.xy[k];
        const uint32_t ki = st.k[k];
        srec[k] = make_float4(X.x, X.y, __uint_as_float(lds_addr(bits + (ki >> 5))), __uint_as_float(1u << (ki & 31u)));
    }
    if (RUNS)
        for (int q = tid; q <= Q; q += BLOCK) sq[q] = st.qidx[q];
    if (tid == 0) s_next = 0;
    const float4 ext0 = *st.ext;
    const float4 ext = make_float4(uniform_f(ext0.x), uniform_f(ext0.y), uniform_f(ext0.z), uniform_f(ext0.w));

    const float z = a.zoom, Rmax = a.r_out_max;
    const PixRegion reg = grain_tile_region(a, ext, X0, Y0, X1, Y1);
    const int xi0 = reg.x0, yi0 = reg.y0, rwi = reg.w, npx = reg.n;
    __syncthreads();

    // widening of the fraction interval: every coordinate of a box is below
    // C in magnitude, so each of its f32 steps is off by at most C * 2^-24
    const float C = (float)max(a.out_w, a.out_h) + fmaxf(fmaxf(fabsf(ext.x), fabsf(ext.y)),
                                                         fmaxf(fabsf(ext.z), fabsf(ext.w))) + Rmax + 8.0f;
    const float eps = uniform_f(C * 9.5367431640625e-07f + 1.52587890625e-05f);  // C * 2^-20 + 2^-16
    // a grain below this radius covers pixels nearest its target alone
    // (0 where a lognormal law has no lists: their room is for a bounded eps)
    const float narrow_r = uniform_f(MODE == kLognormal && !(eps <= kGrainWalkEps) ? 0.0f : 0.5f - (eps + eps));
    // within this of the radius a passing pixel's bounds() box is looked at
    const float edge = uniform_f(C * 4.76837158203125e-07f);  // C * 2^-21
    const float Qf = uniform_f((float)Q);
    uint32_t *queue = s_wave[wid];
    int qcount = 0;
    // the lane's current grain: target origin and output radius
    float gbx = 0.0f, gby = 0.0f, gR = 0.0f;

    auto hit = [&](int tx, int ty, const float4 &r) {
        lds_or(mad_u24((uint32_t)ty, row_b, mad_u24((uint32_t)tx, w4, __float_as_uint(r.z))), __float_as_uint(r.w));
    };
    // The pixels of bounds() of src/grainwise.rs:126-142 before its clamp (the
    // tile lies inside the image, so meeting the tile is the clamp).
    auto bounds = [](float t, float R, float &lo, float &hi) {
        lo = ceilf((t - R) - 0.5f);
        hi = floorf((t + R) - 0.5f);
    };

    // Entries: lane (6 bits) | sorted position << 6 (11 bits) | tile column
    // << 17 (7 bits) | tile row << 24 (8 bits).  The reference's disk test
    // (src/grainwise.rs:82-100) for entries [0, n).
    auto drain = [&](int n) {
        uint32_t e = 0;
        if (lane < n) e = queue[lane];
        if (lane + 64 < qcount) queue[lane] = queue[lane + 64];
        const int l = (int)(e & 63u);
        const float bx = __shfl(gbx, l, 64), by = __shfl(gby, l, 64), R = __shfl(gR, l, 64);
        if (lane >= n) return;
        const int p = (int)((e >> 6) & 0x7FFu), tx = (int)((e >> 17) & 0x7Fu), ty = (int)(e >> 24);
        const float4 r = srec[p];
        const float txp = bx + r.x, typ = by + r.y;
        const float dy = ((float)(Y0 + ty) + 0.5f) - typ;
        const float dx = ((float)(X0 + tx) + 0.5f) - txp;
        if (dx * dx + dy * dy <= R * R) hit(tx, ty, r);
    };
    auto push = [&](bool cand, uint32_t entry) {
        const unsigned long long mask = __ballot(cand);
        const int before = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
        if (cand) queue[qcount + before] = entry;
        qcount += __popcll(mask);
        if (qcount >= 64) {
            drain(64);
            qcount -= 64;
        }
    };

    // Each lane draws the grains of one region pixel at a time; a lane whose
    // pixel has no grain left takes the region's next pixel, so the wave's
    // lanes stay busy until the region runs out (pixel counts differ widely).
    // Grains reach the bitset in another order than the reference's, which
    // changes nothing: the bitset is an OR of the tests.
    Xoshiro rng;
    rng.s0 = rng.s1 = rng.s2 = rng.s3 = 0;
    uint32_t q = 0, done = 0;
    float fx = 0.0f, fy = 0.0f;
    bool more = true;  // uniform: pixels of the region are left
    for (;;) {
        while (more) {
            const bool need = done >= q;
            const unsigned long long m = __ballot(need);
            if (m == 0) break;
            const int cnt = __popcll(m);
            int base = 0;
            if (lane == 0) base = atomicAdd(&s_next, cnt);
            base = __builtin_amdgcn_readfirstlane(base);
            more = base + cnt < npx;
            const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            const int pix = base + rank;
            if (need && pix < npx) {
                const int y = yi0 + pix / rwi, x = xi0 + pix % rwi;
                const size_t pi = (size_t)y * a.in_w + x;
                q = a.pix_q[pi];
                const ulonglong2 s01 = a.pix_s01[pi], s23 = a.pix_s23[pi];
                rng.s0 = s01.x;
                rng.s1 = s01.y;
                rng.s2 = s23.x;
                rng.s3 = s23.y;
                done = 0;
                fx = (float)x;
                fy = (float)y;
            }
        }
        if (!__any(done < q)) break;
        // the lane's next grain (src/grainwise.rs:48-67)
        int p0 = 0, len = 0;
        bool listed = false;
        float bx = 0.0f, by = 0.0f, R = 0.0f;
        if (done < q) {
            const float cx = fx + uniform_f32(rng, 1.0f);
            const float cy = fy + uniform_f32(rng, 1.0f);
            float rad = MODE == kLognormal ? lognormal_f32(rng, a.log_mu, a.log_sigma, d_zig_x, d_zig_f) : a.r_const;
            ++done;
            if (rad > a.rm) rad = a.rm;
            R = rad * z;
            bx = cx * z;
            by = cy * z;
            // skip radii <= 0 and grains whose boxes miss the tile for
            // every sample (bounds() is monotone in the target); one mask,
            // not a chain of branches
            const bool keep = ((int)(rad > 0.0f) & (int)(R > 0.0f) &
                               (int)(floorf(((bx + ext.y) + R) - 0.5f) >= fx0) &
                               (int)(ceilf(((bx + ext.x) - R) - 0.5f) <= fx1) &
                               (int)(floorf(((by + ext.w) + R) - 0.5f) >= fy0) &
                               (int)(ceilf(((by + ext.z) - R) - 0.5f) <= fy1)) != 0;
            const int cls = MODE == kLognormal ? (int)(R * (float)(2 * kGrainClassQ)) : 0;
            listed = LISTS && keep && (MODE == kConstLists || (R < narrow_r && cls < a.gl_classes));
            if (listed) {
                // the list of the grain's class and of the cell of its centre
                // fractions (grain_lists_kernel)
                const float nx = 0.5f - bx, ny = 0.5f - by;
                const float A = nx - floorf(nx), B = ny - floorf(ny);
                const int gq = MODE == kLognormal ? kGrainClassQ : kGrainConstQ;
                const int qa = min((int)(A * (float)gq), gq - 1), qb = min((int)(B * (float)gq), gq - 1);
                const uint2 se = a.gl_cell[(uint32_t)(cls * gq + qb) * (uint32_t)gq + (uint32_t)qa];
                p0 = (int)se.x;
                len = (int)se.y;
            } else if (RUNS && keep) {
                // the run of samples whose box can hold a column
                const float nc = R - (bx - 0.5f);
                const float A = nc - floorf(nc);
                const float lo = (A - (R + R)) - eps, hi = A + eps;
                if (!(lo * Qf > -2.0f * Qf) || !(hi * Qf < 2.0f * Qf) ||
                    (int)floorf(hi * Qf) + 1 - (int)floorf(lo * Qf) >= Q) {
                    len = N;
                } else {
                    int lq = (int)floorf(lo * Qf), hq = (int)floorf(hi * Qf) + 1;
                    if (lq < 0) {
                        lq += Q;
                        hq += Q;
                    }
                    lq = min(max(lq, 0), Q - 1);
                    hq = min(max(hq, lq + 1), 2 * Q);
                    p0 = sq[lq];
                    const int end = hq <= Q ? (int)sq[hq] : N + (int)sq[hq - Q];
                    len = end - p0;
                }
            }
        }
        if (LISTS) {
            const bool walks = listed && len > 0;
            const unsigned long long lmask = __ballot(walks);
            if (lmask) {
                const uint32_t fl = walks ? (uint32_t)len : 0u;
                const uint32_t incl = wave_inclusive_sum(fl);
                const int total = __builtin_amdgcn_readlane((int)incl, 63);
                const int bias = total + 64 * STAGE;
                const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(lmask >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)lmask, 0u));
                float4 *rec = reinterpret_cast<float4 *>(s_wave[wid]);
                if (walks) rec[rank] = make_float4(bx, by, R, __int_as_float(p0 - (int)(incl - fl) + bias));
                const unsigned char *recb = reinterpret_cast<const unsigned char *>(rec);
                const int my_end = walks && (int)incl != total ? (int)incl - 1 : -1;
                const unsigned char *list = reinterpret_cast<const unsigned char *>(a.gl_list);
                // A narrow grain's disk reaches only the pixel whose square
                // holds the target, x = floor(t): a pixel whose centre is
                // within R < 1/2 of t is that one.  It passes the reference's
                // disk test and lies in its bounds() box; where |dx| and |dy|
                // are at most R - C 2^-21 the box follows from them (its two
                // roundings and theirs are at most C 2^-24 each), and only
                // nearer the rim is it evaluated.
                auto narrow = [&](uint32_t own, uint32_t entry) {
                    const float4 g = *reinterpret_cast<const float4 *>(recb + own);
                    const float4 r = *reinterpret_cast<const float4 *>(lds + entry);
                    asm volatile("" ::"v"(r.x), "v"(r.y), "v"(r.z), "v"(r.w));
                    const float txp = g.x + r.x, typ = g.y + r.y;
                    const float px = floorf(txp), py = floorf(typ);
                    const int tx = (int)px - X0, ty = (int)py - Y0;
                    if (((unsigned)tx < (unsigned)(X1 - X0)) & ((unsigned)ty < (unsigned)(Y1 - Y0))) {
                        const float dx = (px + 0.5f) - txp, dy = (py + 0.5f) - typ;
                        if (dx * dx + dy * dy <= g.z * g.z) {
                            bool in = fmaxf(fabsf(dx), fabsf(dy)) <= g.z - edge;
                            if (!in) {
                                float xl, xh, yl, yh;
                                bounds(txp, g.z, xl, xh);
                                bounds(typ, g.z, yl, yh);
                                in = (xl <= px) & (px <= xh) & (yl <= py) & (py <= yh);
                            }
                            if (in) hit(tx, ty, r);
                        }
                    }
                };
                // constant radii close to 1/2 of planes so large that eps is
                // not small against it: every pixel of the box in the lane
                auto general = [&](uint32_t own, uint32_t entry) {
                    const float4 g = *reinterpret_cast<const float4 *>(recb + own);
                    const float4 r = *reinterpret_cast<const float4 *>(lds + entry);
                    const float txp = g.x + r.x, typ = g.y + r.y;
                    float xl, xh, yl, yh;
                    bounds(txp, g.z, xl, xh);
                    bounds(typ, g.z, yl, yh);
                    xl = fmaxf(xl, fx0);
                    xh = fminf(xh, fx1);
                    yl = fmaxf(yl, fy0);
                    yh = fminf(yh, fy1);
                    for (float y = yl; y <= yh; y += 1.0f)
                        for (float x = xl; x <= xh; x += 1.0f) {
                            const float dx = (x + 0.5f) - txp, dy = (y + 0.5f) - typ;
                            if (dx * dx + dy * dy <= g.z * g.z) hit((int)(x - fx0), (int)(y - fy0), r);
                        }
                };
                if (MODE == kConstLists && !(a.r_list < narrow_r)) {
                    uint32_t before = 0;
                    for (int sb = 0; sb < total; sb += 64)
                        walk_batch<1>(sb, total, bias, my_end, s_ends[wid], recb, list, before, general);
                } else {
                    walk_lists<STAGE>(total, bias, my_end, s_ends[wid], recb, list, narrow);
                }
            }
        }
        if (RUNS && __any(!listed && len > 0)) {
            gbx = bx;
            gby = by;
            gR = R;
            // one candidate a lane: sorted position p against the grain of
            // lane g, target origin (ebx, eby) and output radius eR
            auto visit = [&](bool ok, int p, int g, float ebx, float eby, float eR) {
                const float4 r = srec[p];
                const float txp = ebx + r.x, typ = eby + r.y;
                float xl, xh, yl, yh;
                bounds(txp, eR, xl, xh);
                bounds(typ, eR, yl, yh);
                const bool cand = ok & (xl <= xh) & (yl <= yh) & (xl <= fx1) & (xh >= fx0) & (yl <= fy1) & (yh >= fy0);
                // a candidate box of one pixel lies in the tile (it meets
                // it); wider boxes queue their pixels inside the tile
                const bool multi = cand & ((xh > xl) | (yh > yl));
                if (!__any(multi)) {
                    // one pixel per candidate: the drain's test of it, run
                    // here in the lane (same f32 expression)
                    if (cand) {
                        const float dx = (xl + 0.5f) - txp, dy = (yl + 0.5f) - typ;
                        if (dx * dx + dy * dy <= eR * eR) hit((int)(xl - fx0), (int)(yl - fy0), r);
                    }
                } else {
                    const uint32_t base = (uint32_t)g | ((uint32_t)p << 6);
                    const float cxl = fmaxf(xl, fx0), cxh = fminf(xh, fx1);
                    const float cyl = fmaxf(yl, fy0), cyh = fminf(yh, fy1);
                    const int tx = (int)(cxl - fx0), ty = (int)(cyl - fy0);
                    const int bw = cand ? (int)(cxh - cxl) + 1 : 0, bh = cand ? (int)(cyh - cyl) + 1 : 0;
                    const int nb = bw * bh;
                    for (int j = 0; __any(j < nb); ++j) {
                        const bool c = j < nb;
                        const int jy = c ? j / bw : 0, jx = c ? j - jy * bw : 0;
                        push(c, base | ((uint32_t)(tx + jx) << 17) | ((uint32_t)(ty + jy) << 24));
                    }
                }
            };
            // the cyclic run position (lanes past their run read a valid
            // sample and queue nothing)
            auto position = [&](int pr) {
                return (int)min(min((uint32_t)pr, (uint32_t)(pr - N)), (uint32_t)(N - 1));
            };
            if (LISTS) {
                // The round's wide grains one after another, 64 samples of a
                // grain's run a step.  In lockstep, a sample a step for every
                // lane's grain, a few wide grains kept the wave for the
                // longest run while the others' lanes idled, on top of the
                // lists: 700x500 at zoom 3, N = 256, 4.6% wide grains: 25.0
                // ms by runs alone, 30.1 with lists and lockstep, 4.4 now;
                // 400x300 at zoom 2, N = 128, 46%: 2.77, 3.41 and 0.90; 96x64
                // at zoom 4, N = 1024, all wide: 26.1, 26.5 and 3.1.
                for (unsigned long long m = __ballot(!listed && len > 0); m; m &= m - 1ull) {
                    const int g = __ffsll((long long)m) - 1;
                    auto of_g = [&](float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), g)); };
                    const float ubx = of_g(bx), uby = of_g(by), uR = of_g(R);
                    const int up0 = __builtin_amdgcn_readlane(p0, g), ulen = __builtin_amdgcn_readlane(len, g);
                    for (int i0 = 0; i0 < ulen; i0 += 64)
                        visit(i0 + lane < ulen, position(up0 + i0 + lane), g, ubx, uby, uR);
                }
            } else {
                for (int it = 0; __any(it < len); ++it) visit(it < len, position(p0 + it), lane, bx, by, R);
            }
            // the queue refers to the lanes' current grains
            if (qcount > 0) {
                drain(qcount);
                qcount = 0;
            }
        }
    }
    __syncthreads();

    const int tw = X1 - X0, th = Y1 - Y0;
    for (int p = tid; p < tw * th; p += BLOCK) {
        const int ox = p % tw, oy = p / tw;
        const uint32_t *pw = bits + ((size_t)oy * a.tile_w + ox) * words;
        uint32_t count = 0;
        for (int w = 0; w < words; ++w) count += __popc(pw[w]);
        a.out[(size_t)(Y0 + oy) * a.out_w + (X0 + ox)] = (float)count * a.inv_samples;
    }
}

size_t grainwise_sorted_static_lds(int block)
{
    return (size_t)block / 64 * (kGrainWaveWords * 4 + 2 * kGrainStageMax * 4) + 64;
}

size_t grainwise_sorted_lds(int tile_w, int tile_h, int n_samples, int qbuckets)
{
    const size_t words = ((size_t)n_samples + 31) / 32;
    auto a16 = [](size_t b) { return (b + 15) & ~(size_t)15; };
    return a16((size_t)tile_w * tile_h * words * 4) + (size_t)n_samples * 16 + a16((size_t)(qbuckets + 1) * 2);
}

template <int MODE>
static void launch_sorted_mode(const GrainArgs &a, const SampleTable &st, int block, hipStream_t s)
{
    const dim3 grid(a.n_tiles);
    const size_t lds = (size_t)a.lds_bytes;
    if (block == 256)
        hipLaunchKernelGGL((grainwise_sorted<MODE, 256>), grid, dim3(256), lds, s, a, st);
    else
        hipLaunchKernelGGL((grainwise_sorted<MODE, 512>), grid, dim3(512), lds, s, a, st);
}

hipError_t launch_grainwise_sorted(const GrainArgs &a, const SampleTable &st, int dist_kind, int block,
                                   hipStream_t s)
{
    if (dist_kind != 0)
        launch_sorted_mode<kLognormal>(a, st, block, s);
    else if (a.gl_classes > 0)
        launch_sorted_mode<kConstLists>(a, st, block, s);
    else
        launch_sorted_mode<kConstRuns>(a, st, block, s);
    return hipGetLastError();
}

hipError_t launch_grainwise(const GrainArgs &a, int dist_kind, bool with_stats, hipStream_t s)
{
    const dim3 grid(a.n_tiles), block(kBlock);
    const size_t lds = (size_t)a.lds_bytes;
    if (dist_kind == 0) {
        if (with_stats)
            hipLaunchKernelGGL((grainwise_tiles<0, true>), grid, block, lds, s, a);
        else
            hipLaunchKernelGGL((grainwise_tiles<0, false>), grid, block, lds, s, a);
    } else {
        if (with_stats)
            hipLaunchKernelGGL((grainwise_tiles<1, true>), grid, block, lds, s, a);
        else
            hipLaunchKernelGGL((grainwise_tiles<1, false>), grid, block, lds, s, a);
    }
    return hipGetLastError();
}

}  // namespace fg
