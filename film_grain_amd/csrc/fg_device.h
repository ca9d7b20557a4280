// fg_device.h -- device helpers shared by the film-grain kernels.
#ifndef FG_DEVICE_H
#define FG_DEVICE_H

#include "fg_kernels.h"
#include "fg_rng.h"

namespace fg {

static __constant__ double d_zig_x[257] = {FG_ZIG_NORM_X_VALUES};
static __constant__ double d_zig_f[257] = {FG_ZIG_NORM_F_VALUES};

// floor(RN(a / d)) cast like Rust's `as i32`.  With fast set, the quotient
// comes from q0 = a*rd corrected by one FMA residual step, which the host has
// verified equals the IEEE quotient for this d over a whole binade; outside
// [2^-60, 2^60] (where intermediates could leave the normal range) the IEEE
// division is used.
__device__ __forceinline__ int floor_div(float a, float d, float rd, int fast)
{
    float q;
    const float aa = fabsf(a);
    if (fast && aa >= 8.67361737988404e-19f && aa <= 1.152921504606847e18f) {
        const float q0 = a * rd;
        const float r = fmaf(-q0, d, a);
        q = fmaf(r, rd, q0);
    } else {
        q = __fdiv_rn(a, d);
    }
    return sat_i32(floorf(q));
}

// Workgroup exclusive scan of one u32 per thread (kBlock threads); returns the
// exclusive prefix and the workgroup total.  Contains two barriers.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t *s_wave,
                                                         uint32_t &total)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[wid] = x;
    __syncthreads();
    uint32_t before = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) {
        const uint32_t t = s_wave[w];
        before += (w < wid) ? t : 0u;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return before + x - v;
}

// Poisson threshold of one lambda value for the pixel-wise cells
// (src/pixelwise.rs:69-82): 2.0 when the cell is skipped (lambda <= 0 or
// lambda*delta*delta <= 0), exp(-expected) for the Knuth branch (expected < 12),
// and -expected for the rejection branch.  Values outside the accepted range
// (NaN, above kMaxLambda) are skipped too; lambda_invalid flags them.
__device__ __forceinline__ bool lambda_invalid(float lam) { return !(lam <= kMaxLambda); }
__device__ __forceinline__ double cell_threshold(float lam, float delta)
{
    if (!(lam > 0.0f) || !(lam <= kMaxLambda)) return 2.0;
    const float expected = lam * delta * delta;
    if (!(expected > 0.0f)) return 2.0;
    if (expected < 12.0f) return exp_neg_glibc(expected);  // glibc's exp(-expected), exactly
    return -(double)expected;
}

// Poisson count of a cell given its hash and threshold, leaving rng positioned
// after the count draws (as Poisson::sample leaves it).  The common empty cell
// costs only the two seed words the first Xoshiro output depends on.
__device__ __forceinline__ uint32_t cell_count(uint64_t h, double e, Xoshiro &rng)
{
    if (e > 1.5) return 0u;
    if (e >= 0.0) {
        const uint64_t s0 = splitmix64(h), s3 = splitmix64(h + 3 * kGolden);
        const double u1 = standard_f64(rotl64(s0 + s3, 23) + s0);
        if (!(u1 > e)) return 0u;  // Knuth: p = u1 <= exp(-lambda) stops at once
        rng.seed(h);
        (void)rng.next();
        double p = u1;
        uint32_t n = 1;
        while (p > e) {
            p = p * standard_f64(rng.next());
            ++n;
        }
        return n - 1u;
    }
    rng.seed(h);
    const double r = poisson_rejection(rng, -e);
    if (!(r > 0.0)) return 0u;
    if (r >= 4294967295.0) return 0xFFFFFFFFu;
    return (uint32_t)r;
}

// ---------------------------------------------------------------------------
// splat drain, shared by the tile and HBM splat kernels
// ---------------------------------------------------------------------------
struct SplatTile {
    int X0, Y0, X1, Y1;  // output rect
    int I0, J0;          // region origin (cell indices)
    int TW;              // bitset row pitch (tile_w)
    float fx0, fx1, fy0, fy1;  // X0, X1-1, Y0, Y1-1 as floats
};

// Candidate box of grain record B = (cx*zoom - 0.5, cy*zoom - 0.5, r*zoom +
// slack) for sample k with scaled offset (oxz, oyz): the output pixels whose
// sample point can lie in the grain's disk.  The phase that queues candidates
// and the drain that tests them evaluate this with the same operations, so
// they agree on every box.
struct SplatBox {
    float xl, xh, yl, yh;
};
__device__ __forceinline__ SplatBox splat_box(const float4 &B, float oxz, float oyz)
{
    const float cx = B.x + oxz, cy = B.y + oyz;
    SplatBox b;
    b.xl = ceilf(cx - B.z);
    b.xh = floorf(cx + B.z);
    b.yl = ceilf(cy - B.z);
    b.yh = floorf(cy + B.z);
    return b;
}
// The box is non-empty and meets the tile.
__device__ __forceinline__ bool splat_box_hits(const SplatBox &b, const SplatTile &t)
{
    return b.xl <= b.xh && b.xl <= t.fx1 && b.xh >= t.fx0 && b.yl <= b.yh && b.yl <= t.fy1 &&
           b.yh >= t.fy0;
}

// Drains the first n (<= 64) entries (grain | k << 16) of this wave's queue
// through the exact reference test and moves entries [64, count) to the front.
__device__ __forceinline__ void splat_drain(const PixelArgs &a, const SplatTile &t, uint32_t *queue,
                                            int n, int count, const float4 *gA, const float4 *gB,
                                            const float2 *offs, uint32_t *bits)
{
    const int lane = threadIdx.x & 63;
    uint32_t e = 0;
    if (lane < n) e = queue[lane];
    if (lane + 64 < count) queue[lane] = queue[lane + 64];
    if (lane >= n) return;
    const uint32_t g = e & 0xFFFFu;
    const int k = (int)(e >> 16);
    const float2 o = offs[k];
    const SplatBox b = splat_box(gB[g], o.x * a.zoom, o.y * a.zoom);
    const int xlo = (int)fmaxf(b.xl, t.fx0), xhi = (int)fminf(b.xh, t.fx1);
    const int ylo = (int)fmaxf(b.yl, t.fy0), yhi = (int)fminf(b.yh, t.fy1);
    const float4 G = gA[g];
    const uint32_t cell = __float_as_uint(G.w);
    const int gi = t.I0 + (int)(cell & 0xFFFFu), gj = t.J0 + (int)(cell >> 16);
    const float rm = a.rm, delta = a.delta, rd = a.rdelta, iz = a.inv_zoom;
    const int fast = a.div_fast;
    for (int y = ylo; y <= yhi; ++y) {
        const float yg = ((float)y + 0.5f) * iz - o.y;
        const float dy = yg - G.y;
        const float dy2 = dy * dy;
        for (int x = xlo; x <= xhi; ++x) {
            const float xg = ((float)x + 0.5f) * iz - o.x;
            const float dx = xg - G.x;
            if (dx * dx + dy2 <= G.z) {
                // the grain's cell must lie in the point's window
                if (floor_div(xg - rm, delta, rd, fast) <= gi && gi <= floor_div(xg + rm, delta, rd, fast) &&
                    floor_div(yg - rm, delta, rd, fast) <= gj && gj <= floor_div(yg + rm, delta, rd, fast)) {
                    atomicOr(&bits[((y - t.Y0) * t.TW + (x - t.X0)) * a.words + (k >> 5)], 1u << (k & 31));
                }
            }
        }
    }
}

// Cancellation between tiles (a workgroup reads the flag once per tile):
// true when the host has raised *flag; the caller's status then records it.
// The flag lives in coherent host memory, so the load goes to the system
// scope.  Must be called by every thread of the workgroup (it synchronises).
__device__ __forceinline__ bool tile_cancelled(const int *flag, int *status)
{
    __shared__ int s_cancel;
    if (!flag) return false;
    if (threadIdx.x == 0) {
        s_cancel = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (s_cancel) atomicOr(status, kStatusCancelled);
    }
    __syncthreads();
    return s_cancel != 0;
}

// Wave-wide inclusive sum (every lane of the wave active): six DPP adds, within
// rows of 16 lanes and then across them.  By lane exchanges (ds_bpermute) each
// step waits for LDS: the 4096x4096 grain-wise plane, a sum per 64 grains,
// took 20.87 ms and takes 18.79; the 4K RGB frame 16.27 and 16.07.
__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t x)
{
    int v = (int)x;
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 to rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 to rows 2, 3
    return (uint32_t)v;
}

// A wave-uniform float moved to an SGPR (no scalar float ALU on this target:
// a float computed from uniform values lands in a VGPR and holds it).
__device__ __forceinline__ float uniform_f(float v)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// LDS locations as 32-bit LDS addresses: a bitset word's address held in a
// sample record is used as it is, with no workgroup base added per hit
typedef __attribute__((address_space(3))) uint32_t lds_u32;
__device__ __forceinline__ uint32_t lds_addr(uint32_t *p)
{
    return (uint32_t)(uintptr_t)(lds_u32 *)p;
}
__device__ __forceinline__ void lds_or(uint32_t addr, uint32_t v)
{
    __hip_atomic_fetch_or((lds_u32 *)(uintptr_t)addr, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// a * b + c for a, b < 2^24 with one full-rate v_mad_u32_u24 (b uniform).
// Written out because the compiler turns two such terms into two products
// and a three-way add.
__device__ __forceinline__ uint32_t mad_u24(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t d;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(d) : "v"(a), "s"(b), "v"(c));
    return d;
}

// The candidate lists of a wave's grains, concatenated in lane order into one
// stream of `total` entries, walked 64 entries a step.  The grains with a list
// are numbered by their place in that order (their rank); rank k has a 16-byte
// record at rec + 16 k (the wave's own LDS) whose last word is its first list
// position, less its first stream entry, plus bias.  The stream's entry e
// belongs to the grain whose rank is the number of lists that end before e: a
// set bit per list end (its last entry, my_end per lane; -1 for none, and for
// the stream's last list, so that lanes past the stream count as its entries)
// in a bitset of the batch's entries (ends, 2 STAGE words of the wave's LDS),
// so that a step's owners are a count of the set bits below each lane (two
// v_mbcnt) on top of the count before the step.  (Taking the owners from a
// scalar loop over the grains that start within the step was half of the
// walk's scalar instructions: the splat of a 4K RGB frame at N = 256 took
// 13.6 ms and takes 11.2.)
//
// A batch is STAGE steps: their owners first, then all their list loads in
// flight together, then test(owner's record offset, entry) for each: one
// global latency per batch of steps instead of one per step.  Lanes past the
// stream read its last entry (the stream's last pair again: its bit is ORed
// twice, which changes nothing).  A step from s loads stream entry s +
// min(lane, total - 1 - s), and the steps of a batch that start past the
// stream have s < total + 64 (STAGE - 1); with bias = total + 64 STAGE the
// lane's part of the list position is positive: a load takes a base in SGPRs
// (the batch's first entry, less the bias), a valid unsigned 32-bit offset in
// one VGPR and the step's 128 bytes as its immediate offset, no 64-bit address
// arithmetic.  Whole batches come first, then a shorter one where it holds
// the rest: the lists of a small N are a few entries each.
//
// The wave's LDS accesses run in order, so no barrier is needed.
template <int STAGE, class Test>
__device__ __forceinline__ void walk_batch(int sb, int total, int bias, int my_end, uint32_t *ends,
                                           const unsigned char *rec, const unsigned char *list, uint32_t &before,
                                           Test &&test)
{
    const int lane = threadIdx.x & 63;
    if (lane < 2 * STAGE) ends[lane] = 0u;
    __builtin_amdgcn_wave_barrier();
    const int rel = my_end - sb;
    if ((unsigned)rel < 64u * STAGE && my_end >= 0) lds_or(lds_addr(ends + (rel >> 5)), 1u << (rel & 31));
    __builtin_amdgcn_wave_barrier();
    const unsigned char *lbb = list + 2 * ((long long)sb - bias);
    uint32_t own[STAGE], pn[STAGE];
#pragma unroll
    for (int i = 0; i < STAGE; ++i) {
        const uint2 e = *reinterpret_cast<const uint2 *>(ends + 2 * i);
        own[i] = __builtin_amdgcn_mbcnt_hi(e.y, __builtin_amdgcn_mbcnt_lo(e.x, before)) << 4;
        before += __popc(e.x) + __popc(e.y);
    }
#pragma unroll
    for (int i = 0; i < STAGE; ++i) {
        const uint32_t pos = *reinterpret_cast<const uint32_t *>(rec + own[i] + 12) +
                             (uint32_t)min(lane, total - 1 - (sb + 64 * i));
        pn[i] = (uint32_t)*reinterpret_cast<const uint16_t *>(lbb + 128 * i + (pos << 1));
    }
#pragma unroll
    for (int i = 0; i < STAGE; ++i) {
        if (sb + 64 * i >= total) break;
        test(own[i], pn[i]);
    }
    __builtin_amdgcn_wave_barrier();
}

template <int STAGE, class Test>
__device__ __forceinline__ void walk_lists(int total, int bias, int my_end, uint32_t *ends, const unsigned char *rec,
                                           const unsigned char *list, Test &&test)
{
    static_assert(STAGE >= 4, "batches of STAGE, STAGE / 2 and STAGE / 4 steps");
    uint32_t before = 0;  // list ends before the step
    int sb = 0;
    for (; total - sb > 64 * (STAGE / 2); sb += 64 * STAGE)
        walk_batch<STAGE>(sb, total, bias, my_end, ends, rec, list, before, test);
    if (total - sb > 64 * (STAGE / 4))
        walk_batch<STAGE / 2>(sb, total, bias, my_end, ends, rec, list, before, test);
    else if (total - sb > 0)
        walk_batch<STAGE / 4>(sb, total, bias, my_end, ends, rec, list, before, test);
}

}  // namespace fg

#endif
