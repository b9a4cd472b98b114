/*
 * er_post.hip - per-pass post-processing and the volume preprocessing kernels.
 *
 * k_post fuses, per pixel, the three remaining kernels of a pass:
 *   KrnlFilterFrameEstimate (Source/filterframeestimate.cuh:33-64): 3x3 Gaussian, sigma 1,
 *     weights renormalised at the border; alpha is the centre alpha divided by the total
 *     weight (the code sets Sum[3] and then divides all four channels);
 *   KrnlComputeEstimate (Source/estimate.cuh:27-32): R += (F - R) / max(N, 1) with N the
 *     passes completed before this one (Q1);
 *   KrnlToneMap (Source/tonemap.cuh:30-59): XYZ -> linear sRGB, 1 - exp(-c / Exposure),
 *     clamp, x255 truncated; A = R.a x 255.
 * The filtered frame is not written back (the reference copies it over the frame estimate,
 * filterframeestimate.cuh:71-73); the fused kernel reads the 3x3 neighbourhood through an
 * LDS tile with a one-pixel halo.
 *
 * k_bilateral_{h,v}: the separable bilateral filter on the RGBA8 display image (design:
 * Source/filterrunningestimate.cuh:55-191, Source/filter.h:34-40) with taps
 * [max(0, i-R), min(i+R, n-1)) - exclusive upper bound as written (Q27).
 *
 * k_build_cells / k_macro_minmax / k_macro_sigma / k_macro_bits / k_gm_max: volume preprocessing.
 */
#include "er_path.h"

namespace erd {

#define POST_TILE 16

/* One 16 x 16 tile of one pass's post-processing; every thread of the workgroup calls it. */
__device__ __forceinline__ void post_tile(const DevParams& p, const float4* __restrict__ frame, float4* __restrict__ running,
                                          uchar4* __restrict__ display, int no_iterations, int bx, int by,
                                          float4 (*tile)[POST_TILE + 2])
{
    const int W = p.film_w, H = p.film_h;
    for (int k = threadIdx.x; k < (POST_TILE + 2) * (POST_TILE + 2); k += blockDim.x) {
        const int ty = k / (POST_TILE + 2), tx = k % (POST_TILE + 2);
        const int gx = min(max(bx + tx - 1, 0), W - 1), gy = min(max(by + ty - 1, 0), H - 1);
        tile[ty][tx] = frame[(size_t)gy * W + gx];
    }
    __syncthreads();
    const int lx = threadIdx.x % POST_TILE, ly = threadIdx.x / POST_TILE;
    const int x = bx + lx, y = by + ly;
    if (x >= W || y >= H) return;

    /* Gauss2D(1, X, Y) = exp(-(X^2 + Y^2) / 2) */
    const float g0 = erm::expf_(-0.0f), g1 = erm::expf_(-0.5f), g2 = erm::expf_(-1.0f);
    const int x0 = max(x - 1, 0), x1 = min(x + 1, W - 1);
    const int y0 = max(y - 1, 0), y1 = min(y + 1, H - 1);
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f, tw = 0.0f;
    for (int yy = y0; yy <= y1; ++yy) {
        for (int xx = x0; xx <= x1; ++xx) {
            const int d2 = (xx - x) * (xx - x) + (yy - y) * (yy - y);
            const float w = d2 == 0 ? g0 : (d2 == 1 ? g1 : g2);
            const float4 f = tile[yy - by + 1][xx - bx + 1];
            s0 += f.x * w; s1 += f.y * w; s2 += f.z * w; s3 += f.w * w;
            tw += w;
        }
    }
    s3 = tile[ly + 1][lx + 1].w;
    float4 fe;
    if (tw > 0.0f) { fe.x = s0 / tw; fe.y = s1 / tw; fe.z = s2 / tw; fe.w = s3 / tw; }
    else { fe.x = fe.y = fe.z = fe.w = 0.0f; }

    const size_t i = (size_t)y * W + x;
    const float n = fmaxf((float)no_iterations, 1.0f);
    float4 r = running[i];
    r.x = r.x + (fe.x - r.x) / n;
    r.y = r.y + (fe.y - r.y) / n;
    r.z = r.z + (fe.z - r.z) / n;
    r.w = r.w + (fe.w - r.w) / n;
    running[i] = r;

    const float R = 3.240479f * r.x - 1.537150f * r.y - 0.498535f * r.z;
    const float G = -0.969256f * r.x + 1.875991f * r.y + 0.041556f * r.z;
    const float B = 0.055648f * r.x - 0.204043f * r.y + 1.057311f * r.z;
    const float e = p.exposure;
    const float tr = fmaxf(0.0f, fminf(1.0f - erm::expf_(-(R / e)), 1.0f));
    const float tg = fmaxf(0.0f, fminf(1.0f - erm::expf_(-(G / e)), 1.0f));
    const float tb = fmaxf(0.0f, fminf(1.0f - erm::expf_(-(B / e)), 1.0f));
    uchar4 d;
    d.x = (unsigned char)(255.0f * tr);
    d.y = (unsigned char)(255.0f * tg);
    d.z = (unsigned char)(255.0f * tb);
    d.w = (unsigned char)(r.w * 255.0f);
    display[i] = d;
}

__global__ __launch_bounds__(256) void k_post(const DevParams* __restrict__ pp, const float4* __restrict__ frame,
                                             float4* __restrict__ running, uchar4* __restrict__ display, int no_iterations,
                                             unsigned int* __restrict__ qcount)
{
    /* the queues of this pass have been consumed: empty them for the next pass */
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < ER_CNT_LINES) qcount[ER_CNT(threadIdx.x)] = 0u;
    __shared__ float4 tile[POST_TILE + 2][POST_TILE + 2];
    post_tile(*pp, frame, running, display, no_iterations, blockIdx.x * POST_TILE, blockIdx.y * POST_TILE, tile);
}

/* post-processing of a batch round: one workgroup per 16 x 16 tile of each of the na jobs
 * taking part (the first na of the table, whose tiles come first); the job by binary search
 * over the tiles' ascending first indices */
__global__ __launch_bounds__(256) void k_post_b(const BatchJob* __restrict__ J, int na, unsigned int round)
{
    const int b = blockIdx.x;
    if (na == 0) return;
    int lo = 0, hi = na - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (J[mid].post_base <= b) lo = mid; else hi = mid - 1;
    }
    const int job = lo;
    if (b < J[job].post_base || b >= J[job].post_base + J[job].post_ntiles) return;
    const BatchJob& B = J[job];
    const int t = b - B.post_base;
    __shared__ float4 tile[POST_TILE + 2][POST_TILE + 2];
    post_tile(*B.params, B.frame, B.running, B.display, B.no_iter0 + (int)round, (t % B.post_tiles_x) * POST_TILE,
              (t / B.post_tiles_x) * POST_TILE, tile);
}

struct BilateralParams {
    int radius;
    float kd[65];      /* spatial weights, index R + k - i */
    float gs[256];     /* range weights, index (int)|dY| */
};

__device__ __forceinline__ float lum(uchar4 c)
{
    return 0.212671f * (float)c.x + 0.715160f * (float)c.y + 0.072169f * (float)c.z;
}

template<int HORIZONTAL>
__global__ __launch_bounds__(256) void k_bilateral(const BilateralParams* __restrict__ bp, const uchar4* __restrict__ in,
                                                  uchar4* __restrict__ out, int W, int H)
{
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= W || y >= H) return;
    const int R = bp->radius;
    const int i = HORIZONTAL ? x : y;
    const int n = HORIZONTAL ? W : H;
    const int lo = max(0, i - R), hi = min(i + R, n - 1);
    const uchar4 c = in[(size_t)y * W + x];
    const float yc = lum(c);
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, tw = 0.0f;
    for (int k = lo; k < hi; ++k) {
        const uchar4 q = HORIZONTAL ? in[(size_t)y * W + k] : in[(size_t)k * W + x];
        const float w = bp->kd[R + k - i] * bp->gs[(int)fabsf(lum(q) - yc)];
        tw += w;
        s0 += (float)q.x * w; s1 += (float)q.y * w; s2 += (float)q.z * w;
    }
    uchar4 d;
    if (tw > 0.0f) {
        d.x = (unsigned char)fmaxf(0.0f, fminf(s0 / tw, 255.0f));
        d.y = (unsigned char)fmaxf(0.0f, fminf(s1 / tw, 255.0f));
        d.z = (unsigned char)fmaxf(0.0f, fminf(s2 / tw, 255.0f));
    } else {
        d.x = d.y = d.z = 0;
    }
    d.w = 255;
    out[(size_t)y * W + x] = d;
}

/* cell (cx, cy, cz) in [0, R]^3 holds the corners of lattice cell (cx-1, cy-1, cz-1). Bound by the 16-byte records it writes: a thread owns one (cx, cy) column
 * of ER_CELL_RUN cells along z and carries the column's upper corners over to the next cell, so
 * a cell costs four 2-byte loads and no 64-bit division: 256^3 in 70 us, 3.9 TB/s written (the
 * flat form with three divisions 85 us), 512 x 512 x 460 in 540 us (640). */
#define ER_CELL_RUN 8
__global__ __launch_bounds__(256) void k_build_cells(const uint16_t* __restrict__ vox, uint4* __restrict__ cells,
                                                    int rx, int ry, int rz)
{
    const unsigned int sx = (unsigned int)rx + 1u, sy = (unsigned int)ry + 1u;
    const unsigned int n = sx * sy;                                     /* below 2^24 */
    const unsigned int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) {
        const int cy = (int)udiv24(k, sx);
        const int cx = (int)(k - (unsigned int)cy * sx);
        const int x0 = max(cx - 1, 0), x1 = min(cx, rx - 1);
        const int y0 = max(cy - 1, 0), y1 = min(cy, ry - 1);
        const size_t a = (size_t)y0 * rx + x0, b = (size_t)y0 * rx + x1, c = (size_t)y1 * rx + x0, d = (size_t)y1 * rx + x1;
        const size_t plane = (size_t)rx * ry;
        for (int z_first = (int)blockIdx.y * ER_CELL_RUN; z_first <= rz; z_first += (int)gridDim.y * ER_CELL_RUN) {
            const uint16_t* v = vox + plane * (size_t)max(z_first - 1, 0);
            uint32_t lo0 = (uint32_t)v[a] | ((uint32_t)v[b] << 16), lo1 = (uint32_t)v[c] | ((uint32_t)v[d] << 16);
            for (int cz = z_first; cz < min(z_first + ER_CELL_RUN, rz + 1); ++cz) {
                v = vox + plane * (size_t)min(cz, rz - 1);
                const uint32_t hi0 = (uint32_t)v[a] | ((uint32_t)v[b] << 16), hi1 = (uint32_t)v[c] | ((uint32_t)v[d] << 16);
                cells[(size_t)cz * n + k] = make_uint4(lo0, lo1, hi0, hi1);
                lo0 = hi0;
                lo1 = hi1;
            }
        }
    }
}

/* min/max voxel over [m*E, m*E + E] (E = 2^shift, clamped) on each axis: every voxel a sample
 * whose floor(L) >> shift == m (after clamping) can read.
 * k_macro_rows, E <= 8: a workgroup takes a row of macrocells along x; each thread reduces one
 * column of (E + 1)^2 voxels, all loads coalesced along x and independent, and the macrocells
 * then reduce their E + 1 columns from LDS. Bound by the voxel loads: 1.3 passes over the volume.
 * k_macro_minmax, E >= 16: a wave per macrocell, 16 lanes along x and 4 rows at once (few, large
 * macrocells, whose rows alone would not fill the device).
 * 8-cell macrocells of 192^3 / 512 x 512 x 460: 10.5 / 119 us; one lane per macrocell took 94 /
 * 215 us, a wave per macrocell 24 / 400 us. */
#define ER_ROW_COLUMNS 256
__global__ __launch_bounds__(ER_ROW_COLUMNS) void k_macro_rows(const uint16_t* __restrict__ vox, uint32_t* __restrict__ mm,
                                                               int rx, int ry, int rz, int mx, int my, int shift, int mrows)
{
    __shared__ uint32_t clo[ER_ROW_COLUMNS], chi[ER_ROW_COLUMNS];
    const int E = 1 << shift;
    const int per = (ER_ROW_COLUMNS - 1) >> shift;   /* macrocells a workgroup takes, and one more column */
    const int m0 = (int)blockIdx.x * per;
    const int x = min(m0 * E + (int)threadIdx.x, rx - 1);
    for (int row = (int)blockIdx.y; row < mrows; row += (int)gridDim.y) {
        const int by = row % my, bz = row / my;
        const int y1 = min(by * E + E, ry - 1), z1 = min(bz * E + E, rz - 1);
        uint32_t lo = 0xffff, hi = 0;
        if ((int)threadIdx.x <= per * E)
            for (int z = bz * E; z <= z1; ++z) {
                const uint16_t* v = vox + ((size_t)z * ry + by * E) * rx + x;
#pragma unroll 3
                for (int y = by * E; y <= y1; ++y, v += rx) {
                    const uint32_t u = *v;
                    lo = min(lo, u);
                    hi = max(hi, u);
                }
            }
        clo[threadIdx.x] = lo;
        chi[threadIdx.x] = hi;
        __syncthreads();
        const int m = m0 + (int)threadIdx.x;
        if ((int)threadIdx.x < per && m < mx) {
            for (int k = 0; k <= E; ++k) {
                lo = k ? min(lo, clo[threadIdx.x * E + k]) : clo[threadIdx.x * E];
                hi = k ? max(hi, chi[threadIdx.x * E + k]) : chi[threadIdx.x * E];
            }
            mm[(size_t)row * mx + m] = lo | (hi << 16);
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void k_macro_minmax(const uint16_t* __restrict__ vox, uint32_t* __restrict__ mm,
                                                     int rx, int ry, int rz, int mx, int my, int mz, int shift)
{
    const int m = (int)(blockIdx.x * 4 + (threadIdx.x >> 6));
    const int lx = threadIdx.x & 15, lr = (threadIdx.x >> 4) & 3;
    uint32_t lo = 0xffff, hi = 0;
    if (m >= mx * my * mz) return;
    const int E = 1 << shift;
    const int bx = m % mx, by = (m / mx) % my, bz = m / (mx * my);
    const int x0 = bx * E, x1 = min(bx * E + E, rx - 1);
    const int y0 = by * E, y1 = min(by * E + E, ry - 1);
    const int z0 = bz * E, z1 = min(bz * E + E, rz - 1);
    for (int z = z0; z <= z1; ++z)
        for (int y = y0 + lr; y <= y1; y += 4)
            for (int x = x0 + lx; x <= x1; x += 16) {
                const uint32_t v = vox[((size_t)z * ry + y) * rx + x];
                lo = min(lo, v);
                hi = max(hi, v);
            }
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, o));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, o));
    }
    if ((threadIdx.x & 63) == 0) mm[m] = lo | (hi << 16);
}

/* the largest voxel from a macrocell grid's ranges (one workgroup) */
__global__ __launch_bounds__(1024) void k_range_top(const uint32_t* __restrict__ mm, int n, unsigned int* __restrict__ top)
{
    __shared__ uint32_t part[16];
    uint32_t hi = 0;
    for (int k = threadIdx.x; k < n; k += 1024) hi = max(hi, mm[k] >> 16);
    for (int o = 32; o > 0; o >>= 1) hi = max(hi, (uint32_t)__shfl_xor((int)hi, o));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = hi;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) hi = max(hi, part[w]);
        *top = hi;
    }
}

/* the intensities a truncating trilinear sample can take in a macrocell of min/max mm: each of
 * the three lerp levels can lose at most one unit below the smallest corner */
__device__ __forceinline__ void sample_range(uint32_t mm, int lut_max, int& lo, int& hi)
{
    lo = max((int)(mm & 0xffff) - 3, 0);
    hi = min((int)(mm >> 16), lut_max);
}

/* max sigma over those intensities (the Woodcock majorants), 16 lanes to a macrocell: a range
 * may span the whole table, which one lane per macrocell read entry by entry in 230 us */
__global__ __launch_bounds__(256) void k_macro_sigma(const uint32_t* __restrict__ mm, const float* __restrict__ lut,
                                                    int lut_max, float* __restrict__ out, int n)
{
    const int m = (int)(blockIdx.x * (blockDim.x >> 4) + (threadIdx.x >> 4));
    float s = 0.0f;
    if (m < n) {
        int lo, hi;
        sample_range(mm[m], lut_max, lo, hi);
        for (int i = lo + (int)(threadIdx.x & 15); i <= hi; i += 16) s = fmaxf(s, lut[i]);
    }
    for (int o = 8; o > 0; o >>= 1) s = fmaxf(s, __shfl_xor(s, o));
    if (m < n && (threadIdx.x & 15) == 0) out[m] = s;
}

/* occupancy bit of macrocell m: it can hold a sample with sigma > 0 that is not clipped away.
 * next[i] is the smallest intensity >= i whose sigma is positive (0xffffffff: none), so the test
 * over the macrocell's range of intensities is one table read; gone (may be NULL) has bit m set
 * when every sample of macrocell m is clipped away (the host's conservative test; clipping
 * objects apply in the full estimator only); with unclipped, whose bit m is set when no sample of
 * macrocell m is, cut gets the macrocells that can hold such a sample and are not wholly
 * unclipped. One lane per macrocell, a ballot for 64 bits. */
__global__ __launch_bounds__(256) void k_macro_bits(const uint32_t* __restrict__ mm, const uint32_t* __restrict__ next,
                                                   int lut_max, const uint32_t* __restrict__ gone,
                                                   const uint32_t* __restrict__ unclipped, uint32_t* __restrict__ bits,
                                                   uint32_t* __restrict__ cut, int n, int words)
{
    const int m = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    bool occ = false, part = false;
    if (m < n) {
        int lo, hi;
        sample_range(mm[m], lut_max, lo, hi);
        occ = next[lo] <= (uint32_t)hi;
        part = occ && unclipped && !((unclipped[m >> 5] >> (m & 31)) & 1u);
        occ = occ && !(gone && ((gone[m >> 5] >> (m & 31)) & 1u));
    }
    const unsigned long long v = __ballot(occ), c = __ballot(part);
    if ((threadIdx.x & 31) == 0 && (m >> 5) < words) {
        bits[m >> 5] = (uint32_t)(v >> (threadIdx.x & 32));
        if (cut) cut[m >> 5] = (uint32_t)(c >> (threadIdx.x & 32));
    }
}

/* group bits: bit g set iff any macrocell of group g (2^ER_GROUP_SHIFT macrocells a side, clipped to the
 * grid) has its bit set, from word `occ_base` of the same array; the groups' clip-free bits
 * from word `free_base`: bit g set iff no macrocell of group g has its bit in `cut` (k_macro_bits;
 * NULL: no clipping objects, every bit clear), so the march need not test its samples against
 * the clipping objects. One lane per group, which reads
 * its macrocells' bits a row of 4 at a time (one lane per 32 groups, bit by bit, took 340 us for
 * 16^3 groups; this takes 5). */
__device__ __forceinline__ uint32_t bit_run(const uint32_t* __restrict__ w, int first, int count)
{
    const int s = first & 31;
    uint32_t v = w[first >> 5] >> s;
    if (s + count > 32) v |= w[(first >> 5) + 1] << (32 - s);
    return v & ((1u << count) - 1u);
}
__global__ __launch_bounds__(256) void k_group_bits(uint32_t* __restrict__ bits, const uint32_t* __restrict__ cut,
                                                   int mx, int my, int mz, int gx, int gy, int gz, int occ_base,
                                                   int free_base, int words)
{
    const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    bool any = false, free = cut != nullptr;
    if (g < gx * gy * gz) {
        const int E = 1 << ER_GROUP_SHIFT;
        const int x = g % gx, y = (g / gx) % gy, z = g / (gx * gy);
        const int nx = min(E, mx - E * x);
        for (int k = E * z; k < min(E * z + E, mz); ++k)
            for (int j = E * y; j < min(E * y + E, my); ++j) {
                const int m = (k * my + j) * mx + E * x;
                any = any || bit_run(bits, m, nx) != 0u;
                if (cut) free = free && bit_run(cut, m, nx) == 0u;
            }
    } else {
        free = false;
    }
    const unsigned long long va = __ballot(any), vf = __ballot(free);
    if ((threadIdx.x & 31) == 0 && (g >> 5) < words) {
        bits[occ_base + (g >> 5)] = (uint32_t)(va >> (threadIdx.x & 32));
        bits[free_base + (g >> 5)] = (uint32_t)(vf >> (threadIdx.x & 32));
    }
}

/* The empty-space radius of every group: its Chebyshev distance to the nearest occupied group,
 * at most 15 (0 for an occupied group). The distance is taken axis by axis - along a row, the
 * steps to the nearest occupied group; then along each further axis the minimum over its
 * neighbours of the larger of the step and the neighbour's distance so far. AXIS 0 reads the
 * groups' occupancy bits, AXIS 2 packs the result, eight groups to a word. (The host did this,
 * between two copies that waited for the device.) */
template<int AXIS>
__global__ __launch_bounds__(256) void k_group_radii(const uint32_t* __restrict__ occ, const uint8_t* __restrict__ in,
                                                    uint8_t* __restrict__ out, uint32_t* __restrict__ packed, int gx, int gy,
                                                    int gz)
{
    const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int n = gx * gy * gz;
    int d = 15;
    if (g < n) {
        const int dim = AXIS == 0 ? gx : (AXIS == 1 ? gy : gz);
        const int step = AXIS == 0 ? 1 : (AXIS == 1 ? gx : gx * gy);
        const int at = AXIS == 0 ? g % gx : (AXIS == 1 ? (g / gx) % gy : g / (gx * gy));
        /* a neighbour r steps away cannot lower a distance of at most r */
        for (int r = 0; r < d; ++r)
            for (int s = -1; s <= 1; s += 2) {
                if (at + s * r < 0 || at + s * r >= dim) continue;
                const int h = g + s * r * step;
                const int v = AXIS == 0 ? (((occ[h >> 5] >> (h & 31)) & 1u) ? 0 : 15) : (int)in[h];
                d = min(d, max(r, v));
            }
    }
    if (AXIS < 2) {
        if (g < n) out[g] = (uint8_t)d;
    } else {
        uint32_t w = g < n ? (uint32_t)d << ((g & 7) * 4) : 0u;
        for (int o = 1; o < 8; o <<= 1) w |= (uint32_t)__shfl_xor((int)w, o);
        if ((g & 7) == 0 && g < n) packed[g >> 3] = w;
    }
}

/* ---- maximum GradientMagnitude over voxel centres (design: gradientmagnitude.cuh:28-70) ----
 * The six samples of a voxel take some 500 instructions (every voxel of 256^3: 240 us, of
 * 512 x 512 x 460: 1680 us, all of it instruction issue; now 179 and 426 us), and few bricks of 8^3 voxels can hold the maximum: a sample in the brick
 * lies between (the smallest voxel it can read) - 3 (truncating lerps) and the largest, so with R
 * their difference no gradient there exceeds the expression's value for a difference of R on
 * every axis (each operation is monotone). k_gm_bound finds that bound for every brick, one wave
 * per brick; in k_gm_max each wave takes ER_GM_RUN bricks, the one of the largest bound first,
 * offers its result as a lower limit for all waves, and then only the bricks whose bound exceeds
 * the largest offer so far. Which bricks are left out depends on timing, the maximum does not.
 * Few atomics: operations on one address go one after the other, some 6 ns each (an exchange
 * per brick took 790 us). prune = 0, where lattice coordinates are too coarse for the two-voxel
 * margin, takes every brick. */
#define ER_GM_RUN 64
__global__ __launch_bounds__(256) void k_gm_bound(const DevParams* __restrict__ pp, const uint16_t* __restrict__ vox,
                                                 float* __restrict__ bounds, int bx, int by, int nb, int prune)
{
    const DevParams& p = *pp;
    const int rx = p.res[0], ry = p.res[1], rz = p.res[2];
    const int lane = threadIdx.x & 63;
    const int b = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if (b >= nb) return;
    const int X = (b % bx) * 8, Y = ((b / bx) % by) * 8, Z = (b / (bx * by)) * 8;
    /* voxels [X - 2, X + 9], clamped to the volume, 12 on each axis */
    const int x = min(max(X - 2 + min(lane & 15, 11), 0), rx - 1);
    uint32_t lo = 0xffff, hi = 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int y = min(max(Y - 2 + 4 * j + (lane >> 4), 0), ry - 1);
#pragma unroll
        for (int i = 0; i < 12; ++i) {
            const int z = min(max(Z - 2 + i, 0), rz - 1);
            const uint32_t v = vox[((size_t)z * ry + y) * rx + x];
            lo = min(lo, v);
            hi = max(hi, v);
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, o));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, o));
    }
    const float R = (float)(hi - lo + 3u);
    const float g[6] = {0.0f, R, 0.0f, R, 0.0f, R};
    if (lane == 0) bounds[b] = prune ? gradient_magnitude_cd(p, g) : 3.402823466e+38f;
}

__global__ __launch_bounds__(256) void k_gm_max(const DevParams* __restrict__ pp, const float* __restrict__ bounds,
                                               unsigned int* __restrict__ out, int bx, int by, int nb)
{
    const DevParams& p = *pp;
    const int rx = p.res[0], ry = p.res[1], rz = p.res[2];
    const int lane = threadIdx.x & 63;
    const int waves = (int)(gridDim.x * (blockDim.x >> 6));
    const int w = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    /* the wave's bricks: w, w + waves, ...; lane k holds the bound of the k-th (at most ER_GM_RUN) */
    const int mine = w + lane * waves;
    float bound = lane < ER_GM_RUN && mine < nb ? bounds[mine] : -1.0f;
    if (!(bound == bound)) bound = 3.402823466e+38f;   /* a NaN excludes nothing */
    float best = 0.0f, seen = 0.0f;
    for (bool first = true;; first = false) {
        float top = bound;
        for (int o = 32; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
        if (!(top > fmaxf(best, seen))) break;
        const int k = __ffsll((long long)__ballot(bound == top)) - 1;
        const int b = w + k * waves;
        if (lane == k) bound = -1.0f;
        const int X = (b % bx) * 8, Y = ((b / bx) % by) * 8, Z = (b / (bx * by)) * 8;
        const int x = X + (lane & 7), y = Y + (lane >> 3);
        float m = 0.0f;
        if (x < rx && y < ry) {
            for (int z = Z; z < min(Z + 8, rz); ++z) {
                const f3 P = mk(p.minp[0] + p.size[0] * (((float)x + 0.5f) / (float)rx),
                                p.minp[1] + p.size[1] * (((float)y + 0.5f) / (float)ry),
                                p.minp[2] + p.size[2] * (((float)z + 0.5f) / (float)rz));
                m = fmaxf(m, gradient_magnitude(p, P));
            }
        }
        for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        best = fmaxf(best, m);
        if (first) {
            /* non-negative floats order like their bit patterns */
            unsigned int s = 0u;
            if (lane == 0) s = atomicMax(out, __float_as_uint(best));
            seen = __uint_as_float(__builtin_amdgcn_readfirstlane(s));
        }
    }
    if (lane == 0 && best > seen) atomicMax(out, __float_as_uint(best));
}

} /* namespace erd */

extern "C" hipError_t erd_launch_post(const erd::DevParams* p, const float4* frame, float4* running, uchar4* display,
                                      int no_iterations, unsigned int* qcount, int W, int H, hipStream_t st)
{
    dim3 grid((W + POST_TILE - 1) / POST_TILE, (H + POST_TILE - 1) / POST_TILE), block(256);
    hipLaunchKernelGGL(erd::k_post, grid, block, 0, st, p, frame, running, display, no_iterations, qcount);
    return hipGetLastError();
}

extern "C" hipError_t erd_launch_bilateral(const erd::BilateralParams* bp, const uchar4* in, uchar4* tmp, uchar4* out,
                                           int W, int H, hipStream_t st)
{
    dim3 grid((W + 15) / 16, (H + 15) / 16), block(256);
    hipLaunchKernelGGL(erd::k_bilateral<1>, grid, block, 0, st, bp, in, tmp, W, H);
    hipLaunchKernelGGL(erd::k_bilateral<0>, grid, block, 0, st, bp, (const uchar4*)tmp, out, W, H);
    return hipGetLastError();
}

extern "C" size_t erd_bilateral_params_size(void) { return sizeof(erd::BilateralParams); }

extern "C" hipError_t erd_launch_build_cells(const uint16_t* vox, uint4* cells, int rx, int ry, int rz, hipStream_t st)
{
    const unsigned int n = (unsigned int)(rx + 1) * (unsigned int)(ry + 1);
    const int runs = std::min((rz + 1 + ER_CELL_RUN - 1) / ER_CELL_RUN, 32768);   /* the kernel strides over more */
    hipLaunchKernelGGL(erd::k_build_cells, dim3((n + 255) / 256, runs), dim3(256), 0, st, vox, cells, rx, ry, rz);
    return hipGetLastError();
}

extern "C" hipError_t erd_launch_range_top(const uint32_t* mm, int n, unsigned int* top, hipStream_t st)
{
    hipLaunchKernelGGL(erd::k_range_top, dim3(1), dim3(1024), 0, st, mm, n, top);
    return hipGetLastError();
}

extern "C" hipError_t erd_launch_macro_minmax(const uint16_t* vox, uint32_t* mm, int rx, int ry, int rz, int mx, int my,
                                              int mz, int shift, hipStream_t st)
{
    if (shift <= 3) {
        const int per = (ER_ROW_COLUMNS - 1) >> shift;
        hipLaunchKernelGGL(erd::k_macro_rows, dim3((mx + per - 1) / per, std::min(my * mz, 32768)), dim3(ER_ROW_COLUMNS), 0, st,
                           vox, mm, rx, ry, rz, mx, my, shift, my * mz);
    } else {
        hipLaunchKernelGGL(erd::k_macro_minmax, dim3((mx * my * mz + 3) / 4), dim3(256), 0, st, vox, mm, rx, ry, rz, mx, my, mz,
                           shift);
    }
    return hipGetLastError();
}

extern "C" hipError_t erd_launch_macro_bits(const uint32_t* mm, const uint32_t* next, int lut_max, const uint32_t* gone,
                                            const uint32_t* unclipped, uint32_t* bits, uint32_t* cut, int n, int words,
                                            hipStream_t st)
{
    hipLaunchKernelGGL(erd::k_macro_bits, dim3((n + 255) / 256), dim3(256), 0, st, mm, next, lut_max, gone, unclipped, bits, cut,
                       n, words);
    return hipGetLastError();
}

/* the groups' occupancy bits (from word occ_base), clip-free bits (free_base) and radii
 * (radii_base); tmp: two bytes a group */
extern "C" hipError_t erd_launch_group_tables(uint32_t* bits, const uint32_t* cut, uint8_t* tmp, int mx, int my, int mz,
                                              int gx, int gy, int gz, int occ_base, int free_base, int radii_base, int words,
                                              hipStream_t st)
{
    const int n = gx * gy * gz;
    const dim3 grid((n + 255) / 256), block(256);
    uint8_t* tmp2 = tmp + n;
    const uint32_t* occ = bits + occ_base;
    hipLaunchKernelGGL(erd::k_group_bits, grid, block, 0, st, bits, cut, mx, my, mz, gx, gy, gz, occ_base, free_base, words);
    hipLaunchKernelGGL(erd::k_group_radii<0>, grid, block, 0, st, occ, (const uint8_t*)nullptr, tmp, (uint32_t*)nullptr, gx, gy, gz);
    hipLaunchKernelGGL(erd::k_group_radii<1>, grid, block, 0, st, occ, (const uint8_t*)tmp, tmp2, (uint32_t*)nullptr, gx, gy, gz);
    hipLaunchKernelGGL(erd::k_group_radii<2>, grid, block, 0, st, occ, (const uint8_t*)tmp2, tmp, bits + radii_base, gx, gy, gz);
    return hipGetLastError();
}

extern "C" hipError_t erd_launch_macro_sigma(const uint32_t* mm, const float* lut, int lut_max, float* out, int n, hipStream_t st)
{
    hipLaunchKernelGGL(erd::k_macro_sigma, dim3((n + 15) / 16), dim3(256), 0, st, mm, lut, lut_max, out, n);
    return hipGetLastError();
}

/* out: one word, zero before the call; bounds: one float per brick of 8^3 voxels */
extern "C" hipError_t erd_launch_gm_max(const erd::DevParams* p, const uint16_t* vox, float* bounds, unsigned int* out, int rx,
                                        int ry, int rz, int prune, hipStream_t st)
{
    const int bx = (rx + 7) / 8, by = (ry + 7) / 8, nb = bx * by * ((rz + 7) / 8);
    hipLaunchKernelGGL(erd::k_gm_bound, dim3((nb + 3) / 4), dim3(256), 0, st, p, vox, bounds, bx, by, nb, prune);
    /* ER_GM_RUN bricks to a wave, fewer where that would leave the device's 4 waves per CU idle */
    const int waves = std::max((nb + ER_GM_RUN - 1) / ER_GM_RUN, std::min(nb, 1024));
    hipLaunchKernelGGL(erd::k_gm_max, dim3((waves + 3) / 4), dim3(256), 0, st, p, (const float*)bounds, out, bx, by, nb);
    return hipGetLastError();
}

extern "C" hipError_t erd_launch_batch_post(const erd::BatchJob* J, int na, unsigned int round, int active_tiles,
                                            hipStream_t stream)
{
    if (na == 0 || active_tiles == 0) return hipSuccess;
    hipLaunchKernelGGL(erd::k_post_b, dim3(active_tiles), dim3(256), 0, stream, J, na, round);
    return hipGetLastError();
}
