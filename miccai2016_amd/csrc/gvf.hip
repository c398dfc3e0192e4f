// Gradient vector flow on gfx950: explicit-Euler steps on the three SoA
// components, ping-ponging two buffers, mirrored neighbours at the faces;
// one step per launch, or two to four per launch in a sweep along axis 0.
#include <algorithm>

#include "cmf_words.h"
#include "mh_common.h"
#include "mh_reduce.h"

namespace {

struct SumOp {
    __device__ static float identity() { return 0.f; }
    __device__ static float combine(float a, float b) { return a + b; }
};

// One step of one component at one voxel: out = g - dt (r (g - v) - mu lap),
// lap = sum_k rss_k ((g[-e_k] + g[+e_k]) - 2 g) over the axes, with the
// neighbour across a face replaced by the one on the inner side (m_k: the
// lower neighbour, p_k: the upper). Only explicit fused operations, so that
// every kernel below rounds identically. Returns delta.
__device__ __forceinline__ float gvf_voxel(float gi, float m0, float p0, float m1, float p1,
                                           float m2, float p2, float v, float r, float mu,
                                           float dt, float rss0, float rss1, float rss2,
                                           float &out)
{
#pragma clang fp contract(off)
    const float t0 = fmaf(-2.f, gi, m0 + p0);
    const float t1 = fmaf(-2.f, gi, m1 + p1);
    const float t2 = fmaf(-2.f, gi, m2 + p2);
    const float lap = fmaf(t2, rss2, fmaf(t1, rss1, t0 * rss0));
    const float delta = fmaf(-mu, lap, r * (gi - v));
    out = fmaf(-dt, delta, gi);
    return delta;
}

// |delta| of a voxel from its three components
__device__ __forceinline__ float gvf_mag(float d0, float d1, float d2)
{
#pragma clang fp contract(off)
    return sqrtf(fmaf(d2, d2, fmaf(d1, d1, d0 * d0)));
}

// One step over the volume. With `partials`, each block stores the sum of
// |delta| over its voxels.
__global__ void __launch_bounds__(mh::kBlock)
gvf_step_kernel(float *__restrict__ out, const float *__restrict__ g, const float *__restrict__ v,
                const float *__restrict__ r, int d0, int d1, int d2, float mu, float dt, float rss0,
                float rss1, float rss2, float *__restrict__ partials)
{
    const int64_t n = int64_t(d0) * d1 * d2;
    const unsigned b = mh::xcd_block(blockIdx.x, gridDim.x);
    const int64_t i = int64_t(b) * blockDim.x + threadIdx.x;
    float dmag = 0.f;
    if (i < n) {
        const int i2 = int(i % d2);
        const int i1 = int((i / d2) % d1);
        const int i0 = int(i / (int64_t(d2) * d1));
        const int64_t s0 = int64_t(d1) * d2, s1 = d2;
        const int64_t b0 = i0 > 0 ? -s0 : s0, a0 = i0 < d0 - 1 ? s0 : -s0;
        const int64_t b1 = i1 > 0 ? -s1 : s1, a1 = i1 < d1 - 1 ? s1 : -s1;
        const int64_t b2 = i2 > 0 ? -1 : 1, a2 = i2 < d2 - 1 ? 1 : -1;
        const float ri = r[i];
        float dl[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float *gc = g + c * n;
            float o;
            dl[c] = gvf_voxel(gc[i], gc[i + b0], gc[i + a0], gc[i + b1], gc[i + a1], gc[i + b2],
                              gc[i + a2], v[c * n + i], ri, mu, dt, rss0, rss1, rss2, o);
            out[c * n + i] = o;
        }
        dmag = gvf_mag(dl[0], dl[1], dl[2]);
    }
    if (!partials) return;
    dmag = mh::block_reduce<SumOp>(dmag);
    if (threadIdx.x == 0) partials[blockIdx.x] = dmag;
}

// word 3 of a buffer's resource: a 32-bit format, offsets checked against its
// bytes (loads beyond it give zero, stores none)
constexpr int kRawBuffer = 0x00027000;

// L steps per launch, temporally blocked along axis 0 (as the max-flow sweep
// is). A work-group owns an output tile of TY x TX voxels in the (axis 1, axis 2)
// plane and a chunk of planes [z0, z1), one thread per point of the tile widened
// by L on every side. Step z puts g of plane z into LDS and after the step's one
// barrier computes, for l = 1 .. L,
//   level l: the l-th step at plane z - l + 1 on the tile widened by L - l, from
//            level l - 1 of the same plane in LDS (written a step ago; level 0:
//            before the barrier) and of the planes around it in registers,
//            into LDS by plane parity; level L is stored.
// LDS holds two planes of each level (by plane parity), so one barrier per step
// orders every write before the reads that need it and after the reads of the
// plane two steps back. The per-voxel arithmetic is gvf_voxel's, so the result
// equals L launches of gvf_step_kernel bit for bit. With `partials`, each
// work-group stores the sum of |delta| of its last step.
//
// Loads run two planes ahead and go through buffer resources, whose bounds mask
// the lanes outside the volume: without branches around them the compiler knows
// how many are under way and waits for none but the plane it needs. They are
// issued between the levels (all seven at once hold up the waves at the step's
// start: 8 % more). A step of all work-groups takes about 1.0 + 0.25 L us, the first
// part for the loads and stores of 64 threads each (tiles of 24 columns 1.2: rows of
// 128 bytes off their alignment), the second for the arithmetic; so three and four
// levels often win although their halos cost more: 150 x 128 x 141 11.6 us a GVF step
// in four levels, 11.7 in three, 13.2 in two (below), 17.0 in one step per launch.
template <int TY, int TX, int NT, int L>
__global__ void __launch_bounds__(NT)
gvf_sweep_kernel(float *__restrict__ out, const float *__restrict__ g, const float *__restrict__ v,
                 const float *__restrict__ r, int d0, int d1, int d2, float mu, float dt, float rss0,
                 float rss1, float rss2, int zchunk, float *__restrict__ partials)
{
    constexpr int EY = TY + 2 * L, EX = TX + 2 * L, NE = EY * EX;
    static_assert(NE <= NT, "one point per thread");
    extern __shared__ float lds[];  // level l of plane parity q, component c: 3 (2 l + q) + c
    const unsigned b = mh::xcd_block(blockIdx.x, gridDim.x);
    const int ntx = (d2 + TX - 1) / TX, nty = (d1 + TY - 1) / TY;
    const int tx = int(b % unsigned(ntx)), ty = int((b / unsigned(ntx)) % unsigned(nty));
    const int tz = int(b / unsigned(ntx * nty));
    const int z0 = tz * zchunk, z1 = min(z0 + zchunk, d0);
    const int t = int(threadIdx.x);
    const bool live = t < NE;
    const int yy = live ? t / EX : 0, xx = live ? t % EX : 0;
    const int p = yy * EX + xx;
    const int y = ty * TY - L + yy, x = tx * TX - L + xx;
    const bool inv = live && y >= 0 && y < d1 && x >= 0 && x < d2;
    // levels up to this one are computed at this point
    const int most = inv ? min(min(min(yy, EY - 1 - yy), min(xx, EX - 1 - xx)), L) : 0;
    // in-plane neighbours in LDS, mirrored at the faces
    const int pym = y > 0 ? p - EX : p + EX, pyp = y < d1 - 1 ? p + EX : p - EX;
    const int pxm = x > 0 ? p - 1 : p + 1, pxp = x < d2 - 1 ? p + 1 : p - 1;
    const int64_t n = int64_t(d0) * d1 * d2;
    const unsigned st0 = unsigned(d1) * unsigned(d2), plane = 4u * st0;
    // byte offset in a plane; lanes that load or store nothing lie beyond it
    const unsigned here4 = 4u * (unsigned(y) * unsigned(d2) + unsigned(x));
    const unsigned in_g = inv ? here4 : ~0u, in_v = most > 0 ? here4 : ~0u, in_o = most == L ? here4 : ~0u;
    auto load = [&](const float *f, int k, unsigned off) {
        return __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(
                       __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(f) + int64_t(k) * st0, 0,
                                                         int(plane), kRawBuffer),
                       int(off), 0, 0));
    };

    const int zs = max(z0 - (L - 1), 0);   // first plane of level 1
    const int zend = z1 - 1 + (L - 1);     // the last step
    // Planes in registers, by their distance from zs modulo 6 (g, v, r) or 3 (the
    // levels), so that none is ever moved: a move would wait for the loads.
    float G[6][3], V[6][3], R[6], H[L][3][3];  // H[0] is not used
    float dsum = 0.f;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        R[k] = 0.f;
#pragma unroll
        for (int c = 0; c < 3; ++c) G[k][c] = V[k][c] = 0.f;
    }
#pragma unroll
    for (int l = 0; l < L; ++l)
#pragma unroll
        for (int k = 0; k < 9; ++k) H[l][k / 3][k % 3] = 0.f;
    // inputs that step z is the first to use, loaded two steps ahead: g of plane
    // z + 1, v and r of plane z (beyond the volume: the last plane's, not used)
    auto fetch_g = [&](auto PH, int z) {
#pragma unroll
        for (int c = 0; c < 3; ++c) G[(PH + 1) % 6][c] = load(g + c * n, min(z + 1, d0 - 1), in_g);
    };
    auto fetch_v = [&](auto PH, int z) {
#pragma unroll
        for (int c = 0; c < 3; ++c) V[PH][c] = load(v + c * n, min(z, d0 - 1), in_v);
        R[PH] = load(r, min(z, d0 - 1), in_v);
    };
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        G[0][c] = load(g + c * n, zs, in_g);
        G[5][c] = load(g + c * n, max(zs - 1, 0), in_g);
    }
    fetch_g(std::integral_constant<int, 0>{}, zs);
    fetch_v(std::integral_constant<int, 0>{}, zs);
    fetch_g(std::integral_constant<int, 1>{}, zs + 1);
    fetch_v(std::integral_constant<int, 1>{}, zs + 1);
    auto step = [&](auto PH, int z) {
        if (live) {
#pragma unroll
            for (int c = 0; c < 3; ++c) lds[(3 * (PH % 2) + c) * NE + p] = G[PH][c];
        }
        mh::lds_barrier();
        mh::unrolled_while<L>([&](auto LC) {
            constexpr int l = LC + 1, kk = (PH + 13 - l) % 6;  // its plane: z - l + 1
            constexpr int q = kk % 2;
            const int k = z - l + 1;
            float o[3] = {0.f, 0.f, 0.f};
            const bool on = k >= z0 - (L - l) && k >= 0 && k < z1 + (L - l) && k < d0;
            if (on) {
                float(&mid)[3] = l == 1 ? G[kk] : H[l - 1][kk % 3];
                float(&below)[3] = l == 1 ? G[(kk + 5) % 6] : H[l - 1][(kk + 2) % 3];
                float(&above)[3] = l == 1 ? G[(kk + 1) % 6] : H[l - 1][(kk + 1) % 3];
                if (k == 0) {  // mirrored
#pragma unroll
                    for (int c = 0; c < 3; ++c) below[c] = above[c];
                }
                if (k == d0 - 1) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) above[c] = below[c];
                }
                if (most >= l) {
                    const float *S = lds + 3 * (2 * (l - 1) + q) * NE;
                    float dl[3];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        dl[c] = gvf_voxel(mid[c], below[c], above[c], S[c * NE + pym], S[c * NE + pyp],
                                          S[c * NE + pxm], S[c * NE + pxp], V[kk][c], R[kk], mu, dt,
                                          rss0, rss1, rss2, o[c]);
                        if (l < L) lds[(3 * (2 * l + q) + c) * NE + p] = o[c];
                    }
                    if (l == L && partials) dsum += gvf_mag(dl[0], dl[1], dl[2]);
                }
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (l < L)
                    H[l < L ? l : 0][kk % 3][c] = o[c];
                else
                    __builtin_amdgcn_raw_buffer_store_b32(
                        __builtin_bit_cast(unsigned, o[c]),
                        __builtin_amdgcn_make_buffer_rsrc(out + c * n + int64_t(on ? k : 0) * st0, 0,
                                                          on ? int(plane) : 0, kRawBuffer),
                        int(in_o), 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (l == 1) fetch_g(std::integral_constant<int, (PH + 2) % 6>{}, z + 2);
            if (l == 2) fetch_v(std::integral_constant<int, (PH + 2) % 6>{}, z + 2);
            __builtin_amdgcn_sched_barrier(0);
            return true;
        });
    };
    for (int z = zs; z <= zend; z += 6)
        mh::unrolled_while<6>([&](auto PH) {
            step(PH, z + PH);
            return z + PH < zend;
        });
    if (!partials) return;
    dsum = mh::block_reduce<SumOp>(dsum);
    if (t == 0) partials[blockIdx.x] = dsum;
}

// Two steps per launch in the same way with every plane moved on in registers: 55 of
// them, so that a compute unit holds two work-groups and one's loads hide behind the
// other's arithmetic. A plane step of 512 work-groups takes 1.8 us, of 256 1.05; fewer
// levels read and write more often, so it is the faster while the fields stay in the
// last-level cache and its tiles fill the device better (128^3 10.7 us a step against
// 11.3 to 12.8 in three and four levels, 172 x 173 x 122 15.3 and 18.2, 500 x 100 x 60
// 12.8 and 14.6; but 150 x 128 x 141 13.2 and 11.6, 183 x 158 x 191 22.0 and 20.5).
template <int TY, int TX, int NT>
__global__ void __launch_bounds__(NT)
gvf_two_step_kernel(float *__restrict__ out, const float *__restrict__ g, const float *__restrict__ v,
                 const float *__restrict__ r, int d0, int d1, int d2, float mu, float dt, float rss0,
                 float rss1, float rss2, int zchunk, float *__restrict__ partials)
{
    constexpr int EY = TY + 4, EX = TX + 4, NE = EY * EX;
    static_assert(NE <= NT, "one point per thread");
    __shared__ float sG[2][3][NE];  // g of plane z, by plane parity
    __shared__ float sH[2][3][NE];  // level-A result of plane z, by plane parity
    const unsigned b = mh::xcd_block(blockIdx.x, gridDim.x);
    const int ntx = (d2 + TX - 1) / TX, nty = (d1 + TY - 1) / TY;
    const int tx = int(b % unsigned(ntx)), ty = int((b / unsigned(ntx)) % unsigned(nty));
    const int tz = int(b / unsigned(ntx * nty));
    const int x0 = tx * TX, y0 = ty * TY, z0 = tz * zchunk;
    const int z1 = min(z0 + zchunk, d0);
    const int t = int(threadIdx.x);
    const bool live = t < NE;
    const int yy = live ? t / EX : 0, xx = live ? t % EX : 0;
    const int p = yy * EX + xx;
    const int y = y0 - 2 + yy, x = x0 - 2 + xx;
    const bool inv = live && y >= 0 && y < d1 && x >= 0 && x < d2;
    const bool inE1 = inv && yy >= 1 && yy <= TY + 2 && xx >= 1 && xx <= TX + 2;
    const bool inO = inv && yy >= 2 && yy <= TY + 1 && xx >= 2 && xx <= TX + 1;
    // in-plane neighbours in LDS, mirrored at the faces (inside E2 for E1)
    const int pym = y > 0 ? p - EX : p + EX, pyp = y < d1 - 1 ? p + EX : p - EX;
    const int pxm = x > 0 ? p - 1 : p + 1, pxp = x < d2 - 1 ? p + 1 : p - 1;
    const int64_t n = int64_t(d0) * d1 * d2, st0 = int64_t(d1) * d2;
    const int64_t ip = inv ? int64_t(y) * d2 + x : 0;
    auto at = [&](int z) { return int64_t(z) * st0 + ip; };

    const int zs = max(z0 - 1, 0);  // first level-A plane
    const int zend = z1;            // last step (level A only below d0)
    float gm[3], gc[3], gp[3], gn[3];    // g at planes z - 1, z, z + 1 (mirrored), z + 2
    float vA[3], vB[3], vN[3];           // v at planes z, z - 1, z + 1
    float rA = 0.f, rB = 0.f, rN = 0.f;
    float h2[3], h1[3], h0[3];           // level A at planes z - 2, z - 1, z
    float dsum = 0.f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        gm[c] = gc[c] = gp[c] = gn[c] = vA[c] = vB[c] = vN[c] = h2[c] = h1[c] = h0[c] = 0.f;
    }
    if (inv) {
        const int zm = zs > 0 ? zs - 1 : zs + 1, zp = zs < d0 - 1 ? zs + 1 : zs - 1;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            gc[c] = g[c * n + at(zs)];
            gm[c] = g[c * n + at(zm)];
            gp[c] = g[c * n + at(zp)];
        }
    }
    if (inE1) {
#pragma unroll
        for (int c = 0; c < 3; ++c) vA[c] = v[c * n + at(zs)];
        rA = r[at(zs)];
    }
    for (int z = zs; z <= zend; ++z) {
        const bool la = z < d0;                  // level A at plane z
        const bool lb = z - 1 >= z0;             // level B at plane z - 1 (< z1 since z <= z1)
        const int q = z & 1, qb = (z - 1) & 1;
        // inputs of the next step
        if (inv && z + 1 < d0) {
            if (z + 2 < d0) {
#pragma unroll
                for (int c = 0; c < 3; ++c) gn[c] = g[c * n + at(z + 2)];
            } else {  // plane z + 1 is the last: its upper neighbour mirrors to plane z
#pragma unroll
                for (int c = 0; c < 3; ++c) gn[c] = gc[c];
            }
        }
        if (inE1 && z + 1 < d0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) vN[c] = v[c * n + at(z + 1)];
            rN = r[at(z + 1)];
        }
        if (la && live) {
#pragma unroll
            for (int c = 0; c < 3; ++c) sG[q][c][p] = gc[c];
        }
        __syncthreads();
        if (la && inE1) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                h0[c] = 0.f;
                (void)gvf_voxel(gc[c], gm[c], gp[c], sG[q][c][pym], sG[q][c][pyp], sG[q][c][pxm],
                                sG[q][c][pxp], vA[c], rA, mu, dt, rss0, rss1, rss2, h0[c]);
                sH[q][c][p] = h0[c];
            }
        }
        if (lb && inO) {
            const int zb = z - 1;
            float dl[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float below = zb > 0 ? h2[c] : h0[c];
                const float above = zb < d0 - 1 ? h0[c] : h2[c];
                float o;
                dl[c] = gvf_voxel(h1[c], below, above, sH[qb][c][pym], sH[qb][c][pyp],
                                  sH[qb][c][pxm], sH[qb][c][pxp], vB[c], rB, mu, dt, rss0, rss1,
                                  rss2, o);
                out[c * n + at(zb)] = o;
            }
            if (partials) dsum += gvf_mag(dl[0], dl[1], dl[2]);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            gm[c] = gc[c];
            gc[c] = gp[c];
            gp[c] = gn[c];
            h2[c] = h1[c];
            h1[c] = h0[c];
            vB[c] = vA[c];
            vA[c] = vN[c];
        }
        rB = rA;
        rA = rN;
    }
    if (!partials) return;
    dsum = mh::block_reduce<SumOp>(dsum);
    if (threadIdx.x == 0) partials[blockIdx.x] = dsum;
}

struct GvfShape {
    int ty, tx, nt, levels;
    int per_cu;       // resident work-groups of a compute unit
    double unit[2];   // microseconds a plane step takes with one and two of them on each
    int64_t voxels;   // of volumes it is taken for
    const void *kernel;
    int lds() const { return per_cu > 1 ? 0 : 4 * levels * 6 * (ty + 2 * levels) * (tx + 2 * levels); }
};
// (the two-step kernel up to 5.4 million voxels, whose 40 bytes each are 216 MB: at
// 5.3 and 5.1 million it is the faster by 5 and 13 % where it is chosen, at 5.5 and 5.8
// million the slower by 7 and 9 %)
#define GVF_SHAPE(TY, TX, NT, L, UNIT) \
    {TY, TX, NT, L, 1, {UNIT, UNIT}, int64_t(1) << 31, \
     reinterpret_cast<const void *>(&gvf_sweep_kernel<TY, TX, NT, L>)}
#define GVF_PAIR(TY, TX) \
    {TY, TX, 1024, 2, 2, {1.45, 2.55}, 5400000, \
     reinterpret_cast<const void *>(&gvf_two_step_kernel<TY, TX, 1024>)}
const GvfShape kGvfShapes[] = {GVF_PAIR(11, 64), GVF_PAIR(12, 60), GVF_SHAPE(12, 50, 1024, 3, 1.6),
                               GVF_SHAPE(10, 58, 1024, 3, 1.52), GVF_SHAPE(6, 74, 960, 3, 1.34),
                               GVF_SHAPE(24, 24, 1024, 4, 1.95)};
#undef GVF_SHAPE
#undef GVF_PAIR

// Sum of the per-block partials in block order (one work-group).
__global__ void __launch_bounds__(mh::kBlock)
sum_partials_kernel(const float *__restrict__ partials, int nparts, float *__restrict__ out)
{
    float s = 0.f;
    for (int k = threadIdx.x; k < nparts; k += blockDim.x) s += partials[k];
    s = mh::block_reduce<SumOp>(s);
    if (threadIdx.x == 0) *out = s;
}

__global__ void __launch_bounds__(mh::kBlock)
response_kernel(float *__restrict__ r, const float *__restrict__ v, int64_t n)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float a = v[i], b = v[n + i], c = v[2 * n + i];
    r[i] = a * a + b * b + c * c;
}

__global__ void __launch_bounds__(mh::kBlock) normalize_kernel(float *g, int64_t n)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float a = g[i], b = g[n + i], c = g[2 * n + i];
    const float nrm = sqrtf(a * a + b * b + c * c);
    if (nrm != 0.f) {
        const float k = 1.f / nrm;
        g[i] = k * a;
        g[n + i] = k * b;
        g[2 * n + i] = k * c;
    }
}

}  // namespace

MH_EXPORT int64_t mh_gvf_work_floats(const int64_t dims[3])
{
    if (!mh::dims_ok(dims)) return -1;
    return int64_t(mh::blocks_for(dims[0] * dims[1] * dims[2])) + 64;
}

MH_EXPORT int mh_gvf_response(mh_ctx *ctx, float *r, const float *v3, int64_t n, void *stream)
{
    MH_REQUIRE(ctx, r && v3 && n >= 0 && n < (int64_t(1) << 31), "bad arguments");
    if (n == 0) return MH_OK;
    hipLaunchKernelGGL(response_kernel, dim3(mh::blocks_for(n)), dim3(mh::kBlock), 0,
                       (hipStream_t)stream, r, v3, n);
    MH_CHECK_LAUNCH(ctx, "response_kernel");
    return MH_OK;
}

struct GvfPlan {
    const GvfShape *shape = nullptr;  // null: one step per launch
    int zchunk = 0;
    int64_t groups = 0;
};

// The shape and plane chunk that take the fewest microseconds per step on a device
// of `cus` compute units: a launch's work-groups run in ceil(groups / resident ones)
// waves of chunk + 2 (levels - 1) plane steps, and a launch costs 2.5 beside them; the
// chunk must leave at most max_groups groups. One step per launch takes 2.2 + 5.6 per
// million voxels, the less up to about 80^3 (4.9 us a step there, 5.2 in three levels;
// 96^3 6.6 and 5.4, 110^3 9.6 and 6.6, 220 x 215 x 210 93 and 38). `any`: a sweep in
// any case. (Of 95 volumes of 0.15 to 33 million voxels the plan's choice is on
// average 1.0 % off the fastest shape and chunk, at most 13 %.)
GvfPlan gvf_plan(int cus, const int64_t dims[3], int iters, int64_t max_groups, bool any)
{
    GvfPlan best;
    // planes beyond the bytes of a buffer resource: the two-step kernel has none (and
    // volumes of such planes read the less from memory)
    const bool wide = 4 * dims[1] * dims[2] >= (int64_t(1) << 31);
    double cost = any || wide ? 1e30 : 2.2 + 5.6e-6 * double(dims[0]) * double(dims[1]) * double(dims[2]);
    if (cost < 3.0) return best;  // no sweep takes less
    const int d0 = int(dims[0]);
    for (const GvfShape &S : kGvfShapes) {
        if (iters < S.levels) continue;
        if (wide ? S.per_cu == 1 : !any && dims[0] * dims[1] * dims[2] > S.voxels) continue;
        const int64_t tiles = ((dims[2] + S.tx - 1) / S.tx) * ((dims[1] + S.ty - 1) / S.ty);
        const int64_t slots = int64_t(cus) * S.per_cu;
        // as many chunks as fill the device once, twice, ..
        for (int64_t waves = (tiles + cus - 1) / cus, k = 0; k < 8; ++waves, ++k) {
            const int chunks = int(std::min<int64_t>(d0, waves * cus / tiles));
            const int z = (d0 + chunks - 1) / chunks;
            const int64_t groups = tiles * ((d0 + z - 1) / z);
            if (groups > max_groups) break;
            const int64_t rest = groups % slots;
            const double step = double(groups / slots) * S.unit[S.per_cu - 1] +
                                (rest == 0 ? 0.0 : S.unit[rest <= cus ? 0 : 1]);
            const double c = ((z + 2 * (S.levels - 1)) * step + 2.5) / S.levels;
            if (c < cost) {
                cost = c;
                best.shape = &S;
                best.zchunk = z;
                best.groups = groups;
            }
        }
    }
    return best;
}

int gvf_compute_units(mh_ctx *ctx)
{
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess ||
        cus <= 0)
        cus = 256;
    (void)hipGetLastError();
    return cus;
}

MH_EXPORT int mh_gvf_plan(const int64_t dims[3], int iters, int compute_units, int plan[4])
{
    if (!mh::dims_ok(dims) || compute_units < 1) return MH_ERR_ARG;
    const GvfPlan P = gvf_plan(compute_units, dims, iters,
                               int64_t(mh::blocks_for(dims[0] * dims[1] * dims[2])), false);
    if (!P.shape) return 1;
    if (plan) {
        const int v[4] = {P.shape->ty, P.shape->tx, P.zchunk, int(P.groups)};
        std::copy(v, v + 4, plan);
    }
    return P.shape->levels;
}

MH_EXPORT int mh_gvf(mh_ctx *ctx, float *g3, float *swap3, const float *v3, const float *r,
                     const int64_t dims[3], const mh_gvf_params *p, int iters, float *mag,
                     float *work, void *stream)
{
    MH_REQUIRE(ctx, mh::dims_ok(dims), "bad dims");
    MH_REQUIRE(ctx, dims[0] >= 2 && dims[1] >= 2 && dims[2] >= 2, "every dim must be >= 2");
    MH_REQUIRE(ctx, g3 && swap3 && v3 && r && p && iters >= 0, "bad arguments");
    MH_REQUIRE(ctx, !mag || work, "mag_dev needs work_dev");
    const int64_t n = dims[0] * dims[1] * dims[2];
    const unsigned nb = mh::blocks_for(n);
    hipStream_t s = (hipStream_t)stream;
    float *src = g3, *dst = swap3;
    // several steps per launch where that is faster; the partial sums of the
    // last launch fit in the workspace's nb floats
    GvfPlan P;
    if (ctx->gvf_sweep != 1 && iters >= 2)
        P = gvf_plan(gvf_compute_units(ctx), dims, iters, int64_t(nb), ctx->gvf_sweep == 2);
    const int levels = P.shape ? P.shape->levels : 1;
    if (P.shape)
        MH_CHECK(ctx, hipFuncSetAttribute(P.shape->kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                          P.shape->lds()));
    int it = 0;
    auto step = [&](float *parts) {
        hipLaunchKernelGGL(gvf_step_kernel, dim3(nb), dim3(mh::kBlock), 0, s, dst, src, v3, r,
                           int(dims[0]), int(dims[1]), int(dims[2]), p->mu, p->dt, p->rss[0],
                           p->rss[1], p->rss[2], parts);
        if (parts)
            hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(mh::kBlock), 0, s, parts, int(nb), mag);
        float *t = src;
        src = dst;
        dst = t;
        ++it;
    };
    while ((iters - it) % levels) step((mag && it == iters - 1) ? work : nullptr);
    while (P.shape && it < iters) {
        float *parts = (mag && it + levels == iters) ? work : nullptr;
        int d0 = int(dims[0]), d1 = int(dims[1]), d2 = int(dims[2]);
        float mu = p->mu, dt = p->dt, r0 = p->rss[0], r1 = p->rss[1], r2 = p->rss[2];
        void *args[] = {&dst, &src, &v3, &r, &d0, &d1, &d2, &mu, &dt, &r0, &r1, &r2, &P.zchunk, &parts};
        MH_CHECK(ctx, hipLaunchKernel(P.shape->kernel, dim3(unsigned(P.groups)),
                                      dim3(unsigned(P.shape->nt)), args, size_t(P.shape->lds()), s));
        if (parts)
            hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(mh::kBlock), 0, s, parts,
                               int(P.groups), mag);
        float *t = src;
        src = dst;
        dst = t;
        it += levels;
    }
    while (it < iters) step((mag && it == iters - 1) ? work : nullptr);
    MH_CHECK_LAUNCH(ctx, "gvf kernels");
    if (src != g3) MH_CHECK(ctx, hipMemcpyAsync(g3, src, sizeof(float) * 3 * n, hipMemcpyDeviceToDevice, s));
    return MH_OK;
}

MH_EXPORT int mh_gvf_set_sweep(mh_ctx *ctx, int mode)
{
    if (!ctx) return MH_ERR_ARG;
    MH_REQUIRE(ctx, mode >= 0 && mode <= 2, "mode 0 (automatic), 1 (off) or 2 (on)");
    ctx->gvf_sweep = mode;
    return MH_OK;
}

MH_EXPORT int mh_gvf_normalize(mh_ctx *ctx, float *g3, int64_t n, void *stream)
{
    MH_REQUIRE(ctx, g3 && n >= 0 && n < (int64_t(1) << 31), "bad arguments");
    if (n == 0) return MH_OK;
    hipLaunchKernelGGL(normalize_kernel, dim3(mh::blocks_for(n)), dim3(mh::kBlock), 0,
                       (hipStream_t)stream, g3, n);
    MH_CHECK_LAUNCH(ctx, "normalize_kernel");
    return MH_OK;
}
