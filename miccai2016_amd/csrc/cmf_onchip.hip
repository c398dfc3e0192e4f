// Max-flow solves whose whole state stays on the chip.
//
// The state and inputs of a voxel are 12 to 19 floats; the 256 compute units
// hold 128 MB of registers, so a volume of up to 2^21 voxels (128^3) fits. A
// volume is cut into bricks of V planes x b1 x b2 voxels, one work-group per
// brick and compute unit, a thread per in-plane position holding its V voxels
// along axis 0 in registers for the whole solve: the fields are read once, u
// is written once, and an iteration moves nothing through memory but the
// brick faces.
//
// In-plane neighbours go through LDS, axis-0 neighbours are the thread's own
// registers, and the faces of neighbouring bricks travel as tagged words: a
// 64-bit store carries the iteration's tag beside the value, and the receiver
// polls the word itself until the tag is the one it waits for, so that no flag,
// fence or cache flush orders the exchange (one hop measures 1.0 us for 256
// words, 1.3 us for 1024). One iteration is
//   p-step, planes downwards: the top plane's h0, the last row's h1 and the
//     last column's h2 go to the next bricks as they are formed;
//   receive the previous bricks' h0, h1, h2; barrier;
//   u-step, planes upwards: the first plane's, row's and column's residuals go
//     to the previous bricks as they are formed;
//   receive the next bricks' residuals; barrier.
// Every word is written again only after the words it depends on came back, so
// one slot per word suffices (the criterion's two sets alternate). Every wait
// is bounded: after kWaitSpins loads without its word a work-group raises the abort
// flag, every wait ends, and the host restores u and solves another way.
//
// Bound at 128^3 by the issue of 74 vector instructions per voxel, 3.95 of 4.4 to
// 4.6 us an iteration (16.0 in the three-level sweep); below about 80^3 by the two
// exchanges (64^3 2.6 us, 6.1 in the per-iteration kernels). Words are polled as
// their phase ends, by all threads: polled after the barrier by the waves that
// read them 5.3 us at 128^3 (4.8 in the same run); two work-groups of half the size
// per compute unit are no faster (96^3 4.1 against 3.7 us).
//
// The per-voxel arithmetic is cmf_voxel.h's, so the result equals the
// per-iteration kernels' bit for bit; the criterion's sum is taken in another
// order.
#include <algorithm>
#include <climits>
#include <mutex>
#include <vector>

#include "cmf_onchip.h"
#include "cmf_voxel.h"
#include "cmf_words.h"
#include "mh_reduce.h"

namespace {

using namespace mh;

constexpr int kMaxThreads = 1024;
constexpr int kMaxPlanes = 8;   // per thread, constant eigenvalues (l0, l1, l1); else half
constexpr int kCells = 1184;    // LDS cells of a tile and its faces
constexpr int kWords = 2;       // in-plane words a thread receives per phase
constexpr int kRedFloats = 64;  // three sets of the waves' sums, the failure flag last

struct SumOp {
    __device__ static float identity() { return 0.f; }
    __device__ static float combine(float a, float b) { return a + b; }
};

// modes of the p-step
constexpr int kAxial = 0;      // constant eigenvalues (l0, l1, l1)
constexpr int kConst = 1;      // other constant eigenvalues
constexpr int kPointwise = 2;  // eigenvalues of their own at every voxel

struct Args {
    const mh::OnchipSolve *solves;
    int nsolves, nslots;
    mh::OnchipFields F;
    int d0, d1, d2;
    int b1, b2, nt1, nt2, nz;
    int num_iter, update;
    float rcc, inv_rcc, rs0, rs1, rs2, ss0, ss1, ss2, error_bound, inv_n_rcc;
    float sq0, sq1, sq2, rq0, rq1, rq2;
    mh::AxiParams A;
    Word *inbox;      // per brick: [z residuals | z h0 | in-plane residuals | in-plane h1, h2]
    Word *parts;      // criterion partials, two sets per slot
    int *abort;
};

// One volume's solves, or one solve of each of up to N volumes side by side:
// volume v's work-groups are first[v] .. first[v + 1] - 1. An iteration's two
// exchanges take as long for a small volume as for a large one (64^3 2.6 us on
// 128 or 256 compute units), so several share them (packed per-iteration
// kernels: 10.6 us an iteration for a few volumes below 80^3).
template <int N>
struct ArgsOf {
    Args a[N];
    int n, first[N + 1];
};
constexpr int kMany = int(mh::kOnchipMany);

// Where a thread's 128 registers do not hold its planes, cs and ct are in LDS:
// of 8 planes all cs and the upper four's ct (160 KB are then full), of 4 planes
// with pointwise eigenvalues all of both.
constexpr bool caps_in_lds(int v, int mode) { return v == 8 || (v == 4 && mode == kPointwise); }
constexpr int lds_bytes(int v, int mode)
{
    return 4 * (3 * v * kCells + kRedFloats +
                (caps_in_lds(v, mode) ? (v + 4) * kMaxThreads : 0));
}

template <int V, int MODE, bool SUP, bool DEFER, int N = 1>
__global__ void __launch_bounds__(kMaxThreads)
cmf_onchip_kernel(const ArgsOf<N> L)
{
    unsigned b = mh::xcd_block(blockIdx.x, gridDim.x);
    int vol = 0;
    if (N > 1) {
        while (vol + 1 < L.n && int(b) >= L.first[vol + 1]) ++vol;
        vol = __builtin_amdgcn_readfirstlane(vol);
        b -= unsigned(L.first[vol]);
    }
    const Args &A = L.a[vol];
    constexpr int G = V < 4 ? V : 4, NG = V / G;
    constexpr int NF = MODE == kAxial ? 3 : MODE == kConst ? 4 : 7;
    constexpr int kTile = NG * kCells;  // LDS vectors of one field
    constexpr bool kCapLds = caps_in_lds(V, MODE);
    using VecG = Vec<G>;
    extern __shared__ __align__(16) unsigned char lds[];
    const int t = int(threadIdx.x), NT = int(blockDim.x);
    const int b1 = A.b1, b2 = A.b2, nc = b1 * b2;
    // LDS: the residual, h1 and h2 tiles, NG of kCells vectors of G planes
    // each. Cells: the brick's own [0, nc), the row beyond it [nc, nc + b2)
    // (after it for the residual, before it for h1), the column beyond it
    // [nc + b2, nc + b2 + b1) (h2's lies in h1's tile), and a zero at the end.
    VecG *sT = reinterpret_cast<VecG *>(lds);
    float *fT = reinterpret_cast<float *>(sT);
    float *red = fT + (3 * kTile + (kCapLds ? (NG + 1) * kMaxThreads : 0)) * G;
    int *fail = reinterpret_cast<int *>(red + kRedFloats - 1);

    const int per = A.nt1 * A.nt2 * A.nz;
    const int slot = int(b) / per, lb = int(b) - slot * per;
    const int bx = lb % A.nt2, by = (lb / A.nt2) % A.nt1, bz = lb / (A.nt1 * A.nt2);
    const bool live = t < nc;
    const int y = live ? t / b2 : 0, x = live ? t - y * b2 : 0, cell = live ? t : 0;
    const int gy = by * b1 + y, gx = bx * b2 + x, z0 = bz * V;
    const bool inv = live && gy < A.d1 && gx < A.d2;
    const int nz = min(V, A.d0 - z0);
    const int last0 = A.d0 - 1 - z0;  // the volume's last plane, counted from z0
    const bool e1 = gy < A.d1 - 1, e2 = gx < A.d2 - 1;
    const bool zp = z0 + V < A.d0, zm = bz > 0, yp = by + 1 < A.nt1, ym = by > 0,
               xp = bx + 1 < A.nt2, xm = bx > 0;
    VecG *const own = sT + cell;
    const VecG *const t2 = sT + (x < b2 - 1 ? cell + 1 : nc + b2 + y);  // residual at +axis 2
    const VecG *const m1p =                                             // h1 at -axis 1
        sT + kTile + (!inv ? kCells - 1 : y > 0 ? cell - b2 : nc + x);
    const VecG *const m2p =                                             // h2 at -axis 2
        sT + (!inv ? kTile + kCells - 1 : x > 0 ? 2 * kTile + cell - 1 : kTile + nc + b2 + y);

    const unsigned st0 = unsigned(A.d1) * unsigned(A.d2);
    const float inv_b2 = 1.f / float(b2);
    // words between bricks: byte offsets of this brick's inbox and of its parts
    const int Wy = A.nt1 > 1 ? V * b2 : 0, Wx = A.nt2 > 1 ? V * b1 : 0, W = Wy + Wx;
    const unsigned IB = 16u * unsigned(nc + W), box = b * IB, nc8 = 8u * unsigned(nc);
    const unsigned boxT = box + 2u * nc8, boxH = boxT + 8u * unsigned(W);
    const unsigned dz = unsigned(A.nt1 * A.nt2) * IB, dy = unsigned(A.nt2) * IB;
    const unsigned t8 = 8u * unsigned(t);
    const unsigned NT8 = 8u * unsigned(NT);
    // faces this thread sends: residuals of the first plane, row and column,
    // h0 of the last plane, h1 of the last row, h2 of the last column; the
    // waves that send whole rows run first in their phase
    const bool oTz = inv && zm, oTy = inv && y == 0 && ym, oTx = inv && x == 0 && xm;
    const bool oHz = inv && zp, oHy = inv && y == b1 - 1 && yp, oHx = inv && x == b2 - 1 && xp;
    const bool firstT = __any(oTy), firstH = __any(oHy);
    // in-plane words this thread receives (words t, t + NT, .. of the brick's)
    // and the LDS floats they go to, in the residual's tile or h1's
    constexpr int R = kWords;
    int d[R];
    bool rT[R], rH[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int w = t + r * NT;
        const bool isy = w < Wy;
        const int div = isy ? b2 : b1, v = isy ? w : w - Wy, k = v / div, i = v - k * div;
        const bool in = w < W && k < nz && (isy ? bx * b2 + i < A.d2 : by * b1 + i < A.d1);
        d[r] = ((k / G) * kCells + nc + (isy ? 0 : b2) + i) * G + k % G;
        rT[r] = in && (isy ? yp : xp);
        rH[r] = in && (isy ? ym : xm);
    }

    // the faces that have no neighbour, and the zero cells, stay zero
    for (int i = t; i < lds_bytes(V, MODE) / 4; i += NT) fT[i] = 0.f;
    lds_barrier();

    // Receives this thread's words: one load of each as its phase ends, then
    // all of them again until none is missing. (The first load half a phase
    // earlier mostly came too early: 14 % slower at 128^3.) The axis-0 neighbour's value is returned, the in-plane ones go to
    // `tile`.
    Word first[R + 1];
    auto look = [&](unsigned zoff, bool rz, unsigned off, const bool (&rv)[R]) {
        const unsigned o = here(t8);
        first[R] = 0;
        if (rz) first[R] = ld_word(word_at(A.inbox, o + zoff));
#pragma unroll
        for (int r = 0; r < R; ++r) {
            first[r] = 0;
            if (rv[r]) first[r] = ld_word(word_at(A.inbox, o + (off + unsigned(r) * NT8)));
        }
    };
    auto receive = [&](unsigned zoff, bool rz, unsigned off, const bool (&rv)[R], float *tile,
                       unsigned tag) {
        for (int spin = 0;; ++spin) {
            bool missing = rz && unsigned(first[R] >> 32) != tag;
#pragma unroll
            for (int r = 0; r < R; ++r) missing |= rv[r] && unsigned(first[r] >> 32) != tag;
            if (!missing || give_up(spin, A.abort, fail)) break;
            look(zoff, rz, off, rv);
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (rv[r]) tile[d[r]] = __builtin_bit_cast(float, unsigned(first[r]));
        return rz ? __builtin_bit_cast(float, unsigned(first[R])) : 0.f;
    };
    // the row (exact: t < 1024) of this thread's position
    auto row_of = [&](unsigned tt) { return unsigned((float(tt) + 0.5f) * inv_b2); };
    // sends planes [g G, g G + G) of the first or last row (word i of a plane is
    // column i: the senders are consecutive threads) or column (word i: row i)
    auto send_row = [&](bool mine, unsigned off, int g, const float (&v)[G], unsigned tag) {
        if (!mine) return;
        const unsigned o = here(t8) + off;
#pragma unroll
        for (int j = 0; j < G; ++j)
            if (g * G + j < here_s(nz))
                st_word(word_at(A.inbox, o + unsigned(here_s(8 * b2) * (g * G + j))), tag, v[j]);
    };
    auto send_col = [&](bool mine, unsigned off, int g, const float (&v)[G], unsigned tag) {
        if (!mine) return;
        const unsigned o = 8u * row_of(here(t8) >> 3) + off;
#pragma unroll
        for (int j = 0; j < G; ++j)
            if (g * G + j < here_s(nz))
                st_word(word_at(A.inbox, o + unsigned(here_s(8 * b1) * (g * G + j))), tag, v[j]);
    };
    // element index of this thread's first voxel (inside the volume only)
    auto index0 = [&]() {
        const unsigned tt = here(t8) >> 3, yy = row_of(tt), xx = tt - yy * unsigned(b2);
        return unsigned(z0) * st0 + (unsigned(by * b1) + yy) * unsigned(A.d2) + unsigned(bx * b2) + xx;
    };

    unsigned tag = 1;
    int nparts = 0;
    for (int q = slot; q < A.nsolves; q += A.nslots) {
        float h0[V], h1[V], h2[V], pt[V], u[V], al[V], cs[V], ct[V], fr[V][NF];
        unsigned lab = 0;
        {
            const mh::OnchipSolve S = A.solves[q];
#pragma unroll
            for (int k = 0; k < V; ++k) {
                h0[k] = h1[k] = h2[k] = 0.f;
                pt[k] = u[k] = al[k] = cs[k] = ct[k] = 0.f;
#pragma unroll
                for (int f = 0; f < NF; ++f) fr[k][f] = 0.f;
                if (MODE == kPointwise) fr[k][4] = fr[k][5] = fr[k][6] = 1.f;
                if (inv && k < nz) {
                    const unsigned i = index0() + unsigned(k) * st0;
                    u[k] = S.u[i];
                    cs[k] = A.F.cs[i];
                    ct[k] = A.F.ct[i];
                    al[k] = S.alpha[i];
                    const float *e = A.F.eigs + (MODE == kPointwise ? 6u * i + 3u : 3u * i);
                    const mh::Quat qq = mh::expand_squeezed(e[0], e[1], e[2]);
                    if constexpr (MODE == kAxial) {
                        mh::frame_axis(make_float4(qq.w, qq.x, qq.y, qq.z), fr[k][0], fr[k][1], fr[k][2]);
                    } else {
                        fr[k][0] = qq.w;
                        fr[k][1] = qq.x;
                        fr[k][2] = qq.y;
                        fr[k][3] = qq.z;
                    }
                    if constexpr (MODE == kPointwise) {
                        fr[k][4] = e[-3];
                        fr[k][5] = e[-2];
                        fr[k][6] = e[-1];
                    }
                    if (SUP) lab |= unsigned(A.F.labels[i] & 3) << (2 * k);
                    pt[k] = fminf(cs[k], ct[k]);
                }
            }
        }
        // the first residuals
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            VecG T;
#pragma unroll
            for (int j = 0; j < G; ++j) T.v[j] = inv && g * G + j < nz ? -(u[g * G + j] * A.rcc) : 0.f;
            if (g == 0 && oTz) st_word(word_at(A.inbox, here(t8) + (box - dz)), tag, T.v[0]);
            send_row(oTy, boxT - dy, g, T.v, tag);
            send_col(oTx, boxT - IB + 8u * unsigned(Wy), g, T.v, tag);
            if (live) own[g * kCells] = T;
            if (kCapLds && live) {
#pragma unroll
                for (int j = 0; j < G; ++j) T.v[j] = cs[g * G + j];
                own[3 * kTile + g * kMaxThreads] = T;
                if (g == NG - 1) {
#pragma unroll
                    for (int j = 0; j < G; ++j) T.v[j] = ct[g * G + j];
                    own[3 * kTile + NG * kMaxThreads] = T;
                }
            }
        }
        look(box, oHz, boxT, rT);

        // The criterion: the waves' sums, then (thread 0) the brick's sum to
        // everyone, then every brick's sum, added in the same order by every
        // work-group, so that all of them take the same decision. The p-step
        // leaves u as it is, so the decision may wait for the next u-step.
        int stop = 0, ncrit = 0;
        bool pending = false;
        Word *set = nullptr;
        unsigned ptag = 0;
        auto sum16 = [&](const float *v) {  // zero beyond the work-group's waves
            const Vec<4> *w = reinterpret_cast<const Vec<4> *>(v);
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const Vec<4> a = w[k];
                s += (a.v[0] + a.v[1]) + (a.v[2] + a.v[3]);
            }
            return s;
        };
        auto crit_send = [&]() {
            if (per > 1 && here(t8) == 0) st_word(set + lb, ptag, sum16(red + 16 * (nparts & 1)));
        };
        auto crit_receive = [&]() {
            if (per == 1) return;
            float s = 0.f;
            const int tt = int(here(t8) >> 3);
            for (int w = tt; w < per; w += NT) {
                Word v = ld_word(set + w);
                for (int spin = 0; unsigned(v >> 32) != ptag; ++spin) {
                    if (give_up(spin, A.abort, fail)) break;
                    v = ld_word(set + w);
                }
                s += __builtin_bit_cast(float, unsigned(v));
            }
            s = mh::wave_reduce<SumOp>(s);
            if ((tt & 63) == 0) red[32 + (tt >> 6)] = s;
        };
        auto crit_decide = [&]() {
            // (the same in every lane: held and branched on as a scalar)
            const float s = sum16(red + (per > 1 ? 32 : 16 * (nparts & 1))) * A.inv_n_rcc;
            const float crit = __builtin_bit_cast(
                float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, s)));
            if (lb == 0 && here(t8) == 0) {
                const mh::OnchipSolve &S = A.solves[here_s(q)];
                if (ncrit < S.crit_max) S.crit_log[ncrit] = crit;
            }
            ++ncrit;
            pending = false;
            stop = crit != crit ? 1 : crit < A.error_bound ? 2 : 0;
        };
        auto crit_settle = [&]() {
            lds_barrier();
            crit_send();
            crit_receive();
            lds_barrier();
            crit_decide();
        };
        for (int it = 0; it < A.num_iter; ++it) {
            float zin = receive(box, oHz, boxT, rT, fT, tag);
            lds_barrier();
            if (DEFER && pending) crit_send();
            // p-step
            if (firstH) __builtin_amdgcn_s_setprio(2);
#pragma unroll
            for (int g = NG - 1; g >= 0; --g) {
                const VecG To = own[g * kCells], T1 = own[g * kCells + b2], T2 = t2[g * kCells];
                VecG w1, w2;
#pragma unroll
                for (int j = G - 1; j >= 0; --j) {
                    const int k = g * G + j;
                    const float tn = j < G - 1 ? To.v[j < G - 1 ? j + 1 : j] : zin;
                    const float g0 = k < here_s(last0) ? (tn - To.v[j]) * A.ss0 : 0.f;
                    const float g1 = e1 ? (T1.v[j] - To.v[j]) * A.ss1 : 0.f;
                    const float g2 = e2 ? (T2.v[j] - To.v[j]) * A.ss2 : 0.f;
                    if constexpr (MODE == kAxial) {
                        mh::cmf_p_voxel_axi(h0[k], h1[k], h2[k], g0, g1, g2, fr[k][0], fr[k][1],
                                            fr[k][2], A.A, al[k]);
                    } else {
                        const mh::Mat3 M =
                            mh::quat_to_mat(mh::Quat{fr[k][0], fr[k][1], fr[k][2], fr[k][3]});
                        if constexpr (MODE == kConst)
                            mh::cmf_p_voxel_m(h0[k], h1[k], h2[k], g0, g1, g2, M, A.sq0, A.sq1, A.sq2,
                                              A.rq0, A.rq1, A.rq2, al[k]);
                        else
                            mh::cmf_p_voxel_m(h0[k], h1[k], h2[k], g0, g1, g2, M, fr[k][4], fr[k][5],
                                              fr[k][6], 1.f / fr[k][4], 1.f / fr[k][5],
                                              1.f / fr[k][6], al[k]);
                    }
                    w1.v[j] = h1[k];
                    w2.v[j] = h2[k];
                    if (k == V - 1 && oHz)
                        st_word(word_at(A.inbox, here(t8) + (box + dz + nc8)), tag, h0[k]);
                }
                zin = To.v[0];
                send_row(oHy, boxH + dy - 8u * unsigned(nc - b2), g, w1.v, tag);
                send_col(oHx, boxH + IB + 8u * unsigned(Wy), g, w2.v, tag);
                if (live) {
                    own[kTile + g * kCells] = w1;
                    own[2 * kTile + g * kCells] = w2;
                }
            }
            look(box + nc8, oTz, boxH, rH);
            if (firstH) __builtin_amdgcn_s_setprio(0);
            float below = receive(box + nc8, oTz, boxH, rH, fT + kTile * G, tag);
            if (DEFER && pending) crit_receive();
            lds_barrier();
            // A launch that was given up ends here, not after num_iter iterations of
            // waits that each take 16 loads. (Not where the look costs time: with
            // eigenvalues at every voxel 3 to 8 %, 96 x 100 x 100 4.55 -> 4.97 us an
            // iteration, with volumes side by side 1 to 2 %; axial 128^3 4.65 -> 4.57.)
            if (MODE != kPointwise && N == 1 && (it & 63) == 63 && *fail) break;
            if (DEFER && pending) {
                crit_decide();
                if (stop) break;
            }
            // u-step
            ++tag;
            if (firstT) __builtin_amdgcn_s_setprio(2);
            const bool more = it + 1 < A.num_iter;
            float aerr = 0.f;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const VecG m1 = m1p[g * kCells], m2 = m2p[g * kCells];
                VecG T, C, E;
                if (kCapLds) C = own[3 * kTile + g * kMaxThreads];
                if (kCapLds && g == NG - 1) E = own[3 * kTile + NG * kMaxThreads];
#pragma unroll
                for (int j = 0; j < G; ++j) {
                    const int k = g * G + j;
                    const float own0 = k < here_s(last0) ? h0[k] : 0.f;
                    const float x0 = own0 - below;
                    const float x1 = (e1 ? h1[k] : 0.f) - m1.v[j];
                    const float x2 = (e2 ? h2[k] : 0.f) - m2.v[j];
                    below = own0;
                    const float div = mh::cmf_div(x0, x1, x2, A.rs0, A.rs1, A.rs2);
                    float ub = 1.f, uf = 0.f;
                    if (SUP) {
                        const unsigned l = here(lab) >> (2 * k);
                        uf = float(l & 1u);
                        ub = (l & 2u) ? 0.f : 1.f;
                    }
                    const float err = mh::cmf_u_voxel(div, pt[k], u[k], T.v[j], kCapLds ? C.v[j] : cs[k],
                                                      kCapLds && g == NG - 1 ? E.v[j] : ct[k], A.rcc,
                                                      A.inv_rcc, ub, uf);
                    aerr += fabsf(err);
                    if (k == 0 && more && oTz)
                        st_word(word_at(A.inbox, here(t8) + (box - dz)), tag, T.v[0]);
                }
                send_row(oTy && more, boxT - dy, g, T.v, tag);
                send_col(oTx && more, boxT - IB + 8u * unsigned(Wy), g, T.v, tag);
                if (live) own[g * kCells] = T;
            }
            if (more) look(box, oHz, boxT, rT);
            if (firstT) __builtin_amdgcn_s_setprio(0);
            if (it % A.update == 0) {
                ++nparts;
                set = A.parts + (int64_t(slot) * 2 + (nparts & 1)) * per;
                ptag = tag;
                aerr = mh::wave_reduce<SumOp>(inv ? aerr : 0.f);
                const int tt = int(here(t8) >> 3);
                if ((tt & 63) == 0) red[16 * (nparts & 1) + (tt >> 6)] = aerr;
                pending = true;
                if (!DEFER) {
                    crit_settle();
                    if (stop) break;
                }
            }
        }
        if (DEFER && pending) crit_settle();
        ++tag;
        // read before the barrier (every wait of this solve is behind an earlier one):
        // after it, a wave ahead may give up in the next solve
        const int failed = *fail;
        lds_barrier();
        if (failed) return;
        const mh::OnchipSolve &S = A.solves[here_s(q)];
        if (inv) {
            float *out = S.u;
            const unsigned i = index0();
#pragma unroll
            for (int k = 0; k < V; ++k)
                if (k < nz) out[i + unsigned(k) * st0] = u[k];
        }
        if (t == 0) {
            if (lb == 0) {
                *S.stop = stop;
                *S.ncrit = ncrit;
            }
            atomicAdd(S.done, 1);
        }
    }
}

// A few solves reach the device as an argument: a transfer of their table costs
// the host 10 us.
constexpr int kFew = 16;
struct Few {
    mh::OnchipSolve s[kFew];
};

// The inbox and criterion words, the abort and done words to zero; u of every
// solve kept in `keep`; the table of a few solves.
__global__ void __launch_bounds__(mh::kBlock)
onchip_prepare_kernel(Word *words, int64_t nwords, mh::OnchipSolve *table, const Few few, int nsolves,
                      int64_t n, float *keep, int *abort)
{
    const mh::OnchipSolve *solves = nsolves <= kFew ? few.s : table;
    const int64_t step = int64_t(gridDim.x) * blockDim.x;
    const int64_t i0 = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (int64_t i = i0; i < nwords; i += step) words[i] = 0;
    for (int q = 0; q < nsolves; ++q) {
        const float *u = solves[q].u;
        for (int64_t i = i0; i < n; i += step) keep[q * n + i] = u[i];
    }
    if (i0 < nsolves) {
        *solves[i0].done = 0;
        if (nsolves <= kFew) table[i0] = solves[i0];
    }
    if (i0 == 0) *abort = 0;
}

__global__ void __launch_bounds__(mh::kBlock)
onchip_restore_kernel(float *__restrict__ u, const float *__restrict__ keep, int64_t n)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) u[i] = keep[i];
}

int64_t align256(int64_t b) { return (b + 255) & ~int64_t(255); }

int mode_of(const mh_cmf_params *p)
{
    return !p->const_evals ? kPointwise : mh::axi_params(p).on ? kAxial : kConst;
}

int words_of(const mh::OnchipPlan &P)  // in-plane face words of a brick
{
    return (P.nt1 > 1 ? P.v * P.b2 : 0) + (P.nt2 > 1 ? P.v * P.b1 : 0);
}

int threads_of(const mh::OnchipPlan &P) { return (P.b1 * P.b2 + 63) / 64 * 64; }

template <int V, int MODE, bool DEFER>
const void *kernel_sup(bool sup)
{
    return sup ? reinterpret_cast<const void *>(&cmf_onchip_kernel<V, MODE, true, DEFER>)
               : reinterpret_cast<const void *>(&cmf_onchip_kernel<V, MODE, false, DEFER>);
}

// The kernel of a brick of v planes. The criterion is settled during the next
// iteration's p-step, except where that costs registers that are not there and
// a criterion is rare (8 planes, 128^3: 4.6 us per iteration with a criterion
// every 30, 6 % more in the p-step; with one every iteration 6.0 in the p-step, 47 %
// more out of it).
const void *kernel_of(int v, int mode, bool sup, int update)
{
    const bool rare = update >= 8;
    switch (mode * 16 + v) {
    case kAxial * 16 + 1: return kernel_sup<1, kAxial, true>(sup);
    case kAxial * 16 + 2: return kernel_sup<2, kAxial, true>(sup);
    case kAxial * 16 + 4: return kernel_sup<4, kAxial, true>(sup);
    case kAxial * 16 + 8:
        return rare ? kernel_sup<8, kAxial, false>(sup) : kernel_sup<8, kAxial, true>(sup);
    case kConst * 16 + 1: return kernel_sup<1, kConst, true>(sup);
    case kConst * 16 + 2: return kernel_sup<2, kConst, true>(sup);
    case kConst * 16 + 4: return kernel_sup<4, kConst, true>(sup);
    case kPointwise * 16 + 1: return kernel_sup<1, kPointwise, true>(sup);
    case kPointwise * 16 + 2: return kernel_sup<2, kPointwise, true>(sup);
    case kPointwise * 16 + 4:
        return rare ? kernel_sup<4, kPointwise, false>(sup) : kernel_sup<4, kPointwise, true>(sup);
    default: return nullptr;
    }
}

bool plan_fits(const mh::OnchipPlan &P)
{
    const int nc = P.b1 * P.b2;
    return nc <= kMaxThreads && words_of(P) <= kWords * threads_of(P) && nc + P.b1 + P.b2 + 1 <= kCells;
}

// Microseconds of an iteration, fitted to plans as an earlier, up to 7 % slower form
// of the kernel ran them (8 planes of 8 x 128 voxels per brick 4.9, now 4.6; of 8 x 64
// 3.4; 4 of 10 x 96 3.7, of 8 x 64 2.6; 2 of 8 x 64 2.6; 1 of 10 x 37 2.3, of 16 x 64
// 3.4; bricks split along axis 2: 8 of 16 x 64 6.3, 4 of 32 x 32 4.8), whose order is
// what the choice goes by: the two exchanges, the issue of a SIMD's waves
// plane by plane (one wave alone does not hide its own latencies), the axis-0
// words where little work covers them, and along a split axis 2 the words every
// wave sends last.
double iteration_us(const mh::OnchipPlan &P)
{
    if (P.blocks() == 1) return 0.8 + 0.1 * P.v * ((threads_of(P) + 255) / 256);
    const int waves = (threads_of(P) + 255) / 256;
    return 2.0 + 0.09 * P.v * (waves == 1 && P.v > 1 ? 3 : waves) +
           (P.v < 4 ? 0.6 * P.b1 * P.b2 / 1024.0 : 0.0) + (P.nt2 > 1 ? 0.22 * P.v : 0.0);
}

std::mutex g_device_mu[kMaxDevices];

}  // namespace

namespace mh {

std::mutex &device_lock(int device) { return g_device_mu[device]; }

int compute_units(mh_ctx *ctx)
{
    int cus = 0;
    if (ctx->chip_units > 0) return ctx->chip_units;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess) {
        (void)hipGetLastError();
        cus = 0;
    }
    return cus;
}

OnchipPlan onchip_plan(mh_ctx *ctx, const int dims[3], const mh_cmf_params *prm, int solves)
{
    OnchipPlan best;
    const std::array<int, 5> key{dims[0], dims[1], dims[2], mode_of(prm), solves};
    const auto f = ctx->onchip_plans.find(key);
    if (f != ctx->onchip_plans.end()) {
        const auto &c = f->second;
        best.v = c[0], best.b1 = c[1], best.b2 = c[2], best.nt1 = c[3], best.nt2 = c[4], best.nz = c[5];
        return best;
    }
    const int cus = ctx->device < kMaxDevices ? compute_units(ctx) : 0;
    if (cus <= 0) return best;
    const int vmax = mode_of(prm) == kAxial ? kMaxPlanes : kMaxPlanes / 2;
    double best_cost = 0;
    for (int v = 1; v <= vmax; v *= 2) {
        const int nz = (dims[0] + v - 1) / v;
        if (nz > cus) continue;
        for (int n2 = 1; n2 <= std::min(dims[2], 16); ++n2) {
            const int b2 = (dims[2] + n2 - 1) / n2;
            if (b2 > kMaxThreads) continue;
            const int least = (dims[1] + kMaxThreads / b2 - 1) / (kMaxThreads / b2);
            for (int n1 = least; n1 <= std::min(dims[1], least + 16); ++n1) {
                OnchipPlan P;
                P.v = v;
                P.b1 = (dims[1] + n1 - 1) / n1;
                P.b2 = b2;
                P.nt1 = (dims[1] + P.b1 - 1) / P.b1;
                P.nt2 = (dims[2] + b2 - 1) / b2;
                P.nz = nz;
                if (P.blocks() > cus || !plan_fits(P)) continue;
                const int rounds = (solves + cus / P.blocks() - 1) / (cus / P.blocks());
                const double cost = iteration_us(P) * rounds;
                if (best.v == 0 || cost < best_cost) {
                    best = P;
                    best_cost = cost;
                }
            }
        }
    }
    if (ctx->onchip_plans.size() >= 4096) ctx->onchip_plans.clear();  // (formed again in microseconds)
    ctx->onchip_plans[key] = {best.v, best.b1, best.b2, best.nt1, best.nt2, best.nz};
    return best;
}

namespace {
int slots_of(const OnchipPlan &P, int solves, int cus) { return std::min(solves, cus / P.blocks()); }
int64_t nwords_of(const OnchipPlan &P, int slots)
{
    return int64_t(slots) * P.blocks() * (2 * (P.b1 * P.b2 + words_of(P)) + 2);
}
// work-groups launched of so many: all, but for mh_cmf_set_lost_group
unsigned launched(mh_ctx *ctx, int blocks)
{
    return unsigned(ctx->lost_group == 0 ? std::max(1, blocks - 1) : blocks);
}
Args args_of(const OnchipPlan &P, const OnchipFields &F, const int dims[3], const mh_cmf_params *prm)
{
    Args A{};
    A.F = F;
    A.d0 = dims[0];
    A.d1 = dims[1];
    A.d2 = dims[2];
    A.b1 = P.b1;
    A.b2 = P.b2;
    A.nt1 = P.nt1;
    A.nt2 = P.nt2;
    A.nz = P.nz;
    A.num_iter = prm->num_iter;
    A.update = prm->update;
    A.rcc = prm->rcc;
    A.inv_rcc = float(1.0 / double(prm->rcc));
    A.rs0 = prm->rs[0];
    A.rs1 = prm->rs[1];
    A.rs2 = prm->rs[2];
    A.ss0 = prm->ss[0];
    A.ss1 = prm->ss[1];
    A.ss2 = prm->ss[2];
    A.error_bound = prm->error_bound;
    A.inv_n_rcc = float(1.0 / (double(int64_t(dims[0]) * dims[1] * dims[2]) * double(prm->rcc)));
    A.sq0 = prm->sqev[0];
    A.sq1 = prm->sqev[1];
    A.sq2 = prm->sqev[2];
    A.rq0 = float(1.0 / double(prm->sqev[0]));
    A.rq1 = float(1.0 / double(prm->sqev[1]));
    A.rq2 = float(1.0 / double(prm->sqev[2]));
    A.A = axi_params(prm);
    return A;
}
}  // namespace

OnchipPlan onchip_plan_many(mh_ctx *ctx, const int dims[3], const mh_cmf_params *prm)
{
    OnchipPlan best;
    const int cus = ctx->device < kMaxDevices ? compute_units(ctx) : 0;
    double best_cost = 0;
    if (mode_of(prm) != kAxial) return best;
    for (int n2 = 1; n2 <= std::min(dims[2], 16); ++n2) {
        const int b2 = (dims[2] + n2 - 1) / n2;
        if (b2 > kMaxThreads) continue;
        const int least = (dims[1] + kMaxThreads / b2 - 1) / (kMaxThreads / b2);
        for (int n1 = least; n1 <= std::min(dims[1], least + 4); ++n1) {
            OnchipPlan P;
            P.v = kMaxPlanes;
            P.b1 = (dims[1] + n1 - 1) / n1;
            P.b2 = b2;
            P.nt1 = (dims[1] + P.b1 - 1) / P.b1;
            P.nt2 = (dims[2] + b2 - 1) / b2;
            P.nz = (dims[0] + P.v - 1) / P.v;
            const double cost = iteration_us(P) * P.blocks();
            if (P.blocks() <= cus && plan_fits(P) && (best.v == 0 || cost < best_cost)) {
                best = P;
                best_cost = cost;
            }
        }
    }
    return best;
}

int onchip_run_many(mh_ctx *ctx, const OnchipVolume *vols, int nvol, const mh_cmf_params *prm,
                    void *work, int64_t work_bytes, void *heads, hipStream_t s, std::vector<char> *host,
                    bool *ran)
{
    *ran = false;
    const int cus = compute_units(ctx);
    ArgsOf<kMany> L{};
    int64_t words = 0, kept = 0, head_bytes = 0;
    int threads = 64;
    for (int v = 0; v < nvol; ++v) {
        const OnchipVolume &V = vols[v];
        L.first[v + 1] = L.first[v] + V.plan.blocks();
        words += align256(sizeof(Word) * nwords_of(V.plan, 1));
        kept += align256(sizeof(float) * int64_t(V.dims[0]) * V.dims[1] * V.dims[2]);
        threads = std::max(threads, threads_of(V.plan));
        head_bytes += V.head_bytes;
    }
    const int64_t table_bytes = align256(sizeof(OnchipSolve) * kMany);
    if (nvol < 1 || nvol > kMany || L.first[nvol] > cus || prm->num_iter < 1 ||
        prm->num_iter >= INT_MAX / 2 || work_bytes < words + table_bytes + 256 + kept)
        return MH_OK;
    std::unique_lock<std::mutex> lock(device_lock(ctx->device), std::try_to_lock);
    if (!lock.owns_lock()) return MH_OK;
    L.n = nvol;
    char *base = static_cast<char *>(work);
    OnchipSolve *table = reinterpret_cast<OnchipSolve *>(base);
    int *abort = reinterpret_cast<int *>(base + table_bytes);
    base += table_bytes + 256;
    char *keep = base + words;
    for (int v = 0; v < nvol; ++v) {
        const OnchipVolume &V = vols[v];
        const int64_t n = int64_t(V.dims[0]) * V.dims[1] * V.dims[2], nwords = nwords_of(V.plan, 1);
        Args &A = L.a[v];
        A = args_of(V.plan, V.F, V.dims, prm);
        A.inbox = reinterpret_cast<Word *>(base);
        A.parts = A.inbox + nwords - int64_t(V.plan.blocks()) * 2;
        base += align256(sizeof(Word) * nwords);
        A.abort = abort;
        A.solves = table + v;
        A.nsolves = A.nslots = 1;
        Few few{};
        few.s[0] = V.solve;
        hipLaunchKernelGGL(onchip_prepare_kernel,
                           dim3(unsigned(std::min<int64_t>(1024, blocks_for(std::max(n, nwords))))),
                           dim3(kBlock), 0, s, A.inbox, nwords, table + v, few, 1, n,
                           reinterpret_cast<float *>(keep), abort);
        keep += align256(sizeof(float) * n);
    }
    MH_CHECK_LAUNCH(ctx, "onchip prepare");
    const void *kernel = reinterpret_cast<const void *>(&cmf_onchip_kernel<8, kAxial, false, false, kMany>);
    const int lds = lds_bytes(8, kAxial);
    void *args[] = {&L};
    MH_CHECK(ctx, hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    const hipError_t e = hipLaunchCooperativeKernel(kernel, dim3(launched(ctx, L.first[nvol])),
                                                    dim3(unsigned(threads)), args, unsigned(lds), s);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        ++ctx->chip.refused;
        return MH_OK;
    }
    host->resize(size_t(head_bytes));
    MH_CHECK(ctx, hipMemcpyAsync(host->data(), heads, size_t(head_bytes), hipMemcpyDeviceToHost, s));
    MH_CHECK(ctx, hipStreamSynchronize(s));
    *ran = true;
    for (int v = 0; v < nvol; ++v) {
        const OnchipVolume &V = vols[v];
        const int done = *reinterpret_cast<const int *>(host->data() + (reinterpret_cast<char *>(V.solve.done) -
                                                                        static_cast<char *>(heads)));
        *ran = *ran && done == V.plan.blocks();
    }
    if (*ran) {
        ctx->chip.solves += nvol;
        return MH_OK;
    }
    // a work-group gave up: every volume as it was
    ++ctx->chip.given_up;
    keep = base;
    for (int v = 0; v < nvol; ++v) {
        const int64_t n = int64_t(vols[v].dims[0]) * vols[v].dims[1] * vols[v].dims[2];
        hipLaunchKernelGGL(onchip_restore_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, s, vols[v].solve.u,
                           reinterpret_cast<const float *>(keep), n);
        MH_CHECK_LAUNCH(ctx, "onchip restore");
        keep += align256(sizeof(float) * n);
    }
    return MH_OK;
}

int64_t onchip_work_bytes(const OnchipPlan &P, int solves, int cus)
{
    if (P.v == 0) return 0;
    return align256(sizeof(Word) * nwords_of(P, slots_of(P, solves, cus))) +
           align256(sizeof(OnchipSolve) * int64_t(solves)) + 256;
}

int onchip_run(mh_ctx *ctx, const OnchipPlan &P, const OnchipSolve *solves, int nsolves,
               const OnchipFields &F, const int dims[3], const mh_cmf_params *prm, void *work,
               int64_t work_bytes, hipStream_t s, bool *ran, std::vector<int> *finished, void *head,
               size_t head_bytes)
{
    *ran = false;
    if (finished) finished->clear();
    const int64_t n = int64_t(dims[0]) * dims[1] * dims[2];
    const int cus = compute_units(ctx), mode = mode_of(prm);
    if (P.v == 0 || cus <= 0 || prm->num_iter < 1) return MH_OK;
    if (int64_t(nsolves) * (int64_t(prm->num_iter) + 1) > INT_MAX / 2) return MH_OK;  // tags
    const int64_t fixed = onchip_work_bytes(P, nsolves, cus);
    if (work_bytes < fixed + int64_t(sizeof(float)) * n * nsolves) return MH_OK;
    const void *kernel = kernel_of(P.v, mode, F.labels != nullptr, prm->update);
    if (!kernel) return MH_OK;
    std::unique_lock<std::mutex> lock(device_lock(ctx->device), std::try_to_lock);
    if (!lock.owns_lock()) return MH_OK;

    const int slots = slots_of(P, nsolves, cus), lds = lds_bytes(P.v, mode);
    const int64_t nwords = nwords_of(P, slots);
    char *base = static_cast<char *>(work);
    ArgsOf<1> L{};
    Args &A = L.a[0];
    A = args_of(P, F, dims, prm);
    A.inbox = reinterpret_cast<Word *>(base);
    A.parts = A.inbox + nwords - int64_t(slots) * P.blocks() * 2;
    base += align256(sizeof(Word) * nwords);
    OnchipSolve *table = reinterpret_cast<OnchipSolve *>(base);
    base += align256(sizeof(OnchipSolve) * int64_t(nsolves));
    A.abort = reinterpret_cast<int *>(base);
    float *keep = reinterpret_cast<float *>(base + 256);
    A.solves = table;
    A.nsolves = nsolves;
    A.nslots = slots;
    Few few{};
    if (nsolves <= kFew)
        std::copy(solves, solves + nsolves, few.s);
    else
        MH_CHECK(ctx, hipMemcpyAsync(table, solves, sizeof(OnchipSolve) * size_t(nsolves),
                                     hipMemcpyHostToDevice, s));
    const unsigned pb = unsigned(std::min<int64_t>(1024, blocks_for(std::max(n, nwords))));
    hipLaunchKernelGGL(onchip_prepare_kernel, dim3(std::max(pb, blocks_for(nsolves))), dim3(kBlock), 0,
                       s, A.inbox, nwords, table, few, nsolves, n, keep, A.abort);
    MH_CHECK_LAUNCH(ctx, "onchip prepare");
    void *args[] = {&L};
    MH_CHECK(ctx, hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    const hipError_t e = hipLaunchCooperativeKernel(kernel, dim3(launched(ctx, slots * P.blocks())),
                                                    dim3(unsigned(threads_of(P))), args,
                                                    unsigned(lds), s);
    if (e != hipSuccess) {  // the device does not hold every work-group: nothing ran
        (void)hipGetLastError();
        ++ctx->chip.refused;
        return MH_OK;
    }
    // every solve's done word counts the bricks that stored u
    std::vector<int> done(static_cast<size_t>(nsolves), 0);
    if (head)
        MH_CHECK(ctx, hipMemcpyAsync(head, solves[0].stop, head_bytes, hipMemcpyDeviceToHost, s));
    else
        for (int q = 0; q < nsolves; ++q)
            MH_CHECK(ctx, hipMemcpyAsync(&done[size_t(q)], solves[q].done, sizeof(int),
                                         hipMemcpyDeviceToHost, s));
    MH_CHECK(ctx, hipStreamSynchronize(s));
    if (head) done[0] = static_cast<const int *>(head)[solves[0].done - solves[0].stop];
    *ran = true;
    for (int q = 0; q < nsolves; ++q) {
        done[size_t(q)] = done[size_t(q)] == P.blocks();
        ctx->chip.solves += done[size_t(q)];
        if (done[size_t(q)]) continue;
        *ran = false;
        hipLaunchKernelGGL(onchip_restore_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, s, solves[q].u,
                           keep + q * n, n);
        MH_CHECK_LAUNCH(ctx, "onchip restore");
    }
    ctx->chip.given_up += !*ran;
    if (finished) finished->swap(done);
    return MH_OK;
}

}  // namespace mh
