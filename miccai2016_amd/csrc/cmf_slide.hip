// Max-flow passes of many iterations over a volume larger than the chip.
//
// A window of W = 8 slots planes (axis 0) is resident, cut into tiles of b1 x b2
// voxels: a work-group per tile and run of 8 planes, a thread per in-plane
// position holding its 8 planes in registers, as in cmf_onchip.hip. The window
// slides: at step s the planes k = s - 2 l, l = 1 .. levels, advance from
// iteration l - 1 to l of the pass, so that plane k + 1 is always one iteration
// behind plane k and one step old. Every second plane of the window is active,
// plane s is new and plane s - 2 levels leaves. A pass of L levels over D0 planes
// takes D0 + 2 L steps, reads and writes the state once, and recomputes
// nothing: the in-plane faces of neighbouring tiles and the axis-0 faces between
// runs of planes (one run's with itself) travel as tagged words (cmf_words.h).
//
// Step s, all planes of parity s:
//   barrier; p-step: residuals of the plane and the next one (LDS; the run's
//     last plane: a word of step s - 1), h1 of the last row and h2 of the last
//     column to the next tiles, h0 of the run's last plane to the next run;
//   barrier; receive: h1, h2 of the previous tiles (this step's), the residuals
//     of the next tiles that step s + 1 needs (step s - 1's), h0 of the previous
//     run's last plane (step s - 1's). In-plane words go to the thread that reads
//     them, so only the waves of an outer row or column wait (for h1 and h2, half
//     a step after they were sent) while the others compute;
//   planes that come are loaded, then the u-step: residuals of the first row,
//     column and plane to the previous tiles and run; a plane that reached the
//     pass's last level is stored.
// Words keep one slot per plane of the run: a slot's next word is formed from
// values that its reader sent after reading.
//
// Loads, stores and polls of a wave complete in order, so a poll waits for the
// plane that is on its way as well; loads are issued right after one poll, most
// of a step before the next. Measured at 256^3 (tiles 4 x 256, 4 slots, 15
// levels: 286 steps of 3.99 us, 76 us an iteration; the 4-level sweep 138 us):
// arithmetic 1.9 us of a step, sends 0.25, polls 0.75, loads 0.75 and stores 0.4
// (each step's plane is loaded and stored by a quarter of the work-groups).
//
// The per-voxel arithmetic is cmf_voxel.h's, so the result equals the
// per-iteration kernels' bit for bit.
#include <algorithm>
#include <mutex>

#include "cmf_slide.h"
#include "cmf_voxel.h"
#include "cmf_words.h"
#include "mh_reduce.h"

namespace {

using namespace mh;

constexpr int kMaxThreads = 1024;
constexpr int kRun = 8;        // planes per thread
constexpr int kCells = 1360;   // LDS cells of a tile and its faces
constexpr int kRedFloats = 64;
// residuals of both parities, h1 and h2 of one; in float4s; then cs and ct plane
// by plane
constexpr int kLdsVecs = 4 * kCells + 4 * kMaxThreads;

struct SumOp {
    __device__ static float identity() { return 0.f; }
    __device__ static float combine(float a, float b) { return a + b; }
};

typedef float Float4 __attribute__((ext_vector_type(4)));

struct Addresses {  // SlideFields, as kept in LDS
    const float *hp, *tmp, *pt, *u;
    float *hpo, *tmpo, *pto, *uo;
    const Float4 *q4;
    const float *alpha, *cs, *ct;
    const uint8_t *labels;
};
constexpr int kLdsFixed = 16 * kLdsVecs + 4 * kRedFloats + 4 * kMaxThreads + int(sizeof(Addresses));
int lds_bytes(int slots) { return kLdsFixed + 4 * kRun * slots; }
// what the masks may take of a compute unit's LDS (block_reduce holds 64 bytes)
constexpr int kLds = 160 * 1024, kLdsReduce = 64;
constexpr int kMaxSlots = (kLds - kLdsReduce - kLdsFixed) / (4 * kRun);

struct Args {
    SlideFields F;
    SlideControl C;
    int d0, d1, d2;
    int b1, b2, nt1, nt2, slots;
    int levels, it, check, cur;
    float rcc, inv_rcc, rs0, rs1, rs2, ss0, ss1, ss2;
    AxiParams A;
    Word *inbox;  // per work-group: [axis-0 residuals | h0 | rows and columns of residuals | of h]
    unsigned tag0;
    float *partials;
};

// A field whose address is kept in LDS, at byte offset off (below 2^31): the
// address is the same in every lane and goes through scalar registers. Through
// the global address space (a flat access would be waited for with the LDS's).
template <typename T>
using Global = T __attribute__((address_space(1)));
template <typename T>
__device__ __forceinline__ Global<T> *field(T *const &p, unsigned off)
{
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint64_t lo = unsigned(__builtin_amdgcn_readfirstlane(int(unsigned(a))));
    const uint64_t hi = unsigned(__builtin_amdgcn_readfirstlane(int(unsigned(a >> 32))));
    return reinterpret_cast<Global<T> *>((hi << 32 | lo) + uint64_t(off));
}
// the lower or upper two of a cell's four planes
__device__ __forceinline__ Vec<2> &half(Vec<4> *p, int h) { return reinterpret_cast<Vec<2> *>(p)[h]; }
__device__ __forceinline__ const Vec<2> &half(const Vec<4> *p, int h)
{
    return reinterpret_cast<const Vec<2> *>(p)[h];
}

// ONE: one run per tile (an instance of its own: the wrapped positions cost the others
// 1 %)
template <bool SUP, bool ONE>
__global__ void __launch_bounds__(kMaxThreads)
cmf_slide_kernel(const Args A)
{
    if (*A.C.stop) return;
    using Vec4 = Vec<4>;
    using Vec2 = Vec<2>;
    extern __shared__ __align__(16) unsigned char lds[];
    const int t = int(threadIdx.x), NT = int(blockDim.x);
    const int b1 = A.b1, b2 = A.b2, nc = b1 * b2, W = kRun * A.slots;
    // LDS cells, 4 planes of one parity each: the tile's own [0, nc), the row
    // beyond it [nc, nc + b2) (after it for residuals, before it for h1), the
    // column beyond it [nc + b2, nc + b2 + b1) (h2's lies in h1's cells), a zero
    Vec4 *sT = reinterpret_cast<Vec4 *>(lds);
    constexpr int kH1 = 2 * kCells, kH2 = 3 * kCells;
    float *fT = reinterpret_cast<float *>(sT);
    float *sCs = fT + 16 * kCells, *sCt = sCs + kRun * kMaxThreads;
    float *red = fT + 4 * kLdsVecs;
    int *fail = reinterpret_cast<int *>(red + kRedFloats - 1);
    // the fields' addresses, read where a plane is loaded or stored: held in
    // scalar registers all the time they would push others out
    Addresses *sF = reinterpret_cast<Addresses *>(red + kRedFloats);
    float *sE = reinterpret_cast<float *>(sF + 1);  // each thread's sum of |err|
    unsigned *sM = reinterpret_cast<unsigned *>(sE + kMaxThreads);  // W masks

    // A tile's runs side by side, so that each XCD holds some of every run: the
    // run that loads and stores in a step (its planes come and go) spreads over
    // all of them (two of eight XCDs took 1.5 us longer per step at 256^3).
    const unsigned b = xcd_block(blockIdx.x, gridDim.x);
    const int tile = int(b) / A.slots, c = int(b) - tile * A.slots;
    const int bx = tile % A.nt2, by = tile / A.nt2;
    const bool live = t < nc;
    const int y = live ? t / b2 : 0, x = live ? t - y * b2 : 0, cell = live ? t : 0;
    const int gy = by * b1 + y, gx = bx * b2 + x;
    const bool inv = live && gy < A.d1 && gx < A.d2;
    const bool e1 = gy < A.d1 - 1, e2 = gx < A.d2 - 1;
    const bool yp = by + 1 < A.nt1, ym = by > 0, xp = bx + 1 < A.nt2, xm = bx > 0;
    auto own_cell = [&](unsigned t8) { return sT + (here(t8) >> 3); };
    const Vec4 *const t2 = sT + (x < b2 - 1 ? cell + 1 : nc + b2 + y);
    const Vec4 *const m1p = sT + kH1 + (!inv ? kCells - 1 : y > 0 ? cell - b2 : nc + x);
    const Vec4 *const m2p =
        sT + (!inv ? kH1 + kCells - 1 : x > 0 ? kH2 + cell - 1 : kH1 + nc + b2 + y);

    // words: byte offsets of this work-group's inbox and of its parts
    // (a plane's in-plane words: b2 of a row, b1 of a column)
    const int P8 = 8 * (b1 + b2);
    const unsigned IB = 16u * unsigned(nc) + 16u * unsigned(P8), box = b * IB;
    const unsigned nc8 = 8u * unsigned(nc), boxT = box + 2u * nc8, boxH = boxT + 8u * unsigned(P8);
    const unsigned dx = unsigned(A.slots) * IB, dy = unsigned(A.nt2) * dx;
    const unsigned below_run = c > 0 ? box - IB : box + dx - IB;
    const unsigned above_run = c + 1 < A.slots ? box + IB : box + IB - dx;
    const unsigned t8 = 8u * unsigned(t);
    const bool oTy = inv && y == 0 && ym, oTx = inv && x == 0 && xm;
    const bool oHy = inv && y == b1 - 1 && yp, oHx = inv && x == b2 - 1 && xp;
    const bool firstT = __any(oTy), firstH = __any(oHy);
    for (int i = t; i < 4 * kLdsVecs + kRedFloats; i += NT) fT[i] = 0.f;
    if (t == 0)
        *sF = Addresses{A.F.hp, A.F.tmp, A.F.pt, A.F.u, A.F.hpo, A.F.tmpo, A.F.pto, A.F.uo,
                        reinterpret_cast<const Float4 *>(A.F.q4), A.F.alpha, A.F.cs, A.F.ct, A.F.labels};
    sE[t] = 0.f;
    lds_barrier();

    const float inv_b2 = 1.f / float(b2);
    auto row_of = [&](unsigned tt) { return unsigned((float(tt) + 0.5f) * inv_b2); };
    // those of planes i, i + 1 that are in `mask`, of a first or last row
    // (words: the senders are consecutive threads), and of a first or last column
    auto send_row = [&](bool mine, unsigned off, unsigned mask, int i, const float (&v)[2],
                        unsigned tag) {
        if (!mine) return;
        const unsigned o = here(t8) + off;
        if (mask >> 2 * i & 1) st_word(word_at(A.inbox, o + unsigned(here_s(2 * P8) * i)), tag, v[0]);
        if (mask >> 2 * i & 4)
            st_word(word_at(A.inbox, o + unsigned(here_s(2 * P8) * (i + 1))), tag, v[1]);
    };
    auto send_col = [&](bool mine, unsigned off, unsigned mask, int i, const float (&v)[2],
                        unsigned tag) {
        if (!mine) return;
        const unsigned o = 8u * row_of(here(t8) >> 3) + off;
        if (mask >> 2 * i & 1) st_word(word_at(A.inbox, o + unsigned(here_s(2 * P8) * i)), tag, v[0]);
        if (mask >> 2 * i & 4)
            st_word(word_at(A.inbox, o + unsigned(here_s(2 * P8) * (i + 1))), tag, v[1]);
    };

    // the words of the planes in `mask` of the row or column beyond the tile, into
    // the cells past its own
    auto receive = [&](unsigned off, unsigned mask, Vec4 *to, unsigned tag) {
        Word w[4] = {0, 0, 0, 0};
        for (int spin = 0;; ++spin) {
            bool missing = false;
            unrolled_while<4>([&](auto I) {
                if (mask >> 2 * I & 1) w[I] = ld_word(word_at(A.inbox, off + unsigned(here_s(2 * P8) * I)));
                return true;
            });
            unrolled_while<4>([&](auto I) {
                missing |= (mask >> 2 * I & 1) && unsigned(w[I] >> 32) != tag;
                return true;
            });
            if (!missing || give_up(spin, A.C.abort, fail)) break;
        }
        words_arrived();
        Vec4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v.v[i] = __builtin_bit_cast(float, unsigned(w[i]));
        *to = v;
    };
    auto receive_row = [&](bool mine, unsigned off, unsigned mask, int cell0, unsigned tag) {
        if (!mine || !(mask & 0x55u)) return;
        receive(here(t8) + off, mask, own_cell(t8) + cell0, tag);
    };
    auto receive_col = [&](bool mine, unsigned off, unsigned mask, int cell0, unsigned tag) {
        if (!mine || !(mask & 0x55u)) return;
        const unsigned yy = row_of(here(t8) >> 3);
        receive(8u * yy + off, mask, sT + cell0 + yy, tag);
    };

    const unsigned plane4 = 4u * unsigned(A.d1) * unsigned(A.d2);
    const unsigned n4 = plane4 * unsigned(A.d0);
    // byte offset of this thread's voxel in a plane (inside the volume only)
    auto in_plane = [&]() {
        const unsigned tt = here(t8) >> 3, yy = row_of(tt), xx = tt - yy * unsigned(b2);
        return 4u * ((unsigned(by * b1) + yy) * unsigned(A.d2) + unsigned(bx * b2) + xx);
    };
    const int lv2 = 2 * A.levels, send2 = lv2 - 2;

    float h0[kRun], h1[kRun], h2[kRun], pt[kRun], u[kRun], al[kRun], fr[kRun][3];
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
        h0[j] = h1[j] = h2[j] = pt[j] = u[j] = al[j] = 0.f;
        fr[j][0] = fr[j][1] = fr[j][2] = 0.f;
    }
    // A plane's way in: its residual is loaded a step before it joins, the rest
    // of its state in the step it joins in, into registers of their own (a use of
    // a position's registers would wait for loads that might be under way there),
    // and moved to its position a step later.
    float ntmp[2] = {0.f, 0.f};  // by parity of the plane
    float nh0 = 0.f, nh1 = 0.f, nh2 = 0.f, npt = 0.f, nu = 0.f, nal = 0.f, ncs = 0.f,
          nct = 0.f;
    Float4 nq = {0.f, 0.f, 0.f, 0.f};
    unsigned lab = 0, nlab = 0;  // two bits per plane
    auto load_residual = [&](auto PARITY, int k) {
        if (inv) ntmp[PARITY] = __builtin_nontemporal_load(field(sF->tmp, in_plane() + unsigned(k) * plane4));
    };
    auto load_state = [&](int k) {
        if (!inv) return;
        const unsigned o = in_plane() + unsigned(k) * plane4;
        const Addresses &F = *sF;
        nh0 = __builtin_nontemporal_load(field(F.hp, o));
        nh1 = __builtin_nontemporal_load(field(F.hp, o + n4));
        nh2 = __builtin_nontemporal_load(field(F.hp, o + 2u * n4));
        nq = __builtin_nontemporal_load(field(F.q4, 4u * o));
        npt = __builtin_nontemporal_load(field(F.pt, o));
        nu = __builtin_nontemporal_load(field(F.u, o));
        nal = __builtin_nontemporal_load(field(F.alpha, o));
        ncs = __builtin_nontemporal_load(field(F.cs, o));
        nct = __builtin_nontemporal_load(field(F.ct, o));
        if (SUP) nlab = *field(F.labels, o >> 2);
    };
    auto settle = [&](auto J) {
        constexpr int j = J;
        h0[j] = nh0;
        h1[j] = nh1;
        h2[j] = nh2;
        pt[j] = npt;
        u[j] = nu;
        al[j] = nal;
        frame_axis(make_float4(nq[0], nq[1], nq[2], nq[3]), fr[j][0], fr[j][1], fr[j][2]);
        sCs[j * kMaxThreads + (here(t8) >> 3)] = ncs;
        sCt[j * kMaxThreads + (here(t8) >> 3)] = nct;
        if (SUP) lab = (lab & ~(3u << (2 * j))) | ((nlab & 3u) << (2 * j));
    };

    // Position j's plane k at step s: s - k, twice its level, is ph - j - 1 (mod
    // W, from -1 on) with ph = (s + 1 - kRun c) mod W. All four positions of the
    // step's parity are computed; those whose plane does not advance hold values
    // that nothing reads (a plane's state is loaded after the step it joins in).
    // Bits 0-7: the positions that advance at the next step, 8-15: those whose
    // residuals go out, here as if every plane were inside the volume.
    for (int i = t; i < W; i += NT) {
        unsigned m = 0;
        for (int j = 0; j < kRun; ++j) {
            const int rel = i < j ? i - j + W - 1 : i - j - 1;
            m |= (rel >= 1 && rel < lv2 ? 1u : 0u) << j | (rel >= 0 && rel <= send2 ? 256u : 0u) << j;
        }
        sM[i] = m;
    }
    lds_barrier();
    int ph = (1 + W - kRun * c) % W;
    unsigned adv = 0;  // bit j: position j's plane takes a level at step s
    auto step = [&](auto PARC, int s) {
        constexpr int PAR = PARC;
        constexpr unsigned kMine = PAR ? 0xaau : 0x55u;
        const unsigned tag = A.tag0 + unsigned(s) + 1u;
        // the positions that advance next and that send, those with a plane above
        // and (position 0) below
        unsigned mask, e0 = 0xffu;
        bool over0 = true;
        if (s >= W && s + 3 < A.d0) {
            mask = unsigned(__builtin_amdgcn_readfirstlane(int(sM[ph])));
        } else {  // one lane per position
            const int j = int(here(t8) >> 3) & 63;
            const int rel = ph < j ? ph - j + W - 1 : ph - j - 1, k = s - rel;
            const bool in = unsigned(k) < unsigned(A.d0) && j < kRun;
            mask = unsigned(__ballot(in && rel >= 1 && rel < lv2)) |
                   unsigned(__ballot(in && rel >= 0 && rel <= send2)) << 8;
            e0 = unsigned(__ballot(k < A.d0 - 1));
            over0 = (unsigned(__ballot(k > 0)) & 1u) != 0;
        }
        const unsigned act = adv & kMine, out = mask >> 8 & kMine;
        // positions of planes s, s - 1 and s - 2 levels, this run's if 0 .. kRun - 1 (-1
        // and -2 are W - 1 and W - 2, another run's but where the tile has one run)
        const int joins = s < A.d0 ? (ONE && ph < 1 ? W - 1 : ph - 1) : -1;
        const int settles = s <= A.d0 && s > 0 ? (ONE && ph < 2 ? ph - 2 + W : ph - 2) : -1;
        const int leaves = s >= lv2 ? (ph - 1 < lv2 ? ph - 1 - lv2 + W : ph - 1 - lv2) : -1;
        lds_barrier();
        Vec4 *own = own_cell(t8);
        // p-step, two planes at a time: all four's neighbours at once would not
        // fit the registers beside the state
        if (firstH) __builtin_amdgcn_s_setprio(2);
        const bool rz1 = PAR == 1 && (act & 0x80u) && (e0 & 0x80u) && inv;
        auto p_plane = [&](auto I, float to, float t1, float t2v, float tn, float &w1, float &w2) {
            constexpr int j = 2 * I + PAR;
            const float g0 = (e0 >> j & 1) ? (tn - to) * A.ss0 : 0.f;
            const float g1 = e1 ? (t1 - to) * A.ss1 : 0.f;
            const float g2 = e2 ? (t2v - to) * A.ss2 : 0.f;
            cmf_p_voxel_axi(h0[j], h1[j], h2[j], g0, g1, g2, fr[j][0], fr[j][1], fr[j][2], A.A, al[j]);
            w1 = h1[j];
            w2 = h2[j];
        };
        const bool rz = PAR == 0 && (act & 1u) && over0 && inv;
        Word vz = 0;  // sent a step ago
        if (rz) vz = ld_word(word_at(A.inbox, here(t8) + (box + nc8)));
        Word vz1 = 0;
        if (act)
            unrolled_while<2>([&](auto HC) {
                constexpr int i = 2 * HC;
                const Vec2 To = half(own + PAR * kCells, HC), T1 = half(own + PAR * kCells + b2, HC),
                           T2 = half(t2 + PAR * kCells, HC);
                const float *Tn = own[(1 - PAR) * kCells].v;
                const float n0 = Tn[i + PAR];
                float n1 = Tn[i + 1 + PAR < 4 ? i + 1 + PAR : 3];
                Vec2 w1, w2;
                if (PAR == 1 && i == 0 && rz1) vz1 = ld_word(word_at(A.inbox, here(t8) + box));
                p_plane(std::integral_constant<int, i>{}, To.v[0], T1.v[0], T2.v[0], n0, w1.v[0], w2.v[0]);
                if (PAR == 1 && i == 2) {  // position 7: the residual of the next run's first plane
                    for (int spin = 0; rz1 && unsigned(vz1 >> 32) != tag - 1; ++spin) {
                        if (give_up(spin, A.C.abort, fail)) break;
                        vz1 = ld_word(word_at(A.inbox, here(t8) + box));
                    }
                    words_arrived();
                    n1 = __builtin_bit_cast(float, unsigned(vz1));
                }
                p_plane(std::integral_constant<int, i + 1>{}, To.v[1], T1.v[1], T2.v[1], n1, w1.v[1],
                        w2.v[1]);
                if (PAR == 1 && i == 2 && rz1)
                    st_word(word_at(A.inbox, here(t8) + (above_run + nc8)), tag, h0[7]);
                send_row(oHy, boxH + dy + unsigned(PAR * P8) - 8u * unsigned(nc - b2), act >> PAR, i, w1.v, tag);
                send_col(oHx, boxH + dx + unsigned(PAR * P8) + 8u * unsigned(b2), act >> PAR, i, w2.v, tag);
                if (live) {
                    half(own + kH1, HC) = w1;
                    half(own + kH2, HC) = w2;
                }
                __builtin_amdgcn_sched_barrier(0);
                return true;
            });
        if (firstH) __builtin_amdgcn_s_setprio(0);
        lds_barrier();
        // Receive. What a thread receives it alone reads: only the waves of an
        // outer row or column wait, while the others go on.
        receive_row(oTy, boxH + unsigned(PAR * P8), act >> PAR, kH1 + nc, tag);
        receive_col(oTx, boxH + unsigned(PAR * P8) + 8u * unsigned(b2), act >> PAR, kH1 + nc + b2, tag);
        receive_row(oHy, boxT + unsigned((1 - PAR) * P8) - 8u * unsigned(nc - b2), mask >> (1 - PAR),
                    (1 - PAR) * kCells + b2, tag - 1);
        receive_col(oHx, boxT + unsigned((1 - PAR) * P8) + 8u * unsigned(b2), mask >> (1 - PAR),
                    (1 - PAR) * kCells + nc + b2, tag - 1);
        float below = 0.f;
        if (PAR == 0) {
            for (int spin = 0; rz && unsigned(vz >> 32) != tag - 1; ++spin) {
                if (give_up(spin, A.C.abort, fail)) break;
                vz = ld_word(word_at(A.inbox, here(t8) + (box + nc8)));
            }
            below = rz ? __builtin_bit_cast(float, unsigned(vz)) : 0.f;
        }
        words_arrived();
        if (unsigned(settles) < unsigned(kRun))
            unrolled_while<4>([&](auto I) {
                if (settles == 2 * I + 1 - PAR) settle(std::integral_constant<int, 2 * I + 1 - PAR>{});
                return true;
            });
        // (here, so that the next wait for words, which waits for these loads as
        // well, is most of a step away)
        if (unsigned(joins) < unsigned(kRun)) load_state(s);
        if (ph < kRun && s + 1 < A.d0) load_residual(std::integral_constant<int, 1 - PAR>{}, s + 1);
        own = own_cell(t8);
        // u-step
        if (firstT) __builtin_amdgcn_s_setprio(2);
        auto u_plane = [&](auto I, float m1, float m2, float cap_s, float cap_t, float &T) {
            constexpr int j = 2 * I + PAR;
            const float own0 = (e0 >> j & 1) ? h0[j] : 0.f;
            const float x0 = own0 - (j == 0 ? below : h0[j > 0 ? j - 1 : 0]);
            const float x1 = (e1 ? h1[j] : 0.f) - m1;
            const float x2 = (e2 ? h2[j] : 0.f) - m2;
            const float div = cmf_div(x0, x1, x2, A.rs0, A.rs1, A.rs2);
            float ub = 1.f, uf = 0.f;
            if (SUP) {
                const unsigned l = here(lab) >> (2 * j);
                uf = float(l & 1u);
                ub = (l & 2u) ? 0.f : 1.f;
            }
            const float err = cmf_u_voxel(div, pt[j], u[j], T, cap_s, cap_t, A.rcc, A.inv_rcc, ub, uf);
            if (j == leaves && (act >> j & 1)) {
                if (inv) {
                    sE[here(t8) >> 3] += fabsf(err);
                    const unsigned o = in_plane() + unsigned(s - lv2) * plane4;
                    const Addresses &F = *sF;
                    *field(F.hpo, o) = h0[j];
                    *field(F.hpo, o + n4) = h1[j];
                    *field(F.hpo, o + 2u * n4) = h2[j];
                    *field(F.pto, o) = pt[j];
                    *field(F.uo, o) = u[j];
                    *field(F.tmpo, o) = T;
                }
            }
        };
        if (act | out)
            unrolled_while<2>([&](auto HC) {
                constexpr int i = 2 * HC;
                const Vec2 m1 = half(m1p, HC), m2 = half(m2p, HC);
                const float *C = sCs + (2 * i + PAR) * kMaxThreads + (here(t8) >> 3);
                const float *E = C + kRun * kMaxThreads;
                Vec2 T;
                u_plane(std::integral_constant<int, i>{}, m1.v[0], m2.v[0], C[0], E[0], T.v[0]);
                u_plane(std::integral_constant<int, i + 1>{}, m1.v[1], m2.v[1], C[2 * kMaxThreads],
                        E[2 * kMaxThreads], T.v[1]);
                if (joins == 2 * i + PAR) T.v[0] = ntmp[PAR];
                if (joins == 2 * i + 2 + PAR) T.v[1] = ntmp[PAR];
                if (i == 0 && PAR == 0 && (out & 1u) && over0 && inv)
                    st_word(word_at(A.inbox, here(t8) + below_run), tag, T.v[0]);
                send_row(oTy, boxT - dy + unsigned(PAR * P8), out >> PAR, i, T.v, tag);
                send_col(oTx, boxT - dx + unsigned(PAR * P8) + 8u * unsigned(b2), out >> PAR, i, T.v, tag);
                if (live) half(own + PAR * kCells, HC) = T;
                __builtin_amdgcn_sched_barrier(0);
                return true;
            });
        if (firstT) __builtin_amdgcn_s_setprio(0);
        adv = mask & 0xffu;
        ph = ph + 1 == W ? 0 : ph + 1;
    };
    if (c == 0) load_residual(std::integral_constant<int, 0>{}, 0);
    const int last = A.d0 - 1 + lv2;  // the last plane's last level
    for (int s = 0; s <= last; s += 2) {
        step(std::integral_constant<int, 0>{}, s);
        step(std::integral_constant<int, 1>{}, s + 1);
    }
    const float aerr = block_reduce<SumOp>(sE[t]);
    lds_barrier();
    if (t != 0) return;
    if (*fail) {  // this pass's output is not complete: the solve goes on elsewhere
        *A.C.abort_it = A.it;
        *A.C.abort_cur = A.cur;
        *A.C.stop = kSlideAborted;
        return;
    }
    if (A.check) A.partials[b] = aerr;
    if (b == 0) *A.C.parity = 1 - A.cur;
}

__global__ void __launch_bounds__(mh::kBlock) zero_words_kernel(Word *w, int64_t n)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) w[i] = 0;
}

template <bool ONE>
const void *kernel_of(bool sup)
{
    return sup ? reinterpret_cast<const void *>(&cmf_slide_kernel<true, ONE>)
               : reinterpret_cast<const void *>(&cmf_slide_kernel<false, ONE>);
}

int threads_of(const SlidePlan &P) { return (P.b1 * P.b2 + 63) / 64 * 64; }

}  // namespace

namespace mh {

int64_t slide_inbox_bytes(const SlidePlan &P)
{
    return int64_t(P.blocks()) * 16 * (int64_t(P.b1) * P.b2 + 8 * (P.b1 + P.b2));
}

SlidePlan slide_plan(int cus, const int dims[3], const mh_cmf_params *prm, bool sup)
{
    SlidePlan best;
    const int64_t n = int64_t(dims[0]) * dims[1] * dims[2];
    // byte offsets of the AoS x4 frames stay below 2^31
    if (!axi_params(prm).on || n >= (int64_t(1) << 27)) return best;
    // (a window of cus runs of planes holds 4 cus - 1 iterations: a criterion rarer
    // than that, INT_MAX among them, ends no pass)
    const int update = std::min(prm->update, 4 * std::max(cus, 1));
    double best_cost = 0;
    for (int n2 = 1; n2 <= std::min(dims[2], 16); ++n2) {
        const int b2 = (dims[2] + n2 - 1) / n2;
        if (b2 > kMaxThreads) continue;
        const int least = (dims[1] + kMaxThreads / b2 - 1) / (kMaxThreads / b2);
        for (int n1 = least; n1 <= std::min(dims[1], least + 16); ++n1) {
            SlidePlan P;
            P.b1 = (dims[1] + n1 - 1) / n1;
            P.b2 = b2;
            P.nt1 = (dims[1] + P.b1 - 1) / P.b1;
            P.nt2 = (dims[2] + b2 - 1) / b2;
            const int tiles = P.nt1 * P.nt2;
            if (tiles > cus || P.b1 * b2 + P.b1 + b2 + 1 > kCells)
                continue;
            // W = 8 slots planes hold 4 slots - 1 levels; a pass ends at a criterion
            P.slots = std::min({cus / tiles, (update + 4) / 4, kMaxSlots});
            P.levels = std::min(4 * P.slots - 1, update);
            const int passes = (update + P.levels - 1) / P.levels;
            P.levels = (update + passes - 1) / passes;
            P.slots = std::min(P.slots, (P.levels + 4) / 4);
            if (P.levels < 3) continue;
            const int waves = (threads_of(P) / 64 + 3) / 4;
            // microseconds, measured within 10 % for rows of 64 .. 320 voxels;
            // columns of more than 12 words are slow to receive
            const double step = 2.25 + 0.22 * waves + 1.3e-5 * dims[1] * dims[2] +
                                (P.nt2 > 1 ? (P.b1 > 12 ? 3.5 : 0.5) : 0.0);
            const double cost = (dims[0] + 2.0 * P.levels) * step / P.levels;
            if (best.levels == 0 || cost < best_cost) {
                best = P;
                best_cost = cost;
            }
        }
    }
    // Where it wins: against the sweeps, which do up to 1.5e11 voxels and iterations
    // a second while their state stays in the last-level cache (132 x 159 x 155
    // 1.48e11 against 1.46e11 here) and 0.95e11 .. 1.3e11 beyond it (256^3 1.22e11
    // against 2.18e11 here, 192^3 1.28e11 and 1.49e11, 240 x 230 x 190 1.17e11 and
    // 1.63e11, 320^3 1.2e11 and 1.36e11; but 420^3 1.30e11 and 0.92e11, 256^3 with a
    // criterion every 5 iterations 1.1e11 and 0.82e11), and with seeds against the
    // per-iteration kernels (256^3 5.6e10 and 2.08e11; with one run of planes, three
    // iterations a pass, 128 x 512 x 512 5.7e10 and 1.14e11, 40 x 512 x 512 6.0e10 and
    // 1.02e11, 64 x 400 x 400 6.0e10 and 7.9e10, 10 x 500 x 500 6.3e10 and 6.8e10).
    const double others = sup ? 6e4 : n < (int64_t(1) << 22) ? 1.5e5 : 1.3e5;
    if (best.levels && best_cost > double(n) / others) best.levels = 0;
    return best;
}

SlidePlan slide_plan(mh_ctx *ctx, const int dims[3], const mh_cmf_params *prm, bool sup)
{
    return ctx->device < kMaxDevices ? slide_plan(compute_units(ctx), dims, prm, sup) : SlidePlan();
}

int slide_lds_bytes(const SlidePlan &P) { return lds_bytes(P.slots) + kLdsReduce; }

int slide_pass(mh_ctx *ctx, const SlidePlan &P, const SlideFields &F, const int dims[3],
               const mh_cmf_params *prm, int lv, int it, bool check, int cur, bool lost,
               const SlideControl &C, float *partials, void *inbox, size_t inbox_bytes, unsigned *tags,
               hipStream_t s)
{
    MH_REQUIRE(ctx, lv >= 1 && lv <= P.levels, "levels of a pass");
    const unsigned steps = unsigned(dims[0] + 2 * lv + 4);
    if (*tags == 0 || *tags > 0xffffffffu - steps) {  // a new inbox, or the tags start over
        const int64_t words = int64_t(inbox_bytes / sizeof(Word));
        hipLaunchKernelGGL(zero_words_kernel, dim3(blocks_for(words)), dim3(kBlock), 0, s,
                           static_cast<Word *>(inbox), words);
        MH_CHECK_LAUNCH(ctx, "slide inbox");
        *tags = 0;
    }
    Args A{};
    A.F = F;
    A.C = C;
    A.d0 = dims[0];
    A.d1 = dims[1];
    A.d2 = dims[2];
    A.b1 = P.b1;
    A.b2 = P.b2;
    A.nt1 = P.nt1;
    A.nt2 = P.nt2;
    A.slots = P.slots;
    A.levels = lv;
    A.it = it;
    A.check = check;
    A.cur = cur;
    A.rcc = prm->rcc;
    A.inv_rcc = float(1.0 / double(prm->rcc));
    A.rs0 = prm->rs[0];
    A.rs1 = prm->rs[1];
    A.rs2 = prm->rs[2];
    A.ss0 = prm->ss[0];
    A.ss1 = prm->ss[1];
    A.ss2 = prm->ss[2];
    A.A = axi_params(prm);
    A.inbox = static_cast<Word *>(inbox);
    A.tag0 = *tags;
    A.partials = partials;
    *tags += steps;
    const void *kernel = P.slots == 1 ? kernel_of<true>(F.labels != nullptr) : kernel_of<false>(F.labels != nullptr);
    void *args[] = {&A};
    MH_CHECK(ctx, hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes(P.slots)));
    const unsigned blocks = unsigned(P.blocks() - (lost && P.blocks() > 1));
    MH_CHECK(ctx, hipLaunchCooperativeKernel(kernel, dim3(blocks),
                                             dim3(unsigned(threads_of(P))), args,
                                             unsigned(lds_bytes(P.slots)), s));
    return MH_OK;
}

}  // namespace mh

MH_EXPORT int mh_cmf_slide_plan(const int64_t dims[3], const mh_cmf_params *prm, int seeded,
                                int compute_units, int plan[6])
{
    if (!mh::dims_ok(dims) || !prm || prm->update < 1) return MH_ERR_ARG;
    const int d[3] = {int(dims[0]), int(dims[1]), int(dims[2])};
    const mh::SlidePlan P = mh::slide_plan(compute_units, d, prm, seeded != 0);
    if (P.levels && plan) {
        const int v[6] = {P.b1, P.b2, P.nt1, P.nt2, P.slots, mh::slide_lds_bytes(P)};
        std::copy(v, v + 6, plan);
    }
    return P.levels;
}
