// Lattice i-quants: IQ2_XXS, IQ2_XS, IQ2_S (groups of 8 weights) and IQ3_XXS, IQ3_S (groups of 4),
// bit-exact with ggml-quants.c (cited per step).
//
// The reference rounds a sub-block at each of 13 to 31 trial scales; a group whose rounded levels u are
// no codebook point takes the best point of u's neighbour list: the first with the least
// d2 = sum_i sqrt(w_i) (s q_i - x_i)^2 at the trial's scale s. Searched trial by trial (20 to 60 points
// each) this was 75-94% of the kernels' time. Three facts make most of that work unnecessary:
//   * the searches of all trials depend only on u and s, not on which trial is best so far;
//   * u changes only once or twice over the trials of a group, so a run of trials shares one list;
//   * with B = sum v q x and C = sum v q^2 (v = sqrt(w)), d2 = A + 2 s (s C / 2 - B): at a fixed point
//     the order of the points is that of functions linear in s: a point that is best at two scales is
//     best at every scale between them.
// So a wave collects the runs of its 64 sub-blocks (one group index at a time) in an LDS queue, sorted
// by list length, and each lane scans the list of one run once, for its first and its last trial: what
// the trials between take follows from those (search_runs). B and C are integers here: v and v x are
// scaled by powers of two to 22-24 bits, and twelve (six) 4-way byte dot products with a point's bytes
// q and q^2 give both.
// Exactness: the filter's answer counts only where its best point leads the second by more than a bound
// on everything that separates it from the reference's float sums (tolerance() below). Otherwise, and
// for inputs outside the filter's range, the reference's float expression is evaluated for the whole list,
// its first strict minimum winning as in the C code: a few lanes' lists one after another, each by the whole
// wave (exact_neighbour), more of them cut into pieces that are dealt to the lanes (dealt_neighbours).
//
// The SIMDs issue VALU instructions in 84-89% of their quad-cycles, almost never two at once: half of the issue
// limit. With the importance matrix, against one list search per trial and group: IQ2_XS 4096 x 12288 6.10 to
// 3.18 ms (7231 to 2459 lane-instructions a weight), IQ3_XXS 2053 x 3584 1.157 to 0.64 ms; on 4096 x 4096 IQ2_XXS
// 1.48 to 0.94 ms, IQ2_S 0.75 to 0.57 ms, IQ3_S 1.29 to 0.88 ms.
// Weights on a coarse grid, where equal distances are common, need the float sums for up to half of their trials.
// Without the importance matrix, 4096 x 4096, us: one list search per trial and group; undecided lists one after
// another, each by the whole wave; dealt, up to four trials at once:
//   4-bit codes, a scale per 32    IQ2_S 712 / 3790 / 945    IQ3_XXS 1835 / 5220 / 1790    IQ3_S 1290 / 3150 / 1290
//   three values, a scale per 128  IQ2_S 556 / 2600 / 584    IQ3_XXS 1600 / 15460 / 1490   IQ3_S  885 / 2960 /  785
// On normal weights the dealt search, which runs there now and then, its registers and the bound cost 1% to 2%,
// IQ2_S 3%.
//
// Mapping: one lane per sub-block (32 or 16 weights), G = 256/N lanes per super-block, 256-lane
// workgroups, held to three waves per SIMD (8 to 212 bytes of scratch a lane; at two or four waves the kernels
// are 10-20% slower). The groups of the sub-blocks are worked through one by one, a group's weights read again
// for each (they stay in L1/L2) so that only the trials' running sums are held in registers.
#include <type_traits>

#include "../../include/seedpack_amd.h"
#include "common.h"
#include "iq_tables.h"
#include "launch.h"
#include "search.h"

namespace spa {
namespace {

constexpr int WG = 256;
constexpr float FLT_BIG = 3.402823466e+38F;   // FLT_MAX
constexpr uint32_t PREV = 0xffffu;            // a trial's point: that of the trial before it
constexpr uint32_t EXACT = 0xfffeu;           // a trial's point: still to be found by the float sums
// Open points of at most FEW lanes and FEW_TRIALS trials are found one after another, more of them dealt (FEW = 0,
// 2, 6: IQ2_S with normal weights 631, 606, 606 us; 6 is 10-25% slower where weights are on a fine grid).
// A run that is undecided at both ends is left open at once where more than MANY of those searched side by side
// are undecided; so is one that is undecided once more, there and without an importance matrix, where equal weights
// make equal distances common. Elsewhere a near miss of one or two trials is likelier, which a further scan of the run
// costs less (left open: IQ2_XS and IQ2_S with normal weights 1% and 2% slower; scanned again without a matrix:
// weights of three values 14-27% slower).
constexpr int FEW = 2, FEW_TRIALS = 4, MANY = 3;
constexpr int QCAP = 256;                     // runs a wave queues before it searches them
constexpr uint32_t PEELED = 1u << 31;         // a queued run: what is left of one with an undecided end

enum Kind { K_IQ2_XXS, K_IQ2_XS, K_IQ2_S, K_IQ3_XXS, K_IQ3_S };

// D: group size; N: sub-block; BS: block bytes; PTS: codebook points; KMAXQ: levels; trials
// is = IS_LO .. IS_LO + T - 1 in steps of STEP; TWO: sigma2 = 2 sumx2 / 256 (else sumx2 / 256); PARITY:
// an even count of signs per 8 weights; R: list entries per piece (lists of 30 to 60 points, of about 10); EPS: sub-blocks whose max is below it are empty (IQ3_S: max == 0);
// ON0: groups count as on the grid before a trial wins; ALL: every group is redone at the end
template <int K> struct Cfg;
template <> struct Cfg<K_IQ2_XXS> {
    static constexpr int D = 8, N = 32, BS = 66, PTS = 256, KMAXQ = 3, T = 13, R = 8, IS_LO = -6;
    static constexpr float STEP = 0.1f, EPS = GROUP_MAX_EPS, DSCALE = 1.f;
    static constexpr bool TWO = false, PARITY = true, ON0 = false, ALL = true;
};
template <> struct Cfg<K_IQ2_XS> {
    static constexpr int D = 8, N = 16, BS = 74, PTS = 512, KMAXQ = 3, T = 19, R = 8, IS_LO = -9;
    static constexpr float STEP = 0.1f, EPS = GROUP_MAX_EPS, DSCALE = 1.f;
    static constexpr bool TWO = false, PARITY = true, ON0 = true, ALL = false;
};
template <> struct Cfg<K_IQ2_S> {
    static constexpr int D = 8, N = 16, BS = 82, PTS = 1024, KMAXQ = 3, T = 19, R = 4, IS_LO = -9;
    static constexpr float STEP = 0.1f, EPS = 1e-8f, DSCALE = 0.9875f;
    static constexpr bool TWO = true, PARITY = false, ON0 = true, ALL = false;
};
template <> struct Cfg<K_IQ3_XXS> {
    static constexpr int D = 4, N = 32, BS = 98, PTS = 256, KMAXQ = 8, T = 31, R = 4, IS_LO = -15;
    static constexpr float STEP = 0.2f, EPS = 1e-8f, DSCALE = 1.0125f;
    static constexpr bool TWO = true, PARITY = true, ON0 = true, ALL = false;
};
template <> struct Cfg<K_IQ3_S> {
    static constexpr int D = 4, N = 32, BS = 110, PTS = 512, KMAXQ = 8, T = 19, R = 4, IS_LO = -9;
    static constexpr float STEP = 0.2f, EPS = 0.f, DSCALE = 1.033f;
    static constexpr bool TWO = true, PARITY = false, ON0 = false, ALL = true;
};

// ---------------------------------------------------------------- a wave's LDS

// a sub-block's current group for the filter: byte planes of v (scaled by 2^a) and of v x (scaled by
// 2^b, two's complement: the top plane is signed), 4 weights a word, then {max, 2^b / 2^a / 2,
// 2^b / 2 sum v x^2, final scale}
template <int D> struct Record {
    uint4 w[D == 8 ? 4 : 3];
};
template <int K> struct WaveMem {
    using C = Cfg<K>;
    Record<C::D> rec[64];
    uint2 queue[QCAP];                   // {map entry (or rounded levels), lane | first trial << 8 | last << 16}
    uint16_t point[C::T][64];            // per trial and lane: the group's point, PREV or EXACT
    uint16_t best[C::N / C::D][64];      // per group and lane: the point written out
};

// LDS writes of the wave's lanes complete before its later LDS reads, and no compiler reordering
__device__ __forceinline__ void wave_lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ int lanes_below(uint64_t m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
__device__ __forceinline__ float lane_float(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// The device map holds, for levels off the grid, -1 - (list offset / 8 << 9 | list length)
__device__ __forceinline__ int list_offset(int gi) { return ((-1 - gi) >> 9) * 8; }
__device__ __forceinline__ int list_length(int gi) { return (-1 - gi) & 511; }

// a codebook point in LDS: its bytes q = 2l + 1 and their squares; R list entries as they are read
template <int D> struct Point;
template <> struct __align__(16) Point<8> { uint32_t q[2], s[2]; };
template <> struct __align__(8) Point<4> { uint32_t q[1], s[1]; };
template <int R> struct __align__(2 * R) Piece { uint32_t j[R / 2]; };

template <int D>
__device__ __forceinline__ void coords(const Point<D>& p, float (&q)[D]) {
#pragma unroll
    for (int i = 0; i < D; ++i) q[i] = (float)((p.q[i / 4] >> (8 * (i & 3))) & 0xff);
}

// ---------------------------------------------------------------- rounding

// level index of a group rounded at inverse scale id: nearest_int(0.5 (id x - 1)) clamped to the levels,
// B bits per coordinate
template <int D, int KMAXQ>
__device__ __forceinline__ int round_exact(const float (&xval)[D], float id) {
    constexpr int B = D == 8 ? 2 : 3;
    int u = 0;
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const int l = nearest_int(0.5f * (id * xval[i] - 1));
        u |= tmax(0, tmin(KMAXQ - 1, l)) << (B * i);
    }
    return u;
}
// the same number in float for finite |id x| < 2^22: 0.5 (y - 1) rounds as 0.5 y - 0.5 in one step does (a
// factor of two is exact), rint rounds as nearest_int does, and the index is a sum of exact small numbers
template <int D, int KMAXQ>
__device__ __forceinline__ int round_float(const float (&xval)[D], float id) {
    constexpr int B = D == 8 ? 2 : 3;
    float u = 0.f;
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const float y = id * xval[i];
        const float l = rintf(__builtin_amdgcn_fmed3f(__builtin_fmaf(y, 0.5f, -0.5f), 0.f, (float)(KMAXQ - 1)));
        u = __builtin_fmaf(l, (float)(1 << (B * i)), u);
    }
    return (int)u;
}

template <int K>
__host__ __device__ __forceinline__ float trial_num(int t) {
    return (float)(2 * Cfg<K>::KMAXQ - 1) + (float)(t + Cfg<K>::IS_LO) * Cfg<K>::STEP;
}
// trial t's inverse scale num / max, correctly rounded: with rmax = 1 / max correctly rounded, one
// remainder step corrects num rmax to the quotient (checked for every mantissa of max and every num of
// the types; max is within 2^+-60 here, so nothing over- or underflows)
template <int K>
__host__ __device__ __forceinline__ float trial_id(int t, float max, float rmax) {
    const float num = trial_num<K>(t), q = num * rmax;
    return __builtin_fmaf(__builtin_fmaf(-max, q, num), rmax, q);
}

// The trials at which some weight of the group takes another level than at the trial before, as bits (and
// trial 0). A weight's level rises with the trial; level L is reached at the first trial with
// 0.5 (id x - 1) >= L - 0.5 about: num = 2 L max / x, which is right to far less than a trial's step, so
// that the first trial is its ceiling or one beside it, decided by the rounding itself.
template <int K>
__device__ __forceinline__ uint32_t level_changes(const float (&xval)[Cfg<K>::D], float max, float rmax) {
    using C = Cfg<K>;
    auto level = [&](float x, float id) __attribute__((always_inline)) {
        return rintf(__builtin_amdgcn_fmed3f(__builtin_fmaf(id * x, 0.5f, -0.5f), 0.f, (float)(C::KMAXQ - 1)));
    };
    const float id0 = trial_id<K>(0, max, rmax), id1 = trial_id<K>(C::T - 1, max, rmax);
    uint32_t bits = 1;
#pragma unroll
    for (int i = 0; i < C::D; ++i) {
        const float x = xval[i], last = level(x, id1);
        const float rx = 2.f * max * __builtin_amdgcn_rcpf(x) * (1.f / C::STEP);
        for (float l = level(x, id0) + 1.f; __ballot(l <= last); l += 1.f) {
            const float at = ceilf(__builtin_fmaf(l, rx, -trial_num<K>(0) * (1.f / C::STEP)));
            int t = (int)fminf(fmaxf(at, 1.f), (float)(C::T - 1));
            if (level(x, trial_id<K>(t, max, rmax)) < l) ++t;
            else if (level(x, trial_id<K>(t - 1, max, rmax)) >= l) --t;
            if (l <= last) bits |= 1u << t;
        }
    }
    return bits;
}

// ---------------------------------------------------------------- the exact search

// The reference's neighbour (iq2_find_best_neighbour / iq3_find_best_neighbour, ggml-quants.c:3271-3293,
// :3915-3937) of lane o's group: the first listed point with the least d2 < FLT_MAX, each lane taking
// entries of the list; without one the list's first point (the reference asserts there instead). Called
// by the whole wave; xval, v, s and gi are each lane's own, o is uniform.
template <int D>
__device__ __forceinline__ int exact_neighbour(const float (&xval)[D], const float (&v)[D], float s, int gi, int o,
                                            const Point<D>* pts, const uint16_t* __restrict__ nb) {
    float x[D], w[D];
#pragma unroll
    for (int i = 0; i < D; ++i) { x[i] = lane_float(xval[i], o); w[i] = lane_float(v[i], o); }
    const float sc = lane_float(s, o);
    const int g = __builtin_amdgcn_readlane(gi, o);
    const uint16_t* list = nb + list_offset(g);
    const int len = list_length(g);
    float best = FLT_BIG;
    int bj = list[0];
    for (int base = 0; base < len; base += 64) {
        const int pos = base + (int)__lane_id();
        const int j = list[pos < len ? pos : len - 1];
        float q[D];
        coords<D>(pts[j], q);
        float d2 = 0;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const float diff = sc * q[i] - x[i];
            d2 += w[i] * diff * diff;
        }
        if (!(pos < len && d2 < best)) d2 = FLT_BIG;
        float m = d2;
#pragma unroll
        for (int st = 32; st >= 1; st >>= 1) m = fminf(m, __shfl_xor(m, st));
        if (m < best) {
            best = m;
            bj = __builtin_amdgcn_readlane(j, __ffsll((unsigned long long)__ballot(d2 == m)) - 1);
        }
    }
    return bj;
}

// The same for every lane with bits in `sel`, each its own group and list, at NT scales at once: trials t0 to
// t0 + NT - 1, bit i for trial t0 + i (NT = 1: the scale s). The lists are cut into pieces of R entries and dealt to
// the lanes in rounds, so that the wave does not wait for its longest list. A list's winner is the least of d2 as
// bits, position and point (d2 is not negative; infinities and NaN order above FLT_MAX), lowered by atomic minima
// in the words of the queue, which is empty here.
template <int K, int NT>
__device__ __forceinline__ void dealt_neighbours(WaveMem<K>& W, int t0, uint32_t sel, const float (&xval)[Cfg<K>::D],
                                                 const float (&v)[Cfg<K>::D], float max, float s, int gi,
                                                 const Point<Cfg<K>::D>* pts, const uint16_t* __restrict__ nb) {
    constexpr int D = Cfg<K>::D, R = Cfg<K>::R;
    static_assert(64 * NT <= QCAP, "a word for each lane and scale");
    unsigned long long* slots = reinterpret_cast<unsigned long long*>(W.queue);
    const int lane = (int)__lane_id();
    const int np = sel ? (list_length(gi) + R - 1) / R : 0;
    const unsigned long long none = ((unsigned long long)0x7f7fffffu << 32) | (sel ? nb[list_offset(gi)] : 0u);   // (FLT_MAX, position 0)
#pragma unroll
    for (int i = 0; i < NT; ++i) slots[64 * i + lane] = none;
    // inclusive prefix of the piece counts: shifts by 1, 2, 4, 8 within a row of 16 lanes, then the rows below
    int incl = np;
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xf, 0xf, false);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xf, 0xf, false);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xf, 0xf, false);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xf, 0xf, false);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x142, 0xa, 0xf, false);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x143, 0xc, 0xf, false);
    const int total = __builtin_amdgcn_readlane(incl, 63);
    wave_lds_sync();
    for (int base = 0; base < total; base += 64) {
        const int q = base + lane;
        int o = 0;                               // the lane whose pieces hold q: how many end at or before it
#pragma unroll
        for (int st = 32; st >= 1; st >>= 1)
            if (__shfl(incl, o + st - 1) <= q) o += st;
        const int first = __shfl(incl - np, o), g = __shfl(gi, o);
        uint32_t what = (uint32_t)__shfl((int)(sel | (uint32_t)t0 << 8), o);         // by all lanes, before any is left out
        if (q >= total) what = 0u;
        const float m = __shfl(NT == 1 ? s : max, o);
        float x[D], w[D];
#pragma unroll
        for (int i = 0; i < D; ++i) { x[i] = __shfl(xval[i], o); w[i] = __shfl(v[i], o); }
        const int p = q - first, len = list_length(g);
        const uint16_t* list = what ? nb + list_offset(g) + p * R : nb;      // (lists are padded to whole pieces)
        float sc[NT];
        unsigned long long best[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            sc[i] = NT == 1 ? m : 1 / (trial_num<K>((int)(what >> 8) + i) / m);
            best[i] = ~0ull;
        }
#pragma unroll 1
        for (int e = 0; e < R; ++e) {
            const int j = list[e];
            const uint32_t low = (uint32_t)((p * R + e) << 16) | (uint32_t)j;
            float c[D];
            coords<D>(pts[j], c);
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                float d2 = 0;
#pragma unroll
                for (int b = 0; b < D; ++b) {
                    const float diff = sc[i] * c[b] - x[b];
                    d2 += w[b] * diff * diff;
                }
                const unsigned long long key = ((unsigned long long)__float_as_uint(d2) << 32) | low;
                if (p * R + e < len && key < best[i]) best[i] = key;
            }
        }
#pragma unroll
        for (int i = 0; i < NT; ++i)
            if (what >> i & 1) atomicMin(&slots[64 * i + o], best[i]);
    }
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < NT; ++i)
        if (sel >> i & 1) W.point[t0 + i][lane] = (uint16_t)slots[64 * i + lane];
    wave_lds_sync();
}

// ---------------------------------------------------------------- the filter

// Bounds over every list of a lattice type (spa_lattice_bound_host shows them to the tests):
// L1, M2: the largest sums over the coordinates of |q - q'| and |q^2 - q'^2| between a list's first
// point and another of it; P1, P2: between any two points of it.
template <int D> struct ListBound;
template <> struct ListBound<8> { static constexpr float L1 = 20, M2 = 128, P1 = 24, P2 = 144; };
template <> struct ListBound<4> { static constexpr float L1 = 16, M2 = 336, P1 = 24, P2 = 480; };

// How far the filter's second best value has to lie above its best so that the best is the reference's
// strict minimum. The values are F = s' C - B over integers, s' = s 2^b / 2^(a+1), relative to the list's
// first point; d2 = A + 2 s / 2^b F. With u = 2^-24, V = v 2^a <= VMAX = 2^23 (2^22 for D = 4) and
// |P| = |v x 2^b| < 2^23 it covers, for the two points:
//   V rounded to an integer      s' P2 / 2          P rounded to an integer, and v x itself     P1 / 2 + P1 / 2
//   s', within 4 u of the trial's scale (search_runs)                                  4 u VMAX s' P2
//   C and B converted, the fma: 2 u (|s' C| + |B|) for each point                      4 u (VMAX s' M2 + 2^23 L1)
//   the reference's float sum: 14 u d2 + u A for each point (|s q| <= |diff| + |x|; the rounded differences, two
//   products and the additions left to right)                                          28 u d2 + 2 u A
// A and d2 in these units are A 2^b / (2 s) and that plus F. The factors of the last line are rounded up, for the
// second point's larger d2 and the bound's own rounding. At one point every term is convex in s: between two
// scales the bound is no larger than at one of them.
template <int D>
__host__ __device__ __forceinline__ float tolerance(float sp, float rs, float a, float c0, float b0, float best) {
    using L = ListBound<D>;
    constexpr float U = 5.9604645e-8f, UV = D == 8 ? 0.5f : 0.25f;        // UV = u VMAX
    const float d2 = fmaxf(a * rs + sp * c0 - b0 + best, 0.f);
    return 1.01f * (sp * ((0.5f + 4.f * UV) * L::P2 + 4.f * UV * L::M2) + (L::P1 + 2.f * L::L1)) + U * (32.f * d2 + 4.f * (a * rs + sp * c0));
}

// byte planes of four 24-bit integers
__device__ __forceinline__ void planes(const uint32_t (&n)[4], uint32_t& p0, uint32_t& p1, uint32_t& p2) {
    const uint32_t a = __builtin_amdgcn_perm(n[1], n[0], 0x05010400u), b = __builtin_amdgcn_perm(n[3], n[2], 0x05010400u);
    p0 = __builtin_amdgcn_perm(b, a, 0x05040100u);
    p1 = __builtin_amdgcn_perm(b, a, 0x07060302u);
    const uint32_t c = __builtin_amdgcn_perm(n[1], n[0], 0x0c0c0602u), d = __builtin_amdgcn_perm(n[3], n[2], 0x0c0c0602u);
    p2 = __builtin_amdgcn_perm(d, c, 0x05040100u);
}

// this lane's group as the filter's record; false where the filter does not apply (values that are not
// finite or too large or small for its integers)
template <int D>
__device__ __forceinline__ bool make_record(Record<D>& r, const float (&xval)[D], const float (&v)[D], float max, float last) {
    constexpr int VBITS = D == 8 ? 22 : 21;          // V <= 2^23 (2^22): C fits 32 bits, differences 31
    float vmax = 0, pmax = 0, a = 0, vs = 0, p[D];
#pragma unroll
    for (int i = 0; i < D; ++i) {
        p[i] = v[i] * xval[i];
        vmax = fmaxf(vmax, v[i]);
        pmax = fmaxf(pmax, fabsf(p[i]));
        vs += v[i];
        a += fabsf(p[i] * xval[i]);
    }
    constexpr float HI = 1.15292150e18f, LO = 8.67361738e-19f;       // 2^60, 2^-60
    const bool ok = vmax > LO && pmax > LO && vs < HI && a < HI && pmax < HI;
    const int ev = (int)(__float_as_uint(vmax) >> 23) - 127, ep = (int)(__float_as_uint(pmax) >> 23) - 127;
    const int as = ok ? VBITS - ev : 0, bs = ok ? 22 - ep : 0;
    const float fa = __uint_as_float((uint32_t)(as + 127) << 23), fb = __uint_as_float((uint32_t)(bs + 127) << 23);
    uint32_t w[D / 4][6];
#pragma unroll
    for (int h = 0; h < D / 4; ++h) {
        uint32_t vi[4], pi[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            vi[i] = ok ? (uint32_t)rintf(v[4 * h + i] * fa) : 0u;
            pi[i] = ok ? (uint32_t)(int)__builtin_amdgcn_fmed3f(rintf(p[4 * h + i] * fb), -8388607.f, 8388607.f) : 0u;
        }
        planes(vi, w[h][0], w[h][1], w[h][2]);
        planes(pi, w[h][3], w[h][4], w[h][5]);
    }
    const uint32_t ratio = (uint32_t)(bs - as - 1 + 127) << 23;
    const uint4 meta = make_uint4(__float_as_uint(max), ratio, __float_as_uint(a * fb * 0.5f), __float_as_uint(last));
    if constexpr (D == 8) {
        r.w[0] = make_uint4(w[0][0], w[1][0], w[0][1], w[1][1]);
        r.w[1] = make_uint4(w[0][2], w[1][2], w[0][3], w[1][3]);
        r.w[2] = make_uint4(w[0][4], w[1][4], w[0][5], w[1][5]);
        r.w[3] = meta;
    } else {
        r.w[0] = make_uint4(w[0][0], w[0][1], w[0][2], w[0][3]);
        r.w[1] = make_uint4(w[0][4], w[0][5], 0u, 0u);
        r.w[2] = meta;
    }
    return ok;
}

// C and B of a point, less c0 and b0: a plane's products added to 256 times those of the planes above
template <int D>
__device__ __forceinline__ void sums(const uint32_t (&w)[D == 8 ? 12 : 8], const Point<D>& p, int c0, int b0, int& dc, int& db) {
    constexpr int H = D / 4;
    uint32_t c = 0, b = 0;
#pragma unroll
    for (int k = 2; k >= 0; --k) {
        if (k < 2) c = (c << 8) - (k == 0 ? (uint32_t)c0 : 0u);
        if (k < 2) b = (b << 8) - (k == 0 ? (uint32_t)b0 : 0u);
#pragma unroll
        for (int h = 0; h < H; ++h) {
            c = __builtin_amdgcn_udot4(w[H * k + h], p.s[h], c, false);
            if (k == 2) b = (uint32_t)__builtin_amdgcn_sdot4((int)w[H * (3 + k) + h], (int)p.q[h], (int)b, false);
            else b = __builtin_amdgcn_udot4(w[H * (3 + k) + h], p.q[h], b, false);
        }
    }
    dc = (int)c;
    db = (int)b;
}

// The queue's runs searched, 64 at a time (fewer runs: each list shared by 2, 4 or 8 lanes): a run's list
// is scanned at the scales of its first and last trial (FINAL: at the record's final scale) and its points
// written, EXACT where a lead is too small to be sure of. F is linear in s, so
//   * one point best at both ends is best between them, and the bound is no larger there than the larger of
//     the two;
//   * with point g at the first and h at the last trial, every third point lies above the line between the
//     second best values of the two ends. If that line passes over the crossing of g and h, it is above the
//     better of the two all the way: the trials before the crossing take g, the others h. (The crossing is
//     right to 4 u and the line to 4 u of its ends, together less than three times the bound: four times it
//     are asked for, the bound being the largest of the two ends and the crossing.) If it does not, the two
//     trials at the crossing are searched as well (the run queued again with them): g and h there mean the
//     same; anything else leaves a shorter run on one side to be searched the same way.
// A queue entry: {map entry, lane | first trial << 8 | last << 16 | (trial before the crossing + 1) << 24 | PEELED}.
// `ties`: no importance matrix (see MANY). Returns the trials (as bits) of which some point is left open (EXACT).
template <int K, bool FINAL>
__device__ __forceinline__ uint32_t search_runs(WaveMem<K>& W, int count, bool ties, const Point<Cfg<K>::D>* pts, const uint16_t* __restrict__ nb) {
    constexpr int D = Cfg<K>::D, NS = FINAL ? 1 : 2, R = Cfg<K>::R;
    const int lane = (int)__lane_id();
    uint32_t open = 0;
    int tail = count;
    for (int head = 0, n; head < tail; head += n) {
        n = tmin(64, tail - head);
        const int share = n <= 8 ? 3 : (n <= 16 ? 2 : (n <= 32 ? 1 : 0));
        const int part = lane & ((1 << share) - 1);
        const bool act = (lane >> share) < n;
        const uint2 task = W.queue[(head + (act ? lane >> share : 0)) & (QCAP - 1)];
        const int o = (int)(task.y & 63u), r0 = (int)((task.y >> 8) & 31u), r1 = (int)((task.y >> 16) & 31u);
        const bool inner = (task.y >> 24 & 63u) != 0;     // the two trials at a crossing inside r0 .. r1
        const int t0 = inner ? (int)(task.y >> 24 & 63u) - 1 : r0, t1 = inner ? t0 + 1 : r1;
        const int gi = (int)task.x, np = act ? (list_length(gi) + R - 1) / R : 0;
        const uint16_t* list = nb + list_offset(gi);
        const Piece<R>* pieces = reinterpret_cast<const Piece<R>*>(list);
        const int first = list[0];
        Piece<R> next = pieces[part < np ? part : 0];
        uint32_t r[D == 8 ? 12 : 8];
#pragma unroll
        for (int i = 0; i < (D == 8 ? 3 : 2); ++i) {
            const uint4 v = W.rec[o].w[i];
            r[4 * i] = v.x; r[4 * i + 1] = v.y; r[4 * i + 2] = v.z; r[4 * i + 3] = v.w;
        }
        const uint4 meta = W.rec[o].w[D == 8 ? 3 : 2];
        const float max = __uint_as_float(meta.x), ratio = __uint_as_float(meta.y);
        // s' of trial t: max / num within 4 u (3.04 over all mantissas and trials) of the scale 1 / (num / max)
        auto scaled = [&](int t) __attribute__((always_inline)) {
            const float num = trial_num<K>(t), rn = __builtin_amdgcn_rcpf(num);
            return max * __builtin_fmaf(__builtin_fmaf(-num, rn, 1.f), rn, rn) * ratio;
        };
        float sp[NS], m1[NS], m2[NS];
        int id[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            sp[j] = FINAL ? __uint_as_float(meta.w) * ratio : scaled(j == 0 ? t0 : t1);
            m1[j] = m2[j] = FLT_BIG;
            id[j] = 0;
        }
        int c0, b0;
        sums<D>(r, pts[first], 0, 0, c0, b0);
        for (int p = part; __ballot(p < np); p += 1 << share) {
            if (p < np) {
                const Piece<R> cur = next;
                if (p + (1 << share) < np) next = pieces[p + (1 << share)];
                // the piece's points are all requested before the first is used; past the list's end they are
                // the origin, whose F is that of d2 = A
                int jj[R];
                Point<D> pt[R];
#pragma unroll
                for (int e = 0; e < R; ++e) {
                    jj[e] = (int)((e & 1) ? cur.j[e / 2] >> 16 : cur.j[e / 2] & 0xffffu);
                    pt[e] = pts[jj[e]];
                }
#pragma unroll
                for (int e = 0; e < R; ++e) {
                    int dc, db;
                    sums<D>(r, pt[e], c0, b0, dc, db);
                    const float fc = (float)dc, fb = (float)db;
#pragma unroll
                    for (int k = 0; k < NS; ++k) {
                        const float f = __builtin_fmaf(sp[k], fc, -fb);
                        const bool lt = f < m1[k];
                        id[k] = lt ? jj[e] : id[k];
                        m2[k] = __builtin_amdgcn_fmed3f(f, m1[k], m2[k]);
                        m1[k] = lt ? f : m1[k];
                    }
                }
            }
        }
        for (int st = 1; st < 1 << share; st <<= 1) {
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const float a1 = __shfl_xor(m1[k], st), a2 = __shfl_xor(m2[k], st);
                const int ai = __shfl_xor(id[k], st);
                m2[k] = fminf(fmaxf(m1[k], a1), fminf(m2[k], a2));
                id[k] = a1 < m1[k] ? ai : id[k];
                m1[k] = fminf(m1[k], a1);
            }
        }
        const float fc0 = (float)(uint32_t)c0, fb0 = (float)b0, av = __uint_as_float(meta.z);
        auto bound = [&](float s, float f) __attribute__((always_inline)) {
            return tolerance<D>(s, __builtin_amdgcn_rcpf(s) * ratio, av, fc0, fb0, f);
        };
        float tol = 0;
        bool sure[NS], all = true;
#pragma unroll
        for (int k = 0; k < NS; ++k) tol = fmaxf(tol, bound(sp[k], m1[k]));
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            sure[k] = m2[k] - m1[k] > tol && id[k] < Cfg<K>::PTS;
            all = all && sure[k];
        }
        auto leave_open = [&](int from, int to) __attribute__((always_inline)) {
            for (int t = from; t <= to; ++t) {
                W.point[t][o] = (uint16_t)EXACT;
                open |= 1u << t;
            }
        };
        uint32_t again = 0, more = 0;      // runs to queue again
        const bool many = __popcll(__ballot(act && part == 0 && !all)) > MANY;
        if (act && part == 0) {
            if (!sure[0]) open |= 1u << (FINAL ? 0 : t0);
            if (!sure[NS - 1]) open |= 1u << (FINAL ? 0 : t1);
            const uint32_t g = sure[0] ? (uint32_t)id[0] : EXACT, h = sure[NS - 1] ? (uint32_t)id[NS - 1] : EXACT;
            if constexpr (FINAL) {
                W.point[0][o] = (uint16_t)g;
            } else if (!inner) {
                W.point[t0][o] = (uint16_t)g;
                W.point[t1][o] = (uint16_t)h;
                if (t1 - t0 > 1 && !(all && g == h)) {
                    if (all) {
                        int cg, bg, ch, bh;
                        sums<D>(r, pts[g], c0, b0, cg, bg);
                        sums<D>(r, pts[h], c0, b0, ch, bh);
                        const float dc = (float)(cg - ch), db = (float)(bg - bh);       // g less h: s' dc - db
                        const float sx = db * __builtin_amdgcn_rcpf(dc), k = (sx - sp[1]) * __builtin_amdgcn_rcpf(sp[0] - sp[1]);
                        // the trial from which h is taken (a wrong one fails the tests)
                        const float x = (max * ratio * __builtin_amdgcn_rcpf(sx) - trial_num<K>(0)) * (1.f / Cfg<K>::STEP);
                        const int tx = tmax(t0 + 1, tmin(t1, (int)ceilf(fminf(fmaxf(x, -1.f), 64.f))));
                        const float fx = __builtin_fmaf(sx, (float)cg, -(float)bg);
                        const float over = k * m2[0] + (1.f - k) * m2[1] - fx, tolx = over > 4.f * tol ? fmaxf(tol, bound(sx, fx)) : tol;
                        if (k >= 0.f && k <= 1.f && over > 4.f * tolx &&
                            (tx - 1 == t0 || __builtin_fmaf(scaled(tx - 1), dc, -db) < -tolx) &&
                            (tx == t1 || __builtin_fmaf(scaled(tx), dc, -db) > tolx))
                            W.point[tx][o] = (uint16_t)h;
                        else
                            again = (task.y & 0xffffffu) | ((uint32_t)tx << 24);
                    } else if ((task.y & PEELED && (many || ties)) || (many && !sure[0] && !sure[NS - 1])) {
                        // undecided once more, or at both ends in many lanes: equal distances, which last
                        leave_open(t0, t1);
                    } else {
                        again = (uint32_t)o | ((uint32_t)(t0 + 1) << 8) | ((uint32_t)(t1 - 1) << 16) | PEELED;
                    }
                }
            } else {
                // known at the run's ends: g0 and h0
                const uint32_t g0 = W.point[r0][o], h0 = W.point[r1][o];
                if (t0 > r0) W.point[t0][o] = (uint16_t)g;
                if (t1 < r1) W.point[t1][o] = (uint16_t)h;
                const bool left = t0 - r0 > 1 && g != g0, right = r1 - t1 > 1 && h != h0;
                if (left) again = (uint32_t)o | ((uint32_t)r0 << 8) | ((uint32_t)t0 << 16);
                if (right) more = (uint32_t)o | ((uint32_t)t1 << 8) | ((uint32_t)r1 << 16);
            }
        }
        if constexpr (!FINAL) {
            uint64_t m = __ballot(again != 0);
            if (again != 0) W.queue[(tail + lanes_below(m)) & (QCAP - 1)] = make_uint2(task.x, again);
            tail += __popcll(m);
            m = __ballot(more != 0);
            const bool room = tail + __popcll(m) - (head + n) <= QCAP;
            if (more != 0) {
                if (room) {
                    W.queue[(tail + lanes_below(m)) & (QCAP - 1)] = make_uint2(task.x, more);
                } else {
                    leave_open(t1 + 1, r1 - 1);
                }
            }
            tail += room ? __popcll(m) : 0;
        }
        wave_lds_sync();
    }
    uint32_t every = 0;
    for (uint64_t m = __ballot(open != 0); m; m &= m - 1)
        every |= (uint32_t)__builtin_amdgcn_readlane((int)open, __ffsll((unsigned long long)m) - 1);
    return every;
}

// The queued runs' map entries looked up; those on the grid are done, the others stay queued, the longest
// lists first (four classes), so that the lists scanned side by side are of about one length and the last
// ones are short. Returns how many stay.
template <int K>
__device__ __forceinline__ int sort_runs(WaveMem<K>& W, int count, const int32_t* __restrict__ map) {
    const int lane = (int)__lane_id();
    uint2 task[QCAP / 64];
    int cls[QCAP / 64];
    constexpr int C1 = Cfg<K>::D == 8 ? (K == K_IQ2_S ? 8 : 24) : 6;
#pragma unroll
    for (int k = 0; k < QCAP / 64; ++k) {
        cls[k] = -1;
        if (64 * k + lane < count) {
            task[k] = W.queue[64 * k + lane];
            const int gi = map[task[k].x];
            if (gi >= 0) {
                W.point[(task[k].y >> 8) & 31u][task[k].y & 63u] = (uint16_t)gi;
            } else {
                const int len = list_length(gi);
                cls[k] = len > 3 * C1 ? 3 : (len > 2 * C1 ? 2 : (len > C1 ? 1 : 0));
                task[k].x = (uint32_t)gi;
            }
        }
    }
    wave_lds_sync();
    int n = 0;
    for (int c = 3; c >= 0; --c) {
#pragma unroll
        for (int k = 0; k < QCAP / 64; ++k) {
            const uint64_t m = __ballot(cls[k] == c);
            if (cls[k] == c) W.queue[n + lanes_below(m)] = task[k];
            n += __popcll(m);
        }
    }
    wave_lds_sync();
    return n;
}

// ---------------------------------------------------------------- a sub-block

// |x| and the sign bits of 8 weights; with PARITY an odd count of negatives leaves the least important
// weight's sign flipped (ggml-quants.c:3336-3356); without it (IQ2_S, IQ3_S) all are kept (:4222-4231)
template <bool PARITY>
__device__ __forceinline__ uint32_t make_signs(const float* x, const float* w, float* xval) {
    int nflip = 0;
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if (x[i] >= 0) xval[i] = x[i];
        else { xval[i] = -x[i]; ++nflip; s |= 1u << i; }
    }
    if (PARITY && (nflip % 2)) {
        int imin = 0;
        float mn = w[0] * x[0] * x[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) {
            const float ax = w[i] * x[i] * x[i];
            if (ax < mn) { mn = ax; imin = i; }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i == imin) xval[i] = -xval[i];
        s ^= 1u << imin;
    }
    return s;
}

template <int K>
__device__ __forceinline__ float weight_of(float x, float sigma2, const float* qw, int i) {
    if (qw) return qw[i] * sqrtf(sigma2 + x * x);
    return K == K_IQ2_S ? 0.25f * sigma2 + x * x : x * x;
}

// n = 4 or 8 consecutive weights (see load_weights)
template <int D>
__device__ __forceinline__ void load_group(const void* __restrict__ src, int kind, int64_t e, float (&x)[D]) {
    if constexpr (D == 8) {
        load_weights<8>(src, kind, e, x);
    } else if (kind == SRC_F32) {
        const float4 v = *reinterpret_cast<const float4*>(static_cast<const float*>(src) + e);
        x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    } else {
        const uint2 v = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(src) + e);
        const uint32_t h[4] = {v.x & 0xffffu, v.x >> 16, v.y & 0xffffu, v.y >> 16};
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = kind == SRC_BF16 ? bf16_to_f32(h[i]) : f16_to_f32(h[i]);
    }
}

template <int K>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(3))) void k_lattice(const void* __restrict__ src, int kind, uint8_t* __restrict__ dst, int64_t nsb,
                                                int64_t sbpr, const float* __restrict__ imx, IqDeviceTable tab) {
    using C = Cfg<K>;
    constexpr int D = C::D, N = C::N, T = C::T, G = 256 / N, SBW = WG / G, NG = N / D, KMAXQ = C::KMAXQ;
    __shared__ Point<D> pts[C::PTS + 1];          // the point after the last: the origin
    __shared__ __align__(16) uint16_t otile[SBW * C::BS / 2];
    __shared__ __align__(16) WaveMem<K> mem[WG / 64];
    for (int i = threadIdx.x; i < C::PTS * D / 4; i += WG) {
        const uint32_t q = reinterpret_cast<const uint32_t*>(tab.grid)[i];
        uint32_t s = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) { const uint32_t l = (q >> (8 * b)) & 0xff; s |= (l * l) << (8 * b); }
        pts[i / (D / 4)].q[i % (D / 4)] = q;
        pts[i / (D / 4)].s[i % (D / 4)] = s;
    }
    if (threadIdx.x == 0) pts[C::PTS] = Point<D>{};
    for (int i = threadIdx.x; i < SBW * C::BS / 2; i += WG) otile[i] = 0;
    __syncthreads();
    WaveMem<K>& W = mem[threadIdx.x / 64];
    const int lane = (int)__lane_id();
    const int lsb = threadIdx.x / G, sub = threadIdx.x % G;
    const int64_t sb0 = (int64_t)blockIdx.x * SBW;
    const int64_t sb = sb0 + lsb;
    const bool active = sb < nsb;
    const int64_t sbc = active ? sb : nsb - 1;
    const int64_t e0 = sbc * 256 + sub * N;
    const float* qw = imx ? imx + (sbc % sbpr) * 256 + sub * N : nullptr;

    // ---- the sub-block's scale of search, its signs
    float sigma2, max, amax = 0, scale;
    uint32_t sg[N / 8];
    bool finite;
    {
        float x[N], w[N], xval[N];
        load_weights<N>(src, kind, e0, x);
        // the super-block's sum of squares, left to right, handed from lane to lane of the group
        float sumx2 = 0.f;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (sub == g) {
#pragma unroll
                for (int i = 0; i < N; ++i) sumx2 += x[i] * x[i];
            }
            sumx2 = __shfl(sumx2, g, G);
        }
        sigma2 = C::TWO ? 2 * sumx2 / 256 : sumx2 / 256;
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = weight_of<K>(x[i], sigma2, qw, i);
#pragma unroll
        for (int k = 0; k < N / 8; ++k) sg[k] = make_signs<C::PARITY>(x + 8 * k, w + 8 * k, xval + 8 * k);
        max = xval[0];
#pragma unroll
        for (int i = 1; i < N; ++i) max = tmax(max, xval[i]);
#pragma unroll
        for (int i = 0; i < N; ++i) amax = tmax(amax, fabsf(x[i]));
        finite = !not_finite<N>(x);
        scale = max / (float)(2 * KMAXQ - 1);
        if constexpr (K == K_IQ2_XXS) {
            int Lq[N];     // make_qp_quants' levels never reach the output: scale > 0 below refits every group
            scale = make_qp_quants<N>(KMAXQ + 1, xval, Lq, w);
        }
    }
    bool live = C::EPS == 0.f ? !(max == 0.f) : !(max < C::EPS);
    if constexpr (K == K_IQ2_XXS) {
        max = scale * KMAXQ;          // the reference's eff_max
        live = live && max > 0;       // its early exits leave the sub-block empty
    }
    // plain: the float rounding and the filter apply (finite, max within 2^+-60, |x| / max < 2^12)
    const bool plain = finite && max > 8.67361738e-19f && max < 1.15292150e18f && amax < 4096.f * max;
    const bool odd = live && !plain;
    const bool any_odd = __ballot(odd) != 0;
    const float rmax = 1.f / max;

    // group k's weights: x as searched, v = sqrt(w)
    auto group = [&](int k, float (&xval)[D], float (&w)[D], float (&v)[D]) __attribute__((always_inline)) {
        float x[D];
        load_group<D>(src, kind, e0 + D * k, x);
        const float* q = qw ? qw + D * k : nullptr;
        uint32_t s = sg[0];
#pragma unroll
        for (int j = 1; j < N / 8; ++j)
            if (k * D / 8 == j) s = sg[j];
        if (D == 4 && (k & 1)) s >>= 4;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            w[i] = weight_of<K>(x[i], sigma2, q, i);
            v[i] = sqrtf(w[i]);
            // |x|, negated where the stored sign is not x's own
            const bool neg = !(x[i] >= 0);
            const float ax = neg ? -x[i] : x[i];
            xval[i] = neg == (bool)((s >> i) & 1) ? ax : -ax;
        }
    };
    auto round_at = [&](const float (&xval)[D], float id) __attribute__((always_inline)) {
        return any_odd ? round_exact<D, KMAXQ>(xval, id) : round_float<D, KMAXQ>(xval, id);
    };
    auto id_at = [&](int t, float m, float rm) { return any_odd ? trial_num<K>(t) / m : trial_id<K>(t, m, rm); };
    // the points still open (EXACT) of trial t at scale s
    auto settle = [&](bool last, int t, const float (&xval)[D], const float (&v)[D], float s, int u) __attribute__((always_inline)) {
        const bool off = W.point[t][lane] == EXACT;
        uint64_t m = __ballot(off);
        if (!m) return;
        const int gi = tab.map[u];
        if (last && __popcll(m) > FEW) {
            dealt_neighbours<K, 1>(W, 0, off ? 1u : 0u, xval, v, max, s, gi, pts, tab.nb);
            return;
        }
        for (; m; m &= m - 1) {
            const int o = __ffsll((unsigned long long)m) - 1;
            const int j = exact_neighbour<D>(xval, v, s, gi, o, pts, tab.nb);
            if (lane == o) W.point[t][lane] = (uint16_t)j;
        }
        wave_lds_sync();
    };

    // ---- every trial's sums, a group at a time (element order within each trial)
    float sx[T], s2[T];
#pragma unroll
    for (int t = 0; t < T; ++t) { sx[t] = 0; s2[t] = 0; }
    for (int k = 0; k < NG; ++k) {
        float xval[D], w[D], v[D];
        group(k, xval, w, v);
        const bool filter = make_record<D>(W.rec[lane], xval, v, max, 0.f) && plain && live;
        const bool by_hand = live && !filter;
        const bool any_by_hand = __ballot(by_hand) != 0;
#pragma unroll
        for (int t = 0; t < T; ++t) W.point[t][lane] = (uint16_t)PREV;
        wave_lds_sync();
        if (any_by_hand) {
            for (int t = 0; t < T; ++t) {
                const int gi = tab.map[by_hand ? round_at(xval, id_at(t, max, rmax)) : 0];
                if (by_hand) W.point[t][lane] = (uint16_t)(gi >= 0 ? (uint32_t)gi : EXACT);
            }
        }
        uint32_t open = any_by_hand ? ~0u >> (32 - T) : 0u;
        const uint32_t starts = filter ? level_changes<K>(xval, max, rmax) : ~0u;      // of runs of one rounding
        int n = 0;
        for (uint32_t left = filter ? starts : 0u; __ballot(left != 0); ) {
            const int from = __ffs((int)left) - 1, to = (left & (left - 1)) ? __ffs((int)(left & (left - 1))) - 2 : T - 1;
            const int u = round_float<D, KMAXQ>(xval, trial_id<K>(from, max, rmax));
            const uint64_t m = __ballot(left != 0);
            if (left != 0) W.queue[n + lanes_below(m)] = make_uint2((uint32_t)u, (uint32_t)lane | ((uint32_t)from << 8) | ((uint32_t)to << 16));
            n += __popcll(m);
            left &= left - 1;
            if (n > QCAP - 64 || !__ballot(left != 0)) {
                wave_lds_sync();
                n = sort_runs<K>(W, n, tab.map);
                open |= search_runs<K, false>(W, n, !imx, pts, tab.nb);
                n = 0;
            }
        }
        uint32_t mine = 0;
        for (uint32_t m = open; m; m &= m - 1) {
            const int t = __ffs((int)m) - 1;
            mine |= W.point[t][lane] == EXACT ? 1u << t : 0u;
        }
        if (__popcll(__ballot(mine != 0)) > FEW || __popc(open) > FEW_TRIALS) {
            // up to four trials of a run at once
            while (__ballot(mine != 0)) {
                const int t = mine ? __ffs((int)mine) - 1 : 0;
                const uint32_t later = starts & ~1u << t, run = later ? (later & (0u - later)) - 1 : ~0u;     // before the next run
                const uint32_t now = mine & run & 15u << t;
                const int gi = tab.map[round_at(xval, id_at(t, max, rmax))];
                dealt_neighbours<K, 4>(W, t, now >> t, xval, v, max, 0.f, gi, pts, tab.nb);
                mine &= ~now;
            }
        } else {
            for (; open; open &= open - 1) {
                const int t = __ffs((int)open) - 1;
                const float id = id_at(t, max, rmax);
                settle(false, t, xval, v, 1 / id, round_at(xval, id));
            }
        }
        float wx[D];
#pragma unroll
        for (int i = 0; i < D; ++i) wx[i] = w[i] * xval[i];
        int cur = 0;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int p = W.point[t][lane];
            cur = p == (int)PREV ? cur : p;
            float q[D];
            coords<D>(pts[cur], q);
#pragma unroll
            for (int i = 0; i < D; ++i) {
                sx[t] += wx[i] * q[i];
                s2[t] += w[i] * q[i] * q[i];
            }
        }
        wave_lds_sync();
    }
    // ---- the best trial (ggml-quants.c:3391-3400, :3583-3592, :4058-4067)
    float best = 0;
    int bt = -1;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        if (s2[t] > 0 && sx[t] * sx[t] > best * s2[t]) {
            scale = sx[t] / s2[t];
            best = scale * sx[t];
            bt = t;
        }
    }
    // ---- its groups on the grid keep their points; the others (ALL: every group, if one is off) are
    // rounded and searched again at the best scale, and the scale is refitted (:3411-3432, :3595-3616,
    // :4070-4086)
    uint32_t on = 0;
    const float bid = bt >= 0 ? id_at(bt, max, rmax) : 0.f;
    for (int k = 0; k < NG; ++k) {
        float xval[D], w[D], v[D];
        group(k, xval, w, v);
        const int gi = tab.map[bt >= 0 ? round_at(xval, bid) : 0];
        if (bt >= 0 ? gi >= 0 : C::ON0) on |= 1u << k;
        W.best[k][lane] = (uint16_t)(gi >= 0 ? gi : 0);
    }
    constexpr uint32_t EVERY = (1u << NG) - 1;
    const bool some_off = K == K_IQ2_XXS || on != EVERY;
    const bool refit = live && some_off && scale > 0;
    const float id = 1 / scale;
    float sumqx = 0, sumq2 = 0;
    for (int k = 0; k < NG; ++k) {
        float xval[D], w[D], v[D];
        group(k, xval, w, v);
        const bool redo = refit && (C::ALL || !((on >> k) & 1));
        // (a group off the grid at the best trial with scale <= 0 keeps that trial's neighbour)
        const bool keep_off = live && !refit && !((on >> k) & 1) && bt >= 0;
        const int u = redo ? round_exact<D, KMAXQ>(xval, id) : (keep_off ? round_exact<D, KMAXQ>(xval, bid) : 0);
        const int gi = tab.map[u];
        const bool off = (redo || keep_off) && gi < 0;
        const bool filter = make_record<D>(W.rec[lane], xval, v, max, scale) && plain && redo;
        W.point[0][lane] = (uint16_t)(off ? EXACT : (uint32_t)(redo ? gi : (int)W.best[k][lane]));
        const uint64_t m = __ballot(off && filter);
        if (off && filter) W.queue[lanes_below(m)] = make_uint2((uint32_t)u, (uint32_t)lane);
        wave_lds_sync();
        const int n = sort_runs<K>(W, __popcll(m), tab.map);
        search_runs<K, true>(W, n, !imx, pts, tab.nb);
        settle(true, 0, xval, v, redo ? scale : 1 / bid, u);
        const int p = W.point[0][lane];
        W.best[k][lane] = (uint16_t)p;
        float q[D];
        coords<D>(pts[p], q);
#pragma unroll
        for (int i = 0; i < D; ++i) {
            sumqx += w[i] * xval[i] * q[i];
            sumq2 += w[i] * q[i] * q[i];
        }
        wave_lds_sync();
    }
    if (refit && sumq2 > 0) scale = sumqx / sumq2;
    const bool empty = !live;
    uint32_t sgn[N / 8];
#pragma unroll
    for (int k = 0; k < N / 8; ++k) {
        sgn[k] = sg[k];
        if (scale < 0) sgn[k] = ~sgn[k];
        sgn[k] = empty ? 0u : sgn[k] & (C::PARITY ? 127u : 255u);
    }
    if (scale < 0) scale = -scale;

    // ---- the super-block's scale: the largest of its sub-blocks (empty ones count as 0), 4-bit steps
    const float s_own = empty ? 0.f : scale;
    float max_scale = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) max_scale = tmax(max_scale, __shfl(s_own, g, G));
    const bool nz = max_scale != 0.f;   // the reference's `if (!max_scale)` exit
    const float d = max_scale / 31.f;
    int l = 0;
    if (nz) {
        const float ids = 1 / d;
        l = tmax(0, tmin(15, nearest_int(0.5f * (ids * s_own - 1))));
    }
    uint32_t gx[NG];
#pragma unroll
    for (int k = 0; k < NG; ++k) gx[k] = empty ? 0u : (uint32_t)W.best[k][lane];

    // ---- the block's bytes, each lane its sub-block's (the tile starts as zeros)
    TileOut o{otile + lsb * (C::BS / 2)};
    if (nz && sub == 0) o.put16(0, f32_to_f16(K == K_IQ2_XXS || K == K_IQ2_XS ? d : d * C::DSCALE));
    // the scale codes of four sub-blocks as one u16, in the first of them
    const uint32_t l4 = (uint32_t)l | ((uint32_t)__shfl_down(l, 1, G) << 4) | ((uint32_t)__shfl_down(l, 2, G) << 8) |
                        ((uint32_t)__shfl_down(l, 3, G) << 12);
    if constexpr (K == K_IQ2_XXS) {
        // d, then per 32 weights: u32 of 4 grid indices, u32 of 4 x 7 sign bits | scale << 28
        if (nz) {
            o.put4(2 + 8 * sub, gx[0] | (gx[1] << 8) | (gx[2] << 16) | (gx[3] << 24));
            o.put4(6 + 8 * sub, sgn[0] | (sgn[1] << 7) | (sgn[2] << 14) | (sgn[3] << 21) | ((uint32_t)l << 28));
        }
    } else if constexpr (K == K_IQ2_XS) {
        // d, per 16 weights two u16 (9-bit grid index | 7 sign bits << 9), scale nibbles
        if (nz) {
            o.put16(2 + 4 * sub, gx[0] | (sgn[0] << 9));
            o.put16(4 + 4 * sub, gx[1] | (sgn[1] << 9));
            if (sub % 4 == 0) o.put16(66 + sub / 2, l4);
        }
    } else if constexpr (K == K_IQ2_S) {
        // d, qs[32] grid low bytes, qs[32] signs, qh[8] (2 high bits per group), scales[8]
        o.put2(2 + 2 * sub, gx[0] & 255, gx[1] & 255);
        o.put2(34 + 2 * sub, sgn[0], sgn[1]);
        const uint32_t h = (gx[0] >> 8) | ((gx[1] >> 8) << 2);
        const uint32_t h4 = h | ((uint32_t)__shfl_down((int)h, 1, G) << 4) | ((uint32_t)__shfl_down((int)h, 2, G) << 8) |
                            ((uint32_t)__shfl_down((int)h, 3, G) << 12);
        if (sub % 4 == 0) o.put16(66 + sub / 2, h4);
        if (nz && sub % 4 == 0) o.put16(74 + sub / 2, l4);
    } else if constexpr (K == K_IQ3_XXS) {
        // d, 64 grid indices, per 32 weights u32 of 4 x 7 sign bits | scale << 28
        if (nz) {
#pragma unroll
            for (int k = 0; k < 8; k += 2) o.put2(2 + 8 * sub + k, gx[k], gx[k + 1]);
            o.put4(66 + 4 * sub, sgn[0] | (sgn[1] << 7) | (sgn[2] << 14) | (sgn[3] << 21) | ((uint32_t)l << 28));
        }
    } else {
        // d, qs[64], qh[8], signs[32], scales[4]. The reference advances its qs and signs cursors only
        // past sub-blocks that were not empty (ggml-quants.c:4336-4339 sit after the `continue` of
        // :4237), so later sub-blocks land in the earlier free slots; qh is indexed by position.
        const uint32_t full = (uint32_t)((uint64_t)__ballot(!empty) >> (lane & ~(G - 1))) & ((1u << G) - 1);
        const int slot = __popc(full & ((1u << sub) - 1));
        uint32_t h = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) h |= (gx[k] >> 8) << k;
        if (!empty) {
#pragma unroll
            for (int k = 0; k < 8; k += 2) o.put2(2 + 8 * slot + k, gx[k] & 255, gx[k + 1] & 255);
            o.put2(74 + 4 * slot, sgn[0], sgn[1]);
            o.put2(76 + 4 * slot, sgn[2], sgn[3]);
        }
        const uint32_t h2 = h | ((uint32_t)__shfl_down((int)h, 1, G) << 8);
        if (sub % 2 == 0) o.put16(66 + sub, h2);
        if (nz && sub % 4 == 0) o.put16(106 + sub / 2, l4);
    }
    __syncthreads();
    const int nb = (int)(nsb - sb0 < SBW ? nsb - sb0 : SBW);
    store_tile(otile, dst + sb0 * C::BS, nb * C::BS);
}

template <int K>
int run(const QuantArgs& a, int table) {
    IqDeviceTable tab;
    if (int e = iq_device_table(table, &tab, a.stream)) return e;
    using C = Cfg<K>;
    if (tab.size != C::PTS)
        return fail(SPA_ERR_ASSERT, "lattice i-quant type %d: codebook of %d points does not fit the kernel", a.type, tab.size);
    if (a.n_per_row % 256) return fail(SPA_ERR_ARG, "lattice i-quant type %d: n_per_row %% 256", a.type);
    const int64_t nsb = a.nrows * a.n_per_row / 256;
    if (nsb == 0) return 0;
    constexpr int SBW = WG / (256 / C::N);
    hipLaunchKernelGGL(k_lattice<K>, dim3((unsigned)((nsb + SBW - 1) / SBW)), dim3(WG), 0, a.stream, a.src, a.src_kind,
                       (uint8_t*)a.dst, nsb, a.n_per_row / 256, a.imatrix, tab);
    SPA_HIP_TRY(hipGetLastError());
    return 0;
}

// fn(std::integral_constant<int, K>) of a type's kind; false for other types
template <class F>
bool with_kind(int type, F fn) {
    switch (type) {
        case 16: fn(std::integral_constant<int, K_IQ2_XXS>()); return true;
        case 17: fn(std::integral_constant<int, K_IQ2_XS>()); return true;
        case 22: fn(std::integral_constant<int, K_IQ2_S>()); return true;
        case 18: fn(std::integral_constant<int, K_IQ3_XXS>()); return true;
        case 21: fn(std::integral_constant<int, K_IQ3_S>()); return true;
    }
    return false;
}

}  // namespace

int launch_lattice(const QuantArgs& a) {
    const int t = iq_table_index(a.type);
    int e = SPA_OK;
    if (!with_kind(a.type, [&](auto k) { e = run<decltype(k)::value>(a, t); }))
        return fail(SPA_ERR_TYPE, "launch_lattice: type %d", a.type);
    return e;
}

}  // namespace spa

extern "C" int spa_lattice_trials_host(int type, int trial, const float* max, int64_t n, float* id) {
    if (n < 0 || (n > 0 && (!max || !id))) return spa::fail(SPA_ERR_ARG, "spa_lattice_trials_host: null or negative");
    bool in_range = false;
    const bool known = spa::with_kind(type, [&](auto k) {
        constexpr int K = decltype(k)::value;
        in_range = trial >= 0 && trial < spa::Cfg<K>::T;
        for (int64_t i = 0; in_range && i < n; ++i) id[i] = spa::trial_id<K>(trial, max[i], 1.f / max[i]);
    });
    if (!known) return spa::fail(SPA_ERR_TYPE, "spa_lattice_trials_host: type %d", type);
    return in_range ? SPA_OK : spa::fail(SPA_ERR_ARG, "spa_lattice_trials_host: trial %d", trial);
}

extern "C" int spa_lattice_bound_host(int type, const float* f, float* out) {
    if (!f || !out) return spa::fail(SPA_ERR_ARG, "spa_lattice_bound_host: null");
    const bool known = spa::with_kind(type, [&](auto k) {
        constexpr int D = spa::Cfg<decltype(k)::value>::D;
        using L = spa::ListBound<D>;
        out[0] = spa::tolerance<D>(f[0], f[1], f[2], f[3], f[4], f[5]);
        out[1] = L::L1; out[2] = L::M2; out[3] = L::P1; out[4] = L::P2;
    });
    return known ? SPA_OK : spa::fail(SPA_ERR_TYPE, "spa_lattice_bound_host: type %d", type);
}
