// hvc_oct64.hip.h -- FP64 steppers with eight lanes per neuron (an octet).
//
// One network leaves most SIMDs with one wave or none, so a window takes as
// long as one wave's instruction stream: a wave alone on its SIMD issues an
// instruction of any kind (vector, scalar, s_nop) every ~4.3 cycles and a
// dependent FP64 operation every 8.4 (measured on gfx950).  What shortens a
// step is therefore fewer instructions per lane.  An octet spreads a neuron's
// state variables over its lanes -- each lane evaluates one gate, one
// derivative and one stage combination -- and the arithmetic is written so
// that all lanes run one branch-free stream with per-lane constants:
//
//  * quotients by constants take two operations (cdiv2), quotients by values
//    eight (div_inrange) instead of the IEEE sequence's eleven;
//  * exp reads its table from LDS and needs no clamping;
//  * one range test per step instead of one per quotient (StepRange).  A step
//    whose values leave the range is repeated from the saved state in the
//    EXACT form, which uses IEEE division and the clamped exp.
//
// Instructions per step and wave: HVC-I 1 350 (2 400 before, in 96 pieces
// between lane-dependent branches), HVC-RA Debraband 640 (one thread per
// neuron 5 600).  k_integrate per window, before and now: Debraband 100 -> 41
// us at 300 + 30 neurons and 99 -> 42 us at 5 003 + 1 377, RK4 67 -> 42 us at
// 2 000 + 550.  Now the HVC-I wave sets the window; its instructions take 5.2
// cycles each on average.
//
// Every value is the reference's expression tree (HH2_test.cpp:613-754,
// HH2_buffer.cpp:741-874, HHI_buffer.cpp:426-691), so results equal the
// one-thread steppers bit for bit.  Where a lane's form differs from the
// tree it only adds a zero, multiplies by one or changes the sign of a zero
// that is then added to a value.
#pragma once
#ifndef HVC_FP32

namespace hvc {
inline namespace p64 {

// lane LO of the quad of x in an octet's lanes 0-3, lane HI of the quad of y in
// its lanes 4-7 (the second move writes the odd banks of four lanes only)
template <int LO, int HI>
__device__ __forceinline__ double half_bcast(double x, double y)
{
    const long long a = __double_as_longlong(x), b = __double_as_longlong(y);
    int lo = __builtin_amdgcn_mov_dpp((int)a, LO * 0x55, 0xF, 0xF, true);
    int hi = __builtin_amdgcn_mov_dpp((int)(a >> 32), LO * 0x55, 0xF, 0xF, true);
    lo = __builtin_amdgcn_update_dpp(lo, (int)b, HI * 0x55, 0xF, 0xA, false);
    hi = __builtin_amdgcn_update_dpp(hi, (int)(b >> 32), HI * 0x55, 0xF, 0xA, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// keeps a value computed in every lane: a select between lanes otherwise
// becomes a branch around the value, which splits the stage into pieces that
// the scheduler cannot interleave
__device__ __forceinline__ void every_lane(double& x) { asm volatile("" : "+v"(x)); }

// the exp table in LDS: entry j = 2^(j/64) as a double-double
typedef double ExpPair __attribute__((ext_vector_type(2)));
constexpr int kExpTabBytes = 64 * (int)sizeof(ExpPair);

// one entry per thread (blocks of 64 threads or more)
__device__ __forceinline__ ExpPair exp_table_load()
{
    const double* e = kExp2Table + 2 * (threadIdx.x & 63);
    return ExpPair{e[0], e[1]};
}
__device__ __forceinline__ void exp_table_store(ExpPair* tab, ExpPair v) { tab[threadIdx.x & 63] = v; }

// dexp for |x| <= 700 (no clamp needed, results normal): the same operations
__device__ __forceinline__ double exp_inrange(double x, const ExpPair* tab)
{
    const double kd = __builtin_rint(x * HVC_INV_LN2_64);
    const int k = (int)kd;
    const ExpPair t = tab[k & 63];
    double r = __builtin_fma(-kd, HVC_LN2_64_HI, x);
    r = __builtin_fma(-kd, HVC_LN2_64_LO, r);
    const double z = r * r;
    double p = __builtin_fma(r, 1.0 / 720.0, 1.0 / 120.0);
    p = __builtin_fma(r, p, 1.0 / 24.0);
    p = __builtin_fma(r, p, 1.0 / 6.0);
    p = __builtin_fma(r, p, 0.5);
    p = __builtin_fma(z, p, r);
    const double y = t.x + __builtin_fma(t.x, p, t.y);
    return __builtin_ldexp(y, k >> 6);
}

// n / d for 2^-600 <= |d| <= 2^600 and n = 0 or 2^-400 <= |n| <= 2^400:
// Newton's iteration from the hardware reciprocal, then Markstein's final
// correction -- the IEEE sequence without its scaling and special-case steps,
// which change nothing in this range
__device__ __forceinline__ double div_inrange(double n, double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-d, q, n), y, q);
}

// What a step notes of its values: it holds for EXACT = false steps only.
// Stage voltages (summed, so one huge value or a NaN fails) bounded by 2000
// keep every gate's exponential in [2^-600, 2^600] and its quotient in range;
// stage derivatives k in [2^-800, 2^500] keep every quotient of a
// combination in cdiv2's range.  A derivative that is exactly zero fails the
// test too: rare, and the repeated step gives the same bits.
struct StepRange {
    double v = 0.0, k = 0.0, kmin = 1.0;
    __device__ __forceinline__ void volt(double x) { v += __builtin_fabs(x); }
    __device__ __forceinline__ void deriv(double x)
    {
        k += __builtin_fabs(x);
        least(x);
    }
    // kmin = min(kmin, |x|) in one instruction (fmin would first quieten its
    // operands; a NaN is caught by the sums)
    __device__ __forceinline__ void least(double x) { asm("v_min_f64 %0, %0, |%1|" : "+v"(kmin) : "v"(x)); }
    __device__ __forceinline__ bool failed() const { return !(v < 2000.0) || !(k < 0x1p500) || !(kmin > 0x1p-800); }
};

template <bool EXACT>
__device__ __forceinline__ double qdiv(double n, double d)
{
    return EXACT ? n / d : div_inrange(n, d);
}
// a / B, B a literal
template <bool EXACT>
__device__ __forceinline__ double qconst(double a, double B)
{
    return EXACT ? a / B : ::hvc::cdiv2(a, B);
}

template <bool EXACT>
__device__ __forceinline__ double qlane(double a, const LaneDiv& d)
{
    return EXACT ? a / d.B : ::hvc::cdiv_lane(a, d);
}

// ---------------------------------------------------------------------------
// HVC-I, DP8: lane 0 owns V, lanes 1-3 own n, m, h and evaluate an, am, ah,
// lane 7 owns w and evaluates wInf.  Lanes 4-6 evaluate bh, bm, bn for their
// mirror lanes; as their own variable they carry 1 - h, 1 - m, 1 - n, whose
// opening and closing rates are h's, m's and n's exchanged (they come for
// free and are not stored).  Every lane's derivative but V's is
// r (1 + cx x) - b x with the mirror lane's rate b: cx = -1 for the gates; for
// w, cx = 0 and b = 1 (lane 0's rate), which is wInf - w exactly.
// ---------------------------------------------------------------------------
struct IOctConst {
    double d;               // rate = fma(cA, v + d, cC) / fma(sg, E, 1) * fma(cB, E, sB),
    LaneDiv e;              // E = exp((v + d) / e), e negative
    double cA, cC, sg, cB, sB;
    double cx;
};
// the gates of kIOctGates: type 0 (A), 1 (B) or 2 (C), c, d, e
constexpr IOctConst i_oct_const(int type, double c, double d, double e, double cx = -1.0)
{
    return IOctConst{d, lane_div(-e), type == 0 ? c : 0.0, type == 0 ? 0.0 : (type == 2 ? c : 1.0),
                     type == 0 ? -1.0 : (type == 1 ? 0.0 : 1.0), type == 1 ? c : 0.0, type == 1 ? 0.0 : 1.0, cx};
}
static __constant__ IOctConst kIOctConsts[8] = {
    IOctConst{0.0, lane_div(-10.0), 0.0, 1.0, 0.0, 0.0, 1.0, -1.0},   // V: rate 1
    i_oct_const(0, 0.15, 15.0, 10.0), i_oct_const(0, 1.0, 22.0, 10.0), i_oct_const(1, 0.7, 34.0, 20.0),
    i_oct_const(2, 10.0, 4.0, 10.0), i_oct_const(1, 40.0, 47.0, 18.0), i_oct_const(1, 0.2, 25.0, 80.0),
    i_oct_const(2, 1.0, 0.0, 5.0, 0.0)};
struct IOctLane : IOctConst {
    int q;
    const ExpPair* tab;
};

// (a lane's constants come from memory with its state: as selects among
// literals they became a tree of branches)
__device__ __forceinline__ IOctLane i_oct_lane(int q, const ExpPair* tab)
{
    IOctLane L;
    (IOctConst&)L = kIOctConsts[q];
    L.q = q;
    L.tab = tab;
    return L;
}

template <bool EXACT>
__device__ __forceinline__ double i_oct_rate(const IOctLane& L, double v)
{
    const double vd = v + L.d;
    if constexpr (EXACT) {
        const GateSlot& g = kIOctGates[L.q];
        const double E = dexp(-vd / g.e);
        const double num = g.type == 0 ? g.c * vd : g.c;
        const double den = g.type == 0 ? 1 - E : 1 + E;
        return g.type == 1 ? g.c * E : num / den;
    } else {
        const double E = exp_inrange(qlane<false>(vd, L.e), L.tab);
        const double q = div_inrange(__builtin_fma(L.cA, vd, L.cC), __builtin_fma(L.sg, E, 1.0));
        return q * __builtin_fma(L.cB, E, L.sB);
    }
}

// derivative of the lane's variable xo at stage voltage v; n1, m1, h1, w1 are
// the neuron's other variables in lane 0
template <bool EXACT>
__device__ __forceinline__ double i_oct_deriv(StepRange& rg, const IOctLane& L, double Ge, double Gi, double v,
                                              double n1, double m1, double h1, double w1, double xo, double e2,
                                              double e5)
{
    const double r = i_oct_rate<EXACT>(L, v);
    const double n4 = n1 * n1 * n1 * n1;
    const double m3 = m1 * m1 * m1;
    const double vk = v - kI_Ek;
    double kV = -kI_gL * (v - kI_El) - kI_gNa * h1 * m3 * (v - kI_Ena) - kI_gKdr * n4 * vk - kI_gKHT * w1 * vk -
                      (Ge * e2) * v - (Gi * e5) * (v - kI_Ei);
    const double b = oct_mirror(r);
    double k;
    if constexpr (EXACT) {
        k = L.q == 0 ? kV : (L.q == 7 ? r - xo : r * (1 - xo) - b * xo);
    } else {
        double kg = r * __builtin_fma(L.cx, xo, 1.0) - b * xo;
        every_lane(kV);
        every_lane(kg);
        k = L.q == 0 ? kV : kg;
    }
    if constexpr (!EXACT) {
        rg.volt(v);
        rg.deriv(k);
    }
    return k;
}

// numerators and divisors of the DP8 tableau (HHI_buffer.cpp:426-691), stages
// 7-12 and the final combination in the order of their terms
constexpr int kDp8Terms = 47;
constexpr double kDp8N[kDp8Terms] = {
    29443841.0, 77736538.0, 28693883.0, 23124283.0, 16016141.0, 61564180.0, 22789713.0, 545815736.0,
    180193667.0, 39632708.0, 433636366.0, 421739975.0, 100302831.0, 790204164.0, 800635310.0, 246121993.0,
    37695042795.0, 309121744.0, 12992083.0, 6005943493.0, 393006217.0, 123872331.0, -1028468189.0,
    8478235783.0, 1311729495.0, 10304129995.0, 48777925059.0, 15336726248.0, 45442868181.0, 3065993473.0,
    185892177.0, 3185094517.0, 477755414.0, 703635378.0, 5731566787.0, 5232866602.0, 4093664535.0,
    3962137247.0, 65686358.0, 13451932.0, 808719846.0, 1757004468.0, 656045339.0, 3867574721.0, 465885868.0,
    53011238.0, 2.0};
constexpr double kDp8D[kDp8Terms] = {
    614563906.0, 692538347.0, 1125000000.0, 1800000000.0, 946692911.0, 158732637.0, 633445777.0, 2771057229.0,
    1043307555.0, 573591083.0, 683701615.0, 2616292301.0, 723423059.0, 839813087.0, 3783071287.0,
    1340847787.0, 15268766246.0, 1061227803.0, 490766935.0, 2108947869.0, 1396673457.0, 1001029789.0,
    846180014.0, 508512852.0, 1432422823.0, 1701304382.0, 3047939560.0, 1032824649.0, 3398467696.0,
    597172653.0, 718116043.0, 667107341.0, 1098053517.0, 230739211.0, 1027545527.0, 850066563.0, 808688257.0,
    1805957418.0, 487910083.0, 455176623.0, 976000145.0, 5645159321.0, 265891186.0, 1518517206.0, 322736535.0,
    667516719.0, 45.0};

// A term is RN(RN(n k) / d): cdiv2 with its small product taken from k itself,
// k RN(n Yl) instead of RN(n k) Yl, which starts the sum one operation earlier.
// The roundings of n Yl and of n k move the sum by another 2^-106 |q| each, four
// such terms in all: 2^-104 |q|, under 2^-51 ulp, against ulp / (4 d_odd) to a
// rounding boundary.  So the divisors' odd parts must stay below 2^49, and are
// below 2^34.  Three constants a term: what
// the compiler would otherwise build from two scalar moves each at every use
// (227 of a step's 1 490 instructions), the first kDp8Pinned terms keep in
// vector registers (the count that leaves two waves to a SIMD).
constexpr bool dp8_divisors_below(double limit)
{
    for (double d : kDp8D)
        if (!(d < limit)) return false;
    return true;
}
static_assert(dp8_divisors_below(0x1p49), "dp8_term's error bound");
constexpr int kDp8Pinned = 21;
struct Dp8Consts {
    double n[kDp8Pinned], hi[kDp8Pinned], lo[kDp8Pinned];
};
template <int J>
__device__ __forceinline__ void dp8_literals(double& n, double& hi, double& lo)
{
    n = kDp8N[J];
    hi = 1.0 / kDp8D[J];
    lo = kDp8N[J] * (__builtin_fma(-kDp8D[J], 1.0 / kDp8D[J], 1.0) / kDp8D[J]);
}
template <int J = 0>
__device__ __forceinline__ void dp8_pin(Dp8Consts& c)
{
    if constexpr (J < kDp8Pinned) {
        dp8_literals<J>(c.n[J], c.hi[J], c.lo[J]);
        asm volatile("" : "+v"(c.n[J]), "+v"(c.hi[J]), "+v"(c.lo[J]));
        dp8_pin<J + 1>(c);
    }
}
template <int J, bool EXACT>
__device__ __forceinline__ double dp8_term(const Dp8Consts& c, double k)
{
    if constexpr (EXACT) {
        return (kDp8N[J] * k) / kDp8D[J];
    } else {
        double n, hi, lo;
        if constexpr (J < kDp8Pinned) {
            n = c.n[J];
            hi = c.hi[J];
            lo = c.lo[J];
        } else {
            dp8_literals<J>(n, hi, lo);
        }
        return __builtin_fma(n * k, hi, k * lo);
    }
}

// HHI_buffer::DP8_step of one octet: x is the lane's variable, row the step's
// decay factors
template <bool EXACT, class Row>
__device__ __forceinline__ void i_oct_dp8(StepRange& rg, const IOctLane& L, const Dp8Consts& C, double& x_io,
                                          double Ge, double Gi, double dt, const Row& row)
{
    const double x0 = x_io;
    double x = x0, v, n1, m1, h1, w1;
    // V to every lane; n, m, h (quad broadcasts) and w (mirror of lane 7) to lane 0
    auto exchange = [&] {
        const double t = oct_mirror(x);
        v = half_bcast<0, 3>(x, t);
        n1 = quad_bcast<1>(x);
        m1 = quad_bcast<2>(x);
        h1 = quad_bcast<3>(x);
        w1 = t;
    };
#define OCT_K(e2, e5) i_oct_deriv<EXACT>(rg, L, Ge, Gi, v, n1, m1, h1, w1, x, e2, e5)
#define OCT_T(J, k) dp8_term<J, EXACT>(C, k)
    exchange();
    const double k1 = OCT_K(1.0, 1.0);
    x = x0 + qconst<EXACT>(dt * k1, 18);
    exchange();
    const double k2 = OCT_K(row.e2[kOffDp2], row.e5[kOffDp2]);
    x = x0 + qconst<EXACT>(dt * (k1 + 3 * k2), 48);
    exchange();
    const double k3 = OCT_K(row.e2[kOffDp3], row.e5[kOffDp3]);
    x = x0 + dt * (k1 + 3 * k3) * 0.03125;
    exchange();
    const double k4 = OCT_K(row.e2[kOffDp4], row.e5[kOffDp4]);
    x = x0 + dt * (20 * k1 - 75 * k3 + 75 * k4) * 0.015625;
    exchange();
    const double k5 = OCT_K(row.e2[kOffDp5], row.e5[kOffDp5]);
    x = x0 + qconst<EXACT>(dt * (3 * k1 + 15 * k4 + 12 * k5), 80);
    exchange();
    const double k6 = OCT_K(row.e2[kOffDp6], row.e5[kOffDp6]);
    x = x0 + dt * (OCT_T(0, k1) + OCT_T(1, k4) - OCT_T(2, k5) +
                   OCT_T(3, k6));
    exchange();
    const double k7 = OCT_K(row.e2[kOffDp7], row.e5[kOffDp7]);
    x = x0 + dt * (OCT_T(4, k1) + OCT_T(5, k4) + OCT_T(6, k5) +
                   OCT_T(7, k6) - OCT_T(8, k7));
    exchange();
    const double k8 = OCT_K(row.e2[kOffDp8], row.e5[kOffDp8]);
    x = x0 + dt * (OCT_T(9, k1) - OCT_T(10, k4) - OCT_T(11, k5) +
                   OCT_T(12, k6) + OCT_T(13, k7) + OCT_T(14, k8));
    exchange();
    const double k9 = OCT_K(row.e2[kOffDp9], row.e5[kOffDp9]);
    x = x0 + dt * (OCT_T(15, k1) - OCT_T(16, k4) -
                   OCT_T(17, k5) - OCT_T(18, k6) + OCT_T(19, k7) +
                   OCT_T(20, k8) + OCT_T(21, k9));
    exchange();
    const double k10 = OCT_K(row.e2[kOffDp10], row.e5[kOffDp10]);
    x = x0 + dt * (OCT_T(22, k1) + OCT_T(23, k4) +
                   OCT_T(24, k5) - OCT_T(25, k6) -
                   OCT_T(26, k7) + OCT_T(27, k8) -
                   OCT_T(28, k9) + OCT_T(29, k10));
    exchange();
    const double k11 = OCT_K(row.e2[kOffDp11], row.e5[kOffDp11]);
    x = x0 + dt * (OCT_T(30, k1) - OCT_T(31, k4) -
                   OCT_T(32, k5) - OCT_T(33, k6) + OCT_T(34, k7) +
                   OCT_T(35, k8) - OCT_T(36, k9) +
                   OCT_T(37, k10) + OCT_T(38, k11));
    exchange();
    const double k12 = OCT_K(row.e2[kOffDt], row.e5[kOffDt]);
    x_io = x0 + dt * (OCT_T(39, k1) - OCT_T(40, k6) +
                      OCT_T(41, k7) + OCT_T(42, k8) -
                      OCT_T(43, k9) + OCT_T(44, k10) +
                      OCT_T(45, k11) + OCT_T(46, k12));
#undef OCT_K
#undef OCT_T
}

template <class Row>
__device__ __forceinline__ void i_oct_step(const IOctLane& L, const Dp8Consts& C, double& x, double& Ge, double& Gi,
                                           double dt, const Row& row)
{
    StepRange rg;
    const double xs = x;
    i_oct_dp8<false>(rg, L, C, x, Ge, Gi, dt, row);
    if (__any(rg.failed())) {
        x = xs;
        i_oct_dp8<true>(rg, L, C, x, Ge, Gi, dt, row);
    }
    Ge = Ge * row.e2[kOffDt];
    Gi = Gi * row.e5[kOffDt];
}

// ---------------------------------------------------------------------------
// HVC-RA: lane 0 owns Vs and evaluates mInf, lanes 1-3 own n, h, l with nInf,
// hInf, lInf, lane 4 owns r with rInf, lane 5 owns Vd with tauH, lane 6 owns
// Ca with tauN, lane 7 owns c with cInf.  tauN and tauH reach n and h by the
// half-row mirror (1 <-> 6, 2 <-> 5).  The derivatives of n, h, l, r, c and
// the dendrite's calcium-dependent current are one quotient per lane, and the
// two membrane equations one sum with per-lane terms.  l belongs to the
// Debraband model; in the RK4 model its lane runs along and is not stored.
// ---------------------------------------------------------------------------
constexpr int kRAOctNeuronsPerWave = 8;

struct RAOctLane {
    int q;
    bool lo;                 // lanes 0-3: the soma's half
    bool vother;             // tauH, tauN: gates on Vs in the dendrite's half
    double d;                // gate = g0 + c / (1 + exp((v + d) / e)), e signed
    LaneDiv e;
    double g0, c;
    double den;              // divisor of the lane's derivative quotient (constant ones)
    bool dtau, dca;          // ... taken from the mirror lane; 1 + 6 / [Ca]
    double EL, f1, E1, kl;   // membrane sum: leak, first current, l conductance
    double EA, EB;           // reversal of the two synaptic terms in their order
    double mu;
    LaneDiv R;               // coupling: 100000 (v2 - v1) / R
    double ca01;             // -0.1 GCa
    const ExpPair* tab;
};

struct RAOctConst {
    double d;
    LaneDiv e;
    double g0, c, den;       // den: the Debraband model's (the RK4 model's c has 10)
    LaneDiv R;
};
static __constant__ RAOctConst kRAOctConsts[8] = {
    {30.0, lane_div(-9.5), 0.0, 1.0, 1.0, lane_div(275000.0)},     // mInf
    {35.0, lane_div(-10.0), 0.0, 1.0, 1.0, lane_div(275000.0)},    // nInf
    {45.0, lane_div(7.0), 0.0, 1.0, 1.0, lane_div(275000.0)},      // hInf
    {40.0, lane_div(-5.0), 0.0, 1.0, 10.0, lane_div(275000.0)},    // lInf
    {5.0, lane_div(-10.0), 0.0, 1.0, 1.0, lane_div(550000.0)},     // rInf
    {40.5, lane_div(6.0), 0.1, 0.75, 1.0, lane_div(550000.0)},     // tauH
    {27.0, lane_div(15.0), 0.1, 0.5, 1.0, lane_div(550000.0)},     // tauN
    {-10.0, lane_div(-7.0), 0.0, 1.0, 15.0, lane_div(550000.0)}};  // cInf

template <int MODEL>
__device__ __forceinline__ RAOctLane ra_oct_lane(int q, double EL, double GCa, double mu_s, double mu_d,
                                                 const ExpPair* tab)
{
    const RAOctConst c = kRAOctConsts[q];
    RAOctLane L;
    L.q = q;
    L.lo = q < 4;
    L.vother = q == 5 || q == 6;
    L.d = c.d;
    L.e = c.e;
    L.g0 = c.g0;
    L.c = c.c;
    L.den = MODEL == 1 && q == 7 ? 10.0 : c.den;
    L.dtau = q == 1 || q == 2;
    L.dca = q == 5;
    L.EL = EL;
    L.f1 = GCa;
    L.E1 = L.lo ? kRA_EsNa : kRA_EdCa;
    L.kl = L.lo && MODEL == 0 ? kRA_GsKLT : 0.0;
    L.EA = L.lo ? kRA_Egaba : 0.0;
    L.EB = L.lo ? 0.0 : kRA_Egaba;
    L.mu = L.lo ? mu_s : mu_d;
    L.R = c.R;
    L.ca01 = -0.1 * GCa;
    L.tab = tab;
    return L;
}

// derivative of the lane's variable at stage value x; GA, GB: the neuron's
// inhibitory and excitatory soma conductances (lane 0) or excitatory and
// inhibitory dendritic ones (lane 5), E the stage's decay factor
template <int MODEL, bool EXACT>
__device__ __forceinline__ double ra_oct_deriv(StepRange& rg, const RAOctLane& L, double x, double GA, double GB,
                                               double E)
{
    const double t = oct_mirror(x);
    const double P0 = quad_bcast<0>(x), P1 = quad_bcast<1>(x), P2 = quad_bcast<2>(x), P3 = quad_bcast<3>(x);
    const double v1 = L.lo ? P0 : P1;           // the half's own voltage: Vs, Vd
    const double v2 = half_bcast<2, 3>(t, t);   // the other one
    // the lane's gate
    const double vd = (L.vother ? v2 : v1) + L.d;
    const double Eg = EXACT ? dexp(vd / L.e.B) : exp_inrange(qlane<EXACT>(vd, L.e), L.tab);
    const double g = L.g0 + qdiv<EXACT>(L.c, 1 + Eg);
    const double tau = oct_mirror(g);
    // (xInf - x) / tau; in lane 5 the calcium-dependent potassium current
    const double vk = v1 - kRA_EsK;     // E_K is the same in both compartments
    double w6 = 1 + qdiv<EXACT>(6, P2), ica = kRA_GdCaK * vk * P3, gx = g - x;
    every_lane(w6);
    every_lane(ica);
    every_lane(gx);
    const double num = L.dca ? ica : gx;
    const double den = L.dca ? w6 : (L.dtau ? tau : L.den);
    double Q = qdiv<EXACT>(num, den);
    every_lane(Q);
    // membrane sum of the half: u = m (soma) or r (dendrite)
    const double u = L.lo ? g : P0;
    const double uu = u * u;
    double gna = kRA_GsNa * (uu * u), ik = kRA_GsK * (P1 * P1 * P1 * P1) * vk;
    every_lane(gna);
    every_lane(ik);
    const double f1 = L.lo ? gna : L.f1;
    const double f2 = L.lo ? P2 : uu;
    const double ve = v1 - L.E1;
    const double T2 = L.lo ? ik : Q;
    double acc = -kRA_GsL * (v1 - L.EL) - f1 * f2 * ve - T2;
    if (MODEL == 0) {
        if constexpr (EXACT)
            acc = L.lo ? acc - kRA_GsKLT * P3 * vk : acc;
        else
            acc = acc - L.kl * P3 * vk;
    }
    const double dv = v2 - v1;
    double kV = acc - (GA * E) * (v1 - L.EA) - (GB * E) * (v1 - L.EB) + L.mu + qlane<EXACT>(100000 * dv, L.R);
    double kCa = L.ca01 * P0 * P0 * ve - 0.02 * P2;
    every_lane(kV);
    every_lane(kCa);
    const double k = (L.q == 0 || L.q == 5) ? kV : (L.q == 6 ? kCa : Q);
    if constexpr (!EXACT) {
        rg.volt(v1);
        rg.volt(v2);
        rg.least(dv);
        rg.deriv(k);
    }
    return k;
}

// what a Debraband step adds of its white noise to the lane's variable at the
// four stages and at its end (zero but for the two voltages)
struct RANoise {
    double s[4], end, pad;
};

// HH2_test::Debraband_step of one octet
template <bool EXACT>
__device__ __forceinline__ void ra_oct_debraband(StepRange& rg, const RAOctLane& L, double& x, double GA, double GB,
                                                 double dt, const RANoise& nz, double E_dt, double E_half)
{
    const double x0 = x;
#define OCT_K(v, E) ra_oct_deriv<0, EXACT>(rg, L, v, GA, GB, E)
    const double a1 = OCT_K(x0 + nz.s[0], 1.0);
    const double a2 = OCT_K(x0 + dt * a1 + nz.s[1], E_dt);
    const double a3 = OCT_K(x0 + dt * (3 * a1 + a2) * 0.125 + nz.s[2], E_half);
    const double a4 = OCT_K(x0 + dt * (-0.4526683126055039 * a1 - 0.4842227708685013 * a2 + 1.9368910834740051 * a3) +
                                nz.s[3],
                            E_dt);
#undef OCT_K
    x = x0 + dt * (qconst<EXACT>(a1, 6) - 0.005430430675258792 * a2 + qconst<EXACT>(2 * a3, 3) +
                   0.1720970973419255 * a4) +
        nz.end;
}

// HH2_buffer::Runge4_step of one octet
template <bool EXACT>
__device__ __forceinline__ void ra_oct_runge4(StepRange& rg, const RAOctLane& L, double& x, double GA, double GB,
                                              double dt, double E_third, double E_twothird, double E_dt)
{
    const double x0 = x;
#define OCT_K(v, E) ra_oct_deriv<1, EXACT>(rg, L, v, GA, GB, E)
    const double k1 = OCT_K(x0, 1.0);
    const double k2 = OCT_K(x0 + qconst<EXACT>(dt * k1, 3), E_third);
    const double k3 = OCT_K(x0 + dt * (qconst<EXACT>(-k1, 3) + k2), E_twothird);
    const double k4 = OCT_K(x0 + dt * (k1 - k2 + k3), E_dt);
#undef OCT_K
    x = x0 + dt * (k1 + 3 * k2 + 3 * k3 + k4) * 0.125;
}

// one step of MODEL and the decay of the lane's two conductances; nz is the
// step's noise (Debraband)
template <int MODEL, class Row>
__device__ __forceinline__ void ra_oct_step(const RAOctLane& L, double& x, double& GA, double& GB, double dt,
                                            const RANoise& nz, const Row& row)
{
    const double E_dt = row.e5[kOffDt];
    StepRange rg;
    const double xs = x;
    if constexpr (MODEL == 0) {
        const double E_half = row.e5[kOffHalf];
        ra_oct_debraband<false>(rg, L, x, GA, GB, dt, nz, E_dt, E_half);
        if (__any(rg.failed())) {
            x = xs;
            ra_oct_debraband<true>(rg, L, x, GA, GB, dt, nz, E_dt, E_half);
        }
    } else {
        const double E_third = row.e5[kOffThird], E_twothird = row.e5[kOffTwoThird];
        ra_oct_runge4<false>(rg, L, x, GA, GB, dt, E_third, E_twothird, E_dt);
        if (__any(rg.failed())) {
            x = xs;
            ra_oct_runge4<true>(rg, L, x, GA, GB, dt, E_third, E_twothird, E_dt);
        }
    }
    GA = GA * E_dt;
    GB = GB * E_dt;
}

// The Debraband noise of a window.  A step adds a multiple of each
// compartment's pair of point-distribution values, and these take five values
// each, so a block tabulates the 2 x 25 possible RANoise once (kNoiseRows rows
// in LDS, the last one zero) and a step only picks a row.
constexpr int kNoiseClasses = 5;
constexpr int kNoiseRows = 2 * kNoiseClasses * kNoiseClasses + 1;
__device__ __forceinline__ int point_class(uint32_t w)
{
    const int p = point_index(w);
    return p < 2 ? p : (p < 11 ? 2 : (p < 20 ? 3 : 4));
}
__device__ __forceinline__ void stage_noise_rows(RANoise* rows, double sq_sig_s, double sq_sig_d)
{
    for (int r = threadIdx.x; r < kNoiseRows; r += blockDim.x) {
        RANoise z{};
        if (r < kNoiseRows - 1) {
            const int comp = r / (kNoiseClasses * kNoiseClasses), p = r % (kNoiseClasses * kNoiseClasses);
            auto value = [](int c) { return kPointDistribution[c < 2 ? c : (c == 2 ? 2 : (c == 3 ? 11 : 20))]; };
            const double J1 = value(p / kNoiseClasses), J2 = value(p % kNoiseClasses);
            const double sq = comp ? sq_sig_d : sq_sig_s, A = comp ? 10000.0 : 5000.0;
            z.s[0] = sq * (-0.01844540496323970 * J1 - 0.1866426386543421 * J2) / A;
            z.s[1] = sq * (0.8017012756521233 * J1 - 0.8575745885712401 * J2) / A;
            z.s[2] = sq * (0.5092227024816198 * J1 - 0.4723392695015512 * J2) / A;
            z.s[3] = sq * (0.9758794209767762 * J1 + 0.3060354860326548 * J2) / A;
            z.end = sq * J1 * 100000 / A;
        }
        rows[r] = z;
    }
}
// the noise rows of the octet's neuron at the steps t0 .. t0 + n - 1, one
// Philox call per lane and eight steps: at[2 k] the soma's, at[2 k + 1] the
// dendrite's
__device__ __forceinline__ void noise_window(uint8_t* at, int q, const NoiseId& id, int t0, int n)
{
    for (int k = q; k < n; k += 8) {
        const U4 o = philox4x32((uint32_t)(t0 + k), id.local, id.trial, kStreamRAWhite, id.k0, id.k1);
        at[2 * k] = (uint8_t)(point_class(o.x) * kNoiseClasses + point_class(o.y));
        at[2 * k + 1] = (uint8_t)(kNoiseClasses * kNoiseClasses + point_class(o.z) * kNoiseClasses + point_class(o.w));
    }
}

}  // namespace p64
}  // namespace hvc
#endif
