// hvc_integrate.hip.h -- neuron integration kernels of one precision form.
//
// Included once by hvc_kernels.hip (FP64 form, bit-exact) and once by
// hvc_kernels_f32.hip (FP32 form, HVC_FP32 defined); the kernels land in
// hvc::p64 or hvc::p32, the launchers are named launch_* and launch_*_f32.
// Neuron state is stored in HBM as FP64 structure-of-arrays in both forms; the
// FP32 form rounds it to float when a window starts and widens it when the
// window ends.
#pragma once
#include <hip/hip_runtime.h>

#include "hvc_internal.h"
#include "hvc_neuron.hip.h"
#include "hvc_oct64.hip.h"
#include "hvc_stdp.hip.h"

namespace hvc {

static inline int blocks_for(int n, int bs) { return n > 0 ? (n + bs - 1) / bs : 1; }

#ifndef HVC_INBOX_DEFINED
#define HVC_INBOX_DEFINED
// ordered sum of one target's inbox: records sorted by (arrival step, presynaptic id)
__device__ __forceinline__ double inbox_sum(const Inbox& ib, int tgt, int n)
{
    Record* r = ib.rec + (size_t)tgt * ib.cap;
    for (int a = 1; a < n; ++a) {
        Record x = r[a];
        int b = a - 1;
        while (b >= 0 && r[b].key > x.key) {
            r[b + 1] = r[b];
            --b;
        }
        r[b + 1] = x;
    }
    double sum = 0.0;
    for (int a = 0; a < n; ++a) sum += r[a].w;
    return sum;
}

// the previous window's sync for one target (NGS:9309-9366): the ordered sum
// of its inbox, if any, and the inbox emptied
// (n: the inbox's count, loaded ahead)
__device__ __forceinline__ bool inbox_take(const NetDev& nd, const Inbox& ib, int tgt, int n, double& sum)
{
    if (n <= 0) return false;
    if (n > ib.cap) {
        atomicOr(nd.err, (unsigned)kErrInbox);
        n = ib.cap;
    }
    sum = inbox_sum(ib, tgt, n);
    ib.cnt[tgt] = 0;
    return true;
}
#endif

HVC_PREC_BEGIN

// One neuron step.  FP64: with the branch-free constant divisions; if any lane
// of the wave met a quotient outside the proven range, the wave repeats the
// step from the saved state with IEEE division (EXACT), which gives the same
// bits.  FP32: the step as is.
#define HVC_GUARDED_STEP(State, call_fast, call_exact) \
    Guard bad;                                         \
    if constexpr (Guard::kActive) {                    \
        State s0 = s;                                  \
        call_fast;                                     \
        if (__any(bad.failed())) {                     \
            s = s0;                                    \
            call_exact;                                \
        }                                              \
    } else {                                           \
        call_fast;                                     \
    }

__device__ __forceinline__ void ra_step_debraband(RAState& s, real el, real gca, const RAUniform& u, real J1s,
                                                  real J2s, real J1d, real J2d, real E_dt, real E_half)
{
    HVC_GUARDED_STEP(RAState, (ra_debraband<false>(bad, s, el, gca, u, J1s, J2s, J1d, J2d, E_dt, E_half)),
                     (ra_debraband<true>(bad, s, el, gca, u, J1s, J2s, J1d, J2d, E_dt, E_half)))
}

template <bool LANES = false>
__device__ __forceinline__ void ra_step_runge4(RAState& s, real el, real gca, const RAUniform& u, real E_third,
                                               real E_twothird, real E_dt, const RAGateSlot* sl = nullptr)
{
    HVC_GUARDED_STEP(RAState, (ra_runge4<false, LANES>(bad, s, el, gca, u, sl, E_third, E_twothird, E_dt)),
                     (ra_runge4<true, LANES>(bad, s, el, gca, u, sl, E_third, E_twothird, E_dt)))
}

template <int MODEL, class Row>
__device__ __forceinline__ void i_step(IState& s, real dt, const Row& row)
{
    if (MODEL == 0) {
        HVC_GUARDED_STEP(IState, (i_dp8<false>(bad, s, dt, row)), (i_dp8<true>(bad, s, dt, row)))
    } else {
        HVC_GUARDED_STEP(IState, (i_runge4<false>(bad, s, dt, row)), (i_runge4<true>(bad, s, dt, row)))
    }
}

#ifdef HVC_FP32
template <class Row>
__device__ __forceinline__ void i_step_lanes(IState& s, real& xlo, int role, int base, real dt, const Row& row)
{
    Guard bad;
    i_dp8_lanes<false>(bad, s, xlo, role, base, dt, row);
}

template <class Row>
__device__ __forceinline__ void i_step_quad(IState& s, real& xlo, real& wlo, int role, const GateSlot& ga,
                                            const GateSlot& gb, real dt, const Row& row)
{
    Guard bad;
    i_dp8_quad<false>(bad, s, xlo, wlo, role, ga, gb, dt, row);
}
template <class Row>
__device__ __forceinline__ void i_step_oct(IState& s, real& xo, real& xlo, int q, const GateSlot& g, real dt,
                                           const Row& row)
{
    Guard bad;
    i_dp8_oct<false>(bad, s, xo, xlo, q, g, dt, row);
}
template <class Row>
__device__ __forceinline__ void i_step_oct(IState& s, real& xo, real& xlo, int q, const IOctShared& g, real dt,
                                           const Row& row)
{
    i_dp8_shared(s, xo, xlo, q, g, dt, row);
}
__device__ __forceinline__ void i_oct_gate(GateSlot& g, int q) { g = kIOctGates[q]; }
__device__ __forceinline__ void i_oct_gate(IOctShared& g, int q) { g = IOctShared(q); }
#endif
#undef HVC_GUARDED_STEP

// state variables between HBM (FP64) and registers: the FP32 form keeps a
// variable as float hi + float lo (compensated accumulation), which the FP64
// copy in HBM holds exactly
#ifdef HVC_FP32
#define HVC_LOAD(st, f, d)                            \
    {                                                 \
        double d_ = (d);                              \
        st.f = (real)d_;                              \
        st.f##_lo = (real)(d_ - (double)st.f);        \
    }
#define HVC_WIDE(st, f) ((double)st.f + (double)st.f##_lo)
#else
#define HVC_LOAD(st, f, d) st.f = (d);
#define HVC_WIDE(st, f) (st.f)
#endif

// per-network stepper constants in the form's type
__device__ __forceinline__ RAUniform ra_uniform(const NetDev& nd)
{
    return RAUniform{(real)nd.sq_sig_s, (real)nd.sq_sig_d, (real)nd.mu_term_s, (real)nd.mu_term_d, (real)nd.dt};
}

// The coupling window's per-step tables, staged in LDS by k_integrate: decay
// rows of the steps t0..t1 and the clock at t0 - 1 .. t1 (every step of every
// neuron reads them; from HBM / L2 each read would stall the step).
struct Win {
    const WinRow* rows;     // rows[t - t0]
    const double* clock;    // clock[t - t0 + 1] = clock at step t
    int t0;
    double* lds;            // the block's copy: nsteps rows, then the clock
    int nsteps;
    __device__ __forceinline__ const WinRow& row(int t) const { return rows[t - t0]; }
    __device__ __forceinline__ double clk(int t) const { return clock[t - t0 + 1]; }
    // Copy the tables into LDS, by every thread of the block.  load() issues
    // kStagePieces reads of 16 bytes a thread (all of an 18-step window's rows
    // in blocks of 64) and store() writes them, so that the tables arrive
    // together with the neuron's state, which the caller loads before, in one
    // memory latency (the L2s are cold after a kernel boundary); the loop of
    // 8-byte copies waited six times.  From a wave's start to its first step,
    // with the neuron's loads ahead of the tables' and kernarg_touch, FP64
    // HVC-I octets: 9 900 -> 2 550 cycles, 2.8 us of a 47 us window.
    static constexpr int kStagePieces = 4;
    typedef double Piece __attribute__((ext_vector_type(2)));
    static constexpr int kRowPieces = (int)(sizeof(DecayRow) / sizeof(Piece));
    struct Tables {
        Piece v[kStagePieces];
        double c;
    };
    __device__ __forceinline__ const Piece* pieces(const NetDev& nd) const
    {
        return (const Piece*)((const DecayRow*)nd.decay + t0);
    }
    __device__ __forceinline__ Tables load(const NetDev& nd) const
    {
        Tables t;
        const int last = nsteps * kRowPieces - 1;
#pragma unroll
        for (int u = 0; u < kStagePieces; ++u) t.v[u] = pieces(nd)[min((int)(threadIdx.x + u * blockDim.x), last)];
        t.c = nd.clock[t0 - 1 + min((int)threadIdx.x, nsteps)];
        return t;
    }
    __device__ __forceinline__ void put(int p, Piece v) const
    {
#ifdef HVC_FP32
        const int r = p / kRowPieces, o = p - r * kRowPieces;
        WinRow* row = (WinRow*)lds + r;
        ((float2*)row)[o] = make_float2((float)v.x, (float)v.y);   // e5, then e2
        if (o == 0) row->e5dt = v.x;
        if (o == kRowPieces / 2) row->e2dt = v.x;
#else
        ((Piece*)lds)[p] = v;
#endif
    }
    __device__ __forceinline__ void store(const NetDev& nd, const Tables& t) const
    {
        const int n = nsteps * kRowPieces;
        double* wc = (double*)((WinRow*)lds + nsteps);
#pragma unroll
        for (int u = 0; u < kStagePieces; ++u) put(min((int)(threadIdx.x + u * blockDim.x), n - 1), t.v[u]);
        wc[min((int)threadIdx.x, nsteps)] = t.c;
        for (int p = threadIdx.x + kStagePieces * blockDim.x; p < n; p += blockDim.x) put(p, pieces(nd)[p]);
        for (int k = threadIdx.x + blockDim.x; k <= nsteps; k += blockDim.x) wc[k] = nd.clock[t0 - 1 + k];
        __syncthreads();
    }
    __device__ __forceinline__ void stage(const NetDev& nd) const { store(nd, load(nd)); }
};
static_assert(kOffDt == 0 && kNumOffsets % 2 == 0, "put() finds the whole-step factors at the start of each half row");

// The neuron's next two noise events of the chunk (lists are generated by
// k_noise_events).  take() applies every event of step t, in list order; the
// following entry is loaded a step or more before it is looked at, except
// when two events fall on one step.
struct NoiseCursor {
    const NoiseEvent* ev;
    int pos;
    NoiseEvent cur, nxt;
    __device__ __forceinline__ void open(const NoiseEvent* list, int p)
    {
        ev = list;
        pos = p;
        cur = ev[p];
        nxt = ev[p + 1];
    }
    __device__ __forceinline__ void none()
    {
        ev = nullptr;
        pos = 0;
        cur.step = kNoNoiseStep;
        nxt.step = kNoNoiseStep;
    }
    template <class Apply>
    __device__ __forceinline__ void take(int t, Apply apply)
    {
        while (cur.step == t) {
            apply(cur.target, cur.inc);
            cur = nxt;
            ++pos;
            nxt = ev[pos + 1];
        }
    }
};

// append (neuron, step) to a log with one atomic per wave
__device__ __forceinline__ void wave_append(int2* log, int* cnt, int cap, bool pred, int neuron, int step,
                                            unsigned int* err)
{
    uint64_t m = __ballot(pred);
    if (m == 0) return;
    int lane = __lane_id();
    int leader = __ffsll((unsigned long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(cnt, __popcll(m));
    base = __shfl(base, leader);
    if (pred) {
        int pos = base + __popcll(m & ((1ull << lane) - 1ull));
        if (pos < cap)
            log[pos] = make_int2(neuron, step);
        else
            atomicOr(err, (unsigned)kErrSpikeLog);
    }
}

// the window's spikes of the lanes (bit k of mask: step t0 + k) appended after
// the steps, one atomic per wave and round (a lane spikes at most once per
// window in practice, so one round); the host sorts the log
__device__ __forceinline__ void window_append(int2* log, int* cnt, int cap, uint64_t mask, int neuron, int t0,
                                              unsigned int* err)
{
    for (;;) {
        const bool pred = mask != 0;
        if (__ballot(pred) == 0) return;
        const int step = pred ? t0 + __ffsll((unsigned long long)mask) - 1 : 0;
        wave_append(log, cnt, cap, pred, neuron, step, err);
        mask &= mask - 1;
    }
}

// A neuron that spiked in the window goes on the role's delivery list for the
// window (the delivery kernel visits only listed neurons), unless the previous
// window's delivery listed it already (spikes still in flight); `listed` is
// the neuron's list mark, loaded when the window began.  One atomic per wave.
// A list holds each neuron at most once, so it never outgrows its neurons.
__device__ __forceinline__ void wl_enlist(const NetDev& nd, int role, bool spiked, int listed, int neuron)
{
    if (!nd.wl_on) return;
    const int w = nd.window;
    const bool pred = spiked && listed != w;
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    const int lane = __lane_id();
    const int leader = __ffsll((unsigned long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(&nd.wl_cnt[3 * role + w % 3], __popcll(m));
    base = __shfl(base, leader);
    if (pred) {
        const int pos = base + __popcll(m & ((1ull << lane) - 1ull));
        if (pos < nd.wl_cap[role]) {
            nd.wl_list[role][(size_t)(w & 1) * nd.wl_cap[role] + pos] = neuron;
            nd.wl_mark[role][neuron] = w;
        } else {
            atomicOr(nd.err, (unsigned)kErrWorklist);
        }
    }
}

// ---------------------------------------------------------------------------
// integrate: HVC-RA neurons (NGS:8931-9216 minus delivery) and HVC-I neurons
// (NGS:9221-9286 minus delivery) through the steps t0..t1 of one window, in one
// launch.  HVC-I blocks come first: with five lanes per neuron they carry the
// longer per-step work, and the RA blocks run beside them.
// ---------------------------------------------------------------------------
constexpr int kRALanes = 4;                      // lanes per HVC-RA neuron (RK4 form)
constexpr int kRANeuronsPerWave = 64 / kRALanes;  // 16 neurons

// the postsynaptic events of an HVC-RA neuron as a window finds them
struct RAPosts {
    int growth, count;
    double last;      // the latest one's time (count > 0)
};
// post events detected in the previous window become visible now (NGS:9385-9386);
// lead: the lane that keeps neuron ii's events; count, pend: the neuron's
// post_cnt and post_pend, loaded ahead
__device__ __forceinline__ RAPosts ra_posts_begin(const NetDev& nd, const Win& win, int growth, int ii, int t0,
                                                  bool lead, int count, int pend)
{
    RAPosts p{growth, count, 0.0};
    if (growth && lead) {
        if (pend > 0) {
            double cs = win.clk(t0 - 1);
            for (int q = 0; q < pend; ++q) {
                nd.post_ring[(size_t)ii * kPostRing + (p.count % kPostRing)] = cs;
                ++p.count;
            }
            if (pend > 2) atomicOr(nd.err, (unsigned)kErrPostRing);
            nd.post_cnt[ii] = p.count;
            nd.post_pend[ii] = 0;
        }
        if (p.count > 0) p.last = nd.post_ring[(size_t)ii * kPostRing + ((p.count - 1) % kPostRing)];
    }
    return p;
}
// after the steps: the spike logs, the delivery lists and the new postsynaptic
// events (NGS:8956-8967; a window's events become visible in the next window,
// so each spike is tested against the events of earlier windows only, as in
// the step loop).  smask / dmask: the lane's somatic / dendritic spikes of
// neuron i.  Returns the lane's new events.
__device__ __forceinline__ int ra_window_logs(const NetDev& nd, const Win& win, const RAPosts& p, int i, int t0,
                                              uint64_t smask, uint64_t dmask, int listed0, int listed1)
{
    window_append(nd.soma_log, &nd.log_cnt[0], nd.log_cap, smask, i, t0, nd.err);
    window_append(nd.dend_log, &nd.log_cnt[1], nd.log_cap, dmask, i, t0, nd.err);
    wl_enlist(nd, 0, smask != 0, listed0, i);
    wl_enlist(nd, 1, smask != 0, listed1, i);
    int new_posts = 0;
    uint64_t pmask = 0;
    if (p.growth) {
        for (uint64_t m = smask; m; m &= m - 1) {
            const int t = t0 + __ffsll((unsigned long long)m) - 1;
            if (p.count == 0 || win.clk(t) > p.last + 30.0) pmask |= 1ull << (t - t0);
        }
    }
    for (;;) {
        const bool pred = pmask != 0;
        const uint64_t b = __ballot(pred);
        if (b == 0) break;
        const int lane = __lane_id(), lead = __ffsll((unsigned long long)b) - 1;
        int base = 0;
        if (lane == lead) base = atomicAdd(nd.post_list_cnt, __popcll(b));
        base = __shfl(base, lead);
        if (pred) {
            const int t = t0 + __ffsll((unsigned long long)pmask) - 1;
            const int pos = base + __popcll(b & ((1ull << lane) - 1ull));
            if (pos < kPostListCap)
                nd.post_list[pos] = post_key(nd.ra_net[i], t, i);
            else
                atomicOr(nd.err, (unsigned)kErrPostList);
            ++new_posts;
        }
        pmask &= pmask - 1;
    }
    return new_posts;
}

// HVC-RA neurons: one thread per neuron (LANES false, `slot` = neuron index) or,
// RK4 model, four lanes per neuron (LANES true, `slot` = wave index; the quad's
// first lane does the neuron's logging and stores)
template <int MODEL, bool LANES>
__device__ void integrate_ra(const NetDev& nd, const Win& win, int slot, int t0, int t1)
{
    static_assert(!LANES || MODEL == 1, "four lanes per neuron: RK4 form only");
    const int lane = LANES ? __lane_id() : 0;
    const int i = LANES ? slot * kRANeuronsPerWave + (lane >> 2) : slot;
    const bool leader = !LANES || (lane & 3) == 0;
    RAGateSlot gs[2];
    if (LANES) {
        gs[0] = kRAGates[2 * (lane & 3)];
        gs[1] = kRAGates[2 * (lane & 3) + 1];
    }
    const bool live = i < nd.n_ra && (!nd.net_live || nd.net_live[nd.ra_net[i]]);
    const int ii = live ? i : 0;
    const int growth = nd.net_growth[nd.ra_net[ii]];
    const int listed0 = nd.wl_on ? nd.wl_mark[0][ii] : 0, listed1 = nd.wl_on ? nd.wl_mark[1][ii] : 0;
    const RAUniform u = ra_uniform(nd);
    RAState s;
    HVC_LOAD(s, Vs, nd.ra[0][ii]) HVC_LOAD(s, Vd, nd.ra[1][ii]) HVC_LOAD(s, n, nd.ra[2][ii])
    HVC_LOAD(s, l, nd.ra[3][ii]) HVC_LOAD(s, h, nd.ra[4][ii]) HVC_LOAD(s, r, nd.ra[5][ii])
    HVC_LOAD(s, c, nd.ra[6][ii]) HVC_LOAD(s, Ca, nd.ra[7][ii])
    double ge_d = nd.ra[10][ii], gi_d = nd.ra[11][ii];
    s.Ge_s = nd.ra[8][ii]; s.Gi_s = nd.ra[9][ii];
    const int flags = nd.ra_flags[ii];
    const real el = (real)nd.EL[ii], gca = (real)nd.GCa[ii];
    const int kick = nd.kick_step[ii];
    const int n_gi = nd.in_gi_ra.cnt[ii], n_ge = nd.in_ge_ra.cnt[ii];
    const int post_cnt = nd.post_cnt[ii], post_pend = nd.post_pend[ii];
    const bool poisson = MODEL == 1 && nd.ra_poisson;
    const int ev_pos = poisson ? nd.ra_ev_pos[ii] : 0;
    const Win::Tables tab = win.load(nd);
    const NoiseId sid = ra_noise_id(nd, ii);
    NoiseCursor nc;
    if (poisson)
        nc.open(nd.ra_ev + (size_t)ii * nd.ev_cap, ev_pos);
    else
        nc.none();
    win.store(nd, tab);
    // the previous window's sync: raiseI (Gi_d += G), raiseExcWeight (Ge_d += w / Ad)
    if (live && leader) {
        double sum;
        if (inbox_take(nd, nd.in_gi_ra, i, n_gi, sum)) gi_d += sum;
        if (inbox_take(nd, nd.in_ge_ra, i, n_ge, sum)) ge_d += HVC_CDIV(sum, 10000);
    }
    if constexpr (LANES) {
        ge_d = quad_bcast<0>(ge_d);
        gi_d = quad_bcast<0>(gi_d);
    }
    s.Ge_d = ge_d; s.Gi_d = gi_d;
    int fs = flags & 1, fd = (flags >> 1) & 1;

    const RAPosts posts = ra_posts_begin(nd, win, growth, ii, t0, live && leader, post_cnt, post_pend);

    uint64_t smask = 0, dmask = 0;
    for (int t = t0; t <= t1; ++t) {
        if (kick == t) s.Ge_d += 3.0;  // raiseE(G_TRAINING_KICK), NGS:8933-8940
        int f = ra_state_check(s.Vs, s.Vd, fs, fd);
        const WinRow& row = win.row(t);
        if (MODEL == 0) {
            U4 o = philox4x32((uint32_t)t, sid.local, sid.trial, kStreamRAWhite, sid.k0, sid.k1);
            ra_step_debraband(s, el, gca, u, kPointDistribution[point_index(o.x)], kPointDistribution[point_index(o.y)],
                         kPointDistribution[point_index(o.z)], kPointDistribution[point_index(o.w)],
                         row.e5[kOffDt], row.e5[kOffHalf]);
        } else {
            // HH2_buffer noise checks (Gi_s, Gi_d, Ge_s, Ge_d), as listed
            // (selects, not stores through an index: the state stays in registers)
            nc.take(t, [&](int g, double inc) {
                s.Gi_s = g == 0 ? (real)(s.Gi_s + inc) : s.Gi_s;
                s.Gi_d = g == 1 ? (real)(s.Gi_d + inc) : s.Gi_d;
                s.Ge_s = g == 2 ? (real)(s.Ge_s + inc) : s.Ge_s;
                s.Ge_d = g == 3 ? (real)(s.Ge_d + inc) : s.Ge_d;
            });
            ra_step_runge4<LANES>(s, el, gca, u, row.e5[kOffThird], row.e5[kOffTwoThird], row.e5[kOffDt], gs);
        }
        bool soma = live && leader && (f & 1);
        bool dend = live && leader && (f & 2);
        if (soma) smask |= 1ull << (t - t0);
        if (dend) dmask |= 1ull << (t - t0);
    }
    const int new_posts = ra_window_logs(nd, win, posts, i, t0, smask, dmask, listed0, listed1);
    if (live && leader) {
        nd.ra[0][i] = HVC_WIDE(s, Vs); nd.ra[1][i] = HVC_WIDE(s, Vd); nd.ra[2][i] = HVC_WIDE(s, n);
        nd.ra[3][i] = HVC_WIDE(s, l); nd.ra[4][i] = HVC_WIDE(s, h); nd.ra[5][i] = HVC_WIDE(s, r);
        nd.ra[6][i] = HVC_WIDE(s, c); nd.ra[7][i] = HVC_WIDE(s, Ca);
        nd.ra[8][i] = s.Ge_s; nd.ra[9][i] = s.Gi_s; nd.ra[10][i] = s.Ge_d; nd.ra[11][i] = s.Gi_d;
        nd.ra_flags[i] = fs | (fd << 1);
        nd.soma_mask[i] = smask;
        nd.dend_mask[i] = dmask;
        if (growth) nd.post_pend[i] = new_posts;
        if (MODEL == 1 && nd.ra_poisson) nd.ra_ev_pos[i] = nc.pos;
    }
}

// HVC-I, one lane per neuron (RK4 form)
template <int MODEL>
__device__ void integrate_i_thread(const NetDev& nd, const Win& win, int i, int t0, int t1)
{
    const bool live = i < nd.n_i && (!nd.net_live || nd.net_live[nd.i_net[i]]);
    const int ii = live ? i : 0;
    IState s;
    HVC_LOAD(s, V, nd.in[0][ii]) HVC_LOAD(s, n, nd.in[1][ii]) HVC_LOAD(s, m, nd.in[2][ii])
    HVC_LOAD(s, h, nd.in[3][ii]) HVC_LOAD(s, w, nd.in[4][ii])
    const int listed = nd.wl_on ? nd.wl_mark[2][ii] : 0;
    double ge = nd.in[5][ii];
    s.Gi = nd.in[6][ii];
    int flag = nd.i_flag[ii];
    const int n_in = nd.in_ge_i.cnt[ii], ev_pos = nd.i_poisson ? nd.i_ev_pos[ii] : 0;
    const Win::Tables tab = win.load(nd);
    NoiseCursor nc;
    if (nd.i_poisson)
        nc.open(nd.i_ev + (size_t)ii * nd.ev_cap, ev_pos);
    else
        nc.none();
    win.store(nd, tab);
    // the previous window's sync: HHI raiseE (Ge += G)
    if (live) {
        double sum;
        if (inbox_take(nd, nd.in_ge_i, i, n_in, sum)) ge += sum;
    }
    s.Ge = ge;
    uint64_t mask = 0;
    for (int t = t0; t <= t1; ++t) {
        int f = i_state_check(s.V, flag);
        // HHI_buffer noise checks (Ge, Gi), as listed
        nc.take(t, [&](int g, double inc) {
            s.Ge = g == 0 ? (real)(s.Ge + inc) : s.Ge;
            s.Gi = g == 1 ? (real)(s.Gi + inc) : s.Gi;
        });
        i_step<MODEL>(s, (real)nd.dt, win.row(t));
        bool fired = live && f;
        if (fired) mask |= 1ull << (t - t0);
    }
    window_append(nd.i_log, &nd.log_cnt[2], nd.log_cap, mask, i, t0, nd.err);
    wl_enlist(nd, 2, mask != 0, listed, i);
    if (live) {
        nd.in[0][i] = HVC_WIDE(s, V); nd.in[1][i] = HVC_WIDE(s, n); nd.in[2][i] = HVC_WIDE(s, m);
        nd.in[3][i] = HVC_WIDE(s, h); nd.in[4][i] = HVC_WIDE(s, w);
        nd.in[5][i] = s.Ge; nd.in[6][i] = s.Gi;
        nd.i_flag[i] = flag;
        if (nd.i_poisson) nd.i_ev_pos[i] = nc.pos;
        nd.i_mask[i] = mask;
    }
}

#ifdef HVC_FP32
constexpr int kILanes = 5;                    // lanes per HVC-I neuron (DP8)
constexpr int kINeuronsPerWave = 64 / kILanes; // 12 neurons, 4 idle lanes

// HVC-I, five lanes per neuron (DP8 form); one wave holds 12 neurons
__device__ void integrate_i_lanes(const NetDev& nd, const Win& win, int wave, int t0, int t1)
{
    // the four spare lanes 60..63 shadow lanes 55..58 of the last group: same
    // neuron, same roles, results discarded -- their quotients then stay in the
    // range of the real ones and never force the wave to repeat a step
    const int lane = __lane_id();
    const bool spare = lane >= kINeuronsPerWave * kILanes;
    const int role = spare ? lane - kINeuronsPerWave * kILanes : lane % kILanes;
    const int group = spare ? kINeuronsPerWave - 1 : lane / kILanes;
    const int base = group * kILanes;
    const int i = wave * kINeuronsPerWave + group;
    const bool live = (i < nd.n_i) && !spare && (!nd.net_live || nd.net_live[nd.i_net[i]]);
    const int ii = (i < nd.n_i) ? i : 0;
    IState s;
    HVC_LOAD(s, V, nd.in[0][ii]) HVC_LOAD(s, n, nd.in[1][ii]) HVC_LOAD(s, m, nd.in[2][ii])
    HVC_LOAD(s, h, nd.in[3][ii]) HVC_LOAD(s, w, nd.in[4][ii])
    const int listed = nd.wl_on ? nd.wl_mark[2][ii] : 0;
    double ge = nd.in[5][ii];
    s.Gi = nd.in[6][ii];
    int flag = nd.i_flag[ii];
    const int n_in = nd.in_ge_i.cnt[ii], ev_pos = nd.i_poisson ? nd.i_ev_pos[ii] : 0;
    const Win::Tables tab = win.load(nd);
    NoiseCursor nc;
    if (nd.i_poisson)
        nc.open(nd.i_ev + (size_t)ii * nd.ev_cap, ev_pos);
    else
        nc.none();
    win.store(nd, tab);
    // the previous window's sync: HHI raiseE (Ge += G), by the group's first lane
    if (live && role == 0) {
        double sum;
        if (inbox_take(nd, nd.in_ge_i, i, n_in, sum)) ge += sum;
    }
    ge = __shfl(ge, base);
    s.Ge = ge;
    // low part of this lane's own variable
    real xlo = role == 0 ? s.V_lo : (role == 1 ? s.n_lo : (role == 2 ? s.m_lo : (role == 3 ? s.h_lo : s.w_lo)));
    uint64_t mask = 0;
    for (int t = t0; t <= t1; ++t) {
        int f = i_state_check(s.V, flag);
        // HHI_buffer noise checks (Ge, Gi), as listed
        nc.take(t, [&](int g, double inc) {
            s.Ge = g == 0 ? (real)(s.Ge + inc) : s.Ge;
            s.Gi = g == 1 ? (real)(s.Gi + inc) : s.Gi;
        });
        i_step_lanes(s, xlo, role, base, (real)nd.dt, win.row(t));
        bool fired = live && f && role == 0;
        if (fired) mask |= 1ull << (t - t0);
    }
    window_append(nd.i_log, &nd.log_cnt[2], nd.log_cap, mask, i, t0, nd.err);
    wl_enlist(nd, 2, mask != 0, listed, i);
    if (live) {
        // each lane writes its own variable, widened with its low part
        const real xr = role == 0 ? s.V : (role == 1 ? s.n : (role == 2 ? s.m : (role == 3 ? s.h : s.w)));
        nd.in[role][i] = (double)xr + (double)xlo;
    }
    if (live && role == 0) {
        nd.in[5][i] = s.Ge; nd.in[6][i] = s.Gi;
        nd.i_flag[i] = flag;
        if (nd.i_poisson) nd.i_ev_pos[i] = nc.pos;
        nd.i_mask[i] = mask;
    }
}

constexpr int kINeuronsPerQuadWave = 16;       // four lanes per HVC-I neuron

// HVC-I, four lanes per neuron (DP8 form); one wave holds 16 neurons
__device__ void integrate_i_quad(const NetDev& nd, const Win& win, int wave, int t0, int t1)
{
    const int lane = __lane_id();
    const int role = lane & 3;
    const int i = wave * kINeuronsPerQuadWave + (lane >> 2);
    const bool live = i < nd.n_i && (!nd.net_live || nd.net_live[nd.i_net[i]]);
    const int ii = live ? i : 0;
    const GateSlot ga = kIQuadGates[role][0], gb = kIQuadGates[role][1];
    IState s;
    HVC_LOAD(s, V, nd.in[0][ii]) HVC_LOAD(s, n, nd.in[1][ii]) HVC_LOAD(s, m, nd.in[2][ii])
    HVC_LOAD(s, h, nd.in[3][ii]) HVC_LOAD(s, w, nd.in[4][ii])
    const int listed = nd.wl_on ? nd.wl_mark[2][ii] : 0;
    double ge = nd.in[5][ii];
    s.Gi = nd.in[6][ii];
    int flag = nd.i_flag[ii];
    const int n_in = nd.in_ge_i.cnt[ii], ev_pos = nd.i_poisson ? nd.i_ev_pos[ii] : 0;
    const Win::Tables tab = win.load(nd);
    NoiseCursor nc;
    if (nd.i_poisson)
        nc.open(nd.i_ev + (size_t)ii * nd.ev_cap, ev_pos);
    else
        nc.none();
    win.store(nd, tab);
    // the previous window's sync: HHI raiseE (Ge += G), by the quad's first lane
    if (live && role == 0) {
        double sum;
        if (inbox_take(nd, nd.in_ge_i, i, n_in, sum)) ge += sum;
    }
    ge = quad_bcast<0>(ge);
    s.Ge = ge;
    // low parts of this lane's variable and of w
    real xlo = role == 0 ? s.V_lo : (role == 1 ? s.n_lo : (role == 2 ? s.m_lo : s.h_lo));
    real wlo = s.w_lo;
    uint64_t mask = 0;
    for (int t = t0; t <= t1; ++t) {
        int f = i_state_check(s.V, flag);
        // HHI_buffer noise checks (Ge, Gi), as listed
        nc.take(t, [&](int g, double inc) {
            s.Ge = g == 0 ? (real)(s.Ge + inc) : s.Ge;
            s.Gi = g == 1 ? (real)(s.Gi + inc) : s.Gi;
        });
        i_step_quad(s, xlo, wlo, role, ga, gb, (real)nd.dt, win.row(t));
        bool fired = live && f && role == 0;
        if (fired) mask |= 1ull << (t - t0);
    }
    window_append(nd.i_log, &nd.log_cnt[2], nd.log_cap, mask, i, t0, nd.err);
    wl_enlist(nd, 2, mask != 0, listed, i);
    if (live) {
        // each lane writes its own variable, widened with its low part; lane 0 also w
        const real xr = role == 0 ? s.V : (role == 1 ? s.n : (role == 2 ? s.m : s.h));
        nd.in[role][i] = (double)xr + (double)xlo;
        if (role == 0) nd.in[4][i] = (double)s.w + (double)wlo;
    }
    if (live && role == 0) {
        nd.in[5][i] = s.Ge; nd.in[6][i] = s.Gi;
        nd.i_flag[i] = flag;
        if (nd.i_poisson) nd.i_ev_pos[i] = nc.pos;
        nd.i_mask[i] = mask;
    }
}

#endif  // HVC_FP32

constexpr int kINeuronsPerOctWave = 8;       // eight lanes per HVC-I neuron

#ifdef HVC_FP32
// HVC-I, eight lanes per neuron (DP8 form); one wave holds 8 neurons.  Gate:
// the arithmetic of the gates (GateSlot: the octet's own, IOctShared: the one-thread stepper's)
template <class Gate>
__device__ void integrate_i_oct(const NetDev& nd, const Win& win, int wave, int t0, int t1)
{
    const int lane = __lane_id();
    const int q = lane & 7;
    const int i = wave * kINeuronsPerOctWave + (lane >> 3);
    const bool live = i < nd.n_i && (!nd.net_live || nd.net_live[nd.i_net[i]]);
    const int ii = live ? i : 0;
    // the lane's own variable: V (lane 0), n (1, 6), m (2, 5), h (3, 4), w (7)
    const int var = q == 0 ? 0 : (q == 1 || q == 6 ? 1 : (q == 2 || q == 5 ? 2 : (q == 7 ? 4 : 3)));
    IState s;
    HVC_LOAD(s, V, nd.in[0][ii]) HVC_LOAD(s, n, nd.in[1][ii]) HVC_LOAD(s, m, nd.in[2][ii])
    HVC_LOAD(s, h, nd.in[3][ii]) HVC_LOAD(s, w, nd.in[4][ii])
    const int listed = nd.wl_on ? nd.wl_mark[2][ii] : 0;
    double ge = nd.in[5][ii];
    s.Gi = nd.in[6][ii];
    int flag = nd.i_flag[ii];
    const int n_in = nd.in_ge_i.cnt[ii], ev_pos = nd.i_poisson ? nd.i_ev_pos[ii] : 0;
    const Win::Tables tab = win.load(nd);
    Gate g;
    i_oct_gate(g, q);
    NoiseCursor nc;
    if (nd.i_poisson)
        nc.open(nd.i_ev + (size_t)ii * nd.ev_cap, ev_pos);
    else
        nc.none();
    win.store(nd, tab);
    // the previous window's sync: HHI raiseE (Ge += G), by the octet's first lane
    if (live && q == 0) {
        double sum;
        if (inbox_take(nd, nd.in_ge_i, i, n_in, sum)) ge += sum;
    }
    const double ge_lo = quad_bcast<0>(ge), ge_hi = quad_bcast<3>(oct_mirror(ge));
    ge = q < 4 ? ge_lo : ge_hi;
    s.Ge = ge;
    real xo = var == 0 ? s.V : (var == 1 ? s.n : (var == 2 ? s.m : (var == 3 ? s.h : s.w)));
    real xlo = 0;
    xlo = var == 0 ? s.V_lo : (var == 1 ? s.n_lo : (var == 2 ? s.m_lo : (var == 3 ? s.h_lo : s.w_lo)));
    uint64_t mask = 0;
    for (int t = t0; t <= t1; ++t) {
        int f = i_state_check(s.V, flag);
        // HHI_buffer noise checks (Ge, Gi), as listed
        nc.take(t, [&](int gi, double inc) {
            s.Ge = gi == 0 ? (real)(s.Ge + inc) : s.Ge;
            s.Gi = gi == 1 ? (real)(s.Gi + inc) : s.Gi;
        });
        i_step_oct(s, xo, xlo, q, g, (real)nd.dt, win.row(t));
        bool fired = live && f && q == 0;
        if (fired) mask |= 1ull << (t - t0);
    }
    window_append(nd.i_log, &nd.log_cnt[2], nd.log_cap, mask, i, t0, nd.err);
    wl_enlist(nd, 2, mask != 0, listed, i);
    if (live && (q < 4 || q == 7)) {
        // lanes 0-3 write V, n, m, h and lane 7 w, widened with their low parts
        nd.in[var][i] = (double)xo + (double)xlo;
    }
    if (live && q == 0) {
        nd.in[5][i] = s.Ge; nd.in[6][i] = s.Gi;
        nd.i_flag[i] = flag;
        if (nd.i_poisson) nd.i_ev_pos[i] = nc.pos;
        nd.i_mask[i] = mask;
    }
}
#else
// the block's tables of the octet steppers
struct OctLds {
    ExpPair* exp;       // [64]
    RANoise* noise;     // [kNoiseRows], Debraband model
    uint8_t* at;        // 2 kMaxWindowSteps per octet of the block (noise_window)
};

// one of a neuron's state arrays by lane (selects: an indexed read of the
// pointers would be a memory round trip of its own)
template <int N>
__device__ __forceinline__ double* state_array(double* const (&arrays)[N], int k)
{
    double* p = arrays[0];
#pragma unroll
    for (int j = 1; j < N; ++j) p = k == j ? arrays[j] : p;
    return p;
}
// HVC-I octet lane -> V n m h w; HVC-RA octet lane -> Vs Vd n l h r c Ca
__device__ __forceinline__ int i_oct_var(int q) { return q == 0 ? 0 : (q == 7 ? 4 : (q < 4 ? q : 7 - q)); }
__device__ __forceinline__ int ra_oct_var(int q) { return (int)(0x67153420u >> (4 * q)) & 0xf; }

// HVC-I, eight lanes per neuron (DP8 form); one wave holds 8 neurons
__device__ void integrate_i_oct(const NetDev& nd, const Win& win, const OctLds& lds, int wave, int t0, int t1)
{
    const int lane = __lane_id();
    const int q = lane & 7;
    const int i = wave * kINeuronsPerOctWave + (lane >> 3);
    const bool live = i < nd.n_i && (!nd.net_live || nd.net_live[nd.i_net[i]]);
    const int ii = live ? i : 0;
    // everything the window reads of the neuron and its tables, issued together;
    // the lane's constants are made while it is on its way
    double* xp = state_array<7>(nd.in, i_oct_var(q));
    double x = xp[ii];
    const int listed = nd.wl_on ? nd.wl_mark[2][ii] : 0;
    double Ge = nd.in[5][ii], Gi = nd.in[6][ii];
    int flag = nd.i_flag[ii];
    const int n_in = nd.in_ge_i.cnt[ii], ev_pos = nd.i_poisson ? nd.i_ev_pos[ii] : 0;
    const Win::Tables tab = win.load(nd);
    const ExpPair ex = exp_table_load();
    const IOctLane L = i_oct_lane(q, lds.exp);
    Dp8Consts C;
    dp8_pin(C);
    NoiseCursor nc;
    if (nd.i_poisson)
        nc.open(nd.i_ev + (size_t)ii * nd.ev_cap, ev_pos);
    else
        nc.none();
    exp_table_store(lds.exp, ex);
    win.store(nd, tab);
    if (q > 3 && q < 7) x = 1 - x;
    // the previous window's sync: HHI raiseE (Ge += G); only the octet's first
    // lane uses the conductances
    if (live && q == 0) {
        double sum;
        if (inbox_take(nd, nd.in_ge_i, i, n_in, sum)) Ge += sum;
    }
    const double dt = nd.dt;
    uint64_t mask = 0;
    for (int t = t0; t <= t1; ++t) {
        const int f = i_state_check(x, flag);   // of V in lane 0
        // HHI_buffer noise checks (Ge, Gi), as listed
        nc.take(t, [&](int gi, double inc) {
            Ge = gi == 0 ? Ge + inc : Ge;
            Gi = gi == 1 ? Gi + inc : Gi;
        });
        i_oct_step(L, C, x, Ge, Gi, dt, win.row(t));
        if (live && f && q == 0) mask |= 1ull << (t - t0);
    }
    window_append(nd.i_log, &nd.log_cnt[2], nd.log_cap, mask, i, t0, nd.err);
    wl_enlist(nd, 2, mask != 0, listed, i);
    if (live && (q < 4 || q == 7)) xp[i] = x;
    if (live && q == 0) {
        nd.in[5][i] = Ge; nd.in[6][i] = Gi;
        nd.i_flag[i] = flag;
        if (nd.i_poisson) nd.i_ev_pos[i] = nc.pos;
        nd.i_mask[i] = mask;
    }
}

// the spike detection of an HVC-RA octet lane: the soma's in lane 0 (bit 0),
// the dendrite's in lane 5 (bit 1) (ra_state_check, HH2_test.cpp:561-594)
__device__ __forceinline__ int ra_oct_check(int q, double x, int& flag)
{
    int f = 0;
    if (q == 0) {
        if (flag == 1 && x < -30.0 - 5.0) {
            flag = 0;
            f = 1;
        } else if (flag == 0 && x > -30.0) {
            flag = 1;
        }
    } else if (q == 5) {
        if (flag == 0 && x >= -30.0) {
            flag = 1;
            f = 2;
        } else if (flag == 1 && x < -30.0 - 5.0) {
            flag = 0;
        }
    }
    return f;
}

// HVC-RA, eight lanes per neuron; one wave holds 8 neurons.  Lane 0 keeps the
// neuron's events, lane 5 its dendritic spikes.
template <int MODEL>
__device__ void integrate_ra_oct(const NetDev& nd, const Win& win, const OctLds& lds, int wave, int t0, int t1)
{
    const int lane = __lane_id();
    const int q = lane & 7;
    const int i = wave * kRAOctNeuronsPerWave + (lane >> 3);
    const bool live = i < nd.n_ra && (!nd.net_live || nd.net_live[nd.ra_net[i]]);
    const int ii = live ? i : 0;
    const bool soma = live && q == 0, dend = live && q == 5;
    const int growth = nd.net_growth[nd.ra_net[ii]];
    const int listed0 = nd.wl_on ? nd.wl_mark[0][ii] : 0, listed1 = nd.wl_on ? nd.wl_mark[1][ii] : 0;
    double* xp = state_array<12>(nd.ra, ra_oct_var(q));
    double x = xp[ii];
    // the lane's two synaptic conductances (ra_oct_deriv): Gi_s, Ge_s or Ge_d, Gi_d
    double* const gap = q == 0 ? nd.ra[9] : nd.ra[10];
    double* const gbp = q == 0 ? nd.ra[8] : nd.ra[11];
    double GA = gap[ii], GB = gbp[ii];
    const int flags = nd.ra_flags[ii];
    int flag = q == 0 ? flags & 1 : (flags >> 1) & 1;
    const int kick = nd.kick_step[ii];
    const int n_gi = nd.in_gi_ra.cnt[ii], n_ge = nd.in_ge_ra.cnt[ii];
    const int post_cnt = nd.post_cnt[ii], post_pend = nd.post_pend[ii];
    const bool poisson = MODEL == 1 && nd.ra_poisson;
    const int ev_pos = poisson ? nd.ra_ev_pos[ii] : 0;
    const double EL = nd.EL[ii], GCa = nd.GCa[ii];
    const Win::Tables tab = win.load(nd);
    const ExpPair ex = exp_table_load();
    const NoiseId sid = ra_noise_id(nd, ii);
    const RAOctLane L = ra_oct_lane<MODEL>(q, EL, GCa, nd.mu_term_s, nd.mu_term_d, lds.exp);
    uint8_t* at = lds.at + (threadIdx.x >> 3) * (2 * kMaxWindowSteps);
    exp_table_store(lds.exp, ex);
    NoiseCursor nc;
    if constexpr (MODEL == 0) {
        stage_noise_rows(lds.noise, nd.sq_sig_s, nd.sq_sig_d);
        noise_window(at, q, sid, t0, t1 - t0 + 1);
    }
    if (poisson)
        nc.open(nd.ra_ev + (size_t)ii * nd.ev_cap, ev_pos);
    else
        nc.none();
    win.store(nd, tab);
    // the previous window's sync: raiseExcWeight (Ge_d += w / Ad), raiseI (Gi_d += G)
    if (dend) {
        double sum;
        if (inbox_take(nd, nd.in_gi_ra, i, n_gi, sum)) GB += sum;
        if (inbox_take(nd, nd.in_ge_ra, i, n_ge, sum)) GA += HVC_CDIV(sum, 10000);
    }
    const RAPosts posts = ra_posts_begin(nd, win, growth, ii, t0, soma, post_cnt, post_pend);
    const double dt = nd.dt;
    uint64_t mask = 0;   // somatic spikes in lane 0, dendritic ones in lane 5
    for (int t = t0; t <= t1; ++t) {
        if (kick == t && q == 5) GA += 3.0;   // raiseE(G_TRAINING_KICK), NGS:8933-8940
        const int f = ra_oct_check(q, x, flag);
        RANoise nz{};
        if constexpr (MODEL == 0) {
            const int k = 2 * (t - t0);
            nz = lds.noise[q == 0 ? at[k] : (q == 5 ? at[k + 1] : kNoiseRows - 1)];
        } else {
            // HH2_buffer noise checks (Gi_s, Gi_d, Ge_s, Ge_d), as listed
            nc.take(t, [&](int g, double inc) {
                GA = (g == 0 && q == 0) || (g == 3 && q == 5) ? GA + inc : GA;
                GB = (g == 2 && q == 0) || (g == 1 && q == 5) ? GB + inc : GB;
            });
        }
        ra_oct_step<MODEL>(L, x, GA, GB, dt, nz, win.row(t));
        if (live && f) mask |= 1ull << (t - t0);
    }
    const int new_posts = ra_window_logs(nd, win, posts, i, t0, q == 0 ? mask : 0, q == 5 ? mask : 0, listed0, listed1);
    const int fd = __shfl(flag, (lane & ~7) + 5);
    if (live && (MODEL == 0 || q != 3)) xp[i] = x;
    if (soma || dend) {
        gap[i] = GA;
        gbp[i] = GB;
        (soma ? nd.soma_mask : nd.dend_mask)[i] = mask;
    }
    if (soma) {
        nd.ra_flags[i] = flag | (fd << 1);
        if (growth) nd.post_pend[i] = new_posts;
        if (MODEL == 1 && nd.ra_poisson) nd.ra_ev_pos[i] = nc.pos;
    }
}
#endif

// Reads one word of every 64-byte line of the launch arguments, all at once:
// the neuron functions read them in several rounds, and the first wave of a
// compute unit would wait for a line of them in each.
__device__ __forceinline__ void kernarg_touch(const NetDev& nd)
{
    constexpr int kLines = (int)(sizeof(NetDev) / 64);
    const int* w = (const int*)&nd;
    int x[kLines];
#pragma unroll
    for (int k = 0; k < kLines; ++k) x[k] = w[16 * k];
#pragma unroll
    for (int k = 0; k < kLines; ++k) asm volatile("" ::"s"(x[k]));
}

// blocks [0, iblocks) integrate HVC-I, the next rblocks HVC-RA, in the layout
// of LANES; any blocks after them run the previous window's sync-point STDP
// (one row per thread, sa).
// LANES: HVC-I bit 0 = five lanes, bit 2 = four lanes, bit 3 = eight lanes per
// neuron, bit 4 = eight lanes with the one-thread arithmetic (FP32 form), none
// = one thread; HVC-RA bit 1 = four lanes (FP32 form) or eight (FP64 form),
// bit 5 = four lanes (FP64 form), else one thread.  (The layouts are template
// parameters: a kernel holds the register allocation of one layout only.)
template <int RA_MODEL, int I_MODEL, int LANES>
__global__ __launch_bounds__(256) void k_integrate(NetDev nd, int t0, int t1, int iblocks, int rblocks, StdpArgs sa)
{
    if ((int)blockIdx.x >= iblocks + rblocks) {
        __shared__ uint64_t stdp_slice[kStdpSliceCap];
        __shared__ int stdp_count;
        stdp_block(nd, sa, ((int)blockIdx.x - iblocks - rblocks) * blockDim.x, stdp_slice, &stdp_count);
        return;
    }
    kernarg_touch(nd);
    // the window's decay rows and clock, staged in LDS (dynamic shared memory of
    // win_bytes(t1 - t0 + 1) bytes) by Win::stage in the neuron functions
    extern __shared__ __attribute__((aligned(16))) double win_lds[];
    const int nsteps = t1 - t0 + 1;
    const Win win{(const WinRow*)win_lds, (const double*)((const WinRow*)win_lds + nsteps), t0, win_lds, nsteps};
    const int iwave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int rwave = (blockIdx.x - iblocks) * (blockDim.x >> 6) + (threadIdx.x >> 6);
#ifdef HVC_FP32
    if ((int)blockIdx.x < iblocks) {
        if constexpr ((LANES & 16) != 0)
            integrate_i_oct<IOctShared>(nd, win, iwave, t0, t1);
        else if constexpr ((LANES & 8) != 0)
            integrate_i_oct<GateSlot>(nd, win, iwave, t0, t1);
        else if constexpr ((LANES & 4) != 0)
            integrate_i_quad(nd, win, iwave, t0, t1);
        else if constexpr ((LANES & 1) != 0)
            integrate_i_lanes(nd, win, iwave, t0, t1);
        else
            integrate_i_thread<I_MODEL>(nd, win, blockIdx.x * blockDim.x + threadIdx.x, t0, t1);
    } else {
        if constexpr ((LANES & 2) != 0)
            integrate_ra<RA_MODEL, true>(nd, win, rwave, t0, t1);
        else
            integrate_ra<RA_MODEL, false>(nd, win, (blockIdx.x - iblocks) * blockDim.x + threadIdx.x, t0, t1);
    }
#else
    __shared__ ExpPair exp_tab[64];
    __shared__ RANoise noise_rows[RA_MODEL == 0 && (LANES & 2) ? kNoiseRows : 1];
    __shared__ uint8_t noise_at[RA_MODEL == 0 && (LANES & 2) ? 256 / 8 * 2 * kMaxWindowSteps : 1];
    const OctLds lds{exp_tab, noise_rows, noise_at};
    if ((int)blockIdx.x < iblocks) {
        if constexpr ((LANES & 8) != 0)
            integrate_i_oct(nd, win, lds, iwave, t0, t1);
        else
            integrate_i_thread<I_MODEL>(nd, win, blockIdx.x * blockDim.x + threadIdx.x, t0, t1);
    } else {
        if constexpr ((LANES & 2) != 0)
            integrate_ra_oct<RA_MODEL>(nd, win, lds, rwave, t0, t1);
        else if constexpr ((LANES & 32) != 0)
            integrate_ra<RA_MODEL, true>(nd, win, rwave, t0, t1);
        else
            integrate_ra<RA_MODEL, false>(nd, win, (blockIdx.x - iblocks) * blockDim.x + threadIdx.x, t0, t1);
    }
#endif
}

// ---------------------------------------------------------------------------
// single-neuron traces.  A trace is one serial chain of steps per neuron, so
// what a step waits on is what it costs: the decay rows and the clock of
// kTraceChunk steps are staged in LDS, and a step's inputs are loaded a step
// ahead (one thread per neuron) or with the chunk (octets).  One wave per block,
// said so to the compiler (without launch bounds the kernels were held to 128
// registers and spilled 640-780 bytes).  Whole calls, before and now: 16
// HVC-RA neurons x 500 steps FP64 5.6 -> 1.5 ms, 330 HVC-I x 1 250 FP64 33 ->
// 6.8 ms (both octets), 2 000 HVC-RA x 1 500 FP32 (one thread) 3.5 -> 2.2 ms.
// ---------------------------------------------------------------------------
constexpr int kTraceChunk = 32;
constexpr size_t kTraceLds = kTraceChunk * sizeof(WinRow) + (kTraceChunk + 1) * sizeof(double);

// the chunk's tables for the steps t0 .. t1, staged by the block
__device__ __forceinline__ Win trace_window(const NetDev& nd, double* lds, int t0, int t1)
{
    const int nsteps = t1 - t0 + 1;
    const Win win{(const WinRow*)lds, (const double*)((const WinRow*)lds + nsteps), t0, lds, nsteps};
    __syncthreads();   // the previous chunk's tables are done with
    win.stage(nd);
    return win;
}

// the four Poisson channels of an HVC-RA trace (HH2_buffer's initial draws and checks)
struct RATraceNoise {
    PoissonStream ps;
    double nes, nis, ned, nid;
    __device__ __forceinline__ RATraceNoise(const NetDev& nd, uint32_t trial, int k)
        : ps{nd.seed_lo, nd.seed_hi, trial, kStreamRAPoisson, (uint32_t)k, 0u}, nes(0), nis(0), ned(0), nid(0)
    {
        if (nd.ra_poisson) {
            nes = 1000.0 * ps.spike_time(100.0);
            nis = 1000.0 * ps.spike_time(100.0);
            ned = 1000.0 * ps.spike_time(100.0);
            nid = 1000.0 * ps.spike_time(100.0);
        }
    }
    __device__ __forceinline__ void check(double time, double dt, real& Ge_s, real& Gi_s, real& Ge_d, real& Gi_d)
    {
        ra_noise_check(ps, time, dt, Gi_s, 0.035, nis);
        ra_noise_check(ps, time, dt, Gi_d, 0.045, nid);
        ra_noise_check(ps, time, dt, Ge_s, 0.035, nes);
        ra_noise_check(ps, time, dt, Ge_d, 0.045, ned);
    }
};

__global__ __launch_bounds__(64) void k_trace_ra(NetDev nd, int n, int n_steps, uint32_t trial, const double* EL,
                                                 const double* GCa, const double* kick, const double* exc_w,
                                                 const double* inh_g, double* out, uint8_t* fired_out)
{
    extern __shared__ __attribute__((aligned(16))) double trace_lds[];
    const int k0 = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = k0 < n;
    const int k = live ? k0 : n - 1;
    const RAUniform u = ra_uniform(nd);
    // HH2_test::set_to_rest (HH2_test.cpp:196-205)
    RAState s;
    HVC_LOAD(s, Vs, -79.97619025) HVC_LOAD(s, Vd, -79.97268759) HVC_LOAD(s, n, 0.01101284)
    HVC_LOAD(s, l, 0.0) HVC_LOAD(s, h, 0.9932845) HVC_LOAD(s, r, 0.00055429)
    HVC_LOAD(s, c, 0.00000261762353) HVC_LOAD(s, Ca, 0.01689572)
    s.Ge_s = 0; s.Gi_s = 0; s.Ge_d = 0; s.Gi_d = 0;
    int fs = 0, fd = 0;
    const real el = (real)EL[k], gca = (real)GCa[k];
    RATraceNoise pn(nd, trial, k);
    auto dump = [&](int row) {
        if (!live) return;
        double* o = out + ((size_t)row * n + k) * 12;
        o[0] = HVC_WIDE(s, Vs); o[1] = HVC_WIDE(s, Vd); o[2] = HVC_WIDE(s, n); o[3] = HVC_WIDE(s, l);
        o[4] = HVC_WIDE(s, h); o[5] = HVC_WIDE(s, r); o[6] = HVC_WIDE(s, c); o[7] = HVC_WIDE(s, Ca);
        o[8] = s.Ge_s; o[9] = s.Gi_s; o[10] = s.Ge_d; o[11] = s.Gi_d;
    };
    dump(0);
    double kk = kick[k], ig = inh_g[k], ew = exc_w[k];   // the next step's inputs
    for (int t0 = 1; t0 <= n_steps; t0 += kTraceChunk) {
        const int t1 = min(t0 + kTraceChunk - 1, n_steps);
        const Win win = trace_window(nd, trace_lds, t0, t1);
        for (int t = t0; t <= t1; ++t) {
            const size_t idx = (size_t)(t - 1) * n + k, nxt = (size_t)min(t, n_steps - 1) * n + k;
            const double kn = kick[nxt], in = inh_g[nxt], en = exc_w[nxt];
            if (kk != 0.0) s.Ge_d += kk;
            int f = ra_state_check(s.Vs, s.Vd, fs, fd);
            const WinRow& row = win.row(t);
            if (nd.ra_model == 0) {
                U4 o = philox4x32((uint32_t)t, (uint32_t)k, trial, kStreamRAWhite, nd.seed_lo, nd.seed_hi);
                ra_step_debraband(s, el, gca, u, kPointDistribution[point_index(o.x)],
                                  kPointDistribution[point_index(o.y)], kPointDistribution[point_index(o.z)],
                                  kPointDistribution[point_index(o.w)], row.e5[kOffDt], row.e5[kOffHalf]);
            } else {
                if (nd.ra_poisson) pn.check(win.clk(t - 1), nd.dt, s.Ge_s, s.Gi_s, s.Ge_d, s.Gi_d);
                ra_step_runge4(s, el, gca, u, row.e5[kOffThird], row.e5[kOffTwoThird], row.e5[kOffDt]);
            }
            if (live) fired_out[idx] = (uint8_t)f;
            if (ig != 0.0) s.Gi_d += ig;
            if (ew != 0.0) s.Ge_d += ew / 10000.0;
            dump(t);
            kk = kn;
            ig = in;
            ew = en;
        }
    }
}

__global__ __launch_bounds__(64) void k_trace_i(NetDev nd, int n, int n_steps, int first_trial, uint32_t trial,
                                                const double* exc_g, const double* inh_g, double* out,
                                                uint8_t* fired_out)
{
    extern __shared__ __attribute__((aligned(16))) double trace_lds[];
    const int k0 = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = k0 < n;
    const int k = live ? k0 : n - 1;
    // HHI_buffer::set_to_rest (HHI_buffer.cpp:181-185)
    IState s;
    HVC_LOAD(s, V, -66.0) HVC_LOAD(s, n, 0.125) HVC_LOAD(s, m, 0.0) HVC_LOAD(s, h, 0.99) HVC_LOAD(s, w, 0.0)
    s.Ge = 0; s.Gi = 0;
    int flag = 0;
    PoissonStream ps{nd.seed_lo, nd.seed_hi, trial, kStreamIPoisson, (uint32_t)k, 0u};
    double ne = 0, ni = 0;
    if (nd.i_poisson) {
        double init_dt = first_trial ? 0.0 : nd.dt;
        ne = i_init_noise(ps, init_dt);
        ni = i_init_noise(ps, init_dt);
    }
    auto dump = [&](int row) {
        if (!live) return;
        double* o = out + ((size_t)row * n + k) * 7;
        o[0] = HVC_WIDE(s, V); o[1] = HVC_WIDE(s, n); o[2] = HVC_WIDE(s, m); o[3] = HVC_WIDE(s, h);
        o[4] = HVC_WIDE(s, w); o[5] = s.Ge; o[6] = s.Gi;
    };
    dump(0);
    double ig = inh_g[k], eg = exc_g[k];   // the next step's inputs
    for (int t0 = 1; t0 <= n_steps; t0 += kTraceChunk) {
        const int t1 = min(t0 + kTraceChunk - 1, n_steps);
        const Win win = trace_window(nd, trace_lds, t0, t1);
        for (int t = t0; t <= t1; ++t) {
            const size_t idx = (size_t)(t - 1) * n + k, nxt = (size_t)min(t, n_steps - 1) * n + k;
            const double in = inh_g[nxt], en = exc_g[nxt];
            int f = i_state_check(s.V, flag);
            if (nd.i_poisson) {
                const double time = win.clk(t - 1);
                i_noise_check(ps, time, nd.dt, s.Ge, ne);
                i_noise_check(ps, time, nd.dt, s.Gi, ni);
            }
            if (nd.i_model == 0)
                i_step<0>(s, nd.dt, win.row(t));
            else
                i_step<1>(s, (real)nd.dt, win.row(t));
            if (live) fired_out[idx] = (uint8_t)f;
            if (ig != 0.0) s.Gi += ig;
            if (eg != 0.0) s.Ge += eg;
            dump(t);
            ig = in;
            eg = en;
        }
    }
}

#ifndef HVC_FP32
// Traces on octets: eight neurons per block.  Lane q stores its own variable;
// lane 0 (HVC-RA: lanes 0 and 5) also stores the conductances.
__device__ __forceinline__ void trace_inputs(double* lds, const double* src, int k0, int n, int t0, int t1)
{
    for (int r = threadIdx.x; r < 8 * (t1 - t0 + 1); r += blockDim.x)
        lds[r] = src[(size_t)(t0 - 1 + (r >> 3)) * n + min(k0 + (r & 7), n - 1)];
}

template <int MODEL>
__global__ __launch_bounds__(64) void k_trace_ra_oct(NetDev nd, int n, int n_steps, uint32_t trial, const double* EL,
                                                     const double* GCa, const double* kick, const double* exc_w,
                                                     const double* inh_g, double* out, uint8_t* fired_out)
{
    extern __shared__ __attribute__((aligned(16))) double trace_lds[];
    __shared__ ExpPair exp_tab[64];
    __shared__ RANoise noise_rows[MODEL == 0 ? kNoiseRows : 1];
    __shared__ uint8_t noise_at[8 * 2 * kTraceChunk];
    __shared__ double in_kick[8 * kTraceChunk], in_exc[8 * kTraceChunk], in_inh[8 * kTraceChunk];
    const int lane = threadIdx.x, q = lane & 7, g = lane >> 3;
    const bool live = (int)blockIdx.x * 8 + g < n;
    const int k = live ? blockIdx.x * 8 + g : n - 1;
    exp_table_store(exp_tab, exp_table_load());
    if constexpr (MODEL == 0) stage_noise_rows(noise_rows, nd.sq_sig_s, nd.sq_sig_d);
    const RAOctLane L = ra_oct_lane<MODEL>(q, EL[k], GCa[k], nd.mu_term_s, nd.mu_term_d, exp_tab);
    // HH2_test::set_to_rest (HH2_test.cpp:196-205), by state variable
    const int var = ra_oct_var(q);
    double x = var == 0 ? -79.97619025 : var == 1 ? -79.97268759 : var == 2 ? 0.01101284 : var == 3 ? 0.0
             : var == 4 ? 0.9932845 : var == 5 ? 0.00055429 : var == 6 ? 0.00000261762353 : 0.01689572;
    double GA = 0, GB = 0;   // Gi_s, Ge_s in lane 0; Ge_d, Gi_d in lane 5
    int flag = 0;
    RATraceNoise pn(nd, trial, k);
    const NoiseId sid{nd.seed_lo, nd.seed_hi, trial, (uint32_t)k};
    auto dump = [&](int row) {
        if (!live) return;
        double* o = out + ((size_t)row * n + k) * 12;
        o[var] = MODEL == 1 && q == 3 ? 0.0 : x;
        if (q == 0) { o[8] = GB; o[9] = GA; }
        if (q == 5) { o[10] = GA; o[11] = GB; }
    };
    dump(0);
    for (int t0 = 1; t0 <= n_steps; t0 += kTraceChunk) {
        const int t1 = min(t0 + kTraceChunk - 1, n_steps);
        __syncthreads();
        trace_inputs(in_kick, kick, blockIdx.x * 8, n, t0, t1);
        trace_inputs(in_exc, exc_w, blockIdx.x * 8, n, t0, t1);
        trace_inputs(in_inh, inh_g, blockIdx.x * 8, n, t0, t1);
        uint8_t* at = noise_at + g * 2 * kTraceChunk;
        if constexpr (MODEL == 0) noise_window(at, q, sid, t0, t1 - t0 + 1);
        const Win win = trace_window(nd, trace_lds, t0, t1);
        for (int t = t0; t <= t1; ++t) {
            const int r = (t - t0) * 8 + g;
            const double kk = in_kick[r], ig = in_inh[r], ew = in_exc[r];
            if (q == 5 && kk != 0.0) GA += kk;
            const int f = ra_oct_check(q, x, flag);
            RANoise nz{};
            if constexpr (MODEL == 0) {
                const int j = 2 * (t - t0);
                nz = noise_rows[q == 0 ? at[j] : (q == 5 ? at[j + 1] : kNoiseRows - 1)];
            } else if (nd.ra_poisson) {
                double other = 0.0;
                const bool dend = q == 5;
                double ges = dend ? other : GB, gis = dend ? other : GA, ged = dend ? GA : other, gid = dend ? GB : other;
                pn.check(win.clk(t - 1), nd.dt, ges, gis, ged, gid);
                GA = dend ? ged : gis;
                GB = dend ? gid : ges;
            }
            ra_oct_step<MODEL>(L, x, GA, GB, nd.dt, nz, win.row(t));
            const uint64_t fired = __ballot(f != 0) >> (lane & ~7);
            if (live && q == 0)
                fired_out[(size_t)(t - 1) * n + k] = (uint8_t)((fired & 1u) | ((fired >> 4) & 2u));
            if (q == 5) {
                if (ig != 0.0) GB += ig;
                if (ew != 0.0) GA += ew / 10000.0;
            }
            dump(t);
        }
    }
}

__global__ __launch_bounds__(64) void k_trace_i_oct(NetDev nd, int n, int n_steps, int first_trial, uint32_t trial,
                                                    const double* exc_g, const double* inh_g, double* out,
                                                    uint8_t* fired_out)
{
    extern __shared__ __attribute__((aligned(16))) double trace_lds[];
    __shared__ ExpPair exp_tab[64];
    __shared__ double in_exc[8 * kTraceChunk], in_inh[8 * kTraceChunk];
    const int lane = threadIdx.x, q = lane & 7, g = lane >> 3;
    const bool live = (int)blockIdx.x * 8 + g < n;
    const int k = live ? blockIdx.x * 8 + g : n - 1;
    exp_table_store(exp_tab, exp_table_load());
    const IOctLane L = i_oct_lane(q, exp_tab);
    // HHI_buffer::set_to_rest (HHI_buffer.cpp:181-185), by state variable; the
    // mirror lanes 4-6 carry 1 - x
    const int var = i_oct_var(q);
    double x = var == 0 ? -66.0 : var == 1 ? 0.125 : var == 2 ? 0.0 : var == 3 ? 0.99 : 0.0;
    if (q > 3 && q < 7) x = 1 - x;
    double Ge = 0, Gi = 0;
    int flag = 0;
    PoissonStream ps{nd.seed_lo, nd.seed_hi, trial, kStreamIPoisson, (uint32_t)k, 0u};
    double ne = 0, ni = 0;
    if (nd.i_poisson) {
        double init_dt = first_trial ? 0.0 : nd.dt;
        ne = i_init_noise(ps, init_dt);
        ni = i_init_noise(ps, init_dt);
    }
    auto dump = [&](int row) {
        double* o = out + ((size_t)row * n + k) * 7;
        if (live && (q < 4 || q == 7)) o[var] = x;
        if (live && q == 0) { o[5] = Ge; o[6] = Gi; }
    };
    dump(0);
    Dp8Consts C;
    dp8_pin(C);
    for (int t0 = 1; t0 <= n_steps; t0 += kTraceChunk) {
        const int t1 = min(t0 + kTraceChunk - 1, n_steps);
        __syncthreads();
        trace_inputs(in_exc, exc_g, blockIdx.x * 8, n, t0, t1);
        trace_inputs(in_inh, inh_g, blockIdx.x * 8, n, t0, t1);
        const Win win = trace_window(nd, trace_lds, t0, t1);
        for (int t = t0; t <= t1; ++t) {
            const int r = (t - t0) * 8 + g;
            const double ig = in_inh[r], eg = in_exc[r];
            const int f = i_state_check(x, flag);   // of V in lane 0
            if (nd.i_poisson) {
                const double time = win.clk(t - 1);
                i_noise_check(ps, time, nd.dt, Ge, ne);
                i_noise_check(ps, time, nd.dt, Gi, ni);
            }
            i_oct_step(L, C, x, Ge, Gi, nd.dt, win.row(t));
            if (live && q == 0) fired_out[(size_t)(t - 1) * n + k] = (uint8_t)f;
            if (ig != 0.0) Gi += ig;
            if (eg != 0.0) Ge += eg;
            dump(t);
        }
    }
}
#endif

// LDS bytes of k_integrate for a window of n steps
static inline size_t win_bytes(int n) { return (size_t)n * sizeof(WinRow) + (size_t)(n + 1) * sizeof(double); }

}  // namespace p32 / p64

#ifdef HVC_FP32
// HVC-I neurons per context up to which "one thread per neuron" runs on eight
// lanes with the one-thread stepper's arithmetic.  k_integrate per window
// (HVC-RA one thread per neuron beside it, 3.6 times as many; the launch
// included), octets / one thread, us: 25 / 41 at 2 750 HVC-I neurons, 35 / 42
// at 8 745, 41 / 42 at 12 400, 43 / 43 at 16 000.
constexpr int kIOctSharedMaxNeurons = 10240;
#else
// HVC-RA neurons per context up to which a window takes octets without being
// asked.  An octet's wave is short (640 instructions per Debraband step, the
// one-thread wave 5 600 before the two-operation quotients, 4 700 with them)
// but eight times as many are needed.  k_integrate per window beside HVC-I
// octets (n / 3.6 of them), octets / one thread, us: Debraband 81 / 102 at
// 20 000 neurons, 105 / 118 at 30 000, 119 / 120 at 34 000, 135 / 121 at
// 40 000; RK4 76 / 79 at 20 000, 83 / 98 at 24 000, 87 / 98 at 26 000, 99 / 98
// at 28 000, 128 / 99 at 40 000.  (The 20 000 + 5 500 RK4 growth trial in the
// default shape: 164 ms with octets, 172 with one thread.)
constexpr int kRAOctMaxNeurons[2] = {32768, 26624};   // by ra_model
// HVC-RA neurons up to which "several lanes" is eight in the RK4 model, above
// which it is four: half the waves, so two to a SIMD hold out to 21 000 neurons
// instead of 13 000.  k_integrate per window beside HVC-I octets, four lanes /
// eight / one thread, us: 59 / 49 / 77 at 12 000 neurons, 60 / 57 / 77 at
// 14 000, 60 / 71 / 77 at 16 000, 61 / 76 / 79 at 20 000, 87 / 82 / 98 at
// 22 000, 88 / 99 / 98 at 28 000, 111 / 110 / 98 at 32 000.
constexpr int kRAOctMaxOverQuads = 14336;

int ra_lanes_f64(int ra_model, int n_ra, int ra_lanes)
{
    if (ra_model == 1 && ra_lanes) return n_ra <= kRAOctMaxOverQuads ? 8 : 4;
    return ra_lanes || n_ra <= kRAOctMaxNeurons[ra_model == 1] ? 8 : 1;
}
// neurons up to which a trace takes octets (a trace has no launch shape and no
// other neurons beside it), octets / one thread: hvc_trace_ra_noalloc over 64
// steps, us: Debraband 212 / 530 at 8 000 neurons, 270 / 536 at 16 000, 537 /
// 568 at 28 000, 559 / 572 at 32 000, 687 / 591 at 40 000; RK4 223 / 475 at
// 8 000, 485 / 517 at 28 000, 566 / 522 at 32 000; hvc_trace_i over 40 steps, ms,
// most of it the copies: 1.80 / 2.30 at 8 000, 6.8 / 6.9 at 24 000, 8.3 / 8.3 at
// 28 000, 11.2 / 10.9 at 40 000.
constexpr int kRAOctMaxTraces[2] = {32768, 28672};   // by ra_model
constexpr int kIOctMaxTraces = 24576;
#endif

#ifdef HVC_FP32
#define HVC_LAUNCHER(name) name##_f32
#else
#define HVC_LAUNCHER(name) name
#endif

void HVC_LAUNCHER(launch_trace_ra)(hipStream_t st, const NetDev& nd, int n, int n_steps, uint32_t trial, const double* EL,
                     const double* GCa, const double* kick, const double* exc_w, const double* inh_g, double* out,
                     uint8_t* fired)
{
#ifndef HVC_FP32
    if (n <= kRAOctMaxTraces[nd.ra_model == 1]) {
        if (nd.ra_model == 0)
            k_trace_ra_oct<0><<<blocks_for(n, 8), 64, kTraceLds, st>>>(nd, n, n_steps, trial, EL, GCa, kick, exc_w,
                                                                       inh_g, out, fired);
        else
            k_trace_ra_oct<1><<<blocks_for(n, 8), 64, kTraceLds, st>>>(nd, n, n_steps, trial, EL, GCa, kick, exc_w,
                                                                       inh_g, out, fired);
        return;
    }
#endif
    k_trace_ra<<<blocks_for(n, 64), 64, kTraceLds, st>>>(nd, n, n_steps, trial, EL, GCa, kick, exc_w, inh_g, out,
                                                         fired);
}

void HVC_LAUNCHER(launch_trace_i)(hipStream_t st, const NetDev& nd, int n, int n_steps, int first_trial, uint32_t trial,
                    const double* exc_g, const double* inh_g, double* out, uint8_t* fired)
{
#ifndef HVC_FP32
    if (nd.i_model == 0 && n <= kIOctMaxTraces) {
        k_trace_i_oct<<<blocks_for(n, 8), 64, kTraceLds, st>>>(nd, n, n_steps, first_trial, trial, exc_g, inh_g, out,
                                                               fired);
        return;
    }
#endif
    k_trace_i<<<blocks_for(n, 64), 64, kTraceLds, st>>>(nd, n, n_steps, first_trial, trial, exc_g, inh_g, out, fired);
}

void HVC_LAUNCHER(launch_integrate)(hipStream_t st, const NetDev& nd, int t0, int t1, const Tuning& tu,
                                     const StdpArgs& sa, int stdp)
{
    const int bs = tu.integrate_block;
    const int wpb = bs / 64;
#ifdef HVC_FP32
    // HVC-I layout (DP8 only): 0 one thread, 1 five lanes, 2 four lanes, 3 eight lanes per neuron
    // (or 4: the one-thread form's arithmetic on eight lanes, while the HVC-I
    // waves of that layout still find SIMDs to run on)
    const int i_layout = nd.i_model != 0 ? 0 : (tu.i_lanes == 0 && nd.n_i <= kIOctSharedMaxNeurons ? 4 : tu.i_lanes);
    const int ra_lanes = (nd.ra_model == 1 && tu.ra_lanes) ? 1 : 0;
    const int ra_per_block = ra_lanes ? wpb * kRANeuronsPerWave : bs;
    const int i_per_block = i_layout == 1 ? wpb * kINeuronsPerWave
                            : (i_layout == 2 ? wpb * kINeuronsPerQuadWave
                                             : (i_layout >= 3 ? wpb * kINeuronsPerOctWave : bs));
#else
    // the FP64 layouts give the same bits, so every HVC-I layout with several
    // lanes is the octet (45 us per window at 2 000 + 550 neurons; the four-lane
    // and the earlier eight-lane form took 84 and 67 us)
    const int i_layout = nd.i_model == 0 && tu.i_lanes ? 3 : 0;
    const int ra_layout = ra_lanes_f64(nd.ra_model, nd.n_ra, tu.ra_lanes);
    const int ra_per_block = ra_layout == 8 ? wpb * kRAOctNeuronsPerWave : (ra_layout == 4 ? wpb * kRANeuronsPerWave : bs);
    const int i_per_block = i_layout ? wpb * kINeuronsPerOctWave : bs;
#endif
    int iblocks = nd.n_i == 0 ? 0 : (nd.n_i + i_per_block - 1) / i_per_block;
    int rblocks = blocks_for(nd.n_ra, ra_per_block);
    const int sblocks = stdp ? blocks_for(nd.n_ra, bs) : 0;
    dim3 grid(iblocks + rblocks + sblocks);
    const size_t lds = win_bytes(t1 - t0 + 1);
#define HVC_K(R, I, L) k_integrate<R, I, L><<<grid, bs, lds, st>>>(nd, t0, t1, iblocks, rblocks, sa)
#ifdef HVC_FP32
    if (nd.ra_model == 0) {
        if (nd.i_model == 1) HVC_K(0, 1, 0);
        else if (i_layout == 4) HVC_K(0, 0, 16);
        else if (i_layout == 3) HVC_K(0, 0, 8);
        else if (i_layout == 2) HVC_K(0, 0, 4);
        else if (i_layout == 1) HVC_K(0, 0, 1);
        else HVC_K(0, 0, 0);
    } else if (ra_lanes) {
        if (nd.i_model == 1) HVC_K(1, 1, 2);
        else if (i_layout == 4) HVC_K(1, 0, 18);
        else if (i_layout == 3) HVC_K(1, 0, 10);
        else if (i_layout == 2) HVC_K(1, 0, 6);
        else if (i_layout == 1) HVC_K(1, 0, 3);
        else HVC_K(1, 0, 2);
    } else {
        if (nd.i_model == 1) HVC_K(1, 1, 0);
        else if (i_layout == 4) HVC_K(1, 0, 16);
        else if (i_layout == 3) HVC_K(1, 0, 8);
        else if (i_layout == 2) HVC_K(1, 0, 4);
        else if (i_layout == 1) HVC_K(1, 0, 1);
        else HVC_K(1, 0, 0);
    }
#else
    // (four lanes come up with RK4 only)
#define HVC_KR(R)                                     \
    if (nd.i_model == 1) {                            \
        if (ra_layout == 8) HVC_K(R, 1, 2);           \
        else if (ra_layout == 4) HVC_K(1, 1, 32);     \
        else HVC_K(R, 1, 0);                          \
    } else if (i_layout) {                            \
        if (ra_layout == 8) HVC_K(R, 0, 10);          \
        else if (ra_layout == 4) HVC_K(1, 0, 40);     \
        else HVC_K(R, 0, 8);                          \
    } else {                                          \
        if (ra_layout == 8) HVC_K(R, 0, 2);           \
        else if (ra_layout == 4) HVC_K(1, 0, 32);     \
        else HVC_K(R, 0, 0);                          \
    }
    if (nd.ra_model == 0) {
        HVC_KR(0)
    } else {
        HVC_KR(1)
    }
#undef HVC_KR
#endif
#undef HVC_K
}

#undef HVC_LAUNCHER

}  // namespace hvc
