// run1d.hpp -- many RK2 steps of a 1-D block in one launch (mara_block_run,
// mara_block_advance), and of the 1-D solves of a batch (mara_batch_step,
// kb_run1d: the serving mix of 48 solves, 240 steps each, 60 -> 50 ms, the 1-D
// solves' share no longer the longest).
//
// A 1-D step is small: at 1024 zones its two stage kernels and the step
// boundary were 14 us of launches and memory latency around 1 us of
// arithmetic.  Here the block stays on chip for the whole run.  A thread owns
// one zone, whose primitives and conserved state live in its registers; the
// stencil and the fluxes go through LDS; time step, clock and stop condition
// are computed by every work-group alike.  Nothing is read from memory inside
// the loop but what other work-groups send.
//
// Blocks that fit one work-group (up to ONE_MAX zones) exchange nothing: guard
// zones are images of interior zones, written beside them in LDS.  Longer
// blocks are split evenly over work-groups of 256 threads that keep a halo of
// 2 NG zones per side and advance it along in the first stage, so neighbours
// meet once per step: each sends its edge zones and its CFL minimum, and
// receives its halo and everybody's minimum.  Up to GROUPS_MAX work-groups
// (49 600 zones with PLM), which leaves CUs free beside a run; longer blocks
// go by launches per stage.
//
// Measured, us per step, launches (replayed from a graph) -> this: hydro HLLE
// 100 zones 12.5 -> 3.9, 1024 14.5 -> 5.9, 10 007 14.2 -> 5.9, 49 600 14.4 ->
// 7.1; MHD 1024 19.2 -> 10.2; mixed hydro 1024 12.2 -> 4.7.  One exchange
// costs about 2 us; all work-groups on one XCD exchange no faster (and 32 CUs
// hold no more than 32 k zones), so they are spread.  What bounds a step now
// is the latency of its dependent arithmetic at one wavefront per SIMD.
//
// Messages are 64-bit words in device memory that validate themselves: a slot
// holds EMPTY until the word is stored (relaxed, device scope), so one store
// and one polling load carry it, with no flag and no fence between them.  Of
// three slots in rotation, step k uses k % 3 and clears (k + 1) % 3, whose
// words everybody has read (whoever published step k - 1 had finished reading
// step k - 2); the clears are complete (vmcnt 0, barrier) before the
// work-group's minimum of step k is published, and nobody polls slot
// (k + 1) % 3 before having read that minimum.
//
// The work-groups must be resident together, which a plain launch does not
// promise (other work may hold the CUs).  A wait is therefore bounded, and
// the block's arrays and control block are written only at the end: whoever
// gives up moves the decision word from OPEN to GAVE_UP, whoever has passed
// the last exchange moves it from OPEN to DONE, and only DONE writes results.
// After GAVE_UP nothing has changed and the host takes the launches per
// stage.
//
// The arithmetic is pencil_tile's and finish_zone's, function for function,
// so a run is the same bit for bit (a zone whose recovery fails keeps the
// previous value of the buffer the stage writes, as there).
#pragma once

#include <type_traits>

#include "../../include/mara_gpu.h"
#include "kernels.hpp"

namespace mara {
namespace run1d {

constexpr int PL = 256;          // threads of a work-group of a split block
constexpr int GROUPS_MAX = 200;
constexpr int SLOTS = 3;
constexpr unsigned long long EMPTY = 0xfff7a5a5c3c35a5aull;  // a NaN no arithmetic produces
enum : unsigned { OPEN = 0, DONE = 1, GAVE_UP = 2 };
// polls of one word before giving up: about half a second
constexpr int PATIENCE = 1 << 19;

// words one work-group sends per step: its CFL minimum, then its left and
// right edge zones
template <int Law, int Recon> struct Message
{
    static constexpr int H = 2 * Stencil<Recon>::NG;
    static constexpr int EDGE = H * LawNQ<Law>::value;
    static constexpr int WORDS = 1 + 2 * EDGE;
};

__device__ __forceinline__ void post(unsigned long long* p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ unsigned long long peek(const unsigned long long* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a double as a message word (a NaN with EMPTY's bits becomes another NaN)
__device__ __forceinline__ unsigned long long word(double x)
{
    const unsigned long long b = dbits(x);
    return b == EMPTY ? b ^ 1ull : b;
}

// Waits for a word; false if somebody gave up, or after `patience` polls.
__device__ __forceinline__ bool receive(const unsigned long long* p, const unsigned* decision, int patience,
                                        unsigned long long& v)
{
    for (int n = 0; n < patience; ++n)
    {
        v = peek(p);
        if (v != EMPTY) return true;
        if ((n & 255) == 255
            && __hip_atomic_load(decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == GAVE_UP)
            return false;
    }
    return false;
}

// The box and the decision word, before each launch.
static __global__ void __launch_bounds__(256) k_run1d_open(unsigned long long* __restrict__ box, int words,
                                                           unsigned* __restrict__ decision)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < words) box[t] = EMPTY;
    if (t == 0) *decision = OPEN;
}

// The control block, complete in memory, into its copy in host memory, for the
// host to read after the stream has drained (no transfer of its own).
__device__ __forceinline__ void report(const Ctl* ctl, Ctl* host, int m)
{
    constexpr int WORDS = sizeof(Ctl) / 8;
    static_assert(sizeof(Ctl) % 8 == 0, "Ctl is copied in 8-byte words");
    if (m < WORDS)
        reinterpret_cast<unsigned long long*>(host)[m] = peek(reinterpret_cast<const unsigned long long*>(ctl) + m);
}

// Up to max_steps steps of the device-driven loop of k_ctl_step_start /
// k_ctl_step_next, or (given) one step of size dt_given as
// k_ctl_begin_advance starts it, with the control block's copy left in host
// memory.  ONE: a block of one work-group of THREADS threads; only such a
// block takes given steps.
// w of groups: this work-group's part.
template <int Law, int Recon, int Riem, typename R, bool CT, int THREADS, bool ONE>
__device__ __forceinline__ void run(double* __restrict__ Pa, double* __restrict__ Pb, const Geom& G,
                                    Ctl* __restrict__ ctl, int w, int groups, int max_steps, int given,
                                    double dt_given, unsigned long long* __restrict__ box,
                                    unsigned* __restrict__ decision, int patience, Ctl* __restrict__ host)
{
    constexpr int NQ = LawNQ<Law>::value, NG = Stencil<Recon>::NG;
    constexpr int LO = ONE ? NG : 2 * NG;  // local index of the first own zone
    constexpr int WAVES = THREADS / 64;
    using Msg = Message<Law, Recon>;
    __shared__ R sP[NQ][THREADS];
    __shared__ R sF[NQ][THREADS];
    __shared__ double wmin[WAVES];
    __shared__ int wfail[WAVES];
    __shared__ double all_min;
    __shared__ int all_fail, lost, verdict;

    const int m = threadIdx.x, lane = m & 63, wave = m >> 6;
    const int n = G.n[0], g = G.g[0];
    // own zones [r0, r0 + nz) of the interior, spread evenly
    const int q0 = n / groups, extra = n % groups;
    const int nz = q0 + (w < extra ? 1 : 0), r0 = w * q0 + (w < extra ? w : extra);
    const int W = nz + 2 * LO;
    const int r = r0 - LO + m;  // this thread's zone, interior-relative
    const bool wraps = !ONE && G.bc == 0;  // halos beyond the ends are the other end's zones
    const bool own = m >= LO && m < LO + nz;
    // zones the first stage updates, and the faces each stage needs
    const auto first_zone = [&](int l) { return l >= NG && l < W - NG && (wraps || (r0 - LO + l >= 0 && r0 - LO + l < n)); };
    const bool zone1 = first_zone(m);
    const bool face1 = zone1 || (m > 0 && first_zone(m - 1));
    const bool face2 = m >= LO && m <= LO + nz;

    double t = ctl->t;
    const double t_final = ctl->t_final, cfl = ctl->cfl;
    int steps = ctl->steps;
    const int limit = ctl->max_steps;
    unsigned long long bits = DBL_MAX_BITS;
    if (given)
    {
        if (m == 0) begin_advance(ctl, dt_given);
        __builtin_amdgcn_s_waitcnt(0);  // before the counts below, several barriers on
    }
    else
    {
        if (!ctl->active || ctl->c2p_fail || ctl->eigen_fail || ctl->superluminal) return;  // the same for everybody
        bits = wave_min(ctl->cbins[lane * CBIN_STRIDE]);
        bits = (unsigned long long)__shfl((long long)bits, 0, 64);
    }

    // ---- the state: P of this thread's zone, Pk the first stage's previous
    // result (what a failed recovery leaves in the stage buffer)
    double P[NQ], Pk[NQ];
    {
        int z = r;
        if (wraps) z = ((r % n) + n) % n;
        else z = min(max(r, -NG), n - 1 + NG);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            P[q] = m < W ? Pa[q * G.fs + g + z] : 1.0;
            Pk[q] = Law != 0 && m < W ? Pb[q * G.fs + g + z] : 0.0;
        }
    }
    if (m < W)
    {
#pragma unroll
        for (int q = 0; q < NQ; ++q) sP[q][m] = R(P[q]);
        if (wraps && ((r < 0 && r >= -NG) || (r >= n && r < n + NG)))
        {
            // guards that are not the periodic images (as uploaded) count in
            // the first step, which then goes by launches
            bool image = true;
#pragma unroll
            for (int q = 0; q < NQ; ++q) image = image && dbits(Pa[q * G.fs + g + r]) == dbits(P[q]);
            if (!image) atomicCAS(decision, (unsigned)OPEN, (unsigned)GAVE_UP);
        }
    }
    if (m == 0) lost = 0;
    __syncthreads();

    // the faces of a stage from sP into sF
    const auto faces = [&](bool mine) {
        if (!mine) return;
        R S[NQ][2 * NG];
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int k = 0; k < 2 * NG; ++k) S[q][k] = sP[q][m - NG + k];
        R F[NQ];
        face_flux<Law, Recon, Riem, R, LawMath<Law, R>, 0>(S, G, 0, F, ctl);
#pragma unroll
        for (int q = 0; q < NQ; ++q) sF[q][m] = F[q];
    };
    const auto divergence = [&](double* L) {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            const R fr = sF[q][m + 1], fl = sF[q][m];
            if (CT && q >= 5)
            {
                const double x1 = q != 5 ? double(fr) : 0.0, xl = q != 5 ? double(fl) : 0.0;
                L[q] = divergence_ct(G, x1, xl, 0.0, 0.0, 0.0, 0.0);
            }
            else
                L[q] = divergence_R<R>(G, fr, fl, R(0), R(0), R(0), R(0));
        }
    };
    // a zone's new primitives into sP, with its guard images where the guards
    // are filled from inside this work-group
    const auto publish_local = [&](const double* v) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) sP[q][m] = R(v[q]);
        if (wraps || (r >= NG && r < n - NG)) return;
        const auto image = [&](int rr, double sign) {
            const int l = rr - r0 + LO;
            if (l < 0 || l >= W) return;
#pragma unroll
            for (int q = 0; q < NQ; ++q) sP[q][l] = R(q == 1 ? v[q] * sign : v[q]);
        };
        if (G.bc == 0)
        {
            if (r >= n - NG) image(r - n, 1.0);
            if (r < NG) image(r + n, 1.0);
        }
        else if (G.bc == 1)
        {
            if (r == 0)
                for (int l = 1; l <= NG; ++l) image(-l, 1.0);
            if (r == n - 1)
                for (int l = 0; l < NG; ++l) image(n + l, 1.0);
        }
        else
        {
            if (r < NG) image(-1 - r, -1.0);
            if (r >= n - NG) image(2 * n - 1 - r, -1.0);
        }
    };

    double dt = 0.0;
    int failures = 0, floors = 0;
    unsigned long long first_failure = ~0ull;
    int any_fail = 0;
    bool over = false, moved = false;
    for (int k = 0; k < max_steps; ++k)
    {
        // the stop condition and time step of step_start_wave
        if (given) dt = dt_given;
        else
        {
            if (!(t < t_final && steps < limit && !any_fail))
            {
                over = true;
                break;
            }
            const double dt1 = cfl * bitsd(bits);
            const double dt2 = t_final - t;
            dt = dt1 < dt2 ? dt1 : dt2;
        }
        unsigned long long* const slot = box + ((long long)w * SLOTS + k % SLOTS) * Msg::WORDS;
        if constexpr (!ONE)
        {
            unsigned long long* const old = box + ((long long)w * SLOTS + (k + 1) % SLOTS) * Msg::WORDS;
            if (m < Msg::WORDS) post(old + m, EMPTY);
        }
        int failed_here = 0;
        // ---- first stage: U = U0 + dt L
        faces(face1);
        __syncthreads();
        double U1[NQ];
        if (zone1)
        {
            double L[NQ];
            divergence(L);
            ZoneResult<Law> z;
            zone_update<Law, R, LawMath<Law, R>>(
                G, dt, 1.0, 1, P, [](int) { return 0.0; }, [&](int q) { return L[q]; }, z);
#pragma unroll
            for (int q = 0; q < NQ; ++q)
            {
                U1[q] = z.U[q];
                if (!z.failed) Pk[q] = z.P[q];
            }
            if (own)
            {
                floors += z.floor;
                if (z.failed)
                {
                    failures += 1;
                    failed_here = 1;
                    first_failure = min(first_failure, (unsigned long long)r);
                }
            }
            publish_local(Pk);
        }
        __syncthreads();
        // ---- second stage
        faces(face2);
        __syncthreads();
        double dtc = 1.79769313486231570815e+308;
        if (own)
        {
            double L[NQ];
            divergence(L);
            ZoneResult<Law> z;
            zone_update<Law, R, LawMath<Law, R>>(
                G, dt, 0.5, 0, P, [&](int q) { return U1[q]; }, [&](int q) { return L[q]; }, z);
            floors += z.floor;
            if (z.failed)
            {
                failures += 1;
                failed_here = 1;
                first_failure = min(first_failure, (unsigned long long)r);
            }
            else
            {
#pragma unroll
                for (int q = 0; q < NQ; ++q) P[q] = z.P[q];
                int err = 0;
                if (!given) dtc = zone_cfl<Law, R, LawMath<Law, R>>(G, G.Lmin, z, err);
            }
            publish_local(P);
            if constexpr (!ONE)
            {
                if (m < LO + Msg::H)
                {
#pragma unroll
                    for (int q = 0; q < NQ; ++q) post(slot + 1 + (m - LO) * NQ + q, word(P[q]));
                }
                if (m >= LO + nz - Msg::H)
                {
#pragma unroll
                    for (int q = 0; q < NQ; ++q)
                        post(slot + 1 + Msg::EDGE + (m - (LO + nz - Msg::H)) * NQ + q, word(P[q]));
                }
            }
        }
        moved = true;
        steps += 1;
        if (given && ONE)
        {
            any_fail |= failed_here;
            break;
        }
        t += dt;
        // ---- the next step's CFL minimum, over every work-group
        dtc = wave_min(dtc);
        const int fw = __any(failed_here);
        if (lane == 0)
        {
            wmin[wave] = dtc;
            wfail[wave] = fw;
        }
        __builtin_amdgcn_s_waitcnt(0);  // this step's clears are complete
        __syncthreads();
        double mine = 1.79769313486231570815e+308;
        int bad = 0;
        for (int v = 0; v < WAVES; ++v)
        {
            if (wmin[v] < mine) mine = wmin[v];
            bad |= wfail[v];
        }
        if constexpr (ONE)
        {
            bits = dbits(mine);
            any_fail = bad;
        }
        else
        {
            // a failure travels in the sign of the minimum
            if (m == 0) post(slot, dbits(bad ? -mine : mine));
            // halos: the neighbours' facing edges
            const bool left = m < LO && (wraps || w > 0);
            const bool right = m >= LO + nz && m < W && (wraps || w < groups - 1);
            for (;;)
            {
                bool got = true;
                unsigned long long v;
                if (left || right)
                {
                    const int from = left ? (w + groups - 1) % groups : (w + 1) % groups;
                    const unsigned long long* e = box + ((long long)from * SLOTS + k % SLOTS) * Msg::WORDS + 1
                                                  + (left ? Msg::EDGE + m * NQ : (m - (LO + nz)) * NQ);
#pragma unroll
                    for (int q = 0; q < NQ; ++q)
                    {
                        got = got && receive(e + q, decision, patience, v);
                        P[q] = bitsd(v);
                        sP[q][m] = R(P[q]);
                    }
                }
                if (wave == WAVES / 2)
                {
                    double least = 1.79769313486231570815e+308;
                    int f = 0;
                    for (int o = lane; o < groups; o += 64)
                    {
                        got = got && receive(box + ((long long)o * SLOTS + k % SLOTS) * Msg::WORDS, decision, patience, v);
                        const double d = __builtin_fabs(bitsd(v));
                        f |= (int)(v >> 63);
                        if (d < least) least = d;
                    }
                    least = wave_min(least);
                    f = __any(f);
                    if (lane == 0)
                    {
                        all_min = least;
                        all_fail = f;
                    }
                }
                if (!got) lost = 1;
                __syncthreads();
                if (!lost) break;
                // give up, unless the results are decided already: then this
                // is the last exchange, every message of it is there, and the
                // next look finds them
                if (m == 0) verdict = (int)atomicCAS(decision, (unsigned)OPEN, (unsigned)GAVE_UP);
                __syncthreads();
                if (verdict != (int)DONE) return;
                if (m == 0) lost = 0;
                __syncthreads();
            }
            bits = dbits(all_min);
            any_fail = all_fail;
        }
    }
    if (!moved) return;
    if constexpr (!ONE)
    {
        if (m == 0) verdict = (int)atomicCAS(decision, (unsigned)OPEN, (unsigned)DONE);
        __syncthreads();
        if (verdict == (int)GAVE_UP) return;
    }
    // ---- results
    if (own)
    {
        const long long c = g + r;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            Pa[q * G.fs + c] = P[q];
            if (Law != 0) Pb[q * G.fs + c] = Pk[q];
        }
        write_guard_images<NQ>(Pa, G, (int)c, 0, 0, P);
        if (failures)
        {
            atomicAdd(&ctl->c2p_fail, (unsigned long long)failures);
            atomicMin(&ctl->first_fail, first_failure);
        }
        if (floors) atomicAdd(&ctl->floor_applied, (unsigned long long)floors);
    }
    if (given)
    {
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        report(ctl, host, m);
    }
    else if (w == 0)
    {
        if (wave == 0) ctl->cbins[lane * CBIN_STRIDE] = lane == 0 ? bits : DBL_MAX_BITS;
        if (m == 0)
        {
            ctl->t = t;
            ctl->steps = steps;
            ctl->dt = dt;
            if (over) ctl->active = 0;
        }
    }
}

template <int Law, int Recon, int Riem, typename R, bool CT, int THREADS, bool ONE>
static __global__ void __launch_bounds__(THREADS)
k_run1d(double* __restrict__ Pa, double* __restrict__ Pb, const Geom G, Ctl* __restrict__ ctl, int max_steps,
        int given, double dt_given, unsigned long long* __restrict__ box, unsigned* __restrict__ decision,
        int patience, Ctl* __restrict__ host)
{
    run<Law, Recon, Riem, R, CT, THREADS, ONE>(Pa, Pb, G, ctl, (int)blockIdx.x, (int)gridDim.x, max_steps, given,
                                               dt_given, box, decision, patience, host);
}

// The CFL time step of a block of one work-group, in one launch: k_courant
// (or the mixed form's k_courant_form) between k_ctl_begin_courant and
// k_ctl_fold_bins, the control block's copy left in host memory.
template <int Law, typename R>
static __global__ void __launch_bounds__(512)
k_courant_one(const double* __restrict__ P, const Geom G, Ctl* __restrict__ ctl, Ctl* __restrict__ host)
{
    __shared__ double wmin[8];
    constexpr int NQ = LawNQ<Law>::value;
    const int m = threadIdx.x;
    double d = 1.79769313486231570815e+308;
    int err = 0;
    for (int i = m; i < G.n[0]; i += 512)
    {
        double p[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) p[q] = P[q * G.fs + G.g[0] + i];
        const double z = courant_of<Law, R>(p, G, G.Lmin, err);
        if (z < d) d = z;
    }
    d = wave_min(d);
    if ((m & 63) == 0) wmin[m >> 6] = d;
    __syncthreads();
    if (m < CBINS) ctl->cbins[m * CBIN_STRIDE] = DBL_MAX_BITS;
    if (m == 0)
    {
        for (int v = 1; v < 8; ++v)
            if (wmin[v] < d) d = wmin[v];
        ctl->active = 1;
        ctl->eigen_fail = 0;
        ctl->superluminal = 0;
        ctl->courant_bits = d < 1.79769313486231570815e+308 ? dbits(d) : DBL_MAX_BITS;
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    report(ctl, host, m);
}

// ---- host side ---------------------------------------------------------------
// The threads of a block's one work-group (0: it is split), or the work-groups
// it is split over (0: it is not taken).  One work-group of 512 threads, two
// wavefronts per SIMD and no exchange, is level with three of 256 (508 zones,
// hydro 5.7 us a step against 6.3, MHD 10.2 against 9.8); above that the
// split is faster.
inline int one_threads(int cells, int ng)
{
    const int need = cells + 2 * ng;
    return need <= 256 ? 256 : need <= 512 ? 512 : 0;
}

// fs: the field stride of the block's RK state, which holds the messages
inline int split_groups(int cells, int ng, int nq, long long fs)
{
    const int most = PL - 4 * ng;  // own zones of a work-group
    const int groups = (cells + most - 1) / most;
    const long long words = (long long)SLOTS * (1 + 2 * 2 * ng * nq);  // of one work-group
    // every work-group holds at least the zones its neighbours' halos take
    return groups <= GROUPS_MAX && cells / groups >= 2 * ng && groups * words <= nq * fs ? groups : 0;
}

struct Args
{
    const mara_desc* d;
    const Geom* G;
    hipStream_t stream;
    double *Pa, *Pb;
    Ctl* ctl;
    Ctl* host;
    unsigned long long* box;
    unsigned* decision;
    int threads, groups;  // of one_threads, split_groups
    int max_steps, given;
    double dt;
    int patience = PATIENCE;
};

template <int Law, int Recon, int Riem, typename R, bool CT>
void launch_t(const Args& a)
{
    if (a.threads)
    {
        auto go = [&](auto threads) {
            constexpr int T = decltype(threads)::value;
            k_run1d<Law, Recon, Riem, R, CT, T, true><<<1, T, 0, a.stream>>>(
                a.Pa, a.Pb, *a.G, a.ctl, a.max_steps, a.given, a.dt, nullptr, nullptr, a.patience, a.host);
        };
        if (a.threads == 256) go(std::integral_constant<int, 256>{});
        else go(std::integral_constant<int, 512>{});
        return;
    }
    const int words = a.groups * SLOTS * Message<Law, Recon>::WORDS;
    k_run1d_open<<<(words + 255) / 256, 256, 0, a.stream>>>(a.box, words, a.decision);
    k_run1d<Law, Recon, Riem, R, CT, PL, false><<<a.groups, PL, 0, a.stream>>>(
        a.Pa, a.Pb, *a.G, a.ctl, a.max_steps, 0, 0.0, a.box, a.decision, a.patience, nullptr);
}

template <typename R>
void launch(const Args& a)
{
    const mara_desc& d = *a.d;
    const bool hllc = d.riemann == MARA_RIEMANN_HLLC;
    auto go = [&](auto recon) {
        constexpr int Recon = decltype(recon)::value;
        if (d.law == MARA_LAW_HYDRO)
            hllc ? launch_t<0, Recon, 1, R, false>(a) : launch_t<0, Recon, 0, R, false>(a);
        else
            d.field_ct ? launch_t<1, Recon, 0, R, true>(a) : launch_t<1, Recon, 0, R, false>(a);
    };
    if (d.recon == MARA_RECON_PCM) go(std::integral_constant<int, 0>{});
    else if (d.recon == MARA_RECON_PLM) go(std::integral_constant<int, 1>{});
    else go(std::integral_constant<int, 2>{});
}

template <typename R>
void launch_courant(const Args& a)
{
    if (a.d->law == MARA_LAW_HYDRO) k_courant_one<0, R><<<1, 512, 0, a.stream>>>(a.Pa, *a.G, a.ctl, a.host);
    else k_courant_one<1, R><<<1, 512, 0, a.stream>>>(a.Pa, *a.G, a.ctl, a.host);
}

// binary64 fluxes (run1d.hip) and the mixed form's binary32 ones
// (run1d_mixed.hip, compiled with contraction)
void launch_f64(const Args& a);
void launch_f32(const Args& a);
void courant_f64(const Args& a);
void courant_f32(const Args& a);

// Hydro and MHD in RK2 (the buffers' roles in the header comment), without
// cooling; pencil_supported has checked the rest.
inline bool supported(const mara_desc& d)
{
    return d.law != MARA_LAW_RMHD && d.rk_order == 2;
}

} // namespace run1d
} // namespace mara
