// Resident conjugate gradients (resident.hpp): the kernels that run many
// Jacobi-PCG iterations in one launch, their windows and their launchers.
//
// What bounds small and middle-sized solves is not bytes but the distance
// between dependent kernels: with three launches per iteration every one of
// them pays a launch gap, a chain of cold loads and a block reduction (13 to
// 15 us per iteration for 4000 rows, 20 us for 100,000 rows whose data fit
// the caches).  Here an iteration is
//   A  q = A p on the block's rows, p from the LDS window; sum p.q
//   B  r -= alpha q; z = D^-1 r, written to memory; sums r.r, r.z
//   C  window: p = z + beta p
// with two device-wide sums as the only meetings.  A sum is exchanged as one
// pair of 8-byte words per block, each half a double and the epoch of the
// sum: a block publishes its pair and polls the others', one trip through
// the memory-side cache (1.7 us for 16 blocks, 2.2 for 64, 3.2 to 4.2 for
// 256).  z is published before the second sum, so that the sum also tells
// that z is there, and every block updates the p of its window for itself:
// no third meeting for p.
//
// The blocks of a launch wait for each other, so all must be on the chip at
// once: at most one block per compute unit, launches of one process on one
// device ordered behind each other by events, and every wait bounded.  A
// block that gives up says so in Scal::abort and leaves; the others follow,
// and the host repeats the solve with the segment kernels.
//
// Mixed precision: the residual replacements (FP64 residual of the folded
// solution) happen inside the launch as well; leaving it for them cost 48 us
// each, 8 times per solve.
#include <algorithm>
#include <climits>
#include <cstdlib>
#include <mutex>

#include "resident.hpp"

#pragma clang fp contract(on)

namespace ins {

namespace {

template <typename T>
__device__ inline T ld_agent(const T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ inline void st_agent(T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// every store of this wave so far is visible to the whole device (they were
// agent-scope stores, written through)
__device__ inline void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Device-wide sums of a resident launch
struct Meet {
    uint64_t* words;   // [parity][block, then group][2 values][2 halves]
    uint32_t epoch;    // of the next sum
    int polls;         // bound of a wait
    int nb, blk;       // blocks, this block's segment
};

constexpr int MEET_SLOT = (RBMAX + RBMAX / 64) * 4;   // words of one parity
constexpr int MEET_WORDS = 2 * MEET_SLOT;

// publish s as the pair of words at w
__device__ inline void meet_words(const Meet& m, uint64_t* w, double s)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, s);
    const uint64_t e = (uint64_t)m.epoch << 32;
    st_agent(w, e | (uint32_t)u);
    st_agent(w + 1, e | (uint32_t)(u >> 32));
}

// The block's sums of v (waves in order, as block_allsum), published as its
// words of this epoch
template <int NV>
__device__ inline void meet_publish(const Meet& m, double (&v)[NV], double (*sh)[RW])
{
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = wave_sum(v[k]);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) sh[k][threadIdx.x >> 6] = v[k];
    __syncthreads();
    if (threadIdx.x < NV) {
        double s = 0.;
#pragma unroll
        for (int w = 0; w < RW; w++) s += sh[threadIdx.x][w];
        meet_words(m, m.words + (size_t)(m.epoch & 1) * MEET_SLOT + 4 * m.blk + 2 * threadIdx.x, s);
    }
}

// Polls the words of `cnt` publishers from `w` on, one per lane of the calling
// wave, and sums them over the wave (the order of totals()); false: some
// publisher did not arrive in time
template <int NV>
__device__ inline bool meet_poll(const Meet& m, const uint64_t* w, int cnt, double (&s)[NV])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < NV; k++) s[k] = 0.;
    bool ok = true;
    if (lane < cnt) {
        uint64_t a[NV], b[NV];
        int c = 0;
        do {
            ok = true;
#pragma unroll
            for (int k = 0; k < NV; k++) {
                a[k] = ld_agent(w + 4 * lane + 2 * k);
                b[k] = ld_agent(w + 4 * lane + 2 * k + 1);
            }
#pragma unroll
            for (int k = 0; k < NV; k++)
                ok = ok && (uint32_t)(a[k] >> 32) == m.epoch && (uint32_t)(b[k] >> 32) == m.epoch;
        } while (!ok && ++c < m.polls);
#pragma unroll
        for (int k = 0; k < NV; k++)
            s[k] = __builtin_bit_cast(double, (uint64_t)(uint32_t)a[k] | (b[k] << 32));
    }
    return __all(ok);
}

// The totals of all blocks' sums, the same bits in every block (and those of
// totals() over the same partials); false: a block did not arrive in time.
// Two slots by epoch parity are enough: a block reaches epoch e + 2 only
// after all blocks published e + 1, hence after all of them read e.
//
// Beyond 64 blocks in two stages: the first block of every 64 sums its 64
// and publishes that, and all poll the at most 4 group sums.  Every block
// polling every other took 4.1 us at 208 blocks and 3.4 at 123, the polls
// being in each other's way; two stages are two trips of about 1.1 us.
template <int NV>
__device__ inline bool meet_collect(Meet& m, double (&t)[NV], double* tot, int* dead,
                                    bool acquire = false)
{
    uint64_t* base = m.words + (size_t)(m.epoch & 1) * MEET_SLOT;
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        double s[NV];
        bool ok = true;
        if (m.nb <= 64) {
            ok = meet_poll<NV>(m, base, m.nb, s);
        } else {
            uint64_t* grp = base + RBMAX * 4;
            const int g = m.blk >> 6;
            if ((m.blk & 63) == 0) {
                ok = meet_poll<NV>(m, base + g * 256, min(64, m.nb - g * 64), s);
#pragma unroll
                for (int k = 0; k < NV; k++) s[k] = wave_sum(s[k]);
                if (ok && lane == 0)
#pragma unroll
                    for (int k = 0; k < NV; k++) meet_words(m, grp + g * 4 + 2 * k, s[k]);
            }
            if (ok) ok = meet_poll<NV>(m, grp, (m.nb + 63) >> 6, s);
        }
        if (m.nb <= 64) {
#pragma unroll
            for (int k = 0; k < NV; k++) s[k] = wave_sum(s[k]);
        } else {
#pragma unroll
            for (int k = 0; k < NV; k++) {
                double v = lane_value(s[k], 0);
                v += lane_value(s[k], 1);
                v += lane_value(s[k], 2);
                v += lane_value(s[k], 3);
                s[k] = v;
            }
        }
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < NV; k++) tot[k] = s[k];
            if (!ok) *dead = 1;
        }
        // what the others wrote before they published is read by plain loads
        // (agent-scope loads do not need it; 0.3 us at 64 blocks, 1.7 at 256)
        if (acquire) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) t[k] = tot[k];
    m.epoch++;
    return *dead == 0;
}

// The rows' part of a residual replacement: t = b - A x64, r = (float)t; a
// thread's shares of t.t and r.z.
struct RowRep {
    const double* x64;
    const double* b;
    float* r;
    const float* dinv;

    __device__ inline void row(int64_t g, double s, double2& v) const
    {
        const double ti = b[g] - s;
        v.x += ti * ti;
        const float rf = (float)ti;
        r[g] = rf;
        v.y += (double)rf * (double)(dinv[g] * rf);
    }
};

template <int FORM, typename TVR>
__device__ inline double2 resid_sell(Span sp, int64_t n, SellView S,
                                                        const int32_t* u, const TVR* vals,
                                                        RowRep rep, double* part)
{
    double2 v = make_double2(0., 0.);
    seg_products<FORM, TVR, double>(sp, n, S, u, vals, [&](int i) { return rep.x64[i]; }, part,
                                    wave_in_block(), [&](int g, double s) { rep.row(g, s, v); });
    return v;
}

template <int LPR, typename TVR>
__device__ inline double2 resid_csr(int64_t row0, int rows, const int32_t* rp,
                                                       const int32_t* col, const TVR* val,
                                                       RowRep rep)
{
    const int sub = threadIdx.x & (LPR - 1), team = threadIdx.x / LPR;
    double2 v = make_double2(0., 0.);
    for (int i = team; i < rows; i += RT / LPR) {
        const int64_t row = row0 + i;
        const double s = csr_seg_row<LPR, TVR, double>(
            rp[row] + sub, rp[row + 1], val, [&](int32_t k) { return rep.x64[col[k]]; });
        if (sub == 0) rep.row(row, s, v);
    }
    return v;
}

template <typename T>
struct Pair {
    T a, b;
};

// The iterations of one block.  F: the matrix form; NR slices per wave, D
// components per item.  Thread (wave w, lane l) owns items
// (first + w + RW j) * 64 + l of every component.  r stays in registers; x and
// the diagonal too where there are few of them, else they are read and
// written (by their owner only) while a sum travels.
//
// F::SHARE_R: the blocks exchange r instead of z and every one scales the r of
// its window itself, in the expression of the kernels on whole vectors
// (p = D^-1 r + beta p, D^-1 r unrounded; the reason beside SYM_SUM).  A second,
// cached load per place of the window.
template <class F, typename TX>
__device__ inline void cg_resident(const CgArgs<TX>& a, int launch_iters, int seg, F& f,
                                   TX* __restrict__ win)
{
    constexpr int NR = F::NR, D = F::D;
    constexpr bool mixed = sizeof(TX) == 4, KEEP = NR * D * sizeof(TX) <= 12;
    constexpr bool SHARE_R = F::SHARE_R;
    __shared__ double sh[2][RW];
    __shared__ double tot[2][2];
    // scalars that are looked at once an iteration (uniform, but doubles
    // would sit in vector registers)
    __shared__ double s_thr, s_delta2, s_rref, s_rr, s_tt;
    __shared__ int dead;
    Scal* sc = a.sc;
    if (sc->done || sc->stop || sc->abort) return;
    int iters = __builtin_amdgcn_readfirstlane(sc->iters);
    if (iters >= a.limit) return;
    double rho = sc->rho[0];
    Meet m{a.words, a.epoch, a.polls, a.g.B, seg};
    const int wave = wave_in_block();
    const int64_t nn = a.n;
    const Span sp = seg_span(a.g, seg);
    if (threadIdx.x == 0) {
        dead = 0;
        s_thr = sc->thr;
        s_delta2 = sc->delta2;
        s_rref = sc->rref;
        s_rr = sc->rr;
        s_tt = sc->tt;
    }
    // f(j, c, place of the item in the vectors) for this thread's items
    auto items = [&](auto fn) {
        const uint32_t i0 = (uint32_t)((sp.s0 + wave) * 64) + (threadIdx.x & 63);
#pragma unroll
        for (int j = 0; j < NR; j++) {
            const uint32_t i = i0 + (uint32_t)(RW * 64) * j;
            if (wave + RW * j < sp.sl && (int64_t)i < nn)
#pragma unroll
                for (int c = 0; c < D; c++) fn(j, c, (uint32_t)nn * c + i);
        }
    };

    TX x[KEEP ? NR : 1][D], r[NR][D], d[NR][D];
#pragma unroll
    for (int j = 0; j < NR; j++)
#pragma unroll
        for (int c = 0; c < D; c++) {
            r[j][c] = (TX)0;
            d[j][c] = (TX)0;
            if constexpr (KEEP) x[j][c] = (TX)0;
        }
    items([&](int j, int c, uint32_t g) {
        r[j][c] = a.r[g];
        if constexpr (KEEP) {
            x[j][c] = a.x[g];
            d[j][c] = a.dinv[g];
        }
    });
    f.window([&](int64_t g) { return a.p[g]; }, [&](int i, TX v) { win[i] = v; });
    __syncthreads();

    // 1: limit, 2: gave up, 3: breakdown, 4: converged (mixed: on the true residual)
    int state = 0, nrep = 0, it = 0;
    while (state == 0) {
        // (the registers of the form are loaded again after a replacement
        // rather than kept through it)
        f.setup();
        bool conv = false;
        for (;; it++) {
            if (it == launch_iters || iters >= a.limit) {
                state = 1;
                break;
            }
            TX q[NR][D];
            f.products(win, q);
            double v1[1] = {0.};
            items([&](int j, int c, uint32_t) { v1[0] += (double)win[f.own(j, c)] * (double)q[j][c]; });
            meet_publish<1>(m, v1, sh);
            if constexpr (!KEEP) items([&](int j, int c, uint32_t g) { d[j][c] = a.dinv[g]; });
            double t1[1];
            if (!meet_collect<1>(m, t1, tot[0], &dead)) {
                state = 2;
                break;
            }
            if (!(t1[0] > 0.) || !isfinite(t1[0])) {
                state = 3;
                break;
            }
            iters++;
            const TX al = (TX)(rho / t1[0]);
            double v2[2] = {0., 0.};
            items([&](int j, int c, uint32_t g) {
                const TX ri = r[j][c] - al * q[j][c];
                r[j][c] = ri;
                const TX zi = d[j][c] * ri;
                st_agent(&a.z[g], SHARE_R ? ri : zi);
                v2[0] += (double)ri * (double)ri;
                v2[1] += (double)ri * (double)zi;
            });
            stores_done();
            meet_publish<2>(m, v2, sh);
            // while the sums travel: x += alpha p
            items([&](int j, int c, uint32_t g) {
                if constexpr (KEEP) x[j][c] = x[j][c] + al * win[f.own(j, c)];
                else a.x[g] = a.x[g] + al * win[f.own(j, c)];
            });
            double t2[2];
            if (!meet_collect<2>(m, t2, tot[1], &dead)) {
                state = 2;
                break;
            }
            const double rr = t2[0];
            if (threadIdx.x == 0) s_rr = rr;
            if (!isfinite(rr)) {
                state = 3;
                break;
            }
            conv = rr < s_thr;
            if (conv) break;
            const TX be = (TX)(t2[1] / rho);
            rho = t2[1];
            if constexpr (SHARE_R)
                f.window([&](int64_t g) { return Pair<TX>{ld_agent(&a.z[g]), a.dinv[g]}; },
                         [&](int i, Pair<TX> v) { win[i] = v.b * v.a + be * win[i]; });
            else
                f.window([&](int64_t g) { return ld_agent(&a.z[g]); },
                         [&](int i, TX v) { win[i] = v + be * win[i]; });
            const bool pause = mixed && rr < s_delta2 * s_rref;
            __syncthreads();
            if (pause) break;
        }
        if (state != 0) break;
        it++;
        if constexpr (!mixed) {
            state = 4;
        } else {
            // Residual replacement: fold x into x64, t = b - A x64 in FP64,
            // r = (float)t.  x64 and z go through agent-scope stores, two
            // more meetings tell that they are there.
            items([&](int j, int c, uint32_t g) {
                double* p64 = &a.rep.x64[g];
                if constexpr (KEEP) {
                    st_agent(p64, ld_agent(p64) + (double)x[j][c]);
                    x[j][c] = (TX)0;
                } else {
                    st_agent(p64, ld_agent(p64) + (double)a.x[g]);
                    a.x[g] = (TX)0;
                }
            });
            stores_done();
            double v0[1] = {0.}, t0[1];
            meet_publish<1>(m, v0, sh);
            if (!meet_collect<1>(m, t0, tot[0], &dead, true)) {
                state = 2;
                break;
            }
            const RowRep rr{a.rep.x64, a.rep.b, a.r, a.dinv};
            const double2 tz = a.rep.v64 ? f.resid(a.rep.v64, rr) : f.resid(a.rep.v32, rr);
            double v2[2] = {tz.x, tz.y}, t2[2];
            __syncthreads();   // a row's sum may be another thread's
            items([&](int j, int c, uint32_t g) {
                r[j][c] = a.r[g];
                const TX zi = a.dinv[g] * r[j][c];
                st_agent(&a.z[g], SHARE_R ? r[j][c] : zi);
            });
            stores_done();
            meet_publish<2>(m, v2, sh);
            if (!meet_collect<2>(m, t2, tot[1], &dead)) {
                state = 2;
                break;
            }
            const double tt = t2[0];
            nrep++;
            // keep the direction while the recursion still tracks the true
            // residual; once it has converged or drifted, restart from D^-1 r
            const bool restart = conv || tt > a.rep.ratio * s_rr;
            const bool done = tt < s_thr;
            __syncthreads();
            if (threadIdx.x == 0) {
                s_tt = tt;
                s_rr = tt;
                s_rref = tt;
            }
            if (!isfinite(tt)) {
                state = 3;
                break;
            }
            if (done) {
                state = 4;
                break;
            }
            rho = t2[1];
            if (restart) {
                if constexpr (SHARE_R)
                    f.window([&](int64_t g) { return Pair<TX>{ld_agent(&a.z[g]), a.dinv[g]}; },
                             [&](int i, Pair<TX> v) { win[i] = v.b * v.a; });
                else
                    f.window([&](int64_t g) { return ld_agent(&a.z[g]); },
                             [&](int i, TX v) { win[i] = v; });
            }
            __syncthreads();
        }
    }
    if (state == 2) {
        if (threadIdx.x == 0) sc->abort = 1;
        return;
    }
    // hand the iterate back
    items([&](int j, int c, uint32_t g) {
        if constexpr (KEEP) a.x[g] = x[j][c];
        a.r[g] = r[j][c];
        a.p[g] = win[f.own(j, c)];
    });
    __syncthreads();
    if (seg == 0 && threadIdx.x == 0) {
        sc->iters = iters;
        sc->rho[0] = rho;
        sc->rho[1] = rho;
        if (it > 0) sc->rr = s_rr;
        if (nrep > 0) {
            sc->nrep += nrep;
            sc->tt = s_tt;
            sc->rref = s_rref;
        }
        if (state == 3) {
            sc->breakdown = 1;
            sc->done = 1;
        } else if (state == 4 && mixed) {
            sc->done = 1;
            sc->fin = 1;
        } else if (state == 4) {
            sc->stop = 1;
        }
    }
}

// ---------------------------------------------------------------------------
// CSR rows.  The window is a list of columns per block (the columns of its
// rows and the rows themselves, ascending); entries name their place in it.
// Up to NP passes of the block over its rows (RT / LPR rows each, rows of at
// most 4 LPR entries) are held in registers for the whole launch, values and
// window places: A then reads LDS only.  NP = 0: streamed from memory.
template <int LPR, int NP, typename TV, typename TX>
struct CsrForm {
    static constexpr int NR = CSR_ROWS / RT, D = 1;
    static constexpr bool SHARE_R = false;
    const int32_t* rp;
    const int32_t* col;
    const uint16_t* lcol;
    const TV* val;
    const int32_t* list;     // columns of this block's window
    int nw;                  // and their number
    int own0;                // window place of the block's first row
    int rows;                // rows of the block
    int64_t row0;
    TX* qs;                  // LDS: q of the block's rows
    static constexpr int UL = 8;
    int32_t lst[UL];         // this thread's first columns of the list
    TV rv[NP ? NP : 1][4];
    int rl[NP ? NP : 1][4];

    __device__ inline int own(int j, int) const { return own0 + threadIdx.x + RT * j; }

    template <class L, class O>
    __device__ inline void window(L load, O op)
    {
        TX v[UL];
#pragma unroll
        for (int u = 0; u < UL; u++)
            v[u] = (int)threadIdx.x + u * RT < nw ? load((int64_t)lst[u]) : (TX)0;
#pragma unroll
        for (int u = 0; u < UL; u++)
            if ((int)threadIdx.x + u * RT < nw) op(threadIdx.x + u * RT, v[u]);
        for (int i0 = threadIdx.x + UL * RT; i0 < nw; i0 += RT * UL) {
#pragma unroll
            for (int u = 0; u < UL; u++) {
                const int i = i0 + u * RT;
                v[u] = i < nw ? load((int64_t)list[i]) : (TX)0;
            }
#pragma unroll
            for (int u = 0; u < UL; u++) {
                const int i = i0 + u * RT;
                if (i < nw) op(i, v[u]);
            }
        }
    }

    __device__ inline void columns()
    {
#pragma unroll
        for (int u = 0; u < UL; u++) {
            const int i = threadIdx.x + u * RT;
            lst[u] = i < nw ? list[i] : 0;
        }
    }

    __device__ inline void setup()
    {
        if constexpr (NP > 0) {
            const int th = (wave_in_block() << 6) + opaque_lane();
            const int sub = th & (LPR - 1), team = th / LPR;
#pragma unroll
            for (int ps = 0; ps < NP; ps++) {
                const int i = team + ps * (RT / LPR);
                int32_t k0 = 0, e = 0;
                if (i < rows) {
                    k0 = rp[row0 + i] + sub;
                    e = rp[row0 + i + 1];
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int32_t k = k0 + j * LPR;
                    rv[ps][j] = k < e ? val[k] : (TV)0;
                    rl[ps][j] = k < e ? (int)lcol[k] : own0;   // a finite value
                }
            }
        }
    }

    template <typename TVR>
    __device__ inline double2 resid(const TVR* v, const RowRep& rep)
    {
        return resid_csr<LPR, TVR>(row0, rows, rp, col, v, rep);
    }

    __device__ inline void products(const TX* __restrict__ w, TX (&q)[NR][1])
    {
        const int sub = threadIdx.x & (LPR - 1), team = threadIdx.x / LPR;
        if constexpr (NP > 0) {
#pragma unroll
            for (int ps = 0; ps < NP; ps++) {
                const int i = team + ps * (RT / LPR);
                TX s = (TX)0;
#pragma unroll
                for (int j = 0; j < 4; j++) s += (TX)rv[ps][j] * w[rl[ps][j]];
                s = group_sum<LPR>(s);
                if (sub == 0 && i < rows) qs[i] = s;
            }
        } else {
            for (int i = team; i < rows; i += RT / LPR) {
                const int32_t e = rp[row0 + i + 1];
                const TX s = csr_seg_row<LPR, TV, TX>(
                    rp[row0 + i] + sub, e, val, [&](int32_t k) { return w[lcol[k]]; });
                if (sub == 0) qs[i] = s;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NR; j++) {
            const int i = threadIdx.x + RT * j;
            q[j][0] = i < rows ? qs[i] : (TX)0;
        }
    }
};

// LDS: q of up to CSR_ROWS rows, then the window
template <int LPR, int NP, typename TV, typename TX>
__global__ __launch_bounds__(RT) void k_cg_csr(CgArgs<TX> a, int iters, const int32_t* __restrict__ rp,
                                               const int32_t* __restrict__ col,
                                               const uint16_t* __restrict__ lcol,
                                               const TV* __restrict__ val,
                                               const int32_t* __restrict__ list,
                                               const int32_t* __restrict__ woff,
                                               const int32_t* __restrict__ own0)
{
    extern __shared__ unsigned char lds[];
    const int seg = seg_of_block(blockIdx.x, a.g.B);
    CsrForm<LPR, NP, TV, TX> f;
    f.rp = rp;
    f.col = col;
    f.lcol = lcol;
    f.val = val;
    f.list = list + woff[seg];
    f.nw = woff[seg + 1] - woff[seg];
    f.own0 = own0[seg];
    f.row0 = (int64_t)seg * a.g.R * 64;
    const int64_t left = a.n - f.row0;
    f.rows = (int)(left < 0 ? 0 : (left < (int64_t)a.g.R * 64 ? left : (int64_t)a.g.R * 64));
    f.qs = reinterpret_cast<TX*>(lds);
    f.columns();
    cg_resident(a, iters, seg, f, f.qs + CSR_ROWS);
}

// ---------------------------------------------------------------------------
// Symmetric slices of scalar rows and of node blocks.  Every row has the same
// offsets, so the windows of all blocks have one layout: the intervals
// [row0 + d, row0 + d + 64 R) over all offsets d, merged where they touch,
// each cut into pieces of 64.  Entry t of a row finds its p at
// (row - row0) + sh[t].  Places outside the matrix hold 0.
template <int D, typename TX, class L, class O>
__device__ inline void rel_window(const RelWin& W, int64_t row0, int64_t nn, L load, O op)
{
    constexpr int U = D == 1 ? 8 : (sizeof(TX) == 4 ? 3 : 2);
    typedef decltype(load((int64_t)0)) V;   // what is loaded for a place
    const int lane = threadIdx.x & 63;
    for (int c0 = wave_in_block(); c0 < W.npiece; c0 += RW * U) {
        V v[U][D];
        int at[U];
#pragma unroll
        for (int k = 0; k < U; k++) {
            const int c = c0 + k * RW;
            at[k] = -1;
            if (c < W.npiece) {
                const int4 pc = W.piece[c];
                const int64_t g = row0 + pc.x + lane;
                const bool in = lane < pc.z && g >= 0 && g < nn;
                at[k] = lane < pc.z ? pc.y + lane : -1;
#pragma unroll
                for (int d = 0; d < D; d++) {
                    v[k][d] = V{};
                    if (in) v[k][d] = load(d * nn + g);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < U; k++)
            if (at[k] >= 0)
#pragma unroll
                for (int d = 0; d < D; d++) op(at[k] * D + d, v[k][d]);
    }
}

// The entries of the thread's rows are held in registers for the launch.
template <int NU, int NR_, typename TV, typename TX>
struct SymForm {
    static constexpr int NR = NR_, D = 1, NT = 2 * NU - 1;
    static constexpr bool SHARE_R = sizeof(TX) == 4;
    const TV* vals;
    RelWin W;
    int64_t n;
    Span sp;
    bool edge;
    int du[NU], sh[NT];
    TV rv[NR_][NT];

    __device__ inline int own(int j, int) const
    {
        return (wave_in_block() + RW * j) * 64 + (threadIdx.x & 63) + sh[0];
    }
    template <class L, class O>
    __device__ inline void window(L load, O op)
    {
        rel_window<1, TX>(W, sp.s0 * 64, n, load, op);
    }
    __device__ inline bool active(int j) const
    {
        const int sl = wave_in_block() + RW * j;
        return sl < sp.sl && (sp.s0 + sl) * 64 < n;
    }
    __device__ inline void setup()
    {
        const int lane = opaque_lane();
        const int us = W.u[lane < NU ? lane : 0], shs = W.sh[lane < NT ? lane : 0];
#pragma unroll
        for (int k = 0; k < NU; k++) du[k] = __builtin_amdgcn_readlane(us, k);
#pragma unroll
        for (int t = 0; t < NT; t++) sh[t] = __builtin_amdgcn_readlane(shs, t);
        edge = sp.s0 * 64 < du[NU - 1];
#pragma unroll
        for (int j = 0; j < NR; j++) {
#pragma unroll
            for (int t = 0; t < NT; t++) rv[j][t] = (TV)0;
            if (active(j))
                sym_seg_values<NU, TV>(vals, sp.s0 + wave_in_block() + RW * j, lane, du, edge,
                                       rv[j]);
        }
    }
    template <typename TVR>
    __device__ inline double2 resid(const TVR* v, const RowRep& rep)
    {
        return resid_sell<NU == 14 ? SEG_SYM14 : SEG_SYM5, TVR>(sp, n, SellView{}, W.u, v, rep,
                                                                nullptr);
    }
    __device__ inline void products(const TX* __restrict__ w, TX (&q)[NR][1])
    {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int j = 0; j < NR; j++) {
            TX s = (TX)0;
            if (active(j)) {
                const int li = (wave_in_block() + RW * j) * 64 + lane;
                // (all LDS reads first: one at a time they cost their latency)
                TX xv[NT];
#pragma unroll
                for (int t = 0; t < NT; t++) xv[t] = w[li + sh[t]];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k0 = 0; k0 < NU; k0 += SYM_SUM) {
#pragma unroll
                    for (int k = k0; k < k0 + SYM_SUM && k < NU; k++)
                        s += (TX)rv[j][k ? 2 * k - 1 : 0] * xv[k ? 2 * k - 1 : 0];
#pragma unroll
                    for (int k = k0; k < k0 + SYM_SUM && k < NU; k++)
                        if (k) s += (TX)rv[j][2 * k] * xv[2 * k];
                }
            }
            q[j][0] = s;
        }
    }
};

template <int NU, int NR, typename TX>
__device__ inline void run_sym(const CgArgs<TX>& a, int iters, int seg, const TX* __restrict__ vals,
                               const RelWin& W, unsigned char* lds)
{
    SymForm<NU, NR, TX, TX> f;
    f.vals = vals;
    f.W = W;
    f.n = a.n;
    f.sp = seg_span(a.g, seg);
    cg_resident(a, iters, seg, f, reinterpret_cast<TX*>(lds));
}

template <int NU, int NR, typename TX>
__global__ __launch_bounds__(RT) void k_cg_sym(CgArgs<TX> a, int iters,
                                               const TX* __restrict__ vals, RelWin W)
{
    extern __shared__ unsigned char lds[];
    run_sym<NU, NR, TX>(a, iters, seg_of_block(blockIdx.x, a.g.B), vals, W, lds);
}

// Node blocks; the window holds the D components of a node side by side.
// PARTS > 1: task t is part t % PARTS of slice t / PARTS, wave w takes tasks w,
// w + RW, ..; the blocks of TASKS tasks sit in registers, with EXT those of the
// others in LDS
template <int D_, int NU, int NR_, int PARTS, bool EXT, typename TV, typename TX>
struct BsymForm {
    static constexpr int NR = NR_, D = D_, NT = 2 * NU - 1, PER = bsym_per(NT, PARTS);
    static constexpr bool SHARE_R = false;
    // tasks of a wave, and those in registers (all, but for FP32 3 x 3 blocks)
    static constexpr int TW = PARTS == 1 ? 1 : (PARTS == 3 && (EXT || D == 2 || sizeof(TV) == 8) ? 3 : 2);
    static constexpr int TR = EXT ? 2 : TW;
    static_assert(TASKS == 2 * RW && BSYM_TASKS <= 3 * RW);
    static constexpr bool REG = PARTS > 1 && PER * D * D * (int)sizeof(TV) <= 9 * 9 * 4;
    // blocks of loads in flight
    static constexpr int G = sizeof(TV) == 4 ? 3 : 2;
    const TV* vals;
    RelWin W;
    int64_t nn;
    Span sp;
    int sh0;
    TX* part;      // LDS: the parts' sums
    TV* ext;       // LDS: the blocks of tasks from TASKS on
    TV rv[REG ? TR : 1][REG ? PER : 1][D * D];
    int rsh[REG ? TR : 1][REG ? PER : 1];   // shifts of those blocks

    __device__ inline int own(int j, int c) const
    {
        return ((wave_in_block() + RW * j) * 64 + (int)(threadIdx.x & 63) + sh0) * D + c;
    }
    template <class L, class O>
    __device__ inline void window(L load, O op)
    {
        rel_window<D, TX>(W, sp.s0 * 64, nn, load, op);
    }
    __device__ inline bool live(int sl) const { return sl < sp.sl && (sp.s0 + sl) * 64 < nn; }
    __device__ inline void setup()
    {
        sh0 = __builtin_amdgcn_readfirstlane(W.sh[0]);
        if constexpr (REG) {
            const int lane = opaque_lane();
            // offsets and shifts with one load each: reading them one by one
            // made every block wait for the one before
            const int us = W.u[lane < NU ? lane : 0], shs = W.sh[lane < NT ? lane : 0];
            auto off = [&](int t) { return __builtin_amdgcn_readlane(us, (t + 1) >> 1); };
            if constexpr (EXT) {
                const int t = wave_in_block() + TASKS;
                const int sl = t / PARTS, p0 = (t % PARTS) * PER;
                if (t < PARTS * sp.sl && live(sl))
#pragma unroll 1
                    for (int s = 0; s < PER && p0 + s < NT; s++) {
                        TV b[D * D];
                        bsym_seg_block<D, NU, TV>(vals, sp.s0 + sl, lane, p0 + s, off(p0 + s), b);
#pragma unroll
                        for (int e = 0; e < D * D; e++) ext_at(s)[e * 64] = b[e];
                    }
            }
#pragma unroll
            for (int w = 0; w < TR; w++) {
                const int t = wave_in_block() + RW * w;
                const int sl = t / PARTS, p0 = (t % PARTS) * PER;
#pragma unroll
                for (int s = 0; s < PER; s++) {
                    // (past the last block: zeros)
                    rsh[w][s] = __builtin_amdgcn_readlane(shs, p0 + s < NT ? p0 + s : 0);
#pragma unroll
                    for (int e = 0; e < D * D; e++) rv[w][s][e] = (TV)0;
                    if (live(sl) && p0 + s < NT)
                        bsym_seg_block<D, NU, TV>(vals, sp.s0 + sl, lane, p0 + s, off(p0 + s),
                                                  rv[w][s]);
                }
            }
        }
    }
    template <typename TVR>
    __device__ inline double2 resid(const TVR* v, const RowRep& rep)
    {
        return resid_sell<D == 3 ? SEG_BSYM3 : SEG_BSYM2, TVR>(sp, nn, SellView{}, W.u, v, rep,
                                                               reinterpret_cast<double*>(part));
    }
    // block s of this wave's task in LDS
    __device__ inline TV* ext_at(int s) const
    {
        return ext + ((wave_in_block() * PER + s) * D * D) * 64 + (threadIdx.x & 63);
    }
    __device__ inline void ext_sum(const TX* __restrict__ w, int sl, int p0, TX (&out)[D])
    {
        const int li = sl * 64 + (int)(threadIdx.x & 63);
#pragma unroll
        for (int c = 0; c < D; c++) out[c] = (TX)0;
        constexpr int G = 1;
#pragma unroll 1
        for (int s0 = 0; s0 < PER; s0 += G) {
            TV b[G][D * D];
            TX x[G][D];
#pragma unroll
            for (int g = 0; g < G; g++)
                if (s0 + g < PER && p0 + s0 + g < NT) {
                    const TX* __restrict__ xp = w + (li + W.sh[p0 + s0 + g]) * D;
#pragma unroll
                    for (int c = 0; c < D; c++) x[g][c] = xp[c];
#pragma unroll
                    for (int e = 0; e < D * D; e++) b[g][e] = ext_at(s0 + g)[e * 64];
                }
#pragma unroll
            for (int g = 0; g < G; g++)
                if (s0 + g < PER && p0 + s0 + g < NT) bsym_seg_add<D, TV, TX>(b[g], x[g], out);
        }
    }
    // the sum of part p0 of slice sl
    __device__ inline void part_sum(const TX* __restrict__ w, int tw, int sl, int p0, TX (&out)[D])
    {
        const int lane = REG ? (int)(threadIdx.x & 63) : opaque_lane();
        const int li = sl * 64 + lane;
#pragma unroll
        for (int c = 0; c < D; c++) out[c] = (TX)0;
        if constexpr (REG) {
            // LDS reads a few blocks ahead of their use
            constexpr int A = PER < 4 ? PER : 4;
            TX x[PER][D];
#pragma unroll
            for (int s = 0; s < PER + A; s++) {
                if (s < PER) {
                    const TX* __restrict__ xp = w + (li + rsh[tw][s]) * D;
#pragma unroll
                    for (int c = 0; c < D; c++) x[s][c] = xp[c];
                }
                if (s >= A) {
                    bsym_seg_add<D, TV, TX>(rv[tw][s - A], x[s - A], out);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        } else {
#pragma unroll 1
            for (int t0 = p0; t0 < p0 + PER && t0 < NT; t0 += G) {
                TV b[G][D * D];
#pragma unroll
                for (int g = 0; g < G; g++)
                    if (t0 + g < p0 + PER && t0 + g < NT)
                        bsym_seg_block<D, NU, TV>(vals, sp.s0 + sl, lane, t0 + g,
                                                  W.u[(t0 + g + 1) >> 1], b[g]);
#pragma unroll
                for (int g = 0; g < G; g++)
                    if (t0 + g < p0 + PER && t0 + g < NT) {
                        const TX* __restrict__ xp = w + (li + W.sh[t0 + g]) * D;
                        TX x[D];
#pragma unroll
                        for (int c = 0; c < D; c++) x[c] = xp[c];
                        bsym_seg_add<D, TV, TX>(b[g], x, out);
                    }
            }
        }
    }
    __device__ inline void products(const TX* __restrict__ w, TX (&q)[NR][D])
    {
        const int lane = threadIdx.x & 63;
        if constexpr (PARTS == 1) {
#pragma unroll
            for (int j = 0; j < NR; j++) {
                const int sl = wave_in_block() + RW * j;
                if (live(sl)) part_sum(w, 0, sl, 0, q[j]);
                else
#pragma unroll
                    for (int c = 0; c < D; c++) q[j][c] = (TX)0;
            }
        } else {
#pragma unroll
            for (int k = 0; k < TW; k++) {
                const int t = wave_in_block() + RW * k;
                if (t < PARTS * sp.sl && live(t / PARTS)) {
                    TX out[D];
                    if constexpr (REG)
                        if (k >= TR) {
                            if constexpr (EXT) ext_sum(w, t / PARTS, (t % PARTS) * PER, out);
                        } else {
                            part_sum(w, k < TR ? k : 0, t / PARTS, (t % PARTS) * PER, out);
                        }
                    else
                        part_sum(w, 0, t / PARTS, (t % PARTS) * PER, out);
#pragma unroll
                    for (int c = 0; c < D; c++) part[(t * D + c) * 64 + lane] = out[c];
                }
            }
            __syncthreads();
            const int own_sl = wave_in_block();
#pragma unroll
            for (int c = 0; c < D; c++) {
                TX s = (TX)0;
                if (live(own_sl))
#pragma unroll
                    for (int i = 0; i < PARTS; i++) s += part[((own_sl * PARTS + i) * D + c) * 64 + lane];
                q[0][c] = s;
            }
        }
    }
};

__host__ __device__ inline int bsym_sum_lds(int D, int R)
{
    return D > 1 && bsym_parts(R) > 1 ? bsym_parts(R) * R * D * 64 * 8 : 0;
}
// FP32 3 x 3 blocks of tasks from TASKS on
__host__ __device__ inline int bsym_ext_lds(int D, int NU, int R)
{
    const int p = bsym_parts(R), more = p * R - TASKS;
    return D == 3 && p == 3 && more > 0 ? more * bsym_per(2 * NU - 1, p) * D * D * 64 * 4 : 0;
}

// LDS: the parts' sums (FP64 in a residual), the blocks kept there, the window
template <int D, int NU, int NR, int PARTS, bool EXT, typename TX>
__device__ inline void run_bsym(const CgArgs<TX>& a, int iters, int seg,
                                const TX* __restrict__ vals, const RelWin& W, unsigned char* lds)
{
    BsymForm<D, NU, NR, PARTS, EXT, TX, TX> f;
    f.vals = vals;
    f.W = W;
    f.nn = a.n;
    f.sp = seg_span(a.g, seg);
    f.part = reinterpret_cast<TX*>(lds);
    f.ext = reinterpret_cast<TX*>(lds + bsym_sum_lds(D, a.g.R));
    cg_resident(a, iters, seg, f,
                reinterpret_cast<TX*>(lds + bsym_sum_lds(D, a.g.R) +
                                      (EXT ? bsym_ext_lds(D, NU, a.g.R) : 0)));
}

template <int D, int NU, int NR, int PARTS, bool EXT, typename TX>
__global__ __launch_bounds__(RT) void k_cg_bsym(CgArgs<TX> a, int iters,
                                                const TX* __restrict__ vals, RelWin W)
{
    extern __shared__ unsigned char lds[];
    run_bsym<D, NU, NR, PARTS, EXT, TX>(a, iters, seg_of_block(blockIdx.x, a.g.B), vals, W, lds);
}

// ---------------------------------------------------------------------------
// Full slices (SELL): windows are lists as for CSR, built from the ranges
// row + d of every slice and offset; base[(slice_ptr / 64) + k] is the place
// of lane 0's column of entry k.  Lanes whose column lies outside the matrix
// (their value is 0) read a neighbouring place: the window has 64 places of
// zeros on either side.
//
// Slices differ in length (the rows of a degree-2 field have 27 to 125
// entries), and a segment has no multiple of 16 of them, so the waves share
// the segment's entries, not its slices: each takes two of TASKS runs of `run`
// entries (sell_run) and leaves one sum per slice it meets in LDS.  Runs of at most
// MAXE entries are held in registers, the places of lane 0 in lane k % 64 of
// two more (read back as scalars: fetched from memory, 16 bytes at a time,
// they took 7 us of a 24 us iteration).
constexpr int SELL_MAXE = 80;
// sums in LDS: every run adds at most one per slice, and every slice but the
// first of a run starts there
constexpr int SELL_MAXR = 2 * RW;   // slices of a segment (short ones: their windows are wide)
constexpr int SELL_SUMS = (SELL_MAXR + TASKS) * 64;

template <int NR_, int MAXE, typename TV, typename TX>
struct SellForm {
    static constexpr int NR = NR_, D = 1;
    static constexpr bool SHARE_R = false;
    SellView S;
    const TV* vals;
    const int32_t* base;
    const int32_t* list;
    int nw, own0;
    int64_t n;
    Span sp;
    int run, e0, ne;    // entries of a run; the segment's first entry and its entries
    static constexpr int TW = TASKS / RW;
    int k0[TW];         // slices where this wave's runs start
    TX* sums;           // LDS
    int* firsts;        // LDS
    TV rv[MAXE ? TW : 1][MAXE ? MAXE / 4 : 1][4];
    int32_t rb[MAXE ? TW : 1][MAXE ? (MAXE + 63) / 64 : 1];

    __device__ inline int own(int j, int) const
    {
        return own0 + (wave_in_block() + RW * j) * 64 + (threadIdx.x & 63);
    }
    template <class L, class O>
    __device__ inline void window(L load, O op)
    {
        constexpr int U = 8;
        for (int i0 = threadIdx.x; i0 < nw; i0 += RT * U) {
            TX v[U];
            int32_t g[U];
#pragma unroll
            for (int u = 0; u < U; u++) g[u] = i0 + u * RT < nw ? list[i0 + u * RT] : 0;
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = i0 + u * RT < nw ? load((int64_t)g[u]) : (TX)0;
#pragma unroll
            for (int u = 0; u < U; u++)
                if (i0 + u * RT < nw) op(i0 + u * RT, v[u]);
        }
    }
    // first entry of slice k of the segment, from the segment's first
    __device__ inline int first(int k) const { return __builtin_amdgcn_readfirstlane(firsts[k]); }
    // sums: slot of slice k's share of run w (runs and slices both ascend, so
    // w + k names a pair)
    __device__ inline int slot(int w, int k) const { return (w + k) * 64; }

    __device__ inline void setup()
    {
        const int64_t nsl = (n + 63) / 64;
        e0 = (int)(S.sptr[sp.s0 < nsl ? sp.s0 : nsl] >> 6);
        if ((int)threadIdx.x <= sp.sl)
            firsts[threadIdx.x] =
                (int)(S.sptr[sp.s0 + threadIdx.x < nsl ? sp.s0 + threadIdx.x : nsl] >> 6) - e0;
        __syncthreads();
        ne = first(sp.sl);
        run = sell_run(S, sp.s0, sp.s0 + sp.sl, n);
#pragma unroll
        for (int t = 0; t < TW; t++) {
            const int e = (wave_in_block() + RW * t) * run;
            int k = 0;
            while (k + 1 < sp.sl && first(k + 1) <= e) k++;
            k0[t] = k;
            if constexpr (MAXE > 0) {
                const int lane = opaque_lane();
#pragma unroll
                for (int g = 0; g < MAXE / 4; g++)
#pragma unroll
                    for (int i = 0; i < 4; i++) rv[t][g][i] = (TV)0;
#pragma unroll
                for (int g = 0; g < MAXE / 4; g++)
                    if (4 * g < run && e + 4 * g < ne)
                        load4<TV>(vals + ((int64_t)(e0 + e + 4 * g) << 6) + lane * 4, rv[t][g]);
#pragma unroll
                for (int i = 0; i < (MAXE + 63) / 64; i++) {
                    const int kk = 64 * i + lane;
                    rb[t][i] = kk < run && e + kk < ne ? base[e0 + e + kk] : 0;
                }
            }
        }
    }
    template <typename TVR>
    __device__ inline double2 resid(const TVR* v, const RowRep& rep)
    {
        return resid_sell<SEG_SELL, TVR>(sp, n, S, nullptr, v, rep, nullptr);
    }
    __device__ inline void products(const TX* __restrict__ w, TX (&q)[NR][1])
    {
        const int lane = threadIdx.x & 63, wave = wave_in_block();
#pragma unroll
        for (int t = 0; t < TW; t++) {
            const int rn = wave + RW * t;
            const int b = rn * run, e1 = min(b + run, ne);
            if (b >= e1) continue;
            int k = k0[t], next = first(k + 1);
            TX s = (TX)0;
            // a slice ends in the run: leave its sum, go to the next
            auto step = [&](int e) {
                while (e == next) {
                    sums[slot(rn, k) + lane] = s;
                    s = (TX)0;
                    k++;
                    next = first(k + 1);
                }
            };
            if constexpr (MAXE > 0) {
                // LDS reads A groups ahead of their use (places past the run
                // are 0 and read the window's first)
                constexpr int A = 4, NG = MAXE / 4;
                TX xv[NG][4];
#pragma unroll
                for (int g = 0; g < NG + A; g++) {
                    if (g < NG) {
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const int kk = 4 * g + i;
                            xv[g][i] = w[__builtin_amdgcn_readlane(rb[t][kk >> 6], kk & 63) + lane];
                        }
                    }
                    if (g >= A && b + 4 * (g - A) < e1) {
                        step(b + 4 * (g - A));
#pragma unroll
                        for (int i = 0; i < 4; i++) s += (TX)rv[t][g - A][i] * xv[g - A][i];
                    }
                }
            } else {
                const TV* __restrict__ v = vals + ((int64_t)e0 << 6) + opaque_lane() * 4;
                const int32_t* __restrict__ pb = base + e0;
                constexpr int SG = sizeof(TV) == 4 ? 4 : 3;
                for (int e = b; e < e1; e += 4 * SG) {
                    TV vv[SG][4];
                    int pl[SG][4];
#pragma unroll
                    for (int g = 0; g < SG; g++)
                        if (e + 4 * g < e1) {
                            load4<TV>(v + ((int64_t)(e + 4 * g) << 6), vv[g]);
#pragma unroll
                            for (int i = 0; i < 4; i++) pl[g][i] = pb[e + 4 * g + i];
                        }
#pragma unroll
                    for (int g = 0; g < SG; g++)
                        if (e + 4 * g < e1) {
                            step(e + 4 * g);
#pragma unroll
                            for (int i = 0; i < 4; i++) s += (TX)vv[g][i] * w[pl[g][i] + lane];
                        }
                }
            }
            sums[slot(rn, k) + lane] = s;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NR; j++) {
            const int kk = wave + RW * j;
            TX s = (TX)0;
            if (kk < sp.sl && (sp.s0 + kk) * 64 < n) {
                const int f0 = first(kk), f1 = first(kk + 1);
                if (f1 > f0)
                    for (int rn = f0 / run; rn * run < f1; rn++) s += sums[slot(rn, kk) + lane];
            }
            q[j][0] = s;
        }
    }
};

template <int MAXE, typename TX>
__device__ inline void run_sell(const CgArgs<TX>& a, int iters, int seg, const SellView& S,
                                const TX* __restrict__ vals, const int32_t* __restrict__ base,
                                const int32_t* __restrict__ list,
                                const int32_t* __restrict__ woff,
                                const int32_t* __restrict__ own0, unsigned char* lds, int* firsts)
{
    SellForm<SELL_MAXR / RW, MAXE, TX, TX> f;
    f.S = S;
    f.vals = vals;
    f.base = base;
    f.list = list + woff[seg];
    f.nw = woff[seg + 1] - woff[seg];
    f.own0 = own0[seg];
    f.n = a.n;
    f.sp = seg_span(a.g, seg);
    f.sums = reinterpret_cast<TX*>(lds);
    f.firsts = firsts;
    TX* win = f.sums + SELL_SUMS + 64;
    if (threadIdx.x < 64) {
        win[(int)threadIdx.x - 64] = (TX)0;
        win[f.nw + threadIdx.x] = (TX)0;
    }
    cg_resident(a, iters, seg, f, win);
}

template <int MAXE, typename TX>
__global__ __launch_bounds__(RT) void k_cg_sell(CgArgs<TX> a, int iters, SellView S,
                                                const TX* __restrict__ vals,
                                                const int32_t* __restrict__ base,
                                                const int32_t* __restrict__ list,
                                                const int32_t* __restrict__ woff,
                                                const int32_t* __restrict__ own0)
{
    extern __shared__ unsigned char lds[];
    __shared__ int firsts[SELL_MAXR + 1];
    run_sell<MAXE, TX>(a, iters, seg_of_block(blockIdx.x, a.g.B), S, vals, base, list, woff, own0,
                       lds, firsts);
}

// Several requests in one launch: every block works on the request whose
// block range holds it, exactly as in a launch of that request alone.
// A pointer of the table, read as a pointer to global memory: as a generic one
// it would have every access through it, and the waits, take the flat path.
template <typename T>
__device__ inline T* in_global(T* const& field)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return (T*)*reinterpret_cast<__attribute__((address_space(1))) T* const*>(
        reinterpret_cast<const char*>(&field));
#else
    return field;
#endif
}

enum CgVariant { CG_SYM14_2, CG_SYM14_4, CG_SYM5_2, CG_SYM5_4, CG_BSYM3_8, CG_BSYM3_4, CG_BSYM3_3, CG_BSYM3_X,
                 CG_BSYM2_8, CG_BSYM2_4, CG_BSYM2_3, CG_SELL };

__global__ __launch_bounds__(RT) void k_cg_batch(const CgEntry* __restrict__ tab, int n, int iters,
                                                 CgEpochs first)
{
    extern __shared__ unsigned char lds[];
    __shared__ int firsts[SELL_MAXR + 1];
    int s = 0;
    while (s + 1 < n && tab[s + 1].first <= (int)blockIdx.x) s++;
    const CgEntry& e = tab[s];
    CgArgs<float> a;
    a.n = e.a.n;
    a.g = Seg{e.a.g.B, e.a.g.R, in_global(e.a.g.cut)};
    a.x = in_global(e.a.x);
    a.r = in_global(e.a.r);
    a.p = in_global(e.a.p);
    a.z = in_global(e.a.z);
    a.dinv = in_global(e.a.dinv);
    a.rep.v64 = in_global(e.a.rep.v64);
    a.rep.v32 = nullptr;   // served matrices are FP64 assemblies
    a.rep.b = in_global(e.a.rep.b);
    a.rep.x64 = in_global(e.a.rep.x64);
    a.rep.ratio = e.a.rep.ratio;
    a.sc = in_global(e.a.sc);
    a.words = in_global(e.a.words);
    a.epoch = first.e[s];
    a.polls = e.a.polls;
    a.limit = e.a.limit;
    const float* vals = in_global(e.vals);
    const RelWin W{in_global(e.W.piece), e.W.npiece, in_global(e.W.sh), in_global(e.W.u)};
    const int seg = seg_of_block((int)blockIdx.x - e.first, a.g.B);
    switch (e.variant) {
    case CG_SYM14_2: run_sym<14, 2, float>(a, iters, seg, vals, W, lds); break;
    case CG_SYM14_4: run_sym<14, 4, float>(a, iters, seg, vals, W, lds); break;
    case CG_SYM5_2: run_sym<5, 2, float>(a, iters, seg, vals, W, lds); break;
    case CG_SYM5_4: run_sym<5, 4, float>(a, iters, seg, vals, W, lds); break;
    case CG_BSYM3_8: run_bsym<3, 14, 1, 8, false, float>(a, iters, seg, vals, W, lds); break;
    case CG_BSYM3_4: run_bsym<3, 14, 1, 4, false, float>(a, iters, seg, vals, W, lds); break;
    case CG_BSYM3_X: run_bsym<3, 14, 1, 3, true, float>(a, iters, seg, vals, W, lds); break;
    case CG_BSYM3_3: run_bsym<3, 14, 1, 3, false, float>(a, iters, seg, vals, W, lds); break;
    case CG_BSYM2_8: run_bsym<2, 5, 1, 8, false, float>(a, iters, seg, vals, W, lds); break;
    case CG_BSYM2_4: run_bsym<2, 5, 1, 4, false, float>(a, iters, seg, vals, W, lds); break;
    case CG_BSYM2_3: run_bsym<2, 5, 1, 3, false, float>(a, iters, seg, vals, W, lds); break;
    default: {
        const SellView S{nullptr, in_global(e.S.sptr), in_global(e.S.spat), in_global(e.S.pptr),
                         in_global(e.S.plen), in_global(e.S.pdel)};
        run_sell<SELL_MAXE, float>(a, iters, seg, S, vals, in_global(e.base), in_global(e.list),
                                   in_global(e.woff), in_global(e.own0), lds, firsts);
    }
    }
}

// ---------------------------------------------------------------------------
// Windows as lists: a bitmap of the columns of the segment's rows in LDS; a
// column's place is the number of set bits below it.
constexpr int64_t WIN_MAXN = LDS_DYN / 8 * 32;   // columns a bitmap and its counts hold

// what marks and places the columns of a segment: CSR rows, or full slices
struct WinCsr {
    int64_t n;
    int R;
    const int32_t* rp;
    const int32_t* col;
    uint16_t* lcol;

    __device__ inline void span(int seg, int64_t& row0, int& rows) const
    {
        row0 = (int64_t)seg * R * 64;
        const int64_t left = n - row0, most = (int64_t)R * 64;
        rows = (int)(left < 0 ? 0 : (left < most ? left : most));
    }
    __device__ inline void mark(int64_t row0, int rows, uint32_t* bits) const
    {
        const int32_t k1 = rp[row0 + rows];
        for (int32_t k = rp[row0] + threadIdx.x; k < k1; k += RT) {
            const int32_t c = col[k];
            atomicOr(&bits[c >> 5], 1u << (c & 31));
        }
    }
    __device__ inline int longest(int64_t row0, int rows) const
    {
        int len = 0;
        for (int i = threadIdx.x; i < rows; i += RT)
            len = max(len, rp[row0 + i + 1] - rp[row0 + i]);
        return len;
    }
    template <class P>
    __device__ inline void fill(int64_t row0, int rows, P place) const
    {
        const int32_t k1 = rp[row0 + rows];
        for (int32_t k = rp[row0] + threadIdx.x; k < k1; k += RT) lcol[k] = (uint16_t)place(col[k]);
    }
};

struct WinSell {
    int64_t n;
    Seg g;
    SellView S;
    int32_t* base;

    __device__ inline void span(int seg, int64_t& row0, int& rows) const
    {
        const Span s = seg_span(g, seg);
        row0 = s.s0 * 64;
        const int64_t left = n - row0, most = (int64_t)s.sl * 64;
        rows = (int)(left < 0 ? 0 : (left < most ? left : most));
    }
    // f(entry index, first column) of every slice entry, over the block
    template <class F>
    __device__ inline void entries(int64_t row0, int rows, F f) const
    {
        const int lane = threadIdx.x & 63;
        for (int sl = wave_in_block(); sl * 64 < rows; sl += RW) {
            const int64_t slice = row0 / 64 + sl;
            const int pid = S.spat[slice];
            const int32_t* d = S.pdel + S.pptr[pid];
            const int len = S.plen[pid];
            for (int k = lane; k < ((len + 3) & ~3); k += 64)   // padding: any column
                f((S.sptr[slice] >> 6) + k, slice * 64 + (k < len ? d[k] : d[0]));
        }
    }
    __device__ inline void mark(int64_t row0, int rows, uint32_t* bits) const
    {
        entries(row0, rows, [&](int64_t, int64_t c0) {
            const int64_t lo = c0 < 0 ? 0 : c0, hi = c0 + 63 < n ? c0 + 63 : n - 1;
            for (int64_t w = lo >> 5; lo <= hi && w <= hi >> 5; w++) {
                const int b0 = (int)(lo > w * 32 ? lo - w * 32 : 0);
                const int b1 = (int)(hi < w * 32 + 31 ? hi - w * 32 : 31);
                atomicOr(&bits[w], (~0u << b0) & (~0u >> (31 - b1)));
            }
        });
    }
    // (the entries of the segment)
    __device__ inline int longest(int64_t row0, int rows) const
    {
        if (rows <= 0) return 0;
        return (int)((S.sptr[(row0 + rows + 63) / 64] - S.sptr[row0 / 64]) >> 6);
    }
    template <class P>
    __device__ inline void fill(int64_t row0, int rows, P place) const
    {
        entries(row0, rows, [&](int64_t e, int64_t c0) {
            // (no lane inside the matrix: any place)
            const int64_t c = c0 < 0 ? 0 : c0;
            base[e] = c0 <= -64 || c0 >= n ? 0 : place((int32_t)c) - (int32_t)(c - c0);
        });
    }
};

template <class W>
__device__ inline void win_bits(const W& w, int64_t row0, int rows, uint32_t* bits, int words)
{
    for (int i = threadIdx.x; i < words; i += RT) bits[i] = 0u;
    __syncthreads();
    if (rows > 0) {
        for (int i = threadIdx.x; i < rows; i += RT) {
            const int64_t c = row0 + i;
            atomicOr(&bits[c >> 5], 1u << (c & 31));
        }
        w.mark(row0, rows, bits);
    }
    __syncthreads();
}

// per segment: columns of its window; of all, the longest row (CSR) or the most
// entries of a segment (slices)
template <class W>
__global__ __launch_bounds__(RT) void k_win_count(W w, int32_t* __restrict__ wlen,
                                                  int32_t* __restrict__ maxlen)
{
    extern __shared__ uint32_t bits[];
    __shared__ int cnt, longest;
    if (threadIdx.x == 0) cnt = longest = 0;
    const int words = (int)((w.n + 31) / 32);
    int64_t row0;
    int rows;
    w.span(blockIdx.x, row0, rows);
    win_bits(w, row0, rows, bits, words);
    int s = 0;
    for (int i = threadIdx.x; i < words; i += RT) s += __popc(bits[i]);
    atomicAdd(&cnt, s);
    atomicMax(&longest, w.longest(row0, rows));
    __syncthreads();
    if (threadIdx.x == 0) {
        wlen[blockIdx.x] = cnt;
        atomicMax(maxlen, longest);
    }
}

template <class W>
__global__ __launch_bounds__(RT) void k_win_fill(W w, const int32_t* __restrict__ woff,
                                                 int32_t* __restrict__ list,
                                                 int32_t* __restrict__ own0)
{
    extern __shared__ uint32_t bits[];
    __shared__ int wsum[RW];
    const int words = (int)((w.n + 31) / 32);
    int32_t* below = reinterpret_cast<int32_t*>(bits + words);   // set bits before each word
    int64_t row0;
    int rows;
    w.span(blockIdx.x, row0, rows);
    win_bits(w, row0, rows, bits, words);
    // each thread a run of words; scan of the runs' counts over the block
    const int per = (words + RT - 1) / RT;
    const int w0 = min(words, (int)threadIdx.x * per), w1 = min(words, w0 + per);
    int s = 0;
    for (int i = w0; i < w1; i++) s += __popc(bits[i]);
    int inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(inc, o, 64);
        if ((int)(threadIdx.x & 63) >= o) inc += t;
    }
    if ((threadIdx.x & 63) == 63) wsum[threadIdx.x >> 6] = inc;
    __syncthreads();
    int run = inc - s;
    for (int k = 0; k < (int)(threadIdx.x >> 6); k++) run += wsum[k];
    int32_t* out = list + woff[blockIdx.x];
    for (int i = w0; i < w1; i++) {
        below[i] = run;
        uint32_t b = bits[i];
        while (b) {
            out[run++] = i * 32 + __ffs(b) - 1;
            b &= b - 1;
        }
    }
    __syncthreads();
    auto place = [&](int32_t c) {
        return below[c >> 5] + __popc(bits[c >> 5] & ((1u << (c & 31)) - 1u));
    };
    if (rows > 0) w.fill(row0, rows, place);
    if (threadIdx.x == 0) own0[blockIdx.x] = rows > 0 ? place((int32_t)row0) : 0;
}

int env_res(const char* name, int dflt)
{
    const char* v = getenv(name);
    return v && *v ? atoi(v) : dflt;
}

// Launches whose blocks wait for each other must not share the chip: they
// are ordered behind one another on the device, whatever stream or thread
// they come from
constexpr int MAXDEV = 64;
struct Order {
    std::mutex mu;
    hipEvent_t last = nullptr;
    hipStream_t stream = nullptr;
};
Order g_order[MAXDEV];

// Runs launches() on stream st in that order; hipSuccess, or what failed
template <class F>
hipError_t ordered(int device, hipStream_t st, F launches)
{
    Order& o = g_order[device];
    std::lock_guard<std::mutex> lock(o.mu);
    hipError_t e = hipSuccess;
    if (!o.last) e = hipEventCreateWithFlags(&o.last, hipEventDisableTiming);
    else if (o.stream != st) e = hipStreamWaitEvent(st, o.last, 0);
    if (e != hipSuccess) return e;
    // (of several launches the first may run although a later one failed)
    const hipError_t le = launches();
    o.stream = st;
    e = hipEventRecord(o.last, st);
    return le != hipSuccess ? le : e;
}

template <class K, typename... A>
hipError_t launch_alone(hipStream_t st, K kernel, int blocks, size_t lds, A... args)
{
    // one block per compute unit: more than half of its LDS
    lds = std::max<size_t>(lds, LDS_MAX / 2 + 1024);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_DYN);
    if (e != hipSuccess) return e;
    kernel<<<blocks, RT, lds, st>>>(args...);
    return hipGetLastError();
}

template <class K, typename... A>
int launch_ordered(Ctx* c, K kernel, int blocks, size_t lds, A... args)
{
    INS_HIP_CHECK(c, ordered(c->device, c->stream, [&] {
        return launch_alone(c->stream, kernel, blocks, lds, args...);
    }));
    return INS_OK;
}

template <typename TX>
CgArgs<TX> cg_args(Ctx* c, const Seg& g, int64_t n, TX* x, TX* r, TX* p, TX* z, const TX* dinv,
                   const ResRep& rep, Scal* sc, uint32_t epoch, int limit)
{
    // bound of a wait: a poll takes about a microsecond
    const int polls = env_res("INS_RESIDENT_POLLS", 500000);
    return CgArgs<TX>{n, g, x, r, p, z, dinv, rep, sc, c->res.words.p, epoch, polls, limit};
}

}  // namespace

// The words, and the first epoch of a launch of `iters` iterations on stream st:
// each launch has a range of epochs of its own, of all it may use, so whatever
// words a launch left, one that was given up or whose end nobody looked at
// included, are of no epoch that a later one waits for.  Epochs are 32 bits and
// start again, on zeroed words, before they would repeat.
int resident_words(Ctx* c, hipStream_t st, int iters, uint32_t* first)
{
    Resident& S = c->res;
    const int64_t most = 8 * (int64_t)iters + 64;   // replacements included
    const bool fresh = !S.words.p;
    if (fresh) INS_TRY(ensure(c, S.words, MEET_WORDS));
    if (fresh || S.used + most > (int64_t)UINT32_MAX) {
        INS_HIP_CHECK(c, hipMemsetAsync(S.words.p, 0, MEET_WORDS * sizeof(uint64_t), st));
        S.used = 0;
    }
    *first = (uint32_t)S.used + 1u;
    S.used += most;
    return INS_OK;
}

int resident_blocks(int n_cu)
{
    static const int on = env_res("INS_RESIDENT", 1);
    if (!on) return 0;
    return n_cu < NXCD ? 0 : std::min(RBMAX, n_cu / NXCD * NXCD);
}

// Segments of a CSR solve.  Up to 64 blocks, whose sums meet in one stage, while
// eight register passes, 8 RT / LPR rows, hold a segment (1,944 elastic rows:
// 6.4 us per iteration with 31 blocks, 12.3 with 8 of the largest segments;
// 15,000 rows of 27: 4.9 and 5.2); beyond them the sums cost the same up to 256 blocks, so all are
// used (125,000 rows numbered at random, whose windows are gathers of one
// lane per cycle: C 4.9 us with 123 blocks).
//
// Rows that the registers do not hold (more than 4 LPR entries) are streamed
// each iteration.  That pays while values and places, 10 or 6 bytes an entry,
// stay near (the L2s hold 4 MB for 32 compute units): us per iteration, streamed
// and with the three kernels on whole vectors,
//   LPR 16, elastic rows of 78, FP64   27 MB 14.1 / 17.9   35 MB 20.5 / 20.5   45 MB 25.8 / 22.9
//                               FP32   30 MB 17.9 / 21.8   34 MB 26.7 / 23.1   41 MB 33.4 / 26.3
//   LPR 8, scattered rows of 31, FP64  34 MB 34.2 / 54.2   39 MB 38.1 / 57.3
//          rows of 26, one of 200, FP64 34 MB 19.1 / 25.3
// csr_windows looks at the longest row.  FP32 rows of at most 4 LPR entries are
// streamed up to CSR_ROWS per block (258,000 rows of 27: 26.3 / 27.5).  FP64
// segments are a matter of n and nnz alone, for the allocation-free solve knows no
// more and has the same bits: where rows of about equal length are neither held
// nor near there are none.
// passes of a block over its rows, and the most that registers hold
constexpr int CSR_PASSES = 8;
static int csr_passes(const Seg& g, int lpr) { return (g.R * 64 * lpr + RT - 1) / RT; }

static bool csr_near(int64_t nnz, int lpr, int n_cu, int vec_bytes)
{
    return nnz * (vec_bytes + 2) <= (int64_t)n_cu * (lpr >= 16 ? 120 << 10 : 160 << 10);
}

Seg csr_segments(int64_t n, int64_t nnz, int lpr, int n_cu, bool mixed)
{
    const int bmax = resident_blocks(n_cu);
    const int64_t nsl = (n + 63) / 64;
    Seg g;
    if (bmax == 0) return g;
    const int64_t regs = std::max(1, 64 / lpr);
    int64_t R = std::min<int64_t>(regs, (nsl + 63) / 64);
    if (nsl > 64 * R) R = (nsl + bmax - 1) / bmax;
    if (R > (mixed ? CSR_ROWS / 64 : regs)) return g;
    if (!mixed && nnz > 4 * lpr * n && !csr_near(nnz, lpr, n_cu, 8)) return g;
    int64_t B = (nsl + R - 1) / R;
    if (B >= NXCD) B = std::min<int64_t>(bmax, (B + NXCD - 1) / NXCD * NXCD);
    g.R = (int)R;
    g.B = (int)B;
    return g;
}

namespace {
// Lists of the windows of one pattern and segmentation, built once (L.gen);
// prep allocates what the marks' places go to
template <class W, class P>
int list_windows(Ctx* c, WinList& L, const Seg& g, W w, P prep)
{
    if (L.gen == c->pattern_gen && L.B == g.B && L.R == g.R) return INS_OK;
    const size_t words = (size_t)((w.n + 31) / 32);
    L.gen = 0;   // a failure below leaves no list
    INS_TRY(ensure(c, L.wlen, RBMAX + 1));
    INS_HIP_CHECK(c, hipMemsetAsync(L.wlen.p + RBMAX, 0, sizeof(int32_t), c->stream));
    INS_HIP_CHECK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(&k_win_count<W>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, LDS_DYN));
    k_win_count<W><<<g.B, RT, words * 4, c->stream>>>(w, L.wlen.p, L.wlen.p + RBMAX);
    INS_HIP_CHECK(c, hipGetLastError());
    int32_t len[RBMAX + 1], off[RBMAX + 1];
    INS_HIP_CHECK(c, hipMemcpyAsync(len, L.wlen.p, sizeof len, hipMemcpyDeviceToHost, c->stream));
    INS_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    off[0] = 0;
    L.wmax = 0;
    for (int b = 0; b < g.B; b++) {
        off[b + 1] = off[b] + len[b];
        L.wmax = std::max(L.wmax, len[b]);
    }
    L.maxlen = len[RBMAX];
    if (L.wmax <= 65536) {   // more fits no LDS (and places of CSR entries are 16 bits)
        INS_TRY(ensure(c, L.woff, RBMAX + 1));
        INS_TRY(ensure(c, L.own0, RBMAX));
        INS_TRY(ensure(c, L.list, (size_t)off[g.B] + 1));
        INS_TRY(prep(w));
        INS_HIP_CHECK(c, hipMemcpyAsync(L.woff.p, off, (g.B + 1) * sizeof(int32_t),
                                        hipMemcpyHostToDevice, c->stream));
        INS_HIP_CHECK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(&k_win_fill<W>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_DYN));
        k_win_fill<W><<<g.B, RT, words * 8, c->stream>>>(w, L.woff.p, L.list.p, L.own0.p);
        INS_HIP_CHECK(c, hipGetLastError());
        INS_HIP_CHECK(c, hipStreamSynchronize(c->stream));   // off is on this stack
    }
    L.gen = c->pattern_gen;
    L.B = g.B;
    L.R = g.R;
    return INS_OK;
}

size_t rel_lds(const Ctx* c, int D, int R, int vec_bytes)
{
    return (size_t)c->res.rel_w * D * vec_bytes + bsym_sum_lds(D, R) +
           (D > 1 && vec_bytes == 4 ? bsym_ext_lds(D, D == 3 ? 14 : 5, R) : 0);
}

bool lds_fits(int64_t bytes) { return bytes <= (int64_t)LDS_DYN; }
}  // namespace

// Windows of the current CSR pattern; fits: whether they fit the LDS beside
// the block's q, and the registers or the caches the rows
int csr_windows(Ctx* c, const Seg& g, int lpr, int vec_bytes, bool* fits)
{
    Resident& S = c->res;
    INS_TRY(list_windows(c, S.csr, g,
                         WinCsr{c->n_active, g.R, c->row_ptr.p, c->col.p, nullptr},
                         [&](WinCsr& w) -> int {
                             INS_TRY(ensure(c, S.lcol, (size_t)c->nnz + 1));
                             w.lcol = S.lcol.p;
                             return INS_OK;
                         }));
    *fits = lds_fits(((int64_t)CSR_ROWS + S.csr.wmax) * vec_bytes) &&
            (S.csr.maxlen <= 4 * lpr || csr_near(c->nnz, lpr, c->n_cu, vec_bytes));
    return INS_OK;
}

namespace {
template <int LPR, typename TV, typename TX>
int launch_csr_lpr(Ctx* c, const Seg& g, const CgArgs<TX>& a, int iters, const TV* val)
{
    const Resident& S = c->res;
    const size_t lds = (size_t)(CSR_ROWS + S.csr.wmax) * sizeof(TX);
    const int passes = csr_passes(g, LPR);
    const bool regs = S.csr.maxlen <= 4 * LPR;
#define INS_CG_CSR(NP)                                                                       \
    return launch_ordered(c, k_cg_csr<LPR, NP, TV, TX>, g.B, lds, a, iters, (const int32_t*)c->row_ptr.p, \
                          (const int32_t*)c->col.p,                                           \
                          (const uint16_t*)S.lcol.p, val, (const int32_t*)S.csr.list.p,          \
                          (const int32_t*)S.csr.woff.p, (const int32_t*)S.csr.own0.p)
    if (regs && passes <= 2) INS_CG_CSR(2);
    if (regs && passes <= 4) INS_CG_CSR(4);
    if (regs && passes <= CSR_PASSES) INS_CG_CSR(CSR_PASSES);
    INS_CG_CSR(0);
#undef INS_CG_CSR
}
}  // namespace

// up to `iters` iterations of a CSR solve in one launch
template <typename T>
int resident_csr(Ctx* c, const Seg& g, int lpr, const T* val, T* x, T* r, T* p, T* z,
                 const T* dinv, const ResRep& rep, int iters, int limit)
{
    uint32_t epoch;
    INS_TRY(resident_words(c, c->stream, iters, &epoch));
    const CgArgs<T> a =
        cg_args<T>(c, g, c->n_active, x, r, p, z, dinv, rep, c->scal.p, epoch, limit);
    if (lpr == 32) return launch_csr_lpr<32>(c, g, a, iters, val);
    if (lpr == 16) return launch_csr_lpr<16>(c, g, a, iters, val);
    if (lpr == 8) return launch_csr_lpr<8>(c, g, a, iters, val);
    return launch_csr_lpr<4>(c, g, a, iters, val);
}
template int resident_csr<double>(Ctx*, const Seg&, int, const double*, double*, double*, double*,
                                  double*, const double*, const ResRep&, int, int);
template int resident_csr<float>(Ctx*, const Seg&, int, const float*, float*, float*, float*,
                                 float*, const float*, const ResRep&, int, int);

// ---------------------------------------------------------------------------
// SELL solves
SegForm sell_form(const Ctx* c)
{
    const Sell& S = c->sell;
    if (!S.ok) return SEG_NONE;
    if (!S.sym_on) return SEG_SELL;
    if ((S.sdpn > 1) != S.perm_on) return SEG_NONE;
    if (S.sdpn == 1) return S.nu == 14 ? SEG_SYM14 : (S.nu == 5 ? SEG_SYM5 : SEG_NONE);
    if (S.sdpn == 3 && S.nu == 14) return SEG_BSYM3;
    if (S.sdpn == 2 && S.nu == 5) return SEG_BSYM2;
    return SEG_NONE;
}

namespace {
int form_dim(SegForm f) { return f == SEG_BSYM3 ? 3 : (f == SEG_BSYM2 ? 2 : 1); }

// the common window of symmetric slices, for segments of R slices
int rel_windows(Ctx* c, int R)
{
    Resident& S = c->res;
    if (S.rel_gen == c->pattern_gen && S.rel_R == R) return INS_OK;
    S.rel_gen = 0;
    const std::vector<int32_t>& u = c->sell.su_host;
    const int nu = (int)u.size();
    std::vector<int64_t> d;
    for (int k = nu - 1; k > 0; k--) d.push_back(-(int64_t)u[k]);
    for (int k = 0; k < nu; k++) d.push_back(u[k]);
    const int64_t len = (int64_t)R * 64;
    std::vector<int4> piece;
    std::vector<int32_t> sh(2 * nu - 1);
    int64_t start = d[0], place = 0;
    for (size_t i = 0; i < d.size(); i++) {
        if (i > 0 && d[i] > d[i - 1] + len) {   // a gap: the interval ends at d[i-1] + len
            place += d[i - 1] + len - start;
            start = d[i];
        }
        const int64_t s = place + d[i] - start;
        if (s + len > INT32_MAX / 4) return fail(c, INS_ERR_RANGE, "window of a segment");
        const int k = (int)(std::lower_bound(u.begin(), u.end(), (int32_t)std::llabs(d[i])) - u.begin());
        sh[d[i] > 0 ? 2 * k - 1 : 2 * k] = (int32_t)s;
        const bool last = i + 1 == d.size() || d[i + 1] > d[i] + len;
        if (last)
            for (int64_t o = 0; o < d[i] + len - start; o += 64)
                piece.push_back(int4{(int)(start + o), (int)(place + o),
                                     (int)std::min<int64_t>(64, d[i] + len - start - o), 0});
    }
    S.rel_w = (int)(place + d.back() + len - start);
    S.rel_n = (int)piece.size();
    INS_TRY(ensure(c, S.rel_piece, piece.size()));
    INS_TRY(ensure(c, S.rel_sh, sh.size()));
    INS_HIP_CHECK(c, hipMemcpyAsync(S.rel_piece.p, piece.data(), piece.size() * sizeof(int4),
                                    hipMemcpyHostToDevice, c->stream));
    INS_HIP_CHECK(c, hipMemcpyAsync(S.rel_sh.p, sh.data(), sh.size() * sizeof(int32_t),
                                    hipMemcpyHostToDevice, c->stream));
    INS_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    S.rel_gen = c->pattern_gen;
    S.rel_R = R;
    return INS_OK;
}
}  // namespace

namespace {
// Cuts of the full slices into at most bmax segments of about equal numbers
// of entries (slices differ up to five times in length), once per pattern
int sell_cuts(Ctx* c, int bmax, Seg* g)
{
    Resident& S = c->res;
    const int64_t nsl = c->sell.nslices;
    // more slices or entries than all segments hold: no cuts, and no search for any
    const int64_t regs = (int64_t)TASKS * SELL_MAXE;
    if (nsl > (int64_t)bmax * SELL_MAXR || c->sell.nvals / 64 > bmax * regs) return INS_OK;
    if (S.cut_gen != c->pattern_gen) {
        std::vector<int64_t> ptr((size_t)nsl + 1);
        INS_HIP_CHECK(c, hipMemcpyAsync(ptr.data(), c->sell.slice_ptr.p, ptr.size() * sizeof(int64_t),
                                        hipMemcpyDeviceToHost, c->stream));
        INS_HIP_CHECK(c, hipStreamSynchronize(c->stream));
        const int64_t total = ptr[nsl] / 64;
        // 64 blocks while the registers hold their entries, beyond: all blocks
        int64_t most = (total + 63) / 64;
        if (most > regs) most = (total + bmax - 1) / bmax;
        std::vector<int32_t> cut;
        int longest = 0;
        for (int tries = 0; tries < 64; tries++) {
            cut.assign(1, 0);
            longest = 0;
            for (int64_t s = 0; s < nsl;) {
                const int64_t s0 = s;
                do s++;
                while (s < nsl && s - s0 < SELL_MAXR && (ptr[s + 1] - ptr[s0]) / 64 <= most);
                cut.push_back((int32_t)s);
                longest = std::max(longest, (int)(s - s0));
            }
            if ((int)cut.size() - 1 <= bmax) break;
            most += most / 32 + 1;
        }
        S.cut_B = (int)cut.size() - 1;
        S.cut_R = longest;
        S.cut_gen = 0;
        if (S.cut_B > bmax) S.cut_B = 0;
        if (S.cut_B >= NXCD)
            while (S.cut_B % NXCD) {   // empty segments at the end
                cut.push_back((int32_t)nsl);
                S.cut_B++;
            }
        INS_TRY(ensure(c, S.cut, RBMAX + 1));
        if (S.cut_B) {
            INS_HIP_CHECK(c, hipMemcpyAsync(S.cut.p, cut.data(), cut.size() * sizeof(int32_t),
                                            hipMemcpyHostToDevice, c->stream));
            INS_HIP_CHECK(c, hipStreamSynchronize(c->stream));
        }
        S.cut_gen = c->pattern_gen;
    }
    g->B = S.cut_B;
    g->R = S.cut_R;
    g->cut = S.cut.p;
    return INS_OK;
}
}  // namespace

// Segments of a SELL solve.  Few blocks meet cheaply (one stage up to 64), so
// small problems take long segments: 16 slices of scalar rows, 4 of node
// blocks; beyond 64 such segments all compute units are used.
//
// Where the registers no longer hold the entries, streaming them through a
// few waves per compute unit is no better than the three kernels, which sweep
// the slices in the order their mirrors are read.  Measured, us per iteration,
// resident against three kernels, at the last size held and the next:
//   scalar rows FP32 (32 slices)   353k rows 13.1 / 16.6, 525k 31.5 / 20.5
//   scalar rows FP64 (16 slices)   223k rows 10.5 / 23.0, 353k 28.2 / 26.8
//   node blocks FP32 (7 slices)    89k nodes 11.0 / 25.3; streamed from the
//     sixth slice on instead of held in LDS the same size took 24.4
//   full slices FP32 (1280 entries) 223k rows of a degree-2 field 21.8 / 29.0
// FP64 node blocks gain streamed too (2 slices held: 26k nodes 8.7 / 32.9,
// streamed: 42k 20.2 / 36.4, 223k 61.6 / 70.2).
int sell_segments(Ctx* c, bool mixed, Seg* out)
{
    *out = Seg{};
    const SegForm f = sell_form(c);
    const int bmax = resident_blocks(c->n_cu);
    if (f == SEG_NONE || bmax == 0) return INS_OK;
    const int D = form_dim(f), vec = mixed ? 4 : 8;
    const int64_t items = D > 1 ? c->sell.snodes : c->n_active;
    const int64_t nsl = (items + 63) / 64;
    Seg g;
    bool fits = false;
    if (f == SEG_SELL) {
        if (items > WIN_MAXN) return INS_OK;
        INS_TRY(sell_cuts(c, bmax, &g));
        if (!g.B) return INS_OK;
        INS_TRY(sell_windows(c, g, vec, &fits));
        if (fits && c->res.sell.maxlen <= TASKS * SELL_MAXE) *out = g;
        return INS_OK;
    }
    int64_t R = D > 1 ? 4 : 16;
    if (nsl > 64 * R) R = (nsl + bmax - 1) / bmax;
    else if (D > 1 && nsl <= 128) R = 2;
    const int64_t most = D > 1 ? (mixed ? 7 : 4 * RW) : (mixed ? 4 * RW : 2 * RW);
    if (R > most) return INS_OK;
    int64_t B = (nsl + R - 1) / R;
    if (B >= NXCD) B = std::min<int64_t>(bmax, (B + NXCD - 1) / NXCD * NXCD);
    g.B = (int)B;
    g.R = (int)R;
    INS_TRY(sell_windows(c, g, vec, &fits));
    if (fits) *out = g;
    return INS_OK;
}

int sell_windows(Ctx* c, const Seg& g, int vec_bytes, bool* fits)
{
    Resident& S = c->res;
    const SegForm f = sell_form(c);
    if (f == SEG_SELL) {
        const Sell& L = c->sell;
        const SellView v{nullptr, L.slice_ptr.p, L.slice_pat.p, L.pat_ptr.p, L.pat_len.p,
                         L.pat_delta.p};
        INS_TRY(list_windows(c, S.sell, g, WinSell{c->n_active, g, v, nullptr},
                             [&](WinSell& w) -> int {
                                 INS_TRY(ensure(c, S.sell_base, (size_t)(L.nvals / 64) + 1));
                                 w.base = S.sell_base.p;
                                 return INS_OK;
                             }));
        // beside the window: the runs' sums of every slice (SellForm)
        *fits = S.sell.wmax <= 65536 && lds_fits((int64_t)(S.sell.wmax + SELL_SUMS + 128) * vec_bytes);
        return INS_OK;
    }
    INS_TRY(rel_windows(c, g.R));
    const int D = form_dim(f);
    *fits = lds_fits((int64_t)rel_lds(c, D, g.R, vec_bytes));
    return INS_OK;
}

namespace {
template <int NU, typename T>
int launch_sym(Ctx* c, const Seg& g, const CgArgs<T>& a, int iters, const T* vals, const RelWin& W)
{
    const size_t lds = (size_t)c->res.rel_w * sizeof(T);
    if constexpr (sizeof(T) == 4)
        if (g.R > 2 * RW) return launch_ordered(c, k_cg_sym<NU, 4, T>, g.B, lds, a, iters, vals, W);
    return launch_ordered(c, k_cg_sym<NU, 2, T>, g.B, lds, a, iters, vals, W);
}

template <int D, int NU, typename T>
int launch_bsym(Ctx* c, const Seg& g, const CgArgs<T>& a, int iters, const T* vals, const RelWin& W)
{
    const int parts = bsym_parts(g.R);
    const size_t lds = rel_lds(c, D, g.R, sizeof(T));
#define INS_CG_BSYM(NR, PARTS, EXT) \
    return launch_ordered(c, k_cg_bsym<D, NU, NR, PARTS, EXT, T>, g.B, lds, a, iters, vals, W)
    if (parts == 8) INS_CG_BSYM(1, 8, false);
    if (parts == 4) INS_CG_BSYM(1, 4, false);
    if constexpr (sizeof(T) == 8) {
        if (parts == 2) INS_CG_BSYM(1, 2, false);
        if (parts == 1 && g.R <= 2 * RW) INS_CG_BSYM(2, 1, false);
        if (parts == 1) INS_CG_BSYM(4, 1, false);
        INS_CG_BSYM(1, 3, false);
    } else {
        if constexpr (D == 3)
            if (g.R * 3 > TASKS) INS_CG_BSYM(1, 3, true);
        INS_CG_BSYM(1, 3, false);
    }
#undef INS_CG_BSYM
}
}  // namespace

// up to `iters` iterations of a SELL solve in one launch
template <typename T>
int resident_sell(Ctx* c, const Seg& g, T* x, T* r, T* p, T* z, const T* dinv,
                  const ResRep& rep, int iters, int limit)
{
    uint32_t epoch;
    INS_TRY(resident_words(c, c->stream, iters, &epoch));
    Resident& S = c->res;
    const SegForm f = sell_form(c);
    const int64_t items = form_dim(f) > 1 ? c->sell.snodes : c->n_active;
    const CgArgs<T> a = cg_args<T>(c, g, items, x, r, p, z, dinv, rep, c->scal.p, epoch, limit);
    const Sell& L = c->sell;
    const T *sym, *full;
    if constexpr (sizeof(T) == 8) {
        sym = L.vs64.p;
        full = L.v64.p;
    } else {
        sym = L.vs.p;
        full = L.v32.p;
    }
    if (f == SEG_SELL) {
        const SellView v{nullptr, L.slice_ptr.p, L.slice_pat.p, L.pat_ptr.p, L.pat_len.p,
                         L.pat_delta.p};
        const size_t lds = (size_t)(S.sell.wmax + SELL_SUMS + 128) * sizeof(T);
        const int32_t *base = S.sell_base.p, *list = S.sell.list.p, *woff = S.sell.woff.p,
                      *own0 = S.sell.own0.p;
        constexpr int MAXE = sizeof(T) == 4 ? SELL_MAXE : 0;   // FP64: streamed
        return launch_ordered(c, k_cg_sell<MAXE, T>, g.B, lds, a, iters, v, full, base, list, woff,
                              own0);
    }
    const RelWin W{S.rel_piece.p, S.rel_n, S.rel_sh.p, L.su.p};
    if (f == SEG_SYM14) return launch_sym<14>(c, g, a, iters, sym, W);
    if (f == SEG_SYM5) return launch_sym<5>(c, g, a, iters, sym, W);
    if (f == SEG_BSYM3) return launch_bsym<3, 14>(c, g, a, iters, sym, W);
    return launch_bsym<2, 5>(c, g, a, iters, sym, W);
}
template int resident_sell<double>(Ctx*, const Seg&, double*, double*, double*, double*,
                                   const double*, const ResRep&, int, int);
template int resident_sell<float>(Ctx*, const Seg&, float*, float*, float*, float*, const float*,
                                  const ResRep&, int, int);

// ---------------------------------------------------------------------------
// Serving: a mixed SELL solve as an entry of a batch
// (whose limit the host sees to, as for the requests of the batched kernels)
int resident_entry(Ctx* c, const Seg& g, Scal* sc, CgEntry* e, size_t* lds)
{
    Resident& S = c->res;
    const Sell& L = c->sell;
    const SegForm f = sell_form(c);
    const int D = form_dim(f);
    ResRep rep;
    rep.b = c->sb;
    rep.x64 = c->sx64;
    rep.ratio = restart_ratio();
    rep.v64 = f == SEG_SELL ? L.v64.p : L.vs64.p;
    e->a = cg_args<float>(c, g, D > 1 ? L.snodes : c->n_active, c->x32.p, c->r32.p, c->p32.p,
                          c->q32.p, c->sd32, rep, sc, 0u, INT32_MAX);
    e->vals = f == SEG_SELL ? L.v32.p : L.vs.p;
    e->W = RelWin{S.rel_piece.p, S.rel_n, S.rel_sh.p, L.su.p};
    e->S = SellView{nullptr, L.slice_ptr.p, L.slice_pat.p, L.pat_ptr.p, L.pat_len.p, L.pat_delta.p};
    e->base = S.sell_base.p;
    e->list = S.sell.list.p;
    e->woff = S.sell.woff.p;
    e->own0 = S.sell.own0.p;
    const int parts = bsym_parts(g.R);
    const int bv = parts == 8 ? 0 : (parts == 4 ? 1 : (D == 3 && parts * g.R > TASKS ? 3 : 2));
    switch (f) {
    case SEG_SYM14: e->variant = g.R <= 2 * RW ? CG_SYM14_2 : CG_SYM14_4; break;
    case SEG_SYM5: e->variant = g.R <= 2 * RW ? CG_SYM5_2 : CG_SYM5_4; break;
    case SEG_BSYM3: e->variant = CG_BSYM3_8 + bv; break;
    case SEG_BSYM2: e->variant = CG_BSYM2_8 + bv; break;
    default: e->variant = CG_SELL;
    }
    *lds = f == SEG_SELL ? (size_t)(S.sell.wmax + SELL_SUMS + 128) * sizeof(float)
                         : rel_lds(c, D, g.R, 4);
    return INS_OK;
}

int resident_batch(int device, hipStream_t st, const CgEntry* tab, const std::vector<CgGroup>& groups,
                   int iters, const uint32_t* first)
{
    const hipError_t e = ordered(device, st, [&] {
        for (const CgGroup& g : groups) {
            CgEpochs ep;
            std::copy(first + g.first, first + g.first + g.n, ep.e);
            const hipError_t le =
                launch_alone(st, k_cg_batch, g.blocks, g.lds, tab + g.first, g.n, iters, ep);
            if (le != hipSuccess) return le;
        }
        return hipSuccess;
    });
    return e == hipSuccess ? INS_OK : INS_ERR_HIP;
}

}  // namespace ins
