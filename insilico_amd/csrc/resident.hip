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
__device__ inline bool meet_collect(Meet& m, double (&t)[NV], double* tot, int* dead)
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
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) t[k] = tot[k];
    m.epoch++;
    return *dead == 0;
}

// What every form of the resident kernel works on
template <typename TX>
struct CgArgs {
    int64_t n;          // items per component (rows, or nodes of a vector problem)
    int B, R;
    TX* x;
    TX* r;
    TX* p;
    TX* z;              // exchanged
    const TX* dinv;
    double* x64;        // mixed: the FP64 solution x is folded into
    Scal* sc;
    uint64_t* words;
    uint32_t epoch;
    int polls;
    int iters;          // iterations of this launch at most
    int limit;          // of the solve
};

// The iterations of one block.  F: the matrix form; NR slices per wave, D
// components per item.  Thread (wave w, lane l) owns items
// (first + w + RW j) * 64 + l of every component.
template <class F, typename TX>
__device__ inline void cg_resident(const CgArgs<TX>& a, F& f, TX* __restrict__ win)
{
    constexpr int NR = F::NR, D = F::D;
    constexpr bool mixed = sizeof(TX) == 4;
    __shared__ double sh[2][RW];
    __shared__ double tot[2][2];
    __shared__ int dead;
    Scal* sc = a.sc;
    if (sc->done || sc->stop || sc->abort || sc->rep_at != INT_MAX) return;
    int iters = sc->iters;
    if (iters >= a.limit) return;
    const double thr = sc->thr, delta2 = sc->delta2, rref = sc->rref;
    const bool restart = mixed && sc->restart;
    double rho = sc->rho[0];
    const int seg = seg_of_block(blockIdx.x, a.B);
    Meet m{a.words, a.epoch, a.polls, a.B, seg};
    const int lane = threadIdx.x & 63, wave = wave_in_block();
    const int64_t s0 = (int64_t)seg * a.R;
    const int64_t nn = a.n;
    if (threadIdx.x == 0) dead = 0;

    int64_t at[NR];      // own items (-1: none)
    TX x[NR][D], r[NR][D], d[NR][D];
#pragma unroll
    for (int j = 0; j < NR; j++) {
        const int sl = wave + RW * j;
        const int64_t i = (s0 + sl) * 64 + lane;
        at[j] = (sl < a.R && i < nn) ? i : -1;
#pragma unroll
        for (int c = 0; c < D; c++) {
            const bool on = at[j] >= 0;
            x[j][c] = on ? a.x[c * nn + at[j]] : (TX)0;
            r[j][c] = on ? a.r[c * nn + at[j]] : (TX)0;
            d[j][c] = on ? a.dinv[c * nn + at[j]] : (TX)0;
        }
    }
    // the window of the first iteration: p, or after a replacement that
    // restarts the direction D^-1 r
    f.window([&](int64_t g) { return restart ? a.dinv[g] * a.r[g] : a.p[g]; },
             [&](int i, TX v) { win[i] = v; });
    f.setup(s0, win);
    __syncthreads();

    int state = 0;   // 1: limit, 2: gave up, 3: breakdown, 4: converged, 5: replace
    bool conv = false;
    double rr = 0., pq = 0., alpha = 0., beta = 0.;
    for (int it = 0;; it++) {
        if (it == a.iters || iters >= a.limit) {
            state = 1;
            break;
        }
        TX q[NR][D];
        f.products(win, q);
        double v1[1] = {0.};
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int c = 0; c < D; c++)
                if (at[j] >= 0) v1[0] += (double)win[f.own(j, c)] * (double)q[j][c];
        meet_publish<1>(m, v1, sh);
        double t1[1];
        if (!meet_collect<1>(m, t1, tot[0], &dead)) {
            state = 2;
            break;
        }
        pq = t1[0];
        if (!(pq > 0.) || !isfinite(pq)) {
            state = 3;
            break;
        }
        alpha = rho / pq;
        iters++;
        const TX al = (TX)alpha;
        double v2[2] = {0., 0.};
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int c = 0; c < D; c++)
                if (at[j] >= 0) {
                    const TX ri = r[j][c] - al * q[j][c];
                    r[j][c] = ri;
                    const TX zi = d[j][c] * ri;
                    st_agent(&a.z[c * nn + at[j]], zi);
                    v2[0] += (double)ri * (double)ri;
                    v2[1] += (double)ri * (double)zi;
                }
        stores_done();
        meet_publish<2>(m, v2, sh);
        // while the sums travel: x += alpha p
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int c = 0; c < D; c++)
                if (at[j] >= 0) x[j][c] = x[j][c] + al * win[f.own(j, c)];
        double t2[2];
        if (!meet_collect<2>(m, t2, tot[1], &dead)) {
            state = 2;
            break;
        }
        rr = t2[0];
        if (!isfinite(rr)) {
            state = 3;
            break;
        }
        conv = rr < thr;
        if (conv && !mixed) {
            state = 4;
            break;
        }
        const bool pause = mixed && !conv && rr < delta2 * rref;
        if (conv) {
            state = 5;
            break;
        }
        beta = t2[1] / rho;
        rho = t2[1];
        const TX be = (TX)beta;
        f.window([&](int64_t g) { return ld_agent(&a.z[g]); },
                 [&](int i, TX v) { win[i] = v + be * win[i]; });
        __syncthreads();
        if (pause) {
            state = 5;
            break;
        }
    }
    if (state == 2) {
        if (threadIdx.x == 0) sc->abort = 1;
        return;
    }
    // hand the iterate back; before a replacement x is folded into x64
#pragma unroll
    for (int j = 0; j < NR; j++)
#pragma unroll
        for (int c = 0; c < D; c++)
            if (at[j] >= 0) {
                const int64_t g = c * nn + at[j];
                if (mixed && state == 5) {
                    a.x64[g] += (double)x[j][c];
                    a.x[g] = (TX)0;
                } else {
                    a.x[g] = x[j][c];
                }
                a.r[g] = r[j][c];
                a.p[g] = win[f.own(j, c)];
            }
    if (seg == 0 && threadIdx.x == 0) {
        sc->iters = iters;
        sc->rho[0] = rho;
        sc->rho[1] = rho;
        sc->restart = 0;
        sc->pq = pq;
        sc->alpha = alpha;
        sc->beta = beta;
        if (state == 1 || state == 4 || state == 5) sc->rr = rr;
        if (state == 3) {
            sc->breakdown = 1;
            sc->done = 1;
        } else if (state == 4) {
            sc->stop = 1;
        } else if (state == 5) {
            sc->conv32 = conv ? 1 : 0;
            sc->rep_at = RES_REPLACE;
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
    static constexpr int NR = 1, D = 1;
    const int32_t* rp;
    const uint16_t* lcol;
    const TV* val;
    const int32_t* list;     // columns of this block's window
    int nw;                  // and their number
    int own0;                // window place of the block's first row
    int rows;                // rows of the block
    int64_t row0;
    TX* qs;                  // LDS: q of the block's rows
    static constexpr int UL = 4;
    int32_t lst[UL];         // this thread's first columns of the list
    TV rv[NP ? NP : 1][4];
    int rl[NP ? NP : 1][4];

    __device__ inline int own(int, int) const { return own0 + threadIdx.x; }

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

    __device__ inline void setup(int64_t, TX*)
    {
        if constexpr (NP > 0) {
            const int sub = threadIdx.x & (LPR - 1), team = threadIdx.x / LPR;
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

    __device__ inline void products(const TX* __restrict__ w, TX (&q)[1][1])
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
        q[0][0] = (int)threadIdx.x < rows ? qs[threadIdx.x] : (TX)0;
    }
};

// LDS: q of up to RT rows, then the window
template <int LPR, int NP, typename TV, typename TX>
__global__ __launch_bounds__(RT) void k_cg_csr(CgArgs<TX> a, const int32_t* __restrict__ rp,
                                               const uint16_t* __restrict__ lcol,
                                               const TV* __restrict__ val,
                                               const int32_t* __restrict__ list,
                                               const int32_t* __restrict__ woff,
                                               const int32_t* __restrict__ own0)
{
    extern __shared__ unsigned char lds[];
    const int seg = seg_of_block(blockIdx.x, a.B);
    CsrForm<LPR, NP, TV, TX> f;
    f.rp = rp;
    f.lcol = lcol;
    f.val = val;
    f.list = list + woff[seg];
    f.nw = woff[seg + 1] - woff[seg];
    f.own0 = own0[seg];
    f.row0 = (int64_t)seg * a.R * 64;
    const int64_t left = a.n - f.row0;
    f.rows = (int)(left < 0 ? 0 : (left < (int64_t)a.R * 64 ? left : (int64_t)a.R * 64));
    f.qs = reinterpret_cast<TX*>(lds);
    f.columns();
    cg_resident(a, f, f.qs + RT);
}

// ---------------------------------------------------------------------------
// Windows of the CSR rows: a bitmap of the columns of the block's rows in
// LDS; a column's place is the number of set bits below it.
constexpr int WIN_MAXN = 256 * 1024;   // columns a bitmap and its counts hold in 64 KB of LDS

__device__ inline void win_bits(int64_t n, int64_t row0, int rows, const int32_t* __restrict__ rp,
                                const int32_t* __restrict__ col, uint32_t* bits, int words)
{
    for (int i = threadIdx.x; i < words; i += RT) bits[i] = 0u;
    __syncthreads();
    if (rows > 0) {
        for (int i = threadIdx.x; i < rows; i += RT) {
            const int64_t c = row0 + i;
            atomicOr(&bits[c >> 5], 1u << (c & 31));
        }
        const int32_t k1 = rp[row0 + rows];
        for (int32_t k = rp[row0] + threadIdx.x; k < k1; k += RT) {
            const int32_t c = col[k];
            atomicOr(&bits[c >> 5], 1u << (c & 31));
        }
    }
    __syncthreads();
}

// per segment: columns of its window; the longest row of all
__global__ __launch_bounds__(RT) void k_win_count(int64_t n, int R, const int32_t* __restrict__ rp,
                                                  const int32_t* __restrict__ col,
                                                  int32_t* __restrict__ wlen,
                                                  int32_t* __restrict__ maxlen)
{
    extern __shared__ uint32_t bits[];
    __shared__ int cnt, longest;
    if (threadIdx.x == 0) cnt = longest = 0;
    const int words = (int)((n + 31) / 32);
    const int64_t row0 = (int64_t)blockIdx.x * R * 64;
    const int64_t left = n - row0;
    const int rows = (int)(left < 0 ? 0 : (left < (int64_t)R * 64 ? left : (int64_t)R * 64));
    win_bits(n, row0, rows, rp, col, bits, words);
    int s = 0, len = 0;
    for (int i = threadIdx.x; i < words; i += RT) s += __popc(bits[i]);
    for (int i = threadIdx.x; i < rows; i += RT) len = max(len, rp[row0 + i + 1] - rp[row0 + i]);
    atomicAdd(&cnt, s);
    atomicMax(&longest, len);
    __syncthreads();
    if (threadIdx.x == 0) {
        wlen[blockIdx.x] = cnt;
        atomicMax(maxlen, longest);
    }
}

__global__ __launch_bounds__(RT) void k_win_fill(int64_t n, int R, const int32_t* __restrict__ rp,
                                                 const int32_t* __restrict__ col,
                                                 const int32_t* __restrict__ woff,
                                                 int32_t* __restrict__ list,
                                                 uint16_t* __restrict__ lcol,
                                                 int32_t* __restrict__ own0)
{
    extern __shared__ uint32_t bits[];
    __shared__ int wsum[RW];
    const int words = (int)((n + 31) / 32);
    int32_t* below = reinterpret_cast<int32_t*>(bits + words);   // set bits before each word
    const int64_t row0 = (int64_t)blockIdx.x * R * 64;
    const int64_t left = n - row0;
    const int rows = (int)(left < 0 ? 0 : (left < (int64_t)R * 64 ? left : (int64_t)R * 64));
    win_bits(n, row0, rows, rp, col, bits, words);
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
    for (int w = 0; w < (int)(threadIdx.x >> 6); w++) run += wsum[w];
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
    if (rows > 0) {
        const int32_t k1 = rp[row0 + rows];
        for (int32_t k = rp[row0] + threadIdx.x; k < k1; k += RT) lcol[k] = (uint16_t)place(col[k]);
    }
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

template <class K, typename... A>
int launch_ordered(Ctx* c, K kernel, int blocks, size_t lds, A... args)
{
    // one block per compute unit: more than half of its LDS
    lds = std::max<size_t>(lds, LDS_MAX / 2 + 1024);
    INS_HIP_CHECK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    Order& o = g_order[c->device];
    std::lock_guard<std::mutex> lock(o.mu);
    if (!o.last) INS_HIP_CHECK(c, hipEventCreateWithFlags(&o.last, hipEventDisableTiming));
    else if (o.stream != c->stream) INS_HIP_CHECK(c, hipStreamWaitEvent(c->stream, o.last, 0));
    kernel<<<blocks, RT, lds, c->stream>>>(args...);
    INS_HIP_CHECK(c, hipGetLastError());
    INS_HIP_CHECK(c, hipEventRecord(o.last, c->stream));
    o.stream = c->stream;
    return INS_OK;
}

int ensure_words(Ctx* c, int iters)
{
    Resident& S = c->res;
    if (!S.words.p || S.epoch > UINT32_MAX - 4u * (uint32_t)iters - 16u) {
        INS_TRY(ensure(c, S.words, MEET_WORDS));
        INS_HIP_CHECK(c, hipMemsetAsync(S.words.p, 0, MEET_WORDS * sizeof(uint64_t), c->stream));
        S.epoch = 1;
    }
    return INS_OK;
}

template <typename TX>
CgArgs<TX> cg_args(Ctx* c, const Seg& g, int64_t n, TX* x, TX* r, TX* p, TX* z, const TX* dinv,
                   int iters, int limit)
{
    // bound of a wait: a poll takes about a microsecond
    static const int polls = env_res("INS_RESIDENT_POLLS", 500000);
    Resident& S = c->res;
    CgArgs<TX> a{n, g.B, g.R, x, r, p, z, dinv, c->sx64, c->scal.p, S.words.p, S.epoch, polls,
                 iters, limit};
    S.epoch += 2u * (uint32_t)iters + 2u;
    return a;
}

}  // namespace

int resident_blocks(int n_cu)
{
    static const int on = env_res("INS_RESIDENT", 1);
    if (!on) return 0;
    return n_cu < NXCD ? 0 : std::min(RBMAX, n_cu / NXCD * NXCD);
}

// Segments of a CSR solve.  R is what four register passes hold, 4 RT / LPR
// rows, while that makes no more than the 64 blocks whose sums meet in one
// stage; beyond them the sums cost the same up to 256 blocks, so all are
// used (125,000 rows numbered at random, whose windows are gathers of one
// lane per cycle: C 4.9 us with 123 blocks).  At most RT rows per block, and
// then streamed; larger systems keep the three kernels.
Seg csr_segments(int64_t n, int lpr, int n_cu)
{
    const int bmax = resident_blocks(n_cu);
    const int64_t nsl = (n + 63) / 64;
    Seg g;
    if (bmax == 0 || n > WIN_MAXN || nsl > (int64_t)bmax * RW) return g;
    int64_t R = std::max(1, 64 / lpr);
    if (nsl > 64 * R) R = (nsl + bmax - 1) / bmax;
    int64_t B = (nsl + R - 1) / R;
    if (B >= NXCD) B = std::min<int64_t>(bmax, (B + NXCD - 1) / NXCD * NXCD);
    g.R = (int)R;
    g.B = (int)B;
    return g;
}

// Windows of the current CSR pattern, once per pattern; S.csr_ok says
// whether they fit the LDS beside the block's q
int csr_windows(Ctx* c, const Seg& g, int vec_bytes)
{
    Resident& S = c->res;
    if (S.csr_gen == c->pattern_gen && S.csr_seg_B == g.B && S.csr_seg_R == g.R) {
        S.csr_ok = (size_t)(RT + S.csr_wmax) * vec_bytes <= (size_t)LDS_MAX - 4096;
        return INS_OK;
    }
    const int64_t n = c->n_active;
    const size_t words = (size_t)((n + 31) / 32);
    INS_TRY(ensure(c, S.wlen, RBMAX + 1));
    INS_HIP_CHECK(c, hipMemsetAsync(S.wlen.p + RBMAX, 0, sizeof(int32_t), c->stream));
    k_win_count<<<g.B, RT, words * 4, c->stream>>>(n, g.R, c->row_ptr.p, c->col.p, S.wlen.p,
                                                   S.wlen.p + RBMAX);
    INS_HIP_CHECK(c, hipGetLastError());
    int32_t len[RBMAX + 1], off[RBMAX + 1];
    INS_HIP_CHECK(c, hipMemcpyAsync(len, S.wlen.p, sizeof len, hipMemcpyDeviceToHost, c->stream));
    INS_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    off[0] = 0;
    S.csr_wmax = 0;
    for (int b = 0; b < g.B; b++) {
        off[b + 1] = off[b] + len[b];
        S.csr_wmax = std::max(S.csr_wmax, len[b]);
    }
    S.csr_maxlen = len[RBMAX];
    S.csr_gen = c->pattern_gen;
    S.csr_seg_B = g.B;
    S.csr_seg_R = g.R;
    S.csr_ok = (size_t)(RT + S.csr_wmax) * vec_bytes <= (size_t)LDS_MAX - 4096;
    if ((size_t)S.csr_wmax > 65536) return INS_OK;   // places are 16 bits
    INS_TRY(ensure(c, S.woff, RBMAX + 1));
    INS_TRY(ensure(c, S.own0, RBMAX));
    INS_TRY(ensure(c, S.wlist, (size_t)off[g.B] + 1));
    INS_TRY(ensure(c, S.lcol, (size_t)c->nnz + 1));
    INS_HIP_CHECK(c, hipMemcpyAsync(S.woff.p, off, (g.B + 1) * sizeof(int32_t),
                                    hipMemcpyHostToDevice, c->stream));
    INS_HIP_CHECK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(&k_win_fill),
                                         hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)(words * 8)));
    k_win_fill<<<g.B, RT, words * 8, c->stream>>>(n, g.R, c->row_ptr.p, c->col.p, S.woff.p,
                                                  S.wlist.p, S.lcol.p, S.own0.p);
    INS_HIP_CHECK(c, hipGetLastError());
    INS_HIP_CHECK(c, hipStreamSynchronize(c->stream));   // off is on this stack
    return INS_OK;
}

namespace {
template <int LPR, typename TV, typename TX>
int launch_csr_lpr(Ctx* c, const Seg& g, const CgArgs<TX>& a, const TV* val)
{
    const Resident& S = c->res;
    const size_t lds = (size_t)(RT + S.csr_wmax) * sizeof(TX);
    const int passes = (g.R * 64 * LPR + RT - 1) / RT;
    const bool regs = S.csr_maxlen <= 4 * LPR;
#define INS_CG_CSR(NP)                                                                       \
    return launch_ordered(c, k_cg_csr<LPR, NP, TV, TX>, g.B, lds, a, (const int32_t*)c->row_ptr.p, \
                          (const uint16_t*)S.lcol.p, val, (const int32_t*)S.wlist.p,          \
                          (const int32_t*)S.woff.p, (const int32_t*)S.own0.p)
    if (regs && passes <= 1) INS_CG_CSR(1);
    if (regs && passes <= 2) INS_CG_CSR(2);
    if (regs && passes <= 4) INS_CG_CSR(4);
    INS_CG_CSR(0);
#undef INS_CG_CSR
}
}  // namespace

// up to `iters` iterations of a CSR solve in one launch
template <typename T>
int resident_csr(Ctx* c, const Seg& g, int lpr, const T* val, T* x, T* r, T* p, T* z,
                 const T* dinv, int iters, int limit)
{
    INS_TRY(ensure_words(c, iters));
    const CgArgs<T> a = cg_args<T>(c, g, c->n_active, x, r, p, z, dinv, iters, limit);
    if (lpr == 32) return launch_csr_lpr<32>(c, g, a, val);
    if (lpr == 16) return launch_csr_lpr<16>(c, g, a, val);
    if (lpr == 8) return launch_csr_lpr<8>(c, g, a, val);
    return launch_csr_lpr<4>(c, g, a, val);
}
template int resident_csr<double>(Ctx*, const Seg&, int, const double*, double*, double*, double*,
                                  double*, const double*, int, int);
template int resident_csr<float>(Ctx*, const Seg&, int, const float*, float*, float*, float*,
                                 float*, const float*, int, int);

}  // namespace ins
