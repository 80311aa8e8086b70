// Resident conjugate gradients: one launch holds a solve on the chip for many
// iterations.  The rows are cut into segments of R slices (64 rows each), one
// segment per block, at most one block per compute unit.  A block keeps the
// part of p that its rows read (its window) in LDS; what the blocks exchange
// in an iteration are two sums and z = D^-1 r.
//
// The same segments, with the same sums, exist as three plain kernels per
// iteration (seg_*), for callers that cannot run the resident kernel; both
// give the same bits.
#pragma once

#include "cg_device.hpp"

namespace ins {

// Threads of a segment block: 8 waves of up to 256 registers.  (16 waves of 128
// hold as much, but left the compiler no room beside the matrix entries: it
// kept loop invariants in scratch, a microsecond per reload.)
constexpr int RT = 512;
constexpr int RW = RT / 64;       // its waves
constexpr int TASKS = 16;         // shares of a segment that the waves take in turn
constexpr int CSR_ROWS = 1024;    // rows of a CSR segment at most
constexpr int RBMAX = 256;        // most segments of a solve
constexpr int LDS_MAX = 160 * 1024;
// dynamic LDS of a launch at most, beside the kernels' own few KB.  A kernel's
// limit is set to this, never to a launch's own size, which another thread's
// (on another device) could lower before the launch.
constexpr int LDS_DYN = LDS_MAX - 4096;

// Decomposition of one solve into segments (B = 0: none): R slices of 64 rows
// per block, or, where cut is set, slices cut[b] .. cut[b + 1] - 1 (at most R)
struct Seg {
    int B = 0;   // blocks
    int R = 0;
    const int32_t* cut = nullptr;   // device
};

// the slices of one segment
struct Span {
    int64_t s0;
    int sl;
};
__device__ inline Span seg_span(const Seg& g, int seg)
{
    if (!g.cut) return Span{(int64_t)seg * g.R, g.R};
    const int a = g.cut[seg];
    return Span{a, g.cut[seg + 1] - a};
}

// Segment of a block: workgroups go to the XCDs round-robin, so that with B a
// multiple of 8 every XCD gets one contiguous eighth of the rows
__device__ inline int seg_of_block(int id, int B)
{
    return (B % NXCD) ? id : (id % NXCD) * (B / NXCD) + id / NXCD;
}

// The lane, unknown to the optimiser: what is computed from it stays where it
// is used (addresses of a form's setup otherwise move out of the loop around
// the replacements and take registers through the iterations)
__device__ inline int opaque_lane()
{
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    return lane;
}

// ---------------------------------------------------------------------------
// CSR rows: LPR lanes per row, 4 entries per lane in flight (the order of
// csr_row); p(k) gives the vector value of entry k
template <int LPR, typename TV, typename TX, class P>
__device__ inline TX csr_seg_round(int32_t k0, int32_t e, const TV* __restrict__ val, P p, TX s)
{
    for (; k0 < e; k0 += 4 * LPR) {
        TV vv[4];
        TX xx[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int32_t k = k0 + j * LPR;
            vv[j] = (k < e) ? val[k] : (TV)0;
            xx[j] = (k < e) ? p(k) : (TX)0;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) s += (TX)vv[j] * xx[j];
    }
    return s;
}
template <int LPR, typename TV, typename TX, class P>
__device__ inline TX csr_seg_row(int32_t k0, int32_t e, const TV* __restrict__ val, P p)
{
    return group_sum<LPR>(csr_seg_round<LPR, TV, TX>(k0, e, val, p, (TX)0));
}

// rows [0, rows) of a segment by THREADS threads, U of a team's rows in flight:
// f(i, sum) by the first lane of the team
template <int LPR, int THREADS, int U, typename TV, typename TX, class P, class F>
__device__ inline void csr_seg_rows(int rows, const int32_t* __restrict__ rp,
                                    const TV* __restrict__ val, P p, F f)
{
    constexpr int T = THREADS / LPR;
    const int sub = threadIdx.x & (LPR - 1);
    for (int i0 = threadIdx.x / LPR; i0 < rows; i0 += U * T) {
        int32_t k0[U], e[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + u * T;
            k0[u] = i < rows ? rp[i] + sub : 0;
            e[u] = i < rows ? rp[i + 1] : 0;
        }
        TV vv[U][4];
        TX xx[U][4];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int32_t k = k0[u] + j * LPR;
                vv[u][j] = (k < e[u]) ? val[k] : (TV)0;
                xx[u][j] = (k < e[u]) ? p(k) : (TX)0;
            }
#pragma unroll
        for (int u = 0; u < U; u++) {
            TX s = (TX)0;
#pragma unroll
            for (int j = 0; j < 4; j++) s += (TX)vv[u][j] * xx[u][j];
            s = group_sum<LPR>(csr_seg_round<LPR, TV, TX>(k0[u] + 4 * LPR, e[u], val, p, s));
            const int i = i0 + u * T;
            if (sub == 0 && i < rows) f(i, s);
        }
    }
}

// ---------------------------------------------------------------------------
// Symmetric slices (SymLayout): the 2 NU - 1 entries of a row, or blocks of a
// node, are numbered t = 0 the diagonal, 2k - 1 the one at offset u_k, 2k its
// mirror at -u_k.  Blocks are summed in that order.
//
// Scalar rows are summed in the order of the kernels on whole vectors
// (sym_row_v of solve.hip): SYM_SUM offsets at a time, first their own entries,
// then the mirrors.  With that, and with p = D^-1 r + beta p rounded as there
// (update_p_body), a mixed solve takes the same FP32 steps whichever kernels
// run it.  It matters: by rounding alone 16^3 diffusion solves end after about
// 103 iterations and 2e-10 off or, one in thirty, after about 91 and 1e-9 to
// 4e-9 off, both with |b - A x| below the tolerance.
constexpr int SYM_SUM = 8;

// place of a block's (i, j) entry in the upper triangle of the diagonal block
template <int D>
__device__ inline constexpr int sym_tri(int i, int j)
{
    return i <= j ? i * D - i * (i - 1) / 2 + (j - i) : j * D - j * (j - 1) / 2 + (i - j);
}

// entry at offset u_k of the row (slice, lane), and its mirror (edge: it may
// lie before row 0)
template <int NU, typename TV>
__device__ inline TV sym_seg_own(const TV* __restrict__ vals, int64_t slice, int lane, int k)
{
    return vals[slice * (64 * NU) + k * 64 + lane];
}
template <int NU, typename TV>
__device__ inline TV sym_seg_mirror(const TV* __restrict__ vals, int64_t slice, int lane, int k,
                                    int d, bool edge)
{
    constexpr int ld = 64 * NU;
    const int t = lane - d, o = (t >> 6) * ld + k * 64 + (t & 63);
    const TV* __restrict__ base = vals + slice * ld;
    if (!edge) return base[o];
    const bool in = (int)slice * 64 + t >= 0;
    const TV w = base[in ? o : lane];
    return in ? w : (TV)0;
}

// all entries of the row, in their order
template <int NU, typename TV>
__device__ inline void sym_seg_values(const TV* __restrict__ vals, int64_t slice, int lane,
                                      const int (&du)[NU], bool edge, TV (&v)[2 * NU - 1])
{
#pragma unroll
    for (int k = 0; k < NU; k++) {
        v[k ? 2 * k - 1 : 0] = sym_seg_own<NU, TV>(vals, slice, lane, k);
        if (k) v[2 * k] = sym_seg_mirror<NU, TV>(vals, slice, lane, k, du[k], edge);
    }
}

// Block t of the node (slice, lane), row-major as the node's row uses it
// (mirrors transposed); d: its offset u_k
template <int D, int NU, typename TV>
__device__ inline void bsym_seg_block(const TV* __restrict__ vals, int64_t slice, int lane, int t,
                                      int d, TV (&b)[D * D])
{
    constexpr int T = D * (D + 1) / 2, D2 = D * D;
    constexpr int64_t ld = 64 * (T + (NU - 1) * D2);
    if (t == 0) {
        const TV* __restrict__ own = vals + slice * ld + lane;
#pragma unroll
        for (int i = 0; i < D; i++)
#pragma unroll
            for (int j = 0; j < D; j++) b[i * D + j] = own[sym_tri<D>(i, j) * 64];
        return;
    }
    const int k = (t + 1) >> 1;
    if (t & 1) {
        const TV* __restrict__ own = vals + slice * ld + (T + (k - 1) * D2) * 64 + lane;
#pragma unroll
        for (int e = 0; e < D2; e++) b[e] = own[e * 64];
    } else {
        const int m = lane - d;
        const bool in = (int)slice * 64 + m >= 0;
        const int o = in ? (m >> 6) * (int)ld + (m & 63) : lane;
        const TV* __restrict__ q = vals + slice * ld + (T + (k - 1) * D2) * 64;
#pragma unroll
        for (int i = 0; i < D; i++)
#pragma unroll
            for (int j = 0; j < D; j++) {
                const TV w = q[o + (j * D + i) * 64];
                b[i * D + j] = in ? w : (TV)0;
            }
    }
}

template <int D, typename TV, typename TX>
__device__ inline void bsym_seg_add(const TV (&b)[D * D], const TX (&x)[D], TX (&out)[D])
{
#pragma unroll
    for (int i = 0; i < D; i++)
#pragma unroll
        for (int j = 0; j < D; j++) out[i] += (TX)b[i * D + j] * x[j];
}

// A node's blocks are shared out over `parts` tasks where a segment has few
// slices (the parts' sums are added in order; wave w takes tasks w and
// w + RW, ..): with one wave per slice most of the waves would have nothing to do
// and the others a chain of 27 dependent rounds of loads.  3 parts and more
// also hold their blocks on the chip (27 / 3 blocks of 9 FP32 values): those of
// TASKS tasks in registers, of the next few in LDS
__host__ __device__ inline constexpr int bsym_parts(int R)
{
    return R <= 2 ? 8 : (R <= 4 ? 4 : (R <= 7 ? 3 : (R <= 8 ? 2 : 1)));
}
constexpr int BSYM_TASKS = 21;   // at most
// blocks per part
__host__ __device__ inline constexpr int bsym_per(int nt, int parts)
{
    return (nt + parts - 1) / parts;
}

// entries of one task's run in a segment of full slices (whole groups of 4)
__device__ inline int sell_run(const SellView& S, int64_t s0, int64_t s1, int64_t n)
{
    const int64_t nsl = (n + 63) / 64;
    const int64_t e = (S.sptr[s1 < nsl ? s1 : nsl] - S.sptr[s0 < nsl ? s0 : nsl]) >> 6;
    return (int)((e + 4 * TASKS - 1) / (4 * TASKS)) * 4;
}

// The kernels on segments go by units: what one wave of the resident kernel's
// block owns, slices w, w + RW, .. of a segment, is a wave's work there too.  The
// U units of a segment that has any (fewer than RW with few slices) are packed into
// blocks without regard to segments; a wave leaves the sums over its unit, and a
// segment's sum is that of its units in order, as block_allsum adds the waves of the
// resident kernel: the same bits.  With U = RW a block is a segment (two units per
// wave) and leaves its sums itself, which spares the totals most of their loads.
constexpr int UT = 256;   // threads of a block
__host__ __device__ inline int seg_units(int R) { return R < RW ? R : RW; }
__host__ __device__ inline int unit_blocks(int B, int U)
{
    const int b = U == RW ? B : (B * U + UT / 64 - 1) / (UT / 64);
    return b < NXCD ? b : (b + NXCD - 1) / NXCD * NXCD;
}
// partials of a segment with U units
__host__ __device__ inline int unit_per(int U) { return U == RW ? 1 : U; }

struct SegUnit {
    Span s;
    int w;       // the wave of the resident kernel
};

// The calling wave's units in block b of the segments g: w, w + UT / 64, .. below
// end of segment seg (one call of a body: inlined, which two would not be)
struct UnitRange {
    int seg, w, end;
    bool whole;   // the block is a segment
};
__device__ inline UnitRange unit_range(const Seg& g, int U, Blk b)
{
    const int wave = wave_in_block(), id = seg_of_block(b.id, b.n);
    if (U >= RW) return UnitRange{id < g.B ? id : 0, wave, id < g.B ? RW : 0, true};
    const int u = id * (UT / 64) + wave;
    if (u >= g.B * U) return UnitRange{0, 0, 0, false};
    return UnitRange{u / U, u % U, u % U + 1, false};
}

// body(unit) for the units of block b
template <class Body>
__device__ inline void seg_unit_visit(const Seg& g, int U, Blk b, Body body)
{
    const UnitRange k = unit_range(g, U, b);
    const Span s = seg_span(g, k.seg);
#pragma unroll 1
    for (int w = k.w; w < k.end; w += UT / 64) body(SegUnit{s, w});
}

// body(unit, v): the unit's shares v of NV sums; leaves the sums' partials
template <int NV, class Body>
__device__ inline void seg_unit_sums(const Seg& g, int U, Blk b, double* part,
                                     const int (&slot)[NV], Body body)
{
    __shared__ double sh[NV][RW];
    const UnitRange k = unit_range(g, U, b);
    const Span s = seg_span(g, k.seg);
#pragma unroll 1
    for (int w = k.w; w < k.end; w += UT / 64) {
        double v[NV] = {};
        body(SegUnit{s, w}, v);
#pragma unroll
        for (int i = 0; i < NV; i++) {
            v[i] = wave_sum(v[i]);
            if ((threadIdx.x & 63) == 0) {
                if (k.whole) sh[i][w] = v[i];
                else part[slot[i] * MAXG + k.seg * U + w] = v[i];
            }
        }
    }
    if (!k.whole || k.end == 0) return;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; i++)
        if ((int)threadIdx.x == i) {
            double t = 0.;
#pragma unroll
            for (int w = 0; w < RW; w++) t += sh[i][w];
            part[slot[i] * MAXG + k.seg] = t;
        }
}

// this thread's share of the totals of B segments (totals_share), each of `per`
// partials
template <int NV>
__device__ inline void unit_totals_share(const double* part, int B, int per,
                                         const int (&slot)[NV], double (&t)[NV])
{
    if (per == 1) return totals_share<NV>(part, B, slot, t);
#pragma unroll
    for (int k = 0; k < NV; k++) t[k] = 0.;
    for (int i = threadIdx.x; i < B; i += blockDim.x) {
        double v[NV][RW];
#pragma unroll
        for (int k = 0; k < NV; k++)
#pragma unroll
            for (int w = 0; w < RW; w++)
                v[k][w] = w < per ? part[slot[k] * MAXG + i * per + w] : 0.;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            double s = 0.;
#pragma unroll
            for (int w = 0; w < RW; w++) s += v[k][w];
            t[k] += s;
        }
    }
}
// f(i) for every item of the unit, in the order of the resident kernel
// (component c of item a at c * n + a)
template <int D, class F>
__device__ inline void unit_items(const SegUnit& u, int64_t n, F f)
{
    const int lane = threadIdx.x & 63;
    for (int k = u.w; k < u.s.sl; k += RW) {
        const int64_t a = (u.s.s0 + k) * 64 + lane;
        if (a < n)
#pragma unroll
            for (int c = 0; c < D; c++) f(c * n + a);
    }
}

// forms of the SELL storage that have segments
enum SegForm { SEG_NONE = 0, SEG_SYM14, SEG_SYM5, SEG_BSYM3, SEG_BSYM2, SEG_SELL };
__host__ __device__ inline constexpr bool sym_form(int f) { return f == SEG_SYM14 || f == SEG_SYM5; }

// Products of the matrix with x on a segment of a SELL storage, the order of
// every sum as in the resident kernel's form F: f(place of the item, sum) for
// this thread's items; x(i): the vector.  The block's waves together, part: LDS
// for the node blocks' part sums; or, part null (UNIT), a wave its unit alone,
// wave: the resident kernel's
template <int F, typename TV, typename TX, bool UNIT = false, class X, class Fn>
__device__ inline void seg_products(const Span& sp, int64_t n_, const SellView& S,
                                    const int32_t* __restrict__ u, const TV* __restrict__ vals,
                                    X x, TX* part, int wave, Fn f)
{
    const int64_t s0 = sp.s0;
    const int sl = sp.sl, n = (int)n_;
    auto live = [&](int k) { return k < sl && (s0 + k) * 64 < n; };
    // (the lane is hidden from the optimiser once per slice: it would carry
    // a pointer per entry through the loop over the slices, in scratch)
    if constexpr (sym_form(F)) {
        constexpr int NU = F == SEG_SYM14 ? 14 : 5;
        int du[NU];
#pragma unroll
        for (int k = 0; k < NU; k++) du[k] = __builtin_amdgcn_readfirstlane(u[k]);
        const bool edge = s0 * 64 < du[NU - 1];
        for (int k = wave; live(k); k += RW) {
            const int lane = opaque_lane();
            const int row = (int)(s0 + k) * 64 + lane;
            TX s = (TX)0;
            // own entries and mirrors of SYM_SUM offsets in turn (both at once
            // take twice the registers of the resident kernel's loop)
#pragma unroll
            for (int t0 = 0; t0 < NU; t0 += SYM_SUM) {
                TV v[SYM_SUM];
                TX xx[SYM_SUM];
#pragma unroll
                for (int g = 0; g < SYM_SUM; g++)
                    if (t0 + g < NU) {
                        v[g] = sym_seg_own<NU, TV>(vals, s0 + k, lane, t0 + g);
                        xx[g] = x(min(row + du[t0 + g], n - 1));
                    }
#pragma unroll
                for (int g = 0; g < SYM_SUM; g++)
                    if (t0 + g < NU) s += (TX)v[g] * xx[g];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int g = 0; g < SYM_SUM; g++)
                    if (t0 + g > 0 && t0 + g < NU) {
                        const int d = du[t0 + g];
                        v[g] = sym_seg_mirror<NU, TV>(vals, s0 + k, lane, t0 + g, d, edge);
                        xx[g] = x(min(max(row - d, 0), n - 1));
                    }
#pragma unroll
                for (int g = 0; g < SYM_SUM; g++)
                    if (t0 + g > 0 && t0 + g < NU) s += (TX)v[g] * xx[g];
                __builtin_amdgcn_sched_barrier(0);
            }
            if (row < n) f(row, s);
        }
    } else if constexpr (F == SEG_BSYM3 || F == SEG_BSYM2) {
        constexpr int D = F == SEG_BSYM3 ? 3 : 2, NU = F == SEG_BSYM3 ? 14 : 5, NT = 2 * NU - 1;
        const int parts = bsym_parts(sl), per = bsym_per(NT, parts);
        auto sum = [&](int k, int t0, TX(&out)[D]) {
            const int lane = opaque_lane();
            const int a = (int)(s0 + k) * 64 + lane;
#pragma unroll
            for (int c = 0; c < D; c++) out[c] = (TX)0;
            constexpr int G = 2;
#pragma unroll 1
            for (int t = t0; t < t0 + per && t < NT; t += G) {
                TV b[G][D * D];
                TX xx[G][D];
#pragma unroll
                for (int g = 0; g < G; g++)
                    if (t + g < t0 + per && t + g < NT) {
                        const int d = u[(t + g + 1) >> 1];
                        bsym_seg_block<D, NU, TV>(vals, s0 + k, lane, t + g, d, b[g]);
                        const int i = min(max((t + g) & 1 ? a + d : a - d, 0), n - 1);
#pragma unroll
                        for (int c = 0; c < D; c++) xx[g][c] = x(c * n + i);
                    }
#pragma unroll
                for (int g = 0; g < G; g++)
                    if (t + g < t0 + per && t + g < NT) bsym_seg_add<D, TV, TX>(b[g], xx[g], out);
            }
        };
        if (UNIT || parts == 1) {
            for (int k = wave; live(k); k += RW) {
                TX out[D];
                sum(k, 0, out);
                for (int pt = 1; pt < parts; pt++) {
                    TX o[D];
                    sum(k, pt * per, o);
#pragma unroll
                    for (int c = 0; c < D; c++) out[c] += o[c];
                }
                const int a = (int)(s0 + k) * 64 + (int)(threadIdx.x & 63);
                if (a < n)
#pragma unroll
                    for (int c = 0; c < D; c++) f(c * n + a, out[c]);
            }
        } else {
            const int lane = threadIdx.x & 63;
            for (int t = wave; t < parts * sl; t += RW) {
                const int k = t / parts, pt = t % parts;
                if (live(k)) {
                    TX out[D];
                    sum(k, pt * per, out);
#pragma unroll
                    for (int c = 0; c < D; c++) part[(t * D + c) * 64 + lane] = out[c];
                }
            }
            __syncthreads();
            const int a = (int)(s0 + wave) * 64 + lane;
            if (live(wave) && a < n)
#pragma unroll
                for (int c = 0; c < D; c++) {
                    TX s = (TX)0;
                    for (int i = 0; i < parts; i++) s += part[((wave * parts + i) * D + c) * 64 + lane];
                    f(c * n + a, s);
                }
        }
    } else {
        // full slices: the segment's entries (lists padded to 4) in TASKS
        // equal runs of whole groups of 4, as the waves of the resident kernel
        // take them; a row's sum is that of its runs' sums, in order
        const int run = sell_run(S, s0, s0 + sl, n);
        const int64_t e0 = S.sptr[s0] >> 6;
        for (int k = wave; live(k); k += RW) {
            const int lane = opaque_lane();
            const int row = (int)(s0 + k) * 64 + lane;
            const TV* __restrict__ v0 = vals + S.sptr[s0 + k];
            const int32_t* __restrict__ d = S.pdel + S.pptr[S.spat[s0 + k]];
            const int len = S.plen[S.spat[s0 + k]];
            const int first = (int)((S.sptr[s0 + k] >> 6) - e0);
            TX s = (TX)0, r = (TX)0;
            constexpr int G = 2;
            for (int e = 0; e < len; e += 4 * G) {
                TV v[G][4];
                TX xx[G][4];
#pragma unroll
                for (int g = 0; g < G; g++)
                    if (e + 4 * g < len) {
                        load4<TV>(v0 + (e + 4 * g) * 64 + lane * 4, v[g]);
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            xx[g][i] = e + 4 * g + i < len
                                           ? x(min(max(row + d[e + 4 * g + i], 0), n - 1))
                                           : (TX)0;
                    }
#pragma unroll
                for (int g = 0; g < G; g++)
                    if (e + 4 * g < len) {
                        if (e + 4 * g > 0 && (first + e + 4 * g) % run == 0) {
                            s += r;
                            r = (TX)0;
                        }
#pragma unroll
                        for (int i = 0; i < 4; i++) r += (TX)v[g][i] * xx[g][i];
                    }
            }
            s += r;
            if (row < n) f(row, s);
        }
    }
}

// what the residual replacement of a mixed solve works on: the FP64 values of
// the storage (null: the FP32 ones, after an FP32 assembly)
struct ResRep {
    const double* v64 = nullptr;
    const float* v32 = nullptr;
    const double* b = nullptr;
    double* x64 = nullptr;
    double ratio = 0.;   // restarts the direction (INS_RESTART_RATIO)
};

// What every form of the resident kernel works on
template <typename TX>
struct CgArgs {
    int64_t n;          // items per component (rows, or nodes of a vector problem)
    Seg g;
    TX* x;
    TX* r;
    TX* p;
    TX* z;              // exchanged
    const TX* dinv;
    ResRep rep;         // mixed
    Scal* sc;
    uint64_t* words;    // device-wide sums
    uint32_t epoch;     // of the launch's first sum (resident_words)
    int polls;          // bound of a wait
    int limit;          // iterations of the solve at most
};

// The common window of a segment of symmetric slices (see resident.hip)
struct RelWin {
    const int4* piece;      // x: first column - row0, y: place, z: length
    int npiece;
    const int32_t* sh;      // shift of every entry t
    const int32_t* u;       // offsets
};

// One request of a resident batch: its blocks are first .. first + a.g.B - 1
struct CgEntry {
    CgArgs<float> a;
    int first;
    int variant;
    const float* vals;
    RelWin W;
    SellView S;
    const int32_t *base, *list, *woff, *own0;
};

constexpr int CG_MAX = 64;   // requests of a batch at most
// first epochs of the requests of one launch
struct CgEpochs {
    uint32_t e[CG_MAX] = {};
};

// one resident launch of a step: entries cg[first] .. of the table
struct CgGroup {
    int first = 0, n = 0, blocks = 0;
    size_t lds = 0;
};

// launchers (resident.hip)
int resident_blocks(int n_cu);
int resident_words(Ctx* c, hipStream_t st, int iters, uint32_t* first);
double restart_ratio();   // solve.hip
Seg csr_segments(int64_t n, int64_t nnz, int lpr, int n_cu, bool mixed);
int csr_windows(Ctx* c, const Seg& g, int lpr, int vec_bytes, bool* fits);
template <typename T>
int resident_csr(Ctx* c, const Seg& g, int lpr, const T* val, T* x, T* r, T* p, T* z,
                 const T* dinv, const ResRep& rep, int iters, int limit);

// a mixed SELL solve as an entry of a batch, and the LDS it needs
int resident_entry(Ctx* c, const Seg& g, Scal* sc, CgEntry* e, size_t* lds);
int resident_batch(int device, hipStream_t st, const CgEntry* tab, const std::vector<CgGroup>& groups,
                   int iters, const uint32_t* first);
SegForm sell_form(const Ctx* c);
int sell_segments(Ctx* c, bool mixed, Seg* out);
int sell_windows(Ctx* c, const Seg& g, int vec_bytes, bool* fits);
template <typename T>
int resident_sell(Ctx* c, const Seg& g, T* x, T* r, T* p, T* z, const T* dinv,
                  const ResRep& rep, int iters, int limit);

}  // namespace ins
