// Batched uneven 2D Shockley problems, all instances advancing together: every step of the
// Picard loop and of its multigrid-preconditioned CG is one launch over the blocks of all
// unfinished instances, with the CG scalars, stopping decisions and loop errors of each
// instance kept on the device.  The arithmetic per instance is that of k_batch_shockley2d
// (batch_kernels.hpp), which runs a whole instance in one workgroup and remains for the line
// preconditioner and for the meshes that steps_build leaves out: there every pass of an instance
// is a chain of latencies on one CU (a sweep of its coarsest level, 3 columns, used 3 threads for
// hundreds of dependent rows), and a batch took as long as its slowest instances.  Here the
// lines are solved by segments (part_solve), the passes of all instances share the chip, and
// the levels that fit one block's LDS are done in one kernel (k_bs_tail).
// 24 instances of 20-120 x 40-200 nodes, 6 loops: 130 -> 45 ms (one iteration is 11 launches,
// 190 us, 84 of them the tail).  96 of 50-400 x 100-800, 3 loops: 585 -> 138 ms (23 launches, 1.8 ms
// an iteration while all of them iterate, 9.7e6 nodes on the instance grids; 1.14 ms on average).
#pragma once
#include "batch_kernels.hpp"

namespace pf {

constexpr int BS_M = 8;       // planes per line segment
constexpr int BS_T = 512;     // threads of a line-sweep block
constexpr int BS_TAIL = 512;  // threads of a tail block (256 registers, 20 more spilled; with 1024 threads and 128
                              // registers most spill: 95 instead of 49 ms, 24 instances)

// One level of one instance (level 0: the instance grid); offsets into the pools of its kind.
struct BsLevel {
    int n0, n1, P, CB;        // nodes per axis, segments per line, columns per sweep block
    long long node, elem, mask, schur, seg;
    int h0, cx, mx, pad;      // widths; tables of the step to the next coarser level
};

// One block of a launch: which instance and level, its index among their blocks.
struct BsBlock {
    int inst, level, local, nblk;
};

struct BsPool {
    double *b, *x, *r, *la, *lw, *lc, *kh, *kv;
    double *ea, *eb;             // element coefficients (k_bs_coarsen)
    const double *h0, *rm;
    const uint64_t* mask;
    const unsigned char* fixed;  // Dirichlet nodes of each line segment, [segment][column], bit u: plane u
};

// CG state of an instance within one Picard loop (counter: block tickets of its reductions).
struct BsState {
    double rz, rz_prev, alpha, rr, stop2, rr_run, bb, bwd;
    int it, it_run, run, cst;
    int cg;       // 1: iterating
    int pending;  // 1: a run was started and its true residual is not yet taken
    int fin;      // 1: the Picard loop has ended
    int loops;
    unsigned counter[4];
};

struct BsArgs {
    const BatchInst* inst;
    const BsLevel* lev;    // [instance's first level + l]
    const int* lev0;       // first level per instance
    const int* tail;       // first level of k_bs_tail per instance (nlev + 1: none)
    const long long* part; // reduction partials per instance
    BsPool pool[2];        // level 0, coarse levels
    const double* h1;
    const int *cx, *mx;
    const double* wx;
    double *X, *PA, *PB, *cur, *schur, *partials;
    BsState* st;
    BatchStats* stats;
    int* count;            // instances [0] iterating, [1] finished
    int coarse_sweeps, maxit, maxloops, stable, rows;
    double omega, rtol, maxerr;
};

// Fused operand of bs_march
struct MarchP {
    bool on = false;
    double beta = 0.;
    const double* pin = nullptr;
};

// Sums NV values over an instance's blocks of this launch (the last MAXV of them are maxima);
// true in thread 0 of the block that ends them.
template <int NV, int MAXV>
__device__ bool bs_reduce(double (&v)[NV], double* __restrict__ partials, unsigned* counter, unsigned nblk, unsigned bid,
                          double (&tot)[NV]) {
    __shared__ double red[NV][16];
    __shared__ bool last;
    const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wid = tid >> 6, nw = (nthr + 63) >> 6;
    auto wred = [&](int a, double s) { return a < NV - MAXV ? wave_sum(s) : wave_max(s); };
    auto join = [&](int a, double p, double s) { return a < NV - MAXV ? p + s : fmax(p, s); };
#pragma unroll
    for (int a = 0; a < NV; ++a) {
        const double s = wred(a, v[a]);
        if (lane == 0) red[a][wid] = s;
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int a = 0; a < NV; ++a) {
            double s = red[a][0];
            for (int w = 1; w < nw; ++w) s = join(a, s, red[a][w]);
            publish_partial(partials + (size_t)a * nblk + bid, s);
        }
        last = take_ticket(counter) == nblk - 1;
    }
    __syncthreads();
    if (!last) return false;
#pragma unroll
    for (int a = 0; a < NV; ++a) {
        double s = a < NV - MAXV ? 0. : -__builtin_huge_val();
        for (unsigned b = tid; b < nblk; b += nthr) s = join(a, s, read_partial(partials + (size_t)a * nblk + b));
        s = wred(a, s);
        __syncthreads();
        if (lane == 0) red[a][wid] = s;
        __syncthreads();
        if (tid == 0) {
            double t = red[a][0];
            for (int w = 1; w < nw; ++w) t = join(a, t, red[a][w]);
            tot[a] = t;
        }
    }
    if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return tid == 0;
}

__device__ __forceinline__ LView bs_view(const BsArgs& A, const BatchInst& I, const BsLevel& L, int l) {
    const BsPool& P = A.pool[l > 0];
    return LView{L.n0, L.n1, I.cyl, P.h0 + L.h0, A.h1 + I.h1_off, P.rm + L.h0, P.kh + L.elem, P.kv + L.elem,
                 P.mask, L.mask, P.la + L.node, P.lw + L.node, P.lc + L.node};
}

// Rows k0 .. k1 of one column of A x, marching along axis 1 in the sum / difference basis of
// k_apply2d with the element coefficients ea = kx' / 12, eb = ky' / 12 (a layer of two elements
// costs ~25 operations and no division; a node needs three values of x and four coefficients).
// Four rows at a time, their loads issued together.  out(row, own value, (A x)_row, fixed).
// FUSE: the operand is z + beta p_old, formed where it is read (P.on false: z).
template <bool FUSE, typename OUT>
__device__ __forceinline__ void bs_march(const BsLevel& L, const BsPool& P, int i, int k0, int k1,
                                         const double* __restrict__ x, const MarchP& F, OUT&& out) {
    constexpr int U = 4;
    const int n0 = L.n0, n1 = L.n1;
    const int il = max(i - 1, 0), ir = min(i + 1, n0 - 1), eL = max(i - 1, 0), eR = min(i, n0 - 2);
    const double fL = i > 0 ? 1. : 0., fR = i < n0 - 1 ? 1. : 0.;
    const double *ea = P.ea + L.elem, *eb = P.eb + L.elem;
    auto row = [&](int k, double (&v)[3]) {
        const long long o = (long long)min(max(k, 0), n1 - 1) * n0;
        v[0] = x[o + il];
        v[1] = x[o + i];
        v[2] = x[o + ir];
        if (FUSE && F.on) {
            v[0] += F.beta * F.pin[o + il];
            v[1] += F.beta * F.pin[o + i];
            v[2] += F.beta * F.pin[o + ir];
        }
    };
    auto coef = [&](int e, double (&c)[4]) {  // layer e, between rows e and e + 1
        const long long o = (long long)min(max(e, 0), n1 - 2) * (n0 - 1);
        const double f = e >= 0 && e < n1 - 1 ? 1. : 0.;
        c[0] = ea[o + eL] * (fL * f);
        c[1] = eb[o + eL] * (fL * f);
        c[2] = ea[o + eR] * (fR * f);
        c[3] = eb[o + eR] * (fR * f);
    };
    // values a = (left sum, left difference, right sum, right difference) of a row
    auto tf = [](const double (&v)[3], double (&t)[4]) {
        t[0] = v[0] + v[1];
        t[1] = v[1] - v[0];
        t[2] = v[1] + v[2];
        t[3] = v[1] - v[2];
    };
    auto layer = [](const double (&t)[4], const double (&p)[4], const double (&c)[4], double& S, double& D) {
        S = (t[1] + p[1]) * (3. * c[0]) + (t[3] + p[3]) * (3. * c[2]);
        D = (t[0] - p[0]) * (3. * c[1]) + (t[1] - p[1]) * (c[0] + c[1]) + (t[2] - p[2]) * (3. * c[3]) +
            (t[3] - p[3]) * (c[2] + c[3]);
    };
    double v[3], c[4], p[4], t[4], S, D, own, acc;
    row(k0 - 1, v);
    tf(v, p);
    row(k0, v);
    coef(k0 - 1, c);
    tf(v, t);
    layer(t, p, c, S, D);
    own = v[1];
    acc = S + D;  // the layer below row k0
    for (int kb = k0; kb < k1; kb += U) {
        double vr[U][3], cr[U][4];
        bool fx[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            row(kb + u + 1, vr[u]);
            coef(kb + u, cr[u]);
            fx[u] = dbit(P.mask, L.mask + (long long)min(kb + u, n1 - 1) * n0 + i);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int q = 0; q < 4; ++q) p[q] = t[q];
            tf(vr[u], t);
            layer(t, p, cr[u], S, D);
            if (kb + u < k1) out(kb + u, own, acc + (S - D), fx[u]);
            own = vr[u][1];
            acc = S + D;
        }
    }
}

// Operator kernels: an item is one column and A.rows rows, 256 items per block.
//   k_bs_apply    p = z + beta p_old, x += alpha_prev p_old, q = A p, (p, q) -> alpha
//   k_bs_resid    b - A x of a level's first sweep (x in r, the residual to x)
//   k_bs_true     PHASE 0: residual of the start field -> bb; 1: compensated true residual at
//                 the start of a loop -> its stopping level; 2: after a run -> restart or end
//                 (march_rows)
// HBM- (or, on small batches, latency-) bound: 64, 40 and 32 bytes per node; for 9.7e6 nodes
// k_bs_apply takes 164 us (760 MB moved, 4.6 TB/s), k_bs_resid 102 us (446 MB, 4.4 TB/s),
// k_bs_true 165 us (its double-double products); 10, 5 and 13 us for 24 small instances.
// Directions are zero at Dirichlet nodes (residuals are), so the elimination only clears the
// rows there.
__global__ __launch_bounds__(256) void k_bs_apply(BsArgs A, const BsBlock* __restrict__ map) {
    const BsBlock B = map[blockIdx.x];
    BsState& S = A.st[B.inst];
    if (!S.cg) return;
    const BsLevel L = A.lev[A.lev0[B.inst]];
    const bool first = S.it_run == 0;
    double* pa = A.PA + L.node;
    double* pb = A.PB + L.node;
    MarchP P;
    P.on = !first;
    P.beta = first ? 0. : S.rz / S.rz_prev;
    const double alpha = S.alpha;
    const double* __restrict__ pin = (S.it_run & 1) ? pb : pa;
    double* __restrict__ pout = (S.it_run & 1) ? pa : pb;
    P.pin = pin;
    double* __restrict__ xs = A.X + L.node;
    double* __restrict__ q = A.pool[0].r + L.node;
    const int G = (L.n1 + A.rows - 1) / A.rows, w = B.local * 256 + (int)threadIdx.x;
    double acc = 0.;
    if (w < G * L.n0) {
        const int g = w / L.n0, i = w - g * L.n0, k0 = g * A.rows;
        bs_march<true>(L, A.pool[0], i, k0, min(L.n1, k0 + A.rows), A.pool[0].x + L.node, P,
                       [&](int k, double own, double s, bool fixed) {
                           const long long node = (long long)k * L.n0 + i;
                           pout[node] = own;
                           if (!first) xs[node] += alpha * pin[node];
                           const double o = fixed ? own : s;
                           q[node] = o;
                           acc += own * o;
                       });
    }
    double v[1] = {acc}, tot[1];
    if (bs_reduce<1, 0>(v, A.partials + A.part[B.inst], &S.counter[0], B.nblk, B.local, tot)) {
        if (tot[0] > 0.) {
            S.alpha = S.rz / tot[0];
        } else {
            S.alpha = 0.;
            S.cst = -6;
            S.cg = 0;
        }
    }
}

__global__ __launch_bounds__(256) void k_bs_resid(BsArgs A, const BsBlock* __restrict__ map) {
    const BsBlock B = map[blockIdx.x];
    if (!A.st[B.inst].cg) return;
    const BsLevel L = A.lev[A.lev0[B.inst] + B.level];
    const BsPool& P = A.pool[B.level > 0];
    const int G = (L.n1 + A.rows - 1) / A.rows, w = B.local * 256 + (int)threadIdx.x;
    if (w >= G * L.n0) return;
    const int g = w / L.n0, i = w - g * L.n0, k0 = g * A.rows;
    const double* __restrict__ b = P.b + L.node;
    double* __restrict__ r = P.x + L.node;
    bs_march<false>(L, P, i, k0, min(L.n1, k0 + A.rows), P.r + L.node, MarchP(),
                    [&](int k, double, double s, bool fixed) {
                        const long long node = (long long)k * L.n0 + i;
                        r[node] = fixed ? 0. : b[node] - s;
                    });
}

template <int PHASE>
__global__ __launch_bounds__(256) void k_bs_true(BsArgs A, const BsBlock* __restrict__ map) {
    const BsBlock B = map[blockIdx.x];
    BsState& S = A.st[B.inst];
    if (S.fin || (PHASE == 0 && S.loops > 0) || (PHASE == 2 && !S.pending)) return;
    if (PHASE == 2 && S.cst != 0) {  // CG ended without its tolerance: the loop keeps what it has
        if (B.local == 0 && threadIdx.x == 0) S.pending = 0;
        return;
    }
    const BatchInst I = A.inst[B.inst];
    const BsLevel L = A.lev[A.lev0[B.inst]];
    const LView V = bs_view(A, I, L, 0);
    const int G = (L.n1 + A.rows - 1) / A.rows, w = B.local * 256 + (int)threadIdx.x;
    double acc = 0., bw = 0.;
    if (w < G * L.n0) {
        const int g = w / L.n0, i = w - g * L.n0, k0 = g * A.rows;
        acc = march_rows<PHASE == 0 ? 1 : 2>(V, i, k0, min(L.n1, k0 + A.rows), A.X + L.node, nullptr,
                                             A.pool[0].b + L.node, bw);
    }
    double v[2] = {acc, bw}, tot[2];
    if (!bs_reduce<2, 1>(v, A.partials + A.part[B.inst], &S.counter[1], B.nblk, B.local, tot)) return;
    if (PHASE == 0) {
        S.bb = tot[0];
        return;
    }
    const double rr = tot[0];
    S.rr = rr;
    S.bwd = tot[1];
    bool start = false;
    if (PHASE == 1) {
        // each loop solves its own system: its start residual reduced by rtol, but never below
        // rtol 1e-4 of the start field's residual
        S.stop2 = A.rtol * A.rtol * fmax(rr, 1e-8 * (S.bb > 0. ? S.bb : 1.));
        S.it = 0;
        S.run = 0;
        S.cst = 0;
        start = rr > S.stop2;
    } else if (S.run == 0 && rr > S.stop2 && !(rr > 0.25 * S.rr_run)) {
        // the true residual has drifted above the level the recursive one reached: once more
        S.run = 1;
        A.stats[B.inst].restarts += 1;
        start = true;
    }
    S.pending = start ? 1 : 0;
    S.cg = start ? 1 : 0;
    if (start) {
        S.rr_run = rr;
        S.it_run = 0;
        S.alpha = 0.;
    }
}

// First damped line sweeps of a level (from zero): a block takes L.CB columns, 512 threads,
// part_solve.  x = omega M^-1 b goes to the level's r, its residual then to x (k_bs_resid), so
// that the way up reads one array and writes the other (k_bs_up).
//   START  level 0, start of a run: b as it is
//   UPD    level 0, in an iteration: b -= alpha q (q in r, overwritten) before it, (b, b) and
//          the stop test
//   DOWN   coarse level: b = R r of the finer level's residual (stored)
// 36, 52 and 52 bytes per node, 4 of them of the separators.  UPD 223 us for 9.7e6 nodes, 10 us for
// 24 small instances.  What holds it on large ones is HBM, at 2.7 times those bytes (1380 MB, 6.2
// TB/s): a block reads L.CB columns of a row, 5 (40 bytes) at 800 rows, and fetches whole lines.
enum { BS_START = 0, BS_UPD = 1, BS_DOWN = 2 };

template <int MODE>
__global__ __launch_bounds__(BS_T, 4) void k_bs_sweep(BsArgs A, const BsBlock* __restrict__ map) {
    extern __shared__ __align__(16) unsigned char part_smem[];
    const BsBlock B = map[blockIdx.x];
    BsState& S = A.st[B.inst];
    if (!S.cg || (MODE == BS_START && S.it_run > 0)) return;
    const BsLevel* LV = A.lev + A.lev0[B.inst] + B.level;
    const BsLevel L = *LV;
    const BsPool& P = A.pool[B.level > 0];
    const int plane = L.n0;
    const PartPos q = part_pos(L.n0, L.n1, L.P, L.CB, plane, BS_M, B.local);
    double* b = P.b + L.node;
    double* r = P.r + L.node;
    double rv[BS_M], qv[BS_M], av[BS_M], wv[BS_M], cv[BS_M], sv[3];
    double rr = 0.;
    if (MODE == BS_DOWN) {
        const BsLevel F = LV[-1];
        const int c = q.act ? q.col : 0;
        const int *cx = A.cx + F.cx, *mx = A.mx + F.mx;
        const double* wx = A.wx + F.mx;
        int ii[3];
        double wt[3];
        restrict_axis(c, L.n0, cx, mx, wx, ii, wt);
        const double* rf = A.pool[B.level > 1].x + F.node;
        const unsigned fixed = q.act ? P.fixed[L.seg + q.seg * L.n0 + q.col] : 0u;
#pragma unroll
        for (int u = 0; u < BS_M; ++u) {
            rv[u] = 0.;
            if (u < q.len) {
                const long long node = q.base + (long long)u * plane;
                const double* row = rf + (long long)(q.seg * BS_M + u) * F.n0;
                const double s = wt[0] * row[ii[0]] + wt[1] * row[ii[1]] + wt[2] * row[ii[2]];
                rv[u] = (fixed >> u) & 1u ? 0. : s;
                b[node] = rv[u];
            }
        }
    } else {
        part_load<double, BS_M>(q, plane, b, rv);
        if (MODE == BS_UPD) {
            const double alpha = S.alpha;
            part_load<double, BS_M>(q, plane, r, qv);  // level 0: q = A p lies in r
            part_factors<double, BS_M>(q, L.P, L.n0, plane, P.la + L.node, P.lw + L.node, P.lc + L.node, A.schur + L.schur,
                                       av, wv, cv, sv);
#pragma unroll
            for (int u = 0; u < BS_M; ++u) {
                rv[u] -= alpha * qv[u];
                rr += rv[u] * rv[u];
                if (u < q.len) b[q.base + (long long)u * plane] = rv[u];
            }
        }
    }
    if (MODE != BS_UPD)
        part_factors<double, BS_M>(q, L.P, L.n0, plane, P.la + L.node, P.lw + L.node, P.lc + L.node, A.schur + L.schur, av,
                                   wv, cv, sv);
    double zv[BS_M];
    part_solve<double, BS_M>(q, L.P, L.CB, reinterpret_cast<double*>(part_smem), rv, av, wv, cv, sv, zv);
#pragma unroll
    for (int u = 0; u < BS_M; ++u)
        if (u < q.len) r[q.base + (long long)u * plane] = A.omega * zv[u];
    if (MODE == BS_UPD) {
        double v[1] = {rr}, tot[1];
        if (bs_reduce<1, 0>(v, A.partials + A.part[B.inst], &S.counter[2], B.nblk, B.local, tot)) {
            S.rr = tot[0];
            S.it += 1;
            S.it_run += 1;
            if (tot[0] <= S.stop2) {
                S.cg = 0;
            } else if (S.it >= A.maxit) {
                S.cst = 1;
                S.cg = 0;
            }
        }
    }
}

// The coarsest levels of an instance in one block: sweep, residual and restriction on the way
// down, coarse_sweeps on the last level, correction, residual and sweep on the way up, one
// thread per column and segment, iterates and residuals in LDS.  From global memory only the
// levels' factors, conductivities and right-hand sides.  Held by the latency of its ~10 phases
// per level; as separate launches each level took six.
inline bool bs_tail_fits(int n0, int n1, int P, long long nodes) {  // nodes: of the level and all below it
    const int per = std::max(P, part_scan_lanes(P)), ps = part_lds_values(P, n0, BS_TAIL);
    return n0 * per <= BS_TAIL && (long long)n0 * n1 <= ps && (size_t)(nodes + ps) * sizeof(double) <= 150 * 1024;
}

// What a thread keeps of its segment on a level: line factors, element coefficients of the
// layers around it on both sides (0 where there is none), Dirichlet nodes.
struct BsSegment {
    double av[BS_M], wv[BS_M], cv[BS_M], sv[3];
    double c[BS_M + 1][4];
    unsigned fixed;
};

__device__ __forceinline__ void bs_segment(const BsLevel& L, const BsPool& P, const double* schur, const PartPos& q,
                                           BsSegment& G) {
    part_factors<double, BS_M>(q, L.P, L.n0, L.n0, P.la + L.node, P.lw + L.node, P.lc + L.node, schur + L.schur, G.av, G.wv,
                               G.cv, G.sv);
    G.fixed = q.act ? P.fixed[L.seg + q.seg * L.n0 + q.col] : 0u;
    const int i = q.act ? q.col : 0, k0 = q.act ? q.seg * BS_M : 0;
    const int eL = max(i - 1, 0), eR = min(i, L.n0 - 2);
    const double fL = i > 0 ? 1. : 0., fR = i < L.n0 - 1 ? 1. : 0.;
    const double *ea = P.ea + L.elem, *eb = P.eb + L.elem;
#pragma unroll
    for (int p = 0; p <= BS_M; ++p) {
        const int e = k0 - 1 + p;
        const long long o = (long long)min(max(e, 0), L.n1 - 2) * (L.n0 - 1);
        const double f = e >= 0 && e < L.n1 - 1 ? 1. : 0.;
        G.c[p][0] = ea[o + eL] * (fL * f);
        G.c[p][1] = eb[o + eL] * (fL * f);
        G.c[p][2] = ea[o + eR] * (fR * f);
        G.c[p][3] = eb[o + eR] * (fR * f);
    }
}

// r -= A x for a thread's segment, x in LDS: columns il, i, ir of rows n0 values apart, with
// `pad` more per segment; 0 at fixed nodes
__device__ __forceinline__ void bs_lds_residual(const BsLevel& L, const double* xs, int n0, int pad, int il, int i, int ir,
                                                const PartPos& q, const BsSegment& G, double (&r)[BS_M]) {
    if (!q.act) return;
    const int n1 = L.n1, k0 = q.seg * BS_M;
    double p[4], t[4];
    auto row = [&](int kk, double (&t)[4]) {
        const int k = min(max(kk, 0), n1 - 1);
        const double* o = xs + k * n0 + (k / BS_M) * pad;
        const double a = o[il], c = o[i], d = o[ir];
        t[0] = a + c;
        t[1] = c - a;
        t[2] = c + d;
        t[3] = c - d;
    };
    row(k0 - 1, p);
#pragma unroll
    for (int u = 0; u <= BS_M; ++u) {
        row(k0 + u, t);
        const double(&c)[4] = G.c[u];
        const double S = (t[1] + p[1]) * (3. * c[0]) + (t[3] + p[3]) * (3. * c[2]);
        const double D = (t[0] - p[0]) * (3. * c[1]) + (t[1] - p[1]) * (c[0] + c[1]) + (t[2] - p[2]) * (3. * c[3]) +
                         (t[3] - p[3]) * (c[2] + c[3]);
        if (u > 0) r[u - 1] -= S - D;
        if (u < BS_M) r[u] -= S + D;
#pragma unroll
        for (int w = 0; w < 4; ++w) p[w] = t[w];
    }
#pragma unroll
    for (int u = 0; u < BS_M; ++u)
        if (u >= q.len || ((G.fixed >> u) & 1u)) r[u] = 0.;
}

// The way up of one level in one kernel: x' = x + P x_c for a block's columns and one more on
// each side in LDS, then x = x' + omega M^-1 (b - A x') (on level 0 also (b, x) and the next
// beta).  x is read from r (where the way down left it, see steps_vcycle) and written to x, as
// neighbouring blocks read the columns around theirs.  As three kernels (correction, residual,
// sweep) it needs 104 instead of 64 bytes per node and three launches: 157 -> 146 ms for
// 96 uneven instances, 49 -> 46 ms for 24 small ones.  358 us for the 9.7e6 nodes of the instance
// grids, held by HBM at 3.4 times those bytes (2100 MB, 5.9 TB/s): the narrow rows of the sweeps,
// and two columns more per block.  x' is staged rather than read around each
// thread because the columns of a segment are M rows apart; the pad per segment puts the
// segments of a column into different banks.
__host__ __device__ inline int bs_up_pad(int CB) { return ((CB - BS_M * (CB + 2)) % 32 + 32) % 32; }
__host__ __device__ inline int bs_up_lds(int n1, int P, int CB) {
    return n1 * (CB + 2) + P * bs_up_pad(CB) + part_lds_values(P, CB, BS_T);
}

__global__ __launch_bounds__(BS_T, 2) void k_bs_up(BsArgs A, const BsBlock* __restrict__ map) {
    extern __shared__ __align__(16) unsigned char part_smem[];
    const BsBlock B = map[blockIdx.x];
    BsState& S = A.st[B.inst];
    if (!S.cg) return;
    const BsLevel* LV = A.lev + A.lev0[B.inst] + B.level;
    const BsLevel L = LV[0];
    const BsPool& P = A.pool[B.level > 0];
    const PartPos q = part_pos(L.n0, L.n1, L.P, L.CB, L.n0, BS_M, B.local);
    const int HX = L.CB + 2, pad = bs_up_pad(L.CB);
    double* ps = reinterpret_cast<double*>(part_smem);
    double* xt = ps + part_lds_values(L.P, L.CB, BS_T);
    // the segment's own data travels while the tile is staged
    BsSegment G;
    bs_segment(L, P, A.schur, q, G);
    double rv[BS_M], bv[BS_M], zv[BS_M];
#pragma unroll
    for (int u = 0; u < BS_M; ++u) bv[u] = u < q.len ? P.b[L.node + q.base + (long long)u * L.n0] : 0.;
    {
        const int per = BS_T / HX, c = (int)threadIdx.x % HX, k0 = (int)threadIdx.x / HX;
        const int i = B.local * L.CB - 1 + c;
        if (k0 < per) {
            const bool in = i >= 0 && i < L.n0, coarse = B.level < A.inst[B.inst].nlev;
            const int ic = min(max(i, 0), L.n0 - 1);
            const BsLevel C = LV[coarse ? 1 : 0];
            const int J = coarse ? A.mx[L.mx + ic] : 0, J1 = min(J + 1, C.n0 - 1);
            const double a = coarse ? A.wx[L.mx + ic] : 0.;
            const double* x = P.r + L.node + ic;
            const double* xc = A.pool[1].x + C.node;
            constexpr int U = 8;
            for (int kb = k0; kb < L.n1; kb += U * per) {
                double v[U], c0[U], c1[U];
                bool fx[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int k = min(kb + u * per, L.n1 - 1);
                    v[u] = x[(long long)k * L.n0];
                    c0[u] = coarse ? xc[(long long)k * C.n0 + J] : 0.;
                    c1[u] = coarse ? xc[(long long)k * C.n0 + J1] : 0.;
                    fx[u] = (P.fixed[L.seg + (k / BS_M) * L.n0 + ic] >> (k % BS_M)) & 1u;
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int k = kb + u * per;
                    const double o = fx[u] ? v[u] : v[u] + ((1. - a) * c0[u] + a * c1[u]);
                    if (k < L.n1) xt[k * HX + (k / BS_M) * pad + c] = in ? o : 0.;
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BS_M; ++u) rv[u] = bv[u];
    bs_lds_residual(L, xt, HX, pad, q.cl, q.cl + 1, q.cl + 2, q, G, rv);
    part_solve<double, BS_M>(q, L.P, L.CB, ps, rv, G.av, G.wv, G.cv, G.sv, zv);
    double rz = 0.;
#pragma unroll
    for (int u = 0; u < BS_M; ++u) {
        if (u < q.len) {
            const double o = xt[(q.seg * BS_M + u) * HX + q.seg * pad + q.cl + 1] + A.omega * zv[u];
            P.x[L.node + q.base + (long long)u * L.n0] = o;
            rz += bv[u] * o;
        }
    }
    if (B.level == 0) {
        double v[1] = {rz}, tot[1];
        if (bs_reduce<1, 0>(v, A.partials + A.part[B.inst], &S.counter[3], B.nblk, B.local, tot)) {
            S.rz_prev = S.rz;
            S.rz = tot[0];
            if (S.it_run > 0 && !(tot[0] > 0.)) {
                S.cst = -7;
                S.cg = 0;
            }
        }
    }
}

__global__ __launch_bounds__(BS_TAIL) void k_bs_tail(BsArgs A, int ninst) {
    extern __shared__ __align__(16) unsigned char part_smem[];
    const int inst = blockIdx.x;
    const int lt = A.tail[inst], nlev = A.inst[inst].nlev;
    if (!A.st[inst].cg || lt > nlev) return;
    const BsLevel* LV = A.lev + A.lev0[inst];
    const BsPool& P = A.pool[1];
    const BsLevel T0 = LV[lt];
    // LDS: part_solve's values (also the residual between two levels), then x of every level
    double* ps = reinterpret_cast<double*>(part_smem);
    double* xs = ps + part_lds_values(T0.P, T0.n0, BS_TAIL);
    const long long xnode0 = T0.node;  // the levels of an instance are consecutive in the pool
    auto pos = [&](const BsLevel& L) { return part_pos(L.n0, L.n1, L.P, L.n0, L.n0, BS_M, 0); };
    for (int l = lt; l <= nlev; ++l) {
        const BsLevel L = LV[l], F = LV[l - 1];
        const PartPos q = pos(L);
        BsSegment G;
        bs_segment(L, P, A.schur, q, G);
        double* x = xs + (L.node - xnode0);
        double bv[BS_M], rv[BS_M], zv[BS_M];
        {
            const int c = q.act ? q.col : 0;
            int ii[3];
            double wt[3];
            restrict_axis(c, L.n0, A.cx + F.cx, A.mx + F.mx, A.wx + F.mx, ii, wt);
            const double* rf = l == lt ? A.pool[l > 1].x + F.node : ps;
#pragma unroll
            for (int u = 0; u < BS_M; ++u) {
                bv[u] = 0.;
                if (u < q.len) {
                    const double* row = rf + (long long)(q.seg * BS_M + u) * F.n0;
                    const double s = wt[0] * row[ii[0]] + wt[1] * row[ii[1]] + wt[2] * row[ii[2]];
                    bv[u] = (G.fixed >> u) & 1u ? 0. : s;
                    if (l < nlev) P.b[L.node + q.base + (long long)u * L.n0] = bv[u];  // for the way up
                }
            }
        }
        __syncthreads();  // the finer level's residual is read
        part_solve<double, BS_M>(q, L.P, L.n0, ps, bv, G.av, G.wv, G.cv, G.sv, zv);
#pragma unroll
        for (int u = 0; u < BS_M; ++u)
            if (u < q.len) x[q.base + (long long)u * L.n0] = A.omega * zv[u];
        __syncthreads();
        const int sweeps = l == nlev ? A.coarse_sweeps : 2;
        for (int sw = 1; sw < sweeps; ++sw) {
#pragma unroll
            for (int u = 0; u < BS_M; ++u) rv[u] = bv[u];
            bs_lds_residual(L, x, L.n0, 0, max(q.col - 1, 0), q.col, min(q.col + 1, L.n0 - 1), q, G, rv);
            if (l < nlev) {  // to the next coarser level
#pragma unroll
                for (int u = 0; u < BS_M; ++u)
                    if (u < q.len) ps[q.base + (long long)u * L.n0] = rv[u];
                __syncthreads();
                break;
            }
            __syncthreads();
            part_solve<double, BS_M>(q, L.P, L.n0, ps, rv, G.av, G.wv, G.cv, G.sv, zv);
#pragma unroll
            for (int u = 0; u < BS_M; ++u)
                if (u < q.len) x[q.base + (long long)u * L.n0] += A.omega * zv[u];
            __syncthreads();
        }
    }
    for (int l = nlev - 1; l >= lt; --l) {
        const BsLevel L = LV[l], C = LV[l + 1];
        const PartPos q = pos(L);
        BsSegment G;
        bs_segment(L, P, A.schur, q, G);
        double rv[BS_M], zv[BS_M];
#pragma unroll
        for (int u = 0; u < BS_M; ++u) rv[u] = u < q.len ? P.b[L.node + q.base + (long long)u * L.n0] : 0.;
        double* x = xs + (L.node - xnode0);
        const double* xc = xs + (C.node - xnode0);
        const int c = q.act ? q.col : 0;
        const int J = A.mx[L.mx + c], J1 = min(J + 1, C.n0 - 1);
        const double a = A.wx[L.mx + c];
#pragma unroll
        for (int u = 0; u < BS_M; ++u)
            if (u < q.len && !((G.fixed >> u) & 1u)) {
                const int k = q.seg * BS_M + u;
                x[q.base + (long long)u * L.n0] += (1. - a) * xc[k * C.n0 + J] + a * xc[k * C.n0 + J1];
            }
        __syncthreads();
        bs_lds_residual(L, x, L.n0, 0, max(q.col - 1, 0), q.col, min(q.col + 1, L.n0 - 1), q, G, rv);
        part_solve<double, BS_M>(q, L.P, L.n0, ps, rv, G.av, G.wv, G.cv, G.sv, zv);
#pragma unroll
        for (int u = 0; u < BS_M; ++u)
            if (u < q.len) x[q.base + (long long)u * L.n0] += A.omega * zv[u];
        __syncthreads();
    }
    double* out = P.x + T0.node;
    for (int n = threadIdx.x; n < T0.n0 * T0.n1; n += BS_TAIL) out[n] = xs[n];
}

// ---------------------------------------------------------------------------
// set-up of a Picard loop
// ---------------------------------------------------------------------------
// junction update from the current potential (not before the first solve); a block per instance
__global__ __launch_bounds__(256) void k_bs_junction(BsArgs A) {
    const BsState& S = A.st[blockIdx.x];
    const BatchInst I = A.inst[blockIdx.x];
    if (S.fin || S.loops == 0 || I.jhi <= I.jlo) return;
    const double* x = A.X + I.node_off;
    double* sh = A.pool[0].kh + I.elem_off;
    double* sv = A.pool[0].kv + I.elem_off;
    const int n0 = I.n0, nje = (I.jhi - I.jlo) * (n0 - 1);
    for (int t = threadIdx.x; t < nje; t += 256) {
        const int ei = t % (n0 - 1), ek = I.jlo + t / (n0 - 1);
        const long long e = (long long)ek * (n0 - 1) + ei;
        const double U = 0.5 * (x[(long long)I.jhi * n0 + ei] - x[(long long)I.jlo * n0 + ei] +
                                x[(long long)I.jhi * n0 + ei + 1] - x[(long long)I.jlo * n0 + ei + 1]);
        const double jy = fabs(0.1 * sv[e] * U / I.jheight);
        double cond = 10. * jy * I.jheight * I.beta / log(1e7 * jy / I.js + 1.);
        if (A.stable) cond = 0.5 * (sv[e] + cond);
        if (isnan(cond) || fabs(cond) < 1e-16) cond = 1e-16;
        sv[e] = cond;
        sh[e] = 0.;
    }
}

// coarse conductivities of every level (coarsen_k_l's means) and the element coefficients
// ea = kx' / 12, eb = ky' / 12 of every level (kx' = k h / w, ky' = k w / h, times the mid
// radius in cylindrical geometry): element rows are independent, a wave takes one through all
// its levels
__global__ __launch_bounds__(64) void k_bs_coarsen(BsArgs A, const BsBlock* __restrict__ map) {
    extern __shared__ __align__(16) unsigned char part_smem[];
    const BsBlock B = map[blockIdx.x];
    if (A.st[B.inst].fin) return;
    const BatchInst I = A.inst[B.inst];
    const BsLevel* LV = A.lev + A.lev0[B.inst];
    const long long k = B.local;
    double* fh = reinterpret_cast<double*>(part_smem);
    double* fv = fh + (I.n0 - 1);
    double* ch = fv + (I.n0 - 1);
    double* cv = ch + (I.n0 - 1);
    const int tid = threadIdx.x;
    const double h = A.h1[I.h1_off + k];
    auto coef = [&](const BsLevel& L, const BsPool& P, int e, double a, double c) {
        const double w = P.h0[L.h0 + e], r = I.cyl ? P.rm[L.h0 + e] : 1.;
        const long long o = L.elem + k * (L.n0 - 1) + e;
        P.ea[o] = r * a * h / w / 12.;
        P.eb[o] = r * c * w / h / 12.;
    };
    for (int e = tid; e < I.n0 - 1; e += 64) {
        fh[e] = A.pool[0].kh[LV[0].elem + k * (I.n0 - 1) + e];
        fv[e] = A.pool[0].kv[LV[0].elem + k * (I.n0 - 1) + e];
        coef(LV[0], A.pool[0], e, fh[e], fv[e]);
    }
    __syncthreads();
    for (int l = 1; l <= I.nlev; ++l) {
        const BsLevel F = LV[l - 1], C = LV[l];
        const double *h0 = A.pool[l > 1].h0 + F.h0, *rm = A.pool[l > 1].rm + F.h0;
        const int* cx = A.cx + F.cx;
        for (int J = tid; J < C.n0 - 1; J += 64) {
            double sa = 0., sh = 0., sv = 0.;
            for (int ex = cx[J]; ex < cx[J + 1]; ++ex) {
                const double a = h0[ex] * (I.cyl ? rm[ex] : 1.);
                sa += a;
                sh += a * fh[ex];
                sv += a * fv[ex];
            }
            ch[J] = sh / sa;
            cv[J] = sv / sa;
            A.pool[1].kh[C.elem + k * (C.n0 - 1) + J] = ch[J];
            A.pool[1].kv[C.elem + k * (C.n0 - 1) + J] = cv[J];
            coef(C, A.pool[1], J, ch[J], cv[J]);
        }
        __syncthreads();
        double* t = fh;
        fh = ch;
        ch = t;
        t = fv;
        fv = cv;
        cv = t;
    }
}

// line coefficients per node of every level (line_factors_l's); scratch: b and x of the coarse
// levels, q (pool r) and z (pool x) of level 0, all free between the loops
__global__ __launch_bounds__(256) void k_bs_line(BsArgs A, const BsBlock* __restrict__ map) {
    const BsBlock B = map[blockIdx.x];
    if (A.st[B.inst].fin) return;
    const BatchInst I = A.inst[B.inst];
    const BsLevel L = A.lev[A.lev0[B.inst] + B.level];
    const LView V = bs_view(A, I, L, B.level);
    const unsigned u = (unsigned)B.local * 256 + threadIdx.x;
    if (u >= (unsigned)L.n0 * L.n1) return;
    const int k = (int)(u / (unsigned)L.n0), i = (int)(u - (unsigned)k * L.n0);
    double b = 0., c = 0.;
    for (int cc = 0; cc < 4; ++cc) {
        const int ei = i - 1 + (cc & 1), ek = k - 1 + (cc >> 1);
        if (ei < 0 || ek < 0 || ei >= L.n0 - 1 || ek >= L.n1 - 1) continue;
        const long long e = (long long)ek * (L.n0 - 1) + ei;
        const double w = V.h0[ei], h = V.h1[ek], rr = V.cyl ? V.rm[ei] : 1.;
        const double kx1 = rr * V.kh[e] * h / w, ky1 = rr * V.kv[e] * w / h;
        b += (kx1 + ky1) / 3.;
        if (ek == k) c += (kx1 - 2. * ky1) / 6.;
    }
    const bool dk = lbit(V, u);
    if (dk) b = 1.;
    if (dk || k == L.n1 - 1 || lbit(V, (long long)u + L.n0)) c = 0.;
    const BsPool& P = A.pool[B.level > 0];
    (B.level ? P.b : P.r)[L.node + u] = b;
    P.x[L.node + u] = c;
}

// segment factors (part_factor_segment) and, per column, the separators' (part_schur_column);
// segment sums: r of the coarse levels, the direction buffer of level 0
__device__ __forceinline__ double* bs_sums(const BsArgs& A, const BsLevel& L, int l) {
    return (l ? A.pool[1].r : A.PA) + L.node;
}

__global__ __launch_bounds__(256) void k_bs_factor(BsArgs A, const BsBlock* __restrict__ map) {
    const BsBlock B = map[blockIdx.x];
    if (A.st[B.inst].fin) return;
    const BsLevel L = A.lev[A.lev0[B.inst] + B.level];
    const BsPool& P = A.pool[B.level > 0];
    const int t = B.local * 256 + (int)threadIdx.x;
    if (t >= L.P * L.n0) return;
    double* sff = bs_sums(A, L, B.level);
    part_factor_segment<double>(t % L.n0, t / L.n0, L.n0, L.n1, BS_M, L.n0, (B.level ? P.b : P.r) + L.node, P.x + L.node,
                                P.la + L.node, P.lw + L.node, P.lc + L.node, sff, sff + (size_t)L.P * L.n0);
}

__global__ __launch_bounds__(64) void k_bs_schur(BsArgs A, const BsBlock* __restrict__ map) {
    const BsBlock B = map[blockIdx.x];
    if (A.st[B.inst].fin) return;
    const BsLevel L = A.lev[A.lev0[B.inst] + B.level];
    const BsPool& P = A.pool[B.level > 0];
    const int col = B.local * 64 + (int)threadIdx.x;
    if (col >= L.n0) return;
    const double* sff = bs_sums(A, L, B.level);
    part_schur_column<double>(col, L.n0, L.n1, BS_M, L.n0, P.la + L.node, P.lw + L.node, P.lc + L.node, sff,
                              sff + (size_t)L.P * L.n0, A.schur + L.schur);
}

// ---------------------------------------------------------------------------
// end of a run and of a Picard loop
// ---------------------------------------------------------------------------
// the last x += alpha p of a run (the next fused apply would have done it)
__global__ __launch_bounds__(256) void k_bs_fixup(BsArgs A, const BsBlock* __restrict__ map) {
    const BsBlock B = map[blockIdx.x];
    const BsState& S = A.st[B.inst];
    if (!S.pending) return;
    const BsLevel L = A.lev[A.lev0[B.inst]];
    const unsigned u = (unsigned)B.local * 256 + threadIdx.x;
    if (u >= (unsigned)L.n0 * L.n1) return;
    const double* p = ((S.it_run & 1) ? A.PB : A.PA) + L.node;
    if (S.it_run > 0) A.X[L.node + u] += S.alpha * p[u];
}

// element currents and the loop error; the last block of an instance ends its loop
__global__ __launch_bounds__(256) void k_bs_currents(BsArgs A, const BsBlock* __restrict__ map) {
    const BsBlock B = map[blockIdx.x];
    BsState& S = A.st[B.inst];
    if (S.fin) return;
    const BatchInst I = A.inst[B.inst];
    const int n0 = I.n0;
    const unsigned E = (unsigned)(I.n0 - 1) * (I.n1 - 1), e = (unsigned)B.local * 256 + threadIdx.x;
    const bool has_j = I.jhi > I.jlo;
    double dmax = 0., jmax = 0.;
    if (e < E) {
        const int ek = (int)(e / (unsigned)(n0 - 1)), ei = (int)(e - (unsigned)ek * (n0 - 1));
        const double w = A.pool[0].h0[I.h0_off + ei], h = A.h1[I.h1_off + ek];
        const double* x = A.X + I.node_off + (long long)ek * n0 + ei;
        double* cur = A.cur + 2 * (I.elem_off + e);
        const double vll = x[0], vlu = x[1], vul = x[n0], vuu = x[n0 + 1];
        const double jx = A.pool[0].kh[I.elem_off + e] * (-0.05 * (-vll + vlu - vul + vuu) / w);
        const double jy = A.pool[0].kv[I.elem_off + e] * (-0.05 * (-vll - vlu + vul + vuu) / h);
        const double dx = jx - cur[0], dy = jy - cur[1];
        cur[0] = jx;
        cur[1] = jy;
        dmax = dx * dx + dy * dy;
        if (!has_j || (ek >= I.jlo && ek < I.jhi)) jmax = jx * jx + jy * jy;
    }
    double v[2] = {dmax, jmax}, tot[2];
    if (!bs_reduce<2, 2>(v, A.partials + A.part[B.inst], &S.counter[0], B.nblk, B.local, tot)) return;
    BatchStats& T = A.stats[B.inst];
    if (S.cst != 0) T.status = S.cst;
    T.iters += S.it;
    T.rel = sqrt(S.rr / S.stop2) * A.rtol;
    T.bwd = S.bwd;
    T.maxj = sqrt(tot[1]);
    T.err = 100. * sqrt(tot[0]) / fmax(T.maxj, 100e-7);
    S.loops += 1;
    T.loops = S.loops;
    if (T.status < 0 || (T.status == 0 && T.err <= A.maxerr)) {
        S.fin = 1;
    } else if (S.loops == A.maxloops) {
        T.status = 2;
        S.fin = 1;
    }
    S.pending = 0;
}

// total current through the middle junction row (integrateCurrent, electr2d.cpp:466-496)
__global__ __launch_bounds__(256) void k_bs_total(BsArgs A) {
    __shared__ double red[16];
    const BatchInst I = A.inst[blockIdx.x];
    double tot = 0.;
    if (I.jhi > I.jlo) {
        const int level = (I.jlo + I.jhi) / 2;
        for (int ei = threadIdx.x; ei < I.n0 - 1; ei += 256) {
            const double j1 = A.cur[2 * (I.elem_off + (long long)level * (I.n0 - 1) + ei) + 1];
            const double w = A.pool[0].h0[I.h0_off + ei];
            if (I.cyl) {
                const double r0 = A.pool[0].rm[I.h0_off + ei] - 0.5 * w, r1 = A.pool[0].rm[I.h0_off + ei] + 0.5 * w;
                tot += j1 * (r1 * r1 - r0 * r0);
            } else {
                tot += j1 * w;
            }
        }
    }
    tot = wg_sum(tot, red);
    if (threadIdx.x == 0)
        A.stats[blockIdx.x].current = I.cyl ? tot * 3.14159265358979323846 * 0.01 : tot * 0.01;
}

// instances that still iterate (count[0]) and that have ended (count[1]); one block
__global__ __launch_bounds__(256) void k_bs_count(BsArgs A, int ninst) {
    __shared__ double red[16];
    double cg = 0., fin = 0.;
    for (int i = threadIdx.x; i < ninst; i += 256) {
        cg += A.st[i].cg ? 1. : 0.;
        fin += A.st[i].fin ? 1. : 0.;
    }
    cg = wg_sum(cg, red);
    fin = wg_sum(fin, red);
    if (threadIdx.x == 0) {
        A.count[0] = (int)cg;
        A.count[1] = (int)fin;
    }
}

__global__ void k_bs_reset(BsArgs A, int ninst) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ninst; i += gridDim.x * blockDim.x) {
        A.st[i] = BsState{};
        A.stats[i] = BatchStats{};
    }
}

}  // namespace pf
