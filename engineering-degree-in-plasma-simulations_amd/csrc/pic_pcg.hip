// pic_pcg.hip -- Newton + PCG of the gfx950 PIC library.
//
//   k_F          Newton residual F = A phi - b - q n0 e^{(phi-phi0)/Te0}/eps0
//                and the Jacobian diagonal shift (PotentialSolver.cpp:189-217)
//   k_pcg1/2     matrix-free Jacobi PCG (PotentialSolver.cpp:243-313), two
//                fused kernels per iteration, scalars kept on the device
//   k_cg         an iteration in one kernel, for small grids
#include "pic_stencil.h"

namespace {

// ------------------------------------------------------------------------
// Newton residual and Jacobian shift (PotentialSolver.cpp:189-217)
//   b_u = 0 (Neumann), phi_u (Dirichlet), -rho_u/eps0 (regular)
//   F = A phi - b - [regular] q n0 exp((phi-phi0)/Te0)/eps0
//   P = [regular] q n0/(eps0 Te0) exp((phi-phi0)/Te0)
// partial sums F.F (all rows), F.F (regular), b.b (regular)
// START: the set-up of PCG on J y = F from y = 0 instead of F itself: g = -F
// (TF), its Jacobi-scaled s = M g (NEU), and the partial sums g.s and g.g;
// the stop flag of the iterations that follow is cleared.
// ------------------------------------------------------------------------
template <typename TF, bool START, bool NEU>
__global__ void __launch_bounds__(BLOCK)
    k_F(Stencil s, NewtonArgs a, const uint8_t* __restrict__ nt, const double* __restrict__ phi,
        const double* __restrict__ rho, TF* __restrict__ F, TF* __restrict__ sv, double* __restrict__ P,
        double* __restrict__ scratch) {
    double f_all = 0, f_reg = 0, b_reg = 0, gs = 0, gg = 0;
    // one node: its row of F, and what START keeps of it
    auto row = [&](uint8_t t, double Ap, double pu, double rho_u, double& Pu, TF& Fu, TF& su) {
        Pu = 0.0;
        double f;
        if (t == NT_REG) {
            const double b = -rho_u * a.ieps;
            f = Ap - b;
            if (a.n0 != 0.0) {
                const double ex = exp((pu - a.phi0) * a.inv_te0);
                f -= QE * a.n0 * ex * a.ieps;
                Pu = QE * a.n0 * a.ieps * a.inv_te0 * ex;
            }
            f_reg += f * f;
            b_reg += b * b;
        } else {
            f = t == NT_DIR ? 0.0 : Ap;  // a Dirichlet row is phi - phi
        }
        f_all += f * f;
        Fu = START ? -(TF)f : (TF)f;
        if (START) {
            su = (TF)(1.0 / diagA(t, s)) * Fu;
            gs += (double)Fu * (double)su;
            gg += (double)Fu * (double)Fu;
        }
    };
    long long end;
    for (long long m = chunk_begin(s.nn / 4, end) + threadIdx.x; m < end; m += BLOCK) {
        const unsigned u0 = 4u * (unsigned)m;
        const uint32_t t4 = load_types4(nt, u0);
        Ring4<double> g;
        load_ring4(phi, u0, s, g);
        const Q4<double> rh = load4(rho + u0);
        TF f4[4], s4[4];
        double P4[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint8_t t = type_at(t4, q);
            double Ap = 0.0;
            if (t == NT_REG)
                Ap = ring_A(g, q, s);
            else if (NEU && t != NT_DIR)
                Ap = apply_A<double>(t, u0 + q, s, [&](long long v) { return phi[v]; });
            s4[q] = 0;
            row(t, Ap, g.c.a[q], rh.a[q], P4[q], f4[q], s4[q]);
        }
        store4(F + u0, f4);
        if (START && NEU) store4(sv + u0, s4);
        if (P) store4(P + u0, P4);
    }
    if (blockIdx.x == 0 && threadIdx.x < (unsigned)(s.nn & 3)) {  // corner nodes past the last group
        const long long u = (s.nn & ~3ll) + threadIdx.x;
        const uint8_t t = nt[u];
        double Pu;
        TF Fu, su = 0;
        row(t, NEU ? apply_A<double>(t, u, s, [&](long long v) { return phi[v]; }) : 0.0, phi[u], rho[u], Pu, Fu, su);
        F[u] = Fu;
        if (START && NEU) sv[u] = su;
        if (P) P[u] = Pu;
    }
    double t0 = block_sum(f_all), t1 = block_sum(f_reg), t2 = block_sum(b_reg);
    if (threadIdx.x == 0) {
        scratch[PART_F + blockIdx.x] = t0;
        scratch[PART_F + PART_MAX + blockIdx.x] = t1;
        scratch[PART_F + 2 * PART_MAX + blockIdx.x] = t2;
    }
    if (START) {
        double t3 = block_sum(gs), t4 = block_sum(gg);
        if (threadIdx.x == 0) {
            scratch[PART_GS + blockIdx.x] = t3;
            scratch[PART_GG + blockIdx.x] = t4;
            if (blockIdx.x == 0) scratch[PCG_FLAG] = 0.0;
        }
    }
}

// ------------------------------------------------------------------------
// PCG on J y = F, J = A - diag(P), M = 1/diag(A), two kernels per iteration
// over groups of four nodes, sums by partials.  Without Neumann faces M is
// one constant on every row where g is not 0 (Dirichlet rows of F vanish),
// so s = M g is formed from g where it is read; with them (NEU) s is kept.
//
// 128^3 nodes, FP64: k_pcg1 moves 41 B and k_pcg2 48 B per node of
// cache-resident vectors, about 18 us each (5 TB/s); with one node per load,
// eight nodes per thread, s stored and atomics on single words they took 27.8
// and 30.2 us.  97^3 FP32: 5.6 and 5.0 us, close to an empty launch's 4 us,
// against 14.1 and 13.5 us.
// ------------------------------------------------------------------------
template <typename T>
struct PcgVec {
    T *y, *g, *s, *z;  // s: NEU only
    const double* P;   // may be null
};

// d_new = beta d_old - s (beta = gs[t]/gs[t-1], 0 at t = 0); z = J d_new,
// by the recurrence J d_new = beta J d_old - J s: the stencil of s alone
// (one operand's neighbours instead of two), the previous z in place.
// gg[t] is kept for the host's check.  Returns at once when the stop flag is
// set (an earlier iteration converged).
template <typename T, bool NEU>
__global__ void __launch_bounds__(BLOCK)
    k_pcg1(Stencil s, const uint8_t* __restrict__ nt, PcgVec<T> v, const T* __restrict__ dold,
           T* __restrict__ dnew, double* __restrict__ scratch, double* __restrict__ ggh, int t) {
    if (scratch[PCG_FLAG] != 0.0) return;  // (the whole grid)
    const T* __restrict__ src = NEU ? v.s : v.g;
    const T mreg = (T)(1.0 / diagA(NT_REG, s));  // M of a regular row (k_pcg2's s, rounded alike)
    long long end;
    long long m = chunk_begin(s.nn / 4, end) + threadIdx.x;
    Ring4<T> r;
    Q4<T> d4{}, z4{};
    uint32_t t4 = 0;
    auto load = [&]() {
        const unsigned u0 = 4u * (unsigned)m;
        t4 = load_types4(nt, u0);
        load_ring4(src, u0, s, r);
        if (t > 0) {
            d4 = load4(dold + u0);
            z4 = load4(v.z + u0);
        }
    };
    if (m < end) load();
    const double gs = sum_parts(scratch + PART_GS, gridDim.x);
    double beta = 0.0;
    if (t > 0) {
        const double den = scratch[PCG_GS + ((t - 1) & 3)];
        beta = den != 0.0 ? gs / den : 0.0;
    }
    const T bt = (T)beta;
    double acc = 0;
    while (m < end) {
        const unsigned u0 = 4u * (unsigned)m;
        if (!NEU) {  // s = M g
#pragma unroll
            for (int q = 0; q < 4; q++) {
                r.c.a[q] *= mreg;
                r.ym.a[q] *= mreg;
                r.yp.a[q] *= mreg;
                r.zm.a[q] *= mreg;
                r.zp.a[q] *= mreg;
            }
            r.l *= mreg;
            r.r *= mreg;
        }
        T dn[4], zn[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint8_t ty = type_at(t4, q);
            const T su = r.c.a[q];
            T js = su;  // a Dirichlet row
            if (ty == NT_REG)
                js = ring_A(r, q, s);
            else if (NEU && ty != NT_DIR)
                js = apply_A<T>(ty, u0 + q, s, [&](long long w) { return src[w]; });
            if (v.P) js -= (T)v.P[u0 + q] * su;
            dn[q] = -su + bt * d4.a[q];
            zn[q] = -js + bt * z4.a[q];
            acc += (double)dn[q] * (double)zn[q];
        }
        store4(dnew + u0, dn);
        store4(v.z + u0, zn);
        m += BLOCK;
        if (m < end) load();
    }
    if (NEU && blockIdx.x == 0 && threadIdx.x < (unsigned)(s.nn & 3)) {  // corner nodes past the last group
        const long long u = (s.nn & ~3ll) + threadIdx.x;
        const T su = src[u];
        T js = apply_A<T>(nt[u], u, s, [&](long long w) { return src[w]; });
        if (v.P) js -= (T)v.P[u] * su;
        T du = -su, zu = -js;
        if (t > 0) {
            du += bt * dold[u];
            zu += bt * v.z[u];
        }
        dnew[u] = du;
        v.z[u] = zu;
        acc += (double)du * (double)zu;
    }
    const double a = block_sum(acc);
    if (threadIdx.x == 0) scratch[PART_DZ + blockIdx.x] = a;
    if (blockIdx.x == 0) {
        const double gg = sum_parts(scratch + PART_GG, gridDim.x);
        if (threadIdx.x == 0) {
            scratch[PCG_GS + (t & 3)] = gs;
            ggh[t] = gg;
        }
    }
}

// alpha = gs[t]/dz[t]; y += alpha d (y = 0 before t = 0); g += alpha z;
// s = M g; gs[t+1], gg[t+1]
template <typename T, bool NEU>
__global__ void __launch_bounds__(BLOCK)
    k_pcg2(Stencil s, const uint8_t* __restrict__ nt, PcgVec<T> v, const T* __restrict__ d,
           double* __restrict__ scratch, int t) {
    if (scratch[PCG_FLAG] != 0.0) return;  // (the whole grid)
    const T mreg = (T)(1.0 / diagA(NT_REG, s));
    long long end;
    long long m = chunk_begin(s.nn / 4, end) + threadIdx.x;
    Q4<T> g4, z4, y4{}, d4;
    uint32_t t4 = 0;
    auto load = [&]() {
        const unsigned u0 = 4u * (unsigned)m;
        g4 = load4(v.g + u0);
        z4 = load4(v.z + u0);
        if (t > 0) y4 = load4(v.y + u0);
        d4 = load4(d + u0);
        if (NEU) t4 = load_types4(nt, u0);
    };
    if (m < end) load();
    const double den = sum_parts(scratch + PART_DZ, gridDim.x);
    const T alpha = (T)(den != 0.0 ? scratch[PCG_GS + (t & 3)] / den : 0.0);
    double gs = 0, gg = 0;
    auto sums = [&](T gu, T su) {
        gs += (double)gu * (double)su;
        gg += (double)gu * (double)gu;
    };
    while (m < end) {
        const unsigned u0 = 4u * (unsigned)m;
        T gn[4], yn[4], sn[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            gn[q] = g4.a[q] + alpha * z4.a[q];
            yn[q] = y4.a[q] + alpha * d4.a[q];
            sn[q] = (NEU ? (T)(1.0 / diagA(type_at(t4, q), s)) : mreg) * gn[q];
            sums(gn[q], sn[q]);
        }
        store4(v.g + u0, gn);
        store4(v.y + u0, yn);
        if (NEU) store4(v.s + u0, sn);
        m += BLOCK;
        if (m < end) load();
    }
    if (blockIdx.x == 0 && threadIdx.x < (unsigned)(s.nn & 3)) {  // corner nodes past the last group
        const long long u = (s.nn & ~3ll) + threadIdx.x;
        if (NEU) {
            const T gu = v.g[u] + alpha * v.z[u];
            const T su = (T)(1.0 / diagA(nt[u], s)) * gu;
            v.y[u] = (t > 0 ? v.y[u] : (T)0) + alpha * d[u];
            v.g[u] = gu;
            v.s[u] = su;
            sums(gu, su);
        }
    }
    const double a = block_sum(gs), b = block_sum(gg);
    if (threadIdx.x == 0) {
        scratch[PART_GS + blockIdx.x] = a;
        scratch[PART_GG + blockIdx.x] = b;
    }
}

// The same iteration in one kernel (Chronopoulos and Gear's arrangement of CG:
// J. Comput. Appl. Math. 25, 1989), for grids without Neumann faces that a
// launch's latency bounds.  With u = M g, w = J u and the sums gamma = g.u,
// delta = w.u of the last kernel,
//   beta = gamma / gamma_old,  alpha = gamma / (delta - beta gamma / alpha_old)
//   d = -u + beta d,  z = -w + beta z (= J d),  y += alpha d,  g += alpha z
// and then the new w and sums.  The new w needs the new g of the neighbours,
// which every thread makes again from the old g, w and z around its group;
// those three are therefore written to a second set of vectors.  t = -1: w and
// delta of the start.
template <typename T>
struct CgVec {
    T *y, *d, *g[2], *w[2], *z[2];
    const double* P;  // may be null
};
template <typename T>
__global__ void __launch_bounds__(BLOCK)
    k_cg(Stencil s, const uint8_t* __restrict__ nt, CgVec<T> v, double* __restrict__ scratch,
         double* __restrict__ ggh, int t) {
    if (scratch[PCG_FLAG] != 0.0) return;  // (the whole grid)
    const int from = t < 0 ? 0 : t & 1, to = t < 0 ? 0 : (t + 1) & 1;
    const double* __restrict__ pin = scratch + from * PART_SET;
    double* __restrict__ pout = scratch + to * PART_SET;
    const T* __restrict__ gi = v.g[from];
    const T* __restrict__ wi = v.w[from];
    const T* __restrict__ zi = v.z[from];
    const T mreg = (T)(1.0 / diagA(NT_REG, s));  // M of a regular row; g vanishes on the others
    long long end;
    long long m = chunk_begin(s.nn / 4, end) + threadIdx.x;
    Ring4<T> g{}, w{}, z{};
    Q4<T> d4{}, y4{};
    uint32_t t4 = 0;
    auto load = [&]() {
        const unsigned u0 = 4u * (unsigned)m;
        t4 = load_types4(nt, u0);
        load_ring4(gi, u0, s, g);
        if (t >= 0) load_ring4(wi, u0, s, w);
        if (t > 0) {
            load_ring4(zi, u0, s, z);
            d4 = load4(v.d + u0);
            y4 = load4(v.y + u0);
        }
    };
    if (m < end) load();
    double al = 0.0, be = 0.0, gamma = 0.0;
    if (t >= 0) {
        gamma = sum_parts(pin + PART_GS, gridDim.x);
        double den = sum_parts(pin + PART_DZ, gridDim.x);
        if (t > 0) {
            const double go = scratch[PCG_GS + ((t - 1) & 3)], ao = scratch[PCG_AL + ((t - 1) & 3)];
            be = go != 0.0 ? gamma / go : 0.0;
            if (ao != 0.0) den -= be * gamma / ao;
        }
        al = den != 0.0 ? gamma / den : 0.0;
    }
    const T alpha = (T)al, beta = (T)be;
    double gs = 0, gg = 0, dz = 0;
    while (m < end) {
        const unsigned u0 = 4u * (unsigned)m;
        T zn[4], gn[4], wn[4], dn[4], yn[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            zn[q] = -w.c.a[q] + beta * z.c.a[q];
            dn[q] = -(mreg * g.c.a[q]) + beta * d4.a[q];
            yn[q] = y4.a[q] + alpha * dn[q];
        }
        // the new g around the group, then u = M g in its place
        auto next = [&](T& gv, T wv, T zv) { gv = mreg * (gv + alpha * (-wv + beta * zv)); };
        T gc[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            gc[q] = g.c.a[q] + alpha * zn[q];
            g.c.a[q] = mreg * gc[q];
            next(g.ym.a[q], w.ym.a[q], z.ym.a[q]);
            next(g.yp.a[q], w.yp.a[q], z.yp.a[q]);
            next(g.zm.a[q], w.zm.a[q], z.zm.a[q]);
            next(g.zp.a[q], w.zp.a[q], z.zp.a[q]);
        }
        next(g.l, w.l, z.l);
        next(g.r, w.r, z.r);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const T u = g.c.a[q];
            T ju = type_at(t4, q) == NT_REG ? ring_A(g, q, s) : u;
            if (v.P) ju -= (T)v.P[u0 + q] * u;
            wn[q] = ju;
            gn[q] = gc[q];
            gs += (double)gn[q] * (double)u;
            gg += (double)gn[q] * (double)gn[q];
            dz += (double)ju * (double)u;
        }
        store4(v.w[to] + u0, wn);
        if (t >= 0) {
            store4(v.g[to] + u0, gn);
            store4(v.z[to] + u0, zn);
            store4(v.d + u0, dn);
            store4(v.y + u0, yn);
        }
        m += BLOCK;
        if (m < end) load();
    }
    if (blockIdx.x == 0 && threadIdx.x < (unsigned)(s.nn & 3)) {  // corner nodes past the last group: all zero
        const long long u = (s.nn & ~3ll) + threadIdx.x;
        v.w[to][u] = 0;
        if (t >= 0) {
            v.g[to][u] = 0;
            v.z[to][u] = 0;
            v.y[u] = 0;
        }
    }
    const double a = block_sum(gs), b = block_sum(gg), c = block_sum(dz);
    if (threadIdx.x == 0) {
        if (t >= 0) {
            pout[PART_GS + blockIdx.x] = a;
            pout[PART_GG + blockIdx.x] = b;
        }
        pout[PART_DZ + blockIdx.x] = c;
    }
    if (blockIdx.x == 0 && t >= 0) {
        const double g0 = sum_parts(pin + PART_GG, gridDim.x);
        if (threadIdx.x == 0) {
            scratch[PCG_GS + (t & 3)] = gamma;
            scratch[PCG_AL + (t & 3)] = al;
            ggh[t] = g0;
        }
    }
}

// The end of a batch of iterations (t0, t1]: g.g of each to the host (pinned
// memory), and the stop flag when one is within the target.
__global__ void __launch_bounds__(BLOCK)
    k_pcg_check(double* __restrict__ scratch, const double* __restrict__ gg1, const double* __restrict__ ggh, int nb,
                int t0, int t1, double target2, double* host) {
    if (scratch[PCG_FLAG] != 0.0) return;
    const double gg = sum_parts(gg1, nb);  // of iteration t1
    __shared__ int hit;
    if (threadIdx.x == 0) hit = 0;
    __syncthreads();
    for (int q = t0 + 1 + threadIdx.x; q <= t1; q += BLOCK) {
        const double x = q == t1 ? gg : ggh[q];
        host[q - t0 - 1] = x;
        if (x <= target2) hit = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0 && hit) scratch[PCG_FLAG] = 1.0;
}

// phi -= y on non-Dirichlet rows (PotentialSolver.cpp:225-228); with part,
// the partial sums of y.y over them
template <typename T>
__global__ void __launch_bounds__(BLOCK)
    k_update_phi(Stencil s, const uint8_t* __restrict__ nt, double* __restrict__ phi,
                 const T* __restrict__ y, double* __restrict__ part) {
    double yy = 0;
    long long end;
    for (long long u = chunk_begin(s.nn, end) + threadIdx.x; u < end; u += BLOCK) {
        if (nt[u] == NT_DIR) continue;
        double yv = (double)y[u];
        phi[u] -= yv;
        yy += yv * yv;
    }
    if (!part) return;
    double a = block_sum(yy);
    if (threadIdx.x == 0) part[blockIdx.x] = a;
}

}  // namespace

// The iterations of PCG on J y = F after k_F's set-up (vectors of type T, g.g
// = gg0 > target2); stops at the end of the first batch of `check` iterations
// in which g.g reached target2, or at max_it.  The host queues the first
// RUN_AHEAD iterations of the next batch before it waits for one, so the
// device never idles during a check; once a batch has converged the kernels
// behind it return at once (the stop flag), so y is the one of the batch that
// converged.  hp: 2 * check doubles of pinned memory; ggh: max_it + 1 doubles
// on the device.
template <typename T, bool NEU>
static int pcg_inner(pic_ctx* ctx, const Stencil& s, const PcgVec<T>& v, T* d0, T* d1, const CgVec<T>* cg, double* ggh,
                     double* hp, double target2, int max_it, int check, int* iters) {
    const unsigned nb = part_blocks(s.nn);
    if (cg) k_cg<T><<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, *cg, ctx->scratch, ggh, -1);
    for (auto& e : ctx->batch_ev)
        if (!e) PIC_HIP(ctx, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    // profiled runs wait for every batch, so that no returned-at-once
    // iteration is counted
    const int ahead = ctx->prof.on ? 1 : 2;
    int t = 0;                        // iterations queued
    int beg[2], end[2], queued = 0, done = 0;  // batches queued and waited for
    T *dold = d0, *dnew = d1;
    bool conv = false;
    auto wait_oldest = [&]() {  // for the oldest queued batch; conv: it reached target2
        const int q = done & 1;
        const hipError_t e = pic_spin_event(ctx->batch_ev[q]);
        if (e != hipSuccess) return pic_hip_check(ctx, e, "PCG check");
        done++;
        const volatile double* h = hp + (size_t)q * check;
        for (int m = 0; m < end[q] - beg[q]; m++) {
            if (!(h[m] == h[m])) return pic_fail(ctx, PIC_ERR_NUMERIC, "PCG produced NaN");
            if (h[m] <= target2) {
                *iters = end[q];
                conv = true;
                break;
            }
        }
        return (int)PIC_OK;
    };
    for (;;) {
        while (t < max_it && queued - done < ahead) {
            const int q = queued & 1, t0 = t, upto = check < max_it - t ? t + check : max_it;
            for (; t < upto; t++) {  // one profiled "launch" = one PCG iteration (1 or 2 kernels)
                if (t - t0 == RUN_AHEAD && queued > done) {
                    const int rc = wait_oldest();
                    if (rc || conv) return rc;
                }
                PicProfScope ps(ctx, PIC_K_PCG);
                if (cg) {
                    k_cg<T><<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, *cg, ctx->scratch, ggh, t);
                    continue;
                }
                k_pcg1<T, NEU><<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, v, dold, dnew, ctx->scratch, ggh, t);
                k_pcg2<T, NEU><<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, v, dnew, ctx->scratch, t);
                std::swap(dold, dnew);
            }
            k_pcg_check<<<1, BLOCK, 0, ctx->stream>>>(ctx->scratch,
                                                      ctx->scratch + (cg ? (t & 1) * PART_SET : 0) + PART_GG, ggh,
                                                      (int)nb, t0, t, target2, hp + (size_t)q * check);
            PIC_HIP(ctx, hipGetLastError());
            PIC_HIP(ctx, hipEventRecord(ctx->batch_ev[q], ctx->stream));
            beg[q] = t0;
            end[q] = t;
            queued++;
        }
        if (done == queued) {
            *iters = t;
            return PIC_NOT_CONVERGED;
        }
        const int rc = wait_oldest();
        if (rc || conv) return rc;
    }
}

// Nodes up to which an iteration is one kernel (k_cg): one launch's latency
// against three stencil operands instead of one.  Cold solves, two kernels and
// one: FP32-inner 33^3 1.61 and 1.24 ms, 64^3 3.06 and 2.26, a run on 97 x 65 x 49
// 16.3 and 14.4, 100^3 6.5 and 7.5; FP64 33^3 1.37 and 1.13, 50^3 1.84 and 1.60, 70^3
// 3.44 and 3.28, 90^3 5.3 and 6.4.
template <typename T>
constexpr size_t CG_ONE_MAX = sizeof(T) == sizeof(float) ? (size_t)1 << 19 : (size_t)3 << 17;

// Newton + PCG (PotentialSolver.cpp:178-241).  The linear case (n0 == 0)
// needs a single Newton step; each Newton step restarts PCG from y = 0.
template <typename T, bool NEU>
static int solve_pcg_t(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st) {
    const GridC& g = ctx->g;
    constexpr bool mixed = sizeof(T) == sizeof(float);
    size_t nn = (size_t)g.nn;
    Stencil s = make_stencil(g, (p->flags & PIC_SOLVE_AXIS_SWAP) != 0);
    bool nonlinear = p->n0 != 0.0;
    int max_it = p->max_it > 0 ? p->max_it : 10000;
    int check = std::min(p->check_every > 0 ? p->check_every : 8, max_it);
    // y, g, d0, d1, z (s), P, the g.g history; each vector on a 256-byte line
    const size_t vs = (nn * sizeof(T) + 255) & ~(size_t)255;
    const size_t ps = nonlinear ? (nn * sizeof(double) + 255) & ~(size_t)255 : 0;
    const bool one = !NEU && nn <= CG_ONE_MAX<T>;  // one kernel per iteration (k_cg)
    const int nvec = NEU ? 6 : one ? 8 : 5;
    int rc = pic_ensure_work(ctx, nvec * vs + ps + ((size_t)max_it + 2) * sizeof(double));
    if (rc) return rc;
    rc = pic_ensure_pin(ctx, (8 + 2 * (size_t)check) * sizeof(double));
    if (rc) return rc;
    char* wbase = (char*)ctx->work;
    auto vec = [&](int q) { return reinterpret_cast<T*>(wbase + q * vs); };
    double* P = nonlinear ? (double*)(wbase + nvec * vs) : nullptr;
    double* ggh = (double*)(wbase + nvec * vs + ps);
    PcgVec<T> v;
    v.y = vec(0);
    v.g = vec(1);
    v.z = vec(4);
    v.s = NEU ? vec(5) : nullptr;
    v.P = P;
    // k_cg's vectors: g's first is k_F's g
    const CgVec<T> cg{vec(0), vec(2), {vec(1), vec(3)}, {vec(4), vec(5)}, {vec(6), vec(7)}, P};
    volatile double* hp = ctx->pin;  // [0, 5) sums of k_F, [5] y.y, [8, ...) g.g of the batches
    NewtonArgs na;
    na.ieps = 1.0 / EPS0;
    na.phi0 = p->phi0;
    na.n0 = p->n0;
    na.inv_te0 = 1.0 / (p->Te0 != 0 ? p->Te0 : 1.0);
    const unsigned nb = part_blocks(s.nn);
    int total_it = 0, newton = 0;
    bool conv = false, have_r = false;
    double fr[3];
    const int newton_max = nonlinear ? 20 : 1000;  // PotentialSolver.cpp:179
    for (newton = 0; newton < newton_max; newton++) {
        // set-up launches are not counted as PCG iterations
        k_F<T, true, NEU><<<nb, BLOCK, 0, ctx->stream>>>(s, na, ctx->ntype, ctx->phi, ctx->rho, v.g, v.s, P,
                                                         ctx->scratch);
        // F.F (all rows, regular), b.b, and PCG's g.s, g.g
        k_sum_parts<<<5, BLOCK, 0, ctx->stream>>>(ctx->scratch + PART_F, (int)nb, ctx->pin);
        PIC_HIP(ctx, hipGetLastError());
        PIC_HIP(ctx, pic_spin_wait(ctx->stream));
        for (int q = 0; q < 3; q++) fr[q] = hp[q];
        const double gg0 = hp[4];
        // target on the inner residual g (g = -F at y = 0)
        double target2;
        if (p->tol_kind == PIC_TOL_REF_RMS)
            target2 = p->tol * p->tol * (double)nn;
        else
            target2 = p->tol * p->tol * (fr[2] > 0 ? fr[2] : 1.0);
        if (!nonlinear && fr[0] <= target2) {
            conv = have_r = true;
            break;
        }
        // relative criterion on the nonlinear problem: the FP64 residual F
        // of the current phi over the regular rows (the Newton iterate is
        // judged by the residual, not by the size of its last step)
        if (nonlinear && p->tol_kind == PIC_TOL_REL && fr[1] <= target2) {
            conv = have_r = true;
            break;
        }
        double inner_target2 = target2;
        if (mixed) {  // FP32 inner solve: reduce the residual by ~1e-3 per pass
            double floor2 = fr[0] * 1e-6;
            inner_target2 = std::max(target2 * 0.25, floor2);
        } else if (nonlinear && p->tol_kind == PIC_TOL_REL) {
            // inexact Newton: each linear solve to 1e-4 of the current
            // residual, or below the final tolerance
            inner_target2 = std::max(target2 * 0.25, fr[0] * 1e-8);
        }
        double yy = 0;
        if (!(gg0 <= inner_target2)) {  // otherwise y = 0 (a zero right-hand side included)
            int its = 0;
            rc = pcg_inner<T, NEU>(ctx, s, v, vec(2), vec(3), one ? &cg : nullptr, ggh, ctx->pin + 8, inner_target2,
                                   max_it - total_it, check, &its);
            total_it += its;
            if (rc < 0) return rc;
            const bool want_yy = nonlinear && p->tol_kind == PIC_TOL_REF_RMS;
            k_update_phi<T><<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, ctx->phi, v.y,
                                                           want_yy ? ctx->scratch + PART_F : nullptr);
            PIC_HIP(ctx, hipGetLastError());
            if (want_yy) {
                k_sum_parts<<<1, BLOCK, 0, ctx->stream>>>(ctx->scratch + PART_F, (int)nb, ctx->pin + 5);
                PIC_HIP(ctx, hipGetLastError());
                PIC_HIP(ctx, pic_spin_wait(ctx->stream));
                yy = hp[5];
            }
        }
        if (nonlinear && p->tol_kind == PIC_TOL_REF_RMS) {
            if (std::sqrt(yy / (double)nn) < 1e-3) {  // NR_TOL, PotentialSolver.cpp:180, :229-233
                conv = true;
                newton++;
                break;
            }
        }
        if (total_it >= max_it) break;
    }
    double r[3];
    if (have_r && !NEU) {  // k_F's sums are the residual of the final phi
        for (int q = 0; q < 3; q++) r[q] = fr[q];
    } else {
        SorArgs a;
        a.omega = 1;
        a.ieps = 1.0 / EPS0;
        a.itwos = 1.0 / s.twos;
        a.phi0 = p->phi0;
        a.n0 = p->n0;
        a.inv_te0 = na.inv_te0;
        rc = residual_norms(ctx, s, a, r);
        if (rc) return rc;
    }
    st->converged = conv;
    st->iterations = total_it;
    st->newton_iterations = newton;
    st->ref_l2 = std::sqrt(r[0] / (double)nn);
    st->rel_residual = r[2] > 0 ? std::sqrt(r[1] / r[2]) : std::sqrt(r[1]);
    return conv ? PIC_OK : PIC_NOT_CONVERGED;
}

int pic_solve_pcg(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st, bool mixed) {
    if (has_neumann(ctx))
        return mixed ? solve_pcg_t<float, true>(ctx, p, st) : solve_pcg_t<double, true>(ctx, p, st);
    return mixed ? solve_pcg_t<float, false>(ctx, p, st) : solve_pcg_t<double, false>(ctx, p, st);
}

int pic_newton_residual(pic_ctx* ctx, const Stencil& s, const NewtonArgs& a, double* F, double* P, double* sums) {
    const unsigned nb = part_blocks(s.nn);
    k_F<double, false, false><<<nb, BLOCK, 0, ctx->stream>>>(s, a, ctx->ntype, ctx->phi, ctx->rho, F, nullptr, P,
                                                             ctx->scratch);
    k_sum_parts<<<3, BLOCK, 0, ctx->stream>>>(ctx->scratch + PART_F, (int)nb, sums);
    PIC_HIP(ctx, hipGetLastError());
    return PIC_OK;
}

int pic_newton_update(pic_ctx* ctx, const Stencil& s, const double* y, double* sum) {
    const unsigned nb = part_blocks(s.nn);
    k_update_phi<double><<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, ctx->phi, y, ctx->scratch + PART_F);
    k_sum_parts<<<1, BLOCK, 0, ctx->stream>>>(ctx->scratch + PART_F, (int)nb, sum);
    PIC_HIP(ctx, hipGetLastError());
    return PIC_OK;
}
