// pic_solver.hip -- field solve of the gfx950 PIC library: the entry point, the
// E-field and the learned solver (pic_sor.hip and pic_pcg.hip: the others).
//
//   k_efield     E = -grad(phi), FP64 math, FP32 float4 output
//                (PotentialSolver.cpp:354-408)
//   k_fcg_*      flexible CG with the learned two-level preconditioner
#include <vector>

#include "pic_stencil.h"

namespace {

// Node pairs (2h, 2h+1) of every i-line, XCD-contiguous chunks per
// workgroup: f(u, second, red) for the pair's first node u, whether the
// second node exists (odd ni) and whether the first node is red
// ((i + j + k) even; the second node has the other colour).  One (j, k)
// division per pair; a wave's lanes never diverge on the colour.
__device__ inline unsigned pair_count(const Stencil& s) {
    return (unsigned)((s.ni + 1) / 2) * (unsigned)s.nj * (unsigned)s.nk;
}
template <typename F>
__device__ inline void for_pairs(const Stencil& s, F f) {
    const unsigned half = (unsigned)(s.ni + 1) >> 1;
    long long end;
    for (long long m = chunk_begin(pair_count(s), end) + threadIdx.x; m < end; m += BLOCK) {
        unsigned row = (unsigned)m / half;
        unsigned h = (unsigned)m - row * half;
        unsigned k = row / (unsigned)s.nj;
        unsigned j = row - k * (unsigned)s.nj;
        unsigned u = row * (unsigned)s.ni + 2 * h;
        f(u, 2 * h + 1 < (unsigned)s.ni, ((j + k) & 1u) == 0);
    }
}

// ------------------------------------------------------------------------
// E-field
// ------------------------------------------------------------------------
__device__ inline void efield_node(const GridC& g, const double* __restrict__ phi, float4* __restrict__ ef,
                                   long long u, float (&e)[3]) {
    unsigned uu = (unsigned)u, row = uu / (unsigned)g.ni, kk = row / (unsigned)g.nj;
    int i = (int)(uu - row * (unsigned)g.ni), j = (int)(row - kk * (unsigned)g.nj), k = (int)kk;
    int ijk[3] = {i, j, k};
    int n[3] = {g.ni, g.nj, g.nk};
    long long st[3] = {1, g.ni, (long long)g.ni * g.nj};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double inv2 = 1.0 / (2 * g.dx[d]);
        long long s = st[d];
        double v;
        if (ijk[d] == 0)
            v = (3 * phi[u] - 4 * phi[u + s] + phi[u + 2 * s]) * inv2;
        else if (ijk[d] == n[d] - 1)
            v = (-phi[u - 2 * s] + 4 * phi[u - s] - 3 * phi[u]) * inv2;
        else
            v = (phi[u - s] - phi[u + s]) * inv2;
        e[d] = (float)v;
    }
    ef[u] = make_float4(e[0], e[1], e[2], 0.f);
}

// a few nodes per thread (grid-stride): one maximum reduction per workgroup
__global__ void __launch_bounds__(BLOCK)
    k_efield(GridC g, const double* __restrict__ phi, float4* __restrict__ ef, float* __restrict__ emax) {
    float m[3] = {0.f, 0.f, 0.f};
    for (long long u = (long long)blockIdx.x * BLOCK + threadIdx.x; u < g.nn; u += (long long)gridDim.x * BLOCK) {
        float e[3];
        efield_node(g, phi, ef, u, e);
#pragma unroll
        for (int d = 0; d < 3; d++) m[d] = fmaxf(m[d], fabsf(e[d]));
    }
    block_max3_to(m[0], m[1], m[2], emax);  // the push's bound on the kick
}


// warm start of a time loop's solve: phi = 2 phi - prev, prev = the old phi
__global__ void __launch_bounds__(BLOCK)
    k_extrapolate(long long n, double* __restrict__ phi, double* __restrict__ prev) {
    long long end;
    for (long long m = chunk_begin(n, end) + threadIdx.x; m < end; m += BLOCK) {
        const double p = phi[m];
        phi[m] = 2.0 * p - prev[m];
        prev[m] = p;
    }
}

// kernels ending in a single-address grid-wide sum: fewer, longer workgroups
// (eight items per thread) keep the per-workgroup atomics few
unsigned stencil_blocks_red(long long items) {
    long long b = (items + BLOCK * 8 - 1) / (BLOCK * 8);
    if (b > 2048) b = 2048;
    b = (b + NXCD - 1) / NXCD * NXCD;
    return (unsigned)b;
}

// workgroups of the node-pair kernels (for_pairs): one pair per thread
// (measured faster than two)
unsigned pair_blocks(const Stencil& s) { return stencil_blocks(s.nn); }

}  // namespace

// ------------------------------------------------------------------------
extern "C" int pic_efield(pic_ctx* ctx) {
    if (!ctx) return PIC_ERR_ARG;
    {
        PicProfScope ps(ctx, PIC_K_EFIELD);
        PIC_HIP(ctx, hipMemsetAsync(ctx->emax, 0, 4 * sizeof(float), ctx->stream));
        k_efield<<<std::min(grid_for((size_t)ctx->g.nn, BLOCK), 2048u), BLOCK, 0, ctx->stream>>>(
            ctx->g, ctx->phi, ctx->ef, ctx->emax);
    }
    PIC_HIP(ctx, hipGetLastError());
    return PIC_OK;
}

// ------------------------------------------------------------------------
// Flexible CG with the learned two-level preconditioner.  FCG(1) (Notay
// 2000): p_k = z_k - (z_k.A p_{k-1}) / (p_{k-1}.A p_{k-1}) p_{k-1}, which keeps
// CG's descent when the preconditioner varies from step to step.  On a cold
// start (phi = 0) the first step's correction is the preconditioned residual
// -- the network's prediction -- scaled by the optimal step length, so the
// network supplies the initial guess.  Scalars stay on the device in
// per-iteration history slots; the host reads the residual history every
// few iterations.  Plain PCG is the fallback and the final residual is
// recomputed in FP64.
//
// Preconditioner M(r): LEARNED_PRE_SWEEPS red-black Gauss-Seidel sweeps on
// A z = r from z = 0 (red, black), the network's coarse correction of the
// remaining residual, LEARNED_POST_SWEEPS sweeps in the reverse colour order
// (black, red).  A sweep costs ~17 us at 128^3, an iteration ~290 us: three
// sweeps on each side take the 128^3 time loop's solves from 5 iterations
// (one sweep each side) to 2 and cold solves from 11 to 6.  The sweeps after
// the first and the output z are stored in FP32 (FP64 arithmetic).
// ------------------------------------------------------------------------
bool pic_unet_ready(pic_ctx* ctx);
int pic_unet_coarse_correct(pic_ctx* ctx, const float* t, const float* z, float* c, float* res,
                            double* ws, const double* P);

namespace {

constexpr int LEARNED_PRE_SWEEPS = 3, LEARNED_POST_SWEEPS = 3;

// per-iteration striped scalars (slot k at base + k * SSIZE)
struct FcgHist {
    double* rz;  // r_k . z_k
    double* pq;  // p_k . A p_k
    double* zq;  // z_{k+1} . A p_k
    double* rr;  // r_{k+1} . r_{k+1}
};

// The neighbour offsets of node u clamped only at the array's ends: the full
// offsets on every regular (interior) node, in bounds on every node, and
// independent of the node type, so a kernel's neighbour loads are issued
// together with its node-type load instead of after it (values on
// non-regular nodes are discarded)
struct NbrOff {
    unsigned mi, pi, mj, pj, mk, pk;
};
__device__ inline NbrOff nbr_off(const Stencil& s, unsigned u) {
    const unsigned n = (unsigned)s.nn, sj = (unsigned)s.sj, sk = (unsigned)s.sk;
    NbrOff o;
    o.mi = u >= 1u ? 1u : 0u;
    o.pi = u + 1u < n ? 1u : 0u;
    o.mj = u >= sj ? sj : 0u;
    o.pj = u + sj < n ? sj : 0u;
    o.mk = u >= sk ? sk : 0u;
    o.pk = u + sk < n ? sk : 0u;
    return o;
}
// 7-point neighbour sum of f at node u, weighted per axis, with nbr_off's
// offsets (the full stencil on regular nodes)
template <typename F>
__device__ inline double nbr_sum_any(const Stencil& s, unsigned u, F f) {
    const NbrOff o = nbr_off(s, u);
    return (f(u - o.mi) + f(u + o.pi)) * s.cx + (f(u - o.mj) + f(u + o.pj)) * s.cy +
           (f(u - o.mk) + f(u + o.pk)) * s.cz;
}

// r = b - A phi on regular rows (0 elsewhere); out += {r.r, b.b, #(phi != 0)}
__global__ void __launch_bounds__(BLOCK)
    k_fcg_resid(Stencil s, const uint8_t* __restrict__ nt, const double* __restrict__ phi,
                const double* __restrict__ rho, double ieps, double* __restrict__ r,
                double* __restrict__ out) {
    double rr = 0, bb = 0, cold = 0;
    auto ph = [&](unsigned w) { return phi[w]; };
    long long end;
    for (long long m = chunk_begin(s.nn, end) + threadIdx.x; m < end; m += BLOCK) {
        const unsigned u = (unsigned)m;
        const bool reg = nt[u] == NT_REG;  // regular nodes are interior (Dirichlet walls)
        const double pu = phi[u];
        const double b = -rho[u] * ieps;
        const double rv = reg ? b - (nbr_sum_any(s, u, ph) - s.twos * pu) : 0.0;
        if (reg) {
            bb += b * b;
            cold += pu != 0.0;
        }
        r[u] = rv;
        rr += rv * rv;
    }
    double a = block_sum(rr), b2 = block_sum(bb), c = block_sum(cold);
    if (threadIdx.x == 0) {  // striped: out, out + SSIZE, out + 2 SSIZE
        sadd(out, a);
        sadd(out + SSIZE, b2);
        sadd(out + 2 * SSIZE, c);
    }
}

// p_k = z_k + beta p_{k-1} (beta = -zq[k-1] / pq[k-1]; p_0 = z_0), q = A p_k on
// regular rows (by the recurrence A p_k = A z_k + beta A p_{k-1}); pq[k] +=
// p_k.q.  z and p vanish on non-regular nodes, and
// regular nodes are interior (Dirichlet walls), so q is the 7-point stencil.
// Neighbour offsets are zeroed on non-regular nodes so that every load is in
// bounds and the loop has no branches.
__global__ void __launch_bounds__(BLOCK)
    k_fcg_pq(Stencil s, const uint8_t* __restrict__ nt, const float* __restrict__ z,
             const double* __restrict__ pold, double* __restrict__ pnew, double* __restrict__ q,
             FcgHist h, int k, const double* __restrict__ P) {
    double beta = 0.0;
    if (k > 0) {
        double den = sget(h.pq + (k - 1) * SSIZE);
        beta = den != 0.0 ? -sget(h.zq + (k - 1) * SSIZE) / den : 0.0;
    }
    const bool first = k == 0;
    double acc = 0;
    long long end;
    for (long long m = chunk_begin(s.nn, end) + threadIdx.x; m < end; m += BLOCK) {
        const unsigned u = (unsigned)m;
        const bool reg = nt[u] == NT_REG;
        const NbrOff o = nbr_off(s, u);
        // q = A p = A z + beta A p_old: the stencil of z alone (seven loads
        // instead of fourteen), the previous q in place
        const double zu = z[u];
        double az = ((double)z[u - o.mk] + z[u + o.pk]) * s.cz + ((double)z[u - o.mj] + z[u + o.pj]) * s.cy +
                    ((double)z[u - o.mi] + z[u + o.pi]) * s.cx - s.twos * zu;
        if (P) az -= P[u] * zu;  // J = A - diag(P) (the Newton Jacobian)
        double pu = zu, qv = az;
        if (!first) {
            pu += beta * pold[u];
            qv += beta * q[u];
        }
        qv = reg ? qv : 0.0;
        pnew[u] = pu;
        q[u] = qv;
        acc += pu * qv;
    }
    double a = block_sum(acc);
    if (threadIdx.x == 0) sadd(h.pq + k * SSIZE, a);
}

// alpha = rz[k] / pq[k]; x += alpha p; r -= alpha q; rr[k] += r.r
__global__ void __launch_bounds__(BLOCK)
    k_fcg_update(long long n, FcgHist h, int k, double* __restrict__ x, const double* __restrict__ p,
                 double* __restrict__ r, const double* __restrict__ q) {
    double den = sget(h.pq + k * SSIZE);
    double alpha = den != 0.0 ? sget(h.rz + k * SSIZE) / den : 0.0;
    double rr = 0;
    long long end;
    for (long long m = chunk_begin(n, end) + threadIdx.x; m < end; m += BLOCK) {
        const unsigned u = (unsigned)m;
        x[u] += alpha * p[u];
        double rv = r[u] - alpha * q[u];
        r[u] = rv;
        rr += rv * rv;
    }
    double a = block_sum(rr);
    if (threadIdx.x == 0) sadd(h.rr + k * SSIZE, a);
}


// One red-black Gauss-Seidel sweep on A z = r from z = 0, in one pass: the
// red half-sweep gives z = -r / (2 sum 1/dx^2) on red regular nodes
// ((i + j + k) even); the black half-sweep that follows reads only those red
// values, so it is written directly in r.  Non-regular nodes get 0.  z is
// FP32 (the preconditioner's vectors are stored in FP32, its arithmetic is
// FP64); r32 (optional) receives r in FP32 for the closing sweeps.
// 1 / the diagonal of the operator's regular row: 2 sum 1/dx^2, plus P_u
// for the Newton Jacobian J = A - diag(P)
__device__ inline double inv_diag(const Stencil& s, const double* __restrict__ P, unsigned u) {
    return P ? 1.0 / (s.twos + P[u]) : s.itwos;
}

__global__ void __launch_bounds__(BLOCK)
    k_presmooth(Stencil s, const uint8_t* __restrict__ nt, const double* __restrict__ r,
                float* __restrict__ z, double* __restrict__ clear, int nclear,
                const double* __restrict__ P, float* __restrict__ r32) {
    // the coarse correction's striped sums start from zero (no memset node)
    for (int q = blockIdx.x * BLOCK + threadIdx.x; q < nclear; q += gridDim.x * BLOCK) clear[q] = 0.0;
    // r / diag on regular nodes, 0 elsewhere (a red value is -that)
    auto rr = [&](unsigned v) {
        double rv = r[v] * inv_diag(s, P, v);
        return nt[v] == NT_REG ? rv : 0.0;
    };
    auto node = [&](unsigned u, bool red) {
        const bool reg = nt[u] == NT_REG;
        const double id = inv_diag(s, P, u);
        double zu;
        if (red)
            zu = -r[u] * id;
        else
            zu = (-nbr_sum_any(s, u, rr) - r[u]) * id;
        z[u] = reg ? (float)zu : 0.f;
        if (r32) r32[u] = (float)r[u];
    };
    for_pairs(s, [&](unsigned u, bool second, bool red) {
        node(u, red);
        if (second) node(u + 1, !red);
    });
}

// The closing red half-sweep of the preconditioner fused with FCG's dot
// products: red regular nodes get the Gauss-Seidel update (their neighbours
// are black and final); then zq += z.q (when q is given) and rz += z.r.
// z vanishes on non-regular nodes.  z and r in FP32 (r32: r rounded), the
// sums in FP64 of the stored values.
__global__ void __launch_bounds__(BLOCK)
    k_gs_red_dots(Stencil s, const uint8_t* __restrict__ nt, const float* __restrict__ r,
                  float* __restrict__ z, const double* __restrict__ q, double* __restrict__ zq,
                  double* __restrict__ rz, const double* __restrict__ P) {
    double a = 0, b = 0;
    auto zv = [&](unsigned w) { return (double)z[w]; };
    auto node = [&](unsigned u, bool red) {
        double zu = z[u];
        if (red) {
            const bool reg = nt[u] == NT_REG;
            double upd = (nbr_sum_any(s, u, zv) - (double)r[u]) * inv_diag(s, P, u);
            if (reg) {
                const float zf = (float)upd;
                z[u] = zf;
                zu = zf;
            }
        }
        if (q) a += zu * q[u];
        b += zu * (double)r[u];
    };
    for_pairs(s, [&](unsigned u, bool second, bool red) {
        node(u, red);
        if (second) node(u + 1, !red);
    });
    double ta = block_sum(a), tb = block_sum(b);
    if (threadIdx.x == 0) {
        if (zq) sadd(zq, ta);
        sadd(rz, tb);
    }
}

// the coarse correction fused with the next (black) half-sweep:
// z = zin + omega c on red nodes, the Gauss-Seidel update from those values on
// black regular nodes, 0 on non-regular nodes; omega = d[0] / d[1] (A-norm
// optimal step along c).  zin and c (FP32) vanish on non-regular nodes; r
// and z in FP32.
__global__ void __launch_bounds__(BLOCK)
    k_gs_corr(Stencil s, const uint8_t* __restrict__ nt, const float* __restrict__ r,
              const float* __restrict__ zin, const float* __restrict__ c,
              const double* __restrict__ d, float* __restrict__ z, const double* __restrict__ P) {
    const double d1 = sget(d + SSIZE);
    const double om = d1 != 0.0 ? sget(d) / d1 : 0.0;
    auto zc = [&](unsigned w) { return (double)zin[w] + om * c[w]; };
    auto node = [&](unsigned u, bool red) {
        const bool reg = nt[u] == NT_REG;
        double zu;
        if (red)
            zu = zc(u);
        else
            zu = (nbr_sum_any(s, u, zc) - (double)r[u]) * inv_diag(s, P, u);
        z[u] = reg ? (float)zu : 0.f;
    };
    for_pairs(s, [&](unsigned u, bool second, bool red) {
        node(u, red);
        if (second) node(u + 1, !red);
    });
}

// one Gauss-Seidel half-sweep in place: the regular nodes of one colour
// (red: (i + j + k) even) get (sum of neighbours - r) / diag; their
// neighbours have the other colour, so the update is race-free.  r in FP32
// (the solver's rounded copy) or FP64.
template <typename RT>
__global__ void __launch_bounds__(BLOCK)
    k_gs_half(Stencil s, const uint8_t* __restrict__ nt, const RT* __restrict__ r,
              float* __restrict__ z, int red_colour, const double* __restrict__ P) {
    auto zv = [&](unsigned w) { return (double)z[w]; };
    auto node = [&](unsigned u, bool red) {
        if (red != (red_colour != 0)) return;
        const double upd = (nbr_sum_any(s, u, zv) - (double)r[u]) * inv_diag(s, P, u);
        if (nt[u] == NT_REG) z[u] = (float)upd;
    };
    for_pairs(s, [&](unsigned u, bool second, bool red) {
        node(u, red);
        if (second) node(u + 1, !red);
    });
}

// k_gs_half<float> on four consecutive nodes of an i-line per thread (ni a
// multiple of 4): the z rows around the group come in 16-byte loads (the
// i-neighbours at the group's ends as single words), r and the node types
// likewise, and the group goes back in one 16-byte store with the other
// colour's two values unchanged.  The same arithmetic as k_gs_half (equal
// bit for bit); every value an update reads has the other colour, which no
// thread writes.
__global__ void __launch_bounds__(BLOCK)
    k_gs_half4(Stencil s, const uint8_t* __restrict__ nt, const float* __restrict__ r,
               float* __restrict__ z, int red_colour, const double* __restrict__ P) {
    const long long ng = s.nn / 4;
    const unsigned n = (unsigned)s.nn, sj = (unsigned)s.sj, sk = (unsigned)s.sk;
    const unsigned want = red_colour ? 0u : 1u;  // parity (i + j + k) & 1 of the updated nodes
    long long end;
    for (long long m = chunk_begin(ng, end) + threadIdx.x; m < end; m += BLOCK) {
        const unsigned u0 = 4u * (unsigned)m;
        const unsigned row = u0 / (unsigned)s.ni;
        const unsigned i0 = u0 - row * (unsigned)s.ni;
        const unsigned k = row / (unsigned)s.nj, j = row - k * (unsigned)s.nj;
        const unsigned p0 = (i0 + j + k) & 1u;
        // in-bounds addresses everywhere; only regular (interior) nodes are
        // updated, and their neighbours are the unclamped ones
        const float4 zc = *reinterpret_cast<const float4*>(z + u0);
        const float zl = z[u0 >= 1u ? u0 - 1u : u0];
        const float zr = z[u0 + 4u < n ? u0 + 4u : u0];
        const float4 ym = *reinterpret_cast<const float4*>(z + (u0 >= sj ? u0 - sj : u0));
        const float4 yp = *reinterpret_cast<const float4*>(z + (u0 + sj < n ? u0 + sj : u0));
        const float4 zm = *reinterpret_cast<const float4*>(z + (u0 >= sk ? u0 - sk : u0));
        const float4 zp = *reinterpret_cast<const float4*>(z + (u0 + sk < n ? u0 + sk : u0));
        const float4 r4 = *reinterpret_cast<const float4*>(r + u0);
        const uint32_t t4 = *reinterpret_cast<const uint32_t*>(nt + u0);
        const float c[4] = {zc.x, zc.y, zc.z, zc.w};
        const float xm[4] = {zl, zc.x, zc.y, zc.z}, xp[4] = {zc.y, zc.z, zc.w, zr};
        const float ymv[4] = {ym.x, ym.y, ym.z, ym.w}, ypv[4] = {yp.x, yp.y, yp.z, yp.w};
        const float zmv[4] = {zm.x, zm.y, zm.z, zm.w}, zpv[4] = {zp.x, zp.y, zp.z, zp.w};
        const float rv[4] = {r4.x, r4.y, r4.z, r4.w};
        float out[4];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            out[a] = c[a];
            if (((p0 + (unsigned)a) & 1u) != want || ((t4 >> (8 * a)) & 0xFFu) != (uint32_t)NT_REG) continue;
            const double sum = ((double)xm[a] + (double)xp[a]) * s.cx + ((double)ymv[a] + (double)ypv[a]) * s.cy +
                               ((double)zmv[a] + (double)zpv[a]) * s.cz;
            out[a] = (float)((sum - (double)rv[a]) * inv_diag(s, P, u0 + (unsigned)a));
        }
        *reinterpret_cast<float4*>(z + u0) = make_float4(out[0], out[1], out[2], out[3]);
    }
}

// The four-node forms of k_gs_corr and k_gs_red_dots (ni a multiple of 4):
// a group of four consecutive nodes of an i-line per thread, its
// neighbour rows in 16-byte loads, one 16-byte store; the same arithmetic
// (z equal bit for bit; the dot products sum in another order).
struct Group4 {
    unsigned u0, p0;  // first node, its parity (i + j + k) & 1
    unsigned xm, xp, ym, yp, zm, zp;  // clamped addresses: u0 - 1, u0 + 4, u0 -+ sj, u0 -+ sk
};
__device__ inline Group4 group4(const Stencil& s, long long m) {
    Group4 g;
    const unsigned n = (unsigned)s.nn, sj = (unsigned)s.sj, sk = (unsigned)s.sk;
    g.u0 = 4u * (unsigned)m;
    const unsigned row = g.u0 / (unsigned)s.ni;
    const unsigned i0 = g.u0 - row * (unsigned)s.ni;
    const unsigned k = row / (unsigned)s.nj, j = row - k * (unsigned)s.nj;
    g.p0 = (i0 + j + k) & 1u;
    g.xm = g.u0 >= 1u ? g.u0 - 1u : g.u0;
    g.xp = g.u0 + 4u < n ? g.u0 + 4u : g.u0;
    g.ym = g.u0 >= sj ? g.u0 - sj : g.u0;
    g.yp = g.u0 + sj < n ? g.u0 + sj : g.u0;
    g.zm = g.u0 >= sk ? g.u0 - sk : g.u0;
    g.zp = g.u0 + sk < n ? g.u0 + sk : g.u0;
    return g;
}
// a vector's values around a group: [a] = at u0 + a, xm/xp the i-neighbours
// of node a, ym/yp/zm/zp the rows on either side
struct Around4 {
    float c[4], xm[4], xp[4], ym[4], yp[4], zm[4], zp[4];
};
__device__ inline void load_around4(const float* __restrict__ v, const Group4& g, Around4& a) {
    const float4 c = *reinterpret_cast<const float4*>(v + g.u0);
    const float l = v[g.xm], r = v[g.xp];
    const float4 ym = *reinterpret_cast<const float4*>(v + g.ym);
    const float4 yp = *reinterpret_cast<const float4*>(v + g.yp);
    const float4 zm = *reinterpret_cast<const float4*>(v + g.zm);
    const float4 zp = *reinterpret_cast<const float4*>(v + g.zp);
    const float cc[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        a.c[q] = cc[q];
        a.xm[q] = q == 0 ? l : cc[q - 1];
        a.xp[q] = q == 3 ? r : cc[q + 1];
    }
    a.ym[0] = ym.x; a.ym[1] = ym.y; a.ym[2] = ym.z; a.ym[3] = ym.w;
    a.yp[0] = yp.x; a.yp[1] = yp.y; a.yp[2] = yp.z; a.yp[3] = yp.w;
    a.zm[0] = zm.x; a.zm[1] = zm.y; a.zm[2] = zm.z; a.zm[3] = zm.w;
    a.zp[0] = zp.x; a.zp[1] = zp.y; a.zp[2] = zp.z; a.zp[3] = zp.w;
}
unsigned group4_blocks(const Stencil& s) {
    long long b = (s.nn / 4 + BLOCK - 1) / BLOCK;
    return (unsigned)((b + NXCD - 1) / NXCD * NXCD);
}

__global__ void __launch_bounds__(BLOCK)
    k_gs_corr4(Stencil s, const uint8_t* __restrict__ nt, const float* __restrict__ r,
               const float* __restrict__ zin, const float* __restrict__ c,
               const double* __restrict__ d, float* __restrict__ z, const double* __restrict__ P) {
    const double d1 = sget(d + SSIZE);
    const double om = d1 != 0.0 ? sget(d) / d1 : 0.0;
    long long end;
    for (long long m = chunk_begin(s.nn / 4, end) + threadIdx.x; m < end; m += BLOCK) {
        const Group4 g = group4(s, m);
        Around4 zi, cc;
        load_around4(zin, g, zi);
        load_around4(c, g, cc);
        const float4 r4 = *reinterpret_cast<const float4*>(r + g.u0);
        const uint32_t t4 = *reinterpret_cast<const uint32_t*>(nt + g.u0);
        const float rv[4] = {r4.x, r4.y, r4.z, r4.w};
        auto zc = [&](float a, float b) { return (double)a + om * b; };
        float out[4];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const bool red = ((g.p0 + (unsigned)a) & 1u) == 0u;
            const bool reg = ((t4 >> (8 * a)) & 0xFFu) == (uint32_t)NT_REG;
            double zu;
            if (red)
                zu = zc(zi.c[a], cc.c[a]);
            else
                zu = ((zc(zi.xm[a], cc.xm[a]) + zc(zi.xp[a], cc.xp[a])) * s.cx +
                      (zc(zi.ym[a], cc.ym[a]) + zc(zi.yp[a], cc.yp[a])) * s.cy +
                      (zc(zi.zm[a], cc.zm[a]) + zc(zi.zp[a], cc.zp[a])) * s.cz - (double)rv[a]) *
                     inv_diag(s, P, g.u0 + (unsigned)a);
            out[a] = reg ? (float)zu : 0.f;
        }
        *reinterpret_cast<float4*>(z + g.u0) = make_float4(out[0], out[1], out[2], out[3]);
    }
}

__global__ void __launch_bounds__(BLOCK)
    k_gs_red_dots4(Stencil s, const uint8_t* __restrict__ nt, const float* __restrict__ r,
                   float* __restrict__ z, const double* __restrict__ q, double* __restrict__ zq,
                   double* __restrict__ rz, const double* __restrict__ P) {
    double acc_a = 0, acc_b = 0;
    long long end;
    for (long long m = chunk_begin(s.nn / 4, end) + threadIdx.x; m < end; m += BLOCK) {
        const Group4 g = group4(s, m);
        Around4 zz;
        load_around4(z, g, zz);
        const float4 r4 = *reinterpret_cast<const float4*>(r + g.u0);
        const uint32_t t4 = *reinterpret_cast<const uint32_t*>(nt + g.u0);
        const float rv[4] = {r4.x, r4.y, r4.z, r4.w};
        double qv[4] = {0, 0, 0, 0};
        if (q) {
            const double2 q0 = *reinterpret_cast<const double2*>(q + g.u0);
            const double2 q1 = *reinterpret_cast<const double2*>(q + g.u0 + 2);
            qv[0] = q0.x; qv[1] = q0.y; qv[2] = q1.x; qv[3] = q1.y;
        }
        float out[4];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            out[a] = zz.c[a];
            const bool red = ((g.p0 + (unsigned)a) & 1u) == 0u;
            const bool reg = ((t4 >> (8 * a)) & 0xFFu) == (uint32_t)NT_REG;
            if (red && reg) {
                const double sum = ((double)zz.xm[a] + (double)zz.xp[a]) * s.cx +
                                   ((double)zz.ym[a] + (double)zz.yp[a]) * s.cy +
                                   ((double)zz.zm[a] + (double)zz.zp[a]) * s.cz;
                out[a] = (float)((sum - (double)rv[a]) * inv_diag(s, P, g.u0 + (unsigned)a));
            }
            const double zu = out[a];
            if (q) acc_a += zu * qv[a];
            acc_b += zu * (double)rv[a];
        }
        *reinterpret_cast<float4*>(z + g.u0) = make_float4(out[0], out[1], out[2], out[3]);
    }
    double ta = block_sum(acc_a), tb = block_sum(acc_b);
    if (threadIdx.x == 0) {
        if (zq) sadd(zq, ta);
        sadd(rz, tb);
    }
}

// The four-node form of k_presmooth without the Jacobian's diagonal (the
// plain operator): r and the node types of the group's neighbour rows in
// 16-byte loads, z and r32 of the group in 16-byte stores; the same
// arithmetic (equal bit for bit).
__device__ inline void load_around4d(const double* __restrict__ v, const Group4& g, double (&c)[4],
                                     double (&xm)[4], double (&xp)[4], double (&ym)[4], double (&yp)[4],
                                     double (&zm)[4], double (&zp)[4]) {
    auto row = [&](unsigned a, double (&o)[4]) {
        const double2 h0 = *reinterpret_cast<const double2*>(v + a);
        const double2 h1 = *reinterpret_cast<const double2*>(v + a + 2);
        o[0] = h0.x; o[1] = h0.y; o[2] = h1.x; o[3] = h1.y;
    };
    row(g.u0, c);
    row(g.ym, ym);
    row(g.yp, yp);
    row(g.zm, zm);
    row(g.zp, zp);
    const double l = v[g.xm], r = v[g.xp];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        xm[q] = q == 0 ? l : c[q - 1];
        xp[q] = q == 3 ? r : c[q + 1];
    }
}
__device__ inline void load_nt4(const uint8_t* __restrict__ nt, const Group4& g, uint32_t (&c)[4],
                                uint32_t (&xm)[4], uint32_t (&xp)[4], uint32_t (&ym)[4], uint32_t (&yp)[4],
                                uint32_t (&zm)[4], uint32_t (&zp)[4]) {
    auto row = [&](unsigned a, uint32_t (&o)[4]) {
        const uint32_t w = *reinterpret_cast<const uint32_t*>(nt + a);
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = (w >> (8 * q)) & 0xFFu;
    };
    row(g.u0, c);
    row(g.ym, ym);
    row(g.yp, yp);
    row(g.zm, zm);
    row(g.zp, zp);
    const uint32_t l = nt[g.xm], r = nt[g.xp];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        xm[q] = q == 0 ? l : c[q - 1];
        xp[q] = q == 3 ? r : c[q + 1];
    }
}

__global__ void __launch_bounds__(BLOCK)
    k_presmooth4(Stencil s, const uint8_t* __restrict__ nt, const double* __restrict__ r,
                 float* __restrict__ z, double* __restrict__ clear, int nclear, float* __restrict__ r32) {
    for (int q = blockIdx.x * BLOCK + threadIdx.x; q < nclear; q += gridDim.x * BLOCK) clear[q] = 0.0;
    long long end;
    for (long long m = chunk_begin(s.nn / 4, end) + threadIdx.x; m < end; m += BLOCK) {
        const Group4 g = group4(s, m);
        double rc[4], rxm[4], rxp[4], rym[4], ryp[4], rzm[4], rzp[4];
        uint32_t tc[4], txm[4], txp[4], tym[4], typ[4], tzm[4], tzp[4];
        load_around4d(r, g, rc, rxm, rxp, rym, ryp, rzm, rzp);
        load_nt4(nt, g, tc, txm, txp, tym, typ, tzm, tzp);
        // r / diag on regular nodes, 0 elsewhere
        auto rr = [&](double v, uint32_t t) {
            const double rv = v * s.itwos;
            return t == (uint32_t)NT_REG ? rv : 0.0;
        };
        float out[4], o32[4];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const bool red = ((g.p0 + (unsigned)a) & 1u) == 0u;
            double zu;
            if (red)
                zu = -rc[a] * s.itwos;
            else
                zu = (-((rr(rxm[a], txm[a]) + rr(rxp[a], txp[a])) * s.cx +
                        (rr(rym[a], tym[a]) + rr(ryp[a], typ[a])) * s.cy +
                        (rr(rzm[a], tzm[a]) + rr(rzp[a], tzp[a])) * s.cz) -
                      rc[a]) *
                     s.itwos;
            out[a] = tc[a] == (uint32_t)NT_REG ? (float)zu : 0.f;
            o32[a] = (float)rc[a];
        }
        *reinterpret_cast<float4*>(z + g.u0) = make_float4(out[0], out[1], out[2], out[3]);
        *reinterpret_cast<float4*>(r32 + g.u0) = make_float4(o32[0], o32[1], o32[2], o32[3]);
    }
}

// The four-node form of k_fcg_pq (ni a multiple of 4): z's neighbour rows,
// p_old, q and P in 16-byte loads, p_new and q in 16-byte stores; the same
// arithmetic per node (p and q equal bit for bit; pq sums in another order).
__global__ void __launch_bounds__(BLOCK)
    k_fcg_pq4(Stencil s, const uint8_t* __restrict__ nt, const float* __restrict__ z,
              const double* __restrict__ pold, double* __restrict__ pnew, double* __restrict__ q,
              FcgHist h, int k, const double* __restrict__ P) {
    double beta = 0.0;
    if (k > 0) {
        double den = sget(h.pq + (k - 1) * SSIZE);
        beta = den != 0.0 ? -sget(h.zq + (k - 1) * SSIZE) / den : 0.0;
    }
    const bool first = k == 0;
    double acc = 0;
    auto ld4 = [&](const double* v, unsigned a, double (&o)[4]) {
        const double2 h0 = *reinterpret_cast<const double2*>(v + a);
        const double2 h1 = *reinterpret_cast<const double2*>(v + a + 2);
        o[0] = h0.x; o[1] = h0.y; o[2] = h1.x; o[3] = h1.y;
    };
    long long end;
    for (long long m = chunk_begin(s.nn / 4, end) + threadIdx.x; m < end; m += BLOCK) {
        const Group4 g = group4(s, m);
        Around4 zz;
        load_around4(z, g, zz);
        const uint32_t t4 = *reinterpret_cast<const uint32_t*>(nt + g.u0);
        double po[4] = {0, 0, 0, 0}, qo[4] = {0, 0, 0, 0}, pv[4] = {0, 0, 0, 0};
        if (!first) {
            ld4(pold, g.u0, po);
            ld4(q, g.u0, qo);
        }
        if (P) ld4(P, g.u0, pv);
        double pn[4], qn[4];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const bool reg = ((t4 >> (8 * a)) & 0xFFu) == (uint32_t)NT_REG;
            const double zu = zz.c[a];
            double az = ((double)zz.zm[a] + zz.zp[a]) * s.cz + ((double)zz.ym[a] + zz.yp[a]) * s.cy +
                        ((double)zz.xm[a] + zz.xp[a]) * s.cx - s.twos * zu;
            if (P) az -= pv[a] * zu;
            double pu = zu, qv = az;
            if (!first) {
                pu += beta * po[a];
                qv += beta * qo[a];
            }
            qv = reg ? qv : 0.0;
            pn[a] = pu;
            qn[a] = qv;
            acc += pu * qv;
        }
        *reinterpret_cast<double2*>(pnew + g.u0) = make_double2(pn[0], pn[1]);
        *reinterpret_cast<double2*>(pnew + g.u0 + 2) = make_double2(pn[2], pn[3]);
        *reinterpret_cast<double2*>(q + g.u0) = make_double2(qn[0], qn[1]);
        *reinterpret_cast<double2*>(q + g.u0 + 2) = make_double2(qn[2], qn[3]);
    }
    double a = block_sum(acc);
    if (threadIdx.x == 0) sadd(h.pq + k * SSIZE, a);
}

// b = a in FP64
__global__ void __launch_bounds__(BLOCK) k_widen(long long n, const float* __restrict__ a, double* __restrict__ b) {
    for (long long i = (long long)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (long long)gridDim.x * BLOCK)
        b[i] = (double)a[i];
}

}  // namespace

// one half-sweep of the learned cycle on FP32 vectors: the four-node kernel
// where i-lines are a multiple of 4 long, else the per-pair one
static void gs_half32(pic_ctx* ctx, const Stencil& s, const float* r32, float* z, int red_colour,
                      const double* P) {
    if (s.ni % 4 == 0) {
        k_gs_half4<<<group4_blocks(s), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r32, z, red_colour, P);
    } else {
        k_gs_half<float><<<pair_blocks(s), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r32, z, red_colour, P);
    }
}

// z = LEARNED_PRE_SWEEPS red-black Gauss-Seidel sweeps on A z = r from z = 0
// (device vectors): the learned preconditioner's pre-smoother, also used for
// its training pairs
int pic_learned_presmooth(pic_ctx* ctx, const double* r, float* z) {
    Stencil s = make_stencil(ctx->g, false);
    unsigned nb = pair_blocks(s);
    k_presmooth<<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r, z, nullptr, 0, nullptr, nullptr);
    for (int e = 1; e < LEARNED_PRE_SWEEPS; e++) {
        k_gs_half<double><<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r, z, 1, nullptr);
        k_gs_half<double><<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r, z, 0, nullptr);
    }
    PIC_HIP(ctx, hipGetLastError());
    return PIC_OK;
}

// z = M(r) in FP32; tmp holds the four FP32 vectors zpre, c, res and r32
// (r rounded, read by the closing sweeps).  The closing half-sweep also
// accumulates *zq += z.q (q may be null) and *rz += z.r; both must be zeroed
// by the caller.
static int learned_precond(pic_ctx* ctx, const Stencil& s, const double* rin, float* zout,
                           float* tmp, const double* q, double* zq, double* rz,
                           const double* P = nullptr) {
    unsigned nb = pair_blocks(s);
    float* zpre = tmp;
    float* c = tmp + s.nn;
    float* res = c + s.nn;
    float* r32 = res + s.nn;
    double* ws = ctx->scratch + LEARNED_WS;  // the coarse correction's striped sums
    double* dots = ws + 2 * SSIZE;
    const bool v4 = s.ni % 4 == 0;  // the four-node kernels
    if (v4 && !P)
        k_presmooth4<<<group4_blocks(s), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, rin, zpre, ws, 4 * SSIZE, r32);
    else
        k_presmooth<<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, rin, zpre, ws, 4 * SSIZE, P, r32);
    for (int e = 1; e < LEARNED_PRE_SWEEPS; e++) {
        gs_half32(ctx, s, r32, zpre, 1, P);
        gs_half32(ctx, s, r32, zpre, 0, P);
    }
    int e = pic_unet_coarse_correct(ctx, r32, zpre, c, res, ws, P);
    if (e) return e;
    // the closing sweeps: the first black half in k_gs_corr, the last red
    // half in k_gs_red_dots, the half-sweeps between them in place
    if (v4)
        k_gs_corr4<<<group4_blocks(s), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r32, zpre, c, dots, zout, P);
    else
        k_gs_corr<<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r32, zpre, c, dots, zout, P);
    for (int e = 1; e < LEARNED_POST_SWEEPS; e++) {
        gs_half32(ctx, s, r32, zout, 1, P);
        gs_half32(ctx, s, r32, zout, 0, P);
    }
    if (v4)
        k_gs_red_dots4<<<group4_blocks(s), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r32, zout, q, zq, rz, P);
    else
        k_gs_red_dots<<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, r32, zout, q, zq, rz, P);
    PIC_HIP(ctx, hipGetLastError());
    return PIC_OK;
}

static int learned_check(pic_ctx* ctx) {
    if (!pic_unet_ready(ctx))
        return pic_fail(ctx, PIC_ERR_STATE, "learned solver: no trained network for this grid");
    if (has_neumann(ctx))
        return pic_fail(ctx, PIC_ERR_ARG, "learned solver: Dirichlet-walled problems only");
    return PIC_OK;
}

// z = M(r) for host vectors (node order), the preconditioner alone
extern "C" int pic_learned_precondition(pic_ctx* ctx, const double* r, double* z) {
    if (!ctx || !r || !z) return PIC_ERR_ARG;
    int rc = pic_ensure_ntype(ctx);
    if (rc) return rc;
    rc = learned_check(ctx);
    if (rc) return rc;
    size_t nn = (size_t)ctx->g.nn;
    rc = pic_ensure_work(ctx, 5 * nn * sizeof(double));
    if (rc) return rc;
    double* rd = ctx->work;
    float* z32 = reinterpret_cast<float*>(rd + nn);
    double* rz = ctx->scratch + LEARNED_WS + 4 * SSIZE;  // striped
    PIC_HIP(ctx, hipMemcpyAsync(rd, r, nn * 8, hipMemcpyHostToDevice, ctx->stream));
    PIC_HIP(ctx, hipMemsetAsync(rz, 0, SSIZE * sizeof(double), ctx->stream));
    rc = learned_precond(ctx, make_stencil(ctx->g, false), rd, z32, reinterpret_cast<float*>(rd + 2 * nn),
                         nullptr, nullptr, rz);
    if (rc) return rc;
    k_widen<<<grid_for(nn, BLOCK), BLOCK, 0, ctx->stream>>>((long long)nn, z32, rd);  // r is spent
    PIC_HIP(ctx, hipGetLastError());
    PIC_HIP(ctx, hipMemcpyAsync(z, rd, nn * 8, hipMemcpyDeviceToHost, ctx->stream));
    PIC_HIP(ctx, pic_spin_wait(ctx->stream));
    return PIC_OK;
}

// the residual of the linear problem (no Boltzmann term)
static SorArgs plain_args(const Stencil& s) {
    SorArgs a;
    a.omega = 1;
    a.ieps = 1.0 / EPS0;
    a.itwos = 1.0 / s.twos;
    a.phi0 = 0;
    a.n0 = 0;
    a.inv_te0 = 1;
    return a;
}

static int solve_learned(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st) {
    int rc = learned_check(ctx);
    if (rc) return rc;
    const GridC& g = ctx->g;
    size_t nn = (size_t)g.nn;
    Stencil s = make_stencil(g, false);
    const int max_fcg = std::min(p->max_it, 500);
    // after the first check, every iteration: an iteration costs far more
    // than a check (a polled wait on a few bytes)
    const int check = p->check_every > 0 ? p->check_every : 1;
    const size_t hslots = (size_t)(max_fcg + 2) * SSIZE;  // striped history, per quantity
    rc = pic_ensure_work(ctx, 8 * nn * sizeof(double) + 4 * hslots * sizeof(double));
    if (rc) return rc;
    double* r = ctx->work;
    float* z = reinterpret_cast<float*>(r + nn);  // the preconditioned residual, FP32
    double* p0 = r + 2 * nn;
    double* p1 = p0 + nn;
    double* q = p1 + nn;
    float* ftmp = reinterpret_cast<float*>(q + nn);  // four FP32 vectors: 2 nn doubles
    FcgHist h;
    h.rz = q + 3 * nn;  // past the FP32 vectors, inside the 8 nn doubles
    h.pq = h.rz + hslots;
    h.zq = h.pq + hslots;
    h.rr = h.zq + hslots;
    double* sc = ctx->scratch + LEARNED_WS + 5 * SSIZE;  // three striped scalars
    unsigned nb = stencil_blocks(s.nn), nbr = stencil_blocks_red(s.nn);
    auto precond = [&](const double* rin, float* zout, const double* qv, double* zq, double* rz) {
        return learned_precond(ctx, s, rin, zout, ftmp, qv, zq, rz);
    };
    // pinned host copies: [0, 3 S) initial sums, 3 final FP64 residual sums
    // at 3 S, the striped r.r history from 4 S (S = SSIZE doubles)
    rc = pic_ensure_pin(ctx, (4 * SSIZE + hslots) * sizeof(double));
    if (rc) return rc;
    double* hp = ctx->pin;
    double* hrr = hp + 4 * SSIZE;
    PIC_HIP(ctx, hipMemsetAsync(sc, 0, 3 * SSIZE * sizeof(double), ctx->stream));
    k_fcg_resid<<<nb, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, ctx->phi, ctx->rho, 1.0 / EPS0, r, sc);
    PIC_HIP(ctx, hipMemcpyAsync(hp, sc, 3 * SSIZE * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    double bnorm2 = 1.0, target2 = 0.0;
    bool have_b = false;
    auto read_initial = [&]() {  // after a wait that covers the copy above
        const double rr0 = shost(hp), bb = shost(hp + SSIZE);
        bnorm2 = bb > 0 ? bb : 1.0;
        target2 = (p->tol_kind == PIC_TOL_REF_RMS) ? p->tol * p->tol * (double)nn : p->tol * p->tol * bnorm2;
        have_b = true;
        return rr0;
    };
    // A solve that follows another learned solve on this context (a time
    // loop) does not wait for the initial residual: it starts iterating and
    // reads it with the first check, since such a start is almost never
    // converged already (if it is, one iteration runs and the checks below
    // still decide convergence).  Otherwise the host waits for it here.
    const int prev = ctx->learned_last_its;
    int it = 0;
    bool conv = false;
    if (prev == 0) {
        PIC_HIP(ctx, pic_spin_wait(ctx->stream));
        conv = read_initial() <= target2;
    }
    bool have_final = false;  // FP64 residual of the final phi already copied to hp + 3 S
    if (!conv) {
        PIC_HIP(ctx, hipMemsetAsync(h.rz, 0, 4 * hslots * sizeof(double), ctx->stream));
        rc = precond(r, z, nullptr, nullptr, h.rz);  // rz[0] = z.r
        if (rc) return rc;
        double* pold = p0;
        double* pnew = p1;
        int last = 0;
        // the host reads the residual history first at 3/4 of the previous
        // solve's iteration count (a time loop's solves are alike; a later
        // first check would overshoot whenever a solve needs fewer
        // iterations than the last), then every `check` iterations
        int next_check = std::max(check, std::min(3 * prev / 4, max_fcg));
        for (int k = 0; k < max_fcg; k++) {
            {
                PicProfScope ps(ctx, PIC_K_PCG);
                if (s.ni % 4 == 0)
                    k_fcg_pq4<<<group4_blocks(s), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, z, pold, pnew, q, h, k,
                                                                          nullptr);
                else
                    k_fcg_pq<<<nbr, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, z, pold, pnew, q, h, k, nullptr);
                k_fcg_update<<<nb, BLOCK, 0, ctx->stream>>>(s.nn, h, k, ctx->phi, pnew, r, q);
            }
            PIC_HIP(ctx, hipGetLastError());
            it = k + 1;
            if (it >= next_check || it == max_fcg) {
                next_check = it + check;
                PIC_HIP(ctx, hipMemcpyAsync(hrr + (size_t)last * SSIZE, h.rr + (size_t)last * SSIZE,
                                            (size_t)(it - last) * SSIZE * sizeof(double),
                                            hipMemcpyDeviceToHost, ctx->stream));
                // where convergence is expected (the previous solve's count
                // or one more), the final FP64 residual is queued with the
                // check, saving a second wait
                const bool expect = prev > 0 && it >= prev && it <= prev + 1;
                if (expect) {
                    rc = queue_residual(ctx, s, plain_args(s), hp + 3 * SSIZE);
                    if (rc) return rc;
                }
                PIC_HIP(ctx, pic_spin_wait(ctx->stream));
                if (!have_b) read_initial();
                for (int j = last; j < it; j++) {
                    const double rj = shost(hrr + (size_t)j * SSIZE);
                    if (!(rj == rj)) return pic_fail(ctx, PIC_ERR_NUMERIC, "learned PCG produced NaN");
                    if (rj <= target2) conv = true;
                }
                last = it;
                if (conv) {
                    have_final = expect;
                    break;
                }
            }
            if (it == max_fcg) break;
            rc = precond(r, z, q, h.zq + (size_t)k * SSIZE, h.rz + (size_t)(k + 1) * SSIZE);
            if (rc) return rc;
            std::swap(pold, pnew);
        }
    }
    double rn[3];
    if (conv) {
        if (have_final) {
            for (int q2 = 0; q2 < 3; q2++) rn[q2] = hp[3 * SSIZE + q2];
        } else {
            rc = residual_norms(ctx, s, plain_args(s), rn);
            if (rc) return rc;
        }
        // the recursive residual history decided convergence; the FP64
        // residual of the final phi is the judge (CG residual norms are not
        // monotone, and the recursion drifts from the true residual)
        if (!(crit_value(p, rn, (double)nn) <= p->tol)) conv = false;
    }
    if (!conv) {  // plain PCG is the fallback, from the current phi
        pic_solver_params q2 = *p;
        q2.method = PIC_SOLVER_PCG;
        pic_solver_stats s2;
        rc = pic_solve_pcg(ctx, &q2, &s2, false);
        *st = s2;
        st->iterations += it;
        return rc;
    }
    st->converged = 1;
    st->iterations = it;
    ctx->learned_last_its = it;
    st->newton_iterations = 0;
    st->ref_l2 = std::sqrt(rn[0] / (double)nn);
    st->rel_residual = rn[2] > 0 ? std::sqrt(rn[1] / rn[2]) : std::sqrt(rn[1]);
    return PIC_OK;
}

// Newton-Boltzmann (PotentialSolver::solveNRPCG, PotentialSolver.cpp:178-241)
// with the learned preconditioner inside: per Newton step, F and the
// Jacobian shift P from the FP64 phi (k_F), then flexible CG on
// J y = F, J = A - diag(P), preconditioned by the two-level cycle whose
// smoothing sweeps, residual restriction and line search carry diag(P)
// (the network's coarse solve approximates A^-1 and the A-norm optimal step
// becomes the J-norm optimal one); phi -= y.  Converged when the FP64
// residual of the nonlinear problem over the regular rows is within the
// tolerance (PIC_TOL_REL), or, with PIC_TOL_REF_RMS, when RMS(y) < 1e-3 as
// in the reference (:229-233).  Each inner solve reduces its residual by
// 1e-2 (inexact Newton) or to below the tolerance.  Plain Newton-PCG is the
// fallback if the learned iteration stalls; the final residual is FP64.
static int solve_newton_learned(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st) {
    int rc = learned_check(ctx);
    if (rc) return rc;
    const GridC& g = ctx->g;
    const size_t nn = (size_t)g.nn;
    Stencil s = make_stencil(g, false);
    const int max_fcg = std::min(p->max_it, 1000);
    const size_t hslots = (size_t)(max_fcg + 2) * SSIZE;
    // r (F), z, p0, p1, q, y, P (FP64), three FP32 vectors, four histories
    rc = pic_ensure_work(ctx, 9 * nn * sizeof(double) + 4 * hslots * sizeof(double));
    if (rc) return rc;
    double* r = ctx->work;
    float* z = reinterpret_cast<float*>(r + nn);  // the preconditioned residual, FP32
    double* p0 = r + 2 * nn;
    double* p1 = p0 + nn;
    double* q = p1 + nn;
    double* y = q + nn;
    double* P = y + nn;
    float* ftmp = reinterpret_cast<float*>(P + nn);  // four FP32 vectors: 2 nn doubles
    FcgHist h;
    h.rz = P + nn + 2 * nn;
    h.pq = h.rz + hslots;
    h.zq = h.pq + hslots;
    h.rr = h.zq + hslots;
    rc = pic_ensure_pin(ctx, (4 + hslots) * sizeof(double));
    if (rc) return rc;
    double* hf = ctx->pin;       // the Newton residual sums
    double* hrr = ctx->pin + 4;  // the inner residual history (striped)
    NewtonArgs na;
    na.ieps = 1.0 / EPS0;
    na.phi0 = p->phi0;
    na.n0 = p->n0;
    na.inv_te0 = 1.0 / (p->Te0 != 0 ? p->Te0 : 1.0);
    unsigned nb = stencil_blocks(s.nn), nbr = stencil_blocks_red(s.nn);
    int total_it = 0, newton = 0;
    bool conv = false, stalled = false;
    for (newton = 0; newton < 20; newton++) {  // NR_MAX_IT, PotentialSolver.cpp:179
        rc = pic_newton_residual(ctx, s, na, r, P, hf);
        if (rc) return rc;
        PIC_HIP(ctx, pic_spin_wait(ctx->stream));
        const double bb = hf[2] > 0 ? hf[2] : 1.0;
        const double target2 = p->tol_kind == PIC_TOL_REF_RMS ? p->tol * p->tol * (double)nn
                                                              : p->tol * p->tol * bb;
        if (p->tol_kind == PIC_TOL_REL && hf[1] <= target2) {
            conv = true;
            break;
        }
        if (!(hf[0] == hf[0])) return pic_fail(ctx, PIC_ERR_NUMERIC, "Newton residual is NaN");
        // inexact Newton (Eisenstat-Walker style, constant forcing 1e-2):
        // each inner solve reduces its residual 100-fold, or to below the
        // tolerance; a learned iteration costs several PCG iterations, so
        // more, cheaper Newton steps pay
        const double inner2 = std::max(0.25 * target2, hf[0] * 1e-4);
        // flexible CG on J y = F from y = 0 (r = F; F vanishes off the regular rows)
        PIC_HIP(ctx, hipMemsetAsync(y, 0, nn * sizeof(double), ctx->stream));
        PIC_HIP(ctx, hipMemsetAsync(h.rz, 0, 4 * hslots * sizeof(double), ctx->stream));
        rc = learned_precond(ctx, s, r, z, ftmp, nullptr, nullptr, h.rz, P);
        if (rc) return rc;
        double* pold = p0;
        double* pnew = p1;
        int it = 0;
        bool inner_conv = false;
        for (int k = 0; k < max_fcg; k++) {
            {
                PicProfScope ps(ctx, PIC_K_PCG);
                if (s.ni % 4 == 0)
                    k_fcg_pq4<<<group4_blocks(s), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, z, pold, pnew, q, h, k, P);
                else
                    k_fcg_pq<<<nbr, BLOCK, 0, ctx->stream>>>(s, ctx->ntype, z, pold, pnew, q, h, k, P);
                k_fcg_update<<<nb, BLOCK, 0, ctx->stream>>>(s.nn, h, k, y, pnew, r, q);
            }
            PIC_HIP(ctx, hipGetLastError());
            it = k + 1;
            PIC_HIP(ctx, hipMemcpyAsync(hrr + (size_t)k * SSIZE, h.rr + (size_t)k * SSIZE, SSIZE * sizeof(double),
                                        hipMemcpyDeviceToHost, ctx->stream));
            PIC_HIP(ctx, pic_spin_wait(ctx->stream));
            const double rk = shost(hrr + (size_t)k * SSIZE);
            if (!(rk == rk)) return pic_fail(ctx, PIC_ERR_NUMERIC, "learned Newton inner solve produced NaN");
            if (rk <= inner2) {
                inner_conv = true;
                break;
            }
            if (it == max_fcg) break;
            rc = learned_precond(ctx, s, r, z, ftmp, q, h.zq + (size_t)k * SSIZE,
                                 h.rz + (size_t)(k + 1) * SSIZE, P);
            if (rc) return rc;
            std::swap(pold, pnew);
        }
        total_it += it;
        if (!inner_conv) {
            stalled = true;
            break;
        }
        rc = pic_newton_update(ctx, s, y, hf + 3);
        if (rc) return rc;
        double yy;
        PIC_HIP(ctx, pic_spin_wait(ctx->stream));
        yy = hf[3];
        if (p->tol_kind == PIC_TOL_REF_RMS && std::sqrt(yy / (double)nn) < 1e-3) {  // :229-233
            conv = true;
            newton++;
            break;
        }
    }
    if (stalled || !conv) {  // plain Newton-PCG from the current phi is the fallback
        pic_solver_params q2 = *p;
        q2.method = PIC_SOLVER_PCG;
        pic_solver_stats s2;
        rc = pic_solve_pcg(ctx, &q2, &s2, false);
        *st = s2;
        st->iterations += total_it;
        st->newton_iterations += newton;
        return rc;
    }
    SorArgs a;
    a.omega = 1;
    a.ieps = 1.0 / EPS0;
    a.itwos = 1.0 / s.twos;
    a.phi0 = p->phi0;
    a.n0 = p->n0;
    a.inv_te0 = na.inv_te0;
    double rn[3];
    rc = residual_norms(ctx, s, a, rn);
    if (rc) return rc;
    st->converged = 1;
    st->iterations = total_it;
    st->newton_iterations = newton;
    st->ref_l2 = std::sqrt(rn[0] / (double)nn);
    st->rel_residual = rn[2] > 0 ? std::sqrt(rn[1] / rn[2]) : std::sqrt(rn[1]);
    return PIC_OK;
}

// plain red-black SOR to a relative tolerance (used to make training pairs)
extern "C" int pic_poisson(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st) {
    if (!ctx || !p) return PIC_ERR_ARG;
    if (!(p->tol > 0) || p->max_it <= 0) return pic_fail(ctx, PIC_ERR_ARG, "bad solver params");
    int rc = pic_ensure_ntype(ctx);
    if (rc) return rc;
    pic_solver_stats local;
    if (!st) st = &local;
    *st = pic_solver_stats{};
    for (auto& e : ctx->solve_ev)
        if (!e) PIC_HIP(ctx, hipEventCreate(&e));
    hipEvent_t e0 = ctx->solve_ev[0], e1 = ctx->solve_ev[1];
    PIC_HIP(ctx, hipEventRecord(e0, ctx->stream));
    if (p->flags & PIC_SOLVE_EXTRAPOLATE) {
        const size_t nn = (size_t)ctx->g.nn;
        if (!ctx->phi_prev) PIC_HIP(ctx, hipMalloc(&ctx->phi_prev, nn * sizeof(double)));
        if (ctx->phi_prev_valid) {
            k_extrapolate<<<stencil_blocks((long long)nn), BLOCK, 0, ctx->stream>>>((long long)nn, ctx->phi,
                                                                                    ctx->phi_prev);
            PIC_HIP(ctx, hipGetLastError());
        } else {
            PIC_HIP(ctx, hipMemcpyAsync(ctx->phi_prev, ctx->phi, nn * sizeof(double), hipMemcpyDeviceToDevice,
                                        ctx->stream));
            ctx->phi_prev_valid = true;
        }
    }
    switch (p->method) {
        case PIC_SOLVER_SOR_RB: rc = pic_solve_sor(ctx, p, st); break;
        case PIC_SOLVER_PCG: rc = pic_solve_pcg(ctx, p, st, false); break;
        case PIC_SOLVER_PCG_MIXED: rc = pic_solve_pcg(ctx, p, st, true); break;
        case PIC_SOLVER_LEARNED:
            rc = p->n0 != 0.0 ? solve_newton_learned(ctx, p, st) : solve_learned(ctx, p, st);
            break;
        default: rc = pic_fail(ctx, PIC_ERR_ARG, "unknown solver method");
    }
    (void)hipEventRecord(e1, ctx->stream);
    (void)pic_spin_event(e1);  // polled: the solvers' last wait has usually drained the stream
    float ms = 0;
    (void)hipEventElapsedTime(&ms, e0, e1);
    st->seconds = ms * 1e-3;
    return rc;
}
