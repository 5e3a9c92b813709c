// pic_stencil.h -- what the field solvers share: the operator's rows, the
// grid-wide sums, the residual of a potential.
//
// The solvers are translation units of their own (pic_sor.hip, pic_pcg.hip,
// pic_solver.hip): the GPU code of a unit is loaded when the first of its
// kernels is launched, and a process that solves one way does not wait for the
// others'.  A process's first solve, in one unit and here: learned at 128^3 5.3 and
// 3.8 ms, FP64 PCG at 64^3 4.6 and 3.2, SOR 3.6 and 2.5 (0.9 when repeated).
//
// The operator rows follow PotentialSolver::buildMatrix
// (PotentialSolver.cpp:414-471): Dirichlet rows are the identity, Neumann face
// rows are one-sided (1/dx)(phi_u - phi_nbr), regular rows are the 7-point
// Laplacian.  Jacobi M = 1/diag(A) of that operator (PotentialSolver.cpp:470).
//
// All stencil kernels walk the grid in contiguous chunks per workgroup and
// map consecutive chunks to the same XCD (workgroups are dealt round-robin
// over the 8 XCDs), so k-neighbour planes are reused from that XCD's L2.
#pragma once
#include <algorithm>
#include <cmath>

#include "pic_internal.h"

namespace pic {

struct Stencil {
    double cx, cy, cz, twos;  // +-1, +-ni, +-ni*nj coefficients; 2(sum 1/dx^2)
    double itwos;             // 1 / twos
    double idx[3];            // 1/dx per axis (Neumann rows)
    long long sj, sk, nn;
    int ni, nj, nk;
};

struct SorArgs {
    double omega, ieps, itwos, phi0, n0, inv_te0;
    int color;
};

struct NewtonArgs {
    double ieps, phi0, n0, inv_te0;
};

}  // namespace pic

// pic_sor.hip: PIC_SOLVER_SOR_RB
int pic_solve_sor(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st);
// pic_pcg.hip: Newton + PCG, FP64 or (mixed) with FP32 inner vectors
int pic_solve_pcg(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st, bool mixed);
// and its parts for another inner solver (no Neumann faces): the Newton residual F
// of ctx->phi and the Jacobian's shift P, with the sums F.F (all rows), F.F
// (regular), b.b into sums[0..2]; phi -= y, with y.y into *sum.  Queued; the sums
// go to pinned memory.
int pic_newton_residual(pic_ctx* ctx, const pic::Stencil& s, const pic::NewtonArgs& a, double* F, double* P,
                        double* sums);
int pic_newton_update(pic_ctx* ctx, const pic::Stencil& s, const double* y, double* sum);

namespace {

using namespace pic;

constexpr int BLOCK = 256;
constexpr int NXCD = 8;

// gridDim.x is a multiple of NXCD (stencil_blocks), so lb is a bijection
__device__ inline long long chunk_begin(long long nn, long long& end) {
    int nb = gridDim.x;
    int b = blockIdx.x;
    int per_xcd = nb / NXCD;
    int lb = (b % NXCD) * per_xcd + b / NXCD;  // logical, XCD-contiguous
    long long chunk = ((nn + nb - 1) / nb + BLOCK - 1) / BLOCK * BLOCK;
    long long beg = (long long)lb * chunk;
    end = beg + chunk < nn ? beg + chunk : nn;
    return beg;
}

__device__ inline double block_sum(double v) {
    __shared__ double red[BLOCK / 64];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < BLOCK / 64; w++) t += red[w];
    __syncthreads();
    return t;  // valid in thread 0
}

template <typename T>
__device__ inline T nbr_of(uint8_t t, const T* v, long long u, const Stencil& s) {
    switch (t) {
        case NT_NEU_IM: return v[u + 1];
        case NT_NEU_IP: return v[u - 1];
        case NT_NEU_JM: return v[u + s.sj];
        case NT_NEU_JP: return v[u - s.sj];
        case NT_NEU_KM: return v[u + s.sk];
        default: return v[u - s.sk];
    }
}
__device__ inline double neu_coef(uint8_t t, const Stencil& s) {
    return t <= NT_NEU_IP ? s.idx[0] : (t <= NT_NEU_JP ? s.idx[1] : s.idx[2]);
}
// diag(A) for the Jacobi preconditioner
__device__ inline double diagA(uint8_t t, const Stencil& s) {
    if (t == NT_REG) return -s.twos;
    if (t == NT_DIR) return 1.0;
    return neu_coef(t, s);
}

// (A v)_u for a vector given as a functor of the node index
template <typename T, typename F>
__device__ inline T apply_A(uint8_t t, long long u, const Stencil& s, F v) {
    T vu = v(u);
    if (t == NT_REG)
        return (T)s.cz * (v(u - s.sk) + v(u + s.sk)) + (T)s.cy * (v(u - s.sj) + v(u + s.sj)) +
               (T)s.cx * (v(u - 1) + v(u + 1)) - (T)s.twos * vu;
    if (t == NT_DIR) return vu;
    long long o;
    switch (t) {
        case NT_NEU_IM: o = 1; break;
        case NT_NEU_IP: o = -1; break;
        case NT_NEU_JM: o = s.sj; break;
        case NT_NEU_JP: o = -s.sj; break;
        case NT_NEU_KM: o = s.sk; break;
        default: o = -s.sk; break;
    }
    return (T)neu_coef(t, s) * (vu - v(u + o));
}

// Grid-wide sums of the linear solvers: every workgroup stores its partial
// sum at part[blockIdx.x] (a plain store, nothing to clear and no atomics:
// 1000 workgroups adding to one FP64 word took longer than the PCG kernels'
// loads), and every workgroup of the kernel that needs the total adds the
// partials up itself, while its first loads are in flight.
// PART_MAX workgroups at most: four per CU, all resident at once at these
// kernels' 44..107 registers (128^3 FP64 solve of 424 iterations: 20.0 ms with
// up to 2048 workgroups, whose last ones ran as a second, nearly empty wave,
// 18.8 with 1280, 16.1 with 1024, 16.3 with 512)
constexpr int PART_MAX = 1024;
// ctx->scratch offsets of the partials: three residual sums, then PCG's g.s,
// g.g and d.z (a second set of these for k_cg, which reads one and writes the
// other); the stop flag and the rings of g.s and alpha follow
constexpr int PART_F = 16384, PART_GS = PART_F + 3 * PART_MAX, PART_GG = PART_GS + PART_MAX,
              PART_DZ = PART_GG + PART_MAX, PART_SET = 3 * PART_MAX, PCG_FLAG = PART_GS + 2 * PART_SET,
              PCG_GS = PCG_FLAG + 8, PCG_AL = PCG_GS + 4;
static_assert(PCG_AL + 4 <= (int)SCRATCH_DOUBLES, "scratch layout");
__device__ inline double sum_parts(const double* __restrict__ part, int n) {
    __shared__ double red[BLOCK / 64];
    double v = 0;
    for (int q = threadIdx.x; q < n; q += BLOCK) v += part[q];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; w++) t += red[w];
    __syncthreads();
    return t;  // valid in every thread
}
// out[q] = the sum of part[q * PART_MAX ..] (one workgroup per q); out may
// be pinned host memory
__global__ void __launch_bounds__(BLOCK) k_sum_parts(const double* __restrict__ part, int n, double* out) {
    const double t = sum_parts(part + (size_t)blockIdx.x * PART_MAX, n);
    if (threadIdx.x == 0) out[blockIdx.x] = t;
}

// Four consecutive nodes u0 .. u0 + 3 (u0 a multiple of 4) per thread, in
// flat order: a vector's own values in one 16-byte load (two in FP64), the
// rows on either side likewise (unaligned where a row is not a multiple of 4
// long), the i-neighbours beyond the group as single words.  Rows need no
// special care: a group that straddles two i-lines holds face nodes there,
// and face nodes do not use the 7-point stencil.  Addresses are clamped into
// the array for the groups on its first and last planes.
template <typename T>
struct Q4 {
    T a[4];
};
template <typename T>
__device__ inline Q4<T> load4(const T* __restrict__ p) {
    typedef T V __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    const V v = *reinterpret_cast<const V*>(p);
    return Q4<T>{{v[0], v[1], v[2], v[3]}};
}
template <typename T>
__device__ inline void store4(T* __restrict__ p, const T (&a)[4]) {
    typedef T V __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    *reinterpret_cast<V*>(p) = V{a[0], a[1], a[2], a[3]};
}
template <typename T>
struct Ring4 {
    Q4<T> c, ym, yp, zm, zp;
    T l, r;
};
template <typename T>
__device__ inline void load_ring4(const T* __restrict__ v, unsigned u0, const Stencil& s, Ring4<T>& g) {
    const unsigned n = (unsigned)s.nn, sj = (unsigned)s.sj, sk = (unsigned)s.sk, last = n - 4u;
    g.c = load4(v + u0);
    g.ym = load4(v + (u0 >= sj ? u0 - sj : 0u));
    g.yp = load4(v + (u0 + sj <= last ? u0 + sj : last));
    g.zm = load4(v + (u0 >= sk ? u0 - sk : 0u));
    g.zp = load4(v + (u0 + sk <= last ? u0 + sk : last));
    g.l = v[u0 >= 1u ? u0 - 1u : 0u];
    g.r = v[u0 + 4u < n ? u0 + 4u : n - 1u];
}
// the 7-point operator at the group's node q (apply_A's order)
template <typename T>
__device__ inline T ring_A(const Ring4<T>& g, int q, const Stencil& s) {
    const T xm = q == 0 ? g.l : g.c.a[q == 0 ? 0 : q - 1];
    const T xp = q == 3 ? g.r : g.c.a[q == 3 ? 3 : q + 1];
    return (T)s.cz * (g.zm.a[q] + g.zp.a[q]) + (T)s.cy * (g.ym.a[q] + g.yp.a[q]) + (T)s.cx * (xm + xp) -
           (T)s.twos * g.c.a[q];
}
__device__ inline uint32_t load_types4(const uint8_t* __restrict__ nt, unsigned u0) {
    return *reinterpret_cast<const uint32_t*>(nt + u0);
}
__device__ inline uint8_t type_at(uint32_t t4, int q) { return (uint8_t)((t4 >> (8 * q)) & 0xFFu); }

// workgroups of the four-node kernels with partial sums: one group per
// thread up to PART_MAX workgroups
inline unsigned part_blocks(long long nn) {
    long long b = (nn / 4 + BLOCK - 1) / BLOCK;
    if (b > PART_MAX) b = PART_MAX;
    return (unsigned)((b + NXCD - 1) / NXCD * NXCD);
}

// residual of the (Boltzmann) Poisson problem, three partial sums: sum R^2
// over all non-Dirichlet rows (reference RMS numerator), sum R^2 over
// regular rows, sum b^2 over regular rows.
__global__ void __launch_bounds__(BLOCK)
    k_resid(Stencil s, SorArgs a, const uint8_t* __restrict__ nt, const double* __restrict__ phi,
            const double* __restrict__ rho, double* __restrict__ part) {
    double r_all = 0, r_reg = 0, b_reg = 0;
    auto regular = [&](double p, double rho_u, double sx, double sy, double sz) {
        double q = rho_u;
        if (a.n0 != 0.0) q -= QE * (a.n0 * exp((p - a.phi0) * a.inv_te0));
        const double R = -p * s.twos + q * a.ieps + sx * s.cx + sy * s.cy + sz * s.cz;
        const double b = rho_u * a.ieps;
        r_all += R * R;
        r_reg += R * R;
        b_reg += b * b;
    };
    auto face = [&](uint8_t t, long long u) {
        const double R = phi[u] - nbr_of<double>(t, phi, u, s);
        r_all += R * R;
    };
    long long end;
    for (long long m = chunk_begin(s.nn / 4, end) + threadIdx.x; m < end; m += BLOCK) {
        const unsigned u0 = 4u * (unsigned)m;
        const uint32_t t4 = load_types4(nt, u0);
        Ring4<double> g;
        load_ring4(phi, u0, s, g);
        const Q4<double> rh = load4(rho + u0);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint8_t t = type_at(t4, q);
            if (t == NT_REG)
                regular(g.c.a[q], rh.a[q], (q == 0 ? g.l : g.c.a[q == 0 ? 0 : q - 1]) +
                                               (q == 3 ? g.r : g.c.a[q == 3 ? 3 : q + 1]),
                        g.ym.a[q] + g.yp.a[q], g.zm.a[q] + g.zp.a[q]);
            else if (t != NT_DIR)
                face(t, u0 + q);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < (unsigned)(s.nn & 3)) {  // corner nodes past the last group
        const long long u = (s.nn & ~3ll) + threadIdx.x;
        if (nt[u] != NT_REG && nt[u] != NT_DIR) face(nt[u], u);
    }
    double t0 = block_sum(r_all), t1 = block_sum(r_reg), t2 = block_sum(b_reg);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = t0;
        part[PART_MAX + blockIdx.x] = t1;
        part[2 * PART_MAX + blockIdx.x] = t2;
    }
}

inline Stencil make_stencil(const GridC& g, bool axis_swap) {
    Stencil s;
    double d2x = 1.0 / (g.dx[0] * g.dx[0]), d2y = 1.0 / (g.dx[1] * g.dx[1]),
           d2z = 1.0 / (g.dx[2] * g.dx[2]);
    s.cx = axis_swap ? d2z : d2x;
    s.cy = d2y;
    s.cz = axis_swap ? d2x : d2z;
    s.twos = 2.0 * (d2x + d2y + d2z);
    s.itwos = 1.0 / s.twos;
    for (int d = 0; d < 3; d++) s.idx[d] = 1.0 / g.dx[d];
    s.sj = g.ni;
    s.sk = (long long)g.ni * g.nj;
    s.nn = g.nn;
    s.ni = g.ni;
    s.nj = g.nj;
    s.nk = g.nk;
    return s;
}

inline unsigned stencil_blocks(long long items) {
    // about two items per thread: enough workgroups in flight to cover HBM latency
    long long b = (items + BLOCK * 2 - 1) / (BLOCK * 2);
    if (b > 16384) b = 16384;
    b = (b + NXCD - 1) / NXCD * NXCD;  // multiple of NXCD, at least NXCD
    return (unsigned)b;
}

// any Neumann face node (a face node that is neither an object node nor
// flagged Dirichlet); the node types are current
inline bool has_neumann(pic_ctx* ctx) {
    if (pic_ensure_ntype(ctx) != PIC_OK) return true;
    return ctx->has_neumann;
}

// queues the residual sums of phi (k_resid's three) into out (pinned memory)
inline int queue_residual(pic_ctx* ctx, const Stencil& st, const SorArgs& a, double* out) {
    const unsigned nb = part_blocks(st.nn);
    k_resid<<<nb, BLOCK, 0, ctx->stream>>>(st, a, ctx->ntype, ctx->phi, ctx->rho, ctx->scratch + PART_F);
    k_sum_parts<<<3, BLOCK, 0, ctx->stream>>>(ctx->scratch + PART_F, (int)nb, out);
    PIC_HIP(ctx, hipGetLastError());
    return PIC_OK;
}
inline int residual_norms(pic_ctx* ctx, const Stencil& st, const SorArgs& a, double out[3]) {
    int rc = pic_ensure_pin(ctx, 3 * sizeof(double));
    if (!rc) rc = queue_residual(ctx, st, a, ctx->pin);
    if (rc) return rc;
    PIC_HIP(ctx, pic_spin_wait(ctx->stream));
    for (int q = 0; q < 3; q++) out[q] = ctx->pin[q];
    return PIC_OK;
}

inline double crit_value(const pic_solver_params* p, const double r[3], double nn) {
    if (p->tol_kind == PIC_TOL_REF_RMS) return std::sqrt(r[0] / nn);
    return r[2] > 0 ? std::sqrt(r[1] / r[2]) : std::sqrt(r[1]);
}

// Launches (PCG: iterations) that the host queues behind a check before it
// waits for it: enough to keep the device busy while the host sees the check's
// event, and few, because those behind a check that ends the solve are waited
// for although they return at once (2 us each).  32^3 nodes, SOR from the solution,
// a check every 25 and every 1000 sweeps: 44 us with 4; 75 and 2225 with the whole
// interval queued; 47 and 69 with none.  The cold solve 0.38 ms with 2 and with 4, 0.40
// with the whole interval; 128^3 FP64 PCG 12.6 ms with any.
constexpr int RUN_AHEAD = 4;

}  // namespace
