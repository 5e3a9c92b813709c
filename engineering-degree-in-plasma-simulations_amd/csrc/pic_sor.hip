// pic_sor.hip -- red-black SOR of the gfx950 PIC library.
//
//   k_sor_tile   red-black SOR with the Boltzmann electron term
//                (PotentialSolver.cpp:69-166; ch2/v1/PotentialSolver.cpp:8-87),
//                two sweeps per launch on tiles; k_sor: one colour per launch
//   k_neumann    Neumann face copies (PotentialSolver.cpp:96-107)
#include <type_traits>
#include <utility>

#include "pic_stencil.h"

namespace {

// The SOR update of a regular node from its neighbour sums along each axis
// (shared by both sweep kernels, rounded the same way: no contraction).
template <bool BOLTZ>
__device__ inline double sor_node(const Stencil& s, const SorArgs& a, double p, double rho_u, double sx,
                                  double sy, double sz) {
#pragma clang fp contract(off)
    double q = rho_u;
    if (BOLTZ) q -= QE * (a.n0 * exp((p - a.phi0) * a.inv_te0));
    const double nw = (q * a.ieps + sx * s.cx + sy * s.cy + sz * s.cz) * a.itwos;
    return p + a.omega * (nw - p);
}

__global__ void __launch_bounds__(BLOCK)
    k_sor(Stencil s, SorArgs a, const uint8_t* __restrict__ nt, double* __restrict__ phi,
          const double* __restrict__ rho) {
    long long half = (s.ni + 1) / 2;
    long long items = half * s.nj * s.nk;
    long long end;
    for (long long m = chunk_begin(items, end) + threadIdx.x; m < end; m += BLOCK) {
        unsigned row = (unsigned)m / (unsigned)half;
        int h = (int)((unsigned)m - row * (unsigned)half);
        unsigned kk = row / (unsigned)s.nj;
        int j = (int)(row - kk * (unsigned)s.nj), k = (int)kk;
        int i = 2 * h + ((j + k + a.color) & 1);
        if (i >= s.ni) continue;
        long long u = row * s.ni + i;
        if (nt[u] != NT_REG) continue;
        const double sx = phi[u - 1] + phi[u + 1], sy = phi[u - s.sj] + phi[u + s.sj], sz = phi[u - s.sk] + phi[u + s.sk];
        phi[u] = a.n0 != 0.0 ? sor_node<true>(s, a, phi[u], rho[u], sx, sy, sz)
                             : sor_node<false>(s, a, phi[u], rho[u], sx, sy, sz);
    }
}

// ---- tiled sweeps: several half sweeps per launch ----
// A launch per colour is bound by its launch: a half sweep of a 64 x 64 x 256
// grid took 6.9 us (4.1 us at 32^3, an empty launch's time).  k_sor_tile
// therefore keeps a tile of the potential on chip and makes up to SOR_HALO
// half sweeps on it.  The tile's core is what it writes; around it lie
// SOR_HALO more nodes in every direction, because half sweep q + 1 of a node
// needs its neighbours after half sweep q: what a half sweep computes is right
// for nodes at least q + 1 from the tile's edge, so the core is right after
// SOR_HALO of them.  Nodes nearer the edge hold values that nothing correct
// reads.  Where the tile ends at the grid's end there is no halo (face nodes
// are not updated).  The potential goes from one buffer to another, since
// neighbouring tiles read each other's cores.
//
// A thread owns the node pair (2h, 2h + 1) of one j-line of the tile for all
// TK planes, in registers with their charge density and row bits; one of the
// two is red, by the plane's parity.  A wave's j-lines all have the same
// parity, so which one it is is a constant of the wave and the code has no
// selection.  A node's neighbours along k and one of those along i are the
// thread's own; the other three come from LDS, which holds the first and the
// second nodes as [plane][j][pair] (consecutive lanes read consecutive
// words).  The update is sor_node on the same operands as k_sor's (a sum of
// two neighbours does not depend on their order), so every value equals
// k_sor's bit for bit.
//
// Row bits of a node: SOR_REG, and for each neighbour whether it is a Neumann
// face.  Such a face holds a copy of the node next to it from the end of the
// previous sweep (k_neumann), which is the value the node still has when its
// own turn comes, so from the second sweep on (own) the node's value stands
// in for the face's and no copies are made between sweeps.
constexpr int SOR_HALO = 4;
enum : unsigned { SOR_REG = 1, SOR_IM = 2, SOR_IP = 4, SOR_JM = 8, SOR_JP = 16, SOR_KM = 32, SOR_KP = 64 };

__global__ void __launch_bounds__(BLOCK)
    k_sor_bits(Stencil s, const uint8_t* __restrict__ nt, uint8_t* __restrict__ bits) {
    long long end;
    for (long long u = chunk_begin(s.nn, end) + threadIdx.x; u < end; u += BLOCK) {
        unsigned m = 0;
        if (nt[u] == NT_REG) {  // an interior node
            auto neu = [&](long long v) { return nt[v] != NT_REG && nt[v] != NT_DIR; };
            m = SOR_REG | (neu(u - 1) ? SOR_IM : 0) | (neu(u + 1) ? SOR_IP : 0) | (neu(u - s.sj) ? SOR_JM : 0) |
                (neu(u + s.sj) ? SOR_JP : 0) | (neu(u - s.sk) ? SOR_KM : 0) | (neu(u + s.sk) ? SOR_KP : 0);
        }
        bits[u] = (uint8_t)m;
    }
}

// One axis of the tiling: a grid of n nodes in m tiles of t nodes
struct TileAxis {
    int n, t, m;
    __host__ __device__ int start(int q) const {  // even, and the last tile reaches the grid's end
        if (q == 0) return 0;
        const int b = q * (t - 2 * SOR_HALO), e = (n - t + 1) & ~1;
        return b < e ? b : e;
    }
    __host__ __device__ int core(int q) const {  // the first node tile q writes; core(m) = n
        return q == 0 ? 0 : (q == m ? n : q * (t - 2 * SOR_HALO) + SOR_HALO);
    }
};
TileAxis tile_axis(int n, int t) {
    TileAxis a{n, t, 1};
    while ((a.m - 1) * (t - 2 * SOR_HALO) + t < n) a.m++;
    return a;
}

// f(1), ..., f(n) with constant arguments, K = 0 .. n - 1
template <typename F, int... K>
__device__ __attribute__((always_inline)) inline void for_planes(F f, std::integer_sequence<int, K...>) {
    (f(std::integral_constant<int, K + 1>{}), ...);
}

template <int PI, int TJ, int TK, bool NEU, bool BOLTZ>
__global__ void __launch_bounds__(PI* TJ)
    k_sor_tile(Stencil s, SorArgs a, TileAxis ax, TileAxis ay, TileAxis az, const uint8_t* __restrict__ bits,
               const double* __restrict__ in, double* __restrict__ out, const double* __restrict__ rho, int ns,
               int own, const double* __restrict__ stop) {
    constexpr int NT = PI * TJ, LINES = 64 / PI;  // j-lines of a wave
    static_assert(NT % 128 == 0 && TJ % (2 * LINES) == 0, "waves of one parity");
    __shared__ double lds[2][TK][NT];  // [first or second node][plane][j, pair]
    if (*stop != 0.0) return;          // (the whole grid)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int h = lane % PI;
    const int jl = (wave & 1) + 2 * (LINES * (wave >> 1) + lane / PI);  // the wave's lines: every second one
    const int tid = jl * PI + h;
    const unsigned b = (unsigned)xcd_wg();
    const int bx = (int)(b % (unsigned)ax.m), by = (int)(b / (unsigned)ax.m % (unsigned)ay.m),
              bz = (int)(b / (unsigned)(ax.m * ay.m));
    if (bz >= az.m) return;  // (the whole workgroup)
    const int i0 = ax.start(bx), j0 = ay.start(by), k0 = az.start(bz);
    const int i = i0 + 2 * h, j = j0 + jl;
    const bool in1 = i < s.ni && j < s.nj, in2 = i + 1 < s.ni && j < s.nj;
    const unsigned ub = ((unsigned)k0 * (unsigned)s.nj + (unsigned)j) * (unsigned)s.ni + (unsigned)i;
    const unsigned sk = (unsigned)s.sk;
    // Every load before any use, without branches: clamped addresses (a node
    // beyond the grid gets some other node's values and no row bits).
    typedef double D2 __attribute__((ext_vector_type(2), aligned(8)));
    const unsigned top = (unsigned)s.nn - 2u;
    D2 P[TK], R[TK];
    unsigned m[TK];  // row bits: first | second << 8
#pragma unroll
    for (int k = 0; k < TK; k++) {
        const unsigned u = ub + (unsigned)k * sk, v = u < top ? u : top;
        P[k] = *reinterpret_cast<const D2*>(in + v);
        R[k] = *reinterpret_cast<const D2*>(rho + v);
        uint16_t w;
        __builtin_memcpy(&w, bits + v, 2);
        m[k] = w;
    }
    const unsigned keep = (in1 ? 0xFFu : 0u) | (in2 ? 0xFF00u : 0u);
#pragma unroll
    for (int k = 0; k < TK; k++) {
        if (ub + (unsigned)k * sk == top + 1u) {  // the grid's last node: the second of the clamped pair
            P[k][0] = P[k][1];
            m[k] = 0;
        }
        m[k] = k0 + k < s.nk ? m[k] & keep : 0u;
        lds[0][k][tid] = P[k][0];
        lds[1][k][tid] = P[k][1];
    }
    __syncthreads();
    // LDS places of the neighbours (a place beyond the tile: the thread's own,
    // read only for nodes whose value nothing correct reads)
    const int qm = h > 0 ? tid - 1 : tid, qp = h < PI - 1 ? tid + 1 : tid;
    const int jm = jl > 0 ? tid - PI : tid, jp = jl < TJ - 1 ? tid + PI : tid;
    const bool jlo = j0 == 0, jhi = j0 + TJ >= s.nj, klo = k0 == 0, khi = k0 + TK >= s.nk;
    // one node of plane k: the pair's node e
    auto node = [&](auto kc, auto ec, bool fresh) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value, e = decltype(ec)::value;
        const double p = P[k][e];
        double w = P[k][1 - e], wl = P[k - 1][e], wh = P[k + 1][e];
        double q = lds[1 - e][k][e ? qp : qm], yl = lds[e][k][jm], yh = lds[e][k][jp];
        const unsigned mb = m[k] >> (8 * e);
        if (NEU && fresh) {
            unsigned nb = mb;
            // (opaque: the bits' comparisons are made here, not kept in
            // scalar registers for every plane across the half sweeps)
            asm volatile("" : "+v"(nb));
            w = (nb & (e ? SOR_IM : SOR_IP)) ? p : w;
            constexpr unsigned others = (e ? SOR_IP : SOR_IM) | SOR_JM | SOR_JP | SOR_KM | SOR_KP;
            if (__ballot(nb & others) != 0) {  // tiles at the other faces
                q = (nb & (e ? SOR_IP : SOR_IM)) ? p : q;
                yl = (nb & SOR_JM) ? p : yl;
                yh = (nb & SOR_JP) ? p : yh;
                wl = (nb & SOR_KM) ? p : wl;
                wh = (nb & SOR_KP) ? p : wh;
            }
        }
        const double v = sor_node<BOLTZ>(s, a, p, R[k][e], w + q, yl + yh, wl + wh);
        const double n = (mb & SOR_REG) ? v : p;
        P[k][e] = n;
        lds[e][k][tid] = n;
    };
    // Half sweep q: the first nodes of the planes of one parity, the second
    // ones of the other's (first = 1: odd planes' first nodes).  Waves whose
    // lines are too near the tile's ends to be right skip it.  With Neumann
    // bits to look at, such planes are left out too; without, all are made,
    // with no branches, so that their loads and sums overlap (measured both
    // ways: 96^3 walls 2.76 ms against 3.11 with the branches; the plates' 64 x
    // 64 x 256 64.4 ms against 61.1 with them).
    auto half = [&](auto firstc, int q, bool fresh) __attribute__((always_inline)) {
        constexpr int first = decltype(firstc)::value;
        if (!((jlo || jl > q) && (jhi || jl < TJ - 1 - q))) return;
        auto plane = [&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            constexpr int near = SOR_HALO;  // planes that every half sweep makes
            if (NEU && k < near && !(klo || k > q)) return;
            if (NEU && k > TK - 1 - near && !(khi || k < TK - 1 - q)) return;
            node(kc, std::integral_constant<int, ((k & 1) == first) ? 0 : 1>{}, fresh);
        };
        for_planes(plane, std::make_integer_sequence<int, TK - 2>{});
    };
    // planes whose first node is red: even ones where j + k0 is even
    const bool odd = ((j0 + (wave & 1) + k0) & 1) != 0;
    auto sweeps = [&](auto redc) __attribute__((always_inline)) {
        constexpr int red = decltype(redc)::value;
        for (int q = 0; q < ns; q += 2) {
            const bool fresh = own != 0 || q >= 2;
            half(std::integral_constant<int, red>{}, q, fresh);
            __syncthreads();
            half(std::integral_constant<int, 1 - red>{}, q + 1, fresh);
            __syncthreads();
        }
    };
    if (odd)
        sweeps(std::integral_constant<int, 1>{});
    else
        sweeps(std::integral_constant<int, 0>{});
    const int ci = ax.core(bx), ce = ax.core(bx + 1);
    const bool wj = j >= ay.core(by) && j < ay.core(by + 1);
    const bool w1 = wj && i >= ci && i < ce, w2 = wj && i + 1 >= ci && i + 1 < ce;
    const int kc = az.core(bz), ke = az.core(bz + 1);
    if (w1 && w2) {
#pragma unroll
        for (int k = 0; k < TK; k++)
            if (k0 + k >= kc && k0 + k < ke) *reinterpret_cast<D2*>(out + (ub + (unsigned)k * sk)) = P[k];
    } else if (w1 || w2) {  // a core that ends inside a pair
#pragma unroll
        for (int k = 0; k < TK; k++)
            if (k0 + k >= kc && k0 + k < ke) out[ub + (unsigned)k * sk + (w1 ? 0u : 1u)] = w1 ? P[k][0] : P[k][1];
    }
}

// every Neumann face node from the node its chain of copies ends at (an edge
// node copies a face node, which copies an interior one): what k_neumann's
// three phases leave
__global__ void __launch_bounds__(BLOCK)
    k_neumann_all(Stencil s, const uint8_t* __restrict__ nt, double* __restrict__ phi,
                  const double* __restrict__ stop) {
    if (*stop != 0.0) return;
    long long end;
    for (long long u = chunk_begin(s.nn, end) + threadIdx.x; u < end; u += BLOCK) {
        uint8_t t = nt[u];
        if (t == NT_REG || t == NT_DIR) continue;
        long long v = u;
        while (t != NT_REG && t != NT_DIR) {
            switch (t) {
                case NT_NEU_IM: v += 1; break;
                case NT_NEU_IP: v -= 1; break;
                case NT_NEU_JM: v += s.sj; break;
                case NT_NEU_JP: v -= s.sj; break;
                case NT_NEU_KM: v += s.sk; break;
                default: v -= s.sk; break;
            }
            t = nt[v];
        }
        phi[u] = phi[v];
    }
}

// Neumann copies; phase 0 = k faces, 1 = j faces, 2 = i faces, so edge and
// corner chains (an i face reads a j face reads a k face) resolve in order.
__global__ void __launch_bounds__(BLOCK)
    k_neumann(Stencil s, const uint8_t* __restrict__ nt, double* __restrict__ phi, int phase) {
    long long u = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (u >= s.nn) return;
    uint8_t t = nt[u];
    if (t == NT_REG || t == NT_DIR) return;
    int ph = t <= NT_NEU_IP ? 2 : (t <= NT_NEU_JP ? 1 : 0);
    if (ph != phase) return;
    phi[u] = nbr_of<double>(t, phi, u, s);
}

// The end of a batch of SOR sweeps: the residual's three sums to the host
// (pinned memory), and the stop flag when the criterion is met; out[3]: met
__global__ void __launch_bounds__(BLOCK)
    k_sor_check(double* __restrict__ scratch, int nb, int ref_rms, double nn, double tol, double* out) {
    if (scratch[PCG_FLAG] != 0.0) return;
    double r[3];
#pragma unroll
    for (int q = 0; q < 3; q++) r[q] = sum_parts(scratch + PART_F + q * PART_MAX, nb);
    if (threadIdx.x != 0) return;
    const double crit = ref_rms ? sqrt(r[0] / nn) : (r[2] > 0 ? sqrt(r[1] / r[2]) : sqrt(r[1]));
    for (int q = 0; q < 3; q++) out[q] = r[q];
    out[3] = crit < tol ? 1.0 : 0.0;
    if (crit < tol) scratch[PCG_FLAG] = 1.0;
}
__global__ void k_clear_flag(double* __restrict__ scratch) { scratch[PCG_FLAG] = 0.0; }

}  // namespace

static SorArgs sor_args(const pic_solver_params* p, const Stencil& s) {
    SorArgs a;
    a.omega = p->omega > 0 ? p->omega : 1.4;
    a.ieps = 1.0 / EPS0;
    a.itwos = 1.0 / s.twos;
    a.phi0 = p->phi0;
    a.n0 = p->n0;
    a.inv_te0 = 1.0 / (p->Te0 != 0 ? p->Te0 : 1.0);
    a.color = 0;
    return a;
}

// SOR with one launch per colour on the natural layout, in place
// (PIC_SOLVE_SOR_PLAIN); the tiled sweeps give the same values.
static int solve_sor_plain(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st) {
    const GridC& g = ctx->g;
    Stencil s = make_stencil(g, false);
    SorArgs a = sor_args(p, s);
    bool neu = has_neumann(ctx);
    int check = p->check_every > 0 ? p->check_every : 25;
    long long half_items = (long long)((g.ni + 1) / 2) * g.nj * g.nk;
    double r[3] = {0, 0, 0};
    int it;
    bool conv = false, fresh = false;  // fresh: r holds the residual of the current potential
    double crit = 0;
    for (it = 0; it < p->max_it; it++) {
        {
            PicProfScope ps(ctx, PIC_K_SOR);
            for (int c = 0; c < 2; c++) {
                a.color = c;
                k_sor<<<stencil_blocks(half_items), BLOCK, 0, ctx->stream>>>(s, a, ctx->ntype, ctx->phi, ctx->rho);
            }
            if (neu)
                for (int ph = 0; ph < 3; ph++)
                    k_neumann<<<grid_for((size_t)g.nn, BLOCK), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, ctx->phi,
                                                                                        ph);
        }
        PIC_HIP(ctx, hipGetLastError());
        fresh = false;
        if (it % check == 0) {  // PotentialSolver.cpp:124
            int rc = residual_norms(ctx, s, a, r);
            if (rc) return rc;
            fresh = true;
            crit = crit_value(p, r, (double)g.nn);
            if (crit < p->tol) {
                conv = true;
                break;
            }
        }
    }
    if (!fresh) {
        int rc = residual_norms(ctx, s, a, r);
        if (rc) return rc;
    }
    st->converged = conv;
    st->iterations = conv ? it + 1 : it;
    st->newton_iterations = 0;
    st->ref_l2 = std::sqrt(r[0] / (double)g.nn);
    st->rel_residual = r[2] > 0 ? std::sqrt(r[1] / r[2]) : std::sqrt(r[1]);
    return conv ? PIC_OK : PIC_NOT_CONVERGED;
}

// red-black sweeps on tiles: `sweeps` (1 or 2) from in to out
template <int PI, int TJ, int TK>
static void launch_sor_tile(pic_ctx* ctx, const Stencil& s, const SorArgs& a, bool neu, const double* in, double* out,
                            int sweeps, int own) {
    const TileAxis ax = tile_axis(s.ni, 2 * PI), ay = tile_axis(s.nj, TJ), az = tile_axis(s.nk, TK);
    const unsigned nb = ((unsigned)(ax.m * ay.m * az.m) + NXCD - 1) / NXCD * NXCD;
    const double* stop = ctx->scratch + PCG_FLAG;
    auto go = [&](auto kernel) {
        kernel<<<nb, PI * TJ, 0, ctx->stream>>>(s, a, ax, ay, az, ctx->sor_bits, in, out, ctx->rho, 2 * sweeps, own,
                                                stop);
    };
    if (a.n0 != 0.0) {
        if (neu)
            go(k_sor_tile<PI, TJ, TK, true, true>);
        else
            go(k_sor_tile<PI, TJ, TK, false, true>);
    } else {
        if (neu)
            go(k_sor_tile<PI, TJ, TK, true, false>);
        else
            go(k_sor_tile<PI, TJ, TK, false, false>);
    }
}

// The tile by the grid.  Small grids: the smallest tile, up to 400 of them
// (three fit a CU), since a launch then lasts as long as one tile's chain of
// half sweeps: 64^3 with 294 tiles 1.28 ms against 1.53 and 1.59 with the
// larger tiles, 96^3 with 968 tiles 3.56 against 2.75.  Larger grids without
// Neumann faces: 64 x 16 or 32 x 32 nodes of a plane, whichever needs fewer
// tiles (128^3 6.8 ms with 32 x 32, 8.5 with 64 x 16).  With them 64 x 16: whole
// lines put the i faces into the threads' own pairs (64 x 64 x 256 plates 61 ms
// against 98; 97 x 80 x 120 23.5 against 23.8).
static void sor_sweeps(pic_ctx* ctx, const Stencil& s, const SorArgs& a, bool neu, const double* in, double* out,
                       int sweeps, int own) {
    auto tiles = [&](int t, int u, int w) {
        return (long long)tile_axis(s.ni, t).m * tile_axis(s.nj, u).m * tile_axis(s.nk, w).m;
    };
    if (tiles(32, 16, 12) <= 400)
        launch_sor_tile<16, 16, 12>(ctx, s, a, neu, in, out, sweeps, own);
    else if (neu || tiles(64, 16, 16) < tiles(32, 32, 16))
        launch_sor_tile<32, 16, 16>(ctx, s, a, neu, in, out, sweeps, own);
    else
        launch_sor_tile<16, 32, 16>(ctx, s, a, neu, in, out, sweeps, own);
}

// Red-black SOR (PotentialSolver.cpp:69-166) on tiles.  The residual is
// checked after the first sweep and then every `check` sweeps (:124); the
// host queues the first RUN_AHEAD launches of the sweeps up to the next check
// before it waits for the last one, and once a check is met the launches
// behind it return at once (the stop flag), so the potential is the one that
// was checked.  Without memory for the second potential and the row bits the
// sweeps are made in place.
int pic_solve_sor(pic_ctx* ctx, const pic_solver_params* p, pic_solver_stats* st) {
    if (p->flags & PIC_SOLVE_SOR_PLAIN) return solve_sor_plain(ctx, p, st);
    const GridC& g = ctx->g;
    const size_t nn = (size_t)g.nn;
    Stencil s = make_stencil(g, false);
    SorArgs a = sor_args(p, s);
    const bool neu = has_neumann(ctx);
    const int check = p->check_every > 0 ? p->check_every : 25;
    if ((!ctx->sor_phi && hipMalloc(&ctx->sor_phi, nn * sizeof(double)) != hipSuccess) ||
        (!ctx->sor_bits && hipMalloc(&ctx->sor_bits, nn) != hipSuccess)) {
        (void)hipGetLastError();
        return solve_sor_plain(ctx, p, st);  // in place
    }
    int rc = pic_ensure_pin(ctx, 8 * sizeof(double));
    if (rc) return rc;
    for (auto& e : ctx->batch_ev)
        if (!e) PIC_HIP(ctx, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    volatile double* hp = ctx->pin;  // two batches of {three sums, criterion met}
    k_clear_flag<<<1, 1, 0, ctx->stream>>>(ctx->scratch);
    k_sor_bits<<<stencil_blocks(s.nn), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, ctx->sor_bits);
    double* buf[2] = {ctx->phi, ctx->sor_phi};
    const unsigned nbr = part_blocks(s.nn);
    const int ahead = ctx->prof.on ? 1 : 2;  // profiled runs count no launch that returns at once
    int it = 0, launches = 0;                // sweeps and launches queued
    int at[2], par[2], queued = 0, done = 0; // batches queued and waited for; their last sweep and buffer
    bool conv = false;
    int last = 0;
    auto wait_oldest = [&]() {  // for the oldest queued batch; conv: it met the criterion
        last = done & 1;
        const hipError_t e = pic_spin_event(ctx->batch_ev[last]);
        if (e != hipSuccess) return pic_hip_check(ctx, e, "SOR check");
        done++;
        conv = hp[4 * last + 3] != 0.0;
        return (int)PIC_OK;
    };
    while (!conv) {
        while (!conv && it < p->max_it && queued - done < ahead) {
            const int q = queued & 1;
            // sweep numbers 0, check, 2 check, ... are checked, and the last
            // (check may be as large as INT_MAX: only the first sweep and the last)
            const int upto = it == 0 ? 1 : check < p->max_it - it ? it + check : p->max_it;
            for (int m = 0; it < upto; m++) {
                if (m == RUN_AHEAD && queued > done) {
                    rc = wait_oldest();
                    if (rc) return rc;
                    if (conv) break;
                }
                PicProfScope ps(ctx, PIC_K_SOR);
                const int n = std::min(2, upto - it);
                sor_sweeps(ctx, s, a, neu, buf[launches & 1], buf[(launches & 1) ^ 1], n, it > 0);
                launches++;
                it += n;
            }
            if (conv) break;
            double* cur = buf[launches & 1];
            if (neu)
                k_neumann_all<<<stencil_blocks(s.nn), BLOCK, 0, ctx->stream>>>(s, ctx->ntype, cur,
                                                                              ctx->scratch + PCG_FLAG);
            k_resid<<<nbr, BLOCK, 0, ctx->stream>>>(s, a, ctx->ntype, cur, ctx->rho, ctx->scratch + PART_F);
            // only sweeps 0, check, 2 check, ... can end the solve
            const bool can = (it - 1) % check == 0;
            k_sor_check<<<1, BLOCK, 0, ctx->stream>>>(ctx->scratch, (int)nbr, p->tol_kind == PIC_TOL_REF_RMS,
                                                      (double)nn, can ? p->tol : 0.0, ctx->pin + 4 * q);
            PIC_HIP(ctx, hipGetLastError());
            PIC_HIP(ctx, hipEventRecord(ctx->batch_ev[q], ctx->stream));
            at[q] = it;
            par[q] = launches & 1;
            queued++;
        }
        if (conv || done == queued) break;
        rc = wait_oldest();
        if (rc) return rc;
    }
    if (par[last]) std::swap(ctx->phi, ctx->sor_phi);
    double r[3];
    for (int q = 0; q < 3; q++) r[q] = hp[4 * last + q];
    st->converged = conv;
    st->iterations = at[last];
    st->newton_iterations = 0;
    st->ref_l2 = std::sqrt(r[0] / (double)g.nn);
    st->rel_residual = r[2] > 0 ? std::sqrt(r[1] / r[2]) : std::sqrt(r[1]);
    return conv ? PIC_OK : PIC_NOT_CONVERGED;
}

int pic_poisson_internal_sor(pic_ctx* ctx, double tol, int max_it, pic_solver_stats* st) {
    pic_solver_params p{};
    p.method = PIC_SOLVER_SOR_RB;
    p.tol_kind = PIC_TOL_REL;
    p.tol = tol;
    p.max_it = max_it;
    int nmax = std::max(ctx->g.ni, std::max(ctx->g.nj, ctx->g.nk));
    p.omega = 2.0 / (1.0 + std::sin(3.141592653589793 / (nmax - 1)));
    p.check_every = 25;
    int rc = pic_ensure_ntype(ctx);
    if (rc) return rc;
    return pic_solve_sor(ctx, &p, st);
}
