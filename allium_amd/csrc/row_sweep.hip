// Direction sweeps of a 2D axis-aligned box grid, p = 1 and 2 (launch mode 3),
// restating src/sweep.cpp:366-475 for uniform geometry and directions that do
// not couple.
//
// A workgroup sweeps one (direction, group) through all nx + ny - 1 wavefronts of
// the mesh, one lane per row of elements: at step l the lane of row j solves
// element l - j of its row, so the trace in x stays in its registers, the trace
// in y comes from the next lane through LDS, and each lane streams through a row
// of its own.  Meshes with more rows than lanes go strip by strip, the last
// row's traces kept in LDS.
//
// Cell solve.  With t_d = |Omega_d| / h_d, the mass m and the upwind convection C
// of the unit interval, B = m^-1 C, the cell system times the inverse unit mass is
//   vol (t_x B (x) I + t_y I (x) B + sigma).
// B = V L V^-1 with L real: a pair of eigenvalues a +- i b as [[a, b], [-b, a]] and, at
// p = 2, a real one l0 (the roots of x^3 - 9 x^2 + 36 x - 60) that the pair couples
// into: L = [[l0, 1, t], [0, a, b], [0, -b, a]], the real Schur form.  In that basis
// of both axes the system is solved from the pair (x) pair unknowns (two 2 x 2
// rotations in the +- eigenspaces of the product of the two axes' J = [[0, 1], [-1, 0]])
// over pair (x) real (a rotation each) to real (x) real.  V is orthogonal under m but for
// the scales of its columns and a ratio of the pair's two scales (1.9 at p = 1, 1.7 at p = 2).  The traces are passed
// on in the basis of their own axis, so a step's chain from trace to trace is 2 Q^2
// multiply-adds, the solve, and a few additions; the transform of the source, the
// reciprocals and the transform to nodal values hang off it.
//
// Error (2-norm against extended precision): at p = 2 that of the LU (log-normal sigma, 150
// x 97: 2.3e-15, LU 2.9e-15) to twice it (constant sigma, 61 x 47: 4.6e-15, LU 2.2e-15); a
// basis of eigenvectors (condition 7 per axis) needs 12 instructions fewer and was at
// 1.5e-14 on the first.  At p = 1 3.7e-15 there (LU 2.6e-15, box sweeps 2.0e-14): the pair's
// unknowns are three times their trace.
//
// Bound by issue: about 350 (p = 2) and 170 (p = 1) instructions a step in each of a few
// waves per CU, 230 and 101 of them vector ones, one of those per 8 cycles.  A 9 x 9 LU in
// one lane with the traces read back from memory took 3 us a step.  Measured before / after
// (the best launch mode of each, one pair of vectors), us: 150 x 97 p = 2 S12 728 / 187, 300 x
// 300 p = 2 S12 2608 / 1178, 150 x 97 p = 1 S12 271 / 102, 32 x 32 p = 1 S8 45 / 30.
#include <algorithm>

#include "device.hpp"
#include "kernel_common.hpp"

namespace allium {

namespace {

// A trace that crosses an element is multiplied by r(z) = V_P (L + z)^-1 W0 (last row
// of V, first column of W), and a rounding of their constants errs with one sign in
// every element.  So some of them are neighbours (one unit in the last place) of the
// nearest doubles: V11 at p = 1, which leaves 4e-17 instead of 2.7e-16 (z = 0), and t,
// W00 and W20 at p = 2, 5e-18 instead of 1.3e-16.
template <int P>
struct Basis;
template <>
struct Basis<1> {
    static constexpr int R = 0;   // real eigenvalues
    static constexpr double l0 = 0.0, a = 2.0, b = 1.4142135623730950488, t = 0.0;
    static constexpr double V[2][2] = {{1.0, 0.0}, {-1.0, 1.4142135623730949234}};
    static constexpr double W[2][2] = {{4.0, -2.0}, {1.4142135623730950488, 1.4142135623730950488}};   // V^-1 m^-1
};
template <>
struct Basis<2> {
    static constexpr int R = 1;
    static constexpr double l0 = 3.6378342527444958, a = 2.6810828736277523, b = 3.0504301992474105;
    static constexpr double t = 0.24964484560420097115;
    static constexpr double V[3][3] = {{2.2420123818119873, 1.0734624624372482, 1.2377295589054893},
                                       {0.85327257928935929, -1.0240820485688007, -0.068423170697841346},
                                       {8.7090951703964432, 1.0, 0.0}};
    static constexpr double W[3][3] = {{0.2016957935665358026, 0.076762060461610951, 0.78348713677483162},
                                       {1.2434121383604055, -2.1685280900358954, 2.1765359610465764},
                                       {5.8276375688838841782, 0.52978617878836110, -0.88308266220483422}};
};

// largest deviation of W m V from I and of W C V from L
template <int P>
constexpr double basis_error()
{
    using E = Basis<P>;
    constexpr int Q = P + 1, R = E::R;
    constexpr double d1[2][2] = {{0.5, 0.5}, {-0.5, 0.5}};   // C: -(integral of phi_i' phi_j), + 1 at the last node
    constexpr double d2[3][3] = {{0.5, 2.0 / 3.0, -1.0 / 6.0}, {-2.0 / 3.0, 0.0, 2.0 / 3.0}, {1.0 / 6.0, -2.0 / 3.0, 0.5}};
    double worst = 0.0;
    for (int i = 0; i < Q; ++i)
        for (int j = 0; j < Q; ++j) {
            double id = i == j ? -1.0 : 0.0, l = 0.0;
            if (i >= R && j >= R) l = i == j ? E::a : (i < j ? E::b : -E::b);
            else if (i < R) l = j == 0 ? E::l0 : (j == 1 ? 1.0 : E::t);
            l = -l;
            for (int k = 0; k < Q; ++k)
                for (int n = 0; n < Q; ++n) {
                    double c = 0.0;
                    if constexpr (P == 1) c = d1[k][n];
                    else c = d2[k][n];
                    id += E::W[i][k] * unit_mass_1d<P>(k, n) * E::V[n][j];
                    l += E::W[i][k] * c * E::V[n][j];
                }
            worst = id > worst ? id : (-id > worst ? -id : worst);
            worst = l > worst ? l : (-l > worst ? -l : worst);
        }
    return worst;
}
static_assert(basis_error<1>() < 4e-15 && basis_error<2>() < 1e-14, "V, W and L to rounding");

// (c + d J)^-1 (u, v), n = 1 / (c^2 + d^2)
__device__ __forceinline__ void rotate(double c, double d, double n, double &u, double &v)
{
    const double w = fma(c, u, -d * v) * n;
    v = fma(c, v, d * u) * n;
    u = w;
}

// r (rows: basis in y, columns: in x) becomes the solution of the cell system
template <int P>
__device__ __forceinline__ void solve_modes(double sig, double tx, double ty, double (&r)[P + 1][P + 1])
{
    using E = Basis<P>;
    constexpr int R = E::R;
    const double c = fma(tx, E::a, fma(ty, E::a, sig)), dm = (tx - ty) * E::b, dp = (tx + ty) * E::b;
    double p1 = 0.5 * (r[R][R] + r[R + 1][R + 1]), p2 = 0.5 * (r[R][R + 1] - r[R + 1][R]);
    double m1 = 0.5 * (r[R][R] - r[R + 1][R + 1]), m2 = 0.5 * (r[R][R + 1] + r[R + 1][R]);
    rotate(c, dm, fast_rcp(fma(c, c, dm * dm)), p1, p2);
    rotate(c, dp, fast_rcp(fma(c, c, dp * dp)), m1, m2);
    r[R][R] = p1 + m1;
    r[R + 1][R + 1] = p1 - m1;
    r[R][R + 1] = p2 + m2;
    r[R + 1][R] = m2 - p2;
    if constexpr (R == 1) {
        // what the pair of an axis adds to its real eigenvalue
#pragma unroll
        for (int k = 1; k < 3; ++k) {
            r[0][k] = fma(-ty, fma(E::t, r[2][k], r[1][k]), r[0][k]);
            r[k][0] = fma(-tx, fma(E::t, r[k][2], r[k][1]), r[k][0]);
        }
        const double cx = fma(tx, E::a, fma(ty, E::l0, sig)), dx = tx * E::b;
        rotate(cx, dx, fast_rcp(fma(cx, cx, dx * dx)), r[0][1], r[0][2]);
        const double cy = fma(ty, E::a, fma(tx, E::l0, sig)), dy = ty * E::b;
        rotate(cy, dy, fast_rcp(fma(cy, cy, dy * dy)), r[1][0], r[2][0]);
        const double u = fma(E::t, r[2][0], r[1][0]), v = fma(E::t, r[0][2], r[0][1]);
        r[0][0] = fma(-ty, u, fma(-tx, v, r[0][0])) * fast_rcp(fma(tx, E::l0, fma(ty, E::l0, sig)));
    }
}

// s + c x for a constant c, without the term where c is 0
__device__ __forceinline__ double term(double c, double x, double s) { return c == 0.0 ? s : fma(c, x, s); }

// out[k][i] = sum A[k][b] A[i][a] x[b][a]
template <int Q>
__device__ __forceinline__ void both_axes(const double (&A)[Q][Q], const double (&x)[Q][Q], double (&out)[Q][Q])
{
    double h[Q][Q];
#pragma unroll
    for (int b = 0; b < Q; ++b)
#pragma unroll
        for (int i = 0; i < Q; ++i) {
            double s = A[i][0] * x[b][0];
#pragma unroll
            for (int a = 1; a < Q; ++a) s = term(A[i][a], x[b][a], s);
            h[b][i] = s;
        }
#pragma unroll
    for (int k = 0; k < Q; ++k)
#pragma unroll
        for (int i = 0; i < Q; ++i) {
            double s = A[k][0] * h[0][i];
#pragma unroll
            for (int b = 1; b < Q; ++b) s = term(A[k][b], h[b][i], s);
            out[k][i] = s;
        }
}

// the sweep of direction (a, g); SX, SY: Omega_x, Omega_y negative; tx, ty: vol t_d; SRC,
// ISO: which sources there are.  ytr: 2 x blockDim x Q
// traces of the last two steps; yline: nx x Q traces of a strip's last row (several strips)
template <int P, bool SRC, bool ISO, int SX, int SY>
__device__ __forceinline__ void sweep_rows(const SweepParams &p, int a, int g, double tx, double ty, double vol,
                                           double *ytr, double *yline)
{
    using E = Basis<P>;
    constexpr int Q = P + 1, N = Q * Q, D = 3;   // D: cells in registers, the loads of two under way
    const int nx = p.nel[0], ny = p.nel[1], T = (int)blockDim.x, j = (int)threadIdx.x;
    const long long base = ((long long)g * p.Nomega + a) * p.Ndof;
    const double tau = p.timedep ? p.tau : 0.0;
    const double *src = SRC ? p.src + base : nullptr, *iso = ISO ? p.iso + (long long)g * p.Ndof : nullptr;
    const double *sigma = p.sigma + (long long)g * p.Ne;
    for (int s = 0; s < ny; s += T) {
        const int rows = ny - s < T ? ny - s : T, steps = nx + rows - 1;
        const int row = s + j < ny ? s + j : ny - 1, erow = (SY ? ny - 1 - row : row) * nx;
        double q[D][N], w[D][N], sg[D], xt[Q];
        auto load = [&](int l, double (&qb)[N], double (&wb)[N], double &sb) {
            const int i0 = l - j, i = i0 < 0 ? 0 : (i0 < nx ? i0 : nx - 1);
            const int e = erow + (SX ? nx - 1 - i : i);
#pragma unroll
            for (int k = 0; k < N; ++k) {
                if constexpr (SRC) qb[k] = src[(long long)e * N + k];
                if constexpr (ISO) wb[k] = iso[(long long)e * N + k];
            }
            sb = sigma[e];
        };
#pragma unroll
        for (int k = 0; k < Q; ++k) xt[k] = 0.0;
        load(0, q[0], w[0], sg[0]);
        load(1, q[1], w[1], sg[1]);
        auto step = [&](int l, const double (&qb)[N], const double (&wb)[N], double sb) {
            const int i = l - j;
            const bool on = i >= 0 && i < nx && j < rows;
            double x[Q][Q], r[Q][Q];
#pragma unroll
            for (int b = 0; b < Q; ++b)
#pragma unroll
                for (int c = 0; c < Q; ++c) {
                    const int k = (SY ? P - b : b) * Q + (SX ? P - c : c);
                    x[b][c] = SRC && ISO ? qb[k] + wb[k] : (SRC ? qb[k] : wb[k]);
                }
            both_axes<Q>(E::W, x, r);
            // the trace in y: of the row before, one step back
            double yt[Q];
#pragma unroll
            for (int k = 0; k < Q; ++k) yt[k] = 0.0;
            if (j > 0) {
#pragma unroll
                for (int k = 0; k < Q; ++k) yt[k] = ytr[(((l + 1) & 1) * T + j - 1) * Q + k];
            } else if (s > 0 && on) {
#pragma unroll
                for (int k = 0; k < Q; ++k) yt[k] = yline[i * Q + k];
            }
            // (t_d is not taken into the constants: its rounding there would be the same
            // in every element)
#pragma unroll
            for (int k = 0; k < Q; ++k) {
                const double xk = tx * xt[k], yk = ty * yt[k];
#pragma unroll
                for (int c = 0; c < Q; ++c) {
                    r[k][c] = fma(E::W[c][0], xk, r[k][c]);
                    r[c][k] = fma(E::W[c][0], yk, r[c][k]);
                }
            }
            solve_modes<P>((sb + tau) * vol, tx, ty, r);
            double yo[Q];
#pragma unroll
            for (int k = 0; k < Q; ++k) {
                double vx = E::V[P][0] * r[k][0], vy = E::V[P][0] * r[0][k];
#pragma unroll
                for (int c = 1; c < Q; ++c) {
                    vx = term(E::V[P][c], r[k][c], vx);
                    vy = term(E::V[P][c], r[c][k], vy);
                }
                xt[k] = on ? vx : xt[k];
                yo[k] = vy;
            }
            // a lane without a cell writes its own slot too: only such lanes read it
#pragma unroll
            for (int k = 0; k < Q; ++k) ytr[((l & 1) * T + j) * Q + k] = yo[k];
            if (yline && on && j == T - 1) {
#pragma unroll
                for (int k = 0; k < Q; ++k) yline[i * Q + k] = yo[k];
            }
            // orders LDS only: psi stores and the loads under way stay in flight
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            both_axes<Q>(E::V, r, x);
            if (on) {
                double *out = p.psi + base + (long long)(erow + (SX ? nx - 1 - i : i)) * N;
#pragma unroll
                for (int b = 0; b < Q; ++b)
#pragma unroll
                    for (int c = 0; c < Q; ++c) out[(SY ? P - b : b) * Q + (SX ? P - c : c)] = x[b][c];
            }
        };
        for (int l = 0; l < steps; l += D) {   // steps past the end have no cell
            load(l + 2, q[2], w[2], sg[2]);
            step(l, q[0], w[0], sg[0]);
            load(l + 3, q[0], w[0], sg[0]);
            step(l + 1, q[1], w[1], sg[1]);
            load(l + 4, q[1], w[1], sg[1]);
            step(l + 2, q[2], w[2], sg[2]);
        }
    }
}

template <int P, bool SRC, bool ISO>
__global__ void __launch_bounds__(512) k_sweep_rows(SweepParams p, double hx, double hy, int strips)
{
    extern __shared__ double lds[];
    constexpr int Q = P + 1;
    const int a = blockIdx.x, g = blockIdx.y;
    const double ox = p.omega[4 * a], oy = p.omega[4 * a + 1];
    const double tx = fabs(ox) * hy, ty = fabs(oy) * hx, vol = hx * hy;
    double *yline = strips > 1 ? lds + 2 * (int)blockDim.x * Q : nullptr;
    if (ox < 0) {
        if (oy < 0) sweep_rows<P, SRC, ISO, 1, 1>(p, a, g, tx, ty, vol, lds, yline);
        else sweep_rows<P, SRC, ISO, 1, 0>(p, a, g, tx, ty, vol, lds, yline);
    } else {
        if (oy < 0) sweep_rows<P, SRC, ISO, 0, 1>(p, a, g, tx, ty, vol, lds, yline);
        else sweep_rows<P, SRC, ISO, 0, 0>(p, a, g, tx, ty, vol, lds, yline);
    }
}

template <int P>
hipError_t launch_p(const DeviceSweep &ds, const SweepParams &prm, int block, size_t lds, hipStream_t s)
{
    const dim3 grid(prm.Nomega, prm.G);
    const int strips = (prm.nel[1] + block - 1) / block;
    const double hx = ds.h2[0], hy = ds.h2[1];
    if (prm.src && prm.iso)
        hipLaunchKernelGGL((k_sweep_rows<P, true, true>), grid, dim3(block), lds, s, prm, hx, hy, strips);
    else if (prm.src)
        hipLaunchKernelGGL((k_sweep_rows<P, true, false>), grid, dim3(block), lds, s, prm, hx, hy, strips);
    else
        hipLaunchKernelGGL((k_sweep_rows<P, false, true>), grid, dim3(block), lds, s, prm, hx, hy, strips);
    return hipGetLastError();
}

}  // namespace

static long rows_lds(const DeviceSweep &ds, int block)
{
    const int Q = ds.prm.p + 1;
    return 8L * Q * (2L * block + (ds.prm.nel[1] > block ? ds.prm.nel[0] : 0));
}

int row_sweep_block(const DeviceSweep &ds)
{
    const SweepParams &p = ds.prm;
    if (p.dim != 2 || !p.uniform || !ds.angle_independent || ds.lumped || (p.p != 1 && p.p != 2)) return 0;
    const int block = std::max(64, std::min((p.nel[1] + 63) / 64 * 64, std::min(512, ds.dir_block)));
    return rows_lds(ds, block) <= 65536 ? block : 0;
}

hipError_t launch_row_sweep(const DeviceSweep &ds, const SweepParams &prm, hipStream_t s)
{
    const int block = row_sweep_block(ds);
    if (!block) return hipErrorInvalidValue;
    if (!prm.src && !prm.iso) return hipErrorInvalidValue;
    const size_t lds = (size_t)rows_lds(ds, block);
    return prm.p == 1 ? launch_p<1>(ds, prm, block, lds, s) : launch_p<2>(ds, prm, block, lds, s);
}

}  // namespace allium
