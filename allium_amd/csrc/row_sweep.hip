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
// B = V L V^-1 with L real: one eigenvalue l0 (p = 2) and a pair a +- i b as
// [[a, b], [-b, a]].  At p = 2 they are the roots of x^3 - 9 x^2 + 36 x - 60, the
// condition of V is 7.  In that basis of both axes the system falls into scalars,
// 2 x 2 rotations and, for pair and pair, two 2 x 2 rotations in the +- eigenspaces
// of the product of the two axes' J = [[0, 1], [-1, 0]].  The traces are passed on in
// the basis of their own axis, so a step's chain from trace to trace is 2 Q^2
// multiply-adds, the rotations, and 2 Q^2 more; the transform of the source, the
// reciprocals and the transform to nodal values hang off it.
//
// Bound by issue: about 330 (p = 2) and 150 (p = 1) instructions a step in each of a
// few waves per CU, one per about 8 cycles.  A 9 x 9 LU in one lane with the traces
// read back from memory took 3 us a step.  Measured before / after (the best launch
// mode of each), us: 150 x 97 p = 2 S12 728 / 186, 300 x 300 p = 2 S12 2608 / 1200,
// 150 x 97 p = 1 S12 271 / 102, 32 x 32 p = 1 S8 45 / 30.
#include <algorithm>

#include "device.hpp"
#include "kernel_common.hpp"

namespace allium {

namespace {

template <int P>
struct Eig;
template <>
struct Eig<1> {
    static constexpr int R = 0;   // real eigenvalues
    static constexpr double l0 = 0.0, a = 2.0, b = 1.41421356237309504880;
    static constexpr double V[2][2] = {{1.0, 0.0}, {-1.0, 1.41421356237309504880}};
    static constexpr double W[2][2] = {{4.0, -2.0}, {1.41421356237309504880, 1.41421356237309504880}};   // V^-1 m^-1
};
template <>
struct Eig<2> {
    static constexpr int R = 1;
    // A trace that crosses an element is multiplied by
    // r(z) = W00 / (l0 + z) + ((a + z) W10 - b W20) / ((a + z)^2 + b^2), with terms of 5 and
    // -4 for a value of 1: its constants rounded to nearest leave 4.9e-16 in every
    // element, always with one sign.  These are neighbours of the nearest doubles
    // (within 3 units in the last place) with r exact to 4e-17, 5e-18 at z = 0.
    static constexpr double l0 = 3.6378342527444953, a = 2.6810828736277528, b = 3.0504301992474105;
    static constexpr double V[3][3] = {{0.257433446063711987, -0.06871672303185599, 0.388146850560913172},
                                       {0.097974882877588054, 0.011012558561205972, -0.37446069925093946},
                                       {1.0, 1.0, 0.0}};
    static constexpr double W[3][3] = {{18.297498174845845, 1.792695240633402691, 4.710388009495045932},
                                       {-15.297498174845845, -3.29269524063340269, 4.289611990504954067},
                                       {8.34328048949488, -5.63643099835961522, 5.364352843454024324}};
};

// (c + d J)^-1 (u, v), n = 1 / (c^2 + d^2)
__device__ __forceinline__ void rotate(double c, double d, double n, double &u, double &v)
{
    const double w = fma(c, u, -d * v) * n;
    v = fma(c, v, d * u) * n;
    u = w;
}

// r (rows: eigenvectors in y, columns: in x) becomes the solution of the cell system
template <int P>
__device__ __forceinline__ void solve_modes(double sig, double tx, double ty, double (&r)[P + 1][P + 1])
{
    using E = Eig<P>;
    constexpr int R = E::R;
    if constexpr (R == 1) {
        r[0][0] *= fast_rcp(fma(tx, E::l0, fma(ty, E::l0, sig)));
        const double cx = fma(tx, E::a, fma(ty, E::l0, sig)), dx = tx * E::b;
        rotate(cx, dx, fast_rcp(fma(cx, cx, dx * dx)), r[0][R], r[0][R + 1]);
        const double cy = fma(ty, E::a, fma(tx, E::l0, sig)), dy = ty * E::b;
        rotate(cy, dy, fast_rcp(fma(cy, cy, dy * dy)), r[R][0], r[R + 1][0]);
    }
    const double c = fma(tx, E::a, fma(ty, E::a, sig)), dm = (tx - ty) * E::b, dp = (tx + ty) * E::b;
    double p1 = 0.5 * (r[R][R] + r[R + 1][R + 1]), p2 = 0.5 * (r[R][R + 1] - r[R + 1][R]);
    double m1 = 0.5 * (r[R][R] - r[R + 1][R + 1]), m2 = 0.5 * (r[R][R + 1] + r[R + 1][R]);
    rotate(c, dm, fast_rcp(fma(c, c, dm * dm)), p1, p2);
    rotate(c, dp, fast_rcp(fma(c, c, dp * dp)), m1, m2);
    r[R][R] = p1 + m1;
    r[R + 1][R + 1] = p1 - m1;
    r[R][R + 1] = p2 + m2;
    r[R + 1][R] = m2 - p2;
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
    using E = Eig<P>;
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
