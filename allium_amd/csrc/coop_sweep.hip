// Cooperative cell solves of the 3D local DG systems whose matrices do not fit
// one lane (p = 2: 27 x 27) or differ from element to element (p = 1: 8 x 8 on
// general geometry), restating src/sweep.cpp:366-475.
//
// LPC lanes (8 at p = 1, 16 at p = 2) solve one cell (e, a, g): lane t holds rows
// t and, at p = 2, t + 16 of
//   A = sum_d Omega_d G_d + sigma M + tau Mt + sum_{outflow} (Omega.n) F
// and of the right-hand side (source, isotropic source, upwind traces), then
// the cell's lanes run an LU without pivoting (A + A^T is positive definite)
// and a column-oriented back substitution; the pivot row and each solved
// unknown reach the other lanes by DPP row broadcast.  No LDS, no barriers.
//
// Assembly.  The cells of a level are ordered by element, so the 4 (p = 2) or 8
// (p = 1) cells of a wave mostly share their element and differ in direction,
// and column j of all their matrices is one small matrix product: directions
// x (coefficient of each element matrix) times (element matrices) x rows.  That
// is v_mfma_f64_4x4x4_4b: lane i + 4 b + 16 k supplies coefficient k of cell i,
// lane r + 4 b + 16 k entry (row 4 b + r, column j) of element matrix k, and lane
// r + 4 b + 16 i receives the sum for cell i.  One MFMA adds the three gradient
// blocks and the mass, a second the three faces that node j lies on (weight
// max(Omega.n, 0)), a third, with the same face operand and the weighted upwind
// trace at node j as coefficient, the inflow part of the right-hand side.  So a
// matrix entry is loaded once per wave and not once per cell, as columns of
// consecutive lanes.  A wave with several elements repeats the product per
// element with the other cells' coefficients zero.  Reading each row per cell
// (27 doubles 216 B apart in every lane) kept the L1's return path busy 94 % of
// the time.  Measured before / after, ms: 16^3 + 18^3 + 21^3 p = 2 S12 batch 10.7 / 8.2,
// uniform 24^3 p = 2 S12 5.3 / 4.2, 26 x 23 x 29 p = 1 S8 (one lane per cell before)
// 1.80 / 0.90, 48^3 p = 1 S8 8.2 / 3.2.  What is left is issue: 2000 to 2300 vector and
// 162 matrix instructions (a few more where a wave holds several elements) per wave of
// four 27 x 27 cells, counted, at two waves per SIMD.
#include <type_traits>
#include <utility>

#include "device.hpp"
#include "kernel_common.hpp"

namespace allium {

bool coop_supported(int dim, int p) { return dim == 3 && p == 2; }
bool coop_level_supported(int dim, int p, bool uniform) { return dim == 3 && (p == 2 || (p == 1 && !uniform)); }

namespace {

template <int P>
struct Coop {
    static constexpr int Q = P + 1, N = Q * Q * Q, NF = Q * Q;
    static constexpr int LPC = P == 1 ? 8 : 16;             // lanes per cell
    static constexpr int RS = (N + LPC - 1) / LPC;          // rows per lane
    static constexpr int CPW = 64 / LPC;                    // cells per wave
};

// lane L of each cell's LPC lanes, to all of them.  Every lane is active where
// this is called, so the source lane is always valid and bound_ctrl (zero for
// an invalid source) only spares the copy of an old value.
template <int LPC, int L, typename T>
__device__ __forceinline__ T cell_bcast(T x)
{
    static_assert(L >= 0 && L < LPC && (LPC == 8 || LPC == 16), "row_newbcast takes a lane of the row");
    if constexpr (LPC == 16) {
        return __builtin_amdgcn_update_dpp((T)0, x, 0x150 + L, 0xF, 0xF, true);
    } else {
        // two cells in a row of 16: banks 0, 1 take lane L, banks 2, 3 lane L + 8
        const T lo = __builtin_amdgcn_update_dpp((T)0, x, 0x150 + L, 0xF, 0xF, true);
        return __builtin_amdgcn_update_dpp(lo, x, 0x150 + L + 8, 0xF, 0xC, false);
    }
}

// One LU step on W columns (RS rows a lane): each row takes n[r] times the pivot
// row's entry, which the FMA reads from lane L of the cell by DPP.  The compiler
// makes a 64-bit DPP move and an FMA of this; v_fmac_f64_dpp is both (788 FMAs
// and 431 moves of a 27 x 27 solve became 756 FMAs).  A DPP operand may not be
// read in the two instructions after the one that writes it: the s_nop covers
// what ran before, and inside a block no instruction reads what one of the two
// before it wrote.  Nothing here may read an MFMA result directly (the compiler
// inserts the waits for its own instructions only): the first step is plain C++.
// DST: rows of the other row set (never the pivot's), SELF: the pivot's row set.
#define ALLIUM_FMAC(D, S, M, L, B) "v_fmac_f64_dpp %" #D ", %" #S ", %" #M " row_newbcast:%" #L " row_mask:0xf bank_mask:" #B "\n"
template <int L>
__device__ __forceinline__ void fmac_self16(double &a, double &b, double &c, double &d, double n)
{
    asm("s_nop 1\n" ALLIUM_FMAC(0, 0, 4, 5, 0xf) ALLIUM_FMAC(1, 1, 4, 5, 0xf) ALLIUM_FMAC(2, 2, 4, 5, 0xf)
            ALLIUM_FMAC(3, 3, 4, 5, 0xf)
        : "+v"(a), "+v"(b), "+v"(c), "+v"(d)
        : "v"(n), "i"(L));
}
template <int L>
__device__ __forceinline__ void fmac_self16(double &a, double n)
{
    asm("s_nop 1\n" ALLIUM_FMAC(0, 0, 1, 2, 0xf) : "+v"(a) : "v"(n), "i"(L));
}
template <int L>
__device__ __forceinline__ void fmac_cross16(double &a, double &b, double &c, double &d, double sa, double sb, double sc,
                                             double sd, double n)
{
    asm("s_nop 1\n" ALLIUM_FMAC(0, 4, 8, 9, 0xf) ALLIUM_FMAC(1, 5, 8, 9, 0xf) ALLIUM_FMAC(2, 6, 8, 9, 0xf)
            ALLIUM_FMAC(3, 7, 8, 9, 0xf)
        : "+v"(a), "+v"(b), "+v"(c), "+v"(d)
        : "v"(sa), "v"(sb), "v"(sc), "v"(sd), "v"(n), "i"(L));
}
template <int L>
__device__ __forceinline__ void fmac_cross16(double &a, double sa, double n)
{
    asm("s_nop 1\n" ALLIUM_FMAC(0, 1, 2, 3, 0xf) : "+v"(a) : "v"(sa), "v"(n), "i"(L));
}
// two cells in a row of 16: banks 0, 1 take lane L, banks 2, 3 lane L + 8
template <int L>
__device__ __forceinline__ void fmac_self8(double &a, double &b, double &c, double &d, double n)
{
    asm("s_nop 1\n" ALLIUM_FMAC(0, 0, 4, 5, 0x3) ALLIUM_FMAC(1, 1, 4, 5, 0x3) ALLIUM_FMAC(2, 2, 4, 5, 0x3)
            ALLIUM_FMAC(3, 3, 4, 5, 0x3) ALLIUM_FMAC(0, 0, 4, 6, 0xc) ALLIUM_FMAC(1, 1, 4, 6, 0xc)
                ALLIUM_FMAC(2, 2, 4, 6, 0xc) ALLIUM_FMAC(3, 3, 4, 6, 0xc)
        : "+v"(a), "+v"(b), "+v"(c), "+v"(d)
        : "v"(n), "i"(L), "i"(L + 8));
}
template <int L>
__device__ __forceinline__ void fmac_self8(double &a, double n)
{
    asm("s_nop 1\n" ALLIUM_FMAC(0, 0, 1, 2, 0x3) "s_nop 1\n" ALLIUM_FMAC(0, 0, 1, 3, 0xc)
        : "+v"(a)
        : "v"(n), "i"(L), "i"(L + 8));
}
// the value of lane L of the cell where an asm above may have written x
template <int LPC, int L>
__device__ __forceinline__ double cell_bcast_after(double x)
{
    double y;
    if constexpr (LPC == 16)
        asm("s_nop 1\nv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(y) : "v"(x), "i"(L));
    else
        asm("s_nop 1\nv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0x3\n"
            "v_mov_b64_dpp %0, %1 row_newbcast:%3 row_mask:0xf bank_mask:0xc"
            : "=&v"(y)
            : "v"(x), "i"(L), "i"(L + 8));
    return y;
}
#undef ALLIUM_FMAC

template <typename F, int... K>
__device__ __forceinline__ void for_each_k(F &&f, std::integer_sequence<int, K...>)
{
    (f(std::integral_constant<int, K>{}), ...);
}

// Columns J .. of one LU step with pivot K (the last column is the right-hand
// side): M[r][j] += n[r] * (pivot row's M[K / LPC][j]).
template <int LPC, int RS, int NC, int K, int J>
__device__ __forceinline__ void lu_columns(double (&M)[RS][NC], const double (&n)[RS])
{
    constexpr int kr = K / LPC, L = K % LPC, left = NC - J;
    if constexpr (left > 0) {
        constexpr int W = left >= 4 ? 4 : 1;
        constexpr bool self = LPC * kr + LPC - 1 > K, cross = kr + 1 < RS;
        static_assert(RS <= 2, "the other row set is the next one");
        if constexpr (cross) {
            if constexpr (W == 4)
                fmac_cross16<L>(M[kr + 1][J], M[kr + 1][J + 1], M[kr + 1][J + 2], M[kr + 1][J + 3], M[kr][J],
                                M[kr][J + 1], M[kr][J + 2], M[kr][J + 3], n[kr + 1]);
            else
                fmac_cross16<L>(M[kr + 1][J], M[kr][J], n[kr + 1]);
        }
        if constexpr (self) {
            if constexpr (LPC == 16) {
                if constexpr (W == 4) fmac_self16<L>(M[kr][J], M[kr][J + 1], M[kr][J + 2], M[kr][J + 3], n[kr]);
                else fmac_self16<L>(M[kr][J], n[kr]);
            } else {
                if constexpr (W == 4) fmac_self8<L>(M[kr][J], M[kr][J + 1], M[kr][J + 2], M[kr][J + 3], n[kr]);
                else fmac_self8<L>(M[kr][J], n[kr]);
            }
        }
        lu_columns<LPC, RS, NC, K, J + W>(M, n);
    }
}

__device__ __forceinline__ double mfma4(double a, double b, double c)
{
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ T by_axis(int ax, T x, T y, T z)
{
    return ax == 0 ? x : (ax == 1 ? y : z);
}

// m[r][j]: the lanes (16 per axis) whose row of set r has the coordinate of node j
// on the lane's axis
template <int P>
struct SideLanes {
    unsigned long long m[Coop<P>::RS][Coop<P>::N];
};
template <int P>
constexpr SideLanes<P> side_lanes()
{
    using C = Coop<P>;
    constexpr int Q = C::Q;
    SideLanes<P> s{};
    for (int r = 0; r < C::RS; ++r)
        for (int j = 0; j < C::N; ++j)
            for (int l = 0; l < 48; ++l) {
                const int t = l % C::LPC, row = t + C::LPC * r < C::N ? t + C::LPC * r : t;
                const int step = l / 16 == 0 ? 1 : (l / 16 == 1 ? Q : Q * Q);
                if ((row / step) % Q == (j / step) % Q) s.m[r][j] |= 1ull << l;
            }
    return s;
}
template <int P>
constexpr SideLanes<P> kSideLanes = side_lanes<P>();

// the cells of one wave: items first .. first + CPW of the instance's level
template <int P, bool UNI, typename T>
__device__ __forceinline__ void coop_wave(const SweepParams &p, const CoopLevel &cl, int inst, long long wg0)
{
    using C = Coop<P>;
    constexpr int Q = C::Q, N = C::N, NF = C::NF, LPC = C::LPC, RS = C::RS;
    const int nc = cl.ncells[inst], items = nc * p.G;
    const int first = (int)(wg0 - cl.start[inst]) + (int)(threadIdx.x >> 6) * C::CPW;
    if (first >= items) return;   // wave-uniform
    // every table read through p is global memory
    const auto g_cells = as_global(p.cells);
    const auto g_psi = as_global(p.psi);
    // slots past the level's end repeat its last cell and are not stored
    auto cell_at = [&](int slot, int &e, int &a, int &g) {
        const int it = first + slot < items ? first + slot : items - 1;
        g = p.G > 1 ? it / nc : 0;
        const uint32_t cell = g_cells[cl.cbeg[inst] + (it - g * nc)];
        e = (int)(cell >> 10);
        a = (int)(cell & 1023u);
    };

    double A[RS][N], b[RS];
#pragma unroll
    for (int r = 0; r < RS; ++r) {
        b[r] = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j) A[r][j] = 0.0;
    }

    const int lane = threadIdx.x & 63, grp = lane >> 4, half = P == 1 ? (lane >> 3) & 1 : 0, t = lane & (LPC - 1);
    // The cell whose coefficients the lane supplies: coefficient grp of the
    // gradients (Omega_x, Omega_y, Omega_z) and the mass (sigma), axis grp of the faces.
    int eA, aA, gA;
    cell_at((lane & 3) + 4 * half, eA, aA, gA);
    // ... and the cell whose rows it holds
    const int slot = grp + 4 * half;
    const bool store = first + slot < items;
    int eD, aD, gD;
    cell_at(slot, eD, aD, gD);
    const long long off = ((long long)gD * p.Nomega + aD) * p.Ndof + (long long)eD * N;
    const auto g_omega = as_global(p.omega);
    const double om[3] = {g_omega[4 * aA], g_omega[4 * aA + 1], g_omega[4 * aA + 2]};
    const double sig = as_global(p.sigma)[(long long)gA * p.Ne + eA];
    const int ax = grp < 3 ? grp : 0;
    const double om_ax = by_axis(ax, om[0], om[1], om[2]);
    const auto own = g_psi + (((long long)gA * p.Nomega + aA) * p.Ndof + (long long)eA * N);
    const int sax = by_axis(ax, 1, Q, Q * Q);                       // node stride along the axis
    const long long nb = (long long)by_axis(ax, p.stride[0], p.stride[1], p.stride[2]) * N;
    // rows of the lane and their face-lexicographic index
    int row[RS], kt[RS];
#pragma unroll
    for (int r = 0; r < RS; ++r) {
        row[r] = t + LPC * r < N ? t + LPC * r : t;   // a lane without a last row repeats its first
        const int i0 = row[r] % Q, i1 = (row[r] / Q) % Q, i2 = row[r] / (Q * Q);
        kt[r] = by_axis(ax, i1 + Q * i2, i0 + Q * i2, i0 + Q * i1);
    }

    unsigned long long todo = ~0ull;
    while (todo) {
        // a uniform mesh has one element's matrices: one pass for every cell
        const int es = UNI ? eA : __builtin_amdgcn_readlane(eA, __builtin_ctzll(todo));
        const bool mine = UNI || eA == es;
        todo = UNI ? 0 : todo & ~__ballot(mine);
        const int c2 = fast_div(es, p.stride[2], p.inv_nel01), rem = es - c2 * p.stride[2];
        const int c1 = fast_div(rem, p.nel[0], p.inv_nel0), c0 = rem - c1 * p.nel[0];
        const int c_ax = by_axis(ax, c0, c1, c2), last = by_axis(ax, p.nel[0], p.nel[1], p.nel[2]) - 1;
        // the element's faces normal to the lane's axis: table index of the low
        // one and distance to the high one
        int flo, fdh;
        if constexpr (UNI) {
            flo = 2 * ax;
            fdh = 1;
        } else {
            const int f0 = p.foff[0] + c0 + p.fext[0][0] * (c1 + p.fext[0][1] * c2);
            const int f1 = p.foff[1] + c0 + p.fext[1][0] * (c1 + p.fext[1][1] * c2);
            const int f2 = p.foff[2] + c0 + p.fext[2][0] * (c1 + p.fext[2][1] * c2);
            flo = by_axis(ax, f0, f1, f2);
            fdh = by_axis(ax, 1, p.fext[1][0], p.fext[2][0] * p.fext[2][1]);
        }
        // Omega.n on the low and high side
        const bool in_lo = c_ax > 0, in_hi = c_ax < last;
        double dlo, dhi;
        if constexpr (UNI) {
            dlo = -om_ax;
            dhi = om_ax;
        } else {
            const auto fn = as_global(p.fnor) + 3LL * flo, fh = fn + 3LL * fdh;
            dlo = fma(om[2], fn[2], fma(om[1], fn[1], om[0] * fn[0]));
            dhi = fma(om[2], fh[2], fma(om[1], fh[1], om[0] * fh[0]));
            dlo = in_lo ? -dlo : dlo;
        }
        dlo = mine && grp < 3 ? dlo : 0.0;
        dhi = mine && grp < 3 ? dhi : 0.0;
        // where the upwind trace at node j of the side is read: lo + j, hi + j; no
        // inflow there reads zeros (at most 35 past the start, the buffer has 64)
        const auto zero = as_global(p.zeros);
        gptr<const double> lo = zero, hi = zero;
        if (dlo < 0) {
            if (in_lo) lo = own - nb + P * sax;
            else if ((p.refl_mask >> (2 * ax)) & 1)
                lo = g_psi + ((long long)gA * p.Nomega + as_global(p.refl)[aA * 6 + 2 * ax]) * p.Ndof + (long long)eA * N;
        }
        if (dhi < 0) {
            if (in_hi) hi = own + nb - P * sax;
            else if ((p.refl_mask >> (2 * ax + 1)) & 1)
                hi = g_psi + ((long long)gA * p.Nomega + as_global(p.refl)[aA * 6 + 2 * ax + 1]) * p.Ndof +
                     (long long)eA * N;
        }
        const double coef = mine ? (grp < 3 ? om_ax : sig) : 0.0;
        // element matrix grp, column-major, and the face block of the lane's axis
        // (symmetric: entry (k, l) read at l NF + k)
        const long long ee = UNI ? 0 : es;
        auto mat = grp < 3 ? as_global(p.Gd) + (ee * 3 + grp) * (N * N) : as_global(p.Mu) + ee * (N * N);
        auto fb = as_global(p.Fface) + (long long)flo * (NF * NF);
        // table offset of face node (j0, j1, j2) from (0, 0, 0): one part per axis,
        // along the lane's axis the step to the high face
        int fo[3][Q];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int st = d == 0 ? NF : by_axis(ax, d == 1 ? NF : Q * NF, d == 1 ? 0 : Q * NF, Q * NF);
#pragma unroll
            for (int v = 0; v < Q; ++v) fo[d][v] = ax == d ? (v == P ? fdh * NF * NF : 0) : v * st;
        }
        // nodes by their coordinate on the lane's axis: 0 low side, P high side,
        // between them neither
        auto dv = [&](int v) { return v == 0 ? dlo : (v == P ? dhi : 0.0); };
        auto uv = [&](int v) { return v == 0 ? lo : (v == P ? hi : zero); };
        // Columns in node order, CH at a time: the loads of the next chunk are issued
        // before the products of this one (NB = 2 buffers).  At p = 1 all columns fit.
        // (One column at a time, for a third wave in the registers, is slower on uniform
        // meshes too: 24^3 S12 4.76 ms against 4.24, 3^3 S4 106 us against 81.)
        constexpr int CH = P == 1 ? N : Q, NC = N / CH, NB = NC > 1 ? 2 : 1;
        static_assert(N % CH == 0, "whole chunks");
        double u[NB][CH], m[NB][CH][RS], f[NB][CH][RS];
        auto load = [&](auto cc) {
            constexpr int c = decltype(cc)::value, v = c % NB;
            if constexpr (c < NC) {
#pragma unroll
                for (int i = 0; i < CH; ++i) {
                    const int j = c * CH + i, j0 = j % Q, j1 = (j / Q) % Q, j2 = j / (Q * Q);
                    u[v][i] = by_axis(ax, uv(j0), uv(j1), uv(j2))[j];
                    const auto fj = fb + (fo[0][j0] + fo[1][j1] + fo[2][j2]);
#pragma unroll
                    for (int r = 0; r < RS; ++r) {
                        m[v][i][r] = mat[j * N + row[r]];
                        f[v][i][r] = fj[kt[r]];
                    }
                }
            }
        };
        if constexpr (NB == 2) load(std::integral_constant<int, 0>{});
        for_each_k(
            [&](auto cc) {
                constexpr int c = decltype(cc)::value, v = c % NB;
                load(std::integral_constant<int, c + NB - 1>{});
#pragma unroll
                for (int i = 0; i < CH; ++i) {
                    const int j = c * CH + i;
                    const double d = by_axis(ax, dv(j % Q), dv((j / Q) % Q), dv(j / (Q * Q)));
                    const double out = d > 0 ? d : 0.0, inn = -d * u[v][i];
#pragma unroll
                    for (int r = 0; r < RS; ++r) {
                        // the row is on the same side of the lane's axis as the node
                        const double fz =
                            __builtin_amdgcn_inverse_ballot_w64(kSideLanes<P>.m[r][j]) ? f[v][i][r] : 0.0;
                        b[r] = mfma4(inn, fz, b[r]);
                        A[r][j] = mfma4(coef, m[v][i][r], mfma4(out, fz, A[r][j]));
                    }
                }
            },
            std::make_integer_sequence<int, NC>{});
        if (p.timedep) {
            const auto mt = as_global(p.Mt) + ee * (N * N);
            const double tau = mine && grp == 0 ? p.tau : 0.0;
#pragma unroll
            for (int j = 0; j < N; ++j)
#pragma unroll
                for (int r = 0; r < RS; ++r) {
                    const double v = mt[j * N + row[r]];
                    A[r][j] = mfma4(tau, grp == 0 ? v : 0.0, A[r][j]);
                }
        }
    }
#pragma unroll
    for (int r = 0; r < RS; ++r) {
        if (p.src) b[r] += as_global(p.src)[off + row[r]];
        if (p.iso) b[r] += as_global(p.iso)[(long long)gD * p.Ndof + (long long)eD * N + row[r]];
    }

    // ---- LU without pivoting ------------------------------------------------
    // Pivot row k is row set k / LPC of lane k % LPC.  Every lane runs every
    // update; a row at or above the pivot takes multiplier 0.
    // Rows past the last one follow along and are never a pivot.
    constexpr bool kAsm = sizeof(T) == 8;
    T M[RS][N + 1], ninv[RS];   // ninv: minus the reciprocal of the row's own pivot
#pragma unroll
    for (int r = 0; r < RS; ++r) {
        ninv[r] = (T)0;
        M[r][N] = (T)b[r];
#pragma unroll
        for (int j = 0; j < N; ++j) M[r][j] = (T)A[r][j];
    }
    for_each_k(
        [&](auto kc) {
            constexpr int k = decltype(kc)::value, kr = k / LPC, kl = k % LPC;
            T piv;
            if constexpr (kAsm && k > 0) piv = cell_bcast_after<LPC, kl>(M[kr][k]);
            else piv = cell_bcast<LPC, kl>(M[kr][k]);
            const T rp = fast_rcp(piv);
            ninv[kr] = t == kl ? -rp : ninv[kr];
            T n[RS];
#pragma unroll
            for (int r = 0; r < RS; ++r) {
                n[r] = (T)0;
                if (r >= kr) n[r] = -(M[r][k] * rp);
                if (r == kr) n[r] = t > kl ? n[r] : (T)0;
            }
            if constexpr (kAsm && k > 0) {
                lu_columns<LPC, RS, N + 1, k, k + 1>(M, n);
            } else {
#pragma unroll
                for (int j = k + 1; j <= N; ++j) {
                    const T pj = cell_bcast<LPC, kl>(M[kr][j]);
#pragma unroll
                    for (int r = 0; r < RS; ++r)
                        if (LPC * r + LPC - 1 > k) M[r][j] = fma(n[r], pj, M[r][j]);
                }
            }
        },
        std::make_integer_sequence<int, N>{});

    // ---- back substitution, one unknown per step: the rows above k take -U(., k) x_k
    for_each_k(
        [&](auto kc) {
            constexpr int k = N - 1 - decltype(kc)::value, kr = k / LPC, kl = k % LPC;
            const T nown = M[kr][N] * ninv[kr];   // -x_k on its lane
#pragma unroll
            for (int r = 0; r <= kr; ++r) {
                const T c = r < kr || t < kl ? M[r][k] : (T)0;
                if constexpr (kAsm && LPC == 16) fmac_cross16<kl>(M[r][N], nown, c);
                else if constexpr (kAsm) M[r][N] = fma(cell_bcast_after<LPC, kl>(nown), c, M[r][N]);
                else M[r][N] = fma(cell_bcast<LPC, kl>(nown), c, M[r][N]);
            }
        },
        std::make_integer_sequence<int, N>{});
    if (store) {
#pragma unroll
        for (int r = 0; r < RS; ++r)
            if (t + LPC * r < N) g_psi[off + t + LPC * r] = (double)-(M[r][N] * ninv[r]);
    }
}

// BATCH: the instances' parameters are the device array prms (a level of
// several instances); otherwise p0, one instance.  The two are separate
// instantiations so that the parameters' address space is known (a pointer
// selected between the two would be generic and its loads flat).
template <int P, bool UNI, typename T, bool BATCH>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(P == 1 ? 4 : 2)))
k_sweep_coop(SweepParams p0, const SweepParams *__restrict__ prms, CoopLevel cl)
{
    // Workgroups go to the 8 XCDs round robin (blockIdx.x % 8).  Each XCD takes
    // a contiguous run of the level's cells instead, so the cells of one element
    // (adjacent in the element-ordered level) share that XCD's L2.
    const int nwg = (int)gridDim.x, x = (int)(blockIdx.x & 7u), q = (int)(blockIdx.x >> 3);
    const int per = nwg >> 3, rem = nwg & 7;
    const long long wg = (long long)x * per + (x < rem ? x : rem) + q;
    // each instance's items start on a multiple of kCoopCells, so the instance (and
    // with it every parameter read through p) is uniform over the workgroup
    const long long wg0 = wg * (4 * Coop<P>::CPW);
    int inst = 0;
    while (inst + 1 < cl.ninst && wg0 >= cl.start[inst + 1]) ++inst;
    if constexpr (BATCH)
        coop_wave<P, UNI, T>(*(const SweepParams *)as_global(prms + inst), cl, inst, wg0);
    else
        coop_wave<P, UNI, T>(p0, cl, inst, wg0);
}

template <int P, bool UNI>
hipError_t launch_pu(const SweepParams &p0, const SweepParams *d_prms, const CoopLevel &cl, int precision, hipStream_t s)
{
    const long long items = cl.start[cl.ninst];
    if (items <= 0) return hipSuccess;
    constexpr int per = 4 * Coop<P>::CPW;
    static_assert(P != 2 || per == kCoopCells, "instances start on a workgroup");
    const dim3 grid((unsigned)((items + per - 1) / per)), block(256);
    // FP32 solves of uniform p = 2 cells saved nothing (24^3 S12: 4.72 ms against 4.57
    // in FP64, with one column at a time): they are the FP64 ones
    constexpr bool f32 = !(P == 2 && UNI);
    using F = std::conditional_t<f32, float, double>;
    if constexpr (P == 2) {
        if (d_prms) {
            if (precision == 1 && f32)
                hipLaunchKernelGGL((k_sweep_coop<P, UNI, F, true>), grid, block, 0, s, p0, d_prms, cl);
            else
                hipLaunchKernelGGL((k_sweep_coop<P, UNI, double, true>), grid, block, 0, s, p0, d_prms, cl);
            return hipGetLastError();
        }
    } else if (d_prms) {
        return hipErrorInvalidValue;   // batches are p = 2
    }
    if (precision == 1 && f32)
        hipLaunchKernelGGL((k_sweep_coop<P, UNI, F, false>), grid, block, 0, s, p0, d_prms, cl);
    else
        hipLaunchKernelGGL((k_sweep_coop<P, UNI, double, false>), grid, block, 0, s, p0, d_prms, cl);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_coop_level(const SweepParams &p0, const SweepParams *d_prms, const CoopLevel &cl, int dim, int p,
                             bool uniform, int precision, hipStream_t s)
{
    if (!coop_level_supported(dim, p, uniform)) return hipErrorInvalidValue;
    if (p == 1) return launch_pu<1, false>(p0, d_prms, cl, precision, s);
    return uniform ? launch_pu<2, true>(p0, d_prms, cl, precision, s)
                   : launch_pu<2, false>(p0, d_prms, cl, precision, s);
}

}  // namespace allium
