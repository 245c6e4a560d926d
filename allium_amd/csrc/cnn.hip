// Learned low-order flux correction: a 5-layer 3x3x3 convolutional network
// on the element-centred grid, with BF16 MFMA forward and backward kernels
// (FP32 accumulation) for gfx950 and an FP32 Adam optimiser.  No counterpart
// in the reference; it stands in for the diffusion synthetic acceleration of
// src/transport_op.hpp:38-59 inside the source iteration.
//
// Convolution as an implicit GEMM on v_mfma_f32_16x16x32_bf16: a wave owns 4
// tiles of 16 consecutive voxels (rows of the A tiles) and all output channels
// (N tiles of 16); the K dimension runs over (kernel offset, input channel) in
// chunks of 8 channels of one offset, so every A operand is one 16-byte load
// of a channels-last voxel row.  Lane l holds A[l % 16][8 (l / 16) + t],
// B[8 (l / 16) + t][l % 16] and D[4 (l / 16) + r][l % 16].
//
// Weight gradients: a (sample, z) plane is shared by one to four workgroups.  Rows of
// the output gradient and of the input stay channels-last in LDS; rows are visited
// in chains one dilation apart, so a step stages one new row per z plane, and the
// matrix operands (voxels as the K dimension) are read transposed.  The partials of
// the workgroups are reduced in a second pass in a fixed order, so gradients are
// deterministic.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/allium_cnn.h"
#include "cnn_internal.hpp"

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int NL = 5;
constexpr int CI_[NL] = {3, 32, 32, 32, 32};
constexpr int CO_[NL] = {32, 32, 32, 32, 1};
constexpr int CIP_[NL] = {8, 32, 32, 32, 32};
constexpr int COP_[NL] = {32, 32, 32, 32, 16};
constexpr int HID = 32;

struct Geo {
    int B, nz, ny, nx;
    long long T;   // voxels
    int dil;       // dilation of the 3x3x3 taps: offsets are dil * (-1, 0, 1) per axis
};
constexpr int kMaxDil = 8;

// ---------------------------------------------------------------------------
// convolution (forward, and backward-data with flipped/transposed weights)
// MODE 0: + bias, ReLU, bf16 out [T][COP]
// MODE 1: + bias, FP32 out [T] (channel 0)
// MODE 2: masked by (mask[T][COP] > 0), bf16 out [T][COP]
// ---------------------------------------------------------------------------
// A workgroup computes one 8 x 8 x 8 tile of voxels with eight waves; a wave
// owns MT = 4 16-voxel row tiles (two y rows of one z plane each), so every B
// operand it loads (a 16-byte weight row) feeds MT MFMAs.  A dilated 3x3x3
// stencil couples only voxels of one sub-grid (x mod d, y mod d, z mod d),
// where it is an undilated stencil: the tile is taken in one sub-grid and its
// 10 x 10 x 10 halo is loaded into LDS once, so each input voxel feeds its 27
// taps from LDS instead of 27 cache reads.  Each output element accumulates
// its K steps (tap-major, then 8-channel chunks) in order.
//
// Tiles are 8 x 8 x 8 voxels on eight waves, or 4 x 4 x 4 on one wave where a
// sub-grid is too narrow to fill the large one.
constexpr int kConvMT = 4;
template <int TE>
struct Tile {
    static constexpr int E = TE, H = TE + 2, halo = H * H * H, waves = TE * TE * TE / (16 * kConvMT);
    // voxel of row v of a wave's operand tile t: (i, j, k) in the tile
    static __device__ __forceinline__ void voxel(int w, int t, int v, int &i, int &j, int &k)
    {
        if constexpr (TE == 8) { i = v & 7; j = 2 * t + (v >> 3); k = w; }
        else { i = v & 3; j = v >> 2; k = t; }
    }
};

struct TileGeo {
    int nsx, nsy, nsz;   // sub-grid extents (the largest, at offset 0)
    int ntx, nty, ntz;   // tiles per sub-grid axis
};

__host__ __device__ inline TileGeo tile_geo(const Geo &g, int e)
{
    TileGeo t;
    t.nsx = (g.nx + g.dil - 1) / g.dil;
    t.nsy = (g.ny + g.dil - 1) / g.dil;
    t.nsz = (g.nz + g.dil - 1) / g.dil;
    t.ntx = (t.nsx + e - 1) / e;
    t.nty = (t.nsy + e - 1) / e;
    t.ntz = (t.nsz + e - 1) / e;
    return t;
}

template <int CIP, int COP, int MODE, int TE>
__global__ void __launch_bounds__(64 * Tile<TE>::waves) k_conv_t(Geo g, const bf16 *__restrict__ in, const bf16 *__restrict__ W,
                                                const float *__restrict__ bias, bf16 *__restrict__ out_bf,
                                                float *__restrict__ out_f, const bf16 *__restrict__ mask)
{
    constexpr int CH = CIP / 8, NCH = 27 * CH, KS = (NCH + 3) / 4, NT = COP / 16, MT = kConvMT;
    static_assert(CIP % 8 == 0 && COP % 16 == 0, "padded channel counts");
    // voxel stride in LDS: the channels, unpadded (timed against 16, 32 and 48
    // bytes of padding per voxel, which were 28 % slower in a 64^3 inference)
    constexpr int VS = CIP * 2;
    using TL = Tile<TE>;
    static_assert(MT * 16 * TL::waves == TE * TE * TE, "a workgroup's voxels are one tile");
    extern __shared__ __align__(16) unsigned char halo[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, grp = lane >> 4;
    const TileGeo tg = tile_geo(g, TE);
    // workgroup -> (batch, sub-grid offset, tile)
    long long q = blockIdx.x;
    const int tx = (int)(q % tg.ntx); q /= tg.ntx;
    const int ty = (int)(q % tg.nty); q /= tg.nty;
    const int tz = (int)(q % tg.ntz); q /= tg.ntz;
    const int d = g.dil;
    const int sx = (int)(q % d); q /= d;
    const int sy = (int)(q % d); q /= d;
    const int sz = (int)(q % d); q /= d;
    const long long b = q;
    const long long plane = (long long)g.nx * g.ny, vol = plane * g.nz;
    // halo: CH 16-byte chunks per voxel, zeros outside the grid
    for (int c = threadIdx.x; c < TL::halo * CH; c += 64 * TL::waves) {
        const int hv = c / CH, part = c - hv * CH;
        const int hx = hv % TL::H, hy = (hv / TL::H) % TL::H, hz = hv / (TL::H * TL::H);
        const int x = sx + d * (tx * TE + hx - 1), y = sy + d * (ty * TE + hy - 1), z = sz + d * (tz * TE + hz - 1);
        const bool ok = x >= 0 && x < g.nx && y >= 0 && y < g.ny && z >= 0 && z < g.nz;
        const long long m = ok ? b * vol + (long long)z * plane + (long long)y * g.nx + x : 0;
        const bf16x8 v = *reinterpret_cast<const bf16x8 *>(in + m * CIP + part * 8);
        const bf16x8 zero8 = {};
        *reinterpret_cast<bf16x8 *>(halo + hv * VS + part * 16) = ok ? v : zero8;
    }
    __syncthreads();
    // this lane's operand rows
    int hbase[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        int i, j, k;
        TL::voxel(w, t, lane & 15, i, j, k);
        hbase[t] = ((k + 1) * TL::H + (j + 1)) * TL::H + (i + 1);
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[i][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x8 zero8 = {};
    for (int s = 0; s < KS; ++s) {
        const int c = 4 * s + grp;
        const bool cv = c < NCH;
        const int cc = cv ? c : 0;
        const int o = cc / CH;
        const int ci0 = (cc - o * CH) * 8;
        const int dz = o / 9 - 1, dy = (o / 3) % 3 - 1, dx = o % 3 - 1;
        const int doff = (dz * TL::H + dy) * TL::H + dx;
        bf16x8 a[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const bf16x8 v = *reinterpret_cast<const bf16x8 *>(halo + (hbase[i] + doff) * VS + ci0 * 2);
            a[i] = cv ? v : zero8;
        }
        bf16x8 bw[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const bf16x8 v = *reinterpret_cast<const bf16x8 *>(W + ((long long)o * COP + nt * 16 + (lane & 15)) * CIP + ci0);
            bw[nt] = cv ? v : zero8;
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bw[nt], acc[i][nt], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int jc = nt * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // output row 4 grp + r of operand tile t
                int i, j, k;
                TL::voxel(w, t, 4 * grp + r, i, j, k);
                const int x = sx + d * (tx * TE + i), y = sy + d * (ty * TE + j), z = sz + d * (tz * TE + k);
                if (x >= g.nx || y >= g.ny || z >= g.nz) continue;
                const long long mo = b * vol + (long long)z * plane + (long long)y * g.nx + x;
                float val = acc[t][nt][r];
                if constexpr (MODE == 0) {
                    val = fmaxf(val + bias[jc], 0.f);
                    out_bf[mo * COP + jc] = (bf16)val;
                } else if constexpr (MODE == 1) {
                    if (jc == 0) out_f[mo] = val + bias[0];
                } else {
                    val = (float)mask[mo * COP + jc] > 0.f ? val : 0.f;
                    out_bf[mo * COP + jc] = (bf16)val;
                }
            }
        }
}

template <int CIP, int COP, int MODE>
void launch_conv(const Geo &g, const bf16 *in, const bf16 *W, const float *bias, bf16 *out_bf, float *out_f,
                 const bf16 *mask, hipStream_t s)
{
    // Padded voxels of either tiling.  The small tile loads 3.4 halo voxels per output
    // instead of 1.95, so it is taken where it more than halves them
    // (at exactly half, a forward pass on 49 x 15 x 34 took 99 instead of 94 us; with
    // this rule 40 random grids of 8 to 64 took 0.89 to 1.00 times as long as before): a layer with
    // dilation 8 on 32^3 (4^3 sub-grids) computed eight times its voxels (8 x 32^3,
    // 32 to 32 channels: 150 -> 45 us forward, 155 -> 55 us backward; at dilation 1
    // the large tile takes 29 us).
    const long long subs = (long long)g.B * g.dil * g.dil * g.dil;
    const TileGeo t8 = tile_geo(g, 8), t4 = tile_geo(g, 4);
    const long long n8 = subs * t8.ntx * t8.nty * t8.ntz, n4 = subs * t4.ntx * t4.nty * t4.ntz;
    if (n8 * 512 > 2 * n4 * 64)
        hipLaunchKernelGGL((k_conv_t<CIP, COP, MODE, 4>), dim3((unsigned)n4), dim3(64 * Tile<4>::waves),
                           (size_t)Tile<4>::halo * CIP * 2, s, g, in, W, bias, out_bf, out_f, mask);
    else
        hipLaunchKernelGGL((k_conv_t<CIP, COP, MODE, 8>), dim3((unsigned)n8), dim3(64 * Tile<8>::waves),
                           (size_t)Tile<8>::halo * CIP * 2, s, g, in, W, bias, out_bf, out_f, mask);
}

// ---------------------------------------------------------------------------
// weight and bias gradient partials: part[workgroup][28][COP][CIP]; entry 27 is the
// bias gradient in every column
// ---------------------------------------------------------------------------
// eight voxels of the lane's channel: two transposing reads of 4 voxels x 16 channels
// per 16 lanes (lane 4 v + c of a group gives voxel v, channels 4 c .. 4 c + 3, and
// receives channel 4 v + c of the four voxels); every lane of the wave takes part
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bf16x8 tr_pair(const bf16 *lo, const bf16 *hi)
{
    using lds4 = __attribute__((address_space(3))) bf16x4;
    const bf16x4 l = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4 *)lo);
    const bf16x4 h = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4 *)hi);
    return __builtin_shufflevector(l, h, 0, 1, 2, 3, 4, 5, 6, 7);
}

constexpr int kWgradWaves = 8;

// nshare workgroups per (batch, z) plane, which divide its dilation residues of
// y, or its rows where there are fewer residues than shares.  A K step is 32
// voxels of a row; the rows are taken in chains y, y + dil, y + 2 dil, ..., so
// that a step finds two of the three input rows of each of its z planes in LDS (a
// ring of four row sets) and stages one: a third of the reads.  Rows stay in
// memory order (voxel, channel): the matrix operands need eight voxels of one
// channel per lane, which ds_read_b64_tr_b16 takes from four voxels by sixteen
// channels at any voxel offset, so the dx shifts cost nothing.  (With rows
// transposed by the stores and eight 2-byte reads per shifted operand, the LDS
// reads took 116 us of 8 x 32^3, 32 to 32 channels, at 256 workgroups of four
// waves; now 45 us.) The next step's global reads are in flight in registers
// during this step's MFMAs (two steps ahead timed the same); as a store only
// touches the ring's fourth set, one barrier per step is enough.  Eight waves
// share the operand tiles (16 input channels of a tap, or with 8 input channels
// two taps), each for all output channels.
template <int CIP, int COP>
__global__ void __launch_bounds__(64 * kWgradWaves) k_wgrad(Geo g, int nshare, const bf16 *__restrict__ gz,
                                               const bf16 *__restrict__ a, float *__restrict__ part)
{
    constexpr int NW = kWgradWaves, NTH = 64 * NW, NTO = COP / 16, NTI = (CIP + 15) / 16;
    constexpr int TPT = CIP < 16 ? 16 / CIP : 1;          // taps per operand tile
    constexpr int WT = NW / NTI;                          // waves over the taps of an input channel tile
    constexpr int NTT = (27 + TPT - 1) / TPT, NB = (NTT + WT - 1) / WT;   // tap tiles, and per wave
    constexpr int XW = 32, XS = XW + 2 * kMaxDil;         // voxels per K step, staged per row
    constexpr int CHI = CIP / 8, CHO = COP / 8;           // 16-byte chunks per voxel
    constexpr int AV = CIP, GV = COP;   // LDS voxel strides (bf16)
    constexpr int NA = (3 * XS * CHI + NTH - 1) / NTH;
    static_assert(NTT * TPT > 27 || NB * WT * TPT > 27, "a tile is left for the bias gradient");
    static_assert(XW * CHO <= NTH && NW % NTI == 0 && (TPT == 1 || NTI == 1), "one chunk of gz per thread; tiles divide the waves");
    __shared__ __attribute__((aligned(16))) bf16 gR[2][XW * GV];
    __shared__ __attribute__((aligned(16))) bf16 aR[4][3][XS * AV];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int share = blockIdx.x % nshare, pl = blockIdx.x / nshare, z = pl % g.nz, b = pl / g.nz;
    const int dl = g.dil, xr = XW + 2 * dl, nxs = (g.nx + XW - 1) / XW;
    const bool by_res = min(dl, g.ny) >= nshare;
    const int ya = by_res ? 0 : (int)((long long)g.ny * share / nshare);
    const int yb = by_res ? g.ny : (int)((long long)g.ny * (share + 1) / nshare);
    const int r0 = by_res ? share : 0, dr = by_res ? nshare : 1, r1 = min(dl, yb - ya);
    const bf16x8 zero8 = {}, one8 = zero8 + (bf16)1.f;
    struct Regs { bf16x8 a[NA], g; } q;
    // position in the share's steps: x chunk, y residue, row
    struct Pos { int xs, r, y; };
    // reads of a step into registers: gradient row y, input rows y + dil of the three
    // planes; out-of-grid chunks read voxel 0 and are zeroed by a select
    auto load = [&](const Pos &p) {
        const int x0 = p.xs * XW, y = p.y;
        {
            const int xi = threadIdx.x / CHO, c = threadIdx.x % CHO;
            const bool ok = xi < XW && x0 + xi < g.nx && y >= ya;
            const long long v = ok ? (((long long)b * g.nz + z) * g.ny + y) * g.nx + x0 + xi : 0;
            const bf16x8 r = *reinterpret_cast<const bf16x8 *>(gz + v * COP + 8 * c);
            q.g = ok ? r : zero8;
        }
        const int yy = y + dl;
#pragma unroll
        for (int k = 0; k < NA; ++k) {
            const int i = threadIdx.x + NTH * k;
            const int c = i % CHI, rest = i / CHI;
            const int xp = rest % XS, r3 = rest / XS;
            const int xx = x0 - dl + xp, zz = z + (r3 - 1) * dl;
            const bool ok = r3 < 3 && xp < xr && xx >= 0 && xx < g.nx && yy >= 0 && yy < g.ny && zz >= 0 && zz < g.nz;
            const long long v = ok ? (((long long)b * g.nz + zz) * g.ny + yy) * g.nx + xx : 0;
            const bf16x8 r = *reinterpret_cast<const bf16x8 *>(a + v * CIP + 8 * c);
            q.a[k] = ok ? r : zero8;
        }
    };
    // this lane's part of the transposing reads: voxel and channel chunk of its 16-lane
    // group's 4 x 16 block (the group holds voxels 8 grp .. 8 grp + 7 of the step)
    const int rv = 8 * (lane >> 4) + ((lane & 15) >> 2), rc = lane & 3;
    const int cit = w % NTI, tap0 = w / NTI;
    int aoff[NB], adz[NB], ady[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        int o = (tap0 + i * WT) * TPT + (TPT > 1 ? 4 * rc / CIP : 0);
        o = o < 27 ? o : 26;
        adz[i] = o / 9;
        ady[i] = (o / 3) % 3 - 1;
        aoff[i] = (rv + dl * (o % 3)) * AV + (TPT > 1 ? (4 * rc) % CIP : cit * 16 + 4 * rc);
    }
    f32x4 acc[NTO][NB];
#pragma unroll
    for (int m = 0; m < NTO; ++m)
#pragma unroll
        for (int i = 0; i < NB; ++i) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    // a chain (x chunk, y residue r) opens with two steps that only stage rows
    // ya + r - dil and ya + r
    Pos cp = {r1 > r0 ? 0 : nxs, r0, ya + r0 - 2 * dl};
    auto advance = [&](Pos &p) {
        p.y += dl;
        if (p.y >= yb) {
            p.r += dr;
            if (p.r >= r1) { p.r = r0; ++p.xs; }
            p.y = ya + p.r - 2 * dl;
        }
    };
    if (cp.xs < nxs) load(cp);
    for (int e = 0; cp.xs < nxs; ++e) {
        if (threadIdx.x < XW * CHO)
            *reinterpret_cast<bf16x8 *>(&gR[e & 1][(threadIdx.x / CHO) * GV + 8 * (threadIdx.x % CHO)]) = q.g;
#pragma unroll
        for (int k = 0; k < NA; ++k) {
            const int i = threadIdx.x + NTH * k;
            const int c = i % CHI, rest = i / CHI;
            const int xp = rest % XS, r3 = rest / XS;
            if (r3 < 3) *reinterpret_cast<bf16x8 *>(&aR[e & 3][r3][xp * AV + 8 * c]) = q.a[k];
        }
        __syncthreads();
        const bool compute = cp.y >= ya;
        advance(cp);
        if (cp.xs < nxs) load(cp);
        if (!compute) continue;
        bf16x8 av[NTO];
#pragma unroll
        for (int m = 0; m < NTO; ++m) {
            const bf16 *p = &gR[e & 1][rv * GV + m * 16 + 4 * rc];
            av[m] = tr_pair(p, p + 4 * GV);
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const bf16 *p = &aR[(e - 1 + ady[i]) & 3][adz[i]][aoff[i]];
            bf16x8 bv = tr_pair(p, p + 4 * AV);
            // the tap after the last multiplies by ones: the bias gradient
            if ((tap0 + i * WT) * TPT + (TPT > 1 ? (lane & 15) / CIP : 0) == 27) bv = one8;
#pragma unroll
            for (int m = 0; m < NTO; ++m)
                acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv, acc[m][i], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int n = lane & 15, o = (tap0 + i * WT) * TPT + (TPT > 1 ? n / CIP : 0);
        const int ci = TPT > 1 ? n % CIP : cit * 16 + n;
        if (o > 27) continue;
#pragma unroll
        for (int m = 0; m < NTO; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                part[(((long long)blockIdx.x * 28 + o) * COP + m * 16 + 4 * (lane >> 4) + q) * CIP + ci] = acc[m][i][q];
    }
}

// grad[o][co][ci], then the bias gradient [co] (packed, real sizes) = sums of the
// partials.  A block sums 64 outputs: each of its four waves adds every fourth
// partial in four chains (sixteen loads in flight) and the sums are added in a fixed
// order, so the result does not depend on timing.
__global__ void __launch_bounds__(256) k_wgrad_reduce(const float *__restrict__ part, int nparts, int COP, int CIP,
                                                      int CO, int CI, float *__restrict__ grad)
{
    __shared__ float red[4][64];
    const int nw = 27 * CO * CI, n = nw + CO;
    const int jl = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + jl;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    if (i < n) {
        const int o = i < nw ? i / (CO * CI) : 27, rem = i - o * CO * CI;
        const int co = i < nw ? rem / CI : rem, ci = i < nw ? rem - co * CI : 0;
        const long long stride = 28LL * COP * CIP;
        const float *p0 = part + ((long long)o * COP + co) * CIP + ci;
        int p = sl;
#pragma unroll 4
        for (; p + 12 < nparts; p += 16)
#pragma unroll
            for (int k = 0; k < 4; ++k) s[k] += p0[(p + 4 * k) * stride];
        for (; p < nparts; p += 4) s[0] += p0[p * stride];
    }
    red[sl][jl] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (sl == 0 && i < n) grad[i] = ((red[0][jl] + red[1][jl]) + red[2][jl]) + red[3][jl];
}

// x [T][3] float -> [T][8] bf16
__global__ void k_pack_input(long long T, const float *__restrict__ x, bf16 *__restrict__ xb)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < T * 8; i += (long long)gridDim.x * blockDim.x) {
        const long long v = i >> 3;
        const int c = (int)(i & 7);
        xb[i] = c < 3 ? (bf16)x[v * 3 + c] : (bf16)0.f;
    }
}

// master FP32 layer (W[27][CO][CI], b[CO]) -> bf16 forward [27][COP][CIP],
// bf16 backward-data [27][CIP][COP] (offset flipped), FP32 bias [COP]
__global__ void k_pack_layer(const float *__restrict__ Wm, const float *__restrict__ bm, int CO, int CI, int COP,
                             int CIP, bf16 *__restrict__ Wf, bf16 *__restrict__ Wb, float *__restrict__ bias)
{
    const int n = 27 * COP * CIP;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int o = i / (COP * CIP), rem = i - o * COP * CIP, co = rem / CIP, ci = rem - co * CIP;
        const float v = (co < CO && ci < CI) ? Wm[(o * CO + co) * CI + ci] : 0.f;
        Wf[i] = (bf16)v;
        Wb[((26 - o) * CIP + ci) * COP + co] = (bf16)v;
        if (i < COP) bias[i] = i < CO ? bm[i] : 0.f;
    }
}

// loss: g[T][16] bf16 (channel 0 = 2 (out - target) / T), lpart[block] = sum diff^2
__global__ void __launch_bounds__(256) k_loss(long long T, const float *__restrict__ out, const float *__restrict__ tgt,
                                              bf16 *__restrict__ g, double *__restrict__ lpart)
{
    __shared__ double red[256];
    double s = 0.0;
    const float scale = 2.0f / (float)T;
    for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < T; v += (long long)gridDim.x * blockDim.x) {
        const float d = out[v] - tgt[v];
        s += (double)d * d;
        g[v * 16] = (bf16)(scale * d);
#pragma unroll
        for (int c = 1; c < 16; ++c) g[v * 16 + c] = (bf16)0.f;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) lpart[blockIdx.x] = red[0];
}

__global__ void k_adam(long n, float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

// ---- source-iteration correction -------------------------------------------
// ravg[e] = sum_i w_i r[e n + i] ; part[block] = sum ravg^2
__global__ void __launch_bounds__(256) k_elem_avg(long long Ne, int n, const double *__restrict__ w,
                                                  const double *__restrict__ r, double *__restrict__ ravg,
                                                  double *__restrict__ part)
{
    __shared__ double red[256];
    double s = 0.0;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < Ne; e += (long long)gridDim.x * blockDim.x) {
        double v = 0.0;
        for (int i = 0; i < n; ++i) v = fma(w[i], r[e * n + i], v);
        ravg[e] = v;
        s += v * v;
    }
    if (!part) return;   // block-uniform
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// scale = sqrt(mean ravg^2) (one block)
__global__ void k_scale(const double *__restrict__ part, int nb, long long Ne, double *__restrict__ scale)
{
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) scale[0] = sqrt(red[0] / (double)Ne);
}

// network input [Ne][8] bf16: (ravg / scale, log sigma_t, sigma_s / sigma_t)
__global__ void k_make_input(long long Ne, const double *__restrict__ ravg, const double *__restrict__ scale,
                             const double *__restrict__ sigt, const double *__restrict__ sigs, bf16 *__restrict__ xb)
{
    const double s = scale[0];
    const double inv = s > 0.0 ? 1.0 / s : 0.0;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < Ne; e += (long long)gridDim.x * blockDim.x) {
        const double st = sigt[e];
        xb[e * 8 + 0] = (bf16)(float)(ravg[e] * inv);
        xb[e * 8 + 1] = (bf16)(float)log(st);
        xb[e * 8 + 2] = (bf16)(float)(sigs[e] / st);
#pragma unroll
        for (int c = 3; c < 8; ++c) xb[e * 8 + c] = (bf16)0.f;
    }
}

// phi[e n + i] += scale * out[e]
__global__ void k_apply_corr(long long Ne, int n, const float *__restrict__ out, const double *__restrict__ scale,
                             double *__restrict__ phi)
{
    const double s = scale[0];
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < Ne * n; i += (long long)gridDim.x * blockDim.x)
        phi[i] += s * (double)out[i / n];
}

// p = 1 (nodes at the vertices): phi[e, i] += scale * (mean of out over the
// elements that share node i's vertex) -- a continuous trilinear correction
__global__ void k_apply_corr_vertex(int nz, int ny, int nx, const float *__restrict__ out,
                                    const double *__restrict__ scale, double *__restrict__ phi)
{
    const double s = scale[0];
    const long long Ne = (long long)nz * ny * nx;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < Ne * 8; i += (long long)gridDim.x * blockDim.x) {
        const long long e = i >> 3;
        const int loc = (int)(i & 7);
        const int x = (int)(e % nx), y = (int)((e / nx) % ny), z = (int)(e / ((long long)nx * ny));
        const int vx = x + (loc & 1), vy = y + ((loc >> 1) & 1), vz = z + (loc >> 2);
        double sum = 0.0;
        int cnt = 0;
        for (int jz = vz - 1; jz <= vz; ++jz)
            for (int jy = vy - 1; jy <= vy; ++jy)
                for (int jx = vx - 1; jx <= vx; ++jx)
                    if (jx >= 0 && jx < nx && jy >= 0 && jy < ny && jz >= 0 && jz < nz) {
                        sum += (double)out[((long long)jz * ny + jy) * nx + jx];
                        ++cnt;
                    }
        phi[i] += s * sum / (double)cnt;
    }
}

inline int grid_for(long long n, int block = 256, int cap = 4096)
{
    long long g = (n + block - 1) / block;
    if (g < 1) g = 1;
    return (int)(g > cap ? cap : g);
}

thread_local std::string g_cnn_err = "no error";
int cfail(int code, const std::string &m)
{
    g_cnn_err = m;
    allium_cnn_internal::set_last_error(m);
    return code;
}
#define CNN_TRY(expr)                                                                     \
    do {                                                                                  \
        hipError_t _e = (expr);                                                           \
        if (_e != hipSuccess) return cfail(-4, std::string(#expr ": ") + hipGetErrorString(_e)); \
    } while (0)

long layer_offset(int l)
{
    long off = 0;
    for (int k = 0; k < l; ++k) off += 27L * CO_[k] * CI_[k] + CO_[k];
    return off;
}
const long NPARAM = layer_offset(NL);

}  // namespace

struct allium_cnn {
    float *params = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr;
    bf16 *Wf[NL] = {}, *Wb[NL] = {};
    float *bias[NL] = {};
    bool packed = false;
    long long cap = 0;
    long long cap_parts = 0;   // weight-gradient partials
    bf16 *xin = nullptr, *act[NL - 1] = {}, *ga = nullptr, *gb = nullptr;
    float *out = nullptr, *part = nullptr, *xf = nullptr;
    double *lpart = nullptr, *ravg = nullptr, *rpart = nullptr, *scale = nullptr;
    long step = 0;
    int dil[NL] = {1, 1, 1, 1, 1};
    hipStream_t stream = nullptr;
    std::vector<void *> owned;
    ~allium_cnn()
    {
        for (void *p : owned) hipFree(p);
        if (stream) hipStreamDestroy(stream);
    }
    template <typename T>
    hipError_t alloc(T **p, size_t count)
    {
        hipError_t e = hipMalloc((void **)p, sizeof(T) * (count ? count : 1));
        if (e == hipSuccess) owned.push_back(*p);
        return e;
    }
};

namespace {

constexpr int kWgradGroups = 256;
constexpr int kLossBlocks = 512;

// workgroups per plane of the weight gradients: one per CU in all, up to four per
// plane (on 8 x 32^3, 256 planes, two per CU took 39 instead of 45 us a layer, but
// their partials' sum 18 instead of 10 us; sixteen waves instead of eight took 49 us)
int wgrad_shares(const Geo &g)
{
    const long long want = kWgradGroups / ((long long)g.B * g.nz);
    return (int)(want < 1 ? 1 : want > 4 ? 4 : want);
}

// the work buffers of T voxels and so many partials; after a failure the handle holds none
hipError_t alloc_work(allium_cnn *h, long long T, long long parts)
{
    auto free_work = [&] {
        std::vector<void *> keep;
        for (void *p : h->owned) {
            bool work = p == h->xin || p == h->ga || p == h->gb || p == h->out || p == h->part || p == h->xf ||
                        p == h->ravg;
            for (int l = 0; l < NL - 1; ++l) work = work || p == h->act[l];
            if (work) hipFree(p);
            else keep.push_back(p);
        }
        h->owned = keep;
        h->xin = h->ga = h->gb = nullptr;
        h->out = h->part = h->xf = nullptr;
        h->ravg = nullptr;
        for (bf16 *&a : h->act) a = nullptr;
        h->cap = h->cap_parts = 0;
    };
    free_work();
    hipError_t e = h->alloc(&h->xin, (size_t)T * 8);
    for (int l = 0; l < NL - 1 && e == hipSuccess; ++l) e = h->alloc(&h->act[l], (size_t)T * HID);
    if (e == hipSuccess) e = h->alloc(&h->ga, (size_t)T * HID);
    if (e == hipSuccess) e = h->alloc(&h->gb, (size_t)T * HID);
    if (e == hipSuccess) e = h->alloc(&h->out, (size_t)T);
    if (e == hipSuccess) e = h->alloc(&h->xf, (size_t)T * 3);
    if (e == hipSuccess) e = h->alloc(&h->ravg, (size_t)T);
    if (e == hipSuccess) e = h->alloc(&h->part, (size_t)parts * 28 * 32 * 32);
    if (e != hipSuccess) {
        (void)hipGetLastError();   // or the next launch's check reports it
        free_work();
        return e;
    }
    h->cap = T;
    h->cap_parts = parts;
    return hipSuccess;
}

int ensure(allium_cnn *h, const Geo &g)
{
    const long long parts = (long long)g.B * g.nz * wgrad_shares(g);
    if (g.T <= h->cap && parts <= h->cap_parts) return 0;
    // neither size shrinks, so calls that alternate between shapes settle, unless the
    // memory only holds what this call needs
    const long long T1 = g.T > h->cap ? g.T : h->cap, parts1 = parts > h->cap_parts ? parts : h->cap_parts;
    hipError_t e = alloc_work(h, T1, parts1);
    if (e != hipSuccess && (T1 > g.T || parts1 > parts)) e = alloc_work(h, g.T, parts);
    if (e != hipSuccess) return cfail(-4, std::string("network work buffers: ") + hipGetErrorString(e));
    return 0;
}

int pack_weights(allium_cnn *h, hipStream_t s)
{
    if (h->packed) return 0;
    for (int l = 0; l < NL; ++l) {
        const float *Wm = h->params + layer_offset(l);
        const float *bm = Wm + 27L * CO_[l] * CI_[l];
        hipLaunchKernelGGL(k_pack_layer, dim3(grid_for(27L * COP_[l] * CIP_[l])), dim3(256), 0, s, Wm, bm, CO_[l],
                           CI_[l], COP_[l], CIP_[l], h->Wf[l], h->Wb[l], h->bias[l]);
    }
    CNN_TRY(hipGetLastError());
    h->packed = true;
    return 0;
}

// forward from the packed bf16 input h->xin; output FP32 h->out
Geo layer_geo(const allium_cnn *h, const Geo &g, int l)
{
    Geo gl = g;
    gl.dil = h->dil[l];
    return gl;
}

int forward_packed(allium_cnn *h, const Geo &g, hipStream_t s)
{
    launch_conv<8, 32, 0>(layer_geo(h, g, 0), h->xin, h->Wf[0], h->bias[0], h->act[0], nullptr, nullptr, s);
    launch_conv<32, 32, 0>(layer_geo(h, g, 1), h->act[0], h->Wf[1], h->bias[1], h->act[1], nullptr, nullptr, s);
    launch_conv<32, 32, 0>(layer_geo(h, g, 2), h->act[1], h->Wf[2], h->bias[2], h->act[2], nullptr, nullptr, s);
    launch_conv<32, 32, 0>(layer_geo(h, g, 3), h->act[2], h->Wf[3], h->bias[3], h->act[3], nullptr, nullptr, s);
    launch_conv<32, 16, 1>(layer_geo(h, g, 4), h->act[3], h->Wf[4], h->bias[4], nullptr, h->out, nullptr, s);
    CNN_TRY(hipGetLastError());
    return 0;
}

int check_geo(int B, int nz, int ny, int nx, Geo &g)
{
    if (B < 1 || nz < 1 || ny < 1 || nx < 1 || nx > (1 << 20)) return cfail(-1, "bad grid size");
    g.B = B;
    g.nz = nz;
    g.ny = ny;
    g.nx = nx;
    g.T = (long long)B * nz * ny * nx;
    g.dil = 1;
    return 0;
}

// forward + backward into h->grad (device, packed); *loss on the host
int gradient(allium_cnn *h, const Geo &g, const float *d_x, const float *d_t, double *loss, hipStream_t s)
{
    int rc = ensure(h, g);
    if (rc) return rc;
    rc = pack_weights(h, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_pack_input, dim3(grid_for(g.T * 8)), dim3(256), 0, s, g.T, d_x, h->xin);
    rc = forward_packed(h, g, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_loss, dim3(kLossBlocks), dim3(256), 0, s, g.T, h->out, d_t, h->ga, h->lpart);
    const int planes = g.B * g.nz, nshare = wgrad_shares(g);
    // layer 5: gz = ga [T][16]
    const bf16 *gz = h->ga;
    bf16 *gnext = h->gb;
    for (int l = NL - 1; l >= 0; --l) {
        const bf16 *ain = l == 0 ? h->xin : h->act[l - 1];
        float *gW = h->grad + layer_offset(l);
        const Geo gl = layer_geo(h, g, l);
        if (l == NL - 1) {
            hipLaunchKernelGGL((k_wgrad<32, 16>), dim3(planes * nshare), dim3(64 * kWgradWaves), 0, s, gl, nshare, gz, ain, h->part);
        } else if (l == 0) {
            hipLaunchKernelGGL((k_wgrad<8, 32>), dim3(planes * nshare), dim3(64 * kWgradWaves), 0, s, gl, nshare, gz, ain, h->part);
        } else {
            hipLaunchKernelGGL((k_wgrad<32, 32>), dim3(planes * nshare), dim3(64 * kWgradWaves), 0, s, gl, nshare, gz, ain, h->part);
        }
        hipLaunchKernelGGL(k_wgrad_reduce, dim3((unsigned)((27L * CO_[l] * CI_[l] + CO_[l] + 63) / 64)), dim3(256), 0, s,
                           h->part, planes * nshare, COP_[l], CIP_[l], CO_[l], CI_[l], gW);
        if (l > 0) {
            // gradient of the previous pre-activation: conv with flipped weights, ReLU mask of its output
            if (l == NL - 1)
                launch_conv<16, 32, 2>(gl, gz, h->Wb[l], nullptr, gnext, nullptr, h->act[l - 1], s);
            else
                launch_conv<32, 32, 2>(gl, gz, h->Wb[l], nullptr, gnext, nullptr, h->act[l - 1], s);
            const bf16 *t = gnext;
            gnext = const_cast<bf16 *>(gz);
            gz = t;
        }
    }
    CNN_TRY(hipGetLastError());
    std::vector<double> lp(kLossBlocks);
    CNN_TRY(hipMemcpyAsync(lp.data(), h->lpart, sizeof(double) * kLossBlocks, hipMemcpyDeviceToHost, s));
    CNN_TRY(hipStreamSynchronize(s));
    double sum = 0.0;
    for (double v : lp) sum += v;
    if (loss) *loss = sum / (double)g.T;
    return 0;
}

}  // namespace

namespace allium_cnn_internal {

hipError_t elem_avg(long long Ne, int n, const double *d_w, const double *d_x, double *d_out, hipStream_t s)
{
    hipLaunchKernelGGL(k_elem_avg, dim3(grid_for(Ne)), dim3(256), 0, s, Ne, n, d_w, d_x, d_out, nullptr);
    return hipGetLastError();
}

int correct(allium_cnn *h, int nz, int ny, int nx, int n, const double *d_w, const double *d_r,
            const double *d_sigt, const double *d_sigs, double *d_phi, hipStream_t s, int prolong)
{
    Geo g;
    int rc = check_geo(1, nz, ny, nx, g);
    if (rc) return rc;
    rc = ensure(h, g);
    if (rc) return rc;
    rc = pack_weights(h, s);
    if (rc) return rc;
    const int nb = 256;
    hipLaunchKernelGGL(k_elem_avg, dim3(nb), dim3(256), 0, s, g.T, n, d_w, d_r, h->ravg, h->rpart);
    hipLaunchKernelGGL(k_scale, dim3(1), dim3(256), 0, s, h->rpart, nb, g.T, h->scale);
    hipLaunchKernelGGL(k_make_input, dim3(grid_for(g.T)), dim3(256), 0, s, g.T, h->ravg, h->scale, d_sigt, d_sigs,
                       h->xin);
    rc = forward_packed(h, g, s);
    if (rc) return rc;
    if (prolong == 1 && n == 8)
        hipLaunchKernelGGL(k_apply_corr_vertex, dim3(grid_for(g.T * 8)), dim3(256), 0, s, nz, ny, nx, h->out, h->scale,
                           d_phi);
    else
        hipLaunchKernelGGL(k_apply_corr, dim3(grid_for(g.T * n)), dim3(256), 0, s, g.T, n, h->out, h->scale, d_phi);
    CNN_TRY(hipGetLastError());
    return 0;
}

}  // namespace allium_cnn_internal

extern "C" {

long allium_cnn_num_params(void) { return NPARAM; }

int allium_cnn_set_dilation(allium_cnn_t h, const int *dilation)
{
    if (!h || !dilation) return cfail(-1, "null argument");
    for (int l = 0; l < NL; ++l)
        if (dilation[l] < 1 || dilation[l] > kMaxDil) return cfail(-1, "dilation must be 1..8 per layer");
    for (int l = 0; l < NL; ++l) h->dil[l] = dilation[l];
    return 0;
}

int allium_cnn_get_dilation(allium_cnn_t h, int *dilation)
{
    if (!h || !dilation) return cfail(-1, "null argument");
    for (int l = 0; l < NL; ++l) dilation[l] = h->dil[l];
    return 0;
}

int allium_cnn_create(unsigned long long seed, allium_cnn_t *out)
{
    if (!out) return cfail(-1, "null argument");
    *out = nullptr;
    auto *h = new allium_cnn();
    auto bad = [&](hipError_t e) {
        delete h;
        return cfail(-4, std::string("allium_cnn_create: ") + hipGetErrorString(e));
    };
    hipError_t e;
    if ((e = h->alloc(&h->params, NPARAM)) != hipSuccess) return bad(e);
    if ((e = h->alloc(&h->m, NPARAM)) != hipSuccess) return bad(e);
    if ((e = h->alloc(&h->v, NPARAM)) != hipSuccess) return bad(e);
    if ((e = h->alloc(&h->grad, NPARAM)) != hipSuccess) return bad(e);
    for (int l = 0; l < NL; ++l) {
        if ((e = h->alloc(&h->Wf[l], 27L * COP_[l] * CIP_[l])) != hipSuccess) return bad(e);
        if ((e = h->alloc(&h->Wb[l], 27L * COP_[l] * CIP_[l])) != hipSuccess) return bad(e);
        if ((e = h->alloc(&h->bias[l], COP_[l])) != hipSuccess) return bad(e);
    }
    if ((e = h->alloc(&h->lpart, kLossBlocks)) != hipSuccess) return bad(e);
    if ((e = h->alloc(&h->rpart, 256)) != hipSuccess) return bad(e);
    if ((e = h->alloc(&h->scale, 1)) != hipSuccess) return bad(e);
    if ((e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking)) != hipSuccess) return bad(e);
    // He-normal weights, zero biases
    std::vector<float> p(NPARAM, 0.f);
    std::mt19937_64 rng(seed);
    for (int l = 0; l < NL; ++l) {
        std::normal_distribution<double> nd(0.0, std::sqrt(2.0 / (27.0 * CI_[l])));
        float *W = p.data() + layer_offset(l);
        for (long i = 0; i < 27L * CO_[l] * CI_[l]; ++i) W[i] = (float)nd(rng);
    }
    if ((e = hipMemcpy(h->params, p.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice)) != hipSuccess) return bad(e);
    if ((e = hipMemset(h->m, 0, sizeof(float) * NPARAM)) != hipSuccess) return bad(e);
    if ((e = hipMemset(h->v, 0, sizeof(float) * NPARAM)) != hipSuccess) return bad(e);
    *out = h;
    return 0;
}

void allium_cnn_destroy(allium_cnn_t h) { delete h; }

int allium_cnn_get_params(allium_cnn_t h, float *params)
{
    if (!h || !params) return cfail(-1, "null argument");
    CNN_TRY(hipMemcpy(params, h->params, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
    return 0;
}

int allium_cnn_set_params(allium_cnn_t h, const float *params)
{
    if (!h || !params) return cfail(-1, "null argument");
    for (long i = 0; i < NPARAM; ++i)
        if (!std::isfinite(params[i])) return cfail(-6, "non-finite network parameter");
    CNN_TRY(hipMemcpy(h->params, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice));
    CNN_TRY(hipMemset(h->m, 0, sizeof(float) * NPARAM));
    CNN_TRY(hipMemset(h->v, 0, sizeof(float) * NPARAM));
    h->step = 0;
    h->packed = false;
    return 0;
}

int allium_cnn_forward_device(allium_cnn_t h, int batch, int nz, int ny, int nx, const float *d_x, float *d_out,
                              void *stream)
{
    if (!h || !d_x || !d_out) return cfail(-1, "null argument");
    Geo g;
    int rc = check_geo(batch, nz, ny, nx, g);
    if (rc) return rc;
    hipStream_t s = stream ? (hipStream_t)stream : h->stream;
    rc = ensure(h, g);
    if (rc) return rc;
    rc = pack_weights(h, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_pack_input, dim3(grid_for(g.T * 8)), dim3(256), 0, s, g.T, d_x, h->xin);
    rc = forward_packed(h, g, s);
    if (rc) return rc;
    CNN_TRY(hipMemcpyAsync(d_out, h->out, sizeof(float) * g.T, hipMemcpyDeviceToDevice, s));
    CNN_TRY(hipStreamSynchronize(s));
    return 0;
}

int allium_cnn_gradient_device(allium_cnn_t h, int batch, int nz, int ny, int nx, const float *d_x,
                               const float *d_target, float *grad, double *loss)
{
    if (!h || !d_x || !d_target || !grad) return cfail(-1, "null argument");
    Geo g;
    int rc = check_geo(batch, nz, ny, nx, g);
    if (rc) return rc;
    rc = gradient(h, g, d_x, d_target, loss, h->stream);
    if (rc) return rc;
    CNN_TRY(hipMemcpy(grad, h->grad, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
    return 0;
}

int allium_cnn_train_step_device(allium_cnn_t h, int batch, int nz, int ny, int nx, const float *d_x,
                                 const float *d_target, float lr, double *loss)
{
    if (!h || !d_x || !d_target) return cfail(-1, "null argument");
    if (!(lr > 0.f) || !std::isfinite(lr)) return cfail(-1, "learning rate must be positive");
    Geo g;
    int rc = check_geo(batch, nz, ny, nx, g);
    if (rc) return rc;
    double l = 0.0;
    rc = gradient(h, g, d_x, d_target, &l, h->stream);
    if (rc) return rc;
    if (!std::isfinite(l)) return cfail(-6, "non-finite training loss");
    h->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)h->step), c2 = 1.f - std::pow(b2, (float)h->step);
    hipLaunchKernelGGL(k_adam, dim3(grid_for(NPARAM)), dim3(256), 0, h->stream, NPARAM, h->params, h->grad, h->m,
                       h->v, lr, b1, b2, 1e-8f, c1, c2);
    CNN_TRY(hipGetLastError());
    h->packed = false;
    CNN_TRY(hipStreamSynchronize(h->stream));
    if (loss) *loss = l;
    return 0;
}

}  // extern "C"
