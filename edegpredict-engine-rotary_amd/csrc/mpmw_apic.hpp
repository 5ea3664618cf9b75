// mpmw_apic.hpp -- the APIC transfer variant of the particle pass.
//
// Quadratic B-spline weights over 27 nodes with base = floor(x/h - 0.5)
// (getWeightsAndGradients, MPMSolver.cu:20-34), affine momentum
// m w (v + C (x_i - x_p)) in P2G (p2gKernel :370-421) and the affine matrix
// C = 0.99 * 3/h^2 * sum w v_i (x_i - x_p)^T from G2P (g2pKernel :554-592);
// the rest of the step (forces, grid update, contact, diffusion,
// constitutive update, chip pass) is the workpiece solver's.
//
// Same tiles and binning as the trilinear pass, and the same walk: thread =
// cell, slot by slot.  A particle of cell c has its base at c - 1 or c, so the
// node window of a tile of TX x TY x TZ cells spans one node before the tile
// and two after it: QX x QY x QZ nodes, and that of one wave's layer of cells
// QX x QY x 4.  A wave adds the 27 x 8 contributions of its particles into a
// window of its own without atomics (quad_scatter_wave; a register
// accumulation per cell does not fit 27 nodes); the tile's window is the sum
// of its waves' (FP64 adds straight into the tile's window with hardware LDS
// adds, quad_scatter_window), stored, with plain stores, into the tile's slot of the
// per-tile window buffer, and the grid update sums the windows holding each
// node in tile order.  Particles that have left their wave's window are
// queued and added to the tile's window after the walk; those whose stencil
// leaves that too go to the node accumulators with device atomics.
#pragma once

#include "mpmw_tile.hpp"

namespace mpmw {

__device__ __forceinline__ int qnode(int x, int y, int z) { return (z * QY + y) * QX + x; }

// The window of node records that the gather reads: rows of QX nodes, padded
// to 12, so that the 16-byte reads of a wave whose lanes follow the cells of a
// layer meet no bank conflict (rows of 11: 34 clocks a read against 30).
// FP64 rows are not padded: two workgroups of its fused pass just fit a CU.
template <typename R> constexpr int kRowP = sizeof(R) == 4 ? QX + 1 : QX;
template <typename R> __device__ __forceinline__ int qpnode(int x, int y, int z) { return (z * QY + y) * kRowP<R> + x; }

// The per-axis quadratic weights of one particle.  d0 = r - base in
// [0.5, 1.5); node offsets x_i - x_p = (i - d0) h.
template <typename R> struct QFrac {
    int b[3];
    R w[3][3], dw[3][3], d0[3];
};

// getWeightsAndGradients (MPMSolver.cu:20-34) on the three axes; r is
// formed in FP64 as the reference forms x_frac, (x - origin) * invDx.
template <typename R>
__device__ __forceinline__ QFrac<R> quad_frac(const GridView<R> &g, double x, double y, double z) {
    QFrac<R> q;
    const double d[3] = {x - g.ox, y - g.oy, z - g.oz};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double r = d[a] * g.inv_hd;
        const double fl = floor(r - 0.5);
        q.b[a] = (int)fl;
        const R d0 = (R)(r - fl), d1 = d0 - R(1), d2 = d0 - R(2);
        q.d0[a] = d0;
        q.w[a][0] = R(0.5) * (R(1.5) - d0) * (R(1.5) - d0);
        q.w[a][1] = R(0.75) - d1 * d1;
        q.w[a][2] = R(0.5) * (R(1.5) + d2) * (R(1.5) + d2);
        q.dw[a][0] = -(R(1.5) - d0) * g.inv_h;
        q.dw[a][1] = R(-2) * d1 * g.inv_h;
        q.dw[a][2] = (R(1.5) + d2) * g.inv_h;
    }
    return q;
}

// Node (i, j, k) of the stencil: weight, gradient and offset x_i - x_p.
template <typename R>
__device__ __forceinline__ void quad_node(const QFrac<R> &q, int i, int j, int k, R h, R &w, R &gx, R &gy, R &gz,
                                          R &dx, R &dy, R &dz) {
    w = q.w[0][i] * q.w[1][j] * q.w[2][k];
    gx = q.dw[0][i] * q.w[1][j] * q.w[2][k];
    gy = q.w[0][i] * q.dw[1][j] * q.w[2][k];
    gz = q.w[0][i] * q.w[1][j] * q.dw[2][k];
    dx = (R(i) - q.d0[0]) * h;
    dy = (R(j) - q.d0[1]) * h;
    dz = (R(k) - q.d0[2]) * h;
}

// One live node's share of the G2P sums and of B.
template <typename R>
__device__ __forceinline__ void quad_gather_add(const vec4_t<R> &nd, R w, R gx, R gy, R gz, R dx, R dy, R dz,
                                                GatherSums<R> &s, R B[9]) {
    s.v0 += w * nd.x; s.v1 += w * nd.y; s.v2 += w * nd.z;
    s.temp += nd.w * w;
    s.wsum += w;
    const R wx = w * nd.x, wy = w * nd.y, wz = w * nd.z;
    B[0] += wx * dx; B[1] += wx * dy; B[2] += wx * dz;
    B[3] += wy * dx; B[4] += wy * dy; B[5] += wy * dz;
    B[6] += wz * dx; B[7] += wz * dy; B[8] += wz * dz;
    s.L[0] += nd.x * gx; s.L[1] += nd.x * gy; s.L[2] += nd.x * gz;
    s.L[3] += nd.y * gx; s.L[4] += nd.y * gy; s.L[5] += nd.y * gz;
    s.L[6] += nd.z * gx; s.L[7] += nd.z * gy; s.L[8] += nd.z * gz;
}

// A node record as the APIC window holds it: an empty node, or one outside
// the grid, has no velocity and keeps the NaN that marks it (a node's
// temperature may be negative, so no number can).
template <typename R> __device__ __forceinline__ vec4_t<R> quad_record(vec4_t<R> nd) {
    if (!(nd.w == nd.w)) nd.x = nd.y = nd.z = R(0);
    return nd;
}

// G2P gather over the 27 nodes from the LDS window (base node at window
// index wb; records as quad_record writes them, so that no node needs a
// branch) or from device memory
// (nodes outside the grid and empty nodes skipped, g2pKernel :538, with the
// workpiece grid's emptiness test).  From the window the sums are factored:
// a column of three nodes along z is reduced once for its value, its z
// gradient and its z moment, and enters the x and y terms as one (the 27
// nodes one by one took 1.7 times the multiply-adds).  The G2P-only pass of
// 4.2 M particles: 186 us then, 171 now, loads one slot ahead included.
template <typename R>
__device__ __forceinline__ void quad_gather_window(const vec4_t<R> *s_node, int wb, const QFrac<R> &q, R h,
                                                   GatherSums<R> &s, R B[9]) {
    R off[3][3], wz[3];   // x_i - x_p per axis
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int n = 0; n < 3; ++n) off[a][n] = (R(n) - q.d0[a]) * h;
#pragma unroll
    for (int k = 0; k < 3; ++k) wz[k] = q.w[2][k] * off[2][k];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        R sx[3] = {R(0), R(0), R(0)};   // sum over y and z of w v
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            R a[3] = {R(0), R(0), R(0)}, b[3] = {R(0), R(0), R(0)}, c[3] = {R(0), R(0), R(0)}, tz = R(0), wl = R(0);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const vec4_t<R> nd = s_node[wb + qpnode<R>(i, j, k)];
                const R v[3] = {nd.x, nd.y, nd.z};
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    a[r] = fma(q.w[2][k], v[r], a[r]);
                    b[r] = fma(q.dw[2][k], v[r], b[r]);
                    c[r] = fma(wz[k], v[r], c[r]);
                }
                const bool live = nd.w == nd.w;
                tz = fma(q.w[2][k], live ? nd.w : R(0), tz);
                wl += live ? q.w[2][k] : R(0);
            }
            const R w = q.w[0][i] * q.w[1][j], gx = q.dw[0][i] * q.w[1][j], gy = q.w[0][i] * q.dw[1][j];
            s.temp = fma(w, tz, s.temp);
            s.wsum = fma(w, wl, s.wsum);
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const R p = w * a[r];
                sx[r] += p;
                B[3 * r + 1] = fma(off[1][j], p, B[3 * r + 1]);
                B[3 * r + 2] = fma(w, c[r], B[3 * r + 2]);
                s.L[3 * r] = fma(gx, a[r], s.L[3 * r]);
                s.L[3 * r + 1] = fma(gy, a[r], s.L[3 * r + 1]);
                s.L[3 * r + 2] = fma(w, b[r], s.L[3 * r + 2]);
            }
        }
        s.v0 += sx[0]; s.v1 += sx[1]; s.v2 += sx[2];
#pragma unroll
        for (int r = 0; r < 3; ++r) B[3 * r] = fma(off[0][i], sx[r], B[3 * r]);
    }
}

template <typename R>
__device__ __forceinline__ void quad_gather_global(const GridView<R> &g, gp<const vec4_t<R>> node, const QFrac<R> &q,
                                                   R h, GatherSums<R> &s, R B[9]) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int x = q.b[0] + i, y = q.b[1] + j, z = q.b[2] + k;
                if (x < 0 || y < 0 || z < 0 || x >= g.nx || y >= g.ny || z >= g.nz) continue;
                const vec4_t<R> nd = node[((int64_t)z * g.ny + y) * g.nx + x];
                if (nd.w != nd.w) continue;
                R w, gx, gy, gz, dx, dy, dz;
                quad_node(q, i, j, k, h, w, gx, gy, gz, dx, dy, dz);
                quad_gather_add(nd, w, gx, gy, gz, dx, dy, dz, s, B);
            }
}

// What one particle adds in the APIC P2G.
template <typename R> struct QP2G {
    R mass, vol, vx, vy, vz, T;
    R s[6];
    R C[9];
    R fex, fey, fez;
    bool momentum;   // not FIXED_BOUNDARY (p2gKernel :393-398)
    bool stress;     // ACTIVE or FIXED_BOUNDARY: stress force (mpmP2GKernel :121-127)
    bool ext;        // stress or CHIP: external force (:121-132)
};

// A particle's P2G terms in the form the 27 nodes share: with node offset
// x_i - x_p = (idx - d0) h, the affine velocity v + C (x_i - x_p) is
// u + (h C) idx with u = v - (h C) d0, so a node adds (h C) idx to u with
// its small integer idx (the sum over idx x and y is shared by the nodes of
// a column); the stress force is S grad w with S = -V sigma.  A particle
// without momentum or forces has zeros there.
template <typename R> struct QScatter {
    R m, T, u[3], hc[9], S[6], fe[3];
};

template <typename R>
__device__ __forceinline__ QScatter<R> quad_scatter_terms(const QP2G<R> &a, const QFrac<R> &q, R h) {
    QScatter<R> z;
    z.m = a.mass;
    z.T = a.T;
#pragma unroll
    for (int c = 0; c < 9; ++c) z.hc[c] = a.momentum ? a.C[c] * h : R(0);
    const R v[3] = {a.momentum ? a.vx : R(0), a.momentum ? a.vy : R(0), a.momentum ? a.vz : R(0)};
#pragma unroll
    for (int r = 0; r < 3; ++r)
        z.u[r] = v[r] - (z.hc[3 * r] * q.d0[0] + z.hc[3 * r + 1] * q.d0[1] + z.hc[3 * r + 2] * q.d0[2]);
#pragma unroll
    for (int c = 0; c < 6; ++c) z.S[c] = -a.vol * a.s[c];
    z.fe[0] = a.fex; z.fe[1] = a.fey; z.fe[2] = a.fez;
    return z;
}

// The 8 channels of node (i, j, k) of the stencil: mass, momentum, force,
// T * m.
template <typename R>
__device__ __forceinline__ void quad_node_channels(const QScatter<R> &z, int i, int j, int k, R w, R gx, R gy, R gz,
                                                   R c[8]) {
    const R m = z.m * w;
    c[0] = m;
#pragma unroll
    for (int r = 0; r < 3; ++r)
        c[1 + r] = m * (z.u[r] + z.hc[3 * r] * R(i) + z.hc[3 * r + 1] * R(j) + z.hc[3 * r + 2] * R(k));
    c[4] = z.S[0] * gx + z.S[3] * gy + z.S[4] * gz + z.fe[0] * w;
    c[5] = z.S[3] * gx + z.S[1] * gy + z.S[5] * gz + z.fe[1] * w;
    c[6] = z.S[4] * gx + z.S[5] * gy + z.S[2] * gz + z.fe[2] * w;
    c[7] = z.T * m;
}

// Nodes of the window of one wave's layer of cells, and its places for a
// base node.
constexpr int QLZ = 4;
constexpr int QLN = QX * QY * QLZ;   // rows along z inside y: no bank conflict, as above
__device__ __forceinline__ int qlnode(int x, int y, int z) { return (y * QLZ + z) * QX + x; }
constexpr int QLB = (TX + 1) * (TY + 1);

// Orders the wave's LDS accesses before this point against those after it.
// The LDS serves a wave's instructions in order: nothing is waited for.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// u + c n for a step n of the stencil, known to the compiler once unrolled.
template <typename R> __device__ __forceinline__ R quad_along(R u, R c, int n) {
    return n == 0 ? u : n == 1 ? u + c : u + c * R(n);
}

// Scatter of a wave's particles into the wave's window: win[n] is node n's
// mass and momentum, win[QLN + n] its force and T * m.  Particles of one wave
// with different base nodes touch different nodes at every one of the 27
// steps, so a step is a read, an add and a write of two 16-byte records
// instead of eight atomic adds (FP32 words of LDS add one lane at a time, or
// by compare-and-swap of pairs, as this pass did: 4.2 M particles took 596 us
// then, 532 with an FP64 window and its hardware adds, and take 355 now; the
// vector unit is busy 60 % of that, the LDS 40 %).  The three nodes of a
// column along z are read together: a round takes lanes of one base layer
// only, so that none of them touches another's column (one node after
// another: 382 us).
// A lane takes part once it has won its base node's place in `owner`; lanes
// that share a base node take turns.  Slots keep the order in which the
// particles were made, so that a wave's particles mostly sit alike in their
// cells: of 64, 63.99 have bases of their own after 50 steps of a jittered slab
// under a drill.
template <typename R>
__device__ __forceinline__ void quad_scatter_wave(vec4_t<R> *win, uint8_t *owner, int lz, int place, int wb,
                                                  QFrac<R> q, QScatter<R> z) {
    const int lane = (int)threadIdx.x % kWave;
    bool pending = true;
    unsigned long long left = __ballot(true);
    do {
        const bool at = pending && lz == __builtin_amdgcn_readlane(lz, __ffsll(left) - 1);
        if (at) __hip_atomic_store(owner + place, (uint8_t)lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        wave_lds_order();
        const bool won =
            at && __hip_atomic_load(owner + place, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT) == lane;
        wave_lds_order();
        // keeps the 216 terms from being formed ahead of the loop, in as
        // many registers
        asm volatile("" : "+v"(z.u[0]), "+v"(z.u[1]), "+v"(z.u[2]), "+v"(z.T));
#pragma unroll
        for (int d = 0; d < 3; ++d)
            asm volatile("" : "+v"(q.w[d][0]), "+v"(q.w[d][1]), "+v"(q.w[d][2]), "+v"(q.dw[d][0]), "+v"(q.dw[d][1]),
                         "+v"(q.dw[d][2]));
        if (won) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const R w = q.w[0][i] * q.w[1][j], gx = q.dw[0][i] * q.w[1][j], gy = q.w[0][i] * q.dw[1][j];
                    const R m = z.m * w;
                    R u[3], p[3], f[3];   // velocity at k = 0; force per weight and per gradient along z
#pragma unroll
                    for (int r = 0; r < 3; ++r) u[r] = quad_along(quad_along(z.u[r], z.hc[3 * r], i), z.hc[3 * r + 1], j);
                    p[0] = z.S[0] * gx + z.S[3] * gy + z.fe[0] * w;
                    p[1] = z.S[3] * gx + z.S[1] * gy + z.fe[1] * w;
                    p[2] = z.S[4] * gx + z.S[5] * gy + z.fe[2] * w;
                    f[0] = z.S[4] * w; f[1] = z.S[5] * w; f[2] = z.S[2] * w;
                    vec4_t<R> *const o = win + wb + qlnode(i, j, 0);
                    vec4_t<R> a[3], b[3];
#pragma unroll
                    for (int k = 0; k < 3; ++k) { a[k] = o[k * QX]; b[k] = o[QLN + k * QX]; }
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const R mk = m * q.w[2][k];
                        a[k].x += mk;
                        a[k].y += mk * quad_along(u[0], z.hc[2], k);
                        a[k].z += mk * quad_along(u[1], z.hc[5], k);
                        a[k].w += mk * quad_along(u[2], z.hc[8], k);
                        b[k].x = fma(f[0], q.dw[2][k], fma(p[0], q.w[2][k], b[k].x));
                        b[k].y = fma(f[1], q.dw[2][k], fma(p[1], q.w[2][k], b[k].y));
                        b[k].z = fma(f[2], q.dw[2][k], fma(p[2], q.w[2][k], b[k].z));
                        b[k].w += z.T * mk;
                    }
#pragma unroll
                    for (int k = 0; k < 3; ++k) { o[k * QX] = a[k]; o[QLN + k * QX] = b[k]; }
                    wave_lds_order();
                }
            pending = false;
        }
        // the lanes go round together (a loop left by each lane on its own
        // would let the compiler move the adds behind it, where all lanes
        // add at once)
        left = __ballot(pending);
    } while (left != 0);
}

// FP64 scatter into the tile's LDS window (channel stride QN, window index wb
// of the base node): FP64 words of LDS add in hardware and the wave goes on
// without waiting; windows of the waves' own, twice the size of FP32's, made
// 4.2 M particles 50 ms for 50 steps against 46, 0.6 M 14.5 against 11.6.
// A channel that the particle does not add to is not touched.
__device__ __forceinline__ void quad_scatter_window(double *s_acc, int wb, const QFrac<double> &q, double h,
                                                    const QP2G<double> &a) {
    const QScatter<double> z = quad_scatter_terms(a, q, h);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                double w, gx, gy, gz, dx, dy, dz, c[8];
                quad_node(q, i, j, k, h, w, gx, gy, gz, dx, dy, dz);
                quad_node_channels(z, i, j, k, w, gx, gy, gz, c);
                double *const o = s_acc + wb + qnode(i, j, k);
                atomicAdd(o, c[0]);
                if (a.momentum) {
#pragma unroll
                    for (int r = 1; r < 4; ++r) atomicAdd(o + r * QN, c[r]);
                }
                if (a.ext) {
#pragma unroll
                    for (int r = 4; r < 7; ++r) atomicAdd(o + r * QN, c[r]);
                }
                atomicAdd(o + 7 * QN, c[7]);
            }
}

// One particle's share of node n of its stencil into the tile's window
// (records of 8 channels), or, if the window does not hold its stencil,
// into the node accumulators (nodes outside the grid skipped); true if the
// latter.
template <typename R>
__device__ __forceinline__ bool quad_scatter_node(const GridView<R> &g, gp<R> acc, R *win, int lx, int ly, int lz,
                                                  const QFrac<R> &q, R h, const QP2G<R> &a, int n) {
    const bool inw = (unsigned)lx <= (unsigned)TX && (unsigned)ly <= (unsigned)TY && (unsigned)lz <= (unsigned)TZ;
    if (n >= 27) return !inw;
    const int i = n % 3, j = n / 3 % 3, k = n / 9;
    // the weights picked by comparison: an index into the arrays would put
    // them in memory
    R wa[3], ga[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int e = d == 0 ? i : d == 1 ? j : k;
        const R w0 = q.w[d][0], w1 = q.w[d][1], w2 = q.w[d][2];
        const R g0 = q.dw[d][0], g1 = q.dw[d][1], g2 = q.dw[d][2];
        wa[d] = e == 0 ? w0 : e == 1 ? w1 : w2;
        ga[d] = e == 0 ? g0 : e == 1 ? g1 : g2;
    }
    R c[8];
    quad_node_channels(quad_scatter_terms(a, q, h), i, j, k, wa[0] * wa[1] * wa[2], ga[0] * wa[1] * wa[2],
                       wa[0] * ga[1] * wa[2], wa[0] * wa[1] * ga[2], c);
    if (inw) {
        R *const o = win + 8 * (qnode(lx, ly, lz) + qnode(i, j, k));
#pragma unroll
        for (int ch = 0; ch < 8; ++ch) atomicAdd(o + ch, c[ch]);
        return false;
    }
    const int x = q.b[0] + i, y = q.b[1] + j, z = q.b[2] + k;
    if (x >= 0 && y >= 0 && z >= 0 && x < g.nx && y < g.ny && z < g.nz) {
        R *const o = acc + ((int64_t)z * g.ny + y) * g.nx + x;
#pragma unroll
        for (int ch = 0; ch < 8; ++ch) unsafeAtomicAdd(o + ch * g.nn, c[ch]);
    }
    return true;
}

// Scatter into the node accumulators with device atomics (nodes outside the
// grid skipped, as p2gKernel :371-378 skips them).
template <typename R>
__device__ __forceinline__ void quad_scatter_global(const GridView<R> &g, gp<R> acc, const QFrac<R> &q, R h,
                                                    const QP2G<R> &a) {
    const QScatter<R> zt = quad_scatter_terms(a, q, h);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int x = q.b[0] + i, y = q.b[1] + j, z = q.b[2] + k;
                if (x < 0 || y < 0 || z < 0 || x >= g.nx || y >= g.ny || z >= g.nz) continue;
                R w, gx, gy, gz, dx, dy, dz, c[8];
                quad_node(q, i, j, k, h, w, gx, gy, gz, dx, dy, dz);
                quad_node_channels(zt, i, j, k, w, gx, gy, gz, c);
                R *p = acc + ((int64_t)z * g.ny + y) * g.nx + x;
#pragma unroll
                for (int ch = 0; ch < 8; ++ch) unsafeAtomicAdd(p + ch * g.nn, c[ch]);
            }
}

template <typename R> __device__ __forceinline__ void load_affine(const Particles<R> &P, int i, R C[9]) {
#pragma unroll
    for (int c = 0; c < 9; ++c) C[c] = P.aff[c][i];
}

// The APIC P2G inputs of a particle from its state p (after its G2P, or as
// loaded for a P2G-only pass) and its affine matrix.
template <typename R>
__device__ __forceinline__ QP2G<R> quad_inputs(const PState<R> &p, const R C[9], R mass, R vol, R fex, R fey,
                                               R fez) {
    QP2G<R> a;
    a.mass = mass; a.vol = vol;
    a.vx = p.vx; a.vy = p.vy; a.vz = p.vz;
    a.T = p.T;
    a.stress = p.status == kActive || p.status == kFixed;
    a.ext = a.stress || p.status == kChip;
    a.momentum = p.status != kFixed;
#pragma unroll
    for (int c = 0; c < 6; ++c) a.s[c] = a.stress ? p.s[c] : R(0);
#pragma unroll
    for (int c = 0; c < 9; ++c) a.C[c] = C[c];
    a.fex = a.ext ? fex : R(0);
    a.fey = a.ext ? fey : R(0);
    a.fez = a.ext ? fez : R(0);
    return a;
}

// G2P of one particle with the quadratic gather, then its affine matrix:
// C = B * 3/h^2, C *= 0.99 (g2pKernel :577-591; cfac and decay, which the
// textbook form sets to 4/h^2 and 1) unless the particle was CHIP
// (:570-573) or FIXED_BOUNDARY (:516-519) at entry.  C is left in C[] for a
// following P2G.
template <typename R, bool HAS_BACK, typename GatherFn>
__device__ __forceinline__ void apic_g2p(const Particles<R> &P, int i, const G2PIn<R> &in, PState<R> &p,
                                         const Material<R> &M, R dt, double dtd, bool chip_step, bool need_stress,
                                         double zcut, R cfac, R decay, R C[9], GatherFn gather_fn) {
    R B[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) B[c] = R(0);
    g2p_particle<R, HAS_BACK>(P, i, in, p, M, dt, dtd, chip_step, need_stress, zcut,
                              [&](GatherSums<R> &s) { gather_fn(s, B); });
    if (in.status != kChip && in.status != kFixed) {
#pragma unroll
        for (int c = 0; c < 9; ++c) {
            C[c] = B[c] * cfac;
            C[c] = C[c] * decay;
            P.aff[c][i] = C[c];
        }
    } else {
        load_affine(P, i, C);
    }
}

// The walk of a wave over the particles of its layer of cells 64 at a time,
// whatever cells they are of.  In memory a slot's particles follow each other
// in cell order, so the layer's share of a slot is one run, and next() fills
// the lanes with as many of the next runs as it takes (-1 in a lane without a
// particle; all lanes -1 past the last run).  No barriers: the counts of all
// the tile's cells are in the wave's registers.
struct LayerRuns {
    static constexpr int kWaves = kBlock / kWave;
    int cnt[kWaves];            // particles of cell `lane` of each layer
    const int lane, wv;
    int slot = 0, base, off = 0;   // base: first particle of the slot; off: taken of this layer's run

    // (`use` false: no walk, nothing is loaded)
    __device__ __forceinline__ LayerRuns(const int32_t *cells, int first, bool use)
        : lane(threadIdx.x % kWave), wv(threadIdx.x / kWave), base(first) {
        if (use) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) cnt[w] = cells[w * kWave + lane + 1] - cells[w * kWave + lane];
        }
    }

    __device__ __forceinline__ int next() {
        int at = -1, filled = 0;
        while (filled < kWave) {
            int run = 0, before = 0, total = 0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const int c = __popcll(__ballot(cnt[w] > slot));
                if (w == wv) run = c;
                before += w < wv ? c : 0;
                total += c;
            }
            if (run == 0) break;   // no cell of the layer holds more
            const int take = min(run - off, kWave - filled);
            if (lane >= filled && lane < filled + take) at = base + before + off + lane - filled;
            filled += take;
            off += take;
            if (off == run) {
                base += total;
                off = 0;
                ++slot;
            }
        }
        return at;
    }
};

// One workgroup per tile: the APIC G2P and / or P2G.  FP32: thread t owns cell
// t of the tile and walks that cell's particles slot by slot (TileSlots), or, in
// a tile whose non-empty cells hold unequal counts, a wave walks its layer's
// particles 64 at a time (LayerRuns); FP64 takes them in memory order.
// Of a tile shared by `parts` workgroups each takes every parts-th slot, 64
// particles of a layer or run of kBlock particles, and stores a window of its
// own.  The window goes to tpart[block] (QN node records of 8
// channels).  counters[0] counts particles that took device memory in place of
// the tile's window (G2P and P2G each), counters[2] is set when one was
// scattered into the node accumulators, counters[3] counts the queued particles
// that the tile's window holds.
template <typename R, bool DO_G2P, bool DO_P2G, bool HAS_BACK>
__device__ __forceinline__ void apic_tile_block(const Particles<R> &P, const GridView<R> &g, const Grid<R> &G,
                                                const Material<R> &M, R dt, double dtd, double zcut,
                                                G2PFlags flags, double ref_temp, double *part,
                                                const int32_t *cell_start, const TileGeom &tg, int32_t *counters,
                                                R *tpart, int block, int parts) {
    constexpr int kWaves = kBlock / kWave;
    static_assert(TX * TY == kWave && TZ == kWaves, "one cell layer per wave");
    constexpr int kNodeBytes = DO_G2P ? kRowP<R> * QY * QZ * (int)sizeof(vec4_t<R>) : 0;
    constexpr bool kOwn = sizeof(R) == 4;   // windows of the waves' own
    constexpr int kAccBytes = DO_P2G ? (kOwn ? kWaves * 2 * QLN : 2 * QN) * (int)sizeof(vec4_t<R>) : 0;
    __shared__ __align__(32) unsigned char smem[kNodeBytes + kAccBytes];
    __shared__ TileSlotsShared s_slots;   // FP32
    __shared__ uint8_t s_owner[kWaves][DO_P2G && kOwn ? QLB : 1];
    __shared__ int32_t s_q[DO_P2G && kOwn ? kExcQueue : 1];   // particles outside their wave's window
    __shared__ int32_t s_qn;
    vec4_t<R> *s_node = reinterpret_cast<vec4_t<R> *>(smem);
    vec4_t<R> *s_acc = reinterpret_cast<vec4_t<R> *>(smem + kNodeBytes);
    const bool stats = DO_G2P && !DO_P2G && flags.stats != 0;
    const int tid = threadIdx.x, lane = tid % kWave, wv = tid / kWave;
    const int t = block / parts, part0 = block - t * parts;
    const int tx = t % tg.ntx, ty = (t / tg.ntx) % tg.nty, tz = t / (tg.ntx * tg.nty);
    // window node 0 is the node before the tile's first cell
    const int qx0 = tg.ox + tx * TX - 1, qy0 = tg.oy + ty * TY - 1, qz0 = tg.oz + tz * TZ - 1;
    const int b0 = cell_start[t * kTileCells];
    const int b1 = cell_start[(t + 1) * kTileCells];
    const R h = (R)g.hd;
    const R cfac = (R)(g.apic_k * g.inv_hd * g.inv_hd), decay = (R)g.apic_decay;
    double st[kRed];
    stats_identity(st, ref_temp);
    if (b0 < b1) {  // uniform over the workgroup
        if (DO_G2P) {
            for (int w = tid; w < QN; w += kBlock) {
                const int i = qx0 + w % QX, j = qy0 + (w / QX) % QY, k = qz0 + w / (QX * QY);
                vec4_t<R> nd;
                if (i >= 0 && j >= 0 && k >= 0 && i < g.nx && j < g.ny && k < g.nz) {
                    nd = quad_record<R>(G.node[((int64_t)k * g.ny + j) * g.nx + i]);
                } else {
                    nd.x = nd.y = nd.z = R(0);
                    nd.w = R(__builtin_nan(""));
                }
                s_node[qpnode<R>(w % QX, (w / QX) % QY, w / (QX * QY))] = nd;
            }
        }
        vec4_t<R> *const win = s_acc + (DO_P2G && kOwn ? wv * 2 * QLN : 0);
        if (DO_P2G) {
            vec4_t<R> z;
            z.x = z.y = z.z = z.w = R(0);
            if (kOwn) for (int w = lane; w < 2 * QLN; w += kWave) win[w] = z;
            else for (int w = tid; w < 2 * QN; w += kBlock) win[w] = z;
            if (tid == 0) s_qn = 0;
        }
        int my_oow = 0, my_acc = 0, my_queued = 0;
        auto process = [&](const G2PIn<R> &in, int i) {
            PState<R> p;
            p.status = DO_G2P ? in.status : P.status[i];
            if (p.status == kInactive) return;
            const R mass = P.m ? P.m[i] : P.m0, vol = P.m ? P.V[i] : P.V0;
            R fex = R(0), fey = R(0), fez = R(0);
            R C[9];
            if (DO_G2P) {
                const QFrac<R> q = quad_frac(g, in.x, in.y, in.z);
                const int lx = q.b[0] - qx0, ly = q.b[1] - qy0, lz = q.b[2] - qz0;
                const bool inw = (unsigned)lx <= (unsigned)TX && (unsigned)ly <= (unsigned)TY &&
                                 (unsigned)lz <= (unsigned)TZ;
                const int wb = qpnode<R>(lx, ly, lz);
                my_oow += inw ? 0 : 1;
                apic_g2p<R, HAS_BACK>(P, i, in, p, M, dt, dtd, flags.chip != 0, stats, zcut, cfac, decay, C,
                                      [&](GatherSums<R> &s, R B[9]) {
                                          if (inw) quad_gather_window(s_node, wb, q, h, s, B);
                                          else quad_gather_global(g, G.node, q, h, s, B);
                                      });
                if (stats) {
                    const double vx = p.vx, vy = p.vy, vz = p.vz;
                    accumulate_stats(st, p.x, p.y, p.z,
                                     (double)von_mises<R>(p.s[0], p.s[1], p.s[2], p.s[3], p.s[4], p.s[5]),
                                     (double)p.T, 0.5 * (double)mass * (vx * vx + vy * vy + vz * vz));
                }
            } else {
                p.x = P.x[i]; p.y = P.y[i]; p.z = P.z[i];
                load_p2g_state(P, i, p, fex, fey, fez);
                load_affine(P, i, C);
            }
            if (DO_P2G) {
                // after G2P the external force has been consumed (:399)
                const QFrac<R> q = quad_frac(g, p.x, p.y, p.z);
                const int lx = q.b[0] - qx0, ly = q.b[1] - qy0, lz = q.b[2] - qz0;
                const bool inxy = (unsigned)lx <= (unsigned)TX && (unsigned)ly <= (unsigned)TY;
                const QP2G<R> a = quad_inputs(p, C, mass, vol, fex, fey, fez);
                if constexpr (kOwn) {
                    const int layer = lz - wv;
                    if (inxy && (unsigned)layer <= 1u) {
                        quad_scatter_wave(win, s_owner[wv], layer, ly * (TX + 1) + lx, qlnode(lx, ly, layer), q,
                                          quad_scatter_terms(a, q, h));
                        return;
                    }
                    const int at = atomicAdd(&s_qn, 1);
                    if (at < kExcQueue) {
                        s_q[at] = i;
                        my_queued += inxy && (unsigned)lz <= (unsigned)TZ ? 1 : 0;
                        return;
                    }
                } else {
                    if (inxy && (unsigned)lz <= (unsigned)TZ) {
                        quad_scatter_window(reinterpret_cast<double *>(s_acc), qnode(lx, ly, lz), q, h, a);
                        return;
                    }
                }
                my_acc = 1;
                ++my_oow;
                quad_scatter_global(g, G.acc, q, h, a);
            }
        };
        if constexpr (kOwn) {
            // its barriers put the node records and zeros in place
            TileSlots slots(s_slots, b0, cell_start[t * kTileCells + tid + 1] - cell_start[t * kTileCells + tid]);
            // Slot by slot an uneven tile takes as many steps as its fullest
            // cell holds particles, with few of the lanes in most of them.
            // A step, us, slot by slot / 64 at a time (/ the pass of before,
            // any 256 particles at a time with compare-and-swap adds into the
            // tile's window): 786 thousand particles at random 336 / 249
            // (/ 403), 197 thousand at random 155 / 114 (/ 162), 2 % of the
            // cells with 50 particles and the others with one 684 / 223
            // (/ 251), a third missing 195 / 176 (/ 301).  Piles of thousands
            // in a cell share their 8 base nodes and take turns: 20 cells of
            // 4000 33.9 ms / 4.8 (/ 3.5).  In a tile whose cells hold equal
            // counts the slots' particles sit alike in their cells, which
            // keeps their base nodes apart.
            const bool runs_walk = !slots.uniform && !slots.semi;
            LayerRuns runs(cell_start + t * kTileCells, b0, runs_walk);
            // the steps in which the thread has a particle, and the steps
            int cnt = slots.cnt, steps = slots.maxc;
            if (runs_walk) {
                const int layer = cell_start[t * kTileCells + (wv + 1) * kWave] - cell_start[t * kTileCells + wv * kWave];
                cnt = (layer + kWave - 1 - lane) / kWave;
                steps = (layer + kWave - 1) / kWave;
            }
            // particle s of the thread's cell is mine + s * stride
            const int stride = slots.uniform ? kBlock : slots.nnz;
            const int mine = b0 + (slots.uniform ? tid : slots.rank_nz);
            // the thread's particle in step `to`, steps from `from` on not yet passed
            auto index = [&](int from, int to) {
                if (!runs_walk) return mine + to * stride;
                int at = 0;
                for (int k = from; k <= to; ++k) at = runs.next();
                return at;
            };
            // a step's G2P inputs are loaded one step ahead, a step past a
            // thread's last particle loading particle b0, unused
            G2PIn<R> nxt;
            int i_next = index(0, part0);
            if (DO_G2P) load_g2p_in(P, cnt > part0 ? i_next : b0, nxt);
            for (int s = part0; s < steps; s += parts) {
                const G2PIn<R> cur = nxt;
                const int i = i_next;
                i_next = index(s + 1, s + parts);
                if (DO_G2P) load_g2p_in(P, cnt > s + parts ? i_next : b0, nxt);
                if (cnt > s) process(cur, i);
            }
        } else {
            // no window is a wave's own: the particles in memory order, every
            // lane with one
            __syncthreads();
            for (int i = b0 + part0 * kBlock + tid; i < b1; i += kBlock * parts) {
                G2PIn<R> cur;
                if (DO_G2P) load_g2p_in(P, i, cur);
                process(cur, i);
            }
        }
        if constexpr (DO_P2G && !kOwn) {
            __syncthreads();  // every LDS atomic is in
            store_window<R, QN>(tpart + (int64_t)block * (8 * QN), reinterpret_cast<R *>(s_acc), tid);
        }
        if constexpr (DO_P2G && kOwn) {
            __syncthreads();  // every wave's window and the queue are complete
            constexpr int kPer = (QN + kBlock - 1) / kBlock;
            vec4_t<R> a[kPer], b[kPer];
#pragma unroll
            for (int r = 0; r < kPer; ++r) {
                const int w = min(tid + r * kBlock, QN - 1);
                const int x = w % QX, y = (w / QX) % QY, z = w / (QX * QY);
                a[r].x = a[r].y = a[r].z = a[r].w = R(0);
                b[r] = a[r];
#pragma unroll
                for (int v = 0; v < kWaves; ++v) {   // layers z - 3 .. z hold node layer z
                    if ((unsigned)(z - v) < (unsigned)QLZ) {
                        const vec4_t<R> *o = s_acc + v * 2 * QLN + qlnode(x, y, z - v);
                        const vec4_t<R> p0 = o[0], p1 = o[QLN];
                        a[r].x += p0.x; a[r].y += p0.y; a[r].z += p0.z; a[r].w += p0.w;
                        b[r].x += p1.x; b[r].y += p1.y; b[r].z += p1.z; b[r].w += p1.w;
                    }
                }
            }
            const int nq = min(s_qn, kExcQueue);
            if (nq > 0) {  // uniform over the workgroup
                // the tile's window takes the place of the waves'; the queued
                // particles enter it, a lane per node, as the G2P above
                // stored them (the barriers order those stores before these
                // loads); the external force was consumed by the G2P of a
                // fused pass
                __syncthreads();
                vec4_t<R> *const sum = s_acc;
#pragma unroll
                for (int r = 0; r < kPer; ++r) {
                    const int w = tid + r * kBlock;
                    if (w < QN) { sum[2 * w] = a[r]; sum[2 * w + 1] = b[r]; }
                }
                __syncthreads();
                for (int e = tid / 32; e < nq; e += kBlock / 32) {
                    const int i = s_q[e];
                    PState<R> p;
                    p.status = P.status[i];
                    p.x = P.x[i]; p.y = P.y[i]; p.z = P.z[i];
                    R fex = R(0), fey = R(0), fez = R(0), C[9];
                    load_p2g_state(P, i, p, fex, fey, fez);
                    load_affine(P, i, C);
                    if (DO_G2P) fex = fey = fez = R(0);
                    const R mass = P.m ? P.m[i] : P.m0, vol = P.m ? P.V[i] : P.V0;
                    const QFrac<R> q = quad_frac(g, p.x, p.y, p.z);
                    if (quad_scatter_node(g, G.acc, reinterpret_cast<R *>(sum), q.b[0] - qx0, q.b[1] - qy0,
                                          q.b[2] - qz0, q, h, quad_inputs(p, C, mass, vol, fex, fey, fez), tid % 32)) {
                        my_acc = 1;
                        my_oow += tid % 32 == 0;
                    }
                }
                __syncthreads();  // the queued scatters are in
#pragma unroll
                for (int r = 0; r < kPer; ++r) {
                    const int w = min(tid + r * kBlock, QN - 1);
                    a[r] = sum[2 * w];
                    b[r] = sum[2 * w + 1];
                }
            }
            vec4_t<R> *const out = reinterpret_cast<vec4_t<R> *>(tpart + (int64_t)block * (8 * QN));
#pragma unroll
            for (int r = 0; r < kPer; ++r) {
                const int w = tid + r * kBlock;
                if (w < QN) { out[2 * w] = a[r]; out[2 * w + 1] = b[r]; }
            }
        }
        int cntv = my_oow, cnta = my_acc, cntq = my_queued;
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) {
            cntv += __shfl_xor(cntv, o, kWave);
            cnta |= __shfl_xor(cnta, o, kWave);
            cntq += __shfl_xor(cntq, o, kWave);
        }
        if (lane == 0 && cntv) atomicAdd(counters, cntv);
        if (lane == 0 && cntq) atomicAdd(counters + 3, cntq);
        if (lane == 0 && cnta) atomicOr(counters + 2, 1);
    } else if (DO_P2G) {
        zero_window<R, QN>(tpart + (int64_t)block * (8 * QN), tid);
    }
    if (stats) block_reduce_stats(st, part, block);
}

// Waves per SIMD: two, but for FP64's G2P-only pass, which needs more
// registers than that leaves (fused FP64, 4.2 M particles, 50 steps: 43.5 ms;
// one wave 52).
template <typename R, bool DO_G2P, bool DO_P2G, bool HAS_BACK>
__global__ void __launch_bounds__(kBlock, sizeof(R) == 4 || DO_P2G ? 2 : 1) k_apic_tile_batch(const TileWork<R> *__restrict__ items,
                                                                                int nitems, int order) {
    const int b = launch_block(order);
    const int w = find_item(items, nitems, b);
    const TileWork<R> &W = items[w];
    apic_tile_block<R, DO_G2P, DO_P2G, HAS_BACK>(W.P, W.g, W.G, W.M, W.dt, W.dtd, W.zcut, W.flags, W.ref_temp,
                                                 W.part, W.cell_start, W.tg, W.counters, W.tpart, b - W.block0,
                                                 W.parts);
}

// The loose particles of the APIC pass, one thread each, nodes read from
// and accumulated into device memory (sets acc_flag).  Statistics partials
// go to part[blockIdx.x].
template <typename R, bool DO_G2P, bool DO_P2G, bool HAS_BACK>
__global__ void __launch_bounds__(kBlock)
    k_apic_loose(Particles<R> P, GridView<R> g, Grid<R> G, Material<R> M, R dt, double dtd, double zcut,
                 G2PFlags flags, double ref_temp, double *part, int32_t begin, int32_t end, int32_t *acc_flag) {
    double st[kRed];
    stats_identity(st, ref_temp);
    const int i = begin + (int)blockIdx.x * kBlock + (int)threadIdx.x;
    const R h = (R)g.hd;
    const R cfac = (R)(g.apic_k * g.inv_hd * g.inv_hd), decay = (R)g.apic_decay;
    if (i < end) {
        PState<R> p;
        p.status = P.status[i];
        if (p.status != kInactive) {
            const R mass = P.m ? P.m[i] : P.m0, vol = P.m ? P.V[i] : P.V0;
            R fex = R(0), fey = R(0), fez = R(0);
            R C[9];
            if (DO_G2P) {
                G2PIn<R> in;
                load_g2p_in(P, i, in);
                const QFrac<R> q = quad_frac(g, in.x, in.y, in.z);
                apic_g2p<R, HAS_BACK>(P, i, in, p, M, dt, dtd, flags.chip != 0, flags.stats != 0, zcut, cfac, decay, C,
                                      [&](GatherSums<R> &s, R B[9]) { quad_gather_global(g, G.node, q, h, s, B); });
                if (flags.stats) {
                    const double vx = p.vx, vy = p.vy, vz = p.vz;
                    accumulate_stats(st, p.x, p.y, p.z,
                                     (double)von_mises<R>(p.s[0], p.s[1], p.s[2], p.s[3], p.s[4], p.s[5]),
                                     (double)p.T, 0.5 * (double)mass * (vx * vx + vy * vy + vz * vz));
                }
            } else {
                p.x = P.x[i]; p.y = P.y[i]; p.z = P.z[i];
                load_p2g_state(P, i, p, fex, fey, fez);
                load_affine(P, i, C);
            }
            if (DO_P2G) {
                const QFrac<R> q = quad_frac(g, p.x, p.y, p.z);
                quad_scatter_global(g, G.acc, q, h, quad_inputs(p, C, mass, vol, fex, fey, fez));
                atomicOr(acc_flag, 1);
            }
        }
    }
    if (DO_G2P && flags.stats) block_reduce_stats(st, part, (int)blockIdx.x);
}

}  // namespace mpmw
