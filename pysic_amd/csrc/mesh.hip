// mesh.hip -- the reciprocal Ewald sums of large systems over a mesh.
//
// The structure factors S(k) = sum_a q_a e^{i k.r_a} of all half-space
// k-vectors and the per-atom field Phi(r_i) = sum_k 2 c_k Re(S(k) e^{-i k.r_i})
// (with its gradient) are the sums that ewald.hip forms ion by ion in
// O(N N_k).  Here they are non-uniform Fourier transforms: spread the
// charges on a regular mesh with a short kernel, transform the mesh, divide
// by the kernel's transform (Dutt & Rokhlin, SIAM J. Sci. Comput. 14, 1993),
// and the adjoint for the field.  The k-vectors and their coefficients are
// the direct sum's (same set, same cutoff test), so nothing is truncated
// but the kernel's tail: with a window of W = 16 points, a mesh of at least
// 4 K + 4 points per axis and the kernel
//   phi(x) = exp(beta (sqrt(1 - (2x/W)^2) - 1)), beta = 2.55 W
// (Barnett, Magland & af Klinteberg, SIAM J. Sci. Comput. 41, 2019), the
// error against extended precision is the direct FP64 sum's: reciprocal forces
// of disordered ions, 2,500 of K = 28 1.8e-15 against 1.2 to 1.7e-15, 1,200 of
// K = 47 3.6e-15 against 3.5e-15; electronegativities 6e-16 against 8e-16.
// A smaller beta leaves a larger tail, which the forces of the long waves show,
// n / k of it (2.45 W: 5.3e-15 and 5e-15); a larger one costs the band edge.
//
// Everything is FP64 and free of atomics on values: each mesh tile sums its
// atoms in a fixed order, each atom sums its tiles in a fixed order.
//
// Measured, energy + forces of 262,144 ions, 852,533 k-vectors, mesh 304^3:
// the reciprocal part takes 2.2 ms where the direct sums take 125 ms; one
// electronegativity evaluation of 24,576 ions (mesh 128 x 120 x 120) 0.16 ms
// against 0.84 ms.  The direct sums stay where they cost less (mesh_suits):
// few ions or k-vectors, and ions crowded into few mesh tiles.
//
//  k_mesh_bin/scan/fill/order  counting sort of the atoms by mesh tile
//  k_mesh_weights              kernel values (and derivatives) per atom, axis
//  k_mesh_spread               charges to mesh, a contraction over atoms (MFMA)
//  k_dft_forward x 3           separable transform, pruned to |k_d| <= K_d:
//                              dense cosine and sine products per axis (MFMA),
//                              mirrored points folded first
//  k_mesh_combine              S(k), energy, coefficients of the field
//  k_dft_inverse x 3           the adjoint transforms
//  k_mesh_field                field and gradient at the atoms (MFMA)
//  k_mesh_finish               per-atom sums over tiles
#include "ewald.h"

#include <algorithm>
#include <cmath>

namespace {

typedef double mfma_d4 __attribute__((ext_vector_type(4)));

constexpr int W = 16;                       // window points per axis
constexpr double BETA = 2.55 * W;
constexpr int TX = 16, TY = 8, TZ = 8;      // mesh tile of one wave
constexpr int SLOTS = 18;                   // tiles an atom can meet: 2 x 3 x 3
constexpr int MB = 256;
constexpr int MT_MAX = 5;                   // 16-row output tiles per wave of a transform

struct MeshGeo {
    int n[3];     // mesh points
    int nb[3];    // tiles
    double f[9];  // rows of the inverse cell matrix
};

// Fractional coordinate d of r, reduced to [0, 1], and the first point of
// its window (not yet reduced to the mesh).  Used by every kernel that needs
// either, with the operations spelled out, so that all agree.
__device__ __forceinline__ double mesh_frac(const MeshGeo &g, int d, const double4 &r, int *g0)
{
    const double u = fma(g.f[3 * d + 2], r.z, fma(g.f[3 * d + 1], r.y, g.f[3 * d] * r.x));
    double v = u - floor(u);
    if (!(v >= 0.0 && v <= 1.0)) v = 0.0;
    *g0 = (int)ceil(v * g.n[d] - 0.5 * W);
    return v;
}

__global__ __launch_bounds__(MB) void k_mesh_bin(int n, MeshGeo g, const double4 *__restrict__ pos,
                                                 int *__restrict__ bin, int *__restrict__ count)
{
    const int i = blockIdx.x * MB + threadIdx.x;
    if (i >= n) return;
    const double4 r = pos[i];
    int c[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int g0;
        mesh_frac(g, d, r, &g0);
        if (g0 < 0) g0 += g.n[d];
        c[d] = g0 / (d == 0 ? TX : d == 1 ? TY : TZ);
    }
    const int b = c[0] + g.nb[0] * (c[1] + g.nb[1] * c[2]);
    bin[i] = b;
    atomicAdd(count + b, 1);
}

// Exclusive scan of the tile counts, one block; clears the counts for the
// next sort and the fill counters for this one.  The arrays are padded to
// whole int4 per thread (scan_room), so a thread's loads are wide and all in
// flight at once: 27,436 tiles 66 -> 21 us.
__global__ __launch_bounds__(1024) void k_mesh_scan(int nbins, int per4, int4 *__restrict__ count,
                                                    int4 *__restrict__ fill,
                                                    int4 *__restrict__ start,
                                                    int *__restrict__ last)
{
    __shared__ int lds[1024];
    const int t = threadIdx.x;
    int s = 0;
#pragma unroll 8
    for (int b = t * per4; b < (t + 1) * per4; ++b) {
        const int4 c = count[b];
        s += (c.x + c.y) + (c.z + c.w);
    }
    lds[t] = s;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const int x = t >= d ? lds[t - d] : 0;
        __syncthreads();
        lds[t] += x;
        __syncthreads();
    }
    int at = lds[t] - s;
    const int4 zero = make_int4(0, 0, 0, 0);
#pragma unroll 8
    for (int b = t * per4; b < (t + 1) * per4; ++b) {
        const int4 c = count[b];
        start[b] = make_int4(at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z);
        count[b] = zero;
        fill[b] = zero;
        at += (c.x + c.y) + (c.z + c.w);
    }
    __syncthreads();
    if (t == 1023) last[nbins] = lds[1023];   // the end of the last tile
}

__global__ __launch_bounds__(MB) void k_mesh_fill(int n, const int *__restrict__ bin,
                                                  const int *__restrict__ start,
                                                  int *__restrict__ fill, int *__restrict__ claim)
{
    const int i = blockIdx.x * MB + threadIdx.x;
    if (i < n) claim[start[bin[i]] + atomicAdd(fill + bin[i], 1)] = i;
}

// The atoms of a tile in slot order (their claims are unordered): one wave
// per tile, each lane counts the smaller slots.
__global__ __launch_bounds__(64) void k_mesh_order(const int *__restrict__ start,
                                                   const int *__restrict__ claim,
                                                   int *__restrict__ order)
{
    const int a = start[blockIdx.x], b = start[blockIdx.x + 1];
    for (int x = a + threadIdx.x; x < b; x += 64) {
        const int v = claim[x];
        int rank = 0;
        for (int y = a; y < b; ++y) rank += claim[y] < v ? 1 : 0;
        order[a + rank] = v;
    }
}

// phi (D = false) or dphi/dx (D = true) at the window points of atom a along
// each axis: w[a * 48 + 16 d + o].  The distance to the first window point
// is one fma, so it carries no error of the mesh coordinate's size, and the
// exponent is written without the cancellation of sqrt - 1.  The derivative
// has an integrable 1/sqrt edge where phi is e^-beta = 2e-18; the root is
// held at 1e-2 there, which changes dphi by some 1e-15.
// at[a] = (window origin on the mesh, slot).
template <bool D>
__global__ __launch_bounds__(MB) void k_mesh_weights(int n, MeshGeo g,
                                                     const double4 *__restrict__ pos,
                                                     const int *__restrict__ order,
                                                     double *__restrict__ w, int4 *__restrict__ at)
{
    const long e = (long)blockIdx.x * MB + threadIdx.x;
    const int a = (int)(e / 48), c = (int)(e - 48L * a), d = c >> 4, o = c & 15;
    if (a >= n) return;
    const int i = order[a];
    const double4 r = pos[i];
    int g0;
    const double v = mesh_frac(g, d, r, &g0);
    const double y = (fma(-v, (double)g.n[d], (double)g0) + o) * (2.0 / W);
    const double y2 = y * y;
    const double s = sqrt(fmax(1.0 - y2, 0.0));
    const double p = exp(-BETA * y2 / (1.0 + s));
    w[e] = D ? p * (-BETA * (2.0 / W)) * y / fmax(s, 1e-2) : p;
    if (!D && c == 0) {
        int h[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            mesh_frac(g, k, r, h + k);
            if (h[k] < 0) h[k] += g.n[k];
        }
        at[a] = make_int4(h[0], h[1], h[2], i);
    }
}

// Bin s of the 2 x 3 x 3 that end at tile (tx, ty, tz).
__device__ __forceinline__ int stream_bin(const MeshGeo &g, int tx, int ty, int tz, int s)
{
    int bx = tx - (s & 1), by = ty - (s >> 1) % 3, bz = tz - (s >> 1) / 3;
    bx += bx < 0 ? g.nb[0] : 0;
    by += by < 0 ? g.nb[1] : 0;
    bz += bz < 0 ? g.nb[2] : 0;
    return bx + g.nb[0] * (by + g.nb[1] * bz);
}

// The atoms whose windows meet tile (tx, ty, tz): those of its 18 bins.  Lane s < 18 holds bin s; base[s] is the first stream
// position of bin s, base[18] the total.
__device__ __forceinline__ void tile_stream(const MeshGeo &g, int tx, int ty, int tz,
                                            const int *__restrict__ start, int *first, int *base)
{
    const int s = threadIdx.x;
    int len = 0, a = 0;
    if (s < SLOTS) {
        const int b = stream_bin(g, tx, ty, tz, s);
        a = start[b];
        len = start[b + 1] - a;
    }
    int incl = len;
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
        const int x = __shfl_up(incl, d);
        if (s >= d) incl += x;
    }
    if (s < SLOTS) {
        first[s] = a;
        base[s] = incl - len;
    }
    if (s == SLOTS - 1) base[SLOTS] = incl;
}

// tile origin - window origin on a periodic axis of n points: in 0 .. W - 1
// when the tile starts inside the window, else negative, and above minus the
// tile's length exactly when the window starts inside the tile (n >= W + tile,
// so never both)
__device__ __forceinline__ int window_rel(int tile0, int g0, int n)
{
    int o = tile0 - g0;
    o += o < 0 ? n : 0;
    return o >= W ? o - n : o;
}

constexpr int FAR = -100000;   // the rel of an empty place: no window there

// Stream positions c0 .. c0 + 63 of a tile: (rel of each axis, atom), the atom
// -1 past the end, and which of the 18 bins it came from.
__device__ __forceinline__ void tile_chunk(const MeshGeo &g, int tx, int ty, int tz, int c0,
                                           const int *first, const int *base,
                                           const int4 *__restrict__ at, int4 *s_at, int *s_bin,
                                           int *slot)
{
    const int c = c0 + threadIdx.x;
    int4 v = make_int4(FAR, FAR, FAR, 0);
    int bin = -1;
    if (c < base[SLOTS]) {
        bin = 0;
        for (int s = 1; s < SLOTS; ++s) bin = c >= base[s] ? s : bin;
        const int atom = first[bin] + (c - base[bin]);
        const int4 o = at[atom];
        *slot = o.w;
        v = make_int4(window_rel(tx * TX, o.x, g.n[0]), window_rel(ty * TY, o.y, g.n[1]),
                      window_rel(tz * TZ, o.z, g.n[2]), atom);
    }
    s_at[threadIdx.x] = v;
    if (s_bin) s_bin[threadIdx.x] = bin;
}

// A group of 16 atoms in the tile's own coordinates: 16 x, 8 y and 8 z values
// of each atom's kernel at the tile's points, zero outside its window, so the
// product loops read them at fixed offsets and compute no index.  Lane L
// takes entry L % 32 of atoms 2 j + L / 32.  STRIDE doubles a row.
template <int STRIDE>
struct Group {
    double v[8];
    static __device__ __forceinline__ int axis() { return (threadIdx.x & 31) < 16 ? 0 : (threadIdx.x & 31) < 24 ? 1 : 2; }
    __device__ __forceinline__ void load(const int4 *s_at, int t, const double *__restrict__ w)
    {
        const int e = threadIdx.x & 31, ax = axis(), p = e - (ax == 0 ? 0 : ax == 1 ? 16 : 24);
        const int *rec = (const int *)(s_at + 16 * t + (threadIdx.x >> 5));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int o = rec[8 * j + ax] + p;
            const bool in = (unsigned)o < (unsigned)W;
            const double x = w[(size_t)rec[8 * j + 3] * 48 + 16 * ax + (in ? o : 0)];
            v[j] = in ? x : 0.0;
        }
    }
    __device__ __forceinline__ void store(double *lds) const
    {
        double *row = lds + (threadIdx.x >> 5) * STRIDE + (threadIdx.x & 31);
#pragma unroll
        for (int j = 0; j < 8; ++j) row[2 * j * STRIDE] = v[j];
    }
};

// Charges to the mesh.  A wave owns a tile of 16 x 8 x 8 points: for atom a
// the tile gains q_a phi(y) phi(z) (64 rows) times phi(x) (16 columns), so the
// tile is a (64 x atoms) by (atoms x 16) product: FP64 MFMA 16x16x4, four
// row blocks of 4 y by 4 z, 4 atoms a step.  The kernel values of 16 atoms
// are staged in LDS in the tile's coordinates while the next 16 load.
// Bound: half the time the matrix pipe (44 steps of 4 products a tile, 126 us
// in all at its peak), else the wait for the next group's values, which come
// from L2 or beyond.  262,144 ions, 304^3 points: 302 us with five gathers
// from global memory a step, 254 staged.
// Lane L: A row L % 16 (y = L % 4, z = L / 4 % 4) of atom L / 16; B column
// L % 16 (x) of atom L / 16; D row L / 16 + 4 r in register r.
__global__ __launch_bounds__(64) void k_mesh_spread(MeshGeo g, const int *__restrict__ start,
                                                    const int4 *__restrict__ at,
                                                    const double *__restrict__ w,
                                                    const double *__restrict__ q,
                                                    const double *__restrict__ sc,
                                                    double *__restrict__ mesh)
{
    __shared__ int first[SLOTS], base[SLOTS + 1];
    __shared__ int4 s_at[64];
    __shared__ double s_q[64];
    constexpr int STRIDE = 48;   // a step's four rows on alternate halves of the banks
    __shared__ double s_w[16 * STRIDE];
    const int lane = threadIdx.x, col = lane & 15, kq = lane >> 4;
    const int blk = xcd_block(gridDim.x);
    const int tx = blk % g.nb[0], ty = blk / g.nb[0] % g.nb[1], tz = blk / (g.nb[0] * g.nb[1]);
    tile_stream(g, tx, ty, tz, start, first, base);
    __syncthreads();
    const int total = base[SLOTS];
    const double *px = s_w + kq * STRIDE + col, *py = s_w + kq * STRIDE + 16 + (col & 3),
                 *pz = s_w + kq * STRIDE + 24 + (col >> 2);
    mfma_d4 acc[2][2];
#pragma unroll
    for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[z][y] = mfma_d4{0.0, 0.0, 0.0, 0.0};
    for (int c0 = 0; c0 < total; c0 += 64) {
        int slot = -1;
        tile_chunk(g, tx, ty, tz, c0, first, base, at, s_at, nullptr, &slot);
        s_q[lane] = slot >= 0 ? q[slot] * sc[slot] : 0.0;
        __syncthreads();
        const int groups = min(4, (total - c0 + 15) >> 4);
        Group<STRIDE> v;
        v.load(s_at, 0, w);
        for (int t = 0; t < groups; ++t) {
            if ((lane & 31) < 16) {   // the x values carry the charge
#pragma unroll
                for (int j = 0; j < 8; ++j) v.v[j] *= s_q[16 * t + 2 * j + (lane >> 5)];
            }
            v.store(s_w);
            __syncthreads();
            if (t + 1 < groups) v.load(s_at, t + 1, w);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int o = 4 * k * STRIDE;
                const double b = px[o], y0 = py[o], y1 = py[o + 4], z0 = pz[o], z1 = pz[o + 4];
                acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(y0 * z0, b, acc[0][0], 0, 0, 0);
                acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(y1 * z0, b, acc[0][1], 0, 0, 0);
                acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(y0 * z1, b, acc[1][0], 0, 0, 0);
                acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(y1 * z1, b, acc[1][1], 0, 0, 0);
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // row kq + 4 r of the block: y = kq, z = r
                const size_t Y = ty * TY + 4 * y + kq, Z = tz * TZ + 4 * z + r;
                mesh[(Z * g.n[1] + Y) * g.n[0] + tx * TX + col] = acc[z][y][r];
            }
}

// One axis of the transform, mesh to k: for every column c (all other
// indices) of every input array,
//   out_c[k] = sum_g cos(2 pi k g / n) in[g],  out_s[k] = the same with sin,
// k = 0 .. K.  Points g and n - g are folded first, which halves the
// products: cos takes in[g] + in[n - g], sin their difference, g <= n / 2
// (the table halves the two self-mirrored points).  A wave owns MT tiles of
// 16 k by 16 columns of both; lane L: A row L % 16 of point L / 16 (from the
// table in this order, a coalesced 512 bytes), B column L % 16 of point
// L / 16.  Bound: the matrix pipe.
// The table of 4 steps is staged in LDS for the block's four waves, the next
// 4 steps' table and mesh values loading meanwhile: read by every wave for
// itself the table alone is 1.2 GB from L2 a pass on 304^3 points.
// Mesh to k, 304^3 points, K = 74, three axes: 275 -> 245 us; k to mesh 327
// -> 294 us.
constexpr int DS = 4;   // steps per staged table

// table values of steps t0 .. t0 + 3 of the wave's tiles: MT double2 a thread
template <int MT>
__device__ __forceinline__ void table_load(const double *__restrict__ tab, int m0, int mtiles,
                                           int steps, int t0, double2 (&v)[MT])
{
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        // pair e of the staged block: [sine][tile][step][32 pairs]
        const int e = j * MB + threadIdx.x;
        const int p = e & 31, t = t0 + ((e >> 5) & (DS - 1)), m = (e >> 7) % MT, sn = (e >> 7) / MT;
        const bool on = m0 + m < mtiles && t < steps;
        const double2 *src = (const double2 *)tab +
                             (((size_t)sn * mtiles + m0 + (on ? m : 0)) * steps + (on ? t : 0)) * 32 + p;
        const double2 x = *src;
        v[j] = on ? x : make_double2(0.0, 0.0);
    }
}

template <int MT>
__global__ __launch_bounds__(MB) void k_dft_forward(int n, int K, int inner, long cols, int steps,
                                                    int mtiles, const double *__restrict__ tab,
                                                    const double *__restrict__ in, long in_size,
                                                    double *__restrict__ out, long out_size)
{
    __shared__ double2 s_tab[2][MT * MB];
    const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
    const long c = ((long)blockIdx.x * (MB / 64) + (threadIdx.x >> 6)) * 16 + col;
    const long cl = c < cols ? c : cols - 1;   // waves past the columns load the last one
    const int m0 = blockIdx.y * MT;
    const long o = cl / inner, i = cl - o * inner;
    const double *src = in + blockIdx.z * in_size + o * n * inner + i;
    mfma_d4 ac[MT], as[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) ac[m] = as[m] = mfma_d4{0.0, 0.0, 0.0, 0.0};
    const int half = n / 2;
    double x[DS], y[DS];
    auto load = [&](int t0) {
#pragma unroll
        for (int u = 0; u < DS; ++u) {
            const int p = min(4 * (t0 + u) + kq, half);
            x[u] = src[(long)p * inner];
            y[u] = src[(long)(p ? n - p : 0) * inner];
        }
    };
    double2 v[MT];
    table_load<MT>(tab, m0, mtiles, steps, 0, v);
    load(0);
    for (int t0 = 0, b = 0; t0 < steps; t0 += DS, b ^= 1) {
#pragma unroll
        for (int j = 0; j < MT; ++j) s_tab[b][j * MB + threadIdx.x] = v[j];
        double e[DS], d[DS];
#pragma unroll
        for (int u = 0; u < DS; ++u) {
            e[u] = x[u] + y[u];
            d[u] = x[u] - y[u];
        }
        __syncthreads();   // also: the other buffer's readers are done
        if (t0 + DS < steps) {
            table_load<MT>(tab, m0, mtiles, steps, t0 + DS, v);
            load(t0 + DS);
        }
        const double *tc = (const double *)s_tab[b] + lane;
#pragma unroll
        for (int u = 0; u < DS; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                ac[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(tc[(m * DS + u) * 64], e[u], ac[m],
                                                             0, 0, 0);
                as[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(tc[((MT + m) * DS + u) * 64], d[u],
                                                             as[m], 0, 0, 0);
            }
    }
    if (c >= cols) return;
    double *oc = out + 2 * blockIdx.z * out_size + o * (K + 1) * inner + i, *os = oc + out_size;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = (m0 + m) * 16 + kq + 4 * r;
            if (k > K) continue;
            oc[(long)k * inner] = ac[m][r];
            os[(long)k * inner] = as[m][r];
        }
}

// The adjoint axis, k to mesh: out[g] = sum_k cos in_c[k] + sin in_s[k] for
// all g of the axis, from the even part E[g] = sum cos in_c and the odd part
// O[g] = sum sin in_s, g <= n / 2: out[g] = E + O, out[n - g] = E - O.
template <int MT>
__global__ __launch_bounds__(MB) void k_dft_inverse(int n, int K, int inner, long cols, int steps,
                                                    int mtiles, const double *__restrict__ tab,
                                                    const double *__restrict__ in, long in_size,
                                                    double *__restrict__ out, long out_size)
{
    __shared__ double2 s_tab[2][MT * MB];
    const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
    const long c = ((long)blockIdx.x * (MB / 64) + (threadIdx.x >> 6)) * 16 + col;
    const long cl = c < cols ? c : cols - 1;   // waves past the columns load the last one
    const int m0 = blockIdx.y * MT;
    const long o = cl / inner, i = cl - o * inner;
    const double *src = in + 2 * blockIdx.z * in_size + o * (K + 1) * inner + i;
    mfma_d4 ae[MT], ao[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) ae[m] = ao[m] = mfma_d4{0.0, 0.0, 0.0, 0.0};
    double x[DS], y[DS];
    auto load = [&](int t0) {
#pragma unroll
        for (int u = 0; u < DS; ++u) {
            const int k = min(4 * (t0 + u) + kq, K);
            x[u] = src[(long)k * inner];
            y[u] = src[in_size + (long)k * inner];
        }
    };
    double2 v[MT];
    table_load<MT>(tab, m0, mtiles, steps, 0, v);
    load(0);
    for (int t0 = 0, b = 0; t0 < steps; t0 += DS, b ^= 1) {
#pragma unroll
        for (int j = 0; j < MT; ++j) s_tab[b][j * MB + threadIdx.x] = v[j];
        double e[DS], d[DS];
#pragma unroll
        for (int u = 0; u < DS; ++u) {
            e[u] = x[u];
            d[u] = y[u];
        }
        __syncthreads();   // also: the other buffer's readers are done
        if (t0 + DS < steps) {
            table_load<MT>(tab, m0, mtiles, steps, t0 + DS, v);
            load(t0 + DS);
        }
        const double *tc = (const double *)s_tab[b] + lane;
#pragma unroll
        for (int u = 0; u < DS; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                ae[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(tc[(m * DS + u) * 64], e[u], ae[m],
                                                             0, 0, 0);
                ao[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(tc[((MT + m) * DS + u) * 64], d[u],
                                                             ao[m], 0, 0, 0);
            }
    }
    if (c >= cols) return;
    double *dst = out + blockIdx.z * out_size + o * n * inner + i;
    const int half = n / 2;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int p = (m0 + m) * 16 + kq + 4 * r;
            if (p > half) continue;
            dst[(long)p * inner] = ae[m][r] + ao[m][r];
            if (p > 0 && p < half) dst[(long)(n - p) * inner] = ae[m][r] - ao[m][r];
        }
}

// Coefficients c_k of the k-vectors of an octant: coef[4 e + 2 s2 + s1] for
// (k1, k2, k3) = (s1 ? -a : a, s2 ? -b : b, c), e = (c (K2 + 1) + b) (K1 + 1)
// + a; zero beyond the cutoff, at k = 0 and for the second signs of 0.  The
// cutoff test is formed as on the host (no contraction), so the set is the
// direct sum's.
__global__ __launch_bounds__(MB) void k_mesh_coef(int K1, int K2, int K3, double4 b0, double4 b1,
                                                  double4 b2, double kc2, double inv_eps_2v,
                                                  double half_sigma2, double *__restrict__ coef)
{
#pragma clang fp contract(off)
    const int e = blockIdx.x * MB + threadIdx.x;
    if (e >= (K1 + 1) * (K2 + 1) * (K3 + 1)) return;
    const int a = e % (K1 + 1), b = e / (K1 + 1) % (K2 + 1), c = e / ((K1 + 1) * (K2 + 1));
    for (int s = 0; s < 4; ++s) {
        double v = 0.0;
        if (!(a == 0 && (s & 1)) && !(b == 0 && (s & 2)) && (a || b || c)) {
            const int k1 = (s & 1) ? -a : a, k2 = (s & 2) ? -b : b;
            const double x = k1 * b0.x + k2 * b1.x + c * b2.x;
            const double y = k1 * b0.y + k2 * b1.y + c * b2.y;
            const double z = k1 * b0.z + k2 * b1.z + c * b2.z;
            const double kk = x * x + y * y + z * z;
            if (kk < kc2) v = inv_eps_2v * (c == 0 ? 1.0 : 2.0) * exp(-half_sigma2 * kk) / kk;
        }
        coef[4 * (size_t)e + s] = v;
    }
}

// From the octant's eight products of cosines and sines (array 4 z + 2 y + x,
// bit set: sine of that axis) to S(k) of the four sign choices, the energy
// sum c_k |S(k)|^2 (block partials), and back to the octant's coefficients of
// Phi(r) = sum_k 2 c_k Re(S(k) e^{-i k.r}), in place.  dec: the reciprocal
// kernel transforms per axis (once for the spreading, once for the field).
__global__ __launch_bounds__(MB) void k_mesh_combine(int K1, int K2, int K3,
                                                     const double *__restrict__ dec,
                                                     const double *__restrict__ coef,
                                                     double *__restrict__ oct,
                                                     double *__restrict__ part)
{
    __shared__ double red[MB];
    const long size = (long)(K1 + 1) * (K2 + 1) * (K3 + 1);
    const long e = (long)blockIdx.x * MB + threadIdx.x;
    double en = 0.0;
    if (e < size) {
        const int a = e % (K1 + 1), b = e / (K1 + 1) % (K2 + 1), c = e / ((K1 + 1) * (K2 + 1));
        const double dc = dec[a] * dec[K1 + 1 + b] * dec[K1 + K2 + 2 + c];
        double p[8], z[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            p[t] = oct[t * size + e] * dc;
            z[t] = 0.0;
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double ck = coef[4 * e + s];
            const double s1 = (s & 1) ? -1.0 : 1.0, s2 = (s & 2) ? -1.0 : 1.0, s12 = s1 * s2;
            // e^{i(s1 t1 + s2 t2 + t3)}, bits of the array index: 1 x, 2 y, 4 z
            const double re = p[0] - s2 * p[6] - s1 * p[5] - s12 * p[3];
            const double im = s1 * p[1] + s2 * p[2] + p[4] - s12 * p[7];
            en += ck * (re * re + im * im);
            const double zr = 2.0 * ck * dc * re, zi = 2.0 * ck * dc * im;
            z[0] += zr;
            z[6] -= s2 * zr;
            z[5] -= s1 * zr;
            z[3] -= s12 * zr;
            z[1] += s1 * zi;
            z[2] += s2 * zi;
            z[4] += zi;
            z[7] -= s12 * zi;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) oct[t * size + e] = z[t];
    }
    red[threadIdx.x] = en;
    __syncthreads();
    for (int w = MB / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// The field at the atoms, tile by tile: for 16 atoms of the tile's stream and
// its 16 x 8 x 8 points, T[atom][yz] = sum_x phi_x(atom, x) mesh[yz][x] is a
// (16 x 16) by (16 x 64) product on the matrix cores with the mesh values
// held in registers; each lane then contracts its column of T with
// phi(y) phi(z), and the 16 columns are summed through LDS.  With FORCE the
// gradient comes from the kernel's derivative: the same with phi'_x, phi'_y
// and phi'_z, so one mesh serves all three components (three transforms of
// i k Phi would cost three inverse transforms).  part[(a * 18 + slot) * NC]
// takes what this tile gives atom a; every slot is written by one tile.
// The kernel values of the 16 atoms are staged in LDS as in k_mesh_spread;
// the sums reuse that space once the values have been read.
// Bound: 32 products per 16 atoms and tile with FORCE (16 without), 260 us at
// the matrix pipe's peak for 262,144 ions, and as much again in the FP64
// contraction, which shares that pipe, and in waiting for values at two waves
// per SIMD.  Forces of 262,144 ions: 774 us with gathers from global memory,
// 642 staged.
template <bool FORCE>
__global__ __launch_bounds__(64) void k_mesh_field(MeshGeo g, const int *__restrict__ start,
                                                   const int4 *__restrict__ at,
                                                   const double *__restrict__ w,
                                                   const double *__restrict__ dw,
                                                   const double *__restrict__ mesh,
                                                   double *__restrict__ part)
{
    constexpr int NC = FORCE ? 3 : 1;
    __shared__ int first[SLOTS], base[SLOTS + 1];
    __shared__ int4 s_at[64];
    __shared__ int s_bin[64];
    constexpr int STRIDE = 36;   // the 16 rows of an A operand spread over the banks
    constexpr int RED = NC * 16 * 17, VAL = (FORCE ? 2 : 1) * 16 * STRIDE;
    __shared__ double s_w[RED > VAL ? RED : VAL];   // the sums take the staged values' place
    double *s_dw = s_w + (FORCE ? 16 * STRIDE : 0), *red = s_w;
    const int lane = threadIdx.x, col = lane & 15, kq = lane >> 4;
    const int blk = xcd_block(gridDim.x);
    const int tx = blk % g.nb[0], ty = blk / g.nb[0] % g.nb[1], tz = blk / (g.nb[0] * g.nb[1]);
    tile_stream(g, tx, ty, tz, start, first, base);
    __syncthreads();
    const int total = base[SLOTS];
    if (total == 0) return;
    // B operands: point x = 4 s + kq of column (y, z) = col of block (bz, by)
    double f[2][2][4];
#pragma unroll
    for (int z = 0; z < 2; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                f[z][y][s] = mesh[((size_t)(tz * TZ + (col >> 2) + 4 * z) * g.n[1] + ty * TY +
                                   (col & 3) + 4 * y) * g.n[0] + tx * TX + 4 * s + kq];
    for (int c0 = 0; c0 < total; c0 += 64) {
        int slot = -1;
        tile_chunk(g, tx, ty, tz, c0, first, base, at, s_at, s_bin, &slot);
        __syncthreads();
        const int groups = min(4, (total - c0 + 15) >> 4);
        Group<STRIDE> v, dv;
        v.load(s_at, 0, w);
        if (FORCE) dv.load(s_at, 0, dw);
        for (int t = 0; t < groups; ++t) {
            v.store(s_w);
            if (FORCE) dv.store(s_dw);
            __syncthreads();
            if (t + 1 < groups) {
                v.load(s_at, t + 1, w);
                if (FORCE) dv.load(s_at, t + 1, dw);
            }
            mfma_d4 T[2][2], U[2][2];
#pragma unroll
            for (int z = 0; z < 2; ++z)
#pragma unroll
                for (int y = 0; y < 2; ++y) T[z][y] = U[z][y] = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int o = col * STRIDE + kq + 4 * s;
                const double ax = s_w[o];
                const double adx = FORCE ? s_dw[o] : 0.0;
#pragma unroll
                for (int z = 0; z < 2; ++z)
#pragma unroll
                    for (int y = 0; y < 2; ++y) {
                        T[z][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ax, f[z][y][s], T[z][y],
                                                                       0, 0, 0);
                        if (FORCE)
                            U[z][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(adx, f[z][y][s],
                                                                           U[z][y], 0, 0, 0);
                    }
            }
            // T register r: atom kq + 4 r of the group, column col
            double out[NC][4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = (kq + 4 * r) * STRIDE;
                const int iy0 = row + 16 + (col & 3), iy1 = iy0 + 4;
                const int iz0 = row + 24 + (col >> 2), iz1 = iz0 + 4;
                const double y0 = s_w[iy0], y1 = s_w[iy1], z0 = s_w[iz0], z1 = s_w[iz1];
                const double t0 = fma(T[0][1][r], y1, T[0][0][r] * y0);
                const double t1 = fma(T[1][1][r], y1, T[1][0][r] * y0);
                if constexpr (!FORCE) {
                    out[0][r] = fma(t1, z1, t0 * z0);
                } else {
                    const double dy0 = s_dw[iy0], dy1 = s_dw[iy1];
                    const double dz0 = s_dw[iz0], dz1 = s_dw[iz1];
                    const double u0 = fma(U[0][1][r], y1, U[0][0][r] * y0);
                    const double u1 = fma(U[1][1][r], y1, U[1][0][r] * y0);
                    const double v0 = fma(T[0][1][r], dy1, T[0][0][r] * dy0);
                    const double v1 = fma(T[1][1][r], dy1, T[1][0][r] * dy0);
                    out[0][r] = fma(u1, z1, u0 * z0);
                    out[1][r] = fma(v1, z1, v0 * z0);
                    out[2][r] = fma(t1, dz1, t0 * dz0);
                }
            }
            __syncthreads();   // the staged values have been read: their place is red's now
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    red[c * 272 + (kq + 4 * r) * 17 + col] = out[c][r];
            __syncthreads();
            if (lane < 16 * NC) {
                double s = 0.0;
#pragma unroll
                for (int j = 0; j < 16; ++j) s += red[lane * 17 + j];
                const int b = 16 * t + (lane & 15);
                if (s_bin[b] >= 0)
                    part[((size_t)s_at[b].w * SLOTS + s_bin[b]) * NC + (lane >> 4)] = s;
            }
            __syncthreads();
        }
    }
}

// Per atom: the sum over its 18 tiles, and what it is for.  chi_i -= Phi;
// F_i = -q_i s_i grad Phi, with grad Phi = -sum_d n_d (d-th sum) f_d, and
// the reciprocal "stress" of absolute positions (block partials).
template <bool FORCE>
__global__ __launch_bounds__(MB) void k_mesh_finish(int n, MeshGeo g,
                                                    const int4 *__restrict__ at,
                                                    const double *__restrict__ part,
                                                    const double4 *__restrict__ pos,
                                                    const double *__restrict__ q,
                                                    const double *__restrict__ sc,
                                                    double4 *__restrict__ frc,
                                                    double *__restrict__ chi,
                                                    double *__restrict__ bpart)
{
    __shared__ double red[MB][6];
    const int a = blockIdx.x * MB + threadIdx.x;
    double w[6] = {0, 0, 0, 0, 0, 0};
    if (a < n) {
        const int i = at[a].w;
        if (!FORCE) {
            double s = 0.0;
            for (int t = 0; t < SLOTS; ++t) s += part[(size_t)a * SLOTS + t];
            chi[i] -= s;
        } else {
            double s[3] = {0, 0, 0};
            for (int t = 0; t < SLOTS; ++t)
                for (int d = 0; d < 3; ++d) s[d] += part[((size_t)a * SLOTS + t) * 3 + d];
            const double qs = q[i] * sc[i];
            for (int d = 0; d < 3; ++d) s[d] *= qs * g.n[d];
            const double fx = s[0] * g.f[0] + s[1] * g.f[3] + s[2] * g.f[6];
            const double fy = s[0] * g.f[1] + s[1] * g.f[4] + s[2] * g.f[7];
            const double fz = s[0] * g.f[2] + s[1] * g.f[5] + s[2] * g.f[8];
            const double4 f = frc[i], r = pos[i];
            frc[i] = make_double4(f.x + fx, f.y + fy, f.z + fz, 0.0);
            w[0] = r.x * fx; w[1] = r.y * fy; w[2] = r.z * fz;
            w[3] = r.y * fz; w[4] = r.x * fz; w[5] = r.x * fy;
        }
    }
    if (!FORCE) return;
    for (int c = 0; c < 6; ++c) red[threadIdx.x][c] = w[c];
    __syncthreads();
    for (int s = MB / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int c = 0; c < 6; ++c) red[threadIdx.x][c] += red[threadIdx.x + s][c];
        __syncthreads();
    }
    if (threadIdx.x < 6) bpart[(size_t)blockIdx.x * 8 + threadIdx.x] = red[0][threadIdx.x];
}

// The most ions that one tile meets (those of its 18 bins), into peak.
__global__ __launch_bounds__(MB) void k_mesh_crowd(MeshGeo g, int nbins,
                                                   const int *__restrict__ count,
                                                   int *__restrict__ peak)
{
    const int t = blockIdx.x * MB + threadIdx.x;
    int sum = 0;
    if (t < nbins) {
        const int tx = t % g.nb[0], ty = t / g.nb[0] % g.nb[1], tz = t / (g.nb[0] * g.nb[1]);
        for (int s = 0; s < SLOTS; ++s) sum += count[stream_bin(g, tx, ty, tz, s)];
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) sum = max(sum, __shfl_xor(sum, d));
    if ((threadIdx.x & 63) == 0) atomicMax(peak, sum);
}

__global__ void k_mesh_zero(int m, int *__restrict__ a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < m) a[t] = 0;
}

// ---- host side ----------------------------------------------------------------

int round_up(int x, int m) { return (x + m - 1) / m * m; }

// What the sum has decayed to at the band edge of axis d.
double band_decay(const CellGeom &c, const EwaldParams &P, int d)
{
    const double *v = c.v + 3 * d;
    const double len = std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    const double k = std::min(P.kc, 8.0 * std::atan(1.0) * P.K[d] / len);
    return std::exp(-0.5 * P.sigma * P.sigma * k * k);
}

// Mesh points of axis d: 4 K + 4, where aliasing leaves 3e-10 of a term at the
// band edge (2e-17 at half of it), if the sum has decayed to 3e-6 there, else
// 4.5 K + 4, where it leaves 6e-12.
int mesh_points(const CellGeom &c, const EwaldParams &P, int d)
{
    const int least[3] = {2 * TX, 3 * TY, 3 * TZ}, tile[3] = {TX, TY, TZ};
    const int K = P.K[d], n = band_decay(c, P, d) <= 3e-6 ? 4 * K + 4 : (9 * K + 1) / 2 + 4;
    return round_up(std::max(n, least[d]), tile[d]);
}

// ints that k_mesh_scan reads for nbins counts: whole int4 for 1024 threads
int scan_room(int nbins) { return round_up(nbins, 4096); }

// Gauss-Legendre rule over half the kernel's support in extended precision,
// the kernel included in the weights.
struct KernelRule {
    static constexpr int Q = 96;
    static_assert(Q % 2 == 0, "an even rule");
    long double x[Q / 2], v[Q / 2];
    KernelRule()
    {
        const long double pi = 4.0L * std::atan(1.0L);
        for (int j = 0; j < Q / 2; ++j) {
            long double z = std::cos(pi * (j + 0.75L) / (Q + 0.5L)), dp = 1.0L;
            for (int it = 0; it < 60; ++it) {
                long double p0 = 1.0L, p1 = z;
                for (int m = 2; m <= Q; ++m) {
                    const long double p2 = ((2 * m - 1) * z * p1 - (m - 1) * p0) / m;
                    p0 = p1;
                    p1 = p2;
                }
                dp = Q * (z * p1 - p0) / (z * z - 1.0L);
                const long double step = p1 / dp;
                z -= step;
                if (std::fabs(step) < 1e-19L) break;
            }
            const long double s = std::sqrt(1.0L - z * z);
            x[j] = z * (W / 2);
            // both mirror points: twice the half rule's weight times the kernel
            v[j] = 2.0L * (W / 2) * 2.0L / ((1.0L - z * z) * dp * dp) *
                   std::exp((long double)BETA * (s - 1.0L));
        }
    }
};

// Fourier transform of the kernel at frequencies k / n, k = 0 .. K (the kernel
// is analytic inside its support and e^-beta at its ends).
std::vector<double> kernel_transform(int K, int n)
{
    static const KernelRule rule;   // depends on nothing: formed once, 0.15 ms
    const long double pi = 4.0L * std::atan(1.0L);
    std::vector<double> out(K + 1);
    for (int k = 0; k <= K; ++k) {
        long double s = 0.0L;
        for (int j = 0; j < KernelRule::Q / 2; ++j)
            s += rule.v[j] * std::cos(2.0L * pi * k * rule.x[j] / n);
        out[k] = (double)s;
    }
    return out;
}

// Operand tables of one axis in the order the waves load them: tile m, step
// t, lane L.  Forward: row k = 16 m + L % 16, point g = 4 t + L / 16 (the
// self-mirrored points halved, zero past n / 2); inverse: row g, index k.
// Cosines first, then sines.
std::vector<double> axis_table(int K, int n, bool forward, int *mtiles, int *steps)
{
    const long double pi = 4.0L * std::atan(1.0L);
    std::vector<long double> cs(n), sn(n);
    for (int j = 0; j < n; ++j) {
        cs[j] = std::cos(2.0L * pi * j / n);
        sn[j] = std::sin(2.0L * pi * j / n);
    }
    const int half = n / 2, rows = forward ? K + 1 : half + 1, len = forward ? half + 1 : K + 1;
    *mtiles = (rows + 15) / 16;
    *steps = (len + 3) / 4;
    std::vector<double> tab((size_t)2 * *mtiles * *steps * 64, 0.0);
    for (int m = 0; m < *mtiles; ++m)
        for (int t = 0; t < *steps; ++t)
            for (int L = 0; L < 64; ++L) {
                const int r = 16 * m + L % 16, e = 4 * t + L / 16;
                if (r >= rows || e >= len) continue;
                const int k = forward ? r : e, p = forward ? e : r;
                const int j = (int)((long)k * p % n);
                const bool self = p == 0 || p == half;
                const size_t at = ((size_t)m * *steps + t) * 64 + L;
                tab[at] = (double)(forward && self ? 0.5L * cs[j] : cs[j]);
                tab[at + (size_t)*mtiles * *steps * 64] = self ? 0.0 : (double)sn[j];
            }
    return tab;
}

MeshGeo geo_of(const MeshState &M, const double *f)
{
    MeshGeo g;
    for (int d = 0; d < 3; ++d) {
        g.n[d] = M.n[d];
        g.nb[d] = M.nb[d];
    }
    for (int c = 0; c < 9; ++c) g.f[c] = f[c];
    return g;
}

// Output tiles per wave: as many as fit (each loaded mesh value then serves
// all of them), fewer where the columns alone would leave the chip idle.
int tiles_per_wave(int mtiles, long waves)
{
    int passes = (mtiles + MT_MAX - 1) / MT_MAX;
    while (passes < mtiles && waves * passes < 2048) ++passes;
    return (mtiles + passes - 1) / passes;
}

template <class F1, class F2, class F3, class F4, class F5>
void by_tiles(int mt, F1 &&f1, F2 &&f2, F3 &&f3, F4 &&f4, F5 &&f5)
{
    switch (mt) {
    case 1: f1(); break;
    case 2: f2(); break;
    case 3: f3(); break;
    case 4: f4(); break;
    default: f5(); break;
    }
}

void transform(System &S, const MeshState &M, int axis, bool forward, int arrays, long outer,
               int inner, const double *in, double *out)
{
    const int n = M.n[axis], K = M.K[axis];
    const long cols = outer * inner, waves = (cols + 15) / 16;
    const int mtiles = forward ? M.fmt[axis] : M.imt[axis];
    const int steps = forward ? M.fst[axis] : M.ist[axis];
    const double *tab = M.tab.p + (forward ? M.fat[axis] : M.iat[axis]);
    const int mt = tiles_per_wave(mtiles, waves * arrays);
    const dim3 grid((unsigned)((waves + MB / 64 - 1) / (MB / 64)), (mtiles + mt - 1) / mt, arrays);
    const long full = cols * n, cut = cols * (K + 1);
    if (forward) {
        auto go = [&](auto kern) {
            kern<<<grid, MB, 0, S.stream>>>(n, K, inner, cols, steps, mtiles, tab, in, full, out,
                                            cut);
        };
        by_tiles(mt, [&] { go(k_dft_forward<1>); }, [&] { go(k_dft_forward<2>); },
                 [&] { go(k_dft_forward<3>); }, [&] { go(k_dft_forward<4>); },
                 [&] { go(k_dft_forward<5>); });
    } else {
        auto go = [&](auto kern) {
            kern<<<grid, MB, 0, S.stream>>>(n, K, inner, cols, steps, mtiles, tab, in, cut, out,
                                            full);
        };
        by_tiles(mt, [&] { go(k_dft_inverse<1>); }, [&] { go(k_dft_inverse<2>); },
                 [&] { go(k_dft_inverse<3>); }, [&] { go(k_dft_inverse<4>); },
                 [&] { go(k_dft_inverse<5>); });
    }
}

}  // namespace

// The choice is by cost, both sides' times (µs) of S(k) and one pass over the
// atoms as sums of what they grow with.  Fitted to 90 systems of 100 to 262,144
// ions and K = 6 to 74 in cubes, slabs and rods: within 20% of most of what was
// measured, within 30% of all.
//   direct: launches, k-vectors, pairs, ions (phases);
//   mesh:   launches, points (the transforms), and the ions: a tile is one
//           wave's, so the longest chain of a tile or, with tiles for the whole
//           chip, all ions.
// Measured, direct and mesh: 262,144 ions, K = 20: 3755 and 2022 µs; K = 14
// (18,400 ions a tile): 1771 and 4876; 64,000 in an eighth of a cell, K = 14:
// 484 and 7552; in a cell of 304^3 points 500 ions 425 and 675, 2,000 904 and
// 715.  Below MESH_MIN_PAIRS neither is ahead by more than a launch or two.
bool mesh_suits(System &S, const EwaldParams &P, MeshState &M, const double *f, double volume)
{
    // k-vectors of the half space: half a sphere's worth, at most the box
    const double pi = 4.0 * std::atan(1.0), n = S.n;
    const int tile[3] = {TX, TY, TZ};
    MeshGeo g;
    double box = 1.0, points = 1.0, decay = 0.0;
    for (int d = 0; d < 3; ++d) {
        g.n[d] = mesh_points(S.geom, P, d);
        g.nb[d] = g.n[d] / tile[d];
        box *= d == 2 ? P.K[d] + 1 : 2 * P.K[d] + 1;
        points *= g.n[d];
        decay = std::max(decay, band_decay(S.geom, P, d));
    }
    for (int c = 0; c < 9; ++c) g.f[c] = f[c];
    const double nk = std::min(box, volume * P.kc * P.kc * P.kc / (12.0 * pi * pi));
    // (what has not decayed at the band edge would need a finer mesh yet)
    if (decay > 1e-4 || !(n * nk >= MESH_MIN_PAIRS) || points > 268435456.0) return false;
    const double direct = 75.0 + 2e-4 * nk + 4.2e-7 * n * nk + 5e-3 * n;
    auto mesh = [&](double met) {   // ions that the most crowded tile meets
        return 60.0 + 2e-5 * points + std::max(0.25 * met, 3.3e-3 * n);
    };
    const int nbins = g.nb[0] * g.nb[1] * g.nb[2];
    if (mesh(SLOTS * n / nbins) >= direct) return false;
    // where the ions are decides, counted once for each plan
    M.bin.ensure(S.n);
    M.count.ensure(scan_room(nbins));
    M.start.ensure(scan_room(nbins) + 1);
    k_mesh_zero<<<div_up(nbins, 256), 256, 0, S.stream>>>(nbins, M.count.p);
    k_mesh_zero<<<1, 64, 0, S.stream>>>(1, M.start.p);
    k_mesh_bin<<<div_up(S.n, MB), MB, 0, S.stream>>>(S.n, g, S.pos.p, M.bin.p, M.count.p);
    k_mesh_crowd<<<div_up(nbins, MB), MB, 0, S.stream>>>(g, nbins, M.count.p, M.start.p);
    HIP_TRY(hipGetLastError());
    int met = 0;
    HIP_TRY(hipMemcpyAsync(&met, M.start.p, sizeof(int), hipMemcpyDeviceToHost, S.stream));
    HIP_TRY(hipStreamSynchronize(S.stream));
    return mesh(met) < direct;
}

// The operand tables and kernel transforms of M.n and M.K, in one upload: equal
// axes share them.  0.4 ms for a cube of K = 22, 3 ms for three axes of K = 74.
static void mesh_tables(System &S, MeshState &M)
{
    std::vector<double> tab, dec;
    auto put = [&](const std::vector<double> &v) {
        const size_t at = tab.size();
        tab.insert(tab.end(), v.begin(), v.end());
        return at;
    };
    size_t dec_at[3];
    for (int d = 0; d < 3; ++d) {
        int e = 0;
        while (M.n[e] != M.n[d] || M.K[e] != M.K[d]) ++e;
        if (e == d) {
            M.fat[d] = put(axis_table(M.K[d], M.n[d], true, &M.fmt[d], &M.fst[d]));
            M.iat[d] = put(axis_table(M.K[d], M.n[d], false, &M.imt[d], &M.ist[d]));
            dec_at[d] = dec.size();
            for (double v : kernel_transform(M.K[d], M.n[d])) dec.push_back(1.0 / v);
        } else {
            M.fat[d] = M.fat[e];
            M.iat[d] = M.iat[e];
            M.fmt[d] = M.fmt[e];
            M.fst[d] = M.fst[e];
            M.imt[d] = M.imt[e];
            M.ist[d] = M.ist[e];
            dec_at[d] = dec.size();
            for (int k = 0; k <= M.K[d]; ++k) dec.push_back(dec[dec_at[e] + k]);
        }
    }
    M.dat = put(dec);
    M.tab.ensure(tab.size());
    HIP_TRY(hipMemcpyAsync(M.tab.p, tab.data(), sizeof(double) * tab.size(),
                           hipMemcpyHostToDevice, S.stream));
    HIP_TRY(hipStreamSynchronize(S.stream));   // before the host vector goes
}

void mesh_plan(System &S, const EwaldParams &P, MeshState &M, const double *b, double inv_eps_2v)
{
    const int tile[3] = {TX, TY, TZ};
    // A new cell with the same k-vector counts (each step of a relaxation of
    // the cell) keeps the tables and runs k_mesh_coef alone.  Energy and forces
    // in a new cell, 8,000 ions: 1.44 ms with the tables formed again, 0.55 so
    // (1.24 by the direct sums before; in the same cell 0.45).
    bool same = M.tables;
    M.tables = false;
    for (int d = 0; d < 3; ++d) {
        const int n = mesh_points(S.geom, P, d);
        same = same && M.K[d] == P.K[d] && M.n[d] == n;
        M.K[d] = P.K[d];
        M.n[d] = n;
        M.nb[d] = n / tile[d];
    }
    if (!same) mesh_tables(S, M);
    const long oct = (long)(M.K[0] + 1) * (M.K[1] + 1) * (M.K[2] + 1);
    const long n0 = M.n[0], n1 = M.n[1], n2 = M.n[2];
    M.nbins = M.nb[0] * M.nb[1] * M.nb[2];
    M.coef.ensure(4 * oct);
    // the two work arrays of the transforms: the mesh and the half-cut mesh,
    // then the twice-cut mesh and the octant
    M.bufa.ensure(std::max(n0 * n1 * n2, 4 * n0 * (M.K[1] + 1) * (M.K[2] + 1)));
    M.bufb.ensure(2 * n0 * n1 * (M.K[2] + 1));
    M.oct.ensure(8 * oct);
    const int room = scan_room(M.nbins);
    M.count.ensure(room);
    M.fill.ensure(room);
    M.start.ensure(room + 1);
    k_mesh_zero<<<div_up(room, 256), 256, 0, S.stream>>>(room, M.count.p);
    k_mesh_coef<<<div_up((int)oct, MB), MB, 0, S.stream>>>(
        M.K[0], M.K[1], M.K[2], make_double4(b[0], b[1], b[2], 0), make_double4(b[3], b[4], b[5], 0),
        make_double4(b[6], b[7], b[8], 0), P.kc * P.kc, inv_eps_2v, 0.5 * P.sigma * P.sigma,
        M.coef.p);
    HIP_TRY(hipGetLastError());
    M.tables = true;
}

void mesh_place(System &S, MeshState &M, const double *f)
{
    const int n = S.n;
    M.bin.ensure(n);
    M.claim.ensure(n);
    M.order.ensure(n);
    M.at.ensure(n);
    M.w.ensure((size_t)n * 48);
    const MeshGeo g = geo_of(M, f);
    k_mesh_bin<<<div_up(n, MB), MB, 0, S.stream>>>(n, g, S.pos.p, M.bin.p, M.count.p);
    k_mesh_scan<<<1, 1024, 0, S.stream>>>(M.nbins, scan_room(M.nbins) / 4096, (int4 *)M.count.p,
                                          (int4 *)M.fill.p, (int4 *)M.start.p, M.start.p);
    k_mesh_fill<<<div_up(n, MB), MB, 0, S.stream>>>(n, M.bin.p, M.start.p, M.fill.p, M.claim.p);
    k_mesh_order<<<M.nbins, 64, 0, S.stream>>>(M.start.p, M.claim.p, M.order.p);
    const unsigned blocks = (unsigned)(((long)n * 48 + MB - 1) / MB);
    k_mesh_weights<false><<<blocks, MB, 0, S.stream>>>(n, g, S.pos.p, M.order.p, M.w.p, M.at.p);
    HIP_TRY(hipGetLastError());
}

void mesh_structure(System &S, MeshState &M, const double *f, const double *scaler)
{
    const MeshGeo g = geo_of(M, f);
    k_mesh_spread<<<M.nbins, 64, 0, S.stream>>>(g, M.start.p, M.at.p, M.w.p, S.q.p, scaler,
                                                M.bufa.p);
    // mesh[z][y][x] -> [k3][y][x] -> [k3][k2][x] -> [k3][k2][k1]
    transform(S, M, 2, true, 1, 1, M.n[0] * M.n[1], M.bufa.p, M.bufb.p);
    transform(S, M, 1, true, 2, M.K[2] + 1, M.n[0], M.bufb.p, M.bufa.p);
    transform(S, M, 0, true, 4, (long)(M.K[2] + 1) * (M.K[1] + 1), 1, M.bufa.p, M.oct.p);
    const long oct = (long)(M.K[0] + 1) * (M.K[1] + 1) * (M.K[2] + 1);
    M.nepart = (int)((oct + MB - 1) / MB);
    M.epart.ensure(M.nepart);
    k_mesh_combine<<<M.nepart, MB, 0, S.stream>>>(M.K[0], M.K[1], M.K[2], M.tab.p + M.dat,
                                                  M.coef.p,
                                                  M.oct.p, M.epart.p);
    HIP_TRY(hipGetLastError());
}

void mesh_atoms(System &S, MeshState &M, const double *f, const double *scaler, bool force,
                double *chi, double *bpart)
{
    const int n = S.n;
    const MeshGeo g = geo_of(M, f);
    M.part.ensure((size_t)n * SLOTS * (force ? 3 : 1));
    if (force) {
        M.dw.ensure((size_t)n * 48);
        const unsigned blocks = (unsigned)(((long)n * 48 + MB - 1) / MB);
        k_mesh_weights<true><<<blocks, MB, 0, S.stream>>>(n, g, S.pos.p, M.order.p, M.dw.p,
                                                          nullptr);
    }
    transform(S, M, 0, false, 4, (long)(M.K[2] + 1) * (M.K[1] + 1), 1, M.oct.p, M.bufa.p);
    transform(S, M, 1, false, 2, M.K[2] + 1, M.n[0], M.bufa.p, M.bufb.p);
    transform(S, M, 2, false, 1, 1, M.n[0] * M.n[1], M.bufb.p, M.bufa.p);
    const int nb = div_up(n, MB);
    if (force) {
        k_mesh_field<true><<<M.nbins, 64, 0, S.stream>>>(g, M.start.p, M.at.p, M.w.p, M.dw.p,
                                                         M.bufa.p, M.part.p);
        k_mesh_finish<true><<<nb, MB, 0, S.stream>>>(n, g, M.at.p, M.part.p, S.pos.p, S.q.p,
                                                     scaler, S.frc.p, nullptr, bpart);
    } else {
        k_mesh_field<false><<<M.nbins, 64, 0, S.stream>>>(g, M.start.p, M.at.p, M.w.p, nullptr,
                                                          M.bufa.p, M.part.p);
        k_mesh_finish<false><<<nb, MB, 0, S.stream>>>(n, g, M.at.p, M.part.p, S.pos.p, S.q.p,
                                                      scaler, nullptr, chi, nullptr);
    }
    HIP_TRY(hipGetLastError());
}

void mesh_release(MeshState &M)
{
    M.tables = false;
    M.tab.release();
    M.coef.release();
    M.bufa.release();
    M.bufb.release();
    M.oct.release();
    M.count.release();
    M.fill.release();
    M.start.release();
    M.bin.release();
    M.claim.release();
    M.order.release();
    M.at.release();
    M.w.release();
    M.dw.release();
    M.part.release();
    M.epart.release();
}
