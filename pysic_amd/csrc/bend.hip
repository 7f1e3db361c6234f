// bend.hip -- COMB's bond-bending angle term (bond_bend).
//
// The reference finds angles while it walks the pairs (Core.f90:3567-3610,
// 3760-3800): for each pair (atom1, atom2) taken once by pick, first the
// triplets (atom2, atom1, atom3) over atom1's neighbors with
// pick(atom2, atom3), then (atom1, atom2, atom3) over atom2's neighbors with
// pick(atom1, atom3); each is evaluated by the many-body potentials whose
// targets match the atoms in that order (core_evaluate_local_triplet_B,
// Core.f90:6656-7028).  So every angle a-v-b at a vertex v is visited once,
// oriented so that pick(a, b) holds: from the pair (v, a) with v as atom 1
// when pick(v, a) holds (targets matched as (v, a, b)), else from (a, v)
// (targets matched as (a, v, b)).
//
// Here each vertex v gets a short list of the neighbors that can take part
// in an angle at it, or it at them, then G lanes: each lane takes some of the legs and, for each,
// every angle it forms with another leg, oriented and matched against the
// rows as the reference does it.  The force on a leg's atom is stored per
// short-list slot and summed by that atom's own thread afterwards, with the
// vertex's own (minus the sum over its slots): no atomics, fixed order,
// bit-for-bit repeatable.  All arithmetic is FP64.
#include "system.h"

namespace {

constexpr int BB = 256;

// x^n for an integer n by repeated products (Fortran's real**integer)
__device__ __forceinline__ double bend_ipow(double x, int n)
{
    const int m = n < 0 ? -n : n;
    double y = 1.0;
    for (int k = 0; k < m; ++k) y = y * x;
    return n < 0 ? 1.0 / y : y;
}

// One neighbor of the vertex: index, image, species, original index,
// r_j - r_v and its length.
struct Leg {
    int j, img, s, id;
    double3 d;
    double r;
};

__device__ __forceinline__ Leg load_leg(const double4 &pv, int j, int img,
                                        const double4 *__restrict__ pos,
                                        const int *__restrict__ id, const double *cv)
{
    Leg L;
    const double4 pj = pos[j];
    L.j = j;
    L.img = img;
    L.s = (int)pj.w;
    L.id = id[j];
    L.d = separation64(pv, pj, img, cv);
    L.r = sqrt(dot64(L.d));
    return L;
}

// The angle a-v-b of one row (evaluate_energy_bond_bending and
// evaluate_force_bond_bending, Potentials.f90:3196-3328) seen from leg a, with
// da = r_a - r_v and db = r_b - r_v: E = eps (cos^n - c0)^m times both legs'
// f_c and, with FORCE, the force on a, t.  The same for either leg in the
// first place: the angle and its smoothing are symmetric in them.
template <bool FORCE>
__device__ __forceinline__ double bend_term(const BendTerm &P, const double3 &da, double ra,
                                            const double3 &db, double rb, double3 &t)
{
    const double ira = recip64(ra), ratio = ira * recip64(rb);
    const double r3 = da.x * db.x + da.y * db.y + da.z * db.z;
    const double cosine = r3 * ratio;
    double fa = 1.0, dfa = 0.0, fb = 1.0, dfb = 0.0;
    if (P.smooth) {
        smooth64(ra, P.cut, P.soft, &fa, &dfa);
        smooth64(rb, P.cut, P.soft, &fb, &dfb);
    }
    const double e = P.eps * bend_ipow(bend_ipow(cosine, P.n) - P.c0, P.m);
    if (FORCE) {
        const double cospower = bend_ipow(cosine, P.n - 1);
        const double xm = bend_ipow(cospower * cosine - P.c0, P.m - 1);
        // dE/dcos f_c f_c along -(d cos / d r_a), and f_c's own slope
        const double k = ira * ira * r3;
        const double c = ratio * P.eps * (double)(P.m * P.n) * xm * cospower * fa * fb;
        const double s = dfa * ira * fb * e;
        t = make_double3(-c * (db.x - k * da.x) - s * da.x, -c * (db.y - k * da.y) - s * da.y,
                         -c * (db.z - k * da.z) - s * da.z);
    }
    return e * fa * fb;
}

// The short list of each vertex: its neighbors that are a leg of some row's
// angle at the vertex, or it of theirs (species and cutoff, bend_leg2: the
// same answer seen from either end, so a pair is in both atoms' lists).
// Silica within 3.05 A: 3 legs an atom instead of 8 neighbors.
template <class Geo>
__global__ __launch_bounds__(BB) void k_bend_list(int n, Geo geo, const double4 *__restrict__ pos,
                                                  const int *__restrict__ nbr,
                                                  const int *__restrict__ nimg,
                                                  const int *__restrict__ ncnt,
                                                  const PairModel *__restrict__ PM,
                                                  int *__restrict__ bsj, int *__restrict__ bsimg,
                                                  int *__restrict__ bscnt)
{
    const int v = xcd_block(gridDim.x) * BB + threadIdx.x;
    if (v >= n) return;
    const double4 pv = pos[v];
    const double *cv = geo.vec(v);
    const size_t N = (size_t)n;
    const double *leg2 = PM->bend_leg2[(int)pv.w];
    const int nf = ncnt[v];
    int c = 0;
    constexpr int U = 8;   // entries in flight
    for (int t0 = 0; t0 < nf; t0 += U) {
        int jv[U], iv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t at = (size_t)min(t0 + u, nf - 1) * N + v;
            jv[u] = nbr[at];
            iv[u] = nimg[at];
        }
        double4 p[U];
#pragma unroll
        for (int u = 0; u < U; ++u) p[u] = pos[jv[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (t0 + u >= nf) break;
            if (!(dot64(separation64(pv, p[u], iv[u], cv)) < leg2[(int)p[u].w])) continue;
            bsj[(size_t)c * N + v] = jv[u];
            bsimg[(size_t)c * N + v] = iv[u];
            ++c;
        }
    }
    bscnt[v] = c;
}

// G lanes per vertex v; lane l takes the short-list legs ta = l, l + G, ...
// and every angle (ta, tb), tb != ta, so each angle is evaluated by the two
// lanes of its legs.  A lane keeps only its own leg's share: the force on
// that atom (stored per slot), half the energy, and d_ta (x) F_ta of the
// virial (the three forces of an angle sum to zero, so sum r (x) F over its
// atoms is d_a (x) F_a + d_b (x) F_b, taking r_v as the origin).
template <class Geo, int MODE, int G, int H>
__global__ __launch_bounds__(BB) void k_bend_angles(int n, Geo geo, const double4 *__restrict__ pos,
                                                    const int *__restrict__ id,
                                                    const PairModel *__restrict__ PM,
                                                    const int *__restrict__ bsj,
                                                    const int *__restrict__ bsimg,
                                                    const int *__restrict__ bscnt,
                                                    double4 *__restrict__ bG,
                                                    double *__restrict__ partial, int blk0)
{
    constexpr bool FORCE = MODE != PAIR_ENERGY;
    constexpr bool VIR = MODE == PAIR_FORCES;
    __shared__ double red[7][BB];
    __shared__ BendTerm rows[PYSIC_MAXB];
    {
        const int *src = reinterpret_cast<const int *>(&PM->bend[0]);
        int *dst = reinterpret_cast<int *>(&rows[0]);
        const int words = PM->nbend * (int)(sizeof(BendTerm) / sizeof(int));
        for (int w = threadIdx.x; w < words; w += BB) dst[w] = src[w];
    }
    __syncthreads();
    const int blk = xcd_block(gridDim.x);
    const int gid = blk * BB + threadIdx.x;
    // G * H consecutive lanes per vertex: lane l + G h takes the legs
    // l, l + G, ... and, of each, the partner legs h, h + H, ...
    const int v = gid / (G * H), lane = gid % G, part = (gid / G) % H;
    double e = 0.0, w0 = 0.0, w1 = 0.0, w2 = 0.0, w3 = 0.0, w4 = 0.0, w5 = 0.0;
    if (v < n) {
        const double4 pv = pos[v];
        const int sv = (int)pv.w, idv = id[v];
        const double *cv = geo.vec(v);
        const size_t N = (size_t)n;
        const double vmax = PM->bend_maxpot[sv];
        const int c = bscnt[v];
        const int nbend = PM->nbend;
        for (int ta = lane; ta < c; ta += G) {
            const Leg A = load_leg(pv, bsj[(size_t)ta * N + v], bsimg[(size_t)ta * N + v], pos, id,
                                   cv);
            double3 fa = make_double3(0.0, 0.0, 0.0);
            for (int tb = part; tb < c; tb += H) {
                if (tb == ta) continue;
                const Leg B = load_leg(pv, bsj[(size_t)tb * N + v], bsimg[(size_t)tb * N + v],
                                       pos, id, cv);
                // the reference's orientation: first leg with pick(first, last)
                const bool ab = pick_dev(A.id, B.id,
                                         pack_img(img_x(B.img) - img_x(A.img),
                                                  img_y(B.img) - img_y(A.img),
                                                  img_z(B.img) - img_z(A.img)));
                const Leg &Fl = ab ? A : B;
                const Leg &Ll = ab ? B : A;
                // from the pair (v, first) [v atom 1] or (first, v)
                const bool vfirst = pick_dev(idv, Fl.id, Fl.img);
                const int e0 = vfirst ? sv : Fl.s, e1 = vfirst ? Fl.s : sv;
                // the second leg is searched within atom 1's radius, which
                // for (first, v) is the vertex's own largest potential cutoff
                if (!vfirst && !(Ll.r < vmax)) continue;
                const double r1 = Fl.r, r2 = Ll.r;
                // the lanes look for their row first and evaluate it together:
                // a wave's vertices and orientations match different rows
                for (int k = 0;; ++k) {
                    while (k < nbend &&
                           (rows[k].e[0] != e0 || rows[k].e[1] != e1 || rows[k].e[2] != Ll.s ||
                            !(rows[k].cut > r1) || !(rows[k].cut > r2) || rows[k].vertex != sv))
                        ++k;
                    if (k >= nbend) break;
                    double3 t;
                    const double ev = bend_term<FORCE>(rows[k], A.d, A.r, B.d, B.r, t);
                    if (!FORCE) {
                        e += 0.5 * ev;
                        continue;
                    }
                    fa.x += t.x;
                    fa.y += t.y;
                    fa.z += t.z;
                    if (VIR) {
                        const double3 d = A.d;
                        w0 += d.x * t.x;
                        w1 += d.y * t.y;
                        w2 += d.z * t.z;
                        w3 += d.y * t.z;
                        w4 += d.x * t.z;
                        w5 += d.x * t.y;
                    }
                }
            }
            if (FORCE) {
                // the H parts of one leg run the same ta loop, so they are
                // active together here
#pragma unroll
                for (int o = G; o < G * H; o <<= 1) {
                    fa.x += __shfl_xor(fa.x, o);
                    fa.y += __shfl_xor(fa.y, o);
                    fa.z += __shfl_xor(fa.z, o);
                }
                if (part == 0) bG[(size_t)ta * N + v] = make_double4(fa.x, fa.y, fa.z, 0.0);
            }
        }
    }
    if (MODE == PAIR_FORCES_ONLY) return;
    const int tid = threadIdx.x;
    red[0][tid] = e;
    red[1][tid] = w0; red[2][tid] = w1; red[3][tid] = w2;
    red[4][tid] = w3; red[5][tid] = w4; red[6][tid] = w5;
    __syncthreads();
    for (int s = BB / 2; s > 0; s >>= 1) {
        if (tid < s)
            for (int q = 0; q < 7; ++q) red[q][tid] += red[q][tid + s];
        __syncthreads();
    }
    if (tid < 7) partial[(size_t)(blk0 + blk) * 8 + tid] = red[tid][0];
}

// F_a += -(the forces of a's own angles on their outer atoms) + the forces
// a's short-list neighbors' angles put on a (found in each neighbor's short
// list at (a, -o)).  G lanes per atom split a's slots; shuffles sum them.
template <int G>
__global__ __launch_bounds__(BB) void k_bend_gather(int n, const int *__restrict__ bsj,
                                                    const int *__restrict__ bsimg,
                                                    const int *__restrict__ bscnt,
                                                    const double4 *__restrict__ bG,
                                                    double4 *__restrict__ frc,
                                                    double4 *__restrict__ mom, double half_dt,
                                                    int kick)
{
    const int gid = xcd_block(gridDim.x) * BB + threadIdx.x;
    const int a = gid / G, lane = gid % G;
    const size_t N = (size_t)n;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if (a < n) {
        const int c = bscnt[a];
        for (int t = lane; t < c; t += G) {
            const double4 own = bG[(size_t)t * N + a];
            fx -= own.x;
            fy -= own.y;
            fz -= own.z;
            const int v = bsj[(size_t)t * N + a];
            const int want = neg_img(bsimg[(size_t)t * N + a]);
            const int cv = bscnt[v];
            for (int u = 0; u < cv; ++u) {
                if (bsj[(size_t)u * N + v] == a && bsimg[(size_t)u * N + v] == want) {
                    const double4 g = bG[(size_t)u * N + v];
                    fx += g.x;
                    fy += g.y;
                    fz += g.z;
                    break;
                }
            }
        }
    }
    // the lanes of one atom are consecutive threads of one wave; every
    // thread reaches the shuffles
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        fx += __shfl_xor(fx, o);
        fy += __shfl_xor(fy, o);
        fz += __shfl_xor(fz, o);
    }
    if (a >= n || lane != 0) return;
    double4 f = frc[a];
    f.x += fx;
    f.y += fy;
    f.z += fz;
    frc[a] = f;
    if (kick) {
        double4 p = mom[a];
        p.x += half_dt * f.x;
        p.y += half_dt * f.y;
        p.z += half_dt * f.z;
        mom[a] = p;
    }
}

}  // namespace

// lanes per vertex: the two to four legs of an oxide's vertex, one or two a
// lane, and each leg's partners over BG_PARTS lanes.  24,576 atoms of COMB
// silica, the angle kernel alone: 80 us with all neighbors within 3.05 A in
// the lists (16 x 2 lanes) and each lane evaluating its rows as it met them,
// 57 with the legs alone, 44 with the rows found first and evaluated together
// (with the other two chains beside it 55; 8 x 4 lanes 47, 8 x 2 65, 4 x 2 80,
// 2 x 4 87, and the same step time within 2% for all of them).
constexpr int BG_LANES = 4;
constexpr int BG_PARTS = 4;
// lanes per atom in the gather: its slots split over 8 lanes
constexpr int BG_GATHER_LANES = 8;

int bend_blocks(const System &S)
{
    return S.pmodel.nbend > 0 ? div_up(S.n * BG_LANES * BG_PARTS, BB) : 0;
}

void bend_room(System &S)
{
    const size_t cap = (size_t)S.cap * S.n;
    S.bsj.ensure(cap);
    S.bsimg.ensure(cap);
    S.bscnt.ensure(S.n);
    S.bG.ensure(cap);
}

// up to the gather: short lists, each vertex's angles, their partials
void bend_sites(System &S, int mode, int blk0, hipStream_t stream)
{
    const int n = S.n, nb = div_up(n, BB), na = bend_blocks(S);
    bend_room(S);
    with_geo(S, [&](auto geo) {
        using Geo = decltype(geo);
        k_bend_list<Geo><<<nb, BB, 0, stream>>>(n, geo, S.pos.p, S.nbr.p, S.nimg.p, S.ncnt.p,
                                                S.dpmodel.p, S.bsj.p, S.bsimg.p, S.bscnt.p);
        auto go = [&](auto kern) {
            kern<<<na, BB, 0, stream>>>(n, geo, S.pos.p, S.id.p, S.dpmodel.p, S.bsj.p, S.bsimg.p,
                                        S.bscnt.p, S.bG.p, S.gpartial.p, blk0);
        };
        if (mode == PAIR_ENERGY) go(k_bend_angles<Geo, PAIR_ENERGY, BG_LANES, BG_PARTS>);
        else if (mode == PAIR_FORCES) go(k_bend_angles<Geo, PAIR_FORCES, BG_LANES, BG_PARTS>);
        else go(k_bend_angles<Geo, PAIR_FORCES_ONLY, BG_LANES, BG_PARTS>);
    });
    HIP_TRY(hipGetLastError());
}

void bend_gather(System &S, int mode, double half_dt, int kick)
{
    if (mode == PAIR_ENERGY) return;
    k_bend_gather<BG_GATHER_LANES><<<div_up(S.n * BG_GATHER_LANES, BB), BB, 0, S.stream>>>(
        S.n, S.bsj.p, S.bsimg.p, S.bscnt.p, S.bG.p, S.frc.p, S.mom.p, half_dt, kick);
    HIP_TRY(hipGetLastError());
}

void bend_eval(System &S, int mode, int blk0, double half_dt, int kick)
{
    if (S.pmodel.nbend == 0) return;
    hipEvent_t ev{};
    S.timer.begin("bend", S.stream, &ev);
    bend_sites(S, mode, blk0, S.stream);
    bend_gather(S, mode, half_dt, kick);
    S.timer.end("bend", S.stream, ev);
}
