// ewald.h -- Ewald summation and electronegativity equalization on device.
#pragma once

#include "system.h"

#include <vector>

struct EwaldParams {
    int on = 0;
    double rc = 0, kc = 0, sigma = 0, eps = 0;
    int K[3] = {0, 0, 0};
    int has_scaler = 0;
    std::vector<double> scaler;  // original order
};

// Reciprocal sums over a mesh (mesh.hip): the plan of one k-vector set and
// the atoms' places on it.
struct MeshState {
    int n[3] = {0, 0, 0}, K[3] = {0, 0, 0}, nb[3] = {0, 0, 0}, nbins = 0, nepart = 0;
    int fmt[3], fst[3], imt[3], ist[3];   // tiles and steps of the transforms, per axis
    bool tables = false;                  // tab is that of n and K
    DBuf<double> tab;                     // operand tables, reciprocal kernel transforms
    size_t fat[3], iat[3], dat;           // where in tab: forward, inverse, transforms
    DBuf<double> coef;                    // k-vector coefficients
    DBuf<double> bufa, bufb, oct;         // mesh, half-transformed mesh, octant
    DBuf<int> count, fill, start, bin, claim, order;
    DBuf<int4> at;                        // window origin and slot, tile order
    DBuf<double> w, dw;                   // kernel values and derivatives, 48 per atom
    DBuf<double> part, epart;             // per-tile atom sums, energy partials
};

struct EwaldState {
    bool dirty = true;
    bool mesh_on = false;   // the k-vectors' sums go over the mesh
    int planned_n = 0;      // atom count the choice was made for
    MeshState mesh;
    int nk = 0;
    DBuf<double4> kvec;     // kx, ky, kz, coefficient c_k
    DBuf<double2> sk;       // sum q s cos(k.r), sum q s sin(k.r)
    DBuf<double> scaler;    // current (sorted) order
    int ones = 0;           // scaler holds this many ones (0: something else)
    DBuf<double> scaler0;   // the caller's scalers, original order
    DBuf<double> chi;       // electronegativities (sorted order)
    DBuf<double> part;      // block partials
    DBuf<double> red;       // reduced scalars
    DBuf<double2> skpart;   // structure-factor partials over atom chunks
    DBuf<double4> rpart;    // per-atom reciprocal partials over k chunks
    DBuf<double4> th;       // per-atom fractional coordinates and q s
    DBuf<double2> pw;       // per-atom q s exp(2 pi i l u3), 16 per atom
    DBuf<double2> wl;       // per-atom exp(2 pi i 16 u3)
    DBuf<double4> zw;       // coefficients of the per-atom sums (plan order)
    DBuf<int> kpk;          // packed (k1, k2, l0) per plan slot
    DBuf<double> dchi, mx;  // relaxation: differences, their block maxima
    DBuf<int> stop;         // relaxation of a small system: it has ended
    hipEvent_t seen[2] = {nullptr, nullptr};   // its last two evaluations' errors are out
    DBuf<unsigned long long> hpart;   // state fingerprint partials
    // sk and th hold the structure factors of the state whose fingerprint
    // is sk_hash
    bool sk_valid = false;
    unsigned long long sk_hash = 0;
    // k-vector segments: runs of at most 16 consecutive k3 at fixed (k1, k2),
    // {k1, k2, k3_start | len << 16, index of the first k}, natural order;
    // the structure-factor kernel's work plan over them (16 x 4 segments
    // per wave) and its continuation flags
    DBuf<int4> seg;
    DBuf<int> plan, pflags;
    int nseg = 0, nwaves = 0;
    double b[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};   // reciprocal vectors 2 pi M^-1 (rows)
    double f[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};   // M^-1 (rows): fractional coordinates
    double volume = 0;
    int skchunks = 0;
};

// Pairs of an ion and a k-vector from which the mesh may be the faster way: both
// take the same time for 4,096 ions at 1e-6 accuracy (energy + forces 0.51 ms
// direct, 0.53 mesh; 8,000 ions 0.67 and 0.57).
constexpr double MESH_MIN_PAIRS = 1e8;
// Whether the system's reciprocal sums should go over the mesh; counts where the
// ions are (in M's sort buffers, and waits) if its sizes do not settle it.
bool mesh_suits(System &S, const EwaldParams &P, MeshState &M, const double *f, double volume);
// Sizes, tables and coefficients; b: reciprocal vectors (rows).
void mesh_plan(System &S, const EwaldParams &P, MeshState &M, const double *b, double inv_eps_2v);
// Sorts the atoms by tile and forms their kernel values; f: inverse cell rows.
void mesh_place(System &S, MeshState &M, const double *f);
// S(k) of the current charges at the places of the last mesh_place, as
// coefficients of the field, with the energy's block partials (M.epart).
void mesh_structure(System &S, MeshState &M, const double *f, const double *scaler);
// Adds the field's forces into S.frc (virial block partials into bpart, rows
// of 8), or subtracts the field from chi.
void mesh_atoms(System &S, MeshState &M, const double *f, const double *scaler, bool force,
                double *chi, double *bpart);
void mesh_release(MeshState &M);

void ewald_release(EwaldState &E);
// Energy of the charge_self singlets + Ewald (real, reciprocal, self, background).
double ewald_eem_energy(System &S, const EwaldParams &P, EwaldState &E);
// get_ewald_energy (Core.f90:8077-8089): the Ewald sum alone, real space
// included, with the dipole term (the caller passes unit scalers and a state
// of its own, so the cached structure factors of the model's Ewald stay).
double ewald_standalone_energy(System &S, const EwaldParams &P, EwaldState &E);
// Adds Ewald forces into S.frc; stress[6] receives the Ewald part.
void ewald_add_forces(System &S, const EwaldParams &P, EwaldState &E, double *stress);
// Electronegativities (charge_self + Ewald) into E.chi, sorted order, queued
// on the stream.  placed: the atoms have not moved since the previous call.
DBuf<double> &ewald_eem_chi(System &S, const EwaldParams &P, EwaldState &E, bool placed = false);
// Damped charge dynamics on device; S.q and rates (sorted order) updated.
void ewald_relax(System &S, const EwaldParams &P, EwaldState &E, double *rates, int n_steps,
                 double dt, double inertia, double friction, double tolerance, int *steps,
                 double *error);
