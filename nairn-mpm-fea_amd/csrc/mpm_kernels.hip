// mpm_kernels.hip -- gfx950 kernels of NairnMPM's explicit step (USAVG+, FLIP, uGIMP).
//
// Layout: particles stay in structure-of-arrays form; every step they are binned by cell with a
// stable counting sort into tiles of TileGeom<DIM> cells (tile-major cell keys), which gives a
// sorted slot -> particle map (order[]). Particle-to-grid sums never use floating-point atomics:
// each wave of a tile's block takes a layer of the tile's cells, stages its particles' per-axis shape
// factors in LDS, sums each cell's particles at the cell's candidate nodes in sorted order on the
// matrix cores (WaveScatter) and adds the sums to the wave's own LDS copy of the tile's node
// footprint. The copies are added in wave order and the footprint sums of each tile go to a partial
// buffer that a node kernel adds in fixed tile order. Results are therefore deterministic; they
// differ from the reference's single-patch sums by summation order only.
//
// Reference tasks (paths relative to the reference root, NairnMPM/src/NairnMPM_Class/):
//   k_p2g_mass    MassAndMomentumTask.cpp:48-127      (+ InitializationTask xi, :43-85)
//   k_node_mass   PostExtrapolationTask.cpp:46-165 + GridValueCalculation (UpdateStrainsFirstTask.cpp:120)
//   k_usf         UpdateStrainsFirstTask.cpp:101-168
//   k_p2g_force   GridForcesTask.cpp:40-153
//   k_node_force  PostForcesTask.cpp:43-111 + UpdateMomentaTask.cpp:44-64 + GridValueCalculation
//   k_g2p_p2g     UpdateParticlesTask.cpp:44-298 + UpdateStrainsLastContactTask.cpp:60-142
//   k_node_mom2   UpdateStrainsLastContactTask.cpp:139-149 + GridValueCalculation
//   k_usl_reset   UpdateStrainsFirstTask::FullStrainUpdate(last) + ResetElementsTask.cpp:44-265
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "mpm_device.h"
#include "mpm_kernels.h"

#define NT 256
// records (particles, or lCPDI corners) that a wave of a scatter stages at a time, two rounds per 64
// lanes, and the length of its rows: 16 words read from four rows by one instruction lie on different banks
#define WREC 32
#define WROW (WREC + 4)

// The kernels of one tile shape: this file builds shape 0, and mpm_kernels_s1.hip builds shape 1
// by defining MPM_TILE_SHAPE before including it. Each goes into its own namespace.
#ifndef MPM_TILE_SHAPE
#define MPM_TILE_SHAPE 0
#endif
#if MPM_TILE_SHAPE == 0
#define MPM_KNS mpmk_s0
#else
#define MPM_KNS mpmk_s1
#endif
namespace MPM_KNS {

template <int DIM> using TileGeom = TileShape<DIM, MPM_TILE_SHAPE>;
// Waves that share a tile in a scatter, and waves per SIMD their kernels are built for (shape 1's larger
// footprint leaves LDS for two). Eight waves give a few full tiles more parallelism and, where the
// registers allow two such blocks per CU, four waves per SIMD instead of three; each has its own staging
// rows and footprint copy, so they need 1.5 times the LDS, and with 32 particles a wave (2D) half of its
// lanes idle. us per launch with 4 and 8 waves: 7.08M uGIMP particles, update 670 and 600, mass 356 and
// 375, force 540 and 870 (its registers and LDS then leave one block); 87k lCPDI particles, mass 74 and 59,
// force 73 and 59, update 90 and 70 (16 waves: 60, 56, 69); 1.7M 2D particles, mass 73 and 110. The 3D lCPDI
// scatters hold four waves per SIMD with 128 registers and 20 (XPIC) to 88 (mass) bytes of scratch a lane.
// One choice per kernel: the order of a sum must not depend on the number of particles.
#define WAVES4 (MPM_TILE_SHAPE == 0 ? 3 : 2)
#define WAVES8 (MPM_TILE_SHAPE == 0 ? 4 : 2)
constexpr int UGIMP_NW = 4;
constexpr int G2P_NW(int dim) { return dim == 3 ? 8 : 4; }
constexpr int CORNER_NW(int dim) { return dim == 3 ? 8 : 4; }

template <int DIM>
__device__ __forceinline__ void tile_origin(const KGrid &g, int t, int &ox, int &oy, int &oz) {
    using G = TileGeom<DIM>;
    int tx = t % g.ntx;
    int r = t / g.ntx;
    int ty = r % g.nty;
    int tz = r / g.nty;
    ox = tx * G::TX; oy = ty * G::TY; oz = tz * G::TZ;
}

// bin key: field-major, then tile, then cell within the tile, so one (field, tile) pair owns a
// contiguous run of sorted particles
template <int DIM>
__device__ __forceinline__ int cell_key(const KGrid &g, int fld, int ci, int cj, int ck) {
    using G = TileGeom<DIM>;
    int tx = ci / G::TX, ty = cj / G::TY, tz = ck / G::TZ;
    int t = (tz * g.nty + ty) * g.ntx + tx;
    int l = ((ck - tz * G::TZ) * G::TY + (cj - ty * G::TY)) * G::TX + (ci - tx * G::TX);
    return (fld * g.tilesTotal + g.tileBase + t) * G::NC + l;
}

// node arrays of one velocity field
__device__ __forceinline__ KNodes field_view(const KGrid &g, const KNodes &N, int f) {
    KNodes v = N;
    long long nn = g.nstride, b = g.nodeBase;
    v.mass = N.mass + f * nn + b;
    v.pk = N.pk + 3 * f * nn + b;
    v.vk = N.vk + 3 * f * nn + b;
    v.ftot = N.ftot + 3 * f * nn + b;
    if (N.vprev) v.vprev = N.vprev + 3 * f * nn + b;
    v.cnt = N.cnt + f * nn + b;
    if (N.cvol) {
        v.cvol = N.cvol + f * nn + b;
        v.cdisp = N.cdisp + 3 * f * nn + b;
        v.cgrad = N.cgrad + 3 * f * nn + b;
    }
    return v;
}

// A grid read as constant memory, which no kernel writes: an instance's from the table, or the kernel's
// own from its arguments (every kernel's first). With a uniform instance the words come by scalar loads
// into scalar registers; read as ordinary memory they took vector registers (about 90 live through a
// tile kernel, a wave per SIMD), also where there is one grid and the table is never read.
typedef const __attribute__((address_space(4))) KGrid *GridPtr;

template <typename T>
__device__ __forceinline__ T constant_copy(const __attribute__((address_space(4))) T *p) {
    typedef const __attribute__((address_space(4))) unsigned long long *Words;
    static_assert(sizeof(T) % 8 == 0, "whole words");
    const Words s = (Words)p;
    union { T t; unsigned long long w[sizeof(T) / 8]; } u;
#pragma unroll
    for (unsigned k = 0; k < sizeof(T) / 8; k++) u.w[k] = s[k];
    return u.t;
}
__device__ __forceinline__ KGrid grid_copy(GridPtr p) { return constant_copy(p); }
__device__ __forceinline__ int const_int(const int *p) {
    return *(const __attribute__((address_space(4))) int *)p;
}

// grid of the instance that owns context tile tg (the kernel's grid for one instance)
__device__ __forceinline__ GridPtr tile_grid_ptr(const KGrid &g0, int tg) {
    if (!g0.inst) return (GridPtr)__builtin_amdgcn_kernarg_segment_ptr();
    return (GridPtr)(g0.inst + const_int(g0.tileInst + tg));
}

// grid of the instance that owns context node ng (node ranges are padded to NT per instance, so a
// block's nodes belong to one)
__device__ __forceinline__ KGrid node_grid(const KGrid &g0, long long ng) {
    if (!g0.inst) return g0;
    return grid_copy((GridPtr)(g0.inst + const_int(g0.nodeBlockInst + __builtin_amdgcn_readfirstlane((int)(ng / 256)))));
}

// Fields and node coordinates by 32-bit division (a 64-bit one is a hundred operations, and a node pass
// had four): the device's memory holds fewer than 2^32 nodes of the 100 bytes and more that each takes.
__device__ __forceinline__ int node_field(const KGrid &g0, long long nall) {
    return g0.nfields == 1 ? 0 : (int)((unsigned)nall / (unsigned)g0.nstride);
}
__device__ __forceinline__ void node_ijk(const KGrid &g, long long n, int &i, int &j, int &k) {
    const unsigned row = (unsigned)n / (unsigned)g.nnx, plane = row / (unsigned)g.nny;
    i = (int)((unsigned)n - row * (unsigned)g.nnx);
    j = (int)(row - plane * (unsigned)g.nny);
    k = (int)plane;
}

__device__ __forceinline__ void elem_ijk(const KGrid &g, int e, int &i, int &j, int &k) {
    i = e % g.nx;
    int r = e / g.nx;
    j = r % g.ny;
    k = r / g.ny;
}

// natural coordinates in the particle's element (EightNodeIsoparamBrick.cpp:276-281,
// FourNodeIsoparam.cpp:351-356), node coordinates xmin + i*dx (Generators.cpp:1823-1833)
template <int DIM>
__device__ __forceinline__ void particle_xi(const KGrid &g, int ei, int ej, int ek, double x, double y,
                                            double z, double xi[3], double invd[3]) {
    double xmn = g.xmin + (double)ei * g.dx, xmx = g.xmin + (double)(ei + 1) * g.dx;
    double ymn = g.ymin + (double)ej * g.dy, ymx = g.ymin + (double)(ej + 1) * g.dy;
    xi[0] = (2. * x - xmn - xmx) / (xmx - xmn);
    xi[1] = (2. * y - ymn - ymx) / (ymx - ymn);
    invd[0] = 2.0 / (xmx - xmn);
    invd[1] = 2.0 / (ymx - ymn);
    if (DIM == 3) {
        double zmn = g.zmin + (double)ek * g.dz, zmx = g.zmin + (double)(ek + 1) * g.dz;
        xi[2] = (2. * z - zmn - zmx) / (zmx - zmn);
        invd[2] = 2.0 / (zmx - zmn);
    } else {
        xi[2] = 0.;
        invd[2] = 0.;
    }
}

// per-axis factors of one particle: uGIMP, or classic linear (the same kernels serve both; the
// choice is uniform over a launch)
template <int DIM>
__device__ __forceinline__ void particle_factors(const KGrid &g, const KPart &P, int p, const double xi[3],
                                                 double S[3][4], double dS[3][4]) {
    if (g.shape == MPMGPU_SHAPE_LINEAR) {
#pragma unroll
        for (int a = 0; a < DIM; a++) linear_axis(xi[a], S[a], dS[a]);
        return;
    }
    double lpx, lpy, lpz;
    if (g.uniformLp) { lpx = g.lp[0]; lpy = g.lp[1]; lpz = g.lp[2]; }
    else { lpx = P.f(MPF_LP_X)[p]; lpy = P.f(MPF_LP_Y)[p]; lpz = P.f(MPF_LP_Z)[p]; }
    if (DIM == 3) {
        gimp_axis3(xi[0], lpx, 1. / (4. * lpx), S[0], dS[0]);
        gimp_axis3(xi[1], lpy, 1. / (4. * lpy), S[1], dS[1]);
        gimp_axis3(xi[2], lpz, 1. / (4. * lpy), S[2], dS[2]);   // EightNodeIsoparamBrick.cpp:303
    } else {
        gimp_axis2(xi[0], lpx, S[0], dS[0]);
        gimp_axis2(xi[1], lpy, S[1], dS[1]);
    }
}

// ---------------------------------------------------------------------------------------
// lCPDI (MatPoint3D::GetCPDINodesAndWeights, MatPoint3D.cpp:538-627; MatPoint2D.cpp:519-571;
// ElementBase::GetCPDIFunctions, MoreMPMElementBase.cpp:581-656). The semi-side vectors
// r1 = F(psz.x,0,0), r2, r3 are taken once per step, from the start-of-step F, by the first
// scatter and kept in P.cpr; every pass rebuilds the corners from them and the start position.
// A corner's element must be the particle's element or a neighbour of it (the 64-node candidate
// block); otherwise, or when a corner leaves the grid, the error counter is raised and the corner
// is clamped so that every access stays in bounds.
struct CpdiCorners {
    double xi[8][3];           // natural coordinates of each corner in its element
    int off[8][3];             // element of the corner relative to the particle's element (-1..1)
};

// MeshInfo::FindElementFromPoint on one axis of a regular grid (MeshInfo.cpp:597-625)
__device__ __forceinline__ int find_cell(double x, double xmin, double d, int n, bool &ok) {
    int c = (int)((x - xmin) / d);
    if (c < 0 || c >= n) {
        if (x == xmin + n * d) c = n - 1;
        else { ok = false; c = c < 0 ? 0 : n - 1; }
    }
    return c;
}

// semi-side vectors from the particle's F and size (GetSemiSideVectors, GetParticleSize)
template <int DIM>
__device__ __forceinline__ void cpdi_semi_sides_of(const KGrid &g, const KPart &P, int p, int ei, int ej, int ek,
                                                   const double ep[6], const double wr[3], double r[9]) {
    double lpx, lpy, lpz;
    if (g.uniformLp) { lpx = g.lp[0]; lpy = g.lp[1]; lpz = g.lp[2]; }
    else { lpx = P.f(MPF_LP_X)[p]; lpy = P.f(MPF_LP_Y)[p]; lpz = P.f(MPF_LP_Z)[p]; }
    double psx = ((g.xmin + (double)(ei + 1) * g.dx) - (g.xmin + (double)ei * g.dx)) * (0.5 * lpx);
    double psy = ((g.ymin + (double)(ej + 1) * g.dy) - (g.ymin + (double)ej * g.dy)) * (0.5 * lpy);
    double F[3][3];
    get_F3(ep, wr, F);
    if (DIM == 3) {
        double psz = ((g.zmin + (double)(ek + 1) * g.dz) - (g.zmin + (double)ek * g.dz)) * (0.5 * lpz);
        r[0] = F[0][0] * psx; r[1] = F[1][0] * psx; r[2] = F[2][0] * psx;
        r[3] = F[0][1] * psy; r[4] = F[1][1] * psy; r[5] = F[2][1] * psy;
        r[6] = F[0][2] * psz; r[7] = F[1][2] * psz; r[8] = F[2][2] * psz;
    } else {
        r[0] = F[0][0] * psx; r[1] = F[1][0] * psx; r[2] = 0.;
        r[3] = F[0][1] * psy; r[4] = F[1][1] * psy; r[5] = 0.;
        r[6] = r[7] = r[8] = 0.;
    }
}

template <int DIM>
__device__ __forceinline__ void cpdi_semi_sides(const KGrid &g, const KPart &P, int p, int ei, int ej, int ek,
                                                double r[9]) {
    double ep[6] = {P.f(MPF_EP_XX)[p], P.f(MPF_EP_YY)[p], P.f(MPF_EP_ZZ)[p], 0., 0., P.f(MPF_EP_XY)[p]};
    double wr[3] = {0., 0., P.f(MPF_WR_XY)[p]};
    if (DIM == 3) {
        ep[3] = P.f(MPF_EP_YZ)[p]; ep[4] = P.f(MPF_EP_XZ)[p];
        wr[0] = P.f(MPF_WR_YZ)[p]; wr[1] = P.f(MPF_WR_XZ)[p];
    }
    cpdi_semi_sides_of<DIM>(g, P, p, ei, ej, ek, ep, wr, r);
}

// linear function of element node (jx,jy,jz) at natural coordinates x (EightNodeIsoparamBrick.cpp:87-108,
// FourNodeIsoparam.cpp:189-214): 0.125 (1 +- xi)(1 +- eta)(1 +- zeta)
template <int DIM>
__device__ __forceinline__ double cpdi_cfn(const double x[3], int jx, int jy, int jz) {
    double t1 = 1. + (jx ? 1. : -1.) * x[0];
    double t2 = 1. + (jy ? 1. : -1.) * x[1];
    if (DIM == 3) {
        double t3 = 1. + (jz ? 1. : -1.) * x[2];
        return 0.125 * t1 * t2 * t3;
    }
    return 0.25 * t1 * t2;
}


template <int DIM>
__device__ __forceinline__ int foot_slot(int lx, int ly, int lz) {
    using G = TileGeom<DIM>;
    if (DIM == 3) return ((lz + 1) * G::FY + (ly + 1)) * G::FX + (lx + 1);
    return (ly + 1) * G::FX + (lx + 1);
}

// global node index of footprint slot s of a tile with cell origin (ox,oy,oz); -1 outside grid
template <int DIM>
__device__ __forceinline__ long long foot_node(const KGrid &g, int s, int ox, int oy, int oz) {
    using G = TileGeom<DIM>;
    int fx = s % G::FX;
    int fy = (s / G::FX) % G::FY;
    int fz = DIM == 3 ? s / (G::FX * G::FY) : 1;
    int i = ox + fx - 1, j = oy + fy - 1, k = DIM == 3 ? oz + fz - 1 : 0;
    if (i < 0 || i >= g.nnx || j < 0 || j >= g.nny || k < 0 || k >= g.nnz) return -1;
    return ((long long)k * g.nny + j) * g.nnx + i;
}

// corner c of a particle; false if the corner is unusable
template <int DIM>
__device__ __forceinline__ bool cpdi_corner(const KGrid &g, const double pos[3], const double r[9], int ei, int ej,
                                            int ek, int c, double xi[3], int off[3]) {
    bool ok = true;
    const int q = c & 3;
    const double s1 = (q == 1 || q == 2) ? 1. : -1.;
    const double s2 = q >= 2 ? 1. : -1.;
    const double s3 = c >= 4 ? 1. : -1.;
    double cx[3];
    if (DIM == 3) {
#pragma unroll
        for (int a = 0; a < 3; a++) cx[a] = pos[a] + s1 * r[a] + s2 * r[3 + a] + s3 * r[6 + a];
    } else {
        cx[0] = pos[0] + s1 * r[0] + s2 * r[3];
        cx[1] = pos[1] + s1 * r[1] + s2 * r[4];
        cx[2] = 0.;
    }
    const int ci = find_cell(cx[0], g.xmin, g.dx, g.nx, ok);
    const int cj = find_cell(cx[1], g.ymin, g.dy, g.ny, ok);
    const int ck = DIM == 3 ? find_cell(cx[2], g.zmin, g.dz, g.nz, ok) : 0;
    off[0] = ci - ei; off[1] = cj - ej; off[2] = DIM == 3 ? ck - ek : 0;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        if (off[a] < -1 || off[a] > 1) { ok = false; off[a] = off[a] < -1 ? -1 : 1; }
    }
    double invd[3];
    particle_xi<DIM>(g, ei + off[0], ej + off[1], ek + off[2], cx[0], cx[1], cx[2], xi, invd);
    return ok;
}

// corners of particle p for the step: from its saved semi-side vectors and start position
template <int DIM>
__device__ __forceinline__ bool cpdi_particle(const KGrid &g, const KPart &P, int p, int ei, int ej, int ek,
                                              CpdiCorners &cc) {
    double r[9];
#pragma unroll
    for (int a = 0; a < 9; a++) r[a] = P.cpr(a)[p];
    double pos[3] = {P.f(MPF_POS_X)[p], P.f(MPF_POS_Y)[p], DIM == 3 ? P.f(MPF_POS_Z)[p] : 0.};
    bool ok = true;
    constexpr int NCOR = DIM == 3 ? 8 : 4;
#pragma unroll
    for (int c = 0; c < NCOR; c++) ok &= cpdi_corner<DIM>(g, pos, r, ei, ej, ek, c, cc.xi[c], cc.off[c]);
    return ok;
}

// gradient weight of corner c as the reference writes it out per corner (MatPoint3D.cpp:571-594,
// MatPoint2D.cpp:551-566): the same six products summed in the same order, each term's sign taken
// from the corner's signs s1, s2, s3 (the scatters use these; the gathers use cpdi_wg)
template <int DIM>
__device__ __forceinline__ void cpdi_wg_listed(const double r[9], int c, double w[3]) {
    const int q = c & 3;
    const double s1 = (q == 1 || q == 2) ? 1. : -1.;
    const double s2 = q >= 2 ? 1. : -1.;
    if (DIM == 3) {
        const double s3 = c >= 4 ? 1. : -1.;
        const double x1 = r[0], y1 = r[1], z1 = r[2], x2 = r[3], y2 = r[4], z2 = r[5];
        const double x3 = r[6], y3 = r[7], z3 = r[8];
        double Vp = 8. * (x1 * (y2 * z3 - z2 * y3) + y1 * (z2 * x3 - x2 * z3) + z1 * (x2 * y3 - y2 * x3));
        Vp = 1. / Vp;
        w[0] = ((((-s3 * (z1 * y2) + s3 * (y1 * z2)) + s2 * (z1 * y3)) - s1 * (z2 * y3)) - s2 * (y1 * z3) + s1 * (y2 * z3)) * Vp;
        w[1] = ((((s3 * (z1 * x2) - s3 * (x1 * z2)) - s2 * (z1 * x3)) + s1 * (z2 * x3)) + s2 * (x1 * z3) - s1 * (x2 * z3)) * Vp;
        w[2] = ((((-s3 * (y1 * x2) + s3 * (x1 * y2)) + s2 * (y1 * x3)) - s1 * (y2 * x3)) - s2 * (x1 * y3) + s1 * (x2 * y3)) * Vp;
    } else {
        double Ap = 4. * (r[0] * r[4] - r[1] * r[3]);
        Ap = 1. / Ap;
        w[0] = (-s2 * r[1] + s1 * r[4]) * Ap;
        w[1] = (s2 * r[0] - s1 * r[3]) * Ap;
        w[2] = 0.;
    }
}

// linear factors of corner c at its particle's candidate node offsets o1 - 1 per axis (o1 = 0..3): the
// corner's element holds the nodes at offsets off and off + 1, where they are 1 - xi and 1 + xi
template <int DIM>
__device__ __forceinline__ void cpdi_table(const double xi[3], const int off[3], double (*T)[4]) {
#pragma unroll
    for (int a = 0; a < DIM; a++)
#pragma unroll
        for (int o = 0; o < 4; o++)
            T[a][o] = o == off[a] + 1 ? 1. - xi[a] : (o == off[a] + 2 ? 1. + xi[a] : 0.);
}

// gradient weight of corner c as the scatters stage it: times the corner function's factor
template <int DIM>
__device__ __forceinline__ void cpdi_wg_staged(const double r[9], int c, double w[3]) {
    cpdi_wg_listed<DIM>(r, c, w);
#pragma unroll
    for (int a = 0; a < 3; a++) w[a] *= DIM == 3 ? 0.125 : 0.25;
}

// ---------------------------------------------------------------------------------------
// Shape factors of the step's passes (uGIMP and classic). Every pass needs them for every particle,
// and evaluated as the reference writes them (particle_factors below: four candidates per axis, a
// division for each natural coordinate and size, an integer division per axis for the cell) they
// were most of the vector work of a pass (about 700 of the mass scatter's 1,500 VALU operations per
// particle). Here the cell comes from the particle's bin key, the divisions are done with the
// reciprocals of the cell size and the particle size kept in KGrid, and an axis evaluates the
// three nodes that can lie in the support: with a = |xi| they are the near one at distance 1 - a,
// the other node of the cell at 1 + a, and the outer one at 3 - a on the near one's side.

// The rows with an opaque length: their addresses are then formed where a particle's words are read
// (scalar additions) instead of being held in registers over the particle loop.
__device__ __forceinline__ KPart local_rows(const KPart &P) {
    KPart q = P;
    asm volatile("" : "+s"(q.n));
    return q;
}

// the particle's cell within its tile, from its bin key
template <int DIM>
__device__ __forceinline__ void tile_cell(int key, int tall, int &lx, int &ly, int &lz) {
    using G = TileGeom<DIM>;
    const int l = key - tall * G::NC;
    lx = l % G::TX;
    ly = (l / G::TX) % G::TY;
    lz = DIM == 3 ? l / (G::TX * G::TY) : 0;
}

// Natural coordinate of x in cell c of one axis (node coordinates xmin + i*d) and 2 over the cell's
// size. The quotient (2x - xmn - xmx)/(xmx - xmn) is found from r = 1/d: a Newton step gives the
// reciprocal of the cell's own (rounded) size and one more of the quotient gives the correctly
// rounded value, so a particle on the edge of a support lies exactly where the division puts it.
__device__ __forceinline__ double natural_coord(double x, double xmin, double d, double r, int c, double &invd) {
    const double mn = xmin + (double)c * d, mx = xmin + (double)(c + 1) * d;
    const double w = mx - mn, n = 2. * x - mn - mx;
    const double y = fma(r, fma(-w, r, 1.), r);
    const double q = n * y;
    invd = 2. * y;
    return fma(fma(-q, w, n), y, q);
}

// values and derivatives (natural coordinates, towards the near node) at the three nodes of an axis
struct AxisFactors {
    double sn, sm, sx;         // near, the cell's other node, outer
    double dn, dm, dx;       // magnitudes with the sign of the derivative left of the node
    int w;                     // 1 when xi >= 0: near is candidate offset 1, outer 2, other 0
    __device__ __forceinline__ double s4(int o) const {      // factor at candidate offset o - 1
        return o == 0 ? (w ? 0. : sx) : o == 1 ? (w ? sm : sn) : o == 2 ? (w ? sn : sm) : (w ? sx : 0.);
    }
    __device__ __forceinline__ double d4(int o) const {
        return o == 0 ? (w ? 0. : dx) : o == 1 ? (w ? dm : dn) : o == 2 ? (w ? -dn : -dm) : (w ? -dx : 0.);
    }
    __device__ __forceinline__ double s3(int j) const {      // factor at window node w + j
        return j == 1 ? sn : ((j == 0) == (w != 0)) ? sm : sx;
    }
    __device__ __forceinline__ double d3(int j) const {
        return j == 0 ? (w ? dm : dx) : j == 1 ? (w ? -dn : dn) : (w ? -dx : -dm);
    }
};

// uGIMP factor and derivative at distance xp (zero outside, and for a NaN position)
__device__ __forceinline__ void gimp_any(double xp, double lp, double inv, double i2lp, double &s, double &d) {
    const double q1 = 2. - lp, q2 = 2. + lp, arg = (q2 - xp) * inv;
    s = xp < lp ? ((4. - lp) * lp - xp * xp) * inv : xp <= q1 ? 0.5 * (2. - xp) : 2. * lp * arg * arg;
    d = xp < lp ? -xp * i2lp : xp <= q1 ? -0.5 : -arg;
    if (!(xp < q2)) { s = 0.; d = 0.; }
}

// lp: half size of the particle; inv = 1/(4 lp) (the 3D z axis takes lp.y's, as in the reference);
// i2lp = 1/(2 lp) of the axis itself. INSIDE: |xi| <= 1; without it any coordinate (a position
// outside the cell that its element names, or NaN), equal to the other for |xi| <= 1.
template <bool INSIDE>
__device__ __forceinline__ void axis_factors(double xi, double lp, double inv, double i2lp, AxisFactors &f) {
    const double a = fabs(xi);
    f.w = xi >= 0. ? 1 : 0;
    if (!INSIDE) {
        gimp_any(fabs(1. - a), lp, inv, i2lp, f.sn, f.dn);
        gimp_any(1. + a, lp, inv, i2lp, f.sm, f.dm);
        gimp_any(fabs(3. - a), lp, inv, i2lp, f.sx, f.dx);
        if (a > 1.) f.dn = -f.dn;
        if (a > 3.) f.dx = -f.dx;
        return;
    }
    const double x0 = 1. - a, x1 = 1. + a, x2 = 3. - a, q1 = 2. - lp, q2 = 2. + lp;
    const double a1 = (q2 - x1) * inv, a2 = (q2 - x2) * inv;
    f.sn = x0 < lp ? ((4. - lp) * lp - x0 * x0) * inv : 0.5 * (2. - x0);
    f.dn = x0 < lp ? -x0 * i2lp : -0.5;
    f.sm = x1 <= q1 ? 0.5 * (2. - x1) : 2. * lp * a1 * a1;
    f.dm = x1 <= q1 ? -0.5 : -a1;
    f.sx = x2 < q2 ? 2. * lp * a2 * a2 : 0.;
    f.dx = x2 < q2 ? -a2 : 0.;
}

// the element's linear functions (classic MPM)
__device__ __forceinline__ void linear_factors(double xi, AxisFactors &f) {
    const double n = 0.5 * (1. + fabs(xi)), o = 0.5 * (1. - fabs(xi));
    f.w = xi >= 0. ? 1 : 0;
    f.sn = n >= 0. ? n : 0.;
    f.sm = o >= 0. ? o : 0.;
    f.dn = n >= 0. ? -0.5 : 0.;
    f.dm = o >= 0. ? -0.5 : 0.;
    f.sx = f.dx = 0.;
}

// The axes of particle p in cell (cx, cy, cz). The grid's words are read here, through an opaque
// pointer (scalar loads once per 64 particles): held over the particle loop they and the row
// addresses overran the scalar registers.
template <int DIM>
__device__ __forceinline__ void particle_axes(GridPtr gp, const KPart &P, int p, int cx, int cy, int cz,
                                              const double pos[3], AxisFactors f[DIM], double invd[DIM]) {
    asm volatile("" : "+s"(gp));
    double xi[DIM];
    xi[0] = natural_coord(pos[0], gp->xmin, gp->dx, gp->rdx[0], cx, invd[0]);
    xi[1] = natural_coord(pos[1], gp->ymin, gp->dy, gp->rdx[1], cy, invd[1]);
    if constexpr (DIM == 3) xi[2] = natural_coord(pos[2], gp->zmin, gp->dz, gp->rdx[2], cz, invd[2]);
    if (gp->shape == MPMGPU_SHAPE_LINEAR) {
#pragma unroll
        for (int a = 0; a < DIM; a++) linear_factors(xi[a], f[a]);
        return;
    }
    bool inside = true;
#pragma unroll
    for (int a = 0; a < DIM; a++) inside = inside && fabs(xi[a]) <= 1.;
    // z takes 1/(4 lp.y) in 3D (EightNodeIsoparamBrick.cpp:303)
    if (gp->uniformLp && __all(inside)) {
#pragma unroll
        for (int a = 0; a < DIM; a++) axis_factors<true>(xi[a], gp->lp[a], gp->rlp4[a == 2 ? 1 : a], gp->rlp2[a], f[a]);
        return;
    }
    const KPart R = local_rows(P);
#pragma unroll
    for (int a = 0; a < DIM; a++) {
        const double lp = R.f(MPF_LP_X + a)[p], own = 1. / (4. * lp);
        const double inv = a == 2 ? 1. / (4. * R.f(MPF_LP_Y)[p]) : own;
        axis_factors<false>(xi[a], lp, inv, 2. * own, f[a]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Support window of one particle: with a half size lp <= 1 (natural units) a particle with xi < 0
// touches no node at offset 2 and one with xi >= 0 none at offset -1, so three offsets per axis
// starting at w = 0 (offsets -1..1) or w = 1 (0..2) hold every node of its support. The window's
// factors are zero for nodes outside the support, and derivatives times 2/dx.
template <int DIM>
__device__ __forceinline__ void particle_window(const AxisFactors f[DIM], const double invd[DIM], int w[3],
                                                double Sw[3][3], double Dw[3][3]) {
#pragma unroll
    for (int a = 0; a < 3; a++) {
        w[a] = 0;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            if (a >= DIM) { Sw[a][j] = j == 1 ? 1. : 0.; Dw[a][j] = 0.; continue; }
            w[a] = f[a < DIM ? a : 0].w;
            Sw[a][j] = f[a < DIM ? a : 0].s3(j);
            Dw[a][j] = f[a < DIM ? a : 0].d3(j) * invd[a < DIM ? a : 0];
        }
    }
}

// ---------------------------------------------------------------------------------------
// lCPDI, a lane per particle corner: a wave takes eight particles (sixteen in 2D) of its cells at a time
// (their corners are adjacent lanes), and the scatters take the corners as records (WaveScatter, PPR = NCOR).
template <int DIM> struct Corners {
    static constexpr int N = DIM == 3 ? 8 : 4, PB = 64 / N;    // corners, particles per 64 lanes
    static constexpr double W = 1. / N, WW = W * W;             // a corner's share; times its function's factor
};

// n/d from r = 1/d, correctly rounded as a division (an infinite one has no remainder to correct it by)
__device__ __forceinline__ double quotient(double n, double d, double r) {
    const double q = n * r, c = fma(fma(-q, d, n), r, q);
    return c == c ? c : q;
}

// corner c of a particle at pos in cell (cx, cy, cz): cpdi_corner without its divisions
template <int DIM>
__device__ __forceinline__ bool corner_lane(GridPtr gp, const double pos[DIM], const double r[9], int cx, int cy, int cz,
                                            int c, double xi[3], int off[3]) {
    asm volatile("" : "+s"(gp));
    const int q = c & 3;
    const double s1 = (q == 1 || q == 2) ? 1. : -1.;
    const double s2 = q >= 2 ? 1. : -1.;
    const double s3 = c >= 4 ? 1. : -1.;
    const double mn[3] = {gp->xmin, gp->ymin, gp->zmin}, d[3] = {gp->dx, gp->dy, gp->dz};
    const int n[3] = {gp->nx, gp->ny, gp->nz}, cell[3] = {cx, cy, cz};
    bool ok = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        if (a >= DIM) { xi[a] = 0.; off[a] = 0; continue; }
        double x = pos[a < DIM ? a : 0] + s1 * r[a] + s2 * r[3 + a];
        if (DIM == 3) x += s3 * r[6 + a];
        int e = (int)quotient(x - mn[a], d[a], gp->rdx[a]);      // find_cell
        if (e < 0 || e >= n[a]) {
            if (x == mn[a] + n[a] * d[a]) e = n[a] - 1;
            else { ok = false; e = e < 0 ? 0 : n[a] - 1; }
        }
        off[a] = e - cell[a];
        if (off[a] < -1 || off[a] > 1) { ok = false; off[a] = off[a] < -1 ? -1 : 1; }
        double invd;
        xi[a] = natural_coord(x, mn[a], d[a], gp->rdx[a], cell[a] + off[a], invd);
    }
    return ok;
}

// A corner's rows at record i: 1 - xi and 1 + xi at the candidates of its element, zeros elsewhere. The
// reference leaves a corner's node out when its function, the product of the axes' factors, is below 1e-15.
// A factor below 2e-15 makes all its products so (the others are 2 at most) and is staged as zero. A corner
// within about 1e-7 of two edges of its element, or 1e-14 of one, has products below the limit of larger
// factors; the mass scatter, which decides which nodes a particle reaches, and all scatters in 2D leave
// those out too (WaveScatter, CUT). In 3D the other sums take them: where no particle has mass the node
// passes drop them, elsewhere they are weights below the limit beside the ones that count. The factors 1/8
// (2D: 1/4) of the function and of the corner's share are in the payload.
template <int DIM> struct CornerLimit { static constexpr double V = (DIM == 3 ? 8. : 4.) * 1e-15; };

// 3D: whether a node of the corner may have a function below the limit with no factor staged as zero: the
// least product of staged factors is that of the least one of each axis (of one that is staged alone, 2
// less rounding, 1 is taken: what this adds only takes the longer way to the same sums)
__device__ __forceinline__ bool corner_cut(const double xi[3]) {
    double m = 1.;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double f = 1. - fabs(xi[a]);
        m *= f < 2e-15 ? 1. : f;
    }
    return m < CornerLimit<3>::V;
}

template <int DIM, int NU>
__device__ __forceinline__ void stage_corner(double (*S)[WROW], int i, const double xi[3], const int off[3],
                                             const double u[NU]) {
#pragma unroll
    for (int a = 0; a < DIM; a++) {
        double lo = 1. - xi[a], hi = 1. + xi[a];
        lo = lo < 2e-15 ? 0. : lo;
        hi = hi < 2e-15 ? 0. : hi;
#pragma unroll
        for (int o = 0; o < 4; o++) S[a * 4 + o][i] = o == off[a] + 1 ? lo : (o == off[a] + 2 ? hi : 0.);
    }
#pragma unroll
    for (int q = 0; q < NU; q++) S[4 * DIM + q][i] = u[q];
}

// sum over the corner lanes of a particle, the total in each of them
template <int CTRL> __device__ __forceinline__ double dpp_double(double v) {
    union { double d; int i[2]; } t;
    t.d = v;
    t.i[0] = __builtin_amdgcn_update_dpp(0, t.i[0], CTRL, 0xf, 0xf, true);
    t.i[1] = __builtin_amdgcn_update_dpp(0, t.i[1], CTRL, 0xf, 0xf, true);
    return t.d;
}
template <int DIM> __device__ __forceinline__ double corner_sum(double v) {
    v += dpp_double<0xB1>(v);      // quad_perm 1,0,3,2
    v += dpp_double<0x4E>(v);      // quad_perm 2,3,0,1
    if (DIM == 3) v += dpp_double<0x141>(v);   // mirror within eight lanes
    return v;
}

// ---------------------------------------------------------------------------------------
// binning: key + histogram, exclusive scan, scatter, per-cell sort (stable by particle index)

// Runs of equal keys among a wave's active lanes, which are a prefix: whether the lane starts one, and its
// length there. The rows are kept in tile order and a tile's particles are taken in sorted order, so keys
// come in runs; a run takes one atomic, all runs of the wave at once (one after another, they were 40 us
// of k_usl_reset's 830 on 7.08M particles and 17 of 131 on 1.7M in 2D).
__device__ __forceinline__ bool run_start(int key, int &length) {
    const int lane = (int)__lane_id();
    const int prev = __shfl_up(key, 1);
    const bool start = lane == 0 || prev != key;
    const int active = __popcll(__ballot(1));
    const unsigned long long later = __ballot(start) & ~((2ull << lane) - 1ull);
    length = (later ? __ffsll((long long)later) - 1 : active) - lane;
    return start;
}

// count[key] += 1 for every active lane (a prefix of the wave's)
__device__ __forceinline__ void wave_count(int *count, int key) {
    int length;
    if (run_start(key, length)) atomicAdd(&count[key], length);
}

template <int DIM>
__global__ void k_bin_keys(KGrid g0, KPart P, KBins B) {
    long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P.n) return;
    if (B.stop[0]) { B.key[p] = 0; return; }   // input refused on the device: nothing is binned
    // (only the words used are read: a copy of the grid, whose table is indexed by the material, would go
    // through 520 bytes of private memory per particle)
    const int mat = P.mat[p];
    const GridPtr gp = g0.inst ? (GridPtr)(g0.inst + g0.matInst[mat]) : (GridPtr)__builtin_amdgcn_kernarg_segment_ptr();
    const KGrid g = grid_copy(gp);
    int i, j, k;
    elem_ijk(g, P.elem[p], i, j, k);
    // fieldOf covers the materials of one multimaterial context; batch instances are single-field
    // and their material numbers run past its end
    const int fld = g.nfields > 1 ? gp->fieldOf[mat] : 0;
    int key = cell_key<DIM>(g, fld, i, j, DIM == 3 ? k : 0);
    B.key[p] = key;
    wave_count(B.count, key);
}

// Cell starts, in one launch: blocks take runs of SCAN_BLOCK keys in the order in which they start
// (a ticket), publish their sum, and add up the sums before theirs until they meet a block that has
// published its whole prefix (decoupled look-back; a block waits for blocks that started before it
// only, so every wait ends). A run holds whole tiles, so its threads also list the non-empty ones.
// state: 2 flag bits and 30 bits of sum (fewer than 2^30 particles fit in the device's memory), zeroed
// with the ticket by k_bin_sort_cells. Three scan launches and a fourth for the list took 20 us of a
// step on 885k particles (0.7M keys) and 11 on 4k; this one takes 10 and 6. It is latency: tickets on one
// address, then one look at the sums of up to 256 blocks before; runs of 8,192 keys (four times the
// tickets) took 20 us instead of 12 on 2.1M keys, and scans by shuffles instead of data-parallel moves 14.
#define SCAN_NT 1024
#define SCAN_ROUNDS 8              // of 256 keys per wave, four a lane
#define SCAN_BLOCK (SCAN_NT * 4 * SCAN_ROUNDS)
#define SCAN_SUM 0x40000000u
#define SCAN_PREFIX 0x80000000u
#define SCAN_VALUE 0x3fffffffu

__device__ __forceinline__ unsigned scan_wait(const unsigned *state) {
    unsigned v;
    while (!((v = __hip_atomic_load(state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) & (SCAN_SUM | SCAN_PREFIX)))
        __builtin_amdgcn_s_sleep(1);
    return v;
}

// a lane's neighbour's value by a data-parallel move (zero where there is none)
template <int CTRL, int ROWS = 0xf> __device__ __forceinline__ int dpp_int(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
// inclusive sum over the wave's lanes: within rows of 16, then each row's total to those after it
__device__ __forceinline__ int wave_inclusive(int v) {
    v += dpp_int<0x111>(v);
    v += dpp_int<0x112>(v);
    v += dpp_int<0x114>(v);
    v += dpp_int<0x118>(v);
    v += dpp_int<0x142, 0xa>(v);
    v += dpp_int<0x143, 0xc>(v);
    return v;
}
// sum over the aligned 16 or 32 lanes, in each of them
template <int LANES> __device__ __forceinline__ int lanes_sum(int v) {
    static_assert(LANES == 16 || LANES == 32, "a row or two");
    v += dpp_int<0xB1>(v);
    v += dpp_int<0x4E>(v);
    v += dpp_int<0x141>(v);
    v += dpp_int<0x140>(v);
    return LANES == 32 ? v + __shfl_xor(v, 16) : v;
}

template <int NC>
__global__ __launch_bounds__(SCAN_NT) void k_bin_scan(KBins B, int n, int nb) {
    static_assert(256 % NC == 0 && 64 % (NC / 4) == 0, "whole tiles");
    __shared__ int s_sum[SCAN_NT / 64];
    __shared__ int s_block, s_before;
    unsigned *state = reinterpret_cast<unsigned *>(B.blockSums);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    // a single block needs no ticket and has no one to tell: a step on 4k particles 58.9 -> 58.2 us
    if (nb > 1) {
        if (threadIdx.x == 0) s_block = atomicAdd(&B.blockSums[nb], 1);
        __syncthreads();
    }
    const int blk = nb > 1 ? s_block : 0, base = blk * SCAN_BLOCK + w * (256 * SCAN_ROUNDS) + l * 4;   // of this lane's first round
    if (blk >= nb) return;               // (a ticket is taken once per block, so this does not happen)
    const bool stopped = B.stop[0] != 0;
    if (blk == 0) {
        // the tile list is rebuilt; the tile kernels' cursors start again; one more step completed
        if (threadIdx.x < TILE_SLOTS * 8) B.work[threadIdx.x * TILE_SLOT_STRIDE] = 0;
        if (threadIdx.x == 0) {
            __hip_atomic_store(B.ntiles, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (!stopped) B.stop[2] += 1;
        }
    }
    int v[SCAN_ROUNDS][4], own[SCAN_ROUNDS], ex[SCAN_ROUNDS], sum = 0;     // keys, their sum, the wave's sum before
#pragma unroll
    for (int r = 0; r < SCAN_ROUNDS; r++) {
        const int at = base + 256 * r;
        if (at + 4 <= n) __builtin_memcpy(v[r], B.count + at, sizeof(v[r]));
        else {
#pragma unroll
            for (int i = 0; i < 4; i++) v[r][i] = at + i < n ? B.count[at + i] : 0;
        }
    }
#pragma unroll
    for (int r = 0; r < SCAN_ROUNDS; r++) {
        own[r] = v[r][0] + v[r][1] + v[r][2] + v[r][3];
        const int incl = wave_inclusive(own[r]);
        ex[r] = sum + incl - own[r];
        sum += __builtin_amdgcn_readlane(incl, 63);
    }
    if (l == 0) s_sum[w] = sum;
    __syncthreads();
    if (w == 0) {
        // the waves' sums, then the sums of the blocks before
        const int t = l < SCAN_NT / 64 ? s_sum[l] : 0, ti = wave_inclusive(t), total = __builtin_amdgcn_readlane(ti, 63);
        if (l < SCAN_NT / 64) s_sum[l] = ti - t;
        int before = 0;
        if (blk > 0) {
            if (l == 0)
                __hip_atomic_store(&state[blk], SCAN_SUM | (unsigned)total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // four blocks a lane, nearest first; those behind a whole prefix are in it already
            int part = 0;
            for (int at = blk - 1 - 4 * l;; at -= 256) {
                unsigned s[4];
#pragma unroll
                for (int i = 0; i < 4; i++) s[i] = at - i >= 0 ? scan_wait(&state[at - i]) : SCAN_PREFIX;
                bool end = false;
                int own = 0;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    own += end ? 0 : (int)(s[i] & SCAN_VALUE);
                    end = end || (s[i] & SCAN_PREFIX);
                }
                const unsigned long long ends = __ballot(end);
                if (l <= (ends ? __ffsll((long long)ends) - 1 : 63)) part += own;
                if (ends) break;
            }
            before = __builtin_amdgcn_readlane(wave_inclusive(part), 63);
            // the tile list's length was cleared by the first block: its prefix, or one that follows
            // from it, has been read
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        if (l == 0) {
            if (nb > 1)
                __hip_atomic_store(&state[blk], SCAN_PREFIX | (unsigned)(before + total), __ATOMIC_RELEASE,
                                   __HIP_MEMORY_SCOPE_AGENT);
            s_before = before;
        }
    }
    __syncthreads();
    const int before = s_before + s_sum[w];
    constexpr int TL = NC / 4;         // lanes of a tile; its first one lists it
    unsigned on = 0;                   // per round
    int listed = 0;
#pragma unroll
    for (int r = 0; r < SCAN_ROUNDS; r++) {
        const int at = base + 256 * r, t = at / NC;
        int c[4];
        c[0] = before + ex[r];
#pragma unroll
        for (int i = 1; i < 4; i++) c[i] = c[i - 1] + v[r][i - 1];
        if (at + 4 <= n) __builtin_memcpy(B.cellStart + at, c, sizeof(c));
        else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (at + i < n) B.cellStart[at + i] = c[i];
        }
        const int in = lanes_sum<TL>(own[r]);
        const bool mine = l % TL == 0 && t < B.ntall;
        if (mine) B.tileOn[t] = !stopped && in > 0 ? 1 : 0;
        if (mine && !stopped && in > 0) { on |= 1u << r; listed++; }
    }
    const int upto = wave_inclusive(listed), all = __builtin_amdgcn_readlane(upto, 63);
    if (all == 0) return;
    int slot = 0;
    if (l == 0) slot = atomicAdd(B.ntiles, all);
    slot = __shfl(slot, 0) + upto - listed;
#pragma unroll
    for (int r = 0; r < SCAN_ROUNDS; r++)
        if (on >> r & 1u) B.tiles[slot++] = (base + 256 * r) / NC;
}

// Slots by key. The rows are kept in tile order, so the keys of a wave's 64 consecutive rows come
// in runs; the first lane of each run takes the run's slots with one atomic, all runs of the wave
// at once (one round trip per wave, not one per key). The order inside a cell is then fixed by
// k_bin_sort_cells, so the slots' first placement does not change any result.
__device__ __forceinline__ void bin_scatter(const KPart &P, const KBins &B, long long p) {
    if (B.stop[0]) return;
    const bool valid = p < P.n;
    const int key = valid ? B.key[p] : -1;
    const int lane = (int)__lane_id();
    const int prev = __shfl_up(key, 1);
    const bool start = valid && (lane == 0 || prev != key);
    const unsigned long long starts = __ballot(start);
    const int nvalid = 64 - __clzll(__ballot(valid));                 // valid lanes are a prefix
    const unsigned long long upto = (2ull << lane) - 1ull;           // lanes 0..lane
    const int leader = 63 - __clzll(starts & upto);                   // this lane's run start
    int base = 0;
    if (start) {
        const unsigned long long later = starts & ~upto;
        const int end = later ? __ffsll((long long)later) - 1 : nvalid;
        base = B.cellStart[key] + atomicAdd(&B.cursor[key], end - lane);
    }
    base = __shfl(base, leader & 63);
    if (valid) {
        const int slot = base + (lane - leader);
        B.order[slot] = (int)p;
        B.shome[slot] = B.home[p];
    }
}

// the (field, tile) pairs the next node passes visit (node_needed): needed = the pair or one of its
// neighbours is non-empty; needAny = needed now or at the previous binning. A stopped run needs none.
template <int DIM>
__device__ __forceinline__ void tile_need(const KGrid &g0, const KBins &B, int tall) {
    if (tall >= B.ntall) return;
    const int fld = tall / g0.tilesTotal;
    const int tg = tall - fld * g0.tilesTotal;
    const KGrid g = g0.inst ? g0.inst[g0.tileInst[tg]] : g0;   // (a thread per tile)
    const int t = tg - g.tileBase;
    const int tx = t % g.ntx, ty = (t / g.ntx) % g.nty, tz = DIM == 3 ? t / (g.ntx * g.nty) : 0;
    int need = 0;
    if (!B.stop[0]) {
        const int zl = DIM == 3 ? max(tz - 1, 0) : 0, zh = DIM == 3 ? min(tz + 1, g.ntz - 1) : 0;
        for (int z = zl; z <= zh && !need; z++)
            for (int y = max(ty - 1, 0); y <= min(ty + 1, g.nty - 1) && !need; y++)
                for (int x = max(tx - 1, 0); x <= min(tx + 1, g.ntx - 1); x++) {
                    const long long u = (long long)fld * g0.tilesTotal + g.tileBase + (z * g.nty + y) * g.ntx + x;
                    if (B.tileOn[u]) { need = 1; break; }
                }
    }
    B.needAny[tall] = need | B.need[tall];
    B.need[tall] = need;
}

// the first `need` blocks take the pairs, the others the particles (one launch: neither needs the other)
template <int DIM>
__global__ void k_bin_scatter(KGrid g0, KPart P, KBins B, int need) {
    if ((int)blockIdx.x < need) tile_need<DIM>(g0, B, blockIdx.x * blockDim.x + threadIdx.x);
    else bin_scatter(P, B, (long long)(blockIdx.x - need) * blockDim.x + threadIdx.x);
}

// the particles of a cell in upload order (their index at upload, which the memory order of the
// rows does not change), so every sum over a cell's particles has the same order in any layout.
// Up to 16 particles are read with independent loads and, unless they are in order already (they stayed
// put, in rows sorted by upload index), each is written to its rank: the insertion sort in memory, which
// larger cells still take, was a chain of loads and kept 885k particles of 8 a cell for 29 us once the
// rows had moved since their last sort.
template <int MOST>
__device__ __forceinline__ void sort_few(const KBins &B, int b, int e) {
    int h[MOST], o[MOST];
#pragma unroll
    for (int t = 0; t < MOST; t++) h[t] = b + t < e ? B.shome[b + t] : 0x7fffffff;
    bool sorted = true;
#pragma unroll
    for (int t = 1; t < MOST; t++) sorted = sorted && h[t - 1] <= h[t];
    if (sorted) return;
#pragma unroll
    for (int t = 0; t < MOST; t++) o[t] = b + t < e ? B.order[b + t] : 0;
#pragma unroll
    for (int t = 0; t < MOST; t++) {
        int rank = 0;
#pragma unroll
        for (int u = 0; u < MOST; u++) rank += u != t && h[u] < h[t] ? 1 : 0;
        if (b + t < e) { B.order[b + rank] = o[t]; B.shome[b + rank] = h[t]; }
    }
}

__device__ __forceinline__ void sort_cell(const KBins &B, int b, int e) {
    if (e - b <= 8) sort_few<8>(B, b, e);
    else if (e - b <= 16) sort_few<16>(B, b, e);
    else {
        for (int i = b + 1; i < e; i++) {
            const int v = B.order[i];
            const int hv = B.shome[i];
            int j = i - 1;
            while (j >= b && B.shome[j] > hv) {
                B.order[j + 1] = B.order[j];
                B.shome[j + 1] = B.shome[j];
                j--;
            }
            B.order[j + 1] = v;
            B.shome[j + 1] = hv;
        }
    }
}

// Only listed tiles hold particles and counts; a stopped run lists none and clears every count.
// Ends the binning: counts, cursors and the scan's words are zero for the next one.
__global__ void k_bin_sort_cells(KBins B, int nc, int nb) {
    const int i0 = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
    for (int i = i0; i <= nb; i += step) B.blockSums[i] = 0;
    const bool stopped = B.stop[0] != 0;
    const int end = stopped ? B.nkeys : B.ntiles[0] * nc;
    for (int i = i0; i < end; i += step) {
        const int c = stopped ? i : B.tiles[i / nc] * nc + i % nc;
        if (!stopped) sort_cell(B, B.cellStart[c], B.cellStart[c + 1]);
        B.cursor[c] = 0;
        B.count[c] = 0;
    }
}

// A tile kernel's blocks walk the list of non-empty tiles, so no workgroup is spent on an empty
// tile. Block b takes entry b first, then further entries claimed from one of eight cursors (the
// block's cursor is b mod 8, so the blocks sharing a cursor sit on one XCD and a claim never waits
// behind the whole device), entry gridDim.x + c + 8 k for the k-th claim on cursor c. Results do not
// depend on which block takes a tile. A wave's memory operations return in order, so a claim (an atomic
// on a contended word) holds up the loads after it: a 3D tile's is made after its particles, a 2D tile's,
// which are short, before (885k particles in 3D: 548 us per step with it before, 537 after; 1.7M in 2D: 506
// and 511), none where every entry has its block, and claims two tiles ahead cost more than the wait they
// spare (559). The first entry is read beside the list's length: a grid has no more blocks than the list
// has room.
template <int DIM, typename F>
__device__ __forceinline__ void for_each_tile(const KBins &B, F &tile) {
    __shared__ int s_li[2];
    const int n = B.ntiles[0];
    int t = B.tiles[blockIdx.x];
    if ((int)blockIdx.x >= n) return;
    const int cur = blockIdx.x & 7;
    int *cursor = &B.work[(B.slot * 8 + cur) * TILE_SLOT_STRIDE];
    for (int k = 0;; k ^= 1) {
        int next = n > (int)gridDim.x ? -1 : n;            // no claims where every entry has its block
        auto claim = [&] {
            if (threadIdx.x == 0 && next < 0) next = (int)gridDim.x + cur + 8 * atomicAdd(cursor, 1);
        };
        // one tile per block: a scalar for the compiler, so an instance's grid and the node views
        // built from it stay in scalar registers
        if (DIM == 2) claim();
        tile(__builtin_amdgcn_readfirstlane(t), claim);
        claim();                           // unless it has been made
        if (threadIdx.x == 0) s_li[k] = next;
        __syncthreads();                   // (the two slots alternate, so one barrier a tile is enough)
        const int li = __builtin_amdgcn_readfirstlane(s_li[k]);
        if (li >= n) return;
        t = B.tiles[li];
    }
}

// ---------------------------------------------------------------------------------------
// NW waves share a tile in a scatter: each takes a run of the tile's cells, in sorted order, that is a
// layer z or half of one in 3D (NW = 4 or 8) and two rows y in 2D (NW = 4). The wave's copy of the
// footprint covers the planes and rows that its cells reach.
template <int DIM, int NW> struct WaveFoot {
    using G = TileGeom<DIM>;
    static constexpr int RW = DIM == 3 ? G::TY * G::TZ / NW : G::TY / NW;       // rows of cells per wave
    static_assert(RW > 0 && G::TY % RW == 0 && RW * NW == (DIM == 3 ? G::TY * G::TZ : G::TY), "whole rows of a layer");
    static constexpr int WPZ = G::TY / RW;                                      // waves per layer (3D)
    static constexpr int WX = G::FX, WY = RW + 3, WZ = DIM == 3 ? 4 : 1;
    static constexpr int PLANE = WX * WY;
    static constexpr int SIZE = PLANE * WZ;
    // first footprint row and plane of wave w
    static __device__ __forceinline__ int y0(int w) { return DIM == 3 ? w % WPZ * RW : w * RW; }
    static __device__ __forceinline__ int z0(int w) { return DIM == 3 ? w / WPZ : 0; }
};

// Scatters on the matrix cores. A cell's sums over its particles at the candidate nodes are a
// contraction: with per-axis factors X, Y, Z and a payload u_q, node (ix, iy, iz) of component q
// gains sum_p (X_p[ix] Y_p[iy]) (Z_p[iz] u_pq), a 16 x K by K x 16 product over the cell's particles
// with rows (iy, ix) and columns (iz, q): v_mfma_f64_16x16x4 for four particles at a time, with four
// LDS reads and two multiplications, where a lane per node read seven words and issued six FP64
// operations for each particle. In 2D the columns are the components alone: v_mfma_f64_4x4x4, whose
// four blocks take the rows iy. Sums keep a fixed order: a matrix instruction adds its four products
// one after another (measured equal to a chain of FMAs bit for bit; a missing fourth adds zero), a
// cell takes its particles in upload order, and a cell's result is added to the wave's own LDS copy,
// one address per lane, by LDS additions that a wave issues in cell order; the copies are added in
// wave order. Every node value is therefore the same on every run.
//
// A wave works on its own: it takes its particles 64 at a time (a lane each for the loads and the
// shape factors), stages their factors in its own LDS rows and scatters its own cells, so no barrier
// stands between loads, factors and sums and the waves of a CU overlap them. The rows hold WREC
// records, so that three blocks fit in a CU's LDS. On the 128^3 J2 block (kernel traces of 205 steps) the
// mass scatter went from 0.60 to 0.30 ms per launch, the force scatter from 0.76 to 0.45 and the particle
// update from 0.86 to 0.48; on 202k lCPDI particles from 0.147, 0.196 and 0.245 to 0.116, 0.091 and 0.115.
typedef double mat4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void lds_add(double *a, double v) {
    __hip_atomic_fetch_add(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// LDS words written by some lanes of a wave are read by others: a wave's LDS instructions execute in
// order, so only the compiler has to keep them so
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The cells of a wave taken one after another as their particles are staged. bounds: lane it holds the
// start of the wave's it-th cell, lane it + ITS its end; it: the cell reached; open: its sums (in the
// caller's registers) have begun; at: its offset in the wave's copy.
template <int DIM, int NW> struct WaveCells {
    static constexpr int ITS = TileGeom<DIM>::NC / NW;
    static_assert(ITS <= 32, "bounds held by the lanes of a wave");
    int bounds, it, at;
    bool open;
    int b, e;                   // the wave's particles: sorted slots b..e-1
    // starts: the tile's cells' first sorted slots, and the next tile's first
    __device__ __forceinline__ void begin(const int *starts) {
        const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
        bounds = starts[w * ITS + l % ITS + (l / ITS > 0 ? 1 : 0)];
        it = 0;
        open = false;
        b = start(0);
        e = end(ITS - 1);
    }
    // the particle of sorted slot k (none beyond the wave's)
    __device__ __forceinline__ int particle(const KBins &B, int k) const { return k < e ? B.order[k] : -1; }
    __device__ __forceinline__ int start(int i) const { return __builtin_amdgcn_readlane(bounds, i); }
    __device__ __forceinline__ int end(int i) const { return __builtin_amdgcn_readlane(bounds, i + ITS); }
};

// visits the cells with particles among the staged slots r0..r1-1: first(kb, ke, open) begins a cell
// with particles kb..ke-1 of them (open: the one before it still has to be added to the copy),
// more(kb, ke) goes on with one that an earlier round began
template <int DIM, int NW, typename First, typename More>
__device__ __forceinline__ void wave_walk(WaveCells<DIM, NW> &W, int r0, int r1, First first, More more) {
    using G = TileGeom<DIM>;
    while (W.it < WaveCells<DIM, NW>::ITS) {
        const int s = W.start(W.it), e = W.end(W.it);
        if (s >= r1) break;
        const int kb = max(s, r0) - r0, ke = min(e, r1) - r0;
        if (kb < ke) {
            if (s < r0 && W.open) more(kb, ke);
            else {
                first(kb, ke, W.open);
                W.open = true;
                W.at = (W.it / G::TX) * WaveFoot<DIM, NW>::WX + W.it % G::TX;
            }
        }
        if (e > r1) break;
        W.it++;
    }
}

// Mass- and momentum-like sums of NQ components. S: rows STR apart, 4*DIM of factors [axis*4 + candidate]
// [record] and NQ of payload [q][record], rounded up to fours (a row beyond NQ is read and its result
// dropped). Four components are one 16x16x4 product, up to eight are two with the same rows. A
// particle has PPR records: itself, or its lCPDI corners (a corner's linear functions are a product of
// axis factors too, zero at the candidates its element lacks). A cell's first records are read before
// the cell before it is added to the copy, so the reads pass over the matrix instructions' latency.
struct NoExtra {
    template <typename... T> __device__ __forceinline__ void operator()(T &&...) const {}
};
template <int DIM> struct MatSums { typedef mat4d T; };     // of one component block of a cell, per lane
template <> struct MatSums<2> { typedef double T; };

// CUT: the records are lCPDI corners, and products below the limit are left out. In 2D these are the rows'
// products. In 3D a quad of records with such a product (a bit of cut per record) is folded twice, with its
// odd and its even candidates of the z axis in turn: of two neighbouring nodes one is each, so a record has
// one factor along z in either turn, and with it what is left out of a row is known. A column's sum takes
// the same products in the same order as in one turn, and zeros in the other. The mass scatter of 85k
// particles takes 47 us with corners anywhere and 51 in a block whose corners lie on cell edges, where
// half of the quads are folded twice, for 42 without; done in every scatter it took a contact step on
// 150k particles from 645 to 780 us (in the mass scatter alone: to 655).
template <int DIM, int NW, int NQ, int PPR, int STR, bool CUT = false> struct WaveScatter {
    using F = WaveFoot<DIM, NW>;
    static constexpr int NB = (NQ + 3) / 4;
    const double *plo, *phi;    // this lane's record of a quad in the rows of its lo and hi candidate
    double *acc;
    int k4, lo, hi;
    unsigned cut;               // 3D corners: the staged records with a product to leave out
    typename MatSums<DIM>::T c[NB];
    struct Quad { double x, y, z, v[NB]; };
    __device__ __forceinline__ void begin(const double *S, double (*s_acc)[NQ][F::SIZE]) {
        const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
        lo = l & 3;
        hi = (l >> 2) & 3;
        k4 = l >> 4;
        plo = S + lo * STR + k4;
        phi = S + hi * STR + k4;
        // 3D: result register r, lane l: node (ix = k4, iy = r, iz = hi) of component lo (block 1: 4 + lo);
        // 2D: lane l: node (ix = k4, iy = hi)
        acc = &s_acc[w][lo < NQ ? lo : 0][hi * (DIM == 3 ? F::PLANE : F::WX) + k4];
    }
    __device__ __forceinline__ Quad read(int k) const {
        Quad t;
        t.x = plo[k]; t.y = phi[4 * STR + k];
        t.z = DIM == 3 ? phi[8 * STR + k] : 1.;
#pragma unroll
        for (int b = 0; b < NB; b++) t.v[b] = plo[(4 * DIM + 4 * b) * STR + k];
        return t;
    }
    // records k..k+3 of a cell whose records end before e; those beyond the end count as zero
    __device__ __forceinline__ Quad load(int k, int e) const {
        if (PPR % 4 == 0 || k + 4 <= e) return read(k);
        Quad t = read(min(k + k4, e - 1) - k4);
        t.x = k + k4 < e ? t.x : 0.;
        return t;
    }
    __device__ __forceinline__ void fold(const Quad &t, int k) {
        double a = t.x * t.y, tz = t.z;
        if constexpr (CUT && DIM == 2) a = a < CornerLimit<2>::V ? 0. : a;
        if constexpr (CUT && DIM == 3) {
            if (cut >> k & 15u) {
                int l = threadIdx.x;
                asm volatile("" : "+v"(l));                   // formed here, not held over the cells
                const bool oddCol = l & 4;
                const double *z = plo + (8 - (l & 3)) * STR + k;
                const double odd = z[STR] + z[3 * STR];
                const double ao = a * odd < CornerLimit<3>::V ? 0. : a, zo = oddCol ? tz : 0.;
#pragma unroll
                for (int b = 0; b < NB; b++) c[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(ao, zo * t.v[b], c[b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                const double even = z[0] + z[2 * STR];
                a = a * even < CornerLimit<3>::V ? 0. : a;
                tz = oddCol ? 0. : tz;
            }
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if constexpr (DIM == 3) c[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, tz * t.v[b], c[b], 0, 0, 0);
            else c[b] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, t.v[b], c[b], 0, 0, 0);
        }
    }
    __device__ __forceinline__ void flush(int at) const {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (4 * b + lo >= NQ) continue;
            double *p = acc + b * 4 * F::SIZE + at;
            if constexpr (DIM == 3) {
#pragma unroll
                for (int r = 0; r < 4; r++) lds_add(p + r * F::WX, c[b][r]);
            } else lds_add(p, c[b]);
        }
    }
    // particles r0..r1-1 are staged, from record 0; extra(kb, ke, lo, hi, k4, c) after each cell's sums
    template <typename Extra> __device__ __forceinline__ void scatter(WaveCells<DIM, NW> &W, int r0, int r1, Extra extra) {
        auto add = [&](int k, int e) {
#pragma unroll 1
            for (; k < e; k += 4) fold(load(k, e), k);
        };
        wave_walk(W, r0, r1,
            [&](int kb, int ke, bool open) {
                const Quad t0 = load(kb * PPR, ke * PPR);
                if (open) flush(W.at);
#pragma unroll
                for (int b = 0; b < NB; b++) c[b] = typename MatSums<DIM>::T{};
                fold(t0, kb * PPR);
                add(kb * PPR + 4, ke * PPR);
                extra(kb, ke, lo, hi, k4, c[0]);
            },
            [&](int kb, int ke) {
                add(kb * PPR, ke * PPR);
                extra(kb, ke, lo, hi, k4, c[0]);
            });
    }
    __device__ __forceinline__ void scatter(WaveCells<DIM, NW> &W, int r0, int r1) { scatter(W, r0, r1, NoExtra()); }
    __device__ __forceinline__ void finish(const WaveCells<DIM, NW> &W) const {
        if (W.open) flush(W.at);
    }
};

// The force scatter's sums: node (ix, iy, iz) of component q gains, per particle,
// a_q0 X'YZ + a_q1 XY'Z + a_q2 XYZ' (the rows of the symmetric a: xx, yy, xy, zz, xz, yz): three of the
// products above, with rows X'Y, XY' and XY and columns Z a_q0, Z a_q1 and Z' a_q2 (2D: two). F: 4*DIM
// rows of (factor, derivative) pairs [axis*4 + candidate][record]; a: the terms' rows; both STR apart.
// With loads (FX) e holds 3 rows of pFext, added times XYZ, and trac adds a particle's own nodal forces.
template <int DIM, int NW, bool FX, int STR> struct WaveForce {
    using F = WaveFoot<DIM, NW>;
    const double2 *flo, *fhi;
    const double *a0, *a1, *a2, *eq;
    double *acc;
    int k4, q, hi;
    bool on;
    typename MatSums<DIM>::T c;
    struct Quad { double2 x, y, z; double a0, a1, a2, e; };
    __device__ __forceinline__ void begin(const double2 *S, const double *a, const double *e, double (*s_acc)[NQ_FORCE][F::SIZE]) {
        const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
        const int lo = l & 3;
        hi = (l >> 2) & 3;
        k4 = l >> 4;
        on = lo < DIM;
        q = on ? lo : 0;
        flo = S + lo * STR + k4;
        fhi = S + hi * STR + k4;
        a0 = a + (q == 0 ? 0 : q == 1 ? 2 : 4) * STR + k4;
        a1 = a + (q == 0 ? 2 : q == 1 ? 1 : 5) * STR + k4;
        a2 = a + (DIM == 2 ? 0 : q == 0 ? 4 : q == 1 ? 5 : 3) * STR + k4;
        eq = FX ? e + q * STR + k4 : nullptr;
        // 3D: result register r, lane l: node (ix = k4, iy = r, iz = hi); 2D: lane l: node (ix = k4, iy = hi)
        acc = &s_acc[w][q][hi * (DIM == 3 ? F::PLANE : F::WX) + k4];
    }
    __device__ __forceinline__ Quad read(int k) const {
        Quad t;
        t.x = flo[k]; t.y = fhi[4 * STR + k];
        if (DIM == 3) { t.z = fhi[8 * STR + k]; t.a2 = a2[k]; }
        t.a0 = a0[k]; t.a1 = a1[k];
        t.e = FX ? eq[k] : 0.;
        return t;
    }
    __device__ __forceinline__ Quad load(int k, int e) const {
        if (k + 4 <= e) return read(k);
        Quad t = read(min(k + k4, e - 1) - k4);
        if (k + k4 >= e) t.x = make_double2(0., 0.);
        return t;
    }
    __device__ __forceinline__ void fold(const Quad &t) {
        if constexpr (DIM == 3) {
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x.y * t.y.x, t.z.x * t.a0, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x.x * t.y.y, t.z.x * t.a1, c, 0, 0, 0);
            const double b = FX ? fma(t.z.x, t.e, t.z.y * t.a2) : t.z.y * t.a2;
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x.x * t.y.x, b, c, 0, 0, 0);
        } else {
            c = __builtin_amdgcn_mfma_f64_4x4x4f64(t.x.y * t.y.x, t.a0, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f64_4x4x4f64(t.x.x * t.y.y, t.a1, c, 0, 0, 0);
            if (FX) c = __builtin_amdgcn_mfma_f64_4x4x4f64(t.x.x * t.y.x, t.e, c, 0, 0, 0);
        }
    }
    __device__ __forceinline__ void flush(int at) const {
        if (!on) return;
        if constexpr (DIM == 3) {
#pragma unroll
            for (int r = 0; r < 4; r++) lds_add(acc + at + r * F::WX, c[r]);
        } else lds_add(acc + at, c);
    }
    template <typename Trac> __device__ __forceinline__ void scatter(WaveCells<DIM, NW> &W, int r0, int r1, Trac trac) {
        auto add = [&](int k, int e) {
#pragma unroll 1
            for (; k < e; k += 4) fold(load(k, e));
        };
        wave_walk(W, r0, r1,
            [&](int kb, int ke, bool open) {
                const Quad t = load(kb, ke);
                if (open) flush(W.at);
                c = typename MatSums<DIM>::T{};
                fold(t);
                add(kb + 4, ke);
                if (FX) trac(kb, ke, q, hi, k4, c);
            },
            [&](int kb, int ke) {
                add(kb, ke);
                if (FX) trac(kb, ke, q, hi, k4, c);
            });
    }
    __device__ __forceinline__ void finish(const WaveCells<DIM, NW> &W) const {
        if (W.open) flush(W.at);
    }
};

// The contact sums of uGIMP and classic particles: volume and displacement as the mass scatter's components,
// and the volume gradient as the force scatter's with Vp alone (component q takes the derivative along q),
// four products (2D: three) for four particles. F: rows of pairs as in WaveForce; U: 4 rows, the volume and
// the displacement's components. A lane per node took 82 us per launch on 202k particles in 3D and 32 on
// 192k in 2D; four records a particle (its factors, and each axis's derivative in turn beside the others'
// factors), two products each and eight particles a round, 96 and 39; this takes 48 and 18. Bit for bit the
// sums of the four records: a component's terms come in the same order, without the zeros between.
template <int DIM, int NW, int STR> struct WaveContact {
    using F = WaveFoot<DIM, NW>;
    const double2 *flo, *fhi;
    const double *ulo;
    double *acc;
    int k4, lo;
    typename MatSums<DIM>::T c[2];
    struct Quad { double2 x, y, z; double u, v; };
    __device__ __forceinline__ void begin(const double2 *S, const double *U, double (*s_acc)[NQ_CONTACT][F::SIZE]) {
        const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
        const int hi = (l >> 2) & 3;
        lo = l & 3;
        k4 = l >> 4;
        flo = S + lo * STR + k4;
        fhi = S + hi * STR + k4;
        ulo = U + lo * STR + k4;
        // nodes as in WaveScatter
        acc = &s_acc[w][lo][hi * (DIM == 3 ? F::PLANE : F::WX) + k4];
    }
    __device__ __forceinline__ Quad load(int k, int e) const {
        const bool in = k + k4 < e;
        const int at = in ? k : e - 1 - k4;
        Quad t;
        t.x = flo[at]; t.y = fhi[4 * STR + at];
        t.z = DIM == 3 ? fhi[8 * STR + at] : make_double2(1., 0.);
        t.u = ulo[at]; t.v = ulo[at - lo * STR];
        if (!in) t.x = make_double2(0., 0.);
        return t;
    }
    __device__ __forceinline__ void fold(const Quad &t) {
        const double v0 = lo == 0 ? t.v : 0., v1 = lo == 1 ? t.v : 0., v2 = lo == 2 ? t.v : 0.;
        if constexpr (DIM == 3) {
            c[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x.x * t.y.x, t.z.x * t.u, c[0], 0, 0, 0);
            c[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x.y * t.y.x, t.z.x * v0, c[1], 0, 0, 0);
            c[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x.x * t.y.y, t.z.x * v1, c[1], 0, 0, 0);
            c[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x.x * t.y.x, t.z.y * v2, c[1], 0, 0, 0);
        } else {
            c[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(t.x.x * t.y.x, t.u, c[0], 0, 0, 0);
            c[1] = __builtin_amdgcn_mfma_f64_4x4x4f64(t.x.y * t.y.x, v0, c[1], 0, 0, 0);
            c[1] = __builtin_amdgcn_mfma_f64_4x4x4f64(t.x.x * t.y.y, v1, c[1], 0, 0, 0);
        }
    }
    __device__ __forceinline__ void flush(int at) const {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            if (b == 1 && lo >= DIM) continue;
            double *p = acc + b * 4 * F::SIZE + at;
            if constexpr (DIM == 3) {
#pragma unroll
                for (int r = 0; r < 4; r++) lds_add(p + r * F::WX, c[b][r]);
            } else lds_add(p, c[b]);
        }
    }
    __device__ __forceinline__ void scatter(WaveCells<DIM, NW> &W, int r0, int r1) {
        auto add = [&](int k, int e) {
#pragma unroll 1
            for (; k < e; k += 4) fold(load(k, e));
        };
        wave_walk(W, r0, r1,
            [&](int kb, int ke, bool open) {
                const Quad t = load(kb, ke);
                if (open) flush(W.at);
                c[0] = c[1] = typename MatSums<DIM>::T{};
                fold(t);
                add(kb + 4, ke);
            },
            [&](int kb, int ke) { add(kb, ke); });
    }
    __device__ __forceinline__ void finish(const WaveCells<DIM, NW> &W) const {
        if (W.open) flush(W.at);
    }
};

// a wave's own copy (the wave's later LDS instructions follow in order)
template <int DIM, int NW, int NQ>
__device__ __forceinline__ void zero_wave_acc(double (*s_acc)[NQ][(WaveFoot<DIM, NW>::SIZE)]) {
    double *a = &s_acc[threadIdx.x >> 6][0][0];
    for (int i = threadIdx.x & 63; i < NQ * WaveFoot<DIM, NW>::SIZE; i += 64) a[i] = 0.;
    wave_sync();
}

// add the wave copies that cover each footprint node in wave order and store the tile's sums
template <int DIM, int NW, int NQ>
__device__ __forceinline__ void write_partials(const KNodes &N, int t, double (*s_acc)[NQ][WaveFoot<DIM, NW>::SIZE]) {
    using G = TileGeom<DIM>;
    using W = WaveFoot<DIM, NW>;
    for (int s = threadIdx.x; s < G::FOOT; s += 64 * NW) {
        const int x = s % G::FX, y = DIM == 3 ? s / G::FX % G::FY : s / G::FX, z = DIM == 3 ? s / (G::FX * G::FY) : 0;
        // every copy is read (a read in place of those that lack the node), so the reads are in flight together
        int at[NW];
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const int r = y - W::y0(w), c = z - W::z0(w);
            at[w] = r < 0 || r >= W::WY || c < 0 || c >= W::WZ ? -1 : c * W::PLANE + r * W::WX + x;
        }
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            double a[NW], v = 0.;
#pragma unroll
            for (int w = 0; w < NW; w++) a[w] = s_acc[w][q][at[w] < 0 ? 0 : at[w]];
#pragma unroll
            for (int w = 0; w < NW; w++) v = at[w] < 0 ? v : v + a[w];
            N.part[((size_t)t * NQMAX + q) * G::FOOT + s] = v;
        }
    }
}

// ---------------------------------------------------------------------------------------
// P2G #1: mass and momentum (MassAndMomentumTask -> NodalPoint::AddMassMomentum,
// NodalPointMPM.cpp:419-453). The point count of a node is not summed: every particle has
// mp > 0 and every in-support weight is > 0, so numberPoints > 0 exactly when the mass is > 0.

// uGIMP and classic: the words of a lane's particle that the mass scatter and the particle update need
template <int DIM> struct MassWords { int p, key; double x[DIM], m, v[DIM]; };

template <int DIM>
__device__ __forceinline__ void load_mass_words(const KPart &rows, const KBins &B, int p, MassWords<DIM> &t) {
    const KPart P = local_rows(rows);
    t.p = p;
    if (t.p < 0) return;
    t.key = B.key[t.p];
#pragma unroll
    for (int a = 0; a < DIM; a++) {
        t.x[a] = P.f(MPF_POS_X + a)[t.p];
        t.v[a] = P.f(MPF_VEL_X + a)[t.p];
    }
    t.m = P.f(MPF_MASS)[t.p];
}

// a particle's factor rows and payload at record i of its wave's rows
template <int DIM, int NU>
__device__ __forceinline__ void stage_factors(double (*S)[WROW], int i, const AxisFactors f[DIM], const double u[NU]) {
#pragma unroll
    for (int a = 0; a < DIM; a++) {
        AxisFactors t = f[a];
        asm volatile("" : "+v"(t.w));          // formed here, not held from before the rounds
#pragma unroll
        for (int o = 0; o < 4; o++) S[a * 4 + o][i] = t.s4(o);
    }
#pragma unroll
    for (int q = 0; q < NU; q++) S[4 * DIM + q][i] = u[q];
}

template <int DIM>
__global__ __launch_bounds__(64 * UGIMP_NW, WAVES4) void k_p2g_mass(KGrid g0, KPart P, KBins B, KNodes N) {
    using G = TileGeom<DIM>;
    constexpr int NW = UGIMP_NW;
    __shared__ double s_S[NW][4 * DIM + 4][WROW];       // per wave: [axis*4 + offset][record], then mass and momentum
    __shared__ double s_acc[NW][NQ_MASS][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        const int tc = tall % g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveScatter<DIM, NW, NQ_MASS, 1, WROW> sc;
        sc.begin(&s_S[w][0][0], s_acc);
        MassWords<DIM> cur;
        int ahead = W.particle(B, W.b + 64 + l);       // the order is read a round before the words
        load_mass_words<DIM>(P, B, W.particle(B, W.b + l), cur);
        zero_wave_acc<DIM, NW, NQ_MASS>(s_acc);
        for (int r = W.b; r < W.e; r += 64) {
            AxisFactors f[DIM];
            double u[4];
            if (cur.p >= 0) {
                int lx, ly, lz;
                double invd[DIM];
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                particle_axes<DIM>(gp, P, cur.p, ox + lx, oy + ly, oz + lz, cur.x, f, invd);
                u[0] = cur.m;
#pragma unroll
                for (int a = 0; a < 3; a++) u[1 + a] = a < DIM ? cur.m * cur.v[a < DIM ? a : 0] : 0.;
            }
            for (int r0 = r; r0 < min(r + 64, W.e); r0 += WREC) {
                if (l / WREC == (r0 - r) / WREC && cur.p >= 0) stage_factors<DIM, 4>(s_S[w], l % WREC, f, u);
                // the next particles' loads pass over the last scatter
                if (r0 + WREC >= min(r + 64, W.e)) {
                    load_mass_words<DIM>(P, B, ahead, cur);
                    ahead = W.particle(B, r + 2 * 64 + l);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC, W.e));
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_MASS>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// strains and rotations in the order of get_F3 (2D: those out of the plane are zero)
template <int DIM>
__device__ __forceinline__ void load_deformation(const KPart &P, int p, double ep[6], double wr[3]) {
#pragma unroll
    for (int a = 0; a < 6; a++) ep[a] = DIM == 3 || a < 3 || a == 5 ? P.f(MPF_EP_XX + a)[p] : 0.;
#pragma unroll
    for (int a = 0; a < 3; a++) wr[a] = DIM == 3 || a == 2 ? P.f(MPF_WR_YZ + a)[p] : 0.;
}

// lCPDI: the words of a lane's particle; F gives the semi-side vectors of the step
template <int DIM> struct CornerMassWords { int p, key; double x[DIM], m, v[DIM], ep[6], wr[3]; };

template <int DIM>
__device__ __forceinline__ void load_corner_mass(const KPart &rows, const KBins &B, int p, CornerMassWords<DIM> &t) {
    const KPart P = local_rows(rows);
    t.p = p;
    if (t.p < 0) return;
    t.key = B.key[t.p];
#pragma unroll
    for (int a = 0; a < DIM; a++) {
        t.x[a] = P.f(MPF_POS_X + a)[t.p];
        t.v[a] = P.f(MPF_VEL_X + a)[t.p];
    }
    load_deformation<DIM>(P, t.p, t.ep, t.wr);
    t.m = P.f(MPF_MASS)[t.p];
}

template <int DIM>
__global__ __launch_bounds__(64 * CORNER_NW(DIM), WAVES8) void k_p2g_mass_corners(KGrid g0, KPart P, KBins B, KNodes N, KStats st) {
    using G = TileGeom<DIM>;
    constexpr int NW = CORNER_NW(DIM);
    __shared__ double s_S[NW][4 * DIM + 4][WROW];       // per wave: [axis*4 + offset][corner], then mass and momentum over 64
    __shared__ double s_acc[NW][NQ_MASS][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l / Corners<DIM>::N, c = l % Corners<DIM>::N;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        const int tc = tall % g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveScatter<DIM, NW, NQ_MASS, Corners<DIM>::N, WROW, true> sc;
        sc.begin(&s_S[w][0][0], s_acc);
        CornerMassWords<DIM> cur;
        int ahead = W.particle(B, W.b + Corners<DIM>::PB + i);       // the order is read a round before the words
        load_corner_mass<DIM>(P, B, W.particle(B, W.b + i), cur);
        zero_wave_acc<DIM, NW, NQ_MASS>(s_acc);
        for (int r = W.b; r < W.e; r += Corners<DIM>::PB) {
            double xi[3], u[4];
            int off[3];
            bool ok = true;
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                // InitializationTask -> GetCPDINodesAndWeights: semi-side vectors of the step (each
                // corner's lane builds them; the first keeps them for the step's other passes)
                double s[9];
                cpdi_semi_sides_of<DIM>(g, P, cur.p, ox + lx, oy + ly, oz + lz, cur.ep, cur.wr, s);
                ok = corner_lane<DIM>(gp, cur.x, s, ox + lx, oy + ly, oz + lz, c, xi, off);
                if (c == 0) {
#pragma unroll
                    for (int a = 0; a < 9; a++) P.cpr(a)[cur.p] = s[a];
                }
                u[0] = Corners<DIM>::WW * cur.m;
#pragma unroll
                for (int a = 0; a < 3; a++) u[1 + a] = a < DIM ? u[0] * cur.v[a < DIM ? a : 0] : 0.;
            }
            // one count per particle with an unusable corner
            const unsigned long long bad = __ballot(!ok);
            if (c == 0 && ((bad >> l) & ((1ull << Corners<DIM>::N) - 1))) atomicAdd(st.cpdiErr, 1ull);
            for (int r0 = r; r0 < min(r + Corners<DIM>::PB, W.e); r0 += WREC / Corners<DIM>::N) {
                bool cut = false;
                if (l / WREC == (r0 - r) / (WREC / Corners<DIM>::N) && cur.p >= 0) {
                    stage_corner<DIM, 4>(s_S[w], l % WREC, xi, off, u);
                    if (DIM == 3) cut = corner_cut(xi);
                }
                const unsigned long long cuts = __ballot(cut);
                sc.cut = (unsigned)cuts | (unsigned)(cuts >> 32);       // (one half of the lanes is staged)
                // the next particles' loads pass over the last scatter
                if (r0 + WREC / Corners<DIM>::N >= min(r + Corners<DIM>::PB, W.e)) {
                    load_corner_mass<DIM>(P, B, ahead, cur);
                    ahead = W.particle(B, r + 2 * Corners<DIM>::PB + i);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC / Corners<DIM>::N, W.e));
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_MASS>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// sum the partials of the tiles that cover node (i,j,k), in fixed tile order
template <int DIM, int NQ>
__device__ __forceinline__ void gather_partials(const KGrid &g, const KBins &B, const KNodes &N, int fld, int i,
                                                int j, int k, double out[NQ]) {
    using G = TileGeom<DIM>;
    constexpr int NP = DIM == 3 ? 8 : 4;       // footprints overlap by less than a tile: two tiles an axis at most
    const int txh = min(g.ntx - 1, (i + 1) / G::TX), txl = i >= G::TX + 1 ? (i - 2) / G::TX : 0;
    const int tyh = min(g.nty - 1, (j + 1) / G::TY), tyl = j >= G::TY + 1 ? (j - 2) / G::TY : 0;
    int tzh = 0, tzl = 0;
    if (DIM == 3) { tzh = min(g.ntz - 1, (k + 1) / G::TZ); tzl = k >= G::TZ + 1 ? (k - 2) / G::TZ : 0; }
    // the flags of all the tiles, then the sums of those that have particles, are read together
    int t[NP];
    bool on[NP];
#pragma unroll
    for (int c = 0; c < NP; c++) {
        const int tx = txl + (c & 1), ty = tyl + (c >> 1 & 1), tz = tzl + (c >> 2);
        const bool in = tx <= txh && ty <= tyh && tz <= tzh;
        t[c] = (min(tz, tzh) * g.nty + min(ty, tyh)) * g.ntx + min(tx, txh) + g.tileBase + fld * g.tilesTotal;
        on[c] = in & (B.tileOn[t[c]] != 0);
    }
    double v[NP][NQ];
#pragma unroll
    for (int c = 0; c < NP; c++) {
#pragma unroll
        for (int q = 0; q < NQ; q++) v[c][q] = 0.;
        if (!on[c]) continue;
        const int fx = i - ((txl + (c & 1)) * G::TX - 1), fy = j - ((tyl + (c >> 1 & 1)) * G::TY - 1);   // slot in the footprint
        int s = fy * G::FX + fx;
        if (DIM == 3) s += (k - ((tzl + (c >> 2)) * G::TZ - 1)) * G::FX * G::FY;
#pragma unroll
        for (int q = 0; q < NQ; q++) v[c][q] = N.part[((size_t)t[c] * NQMAX + q) * G::FOOT + s];
    }
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        out[q] = v[0][q];
#pragma unroll
        for (int c = 1; c < NP; c++) out[q] += v[c][q];
    }
}

// Node passes visit the nodes of the (field, tile) pairs that a non-empty pair's footprint reached at
// this binning or the one before (tile_need): a node of any other pair was cleared when its pair
// last was visited, or was never written, so it is skipped and stays zero. A node's own pair is the
// tile holding it (the grid's last node row belongs to the last tile); the pairs whose footprints
// can reach it are that tile and its neighbours.
template <int DIM>
__device__ __forceinline__ bool node_needed(const KGrid &g, const KBins &B, int fld, int i, int j, int k) {
    using G = TileGeom<DIM>;
    const int tx = min(i / G::TX, g.ntx - 1), ty = min(j / G::TY, g.nty - 1);
    const int tz = DIM == 3 ? min(k / G::TZ, g.ntz - 1) : 0;
    return B.needAny[fld * g.tilesTotal + g.tileBase + (tz * g.nty + ty) * g.ntx + tx] != 0;
}

// node pass after P2G #1: mass, momentum, count and v = p/m (MatVelocityField.cpp:158-164,239-251)
template <int DIM>
__global__ void k_node_mass(KGrid g0, KBins B, KNodes N) {
    long long nall = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (nall >= g0.nstride * g0.nfields) return;
    const int fld = node_field(g0, nall);
    const long long ng = nall - (long long)fld * g0.nstride;
    const KGrid g = node_grid(g0, ng);
    const long long n = ng - g.nodeBase;
    if (n >= g.nnodes) return;                // padding between instances
    const KNodes Nf = field_view(g, N, fld);
    if (nall == 0 && N.clist) N.clist[0] = 0;   // contact-node list of the step (regression normals)
    int i, j, k;
    node_ijk(g, n, i, j, k);
    if (!node_needed<DIM>(g, B, fld, i, j, k)) return;
    double a[NQ_MASS];
    gather_partials<DIM, NQ_MASS>(g, B, N, fld, i, j, k, a);
    long long nn = g.nstride;
    Nf.mass[n] = a[0];
    Nf.pk[n] = a[1]; Nf.pk[nn + n] = a[2]; Nf.pk[2 * nn + n] = a[3];
    int cnt = a[0] > 0. ? 1 : 0;       // numberPoints > 0 <=> mass > 0 (all mp > 0)
    Nf.cnt[n] = cnt;
    double vx = 0., vy = 0., vz = 0.;
    if (cnt > 0 && a[0] != 0.) {
        double s = 1. / a[0];
        vx = s * a[1]; vy = s * a[2]; vz = s * a[3];
    }
    Nf.vk[n] = vx; Nf.vk[nn + n] = vy; Nf.vk[2 * nn + n] = vz;
    Nf.ftot[n] = 0.; Nf.ftot[nn + n] = 0.; Nf.ftot[2 * nn + n] = 0.;
}

// ---------------------------------------------------------------------------------------
// load the footprint node vectors of a tile into LDS (zero outside the grid)
template <int DIM, int NV>
__device__ __forceinline__ void load_foot(const KGrid &g, int ox, int oy, int oz, const double *src[NV],
                                          const long long stride[NV], double (*dst)[TileGeom<DIM>::FOOT]) {
    using G = TileGeom<DIM>;
    for (int s = threadIdx.x; s < G::FOOT; s += NT) {
        long long n = foot_node<DIM>(g, s, ox, oy, oz);
#pragma unroll
        for (int v = 0; v < NV; v++) dst[v][s] = n >= 0 ? src[v][n + stride[v]] : 0.;
    }
}

// lCPDI gathers corner by corner. A node's merged weight and gradient are sums over the corners
// whose element holds it, so a gather over the merged node list is the same sum taken
// corner by corner: sum_n w(n) v(n) = ws sum_c sum_j cfn_c(j) v(n_cj) and
// sum_n v(n) grad(n) = sum_c (sum_j cfn_c(j) v(n_cj)) wg_c, where j runs over the nodes of corner c's
// element (cfn below 1e-15 left out, as in the reference's list). Each corner is built on the fly.

// gradient weight of corner c: the reference's per-corner expressions (MatPoint3D.cpp:571-594,
// MatPoint2D.cpp:551-566) collected as (s3 r1 x r2 - s2 r1 x r3 + s1 r2 x r3) / (8 V) in 3D and
// (s1 r2y - s2 r1y, s2 r1x - s1 r2x) / (4 A) in 2D; inv = 1/(8 V) or 1/(4 A)
template <int DIM>
__device__ __forceinline__ void cpdi_wg(const double r[9], double inv, int c, double w[3]) {
    const int q = c & 3;
    const double s1 = (q == 1 || q == 2) ? 1. : -1.;
    const double s2 = q >= 2 ? 1. : -1.;
    if (DIM == 3) {
        const double s3 = c >= 4 ? 1. : -1.;
        const double *r1 = r, *r2 = r + 3, *r3 = r + 6;
        const double c12[3] = {r1[1] * r2[2] - r1[2] * r2[1], r1[2] * r2[0] - r1[0] * r2[2], r1[0] * r2[1] - r1[1] * r2[0]};
        const double c13[3] = {r1[1] * r3[2] - r1[2] * r3[1], r1[2] * r3[0] - r1[0] * r3[2], r1[0] * r3[1] - r1[1] * r3[0]};
        const double c23[3] = {r2[1] * r3[2] - r2[2] * r3[1], r2[2] * r3[0] - r2[0] * r3[2], r2[0] * r3[1] - r2[1] * r3[0]};
#pragma unroll
        for (int a = 0; a < 3; a++) w[a] = (s3 * c12[a] - s2 * c13[a] + s1 * c23[a]) * inv;
    } else {
        w[0] = (s1 * r[4] - s2 * r[1]) * inv;
        w[1] = (s2 * r[0] - s1 * r[3]) * inv;
        w[2] = 0.;
    }
}

// 1/(8 V) (3D) or 1/(4 A) (2D) of the particle domain with semi-side vectors r
template <int DIM>
__device__ __forceinline__ double cpdi_inv_measure(const double r[9]) {
    if (DIM == 3)
        return 1. / (8. * (r[0] * (r[4] * r[8] - r[5] * r[7]) + r[1] * (r[5] * r[6] - r[3] * r[8]) +
                           r[2] * (r[3] * r[7] - r[4] * r[6])));
    return 1. / (4. * (r[0] * r[4] - r[1] * r[3]));
}

// sum over the nodes of corner c's element of cfn * rows[v][node], footprint slots relative to the
// particle's cell (lx, ly, lz) in its tile
template <int DIM, int NV>
__device__ __forceinline__ void cpdi_corner_sum(const double xi[3], const int off[3], int lx, int ly, int lz,
                                                const double (*rows)[TileGeom<DIM>::FOOT], double out[NV]) {
#pragma unroll
    for (int v = 0; v < NV; v++) out[v] = 0.;
    constexpr int NN = DIM == 3 ? 8 : 4;
#pragma unroll
    for (int jn = 0; jn < NN; jn++) {
        const int q = jn & 3;
        const int jx = (q == 1 || q == 2) ? 1 : 0, jy = q >= 2 ? 1 : 0, jz = jn >= 4 ? 1 : 0;
        double cfn = cpdi_cfn<DIM>(xi, jx, jy, jz);
        cfn = cfn < 1e-15 ? 0. : cfn;
        const int sl = foot_slot<DIM>(lx + off[0] + jx, ly + off[1] + jy, DIM == 3 ? lz + off[2] + jz : 0);
#pragma unroll
        for (int v = 0; v < NV; v++) out[v] = fma(cfn, rows[v][sl], out[v]);
    }
}

// velocity gradient of one particle from footprint velocities over its support window
// (MatPoint3D::ExtrapVelocityGradient, MatPoint3D.cpp:62-94; MatPoint2D.cpp:57-89)
template <int DIM>
__device__ __forceinline__ void velocity_gradient(const int w[3], const double Sw[3][3], const double Dw[3][3], int lx,
                                                  int ly, int lz, const double (*s_v)[TileGeom<DIM>::FOOT],
                                                  double L[3][3]) {
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) L[a][b] = 0.;
    constexpr int NZ = DIM == 3 ? 3 : 1;
#pragma unroll 1
    for (int jz = 0; jz < NZ; jz++)
#pragma unroll
        for (int jy = 0; jy < 3; jy++)
#pragma unroll
            for (int jx = 0; jx < 3; jx++) {
                const int zz = DIM == 3 ? jz : 1;
                const double syz = Sw[1][jy] * Sw[2][zz], sxz = Sw[0][jx] * Sw[2][zz], sxy = Sw[0][jx] * Sw[1][jy];
                const double gx = Dw[0][jx] * syz, gy = Dw[1][jy] * sxz, gz = Dw[2][zz] * sxy;
                const int s = foot_slot<DIM>(lx + w[0] + jx - 1, ly + w[1] + jy - 1, DIM == 3 ? lz + w[2] + jz - 1 : 0);
                const double vx = s_v[0][s], vy = s_v[1][s];
                L[0][0] = fma(vx, gx, L[0][0]); L[0][1] = fma(vx, gy, L[0][1]);
                L[1][0] = fma(vy, gx, L[1][0]); L[1][1] = fma(vy, gy, L[1][1]);
                if (DIM == 3) {
                    const double vz = s_v[2][s];
                    L[0][2] = fma(vx, gz, L[0][2]); L[1][2] = fma(vy, gz, L[1][2]);
                    L[2][0] = fma(vz, gx, L[2][0]); L[2][1] = fma(vz, gy, L[2][1]); L[2][2] = fma(vz, gz, L[2][2]);
                }
            }
}

// Matrix3::Scale (Matrix3.cpp:410-424)
template <int DIM>
__device__ __forceinline__ void scale_gradient(double L[3][3], double f) {
    L[0][0] *= f; L[0][1] *= f; L[1][0] *= f; L[1][1] *= f; L[2][2] *= f;
    if (DIM == 3) { L[0][2] *= f; L[1][2] *= f; L[2][0] *= f; L[2][1] *= f; }
}

// velocity gradient of particle p from footprint velocities (lx,ly,lz = its cell in the tile):
// the support window of its shape functions, or lCPDI nodes in list order
template <int DIM, int SH>
__device__ __forceinline__ void particle_gradient(const KGrid &g, GridPtr gp, const KPart &P, int p, int ei, int ej, int ek,
                                                  int lx, int ly, int lz, const double (*s_v)[TileGeom<DIM>::FOOT],
                                                  double L[3][3]) {
    if (SH == MPMGPU_SHAPE_LCPDI) {
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = 0; b < 3; b++) L[a][b] = 0.;
        double r[9];
#pragma unroll
        for (int a = 0; a < 9; a++) r[a] = P.cpr(a)[p];
        const double pos[3] = {P.f(MPF_POS_X)[p], P.f(MPF_POS_Y)[p], DIM == 3 ? P.f(MPF_POS_Z)[p] : 0.};
        const double inv = cpdi_inv_measure<DIM>(r);
        constexpr int NCOR = DIM == 3 ? 8 : 4;
#pragma unroll 1
        for (int c = 0; c < NCOR; c++) {
            double xi[3], vc[3], w[3];
            int off[3];
            cpdi_corner<DIM>(g, pos, r, ei, ej, ek, c, xi, off);
            cpdi_corner_sum<DIM, 3>(xi, off, lx, ly, lz, s_v, vc);
            cpdi_wg<DIM>(r, inv, c, w);
#pragma unroll
            for (int a = 0; a < DIM; a++)
#pragma unroll
                for (int b = 0; b < DIM; b++) L[a][b] = fma(vc[a], w[b], L[a][b]);
        }
    } else {
        const double pos[3] = {P.f(MPF_POS_X)[p], P.f(MPF_POS_Y)[p], DIM == 3 ? P.f(MPF_POS_Z)[p] : 0.};
        AxisFactors f[DIM];
        double invd[DIM], Sw[3][3], Dw[3][3];
        int w[3];
        particle_axes<DIM>(gp, P, p, ei, ej, ek, pos, f, invd);
        particle_window<DIM>(f, invd, w, Sw, Dw);
        velocity_gradient<DIM>(w, Sw, Dw, lx, ly, lz, s_v, L);
    }
}

// IsoPlasticity: the plastic strain (alt rows) and the cumulative plastic strain alpha (hist0) grow
// together, and rotating a zero plastic strain keeps it zero, so a particle with alpha = 0 has
// zero plastic strain: its alt rows (and alpha) are neither read nor written until it yields.
// Upload checks that the state keeps to this.
__device__ __forceinline__ bool alt_rows(int type, double h0) {
    return type != MPMGPU_MAT_ISOPLASTICITY || h0 != 0.;
}

template <int DIM>
__device__ __forceinline__ void load_state(const KPart &rows, int p, int type, PState &s) {
    const KPart P = local_rows(rows);
    s.ep[0] = P.f(MPF_EP_XX)[p]; s.ep[1] = P.f(MPF_EP_YY)[p]; s.ep[2] = P.f(MPF_EP_ZZ)[p];
    s.ep[5] = P.f(MPF_EP_XY)[p]; s.wr[2] = P.f(MPF_WR_XY)[p];
    s.sp[0] = P.f(MPF_SP_XX)[p]; s.sp[1] = P.f(MPF_SP_YY)[p]; s.sp[2] = P.f(MPF_SP_ZZ)[p];
    s.sp[5] = P.f(MPF_SP_XY)[p];
    if (DIM == 3) {
        s.ep[3] = P.f(MPF_EP_YZ)[p]; s.ep[4] = P.f(MPF_EP_XZ)[p];
        s.wr[0] = P.f(MPF_WR_YZ)[p]; s.wr[1] = P.f(MPF_WR_XZ)[p];
        s.sp[3] = P.f(MPF_SP_YZ)[p]; s.sp[4] = P.f(MPF_SP_XZ)[p];
    } else {
        s.ep[3] = s.ep[4] = 0.; s.wr[0] = s.wr[1] = 0.; s.sp[3] = s.sp[4] = 0.;
    }
    s.P = 0.; s.h0 = 0.; s.h1 = 0.;
#pragma unroll
    for (int c = 0; c < 6; c++) s.alt[c] = 0.;
    if (type != MPMGPU_MAT_ISOTROPIC) {
        s.P = P.f(MPF_PRESSURE)[p];
        s.h0 = P.f(MPF_HIST0)[p];
        if (alt_rows(type, s.h0)) {
            s.alt[0] = P.f(MPF_ALT_XX)[p]; s.alt[1] = P.f(MPF_ALT_YY)[p]; s.alt[2] = P.f(MPF_ALT_ZZ)[p];
            s.alt[5] = P.f(MPF_ALT_XY)[p];
            if (DIM == 3) { s.alt[3] = P.f(MPF_ALT_YZ)[p]; s.alt[4] = P.f(MPF_ALT_XZ)[p]; }
        }
        if (type == MPMGPU_MAT_NEOHOOKEAN || type == MPMGPU_MAT_MOONEY) s.h1 = P.f(MPF_HIST1)[p];
    }
}

template <int DIM>
__device__ __forceinline__ void store_state(const KPart &rows, int p, int type, const PState &s) {
    const KPart P = local_rows(rows);
    P.f(MPF_EP_XX)[p] = s.ep[0]; P.f(MPF_EP_YY)[p] = s.ep[1]; P.f(MPF_EP_ZZ)[p] = s.ep[2];
    P.f(MPF_EP_XY)[p] = s.ep[5]; P.f(MPF_WR_XY)[p] = s.wr[2];
    P.f(MPF_SP_XX)[p] = s.sp[0]; P.f(MPF_SP_YY)[p] = s.sp[1]; P.f(MPF_SP_ZZ)[p] = s.sp[2];
    P.f(MPF_SP_XY)[p] = s.sp[5];
    if (DIM == 3) {
        P.f(MPF_EP_YZ)[p] = s.ep[3]; P.f(MPF_EP_XZ)[p] = s.ep[4];
        P.f(MPF_WR_YZ)[p] = s.wr[0]; P.f(MPF_WR_XZ)[p] = s.wr[1];
        P.f(MPF_SP_YZ)[p] = s.sp[3]; P.f(MPF_SP_XZ)[p] = s.sp[4];
    }
    if (type != MPMGPU_MAT_ISOTROPIC) {
        P.f(MPF_PRESSURE)[p] = s.P;
        if (alt_rows(type, s.h0)) {
            P.f(MPF_ALT_XX)[p] = s.alt[0]; P.f(MPF_ALT_YY)[p] = s.alt[1]; P.f(MPF_ALT_ZZ)[p] = s.alt[2];
            P.f(MPF_ALT_XY)[p] = s.alt[5];
            if (DIM == 3) { P.f(MPF_ALT_YZ)[p] = s.alt[3]; P.f(MPF_ALT_XZ)[p] = s.alt[4]; }
            P.f(MPF_HIST0)[p] = s.h0;
        }
        if (type == MPMGPU_MAT_NEOHOOKEAN || type == MPMGPU_MAT_MOONEY) P.f(MPF_HIST1)[p] = s.h1;
    }
}

// ---------------------------------------------------------------------------------------
// USF strain update, first half step (UpdateStrainsFirstTask::FullStrainUpdate,
// UpdateStrainsFirstTask.cpp:101-168 -> MatPoint3D::UpdateStrain, MatPoint3D.cpp:45-60). Bound by
// memory: 735 MB for 2.1M J2 particles in 0.148 ms, 5.0 TB/s, with three waves per SIMD (two: 0.154).
// The state is loaded before the gradient, which hides its latency (885k rubber particles: 123 and 120 us);
// lCPDI's gradient is long and its registers are worth more.
template <int DIM, int MAT, int SH>
__global__ __launch_bounds__(NT, MAT == MPMGPU_MAT_ISOTROPIC || MAT == MPMGPU_MAT_ISOPLASTICITY ? 3 : 2) void k_usf(KGrid g0, KPart P, KBins B, KNodes N, const MpmMaterial *mats,
                                               int only) {
    using G = TileGeom<DIM>;
    __shared__ double s_v[3][G::FOOT];
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        if (only >= 0 && g0.tileType[tall % g0.tilesTotal] != only) return;   // another launch's type
        const int fld = tall / g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tall - fld * g0.tilesTotal);
        const KGrid g = grid_copy(gp);
        const int t = tall - fld * g0.tilesTotal - g.tileBase;
        const KNodes Nf = field_view(g, N, fld);
        const int tb = const_int(B.cellStart + (size_t)tall * G::NC), te = const_int(B.cellStart + (size_t)(tall + 1) * G::NC);
        int ox, oy, oz;
        tile_origin<DIM>(g, t, ox, oy, oz);
        int p = tb + (int)threadIdx.x < te ? B.order[tb + threadIdx.x] : -1;
        {
            const double *src[3] = {Nf.vk, Nf.vk, Nf.vk};
            const long long st[3] = {0, g.nstride, 2 * g.nstride};
            load_foot<DIM, 3>(g, ox, oy, oz, src, st, s_v);
        }
        __syncthreads();
        for (int k = tb + threadIdx.x; k < te; k += NT, p = k < te ? B.order[k] : -1) {
            const int mat = P.mat[p];
            int lx, ly, lz;
            tile_cell<DIM>(B.key[p], tall, lx, ly, lz);
            const MpmMaterial &m = mats[mat];
            const int mtype = MAT ? MAT : m.type;
            PState s;
            if (SH != MPMGPU_SHAPE_LCPDI) load_state<DIM>(P, p, mtype, s);
            double L[3][3];
            particle_gradient<DIM, SH>(g, gp, P, p, ox + lx, oy + ly, oz + lz, lx, ly, lz, s_v, L);
            scale_gradient<DIM>(L, g.strainFirst);
            if (SH == MPMGPU_SHAPE_LCPDI) load_state<DIM>(P, p, mtype, s);
            constitutive<DIM, MAT>(L, m, s);
            store_state<DIM>(P, p, mtype, s);
        }
    };
    for_each_tile<DIM>(B, tile);
}

// internal-force scatter (GridForcesTask::Execute, GridForcesTask.cpp:40-153 ->
// MatPoint3D::GetFintPlusFext, MatPoint3D.cpp:248-270; MatPoint2D.cpp:242-263) with the stress
// just updated by k_usf; FX adds N * pFext of the loaded particles (pFext is zero otherwise)

// uGIMP and classic: the (factor, derivative) pairs of one particle at record i of its wave's rows
template <int DIM>
__device__ __forceinline__ void stage_pairs(double2 (*F)[WROW], int i, const AxisFactors f[DIM], const double invd[DIM]) {
#pragma unroll
    for (int a = 0; a < DIM; a++) {
        AxisFactors t = f[a];
        asm volatile("" : "+v"(t.w));          // formed here, not held from before the rounds (48 registers)
#pragma unroll
        for (int o = 0; o < 4; o++) F[a * 4 + o][i] = make_double2(t.s4(o), t.d4(o) * invd[a]);
    }
}

// and -mp times the stress terms (xx, yy, xy, zz, xz, yz of sigma - P; 2D: three)
template <int DIM>
__device__ __forceinline__ void stage_force(double2 (*F)[WROW], double (*A)[WROW], int i, const AxisFactors f[DIM],
                                            const double invd[DIM], const double s[6]) {
    stage_pairs<DIM>(F, i, f, invd);
#pragma unroll
    for (int c = 0; c < (DIM == 3 ? 6 : 3); c++) A[c][i] = s[c];
}

// lane (q, iz, ix) of a scatter adds the traction tables of a cell's staged particles to its nodes
__device__ __forceinline__ void add_tractions(const KLoads &L, const int *tt, int kb, int ke, int q, int iz, int ix,
                                              mat4d &c) {
    if (q > 2) return;
    for (int s = kb; s < ke; s++) {
        if (tt[s] < 0) continue;
        const double *tab = L.ttab + (size_t)(3 * tt[s] + q) * TRAC_NODES + iz * 16 + ix;
#pragma unroll
        for (int r = 0; r < 4; r++) c[r] += tab[r * 4];
    }
}

// 2D: lane (q, iy, ix)
__device__ __forceinline__ void add_tractions(const KLoads &L, const int *tt, int kb, int ke, int q, int iy, int ix,
                                              double &c) {
    if (q > 1) return;
    for (int s = kb; s < ke; s++)
        if (tt[s] >= 0) c += L.ttab[(size_t)(3 * tt[s] + q) * TRAC_NODES + iy * 4 + ix];
}

template <int DIM> struct ForceWords { int p, key; double x[DIM], m, pr, s[6]; };

template <int DIM>
__device__ __forceinline__ void load_force_words(const KPart &rows, const KBins &B, int p, ForceWords<DIM> &t) {
    const KPart P = local_rows(rows);
    t.p = p;
    if (t.p < 0) return;
    t.key = B.key[t.p];
#pragma unroll
    for (int a = 0; a < DIM; a++) t.x[a] = P.f(MPF_POS_X + a)[t.p];
    t.m = P.f(MPF_MASS)[t.p];
    t.pr = P.f(MPF_PRESSURE)[t.p];         // stays 0 for small-strain elastic particles
    t.s[0] = P.f(MPF_SP_XX)[t.p]; t.s[1] = P.f(MPF_SP_YY)[t.p]; t.s[2] = P.f(MPF_SP_XY)[t.p];
    if (DIM == 3) { t.s[3] = P.f(MPF_SP_ZZ)[t.p]; t.s[4] = P.f(MPF_SP_XZ)[t.p]; t.s[5] = P.f(MPF_SP_YZ)[t.p]; }
}

template <int DIM, bool FX>
__global__ __launch_bounds__(64 * UGIMP_NW, FX ? 2 : WAVES4) void k_p2g_force(KGrid g0, KPart P, KBins B, KNodes N, KLoads L,
                                                                       const int *loaded) {
    using G = TileGeom<DIM>;
    constexpr int NW = UGIMP_NW;
    __shared__ double2 s_F[NW][4 * DIM][WROW]; // per wave: [axis*4 + offset][record] (factor, derivative)
    __shared__ double s_a[NW][6][WROW];
    __shared__ double s_e[FX ? NW : 1][3][WROW];   // pFext of the staged particles
    __shared__ int s_tt[FX ? NW : 1][WREC];        // their traction tables (-1: none)
    __shared__ double s_acc[NW][NQ_FORCE][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        // with loads: the launch with the load term takes the marked tiles, the other the rest
        if (loaded && (loaded[tall] != 0) != FX) return;
        const int tc = tall % g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveForce<DIM, NW, FX, WROW> sc;
        sc.begin(&s_F[w][0][0], &s_a[w][0][0], &s_e[FX ? w : 0][0][0], s_acc);
        // tractions: lane (q, iz, ix), in 2D (q, iy, ix), adds the tables of the cell's particles to its nodes
        auto trac = [&](int kb, int ke, int q, int hi, int ix, auto &c) {
            if (L.nt == 0) return;
            add_tractions(L, s_tt[FX ? w : 0], kb, ke, q, hi, ix, c);
        };
        zero_wave_acc<DIM, NW, NQ_FORCE>(s_acc);
        int ahead = W.particle(B, W.b + l);
        for (int r = W.b; r < W.e; r += 64) {
            ForceWords<DIM> cur;        // (loading them a round ahead costs the registers of the third wave per SIMD)
            load_force_words<DIM>(P, B, ahead, cur);
            ahead = W.particle(B, r + 64 + l);
            AxisFactors f[DIM];
            double invd[DIM], s[6];
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                particle_axes<DIM>(gp, P, cur.p, ox + lx, oy + ly, oz + lz, cur.x, f, invd);
                s[0] = -cur.m * (cur.s[0] - cur.pr);
                s[1] = -cur.m * (cur.s[1] - cur.pr);
                s[2] = -cur.m * cur.s[2];
                if (DIM == 3) {
                    s[3] = -cur.m * (cur.s[3] - cur.pr);
                    s[4] = -cur.m * cur.s[4];
                    s[5] = -cur.m * cur.s[5];
                }
            }
            for (int r0 = r; r0 < min(r + 64, W.e); r0 += WREC) {
                if (l / WREC == (r0 - r) / WREC && cur.p >= 0) {
                    stage_force<DIM>(s_F[w], s_a[w], l % WREC, f, invd, s);
                    if constexpr (FX) {
                        // MatPtLoadBC's pFext of the particle (0 when it carries no load) and its traction table
                        const int q = L.map[B.home[cur.p]];
#pragma unroll
                        for (int c = 0; c < 3; c++) s_e[w][c][l % WREC] = q >= 0 ? L.fext[3 * q + c] : 0.;
                        s_tt[w][l % WREC] = q >= 0 && L.nt > 0 ? L.tslot[q] : -1;
                    }
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC, W.e), trac);
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_FORCE>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// The first strain half step and the internal forces of uGIMP and classic particles without loads, in one
// pass: nothing on the grid changes between the two, so a particle's words, cell and shape factors are
// taken once and the stress goes to the scatter from registers. The same operations in the same order as
// k_usf and k_p2g_force, to the bit (task by task, with profiling, loads or lCPDI those two run). Its LDS
// holds two blocks a CU where the two kernels have three, yet steps gain, apart and in one pass: 4k 2D
// elastic 66 and 63 us, 1.7M 2D 529 and 516, 74k J2 129 and 122.5, 885k neo-Hookean 568 and 542, 7.08M J2
// 3,341 and 3,254; only tiles that three blocks a CU take in one go and two do not lose (262k J2 with
// XPIC(2) 253 and 259; it is taken there too, as the launch does not know how many tiles hold particles).
// On the 128^3 J2 block it moves 2.7 GB in 0.974 ms, 2.75 TB/s: 249 to 254 registers and 61.6 KB of LDS leave
// two waves per SIMD. Three waves per SIMD hold the 2D laws without volume terms (1.7M: 516, two 530).
template <int DIM, int MAT>
__global__ __launch_bounds__(64 * UGIMP_NW, DIM == 2 && (MAT == MPMGPU_MAT_ISOTROPIC || MAT == MPMGPU_MAT_ISOPLASTICITY) ? 3 : 2)
void k_usf_force(KGrid g0, KPart P, KBins B, KNodes N, const MpmMaterial *mats, int only) {
    using G = TileGeom<DIM>;
    constexpr int NW = UGIMP_NW;
    __shared__ double s_v[3][G::FOOT];
    __shared__ double2 s_F[NW][4 * DIM][WROW]; // as in k_p2g_force
    __shared__ double s_a[NW][6][WROW];
    __shared__ double s_acc[NW][NQ_FORCE][WaveFoot<DIM, NW>::SIZE];
    static_assert(64 * NW == NT, "load_foot's threads");
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        if (only >= 0 && g0.tileType[tall % g0.tilesTotal] != only) return;   // another launch's type
        const int fld = tall / g0.tilesTotal;
        const int tc = tall - fld * g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        const KNodes Nf = field_view(g, N, fld);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveForce<DIM, NW, false, WROW> sc;
        sc.begin(&s_F[w][0][0], &s_a[w][0][0], nullptr, s_acc);
        int p = W.particle(B, W.b + l);
        {
            const double *src[3] = {Nf.vk, Nf.vk, Nf.vk};
            const long long st[3] = {0, g.nstride, 2 * g.nstride};
            load_foot<DIM, 3>(g, ox, oy, oz, src, st, s_v);
        }
        zero_wave_acc<DIM, NW, NQ_FORCE>(s_acc);
        __syncthreads();
        for (int r = W.b; r < W.e; r += 64) {
            AxisFactors f[DIM];
            double invd[DIM], a[6];
            if (p >= 0) {
                const int mat = P.mat[p];
                int lx, ly, lz;
                tile_cell<DIM>(B.key[p], tall, lx, ly, lz);
                double pos[3];
#pragma unroll
                for (int c = 0; c < 3; c++) pos[c] = c < DIM ? P.f(MPF_POS_X + c)[p] : 0.;
                const double nm = -P.f(MPF_MASS)[p];
                const MpmMaterial &m = mats[mat];
                const int mtype = MAT ? MAT : m.type;
                // (stays 0 for small-strain elastic particles, whose law does not touch it)
                double pr = mtype == MPMGPU_MAT_ISOTROPIC ? P.f(MPF_PRESSURE)[p] : 0.;
                PState s;
                load_state<DIM>(P, p, mtype, s);
                double L[3][3];
                {
                    double Sw[3][3], Dw[3][3];
                    int wd[3];
                    particle_axes<DIM>(gp, P, p, ox + lx, oy + ly, oz + lz, pos, f, invd);
                    particle_window<DIM>(f, invd, wd, Sw, Dw);
                    velocity_gradient<DIM>(wd, Sw, Dw, lx, ly, lz, s_v, L);
                }
                scale_gradient<DIM>(L, g.strainFirst);
                constitutive<DIM, MAT>(L, m, s);
                store_state<DIM>(P, p, mtype, s);
                if (mtype != MPMGPU_MAT_ISOTROPIC) pr = s.P;
                a[0] = nm * (s.sp[0] - pr);
                a[1] = nm * (s.sp[1] - pr);
                a[2] = nm * s.sp[5];
                if (DIM == 3) {
                    a[3] = nm * (s.sp[2] - pr);
                    a[4] = nm * s.sp[4];
                    a[5] = nm * s.sp[3];
                }
            }
            for (int r0 = r; r0 < min(r + 64, W.e); r0 += WREC) {
                if (l / WREC == (r0 - r) / WREC && p >= 0) stage_force<DIM>(s_F[w], s_a[w], l % WREC, f, invd, a);
                if (r0 + WREC >= min(r + 64, W.e)) p = W.particle(B, r + 64 + l);
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC, W.e), NoExtra());
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_FORCE>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// lCPDI: a corner's payload is the force -mp (sigma - P) . its gradient weight (+ pFext)
template <int DIM> struct CornerForceWords { int p, key; double x[DIM], m, pr, s[6], r[9]; };

template <int DIM>
__device__ __forceinline__ void load_corner_force(const KPart &rows, const KBins &B, int p, CornerForceWords<DIM> &t) {
    const KPart P = local_rows(rows);
    t.p = p;
    if (t.p < 0) return;
    t.key = B.key[t.p];
#pragma unroll
    for (int a = 0; a < DIM; a++) t.x[a] = P.f(MPF_POS_X + a)[t.p];
#pragma unroll
    for (int a = 0; a < 9; a++) t.r[a] = DIM == 3 || (a < 6 && a % 3 < 2) ? P.cpr(a)[t.p] : 0.;
    t.m = P.f(MPF_MASS)[t.p];
    t.pr = P.f(MPF_PRESSURE)[t.p];
    t.s[0] = P.f(MPF_SP_XX)[t.p]; t.s[1] = P.f(MPF_SP_YY)[t.p]; t.s[2] = P.f(MPF_SP_XY)[t.p];
    if (DIM == 3) { t.s[3] = P.f(MPF_SP_ZZ)[t.p]; t.s[4] = P.f(MPF_SP_XZ)[t.p]; t.s[5] = P.f(MPF_SP_YZ)[t.p]; }
}

template <int DIM, bool FX>
__global__ __launch_bounds__(64 * CORNER_NW(DIM), FX ? 2 : WAVES8) void k_p2g_force_corners(KGrid g0, KPart P, KBins B, KNodes N, KLoads L,
                                                                        const int *loaded) {
    using G = TileGeom<DIM>;
    constexpr int NW = CORNER_NW(DIM);
    __shared__ double s_S[NW][4 * DIM + 4][WROW];
    __shared__ int s_tt[FX ? NW : 1][WREC / Corners<DIM>::N];    // traction tables of the staged particles (-1: none)
    __shared__ double s_acc[NW][NQ_FORCE][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l / Corners<DIM>::N, c = l % Corners<DIM>::N;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        if (loaded && (loaded[tall] != 0) != FX) return;
        const int tc = tall % g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveScatter<DIM, NW, NQ_FORCE, Corners<DIM>::N, WROW, DIM == 2> sc;
        sc.begin(&s_S[w][0][0], s_acc);
        auto trac = [&](int kb, int ke, int q, int hi, int ix, auto &f) {
            if (!FX || L.nt == 0) return;
            add_tractions(L, s_tt[FX ? w : 0], kb, ke, q, hi, ix, f);
        };
        zero_wave_acc<DIM, NW, NQ_FORCE>(s_acc);
        CornerForceWords<DIM> cur;
        int ahead = W.particle(B, W.b + Corners<DIM>::PB + i);       // the order is read a round before the words
        load_corner_force<DIM>(P, B, W.particle(B, W.b + i), cur);
        for (int r = W.b; r < W.e; r += Corners<DIM>::PB) {
            double xi[3], u[3];
            int off[3], tt = -1;
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                corner_lane<DIM>(gp, cur.x, cur.r, ox + lx, oy + ly, oz + lz, c, xi, off);
                double wg[3];
                cpdi_wg_staged<DIM>(cur.r, c, wg);
                const double xx = -cur.m * (cur.s[0] - cur.pr), yy = -cur.m * (cur.s[1] - cur.pr), xy = -cur.m * cur.s[2];
                if constexpr (DIM == 3) {
                    const double zz = -cur.m * (cur.s[3] - cur.pr), xz = -cur.m * cur.s[4], yz = -cur.m * cur.s[5];
                    u[0] = fma(xx, wg[0], fma(xy, wg[1], xz * wg[2]));
                    u[1] = fma(xy, wg[0], fma(yy, wg[1], yz * wg[2]));
                    u[2] = fma(xz, wg[0], fma(yz, wg[1], zz * wg[2]));
                } else {
                    u[0] = fma(xx, wg[0], xy * wg[1]);
                    u[1] = fma(xy, wg[0], yy * wg[1]);
                    u[2] = 0.;
                }
                if constexpr (FX) {
                    const int q = L.map[B.home[cur.p]];
#pragma unroll
                    for (int a = 0; a < 3; a++) u[a] = q >= 0 ? fma(Corners<DIM>::WW, L.fext[3 * q + a], u[a]) : u[a];
                    tt = q >= 0 && L.nt > 0 ? L.tslot[q] : -1;
                }
            }
            for (int r0 = r; r0 < min(r + Corners<DIM>::PB, W.e); r0 += WREC / Corners<DIM>::N) {
                if (l / WREC == (r0 - r) / (WREC / Corners<DIM>::N) && cur.p >= 0) {
                    stage_corner<DIM, 3>(s_S[w], l % WREC, xi, off, u);
                    if (FX && c == 0) s_tt[FX ? w : 0][i % (WREC / Corners<DIM>::N)] = tt;
                }
                if (r0 + WREC / Corners<DIM>::N >= min(r + Corners<DIM>::PB, W.e)) {
                    load_corner_force<DIM>(P, B, ahead, cur);
                    ahead = W.particle(B, r + 2 * Corners<DIM>::PB + i);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC / Corners<DIM>::N, W.e), trac);
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_FORCE>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// node pass after the forces: ftot, restore p (identity without BCs), p += f dt, v = p/m
// (PostForcesTask.cpp:46-48, MatVelocityField.cpp:301-314, :239-251)
template <int DIM>
__global__ void k_node_force(KGrid g0, KBins B, KNodes N) {
    long long nall = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (nall >= g0.nstride * g0.nfields) return;
    const int fld = node_field(g0, nall);
    const long long ng = nall - (long long)fld * g0.nstride;
    const KGrid g = node_grid(g0, ng);
    const long long n = ng - g.nodeBase;
    if (n >= g.nnodes) return;                // padding between instances
    const KNodes Nf = field_view(g, N, fld);
    int i, j, k;
    node_ijk(g, n, i, j, k);
    if (!node_needed<DIM>(g, B, fld, i, j, k)) return;
    double f[NQ_FORCE];
    gather_partials<DIM, NQ_FORCE>(g, B, N, fld, i, j, k, f);
    long long nn = g.nstride;
    if (DIM == 2) f[2] = 0.;
    int cnt = Nf.cnt[n];
    if (DIM == 3 && cnt <= 0 && g.shape == MPMGPU_SHAPE_LCPDI && Nf.mass[n] == 0.) f[0] = f[1] = f[2] = 0.;   // (stage_corner)
    if (g.hasGravity && cnt > 0) {         // PostForcesTask.cpp:62-91 -> AddGravityAndBodyForceTask3
        const double m = Nf.mass[n];       // (MatVelocityField.cpp:254-258): ftot += mass g
        for (int c = 0; c < 3; c++) f[c] += m * g.gravity[c];
    }
    Nf.ftot[n] = f[0]; Nf.ftot[nn + n] = f[1]; Nf.ftot[2 * nn + n] = f[2];
    if (cnt <= 0) return;
    double dt = g.timestep;
    double px = Nf.pk[n] + f[0] * dt;
    double py = Nf.pk[nn + n] + f[1] * dt;
    double pz = Nf.pk[2 * nn + n] + f[2] * dt;
    Nf.pk[n] = px; Nf.pk[nn + n] = py; Nf.pk[2 * nn + n] = pz;
    double m = Nf.mass[n];
    if (m != 0.) {
        double s = 1. / m;
        Nf.vk[n] = s * px; Nf.vk[nn + n] = s * py; Nf.vk[2 * nn + n] = s * pz;
    }
}

// ---------------------------------------------------------------------------------------
// sums of NV footprint rows over a particle's support window
template <int DIM, int NV>
__device__ __forceinline__ void gather_window(const int w[3], const double Sw[3][3], int lx, int ly, int lz,
                                              const double (*s_n)[TileGeom<DIM>::FOOT], double out[NV]) {
#pragma unroll
    for (int v = 0; v < NV; v++) out[v] = 0.;
    constexpr int NZ = DIM == 3 ? 3 : 1;
#pragma unroll
    for (int jz = 0; jz < NZ; jz++) {
#pragma unroll
        for (int jy = 0; jy < 3; jy++)
#pragma unroll
            for (int jx = 0; jx < 3; jx++) {
                const double fi = DIM == 3 ? Sw[0][jx] * (Sw[1][jy] * Sw[2][jz]) : Sw[0][jx] * Sw[1][jy];
                const int s = foot_slot<DIM>(lx + w[0] + jx - 1, ly + w[1] + jy - 1, DIM == 3 ? lz + w[2] + jz - 1 : 0);
#pragma unroll
                for (int v = 0; v < NV; v++) out[v] = fma(s_n[v][s], fi, out[v]);
            }
        __builtin_amdgcn_sched_barrier(0);     // a plane's reads at a time: all 27 nodes' would not fit in registers
    }
    // the sums are formed here, not put off past a branch that follows (with the words held meanwhile)
#pragma unroll
    for (int v = 0; v < NV; v++) asm volatile("" : "+v"(out[v]));
}

// footprint velocities and accelerations f/m (zero outside the grid and on nodes without mass, which
// no particle of the tile touches)
template <int DIM, int NW>
__device__ __forceinline__ void load_foot_va(const KGrid &g, const KNodes &Nf, int ox, int oy, int oz,
                                             double (*s_n)[TileGeom<DIM>::FOOT]) {
    const long long nn = g.nstride;
    for (int s = threadIdx.x; s < TileGeom<DIM>::FOOT; s += 64 * NW) {
        const long long n = foot_node<DIM>(g, s, ox, oy, oz);
        const double m = n >= 0 ? Nf.mass[n] : 0.;
        const double r = m > 0. ? 1. / m : 0.;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            s_n[c][s] = n >= 0 ? Nf.vk[c * nn + n] : 0.;
            s_n[3 + c][s] = n >= 0 ? Nf.ftot[c * nn + n] * r : 0.;
        }
    }
}

// the same as (velocity, acceleration) pairs, one 16-byte LDS read each (the gather's reads kept the
// LDS busy for almost half of the kernel's time)
template <int DIM, int NW>
__device__ __forceinline__ void load_foot_pairs(const KGrid &g, const KNodes &Nf, int ox, int oy, int oz,
                                                double2 (*s_n)[TileGeom<DIM>::FOOT]) {
    const long long nn = g.nstride;
    for (int s = threadIdx.x; s < TileGeom<DIM>::FOOT; s += 64 * NW) {
        const long long n = foot_node<DIM>(g, s, ox, oy, oz);
        const double m = n >= 0 ? Nf.mass[n] : 0.;
        const double r = m > 0. ? 1. / m : 0.;
#pragma unroll
        for (int c = 0; c < 3; c++)
            s_n[c][s] = n >= 0 ? make_double2(Nf.vk[c * nn + n], Nf.ftot[c * nn + n] * r) : make_double2(0., 0.);
    }
}

template <int DIM>
__device__ __forceinline__ void gather_pairs(const int w[3], const double Sw[3][3], int lx, int ly, int lz,
                                             const double2 (*s_n)[TileGeom<DIM>::FOOT], double v[3], double a[3]) {
#pragma unroll
    for (int c = 0; c < 3; c++) v[c] = a[c] = 0.;
    constexpr int NZ = DIM == 3 ? 3 : 1;
#pragma unroll
    for (int jz = 0; jz < NZ; jz++) {
#pragma unroll
        for (int jy = 0; jy < 3; jy++)
#pragma unroll
            for (int jx = 0; jx < 3; jx++) {
                const double fi = DIM == 3 ? Sw[0][jx] * (Sw[1][jy] * Sw[2][jz]) : Sw[0][jx] * Sw[1][jy];
                const int s = foot_slot<DIM>(lx + w[0] + jx - 1, ly + w[1] + jy - 1, DIM == 3 ? lz + w[2] + jz - 1 : 0);
#pragma unroll
                for (int c = 0; c < DIM; c++) {
                    const double2 t = s_n[c][s];
                    v[c] = fma(t.x, fi, v[c]);
                    a[c] = fma(t.y, fi, a[c]);
                }
            }
        __builtin_amdgcn_sched_barrier(0);     // a plane's reads at a time: all 27 nodes' would not fit in registers
    }
    // the sums are formed here, not put off past a branch that follows (with the words held meanwhile)
#pragma unroll
    for (int c = 0; c < 3; c++) asm volatile("" : "+v"(v[c]), "+v"(a[c]));
}

// footprint XPIC increments (zero outside the grid and on nodes without particles)
template <int DIM, int NW>
__device__ __forceinline__ void load_foot_prev(const KGrid &g, const KNodes &Nf, int ox, int oy, int oz,
                                               double (*s_n)[TileGeom<DIM>::FOOT]) {
    const long long nn = g.nstride;
    for (int s = threadIdx.x; s < TileGeom<DIM>::FOOT; s += 64 * NW) {
        const long long n = foot_node<DIM>(g, s, ox, oy, oz);
        const bool on = n >= 0 && Nf.cnt[n] > 0;
#pragma unroll
        for (int c = 0; c < 3; c++) s_n[c][s] = on ? Nf.vprev[c * nn + n] : 0.;
    }
}

// Particle update (FLIP, no damping) fused with the momentum re-extrapolation of the USL pass
// with start-of-step shape functions (MatVelocityField::IncrementNodalVelAcc,
// MatVelocityField.cpp:410-426; MatPoint3D::MoveParticle, MatPoint3D.cpp:104-194;
// NodalPoint::AddMassMomentumLast, NodalPointMPM.cpp:470-486)
// MOVE: G2P_FLIP (no damping), G2P_FLIP_DAMPED, or G2P_SERIES, which moves by FMPM(mode) for
// mode > 0 and by XPIC(-mode) for mode < 0 with the damping of the grid (zero damping gives the
// same numbers as none). The FLIP instances keep their registers for the common update.
enum { G2P_FLIP = 0, G2P_FLIP_DAMPED = 1, G2P_SERIES = 2 };
template <int DIM, int MOVE>
__device__ __forceinline__ void move_particle(const KGrid &g, const KPart &P, const MpmMaterial *mats, int mode, int p,
                                              const double pos[3], const double vold[3], const double Svk[3],
                                              const double Sacc[3], double vnew[3], double xnew[3]) {
    constexpr bool DAMP = MOVE != G2P_FLIP;
    const double dt = g.timestep;
    // particle damping: the material's own <PDamping> in place of the run's
    // (MaterialBase::GetMaterialDamping, MaterialBaseMPM.cpp:742-744)
    double alphaP = 0.;
    if (DAMP) {
        const MpmMaterial &mt = mats[P.mat[p]];
        alphaP = mt.usePDamping ? mt.pdamping : g.particleDamping;
    }
    // MatPoint3D::MoveParticle (MatPoint3D.cpp:104-194): Adamp0 = alpha_p v + alpha_g vm
    // (the DAMP instance; zero damping gives delV = Sacc dt for FLIP)
    if (MOVE != G2P_SERIES) {
        // FLIP: vm = S(v - a dt), v += (Sa - Adamp0) dt, x += (vm + delV/2) dt (:104-160)
#pragma unroll
        for (int c = 0; c < DIM; c++) {
            double vm = Svk[c] - Sacc[c] * dt;
            double delV = DAMP ? (Sacc[c] - (vold[c] * alphaP + vm * g.gridDamping)) * dt
                               : Sacc[c] * dt;
            vnew[c] = vold[c] + delV;
            double delXRate = vm + 0.5 * delV;
            xnew[c] = pos[c] + delXRate * dt;
        }
    } else {
        // FMPM(k) (mode k): vm = S v+(k), v = vm - Adamp0 dt, x += (v(n) + v(n+1)) dt/2
        // (:122-137); XPIC(k) (mode -k): vm = S(v(k) + a dt), v = vm - Adamp0 dt,
        // x += (vm + delV/2) dt (:152-170)
#pragma unroll
        for (int c = 0; c < DIM; c++) {
            const double vm = Svk[c];
            const double adamp = DAMP ? vold[c] * alphaP + vm * g.gridDamping : 0.;
            if (mode > 0) {
                vnew[c] = vm + adamp * -dt;
                const double delXRate = vold[c] + vnew[c];
                xnew[c] = pos[c] + delXRate * (0.5 * dt);
            } else {
                vnew[c] = vm - adamp * dt;
                const double delV = vnew[c] - vold[c];
                const double delXRate = vm + 0.5 * delV;
                xnew[c] = pos[c] + delXRate * dt;
            }
        }
    }
}

template <int DIM>
__device__ __forceinline__ void store_move(const KPart &rows, int p, const double vnew[3], const double xnew[3]) {
    const KPart P = local_rows(rows);
#pragma unroll
    for (int c = 0; c < DIM; c++) {
        P.f(MPF_VEL_X + c)[p] = vnew[c];
        P.posn(c)[p] = xnew[c];
    }
}

// uGIMP and classic: a wave gathers, moves and scatters its particles 64 at a time
template <int DIM, int MOVE>
__global__ __launch_bounds__(64 * G2P_NW(DIM), WAVES8) void k_g2p_p2g(KGrid g0, KPart P, KBins B, KNodes N, const MpmMaterial *mats,
                                                            int mode) {
    using G = TileGeom<DIM>;
    constexpr int NW = G2P_NW(DIM);
    __shared__ double2 s_n[3][G::FOOT];        // (velocity, f/m) of each component
    __shared__ double s_S[NW][4 * DIM + 4][WROW];       // [axis*4 + offset][record], then the momentum (the last row is not used)
    __shared__ double s_acc[NW][NQ_MOM][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        const int fld = tall / g0.tilesTotal;
        const int tc = tall - fld * g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        const KNodes Nf = field_view(g, N, fld);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveScatter<DIM, NW, NQ_MOM, 1, WROW> sc;
        sc.begin(&s_S[w][0][0], s_acc);
        MassWords<DIM> cur;
        int ahead = W.particle(B, W.b + 64 + l);       // the order is read a round before the words
        load_mass_words<DIM>(P, B, W.particle(B, W.b + l), cur);
        load_foot_pairs<DIM, NW>(g, Nf, ox, oy, oz, s_n);
        zero_wave_acc<DIM, NW, NQ_MOM>(s_acc);
        __syncthreads();
        for (int r = W.b; r < W.e; r += 64) {
            AxisFactors f[DIM];
            double u[3];
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                int wd[3];
                double invd[DIM], Svk[3], Sacc[3], vnew[3], xnew[3];
                {
                    double Sw[3][3], Dw[3][3];
                    particle_axes<DIM>(gp, P, cur.p, ox + lx, oy + ly, oz + lz, cur.x, f, invd);
                    particle_window<DIM>(f, invd, wd, Sw, Dw);
                    gather_pairs<DIM>(wd, Sw, lx, ly, lz, s_n, Svk, Sacc);
                }
                move_particle<DIM, MOVE>(g, P, mats, mode, cur.p, cur.x, cur.v, Svk, Sacc, vnew, xnew);
                store_move<DIM>(P, cur.p, vnew, xnew);
#pragma unroll
                for (int c = 0; c < 3; c++) u[c] = c < DIM ? cur.m * vnew[c] : 0.;
            }
            for (int r0 = r; r0 < min(r + 64, W.e); r0 += WREC) {
                if (l / WREC == (r0 - r) / WREC && cur.p >= 0) stage_factors<DIM, 3>(s_S[w], l % WREC, f, u);
                // the next particles' loads pass over the last scatter
                if (r0 + WREC >= min(r + 64, W.e)) {
                    load_mass_words<DIM>(P, B, ahead, cur);
                    ahead = W.particle(B, r + 2 * 64 + l);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC, W.e));
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_MOM>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// lCPDI: the gather is taken corner by corner, a lane each, and added over the particle's lanes
template <int DIM> struct CornerMoveWords { int p, key; double x[DIM], m, v[DIM], r[9]; };

template <int DIM>
__device__ __forceinline__ void load_corner_move(const KPart &rows, const KBins &B, int p, CornerMoveWords<DIM> &t) {
    const KPart P = local_rows(rows);
    t.p = p;
    if (t.p < 0) return;
    t.key = B.key[t.p];
#pragma unroll
    for (int a = 0; a < DIM; a++) {
        t.x[a] = P.f(MPF_POS_X + a)[t.p];
        t.v[a] = P.f(MPF_VEL_X + a)[t.p];
    }
#pragma unroll
    for (int a = 0; a < 9; a++) t.r[a] = DIM == 3 || (a < 6 && a % 3 < 2) ? P.cpr(a)[t.p] : 0.;
    t.m = P.f(MPF_MASS)[t.p];
}

template <int DIM, int MOVE>
__global__ __launch_bounds__(64 * CORNER_NW(DIM), WAVES8) void k_g2p_p2g_corners(KGrid g0, KPart P, KBins B, KNodes N,
                                                             const MpmMaterial *mats, int mode) {
    using G = TileGeom<DIM>;
    constexpr int NW = CORNER_NW(DIM);
    __shared__ double s_n[6][G::FOOT];         // v(3), f/m(3)
    __shared__ double s_S[NW][4 * DIM + 4][WROW];
    __shared__ double s_acc[NW][NQ_MOM][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l / Corners<DIM>::N, c = l % Corners<DIM>::N;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        const int fld = tall / g0.tilesTotal;
        const int tc = tall - fld * g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        const KNodes Nf = field_view(g, N, fld);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveScatter<DIM, NW, NQ_MOM, Corners<DIM>::N, WROW, DIM == 2> sc;
        sc.begin(&s_S[w][0][0], s_acc);
        CornerMoveWords<DIM> cur;
        int ahead = W.particle(B, W.b + Corners<DIM>::PB + i);       // the order is read a round before the words
        load_corner_move<DIM>(P, B, W.particle(B, W.b + i), cur);
        load_foot_va<DIM, NW>(g, Nf, ox, oy, oz, s_n);
        zero_wave_acc<DIM, NW, NQ_MOM>(s_acc);
        __syncthreads();
        for (int r = W.b; r < W.e; r += Corners<DIM>::PB) {
            double xi[3], u[3];
            int off[3];
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                corner_lane<DIM>(gp, cur.x, cur.r, ox + lx, oy + ly, oz + lz, c, xi, off);
                double vc[6], Svk[3], Sacc[3], vnew[3], xnew[3];
                cpdi_corner_sum<DIM, 6>(xi, off, lx, ly, lz, s_n, vc);
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    Svk[a] = Corners<DIM>::W * corner_sum<DIM>(vc[a]);
                    Sacc[a] = Corners<DIM>::W * corner_sum<DIM>(vc[3 + a]);
                }
                move_particle<DIM, MOVE>(g, P, mats, mode, cur.p, cur.x, cur.v, Svk, Sacc, vnew, xnew);
                if (c == 0) store_move<DIM>(P, cur.p, vnew, xnew);
#pragma unroll
                for (int a = 0; a < 3; a++) u[a] = a < DIM ? Corners<DIM>::WW * cur.m * vnew[a] : 0.;
            }
            for (int r0 = r; r0 < min(r + Corners<DIM>::PB, W.e); r0 += WREC / Corners<DIM>::N) {
                if (l / WREC == (r0 - r) / (WREC / Corners<DIM>::N) && cur.p >= 0) stage_corner<DIM, 3>(s_S[w], l % WREC, xi, off, u);
                if (r0 + WREC / Corners<DIM>::N >= min(r + Corners<DIM>::PB, W.e)) {
                    load_corner_move<DIM>(P, B, ahead, cur);
                    ahead = W.particle(B, r + 2 * Corners<DIM>::PB + i);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC / Corners<DIM>::N, W.e));
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_MOM>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// node pass of the USL re-extrapolation: p (rezeroed, RezeroNodeTask6) and v = p/m
template <int DIM>
__global__ void k_node_mom2(KGrid g0, KBins B, KNodes N) {
    long long nall = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (nall >= g0.nstride * g0.nfields) return;
    const int fld = node_field(g0, nall);
    const long long ng = nall - (long long)fld * g0.nstride;
    const KGrid g = node_grid(g0, ng);
    const long long n = ng - g.nodeBase;
    if (n >= g.nnodes) return;                // padding between instances
    const KNodes Nf = field_view(g, N, fld);
    int cnt = Nf.cnt[n];
    if (cnt <= 0) return;
    int i, j, k;
    node_ijk(g, n, i, j, k);
    if (!node_needed<DIM>(g, B, fld, i, j, k)) return;
    double a[NQ_MOM];
    gather_partials<DIM, NQ_MOM>(g, B, N, fld, i, j, k, a);
    long long nn = g.nstride;
    Nf.pk[n] = a[0]; Nf.pk[nn + n] = a[1]; Nf.pk[2 * nn + n] = a[2];
    double m = Nf.mass[n];
    if (m != 0.) {
        double s = 1. / m;
        Nf.vk[n] = s * a[0]; Nf.vk[nn + n] = s * a[1]; Nf.vk[2 * nn + n] = s * a[2];
    }
}

// ---------------------------------------------------------------------------------------
// XPIC(k) and FMPM(k) grid velocities (XPICExtrapolationTask::Execute, XPICExtrapolationTask.cpp:50-164)
// for one material velocity field per material: v(k) = sum_{r<k} (P(I - A))^r v0 with
// A = diag(1/m) S^T Mp S, built as vk = v0 + Delta v(2) + ... + Delta v(k), each increment
// Delta v(r) = (I - A) Delta v(r-1) with the held components of the conditions zeroed.

// InitializeXPICData -> MatVelocityField::XPICSupport(INITIALIZE_XPIC) (MatVelocityField.cpp:321-345):
// FMPM starts from v0 = pk/m (the momenta the caller's pass left), XPIC from the velocities
// before the momentum update, v0 = (pk - ftot dt)/m, with ftot dt/m added to vk so the result
// is v(k) + a dt. vprev = v0 on every node with particles.
template <int DIM>
__global__ void k_xpic_init(KGrid g0, KBins B, KNodes N, int fmpm) {
    long long nall = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (nall >= g0.nstride * g0.nfields) return;
    const int fld = node_field(g0, nall);
    const long long ng = nall - (long long)fld * g0.nstride;
    const KGrid g = node_grid(g0, ng);
    const long long n = ng - g.nodeBase;
    if (n >= g.nnodes) return;
    const KNodes Nf = field_view(g, N, fld);
    if (Nf.cnt[n] <= 0) return;
    const long long nn = g.nstride;
    const double m = Nf.mass[n], dt = g.timestep, sc = 1. / m;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const double p = Nf.pk[c * nn + n];
        double vp, vs;
        if (fmpm) {
            vp = sc * p;
            vs = vp;
        } else {
            const double f = Nf.ftot[c * nn + n];
            vp = (p + f * -dt) * sc;
            vs = vp + f * (dt / m);
        }
        Nf.vprev[c * nn + n] = vp;
        Nf.vk[c * nn + n] = vs;
    }
}

// Particle loop of one increment (XPICExtrapolationTask::XPICDoubleLoop, XPICExtrapolationTask.cpp:182-211):
// node i gains sum_p mp S_ip (sum_j S_jp vprev_j), the particle's gather of the last increment
// scattered as a momentum; the node pass divides by m_i. Shape functions are those of the step's
// start, as in every pass of the step.
// uGIMP and classic: a wave gathers and scatters its particles 64 at a time
template <int DIM>
__global__ __launch_bounds__(64 * UGIMP_NW, WAVES4) void k_xpic_p2g(KGrid g0, KPart P, KBins B, KNodes N) {
    using G = TileGeom<DIM>;
    constexpr int NW = UGIMP_NW;
    __shared__ double s_n[3][G::FOOT];         // vprev
    __shared__ double s_S[NW][4 * DIM + 4][WROW];       // [axis*4 + offset][record], then the momentum (the last row is not used)
    __shared__ double s_acc[NW][NQ_MOM][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        const int fld = tall / g0.tilesTotal;
        const int tc = tall - fld * g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        const KNodes Nf = field_view(g, N, fld);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveScatter<DIM, NW, NQ_MOM, 1, WROW> sc;
        sc.begin(&s_S[w][0][0], s_acc);
        MassWords<DIM> cur;
        int ahead = W.particle(B, W.b + 64 + l);       // the order is read a round before the words
        load_mass_words<DIM>(P, B, W.particle(B, W.b + l), cur);
        load_foot_prev<DIM, NW>(g, Nf, ox, oy, oz, s_n);
        zero_wave_acc<DIM, NW, NQ_MOM>(s_acc);
        __syncthreads();
        for (int r = W.b; r < W.e; r += 64) {
            AxisFactors f[DIM];
            double u[3];
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                int wd[3];
                double invd[DIM], Sw[3][3], Dw[3][3], v[3];
                particle_axes<DIM>(gp, P, cur.p, ox + lx, oy + ly, oz + lz, cur.x, f, invd);
                particle_window<DIM>(f, invd, wd, Sw, Dw);
                gather_window<DIM, 3>(wd, Sw, lx, ly, lz, s_n, v);
#pragma unroll
                for (int c = 0; c < 3; c++) u[c] = c < DIM ? cur.m * v[c] : 0.;
            }
            for (int r0 = r; r0 < min(r + 64, W.e); r0 += WREC) {
                if (l / WREC == (r0 - r) / WREC && cur.p >= 0) stage_factors<DIM, 3>(s_S[w], l % WREC, f, u);
                // the next particles' loads pass over the last scatter
                if (r0 + WREC >= min(r + 64, W.e)) {
                    load_mass_words<DIM>(P, B, ahead, cur);
                    ahead = W.particle(B, r + 2 * 64 + l);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC, W.e));
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_MOM>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

template <int DIM>
__global__ __launch_bounds__(64 * CORNER_NW(DIM), WAVES8) void k_xpic_p2g_corners(KGrid g0, KPart P, KBins B, KNodes N) {
    using G = TileGeom<DIM>;
    constexpr int NW = CORNER_NW(DIM);
    __shared__ double s_n[3][G::FOOT];         // vprev
    __shared__ double s_S[NW][4 * DIM + 4][WROW];
    __shared__ double s_acc[NW][NQ_MOM][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l / Corners<DIM>::N, c = l % Corners<DIM>::N;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        const int fld = tall / g0.tilesTotal;
        const int tc = tall - fld * g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        const KNodes Nf = field_view(g, N, fld);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveScatter<DIM, NW, NQ_MOM, Corners<DIM>::N, WROW, DIM == 2> sc;
        sc.begin(&s_S[w][0][0], s_acc);
        CornerMoveWords<DIM> cur;
        int ahead = W.particle(B, W.b + Corners<DIM>::PB + i);       // the order is read a round before the words
        load_corner_move<DIM>(P, B, W.particle(B, W.b + i), cur);
        load_foot_prev<DIM, NW>(g, Nf, ox, oy, oz, s_n);
        zero_wave_acc<DIM, NW, NQ_MOM>(s_acc);
        __syncthreads();
        for (int r = W.b; r < W.e; r += Corners<DIM>::PB) {
            double xi[3], u[3];
            int off[3];
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                corner_lane<DIM>(gp, cur.x, cur.r, ox + lx, oy + ly, oz + lz, c, xi, off);
                double vc[3];
                cpdi_corner_sum<DIM, 3>(xi, off, lx, ly, lz, s_n, vc);
#pragma unroll
                for (int a = 0; a < 3; a++) u[a] = a < DIM ? Corners<DIM>::WW * cur.m * (Corners<DIM>::W * corner_sum<DIM>(vc[a])) : 0.;
            }
            for (int r0 = r; r0 < min(r + Corners<DIM>::PB, W.e); r0 += WREC / Corners<DIM>::N) {
                if (l / WREC == (r0 - r) / (WREC / Corners<DIM>::N) && cur.p >= 0) stage_corner<DIM, 3>(s_S[w], l % WREC, xi, off, u);
                if (r0 + WREC / Corners<DIM>::N >= min(r + Corners<DIM>::PB, W.e)) {
                    load_corner_move<DIM>(P, B, ahead, cur);
                    ahead = W.particle(B, r + 2 * Corners<DIM>::PB + i);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC / Corners<DIM>::N, W.e));
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_MOM>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// Node pass of one increment (GetDeltaV and UpdateXStar, XPICExtrapolationTask.cpp:222-240;
// MatVelocityField::XPICSupport GET_DELTAV and UPDATE_VSTAR, MatVelocityField.cpp:347-378):
// vprev -= (the scatter's sum)/m, vk += vprev. The XPIC pass of the velocity conditions then zeroes
// the held components of vprev and takes them back out of vk. Block 0 clears the cursors of the
// XPIC tile slot for the next increment's scatter (the scatter before this pass has finished).
template <int DIM>
__global__ void k_xpic_node(KGrid g0, KBins B, KNodes N) {
    if (blockIdx.x == 0 && threadIdx.x < 8) B.work[(TILE_SLOT_XPIC * 8 + threadIdx.x) * TILE_SLOT_STRIDE] = 0;
    long long nall = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (nall >= g0.nstride * g0.nfields) return;
    const int fld = node_field(g0, nall);
    const long long ng = nall - (long long)fld * g0.nstride;
    const KGrid g = node_grid(g0, ng);
    const long long n = ng - g.nodeBase;
    if (n >= g.nnodes) return;
    const KNodes Nf = field_view(g, N, fld);
    if (Nf.cnt[n] <= 0) return;
    int i, j, k;
    node_ijk(g, n, i, j, k);
    double a[NQ_MOM];
    gather_partials<DIM, NQ_MOM>(g, B, N, fld, i, j, k, a);
    const long long nn = g.nstride;
    const double m = Nf.mass[n];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const double d = Nf.vprev[c * nn + n] - a[c] / m;
        Nf.vprev[c * nn + n] = d;
        Nf.vk[c * nn + n] += d;
    }
}

// ---------------------------------------------------------------------------------------
// element test of a rectangle (EightNodeIsoparamBrick.cpp:207-213, FourNodeIsoparam.cpp:413-423)
template <int DIM>
__device__ __forceinline__ bool pt_in_elem(const KGrid &g, int ei, int ej, int ek, const double p[3]) {
    double xmn = g.xmin + (double)ei * g.dx, xmx = g.xmin + (double)(ei + 1) * g.dx;
    if (p[0] < xmn || p[0] >= xmx) return false;
    double ymn = g.ymin + (double)ej * g.dy, ymx = g.ymin + (double)(ej + 1) * g.dy;
    if (p[1] < ymn || p[1] >= ymx) return false;
    if (DIM == 3) {
        double zmn = g.zmin + (double)ek * g.dz, zmx = g.zmin + (double)(ek + 1) * g.dz;
        if (p[2] < zmn || p[2] >= zmx) return false;
    }
    return true;
}

// USL strain update (second half step) and ResetElementsTask; also the cell key and histogram
// of the next binning
template <int DIM, int MAT, int SH>
__global__ __launch_bounds__(NT, 2) void k_usl_reset(KGrid g0, KPart P, KBins B, KNodes N, const MpmMaterial *mats,
                                                  KStats st, int only) {
    using G = TileGeom<DIM>;
    __shared__ double s_v[3][G::FOOT];
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        if (only >= 0 && g0.tileType[tall % g0.tilesTotal] != only) return;   // another launch's type
        const int fld = tall / g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tall - fld * g0.tilesTotal);
        const KGrid g = grid_copy(gp);
        const int t = tall - fld * g0.tilesTotal - g.tileBase;
        const KNodes Nf = field_view(g, N, fld);
        const int tb = const_int(B.cellStart + (size_t)tall * G::NC), te = const_int(B.cellStart + (size_t)(tall + 1) * G::NC);
        int ox, oy, oz;
        tile_origin<DIM>(g, t, ox, oy, oz);
        int p = tb + (int)threadIdx.x < te ? B.order[tb + threadIdx.x] : -1;
        {
            const double *src[3] = {Nf.vk, Nf.vk, Nf.vk};
            const long long stt[3] = {0, g.nstride, 2 * g.nstride};
            load_foot<DIM, 3>(g, ox, oy, oz, src, stt, s_v);
        }
        __syncthreads();
        for (int k = tb + threadIdx.x; k < te; k += NT, p = k < te ? B.order[k] : -1) {
            const int mat = P.mat[p];
            int lx, ly, lz;
            tile_cell<DIM>(B.key[p], tall, lx, ly, lz);
            // the end-of-step position is loaded here, before the state stores below, so its load is
            // issued with the others instead of after them
            double pos[3] = {P.posn(0)[p], P.posn(1)[p], DIM == 3 ? P.posn(2)[p] : 0.};
            int ei = ox + lx, ej = oy + ly, ek = oz + lz;
            const MpmMaterial &m = mats[mat];
            const int mtype = MAT ? MAT : m.type;
            PState s;
            if (SH != MPMGPU_SHAPE_LCPDI) load_state<DIM>(P, p, mtype, s);
            double L[3][3];
            particle_gradient<DIM, SH>(g, gp, P, p, ei, ej, ek, lx, ly, lz, s_v, L);
            scale_gradient<DIM>(L, g.strainLast);
            if (SH == MPMGPU_SHAPE_LCPDI) load_state<DIM>(P, p, mtype, s);
            constitutive<DIM, MAT>(L, m, s);
            store_state<DIM>(P, p, mtype, s);

            // ResetElementsTask::ResetElement (ResetElementsTask.cpp:196-228)
            if (pos[0] != pos[0] || pos[1] != pos[1] || pos[2] != pos[2]) {
                atomicAdd(st.nanCount, 1ull);
                if (g.stopOnNan) stop_run(B, STOP_NAN, -1);
            } else if (!pt_in_elem<DIM>(g, ei, ej, ek, pos)) {
                // MeshInfo::FindElementFromPoint (MeshInfo.cpp:593-640) and EdgeElement2D/3D (:171-199)
                bool left = false;
                long long horiz = g.nx, vert = g.ny, depth = DIM == 3 ? g.nz : 1;
                long long total = horiz * vert * depth;
                long long col = (long long)(int)((pos[0] - g.xmin) / g.dx);
                if (col < 0 || col >= horiz) {
                    if (pos[0] == g.xmin + horiz * g.dx) col = horiz - 1; else left = true;
                }
                long long row = 0, zrow = 0;
                if (!left) {
                    row = (long long)(int)((pos[1] - g.ymin) / g.dy);
                    if (row < 0 || row >= vert) {
                        if (pos[1] == g.ymin + vert * g.dy) row = vert - 1; else left = true;
                    }
                }
                if (!left && DIM == 3) {
                    zrow = (long long)(int)((pos[2] - g.zmin) / g.dz);
                    if (zrow < 0 || zrow >= depth) {
                        if (pos[2] == g.zmin + depth * g.dz) zrow = depth - 1; else left = true;
                    }
                }
                long long num = 0;
                if (!left) {
                    num = (DIM == 3 ? horiz * (zrow * vert + row) + col : row * horiz + col) + 1;
                    if (DIM == 3) {
                        if (num <= horiz * vert || num > total - horiz * vert) left = true;
                        else if (num % horiz <= 1) left = true;
                        else {
                            long long xz = num % (horiz * vert);
                            if (xz <= horiz || xz > horiz * (vert - 1)) left = true;
                        }
                    } else {
                        if (num <= horiz || num > total - horiz) left = true;
                        else if (num % horiz <= 1) left = true;
                    }
                }
                if (!left) {
                    const int e = (int)(num - 1);
                    P.elem[p] = e;
                    elem_ijk(g, e, ei, ej, ek);
                } else {
                    // the warning count comes first, then the deletion (ResetElementsTask.cpp:71-104)
                    if (!P.left[p]) {
                        P.left[p] = 1;
                        const unsigned long long before = atomicAdd(st.leftGrid, 1ull);
                        if (g.maxLeaving > 0 && before + 1ull >= (unsigned long long)g.maxLeaving)
                            stop_run(B, STOP_TOO_MANY_LEFT, (long long)before);
                        else if (g.deleteLeaving)
                            stop_run(B, STOP_DELETE, (long long)before);
                    } else if (g.deleteLeaving) {
                        stop_run(B, STOP_DELETE, (long long)(*st.leftGrid));
                    }
                    // ReturnToElement (ResetElementsTask.cpp:232-265)
                    double dtt = g.timestep;
                    double outside[3] = {pos[0], pos[1], pos[2]};
                    double inside[3];
                    inside[0] = outside[0] - dtt * P.f(MPF_VEL_X)[p];
                    inside[1] = outside[1] - dtt * P.f(MPF_VEL_Y)[p];
                    inside[2] = DIM == 3 ? outside[2] - dtt * P.f(MPF_VEL_Z)[p] : 0.;
                    if (!pt_in_elem<DIM>(g, ei, ej, ek, inside)) {
                        inside[0] = ((g.xmin + (double)ei * g.dx) + (g.xmin + (double)(ei + 1) * g.dx)) / 2.;
                        inside[1] = ((g.ymin + (double)ej * g.dy) + (g.ymin + (double)(ej + 1) * g.dy)) / 2.;
                        inside[2] = DIM == 3 ? ((g.zmin + (double)ek * g.dz) + (g.zmin + (double)(ek + 1) * g.dz)) / 2. : 0.;
                    }
                    for (int pass = 1; pass <= 10; pass++) {
                        double mid[3] = {(outside[0] + inside[0]) / 2., (outside[1] + inside[1]) / 2.,
                                         (outside[2] + inside[2]) / 2.};
                        if (pt_in_elem<DIM>(g, ei, ej, ek, mid)) { inside[0] = mid[0]; inside[1] = mid[1]; inside[2] = mid[2]; }
                        else { outside[0] = mid[0]; outside[1] = mid[1]; outside[2] = mid[2]; }
                    }
                    P.posn(0)[p] = inside[0];
                    P.posn(1)[p] = inside[1];
                    if (DIM == 3) P.posn(2)[p] = inside[2];
                }
            }
            int key = cell_key<DIM>(g, fld, ei, ej, DIM == 3 ? ek : 0);
            B.key[p] = key;
            wave_count(B.count, key);
        }
    };
    for_each_tile<DIM>(B, tile);
}

// ---------------------------------------------------------------------------------------
// Multimaterial contact extrapolations (NodalPoint::AddMassMomentum / AddMassMomentumLast extras,
// NodalPointMPM.cpp:428-437,477-485 -> CrackVelocityField::AddVolumeDisplacement,
// CrackVelocityField.cpp:395-402, CrackVelocityFieldMulti::AddVolumeGradient, :108-112): per field,
// volume sum N Vp, displacement sum (x - x0) N mp and volume gradient sum grad N Vp, with
// Vp = det(F) mp / rho (MatPoint3D::GetVolume, MatPoint2D::GetVolume) and the start-of-step
// shape functions. The displacement uses the new positions in the USL pass.
template <int DIM> struct ContactWords { int p, key; double x[DIM], m, ep[6], wr[3], u[DIM], rho; };

template <int DIM>
__device__ __forceinline__ void load_contact_words(const KPart &rows, const KBins &B, const MpmMaterial *mats, int newPositions,
                                                   int p, ContactWords<DIM> &t) {
    const KPart P = local_rows(rows);
    t.p = p;
    if (t.p < 0) return;
    t.key = B.key[t.p];
#pragma unroll
    for (int a = 0; a < DIM; a++) {
        t.x[a] = P.f(MPF_POS_X + a)[t.p];
        t.u[a] = (newPositions ? P.posn(a)[t.p] : t.x[a]) - P.f(MPF_ORIG_X + a)[t.p];
    }
    load_deformation<DIM>(P, t.p, t.ep, t.wr);
    t.m = P.f(MPF_MASS)[t.p];
    t.rho = mats[P.mat[t.p]].rho;
}

// Vp of the words' particle
template <int DIM>
__device__ __forceinline__ double contact_volume(const ContactWords<DIM> &t) {
    double Fm[3][3], J;
    get_F3(t.ep, t.wr, Fm);
    if (DIM == 3)
        J = Fm[0][0] * (Fm[1][1] * Fm[2][2] - Fm[2][1] * Fm[1][2])
            - Fm[0][1] * (Fm[1][0] * Fm[2][2] - Fm[2][0] * Fm[1][2])
            + Fm[0][2] * (Fm[1][0] * Fm[2][1] - Fm[2][0] * Fm[1][1]);
    else J = Fm[0][0] * Fm[1][1] - Fm[1][0] * Fm[0][1];
    return J * t.m / t.rho;
}

// uGIMP and classic
template <int DIM>
__global__ __launch_bounds__(64 * UGIMP_NW, MPM_TILE_SHAPE == 0 ? 2 : 1) void k_p2g_contact(KGrid g0, KPart P, KBins B, KNodes N, const MpmMaterial *mats,
                                                        int newPositions) {
    using G = TileGeom<DIM>;
    constexpr int NW = UGIMP_NW;
    __shared__ double2 s_F[NW][4 * DIM][WROW]; // per wave: [axis*4 + offset][record] (factor, derivative)
    __shared__ double s_u[NW][4][WROW];        // volume and displacement
    __shared__ double s_acc[NW][NQ_CONTACT][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        const int tc = tall % g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveContact<DIM, NW, WROW> sc;
        sc.begin(&s_F[w][0][0], &s_u[w][0][0], s_acc);
        ContactWords<DIM> cur;
        int ahead = W.particle(B, W.b + 64 + l);       // the order is read a round before the words
        load_contact_words<DIM>(P, B, mats, newPositions, W.particle(B, W.b + l), cur);
        zero_wave_acc<DIM, NW, NQ_CONTACT>(s_acc);
        for (int r = W.b; r < W.e; r += 64) {
            AxisFactors f[DIM];
            double invd[DIM], u[4];
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                u[0] = contact_volume<DIM>(cur);
#pragma unroll
                for (int a = 0; a < 3; a++) u[1 + a] = a < DIM ? cur.m * cur.u[a < DIM ? a : 0] : 0.;
                particle_axes<DIM>(gp, P, cur.p, ox + lx, oy + ly, oz + lz, cur.x, f, invd);
            }
            for (int r0 = r; r0 < min(r + 64, W.e); r0 += WREC) {
                if (l / WREC == (r0 - r) / WREC && cur.p >= 0) {
                    stage_pairs<DIM>(s_F[w], l % WREC, f, invd);
#pragma unroll
                    for (int q = 0; q < 4; q++) s_u[w][q][l % WREC] = u[q];
                }
                // the next particles' loads pass over the last scatter
                if (r0 + WREC >= min(r + 64, W.e)) {
                    load_contact_words<DIM>(P, B, mats, newPositions, ahead, cur);
                    ahead = W.particle(B, r + 2 * 64 + l);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC, W.e));
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_CONTACT>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

// lCPDI: seven components are two products with the same rows, a particle's corners its records (weights and
// the gradient weight times Vp)
template <int DIM>
__global__ __launch_bounds__(64 * UGIMP_NW, MPM_TILE_SHAPE == 0 ? 2 : 1) void k_p2g_contact_corners(KGrid g0, KPart P, KBins B, KNodes N,
                                                        const MpmMaterial *mats, int newPositions) {
    using G = TileGeom<DIM>;
    constexpr int NW = UGIMP_NW;
    constexpr int PPR = Corners<DIM>::N, PB = Corners<DIM>::PB;
    __shared__ double s_S[NW][4 * DIM + 8][WROW];
    __shared__ double s_acc[NW][NQ_CONTACT][WaveFoot<DIM, NW>::SIZE];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l / PPR, c = l % PPR;
    auto tile = [&](const int tall, auto &&claim) {      // (field, context tile) pair
        const int tc = tall % g0.tilesTotal;
        const GridPtr gp = tile_grid_ptr(g0, tc);
        const KGrid g = grid_copy(gp);
        int ox, oy, oz;
        tile_origin<DIM>(g, tc - g.tileBase, ox, oy, oz);
        WaveCells<DIM, NW> W;
        W.begin(B.cellStart + (size_t)tall * G::NC);
        WaveScatter<DIM, NW, NQ_CONTACT, PPR, WROW, DIM == 2> sc;
        sc.begin(&s_S[w][0][0], s_acc);
        ContactWords<DIM> cur;
        int ahead = W.particle(B, W.b + PB + i);       // the order is read a round before the words
        load_contact_words<DIM>(P, B, mats, newPositions, W.particle(B, W.b + i), cur);
        zero_wave_acc<DIM, NW, NQ_CONTACT>(s_acc);
        for (int r = W.b; r < W.e; r += PB) {
            double xi[3], u[NQ_CONTACT];
            int off[3];
            if (cur.p >= 0) {
                int lx, ly, lz;
                tile_cell<DIM>(cur.key, tall, lx, ly, lz);
                const double Vp = contact_volume<DIM>(cur);
                double s[9], wg[3];
#pragma unroll
                for (int a = 0; a < 9; a++) s[a] = DIM == 3 || (a < 6 && a % 3 < 2) ? P.cpr(a)[cur.p] : 0.;
                corner_lane<DIM>(gp, cur.x, s, ox + lx, oy + ly, oz + lz, c, xi, off);
                cpdi_wg_staged<DIM>(s, c, wg);
                u[0] = Corners<DIM>::WW * Vp;
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    u[1 + a] = a < DIM ? Corners<DIM>::WW * cur.m * cur.u[a < DIM ? a : 0] : 0.;
                    u[4 + a] = wg[a] * Vp;
                }
            }
            for (int r0 = r; r0 < min(r + PB, W.e); r0 += WREC / PPR) {
                if (l / WREC == (r0 - r) / (WREC / PPR) && cur.p >= 0) stage_corner<DIM, NQ_CONTACT>(s_S[w], l % WREC, xi, off, u);
                if (r0 + WREC / PPR >= min(r + PB, W.e)) {
                    load_contact_words<DIM>(P, B, mats, newPositions, ahead, cur);
                    ahead = W.particle(B, r + 2 * PB + i);
                }
                wave_sync();
                sc.scatter(W, r0, min(r0 + WREC / PPR, W.e));
                wave_sync();
            }
        }
        claim();
        sc.finish(W);
        __syncthreads();
        write_partials<DIM, NW, NQ_CONTACT>(N, tall, s_acc);
    };
    for_each_tile<DIM>(B, tile);
}

template <int DIM>
__global__ void k_node_contact(KGrid g0, KBins B, KNodes N) {
    long long nall = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (nall >= g0.nstride * g0.nfields) return;
    const int fld = node_field(g0, nall);
    const long long ng = nall - (long long)fld * g0.nstride;
    const KGrid g = node_grid(g0, ng);
    const long long n = ng - g.nodeBase;
    if (n >= g.nnodes) return;                // padding between instances
    const KNodes Nf = field_view(g, N, fld);
    int i, j, k;
    node_ijk(g, n, i, j, k);
    if (!node_needed<DIM>(g, B, fld, i, j, k)) return;
    double a[NQ_CONTACT];
    gather_partials<DIM, NQ_CONTACT>(g, B, N, fld, i, j, k, a);
    long long nn = g.nstride;
    if (DIM == 3 && g.shape == MPMGPU_SHAPE_LCPDI && Nf.mass[n] == 0.)       // (stage_corner)
#pragma unroll
        for (int q = 0; q < NQ_CONTACT; q++) a[q] = 0.;
    Nf.cvol[n] = a[0];
    Nf.cdisp[n] = a[1]; Nf.cdisp[nn + n] = a[2]; Nf.cdisp[2 * nn + n] = a[3];
    Nf.cgrad[n] = a[4]; Nf.cgrad[nn + n] = a[5]; Nf.cgrad[2 * nn + n] = a[6];
}

__device__ __forceinline__ double dot3(const double *a, const double *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

// CoulombFriction::GetFrictionalDeltaMomentum and GetSslideAcDt (CoulombFriction.cpp:146-282);
// false leaves the momenta unchanged
__device__ __forceinline__ bool coulomb_delta(const KGrid &g, double *delPi, const double *norm, double dotn,
                                              double deltaDotn, double mred, const double *delFi) {
    double coeff = g.friction, coeffStatic = g.frictionStatic;
    int style = coeff < 0. ? 0 : (coeff == 0. ? 1 : 2);      // STICK, FRICTIONLESS, FRICTIONAL
    if (coeffStatic > 0. && style == 1) style = 2;
    if (style == 0) return true;
    double deltime = g.timestep;
    if (delFi) {
        double fn = dot3(delFi, norm);
        deltaDotn += deltime * (dotn - 0.5 * fn * deltime) / mred;
    }
    bool inContact = deltaDotn < 0. && dotn < 0.;
    if (style == 1) {
        if (inContact) { for (int c = 0; c < 3; c++) delPi[c] = norm[c] * dotn; return true; }
        return false;
    }
    if (!inContact) return false;
    double dott = 0., tang[3];
    for (int c = 0; c < 3; c++) tang[c] = delPi[c];
    for (int c = 0; c < 3; c++) tang[c] += norm[c] * (-dotn);
    double tangMag = sqrt(dot3(tang, tang));
    if (tangMag > 0.) {
        double sc = 1. / tangMag;
        for (int c = 0; c < 3; c++) tang[c] *= sc;
        dott = dot3(delPi, tang);
        if (dott < 0.) { for (int c = 0; c < 3; c++) tang[c] *= -1.; dott = -dott; }
    }
    double NAcDt = -dotn, SslideAcDt;
    if (coeffStatic > 0. && dott <= coeffStatic * NAcDt) SslideAcDt = coeffStatic * NAcDt;
    else SslideAcDt = coeff * NAcDt;
    if (SslideAcDt <= 0.) {
        for (int c = 0; c < 3; c++) delPi[c] = norm[c] * dotn;
    } else if (dott > SslideAcDt) {
        for (int c = 0; c < 3; c++) delPi[c] = norm[c] * dotn;
        for (int c = 0; c < 3; c++) delPi[c] += tang[c] * SslideAcDt;
    }
    return true;
}

// MatVelocityField::ChangeMatMomentum (MatVelocityField.cpp:197-224) on field f of node n, then
// the field's velocity for the next gather (GridValueCalculation, :239-251)
__device__ __forceinline__ void change_momentum(const KGrid &g, const KNodes &N, int f, long long n,
                                                const double *delP, int callType) {
    long long nn = g.nstride, b = 3 * f * nn + n;
    double p[3];
    for (int c = 0; c < 3; c++) { p[c] = N.pk[b + c * nn] + delP[c]; N.pk[b + c * nn] = p[c]; }
    if (callType == CONTACT_UPDATE_MOMENTUM) {
        double sc = 1. / g.timestep;
        for (int c = 0; c < 3; c++) N.ftot[b + c * nn] += delP[c] * sc;
    }
    double m = N.mass[f * nn + n];
    if (N.cnt[f * nn + n] > 0 && m != 0.) {
        double s = 1. / m;
        for (int c = 0; c < 3; c++) N.vk[b + c * nn] = s * p[c];
    }
}

// MaterialContactNode::ContactOnKnownNodes -> CrackVelocityFieldMulti::MaterialContactOnCVFLumped
// (CrackVelocityFieldMulti.cpp:302-671) for non-rigid materials, contact by displacements, normals
// by GetNormalVector (:960-1069) methods 0-3, no symmetry planes. One thread per node; nodes with
// fewer than two materials return at once.
template <int DIM>
__global__ void k_contact(KGrid g, KNodes N, int callType) {
    long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nnodes) return;
    const long long nn = g.nstride;
    int act[MPMGPU_MAX_MATERIALS];
    int numMats = 0;
    for (int f = 0; f < g.nfields; f++)
        if (N.cnt[f * nn + n] > 0) act[numMats++] = f;
    if (numMats <= 1) return;
    double Pc[3] = {0., 0., 0.}, Mc = 0.;
    for (int a = 0; a < numMats; a++) {
        long long b = 3 * act[a] * nn + n;
        for (int c = 0; c < 3; c++) Pc[c] += N.pk[b + c * nn];
        Mc += N.mass[act[a] * nn + n];
    }
    const int normals = g.normals;
    const bool doingPairs = numMats == 2 && normals != 3;
    const int miMax = doingPairs ? numMats - 1 : numMats;
    const bool postUpdate = callType == CONTACT_UPDATE_MOMENTUM;
    double dispc[3] = {0., 0., 0.};
    for (int a = 0; a < numMats; a++)
        for (int c = 0; c < 3; c++) dispc[c] += N.cdisp[(3 * act[a] + c) * nn + n];
    double sMc = 1. / Mc;
    for (int c = 0; c < 3; c++) dispc[c] *= sMc;
    double volAll = 0.;
    for (int a = 0; a < numMats; a++) volAll += N.cvol[act[a] * nn + n];
    for (int mi = 0; mi < miMax; mi++) {
        const int i = act[mi];
        double massi = N.mass[i * nn + n];
        double voli = N.cvol[i * nn + n];
        double volj = volAll - voli;
        int j = -1;
        double gradj[3] = {0., 0., 0.};
        double maxOther = 0.;
        for (int kj = 0; kj < numMats; kj++) {
            if (kj == mi) continue;
            int jj = act[kj];
            double mv = N.cvol[jj * nn + n];
            if (mv > maxOther) { maxOther = mv; j = jj; }
            for (int c = 0; c < 3; c++) gradj[c] += N.cgrad[(3 * jj + c) * nn + n] * -1.;
        }
        if (j < 0) continue;
        double massRatio = massi / Mc;
        double mred = 1. - massRatio;
        double delPi[3];
        for (int c = 0; c < 3; c++) delPi[c] = N.pk[(3 * i + c) * nn + n] * -1.;
        for (int c = 0; c < 3; c++) delPi[c] += Pc[c] * massRatio;
        if (!g.ignoreContact) {
            double gradi[3], norm[3];
            for (int c = 0; c < 3; c++) gradi[c] = N.cgrad[(3 * i + c) * nn + n] * 1.;
            if (normals == 0) {
                double magi = sqrt(dot3(gradi, gradi)), magj = sqrt(dot3(gradj, gradj));
                if (magi >= 1. * magj) { double sc = 1. / magi; for (int c = 0; c < 3; c++) norm[c] = gradi[c] * sc; }
                else { double sc = 1. / magj; for (int c = 0; c < 3; c++) norm[c] = gradj[c] * sc; }
            } else if (normals == 1) {
                if (voli >= volj) for (int c = 0; c < 3; c++) norm[c] = gradi[c];
                else for (int c = 0; c < 3; c++) norm[c] = gradj[c];
                double sc = 1. / sqrt(dot3(norm, norm));
                for (int c = 0; c < 3; c++) norm[c] = norm[c] * sc;
            } else if (normals == 2) {
                for (int c = 0; c < 3; c++) norm[c] = gradi[c];
                for (int c = 0; c < 3; c++) norm[c] += gradj[c];
                double sc = 1. / sqrt(dot3(norm, norm));
                for (int c = 0; c < 3; c++) norm[c] *= sc;
            } else if (normals == 3) {
                for (int c = 0; c < 3; c++) norm[c] = gradi[c];
                double sc = 1. / sqrt(dot3(norm, norm));
                for (int c = 0; c < 3; c++) norm[c] *= sc;
            } else if (normals == 4) {            // SPECIFIED_NORMAL (no symmetry planes)
                for (int c = 0; c < 3; c++) norm[c] = g.contactNormal[c];
            } else {                              // regression: k_contact_normals found it
                for (int c = 0; c < 3; c++) norm[c] = N.cnorm[(4 * i + c) * nn + n];
            }
            if (norm[0] != norm[0] || norm[1] != norm[1] || norm[2] != norm[2]) continue;
            double dotn = dot3(delPi, norm);
            double dispa[3], sa = 1. / massi;
            for (int c = 0; c < 3; c++) dispa[c] = N.cdisp[(3 * i + c) * nn + n] * sa;
            double delta[3], sr = 1. / mred;
            for (int c = 0; c < 3; c++) delta[c] = dispc[c];
            for (int c = 0; c < 3; c++) delta[c] -= dispa[c];
            for (int c = 0; c < 3; c++) delta[c] *= sr;
            double dispb[3];
            for (int c = 0; c < 3; c++) dispb[c] = delta[c];
            for (int c = 0; c < 3; c++) dispb[c] += dispa[c];
            // the regression normals come with the separation of the point cloud
            double deln = normals >= 5 ? N.cnorm[(4 * i + 3) * nn + n] : dot3(dispb, norm) - dot3(dispa, norm);
            mred *= massi;
            double delFi[3];
            if (postUpdate) {
                double fs[3] = {0., 0., 0.};
                for (int a = 0; a < numMats; a++)
                    for (int c = 0; c < 3; c++) fs[c] += N.ftot[(3 * act[a] + c) * nn + n];
                double sc = massi / Mc;
                for (int c = 0; c < 3; c++) delFi[c] = fs[c] * sc;
                for (int c = 0; c < 3; c++) delFi[c] += N.ftot[(3 * i + c) * nn + n] * -1.;
            }
            // the separation's momentum-update term is skipped for regression normals (CoulombFriction.cpp:162)
            if (!coulomb_delta(g, delPi, norm, dotn, deln, mred, postUpdate && normals < 5 ? delFi : nullptr)) continue;
        }
        change_momentum(g, N, i, n, delPi, callType);
        if (doingPairs) {
            for (int c = 0; c < 3; c++) delPi[c] *= -1.;
            change_momentum(g, N, j, n, delPi, callType);
        }
    }
}

// ---------------------------------------------------------------------------------------
// Regression contact normals (normals methods 5 and 6): CrackVelocityFieldMulti::
// LinearRegressionNormal and LogisticRegressionNormal (Nodes/MachineLearning.cpp:58-633) over the
// particles that see each contact node (MaterialContactNode::GetMaterialContactData,
// MaterialContactNode.cpp:253-350). A wave takes one contact node at a time: it lists the node's
// particles in LDS (cells and fields in a fixed order, particles of a cell in upload order), then
// the lanes split the list for every sum of the fit and a fixed reduction tree adds their parts,
// so each node's result is the same on every run.

// contact nodes of the step: two or more fields with particles (CalcTotalMassAndCount,
// PostExtrapolationTask.cpp:62-80); the count is cleared by the mass node pass before
template <int DIM>
__global__ void k_contact_list(KGrid g, KNodes N) {
    const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    bool on = false;
    if (n < g.nnodes) {
        int numMats = 0;
        for (int f = 0; f < g.nfields; f++) numMats += N.cnt[f * g.nstride + n] > 0 ? 1 : 0;
        on = numMats > 1;
    }
    const unsigned long long m = __ballot(on);
    if (m == 0ull) return;
    const int lane = (int)__lane_id();
    const int leader = __ffsll((long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(&N.clist[0], __popcll(m));
    base = __shfl(base, leader);
    if (on) N.clist[1 + base + __popcll(m & ((1ull << lane) - 1ull))] = (int)n;
}

// node (i,j,k) in particle p's shape-function node list (start-of-step shape functions):
// uGIMP/classic: inside the support on every axis; lCPDI: a corner's function at the node is
// at least 1e-15 (GetCPDIFunctions, MoreMPMElementBase.cpp:581-656)
template <int DIM, int SH>
__device__ __forceinline__ bool lr_member(const KGrid &g, const KPart &P, int p, int i, int j, int k) {
    int ei, ej, ek;
    elem_ijk(g, P.elem[p], ei, ej, ek);
    const int o[3] = {i - ei + 1, j - ej + 1, DIM == 3 ? k - ek + 1 : 1};
#pragma unroll
    for (int a = 0; a < DIM; a++)
        if (o[a] < 0 || o[a] > 3) return false;
    if (SH == MPMGPU_SHAPE_LCPDI) {
        CpdiCorners cc;
        cpdi_particle<DIM>(g, P, p, ei, ej, ek, cc);
        constexpr int NCOR = DIM == 3 ? 8 : 4;
        constexpr double thr = (DIM == 3 ? 8. : 4.) * 1e-15;
        bool in = false;
#pragma unroll
        for (int c = 0; c < NCOR; c++) {
            double T[DIM][4];
            cpdi_table<DIM>(cc.xi[c], cc.off[c], T);
            const double f = DIM == 3 ? T[0][o[0]] * T[1][o[1]] * T[2][o[2]] : T[0][o[0]] * T[1][o[1]];
            in |= f >= thr;
        }
        return in;
    }
    double xi[3], invd[3], S[3][4], dS[3][4];
    particle_xi<DIM>(g, ei, ej, ek, P.f(MPF_POS_X)[p], P.f(MPF_POS_Y)[p], DIM == 3 ? P.f(MPF_POS_Z)[p] : 0., xi, invd);
    particle_factors<DIM>(g, P, p, xi, S, dS);
    bool in = true;
#pragma unroll
    for (int a = 0; a < DIM; a++) in &= S[a][o[a]] >= 0.;
    return in;
}

// sum over the wave in a fixed tree, the total in every lane
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_down(v, off);
    return __shfl(v, 0);
}
__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmin(v, __shfl_down(v, off));
    return __shfl(v, 0);
}

// Matrix4::cofactor, determinant, Inverse and Times (Matrix4.cpp:96-103,133-140,206-231): the
// inverse as signed cofactors scaled by 1/det, then times rhs
__device__ __forceinline__ double lr_cofactor4(const double m[4][4], int row, int col) {
    double c[3][3];
    int cr = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (i == row) continue;
        int cc = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j == col) continue;
            c[cr][cc++] = m[i][j];
        }
        cr++;
    }
    return c[0][0] * (c[1][1] * c[2][2] - c[2][1] * c[1][2]) - c[1][0] * (c[0][1] * c[2][2] - c[2][1] * c[0][2]) +
           c[2][0] * (c[0][1] * c[1][2] - c[1][1] * c[0][2]);
}
__device__ __forceinline__ void lr_solve4(const double m[4][4], const double rhs[4], double out[4]) {
    const double det = m[0][0] * lr_cofactor4(m, 0, 0) - m[1][0] * lr_cofactor4(m, 1, 0) +
                       m[2][0] * lr_cofactor4(m, 2, 0) - m[3][0] * lr_cofactor4(m, 3, 0);
    const double f = 1. / det;
    double inv[4][4];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int c = 0; c < 4; c++) inv[r][c] = ((r + c) & 1 ? -lr_cofactor4(m, c, r) : lr_cofactor4(m, c, r)) * f;
#pragma unroll
    for (int r = 0; r < 4; r++) out[r] = inv[r][0] * rhs[0] + inv[r][1] * rhs[1] + inv[r][2] * rhs[2] + inv[r][3] * rhs[3];
}
// symmetric Matrix3 (Matrix3.cpp:107-121) Inverse (3D form, :446-460) times rhs (:394-408)
__device__ __forceinline__ void lr_solve3(const double s[6], const double rhs[3], double out[3]) {
    const double m[3][3] = {{s[0], s[1], s[2]}, {s[1], s[3], s[4]}, {s[2], s[4], s[5]}};
    double inv[3][3] = {{m[1][1] * m[2][2] - m[2][1] * m[1][2], -(m[0][1] * m[2][2] - m[2][1] * m[0][2]),
                         m[0][1] * m[1][2] - m[1][1] * m[0][2]},
                        {-(m[1][0] * m[2][2] - m[2][0] * m[1][2]), m[0][0] * m[2][2] - m[2][0] * m[0][2],
                         -(m[0][0] * m[1][2] - m[1][0] * m[0][2])},
                        {m[1][0] * m[2][1] - m[2][0] * m[1][1], -(m[0][0] * m[2][1] - m[2][0] * m[0][1]),
                         m[0][0] * m[1][1] - m[1][0] * m[0][1]}};
    const double det = m[0][0] * (m[1][1] * m[2][2] - m[2][1] * m[1][2]) -
                       m[1][0] * (m[0][1] * m[2][2] - m[2][1] * m[0][2]) + m[2][0] * (m[0][1] * m[1][2] - m[1][1] * m[0][2]);
    const double f = 1. / det;
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) inv[r][c] *= f;
#pragma unroll
    for (int r = 0; r < 3; r++) out[r] = inv[r][0] * rhs[0] + inv[r][1] * rhs[1] + inv[r][2] * rhs[2];
}

// MatPoint3D/MatPoint2D::GetDeformedRadius, ellipse methods (MatPoint3D.cpp:497-510,
// MatPoint2D.cpp:482-497): the distance from the particle's center to its deformed domain's
// surface along the unit vector n (2D applies F^-T where 3D applies F^-1, as the reference does)
template <int DIM>
__device__ __forceinline__ double lr_radius(const KGrid &g, const KPart &P, int p, const double n[3]) {
    double lpx, lpy, lpz;
    if (g.uniformLp) { lpx = g.lp[0]; lpy = g.lp[1]; lpz = g.lp[2]; }
    else { lpx = P.f(MPF_LP_X)[p]; lpy = P.f(MPF_LP_Y)[p]; lpz = P.f(MPF_LP_Z)[p]; }
    const double psx = g.dx * (0.5 * lpx), psy = g.dy * (0.5 * lpy);      // GetParticleSize
    if (DIM == 2) {
        const double exx = P.f(MPF_EP_XX)[p], eyy = P.f(MPF_EP_YY)[p], exy = P.f(MPF_EP_XY)[p], wxy = P.f(MPF_WR_XY)[p];
        const double F00 = 1. + exx, F01 = 0.5 * (exy - wxy), F10 = 0.5 * (exy + wxy), F11 = 1. + eyy;
        const double rdet2D = 1. / (F00 * F11 - F01 * F10);
        const double n0x = (F11 * n[0] - F10 * n[1]) * rdet2D;
        const double n0y = (-F01 * n[0] + F00 * n[1]) * rdet2D;
        return 1. / sqrt(n0x * n0x / (psx * psx) + n0y * n0y / (psy * psy));
    }
    const double psz = g.dz * (0.5 * lpz);
    double ep[6], wr[3], m[3][3];
#pragma unroll
    for (int c = 0; c < 6; c++) ep[c] = P.f(MPF_EP_XX + c)[p];
#pragma unroll
    for (int c = 0; c < 3; c++) wr[c] = P.f(MPF_WR_YZ + c)[p];
    get_F3(ep, wr, m);
    double inv[3][3] = {{m[1][1] * m[2][2] - m[2][1] * m[1][2], -(m[0][1] * m[2][2] - m[2][1] * m[0][2]),
                         m[0][1] * m[1][2] - m[1][1] * m[0][2]},
                        {-(m[1][0] * m[2][2] - m[2][0] * m[1][2]), m[0][0] * m[2][2] - m[2][0] * m[0][2],
                         -(m[0][0] * m[1][2] - m[1][0] * m[0][2])},
                        {m[1][0] * m[2][1] - m[2][0] * m[1][1], -(m[0][0] * m[2][1] - m[2][0] * m[0][1]),
                         m[0][0] * m[1][1] - m[1][0] * m[0][1]}};
    const double det = m[0][0] * (m[1][1] * m[2][2] - m[2][1] * m[1][2]) -
                       m[1][0] * (m[0][1] * m[2][2] - m[2][1] * m[0][2]) + m[2][0] * (m[0][1] * m[1][2] - m[1][1] * m[0][2]);
    const double f = 1. / det;
    double n0[3];
#pragma unroll
    for (int r = 0; r < 3; r++) n0[r] = (inv[r][0] * f) * n[0] + (inv[r][1] * f) * n[1] + (inv[r][2] * f) * n[2];
    return 1. / sqrt(n0[0] * n0[0] / (psx * psx) + n0[1] * n0[1] / (psy * psy) + n0[2] * n0[2] / (psz * psz));
}

#define LR_MAX 1024        // particles listed at one contact node (a wave's LDS list)

template <int DIM, int SH>
__global__ __launch_bounds__(NT) void k_contact_normals(KGrid g, KPart P, KBins B, KNodes N, const MpmMaterial *mats,
                                                        KStats st, int newPos) {
    constexpr int NW = NT / 64;
    __shared__ int s_list[NW][LR_MAX];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int *list = s_list[w];
    const int count = N.clist[0];
    const long long nn = g.nstride;
    const double *px = newPos ? P.posn(0) : P.f(MPF_POS_X);
    const double *py = newPos ? P.posn(1) : P.f(MPF_POS_Y);
    const double *pz = DIM == 3 ? (newPos ? P.posn(2) : P.f(MPF_POS_Z)) : nullptr;
    const bool logistic = g.normals == 6;
    for (int e = blockIdx.x * NW + w; e < count; e += gridDim.x * NW) {
        const long long n = N.clist[1 + e];
        const int i = (int)(n % g.nnx), j = (int)((n / g.nnx) % g.nny), k = DIM == 3 ? (int)(n / ((long long)g.nnx * g.nny)) : 0;
        const double nd[3] = {g.xmin + (double)i * g.dx, g.ymin + (double)j * g.dy, DIM == 3 ? g.zmin + (double)k * g.dz : 0.};
        int act[MPMGPU_MAX_MATERIALS];
        int numMats = 0;
        for (int f = 0; f < g.nfields; f++)
            if (N.cnt[f * nn + n] > 0) act[numMats++] = f;
        // the particles seeing the node: cells i-2..i+1 (per axis) of every field, in (field, z, y, x)
        // cell order and sorted order inside a cell. Lane q < 4^DIM holds cell q's slot range; a wave
        // prefix sum of the counts lays the field's particles out one after another, so every pass
        // tests 64 of them whatever the cells hold (the list comes out in the same order).
        constexpr int NCELL = DIM == 3 ? 64 : 16;
        int nl = 0;
        for (int f = 0; f < g.nfields; f++) {
            int cb = 0, cn = 0;
            if (lane < NCELL) {
                const int cx = i - 2 + (lane & 3), cy = j - 2 + ((lane >> 2) & 3);
                const int cz = DIM == 3 ? k - 2 + (lane >> 4) : 0;
                if (cx >= 0 && cx < g.nx && cy >= 0 && cy < g.ny && cz >= 0 && cz < g.nz) {
                    const int key = cell_key<DIM>(g, f, cx, cy, cz);
                    cb = B.cellStart[key];
                    cn = B.cellStart[key + 1] - cb;
                }
            }
            int incl = cn;                                   // inclusive prefix over the lanes
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int u = __shfl_up(incl, d);
                if (lane >= d) incl += u;
            }
            const int total = __shfl(incl, 63);
            for (int t0 = 0; t0 < total; t0 += 64) {
                const int t = t0 + lane;
                // the cell of flattened index t: the first lane whose inclusive prefix exceeds t
                int lo = 0, hi = NCELL - 1;
#pragma unroll
                for (int it = 0; it < (DIM == 3 ? 6 : 4); it++) {
                    const int mid = (lo + hi) >> 1;
                    if (__shfl(incl, mid) > t) hi = mid;
                    else lo = mid + 1;
                }
                const int qb = __shfl(cb, lo), qe = __shfl(incl - cn, lo);
                const int p = t < total ? B.order[qb + (t - qe)] : -1;
                const bool in = p >= 0 && lr_member<DIM, SH>(g, P, p, i, j, DIM == 3 ? k : 0);
                const unsigned long long m = __ballot(in);
                if (in) {
                    const int idx = nl + __popcll(m & ((1ull << lane) - 1ull));
                    if (idx < LR_MAX) list[idx] = p;
                }
                nl += __popcll(m);
            }
        }
        if (nl > LR_MAX) {
            if (lane == 0) atomicAdd(st.lrOverflow, 1ull);   // a fatal error, reported after the step
            nl = LR_MAX;
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int miMax = numMats == 2 ? 1 : numMats;
        for (int mi = 0; mi < miMax; mi++) {
            const int a = act[mi];
            double norm[3] = {0., 0., 0.}, linNorm[3] = {0., 0., 0.};
            const double cell = fmin(g.dx, fmin(g.dy, DIM == 3 ? g.dz : g.dy));     // GetMinCellDimension
            const double normPenalty = 1.e-7 * (cell * cell);
            if (DIM == 3) {
                double mt[10], rhs[4], lambda[4];
                if (logistic) { lambda[0] = lambda[1] = lambda[2] = normPenalty; lambda[3] = 0.; }
                else { lambda[0] = lambda[1] = lambda[2] = 0.; lambda[3] = 0.1; }
                for (int q = 0; q < 10; q++) mt[q] = 0.;
                for (int q = 0; q < 4; q++) rhs[q] = 0.;
                for (int t = lane; t < nl; t += 64) {
                    const int p = list[t];
                    const double mi_ = mats[P.mat[p]].field == a ? -1. : 1.;
                    const double x = px[p] - nd[0], y = py[p] - nd[1], z = pz[p] - nd[2];
                    mt[0] += x * x; mt[1] += x * y; mt[2] += x * z; mt[3] += x;
                    mt[4] += y * y; mt[5] += y * z; mt[6] += y;
                    mt[7] += z * z; mt[8] += z; mt[9] += 1.;
                    rhs[0] += mi_ * x; rhs[1] += mi_ * y; rhs[2] += mi_ * z; rhs[3] += mi_;
                }
                for (int q = 0; q < 10; q++) mt[q] = wave_sum(mt[q]);
                for (int q = 0; q < 4; q++) rhs[q] = wave_sum(rhs[q]);
                auto mat4 = [&](double M[4][4]) {
                    M[0][0] = mt[0] + lambda[0]; M[0][1] = mt[1]; M[0][2] = mt[2]; M[0][3] = mt[3];
                    M[1][0] = mt[1]; M[1][1] = mt[4] + lambda[1]; M[1][2] = mt[5]; M[1][3] = mt[6];
                    M[2][0] = mt[2]; M[2][1] = mt[5]; M[2][2] = mt[7] + lambda[2]; M[2][3] = mt[8];
                    M[3][0] = mt[3]; M[3][1] = mt[6]; M[3][2] = mt[8]; M[3][3] = mt[9] + lambda[3];
                };
                double M[4][4], beta[4];
                mat4(M);
                lr_solve4(M, rhs, beta);
                if (!logistic) {
                    const double magi = sqrt(beta[0] * beta[0] + beta[1] * beta[1] + beta[2] * beta[2]);
                    for (int c = 0; c < 3; c++) norm[c] = beta[c] * (1. / magi);
                } else {
                    for (int q = 0; q < 4; q++) beta[q] *= 2.;
                    double prevNorm[3] = {beta[0], beta[1], beta[2]};
                    double nmag = sqrt(dot3(prevNorm, prevNorm));
                    for (int c = 0; c < 3; c++) prevNorm[c] *= 1. / nmag;
                    for (int c = 0; c < 3; c++) linNorm[c] = prevNorm[c];
                    double delta = 1.;
                    int iter = 0;
                    while (delta > 1.e-5 && iter < 15) {
                        for (int q = 0; q < 10; q++) mt[q] = 0.;
                        for (int q = 0; q < 4; q++) rhs[q] = 0.;
                        for (int t = lane; t < nl; t += 64) {
                            const int p = list[t];
                            const double mi_ = mats[P.mat[p]].field == a ? -1. : 1.;
                            const double x = px[p] - nd[0], y = py[p] - nd[1], z = pz[p] - nd[2];
                            const double dotp = x * beta[0] + y * beta[1] + z * beta[2] + beta[3];
                            const double arg = 1. + exp(-dotp);
                            const double phi = 2. * (arg - 1.) / (arg * arg);
                            const double phi2 = phi * phi;
                            mt[0] += phi2 * x * x; mt[1] += phi2 * x * y; mt[2] += phi2 * x * z; mt[3] += phi2 * x;
                            mt[4] += phi2 * y * y; mt[5] += phi2 * y * z; mt[6] += phi2 * y;
                            mt[7] += phi2 * z * z; mt[8] += phi2 * z; mt[9] += phi2;
                            const double mifi = (mi_ - 2. / arg + 1.) * phi;
                            rhs[0] += mifi * x; rhs[1] += mifi * y; rhs[2] += mifi * z; rhs[3] += mifi;
                        }
                        for (int q = 0; q < 10; q++) mt[q] = wave_sum(mt[q]);
                        // the penalty term starts the right-hand side (MachineLearning.cpp:327-328)
                        for (int q = 0; q < 4; q++) rhs[q] = -lambda[q] * beta[q] + wave_sum(rhs[q]);
                        mat4(M);
                        double dbeta[4];
                        lr_solve4(M, rhs, dbeta);
                        for (int q = 0; q < 4; q++) beta[q] += dbeta[q];
                        for (int c = 0; c < 3; c++) norm[c] = beta[c];
                        nmag = sqrt(dot3(norm, norm));
                        for (int c = 0; c < 3; c++) norm[c] *= 1. / nmag;
                        delta = 1. - dot3(norm, prevNorm);
                        iter++;
                        for (int c = 0; c < 3; c++) prevNorm[c] = norm[c];
                    }
                }
            } else {
                double mt[6], rhs[3];
                double lambda[3] = {0., 0., 0.1};
                if (logistic) { lambda[0] = normPenalty; lambda[1] = normPenalty; lambda[2] = 0.; }
                for (int q = 0; q < 6; q++) mt[q] = 0.;
                for (int q = 0; q < 3; q++) rhs[q] = 0.;
                for (int t = lane; t < nl; t += 64) {
                    const int p = list[t];
                    const double mi_ = mats[P.mat[p]].field == a ? -1. : 1.;
                    const double x = px[p] - nd[0], y = py[p] - nd[1];
                    mt[0] += x * x; mt[1] += x * y; mt[2] += x;
                    mt[3] += y * y; mt[4] += y; mt[5] += 1.;
                    rhs[0] += mi_ * x; rhs[1] += mi_ * y; rhs[2] += mi_;
                }
                for (int q = 0; q < 6; q++) mt[q] = wave_sum(mt[q]);
                for (int q = 0; q < 3; q++) rhs[q] = wave_sum(rhs[q]);
                double beta[3];
                double S[6] = {mt[0] + lambda[0], mt[1], mt[2], mt[3] + lambda[1], mt[4], mt[5] + lambda[2]};
                lr_solve3(S, rhs, beta);
                if (!logistic) {
                    norm[0] = beta[0]; norm[1] = beta[1];
                    const double magi = sqrt(dot3(norm, norm));
                    for (int c = 0; c < 3; c++) norm[c] *= 1. / magi;
                } else {
                    for (int q = 0; q < 3; q++) beta[q] *= 2.;
                    double prevNorm[3] = {beta[0], beta[1], beta[2]};
                    double nmag = sqrt(beta[0] * beta[0] + beta[1] * beta[1]);
                    prevNorm[0] /= nmag; prevNorm[1] /= nmag;
                    linNorm[0] = prevNorm[0]; linNorm[1] = prevNorm[1];
                    double delta = 1., nv[3] = {0., 0., 0.};
                    int iter = 0;
                    while (delta > 1.e-5 && iter < 15) {
                        for (int q = 0; q < 6; q++) mt[q] = 0.;
                        for (int q = 0; q < 3; q++) rhs[q] = 0.;
                        for (int t = lane; t < nl; t += 64) {
                            const int p = list[t];
                            const double mi_ = mats[P.mat[p]].field == a ? -1. : 1.;
                            const double x = px[p] - nd[0], y = py[p] - nd[1], z = 1.;
                            const double arg = 1. + exp(-(x * beta[0] + y * beta[1] + z * beta[2]));
                            const double phi = 2. * (arg - 1.) / (arg * arg);
                            const double phi2 = phi * phi;
                            mt[0] += phi2 * x * x; mt[1] += phi2 * x * y; mt[2] += phi2 * x;
                            mt[3] += phi2 * y * y; mt[4] += phi2 * y; mt[5] += phi2;
                            const double mifi = (mi_ - 2. / arg + 1.) * phi;
                            rhs[0] += mifi * x; rhs[1] += mifi * y; rhs[2] += mifi;
                        }
                        for (int q = 0; q < 6; q++) mt[q] = wave_sum(mt[q]);
                        for (int q = 0; q < 3; q++) rhs[q] = -lambda[q] * beta[q] + wave_sum(rhs[q]);
                        double S2[6] = {mt[0] + lambda[0], mt[1], mt[2], mt[3] + lambda[1], mt[4], mt[5] + lambda[2]};
                        double dbeta[3];
                        lr_solve3(S2, rhs, dbeta);
                        for (int q = 0; q < 3; q++) beta[q] += dbeta[q];
                        for (int q = 0; q < 3; q++) nv[q] = beta[q];
                        nmag = sqrt(nv[0] * nv[0] + nv[1] * nv[1]);
                        nv[0] /= nmag; nv[1] /= nmag;
                        delta = 1. - nv[0] * prevNorm[0] - nv[1] * prevNorm[1];
                        iter++;
                        for (int q = 0; q < 3; q++) prevNorm[q] = nv[q];
                    }
                    norm[0] = nv[0]; norm[1] = nv[1]; norm[2] = 0.;
                }
            }
            if (logistic && norm[0] != norm[0])
                for (int c = 0; c < 3; c++) norm[c] = linNorm[c];
            // separation from the point cloud (MachineLearning.cpp:195-226, 614-633)
            double supA = 1.e30, supB = 1.e30;
            for (int t = lane; t < nl; t += 64) {
                const int p = list[t];
                const double xp[3] = {px[p], py[p], DIM == 3 ? pz[p] : 0.};
                const double r = lr_radius<DIM>(g, P, p, norm);
                if (mats[P.mat[p]].field == a) supA = fmin(supA, -dot3(norm, xp) - r);
                else supB = fmin(supB, dot3(norm, xp) - r);
            }
            supA = wave_min(supA);
            supB = wave_min(supB);
            if (lane == 0) {
#pragma unroll
                for (int c = 0; c < 3; c++) N.cnorm[(4 * a + c) * nn + n] = norm[c];
                N.cnorm[(4 * a + 3) * nn + n] = supA + supB;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ---------------------------------------------------------------------------------------
// launchers
static int g_cus = 256;
static inline unsigned blocks_for(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

void launch_bin_keys(int dim, const KGrid &g, const KPart &p, const KBins &b, hipStream_t s) {
    if (p.n == 0) return;
    if (dim == 3) hipLaunchKernelGGL(k_bin_keys<3>, dim3(blocks_for(p.n, NT)), dim3(NT), 0, s, g, p, b);
    else hipLaunchKernelGGL(k_bin_keys<2>, dim3(blocks_for(p.n, NT)), dim3(NT), 0, s, g, p, b);
}

void launch_bin_finish(int dim, const KGrid &g, const KPart &p, const KBins &b, hipStream_t s) {
    const int n = b.nkeys + 1;    // count[nkeys] stays zero, so cellStart[nkeys] = total
    const int nb = (n + SCAN_BLOCK - 1) / SCAN_BLOCK;
    constexpr int NC3 = TileGeom<3>::NC, NC2 = TileGeom<2>::NC;
    const unsigned need = blocks_for(b.ntall, NT), rows = blocks_for(p.n, NT);
    if (dim == 3) {
        hipLaunchKernelGGL(k_bin_scan<NC3>, dim3(nb), dim3(SCAN_NT), 0, s, b, n, nb);
        hipLaunchKernelGGL(k_bin_scatter<3>, dim3(need + rows), dim3(NT), 0, s, g, p, b, (int)need);
    } else {
        hipLaunchKernelGGL(k_bin_scan<NC2>, dim3(nb), dim3(SCAN_NT), 0, s, b, n, nb);
        hipLaunchKernelGGL(k_bin_scatter<2>, dim3(need + rows), dim3(NT), 0, s, g, p, b, (int)need);
    }
    const unsigned cells = std::min<unsigned>(blocks_for(b.nkeys, NT), 16 * g_cus);
    hipLaunchKernelGGL(k_bin_sort_cells, dim3(cells), dim3(NT), 0, s, b, dim == 3 ? NC3 : NC2, nb);
}

void set_tile_cus(int cus) { g_cus = cus > 0 ? cus : 256; }

// Workgroups of one tile-kernel launch, at most one per (field, tile) pair. Kernels that fill a CU with one
// or two blocks take no more than the device holds at once: further blocks would wait for the end of those
// to find no tile left (262k particles in 512 tiles: 204 us per step with twice as many, 195 without).
// Others take twice as many, whose start hides the claims between short tiles (1.7M particles of 2D
// instances: 523 without, 516; eight blocks per CU for every kernel: 518, and 885k particles 449 for 445).
static int kernel_blocks(const void *kernel, int threads) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) != hipSuccess || n < 1) return 8;
    return n <= 2 ? n : 2 * n;
}
static dim3 tile_grid_dim(const KBins &b, int perCu) {
    const long long want = (long long)perCu * g_cus;
    return dim3((unsigned)(b.ntall < want ? b.ntall : want));
}
static KBins tile_bins(const KBins &b, int slot) {
    KBins r = b;
    r.slot = slot;
    return r;
}
#define TILE_LAUNCH_NT(NT, KERNEL, B, S, ...)                                                                    \
    do {                                                                                                         \
        static const int perCu = kernel_blocks(reinterpret_cast<const void *>(&KERNEL), NT);                     \
        hipLaunchKernelGGL(KERNEL, tile_grid_dim(B, perCu), dim3(NT), 0, S, __VA_ARGS__);                        \
    } while (0)
#define TILE_LAUNCH(KERNEL, B, S, ...) TILE_LAUNCH_NT(NT, KERNEL, B, S, __VA_ARGS__)

void launch_p2g_mass(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                     const MpmMaterial *mats, const KStats &st, hipStream_t s) {
    const KBins tb = tile_bins(b, TILE_SLOT_MASS);
    (void)mats;
    const bool cp = g.shape == MPMGPU_SHAPE_LCPDI;
    if (dim == 3) {
        if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(3), k_p2g_mass_corners<3>, tb, s, g, p, tb, nd, st);
        else TILE_LAUNCH_NT(64 * UGIMP_NW, k_p2g_mass<3>, tb, s, g, p, tb, nd);
    } else {
        if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(2), k_p2g_mass_corners<2>, tb, s, g, p, tb, nd, st);
        else TILE_LAUNCH_NT(64 * UGIMP_NW, k_p2g_mass<2>, tb, s, g, p, tb, nd);
    }
}

void launch_node_mass(int dim, const KGrid &g, const KBins &b, const KNodes &nd, hipStream_t s) {
    if (dim == 3) hipLaunchKernelGGL(k_node_mass<3>, dim3(blocks_for(g.nstride * g.nfields, NT)), dim3(NT), 0, s, g, b, nd);
    else hipLaunchKernelGGL(k_node_mass<2>, dim3(blocks_for(g.nstride * g.nfields, NT)), dim3(NT), 0, s, g, b, nd);
}

template <int DIM, int SH>
static void usf_mat(int mat, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                    const MpmMaterial *mats, int only, int slot, hipStream_t s) {
    const KBins tb = tile_bins(b, slot);
    switch (mat) {
        case MPMGPU_MAT_ISOTROPIC:
            TILE_LAUNCH((k_usf<DIM, MPMGPU_MAT_ISOTROPIC, SH>), tb, s, g, p, tb, nd, mats, only); break;
        case MPMGPU_MAT_ISOPLASTICITY:
            TILE_LAUNCH((k_usf<DIM, MPMGPU_MAT_ISOPLASTICITY, SH>), tb, s, g, p, tb, nd, mats, only); break;
        case MPMGPU_MAT_NEOHOOKEAN:
            TILE_LAUNCH((k_usf<DIM, MPMGPU_MAT_NEOHOOKEAN, SH>), tb, s, g, p, tb, nd, mats, only); break;
        case MPMGPU_MAT_MOONEY:
            TILE_LAUNCH((k_usf<DIM, MPMGPU_MAT_MOONEY, SH>), tb, s, g, p, tb, nd, mats, only); break;
        default:
            TILE_LAUNCH((k_usf<DIM, 0, SH>), tb, s, g, p, tb, nd, mats, only); break;
    }
}

// the strain updates of a launch: one launch with the law of every particle when they share a
// type (or the grid has no per-tile types), else one launch per type present, each taking only the
// tiles of its type, and one with every law for tiles whose instance mixes types
template <typename L>
static void by_type(const KGrid &g, int firstTypedSlot, int plainSlot, L launch) {
    if (g.matType != 0 || !g.tileType) {
        launch(g.matType, -1, plainSlot);
        return;
    }
    for (int j = 0; j < g.ntypes; j++) launch(g.types[j], g.types[j], firstTypedSlot + j);
    if (g.anyMixed) launch(0, 0, plainSlot);
}

template <int DIM>
static void usf_force_mat(int mat, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd, const MpmMaterial *mats,
                          int only, int slot, hipStream_t s) {
    const KBins tb = tile_bins(b, slot);
#define FUSED_LAUNCH(MAT) TILE_LAUNCH_NT(64 * UGIMP_NW, (k_usf_force<DIM, MAT>), tb, s, g, p, tb, nd, mats, only)
    switch (mat) {
        case MPMGPU_MAT_ISOTROPIC: FUSED_LAUNCH(MPMGPU_MAT_ISOTROPIC); break;
        case MPMGPU_MAT_ISOPLASTICITY: FUSED_LAUNCH(MPMGPU_MAT_ISOPLASTICITY); break;
        case MPMGPU_MAT_NEOHOOKEAN: FUSED_LAUNCH(MPMGPU_MAT_NEOHOOKEAN); break;
        case MPMGPU_MAT_MOONEY: FUSED_LAUNCH(MPMGPU_MAT_MOONEY); break;
        default: FUSED_LAUNCH(0); break;
    }
#undef FUSED_LAUNCH
}

bool launch_usf_force(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd, const KLoads &L,
                      const MpmMaterial *mats, hipStream_t s) {
    if (g.shape == MPMGPU_SHAPE_LCPDI || L.nl > 0) return false;
    by_type(g, TILE_SLOT_TYPED, TILE_SLOT_USF, [&](int mat, int only, int slot) {
        if (dim == 3) usf_force_mat<3>(mat, g, p, b, nd, mats, only, slot, s);
        else usf_force_mat<2>(mat, g, p, b, nd, mats, only, slot, s);
    });
    return true;
}

void launch_usf(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                const MpmMaterial *mats, hipStream_t s) {
    const bool cp = g.shape == MPMGPU_SHAPE_LCPDI;
    by_type(g, TILE_SLOT_TYPED, TILE_SLOT_USF, [&](int mat, int only, int slot) {
        if (dim == 3) {
            if (cp) usf_mat<3, MPMGPU_SHAPE_LCPDI>(mat, g, p, b, nd, mats, only, slot, s);
            else usf_mat<3, MPMGPU_SHAPE_UGIMP>(mat, g, p, b, nd, mats, only, slot, s);
        } else {
            if (cp) usf_mat<2, MPMGPU_SHAPE_LCPDI>(mat, g, p, b, nd, mats, only, slot, s);
            else usf_mat<2, MPMGPU_SHAPE_UGIMP>(mat, g, p, b, nd, mats, only, slot, s);
        }
    });
}

// BoundaryCondition::GetNodeNum and BCValue (BoundaryCondition.cpp:72-140): 1 if the condition
// acts at time t, its value in v
__device__ __forceinline__ int style_value(int style, double val, double ft, double t, double &v) {
    v = 0.;
    switch (style) {
        case 1: if (t >= ft) { v = val; return 1; } return 0;
        case 2: if (t >= ft) { v = 0. + val * (t - ft); return 1; } return 0;
        case 3: v = val * sin(t * ft); return 1;
        case 4: v = val * cos(t * ft); return 1;
        default: return 0;
    }
}

// ---------------------------------------------------------------------------------------
// Traction conditions (MatPtTractionBC::AddMPFluxBC, MatPtTractionBC.cpp:64-227: planar and 3D,
// no cracks, no ExactTractions). GetSurfaceInfo (MatPoint2D.cpp:1138-1300, MatPoint3D.cpp:628-851)
// gives the corners of the loaded face and hat n times its weight: uGIMP and classic particles
// take the corners of the undeformed particle and the size of the deformed face, lCPDI particles
// the deformed corners and their own face. Each corner's element adds its linear shape functions
// at the corner (GetShapeFunctionsForTractions, MoreMPMElementBase.cpp:91-107) times
// tmag * weight to the particle's material field at the element's nodes where that field has
// points (NodalPoint::AddTractionTask3, NodalPointMPM.cpp:644-650).

// signs of r1, r2 (and r3) at the corners of each face, in the reference's corner order
__constant__ signed char k_face_corners2[4][2][2] = {
    {{-1, -1}, {1, -1}}, {{1, -1}, {1, 1}}, {{1, 1}, {-1, 1}}, {{-1, 1}, {-1, -1}}};
__constant__ signed char k_face_corners3[6][4][3] = {
    {{-1, -1, -1}, {1, -1, -1}, {1, -1, 1}, {-1, -1, 1}},    // 1: -y, nodes 1, 2, 6, 5
    {{1, -1, -1}, {1, 1, -1}, {1, 1, 1}, {1, -1, 1}},        // 2: +x, nodes 2, 3, 7, 6
    {{1, 1, -1}, {-1, 1, -1}, {-1, 1, 1}, {1, 1, 1}},        // 3: +y, nodes 3, 4, 8, 7
    {{-1, 1, -1}, {-1, -1, -1}, {-1, -1, 1}, {-1, 1, 1}},    // 4: -x, nodes 4, 1, 5, 8
    {{1, -1, -1}, {-1, -1, -1}, {-1, 1, -1}, {1, 1, -1}},    // 5: -z, nodes 2, 1, 4, 3
    {{-1, -1, 1}, {1, -1, 1}, {1, 1, 1}, {-1, 1, 1}}};       // 6: +z, nodes 5, 6, 7, 8

__device__ __forceinline__ void cross3(const double a[3], const double b[3], double c[3]) {
    c[0] = a[1] * b[2] - b[1] * a[2];          // CrossProduct (CommonUtilities.cpp:215-221)
    c[1] = b[0] * a[2] - a[0] * b[2];
    c[2] = a[0] * b[1] - b[0] * a[1];
}

// corners (cx[k]) and weighted normal (wn) of one face; returns the corner count
template <int DIM>
__device__ int surface_info(const KGrid &g, const KPart &P, int p, int ei, int ej, int ek, int face, int dof,
                            double thick, double cx[4][3], double wn[3]) {
    double r[9];
    cpdi_semi_sides<DIM>(g, P, p, ei, ej, ek, r);            // deformed semi sides F (psz)
    double *r1 = r, *r2 = r + 3, *r3 = r + 6;
    double uG = -1.;
    if (g.shape != MPMGPU_SHAPE_LCPDI) {
        if (DIM == 3) {
            double ap[3];
            if (face == 1 || face == 3) cross3(r1, r3, ap);
            else if (face == 2 || face == 4) cross3(r2, r3, ap);
            else cross3(r1, r2, ap);
            uG = sqrt(ap[0] * ap[0] + ap[1] * ap[1] + ap[2] * ap[2]);
        } else {
            const double *rs = (face == 1 || face == 3) ? r1 : r2;
            uG = sqrt(rs[0] * rs[0] + rs[1] * rs[1] + rs[2] * rs[2]);
        }
        // the undeformed semi sides (GetUndeformedSemiSides)
        double lpx, lpy, lpz;
        if (g.uniformLp) { lpx = g.lp[0]; lpy = g.lp[1]; lpz = g.lp[2]; }
        else { lpx = P.f(MPF_LP_X)[p]; lpy = P.f(MPF_LP_Y)[p]; lpz = P.f(MPF_LP_Z)[p]; }
        const double ux = ((g.xmin + (double)(ei + 1) * g.dx) - (g.xmin + (double)ei * g.dx)) * (0.5 * lpx);
        const double uy = ((g.ymin + (double)(ej + 1) * g.dy) - (g.ymin + (double)ej * g.dy)) * (0.5 * lpy);
        const double uz = DIM == 3 ? ((g.zmin + (double)(ek + 1) * g.dz) - (g.zmin + (double)ek * g.dz)) * (0.5 * lpz) : 0.;
#pragma unroll
        for (int a = 0; a < 9; a++) r[a] = 0.;
        r1[0] = ux; r2[1] = uy; r3[2] = uz;
    }
    const double pos[3] = {P.f(MPF_POS_X)[p], P.f(MPF_POS_Y)[p], DIM == 3 ? P.f(MPF_POS_Z)[p] : 0.};
    const int nc = DIM == 3 ? 4 : 2;
    for (int k = 0; k < nc; k++) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            if (DIM == 3) {
                const signed char *sg = k_face_corners3[face - 1][k];
                cx[k][a] = ((pos[a] + (double)sg[0] * r1[a]) + (double)sg[1] * r2[a]) + (double)sg[2] * r3[a];
            } else {
                const signed char *sg = k_face_corners2[face - 1][k];
                cx[k][a] = a < 2 ? (pos[a] + (double)sg[0] * r1[a]) + (double)sg[1] * r2[a] : 0.;
            }
        }
    }
    wn[0] = wn[1] = wn[2] = 0.;
    double r0[3];
#pragma unroll
    for (int a = 0; a < 3; a++) r0[a] = 0.5 * (cx[1][a] - cx[0][a]);
    if (DIM == 3) {
        double r1f[3], ap[3];
#pragma unroll
        for (int a = 0; a < 3; a++) r1f[a] = 0.5 * (cx[3][a] - cx[0][a]);
        cross3(r0, r1f, ap);
        const double am = sqrt(ap[0] * ap[0] + ap[1] * ap[1] + ap[2] * ap[2]);
        const double faceWt = uG < 0. ? am : uG;
        if (dof == 1) wn[0] = faceWt;
        else if (dof == 2) wn[1] = faceWt;
        else if (dof == 11) {
            const double sc = uG > 0. ? uG / am : 1.;
#pragma unroll
            for (int a = 0; a < 3; a++) wn[a] = uG > 0. ? ap[a] * sc : ap[a];
        } else wn[2] = faceWt;
    } else {
        double faceWt = uG < 0. ? sqrt(r0[0] * r0[0] + r0[1] * r0[1] + r0[2] * r0[2]) : uG;
        faceWt *= thick;
        if (dof == 1) wn[0] = faceWt;
        else if (dof == 2) wn[1] = faceWt;
        else if (dof == 11 || dof == 12) {
            const double ex = dof == 11 ? r0[1] : r0[0], ey = dof == 11 ? -r0[0] : r0[1];
            const double en = sqrt(ex * ex + ey * ey);
            wn[0] = ex * faceWt / en;
            wn[1] = ey * faceWt / en;
        } else wn[2] = faceWt;
    }
    return nc;
}

// the nodal traction forces of traction table t (particle p) at step time tt
template <int DIM>
__device__ void particle_tractions(const KGrid &g, const KPart &P, const KNodes &N, const KLoads &L, int p, int t,
                                   double tt) {
    double *tab = L.ttab + (size_t)3 * t * TRAC_NODES;
    for (int o = 0; o < 3 * TRAC_NODES; o++) tab[o] = 0.;
    int ei, ej, ek;
    elem_ijk(g, P.elem[p], ei, ej, ek);
    const int fld = g.fieldOf[P.mat[p]];
    const KNodes Nf = field_view(g, N, fld);
    for (int e = L.tstart[t]; e < L.tstart[t + 1]; e++) {
        double tmag;
        style_value(L.tstyle[e], L.tvalue[e], L.tftime[e], tt, tmag);
        double cx[4][3], wn[3];
        const int nc = surface_info<DIM>(g, P, p, ei, ej, ek, L.tface[e], L.tdir[e], L.tthick[t], cx, wn);
        for (int k = 0; k < nc; k++) {
            bool ok = true;
            const int ci = find_cell(cx[k][0], g.xmin, g.dx, g.nx, ok);
            const int cj = find_cell(cx[k][1], g.ymin, g.dy, g.ny, ok);
            const int ck = DIM == 3 ? find_cell(cx[k][2], g.zmin, g.dz, g.nz, ok) : 0;
            const int ox = ci - ei, oy = cj - ej, oz = DIM == 3 ? ck - ek : 0;
            if (!ok || ox < -1 || ox > 1 || oy < -1 || oy > 1 || oz < -1 || oz > 1) {
                atomicAdd(L.terr, 1ull);          // a fatal error, reported after the step
                continue;
            }
            double xi[3], invd[3];
            particle_xi<DIM>(g, ci, cj, ck, cx[k][0], cx[k][1], cx[k][2], xi, invd);
            for (int jz = 0; jz < (DIM == 3 ? 2 : 1); jz++)
                for (int jy = 0; jy < 2; jy++)
                    for (int jx = 0; jx < 2; jx++) {
                        const long long n = ((long long)(ck + jz) * g.nny + (cj + jy)) * g.nnx + (ci + jx);
                        if (Nf.cnt[n] <= 0) continue;
                        const double fn = cpdi_cfn<DIM>(xi, jx, jy, jz);
                        const int o = DIM == 3 ? ((oz + jz + 1) * 4 + (oy + jy + 1)) * 4 + (ox + jx + 1)
                                               : (oy + jy + 1) * 4 + (ox + jx + 1);
#pragma unroll
                        for (int c = 0; c < DIM; c++) tab[c * TRAC_NODES + o] += wn[c] * (tmag * fn);
                    }
        }
    }
}

// marks the (field, tile) of every loaded particle in slot par, clears slot par ^ 1 for the next
// step, and fills the traction tables of the step (PostForcesTask.cpp:51, after the grid forces'
// strain update and the mass pass that sets the point counts)
template <int DIM>
__global__ void k_mark_load_tiles(KGrid g, KPart P, KBins B, KNodes N, KLoads L, int par) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < B.ntall) L.tflag[par ^ 1][p] = 0;
    if (p >= P.n) return;
    const int q = L.map[B.home[p]];
    if (q < 0) return;
    L.tflag[par][B.key[p] / TileGeom<DIM>::NC] = 1;
    if (L.nt > 0 && L.tslot[q] >= 0) particle_tractions<DIM>(g, P, N, L, (int)p, L.tslot[q], L.time[par]);
}

void launch_p2g_force(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd, const KLoads &L,
                      int par, hipStream_t s) {
    const KBins tb = tile_bins(b, TILE_SLOT_FORCE);
    const bool cp = g.shape == MPMGPU_SHAPE_LCPDI;
    const int *loaded = nullptr;
    if (L.nl > 0) {
        const long long n = std::max<long long>(p.n, b.ntall);
        if (dim == 3) hipLaunchKernelGGL(k_mark_load_tiles<3>, dim3(blocks_for(n, NT)), dim3(NT), 0, s, g, p, b, nd, L, par);
        else hipLaunchKernelGGL(k_mark_load_tiles<2>, dim3(blocks_for(n, NT)), dim3(NT), 0, s, g, p, b, nd, L, par);
        loaded = L.tflag[par];
        const KBins tl = tile_bins(b, TILE_SLOT_FORCE_LOADS);
        if (dim == 3) {
            if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(3), (k_p2g_force_corners<3, true>), tl, s, g, p, tl, nd, L, loaded);
            else TILE_LAUNCH_NT(64 * UGIMP_NW, (k_p2g_force<3, true>), tl, s, g, p, tl, nd, L, loaded);
        } else {
            if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(2), (k_p2g_force_corners<2, true>), tl, s, g, p, tl, nd, L, loaded);
            else TILE_LAUNCH_NT(64 * UGIMP_NW, (k_p2g_force<2, true>), tl, s, g, p, tl, nd, L, loaded);
        }
    }
    if (dim == 3) {
        if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(3), (k_p2g_force_corners<3, false>), tb, s, g, p, tb, nd, L, loaded);
        else TILE_LAUNCH_NT(64 * UGIMP_NW, (k_p2g_force<3, false>), tb, s, g, p, tb, nd, L, loaded);
    } else {
        if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(2), (k_p2g_force_corners<2, false>), tb, s, g, p, tb, nd, L, loaded);
        else TILE_LAUNCH_NT(64 * UGIMP_NW, (k_p2g_force<2, false>), tb, s, g, p, tb, nd, L, loaded);
    }
}

void launch_node_force(int dim, const KGrid &g, const KBins &b, const KNodes &nd, hipStream_t s) {
    if (dim == 3) hipLaunchKernelGGL(k_node_force<3>, dim3(blocks_for(g.nstride * g.nfields, NT)), dim3(NT), 0, s, g, b, nd);
    else hipLaunchKernelGGL(k_node_force<2>, dim3(blocks_for(g.nstride * g.nfields, NT)), dim3(NT), 0, s, g, b, nd);
}

template <int MOVE>
static void g2p_move(int dim, const KGrid &g, const KPart &p, const KBins &tb, const KNodes &nd,
                     const MpmMaterial *mats, int mode, hipStream_t s) {
    const bool cp = g.shape == MPMGPU_SHAPE_LCPDI;
    if (dim == 3) {
        if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(3), (k_g2p_p2g_corners<3, MOVE>), tb, s, g, p, tb, nd, mats, mode);
        else TILE_LAUNCH_NT(64 * G2P_NW(3), (k_g2p_p2g<3, MOVE>), tb, s, g, p, tb, nd, mats, mode);
    } else {
        if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(2), (k_g2p_p2g_corners<2, MOVE>), tb, s, g, p, tb, nd, mats, mode);
        else TILE_LAUNCH_NT(64 * G2P_NW(2), (k_g2p_p2g<2, MOVE>), tb, s, g, p, tb, nd, mats, mode);
    }
}

void launch_g2p_p2g(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                    const MpmMaterial *mats, int mode, hipStream_t s) {
    const KBins tb = tile_bins(b, TILE_SLOT_G2P);
    // damping and the FMPM/XPIC moves have their own instances, so the plain FLIP update keeps its registers
    if (mode != 0) g2p_move<G2P_SERIES>(dim, g, p, tb, nd, mats, mode, s);
    else if (g.damped) g2p_move<G2P_FLIP_DAMPED>(dim, g, p, tb, nd, mats, mode, s);
    else g2p_move<G2P_FLIP>(dim, g, p, tb, nd, mats, mode, s);
}

void launch_node_mom2(int dim, const KGrid &g, const KBins &b, const KNodes &nd, hipStream_t s) {
    if (dim == 3) hipLaunchKernelGGL(k_node_mom2<3>, dim3(blocks_for(g.nstride * g.nfields, NT)), dim3(NT), 0, s, g, b, nd);
    else hipLaunchKernelGGL(k_node_mom2<2>, dim3(blocks_for(g.nstride * g.nfields, NT)), dim3(NT), 0, s, g, b, nd);
}

template <int DIM, int SH>
static void usl_reset_mat(int mat, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                          const MpmMaterial *mats, const KStats &st, int only, int slot, hipStream_t s) {
    const KBins tb = tile_bins(b, slot);
    switch (mat) {
        case MPMGPU_MAT_ISOTROPIC:
            TILE_LAUNCH((k_usl_reset<DIM, MPMGPU_MAT_ISOTROPIC, SH>), tb, s, g, p, tb, nd, mats, st, only); break;
        case MPMGPU_MAT_ISOPLASTICITY:
            TILE_LAUNCH((k_usl_reset<DIM, MPMGPU_MAT_ISOPLASTICITY, SH>), tb, s, g, p, tb, nd, mats, st, only); break;
        case MPMGPU_MAT_NEOHOOKEAN:
            TILE_LAUNCH((k_usl_reset<DIM, MPMGPU_MAT_NEOHOOKEAN, SH>), tb, s, g, p, tb, nd, mats, st, only); break;
        case MPMGPU_MAT_MOONEY:
            TILE_LAUNCH((k_usl_reset<DIM, MPMGPU_MAT_MOONEY, SH>), tb, s, g, p, tb, nd, mats, st, only); break;
        default:
            TILE_LAUNCH((k_usl_reset<DIM, 0, SH>), tb, s, g, p, tb, nd, mats, st, only); break;
    }
}

void launch_usl_reset(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                      const MpmMaterial *mats, const KStats &st, hipStream_t s) {
    const bool cp = g.shape == MPMGPU_SHAPE_LCPDI;
    by_type(g, TILE_SLOT_TYPED + 4, TILE_SLOT_USL, [&](int mat, int only, int slot) {
        if (dim == 3) {
            if (cp) usl_reset_mat<3, MPMGPU_SHAPE_LCPDI>(mat, g, p, b, nd, mats, st, only, slot, s);
            else usl_reset_mat<3, MPMGPU_SHAPE_UGIMP>(mat, g, p, b, nd, mats, st, only, slot, s);
        } else {
            if (cp) usl_reset_mat<2, MPMGPU_SHAPE_LCPDI>(mat, g, p, b, nd, mats, st, only, slot, s);
            else usl_reset_mat<2, MPMGPU_SHAPE_UGIMP>(mat, g, p, b, nd, mats, st, only, slot, s);
        }
    });
}

void launch_p2g_contact(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                        const MpmMaterial *mats, bool newPositions, hipStream_t s) {
    const KBins tb = tile_bins(b, newPositions ? TILE_SLOT_CONTACT_LAST : TILE_SLOT_CONTACT_FIRST);
    int np = newPositions ? 1 : 0;
    const bool cp = g.shape == MPMGPU_SHAPE_LCPDI;
    if (dim == 3) {
        if (cp) TILE_LAUNCH_NT(64 * UGIMP_NW, k_p2g_contact_corners<3>, tb, s, g, p, tb, nd, mats, np);
        else TILE_LAUNCH_NT(64 * UGIMP_NW, k_p2g_contact<3>, tb, s, g, p, tb, nd, mats, np);
    } else {
        if (cp) TILE_LAUNCH_NT(64 * UGIMP_NW, k_p2g_contact_corners<2>, tb, s, g, p, tb, nd, mats, np);
        else TILE_LAUNCH_NT(64 * UGIMP_NW, k_p2g_contact<2>, tb, s, g, p, tb, nd, mats, np);
    }
}

void launch_node_contact(int dim, const KGrid &g, const KBins &b, const KNodes &nd, hipStream_t s) {
    if (dim == 3) hipLaunchKernelGGL(k_node_contact<3>, dim3(blocks_for(g.nstride * g.nfields, NT)), dim3(NT), 0, s, g, b, nd);
    else hipLaunchKernelGGL(k_node_contact<2>, dim3(blocks_for(g.nstride * g.nfields, NT)), dim3(NT), 0, s, g, b, nd);
}

// ---------------------------------------------------------------------------------------
// Grid velocity conditions (NodalVelBC::GridVelocityConditions -> VelocityBCLoop,
// NodalVelBC.cpp:321-400; MatVelocityField::ZeroVelocityBC and AddVelocityBC,
// MatVelocityField.cpp:490-575, norm a unit axis). The reference zeroes for every condition of
// the list, then adds for every one; conditions on different nodes touch different values, so
// taking each node's conditions in list order, zeroes first, gives the same numbers.

__device__ __forceinline__ int bc_value(const KBcs &bc, int e, double t, double &v) {
    return style_value(bc.style[e], bc.value[e], bc.ftime[e], t, v);
}

// one pass on momenta p and forces fo of one field of one node (ZeroVelocityBC, then AddVelocityBC)
template <int PASS>
__device__ __forceinline__ void bc_pass(const KBcs &bc, int e0, int e1, double t, double m, double dt,
                                        double p[3], double fo[3]) {
    for (int e = e0; e < e1; e++) {
        double v;
        const int on = PASS == BC_PASS_MASS_MOMENTUM ? bc_value(bc, e, t, v) : bc.act[e];
        if (!on) continue;
        const int a = bc.dir[e];
        if (PASS == BC_PASS_GRID_FORCES) {
            const double dotf = fo[a], dotp = p[a];
            fo[a] += -dotf - dotp / dt;
        } else {
            const double dotn = p[a];
            p[a] += -dotn;
            if (PASS == BC_PASS_UPDATE_MOMENTUM) fo[a] += -dotn / dt;
        }
    }
    for (int e = e0; e < e1; e++) {
        double v;
        int on;
        if (PASS == BC_PASS_MASS_MOMENTUM) on = bc_value(bc, e, t, v);
        else { on = bc.act[e]; v = bc.cur[e]; }
        if (!on) continue;
        const int a = bc.dir[e];
        const double mv = m * v;
        if (PASS == BC_PASS_GRID_FORCES) {
            fo[a] += mv / dt;
        } else {
            p[a] += mv;
            if (PASS == BC_PASS_UPDATE_MOMENTUM) fo[a] += mv / dt;
        }
    }
}

// one thread per (node with conditions, field). MASS_MOMENTUM (after the contact pass, before the
// first strain update) keeps the momenta it starts from; GRID_FORCES starts from those again
// (MatVelocityField::RestoreMomenta), sets the forces and redoes the momentum update of the node
// (pk + ftot*dt, as k_node_force). The mass-momentum pass reads the step's start time from slot
// par and writes the next step's into slot par ^ 1, which no thread of this step reads.
template <int PASS>
__global__ void k_vel_bcs(KGrid g, KNodes N, KBcs bc, int par) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (PASS == BC_PASS_MASS_MOMENTUM && idx == 0) bc.time[par ^ 1] = bc.time[par] + g.timestep;
    if (idx >= (long long)bc.nb * g.nfields) return;
    const int f = (int)(idx / bc.nb);
    const int b = (int)(idx - (long long)f * bc.nb);
    const int e0 = bc.start[b], e1 = bc.start[b + 1];
    double t = 0.;
    if (PASS == BC_PASS_MASS_MOMENTUM) {
        t = bc.time[par];
        if (f == 0)
            for (int e = e0; e < e1; e++) {
                double v;
                bc.act[e] = bc_value(bc, e, t, v);
                bc.cur[e] = v;
            }
    }
    const KNodes Nf = field_view(g, N, f);
    const long long n = bc.node[b], nn = g.nstride;
    if (Nf.cnt[n] <= 0) return;
    const double m = Nf.mass[n], dt = g.timestep;
    if (PASS == BC_PASS_XPIC || PASS == BC_PASS_XPIC_FORCE) {
        // NodalVelBC::GridVelocityConditions for the XPIC passes (NodalVelBC.cpp:327-335) ->
        // MatVelocityField::ZeroVelocityBC (MatVelocityField.cpp:523-534) on the increment
        for (int e = e0; e < e1; e++) {
            if (!bc.act[e]) continue;
            const int a = bc.dir[e];
            const double dotn = Nf.vprev[a * nn + n];
            Nf.vprev[a * nn + n] = 0.;
            Nf.vk[a * nn + n] -= dotn;
            if (PASS == BC_PASS_XPIC_FORCE) Nf.ftot[a * nn + n] += -m * dotn / dt;
        }
        return;
    }
    double p[3] = {Nf.pk[n], Nf.pk[nn + n], Nf.pk[2 * nn + n]};
    double fo[3] = {Nf.ftot[n], Nf.ftot[nn + n], Nf.ftot[2 * nn + n]};
    double *sv = bc.save + ((long long)f * bc.nb + b) * 3;
    if (PASS == BC_PASS_MASS_MOMENTUM) {
        sv[0] = p[0]; sv[1] = p[1]; sv[2] = p[2];
        bc_pass<BC_PASS_MASS_MOMENTUM>(bc, e0, e1, t, m, dt, p, fo);
    } else if (PASS == BC_PASS_GRID_FORCES || PASS == BC_PASS_FORCES_MOMENTA) {
        p[0] = sv[0]; p[1] = sv[1]; p[2] = sv[2];
        bc_pass<BC_PASS_GRID_FORCES>(bc, e0, e1, t, m, dt, p, fo);
        for (int c = 0; c < 3; c++) p[c] = p[c] + fo[c] * dt;
        if (PASS == BC_PASS_FORCES_MOMENTA) bc_pass<BC_PASS_UPDATE_MOMENTUM>(bc, e0, e1, t, m, dt, p, fo);
    } else {
        bc_pass<PASS>(bc, e0, e1, t, m, dt, p, fo);
    }
    Nf.pk[n] = p[0]; Nf.pk[nn + n] = p[1]; Nf.pk[2 * nn + n] = p[2];
    if (PASS != BC_PASS_MASS_MOMENTUM && PASS != BC_PASS_UPDATE_STRAINS_LAST) {
        Nf.ftot[n] = fo[0]; Nf.ftot[nn + n] = fo[1]; Nf.ftot[2 * nn + n] = fo[2];
    }
    if (m != 0.) {
        const double s = 1. / m;
        Nf.vk[n] = s * p[0]; Nf.vk[nn + n] = s * p[1]; Nf.vk[2 * nn + n] = s * p[2];
    }
}

void launch_vel_bcs(const KGrid &g, const KNodes &nd, const KBcs &bc, int pass, int par, hipStream_t s) {
    const dim3 grid(blocks_for((long long)bc.nb * g.nfields, NT)), blk(NT);
    switch (pass) {
        case BC_PASS_MASS_MOMENTUM: hipLaunchKernelGGL(k_vel_bcs<BC_PASS_MASS_MOMENTUM>, grid, blk, 0, s, g, nd, bc, par); break;
        case BC_PASS_GRID_FORCES: hipLaunchKernelGGL(k_vel_bcs<BC_PASS_GRID_FORCES>, grid, blk, 0, s, g, nd, bc, par); break;
        case BC_PASS_UPDATE_MOMENTUM: hipLaunchKernelGGL(k_vel_bcs<BC_PASS_UPDATE_MOMENTUM>, grid, blk, 0, s, g, nd, bc, par); break;
        case BC_PASS_FORCES_MOMENTA: hipLaunchKernelGGL(k_vel_bcs<BC_PASS_FORCES_MOMENTA>, grid, blk, 0, s, g, nd, bc, par); break;
        case BC_PASS_XPIC: hipLaunchKernelGGL(k_vel_bcs<BC_PASS_XPIC>, grid, blk, 0, s, g, nd, bc, par); break;
        case BC_PASS_XPIC_FORCE: hipLaunchKernelGGL(k_vel_bcs<BC_PASS_XPIC_FORCE>, grid, blk, 0, s, g, nd, bc, par); break;
        default: hipLaunchKernelGGL(k_vel_bcs<BC_PASS_UPDATE_STRAINS_LAST>, grid, blk, 0, s, g, nd, bc, par); break;
    }
}

void launch_xpic(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd, const KBcs &bc,
                 int order, bool fmpm, bool forcePass, int par, hipStream_t s) {
    const dim3 ng(blocks_for(g.nstride * g.nfields, NT)), blk(NT);
    const KBins tb = tile_bins(b, TILE_SLOT_XPIC);
    const bool cp = g.shape == MPMGPU_SHAPE_LCPDI;
    if (dim == 3) hipLaunchKernelGGL(k_xpic_init<3>, ng, blk, 0, s, g, b, nd, fmpm ? 1 : 0);
    else hipLaunchKernelGGL(k_xpic_init<2>, ng, blk, 0, s, g, b, nd, fmpm ? 1 : 0);
    for (int it = 2; it <= order; it++) {
        if (dim == 3) {
            if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(3), k_xpic_p2g_corners<3>, tb, s, g, p, tb, nd);
            else TILE_LAUNCH_NT(64 * UGIMP_NW, k_xpic_p2g<3>, tb, s, g, p, tb, nd);
            hipLaunchKernelGGL(k_xpic_node<3>, ng, blk, 0, s, g, tb, nd);
        } else {
            if (cp) TILE_LAUNCH_NT(64 * CORNER_NW(2), k_xpic_p2g_corners<2>, tb, s, g, p, tb, nd);
            else TILE_LAUNCH_NT(64 * UGIMP_NW, k_xpic_p2g<2>, tb, s, g, p, tb, nd);
            hipLaunchKernelGGL(k_xpic_node<2>, ng, blk, 0, s, g, tb, nd);
        }
        if (bc.nb) MPM_KNS::launch_vel_bcs(g, nd, bc, forcePass && !fmpm ? BC_PASS_XPIC_FORCE : BC_PASS_XPIC, par, s);
    }
}

// MatPtLoadBC::SetParticleFext (MatPtLoadBC.cpp:210-221, called from InitializationTask.cpp:91):
// one thread per loaded particle zeroes its pFext and adds each of its loads' value at the
// step's start time (BCValue, zero before a constant or linear load starts), in list order.
// Like the mass-momentum velocity pass it writes the next step's start time into slot par ^ 1.
__global__ void k_particle_loads(KGrid g, KLoads L, int par) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const double t = L.time[par];
    if (q == 0) L.time[par ^ 1] = t + g.timestep;
    if (q >= L.nl) return;
    double fe[3] = {0., 0., 0.};
    for (int e = L.start[q]; e < L.start[q + 1]; e++) {
        double v;
        style_value(L.style[e], L.value[e], L.ftime[e], t, v);
        fe[L.dir[e]] += v;
    }
    for (int c = 0; c < 3; c++) L.fext[3 * q + c] = fe[c];
}

void launch_particle_loads(const KGrid &g, const KLoads &L, int par, hipStream_t s) {
    hipLaunchKernelGGL(k_particle_loads, dim3(blocks_for(L.nl, NT)), dim3(NT), 0, s, g, L, par);
}

void launch_contact_normals(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                            const MpmMaterial *mats, const KStats &st, int callType, hipStream_t s) {
    if (g.normals < 5 || !nd.cnorm) return;
    if (callType == CONTACT_MASS_MOMENTUM) {
        if (dim == 3) hipLaunchKernelGGL(k_contact_list<3>, dim3(blocks_for(g.nnodes, NT)), dim3(NT), 0, s, g, nd);
        else hipLaunchKernelGGL(k_contact_list<2>, dim3(blocks_for(g.nnodes, NT)), dim3(NT), 0, s, g, nd);
    }
    const int np = callType == CONTACT_UPDATE_STRAINS_LAST ? 1 : 0;
    const dim3 grid(4 * g_cus);
    const bool cp = g.shape == MPMGPU_SHAPE_LCPDI;
    if (dim == 3) {
        if (cp) hipLaunchKernelGGL((k_contact_normals<3, MPMGPU_SHAPE_LCPDI>), grid, dim3(NT), 0, s, g, p, b, nd, mats, st, np);
        else hipLaunchKernelGGL((k_contact_normals<3, MPMGPU_SHAPE_UGIMP>), grid, dim3(NT), 0, s, g, p, b, nd, mats, st, np);
    } else {
        if (cp) hipLaunchKernelGGL((k_contact_normals<2, MPMGPU_SHAPE_LCPDI>), grid, dim3(NT), 0, s, g, p, b, nd, mats, st, np);
        else hipLaunchKernelGGL((k_contact_normals<2, MPMGPU_SHAPE_UGIMP>), grid, dim3(NT), 0, s, g, p, b, nd, mats, st, np);
    }
}

void launch_contact(int dim, const KGrid &g, const KNodes &nd, int callType, hipStream_t s) {
    if (dim == 3) hipLaunchKernelGGL(k_contact<3>, dim3(blocks_for(g.nnodes, NT)), dim3(NT), 0, s, g, nd, callType);
    else hipLaunchKernelGGL(k_contact<2>, dim3(blocks_for(g.nnodes, NT)), dim3(NT), 0, s, g, nd, callType);
}

// ---------------------------------------------------------------------------------------
// particle runs between contexts: one thread per (particle, row); rows 0..MPF_NUM_FIELDS-1 are
// the double fields, the next MPI_NUM_FIELDS the int fields

__global__ void k_move(KMove m) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int r = blockIdx.y;
    if (p >= m.cnt) return;
    if (r < MPF_NUM_FIELDS) {
        const double *src = (r >= MPF_POS_X && r <= MPF_POS_Z) ? m.spos[r - MPF_POS_X] : m.sd + r * m.sn;
        m.dd[r * m.dn + m.doff + p] = src[m.soff + p];
    } else {
        // int rows MPI_*, then the upload-index row (MPI_NUM_FIELDS + 2)
        const int q = r - MPF_NUM_FIELDS < MPI_NUM_FIELDS ? r - MPF_NUM_FIELDS : MPI_NUM_FIELDS + 2;
        int v = m.si[q * m.sn + m.soff + p];
        if (q == MPI_MAT) v += m.matShift;
        if (q == MPI_NUM_FIELDS + 2) v += m.homeShift;
        m.di[q * m.dn + m.doff + p] = v;
    }
}

void launch_move(const KMove &m, hipStream_t s) {
    if (m.cnt <= 0) return;
    hipLaunchKernelGGL(k_move, dim3(blocks_for(m.cnt, NT), MPF_NUM_FIELDS + MPI_NUM_FIELDS + 1), dim3(NT), 0, s, m);
}

__global__ void k_iota(int *a, long long n, int base) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) a[k] = base + (int)k;
}

void launch_iota(int *a, long long n, int base, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_iota, dim3(blocks_for(n, NT)), dim3(NT), 0, s, a, n, base);
}

}  // namespace mpmk_s0 / mpmk_s1
