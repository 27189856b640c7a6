// mpm_launch.hip -- the launchers the context calls: each runs the kernels compiled for the tile
// shape of its grid argument (namespace mpmk_s0 or mpmk_s1); launchers without a grid argument do
// not depend on the shape and run shape 0's copy.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mpm_kernels.h"

#define BY_SHAPE(G, CALL) ((G).tileShape ? mpmk_s1::CALL : mpmk_s0::CALL)

void set_tile_cus(int cus) {
    mpmk_s0::set_tile_cus(cus);
    mpmk_s1::set_tile_cus(cus);
}
void launch_bin_keys(int dim, const KGrid &g, const KPart &p, const KBins &b, hipStream_t s) {
    BY_SHAPE(g, launch_bin_keys(dim, g, p, b, s));
}
void launch_bin_finish(int dim, const KGrid &g, const KPart &p, const KBins &b, hipStream_t s) {
    BY_SHAPE(g, launch_bin_finish(dim, g, p, b, s));
}
void launch_p2g_mass(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                     const MpmMaterial *mats, const KStats &st, hipStream_t s) {
    BY_SHAPE(g, launch_p2g_mass(dim, g, p, b, nd, mats, st, s));
}
void launch_node_mass(int dim, const KGrid &g, const KBins &b, const KNodes &nd, hipStream_t s) {
    BY_SHAPE(g, launch_node_mass(dim, g, b, nd, s));
}
bool launch_usf_force(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd, const KLoads &L,
                      const MpmMaterial *mats, hipStream_t s) {
    return BY_SHAPE(g, launch_usf_force(dim, g, p, b, nd, L, mats, s));
}
void launch_usf(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                const MpmMaterial *mats, hipStream_t s) {
    BY_SHAPE(g, launch_usf(dim, g, p, b, nd, mats, s));
}
void launch_p2g_force(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd, const KLoads &L,
                      int par, hipStream_t s) {
    BY_SHAPE(g, launch_p2g_force(dim, g, p, b, nd, L, par, s));
}
void launch_node_force(int dim, const KGrid &g, const KBins &b, const KNodes &nd, hipStream_t s) {
    BY_SHAPE(g, launch_node_force(dim, g, b, nd, s));
}
void launch_g2p_p2g(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                    const MpmMaterial *mats, int mode, hipStream_t s) {
    BY_SHAPE(g, launch_g2p_p2g(dim, g, p, b, nd, mats, mode, s));
}
void launch_node_mom2(int dim, const KGrid &g, const KBins &b, const KNodes &nd, hipStream_t s) {
    BY_SHAPE(g, launch_node_mom2(dim, g, b, nd, s));
}
void launch_usl_reset(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                      const MpmMaterial *mats, const KStats &st, hipStream_t s) {
    BY_SHAPE(g, launch_usl_reset(dim, g, p, b, nd, mats, st, s));
}
void launch_p2g_contact(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                        const MpmMaterial *mats, bool newPositions, hipStream_t s) {
    BY_SHAPE(g, launch_p2g_contact(dim, g, p, b, nd, mats, newPositions, s));
}
void launch_node_contact(int dim, const KGrid &g, const KBins &b, const KNodes &nd, hipStream_t s) {
    BY_SHAPE(g, launch_node_contact(dim, g, b, nd, s));
}
void launch_contact(int dim, const KGrid &g, const KNodes &nd, int callType, hipStream_t s) {
    BY_SHAPE(g, launch_contact(dim, g, nd, callType, s));
}
void launch_contact_normals(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd,
                            const MpmMaterial *mats, const KStats &st, int callType, hipStream_t s) {
    BY_SHAPE(g, launch_contact_normals(dim, g, p, b, nd, mats, st, callType, s));
}
void launch_vel_bcs(const KGrid &g, const KNodes &nd, const KBcs &bc, int pass, int par, hipStream_t s) {
    BY_SHAPE(g, launch_vel_bcs(g, nd, bc, pass, par, s));
}
void launch_xpic(int dim, const KGrid &g, const KPart &p, const KBins &b, const KNodes &nd, const KBcs &bc,
                 int order, bool fmpm, bool forcePass, int par, hipStream_t s) {
    BY_SHAPE(g, launch_xpic(dim, g, p, b, nd, bc, order, fmpm, forcePass, par, s));
}
void launch_particle_loads(const KGrid &g, const KLoads &L, int par, hipStream_t s) {
    BY_SHAPE(g, launch_particle_loads(g, L, par, s));
}
void launch_move(const KMove &m, hipStream_t s) { mpmk_s0::launch_move(m, s); }
void launch_iota(int *a, long long n, int base, hipStream_t s) { mpmk_s0::launch_iota(a, n, base, s); }

namespace {

// Rows of n words taken in another order, and back: dst[a][k] = src[a][at[k]], or dst[a][at[k]] = src[a][k].
// A run that has stopped (*stop set, if stop is given) keeps its rows where they are: its last positions
// may be in the buffer that serves as scratch.
template <typename T, bool BACK>
__global__ void k_reorder_rows(const T *src, T *dst, const int *at, int rows, long long n, const unsigned long long *stop) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n || (stop && *stop)) return;
    const long long from = BACK ? k : at[k], to = BACK ? at[k] : k;
    for (int a = 0; a < rows; a++) dst[a * n + to] = src[a * n + from];
}

template <typename T>
__global__ void k_copy_unless(const T *src, T *dst, long long n, const unsigned long long *stop) {
    if (stop && *stop) return;
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x)
        dst[k] = src[k];
}

template <typename T>
void reorder(bool back, T *rows, T *tmp, const int *at, int m, long long n, const unsigned long long *stop, hipStream_t s) {
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    if (back) hipLaunchKernelGGL((k_reorder_rows<T, true>), grid, block, 0, s, rows, tmp, at, m, n, stop);
    else hipLaunchKernelGGL((k_reorder_rows<T, false>), grid, block, 0, s, rows, tmp, at, m, n, stop);
    hipLaunchKernelGGL(k_copy_unless<T>, dim3((unsigned)std::min<long long>((m * n + 255) / 256, 2048)), block, 0, s, tmp, rows,
                       m * n, stop);
}

}  // namespace

void launch_reorder_rows(bool back, double *rows, double *tmp, const int *at, int m, long long n,
                         const unsigned long long *stop, hipStream_t s) {
    reorder(back, rows, tmp, at, m, n, stop, s);
}
void launch_reorder_rows(bool back, int *rows, int *tmp, const int *at, int m, long long n,
                         const unsigned long long *stop, hipStream_t s) {
    reorder(back, rows, tmp, at, m, n, stop, s);
}
void launch_copy_row(const double *src, double *dst, long long n, const unsigned long long *stop, hipStream_t s) {
    hipLaunchKernelGGL(k_copy_unless<double>, dim3((unsigned)std::min<long long>((n + 255) / 256, 2048)), dim3(256), 0, s, src, dst, n, stop);
}
