// Newton-step support kernels: nodal loads, FP64 max-norm scans, displacement
// update and the Rodrigues commit of the nodes.
//
// Reference: NodalLoad::Mount src/NodalLoad.cpp:322-401,
// NodalFollowerLoad::Mount src/NodalFollowerLoad.cpp:243-326,
// Table::GetValueAt src/Table.cpp:73-101,
// ConvergenceCriteria scans src/ConvergenceCriteria.cpp:187-288, 289-459, 460-598,
// Solution::UpdateDisps src/Solution.cpp:390-423,
// Node::SaveConfiguration src/Node.cpp:325-384.
#include "gf_internal.h"

#include <algorithm>
#include "gf_device.h"
#include "gf_loads.h"

namespace {

__global__ void fill_kernel(double *p, size_t n, double v)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// Zeroes three ranges; in the second, the entries dfirst + k dstride (k < dcount)
// get 1 instead (the unit diagonal of the padding rows of the global matrix).
__device__ __forceinline__ void clear3(size_t gid, size_t step, double *a, size_t na, double *b, size_t nb, double *c,
                                       size_t nc, size_t dfirst, size_t dstride, size_t dcount)
{
    const size_t n = na + nb + nc;
    for (size_t i = gid; i < n; i += step) {
        double *p = i < na ? a + i : i < na + nb ? b + (i - na) : c + (i - na - nb);
        double v = 0.0;
        if (i >= na + dfirst && i < na + nb) {
            const size_t d = i - na - dfirst;
            if (d % dstride == 0 && d / dstride < dcount) v = 1.0;
        }
        *p = v;
    }
}
__global__ __launch_bounds__(256) void clear3_kernel(double *a, size_t na, double *b, size_t nb, double *c, size_t nc,
                                                     size_t dfirst, size_t dstride, size_t dcount)
{
    clear3(blockIdx.x * (size_t)256 + threadIdx.x, (size_t)gridDim.x * 256, a, na, b, nb, c, nc, dfirst, dstride, dcount);
}

// Zeroes a and c, and the band entries (row, cols[k]) for k in [ptr[row],
// ptr[row + 1]) of rows < nrows (the positions the element scatter writes): one
// wavefront per band row, the short ranges by every thread.
__device__ __forceinline__ void clear_csr(size_t gid, double *a, size_t na, double *c, size_t nc, double *ab, int ld,
                                          int hb, const int *ptr, const int *cols, int nrows)
{
    if (gid < na) a[gid] = 0.0;
    if (gid < nc) c[gid] = 0.0;
    const int row = (int)(gid >> 6), lane = threadIdx.x & 63;
    if (row >= nrows) return;
    double *base = ab + (size_t)row * (size_t)ld + (size_t)hb;
    for (int k = ptr[row] + lane; k < ptr[row + 1]; k += 64) base[cols[k]] = 0.0;
}
__global__ __launch_bounds__(256) void clear_csr_kernel(double *a, size_t na, double *c, size_t nc, double *ab,
                                                         int ld, int hb, const int *ptr, const int *cols, int nrows)
{
    clear_csr(blockIdx.x * (size_t)256 + threadIdx.x, a, na, c, nc, ab, ld, hb, ptr, cols, nrows);
}

__global__ void fill_u32_kernel(unsigned *p, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = 0u;
}


// One thread per loaded node.  (Models with beams take them with the first beam
// launch and the scan instead.)
__global__ __launch_bounds__(128) void nodal_loads_kernel(gf_nodal L, const int *__restrict__ dof, gf_gmat gm, double *r)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= L.n) return;
    double q[GF_NODAL_OUT], q6[6], V18[18];
    gf_nodal_item(L, k, q);
    int R[6], R18[18], C18[18];
#pragma unroll
    for (int i = 0; i < 6; i++) {
        R[i] = dof[6 * L.node[k] + i];
        q6[i] = q[i];
    }
    vec_add_n<6>(r, R, q6);
#pragma unroll
    for (int i = 0; i < 18; i++) {
        R18[i] = R[i / 3];
        C18[i] = R[3 + i % 3];
        V18[i] = q[6 + i];
    }
    gm_add_n<18>(gm, R18, C18, V18);
}

// Max-norms of a vector over band rows split by DOF kind (translation /
// rotation) plus a non-finite flag.  out (as unsigned long long bits of
// non-negative doubles): [0] trans, [1] rot, [2] flag.
__device__ __forceinline__ unsigned long long amax(unsigned long long *p, double v)
{
    return atomicMax(p, (unsigned long long)__double_as_longlong(v));
}

// Workgroup max of NV non-negative values (256 lanes): wave shuffles, then LDS
// across the 4 waves, then one atomic per value and workgroup.
template <int NV> __device__ __forceinline__ void block_amax(double (&v)[NV], unsigned long long *out)
{
    __shared__ double sred[4][NV];
#pragma unroll
    for (int k = 0; k < NV; k++)
        for (int off = 32; off > 0; off >>= 1) v[k] = fmax(v[k], __shfl_xor(v[k], off));
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) sred[wave][k] = v[k];
    __syncthreads();
    if (threadIdx.x < NV) {
        double mx = sred[0][threadIdx.x];
        for (int w = 1; w < 4; w++) mx = fmax(mx, sred[w][threadIdx.x]);
        // the result is waited for: what this wavefront does next comes after the maximum
        const unsigned long long old = amax(out + threadIdx.x, mx);
        asm volatile("" ::"v"(old));
    }
}

// max |r| over translational and rotational free DOFs, and a non-finite flag, into
// scal[GF_SCAL_RES ..].  The workgroup that finishes last (a ticket in
// scal[GF_SCAL_TICKET]; none waits) then writes the scalar block to the host's
// pinned mirror and clears the increment norms and the failure flag for the next
// solve: the copy and the fill that did this were two more dependent launches of
// each Newton iteration (3.9 and 1.6 us).  Only atomics pass between the
// workgroups, so no fence: one here writes an XCD's whole L2 back (8 us after a
// 10,000-element assembly).
//
// LOADS: the nodal loads, formed beside the first beam launch (ln_out), are added here,
// row by row: row i takes entry row_load[i] (6 k + component, or -1) and its three
// tangent entries, where they are not zero.  (As a launch of their own the loads are a
// chain of six dependent reads: 7.4 us at 777 loaded elements, 10.4 at 10,000; so they
// cost the scan 0.1 and 2.4 us and the beam launch 0.1 and 1.)
template <bool LOADS>
__global__ __launch_bounds__(256) void scan_kernel(int n, double *__restrict__ v, const int *__restrict__ row_nc,
                                                   unsigned long long *scal, unsigned long long *host,
                                                   const int *__restrict__ row_load, const double *__restrict__ ln_out,
                                                   const int *__restrict__ dof, gf_gmat gm)
{
    unsigned long long *out = scal + GF_SCAL_RES;
    double m[3] = {0.0, 0.0, 0.0};  // translations, rotations, non-finite
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        double a = v[i];
        if (LOADS) {
            const int li = row_load[i];
            if (li >= 0) {
                const int k = li / 6, c = li - 6 * k, node = row_nc[i] / 6;
                const double *o = ln_out + (size_t)GF_NODAL_OUT * k;
                a += o[c];
                v[i] = a;
                const double K3[3] = {o[6 + 3 * c], o[7 + 3 * c], o[8 + 3 * c]};
                if (K3[0] != 0.0 || K3[1] != 0.0 || K3[2] != 0.0) {
                    const int R3[3] = {i, i, i}, C3[3] = {dof[6 * node + 3], dof[6 * node + 4], dof[6 * node + 5]};
                    gm_add_n<3>(gm, R3, C3, K3);
                }
            }
        }
        a = fabs(a);
        if (!(a == a) || a >= 1e300) m[2] = 1.0;
        else if (row_nc[i] % 6 < 3) m[0] = fmax(m[0], a);
        else m[1] = fmax(m[1], a);
    }
    block_amax<3>(m, out);
    // (the wavefront that added this workgroup's maxima takes its ticket)
    if (threadIdx.x >= 64) return;
    unsigned ticket = 0;
    if (threadIdx.x == 0) ticket = atomicAdd((unsigned *)(scal + GF_SCAL_TICKET), 1u);
    if ((unsigned)__builtin_amdgcn_readfirstlane((int)ticket) != gridDim.x - 1) return;
    if (threadIdx.x < GF_SCAL_RES + 3) {
        host[threadIdx.x] = atomicOr(scal + threadIdx.x, 0ull);  // read where the maxima were formed
        if (threadIdx.x <= GF_SCAL_FLAG) scal[threadIdx.x] = 0;
    }
    if (threadIdx.x == 0) scal[GF_SCAL_TICKET] = 0;
}

// d += x on free DOFs; scans |x| and the updated |d| (CheckGLConvergence).
// Workgroups `block` of `blocks`.
__device__ __forceinline__ void update_rows(int block, int blocks, int n, const double *__restrict__ x,
                                            const int *__restrict__ row_nc, double *__restrict__ disp,
                                            unsigned long long *out)
{
    double m[5] = {0.0, 0.0, 0.0, 0.0, 0.0};  // |x| t/r, |d| t/r, non-finite
    for (int i = block * blockDim.x + threadIdx.x; i < n; i += blocks * blockDim.x) {
        int nc = row_nc[i];
        double xi = x[i];
        double dn = disp[nc] + xi;
        disp[nc] = dn;
        double ax = fabs(xi), ad = fabs(dn);
        if (!(ax == ax) || ax >= 1e300) m[4] = 1.0;
        if (nc % 6 < 3) { m[0] = fmax(m[0], ax); m[2] = fmax(m[2], ad); }
        else { m[1] = fmax(m[1], ax); m[3] = fmax(m[3], ad); }
    }
    block_amax<5>(m, out);
}
__global__ __launch_bounds__(256) void update_kernel(int n, const double *__restrict__ x,
                                                     const int *__restrict__ row_nc, double *__restrict__ disp,
                                                     unsigned long long *out)
{
    update_rows(blockIdx.x, gridDim.x, n, x, row_nc, disp, out);
}

// The update and the clear that the next assembly begins with, in one launch
// (neither touches what the other does): the first `ub` workgroups update, the
// others clear.  CSR: as clear_csr_kernel, else as clear3_kernel.
struct ClearArgs {
    double *a, *b, *c;
    size_t na, nb, nc;
    size_t dfirst, dstride, dcount;   // clear3
    int ld, hb, nrows;                // csr (b: the band)
    const int *ptr, *cols;
};
template <bool CSR>
__global__ __launch_bounds__(256) void update_clear_kernel(int ub, int n, const double *__restrict__ x,
                                                           const int *__restrict__ row_nc, double *__restrict__ disp,
                                                           unsigned long long *out, ClearArgs q)
{
    if ((int)blockIdx.x < ub) {
        update_rows(blockIdx.x, ub, n, x, row_nc, disp, out);
        return;
    }
    const size_t gid = (blockIdx.x - ub) * (size_t)256 + threadIdx.x;
    if constexpr (CSR) clear_csr(gid, q.a, q.na, q.c, q.nc, q.b, q.ld, q.hb, q.ptr, q.cols, q.nrows);
    else clear3(gid, (size_t)(gridDim.x - ub) * 256, q.a, q.na, q.b, q.nb, q.c, q.nc, q.dfirst, q.dstride, q.dcount);
}

// Node::SaveConfiguration: x += u, alpha <- compose(alpha_delta, alpha), Euler vector.
__global__ void node_commit_kernel(int nn, double *__restrict__ copy, const double *__restrict__ disp,
                                   double *__restrict__ euler)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nn) return;
    double *c = copy + 6 * (size_t)i;
    const double *d = disp + 6 * (size_t)i;
    c[0] += d[0]; c[1] += d[1]; c[2] += d[2];
    v3<double> a3 = compose(mk3(d[3], d[4], d[5]), mk3(c[3], c[4], c[5]));
    c[3] = a3.x; c[4] = a3.y; c[5] = a3.z;
    double na = sqrt(dot3(a3, a3));
    double th = 2.0 * atan(na / 2.0);
    double s = na != 0.0 ? th / na : 0.0;
    euler[3 * (size_t)i + 0] = s * a3.x;
    euler[3 * (size_t)i + 1] = s * a3.y;
    euler[3 * (size_t)i + 2] = s * a3.z;
}

// Unit diagonal for the padding rows past n_free.

}  // namespace

static inline int grid_for(size_t n, int block, int cap = 4096)
{
    size_t g = (n + block - 1) / block;
    if (g < 1) g = 1;
    if (g > (size_t)cap) g = cap;
    return (int)g;
}

int gf_launch_fill(hipStream_t s, double *p, size_t n, double v)
{
    if (n == 0) return GF_OK;
    hipLaunchKernelGGL(fill_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, v);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

int gf_launch_clear_csr(hipStream_t s, double *a, size_t na, double *c, size_t nc, double *ab, int ld, int hb,
                        const int *ptr, const int *cols, int nrows)
{
    const size_t n = std::max((size_t)nrows * 64, std::max(na, nc));
    hipLaunchKernelGGL(clear_csr_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, na, c, nc, ab, ld, hb,
                       ptr, cols, nrows);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

int gf_launch_clear3(hipStream_t s, double *a, size_t na, double *b, size_t nb, double *c, size_t nc, size_t dfirst,
                     size_t dstride, size_t dcount)
{
    const size_t n = na + nb + nc;
    if (n == 0) return GF_OK;
    if (dstride == 0) dcount = 0, dstride = 1;
    hipLaunchKernelGGL(clear3_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, a, na, b, nb, c, nc, dfirst, dstride,
                       dcount);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

namespace {
__global__ void set2_kernel(double *p, double a, double b)
{
    if (threadIdx.x == 0) {
        p[0] = a;
        p[1] = b;
    }
}
}  // namespace

int gf_launch_set2(hipStream_t s, double *p, double a, double b)
{
    hipLaunchKernelGGL(set2_kernel, dim3(1), dim3(64), 0, s, p, a, b);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

int gf_launch_fill_bytes(hipStream_t s, void *p, size_t bytes)
{
    size_t n = bytes / 4;
    if (n == 0) return GF_OK;
    hipLaunchKernelGGL(fill_u32_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, (unsigned *)p, n);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

int gf_nodal_loads(gf_model *m, const double *tp)
{
    if (m->n_load_nodes == 0) return GF_OK;
    hipLaunchKernelGGL(nodal_loads_kernel, dim3((m->n_load_nodes + 127) / 128), dim3(128), 0, m->stream,
                       gf_nodal_of(m, tp), m->d_dof, gf_model_gmat(m), m->d_r);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

// The norms land in d_scal[GF_SCAL_RES..+2], which the assembly's clear zeroed, and
// with the rest of the scalar block in h_scal; the increment norms and the flag
// are zero afterwards.
int gf_scan_residual(gf_model *m)
{
    hipLaunchKernelGGL(m->d_ln_out ? scan_kernel<true> : scan_kernel<false>, dim3(grid_for(m->n_free, 256, 128)),
                       dim3(256), 0, m->stream, m->n_free, m->d_r, m->d_row_nc, (unsigned long long *)m->d_scal,
                       (unsigned long long *)m->h_scal, (const int *)m->d_row_load, (const double *)m->d_ln_out,
                       (const int *)m->d_dof, gf_model_gmat(m));
    GF_HIP(hipGetLastError());
    return GF_OK;
}

// zero_norms: clear d_scal[0..7] first (callers that cleared it pass false).
int gf_update_disp(gf_model *m, bool zero_norms)
{
    if (zero_norms) {
        int st = gf_launch_fill_bytes(m->stream, m->d_scal, GF_SCAL_FLAG * sizeof(double));
        if (st) return st;
    }
    hipLaunchKernelGGL(update_kernel, dim3(grid_for(m->n_free, 256, 128)), dim3(256), 0, m->stream, m->n_free,
                       m->d_x, m->d_row_nc, m->d_disp, (unsigned long long *)m->d_scal);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

// UpdateDisps (norms cleared by the caller) with the clear of the next assembly.
int gf_update_clear(gf_model *m)
{
    if (m->shell_gather) return gf_update_disp(m, false);  // (needs no clear)
    ClearArgs q{};
    gf_assemble_clear_ranges(m, q.b, q.nb, q.dfirst, q.dstride, q.dcount);
    q.a = m->d_r;
    q.na = (size_t)m->npad;
    q.c = m->d_scal + GF_SCAL_RES;
    q.nc = 8;
    const int ub = grid_for(m->n_free, 256, 128);
    unsigned long long *out = (unsigned long long *)m->d_scal;
    if (m->fronts_on) {
        q.ld = m->band_ld;
        q.hb = m->half_band;
        q.ptr = m->d_csr_ptr;
        q.cols = m->d_csr_col;
        q.nrows = m->n_free;
        const size_t n = std::max((size_t)q.nrows * 64, std::max(q.na, q.nc));
        hipLaunchKernelGGL(update_clear_kernel<true>, dim3(ub + (unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, ub,
                           m->n_free, m->d_x, m->d_row_nc, m->d_disp, out, q);
    } else {
        hipLaunchKernelGGL(update_clear_kernel<false>, dim3(ub + grid_for(q.na + q.nb + q.nc, 256)), dim3(256), 0,
                           m->stream, ub, m->n_free, m->d_x, m->d_row_nc, m->d_disp, out, q);
    }
    GF_HIP(hipGetLastError());
    return GF_OK;
}

int gf_node_commit(gf_model *m)
{
    hipLaunchKernelGGL(node_commit_kernel, dim3((m->nn + 255) / 256), dim3(256), 0, m->stream, m->nn, m->d_copy,
                       m->d_disp, m->d_euler);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

