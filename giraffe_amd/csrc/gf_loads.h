// Nodal loads of the static analysis: one item per loaded node.
#pragma once
#include "gf_internal.h"
#include "gf_device.h"

struct gf_nodal {
    int n;                                   // loaded nodes
    const int *node, *off, *ids;             // loads ids[off[k] .. off[k + 1]) of node[k]
    const double *rec, *tab_t, *tab_v, *disp, *copy, *tp;
    double *out;                             // (or null) [n][24]: GF_NODAL_OUT
};

// All loads on loaded node k, in load order: the force and pseudo-moment (6), and what
// the tangent gains in the rows of the displacements (9) and of the rotations (9), both
// by the rotations' columns.
constexpr int GF_NODAL_OUT = 24;
__device__ __forceinline__ void gf_nodal_item(const gf_nodal &L, int k, double (&out)[GF_NODAL_OUT])
{
    const double t = *L.tp;  // load time, device-resident (a captured Newton step reads the current one)
    const int node = L.node[k];
#pragma unroll
    for (int i = 0; i < GF_NODAL_OUT; i++) out[i] = 0.0;
    v3<double> alpha = mk3(L.disp[6 * node + 3], L.disp[6 * node + 4], L.disp[6 * node + 5]);
    for (int q = L.off[k]; q < L.off[k + 1]; q++) {
        const double *W = L.rec + (size_t)L.ids[q] * NL_REC;
        int kind = (int)W[NL_KIND];
        m3<double> CS;
#pragma unroll
        for (int i = 0; i < 9; i++) CS.a[i] = W[NL_CS + i];
        int r0 = (int)W[NL_TAB0], nt = (int)W[NL_TABN];
        double tv6[6];
        gf_table_values6(L.tab_t, L.tab_v, r0, nt, t, tv6);
        v3<double> f = mk3(W[NL_MULT + 0] * tv6[0], W[NL_MULT + 1] * tv6[1], W[NL_MULT + 2] * tv6[2]);
        v3<double> mo = mk3(W[NL_MULT + 3] * tv6[3], W[NL_MULT + 4] * tv6[4], W[NL_MULT + 5] * tv6[5]);
        if (kind == GF_LOAD_NODAL) {
            // dead force + pseudo-moment Xi^T m with stiffness -V(alpha, Xi^T m)
            f = mtv(CS, f);
            mo = mtv(CS, mo);
            m3<double> Q, Xi;
            double g;
            rodrigues(alpha, Q, Xi, g);
            mo = mtv(Xi, mo);
            m3<double> S = opV(alpha, mo);
            const double q6[6] = {f.x, f.y, f.z, mo.x, mo.y, mo.z};
#pragma unroll
            for (int i = 0; i < 6; i++) out[i] += q6[i];
#pragma unroll
            for (int i = 0; i < 9; i++) out[15 + i] -= S.a[i];
        } else if (kind == GF_LOAD_NODAL_FOLLOWER) {
            v3<double> ai = mk3(L.copy[6 * node + 3], L.copy[6 * node + 4], L.copy[6 * node + 5]);
            m3<double> Qi, Xii, Q, Xi;
            double gi, g;
            rodrigues(ai, Qi, Xii, gi);
            Qi = mm3(Qi, tr3(CS));
            rodrigues(alpha, Q, Xi, g);
            v3<double> fip = mv(mm3(Q, Qi), f);
            v3<double> Qim = mv(Qi, mo);
            v3<double> mip = mv(Xi, Qim);
            m3<double> K12 = mscl(-1.0, mm3(skew3(fip), Xi));
            m3<double> dy;
#pragma unroll
            for (int i = 0; i < 9; i++) dy.a[i] = 0.0;
            add_outer(dy, 1.0, Qim, alpha);
            m3<double> K22 = mscl(-0.5 * g, madd(skew3(Qim), mm3(Xi, dy)));
            const double q6[6] = {fip.x, fip.y, fip.z, mip.x, mip.y, mip.z};
#pragma unroll
            for (int i = 0; i < 6; i++) out[i] += q6[i];
#pragma unroll
            for (int i = 0; i < 9; i++) {
                out[6 + i] -= K12.a[i];
                out[15 + i] -= K22.a[i];
            }
        }
    }
}

inline gf_nodal gf_nodal_of(const gf_model *m, const double *tp)
{
    return {m->n_load_nodes, m->d_ln_node, m->d_ln_off, m->d_ln_ids, m->d_lrec, m->d_tab_t,
            m->d_tab_v,      m->d_disp,    m->d_copy,   tp,          m->d_ln_out};
}
