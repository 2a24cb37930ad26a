// Shell_1 on gfx950: element tangent + internal force fused with the
// conflict-free scatter, follower pressure, and the Gauss-point commit.
//
// Reference: Shell_1::Mount src/Shell_1.cpp:899-1332 (through-thickness
// hyperelastic integration :1064-1162, drilling stiffness :1212-1217,
// Psi :1239-1268, G :1277-1319), MountFieldLoads (self-weight, twice)
// :1335-1381, MountShellSpecialLoads :1392-1467, SaveLagrange :1650-1664,
// PreCalc :1666-2365, MountGlobal DOF order :1513-1648.
//
// Notation: the 15 rows of dN are five 3-row blocks R = 0 u_x1, 1 alpha_x1,
// 2 u_x2, 3 alpha_x2, 4 alpha; the 27 element DOFs are nine 3-column blocks
// I = 0..5 (u of nodes 1..6) and 6..8 (alpha of nodes 4..6).  dN block (R, I)
// is c_I^R times the identity, so K_IJ = sum_gp w sum_RS c_I^R c_J^S M_RS with
// M = Psi^T D Psi + G assembled block-wise (Psi has two non-zero blocks per
// block row: (R, R) and (R, 4)).
//
// Workgroup: 256 lanes, SEPB = 4 elements; LDS holds per Gauss point the
// 16 blocks of D, Psi, G, M and Psi^T sigma (48 KB), and the elements' constants.
// In the Newton loop phase 1
// runs for all elements in one launch with every lane busy (shell_record_kernel),
// the follower pressure's terms likewise (shell_pressure_record_kernel), then one
// launch of phases 2-4 for all elements writes each element's K and f to HBM,
// and they are added, with the pressure terms and the self-weight, into the tangent
// and residual: gathered by rows where the tangent's structure is at hand
// (shell_gather_kernel), else by a light scatter launch per colour
// (shell_scatter_kernel).
//   phase 1  lane per (element, gp): kinematics, 3-point thickness integration
//   phase 2  lane per (element, gp, block RS): the 25 blocks of M
//   phase 3  lane per (element, I, J), a wavefront's of one form: K_IJ, rotated to global
//   phase 4  lane per (element, I): internal force
#include "gf_internal.h"
#include "gf_device.h"

namespace {

constexpr int SEPB = 4;
constexpr int SWG = 256;
constexpr int L_D = 0;     // 16 blocks D(i,j), rows [n1 m1 n2 m2] x cols [eta1 k1 eta2 k2]
constexpr int L_P = 144;   // Psi(R,R), R = 0..3
constexpr int L_W = 180;   // Psi(R,4), R = 0..3
constexpr int L_G = 216;   // Gua1, Gua2, Vm1, Vm2, Gaa
constexpr int L_S = 261;   // Psi^T sigma (15)
constexpr int L_M = 276;   // M blocks (R,S), 25 x 9
constexpr int L_GP = 501;
constexpr int SPR = 57;    // pressure record of (element, u-node a): P_a (3), then K_p rows of a (3 x 18)

__device__ __forceinline__ m3<double> ld3(const double *p)
{
    m3<double> r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.a[i] = p[i];
    return r;
}
__device__ __forceinline__ void st3(double *p, const m3<double> &m)
{
#pragma unroll
    for (int i = 0; i < 9; i++) p[i] = m.a[i];
}
__device__ __forceinline__ void acc3(double *p, double s, const m3<double> &m)
{
#pragma unroll
    for (int i = 0; i < 9; i++) p[i] += s * m.a[i];
}
// X E3 and E3 X with E3 = skew(e3), e3 = (0,0,1)
__device__ __forceinline__ m3<double> mE3(const m3<double> &X)
{
    m3<double> r;
#pragma unroll
    for (int i = 0; i < 3; i++) { r.a[3 * i] = X.a[3 * i + 1]; r.a[3 * i + 1] = -X.a[3 * i]; r.a[3 * i + 2] = 0.0; }
    return r;
}
__device__ __forceinline__ m3<double> E3m(const m3<double> &X)
{
    m3<double> r;
#pragma unroll
    for (int j = 0; j < 3; j++) { r.a[j] = -X.a[3 + j]; r.a[3 + j] = X.a[j]; r.a[6 + j] = 0.0; }
    return r;
}

// Geometric block G(idx, 4) (row4 = false) or G(4, idx) (row4 = true), idx < 4:
// G(R,4) = Gua1, Vm1^T, Gua2, Vm2^T and G(4,S) = Gua1^T, Vm1, Gua2^T, Vm2, read
// from the Gua1 | Gua2 | Vm1 | Vm2 blocks at L_G with one indexed load per entry.
__device__ __forceinline__ m3<double> g_block(const double *o, int idx, bool row4)
{
    const int off = L_G + ((idx & 1) ? 18 + 9 * (idx >> 1) : 9 * (idx >> 1));
    const bool transpose = ((idx & 1) != 0) != row4;
    m3<double> r;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) r.a[3 * i + j] = o[off + (transpose ? 3 * j + i : 3 * i + j)];
    return r;
}

struct ShellKin {
    v3<double> u, u1, u2, a, a1, a2, z1, z2, eta1, eta2, k1, k2;
    m3<double> Q, Xi, Xi1, Xi2, QQ;
    double g;
};

// ZERO: the incremental displacements are taken as zero (disp and conn unused).
template <bool ZERO = false>
__device__ void shell_kin(const double *__restrict__ cst, const double *__restrict__ gps, size_t ld, int e, int gp,
                          const double *__restrict__ disp, const int *__restrict__ conn, ShellKin &k)
{
    double u[3] = {0, 0, 0}, u1[3] = {0, 0, 0}, u2[3] = {0, 0, 0};
    for (int a = 0; a < (ZERO ? 0 : 6); a++) {
        const double *p = disp + 6 * (size_t)conn[a * ld + e];
        double c0 = cst[(SC_NU + 6 * gp + a) * ld + e], c1 = cst[(SC_NU1 + 6 * gp + a) * ld + e],
               c2 = cst[(SC_NU2 + 6 * gp + a) * ld + e];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double v = p[i];
            u[i] += v * c0;
            u1[i] += v * c1;
            u2[i] += v * c2;
        }
    }
    double al[3] = {0, 0, 0}, al1[3] = {0, 0, 0}, al2[3] = {0, 0, 0};
    for (int b = 0; b < (ZERO ? 0 : 3); b++) {
        const double *p = disp + 6 * (size_t)conn[(3 + b) * ld + e] + 3;
        double c0 = cst[(SC_NA + 3 * gp + b) * ld + e], c1 = cst[(SC_NA1 + 3 * gp + b) * ld + e],
               c2 = cst[(SC_NA2 + 3 * gp + b) * ld + e];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double v = p[i];
            al[i] += v * c0;
            al1[i] += v * c1;
            al2[i] += v * c2;
        }
    }
    m3<double> T3;
#pragma unroll
    for (int i = 0; i < 9; i++) T3.a[i] = cst[(SC_T3 + i) * ld + e];
    k.u = mv(T3, mk3(u[0], u[1], u[2]));
    k.u1 = mv(T3, mk3(u1[0], u1[1], u1[2]));
    k.u2 = mv(T3, mk3(u2[0], u2[1], u2[2]));
    k.a = mv(T3, mk3(al[0], al[1], al[2]));
    k.a1 = mv(T3, mk3(al1[0], al1[1], al1[2]));
    k.a2 = mv(T3, mk3(al2[0], al2[1], al2[2]));
    rodrigues(k.a, k.Q, k.Xi, k.g);
    m3<double> A1 = skew3(k.a1), A2 = skew3(k.a2);
    double p1 = dot3(k.a, k.a1), p2 = dot3(k.a, k.a2);
#pragma unroll
    for (int i = 0; i < 9; i++) {
        k.Xi1.a[i] = -0.5 * k.g * (p1 * k.Xi.a[i] - A1.a[i]);
        k.Xi2.a[i] = -0.5 * k.g * (p2 * k.Xi.a[i] - A2.a[i]);
    }
    const size_t o = (size_t)SG_PER_GP * gp;
    m3<double> Qi;
#pragma unroll
    for (int i = 0; i < 9; i++) Qi.a[i] = gps[(o + i) * ld + e];
    v3<double> kr1 = mk3(gps[(o + 9) * ld + e], gps[(o + 10) * ld + e], gps[(o + 11) * ld + e]);
    v3<double> kr2 = mk3(gps[(o + 12) * ld + e], gps[(o + 13) * ld + e], gps[(o + 14) * ld + e]);
    v3<double> zx1 = mk3(gps[(o + 15) * ld + e], gps[(o + 16) * ld + e], gps[(o + 17) * ld + e]);
    v3<double> zx2 = mk3(gps[(o + 18) * ld + e], gps[(o + 19) * ld + e], gps[(o + 20) * ld + e]);
    k.z1 = add3(k.u1, zx1);
    k.z2 = add3(k.u2, zx2);
    k.QQ = mm3(k.Q, Qi);
    k.eta1 = mtv(k.QQ, k.z1);
    k.eta2 = mtv(k.QQ, k.z2);
    k.eta1.x -= 1.0;
    k.eta2.y -= 1.0;
    k.k1 = add3(mtv(Qi, mtv(k.Xi, k.a1)), kr1);
    k.k2 = add3(mtv(Qi, mtv(k.Xi, k.a2)), kr2);
}

// One point of the through-thickness rule (src/Shell_1.cpp:1083-1145): the
// strains gamma_a = eta_a + zeta kappa_a x e3 (e3 = (0,0,1)), v and dv of the
// hyperelastic law at jbar = det of the in-plane stretch, and the stress vectors
// tau_1, tau_2.
struct ShellPt {
    double g11, g12, g13, g21, g22, g23, v, dv;
    v3<double> tau1, tau2;
};
__device__ __forceinline__ ShellPt shell_point(const ShellKin &k, double mu, double la, double zeta)
{
    ShellPt p;
    p.g11 = k.eta1.x + zeta * k.k1.y;
    p.g12 = k.eta1.y - zeta * k.k1.x;
    p.g13 = k.eta1.z;
    p.g21 = k.eta2.x + zeta * k.k2.y;
    p.g22 = k.eta2.y - zeta * k.k2.x;
    p.g23 = k.eta2.z;
    const double jb = (1.0 + p.g11) * (1.0 + p.g22) - p.g12 * p.g21;
    p.v = (la * (jb * jb * jb - 1.0) + 2.0 * mu * (jb - 1.0)) / (la * jb * jb * jb + 2.0 * mu * jb);
    p.dv = ((la + 2.0 * mu) * (3.0 * la * jb * jb + 2.0 * mu)) /
           (jb * jb * (la * jb * jb + 2.0 * mu) * (la * jb * jb + 2.0 * mu));
    p.tau1 = mk3(mu * p.v * (1.0 + p.g22) + mu * (p.g11 - p.g22), mu * p.v * (-p.g21) + mu * (p.g12 + p.g21),
                 mu * p.g13);
    p.tau2 = mk3(mu * p.v * (-p.g12) + mu * (p.g12 + p.g21), mu * p.v * (1.0 + p.g11) + mu * (p.g22 - p.g11),
                 mu * p.g23);
    return p;
}

// DOF block I of an element -> (node, first component)
__device__ __forceinline__ void dof_block(const int *__restrict__ conn, size_t ld, int e, int I, int &node, int &c0)
{
    if (I < 6) { node = conn[I * ld + e]; c0 = 0; }
    else { node = conn[(3 + I - 6) * ld + e]; c0 = 3; }
}

// Phase 1 of Shell_1::Mount for one (element, Gauss point) in two parts: the
// 3-point thickness integration, which writes the D blocks oD[0 .. 144) and the
// stress resultants, and the rest of the record (Psi, G blocks, Psi^T sigma) that
// the later phases read, o[L_P .. L_M).
//
// The D blocks are sums over the points of w zeta^p C (p = 0, 1, 2) with C11, C12,
// C22 full only in their upper 2 x 2 and (2, 2): 32 sums in registers and one write
// of each entry, instead of 3 x 144 read-modify-writes of LDS.
struct ShellRes {
    v3<double> n1, n2, m1, m2;
};
__device__ __forceinline__ void shell_gp_moduli(const double *__restrict__ cst, size_t ld, int e, const ShellKin &k,
                                                double *oD, ShellRes &sr)
{
    const double mu = cst[SC_MU * ld + e], la = cst[SC_LAMBDA * ld + e], th = cst[SC_THICK * ld + e];
    const double drill = cst[SC_DRILL * ld + e];
    v3<double> n1 = mk3(0.0, 0.0, 0.0), n2 = n1, m1 = n1, m2 = n1;
    const double xi[3] = {-0.77459666924148337703585307995648, 0.0, 0.77459666924148337703585307995648};
    const double wt[3] = {0.55555555555555555555555555555556, 0.88888888888888888888888888888889,
                          0.55555555555555555555555555555556};
    const double J = th / 2.0;
    m3<double> C11[3], C12[3], C22[3];
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
        for (int i = 0; i < 9; i++) C11[p].a[i] = C12[p].a[i] = C22[p].a[i] = 0.0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        double zeta = th * xi[q] / 2.0;
        const ShellPt pt = shell_point(k, mu, la, zeta);
        const double g11 = pt.g11, g12 = pt.g12, g21 = pt.g21, g22 = pt.g22, v = pt.v, dv = pt.dv;
        const v3<double> tau1 = pt.tau1, tau2 = pt.tau2;
        const double a0 = mu * ((1.0 + g22) * (1.0 + g22) * dv + 1.0), a1 = -mu * (1.0 + g22) * g21 * dv,
                     a4 = mu * (g21 * g21 * dv + 1.0);
        const double c0 = mu * (g12 * g12 * dv + 1.0), c1 = -mu * ((1.0 + g11) * g12 * dv),
                     c4 = mu * ((1.0 + g11) * (1.0 + g11) * dv + 1.0);
        const double b0 = -mu * ((1.0 + g22) * g12 * dv), b1 = mu * (v - 1.0 + (1.0 + g11) * (1.0 + g22) * dv),
                     b3 = mu * (1.0 - v + g12 * g21 * dv), b4 = -mu * ((1.0 + g11) * g21 * dv);
        double w = wt[q] * J;
        const double wz[3] = {w, w * zeta, w * zeta * zeta};
#pragma unroll
        for (int p = 0; p < 3; p++) {
            C11[p].a[0] += wz[p] * a0;
            C11[p].a[1] += wz[p] * a1;
            C11[p].a[4] += wz[p] * a4;
            C12[p].a[0] += wz[p] * b0;
            C12[p].a[1] += wz[p] * b1;
            C12[p].a[3] += wz[p] * b3;
            C12[p].a[4] += wz[p] * b4;
            C22[p].a[0] += wz[p] * c0;
            C22[p].a[1] += wz[p] * c1;
            C22[p].a[4] += wz[p] * c4;
        }
        C11[0].a[8] += w * mu;  // (E3's products drop it where zeta stands)
        n1 = add3(n1, scl3(w, tau1));
        n2 = add3(n2, scl3(w, tau2));
        // e3 x tau = (-tau.y, tau.x, 0)
        m1 = add3(m1, scl3(w * zeta, mk3(-tau1.y, tau1.x, 0.0)));
        m2 = add3(m2, scl3(w * zeta, mk3(-tau2.y, tau2.x, 0.0)));
    }
    C22[0].a[8] = C11[0].a[8];
#pragma unroll
    for (int p = 0; p < 3; p++) {
        C11[p].a[3] = C11[p].a[1];
        C22[p].a[3] = C22[p].a[1];
    }
    auto blocks = [](double *o, const m3<double> &X0, const m3<double> &X1, const m3<double> &X2)
        __attribute__((always_inline)) {
        st3(o + 9 * 0, X0);                              // dn/deta
        st3(o + 9 * 1, mscl(-1.0, mE3(X1)));             // dn/dk
        st3(o + 9 * 4, E3m(X1));                         // dm/deta
        st3(o + 9 * 5, mscl(-1.0, mE3(E3m(X2))));        // dm/dk
    };
    blocks(oD + 9 * 0, C11[0], C11[1], C11[2]);
    blocks(oD + 9 * 2, C12[0], C12[1], C12[2]);
    blocks(oD + 9 * 8, tr3(C12[0]), tr3(C12[1]), tr3(C12[2]));
    blocks(oD + 9 * 10, C22[0], C22[1], C22[2]);
    // drilling (overwrites, as the reference)
    oD[9 * 5 + 8] = drill;   // D(5,5): block (1,1) entry (2,2)
    oD[9 * 15 + 8] = drill;  // D(11,11): block (3,3) entry (2,2)
    m1.z = drill * k.k1.z;
    m2.z = drill * k.k2.z;
    sr.n1 = n1;
    sr.n2 = n2;
    sr.m1 = m1;
    sr.m2 = m2;
}

__device__ __forceinline__ void shell_gp_rest(const ShellKin &k, const ShellRes &sr, double *o)
{
    const v3<double> n1 = sr.n1, n2 = sr.n2, m1 = sr.m1, m2 = sr.m2;
    m3<double> Qt = tr3(k.QQ);
    m3<double> QtXi = mm3(Qt, k.Xi);
    m3<double> Z1 = skew3(k.z1), Z2 = skew3(k.z2);
    m3<double> W0 = mm3(mm3(Qt, Z1), k.Xi), W1 = mm3(Qt, k.Xi1);
    m3<double> W2 = mm3(mm3(Qt, Z2), k.Xi), W3 = mm3(Qt, k.Xi2);
    st3(o + L_P + 0, Qt);
    st3(o + L_P + 9, QtXi);
    st3(o + L_P + 18, Qt);
    st3(o + L_P + 27, QtXi);
    st3(o + L_W + 0, W0);
    st3(o + L_W + 9, W1);
    st3(o + L_W + 18, W2);
    st3(o + L_W + 27, W3);
    // Psi^T sigma
    v3<double> s0 = mtv(Qt, n1), s1 = mtv(QtXi, m1), s2 = mtv(Qt, n2), s3 = mtv(QtXi, m2);
    v3<double> s4 = add3(add3(mtv(W0, n1), mtv(W1, m1)), add3(mtv(W2, n2), mtv(W3, m2)));
    double *S = o + L_S;
    S[0] = s0.x; S[1] = s0.y; S[2] = s0.z; S[3] = s1.x; S[4] = s1.y; S[5] = s1.z;
    S[6] = s2.x; S[7] = s2.y; S[8] = s2.z; S[9] = s3.x; S[10] = s3.y; S[11] = s3.z;
    S[12] = s4.x; S[13] = s4.y; S[14] = s4.z;
    // geometric blocks
    v3<double> n_1 = mv(k.QQ, n1), n_2 = mv(k.QQ, n2), m_1 = mv(k.QQ, m1), m_2 = mv(k.QQ, m2);
    m3<double> Gua1 = mscl(-1.0, mm3(skew3(n_1), k.Xi));
    m3<double> Gua2 = mscl(-1.0, mm3(skew3(n_2), k.Xi));
    m3<double> Vm1 = opV(k.a, m_1), Vm2 = opV(k.a, m_2);
    m3<double> XiT = tr3(k.Xi);
    m3<double> Ga1 = msub(mm3(XiT, mm3(mm3(Z1, skew3(n_1)), k.Xi)), opV(k.a, mv(Z1, n_1)));
    Ga1 = madd(Ga1, msub(opdV(k.a, k.a1, m_1), mtm3(k.Xi1, mm3(skew3(m_1), k.Xi))));
    m3<double> Ga2 = msub(mm3(XiT, mm3(mm3(Z2, skew3(n_2)), k.Xi)), opV(k.a, mv(Z2, n_2)));
    Ga2 = madd(Ga2, msub(opdV(k.a, k.a2, m_2), mtm3(k.Xi2, mm3(skew3(m_2), k.Xi))));
    st3(o + L_G + 0, Gua1);
    st3(o + L_G + 9, Gua2);
    st3(o + L_G + 18, Vm1);
    st3(o + L_G + 27, Vm2);
    st3(o + L_G + 36, madd(Ga1, Ga2));
}

// An element's constants in LDS: dN coefficients NU1, NU2, NA1, NA2, NA by Gauss
// point, T3, the Gauss weight.
constexpr int CF_NA1 = 36, CF_NA2 = 45, CF_NA = 54, CF_T3 = 63, CF_W = 72, CF_N = 73, CF_LD = 73;
static_assert(SC_NU2 == SC_NU1 + 18, "NU1 and NU2 follow one another");

__device__ __forceinline__ m3<double> mzero()
{
    m3<double> r;
#pragma unroll
    for (int q = 0; q < 9; q++) r.a[q] = 0.0;
    return r;
}
// x of one lane of each four (CTRL: quad_perm of four times the same lane)
template <int CTRL> __device__ __forceinline__ double quad_get(double x)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// K_IJ of element e, rotated to global
__device__ __forceinline__ void k_store(double *__restrict__ Kout, int e, int I, int J, const double *t3, const m3<double> &Kl)
{
    const m3<double> T3 = ld3(t3), K = mtm3(T3, mm3(Kl, T3));
    double *Ke = Kout + (size_t)e * 729;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) Ke[(3 * I + i) * 27 + 3 * J + j] = K.a[3 * i + j];
}

// Bound by its products' LDS reads (9 or 18 a product of 27 multiply-adds): 338 elements
// 28 us -> 9, 8,192 90 -> 40, since each wavefront runs one form of its phase and the
// constants are read once.
template <bool PRE>
__global__ __launch_bounds__(SWG, PRE ? 3 : 1) void shell_element_kernel(
    int e0, int e1, size_t ld, const int *__restrict__ conn, const double *__restrict__ cst,
    const double *__restrict__ gps, const double *__restrict__ disp, double *__restrict__ Kout,
    double *__restrict__ fout, const double *__restrict__ pre)
{
    __shared__ double sm[SEPB * 3 * L_GP + SEPB * CF_LD];
    const int tid = threadIdx.x;
    const int ebase = e0 + blockIdx.x * SEPB;

    const int lane = tid & 63, wave = tid >> 6, nv = min(SEPB, e1 - ebase);

    // ---- the elements' constants; phase 1 (or its records from shell_record_kernel) ----
    double *cf = sm + SEPB * 3 * L_GP;
    for (int t = tid; t < SEPB * CF_N; t += SWG) {
        const int le = t % SEPB, c = t / SEPB;
        const int src = c < CF_NA1   ? SC_NU1 + c  // (NU1 and NU2 follow one another)
                        : c < CF_NA2 ? SC_NA1 + c - CF_NA1
                        : c < CF_NA  ? SC_NA2 + c - CF_NA2
                        : c < CF_T3  ? SC_NA + c - CF_NA
                        : c < CF_W   ? SC_T3 + c - CF_T3
                                     : SC_ALPHA1;
        if (le < nv) cf[le * CF_LD + c] = cst[(size_t)src * ld + ebase + le];
    }
    if constexpr (PRE) {
        const double *src = pre + (size_t)ebase * 3 * L_M;
        constexpr int NL = (SEPB * 3 * L_M + SWG - 1) / SWG;
        double v[NL];
#pragma unroll
        for (int i = 0; i < NL; i++) v[i] = src[min(tid + SWG * i, nv * 3 * L_M - 1)];
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int t = tid + SWG * i;
            if (t < nv * 3 * L_M) sm[(t / L_M) * L_GP + t % L_M] = v[i];
        }
    } else if (tid < 3 * SEPB) {
        int le = tid / 3, gp = tid - 3 * (tid / 3);
        int e = ebase + le;
        double *o = sm + (le * 3 + gp) * L_GP;
        if (e < e1) {
            ShellKin k;
            ShellRes sr;
            shell_kin(cst, gps, ld, e, gp, disp, conn, k);
            shell_gp_moduli(cst, ld, e, k, o + L_D, sr);
            shell_gp_rest(k, sr, o);
        }
    }
    __syncthreads();

    // ---- phase 2: M blocks ---------------------------------------------------
    // (R, S), R, S < 4: three wavefronts, two products a lane, after which the first
    // takes the (4, S); the fourth the (R, 4), whose W_R^T V_R add up to (4, 4).
    // (One lane a block in order sent every wavefront through all four forms: 20
    // products for (4, 4) alone, twice where 300 tasks meet 256 lanes.)
    if (wave < 3) {
        const int p = tid >> 4, R = (tid >> 2) & 3, S = tid & 3;
        if (p < 3 * nv) {
            double *o = sm + p * L_GP;
            st3(o + L_M + 9 * (5 * R + S),
                mtm3(ld3(o + L_P + 9 * R), mm3(ld3(o + L_D + 9 * (4 * R + S)), ld3(o + L_P + 9 * S))));
        }
        if (wave == 0 && (lane >> 2) < 3 * nv) {
            double *o = sm + (lane >> 2) * L_GP;
            m3<double> V = mtm3(ld3(o + L_W), ld3(o + L_D + 9 * S));
#pragma unroll
            for (int i = 1; i < 4; i++) V = madd(V, mtm3(ld3(o + L_W + 9 * i), ld3(o + L_D + 9 * (4 * i + S))));
            st3(o + L_M + 9 * (20 + S), madd(mm3(V, ld3(o + L_P + 9 * S)), g_block(o, S, true)));
        }
    } else if ((lane >> 2) < 3 * nv) {
        const int R = lane & 3;
        double *o = sm + (lane >> 2) * L_GP;
        m3<double> V = mm3(ld3(o + L_D + 9 * (4 * R)), ld3(o + L_W));
#pragma unroll
        for (int j = 1; j < 4; j++) V = madd(V, mm3(ld3(o + L_D + 9 * (4 * R + j)), ld3(o + L_W + 9 * j)));
        st3(o + L_M + 9 * (5 * R + 4), madd(mtm3(ld3(o + L_P + 9 * R), V), g_block(o, R, false)));
        const m3<double> U = mtm3(ld3(o + L_W + 9 * R), V);
        m3<double> acc;
#pragma unroll
        for (int q = 0; q < 9; q++)
            acc.a[q] = ((quad_get<0x00>(U.a[q]) + quad_get<0x55>(U.a[q])) + quad_get<0xAA>(U.a[q])) + quad_get<0xFF>(U.a[q]);
        if (R == 0) st3(o + L_M + 9 * 24, madd(acc, ld3(o + L_G + 36)));
    }
    __syncthreads();

    // ---- phase 3: K_IJ, by the number of M blocks it takes (9, 6, 4 a Gauss point) --
    if (wave == 0) {
        const int le = lane / 9, I = (lane - 9 * le) / 3, J = lane % 3;
        if (le < nv) {
            m3<double> K = mzero();
            for (int gp = 0; gp < 3; gp++) {
                const double *M = sm + (le * 3 + gp) * L_GP + L_M, *c = cf + le * CF_LD + CF_NA1 + 3 * gp;
#pragma unroll
                for (int a = 0; a < 3; a++)
#pragma unroll
                    for (int b = 0; b < 3; b++)
                        acc3(K.a, cf[le * CF_LD + CF_W] * c[9 * a + I] * c[9 * b + J],
                             ld3(M + 9 * (5 * (a == 2 ? 4 : 1 + 2 * a) + (b == 2 ? 4 : 1 + 2 * b))));
            }
            k_store(Kout, ebase + le, 6 + I, 6 + J, cf + le * CF_LD + CF_T3, K);
        }
    } else if (wave < 3) {
        // displacement I against rotation J (18 a element), then the other way round
        for (int t = lane + 64 * (wave - 1); t < 36 * SEPB; t += 128) {
            const int le = t / 36, x = t - 36 * le, d = (x % 18) / 3, r = x % 3;
            const bool rows = x < 18;  // displacement rows
            if (le >= nv) break;
            m3<double> K = mzero();
            const int sd = rows ? 45 : 9, sr = rows ? 9 : 45;  // strides of M by the displacement's and the rotation's row
            for (int gp = 0; gp < 3; gp++) {
                const double *M = sm + (le * 3 + gp) * L_GP + L_M, *cd = cf + le * CF_LD + 6 * gp + d,
                             *cr = cf + le * CF_LD + CF_NA1 + 3 * gp + r;
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < 3; b++)
                        acc3(K.a, cf[le * CF_LD + CF_W] * cd[18 * a] * cr[9 * b],
                             ld3(M + 2 * a * sd + (b == 2 ? 4 : 1 + 2 * b) * sr));
            }
            k_store(Kout, ebase + le, rows ? d : 6 + r, rows ? 6 + r : d, cf + le * CF_LD + CF_T3, K);
        }
        // ---- phase 4: internal force ----------------------------------------
        if (wave == 2 && lane < 9 * nv) {
            const int le = lane / 9, I = lane - 9 * le;
            const double *c = cf + le * CF_LD;
            const double w = c[CF_W];
            v3<double> f = mk3(0.0, 0.0, 0.0);
            for (int gp = 0; gp < 3; gp++) {
                const double *S = sm + (le * 3 + gp) * L_GP + L_S;
                auto add = [&](double x, int R) { f = add3(f, scl3(w * x, mk3(S[3 * R], S[3 * R + 1], S[3 * R + 2]))); };
                if (I < 6) {
                    add(c[6 * gp + I], 0);
                    add(c[18 + 6 * gp + I], 2);
                } else {
                    add(c[CF_NA1 + 3 * gp + I - 6], 1);
                    add(c[CF_NA2 + 3 * gp + I - 6], 3);
                    add(c[CF_NA + 3 * gp + I - 6], 4);
                }
            }
            f = mtv(ld3(c + CF_T3), f);
            double *fo = fout + (size_t)(ebase + le) * 27 + 3 * I;
            fo[0] = f.x;
            fo[1] = f.y;
            fo[2] = f.z;
        }
    } else {
        for (int t = lane; t < 36 * SEPB; t += 64) {
            const int le = t / 36, I = (t - 36 * le) / 6, J = t % 6;
            if (le >= nv) break;
            m3<double> K = mzero();
            for (int gp = 0; gp < 3; gp++) {
                const double *M = sm + (le * 3 + gp) * L_GP + L_M, *c = cf + le * CF_LD + 6 * gp;
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < 2; b++)
                        acc3(K.a, cf[le * CF_LD + CF_W] * c[18 * a + I] * c[18 * b + J], ld3(M + 9 * (10 * a + 2 * b)));
            }
            k_store(Kout, ebase + le, I, J, cf + le * CF_LD + CF_T3, K);
        }
    }
}

// Follower pressure (MountShellSpecialLoads) of all elements, PE a workgroup: a lane
// per (element, point) finds the surface's tangents and normal there, then a lane per
// (element, u-nodes a, b) sums the points.  The record out[(6 e + a) SPR ...] holds
// the unbalanced-force change P_a (3) and the load stiffness rows of node a (3 x 18,
// global frame); zeros for an element without pressure.  The assembly (by rows or by
// colour) adds them to the element's own.  A lane per (element, a) with all of it took
// 18 us at 338 elements (its 6 x 6 products one after another), 26 us at 8,192; a lane
// per (element, a, b) that finds the tangents itself 11 and 40 us; this one 9 and 25.
constexpr int PE = 7;

__global__ __launch_bounds__(256) void shell_pressure_record_kernel(
    int ns, size_t ld, const int *__restrict__ conn, const double *__restrict__ cst,
    const double *__restrict__ pc, const double *__restrict__ disp, const double *__restrict__ copy,
    const double *__restrict__ copy0, const int *__restrict__ pload, const int *__restrict__ pflag,
    const double *__restrict__ lrec, const double *__restrict__ tab_t, const double *__restrict__ tab_v, const double *__restrict__ tp,
    double *__restrict__ out)
{
    __shared__ double sp[PE * 6][31];  // t1, t2, n, |t1 x t2|, w4, p; N, N1, N2 of the six nodes
    const double time = *tp;  // load time, device-resident (a captured Newton step reads the current one)
    const int tid = threadIdx.x, e0 = blockIdx.x * PE;
    const int le = tid / 36, ab = tid - 36 * le, a = ab / 6, b = ab - 6 * a, e = e0 + le;
    const bool act = le < PE && e < ns;
    const int L = act ? pload[e] : -1;
    for (int t = tid; t < PE * 108; t += 256) {
        const int c = t / PE, l = t - PE * c, f = c / 36, ga = c - 36 * f;
        const int row = (f == 0 ? SP_N4U : f == 1 ? SP_N4U1 : SP_N4U2) + ga;
        sp[6 * l + ga / 6][12 + 6 * f + ga % 6] = pc[(size_t)row * ld + min(e0 + l, ns - 1)];
    }
    if (tid < 6 * PE && e0 + tid / 6 < ns) {
        const int eg = e0 + tid / 6, g = tid % 6, Lg = pload[eg];
        if (Lg >= 0) {
            const double *rec = lrec + (size_t)Lg * NL_REC;
            const double p = gf_table_value(tab_t, tab_v, (int)rec[NL_TAB0], (int)rec[NL_TABN], time, 0);
            v3<double> t1 = mk3(cst[(SC_T3 + 0) * ld + eg], cst[(SC_T3 + 1) * ld + eg], cst[(SC_T3 + 2) * ld + eg]);
            v3<double> t2 = mk3(cst[(SC_T3 + 3) * ld + eg], cst[(SC_T3 + 4) * ld + eg], cst[(SC_T3 + 5) * ld + eg]);
#pragma unroll
            for (int c = 0; c < 6; c++) {
                const size_t nd = 6 * (size_t)conn[c * ld + eg];
                const double d1 = pc[(SP_N4U1 + 6 * g + c) * ld + eg], d2 = pc[(SP_N4U2 + 6 * g + c) * ld + eg];
                const v3<double> pu = mk3((copy[nd] - copy0[nd]) + disp[nd], (copy[nd + 1] - copy0[nd + 1]) + disp[nd + 1],
                                          (copy[nd + 2] - copy0[nd + 2]) + disp[nd + 2]);
                t1 = add3(t1, scl3(d1, pu));
                t2 = add3(t2, scl3(d2, pu));
            }
            const v3<double> cr = cross3(t1, t2);
            const double ncr = sqrt(dot3(cr, cr));
            const v3<double> n = scl3(1.0 / ncr, cr);
            double *o = sp[tid];
            o[0] = t1.x; o[1] = t1.y; o[2] = t1.z;
            o[3] = t2.x; o[4] = t2.y; o[5] = t2.z;
            o[6] = n.x; o[7] = n.y; o[8] = n.z;
            o[9] = ncr;
            o[10] = pc[(SP_W4 + g) * ld + eg];
            o[11] = p;
        }
    }
    __syncthreads();
    if (!act) return;
    double *o = out + ((size_t)6 * e + a) * SPR;
    if (L < 0) {
        for (int q = b; q < SPR; q += 6) o[q] = 0.0;
        return;
    }
    const int au = pflag[e];
    double Kr[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    v3<double> Pa = mk3(0.0, 0.0, 0.0);
#pragma unroll 2
    for (int g = 0; g < 6; g++) {
        const double *q = sp[6 * le + g];
        const v3<double> t1 = mk3(q[0], q[1], q[2]), t2 = mk3(q[3], q[4], q[5]), n = mk3(q[6], q[7], q[8]);
        const double ncr = q[9], w4 = q[10], p = q[11], Na = q[12 + a], c1 = q[18 + b], c2 = q[24 + b];
        const double jac = au ? ncr : 1.0;
        // unbalanced force change: P -= w4 jac N4^T q with q = -p n
        Pa = add3(Pa, scl3(w4 * jac * Na * p, n));
        const m3<double> S1 = skew3(t1), S2 = skew3(t2);
        m3<double> B = msub(mscl(c2, S1), mscl(c1, S2));
        if (!au) {
            m3<double> Pm;
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    double ni = i == 0 ? n.x : (i == 1 ? n.y : n.z), nj = j == 0 ? n.x : (j == 1 ? n.y : n.z);
                    Pm.a[3 * i + j] = ((i == j ? 1.0 : 0.0) - ni * nj) / ncr;
                }
            B = mm3(Pm, B);
        }
        const double s = w4 * 1.0 * p * Na;
#pragma unroll
        for (int i = 0; i < 9; i++) Kr[i] += s * B.a[i];
    }
    // the element's unbalanced force grows by Pa (the residual takes its negative)
    if (b < 3) o[b] = b == 0 ? Pa.x : b == 1 ? Pa.y : Pa.z;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) o[3 + 18 * i + 3 * b + j] = Kr[3 * i + j];
}

// Phase 1 of every element's Gauss points in one launch: lane per (element, gp),
// NP points a wavefront.  A wavefront's instructions bound it (stores of 8 bytes in 64
// lines, and sums in LDS, took half of 26 us at 338 elements, 37 at 8,192; now 12 and
// 22).  Both parts of the record pass through LDS and are copied
// out by all 64 lanes, in rows (a lane's stride is odd: a wavefront's accesses stay
// off shared banks).  The element kernel reads the records instead of recomputing
// phase 1 on 12 lanes per workgroup.
constexpr int REC_DS = 145;

__device__ __forceinline__ void record_rows(double *dst, const double *src, int stride, int width, int nt)
{
    int i = threadIdx.x, r = 0;  // (width > 64: an entry is at most one row further)
    const int n = nt * width;
#pragma unroll 4
    for (int q = threadIdx.x; q < n; q += 64) {
        dst[(size_t)r * L_M + i] = src[r * stride + i];
        i += 64;
        if (i >= width) {
            i -= width;
            r++;
        }
    }
}

template <int NP>
__global__ __launch_bounds__(64) void shell_record_kernel(int ns, size_t ld, const int *__restrict__ conn,
                                                          const double *__restrict__ cst,
                                                          const double *__restrict__ gps,
                                                          const double *__restrict__ disp, double *__restrict__ rec)
{
    __shared__ double sD[NP * REC_DS];
    const int t0 = blockIdx.x * NP, t = t0 + threadIdx.x;
    const int nt = min(NP, 3 * ns - t0);
    const bool act = (int)threadIdx.x < nt;
    const int e = t / 3, gp = t - 3 * (t / 3);
    double *own = sD + threadIdx.x * REC_DS, *out = rec + (size_t)t0 * L_M;
    ShellKin k;
    ShellRes sr;
    if (act) {
        shell_kin(cst, gps, ld, e, gp, disp, conn, k);
        shell_gp_moduli(cst, ld, e, k, own, sr);
    }
    __syncthreads();
    record_rows(out + L_D, sD, REC_DS, L_P - L_D, nt);
    __syncthreads();
    if (act) shell_gp_rest(k, sr, own - L_P);
    __syncthreads();
    record_rows(out + L_P, sD, REC_DS, L_M - L_P, nt);
}

__global__ __launch_bounds__(256) void shell_commit_kernel(int ns, size_t ld, const int *__restrict__ conn,
                                                           const double *__restrict__ cst, double *__restrict__ gps,
                                                           const double *__restrict__ disp)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 3 * ns) return;
    int e = t / 3, gp = t - 3 * (t / 3);
    ShellKin k;
    shell_kin(cst, gps, ld, e, gp, disp, conn, k);
    const size_t o = (size_t)SG_PER_GP * gp;
    m3<double> Qi;
#pragma unroll
    for (int i = 0; i < 9; i++) Qi.a[i] = gps[(o + i) * ld + e];
    m3<double> Qn = mm3(k.Q, Qi);
#pragma unroll
    for (int i = 0; i < 9; i++) gps[(o + i) * ld + e] = Qn.a[i];
    gps[(o + 9) * ld + e] = k.k1.x;
    gps[(o + 10) * ld + e] = k.k1.y;
    gps[(o + 11) * ld + e] = k.k1.z;
    gps[(o + 12) * ld + e] = k.k2.x;
    gps[(o + 13) * ld + e] = k.k2.y;
    gps[(o + 14) * ld + e] = k.k2.z;
    gps[(o + 15) * ld + e] += k.u1.x;
    gps[(o + 16) * ld + e] += k.u1.y;
    gps[(o + 17) * ld + e] += k.u1.z;
    gps[(o + 18) * ld + e] += k.u2.x;
    gps[(o + 19) * ld + e] += k.u2.y;
    gps[(o + 20) * ld + e] += k.u2.z;
}

// Results of the committed state (Shell_1::WriteResults src/Shell_1.cpp:624-666):
// per element the means over the three Gauss points of n_r1, m_r1, n_r2, m_r2,
// eta_r1, kappa_r1, eta_r2, kappa_r2.  With zero incremental displacements the
// kinematics reduce to the committed Q_i, kappa_i, z_x1, z_x2, which hold the
// converged configuration of the last Mount.  out: [ns][24], colour-sorted.
__global__ __launch_bounds__(256) void shell_results_kernel(int ns, size_t ld, const double *__restrict__ cst,
                                                            const double *__restrict__ gps, double *__restrict__ out)
{
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ns) return;
    const double mu = cst[SC_MU * ld + e], la = cst[SC_LAMBDA * ld + e], th = cst[SC_THICK * ld + e];
    const double drill = cst[SC_DRILL * ld + e];
    const double xi[3] = {-0.77459666924148337703585307995648, 0.0, 0.77459666924148337703585307995648};
    const double wt[3] = {0.55555555555555555555555555555556, 0.88888888888888888888888888888889,
                          0.55555555555555555555555555555556};
    const double J = th / 2.0;
    v3<double> avg[8];
#pragma unroll
    for (int i = 0; i < 8; i++) avg[i] = mk3(0.0, 0.0, 0.0);
    for (int gp = 0; gp < 3; gp++) {
        ShellKin k;
        shell_kin<true>(cst, gps, ld, e, gp, nullptr, nullptr, k);
        v3<double> n1 = mk3(0.0, 0.0, 0.0), n2 = n1, m1 = n1, m2 = n1;
        for (int q = 0; q < 3; q++) {
            const double zeta = th * xi[q] / 2.0;
            const ShellPt pt = shell_point(k, mu, la, zeta);
            const double w = wt[q] * J;
            n1 = add3(n1, scl3(w, pt.tau1));
            n2 = add3(n2, scl3(w, pt.tau2));
            m1 = add3(m1, scl3(w * zeta, mk3(-pt.tau1.y, pt.tau1.x, 0.0)));
            m2 = add3(m2, scl3(w * zeta, mk3(-pt.tau2.y, pt.tau2.x, 0.0)));
        }
        m1.z = drill * k.k1.z;
        m2.z = drill * k.k2.z;
        const v3<double> r[8] = {n1, m1, n2, m2, k.eta1, k.k1, k.eta2, k.k2};
#pragma unroll
        for (int i = 0; i < 8; i++) avg[i] = add3(avg[i], scl3(1.0 / 3.0, r[i]));
    }
    double *o = out + 24 * (size_t)e;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        o[3 * i] = avg[i].x;
        o[3 * i + 1] = avg[i].y;
        o[3 * i + 2] = avg[i].z;
    }
}

}  // namespace

// ---- host: constants (Shell_1::PreCalc restated for the device layout) ---------
static void vsub(const double *a, const double *b, double *c) { for (int i = 0; i < 3; i++) c[i] = a[i] - b[i]; }
static void vcross(const double *a, const double *b, double *c)
{
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}
static double vdot(const double *a, const double *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
static double vnorm(const double *a) { return std::sqrt(vdot(a, a)); }

static void tri_shapes(double L1, double L2, double L3, const double *dx, const double *dy, double *Nu, double *Nu1,
                       double *Nu2, double *Na, double *Na1, double *Na2)
{
    double L1x = dx[0], L2x = dx[1], L3x = dx[2], L1y = dy[0], L2y = dy[1], L3y = dy[2];
    Nu[0] = (2 * L1 - 1) * L1; Nu[1] = (2 * L2 - 1) * L2; Nu[2] = (2 * L3 - 1) * L3;
    Nu[3] = 4 * L1 * L2; Nu[4] = 4 * L2 * L3; Nu[5] = 4 * L3 * L1;
    Nu1[0] = 4 * L1x * L1 - L1x; Nu1[1] = 4 * L2x * L2 - L2x; Nu1[2] = 4 * L3x * L3 - L3x;
    Nu1[3] = 4 * L1x * L2 + 4 * L1 * L2x; Nu1[4] = 4 * L2x * L3 + 4 * L2 * L3x; Nu1[5] = 4 * L3x * L1 + 4 * L3 * L1x;
    Nu2[0] = 4 * L1y * L1 - L1y; Nu2[1] = 4 * L2y * L2 - L2y; Nu2[2] = 4 * L3y * L3 - L3y;
    Nu2[3] = 4 * L1y * L2 + 4 * L1 * L2y; Nu2[4] = 4 * L2y * L3 + 4 * L2 * L3y; Nu2[5] = 4 * L3y * L1 + 4 * L3 * L1y;
    if (Na) {
        Na[0] = 1 - 2 * L3; Na[1] = 1 - 2 * L1; Na[2] = 1 - 2 * L2;
        Na1[0] = -2 * L3x; Na1[1] = -2 * L1x; Na1[2] = -2 * L2x;
        Na2[0] = -2 * L3y; Na2[1] = -2 * L1y; Na2[2] = -2 * L2y;
    }
}

void gf_shell_host_const(const double *x, const double *prop, double *rec, double *prec, double *gp)
{
    for (int i = 0; i < SC_COUNT; i++) rec[i] = 0.0;
    for (int i = 0; i < SP_COUNT; i++) prec[i] = 0.0;
    const double *x1 = x, *x2 = x + 3, *x3 = x + 6;
    double d21[3], d31[3], nrm[3];
    vsub(x2, x1, d21);
    vsub(x3, x1, d31);
    vcross(d21, d31, nrm);
    double nn = vnorm(nrm);
    double A = 0.5 * nn;
    double e3[3] = {nrm[0] / nn, nrm[1] / nn, nrm[2] / nn};
    double eg[3] = {1.0, 0.0, 0.0};
    if (std::fabs(vdot(eg, e3)) >= 1.0 - 1e-4) { eg[0] = 0.0; eg[1] = 1.0; }
    double pr = vdot(eg, e3), e1[3], e2[3];
    for (int i = 0; i < 3; i++) e1[i] = eg[i] - pr * e3[i];
    double n1 = vnorm(e1);
    for (int i = 0; i < 3; i++) e1[i] = (1.0 / n1) * e1[i];
    vcross(e3, e1, e2);
    for (int i = 0; i < 3; i++) { rec[SC_T3 + i] = e1[i]; rec[SC_T3 + 3 + i] = e2[i]; rec[SC_T3 + 6 + i] = e3[i]; }
    double E = prop[0], nu = prop[1], rho = prop[2], t = prop[3];
    double mu = E / (2.0 * (1 + nu));
    rec[SC_MU] = mu;
    rec[SC_LAMBDA] = 2.0 * mu * nu / (1 - 2.0 * nu);
    rec[SC_THICK] = t;
    rec[SC_DRILL] = E * t * t * t;
    rec[SC_RHO] = rho;
    rec[SC_ALPHA1] = A / 3.0;
    double t23[3], t31[3], t12[3], t32[3], t13[3], t21[3];
    vsub(x2, x3, t23); vsub(x3, x1, t31); vsub(x1, x2, t12);
    vsub(x3, x2, t32); vsub(x1, x3, t13); vsub(x2, x1, t21);
    double dx[3] = {0.5 * vdot(t23, e2) / A, 0.5 * vdot(t31, e2) / A, 0.5 * vdot(t12, e2) / A};
    double dy[3] = {0.5 * vdot(t32, e1) / A, 0.5 * vdot(t13, e1) / A, 0.5 * vdot(t21, e1) / A};
    for (int g = 0; g < 3; g++) {
        const double *xp = x + 3 * (3 + g);
        double a2[3], a3[3], cr[3], L[3];
        vsub(x2, xp, a2); vsub(x3, xp, a3); vcross(a2, a3, cr); L[0] = 0.5 * vnorm(cr) / A;
        vsub(x3, xp, a2); vsub(x1, xp, a3); vcross(a2, a3, cr); L[1] = 0.5 * vnorm(cr) / A;
        vsub(x1, xp, a2); vsub(x2, xp, a3); vcross(a2, a3, cr); L[2] = 0.5 * vnorm(cr) / A;
        tri_shapes(L[0], L[1], L[2], dx, dy, rec + SC_NU + 6 * g, rec + SC_NU1 + 6 * g, rec + SC_NU2 + 6 * g,
                   rec + SC_NA + 3 * g, rec + SC_NA1 + 3 * g, rec + SC_NA2 + 3 * g);
    }
    // Cowper (1973) six-point rule, constants as src/Shell_1.cpp:2190-2233
    static const double cw[6][4] = {
        {0.816847572980459, 0.091576213509771, 0.091576213509771, 0.109951743655322},
        {0.091576213509771, 0.816847572980459, 0.091576213509771, 0.109951743655322},
        {0.091576213509771, 0.091576213509771, 0.816847572980459, 0.109951743655322},
        {0.108103018168070, 0.445948490915965, 0.445948490915965, 0.223381589678011},
        {0.445948490915965, 0.108103018168070, 0.445948490915965, 0.223381589678011},
        {0.445948490915965, 0.445948490915965, 0.108103018168070, 0.223381589678011}};
    for (int g = 0; g < 6; g++) {
        prec[SP_W4 + g] = A * cw[g][3];
        tri_shapes(cw[g][0], cw[g][1], cw[g][2], dx, dy, prec + SP_N4U + 6 * g, prec + SP_N4U1 + 6 * g,
                   prec + SP_N4U2 + 6 * g, nullptr, nullptr, nullptr);
    }
    for (int a = 0; a < 6; a++) {
        double s = 0.0;
        for (int g = 0; g < 6; g++) s += prec[SP_W4 + g] * prec[SP_N4U + 6 * g + a];
        rec[SC_GW + a] = s;
    }
    for (int g = 0; g < 3; g++) {
        double *st = gp + SG_PER_GP * g;
        for (int i = 0; i < SG_PER_GP; i++) st[i] = 0.0;
        st[0] = st[4] = st[8] = 1.0;
        st[15] = 1.0;  // z_x1_i = e1 (local)
        st[19] = 1.0;  // z_x2_i = e2 (local)
    }
}

// Scatter of one colour's element matrices and forces (written for all elements by
// shell_element_kernel): lane per (element, I, J) adding K_IJ, plus the follower
// pressure stiffness of u-node pair (I, J), into the tangent; lane per (element, I)
// adding -(f_I - self-weight + P_I) into r.  Elements of a colour share no node, and
// an element's lanes touch distinct entries, so no two lanes write the same place.
__global__ __launch_bounds__(256) void shell_scatter_kernel(int e0, int e1, size_t ld, const int *__restrict__ conn,
                                                            const double *__restrict__ cst, const int *__restrict__ dof,
                                                            gf_gmat gm, double *__restrict__ r,
                                                            const double *__restrict__ Ke, const double *__restrict__ fe,
                                                            const double *__restrict__ ppre, const double *__restrict__ lfp,
                                                            double gx, double gy, double gz)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int ne = e1 - e0;
    if (t < 81 * ne) {
        const int e = e0 + t / 81, ij = t - 81 * (t / 81);
        const int I = ij / 9, J = ij - 9 * (ij / 9);
        const double *k = Ke + (size_t)e * 729 + (3 * I) * 27 + 3 * J;
        double V9[9];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) V9[3 * i + j] = k[27 * i + j];
        if (ppre && I < 6 && J < 6) {
            const double *kp = ppre + ((size_t)e * 6 + I) * SPR + 3 + 3 * J;
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
                for (int j = 0; j < 3; j++) V9[3 * i + j] += kp[18 * i + j];
        }
        int na, ca, nb_, cb;
        dof_block(conn, ld, e, I, na, ca);
        dof_block(conn, ld, e, J, nb_, cb);
        int R9[9], C9[9];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) {
                R9[3 * i + j] = dof[6 * na + ca + i];
                C9[3 * i + j] = dof[6 * nb_ + cb + j];
            }
        gm_add_n<9>(gm, R9, C9, V9);
        return;
    }
    const int u = t - 81 * ne;
    if (u >= 9 * ne) return;
    const int e = e0 + u / 9, I = u - 9 * (u / 9);
    const double lf = lfp ? *lfp : 0.0;
    const double *fp = fe + (size_t)e * 27 + 3 * I;
    v3<double> f = mk3(fp[0], fp[1], fp[2]);
    if (I < 6 && lf != 0.0) {
        // self-weight, accumulated twice as src/Shell_1.cpp:1340-1375 does
        double mult = lf * cst[SC_RHO * ld + e] * cst[SC_THICK * ld + e];
        double gw = cst[(SC_GW + I) * ld + e];
        for (int rep = 0; rep < 2; rep++) {
            f.x -= gw * mult * gx;
            f.y -= gw * mult * gy;
            f.z -= gw * mult * gz;
        }
    }
    int node, c0;
    dof_block(conn, ld, e, I, node, c0);
    int R3[3];
    double V3[3] = {-f.x, -f.y, -f.z};
    if (ppre && I < 6) {
        const double *pa = ppre + ((size_t)e * 6 + I) * SPR;
#pragma unroll
        for (int i = 0; i < 3; i++) V3[i] -= pa[i];
    }
#pragma unroll
    for (int i = 0; i < 3; i++) R3[i] = dof[6 * node + c0 + i];
    vec_add_n<3>(r, R3, V3);
}

// ---- assembly by rows -------------------------------------------------------------
// Where the tangent's structure is at hand (multifrontal models of shells alone),
// the element matrices are gathered instead of scattered: one wavefront a DOF
// block (three rows: a node's displacements, or a mid-side node's rotations) adds
// its elements' rows in LDS, in the colour order of the scatter, and writes its
// three rows of the band and of the residual once.  One launch, no read of the
// band and no clear before it, in place of a clear and a scatter launch per
// colour that each read and write what they add to: 64 x 64 plate 30 + 75 us ->
// 60 us (bound by the band's writes, 24 or 48 bytes apart from the next), 13 x 13
// plate 5 + 36 -> 8 us (the chain list, matrix, LDS of one wavefront).  Beams share
// their DOFs with shells in no order of their own, and the block-tridiagonal form
// has no list of columns: both keep the scatter.

constexpr int SGMAX = 255;  // columns of a row (positions are bytes; 255: constrained)

// Position of every element matrix column in its row's list of columns, once per
// model: pos[(9 e + I) 27 + l] for column l of the rows of DOF block I.
__global__ __launch_bounds__(256) void shell_pos_kernel(int ns, size_t ld, const int *__restrict__ conn,
                                                        const int *__restrict__ dof, const int *__restrict__ ptr,
                                                        const int *__restrict__ cols, unsigned char *__restrict__ pos)
{
    const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (t >= 243 * (size_t)ns) return;
    const int e = (int)(t / 243), I = (int)(t - 243 * (size_t)e) / 27, l = (int)(t % 27);
    int n, c0, nj, cj;
    dof_block(conn, ld, e, I, n, c0);
    dof_block(conn, ld, e, l / 3, nj, cj);
    int row = -1;
    for (int i = 2; i >= 0; i--) row = dof[6 * n + c0 + i] >= 0 ? dof[6 * n + c0 + i] : row;
    const int c = dof[6 * nj + cj + l % 3];
    int p = 255;
    if (row >= 0 && c >= 0) {
        int lo = ptr[row], hi = ptr[row + 1];
        const int first = lo;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (cols[mid] < c) lo = mid + 1;
            else hi = mid;
        }
        p = lo - first;
    }
    pos[t] = (unsigned char)p;
}

// list[ptr[b] .. ptr[b + 1]): the (16 e + I) of DOF block b = 2 node + (rotations),
// e ascending; the elements are sorted by colour.  res: the residual norms to clear.
// Loads of SGU elements are in flight at once: a wavefront has no other work beside
// the six or so elements of its node (one at a time: 65 us at 64 x 64, 10.5 at 13 x 13).
constexpr int SGU = 4;

template <bool PRESS>
__global__ __launch_bounds__(256) void shell_gather_kernel(
    int nblk, size_t ld, const int *__restrict__ bptr, const int *__restrict__ list,
    const unsigned char *__restrict__ pos, const double *__restrict__ cst, const int *__restrict__ dof,
    const int *__restrict__ ptr, const int *__restrict__ cols, double *__restrict__ ab, int bld, int hb,
    double *__restrict__ r, const double *__restrict__ Ke, const double *__restrict__ fe,
    const double *__restrict__ ppre, const double *__restrict__ lfp, double gx, double gy, double gz, double *res)
{
    __shared__ double sm[4][3 * SGMAX];
    if (blockIdx.x == 0 && threadIdx.x < 8) res[threadIdx.x] = 0.0;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), b = blockIdx.x * 4 + wave;
    if (b >= nblk) return;  // (no barrier below: a wavefront works by itself)
    const int q0 = bptr[b], n = bptr[b + 1] - q0;
    if (n == 0) return;  // (no free DOF either: an element activates what it adds to)
    int R[3], row = -1;
#pragma unroll
    for (int i = 2; i >= 0; i--) {
        R[i] = dof[3 * b + i];
        row = R[i] >= 0 ? R[i] : row;
    }
    if (row < 0) return;
    double *acc = sm[wave];
    const int p0 = ptr[row], len = ptr[row + 1] - p0;
    const double lf = lfp ? *lfp : 0.0;
    for (int t = lane; t < 3 * len; t += 64) acc[t] = 0.0;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // the 81 entries of an element's three rows: lane t takes t and t + 64
    const int i0 = lane / 27, l0 = lane - 27 * i0, l1 = lane + 10;  // (t + 64 = 2 * 27 + (t + 10))
    const bool two = lane < 17, vec = lane < 3;
    const double gl = (lane == 0 ? gx : 0.0) + (lane == 1 ? gy : 0.0) + (lane == 2 ? gz : 0.0);
    double rv = 0.0;
    for (int q = 0; q < n; q += SGU) {
        int el[SGU], c0[SGU], c1[SGU];
        double k0[SGU], k1[SGU], f[SGU], a0[SGU], a1[SGU], af[SGU];
#pragma unroll
        for (int u = 0; u < SGU; u++) el[u] = list[q0 + min(q + u, n - 1)];
#pragma unroll
        for (int u = 0; u < SGU; u++) {
            const int e = el[u] >> 4, I = el[u] & 15;
            const double *K = Ke + (size_t)e * 729 + 81 * I;
            const unsigned char *ps = pos + (size_t)(9 * (size_t)e + I) * 27;
            k0[u] = K[lane];
            k1[u] = K[two ? lane + 64 : lane];
            f[u] = fe[(size_t)e * 27 + 3 * I + (vec ? lane : 0)];
            c0[u] = ps[l0];
            c1[u] = ps[two ? l1 : l0];
            if (PRESS) {
                // (rotations carry no pressure: their slots read block 5's and drop it)
                const double *kp = ppre + ((size_t)e * 6 + min(I, 5)) * SPR;
                a0[u] = kp[l0 < 18 ? 3 + 18 * i0 + l0 : 0];
                a1[u] = kp[two && l1 < 18 ? 3 + 36 + l1 : 0];
                af[u] = kp[vec ? lane : 0];
            }
        }
#pragma unroll
        for (int u = 0; u < SGU; u++) {
            if (q + u >= n) break;
            const int e = el[u] >> 4, I = el[u] & 15;
            if (PRESS && I < 6) {
                if (l0 < 18) k0[u] += a0[u];
                if (l1 < 18) k1[u] += a1[u];
            }
            if (I < 6 && lf != 0.0) {
                // self-weight, accumulated twice as src/Shell_1.cpp:1340-1375 does
                const double mult = lf * cst[SC_RHO * ld + e] * cst[SC_THICK * ld + e];
                const double gw = cst[(SC_GW + I) * ld + e];
                for (int rep = 0; rep < 2; rep++) f[u] -= gw * mult * gl;
            }
            // (different lanes hold different entries of the three rows)
            if (c0[u] != 255) acc[i0 * len + c0[u]] += k0[u];
            if (two && c1[u] != 255) acc[2 * len + c1[u]] += k1[u];
            rv -= f[u];
            if (PRESS && I < 6) rv -= af[u];
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        if (R[i] < 0) continue;
        double *base = ab + (size_t)R[i] * (size_t)bld + (size_t)hb;
        for (int k = lane; k < len; k += 64) base[cols[p0 + k]] = acc[i * len + k];
        if (lane == i) r[R[i]] = rv;
    }
}

// The tables of the assembly by rows; conn as uploaded (colour order).
int gf_shell_gather_setup(gf_model *m, const std::vector<int> &conn)
{
    const size_t ns = (size_t)m->ns, nb2 = 2 * (size_t)m->nn;
    int longest = 0;
    for (size_t i = 0; i + 1 < m->csr_ptr.size(); i++) longest = std::max(longest, m->csr_ptr[i + 1] - m->csr_ptr[i]);
    if (!m->fronts_on || m->nb > 0 || m->ns == 0 || longest > SGMAX) return GF_OK;
    std::vector<int> ptr(nb2 + 1, 0), list(9 * ns);
    auto block = [&](size_t e, int I) { return 2 * (size_t)conn[(I < 6 ? I : I - 3) * ns + e] + (I < 6 ? 0 : 1); };
    for (size_t e = 0; e < ns; e++)
        for (int I = 0; I < 9; I++) ptr[block(e, I) + 1]++;
    for (size_t b = 0; b < nb2; b++) ptr[b + 1] += ptr[b];
    std::vector<int> at(ptr.begin(), ptr.end() - 1);
    for (size_t e = 0; e < ns; e++)
        for (int I = 0; I < 9; I++) list[at[block(e, I)]++] = (int)(16 * e) + I;
    GF_TRY(gf_pool_alloc((void **)&m->d_sg_ptr, ptr.size() * 4));
    GF_TRY(gf_pool_alloc((void **)&m->d_sg_list, list.size() * 4));
    GF_TRY(gf_pool_alloc((void **)&m->d_sg_pos, 243 * ns));
    GF_HIP(hipMemcpyAsync(m->d_sg_ptr, ptr.data(), ptr.size() * 4, hipMemcpyHostToDevice, m->stream));
    GF_HIP(hipMemcpyAsync(m->d_sg_list, list.data(), list.size() * 4, hipMemcpyHostToDevice, m->stream));
    hipLaunchKernelGGL(shell_pos_kernel, dim3((unsigned)((243 * ns + 255) / 256)), dim3(256), 0, m->stream, m->ns, ns,
                       m->d_sconn, m->d_dof, m->d_csr_ptr, m->d_csr_col, m->d_sg_pos);
    GF_HIP(hipGetLastError());
    // the rows that no DOF has stay as they are from here on
    GF_TRY(gf_launch_fill(m->stream, m->d_r, (size_t)m->npad, 0.0));
    GF_HIP(hipStreamSynchronize(m->stream));  // (the uploads' host arrays end here)
    m->shell_gather = true;
    return GF_OK;
}

// ---- launchers --------------------------------------------------------------
int gf_shell_assemble(gf_model *m, const double *lfp, const double *tp)
{
    const size_t ld = (size_t)m->ns;
    int ncol = (int)m->shell_color_off.size() - 1;
    int launches = 0;
    if (m->ns == 0) return 0;
    // phase 1 of every element and the pressure terms
    // (a wavefront's time hardly depends on its points but for the copy: as few as leave one wavefront a SIMD)
    const int np = 3 * m->ns, per = np <= 16 * 1024 ? 16 : np <= 32 * 1024 ? 32 : 64;
    hipLaunchKernelGGL(per == 16 ? shell_record_kernel<16> : per == 32 ? shell_record_kernel<32> : shell_record_kernel<64>,
                       dim3((np + per - 1) / per), dim3(64), 0, m->stream, m->ns, ld, m->d_sconn, m->d_sconst, m->d_sgp,
                       m->d_disp, m->d_shell_rec);
    launches++;
    if (m->any_pressure) {
        hipLaunchKernelGGL(shell_pressure_record_kernel, dim3((m->ns + PE - 1) / PE), dim3(256), 0, m->stream,
                           m->ns, ld, m->d_sconn, m->d_sconst, m->d_spconst, m->d_disp, m->d_copy, m->d_copy0,
                           m->d_spload, m->d_spflag, m->d_lrec, m->d_tab_t, m->d_tab_v, tp, m->d_shell_prec);
        launches++;
    }
    // every element's K and f (phases 2-4 from the records), then their sum by rows or one
    // scatter launch per colour
    {
        const int pr = gf_probe_begin(m->stream, GF_KC_SHELL_ASSEMBLE);
        hipLaunchKernelGGL(shell_element_kernel<true>, dim3((m->ns + SEPB - 1) / SEPB), dim3(SWG), 0, m->stream, 0,
                           m->ns, ld, m->d_sconn, m->d_sconst, m->d_sgp, m->d_disp, m->d_shell_K, m->d_shell_f,
                           (const double *)m->d_shell_rec);
        gf_probe_end(m->stream, pr, m->ns);
        launches++;
    }
    const double *ppre = m->any_pressure ? m->d_shell_prec : nullptr;
    if (m->shell_gather) {
        hipLaunchKernelGGL(ppre ? shell_gather_kernel<true> : shell_gather_kernel<false>, dim3((2 * m->nn + 3) / 4),
                           dim3(256), 0, m->stream, 2 * m->nn, ld, (const int *)m->d_sg_ptr,
                           (const int *)m->d_sg_list, (const unsigned char *)m->d_sg_pos, m->d_sconst, m->d_dof,
                           (const int *)m->d_csr_ptr, (const int *)m->d_csr_col, m->d_band, m->band_ld, m->half_band,
                           m->d_r, (const double *)m->d_shell_K, (const double *)m->d_shell_f, ppre, lfp,
                           m->gravity[0], m->gravity[1], m->gravity[2], m->d_scal + GF_SCAL_RES);
        GF_HIP(hipGetLastError());
        return launches + 1;
    }
    for (int c = 0; c < ncol; c++) {
        int e0 = m->shell_color_off[c], e1 = m->shell_color_off[c + 1];
        if (e1 <= e0) continue;
        launches++;
        const int threads = 90 * (e1 - e0);
        hipLaunchKernelGGL(shell_scatter_kernel, dim3((threads + 255) / 256), dim3(256), 0, m->stream, e0, e1, ld,
                           m->d_sconn, m->d_sconst, m->d_dof, gf_model_gmat(m), m->d_r, (const double *)m->d_shell_K,
                           (const double *)m->d_shell_f, ppre, lfp, m->gravity[0], m->gravity[1], m->gravity[2]);
    }
    GF_HIP(hipGetLastError());
    return launches;
}

int gf_shell_commit(gf_model *m)
{
    if (m->ns == 0) return GF_OK;
    hipLaunchKernelGGL(shell_commit_kernel, dim3((3 * m->ns + 255) / 256), dim3(256), 0, m->stream, m->ns,
                       (size_t)m->ns, m->d_sconn, m->d_sconst, m->d_sgp, m->d_disp);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

int gf_shell_results(gf_model *m, double *d_out)
{
    if (m->ns == 0) return GF_OK;
    hipLaunchKernelGGL(shell_results_kernel, dim3((m->ns + 255) / 256), dim3(256), 0, m->stream, m->ns, (size_t)m->ns,
                       m->d_sconst, m->d_sgp, d_out);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

int gf_shell_eval_device(int count, const double *x, const double *prop, const double *d, const double *gp,
                         double *K_out, double *f_out)
{
    if (count <= 0) return GF_OK;
    size_t ld = (size_t)count;
    std::vector<int> conn(6 * ld);
    std::vector<double> cst(SC_COUNT * ld), gps(SG_COUNT * ld), disp(36 * ld);
    std::vector<double> rec(SC_COUNT), prec(SP_COUNT), g0(SG_COUNT);
    for (int e = 0; e < count; e++) {
        gf_shell_host_const(x + 18 * (size_t)e, prop + GF_SHELL_NPROP * (size_t)e, rec.data(), prec.data(), g0.data());
        for (int k = 0; k < SC_COUNT; k++) cst[k * ld + e] = rec[k];
        for (int k = 0; k < SG_COUNT; k++) gps[k * ld + e] = gp[(size_t)e * SG_COUNT + k];
        for (int a = 0; a < 6; a++) conn[a * ld + e] = 6 * e + a;
        for (int k = 0; k < 36; k++) disp[36 * (size_t)e + k] = d[36 * (size_t)e + k];
    }
    int *d_conn = nullptr;
    double *d_cst = nullptr, *d_gps = nullptr, *d_disp = nullptr, *d_K = nullptr, *d_f = nullptr;
    hipStream_t s;
    GF_HIP(hipStreamCreate(&s));
    GF_HIP(hipMalloc(&d_conn, sizeof(int) * conn.size()));
    GF_HIP(hipMalloc(&d_cst, sizeof(double) * cst.size()));
    GF_HIP(hipMalloc(&d_gps, sizeof(double) * gps.size()));
    GF_HIP(hipMalloc(&d_disp, sizeof(double) * disp.size()));
    GF_HIP(hipMalloc(&d_K, sizeof(double) * 729 * ld));
    GF_HIP(hipMalloc(&d_f, sizeof(double) * 27 * ld));
    GF_HIP(hipMemcpyAsync(d_conn, conn.data(), sizeof(int) * conn.size(), hipMemcpyHostToDevice, s));
    GF_HIP(hipMemcpyAsync(d_cst, cst.data(), sizeof(double) * cst.size(), hipMemcpyHostToDevice, s));
    GF_HIP(hipMemcpyAsync(d_gps, gps.data(), sizeof(double) * gps.size(), hipMemcpyHostToDevice, s));
    GF_HIP(hipMemcpyAsync(d_disp, disp.data(), sizeof(double) * disp.size(), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(shell_element_kernel<false>, dim3((count + SEPB - 1) / SEPB), dim3(SWG), 0, s, 0, count, ld,
                       d_conn, d_cst, d_gps, d_disp, d_K, d_f, (const double *)nullptr);
    GF_HIP(hipGetLastError());
    GF_HIP(hipMemcpyAsync(K_out, d_K, sizeof(double) * 729 * ld, hipMemcpyDeviceToHost, s));
    GF_HIP(hipMemcpyAsync(f_out, d_f, sizeof(double) * 27 * ld, hipMemcpyDeviceToHost, s));
    GF_HIP(hipStreamSynchronize(s));
    (void)hipFree(d_conn); (void)hipFree(d_cst); (void)hipFree(d_gps);
    (void)hipFree(d_disp); (void)hipFree(d_K); (void)hipFree(d_f);
    (void)hipStreamDestroy(s);
    return GF_OK;
}
