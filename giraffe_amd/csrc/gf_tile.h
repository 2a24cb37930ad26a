// 64 x 64 tile machinery shared by the wide-band and the multifrontal
// factorisations on gfx950: FP64 / FP32 MFMA 16x16x4 products of 64 x 64
// tiles staged through LDS, the in-register 16 x 16 Gauss-Jordan leaf and the
// 64 x 64 block inverse with pivot perturbation, row-major tile transfers.
// Device code only; every definition has internal linkage.
#pragma once
#include "gf_dpp.h"

namespace {

constexpr int NB = 64;   // block size
constexpr int KT = 32;   // k-chunk of the staged MFMA products
// LDS strides (elements) chosen for the MFMA operand patterns in FP64 (64
// banks of 4 bytes, 32 lanes of 8-byte reads per cycle): an A operand reads
// rows i = 0..15 at column offsets c = 0..1, a B operand rows c at columns
// j = 0..15.  Row stride 66 (2 mod 32) and 34 spread A reads over all banks,
// 80 (16 mod 32) does the same for B reads, 18 for the saved 16 x 16 blocks.
constexpr int LDT = NB + 2, LDQ = NB + 16;
constexpr int SA_LD = KT + 2, SB_LD = NB + 16, TMP_LD = 18;

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// 16x16x4 MFMA.  Operands: A(i, k) in lane i + 16 k, B(k, j) in lane j + 16 k.
// Result item v of lane l: row 4 v + l / 16 (f64) or 4 (l / 16) + v (f32),
// column l % 16 (checked on gfx950).
template <typename T> struct mfma;
template <> struct mfma<double> {
    typedef v4d acc_t;
    static __device__ __forceinline__ acc_t run(double a, double b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int v) { return 4 * v + (lane >> 4); }
};
template <> struct mfma<float> {
    typedef v4f acc_t;
    static __device__ __forceinline__ acc_t run(float a, float b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// Per-wave part of a 64 x 64 result: rows wr + 16a + row(lane, v), columns wc + 16b + lane % 16.
template <typename T> struct Acc {
    typename mfma<T>::acc_t a[2][2];
    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int y = 0; y < 2; y++) a[x][y] = typename mfma<T>::acc_t{};
    }
};
__device__ __forceinline__ int acc_row(int wave) { return (wave >> 1) * 32; }
__device__ __forceinline__ int acc_col(int wave) { return (wave & 1) * 32; }
template <typename T, typename F> __device__ __forceinline__ void acc_each(F f)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                f(x, y, v, acc_row(wave) + 16 * x + mfma<T>::row(lane, v), acc_col(wave) + 16 * y + (lane & 15));
}

// acc += P Q (64 x 64 x 64, 256 threads).  P and Q are read through loaders,
// every load of both K-chunks issued before the first LDS store (one memory
// round trip per product), then per chunk of KT the four waves run their
// 2 x 2 MFMA tiles from LDS.
template <typename T, typename LP, typename LQ>
__device__ __forceinline__ void tile_mm(Acc<T> &acc, T *sa, T *sb, LP loadP, LQ loadQ)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = acc_row(wave), wc = acc_col(wave);
    constexpr int PER = NB * KT / 256, NCH = NB / KT;
    T pv[NCH][PER], qv[NCH][PER];
#pragma unroll
    for (int c = 0; c < NCH; c++)
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int t = tid + 256 * r;
            pv[c][r] = loadP(t / KT, c * KT + t % KT);
            qv[c][r] = loadQ(c * KT + t / NB, t % NB);
        }
#pragma unroll
    for (int c = 0; c < NCH; c++) {
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int t = tid + 256 * r;
            sa[(t / KT) * SA_LD + t % KT] = pv[c][r];
            sb[(t / NB) * SB_LD + t % NB] = qv[c][r];
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < KT; kk += 4) {
            T av[2], bv[2];
#pragma unroll
            for (int x = 0; x < 2; x++) av[x] = sa[(wr + 16 * x + (lane & 15)) * SA_LD + kk + (lane >> 4)];
#pragma unroll
            for (int y = 0; y < 2; y++) bv[y] = sb[(kk + (lane >> 4)) * SB_LD + wc + 16 * y + (lane & 15)];
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++) acc.a[x][y] = mfma<T>::run(av[x], bv[y], acc.a[x][y]);
        }
        __syncthreads();
    }
}

// acc += P Q with both operands in LDS (64 x 64, row strides lp and lq); no
// barrier inside.
template <typename T> __device__ __forceinline__ void lds_mm(Acc<T> &acc, const T *P, int lp, const T *Q, int lq)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = acc_row(wave), wc = acc_col(wave);
#pragma unroll 4
    for (int k = 0; k < NB; k += 4) {
        T av[2], bv[2];
#pragma unroll
        for (int x = 0; x < 2; x++) av[x] = P[(wr + 16 * x + (lane & 15)) * lp + k + (lane >> 4)];
#pragma unroll
        for (int y = 0; y < 2; y++) bv[y] = Q[(k + (lane >> 4)) * lq + wc + 16 * y + (lane & 15)];
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int y = 0; y < 2; y++) acc.a[x][y] = mfma<T>::run(av[x], bv[y], acc.a[x][y]);
    }
}

template <typename T> __device__ __forceinline__ T rcp_of(T p);
template <> __device__ __forceinline__ double rcp_of<double>(double p) { return pivot_rcp(p); }
template <> __device__ __forceinline__ float rcp_of<float>(float p) { return pivot_rcp(p); }

template <typename T> struct PivotGuard {
    T rel, huge;
    __device__ __forceinline__ PivotGuard() : rel(sizeof(T) == 8 ? T(1e-13) : T(1e-6)), huge(sizeof(T) == 8 ? T(1e300) : T(1e37)) {}
};

// Cross-lane moves of the 16 x 16 inverse.  A wavefront is four DPP rows of
// 16 lanes.  row_newbcast:K (DPP) gives every lane the value of lane K of its
// own row; rowcast<R> gives every lane the value at the same position of row R
// (v_permlane16_swap: each pair of rows swaps its odd row with the even one,
// so one of the two results holds the pair's even row twice, the other its
// odd row; v_permlane32_swap does the same for the two halves).  Register
// moves only: no LDS round trip on the pivot chain.
template <int CTRL> __device__ __forceinline__ double dpp_mov(double v)
{
    // one 64-bit move where the control allows it (row_newbcast), else two 32-bit ones
    return __builtin_amdgcn_update_dpp(0.0, v, CTRL, 0xF, 0xF, false);
}
template <int CTRL> __device__ __forceinline__ float dpp_mov(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int R> __device__ __forceinline__ unsigned rowcast_u32(unsigned v)
{
    const auto h = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    const unsigned t = (R & 1) ? h[1] : h[0];
    const auto w = __builtin_amdgcn_permlane32_swap(t, t, false, false);
    return (R & 2) ? w[1] : w[0];
}
template <int R> __device__ __forceinline__ double rowcast(double v)
{
    const unsigned lo = rowcast_u32<R>((unsigned)__double2loint(v)), hi = rowcast_u32<R>((unsigned)__double2hiint(v));
    return __hiloint2double((int)hi, (int)lo);
}
template <int R> __device__ __forceinline__ float rowcast(float v)
{
    return __uint_as_float(rowcast_u32<R>(__float_as_uint(v)));
}
// Pivot K of the in-place Gauss-Jordan inverse of a 16 x 16 block held by one
// wavefront: lane 16 q + i holds row i, columns 4 q .. 4 q + 3 (a[0..3]).  Rows
// are kept scaled: the true row i is s_i times the stored one, s_i = 1 until
// row i has been the pivot row and the pivot's reciprocal after, so the pivot
// row itself is left as it is (its diagonal entry set to 1) and every other
// row takes one FMA per entry, a(i, j) -= (a(i, K) / p) a(K, j); the scales
// are applied once at the end.  Row K is unscaled when it is the pivot row, so
// its entries and the pivot are true values.  The pivot reaches every lane by
// two register moves (column K of the lane's row from row block K / 4, then
// lane K of each DPP row): no readlane, no LDS access on the pivot chain.  A
// pivot below a threshold eps_K (|p| / eps_K < 1; ieps[K] = 1 / eps_K in LDS,
// read per pivot off the dependent chain) takes the reciprocal of +-eps_K, a
// non-finite one the reciprocal 1.
template <typename T, int K>
__device__ __forceinline__ void inv16_pivot(T (&a)[4], T &sc, int i, int q, const T *ieps, T huge, bool &bad,
                                            bool &pert)
{
    constexpr int KQ = K >> 2, KE = K & 3;
    const T ie = ieps[K];
    T rk[4];
#pragma unroll
    for (int e = 0; e < 4; e++) rk[e] = dpp_mov<0x150 + K>(a[e]);  // row K, this lane's columns
    const T f = rowcast<KQ>(a[KE]);                                  // row i, column K
    const T p = dpp_mov<0x150 + K>(f);                               // the pivot
    const T r0 = rcp_of<T>(p);  // replaced below when p is tiny or not finite
    const T ap = fabs(p);
    const bool nonfinite = !(ap < huge);
    const bool small = !nonfinite && ap * ie < T(1);
    bad |= nonfinite;
    pert |= small;
    // rcp(-x) = -rcp(x) exactly, rcp(1) = 1
    const T ip = nonfinite ? T(1) : small ? (p >= T(0) ? ie : -ie) : r0;
    const bool isk = i == K;
    const T h = isk ? T(0) : f * ip;  // row K keeps its entries
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const T upd = fma(-h, rk[e], a[e]);
        if (e == KE)
            a[e] = q == KQ ? (isk ? T(1) : -h) : upd;  // column K: -a(i, K) / p; s_K / s_K on the diagonal
        else
            a[e] = upd;
    }
    sc = isk ? ip : sc;
    if constexpr (K + 1 < 16) inv16_pivot<T, K + 1>(a, sc, i, q, ieps, huge, bad, pert);
}

// FP64: the same inverse with every lane holding the whole of its row (the four
// DPP rows hold copies), so that a row's multiplier is its own lane's and the
// pivot row comes inside the multiply-add: about 27 instructions a pivot against
// 70, with the next pivot's reciprocal formed among them.  Pivots are taken as
// they are; sc (their reciprocals, row by row) tells at the end whether one was
// below its threshold or not finite.
template <int K>
__device__ __forceinline__ void inv16_row_pivot(double (&a)[16], double &sc, double ip, double g)
{
    const bool isk = __builtin_amdgcn_inverse_ballot_w64(lanes_at<K>());
    const double h = isk ? 0.0 : g;
    sc = isk ? ip : sc;
    a[K] = __hiloint2double(isk ? 0x3ff00000 : __double2hiint(h), __double2loint(h));  // row K: 1, else -a(i, K) / p
    double t[15];
#pragma unroll
    for (int j = 0; j < 15; j++) t[j] = a[(K + 1 + j) & 15];
    if constexpr (K + 1 < 16) nb_pivot15<K>(t, h, ip, g);
    else nb_self<K, 15>(t, h);
#pragma unroll
    for (int j = 0; j < 15; j++) a[(K + 1 + j) & 15] = t[j];
    if constexpr (K + 1 < 16) inv16_row_pivot<K + 1>(a, sc, ip, g);
}
__device__ __forceinline__ bool inv16_rows(double *b, const double *ieps, double huge)
{
    const int lane = threadIdx.x & 63, i = lane & 15;
    double a[16], sc = 1.0;
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        const double2 w = *reinterpret_cast<const double2 *>(b + i * LDT + e);
        a[e] = w.x;
        a[e + 1] = w.y;
    }
    const double ie = ieps[i], p0 = nb_get<0>(a[0]), ip0 = pivot_rcp(p0);
    inv16_row_pivot<0>(a, sc, ip0, -(a[0] * ip0));
    // |p| >= eps and |p| < huge for every pivot p = 1 / sc
    const double as = fabs(sc);
    if (__any(!(as <= ie && as * huge > 1.0))) return false;
    if (lane < 16) {
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
            double2 w;
            w.x = sc * a[e];
            w.y = sc * a[e + 1];
            *reinterpret_cast<double2 *>(b + i * LDT + e) = w;
        }
    }
    return true;
}
__device__ __forceinline__ bool inv16_rows(float *, const float *, float) { return false; }

// One wavefront: in-place Gauss-Jordan inverse (no interchanges) of the 16 x 16
// block at b (stride LDT); the 16 pivots run in registers with DPP and
// permlane moves, no barrier and no LDS access on the pivot chain.  ieps: the
// reciprocals of the sixteen pivot thresholds (LDS).  FP64 blocks come here only
// where inv16_rows met a pivot that has to be replaced.
template <typename T>
__device__ __forceinline__ void inv16(T *b, const T *ieps, T huge, bool &bad, bool &pert)
{
    if (__builtin_expect(inv16_rows(b, ieps, huge), 1)) return;
    const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    T a[4], sc = T(1);
#pragma unroll
    for (int e = 0; e < 4; e++) a[e] = b[i * LDT + 4 * q + e];
    inv16_pivot<T, 0>(a, sc, i, q, ieps, huge, bad, pert);
#pragma unroll
    for (int e = 0; e < 4; e++) b[i * LDT + 4 * q + e] = sc * a[e];
}

// acc = P Q for 16 x 16 blocks in LDS (strides lp, lq); one wavefront.
template <typename T>
__device__ __forceinline__ typename mfma<T>::acc_t mm16(const T *P, int lp, const T *Q, int lq)
{
    const int lane = threadIdx.x & 63;
    typename mfma<T>::acc_t acc[2] = {};  // two chains of two
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4)
        acc[k0 >> 2 & 1] = mfma<T>::run(P[(lane & 15) * lp + k0 + (lane >> 4)], Q[(k0 + (lane >> 4)) * lq + (lane & 15)],
                                        acc[k0 >> 2 & 1]);
    return acc[0] + acc[1];
}

// Scratch of inverse64: two sets of three saved 16 x 16 column blocks, and one
// more block.
constexpr int INV_TMP = (2 * 3 + 1) * 16 * TMP_LD;

// LDS writes of a wavefront before its own later reads.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// In-place inverse of the 64 x 64 matrix M ([64][LDT], 16-byte aligned) by 256 threads: block
// Gauss-Jordan over 16 x 16 blocks.  Step kb, with the pivot block P already
// inverted in place and the column blocks C_i = M(i, kb) (i != kb) saved: row
// blocks R_j = P^-1 M(kb, j), M(i, j) -= C_i R_j, M(i, kb) = -C_i P^-1 (MFMA
// 16x16x4).  The chain is the next pivot block: wave 0 forms its R itself,
// updates that block and inverts it (inv16) while waves 1-3 each take a column
// (its R, then its blocks; wave 3 the rest of the next pivot's column, which it
// saves for the next step, and the pivot column), so no wave needs another's
// result within a step: one barrier per step.  M(kb, kb + 1) itself keeps its
// old value (the next step overwrites it from the saved blocks).  No
// interchanges: a pivot smaller than 1e-13
// (FP32: 1e-6) of its row's original diagonal entry (of the block's largest
// entry where that is zero) -- a threshold that does not depend on how rows and
// columns are scaled -- is replaced by that size with its sign (bit 2 of
// *flag); a non-finite pivot or an all-zero block sets bit 1.  (An FP32 factor
// with perturbed pivots is still refined against the FP64 tangent, which
// decides whether it was good enough.)  tmp: INV_TMP entries; aux: 4 + 64
// entries.  Runs on the first four wavefronts; those of a larger workgroup only
// take part in the barriers.  nk: only the first nk row and column blocks are
// inverted (the rest is identity, decoupled).
template <typename T> __device__ __forceinline__ void inverse64(T *M, T *tmp, T *aux, int *flag, int nk = 4)
{
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool act = tid < 256;
    const PivotGuard<T> pg;
    auto wave_max = [&](T v) {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) v = fmax(v, __shfl_xor(v, o));
        return v;
    };
    // wave 0: pivot thresholds of block kb (their reciprocals replace the
    // original diagonal in aux; written and read by this wave only), then the
    // inverse of the block in place
    bool bad = false, pert = false;
    auto pivot_block = [&](int kb) {
        T *ie = aux + 4 + 16 * kb;
        T dk = ie[lane & 15];
        if (__any(!(dk > T(0)))) {
            // the largest entry of the original block: while it is still whole, then
            // from the scan beside the first inverse
            T mx = T(0);
            if (kb == 0) {
#pragma unroll 1
                for (int t = lane; t < NB * NB; t += 64) mx = fmax(mx, fabs(M[(t >> 6) * LDT + (t & 63)]));
                mx = wave_max(mx);
            } else {
                for (int k = 0; k < 4; k++) mx = fmax(mx, aux[k]);
            }
            dk = dk > T(0) ? dk : mx;
        }
        if (lane < 16) ie[lane] = rcp_of<T>(pg.rel * dk);
        wave_lds_fence();
        inv16<T>(M + 16 * kb * LDT + 16 * kb, ie, pg.huge, bad, pert);
    };
    constexpr int CS = 16 * TMP_LD, CB = 3 * CS;  // one saved block, one set
    auto block = [&](int i, int j) { return M + 16 * i * LDT + 16 * j; };
    auto put = [&](T *dst, int ld, const typename mfma<T>::acc_t &v) {
#pragma unroll
        for (int e = 0; e < 4; e++) dst[mfma<T>::row(lane, e) * ld + (lane & 15)] = v[e];
    };
    // M(i, j) -= C R (saved copy to sv when given)
    auto update = [&](int i, int j, const T *Ci, const T *R, int ldr, T *sv) {
        T *Mij = block(i, j);
        const typename mfma<T>::acc_t acc = mm16<T>(Ci, TMP_LD, R, ldr);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int r = mfma<T>::row(lane, e), c = lane & 15;
            const T x = Mij[r * LDT + c] - acc[e];
            Mij[r * LDT + c] = x;
            if (sv) sv[r * TMP_LD + c] = x;
        }
    };
    // step 0's pivot block and column blocks; beside the pivot block's inverse the
    // largest magnitudes of the row blocks (wave 0: of its own block), which tell
    // an all-zero block and one with infinite entries
    if (wave == 0) {
        aux[4 + lane] = fabs(M[lane * LDT + lane]);
        T mx = T(0);
#pragma unroll
        for (int t = 0; t < 4; t++) mx = fmax(mx, fabs(M[(lane & 15) * LDT + 4 * (lane >> 4) + t]));
        mx = wave_max(mx);
        if (lane == 0) aux[0] = mx;
        wave_lds_fence();
        pivot_block(0);
    } else if (act) {
        const T *src = block(wave, 0);
#pragma unroll 2
        for (int t = lane; t < 256; t += 64) tmp[(wave - 1) * CS + (t >> 4) * TMP_LD + (t & 15)] = src[(t >> 4) * LDT + (t & 15)];
        T mx = T(0);
#pragma unroll 2
        for (int t = lane; t < 16 * NB; t += 64) mx = fmax(mx, fabs(src[(t >> 6) * LDT + (t & 63)]));
        // row block 0 right of the pivot block
#pragma unroll 2
        for (int t = lane; t < 256; t += 64) mx = fmax(mx, fabs(M[(t >> 4) * LDT + 16 * wave + (t & 15)]));
        mx = wave_max(mx);
        if (lane == 0) aux[wave] = mx;
    }
    __syncthreads();
#pragma unroll 1
    for (int kb = 0; kb < nk; kb++) {
        const T *cur = tmp + (kb & 1) * CB, *P = block(kb, kb);
        T *nxt = tmp + ((kb + 1) & 1) * CB;
        const int nb = kb + 1;
        auto saved = [&](int i) { return cur + (i < kb ? i : i - 1) * CS; };  // C_i
        auto column = [&](int j) {
            T *R = block(kb, j);
            put(R, LDT, mm16<T>(P, LDT, R, LDT));
            wave_lds_fence();
#pragma unroll 1
            for (int i = 0; i < nk; i++)
                if (i != kb) update(i, j, saved(i), R, LDT, nullptr);
        };
        auto pivot_column = [&] {
#pragma unroll 1
            for (int i = 0; i < nk; i++)
                if (i != kb) {
                    typename mfma<T>::acc_t acc = mm16<T>(saved(i), TMP_LD, P, LDT);
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[e] = -acc[e];
                    put(block(i, kb), LDT, acc);
                }
        };
        if (nb == nk) {
            if (wave < nb - 1) column(wave);
            else if (wave == nb - 1) pivot_column();
        } else if (wave == 0) {
            T *R = nxt + kb * CS;
            put(R, TMP_LD, mm16<T>(P, LDT, block(kb, nb), LDT));
            wave_lds_fence();
            update(nb, nb, saved(nb), R, TMP_LD, nullptr);
            wave_lds_fence();
            pivot_block(nb);
        } else if (wave < 3) {
            // the columns other than kb and nb, in cyclic order
            const int j = (kb + 1 + wave) % nk;
            if (1 + wave < nk) column(j);
        } else if (act) {
            T *R = tmp + 2 * CB;
            put(R, TMP_LD, mm16<T>(P, LDT, block(kb, nb), LDT));
            wave_lds_fence();
            for (int i = 0; i < nk; i++)
                if (i != kb && i != nb) update(i, nb, saved(i), R, TMP_LD, nxt + (i < nb ? i : i - 1) * CS);
            pivot_column();
        }
        __syncthreads();
    }
    if (tid == 0) {
        const T mx = fmax(fmax(aux[0], aux[1]), fmax(aux[2], aux[3]));
        bad |= !(mx > T(0)) || !(mx < pg.huge);
        const int bits = (bad ? 1 : 0) | (pert ? 2 : 0);
        if (bits) atomicOr(flag, bits);
    }
}

// Row-major 64 x 64 tile through registers: thread t holds elements t + 256 r
// (each row of 64 read or written by one 64-lane wave, coalesced).
template <typename T, typename F> __device__ __forceinline__ void tile_load(T (&v)[16], F load)
{
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int t = threadIdx.x + 256 * r;
        v[r] = load(t >> 6, t & 63);
    }
}
template <typename T> __device__ __forceinline__ void tile_put(T *dst, int ld, const T (&v)[16])
{
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int t = threadIdx.x + 256 * r;
        dst[(t >> 6) * ld + (t & 63)] = v[r];
    }
}

// LDS of the step kernel: P holds A operands (E_p, then L(i, p); the diagonal
// block D for the inverse), Q B operands (A'(p, j), then U(p, j)); the
// inverse's scratch reuses Q.  75 KB in FP64, so two workgroups share a CU and
// a launch's tiles are all resident at once.
template <typename T> struct alignas(16) StepSmem {
    T P[NB * LDT];
    union {
        T Q[NB * LDQ];
        T tmp[INV_TMP];
    };
    T aux[4 + NB];
};

// Wavefront sum.
template <typename V> __device__ __forceinline__ V sum64(V s)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
    return s;
}

}  // namespace
