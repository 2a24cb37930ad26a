// Multifrontal tangent solve on gfx950: the nested-dissection counterpart of
// sparsesystem -> MKL PARDISO (src/SparseMatrix.cpp:74-166; PARDISO orders by
// nested dissection, iparm[1] = 3, and factors supernode by supernode).
//
// Fronts (plan: gf_nd.cpp) are dense row-major matrices [mp][mp] over a
// supernode's own DOFs (kp = 64 kb rows, the last kp - k of them identity
// padding) followed by its update DOFs.  Per level of the supernode tree:
//
//   assemble  F(i, j) = sum over children c of U_c(a_c(i), a_c(j)) (the child's
//             Schur complement rows that map to i and j, in child order), plus
//             the tangent entry K(i, j) read from the band storage when row i or
//             column j is one of the front's own DOFs (the front of the first of
//             the two in elimination order holds it).  Every entry is written by
//             one thread, in a fixed order: no atomics, bit-reproducible.
//             The workgroup of each front's first diagonal block also inverts it
//             (E_0).  Only the tiles of the own rows and columns are written: step 0
//             forms the others itself.
//   factor    the block LU of the band solver on each front, restricted to its
//             kb own block columns, over all fronts of the level at once:
//             launch p = 0 .. kb - 1 updates A(i, j) -= A(i, p) (E_p A'(p, j))
//             for i, j > p (the update blocks included: after the last own step
//             they hold the Schur complement the parent assembles), inverts the
//             next diagonal block (E_{p+1}) and converts row p - 1 to U.  The
//             last own block row stays A'(kb - 1, .) = D U(kb - 1, .): the
//             backward solve applies E_{kb-1} to it, which saves a launch per
//             level.  Pivots: as the band solver (perturbation below 1e-13 of the
//             block's diagonal, flag bit 2; non-finite, bit 1).
//
// Solve, with A = L U (L(p, p) = D_p = E_p^-1, U block unit upper):
//   forward   per level: a front gathers its own right-hand side and its
//             children's update vectors, solves with its own L blocks (one
//             workgroup, rows kept in LDS), then every update row tile forms
//             its update vector  c = sum_children c_child - L(t, own) y.
//   backward  per level from the root: x_own = y - U(own, update) x_update
//             (row tiles in parallel, x_update read from the ancestors' rows of
//             x), then the own-block back substitution and the scatter of x; in
//             one launch where the plan finds the rows few.
#include "gf_tile.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int KMAX = GF_FRONT_KMAX;  // largest own block (rows in LDS of the solve); the plan splits larger supernodes

struct FrontTab {
    const gf_front_dev *fr;
    const int *rows, *child, *inv, *items;
    const long long *child_inv;
    const int *orig, *asm_orig;
};

// Update vector entry of front position i gathered from the children.
__device__ __forceinline__ double child_sum(const FrontTab &t, const gf_front_dev &F, int i, const double *Vb)
{
    double w = 0.0;
    for (int c = F.ch0; c < F.ch1; c++) {
        const int a = t.inv[t.child_inv[c] + i];
        if (a >= 0) {
            const gf_front_dev C = t.fr[t.child[c]];
            w += Vb[C.V + NB * C.kb + a];
        }
    }
    return w;
}

// LDS of the assembly kernel: the first diagonal block of a front and the
// inverse's scratch.
template <typename T> struct alignas(16) AsmSmem {
    T P[NB * LDT];
    T tmp[INV_TMP];
    T aux[4 + NB];
};

// 512 threads (eight wavefronts) per tile: the inverse's 48 KB of LDS then still
// leaves 24 wavefronts per CU to overlap the gathers.
constexpr int ASM_T = 512, ASM_R = NB * NB / ASM_T;

template <typename T>
__global__ __launch_bounds__(ASM_T, 6) void front_assemble_kernel(FrontTab t, int first, const double *ab, int ld, int hb,
                                                               const double *D, T *Fb, T *Eb, int *flag,
                                                               const double *rhs, double *Vb)
{
    __shared__ AsmSmem<T> sm;
    const int *it = t.items + 4 * (size_t)(first + blockIdx.x);
    const int f = it[0];
    const gf_front_dev F = t.fr[f];
    const int r0 = NB * it[1], c0 = NB * it[2];
    const int tid = threadIdx.x, j = tid & 63, i0 = tid >> 6;
    constexpr int RS = ASM_T / NB;  // row stride of a thread's rows
    const int cj = c0 + j;
    const int *rows = t.rows + F.rows;
    // Few tiles (the upper levels, small plates) are a chain of dependent loads:
    // item, front, child's map, child's entries, and entry list, band.  The two
    // chains run together: a thread's first PQ list entries are read to the band's
    // value while the children's maps arrive (a launch of a few tiles 21.5 -> 19.7
    // us, level 2 of the 64 x 64 plate 29.7 -> 23.6).
    constexpr int PQ = 2;
    const int *ol = t.orig + 3 * (size_t)t.asm_orig[2 * (size_t)(first + blockIdx.x)];
    const int no = t.asm_orig[2 * (size_t)(first + blockIdx.x) + 1];
    auto entry = [&](int oi, int oc) {
        const double a = ab[(size_t)oi * (size_t)ld + (size_t)(oc + hb)];
        return D ? D[oi] * a * D[oc] : a;
    };
    int pos[PQ], oi[PQ], oc[PQ];
#pragma unroll
    for (int k = 0; k < PQ; k++) {
        const int q = min(tid + ASM_T * k, max(no - 1, 0));
        pos[k] = no ? ol[3 * q] : 0;
        oi[k] = no ? ol[3 * q + 1] : 0;
        oc[k] = no ? ol[3 * q + 2] : 0;
    }
    T v[ASM_R];
#pragma unroll
    for (int r = 0; r < ASM_R; r++) v[r] = T(0);
    double pre[PQ];
    for (int c = F.ch0; c < F.ch1 || c == F.ch0; c++) {
        const bool have = c < F.ch1;
        const gf_front_dev C = t.fr[have ? t.child[c] : f];
        const int *im = t.inv + (have ? t.child_inv[c] : 0);
        int b = -1, a[ASM_R];
        if (have) {
            b = im[cj];
#pragma unroll
            for (int r = 0; r < ASM_R; r++) a[r] = im[r0 + i0 + RS * r];
        }
        if (c == F.ch0)
#pragma unroll
            for (int k = 0; k < PQ; k++) pre[k] = no ? entry(oi[k], oc[k]) : 0.0;
        if (b < 0) continue;
        const T *U = Fb + C.F + (size_t)(NB * C.kb) * C.mp + NB * C.kb + b;
#pragma unroll
        for (int r = 0; r < ASM_R; r++)
            if (a[r] >= 0) v[r] += U[(size_t)a[r] * C.mp];
    }
    // the children's sums into the tile in LDS, the tile's tangent entries (its
    // precomputed list) added there, then the tile written out row by row
#pragma unroll
    for (int r = 0; r < ASM_R; r++) {
        const int ri = r0 + i0 + RS * r;
        if (ri == cj && ri >= F.k && ri < NB * F.kb) v[r] = T(1);  // padding of the own block: identity
        sm.P[(i0 + RS * r) * LDT + j] = v[r];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PQ; k++)
        if (tid + ASM_T * k < no) sm.P[(pos[k] >> 6) * LDT + (pos[k] & 63)] += (T)pre[k];
    for (int q = tid + ASM_T * PQ; q < no; q += ASM_T) {
        const int ps = ol[3 * q];
        sm.P[(ps >> 6) * LDT + (ps & 63)] += (T)entry(ol[3 * q + 1], ol[3 * q + 2]);
    }
    __syncthreads();
    T *out = Fb + F.F + cj;
#pragma unroll
    for (int r = 0; r < ASM_R; r++) {
        v[r] = sm.P[(i0 + RS * r) * LDT + j];
        out[(size_t)(r0 + i0 + RS * r) * F.mp] = v[r];
    }
    if (rhs && it[2] == 0 && tid < NB) {
        // the right-hand side rides along the factorisation: the front vector starts
        // as the own rows of b plus the children's update vectors
        const int i = r0 + tid, o = rows[i];
        Vb[F.V + i] = (i < F.k && o >= 0 ? rhs[o] : 0.0) + child_sum(t, F, i, Vb);
    }
    if (it[3] == 0) return;
    // the front's first diagonal block (already in LDS): E_0
    inverse64<T>(sm.P, sm.tmp, sm.aux, flag, min(NB, (F.k + 15) & ~15) >> 4);
    T *E = Eb + F.E;
    for (int q = threadIdx.x; q < NB * NB; q += ASM_T) E[q] = sm.P[(q / NB) * LDT + q % NB];
}

// LDS of the step kernel, 52.6 KB in FP64 so that three workgroups share a CU: X
// holds one full 64 x 64 operand (E_p, then U(p, j) transposed) and C a 32-deep
// chunk of the other (A'(p, j) transposed, then L(i, p)), both at row strides
// for which the MFMA operand reads (16 rows x 4 consecutive entries) hit distinct
// banks; a B operand is kept transposed so that it is read the same way.  The
// inverse's scratch reuses C.
template <typename T> struct alignas(16) FStepSmem {
    T X[NB * LDT];
    union {
        T C[NB * SA_LD];
        T tmp[INV_TMP];
    };
    T aux[4 + NB];
};

// acc += X(:, k0 .. k0+31) * CT^T, X [i][k] (stride LDT), CT [j][k - k0] (stride
// SA_LD); only k < ka and rows < ka (a multiple of 16) take part.
template <typename T> __device__ __forceinline__ void mm_xc(Acc<T> &acc, const T *X, const T *CT, int k0, int ka)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = acc_row(wave), wc = acc_col(wave);
    if (wr >= ka) return;
#pragma unroll
    for (int k16 = 0; k16 < KT; k16 += 16) {
        if (k0 + k16 >= ka) return;
#pragma unroll
        for (int kk = k16; kk < k16 + 16; kk += 4) {
            T av[2], bv[2];
#pragma unroll
            for (int x = 0; x < 2; x++) av[x] = X[(wr + 16 * x + (lane & 15)) * LDT + k0 + kk + (lane >> 4)];
#pragma unroll
            for (int y = 0; y < 2; y++) bv[y] = CT[(wc + 16 * y + (lane & 15)) * SA_LD + kk + (lane >> 4)];
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++) acc.a[x][y] = mfma<T>::run(av[x], bv[y], acc.a[x][y]);
        }
    }
}
// acc += C * XT(:, k0 .. k0+31)^T, C [i][k - k0] (stride SA_LD), XT [j][k] (stride
// LDT); only k < ka.
template <typename T> __device__ __forceinline__ void mm_cx(Acc<T> &acc, const T *C, const T *XT, int k0, int ka)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = acc_row(wave), wc = acc_col(wave);
#pragma unroll
    for (int k16 = 0; k16 < KT; k16 += 16) {
        if (k0 + k16 >= ka) return;
#pragma unroll
        for (int kk = k16; kk < k16 + 16; kk += 4) {
            T av[2], bv[2];
#pragma unroll
            for (int x = 0; x < 2; x++) av[x] = C[(wr + 16 * x + (lane & 15)) * SA_LD + kk + (lane >> 4)];
#pragma unroll
            for (int y = 0; y < 2; y++) bv[y] = XT[(wc + 16 * y + (lane & 15)) * LDT + k0 + kk + (lane >> 4)];
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++) acc.a[x][y] = mfma<T>::run(av[x], bv[y], acc.a[x][y]);
        }
    }
}
// A 32 x 64 row chunk (rows r0 .. r0+31 of a row-major tile at src, stride ld) into
// registers (thread t holds t + 256 r: row (t + 256 r) / 64, column t % 64), and
// into C transposed (C [column][row]).
// (Here and below a thread's offset into the tile is one 32-bit register, in
// bytes, and its rows' steps go to the scalar base: per-thread addresses would
// spill.)
template <typename T> __device__ __forceinline__ T &at(T *base, unsigned bytes)
{
    return *reinterpret_cast<T *>(reinterpret_cast<char *>(const_cast<std::remove_const_t<T> *>(base)) + bytes);
}
template <typename T> __device__ __forceinline__ void rowchunk_load(T (&v)[8], const T *src, unsigned ld, int r0)
{
    const unsigned o = ((threadIdx.x >> 6) * ld + (threadIdx.x & 63)) * sizeof(T);
#pragma unroll
    for (int r = 0; r < 8; r++) v[r] = at(src + (size_t)((r0 + 4 * r) * ld), o);
}
template <typename T> __device__ __forceinline__ void rowchunk_put_t(T *C, const T (&v)[8])
{
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const int t = threadIdx.x + 256 * r;
        C[(t & 63) * SA_LD + (t >> 6)] = v[r];
    }
}
// A 64 x 32 column chunk (columns c0 .. c0+31) into registers (thread t holds
// t + 256 r: row (t + 256 r) / 32, column t % 32), and into C as it is.
template <typename T> __device__ __forceinline__ void colchunk_load(T (&v)[8], const T *src, unsigned ld, int c0)
{
    const unsigned o = ((threadIdx.x >> 5) * ld + (threadIdx.x & 31)) * sizeof(T);
#pragma unroll
    for (int r = 0; r < 8; r++) v[r] = at(src + (size_t)(8 * r * ld) + c0, o);
}
template <typename T> __device__ __forceinline__ void colchunk_put(T *C, const T (&v)[8])
{
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const int t = threadIdx.x + 256 * r;
        C[(t >> 5) * SA_LD + (t & 31)] = v[r];
    }
}

// The tile element of result item (x, y, v) of a thread: tile + acc_at(x, y, v, ld)
// at byte offset acc_off(ld).
template <typename T> __device__ __forceinline__ unsigned acc_off(unsigned ld)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    return ((acc_row(wave) + mfma<T>::row(lane, 0)) * ld + acc_col(wave) + (lane & 15)) * sizeof(T);
}
template <typename T> __device__ __forceinline__ size_t acc_at(int x, int y, int v, unsigned ld)
{
    return (size_t)((16 * x + mfma<T>::row(0, v)) * ld) + 16 * y;
}

// Rows (a multiple of 16) of own block p that hold DOFs: the rest of the last
// block is identity padding, its rows and columns elsewhere zero.
__device__ __forceinline__ int live_rows(const gf_front_dev &F, int p) { return min(NB, (F.k - NB * p + 15) & ~15); }

// A child's Schur complement entries of a tile at a thread's result positions:
// first the positions in the child's update rows, then, behind a product, the
// entries (at 64-bit addresses: a front may pass 4 GB, and 32-bit offsets were no
// faster, 153.2 ms a 64 x 64 plate solve against 152.9).
template <typename T> struct ChildTile {
    int a[2][4], b[2];
    __device__ __forceinline__ void positions(const FrontTab &t, int c, int R0, int C0)
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int *im = t.inv + t.child_inv[c];
#pragma unroll
        for (int y = 0; y < 2; y++) b[y] = im[C0 + acc_col(wave) + 16 * y + (lane & 15)];
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int v = 0; v < 4; v++) a[x][v] = im[R0 + acc_row(wave) + 16 * x + mfma<T>::row(lane, v)];
    }
    __device__ __forceinline__ void entries(const FrontTab &t, int c, const T *Fb, T (&u)[2][2][4])
    {
        const gf_front_dev C = t.fr[t.child[c]];
        const T *U = Fb + C.F + gf_front_at(NB * C.kb, NB * C.kb, C.mp);
        acc_each<T>([&](int x, int y, int v, int, int) {
            u[x][y][v] = T(0);
            if (a[x][v] >= 0 && b[y] >= 0)
                u[x][y][v] = U[gf_front_at(a[x][v], b[y], C.mp)];
        });
    }
};

// Launch p >= 0 of a level's factorisation (the band step on every front of the
// level; see the file header).  Items (front, tile row, tile column, kind | rows
// << 8), kinds: 0 diagonal, 1 update, 2 conversion.  Each product runs in two
// 32-deep chunks; all of a workgroup's loads are issued before the first product.
// An update item covers `rows` tiles of one column: W = E_p A'(p, j) is formed
// once for them.  One tile is two products of 64^3, of which W is half; launches
// of more tiles than the device holds at once are bound by those products (45 %
// of the MFMA rate at one tile an item), so the plan gives them items of several
// rows while the items still make three rounds (fewer leave the last round
// empty: 3,584 items of one tile 82 us, 2,560 of two 89); the others are bound by
// the chain of one workgroup and take one row an item.
// Padding: a block's products stop at its live rows (33 DOFs of a mesh line fill
// half of a block).  Launch 0 takes the old value of a tile outside the own rows
// and columns straight from the children, summed in their order (GATHER; zero
// for a leaf): the assembly does not write those tiles.  64 x 64 plate, levels 1
// to 3: assembly 78, 53, 50 -> 43, 29, 35 us, this launch 58, 51, 58 -> 64, 52, 64.
template <typename T, bool GATHER>
__global__ __launch_bounds__(256, 3) void front_step_kernel(FrontTab t, int first, int p, T *Fb, T *Eb, int *flag,
                                                         double *Vb)
{
    __shared__ FStepSmem<T> sm;
    __shared__ double rv[2][NB];  // the right-hand side block of row p (or p - 1) and E times it
    const int *it = t.items + 4 * (size_t)(first + blockIdx.x);
    const int f = it[0];
    if (f < 0) return;
    const int ti = it[1], tj = it[2], rows = it[3] >> 8;
    const int kind = GATHER ? it[3] & 1 : it[3] & 255;  // (launch 0 converts no row)
    if (kind == 0) __builtin_amdgcn_s_setprio(3);
    const gf_front_dev F = t.fr[f];
    T *A = Fb + F.F;
    const unsigned ld = F.mp, ao = acc_off<T>(ld);
    T *Ef = Eb + F.E;
    const int tid = threadIdx.x;
    const int C0 = tj * NB;
    // with the right-hand side in the front vector (Vb): the first conversion tile of
    // row p - 1 converts its block, y = E_{p-1} b_{p-1}; the first update tile of row
    // i subtracts L(i, p) y_p, y_p = E_p b_p, from block i (each block written by one
    // workgroup; b_p itself is final and unconverted during launch p)
    const bool rhs_row = Vb && tj == (kind == 2 ? p : p + 1);
    // product 1: W = E_q A'(q, j), q = p (update, diagonal) or p - 1 (conversion)
    const int q = kind == 2 ? ti : p, ka = live_rows(F, q);
    const T *E = Ef + (size_t)q * NB * NB;
    const T *Aq = A + gf_front_at(q * NB, C0, F.mp);  // A'(q, j)
    T e[16], a0[8], a1[8];
#pragma unroll
    for (int r = 0; r < 16; r++) e[r] = at(E + 256 * r, tid * (unsigned)sizeof(T));
    rowchunk_load(a0, Aq, ld, 0);
    rowchunk_load(a1, Aq, ld, KT);
    if (rhs_row && tid < NB) rv[0][tid] = Vb[F.V + (size_t)(q * NB) + tid];
    tile_put(sm.X, LDT, e);
    rowchunk_put_t(sm.C, a0);
    __syncthreads();
    T l0[8], l1[8], old[2][2][4];
    const T *Lp = A + gf_front_at(ti * NB, p * NB, F.mp);  // L(i, p)
    colchunk_load(l0, Lp, ld, 0);  // (a conversion item does not use it)
    if (rhs_row && tid < NB) {
        double yv = 0.0;
        for (int c = 0; c < NB; c++) yv += (double)sm.X[tid * LDT + c] * rv[0][c];
        if (kind == 2) Vb[F.V + (size_t)(q * NB) + tid] = yv;
        else rv[1][tid] = yv;  // y_p
    }
    auto tile = [&](int i0) { return A + gf_front_at(i0 * NB, C0, F.mp); };
    Acc<T> w;
    w.zero();
    mm_xc<T>(w, sm.X, sm.C, 0, ka);
    if (ka > KT) {
        __syncthreads();
        rowchunk_put_t(sm.C, a1);
        __syncthreads();
    }
    colchunk_load(l1, Lp, ld, KT);  // behind the second half of product 1
    if (ka > KT) mm_xc<T>(w, sm.X, sm.C, KT, ka);
    if (__builtin_expect(kind == 2, 1)) {
        acc_each<T>([&](int x, int y, int v, int, int) { at(tile(ti) + acc_at<T>(x, y, v, ld), ao) = w.a[x][y][v]; });
        return;
    }
    __syncthreads();
    // product 2: old - L(i, p) W, W kept transposed in X
    acc_each<T>([&](int x, int y, int v, int i, int j) { sm.X[j * LDT + i] = w.a[x][y][v]; });
    Acc<T> acc;
    for (int r = 0;; r++) {
        const int R0 = (ti + r) * NB;
        colchunk_put(sm.C, l0);
        __syncthreads();
        // the old value behind product 2
        const bool unset = p == 0 && ti + r >= F.kb && tj >= F.kb;
        ChildTile<T> ct;
        if (!unset)
            acc_each<T>([&](int x, int y, int v, int, int) { old[x][y][v] = at(tile(ti + r) + acc_at<T>(x, y, v, ld), ao); });
        else if (GATHER) ct.positions(t, F.ch0, R0, C0);
        else acc_each<T>([&](int x, int y, int v, int, int) { old[x][y][v] = T(0); });
        double s = 0.0;
        if (rhs_row && tid < NB)
            for (int c = 0; c < KT; c++) s += (double)sm.C[tid * SA_LD + c] * rv[1][c];
        acc.zero();
        mm_cx<T>(acc, sm.C, sm.X, 0, ka);
        if (ka > KT) {
            __syncthreads();
            colchunk_put(sm.C, l1);
            __syncthreads();
        }
        if (GATHER && unset) {
            ct.entries(t, F.ch0, Fb, old);
            if (F.ch0 + 1 < F.ch1) ct.positions(t, F.ch0 + 1, R0, C0);
        }
        if (ka > KT) {
            if (rhs_row && tid < NB)
                for (int c = 0; c < KT; c++) s += (double)sm.C[tid * SA_LD + c] * rv[1][KT + c];
            mm_cx<T>(acc, sm.C, sm.X, KT, ka);
        }
        if (rhs_row && tid < NB) Vb[F.V + R0 + tid] -= s;  // b_i -= L(i, p) y_p
        if (kind == 0) break;
        if (GATHER && unset)
            for (int c = F.ch0 + 1; c < F.ch1; c++) {
                T u[2][2][4];
                if (c > F.ch0 + 1) ct.positions(t, c, R0, C0);
                ct.entries(t, c, Fb, u);
                acc_each<T>([&](int x, int y, int v, int, int) { old[x][y][v] += u[x][y][v]; });
            }
        acc_each<T>([&](int x, int y, int v, int, int) {
            at(tile(ti + r) + acc_at<T>(x, y, v, ld), ao) = old[x][y][v] - acc.a[x][y][v];
        });
        if (r + 1 >= rows) return;
        Lp += (size_t)(NB * ld);
        colchunk_load(l0, Lp, ld, 0);
        colchunk_load(l1, Lp, ld, KT);
        __syncthreads();
    }
    __syncthreads();
    acc_each<T>([&](int x, int y, int v, int i, int j) { sm.X[i * LDT + j] = old[x][y][v] - acc.a[x][y][v]; });
    __syncthreads();
    inverse64<T>(sm.X, sm.tmp, sm.aux, flag, live_rows(F, ti) >> 4);  // E_{p+1}
    T *En = Ef + (size_t)ti * NB * NB;
    for (int q2 = tid; q2 < NB * NB; q2 += 256) En[q2] = sm.X[(q2 / NB) * LDT + q2 % NB];
}

// ---- solve -----------------------------------------------------------------------
// Tile rows are summed by quads of lanes: thread t takes row t / 4 of a 64-row
// tile and its 16 columns 16 (t % 4) .. 16 (t % 4) + 15 (one 128-byte run of an
// FP64 row, read with 16-byte vector loads), so a row's partial sums sit in four
// neighbouring lanes and two DPP moves reduce them.  Front rows are 512-byte
// aligned (fronts and diagonal inverses start at multiples of 64 x 64 entries,
// rows are multiples of 64 entries long).

template <typename T> __device__ __forceinline__ void load16(const T *p, T (&v)[16]);
template <> __device__ __forceinline__ void load16<double>(const double *p, double (&v)[16])
{
    const double2 *q = reinterpret_cast<const double2 *>(p);
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const double2 w = q[e];
        v[2 * e] = w.x;
        v[2 * e + 1] = w.y;
    }
}
template <> __device__ __forceinline__ void load16<float>(const float *p, float (&v)[16])
{
    const float4 *q = reinterpret_cast<const float4 *>(p);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float4 w = q[e];
        v[4 * e] = w.x;
        v[4 * e + 1] = w.y;
        v[4 * e + 2] = w.z;
        v[4 * e + 3] = w.w;
    }
}
template <typename T> __device__ __forceinline__ double dot16(const T (&v)[16], const double *y)
{
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < 16; e++) s += (double)v[e] * y[e];
    return s;
}
// Sum over the four lanes of a quad (DPP quad_perm [1,0,3,2] then [2,3,0,1]).
__device__ __forceinline__ double quad_sum(double s)
{
    s += dpp_mov<0xB1>(s);
    return s + dpp_mov<0x4E>(s);
}

// Own rows of a front: w = b_own + children's update vectors, then
// y_p = E_p (w_p - sum_{q<p} L(p, q) y_q) block by block (one workgroup, y in LDS).
template <typename T>
__global__ __launch_bounds__(256) void front_fwd_own_kernel(FrontTab t, int f0, const T *Fb, const T *Eb,
                                                            const double *rhs, double *Vb)
{
    __shared__ double y[KMAX];
    __shared__ double tmp[NB];
    const int f = f0 + blockIdx.x;
    const gf_front_dev F = t.fr[f];
    const int kp = NB * F.kb, tid = threadIdx.x, r = tid >> 2, sg = 16 * (tid & 3);
    const int *rows = t.rows + F.rows;
    const size_t ld = (size_t)F.mp;
    for (int i = tid; i < kp; i += 256) {
        const int o = rows[i];
        y[i] = (o >= 0 ? rhs[o] : 0.0) + child_sum(t, F, i, Vb);
    }
    __syncthreads();
    for (int p = 0; p < F.kb; p++) {
        T e[16];
        load16(Eb + F.E + (size_t)p * NB * NB + r * NB + sg, e);
        const T *L = Fb + F.F + (size_t)(NB * p + r) * ld + sg;
        double part = 0.0;
        for (int q = 0; q < p; q++) {
            T v[16];
            load16(L + NB * q, v);
            part += dot16(v, y + NB * q + sg);
        }
        part = quad_sum(part);
        if ((tid & 3) == 0) tmp[r] = y[NB * p + r] - part;
        __syncthreads();
        part = quad_sum(dot16(e, tmp + sg));
        if ((tid & 3) == 0) y[NB * p + r] = part;
        __syncthreads();
    }
    for (int i = tid; i < kp; i += 256) Vb[F.V + i] = y[i];
}

// Update row tile t of a front: c = sum_children c_child - L(t, own) y_own.
template <typename T>
__global__ __launch_bounds__(256) void front_fwd_upd_kernel(FrontTab t, int first, const T *Fb, double *Vb)
{
    __shared__ double y[KMAX];
    const int *it = t.items + 4 * (size_t)(first + blockIdx.x);
    const gf_front_dev F = t.fr[it[0]];
    const int tr = it[1], tid = threadIdx.x, r = tid >> 2, sg = 16 * (tid & 3);
    const int kp = NB * F.kb, i = NB * tr + r;
    for (int j = tid; j < kp; j += 256) y[j] = Vb[F.V + j];
    const double c = (tid & 3) == 0 ? child_sum(t, F, i, Vb) : 0.0;
    __syncthreads();
    const T *L = Fb + F.F + (size_t)i * F.mp + sg;
    double part = 0.0;
    for (int q = 0; q < F.kb; q++) {
        T v[16];
        load16(L + NB * q, v);
        part += dot16(v, y + NB * q + sg);
    }
    part = quad_sum(part);
    if ((tid & 3) == 0) Vb[F.V + i] = c - part;
}

// The backward kernels (one workgroup of four wavefronts a row tile or front)
// read tiles whole rows at a time: wavefront w takes rows 16 w .. 16 w + 15 in
// pairs, lane l the columns 2 (l % 32) and the next of row l / 32 of a pair, so a
// load instruction covers 1 KB in eight lines.  With a quad of lanes a row, each
// lane 128 contiguous bytes, every instruction touched 64 lines and a tile took
// four times as long to come through the CU's cache, which is what these few
// workgroups are bound by: a row of 9 update tiles 15 -> 9.5 us, the 64 x 64
// plate's root (9 own blocks, 36 tiles) 44 -> 29 us, its leaves 28 -> 22 us.  (Four
// quad-row groups on more tiles at once made the root 66 us: same bound.)  A lane
// keeps the partial sums of its eight rows over
// all tiles; the 32 lanes of a row are summed once at the end.
template <typename T> struct RowTile {
    T v[16];
    __device__ __forceinline__ void load(const T *tile, unsigned ld)
    {
        typedef T pair_t __attribute__((ext_vector_type(2)));
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const unsigned o = ((16 * wave + (lane >> 5)) * ld + 2 * (lane & 31)) * sizeof(T);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const pair_t w = *reinterpret_cast<const pair_t *>(&at(tile + (size_t)(2 * k * ld), o));
            v[2 * k] = w.x;
            v[2 * k + 1] = w.y;
        }
    }
    // acc[k] += this lane's part of row 2 k + l / 32 times y (LDS, 16-byte aligned; the tile's
    // 64 columns)
    __device__ __forceinline__ void dot(double (&acc)[8], const double *y) const
    {
        const double2 w = *reinterpret_cast<const double2 *>(y + 2 * (threadIdx.x & 31));
#pragma unroll
        for (int k = 0; k < 8; k++) acc[k] = fma((double)v[2 * k + 1], w.y, fma((double)v[2 * k], w.x, acc[k]));
    }
};
// Sum of the partials over the 32 lanes of a row; the lane gets that of tile row
// tile_row() (four lanes share one).
__device__ __forceinline__ int tile_row()
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    return 16 * wave + 2 * ((lane >> 4 & 1) * 4 + (lane >> 3 & 1) * 2 + (lane >> 2 & 1)) + (lane >> 5);
}
__device__ __forceinline__ double tile_sum(double (&acc)[8])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int n = 4; n >= 1; n >>= 1) {  // halve the rows, xor 16, 8, 4
        const bool up = lane & (4 * n);
#pragma unroll
        for (int k = 0; k < n; k++) {
            const double give = up ? acc[k] : acc[k + n], keep = up ? acc[k + n] : acc[k];
            acc[k] = keep + __shfl_xor(give, 4 * n);
        }
    }
    return quad_sum(acc[0]);
}

// Own row tile p of a front with an update part: z_p = y_p - U(p, update) x_update
// (x_update gathered from the ancestors' rows of x into LDS, 1024 at a time).
template <typename T>
__global__ __launch_bounds__(256) void front_bwd_upd_kernel(FrontTab t, int first, const T *Fb, const T *Eb,
                                                            const double *x, double *Vb, int raw_last)
{
    __shared__ alignas(16) double xu[KMAX];
    const int *it = t.items + 4 * (size_t)(first + blockIdx.x);
    const gf_front_dev F = t.fr[it[0]];
    const int p = it[1], tid = threadIdx.x, r = tile_row();
    const int *rows = t.rows + F.rows;
    const unsigned ld = F.mp;
    const T *U = Fb + F.F + (size_t)(NB * p * ld);
    const bool last = p == F.kb - 1, lead = (tid & 3) == 0;
    double acc[8] = {}, *z = Vb + F.V + NB * p;
    RowTile<T> a;
    a.load(U + NB * F.kb, ld);
    const double y = lead ? z[r] : 0.0;
    for (int c0 = NB * F.kb; c0 < F.mp; c0 += KMAX) {
        const int cn = min(KMAX, F.mp - c0);
        __syncthreads();
        for (int j = tid; j < cn; j += 256) {
            const int o = rows[c0 + j];
            xu[j] = o >= 0 ? x[o] : 0.0;
        }
        __syncthreads();
        for (int q = 0; q < cn; q += NB) {
            RowTile<T> b;
            if (c0 + q + NB < F.mp) b.load(U + c0 + q + NB, ld);
            a.dot(acc, xu + q);
            a = b;
        }
    }
    // the last own block row holds A'(p, .) = D_p U(p, .): subtract E_p (A' x); when
    // the factorisation carried the right-hand side, its block is unconverted too:
    // z_p = E_p (b_p - A' x)
    if (last) a.load(Eb + F.E + (size_t)(p * NB * NB), NB);
    const double part = tile_sum(acc);
    if (!last) {
        if (lead) z[r] = y - part;
        return;
    }
    __syncthreads();
    if (lead) xu[r] = raw_last ? y - part : part;
    __syncthreads();
    double e[8] = {};
    a.dot(e, xu);
    const double s = tile_sum(e);
    if (lead) z[r] = raw_last ? s : y - s;
}

// Own-block back substitution x_p = z_p - sum_{p < j < kb} U(p, j) x_j, then the
// scatter of the own rows of x.
template <typename T>
__global__ __launch_bounds__(256) void front_bwd_own_kernel(FrontTab t, int f0, const T *Fb, const T *Eb,
                                                            const double *Vb, double *x, int raw_last)
{
    __shared__ alignas(16) double y[KMAX];
    const int f = f0 + blockIdx.x;
    const gf_front_dev F = t.fr[f];
    const int kp = NB * F.kb, tid = threadIdx.x, r = tile_row();
    const int *rows = t.rows + F.rows;
    const unsigned ld = F.mp;
    const T *U = Fb + F.F;
    const bool lead = (tid & 3) == 0;
    // each row's first tile is loaded before the row it waits for is done
    RowTile<T> a;
    if (F.kb > 1) a.load(U + (size_t)(NB * (F.kb - 2) * ld) + NB * (F.kb - 1), ld);
    for (int i = tid; i < kp; i += 256) y[i] = Vb[F.V + i];
    __syncthreads();
    if (raw_last && F.mb == F.kb) {
        // no update part, so no front_bwd_upd_kernel converted the last block: y = E b
        RowTile<T> e;
        double acc[8] = {};
        e.load(Eb + F.E + (size_t)((F.kb - 1) * NB * NB), NB);
        e.dot(acc, y + NB * (F.kb - 1));
        const double s = tile_sum(acc);
        __syncthreads();
        if (lead) y[NB * (F.kb - 1) + r] = s;
        __syncthreads();
    }
    for (int p = F.kb - 2; p >= 0; p--) {
        const T *Up = U + (size_t)(NB * p * ld);
        double acc[8] = {};
        for (int j = p + 1; j < F.kb; j++) {
            RowTile<T> b;
            if (j + 1 < F.kb) b.load(Up + NB * (j + 1), ld);
            else if (p > 0) b.load(Up - (size_t)(NB * ld) + NB * p, ld);
            a.dot(acc, y + NB * j);
            a = b;
        }
        const double s = tile_sum(acc);
        if (lead) y[NB * p + r] -= s;
        __syncthreads();
    }
    for (int i = tid; i < F.k; i += 256) x[rows[i]] = y[i];
}

// Next tile of the upper block rows in the order of use: row p's columns p + 1 .. mb - 1,
// p from the last down; past the last, that one again.
template <typename T>
__device__ __forceinline__ void bwd_fetch(RowTile<T> &a, const T *U, unsigned ld, int mb, int &p, int &j)
{
    a.load(U + (size_t)(NB * p * ld) + NB * j, ld);
    const bool end = j + 1 >= mb;
    j = !end ? j + 1 : p > 0 ? p : j;
    p = end && p > 0 ? p - 1 : p;
}
// Row's end: y -= sums, which are cleared.
__device__ __forceinline__ void bwd_row(double (&acc)[8], double *y)
{
    const double s = tile_sum(acc);
    if ((threadIdx.x & 3) == 0) y[tile_row()] -= s;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++) acc[k] = 0.0;
}
// The last own row's end (see front_bwd_upd_kernel); w: 64 doubles of LDS.
template <typename T>
__device__ __forceinline__ void bwd_last(double (&acc)[8], const RowTile<T> &e, double *y, double *w, int raw)
{
    const int r = tile_row();
    const bool lead = (threadIdx.x & 3) == 0;
    const double part = tile_sum(acc), y0 = lead ? y[r] : 0.0;
    if (lead) w[r] = raw ? y0 - part : part;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++) acc[k] = 0.0;
    e.dot(acc, w);
    const double s = tile_sum(acc);
    if (lead) y[r] = raw ? s : y0 - s;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++) acc[k] = 0.0;
}

// The two above in one, a workgroup a front, for the levels where the plan says so
// (bwd_one): x_p = z_p - U(p, p+1 ..) (x_own | x_update), p from the last row up, over
// one vector in LDS.  Three tiles are in flight, without a move or a branch between
// a load and its use (past the last tile the last one is loaded again).  Bound by its
// launch and the chain front record, rows, x: 7 us for a level of small fronts in
// place of 5.1 + 4.6, a root of 9 own blocks 25.6 us where one tile in flight took 28.7.
template <typename T>
__global__ __launch_bounds__(256) void front_bwd_kernel(FrontTab t, int f0, const T *Fb, const T *Eb, const double *Vb,
                                                        double *x, int raw_last)
{
    __shared__ alignas(16) double v[KMAX];
    __shared__ alignas(16) double w[NB];
    const gf_front_dev F = t.fr[f0 + blockIdx.x];
    const int kp = NB * F.kb, tid = threadIdx.x;
    const int *rows = t.rows + F.rows;
    const unsigned ld = F.mp;
    const T *U = Fb + F.F;
    const bool upd = F.mb > F.kb;
    int p = upd ? F.kb - 1 : F.kb - 2, j = p + 1;  // next tile to use
    int lp = max(p, 0), lj = min(lp + 1, F.mb - 1);    // next tile to load
    RowTile<T> a, b, c, e;
    bwd_fetch(a, U, ld, F.mb, lp, lj);
    e.load(Eb + F.E + (size_t)((F.kb - 1) * NB * NB), NB);
    bwd_fetch(b, U, ld, F.mb, lp, lj);
    bwd_fetch(c, U, ld, F.mb, lp, lj);
    for (int i = tid; i < F.mp; i += 256) {
        const int o = i < kp ? 0 : rows[i];
        v[i] = i < kp ? Vb[F.V + i] : o >= 0 ? x[o] : 0.0;
    }
    __syncthreads();
    double acc[8] = {};
    if (!upd && raw_last) bwd_last(acc, e, v + kp - NB, w, raw_last);
    while (p >= 0) {
        a.dot(acc, v + NB * j);
        bwd_fetch(a, U, ld, F.mb, lp, lj);
        if (++j == F.mb) {
            if (p == F.kb - 1) bwd_last(acc, e, v + kp - NB, w, raw_last);
            else bwd_row(acc, v + NB * p);
            j = p--;
        }
        if (p < 0) break;
        b.dot(acc, v + NB * j);
        bwd_fetch(b, U, ld, F.mb, lp, lj);
        if (++j == F.mb) {
            if (p == F.kb - 1) bwd_last(acc, e, v + kp - NB, w, raw_last);
            else bwd_row(acc, v + NB * p);
            j = p--;
        }
        if (p < 0) break;
        c.dot(acc, v + NB * j);
        bwd_fetch(c, U, ld, F.mb, lp, lj);
        if (++j == F.mb) {
            if (p == F.kb - 1) bwd_last(acc, e, v + kp - NB, w, raw_last);
            else bwd_row(acc, v + NB * p);
            j = p--;
        }
    }
    for (int i = tid; i < F.k; i += 256) x[rows[i]] = v[i];
}

FrontTab tab_of(const gf_fronts &fp)
{
    FrontTab t;
    t.fr = fp.d_fr;
    t.rows = fp.d_rows;
    t.child = fp.d_child;
    t.inv = fp.d_inv;
    t.items = fp.d_items;
    t.child_inv = fp.d_child_inv;
    t.orig = fp.d_orig;
    t.asm_orig = fp.d_asm_orig;
    return t;
}

template <typename T>
int front_factor_t(const gf_fronts &fp, const double *ab, int ld, int hb, const double *D, T *F, T *E, hipStream_t s,
                   int *flag, const double *rhs, double *V)
{
    const FrontTab t = tab_of(fp);
    int launches = 0;
    for (int l = 0; l < fp.n_level; l++) {
        int pr = gf_probe_begin(s, GF_KC_FRONT_ASSEMBLE);
        hipLaunchKernelGGL(front_assemble_kernel<T>, dim3(fp.asm_count[l]), dim3(ASM_T), 0, s, t, fp.asm_first[l], ab, ld,
                           hb, D, F, E, flag, rhs, V);
        gf_probe_end(s, pr, (double)fp.asm_count[l] * NB * NB);
        launches++;
        for (int k = fp.lev_step[l]; k < fp.lev_step[l + 1]; k++) {
            if (fp.step_count[k] == 0) continue;
            const int p = k - fp.lev_step[l];
            pr = gf_probe_begin(s, GF_KC_FRONT_STEP);
            // (leaves are the fronts of level 0)
            if (p == 0 && l > 0)
                hipLaunchKernelGGL((front_step_kernel<T, true>), dim3(fp.step_count[k]), dim3(256), 0, s, t,
                                   fp.step_first[k], p, F, E, flag, rhs ? V : nullptr);
            else
                hipLaunchKernelGGL((front_step_kernel<T, false>), dim3(fp.step_count[k]), dim3(256), 0, s, t,
                                   fp.step_first[k], p, F, E, flag, rhs ? V : nullptr);
            gf_probe_end(s, pr, fp.step_flops[k]);
            launches++;
        }
    }
    GF_HIP(hipGetLastError());
    return launches;
}

template <typename T>
int front_solve_t(const gf_fronts &fp, const T *F, const T *E, const double *rhs, double *x, double *V, hipStream_t s,
                  bool carried)
{
    const FrontTab t = tab_of(fp);
    int launches = 0;
    // probe units: factor bytes each launch reads (the own triangle with the
    // diagonal inverses, or the update panel)
    auto own_bytes = [&](int l, bool fwd) {
        double b = 0.0;
        for (int f = fp.lev_off[l]; f < fp.lev_off[l + 1]; f++) {
            const double kp = NB * fp.fr[f].kb;
            b += fwd ? kp * (kp + NB) / 2.0 : kp * (kp - NB) / 2.0;
        }
        return b * sizeof(T);
    };
    auto panel_bytes = [&](int l) {
        double b = 0.0;
        for (int f = fp.lev_off[l]; f < fp.lev_off[l + 1]; f++)
            b += (double)NB * fp.fr[f].kb * (fp.fr[f].mp - NB * fp.fr[f].kb);
        return b * sizeof(T);
    };
    for (int l = 0; l < fp.n_level && !carried; l++) {
        const int nf = fp.lev_off[l + 1] - fp.lev_off[l];
        int pr = gf_probe_begin(s, GF_KC_FRONT_SOLVE);
        hipLaunchKernelGGL(front_fwd_own_kernel<T>, dim3(nf), dim3(256), 0, s, t, fp.lev_off[l], F, E, rhs, V);
        gf_probe_end(s, pr, pr >= 0 ? own_bytes(l, true) : 0.0);
        launches++;
        if (fp.fupd_count[l] > 0) {
            pr = gf_probe_begin(s, GF_KC_FRONT_SOLVE);
            hipLaunchKernelGGL(front_fwd_upd_kernel<T>, dim3(fp.fupd_count[l]), dim3(256), 0, s, t, fp.fupd_first[l], F, V);
            gf_probe_end(s, pr, pr >= 0 ? panel_bytes(l) : 0.0);
            launches++;
        }
    }
    for (int l = fp.n_level - 1; l >= 0; l--) {
        const int nf = fp.lev_off[l + 1] - fp.lev_off[l];
        int pr;
        if (fp.bwd_one[l]) {
            pr = gf_probe_begin(s, GF_KC_FRONT_SOLVE);
            hipLaunchKernelGGL(front_bwd_kernel<T>, dim3(nf), dim3(256), 0, s, t, fp.lev_off[l], F, E, (const double *)V, x,
                               carried ? 1 : 0);
            gf_probe_end(s, pr, pr >= 0 ? panel_bytes(l) + own_bytes(l, false) : 0.0);
            launches++;
            continue;
        }
        if (fp.bupd_count[l] > 0) {
            pr = gf_probe_begin(s, GF_KC_FRONT_SOLVE);
            hipLaunchKernelGGL(front_bwd_upd_kernel<T>, dim3(fp.bupd_count[l]), dim3(256), 0, s, t, fp.bupd_first[l], F,
                               E, (const double *)x, V, carried ? 1 : 0);
            gf_probe_end(s, pr, pr >= 0 ? panel_bytes(l) : 0.0);
            launches++;
        }
        pr = gf_probe_begin(s, GF_KC_FRONT_SOLVE);
        hipLaunchKernelGGL(front_bwd_own_kernel<T>, dim3(nf), dim3(256), 0, s, t, fp.lev_off[l], F, E, (const double *)V,
                           x, carried ? 1 : 0);
        gf_probe_end(s, pr, pr >= 0 ? own_bytes(l, false) : 0.0);
        launches++;
    }
    GF_HIP(hipGetLastError());
    return launches;
}

template <typename T> int put(T **dst, const std::vector<T> &src, hipStream_t s)
{
    const size_t n = std::max<size_t>(src.size(), 1);
    GF_TRY(gf_pool_alloc((void **)dst, n * sizeof(T)));
    if (!src.empty()) GF_HIP(hipMemcpyAsync(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice, s));
    return GF_OK;
}

}  // namespace

int gf_front_upload(gf_fronts &fp, hipStream_t s)
{
    if (fp.max_k > KMAX) {
        gf_set_error("multifrontal plan: supernode larger than the solve supports");
        return GF_E_STATE;
    }
    GF_TRY(put(&fp.d_fr, fp.fr, s));
    GF_TRY(put(&fp.d_rows, fp.rows, s));
    GF_TRY(put(&fp.d_child, fp.child, s));
    GF_TRY(put(&fp.d_child_inv, fp.child_inv, s));
    GF_TRY(put(&fp.d_inv, fp.inv, s));
    GF_TRY(put(&fp.d_items, fp.items, s));
    GF_TRY(put(&fp.d_orig, fp.orig, s));
    GF_TRY(put(&fp.d_asm_orig, fp.asm_orig, s));
    return GF_OK;
}

void gf_front_free(gf_fronts &fp)
{
    void *p[] = {fp.d_fr, fp.d_rows, fp.d_child, fp.d_child_inv, fp.d_inv, fp.d_items, fp.d_orig, fp.d_asm_orig};
    for (void *q : p) gf_pool_free(q);
    fp.d_fr = nullptr;
    fp.d_rows = fp.d_child = fp.d_inv = fp.d_items = fp.d_orig = fp.d_asm_orig = nullptr;
    fp.d_child_inv = nullptr;
}

int gf_front_factor(const gf_fronts &fp, int elem_size, const double *ab, int ld, int hb, const double *D, void *F,
                    void *E, hipStream_t s, int *flag, const double *rhs, double *V)
{
    if (elem_size == 8) return front_factor_t<double>(fp, ab, ld, hb, D, (double *)F, (double *)E, s, flag, rhs, V);
    return front_factor_t<float>(fp, ab, ld, hb, D, (float *)F, (float *)E, s, flag, rhs, V);
}

int gf_front_solve(const gf_fronts &fp, int elem_size, const void *F, const void *E, const double *rhs, double *x,
                   double *V, hipStream_t s, bool carried)
{
    if (elem_size == 8) return front_solve_t<double>(fp, (const double *)F, (const double *)E, rhs, x, V, s, carried);
    return front_solve_t<float>(fp, (const float *)F, (const float *)E, rhs, x, V, s, carried);
}
