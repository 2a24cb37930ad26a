// FP64 block-tridiagonal factorisation and solve in one pass on gfx950 (the
// narrow-band counterpart of sparsesystem -> MKL PARDISO,
// src/SparseMatrix.cpp:74-166): cyclic reduction over chunks of block rows, one
// workgroup per chunk, several reduction levels per launch.
//
// Block row e couples to its neighbours through A_e (left), B_e and C_e (right).
// Eliminating it between the kept rows a (left) and b (right):
//   X_e = B_e^-1 A_e,  Y_e = B_e^-1 C_e,  z_e = B_e^-1 f_e
//   B_b -= A_b Y_e,  A_b <- -A_b X_e,  f_b -= A_b z_e
//   B_a -= C_a X_e,  C_a <- -C_a Y_e,  f_a -= C_a z_e
// A launch cuts the n rows into chunks of at most R and eliminates every row of
// a chunk but its last one (the separator), in log2 R levels separated by
// barriers: with d the distance from the separator, level j eliminates the odd
// multiples of 2^j.  What a chunk adds to the separator at its left (which the
// chunk before it owns) goes to arrays of its own (dB, df, and the coupling C),
// so no workgroup waits on or writes to another's rows; the next launch adds
// them when it loads its rows.  Once at most R rows are left one workgroup
// finishes: the last row is solved and the rows of that launch substituted
// back; one launch per earlier level then substitutes its chunks back.
//
// What bounds it: the dependent pivots.  One elimination is one wavefront's
// Gauss-Jordan sweep over [B | A | C | f] with the matrix in registers: lane
// 16 q + i holds row i (and i + 16 for blocks wider than 16) of all of B and of
// the columns of A (q < 2) or C (q >= 2) that are its share, so the multiplier
// of a row sits in the row's own lane and the pivot row arrives inside the
// multiply-add (gf_dpp.h): about 35 issued instructions per pivot.  The
// products with A_b and C_a use the same multiply-adds on the X, Y just
// computed (FP64 vector and matrix rates are equal on this device, and this
// way X and Y never pass through LDS).  Where a level has fewer rows than the
// workgroup has wavefronts, several wavefronts share a row, each with part of
// the columns.
#include "gf_dpp.h"

#include <algorithm>

namespace {

// H: rows per lane (blocks of up to 16 H rows).  R: most rows of a chunk; W:
// wavefronts; LV: levels.  The kept rows' blocks live in LDS.
template <int H, int R_> struct crc {
    static constexpr int R = R_, W = H == 1 ? R / 2 : R, LV = R == 8 ? 3 : 5, SLOTS = R / 2 + 1;
    static_assert(R == 8 || (H == 1 && R == 32), "chunk sizes");
};

struct CrArgs {
    const double *A, *B, *C, *f;   // block rows; C of row i at C + (i + coff) m m
    const double *B2, *f2;         // (null, or) what the next chunk added to row i, at index i + 1
    int coff, n, R, m;
    double *XY, *x;                // eliminated rows: X | Y by columns [n][2 m][m]; z, then x [n][m]
    double *oA, *oB, *odB, *oC, *of, *odf;  // reduced rows, one per chunk
    int *flag;
};

typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

template <int H, int R> struct alignas(16) CrSmem {
    static constexpr int MT = 16 * H, LD = MT + 2, SLOTS = crc<H, R>::SLOTS;
    // strides of 2 mod 16 doubles: sixteen lanes reading 16 bytes of sixteen rows hit distinct banks
    double A[SLOTS][MT * LD], B[SLOTS][MT * LD], C[SLOTS][MT * LD];
    double f[SLOTS][MT];
    double x[R + 1][MT];
};

// Interchange of row K with the largest row of column K (rows >= K), when the
// pivot is less than half of it.  Rare and wave-uniform.
template <int H, int NC, int K>
__device__ __forceinline__ void row_interchange(double (&r)[H][NC], unsigned long long at, unsigned long long after)
{
    constexpr int h = K >> 4, kk = K & 15;
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane & 48;
    double best = -1.0;
    int row = K;
#pragma unroll
    for (int hh = h; hh < H; hh++) {
        const bool live = hh > h || __builtin_amdgcn_inverse_ballot_w64(at | after);
        const double v = live ? fabs(r[hh][K]) : -1.0;
        if (v > best) {
            best = v;
            row = 16 * hh + i;
        }
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
        const double ob = __shfl_xor(best, o);
        const int orow = __shfl_xor(row, o);
        if (ob > best || (ob == best && orow < row)) {
            best = ob;
            row = orow;
        }
    }
    row = __builtin_amdgcn_readfirstlane(row);
    const int hp = row >> 4, pp = row & 15;
#pragma unroll
    for (int c = K; c < NC; c++) {
        double rp = r[h][c];
        if constexpr (H > 1) rp = hp == h ? rp : r[H - 1][c];
        const double vk = __shfl(r[h][c], g + kk), vp = __shfl(rp, g + pp);
        if (i == pp) {
            if (H == 1 || hp == h) r[h][c] = vk;
            else r[H - 1][c] = vk;
        }
        if (__builtin_amdgcn_inverse_ballot_w64(at)) r[h][c] = vp;
    }
}

// Pivot K of the sweep over the columns of r: NC of them, the first 16 H are B.
// Rows are kept unscaled: a pivot row stays as it is and sc holds its pivot's
// reciprocal, applied to the right-hand columns at the end.  No branch and no
// interchange: `swap` collects the lanes that ask for one (a row below more than
// 16 times the pivot), and the sweep is done again with interchanges if there
// were any (cr_sweep; a compare that steers a branch costs about 45 cycles of a wavefront's
// issue, a third of a pivot).  Blocks of
// up to 16 rows: p, ip, g and larger are the pivot's, formed by the pivot before.
template <int NC, int K>
__device__ __forceinline__ void cr_pivot1(double (&r)[1][NC], double &sc, int m, unsigned long long &swap,
                                          unsigned long long after, double ip, double g, unsigned long long larger)
{
    if constexpr (K % 4 == 0 && K > 0) {
        asm volatile("" : "+s"(m));  // (the exits' conditions are not kept)
        if (K >= m) return;          // identity padding from here on
    }
    const unsigned long long at = lanes_at<K>();
    after &= ~at;  // rows below the pivot
    swap |= larger & after;
    const bool isk = __builtin_amdgcn_inverse_ballot_w64(at);
    const double h = isk ? 0.0 : g;
    sc = isk ? ip : sc;
    if constexpr (K + 1 < 16) {
        double p;
        nb_pivot<K, NC - K - 1>(&r[0][K + 1], h, p, ip, g, larger);
        cr_pivot1<NC, K + 1>(r, sc, m, swap, after, ip, g, larger);
    } else {
        nb_self<K, NC - K - 1>(&r[0][K + 1], h);
    }
}
// SWAP: with an interchange wherever a row below is more than twice the pivot;
// else as cr_pivot1.
template <int H, int NC, int K, bool SWAP>
__device__ __forceinline__ void cr_pivot(double (&r)[H][NC], double (&sc)[H], int m, unsigned long long &swap,
                                         unsigned long long after)
{
    constexpr int h = K >> 4, kk = K & 15;
    if constexpr (K % 4 == 0) {
        asm volatile("" : "+s"(m));
        if (K >= m) return;
    }
    const unsigned long long at = lanes_at<kk>();
    after = (kk == 0 ? ~0ull : after) & ~at;  // rows of this half below the pivot
    double p = nb_get<kk>(r[h][K]);
    const double lim = (SWAP ? 2.0 : 16.0) * fabs(p);
    unsigned long long larger = __ballot(fabs(r[h][K]) > lim) & after;
    if constexpr (h + 1 < H) larger |= __ballot(fabs(r[H - 1][K]) > lim);
    if constexpr (SWAP) {
        if (larger != 0) {
            row_interchange<H, NC, K>(r, at, after);
            p = nb_get<kk>(r[h][K]);
        }
    } else {
        swap |= larger;
    }
    const double ip = pivot_rcp(p);
    const bool isk = __builtin_amdgcn_inverse_ballot_w64(at);
    if constexpr (H > 1) nb_from<kk, NC - K - 1>(&r[1 - h][K + 1], &r[h][K + 1], -(r[1 - h][K] * ip));
    nb_self<kk, NC - K - 1>(&r[h][K + 1], isk ? 0.0 : -(r[h][K] * ip));
    sc[h] = isk ? ip : sc[h];
    if constexpr (K + 1 < 16 * H) cr_pivot<H, NC, K + 1, SWAP>(r, sc, m, swap, after);
}

// [B | W] -> W = B^-1 W for the NC - 16 H columns W.  The diagonal pivots serve
// while no entry below one is more than 16 times as large and none has grown to
// more than twice its row's diagonal entry in B; else the sweep is done over,
// taking the column's largest entry wherever it is more than twice the diagonal
// one.  Multipliers of up to 16 alone would let entries grow by 17 a pivot (unit
// rows with -8 below the diagonal and ones in the last column lose every digit
// in 16 pivots); with both limits the entries of a column are at most 32 times its
// original diagonal entry when it is eliminated, however rows and columns are
// scaled.  Errors against long double of 100,000 random, sparse, graded and symmetric
// blocks of 3 to 32 rows, in ulp times the condition: the 99th percentile of
// those that pass both limits is 1.4 to 3.3 by family, with interchanges for the
// same blocks 1.9 to 13; and no row of risers and roll-ups fails the second limit.
// (At a limit of 2 on the multipliers three quarters of a riser's rows would be
// done over, at 16 one in 75 to 15.)  A system whose every block is done over takes
// three times as long: 900 blocks of 12 rows 198 us, 64 with dominant diagonals.
// load(r, dg) fills r and, in dg, the high words of the lane's diagonal
// entries of B (1 beyond its rows), again if the sweep is done over; loaded() runs once after it.  A
// pivot below 1e-300, at least 1e300 or not a number sets the flag.
template <int H, int NC, typename F, typename G>
__device__ __forceinline__ void cr_sweep(double (&r)[H][NC], int m, int *flag, F load, G loaded)
{
    double sc[H];
    int dg[H];
    unsigned long long swap = 0;
    load(r, dg);
    loaded();
#pragma unroll
    for (int h = 0; h < H; h++) sc[h] = 1.0;
    if constexpr (H == 1) {
        const double p = nb_get<0>(r[0][0]), ip = pivot_rcp(p);
        const unsigned long long larger = __ballot(fabs(r[0][0]) > 16.0 * fabs(p));
        cr_pivot1<NC, 0>(r, sc[0], m, swap, ~0ull, ip, -(r[0][0] * ip), larger);
    } else {
        cr_pivot<H, NC, 0, false>(r, sc, m, swap, 0);
    }
#pragma unroll
    for (int h = 0; h < H; h++) swap |= __ballot(fabs(sc[h] * __hiloint2double(dg[h], 0)) < 0.5);  // (sc: the pivots' reciprocals)
    if (__builtin_expect(swap != 0, 0)) {
        load(r, dg);
#pragma unroll
        for (int h = 0; h < H; h++) sc[h] = 1.0;
        cr_pivot<H, NC, 0, true>(r, sc, m, swap, 0);
    }
    bool bad = false;
#pragma unroll
    for (int h = 0; h < H; h++) {
        bad |= !(fabs(sc[h]) <= 1e300 && fabs(sc[h]) > 1e-300);
#pragma unroll
        for (int c = 16 * H; c < NC; c++) r[h][c] *= sc[h];
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicExch(flag, 1);
}

// acc(row, c) = sum_k M(row, k) W(k, c) for the CN columns W in r from column
// 16 H on; M in LDS (stride LD).
template <int H, int NC, int CN, int K>
__device__ __forceinline__ void cr_product(double (&acc)[H][CN], const double *M, const double (&r)[H][NC], int m)
{
    constexpr int LD = 16 * H + 2;
    if (K >= m) return;
    const int i = threadIdx.x & 15;
#pragma unroll
    for (int h = 0; h < H; h++) {
        const double2 u = *reinterpret_cast<const double2 *>(M + (16 * h + i) * LD + K);
        const double2 v = *reinterpret_cast<const double2 *>(M + (16 * h + i) * LD + K + 2);
        const double m4[4] = {u.x, u.y, v.x, v.y};
        nb_mac4<K & 15, CN>(acc[h], &r[K >> 4][16 * H], m4);
    }
    if constexpr (K + 4 < 16 * H) cr_product<H, NC, CN, K + 4>(acc, M, r, m);
}

// N columns from col0 on of row `row` of the m x m block at p (plus the block at
// p2 when it is given); what lies beyond m is `pad` on the diagonal, else zero.
template <int H, int N>
__device__ __forceinline__ void cr_load_row(double *v, const double *p, const double *p2, int row, int col0, int m,
                                            bool live, double pad)
{
    constexpr int MT = 16 * H;
    if (m == MT) {
        const double *s = p + (size_t)row * MT + col0;
        if constexpr (N % 2 == 0) {
#pragma unroll
            for (int c = 0; c < N; c += 2) {
                const d2u w = *reinterpret_cast<const d2u *>(s + c);
                v[c] = w.x;
                v[c + 1] = w.y;
            }
        } else {
#pragma unroll
            for (int c = 0; c < N; c++) v[c] = s[c];
        }
        if (p2) {
#pragma unroll
            for (int c = 0; c < N; c++) v[c] += p2[(size_t)row * MT + col0 + c];
        }
#pragma unroll
        for (int c = 0; c < N; c++) v[c] = live ? v[c] : 0.0;
        return;
    }
    const size_t ro = (size_t)(row < m ? row : m - 1) * m;
#pragma unroll
    for (int c = 0; c < N; c++) v[c] = p[ro + (col0 + c < m ? col0 + c : m - 1)];
    if (p2) {
#pragma unroll
        for (int c = 0; c < N; c++) v[c] += p2[ro + (col0 + c < m ? col0 + c : m - 1)];
    }
#pragma unroll
    for (int c = 0; c < N; c++) {
        asm volatile("" : "+v"(row));  // (a mask per column would not fit the scalar registers)
        v[c] = row < m && col0 + c < m ? (live ? v[c] : 0.0) : row == col0 + c ? pad : 0.0;
    }
}

// N columns from col0 on of a row of a block in LDS.
template <int N> __device__ __forceinline__ void lds_row(double *v, const double *s)
{
    if constexpr (N % 2 == 0) {
#pragma unroll
        for (int c = 0; c < N; c += 2) {
            const double2 w = *reinterpret_cast<const double2 *>(s + c);
            v[c] = w.x;
            v[c + 1] = w.y;
        }
    } else {
#pragma unroll
        for (int c = 0; c < N; c++) v[c] = s[c];
    }
}

// Level j of a chunk of nr rows: eliminates the rows at distance d = (2 k + 1)
// 2^j from the separator; S wavefronts share a row.  FIRST: level 0, whose
// eliminated rows come straight from memory.  Slot d / 2 of the LDS
// blocks holds the kept row at even distance d, slot R / 2 the separator at the
// chunk's left (hasL).
template <int H, int R, bool TAIL, int S, bool FIRST, typename G>
__device__ __forceinline__ void cr_level(const CrArgs &a, CrSmem<H, R> &sm, int j, int base, int nr, bool hasL,
                                         G loaded)
{
    constexpr int MT = 16 * H, LD = MT + 2, LS = R / 2;
    constexpr int CW = MT / 2 / S, NC = MT + CW + 1, CN = CW + 1;
    const int step = 1 << j;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4, i = lane & 15;
    const int m = a.m, k = wave / S, sub = wave % S, d = (2 * k + 1) * step;
    const size_t bs = (size_t)m * m;
    const bool act = d < nr;
    const int e = base + nr - 1 - d;                      // block row
    const int sb = (d - step) / 2;                        // slot of the right neighbour
    const bool hasA = d + step < nr || hasL;
    const int sa = d + step < nr ? (d + step) / 2 : LS;   // slot of the left one
    const int col0 = ((q & 1) * S + sub) * CW;
    double r[H][NC];
    auto load = [&](double (&v)[H][NC], int (&dg)[H]) {
#pragma unroll
        for (int h = 0; h < H; h++) {
            const int row = 16 * h + i;
            if constexpr (FIRST) {
                const size_t od = (size_t)(row < m ? row : m - 1) * (m + 1);
                double d = a.B[e * bs + od];
                if (a.B2) d += a.B2[(e + 1) * bs + od];
                dg[h] = __double2hiint(row < m ? d : 1.0);
                cr_load_row<H, MT>(v[h], a.B + e * bs, a.B2 ? a.B2 + (e + 1) * bs : nullptr, row, 0, m, true, 1.0);
                cr_load_row<H, CW>(v[h] + MT, q < 2 ? a.A + e * bs : a.C + (e + a.coff) * bs, nullptr, row, col0, m,
                                   q >= 2 || hasA, 0.0);
                const size_t o = (size_t)e * m + (row < m ? row : m - 1);
                double f = a.f[o];
                if (a.f2) f += a.f2[o + m];
                v[h][MT + CW] = row < m ? f : 0.0;
            } else {
                const int s = d / 2;
                dg[h] = __double2hiint(sm.B[s][row * (LD + 1)]);
                lds_row<MT>(v[h], &sm.B[s][row * LD]);
                lds_row<CW>(v[h] + MT, (q < 2 ? &sm.A[s][row * LD] : &sm.C[s][row * LD]) + col0);
                v[h][MT + CW] = sm.f[s][row];
                if (!hasA && q < 2)
#pragma unroll
                    for (int c = 0; c < CW; c++) v[h][MT + c] = 0.0;
            }
        }
    };
    if (act) {
        cr_sweep<H, NC>(r, m, a.flag, load, loaded);
    } else {
        loaded();
    }
    if (act) {
#pragma unroll
        for (int h = 0; h < H; h++) {
            int row = 16 * h + i;
            double *o = a.XY + 2 * bs * e + (q < 2 ? 0 : bs) + row;
#pragma unroll
            for (int c = 0; c < CW; c++) {
                asm volatile("" : "+v"(row));
                if (row < m && col0 + c < m) o[(size_t)(col0 + c) * m] = r[h][MT + c];
            }
            if (q == 0 && sub == 0) {
                if (TAIL) sm.x[d][row] = r[h][MT + CW];
                else if (row < m) a.x[(size_t)e * m + row] = r[h][MT + CW];
            }
        }
    }
    if constexpr (FIRST) __syncthreads();  // the kept rows are in LDS
    double acc[H][CN];
    auto product = [&](const double *M) {
#pragma unroll
        for (int h = 0; h < H; h++)
#pragma unroll
            for (int c = 0; c < CN; c++) acc[h][c] = 0.0;
        cr_product<H, NC, CN, 0>(acc, M, r, m);
    };
    if (act) product(sm.A[sb]);
    __syncthreads();  // A_b has been read by every wavefront that shares it
    if (act) {
#pragma unroll
        for (int h = 0; h < H; h++) {
            const int o = (16 * h + i) * LD + col0;
#pragma unroll
            for (int c = 0; c < CW; c++) {
                if (q < 2) sm.A[sb][o + c] = -acc[h][c];
                else sm.B[sb][o + c] -= acc[h][c];
            }
            if (q == 0 && sub == 0) sm.f[sb][16 * h + i] -= acc[h][CW];
        }
        if (hasA) product(sm.C[sa]);
    }
    __syncthreads();  // likewise C_a; and a kept row takes its two neighbours' terms one after the other
    if (act && hasA) {
#pragma unroll
        for (int h = 0; h < H; h++) {
            const int o = (16 * h + i) * LD + col0;
#pragma unroll
            for (int c = 0; c < CW; c++) {
                if (q < 2) sm.B[sa][o + c] -= acc[h][c];
                else sm.C[sa][o + c] = -acc[h][c];
            }
            if (q == 0 && sub == 0) sm.f[sa][16 * h + i] -= acc[h][CW];
        }
    }
    __syncthreads();
}

// The levels of a chunk.  The issue slots of a SIMD are what a level with a
// wavefront or more on each of them is bound by, so wavefronts share a row only
// on the levels of one and two rows (each of them repeats the sweep over B).
// Levels of one sharing factor run through one copy of the code.
template <int H, int R, bool TAIL, typename G>
__device__ __forceinline__ void cr_levels(const CrArgs &a, CrSmem<H, R> &sm, int base, int nr, bool hasL, G stage)
{
    constexpr int LV = crc<H, R>::LV;
    auto none = [] {};
    if (nr == 1) stage();
    if constexpr (H == 1) {
        if (nr > 1) cr_level<H, R, TAIL, 1, true>(a, sm, 0, base, nr, hasL, stage);
        for (int j = 1; j < LV - 2 && (1 << j) < nr; j++) cr_level<H, R, TAIL, 1, false>(a, sm, j, base, nr, hasL, none);
        if (nr > R / 4) cr_level<H, R, TAIL, 2, false>(a, sm, LV - 2, base, nr, hasL, none);
        if (nr > R / 2) cr_level<H, R, TAIL, 4, false>(a, sm, LV - 1, base, nr, hasL, none);
    } else {
        if (nr > 1) cr_level<H, R, TAIL, 2, true>(a, sm, 0, base, nr, hasL, stage);
        for (int j = 1; (1 << j) < nr; j++) cr_level<H, R, TAIL, 2, false>(a, sm, j, base, nr, hasL, none);
    }
}

// Sum over the four DPP rows (lanes 16 apart).
__device__ __forceinline__ double row_sum(double v)
{
    unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
    auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false), b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    v = __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
    lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
    a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false), b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
}

// ---- back-substitution of a chunk ------------------------------------------------
// Row d of the chunk (distance from the separator) belongs to wavefront d / RPW,
// whose lane 16 q + i holds row i (i + 16) of the columns MT/2 (q % 2) .. of X_e
// (q < 2) or Y_e, all read before the first level.
template <int H, int R> struct CrBack {
    static constexpr int MT = 16 * H, RPW = R / crc<H, R>::W;
    double w[RPW][H][MT / 2];
    __device__ __forceinline__ void load(const CrArgs &a, int base, int nr)
    {
        const int lane = threadIdx.x & 63, q = lane >> 4, i = lane & 15, m = a.m;
        const size_t bs = (size_t)m * m;
#pragma unroll
        for (int t = 0; t < RPW; t++) {
            const int d = RPW * (threadIdx.x >> 6) + t, dd = d < nr ? d : 0;  // (d = 0 reads within its row, unused)
            const double *p = a.XY + 2 * bs * (base + nr - 1 - dd) + (q < 2 ? 0 : bs);
#pragma unroll
            for (int h = 0; h < H; h++) {
                const int row = 16 * h + i;
#pragma unroll
                for (int c = 0; c < MT / 2; c++) {
                    const int col = MT / 2 * (q & 1) + c;
                    const double v = p[(size_t)(col < m ? col : m - 1) * m + (row < m ? row : m - 1)];
                    w[t][h][c] = d > 0 && d < nr && col < m && row < m ? v : 0.0;
                }
            }
        }
    }
    // x_e = z_e - X_e x_left - Y_e x_right, from the last level's rows to the first's
    __device__ __forceinline__ void run(double (*x)[MT], int nr)
    {
        const int lane = threadIdx.x & 63, q = lane >> 4, i = lane & 15;
        for (int j = crc<H, R>::LV - 1; j >= 0; j--) {
            const int step = 1 << j;
            if (step >= nr) continue;
#pragma unroll
            for (int t = 0; t < RPW; t++) {
                const int d = RPW * (threadIdx.x >> 6) + t;
                if (d > 0 && d < nr && (d & (2 * step - 1)) == step) {
                    const int nb = q < 2 ? (d + step < nr ? d + step : R) : d - step;
                    const double *xn = &x[nb][MT / 2 * (q & 1)];
                    double s[H];
#pragma unroll
                    for (int h = 0; h < H; h++) s[h] = 0.0;
#pragma unroll
                    for (int c = 0; c < MT / 2; c++) {
                        const double xv = xn[c];
#pragma unroll
                        for (int h = 0; h < H; h++) s[h] = fma(w[t][h][c], xv, s[h]);
                    }
#pragma unroll
                    for (int h = 0; h < H; h++) {
                        s[h] = row_sum(s[h]);
                        if (q == 0) x[d][16 * h + i] -= s[h];
                    }
                }
            }
            __syncthreads();
        }
    }
};

// Reduction of the chunks of one level (TAIL: the whole remaining system in one
// chunk, solved and substituted back here).
template <int H, int R, bool TAIL> __global__ __launch_bounds__((64 * crc<H, R>::W)) void cr_reduce_kernel(CrArgs a)
{
    constexpr int MT = 16 * H, LD = MT + 2, W = crc<H, R>::W, LS = R / 2, KV = MT * MT / 64;
    __shared__ CrSmem<H, R> sm;
    const int m = a.m, base = blockIdx.x * a.R, nr = min(a.R, a.n - base);
    const bool hasL = !TAIL && base > 0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t bs = (size_t)m * m;
    // the kept rows (even distance) and the left separator's coupling: every load
    // of a wavefront in flight together (and with them the level's own, blocks of
    // up to 16 rows), into LDS as the first level's wait for its rows ends
    constexpr int TASKS = (3 * (LS + 1) + W - 1) / W;
    double v[TASKS][KV], fv = 0.0;
    const int fs = threadIdx.x / MT, fr = threadIdx.x % MT;  // (64 W threads cover the (LS + 1) MT entries)
    static_assert(64 * W >= (LS + 1) * MT, "one entry of f a thread");
    auto block = [&](int u, const double *A, const double *B, const double *C, int o) {
        const int t = wave + u * W, s = t / 3, kind = t - 3 * s, row = base + nr - 1 - 2 * s;
        const bool kept = s < LS && 2 * s < nr;
        return kind == 2 && s == LS && hasL ? C + (size_t)(base - 1 + a.coff) * bs
               : kind == 2 && kept && s > 0 ? C + (size_t)(row + a.coff) * bs
               : kind == 0 && kept          ? A + (size_t)row * bs
                                            : B + (size_t)(kept && row + o < a.n ? row + o : base) * bs;
    };
    auto offset = [&](int j) {
        const int x = lane + 64 * j, r = x / MT, c = x % MT;
        return (size_t)(r < m ? r : m - 1) * m + (c < m ? c : m - 1);
    };
#pragma unroll
    for (int u = 0; u < TASKS; u++) {
        const double *p = block(u, a.A, a.B, a.C, 0);
#pragma unroll
        for (int j = 0; j < KV; j++) v[u][j] = p[offset(j)];
    }
    const int frow = base + nr - 1 - 2 * fs;
    const bool flive = fs < LS && 2 * fs < nr && fr < m;
    if (flive) fv = a.f[(size_t)frow * m + fr];
    if (a.B2) {
#pragma unroll
        for (int u = 0; u < TASKS; u++) {
            const int t = wave + u * W, s = t / 3, kind = t - 3 * s, row = base + nr - 1 - 2 * s;
            const double *p = block(u, a.B2, a.B2, a.B2, 1);
            if (kind == 1 && s < LS && 2 * s < nr && row + 1 < a.n)
#pragma unroll
                for (int j = 0; j < KV; j++) v[u][j] += p[offset(j)];
        }
        if (flive && frow + 1 < a.n) fv += a.f2[(size_t)(frow + 1) * m + fr];
    }
    auto stage = [&] {
#pragma unroll
        for (int u = 0; u < TASKS; u++) {
            const int t = wave + u * W, s = t / 3, kind = t - 3 * s, row = base + nr - 1 - 2 * s;
            double *dst = kind == 0 ? sm.A[s] : kind == 1 ? sm.B[s] : sm.C[s];
            const bool live = s == LS ? kind == 2 && hasL
                                      : 2 * s < nr && (kind == 1 || (kind == 0 ? row > 0 : s > 0));
            if (s <= LS)
#pragma unroll
                for (int j = 0; j < KV; j++) {
                    const int x = lane + 64 * j, r = x / MT, c = x % MT;
                    dst[r * LD + c] = r < m && c < m ? (live ? v[u][j] : 0.0) : r == c && kind == 1 && s < LS ? 1.0 : 0.0;
                }
        }
        if (fs <= LS) sm.f[fs][fr] = fv;
    };
    if constexpr (H > 1) stage();  // (not beside the first level's rows: they do not both fit the registers)
    auto none = [] {};
    if constexpr (H == 1) cr_levels<H, R, TAIL>(a, sm, base, nr, hasL, stage);
    else cr_levels<H, R, TAIL>(a, sm, base, nr, hasL, none);
    if (nr == 1) __syncthreads();  // (no level did)
    if constexpr (!TAIL) {
        // the reduced row of this chunk, and what it adds to the one before
        const size_t o = blockIdx.x * bs;
        if (wave < 4 && (wave < 2 || hasL)) {
            const double *src = wave == 0 ? sm.A[0] : wave == 1 ? sm.B[0] : wave == 2 ? sm.B[LS] : sm.C[LS];
            double *dst = (wave == 0 ? a.oA : wave == 1 ? a.oB : wave == 2 ? a.odB : a.oC) + o;
            for (int u = lane; u < MT * MT; u += 64) {
                const int r = u / MT, c = u % MT;
                if (r < m && c < m) dst[(size_t)r * m + c] = src[r * LD + c];
            }
            if (wave == 1 && lane < m) a.of[(size_t)blockIdx.x * m + lane] = sm.f[0][lane];
            if (wave == 2 && lane < m) a.odf[(size_t)blockIdx.x * m + lane] = sm.f[LS][lane];
        }
    } else {
        CrBack<H, R> back;
        back.load(a, base, nr);
        if (wave == 0) {
            constexpr int NC = MT + 1;
            double r[H][NC];
            const int i = lane & 15;
            cr_sweep<H, NC>(r, m, a.flag, [&](double (&v)[H][NC], int (&dg)[H]) {
#pragma unroll
                for (int h = 0; h < H; h++) {
                    dg[h] = __double2hiint(sm.B[0][(16 * h + i) * (LD + 1)]);
                    lds_row<MT>(v[h], &sm.B[0][(16 * h + i) * LD]);
                    v[h][MT] = sm.f[0][16 * h + i];
                }
            }, none);
            if (lane < 16)
#pragma unroll
                for (int h = 0; h < H; h++) sm.x[0][16 * h + lane] = r[h][MT];
        } else if (wave == 1 && lane < MT) {
            sm.x[R][lane] = 0.0;  // no row at the left
        }
        __syncthreads();
        back.run(sm.x, nr);
        for (int t = threadIdx.x; t < nr * MT; t += 64 * W) {
            const int d = t / MT, r = t % MT;
            if (r < m) a.x[(size_t)(nr - 1 - d) * m + r] = sm.x[d][r];
        }
    }
}

// Back-substitution of the chunks of one level; xup: the separators' solution.
template <int H, int R> __global__ __launch_bounds__((64 * crc<H, R>::W)) void cr_back_kernel(CrArgs a, const double *xup)
{
    constexpr int MT = 16 * H, W = crc<H, R>::W;
    __shared__ double x[R + 1][MT];
    const int m = a.m, base = blockIdx.x * a.R, nr = min(a.R, a.n - base);
    CrBack<H, R> back;
    back.load(a, base, nr);
    for (int t = threadIdx.x; t < (R + 1) * MT; t += 64 * W) {
        const int d = t / MT, r = t % MT;
        double v = 0.0;
        if (r < m) {
            if (d == 0) v = xup[(size_t)blockIdx.x * m + r];
            else if (d < nr) v = a.x[(size_t)(base + nr - 1 - d) * m + r];
            else if (d == R && base > 0) v = xup[(size_t)(blockIdx.x - 1) * m + r];
        }
        x[d][r] = v;
    }
    __syncthreads();
    back.run(x, nr);
    for (int t = threadIdx.x; t < nr * MT; t += 64 * W) {
        const int d = t / MT, r = t % MT;
        if (r < m) a.x[(size_t)(base + nr - 1 - d) * m + r] = x[d][r];
    }
}

template <int H, bool TAIL> void launch_reduce(int chunks, hipStream_t s, const CrArgs &a)
{
    if constexpr (H == 1) {
        if (a.R > 8)
            hipLaunchKernelGGL((cr_reduce_kernel<H, 32, TAIL>), dim3(chunks), dim3(64 * crc<H, 32>::W), 0, s, a);
        else hipLaunchKernelGGL((cr_reduce_kernel<H, 8, TAIL>), dim3(chunks), dim3(64 * crc<H, 8>::W), 0, s, a);
    } else {
        hipLaunchKernelGGL((cr_reduce_kernel<H, 8, TAIL>), dim3(chunks), dim3(64 * crc<H, 8>::W), 0, s, a);
    }
}
template <int H> void launch_back(int chunks, hipStream_t s, const CrArgs &a, const double *xup)
{
    if constexpr (H == 1) {
        if (a.R > 8)
            hipLaunchKernelGGL((cr_back_kernel<H, 32>), dim3(chunks), dim3(64 * crc<H, 32>::W), 0, s, a, xup);
        else hipLaunchKernelGGL((cr_back_kernel<H, 8>), dim3(chunks), dim3(64 * crc<H, 8>::W), 0, s, a, xup);
    } else {
        hipLaunchKernelGGL((cr_back_kernel<H, 8>), dim3(chunks), dim3(64 * crc<H, 8>::W), 0, s, a, xup);
    }
}

template <int H> int cr_run(const gf_btd &b, hipStream_t s, int *flag, const double *rhs, double *x)
{
    const int m = b.m;
    const size_t bs = b.bsz;
    std::vector<CrArgs> lv;
    int launches = 0, halvings = 0;
    double *w = b.cr_work, halved = 0.0;
    for (int n = b.nblk; n > 16; n /= 2, halvings++) halved += n / 2;  // the probe counts in these (giraffe_amd.h)
    CrArgs a{};
    a.A = (const double *)b.A;
    a.B = (const double *)b.B;
    a.C = (const double *)b.C;
    a.f = rhs;
    a.x = x;
    a.m = m;
    a.flag = flag;
    for (size_t l = 0; l < b.cr_n.size(); l++) {
        const int n = b.cr_n[l], R = b.cr_R[l], nch = (n + R - 1) / R;
        a.n = n;
        a.R = R;
        a.XY = w;
        w += 2 * bs * n;
        const bool last = l + 1 == b.cr_n.size();
        if (!last) {
            a.oA = w;
            a.oB = a.oA + bs * nch;
            a.odB = a.oB + bs * nch;
            a.oC = a.odB + bs * nch;
            a.of = a.oC + bs * nch;
            a.odf = a.of + (size_t)m * nch;
            w = a.odf + 2 * (size_t)m * nch;  // and the next level's x
            const int pr = gf_probe_begin(s, GF_KC_BTD_LEVEL);
            launch_reduce<H, false>(nch, s, a);
            gf_probe_end(s, pr, halved, halvings);
            halved = halvings = 0;
        } else {
            const int pr = gf_probe_begin(s, GF_KC_BTD_TAIL);
            launch_reduce<H, true>(1, s, a);
            gf_probe_end(s, pr, n);
        }
        launches++;
        lv.push_back(a);
        CrArgs nx{};
        nx.A = a.oA;
        nx.B = a.oB;
        nx.B2 = a.odB;
        nx.C = a.oC;
        nx.coff = 1;
        nx.f = a.of;
        nx.f2 = a.odf;
        nx.x = a.odf ? a.odf + (size_t)m * nch : nullptr;
        nx.m = m;
        nx.flag = flag;
        a = nx;
    }
    for (int l = (int)lv.size() - 2; l >= 0; l--) {
        const int nch = (lv[l].n + lv[l].R - 1) / lv[l].R;
        launch_back<H>(nch, s, lv[l], lv[l + 1].x);
        launches++;
    }
    GF_HIP(hipGetLastError());
    return launches;
}

}  // namespace

// Chunk sizes of every level (no device call) and the workspace, in doubles.
// Blocks of up to 16 rows: chunks of 8 (a wavefront per SIMD at most, several
// chunks a CU) while the device has CUs to spare, chunks of 32 (a CU each, fewer
// launches) from 4,096 rows on, and one workgroup for the last 16.  Measured per
// solve, 16-row blocks: 583 rows 64 us in chunks of 8, 72 us in chunks of 32;
// 2,250 rows 83 and 94; 7,500 rows 113 and 109; 15 rows in one workgroup 24 us,
// split once 26; 30 rows 34 and 31.
size_t gf_cr_plan(gf_btd &b, int m, int nblk)
{
    const size_t bs = (size_t)m * m;
    size_t work = 0;
    b.cr_n.clear();
    b.cr_R.clear();
    for (int n = nblk;;) {
        const int rmax = m > 16 ? 8 : n >= 4096 ? 32 : n > 16 ? 8 : 16;
        const int nch = (n + rmax - 1) / rmax, R = (n + nch - 1) / nch;
        b.cr_n.push_back(n);
        b.cr_R.push_back(R);
        work += 2 * bs * n;
        if (nch == 1) break;
        n = (n + R - 1) / R;  // chunks of R rows
        work += (4 * bs + 3 * (size_t)m) * n;
    }
    return work;
}

// x = K^-1 rhs with K = (A, B, C) of b, which stay as they are; x must differ
// from rhs.  Returns the number of launches or a negative status.
int gf_btd_factor_solve(const gf_btd &b, hipStream_t s, int *d_flag, const double *rhs, double *x)
{
    if (rhs == x) {
        gf_set_error("block-tridiagonal factor_solve: x must differ from rhs");
        return GF_E_ARG;
    }
    return b.m <= 16 ? cr_run<1>(b, s, d_flag, rhs, x) : cr_run<2>(b, s, d_flag, rhs, x);
}
