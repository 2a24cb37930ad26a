// Index arithmetic of the tangent's storage.  Host and device, and free of HIP
// headers, so that it can be checked on the host at sizes no test would allocate.
#pragma once
#include <cstddef>

#ifdef __HIPCC__
#define GF_HD __host__ __device__ __forceinline__
#else
#define GF_HD inline
#endif

// GM_BTD : block-tridiagonal blocks A (sub), B (diag), C (super), [nblk][m][m]
//          row-major, consecutive in one allocation (B = A + nblk m m,
//          C = B + nblk m m); used when the half-bandwidth fits a block of m <= 32.
// GM_BAND: skewed dense band, entry (i, c) with -hb <= c - i <= ku at
//          ab[i * ld + c + hb], ld = hb + ku (each row a contiguous window of
//          ld + 1); ku = gf_band_ku(hb) leaves room for the factorisation's
//          fill.  Sub-matrices inside the band are plain strided matrices with
//          leading dimension ld, which is what the band LU tiles use.
enum { GM_BTD = 0, GM_BAND = 1 };
struct gf_gmat {
    int layout;
    int m;
    double *A, *B, *C;
    double *ab;
    int hb;
    int ld;
};

// Block index q = floor(x / m) for 0 <= x < 2^24 and m <= 32, through a float
// product (one rounding, then one correction step each way): no integer divide.
GF_HD int gm_block_of(int x, int m, float inv_m)
{
    int q = (int)(((float)x + 0.5f) * inv_m);
    q -= q * m > x ? 1 : 0;
    q += (q + 1) * m <= x ? 1 : 0;
    return q;
}

// Addresses of N entries (R, Cc); a constrained entry (R or Cc negative) gets a
// valid stand-in address whose value is never stored back.  The layout test is
// one uniform branch around the whole batch, so loads through the addresses are
// straight-line code and all in flight together.
template <int N> GF_HD void gm_addr_n(const gf_gmat &g, const int (&R)[N], const int (&Cc)[N], double *(&p)[N])
{
    if (g.layout == GM_BTD) {
        const int m = g.m;
        const float inv_m = 1.0f / (float)m;
        const ptrdiff_t stride = g.B - g.A;
#pragma unroll
        for (int k = 0; k < N; k++) {
            const bool ok = R[k] >= 0 && Cc[k] >= 0;
            const int r = ok ? R[k] : 0, c = ok ? Cc[k] : 0;
            const int bi = gm_block_of(r, m, inv_m), bj = gm_block_of(c, m, inv_m);
            const size_t off = ((size_t)bi * m + (r - bi * m)) * m + (c - bj * m);
            // A, B and C are one allocation in that order (gf_btd_alloc): the block
            // kind selects an offset; a selected pointer would be re-read from the
            // kernel arguments, one dependent load per entry
            const ptrdiff_t kind = bj < bi ? 0 : (bj == bi ? 1 : 2);
            p[k] = g.A + kind * stride + off;
        }
    } else {
#pragma unroll
        for (int k = 0; k < N; k++) {
            const bool ok = R[k] >= 0 && Cc[k] >= 0;
            const int r = ok ? R[k] : 0, c = ok ? Cc[k] : 0;
            p[k] = g.ab + (size_t)r * (size_t)g.ld + (size_t)(c + g.hb);
        }
    }
}

// The same for the 36 entries (R[i], C[j]) of a node pair that a kernel keeps from
// their loads to their stores: entry (i, j) is gm_base(g)[row[i] + step[6 i + j]].
// A band may hold more than 2^32 entries (its size has no bound but memory), so the
// rows' positions take 64 bits; a step stays inside a row's window of ld + 1 entries
// or, in the block-tridiagonal form (rows below 2^24, blocks of up to 32), below
// 2 (B - A) + 32 <= 2^30 + 32.  A constrained row stands at row 0, a constrained
// column on the diagonal.
GF_HD double *gm_base(const gf_gmat &g) { return g.layout == GM_BTD ? g.A : g.ab; }
GF_HD void gm_pair(const gf_gmat &g, const int (&R)[6], const int (&C)[6], size_t (&row)[6], unsigned (&step)[36])
{
    if (g.layout == GM_BTD) {
        const int m = g.m;
        const float inv_m = 1.0f / (float)m;
        const unsigned stride = (unsigned)(g.B - g.A);
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int r = R[i] >= 0 ? R[i] : 0, bi = gm_block_of(r, m, inv_m);
            row[i] = (size_t)r * m;
#pragma unroll
            for (int j = 0; j < 6; j++) {
                const int c = R[i] >= 0 && C[j] >= 0 ? C[j] : r, bj = gm_block_of(c, m, inv_m);
                step[6 * i + j] = (bj < bi ? 0u : bj == bi ? stride : 2 * stride) + (unsigned)(c - bj * m);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int r = R[i] >= 0 ? R[i] : 0;
            row[i] = (size_t)r * ((size_t)g.ld + 1);
#pragma unroll
            for (int j = 0; j < 6; j++)
                step[6 * i + j] = (unsigned)((R[i] >= 0 && C[j] >= 0 ? C[j] : r) - r + g.hb);
        }
    }
}

// Entry (i, j) of a front with rows of mp entries: 64 bits, as fronts of more than
// 23,170 rows pass 4 GB (forced multifrontal plans of meshes whose coordinates do not
// separate them) and of more than 65,535 rows 2^32 entries.
GF_HD size_t gf_front_at(int i, int j, int mp) { return (size_t)i * (size_t)mp + (size_t)j; }
