// FP64 fused multiply-adds whose first factor comes from one lane of the
// reader's own 16-lane DPP row (v_fmac_f64 with row_newbcast), on gfx950: the
// register-resident eliminations keep one matrix row per lane and take the
// pivot row's entry, or the other factor's row, in the multiply-add itself.
// The compiler emits a v_mov_b64_dpp and a v_fma_f64 for the same expression
// (twice the issue slots: these loops are issue-bound), so the groups below
// are written out.
//
// A DPP source may not be written by a VALU instruction in the two wait states
// before it is read.  Every group starts with s_nop 1 and reads through DPP
// only registers that no instruction of the group has written before, so it is
// safe wherever the compiler schedules it.
#pragma once
#include "gf_internal.h"

namespace {

#define GF_NB(d, s, m, k) "v_fmac_f64_dpp " d ", " s ", " m " row_newbcast:" k " row_mask:0xf bank_mask:0xf\n\t"

// v from lane K of the lane's DPP row
template <int K> __device__ __forceinline__ double nb_get(double v)
{
    double r;
    asm("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(v), "n"(K));
    return r;
}

// r[i] += r[i](lane K) h, N entries from r[0]
template <int K> __device__ __forceinline__ void nb_self1(double *r, double h)
{
    asm("s_nop 1\n\t" GF_NB("%0", "%0", "%1", "%2") : "+&v"(r[0]) : "v"(h), "n"(K));
}
template <int K> __device__ __forceinline__ void nb_self4(double *r, double h)
{
    asm("s_nop 1\n\t" GF_NB("%0", "%0", "%4", "%5") GF_NB("%1", "%1", "%4", "%5") GF_NB("%2", "%2", "%4", "%5")
            GF_NB("%3", "%3", "%4", "%5")
        : "+&v"(r[0]), "+&v"(r[1]), "+&v"(r[2]), "+&v"(r[3])
        : "v"(h), "n"(K));
}
template <int K> __device__ __forceinline__ void nb_self8(double *r, double h)
{
    asm("s_nop 1\n\t" GF_NB("%0", "%0", "%8", "%9") GF_NB("%1", "%1", "%8", "%9") GF_NB("%2", "%2", "%8", "%9")
            GF_NB("%3", "%3", "%8", "%9") GF_NB("%4", "%4", "%8", "%9") GF_NB("%5", "%5", "%8", "%9")
                GF_NB("%6", "%6", "%8", "%9") GF_NB("%7", "%7", "%8", "%9")
        : "+&v"(r[0]), "+&v"(r[1]), "+&v"(r[2]), "+&v"(r[3]), "+&v"(r[4]), "+&v"(r[5]), "+&v"(r[6]), "+&v"(r[7])
        : "v"(h), "n"(K));
}
template <int K, int N> __device__ __forceinline__ void nb_self(double *r, double h)
{
    if constexpr (N >= 8) {
        nb_self8<K>(r, h);
        nb_self<K, N - 8>(r + 8, h);
    } else if constexpr (N >= 4) {
        nb_self4<K>(r, h);
        nb_self<K, N - 4>(r + 4, h);
    } else if constexpr (N >= 1) {
        nb_self1<K>(r, h);
        nb_self<K, N - 1>(r + 1, h);
    }
}

// d[i] += s[i](lane K) h, N entries
template <int K> __device__ __forceinline__ void nb_from1(double *d, const double *s, double h)
{
    asm("s_nop 1\n\t" GF_NB("%0", "%1", "%2", "%3") : "+&v"(d[0]) : "v"(s[0]), "v"(h), "n"(K));
}
template <int K> __device__ __forceinline__ void nb_from4(double *d, const double *s, double h)
{
    asm("s_nop 1\n\t" GF_NB("%0", "%4", "%8", "%9") GF_NB("%1", "%5", "%8", "%9") GF_NB("%2", "%6", "%8", "%9")
            GF_NB("%3", "%7", "%8", "%9")
        : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2]), "+&v"(d[3])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]), "v"(h), "n"(K));
}
template <int K, int N> __device__ __forceinline__ void nb_from(double *d, const double *s, double h)
{
    if constexpr (N >= 4) {
        nb_from4<K>(d, s, h);
        nb_from<K, N - 4>(d + 4, s + 4, h);
    } else if constexpr (N >= 1) {
        nb_from1<K>(d, s, h);
        nb_from<K, N - 1>(d + 1, s + 1, h);
    }
}

// d[c] += sum over k = K .. K + 3 of m[k - K] s[c](lane k), N columns
template <int K> __device__ __forceinline__ void nb_mac4_1(double *d, const double *s, const double (&m)[4])
{
    asm("s_nop 1\n\t" GF_NB("%0", "%1", "%2", "%6") GF_NB("%0", "%1", "%3", "%7") GF_NB("%0", "%1", "%4", "%8")
            GF_NB("%0", "%1", "%5", "%9")
        : "+&v"(d[0])
        : "v"(s[0]), "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "n"(K), "n"(K + 1), "n"(K + 2), "n"(K + 3));
}
template <int K> __device__ __forceinline__ void nb_mac4_2(double *d, const double *s, const double (&m)[4])
{
    asm("s_nop 1\n\t" GF_NB("%0", "%2", "%4", "%8") GF_NB("%1", "%3", "%4", "%8") GF_NB("%0", "%2", "%5", "%9")
            GF_NB("%1", "%3", "%5", "%9") GF_NB("%0", "%2", "%6", "%10") GF_NB("%1", "%3", "%6", "%10")
                GF_NB("%0", "%2", "%7", "%11") GF_NB("%1", "%3", "%7", "%11")
        : "+&v"(d[0]), "+&v"(d[1])
        : "v"(s[0]), "v"(s[1]), "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "n"(K), "n"(K + 1), "n"(K + 2), "n"(K + 3));
}
template <int K> __device__ __forceinline__ void nb_mac4_4(double *d, const double *s, const double (&m)[4])
{
#define GF_NB4(mm, kk) \
    GF_NB("%0", "%4", mm, kk) GF_NB("%1", "%5", mm, kk) GF_NB("%2", "%6", mm, kk) GF_NB("%3", "%7", mm, kk)
    asm("s_nop 1\n\t" GF_NB4("%8", "%12") GF_NB4("%9", "%13") GF_NB4("%10", "%14") GF_NB4("%11", "%15")
        : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2]), "+&v"(d[3])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]), "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "n"(K), "n"(K + 1),
          "n"(K + 2), "n"(K + 3));
#undef GF_NB4
}
template <int K, int N> __device__ __forceinline__ void nb_mac4(double *d, const double *s, const double (&m)[4])
{
    if constexpr (N >= 4) {
        nb_mac4_4<K>(d, s, m);
        nb_mac4<K, N - 4>(d + 4, s + 4, m);
    } else if constexpr (N >= 2) {
        nb_mac4_2<K>(d, s, m);
        nb_mac4<K, N - 2>(d + 2, s + 2, m);
    } else if constexpr (N == 1) {
        nb_mac4_1<K>(d, s, m);
    }
}

// One pivot of a sweep whose rows are the lanes: r[i] += r[i](lane K) h for N
// columns, with the next pivot (column r[0], lane (K + 1) % 16) formed among
// them: a wavefront issues in order, so the pivot's dependent instructions are
// placed between the multiply-adds that do not need them.  Out: the next pivot
// p, its reciprocal ip (hardware estimate of 24 bits or more and one cubic step:
// within an ulp), g = -r[0] ip, and the lanes where |r[0]| > 16 |p|.
#define GF_F(i) GF_NB("%[r" #i "]", "%[r" #i "]", "%[h]", "%[k]")
#define GF_R(i) [r##i] "+&v"(r[i])
#define GF_PMOV "v_mov_b64_dpp %[p], %[r0] row_newbcast:%[k1] row_mask:0xf bank_mask:0xf\n\t"
#define GF_PRCP "v_rcp_f64 %[ip], %[p]\n\tv_ldexp_f64 %[t], |%[p]|, 4\n\t"
#define GF_PCMP "v_cmp_gt_f64 %[lg], |%[r0]|, %[t]\n\t"
#define GF_PE1 "v_fma_f64 %[t], -%[p], %[ip], 1.0\n\t"
#define GF_PE2 "v_fma_f64 %[t], %[t], %[t], %[t]\n\t"
#define GF_PE3 "v_fma_f64 %[ip], %[ip], %[t], %[ip]\n\t"
#define GF_PG "v_mul_f64 %[g], -%[r0], %[ip]"
#define GF_PG_NL GF_PG "\n\t"
#define GF_POUT [p] "=&v"(p), [ip] "=&v"(ip), [t] "=&v"(t), [g] "=&v"(g), [lg] "=&s"(larger)
#define GF_PIN : [h] "v"(h), [k] "n"(K), [k1] "n"((K + 1) & 15)
template <int K, int N>
__device__ __forceinline__ void nb_pivot(double *r, double h, double &p, double &ip, double &g,
                                         unsigned long long &larger)
{
    double t;
    static_assert(N >= 2 && N <= 24, "columns of a pivot");
    if constexpr (N == 2)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) "s_nop 1\n\t" GF_PMOV GF_PRCP GF_PCMP GF_PE1 GF_PE2 GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_POUT GF_PIN);
    else if constexpr (N == 3)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_PRCP GF_PCMP GF_PE1 GF_PE2 GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_POUT GF_PIN);
    else if constexpr (N == 4)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_PRCP GF_PCMP GF_PE1 GF_PE2 GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_POUT GF_PIN);
    else if constexpr (N == 5)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_PCMP GF_PE1 GF_PE2 GF_PE3
            GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_POUT GF_PIN);
    else if constexpr (N == 6)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_PE1
            GF_PE2 GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_POUT GF_PIN);
    else if constexpr (N == 7)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_PE2 GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_POUT GF_PIN);
    else if constexpr (N == 8)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_PE2 GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_POUT GF_PIN);
    else if constexpr (N == 9)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_POUT
              GF_PIN);
    else if constexpr (N == 10)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_POUT GF_PIN);
    else if constexpr (N == 11)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_POUT GF_PIN);
    else if constexpr (N == 12)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_POUT GF_PIN);
    else if constexpr (N == 13)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_POUT GF_PIN);
    else if constexpr (N == 14)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_POUT GF_PIN);
    else if constexpr (N == 15)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_POUT GF_PIN);
    else if constexpr (N == 16)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_POUT GF_PIN);
    else if constexpr (N == 17)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15) GF_F(16)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_R(16), GF_POUT GF_PIN);
    else if constexpr (N == 18)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15) GF_F(16) GF_F(17)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_R(16), GF_R(17), GF_POUT GF_PIN);
    else if constexpr (N == 19)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15) GF_F(16) GF_F(17) GF_F(18)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_R(16), GF_R(17), GF_R(18),
              GF_POUT GF_PIN);
    else if constexpr (N == 20)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15) GF_F(16) GF_F(17) GF_F(18) GF_F(19)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_R(16), GF_R(17), GF_R(18),
              GF_R(19), GF_POUT GF_PIN);
    else if constexpr (N == 21)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15) GF_F(16) GF_F(17) GF_F(18) GF_F(19) GF_F(20)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_R(16), GF_R(17), GF_R(18),
              GF_R(19), GF_R(20), GF_POUT GF_PIN);
    else if constexpr (N == 22)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15) GF_F(16) GF_F(17) GF_F(18) GF_F(19) GF_F(20) GF_F(21)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_R(16), GF_R(17), GF_R(18),
              GF_R(19), GF_R(20), GF_R(21), GF_POUT GF_PIN);
    else if constexpr (N == 23)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15) GF_F(16) GF_F(17) GF_F(18) GF_F(19) GF_F(20) GF_F(21) GF_F(22)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_R(16), GF_R(17), GF_R(18),
              GF_R(19), GF_R(20), GF_R(21), GF_R(22), GF_POUT GF_PIN);
    else if constexpr (N == 24)
        asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) GF_PRCP GF_F(5) GF_PCMP GF_F(6)
            GF_PE1 GF_F(7) GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
            GF_F(15) GF_F(16) GF_F(17) GF_F(18) GF_F(19) GF_F(20) GF_F(21) GF_F(22) GF_F(23)
            : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9),
              GF_R(10), GF_R(11), GF_R(12), GF_R(13), GF_R(14), GF_R(15), GF_R(16), GF_R(17), GF_R(18),
              GF_R(19), GF_R(20), GF_R(21), GF_R(22), GF_R(23), GF_POUT GF_PIN);
}
// The same for 15 columns without the compare.
template <int K> __device__ __forceinline__ void nb_pivot15(double *r, double h, double &ip, double &g)
{
    double p, t;
    asm("s_nop 1\n\t" GF_F(0) GF_F(1) GF_F(2) GF_PMOV GF_F(3) GF_F(4) "v_rcp_f64 %[ip], %[p]\n\t" GF_F(5) GF_F(6)
            GF_F(7) GF_PE1 GF_F(8) GF_PE2 GF_F(9) GF_F(10) GF_PE3 GF_F(11) GF_F(12) GF_PG_NL GF_F(13) GF_F(14)
        : GF_R(0), GF_R(1), GF_R(2), GF_R(3), GF_R(4), GF_R(5), GF_R(6), GF_R(7), GF_R(8), GF_R(9), GF_R(10),
          GF_R(11), GF_R(12), GF_R(13), GF_R(14), [p] "=&v"(p), [ip] "=&v"(ip), [t] "=&v"(t), [g] "=&v"(g) GF_PIN);
}
#undef GF_F
#undef GF_R
#undef GF_PMOV
#undef GF_PRCP
#undef GF_PCMP
#undef GF_PE1
#undef GF_PE2
#undef GF_PE3
#undef GF_PG
#undef GF_PG_NL
#undef GF_POUT
#undef GF_PIN

#undef GF_NB

// Lanes i == K of every DPP row, as a wavefront mask.  Formed in place by one
// scalar instruction: as a compare or a constant the compiler keeps all sixteen,
// which the scalar registers do not hold.
template <int K> __device__ __forceinline__ unsigned long long lanes_at()
{
    unsigned long long v;
    asm volatile("s_lshl_b64 %0, %1, %2" : "=s"(v) : "s"(0x0001000100010001ull), "n"(K) : "scc");
    return v;
}

}  // namespace
