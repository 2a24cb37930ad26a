// gf_btdsystem_noalloc: the block-tridiagonal solve of gf_btdsystem for callers
// that cannot allocate device memory (code under HIP graph capture, tight
// serving loops).  Inputs and outputs are the caller's device buffers, read and
// written in place; the workspace (the eliminated rows' X and Y, the reduced
// rows of each level and their solution) lives in `scratch`, a file-scope device
// array of fixed size that every GPU the library runs on holds until the
// process ends.  Nothing here calls hipMalloc, hipFree or an allocating
// library routine, and nothing waits on the host: the work is enqueued on the
// caller's stream, fills are kernels (no memset nodes in a captured graph).
//
// Every call on one GPU shares that GPU's scratch and leaves its contents
// behind; a call reads nothing there that it has not written.  Calls that overlap on one GPU (other
// streams, other threads) race on the scratch.
#include "gf_internal.h"

#include <mutex>

namespace {

// Capacity: nblk * m * m <= 2^17 block entries (so n = nblk m <= 2^17 rows).
constexpr size_t NA_ELEMS = (size_t)1 << 17;
// X|Y of every row (2 E), then the reduced rows of each level (at most a quarter
// of the rows before): under 2.93 E over all sizes within the capacity.  Then a
// stand-in for a solution or flag that overlaps the inputs (at most E, and a
// line): 4.2 MB in all.
constexpr size_t NA_WORK = 3 * NA_ELEMS, NA_SCRATCH = 4 * NA_ELEMS + 32;

static __device__ __align__(256) double scratch[NA_SCRATCH];

constexpr int NA_MAX_DEV = 64;
std::mutex na_mu;
double *na_ptr[NA_MAX_DEV] = {};

// Device address of this GPU's scratch (hipGetSymbolAddress once per device,
// with that device current); the array's name is a host-side stand-in only.
int scratch_of(int dev, double **out)
{
    if (dev < 0 || dev >= NA_MAX_DEV) {
        gf_set_error("gf_btdsystem_noalloc: device ordinal out of range");
        return GF_E_ARG;
    }
    std::lock_guard<std::mutex> lk(na_mu);
    if (!na_ptr[dev]) {
        void *p = nullptr;
        GF_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        na_ptr[dev] = (double *)p;
    }
    *out = na_ptr[dev];
    return GF_OK;
}

bool overlap(const void *p, size_t np, const void *q, size_t nq)
{
    const char *a = (const char *)p, *b = (const char *)q;
    return a < b + nq && b < a + np;
}

}  // namespace

extern "C" int gf_btdsystem_noalloc(int m, int nblk, const double *A, const double *B, const double *C,
                                    const double *b, double *x, int *info_fail, void *stream)
{
    if (m < 1 || m > 32 || nblk < 1 || !A || !B || !C || !b || !x || !info_fail) return GF_E_ARG;
    if (b == x) {  // (before anything is enqueued: the flag of a refused call is not written)
        gf_set_error("gf_btdsystem_noalloc: x must differ from b");
        return GF_E_ARG;
    }
    if ((size_t)nblk * m * m > NA_ELEMS) {
        gf_set_error("gf_btdsystem_noalloc: nblk * m * m exceeds the scratch capacity of 131072");
        return GF_E_CAPACITY;
    }
    int dev = 0;
    GF_HIP(hipGetDevice(&dev));
    double *sp = nullptr;
    GF_TRY(scratch_of(dev, &sp));
    hipStream_t s = (hipStream_t)stream;
    gf_btd t;
    t.m = m;
    t.nblk = nblk;
    t.bsz = (size_t)m * m;
    t.A = const_cast<double *>(A);
    t.B = const_cast<double *>(B);
    t.C = const_cast<double *>(C);
    t.cr_work = sp;
    if (gf_cr_plan(t, m, nblk) > NA_WORK) {
        gf_set_error("gf_btdsystem_noalloc: scratch layout overflow");
        return GF_E_CAPACITY;
    }
    // the flag and the solution are written while the inputs are still being read:
    // one that overlaps them is kept in the scratch until the end
    const size_t E = (size_t)nblk * t.bsz * 8, n = (size_t)nblk * m * 8;
    auto meets = [&](const void *p, size_t np) {
        return overlap(p, np, A, E) || overlap(p, np, B, E) || overlap(p, np, C, E) || overlap(p, np, b, n);
    };
    double *xs = meets(x, n) ? sp + NA_WORK : x;
    int *flag = meets(info_fail, 4) ? (int *)(sp + NA_WORK + NA_ELEMS) : info_fail;
    GF_TRY(gf_launch_fill_bytes(s, flag, 4));
    const int l = gf_btd_factor_solve(t, s, flag, b, xs);
    if (l < 0) return l;
    if (xs != x) GF_HIP(hipMemcpyAsync(x, xs, n, hipMemcpyDeviceToDevice, s));
    if (flag != info_fail) GF_HIP(hipMemcpyAsync(info_fail, flag, 4, hipMemcpyDeviceToDevice, s));
    return GF_OK;
}
