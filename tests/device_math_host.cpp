// The scalar device arithmetic of compas_amd/csrc (cmp_device.hpp, the index helpers of cmp_kernels.hpp) compiled for
// the host, for tests/test_device_math.py. The two hardware approximations it starts from are replaced by the exact value
// with a relative error of the caller's, so that their whole error bound can be covered.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>

#include <hip/hip_runtime.h>

using std::max;
using std::min;

static double rcp_error = 0.0, rsq_error = 0.0;
static double __builtin_amdgcn_rcp(double d) { return (1.0 / d) * (1.0 + rcp_error); }
static double __builtin_amdgcn_rsq(double d) { return (1.0 / std::sqrt(d)) * (1.0 + rsq_error); }
static void __builtin_amdgcn_sched_barrier(int) {}
static uint64_t bits(double d)
{
    uint64_t u;
    std::memcpy(&u, &d, 8);
    return u;
}
static int __double2hiint(double d) { return (int)(bits(d) >> 32); }
static int __double2loint(double d) { return (int)bits(d); }
static double __hiloint2double(int h, int l)
{
    const uint64_t u = ((uint64_t)(uint32_t)h << 32) | (uint32_t)l;
    double d;
    std::memcpy(&d, &u, 8);
    return d;
}

static double __shfl_xor(double v, int, int) { return v; }
static const dim3 blockIdx, threadIdx;

#include "../compas_amd/csrc/cmp_device.hpp"
#include "../compas_amd/csrc/cmp_kernels.hpp"

extern "C" {
void host_errors(double rcp, double rsq) { rcp_error = rcp; rsq_error = rsq; }
void host_quot(long n, const double* a, const double* b, double* q)
{
    for (long i = 0; i < n; ++i) q[i] = cmp::quot(a[i], b[i]);
}
void host_sqrt(long n, const double* a, double* r)
{
    for (long i = 0; i < n; ++i) r[i] = cmp::sqrt_fast(a[i]);
}
// v: n stencils of six cells; L, R: the states of the face in their middle
void host_weno5_faces(long n, const double* v, double* L, double* R)
{
    for (long i = 0; i < n; ++i) {
        auto s = [&](int t, int) { return v[6 * i + t]; };
        cmp::weno5_faces<0, 0>(s, L + i, R + i);
    }
}
// the offset between cells (i, j, k) and (i + d[0], j + d[1], k + d[2]) of a fab with rows of sj and planes of sk
// cells: by the staging's step, and by the cells' own indices
void host_fab_step(long long sj, long long sk, const int* c, const int* d, long long* step, long long* index)
{
    cmp::BoxDev bx{};
    bx.sj = sj;
    bx.sk = sk;
    *step = sk ? cmp::fab_step<3>(bx, d[0], d[1], d[2]) : cmp::fab_step<2>(bx, d[0], d[1], 0);
    *index = cmp::fab_index(bx, c[0] + d[0], c[1] + d[1], c[2] + d[2]) - cmp::fab_index(bx, c[0], c[1], c[2]);
}
// one side at a time (the N-phase model)
void host_weno5(long n, const double* v, double* L, double* R)
{
    for (long i = 0; i < n; ++i) {
        const double* s = v + 6 * i;
        L[i] = cmp::weno5<1>(s[0], s[1], s[2], s[3], s[4]);
        R[i] = cmp::weno5<-1>(s[1], s[2], s[3], s[4], s[5]);
    }
}
}
