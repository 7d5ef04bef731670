// Quotients by the shared reciprocal (Recip, rdiv) on the operands where a
// reciprocal that is not the nearest double could give another quotient than
// the division: prints the denominators and pairs enumerated, the pairs that a
// wrongly rounded reciprocal gets wrong (host), and those the device gets wrong.
//
// With D, N in [2^52, 2^53) the quotient of the last step is
// RN(n/d + (n/d - q0)(D y - 1)), and n/d is at least 1/(2D) ulp from a rounding
// boundary M.  A correctly rounded y has |D y - 1| <= D 2^-106, which is too
// little to cross it.  A y within x ulp of 1/D before its rounding is the other
// neighbour only where 1/D lies within x of the middle between two doubles, and
// then the boundary is crossed only if N 2^53 (or 2^54) - D M = +-1 and
// D >= 2^53 (1 - x): D = 2^53 - j with odd j <= 2^53 x and j^2 2^-54 + ... within x
// of an integer.  Enumerated for x = 2^-15: what one cubic step from v_rcp's 2^-23
// would need; recip takes two Newton steps, whose x is below 2^-39.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "swe_core.hpp"

using namespace rk;
typedef unsigned __int128 u128;

__global__ void k_quotients(const double* n, const double* d, double* q, double* p, int count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) { q[i] = rdiv<false>(n[i], recip(d[i])); p[i] = n[i] / d[i]; }
}

// The neighbour of 1/D in doubles that is farther from it, and the nearer one.
static void reciprocals(uint64_t D, double& near_, double& far_) {
    const double d = (double)D;
    near_ = 1.0 / d;
    const double r = std::fma(-d, near_, 1.0);   // sign of 1/d - near_
    far_ = r > 0.0 ? std::nextafter(near_, 1.0) : std::nextafter(near_, 0.0);
}

static double with(double n, double d, double y) {
    const double q0 = n * y;
    return std::fma(-std::fma(d, q0, -n), y, q0);
}

int main() {
    std::vector<double> n, d;
    long long denominators = 0, wrong_far = 0;
    const u128 P106 = (u128)1 << 106;
    auto visit = [&](uint64_t j) {
        const uint64_t D = (1ull << 53) - j;
        const uint64_t Q = (uint64_t)((P106 / D) & 1), R = (uint64_t)(P106 % D);
        const uint64_t off = Q ? R : D - R;              // 2^106 / D from an odd integer, times D
        if (off > (D >> 14)) return;
        ++denominators;
        uint64_t inv = D;
        for (int k = 0; k < 6; ++k) inv *= 2 - D * inv;   // 1/D modulo 2^64
        double y0, y1;
        reciprocals(D, y0, y1);
        for (int sign = -1; sign <= 1; sign += 2)
            for (int sh = 53; sh <= 54; ++sh) {
                uint64_t M = (sign < 0 ? inv : (uint64_t)0 - inv) & ((1ull << sh) - 1);
                if (sh == 53) M += 1ull << 53;
                const u128 p = (u128)D * M;
                const uint64_t N = (uint64_t)((sign < 0 ? p - 1 : p + 1) >> sh);
                if (M < (1ull << 53) || N < (1ull << 52) || N >= (1ull << 53) || (sh == 53) != (N >= D)) continue;
                n.push_back((double)N);
                d.push_back((double)D);
                const double q = (double)N / (double)D;
                if (with((double)N, (double)D, y0) != q) { printf("nearest reciprocal wrong\n"); return; }
                wrong_far += with((double)N, (double)D, y1) != q;
            }
    };
    for (uint64_t j = 1; j < (1ull << 20); j += 2) visit(j);
    uint64_t done = 1ull << 20;
    for (uint64_t T = 0; T < (1ull << 22); ++T) {
        const long double t = (long double)T, c = 4503599627370496.0L;   // 2^52 z^2 / (1 - z) = T, z = j 2^-53
        const long double z = 2.0L * t / (t + sqrtl(t * t + 4.0L * c * t) + 1e-300L);
        const long double jc = z * 9007199254740992.0L;
        if (jc < 1.0L) continue;
        const long double w = 0x1p-14L * 9007199254740992.0L / jc + 6.0L;
        uint64_t lo = jc > w ? (uint64_t)(jc - w) : 1;
        const uint64_t hi = (uint64_t)(jc + w);
        if (lo < done) lo = done;
        for (uint64_t j = lo | 1; j <= hi && j < (1ull << 38); j += 2) visit(j);
        if (hi + 1 > done) done = hi + 1;
    }
    printf("denominators %lld pairs %zu wrong_with_the_other_neighbour %lld\n", denominators, n.size(), wrong_far);
    int devices = 0;
    if (hipGetDeviceCount(&devices) != hipSuccess || devices == 0) return 0;
    const int count = (int)n.size();
    double *dn, *dd, *dq, *dp;
    std::vector<double> a(count), b(count), q(count), p(count);
    if (hipMalloc((void**)&dn, count * 8) != hipSuccess || hipMalloc((void**)&dd, count * 8) != hipSuccess ||
        hipMalloc((void**)&dq, count * 8) != hipSuccess || hipMalloc((void**)&dp, count * 8) != hipSuccess)
        return 1;
    for (int e : {-72, -53, -52, -40, -13}) {   // denominators from 2^-19 to 2^40
        for (int i = 0; i < count; ++i) { a[i] = std::ldexp(n[i], -50); b[i] = std::ldexp(d[i], e); }
        if (hipMemcpy(dn, a.data(), count * 8, hipMemcpyHostToDevice) != hipSuccess) return 1;
        if (hipMemcpy(dd, b.data(), count * 8, hipMemcpyHostToDevice) != hipSuccess) return 1;
        hipLaunchKernelGGL(k_quotients, dim3((count + 255) / 256), dim3(256), 0, 0, dn, dd, dq, dp, count);
        if (hipMemcpy(p.data(), dp, count * 8, hipMemcpyDeviceToHost) != hipSuccess) return 1;
        if (hipMemcpy(q.data(), dq, count * 8, hipMemcpyDeviceToHost) != hipSuccess) return 1;
        long long wrong = 0, division = 0;
        for (int i = 0; i < count; ++i) {
            wrong += q[i] != p[i];
            division += p[i] != a[i] / b[i];
            if (p[i] != a[i] / b[i] && e == -53)
                printf("the device's division: %a / %a = %a, nearest %a\n", a[i], b[i], p[i], a[i] / b[i]);
        }
        printf("device exponent %d wrong %lld (the device's division against the nearest double: %lld)\n", e, wrong, division);
    }
    return 0;
}
