// ftdma_device.h -- device helpers shared by the kernel sources (internal).
#pragma once

#include <hip/hip_runtime.h>

#include <stddef.h>

namespace ftd {

// para_range over [0, n) in P parts (libs/pascal_tdma/cpu/para_range.cpp:4-9)
__host__ __device__ inline void part_of(int n, int P, int p, int& s, int& m) {
    int base = n / P, rem = n % P;
    s = p * base + (p < rem ? p : rem);
    m = base + (p < rem ? 1 : 0);
}

// float -> int truncation that saturates instead of being undefined, NaN -> 0
__device__ inline long long trunc_sat(double x) {
    if (x != x) return 0;
    if (x >= 2147483647.0) return 2147483647LL;
    if (x <= -2147483648.0) return -2147483648LL;
    return (long long)(int)x;
}

// k_cal_J_rhs_bound's formula (filtered_tdma_kernels.cuh:245-259) with the
// clamp to [0, n_row-1]
__device__ inline int cal_J_gpu(double rho, double max_b, double eps, int n_row) {
    if (rho == 0.0 || rho >= 0.5) return n_row - 1;
    double lambda_p = (1.0 + sqrt(1.0 - 4.0 * rho * rho)) * 0.5;
    double q = rho / lambda_p;
    double Bv = q * (2.0 + q) / ((1.0 - q) * (1.0 - 2.0 * rho)) * max_b;
    long long J = trunc_sat(log(eps / Bv) / log(q)) + 1;
    if (J > n_row - 1) J = n_row - 1;
    if (J < 0) J = 0;
    return (int)J;
}

// max over aligned groups of `width` lanes (width a power of two <= 64)
__device__ inline double group_max(double v, int width) {
    for (int off = width >> 1; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    return v;
}

// Reduced system of NR rows (B == 1) in LDS, row k of this lane's system at
// index k * S, solved by Thomas in place (x to Dr). 4 rows at a time: their
// values are read into registers first and c', d' are carried in registers,
// so the serial chain is the arithmetic, not an LDS round trip per row.
__device__ __forceinline__ void reduced_thomas_lds(double* Ar, double* Cr, double* Dr, int NR,
                                                   int S) {
    double cp = Cr[0], dp = Dr[0];
    int k = 1;
    for (; k + 4 <= NR; k += 4) {
        double ak[4], ck[4], dk[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ak[u] = Ar[(k + u) * S];
            ck[u] = Cr[(k + u) * S];
            dk[u] = Dr[(k + u) * S];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const double inv = 1.0 / (1.0 - ak[u] * cp);
            dp = inv * (dk[u] - ak[u] * dp);
            cp = inv * ck[u];
            Dr[(k + u) * S] = dp;
            Cr[(k + u) * S] = cp;
        }
    }
    for (; k < NR; ++k) {
        const double ak = Ar[k * S];
        const double inv = 1.0 / (1.0 - ak * cp);
        dp = inv * (Dr[k * S] - ak * dp);
        cp = inv * Cr[k * S];
        Dr[k * S] = dp;
        Cr[k * S] = cp;
    }
    double dn = dp;
    k = NR - 2;
    for (; k >= 3; k -= 4) {
        double ck[4], dk[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ck[u] = Cr[(k - u) * S];
            dk[u] = Dr[(k - u) * S];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            dn = dk[u] - ck[u] * dn;
            Dr[(k - u) * S] = dn;
        }
    }
    for (; k >= 0; --k) {
        dn = Dr[k * S] - Cr[k * S] * dn;
        Dr[k * S] = dn;
    }
}

// The periodic reduced system (row 0 coupled to row NR - 1): y to Dr and the
// coefficient e of x_0 to Er for rows 1..NR-1, x_0 to Dr[0] with Er[0] = 0;
// then x_k = y_k + x_0 e_k, which each partition forms for its own two rows.
// The running c, d, e stay in registers.
__device__ __forceinline__ void reduced_cyclic_lds(double* Ar, double* Cr, double* Dr, double* Er,
                                                   int NR, int S) {
    const double e_last = -Cr[(NR - 1) * S];
    double cp = Cr[1 * S], dp = Dr[1 * S], ep = -Ar[1 * S];
    Er[1 * S] = ep;
#pragma unroll 2
    for (int k = 2; k < NR; ++k) {
        const double ak = Ar[k * S];
        const double inv = 1.0 / (1.0 - ak * cp);
        const double ek = (k == NR - 1) ? e_last : 0.0;
        dp = inv * (Dr[k * S] - ak * dp);
        ep = inv * (ek - ak * ep);
        cp = inv * Cr[k * S];
        Dr[k * S] = dp;
        Er[k * S] = ep;
        Cr[k * S] = cp;
    }
    double dn = dp, en = ep;
#pragma unroll 2
    for (int k = NR - 2; k >= 1; --k) {
        const double ck = Cr[k * S];
        dn = Dr[k * S] - ck * dn;
        en = Er[k * S] - ck * en;
        Dr[k * S] = dn;
        Er[k * S] = en;
    }
    const double x0 =
        (Dr[0] - Ar[0] * dp - Cr[0] * Dr[1 * S]) / (1.0 + Ar[0] * ep + Cr[0] * Er[1 * S]);
    Dr[0] = x0;
    Er[0] = 0.0;
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N <= 63, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(3))) double* lds_cdptr_t;

// workgroup barrier for LDS traffic only: the LDS writes are complete, the
// DMAs in flight are left alone (__syncthreads would wait for them as well)
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace ftd
