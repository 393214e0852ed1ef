// ftdma_lines.hip -- the streamed exact solve of long systems (513 to 4096
// rows) over the engine's own partitions, for any number of systems.
//
// The arithmetic is k_pascal_fused's (modified Thomas per partition in
// registers, the reduced system in LDS, the interior update) over a
// global->LDS ring as in k_pascal_stream. A workgroup is 256 lanes: four
// waves, one per SIMD, since 64 rows of a', c', d' fill a lane's registers.
// It holds S systems x Q = 256 / S partitions, so the longer the system, the
// fewer systems of a row it reads together:
//
//   S = 16: up to 1024 rows (Q = 16), 128-byte rows of a tile
//   S =  8: up to 2048 rows (Q = 32),  64-byte
//   S =  4: up to 4096 rows (Q = 64),  32-byte
//
// The whole state of a system stays on the chip between its sweeps: 40 B/row,
// where the lane-per-system Thomas that took such systems moves 72 and runs
// all rows in one chain (4096 x 2048: 1160 us with the operands in the caches,
// 1630 out of them; here 75 and 109). Tiles share cache
// lines below 16 systems, and wherever n_sys is not a multiple of 16, so the
// tiles that run at one time on one XCD are adjacent (xcd_tile), and their
// loads and stores stay in its L2 until the neighbours have used the rest
// of the line; whole-line tiles keep the nontemporal hint (NT). A ring of 4
// row-steps is the fastest for that reason: what is in flight for 32
// neighbouring tiles has to stay in one 4 MB L2 (operands out of the caches,
// 4096 x 2048: 4 / 8 / 16 row-steps 108 / 120 / 124 us; 131072 x 1024: 1115 /
// 1133 / 1208 us). What bounds it: out of the caches, lines fetched by two
// tiles at S < 16 (2.5-3.3 TB/s); at few tiles a lane's chain of divisions, one
// wave per SIMD (1024 x 2048: 35 us in the caches, 47 out of them).
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "ftdma_device.h"
#include "ftdma_kernels.h"
#include "ftdma_xcd.h"

namespace ftd {

namespace {

constexpr int M = 64;        // rows a lane holds
constexpr int R = 4;         // ring depth in row-steps
constexpr int kStep = 2;     // row-steps come in pairs
constexpr int kSlot = 2048;  // bytes of a ring slot: one row-step of a wave
constexpr int kThreads = 256;

typedef double dbl2 __attribute__((ext_vector_type(2)));

// The operands of two row-steps from two ring slots (addresses of this
// lane's a in each: b is 512 bytes on, c and d 1024 and 1536), one wait for
// both. Inline asm for the reason given at k_pascal_stream's ring_read.
__device__ __forceinline__ void slots_read(const uint32_t (&p)[2], dbl2 (&ab)[2], dbl2 (&cd)[2]) {
    asm volatile(
        "ds_read2st64_b64 %0, %4 offset1:1\n\t"
        "ds_read2st64_b64 %1, %4 offset0:2 offset1:3\n\t"
        "ds_read2st64_b64 %2, %5 offset1:1\n\t"
        "ds_read2st64_b64 %3, %5 offset0:2 offset1:3\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(ab[0]), "=&v"(cd[0]), "=&v"(ab[1]), "=&v"(cd[1])
        : "v"(p[0]), "v"(p[1])
        : "memory");
}

// One wave's DMA sources: lane l brings two neighbouring systems of one
// array and partition per block (block 0: A then B, block 1: C then D).
template <int S, int AUX>
struct Feed {
    static constexpr int PW = 64 / S;  // partitions per wave
    const double* src0;
    const double* src1;
    unsigned char* ring;  // this wave's slots
    uint32_t ld;
    int cnt;  // rows of this lane's source partition
    int n_sys, c0;

    __device__ __forceinline__ void init(unsigned char* wave_ring, const double* A,
                                         const double* B, const double* C, const double* D,
                                         int nsys, int n_row, int w, int l) {
        ring = wave_ring;
        ld = (uint32_t)nsys;
        n_sys = nsys;
        const int g = 2 * l / S;  // sub-row: array (g / PW), partition (g % PW)
        int r0;
        part_of(n_row, kThreads / S, w * PW + g % PW, r0, cnt);
        src0 = (g < PW ? A : B) + (size_t)r0 * ld;
        src1 = (g < PW ? C : D) + (size_t)r0 * ld;
        c0 = 2 * l % S;
    }
    // first system of this lane's pair in tile T; past the last pair, the
    // last one (no load leaves its row)
    __device__ __forceinline__ uint32_t col(int T) const {
        const int c = T * S + c0;
        return (uint32_t)(c <= n_sys - 2 ? c : n_sys - 2);
    }
    // row j (clamped to the partition) at column c into slot k
    __device__ __forceinline__ void dma(int j, uint32_t c, int k) const {
        const uint32_t jj = (uint32_t)(j < cnt ? j : cnt - 1);
        const size_t o = (size_t)jj * ld + c;
        unsigned char* const s = ring + k * kSlot;
        __builtin_amdgcn_global_load_lds((const void*)(src0 + o), (lds_ptr_t)s, 16, 0, AUX);
        __builtin_amdgcn_global_load_lds((const void*)(src1 + o), (lds_ptr_t)(s + 1024), 16, 0,
                                         AUX);
    }
};

// The forward sweep of one tile from row-step J0 on, two row-steps at a
// time: modified elimination (rows 0, 1 divided by b) of the rows j < cnt.
// Row j sits in slot (base + j) % R; a step refills its slot with the row R
// steps ahead, the next tile's once this tile's are all requested.
template <int J0>
struct Forward {
    template <int S, int AUX>
    __device__ __forceinline__ static void run(const Feed<S, AUX>& f, int ns, bool first, int cnt,
                                               int base, uint32_t col, uint32_t ncol,
                                               uint32_t lane, double (&a)[M], double (&c)[M],
                                               double (&d)[M], double& aN, double& cN,
                                               double& dN) {
        if (J0 < ns) {
            // Two DMAs per row-step: while either row's are pending, the
            // 2 (R - 2) of the row-steps after them are too (loads complete in
            // order), so vmcnt(2 (R - 2)) means both have landed. Rows below R
            // of a later tile landed before the previous tile's stores. (Past
            // row ns - 1 a slot holds the next tile's first row: read and
            // dropped.)
            if (J0 >= R || first) wait_vmcnt<2 * (R - kStep)>();
            uint32_t p[kStep];
            dbl2 ab[kStep], cd[kStep];
#pragma unroll
            for (int u = 0; u < kStep; ++u) p[u] = lane + (uint32_t)((base + J0 + u) % R * kSlot);
            slots_read(p, ab, cd);
#pragma unroll
            for (int u = 0; u < kStep; ++u) {
                const int j = J0 + u;
                if (u == 0 || j < ns) {
                    const bool own = j + R < ns;
                    f.dma(own ? j + R : j + R - ns, own ? col : ncol, (base + j) % R);
                }
            }
#pragma unroll
            for (int u = 0; u < kStep; ++u) {
                const int j = J0 + u;
                const double aj = ab[u].x, bj = ab[u].y, cj = cd[u].x, dj = cd[u].y;
                if (j < cnt) {
                    if (j < 2) {
                        a[j] = aj / bj;
                        c[j] = cj / bj;
                        d[j] = dj / bj;
                    } else {
                        const double inv = 1.0 / (bj - aj * c[j - 1]);
                        d[j] = inv * (dj - aj * d[j - 1]);
                        c[j] = inv * cj;
                        a[j] = -inv * aj * a[j - 1];
                    }
                    if (j == cnt - 1) {
                        aN = a[j];
                        cN = c[j];
                        dN = d[j];
                    }
                }
            }
            Forward<J0 + kStep>::run(f, ns, first, cnt, base, col, ncol, lane, a, c, d, aN, cN,
                                     dN);
        }
    }
};
template <>
struct Forward<M> {
    template <int S, int AUX>
    __device__ __forceinline__ static void run(const Feed<S, AUX>&, int, bool, int, int, uint32_t,
                                               uint32_t, uint32_t, double (&)[M],
                                               double (&)[M], double (&)[M], double&, double&,
                                               double&) {}
};

// ns: row-steps per tile, the longest partition's rows, odd numbers too, and at
// least R (a tile refills the ring for the next one); at most M. With an odd
// ns the last pair's second read takes the slot that already holds, or will
// hold, the next tile's first row, and drops it; only the first is refilled.
template <int S, bool CYCLIC, bool NT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1))) void k_pascal_lines(
    const double* __restrict__ A, const double* __restrict__ B, const double* __restrict__ C,
    double* D, int n_sys, int n_row, int n_tiles, int ns) {
    constexpr int Q = kThreads / S, NR = 2 * Q, PW = 64 / S;
    __shared__ __attribute__((aligned(16))) unsigned char ring[4][R * kSlot];
    __shared__ double red[CYCLIC ? 4 : 3][NR][S];

    const int t = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l = t & 63;
    const int q = w * PW + l / S;
    const int sl = l % S;
    const size_t ld = (size_t)n_sys;
    Feed<S, NT ? 2 : 0> f;
    f.init(ring[w], A, B, C, D, n_sys, n_row, w, l);
    int r0, cnt0;
    part_of(n_row, Q, q, r0, cnt0);

    // concurrent workgroups of one XCD hold adjacent tiles
    int tile = xcd_tile(blockIdx.x, gridDim.x);
    {
        const uint32_t c = f.col(tile);
#pragma unroll
        for (int j = 0; j < R; ++j) f.dma(j, c, j);
    }
    int slot0 = 0;  // the slot that holds the tile's first row
    bool first = true;
    for (; tile < n_tiles; tile += gridDim.x) {
        // opaque per tile: keeps the row tests from being hoisted out of the
        // tile loop as live values
        int cnt = cnt0;
        asm volatile("" : "+v"(cnt), "+v"(f.cnt));
        const int next = tile + (int)gridDim.x;
        const uint32_t col = f.col(tile), ncol = f.col(next < n_tiles ? next : tile);
        // lanes past the last system repeat it, in every value and store;
        // an odd last system sits second in the pair that ends its rows
        const int i = min(tile * S + sl, n_sys - 1);
        const int at = i - tile * S;
        const int pos = at + (((n_sys & 1) && i == n_sys - 1 && !(at & 1)) ? 1 : 0);
        const uint32_t lane =
            (uint32_t)(uintptr_t)(lds_cdptr_t)(const double*)(ring[w] + 8 * ((l / S) * S + pos));
        const size_t base = (size_t)r0 * ld + (size_t)i;

        double a[M], c[M], d[M];
        double aN = 0.0, cN = 0.0, dN = 0.0;
        Forward<0>::run(f, ns, first, cnt, slot0, col, ncol, lane, a, c, d, aN, cN, dN);
        slot0 = (slot0 + ns) % R;
#pragma unroll
        for (int j = M - 3; j >= 1; --j) {
            if (j <= cnt - 3) {
                const double cj = c[j];
                d[j] = d[j] - cj * d[j + 1];
                a[j] = a[j] - cj * a[j + 1];
                c[j] = -cj * c[j + 1];
            }
        }
        const double r = 1.0 / (1.0 - a[1] * c[0]);
        const double d0 = r * (d[0] - c[0] * d[1]);
        const double a0 = r * a[0];
        const double c0 = -r * c[0] * c[1];

        lds_barrier();  // the previous tile's readers of red[] are done
        red[0][2 * q][sl] = a0;
        red[1][2 * q][sl] = c0;
        red[2][2 * q][sl] = d0;
        red[0][2 * q + 1][sl] = aN;
        red[1][2 * q + 1][sl] = cN;
        red[2][2 * q + 1][sl] = dN;
        lds_barrier();
        if (q == 0) {
            double* Ar = &red[0][0][sl];
            double* Cr = &red[1][0][sl];
            double* Dr = &red[2][0][sl];
            // an opaque count: unrolled whole, its rows would be held beside
            // the partition's
            int nr = NR;
            asm volatile("" : "+s"(nr));
            if constexpr (!CYCLIC)
                reduced_thomas_lds(Ar, Cr, Dr, nr, S);
            else
                reduced_cyclic_lds(Ar, Cr, Dr, &red[3][0][sl], nr, S);
        }
        lds_barrier();
        // the next tile's first rows have landed before this tile's stores
        wait_vmcnt<0>();
        double x0 = red[2][2 * q][sl];
        double xN = red[2][2 * q + 1][sl];
        if constexpr (CYCLIC) {
            // x_k = y_k + x_0 e_k; row 0 of the reduced system is x_0 itself
            const double x0r = red[2][0][sl];
            const double y0 = x0 + x0r * red[3][2 * q][sl];
            xN = xN + x0r * red[3][2 * q + 1][sl];
            x0 = q == 0 ? x0 : y0;
        }
        // rows past m_p store row m_p - 1 (x_N) again
        double* const xlast = D + base + (size_t)(cnt - 1) * ld;
#pragma unroll
        for (int j = 0; j < M; ++j) {
            if (j % kStep == 0 && j >= ns) break;
            double x;
            if (j == 0)
                x = x0;
            else if (j >= cnt - 1)
                x = xN;
            else
                x = d[j] - (a[j] * x0 + c[j] * xN);
            double* const p = j < cnt - 1 ? D + base + (size_t)j * ld : xlast;
            if (NT)
                __builtin_nontemporal_store(x, p);
            else
                *p = x;
        }
        first = false;
    }
    wait_vmcnt<0>();  // no DMA into LDS outlives the wave
}

template <int S, bool CYCLIC, bool NT>
hipError_t launch_t(const double* A, const double* B, const double* C, double* D, int n_sys,
                    int n_row, hipStream_t st) {
    constexpr int Q = kThreads / S;
    const int n_tiles = (n_sys - 1) / S + 1;
    const int m = (n_row + Q - 1) / Q;
    if (n_sys < 2 || m > M || n_row / Q < 3) return hipErrorInvalidValue;
    const int grid =
        resident_grid((const void*)k_pascal_lines<S, CYCLIC, NT>, kThreads, n_tiles);
    hipLaunchKernelGGL((k_pascal_lines<S, CYCLIC, NT>), dim3(grid), dim3(kThreads), 0, st, A, B,
                       C, D, n_sys, n_row, n_tiles, std::max(R, m));
    return hipGetLastError();
}

}  // namespace

int lines_systems(int n_sys, int n_row) {
    return n_sys < 2 || n_row <= 512 ? 0
           : n_row <= 1024           ? 16
           : n_row <= 2048           ? 8
           : n_row <= 4096           ? 4
                                     : 0;
}

hipError_t launch_pascal_lines(int S, const double* A, const double* B, const double* C, double* D,
                               int n_sys, int n_row, int cyclic, hipStream_t st) {
    const bool nt = n_sys % 16 == 0 && S == 16;
#define X(s_, nt_)                                                                            \
    if (S == s_ && nt == nt_)                                                                 \
        return cyclic ? launch_t<s_, true, nt_>(A, B, C, D, n_sys, n_row, st)                 \
                      : launch_t<s_, false, nt_>(A, B, C, D, n_sys, n_row, st);
    X(16, true)
    X(16, false)
    X(8, false)
    X(4, false)
#undef X
    return hipErrorInvalidValue;
}

}  // namespace ftd
