// Register-resident red-black SOR sweeps for gfx950 (CDNA4).
//
// A block of NW wavefronts holds a 128-column tile of chi and B, its halo
// included, in registers: lane l has columns 2l and 2l + 1 of R consecutive
// rows, so a half sweep's cells of one row are one value per lane, their
// north and south neighbours are the same lane's values of the rows beside,
// one of the east and west neighbours is the lane's own other column and the
// other is one DPP shift away.  LDS carries only the rows on either side of a
// wavefront boundary, and the per-row coefficients are wave-uniform scalars.
#pragma once
#include <type_traits>
#include <utility>

#include "swm_kernels.h"

namespace swm {

// Per-cell code of the sweeps: ov | ov(i,j+1) << 1 | (ou(i+1,j) + ou) << 2 |
// ou(i+1,j) << 4 | ou << 5 | ocean eta << 6; the low four bits index c5.
enum : int { SC_OV = 0, SC_OVN = 1, SC_OUE = 4, SC_OU = 5, SC_OE = 6, SC_PLAIN = 0x7b };

__global__ void __launch_bounds__(256) sor_code_kernel(int Nx, int Ny, int P, const uint8_t* mask, uint8_t* code) {
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long)Nx * Ny) return;
    const int j = (int)(idx / Nx), i = (int)(idx - (long)j * Nx);
    const int ip = i + 1 == Nx ? 0 : i + 1, jp = j + 1 == Ny ? 0 : j + 1;
    const int m = mask[(size_t)j * P + i], me = mask[(size_t)j * P + ip], mn = mask[(size_t)jp * P + i];
    const int oue = (me >> 1) & 1, ou = (m >> 1) & 1, ovn = (mn >> 2) & 1, ov = (m >> 2) & 1;
    code[(size_t)j * P + i] = (uint8_t)(ov << SC_OV | ovn << SC_OVN | (oue + ou) << 2 | oue << SC_OUE | ou << SC_OU |
                                        ((m & OC_E) ? 1 << SC_OE : 0));
}

constexpr int kSorMaxSweeps = 4;   // sweeps of one launch, at most
constexpr int kSorPad = 16;        // rows of the coefficient tables before row 0 (and, with the tallest tile, past Ny)

template <typename T>
struct SorRowsArgs {
    int Nx, Ny, P;
    int H, nsw;                 // halo cells (2 x the sweeps a launch may do); sweeps of this launch
    int ntx, ntile;             // tile columns, tiles
    int dead_x, dead_y;         // odd extent closed at its seam: cells past it are never updated
    const T* B;
    const uint8_t* code;        // sor_code_kernel
    const T* rowc;              // [row][8]: c1, c3, c4, c5 and 1/c5 of an all-ocean cell, from row -kSorPad on
    const T* c5;                // [row][12][2]: c5, 1/c5 by the code's low four bits, from row -kSorPad on
    const double* relax;        // omega per half sweep (reference mode), clamped at nrelax
    int nrelax, sweep;          // sweep: the launch's first sweep (from 1)
    double omega;               // fixed omega when relax == nullptr
    int residual_mode;          // 0: sum res^2 (reference), 1: sum (L chi - B)^2
    int test, prev_test;        // bit q: the q-th sweep of this / the previous launch is tested
    double* partial;            // [nsw][ntile] sums over the tested sweeps
    const double* prev_partial;
    int prev_sweep;             // first sweep of the previous launch
    double eps, bnorm;
    int* done;
    long long* iters;
    double* norm_out;
};

// The tests of the previous launch's sweeps, in order, by one block of NT
// threads: the partial sums are added in a fixed order; the first norm below
// eps sets *done.  *iters and *norm_out hold the last sweep tested.
template <int NT>
__device__ __forceinline__ void sor_tests(const double* partial, int n, int test, int sweep, double eps, double bnorm,
                                          int mode, int* done, long long* iters, double* norm_out) {
    __shared__ double red[NT / 64];
    __shared__ int pass;
    if (*done) return;
    for (int q = 0; q < kSorMaxSweeps; ++q) {
        if (!((test >> q) & 1)) continue;
        double acc = 0.0;
        for (int b = threadIdx.x; b < n; b += NT) acc += partial[(size_t)q * n + b];
        for (int s = 32; s >= 1; s >>= 1) acc += __shfl_xor(acc, s, 64);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
        __syncthreads();
        if (threadIdx.x == 0) {
            double nrm = red[0];
            for (int w = 1; w < NT / 64; ++w) nrm += red[w];
            nrm = sqrt(nrm);
            if (mode == 1) nrm = bnorm > 0.0 ? nrm / bnorm : nrm;
            *norm_out = nrm;
            *iters = sweep + q;
            pass = nrm < eps;
            if (nrm < eps) *done = 1;
        }
        __syncthreads();
        if (pass) return;
    }
}

// The tests that close a host batch of launches.
__global__ void __launch_bounds__(256) sor_tests_kernel(const double* partial, int n, int test, int sweep, double eps,
                                                        double bnorm, int mode, int* done, long long* iters,
                                                        double* norm_out) {
    sor_tests<256>(partial, n, test, sweep, eps, bnorm, mode, done, iters, norm_out);
}

// c where m is all ones, +0 where m is 0
__device__ __forceinline__ double keep(double c, int m) {
    const long long b = __double_as_longlong(c);
    return __longlong_as_double(((long long)((int)(b >> 32) & m) << 32) | (unsigned)((int)b & m));
}
__device__ __forceinline__ float keep(float c, int m) { return __int_as_float(__float_as_int(c) & m); }
// dvr with its last choice, q0 where it is zero or infinite, made through a lane
// mask in a scalar register pair by the selects' 64-bit encoding: the 32-bit
// one, which reads vcc, holds a wavefront up for some 19 cycles when two of them
// follow each other, as a double's two halves do; this one takes 4.
// A vector instruction may read a scalar register that another one wrote only two
// wait states later.  The compiler keeps that distance in its own code but not
// between asm statements, so the mask is written and read in one (2048 x 1024
// FP64, a solve of 5000 sweeps: 34.9 ms, and 34.8 with other instructions there).
__device__ __forceinline__ double dvr_e64(double a, double b, double y) {
    const double q0 = a * y;
    double r = __builtin_fma(-b, q0, a);
    const double q1 = __builtin_fma(r, y, q0);
    r = __builtin_fma(-b, q1, a);
    const double q2 = __builtin_fma(r, y, q1);
    const long long x = __double_as_longlong(q0), z = __double_as_longlong(q2);
    int lo = (int)z, hi = (int)(z >> 32);
    unsigned long long m;
    asm("v_cmp_class_f64_e64 %0, %3, %6\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %1, %1, %4, %0\n\t"
        "v_cndmask_b32_e64 %2, %2, %5, %0"
        : "=&s"(m), "+&v"(lo), "+&v"(hi)
        : "v"(q0), "v"((int)x), "v"((int)(x >> 32)), "s"(0x264));   // 0x264: -inf, -0, +0, +inf
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ float dvr_e64(float a, float b, float y) { return a * y; }
// value of the lane to the left (wave_shr:1) / right (wave_shl:1), 0 at the wavefront's ends
template <int CTRL>
__device__ __forceinline__ int dpp_i(int x) { return __builtin_amdgcn_mov_dpp(x, CTRL, 0xf, 0xf, true); }
template <int CTRL>
__device__ __forceinline__ float dpp(float x) { return __int_as_float(dpp_i<CTRL>(__float_as_int(x))); }
template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = dpp_i<CTRL>((int)b), hi = dpp_i<CTRL>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <typename T>
__device__ __forceinline__ T from_left(T x) { return dpp<0x138>(x); }
template <typename T>
__device__ __forceinline__ T from_right(T x) { return dpp<0x130>(x); }

template <typename T>
struct alignas(2 * sizeof(T)) Pair {
    T x, y;
};

// two neighbouring values of a row and two neighbouring codes, in one load (row:
// wave-uniform; the lane's place in it is a 32-bit byte offset)
template <typename T>
struct V2 {
    typedef T type __attribute__((ext_vector_type(2), aligned(sizeof(T))));   // dword alignment is enough
};
template <typename T>
__device__ __forceinline__ Pair<T> ldp(const T* row, unsigned i) {
    using V = typename V2<T>::type;
    const V v = *(const __attribute__((address_space(1))) V*)((const __attribute__((address_space(1))) char*)row + i * (unsigned)sizeof(T));
    return Pair<T>{v.x, v.y};
}
template <typename T>
__device__ __forceinline__ void stp(T* row, unsigned i, Pair<T> p) {
    using V = typename V2<T>::type;
    *(__attribute__((address_space(1))) V*)((__attribute__((address_space(1))) char*)row + i * (unsigned)sizeof(T)) = V{p.x, p.y};
}
__device__ __forceinline__ unsigned ldh(const uint8_t* row, unsigned i) {
    typedef unsigned short H __attribute__((aligned(1)));
    return *(const __attribute__((address_space(1))) H*)((const __attribute__((address_space(1))) uint8_t*)row + i);
}

// f(0), f(1), .. f(N - 1) with compile-time arguments
template <typename F, int... k>
__device__ __forceinline__ void pairs_(F&& f, std::integer_sequence<int, k...>) {
    (f(std::integral_constant<int, k>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void pairs(F&& f) {
    pairs_(f, std::make_integer_sequence<int, N>{});
}

// nsw sweeps (at most H / 2) of one tile per block; the last block of the grid
// tests the previous launch's sweeps meanwhile.  Every staged cell is updated
// in every half sweep of its colour; what a missing neighbour at the tile's
// rim spoils moves inwards by one cell per half sweep, so the cells H or more
// inside it are exactly those of global red-black sweeps, operation by
// operation those of sor_sweep.
//
// Bound: vector issue of the sweeps (23 instructions a cell where every
// neighbour is ocean, 18 of them FP64 at 4 cycles; 41 where a wavefront holds
// land, whose coefficients are masked lane by lane) and, a third of a launch,
// the tile's loads, which nothing overlaps when a CU has one block.  The LDS
// tiles of sor_block spend about 130 instructions a cell and sweep on
// addresses, masks and LDS traffic.  Four sweeps a launch, us per launch in the
// kernel trace, LDS tiles -> here: 51.6 -> 27.1 at 2048 x 1024 FP64, 33.6 -> 11.2
// at 1201 x 800 FP32, 36.4 -> 12.0 at 720 x 361 FP64 (reference mode).
template <typename T, int NW, int R>
__global__ void __launch_bounds__(NW * 64)
sor_rows(const SorRowsArgs<T> a, const T* __restrict__ chi_in, T* __restrict__ chi_out) {
    static_assert(R % 2 == 0, "colours by the row's parity in its wavefront");
    constexpr int W = 128, HH = NW * R;
    if ((int)blockIdx.x == a.ntile) {   // uniform
        if (a.prev_test)
            sor_tests<NW * 64>(a.prev_partial, a.ntile, a.prev_test, a.prev_sweep, a.eps, a.bnorm, a.residual_mode,
                               a.done, a.iters, a.norm_out);
        return;
    }
    if (*a.done) return;
    __shared__ T s_edge[2][NW][2][64];   // by half-sweep parity: each wavefront's first and last row
    __shared__ Pair<T> s_c5[HH * 12];
    __shared__ double red[kSorMaxSweeps][NW];
    const int Nx = a.Nx, Ny = a.Ny, P = a.P, H = a.H;
    const int TX = W - 2 * H, TY = HH - 2 * H;
    const int tile = xcd_tile(blockIdx.x, a.ntile);
    const int i0 = (tile % a.ntx) * TX, j0 = (tile / a.ntx) * TY;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gi0 = i0 - H + 2 * lane;
    // A pair of columns is one load: with even Nx it never straddles the seam;
    // with odd Nx the pair (Nx - 1, 0) reads the row's padding and takes column
    // 0 by a load of its own.
    const unsigned ga = (unsigned)wrap(gi0, Nx);
    const unsigned in_x = (!a.dead_x || (gi0 >= 0 && gi0 < Nx) ? 0xff00ffu : 0u) |
                          (!a.dead_x || (gi0 + 1 >= 0 && gi0 + 1 < Nx) ? 0xff00ff00u : 0u);
    const unsigned gc = in_x & 1u ? ga : 0u;
    T A[R], Bc[R], fA[R], fB[R];
    unsigned cw[R / 2];   // codes: row r's two columns in the half word r & 1 of cw[r / 2]
    unsigned cc[R];
    const int y0 = j0 - H + wv * R, g0 = wrap(y0, Ny);   // this wavefront's first row
    int gj = g0;
#pragma unroll
    for (int r = 0; r < R; ++r, gj = gj + 1 == Ny ? 0 : gj + 1) {   // every load of the tile in flight at once
        const size_t ro = (size_t)gj * P;
        const Pair<T> x = ldp(chi_in + ro, ga), f = ldp(a.B + ro, ga);
        A[r] = x.x; Bc[r] = x.y; fA[r] = f.x; fB[r] = f.y;
        cc[r] = ldh(a.code + ro, gc);
    }
    if (a.dead_x && ga + 1 == (unsigned)Nx) {
        gj = g0;
#pragma unroll
        for (int r = 0; r < R; ++r, gj = gj + 1 == Ny ? 0 : gj + 1) Bc[r] = ldg(chi_in + (size_t)gj * P, 0u);
    }
    unsigned odd0 = 0, odd1 = 0;   // bits of a code that is not SC_PLAIN, by colour
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
        const unsigned in_y = !a.dead_y ? ~0u
                            : (y0 + 2 * k >= 0 && y0 + 2 * k < Ny ? 0xffffu : 0u) |
                              (y0 + 2 * k + 1 >= 0 && y0 + 2 * k + 1 < Ny ? 0xffff0000u : 0u);
        cw[k] = (cc[2 * k] | cc[2 * k + 1] << 16) & in_x & in_y;
        const unsigned x = cw[k] ^ (SC_PLAIN * 0x01010101u);
        odd0 |= x & 0xff0000ffu;   // colour 0: column 0 of even rows, column 1 of odd ones
        odd1 |= x & 0x00ffff00u;
    }
    const bool plain0 = __all(odd0 == 0), plain1 = __all(odd1 == 0);
    // bit r: row r is one of the tile's output rows
    const int r_lo = max(H - wv * R, 0), r_hi = min(min(HH - H - wv * R, Ny - y0), R);
    const int rowok = r_hi > r_lo ? ((1 << r_hi) - 1) & ~((1 << r_lo) - 1) : 0;
    const T* const rowc = a.rowc + (size_t)(y0 + kSorPad) * 8;
    // a wavefront that holds other cells stages its rows' c5 for itself
    if (!plain0 || !plain1) {
        const Pair<T>* const c5g = (const Pair<T>*)a.c5 + (size_t)(y0 + kSorPad) * 12;
#pragma unroll
        for (int q = 0; q < R * 12; q += 64)
            if (q + lane < R * 12) s_c5[wv * R * 12 + q + lane] = c5g[q + lane];
    }
    // colour 1's edge rows for the first half sweep (row 0: column 1, row R - 1: column 0)
    s_edge[1][wv][0][lane] = Bc[0];
    s_edge[1][wv][1][lane] = A[R - 1];
    __syncthreads();
    double accA = 0.0, accB = 0.0;
    double sums[kSorMaxSweeps] = {};   // of the sweeps done, the last one first

    struct RowC {
        T c1, c3, c4, c5, c5r;
    };
    auto row_coef = [&](int r) {
        return RowC{ldc(rowc, r * 8), ldc(rowc, r * 8 + 1), ldc(rowc, r * 8 + 2), ldc(rowc, r * 8 + 3), ldc(rowc, r * 8 + 4)};
    };
    // one half sweep of colour C; MODE 0: no residual sum, 1: res, 2: r
    auto half = [&](auto cc, auto mm, const T om) {
        constexpr int C = decltype(cc)::value, MODE = decltype(mm)::value;
        const T up = s_edge[1 - C][wv + 1 < NW ? wv + 1 : wv][0][lane];   // row R
        const T dn = s_edge[1 - C][wv > 0 ? wv - 1 : wv][1][lane];        // row -1
        auto row = [&](auto rr, auto pp, const RowC& rc) {
            constexpr int r = decltype(rr)::value;
            constexpr bool PLAIN = decltype(pp)::value;
            constexpr int off = (r + C) & 1;
            const T x = off ? Bc[r] : A[r];
            const T E = off ? from_right(A[r]) : Bc[r];
            const T Wn = off ? A[r] : from_left(Bc[r]);
            const T N = r + 1 < R ? (off ? Bc[r + 1 < R ? r + 1 : r] : A[r + 1 < R ? r + 1 : r]) : up;
            const T S = r > 0 ? (off ? Bc[r > 0 ? r - 1 : r] : A[r > 0 ? r - 1 : r]) : dn;
            const T f = off ? fB[r] : fA[r];
            T k1 = rc.c1, k2 = rc.c1, k3 = rc.c3, k4 = rc.c4, c5 = rc.c5, c5r = rc.c5r;
            bool oc = true;
            if constexpr (!PLAIN) {
                constexpr int sh = 16 * (r & 1) + 8 * off;
                const int code = (int)cw[r / 2];
                auto bit = [&](int b) -> int { return (code << (31 - sh - b)) >> 31; };
                k1 = keep(rc.c1, bit(SC_OUE));
                k2 = keep(rc.c1, bit(SC_OU));
                k3 = keep(rc.c3, bit(SC_OVN));
                k4 = keep(rc.c4, bit(SC_OV));
                const Pair<T> p = s_c5[(wv * R + r) * 12 + ((code >> sh) & 15)];
                c5 = p.x;
                c5r = p.y;
                oc = bit(SC_OE) != 0;
            }
            const T lhs = (((k1 * E + k2 * Wn) + k3 * N) + k4 * S) + c5 * x;
            const T res_r = lhs - f;
            const T res = dvr_e64(om * res_r, c5, c5r);
            const T nv = oc ? x - res : x;
            if (off) Bc[r] = nv;
            else A[r] = nv;
            if constexpr (MODE != 0) {
                const double q = oc ? (double)(MODE == 2 ? res_r : res) : 0.0;
                const double qs = (rowok >> r) & 1 ? q : 0.0;
                if (off) accB = __builtin_fma(qs, q, accB);
                else accA = __builtin_fma(qs, q, accA);
            }
        };
        auto rows = [&](auto pp) {
            pairs<R / 2>([&](auto kk) {
                constexpr int k = decltype(kk)::value;
                row(std::integral_constant<int, 2 * k>{}, pp, row_coef(2 * k));
                row(std::integral_constant<int, 2 * k + 1>{}, pp, row_coef(2 * k + 1));
                __builtin_amdgcn_sched_barrier(0);   // two rows' temporaries at a time
            });
        };
        if (C ? plain1 : plain0) {
            rows(std::true_type{});
        } else {
            // the mask bits are expanded here, each time, not once into registers
#pragma unroll
            for (int k = 0; k < R / 2; ++k) asm volatile("" : "+v"(cw[k]));
            rows(std::false_type{});
        }
        s_edge[C][wv][0][lane] = C ? Bc[0] : A[0];
        s_edge[C][wv][1][lane] = C ? A[R - 1] : Bc[R - 1];
        __syncthreads();
    };
    const bool va = 2 * lane >= H && 2 * lane < W - H && gi0 < Nx, vb = va && gi0 + 1 < Nx;
    for (int sw = 0; sw < a.nsw; ++sw) {
        T om[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            om[c] = T(a.omega);
            if (a.relax) {   // Chebyshev schedule, held once stationary
                const int h = 2 * (a.sweep + sw - 1) + c;
                om[c] = T(ldc(a.relax, h < a.nrelax ? h : a.nrelax - 1));
            }
        }
        using std::integral_constant;
        if (!((a.test >> sw) & 1)) {
            half(integral_constant<int, 0>{}, integral_constant<int, 0>{}, om[0]);
            half(integral_constant<int, 1>{}, integral_constant<int, 0>{}, om[1]);
        } else if (a.residual_mode) {
            half(integral_constant<int, 0>{}, integral_constant<int, 2>{}, om[0]);
            half(integral_constant<int, 1>{}, integral_constant<int, 2>{}, om[1]);
        } else {
            half(integral_constant<int, 0>{}, integral_constant<int, 1>{}, om[0]);
            half(integral_constant<int, 1>{}, integral_constant<int, 1>{}, om[1]);
        }
#pragma unroll
        for (int k = kSorMaxSweeps - 1; k > 0; --k) sums[k] = sums[k - 1];
        sums[0] = (va ? accA : 0.0) + (vb ? accB : 0.0);
        accA = accB = 0.0;
    }
    if (va) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if ((rowok >> r) & 1) {
                T* const o = chi_out + (size_t)(y0 + r) * P;
                if (vb) stp(o, (unsigned)gi0, Pair<T>{A[r], Bc[r]});
                else stg(o, (unsigned)gi0, A[r]);
            }
    }
    if (!a.test) return;   // uniform
    // fixed-order block sums: wavefront butterfly, then the wavefronts in order
#pragma unroll
    for (int k = 0; k < kSorMaxSweeps; ++k) {
        double v = sums[k];
        for (int s = 32; s >= 1; s >>= 1) v += __shfl_xor(v, s, 64);
        if (lane == 0) red[k][wv] = v;
    }
    __syncthreads();
    if (tid < a.nsw) {   // sweep tid's sum is sums[nsw - 1 - tid]
        double t = red[a.nsw - 1 - tid][0];
        for (int w = 1; w < NW; ++w) t += red[a.nsw - 1 - tid][w];
        a.partial[(size_t)tid * a.ntile + blockIdx.x] = t;
    }
}

}  // namespace swm
