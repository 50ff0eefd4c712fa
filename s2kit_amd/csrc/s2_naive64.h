// FP64 Legendre transforms as dense GEMMs on FP64 MFMA (bw in [16, 512]):
// every order projects its ring samples on (forward) or sums (inverse) the
// sampled functions P_l^m(theta_j) (naive.c:34-95), folded over the equator:
// P_l^m(theta_{N-1-j}) = (-1)^(l-m) P_l^m(theta_j) and the weights are
// symmetric, so degrees of even l-m see x_j + x_{N-1-j} and odd ones
// x_j - x_{N-1-j}, j < bw.  Per order m, with data columns (field, +m or -m
// row, re or im):
//   forward  C[col][l]   = sum_{j<bw} fold_p(X[col])[j] * w_j P_l^m(theta_j)
//   inverse  E/O[col][j] = sum_i coef[col][m+p+2i] * P_{m+p+2i}^m(theta_j)/sqrt(2pi)
// with ring j <- E+O and ring N-1-j <- E-O.
//
// Why dense and not the seminaive sums: the seminaive form does a third of
// the multiplications but needs a DCT pass over the order rows each way
// (24 N^2 bytes per field at the HBM rate), and its staircase tables left the
// matrix cores mostly waiting.  bw=256 x 1024 fields, DCT + seminaive GEMM
// against one dense GEMM: forward 1.46 + 1.36 -> 1.57 ms, inverse 1.16 + 1.55
// -> 1.75 ms (step 8.28 -> 6.19 ms); bw=512 x 128 2.0 -> 1.41, 1.7 -> 1.39 ms;
// bw=64 x1 16 -> 7, 17 -> 6 us.  The dense sums have no cosine-space
// cancellation: error against 64-bit definitions 4.1e-14 -> 1.4e-14.
//
// Both kernel families take each accumulator's K steps (4 rings, or 4 degrees
// of one parity) in the same ascending order, so a field's results do not
// depend on the field count of the call.
//
// Tables, in MFMA operand order (lane = 16 * (k mod 4) + n mod 16):
//   NF(q) [K step j/4 < bp/4][p][16-degree tile < nt][64]: w_j P_{m+p+2i}^m(theta_j) of the order pair
//         m = q (its n0 tiles first) and bw-1-q, nt tiles per parity together
//   NI(m) [K step i/4 < ki][p][16-ring tile < bp/16][64]: P_{m+p+2i}^m(theta_j)/sqrt(2pi)
// bp = bw rounded up to 16; entries past the last ring or degree are zero.
#pragma once

#include <type_traits>

#include "s2_mix_common.h"
#include "s2_recurrence.h"

namespace s2 {

typedef double dvec2 __attribute__((ext_vector_type(2)));

__host__ __device__ inline int n64_bp(int B) { return (B + 15) & ~15; }
// K steps of order m's inverse: its even degrees in fours, rounded up to whole stages of two steps
__host__ __device__ inline int n64_ki(int m, int B) { return 2 * ((gm_lp(m, 0, B) + 7) / 8); }
// 16-degree tiles per parity of the order pair (q, bw-1-q), rounded up to the
// halves of the K-chunked forward (two for bw > 256); the middle order of an
// odd bw, which pairs with itself, keeps empty tiles in its partner's place.
__host__ __device__ inline int n64_halves(int B) { return B <= 256 ? 1 : 2; }
__host__ __device__ inline int n64_nt(int q, int B) {
    const int n = mix_n0(q, B) + mix_n0(B - 1 - q, B);
    return n64_halves(B) == 1 ? n : (n + 1) & ~1;
}

// VALU and MFMA instructions of a SIMD's waves do not overlap here: every VALU
// instruction adds about 3.5 cycles to the MFMA time (measured: FP32 16x16x4
// MFMAs at 4 waves per SIMD 13.7 ns, 16.6 / 18.7 / 24.4 ns with 2 / 4 / 8
// v_add_u32 between them).  The K loops therefore keep to a dozen VALU
// instructions per stage: addresses are uniform bases in scalar registers
// plus per-lane offsets fixed before the loop, and stages alternate between
// two buffers by unrolling, not by address arithmetic.
__device__ __forceinline__ int n64_uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
template <typename T>
__device__ __forceinline__ T n64_ld(const char* base, unsigned off) {  // uniform base, per-lane offset
    return *reinterpret_cast<const T*>(base + off);
}
// 1 KiB global -> LDS: lane l's 16 bytes from src + off (per lane) to dst + 16 l
__device__ __forceinline__ void n64_dma(const char* src, unsigned off, double* dst) {
    __builtin_amdgcn_global_load_lds((const void*)(src + off), (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// Row of data column `rem` (of cpf) of a field: order m or -m.
__device__ __forceinline__ int n64_row(int rem, int m, int N) { return (rem >> 1) ? N - m : m; }

// Where data column c of order m writes its coefficients: o1 the run of its
// order (sign s1), o2 the mirror run of REAL data (sign s2) or null.
struct N64Out {
    double *o1, *o2;
    double s1, s2;
};
__device__ __forceinline__ N64Out n64_out(int c, int m, int cpf, int B, int fmt, double* cre, double* cim) {
    const int f = c >> (cpf >> 1), rem = c & (cpf - 1), comp = rem & 1;  // cpf is 2 or 4
    double* base = (comp ? cim : cre) + (size_t)f * B * B;
    const bool neg = (rem >> 1) != 0, odd = m & 1;
    N64Out o;
    o.o1 = base + (neg ? index_of_coeff(-m, m, B) : index_of_coeff(m, m, B));
    o.s1 = (neg && odd) ? -1.0 : 1.0;  // rows -m carry (-1)^m
    o.o2 = (!neg && fmt == 1 && m > 0) ? base + index_of_coeff(-m, m, B) : nullptr;
    o.s2 = ((comp != 0) != odd) ? -1.0 : 1.0;  // REAL data: f(l,-m) = (-1)^m conj f(l,m)
    return o;
}

// Inverse epilogue of one MFMA row pair: accumulator registers r, r+1 are the
// re and im sums of column pair c (times sg), lane x16 the ring j of the first tile.
template <int T>
__device__ __forceinline__ void n64_inv_store(const dvec4 (&e)[T], const dvec4 (&o)[T], double2* __restrict__ X, int m,
                                              int c, int r, double sg, int j, int B, int cpf) {
    const int N = 2 * B;
    const int f = c >> (cpf >> 1), rem = c & (cpf - 1);  // cpf is 2 or 4
    double2* xr = X + ((size_t)f * N + n64_row(rem, m, N)) * N;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int jt = j + 16 * t;
        if (jt >= B) continue;
        const double2 lo = make_double2(sg * (e[t][r] + o[t][r]), sg * (e[t][r + 1] + o[t][r + 1]));
        const double2 hi = make_double2(sg * (e[t][r] - o[t][r]), sg * (e[t][r + 1] - o[t][r + 1]));
        xr[jt] = lo;
        xr[N - 1 - jt] = hi;
    }
}
// The inverse's operand row for accumulator row x16: lane (x16, kq) then holds
// columns 4kq .. 4kq+3 of its tile in registers 0 .. 3 (FP64 MFMA results sit
// at rows kq + 4r), so re and im of a value share a lane.
__device__ __forceinline__ int n64_col(int x16) { return 4 * (x16 & 3) + (x16 >> 2); }

// ---------------------------------------------------------------------------
// direct: no LDS, no barrier; one wave per item
// ---------------------------------------------------------------------------
// A wave owns NTW degree (ring) tiles, both parities, and CT column tiles of
// one order and streams its operands from global memory in batches of S K
// steps, NB batches in flight.  For calls of few fields, which are bound by the
// latency of that stream, and for small bandwidths.
template <int CT, int NTW>
constexpr int n64_nb() {
    return CT * NTW == 1 ? 3 : 2;
}

template <int CT, int NTW>
__device__ __forceinline__ void naive64_fwd_direct(const double2* __restrict__ X, const double* __restrict__ NF,
                                                   const GemmMeta* __restrict__ meta, double* __restrict__ cre,
                                                   double* __restrict__ cim, int m, int item, int B, int F, int fmt) {
    constexpr int S = 4, NB = n64_nb<CT, NTW>();
    const GemmMeta g = meta[2 * m];
    const int N = 2 * B, n0 = g.n0, nt = g.Kf;
    const int cpf = mix_cpf(m, fmt), ncols = F * cpf;
    const int ntg = (n0 + NTW - 1) / NTW, cg = item / ntg, t0 = (item - cg * ntg) * NTW;
    if (cg * 16 * CT >= ncols) return;
    const int lane = threadIdx.x & 63, x16 = lane & 15, kq = lane >> 4;
    const int fb = cg * 16 * CT >> (cpf >> 1);  // the item's first field
    const char* xbase = reinterpret_cast<const char*>(X + (size_t)fb * N * N);
    unsigned oa[CT], ob[CT];  // this lane's column at rings kq and N-1-kq
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int col = (cg * CT + c) * 16 + x16, k = col < ncols ? col : fb * cpf;
        const int f = k >> (cpf >> 1), rem = k & (cpf - 1);  // cpf is 2 or 4
        const unsigned row = (unsigned)((f - fb) * N + n64_row(rem, m, N)) * N;
        oa[c] = (row + kq) * 16u + 8 * (rem & 1);
        ob[c] = (row + N - 1 - kq) * 16u + 8 * (rem & 1);
    }
    const char* tsrc = reinterpret_cast<const char*>(NF + g.offF);
    const int nb = (n64_bp(B) >> 2) / S;
    struct Batch {
        double a[S][CT], b[S][CT], t[S][2][NTW];
    } buf[NB];
    auto load = [&](int b, Batch& q) __attribute__((always_inline)) {
        const int k0 = min(b, nb - 1) * S;  // past the end: the last batch again, unused
        const char* xa = xbase + k0 * 64;
        const char* xb = xbase - k0 * 64;
        const char* tk = tsrc + (size_t)k0 * (nt * 1024);
#pragma unroll
        for (int s = 0; s < S; ++s) {
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                q.a[s][c] = n64_ld<double>(xa + 64 * s, oa[c]);
                q.b[s][c] = n64_ld<double>(xb - 64 * s, ob[c]);
            }
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int t = 0; t < NTW; ++t)
                    q.t[s][p][t] = n64_ld<double>(tk + ((s * 2 + p) * nt + min(t0 + t, n0 - 1)) * 512, lane * 8);
        }
    };
    dvec4 acc[CT][2][NTW] = {};
    auto mma = [&](const Batch& q) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const double e = q.a[s][c] + q.b[s][c], o = q.a[s][c] - q.b[s][c];
#pragma unroll
                for (int t = 0; t < NTW; ++t) {
                    acc[c][0][t] = Mma<double>::mma(e, q.t[s][0][t], acc[c][0][t]);
                    acc[c][1][t] = Mma<double>::mma(o, q.t[s][1][t], acc[c][1][t]);
                }
            }
    };
#pragma unroll
    for (int u = 0; u < NB; ++u) load(u, buf[u]);
    int b = 0;
    for (; b + NB <= nb; b += NB)
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            mma(buf[u]);
            load(b + u + NB, buf[u]);
        }
#pragma unroll
    for (int u = 0; u < NB; ++u)
        if (b + u < nb) mma(buf[u]);
    const int L = B - m;
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int col = (cg * CT + c) * 16 + Mma<double>::row(lane, r);
            if (col >= ncols) continue;
            const N64Out w = n64_out(col, m, cpf, B, fmt, cre, cim);
#pragma unroll
            for (int t = 0; t < NTW; ++t) {
                const int d = 32 * (t0 + t) + 2 * x16;
                const double v0 = acc[c][0][t][r], v1 = acc[c][1][t][r];
                if (d + 1 < L) {
                    *reinterpret_cast<dpair8*>(w.o1 + d) = dpair8{w.s1 * v0, w.s1 * v1};
                    if (w.o2) *reinterpret_cast<dpair8*>(w.o2 + d) = dpair8{w.s2 * v0, w.s2 * v1};
                } else if (d < L) {
                    w.o1[d] = w.s1 * v0;
                    if (w.o2) w.o2[d] = w.s2 * v0;
                }
            }
        }
}

// Inverse: CT column tiles and RTW ring tiles of one order per wave.
template <int CT, int RTW>
__device__ __forceinline__ void naive64_inv_direct(const double* __restrict__ cre, const double* __restrict__ cim,
                                                   const double* __restrict__ NI, const GemmMeta* __restrict__ meta,
                                                   double2* __restrict__ X, int m, int item, int B, int F, int fmt) {
    constexpr int S = 2, NB = n64_nb<CT, RTW>() + 1;
    const GemmMeta g = meta[2 * m];
    const int RT = n64_bp(B) >> 4, L = B - m;
    const int cpf = mix_cpf(m, fmt), ncols = F * cpf;
    const int nrg = (RT + RTW - 1) / RTW, cg = item / nrg, rt0 = (item - cg * nrg) * RTW;
    if (cg * 16 * CT >= ncols) return;
    const int lane = threadIdx.x & 63, x16 = lane & 15, kq = lane >> 4;
    const double* cp[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int col = (cg * CT + c) * 16 + n64_col(x16), k = col < ncols ? col : 0;
        const int f = k >> (cpf >> 1), rem = k & (cpf - 1);
        cp[c] = ((rem & 1) ? cim : cre) + (size_t)f * B * B + index_of_coeff((rem >> 1) ? -m : m, m, B);
    }
    const char* tsrc = reinterpret_cast<const char*>(NI + g.offI);
    const int nb = g.ki / S;
    struct Batch {
        dpair8 a[S][CT];
        double t[S][2][RTW];
    } buf[NB];
    auto load = [&](int b, Batch& q) __attribute__((always_inline)) {
        const int k0 = min(b, nb - 1) * S;
        const char* tk = tsrc + (size_t)k0 * (RT * 1024);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            // the run's last pair when this lane's degrees lie past it (mma() selects); the
            // one-degree run of m = bw-1 is never the array's first, so -1 is inside it
            const int d = min(2 * (4 * (k0 + s) + kq), L - 2);
#pragma unroll
            for (int c = 0; c < CT; ++c) q.a[s][c] = *reinterpret_cast<const dpair8*>(cp[c] + d);
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int t = 0; t < RTW; ++t)
                    q.t[s][p][t] = n64_ld<double>(tk + ((s * 2 + p) * RT + min(rt0 + t, RT - 1)) * 512, lane * 8);
        }
    };
    dvec4 acc[CT][2][RTW] = {};
    auto mma = [&](int b, const Batch& q) __attribute__((always_inline)) {
        const bool whole = 8 * S * (b + 1) <= L;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int d = 2 * (4 * (b * S + s) + kq);
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                double e = q.a[s][c].x, o = q.a[s][c].y;
                if (!whole) {  // the run ends in this batch
                    e = d + 1 < L ? e : d < L ? o : 0.0;
                    o = d + 1 < L ? o : 0.0;
                }
#pragma unroll
                for (int t = 0; t < RTW; ++t) {
                    acc[c][0][t] = Mma<double>::mma(e, q.t[s][0][t], acc[c][0][t]);
                    acc[c][1][t] = Mma<double>::mma(o, q.t[s][1][t], acc[c][1][t]);
                }
            }
        }
    };
#pragma unroll
    for (int u = 0; u < NB; ++u) load(u, buf[u]);
    int b = 0;
    for (; b + NB <= nb; b += NB)
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            mma(b + u, buf[u]);
            load(b + u + NB, buf[u]);
        }
#pragma unroll
    for (int u = 0; u < NB; ++u)
        if (b + u < nb) mma(b + u, buf[u]);
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
            const int col = (cg * CT + c) * 16 + 4 * kq + 2 * rr;
            const double sg = ((col & (cpf - 1)) >> 1) && (m & 1) ? -1.0 : 1.0;  // rows -m carry (-1)^m
            if (col < ncols)
                n64_inv_store<RTW>(acc[c][0], acc[c][1], X, m, col, 2 * rr, sg, 16 * rt0 + x16, B, cpf);
        }
}

}  // namespace s2
