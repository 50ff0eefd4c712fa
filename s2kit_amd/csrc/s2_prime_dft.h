// FP64 ring FFTs of lengths N = R P <= 1024 with a prime factor P >= 23 (R
// has none): the Good-Thomas split into P-point and R-point DFTs, which needs
// no twiddles between the two, with the P-point DFTs as GEMMs on FP64 MFMA.
//
// Index maps, for y_k = sum_n x_n w^{nk}, w = exp(SIGN 2 pi i/N): one side by
// residues (n1 = n mod R, n2 = n mod P), the other as k = k1 P + k2 R mod N;
// then w^{nk} = w_R^{n1 k1} w_P^{n2 k2}.  The kernels take residues on the
// side that is contiguous in memory (the ring) and the sum on the order rows.
//
// P-point DFT by conjugate pairs, H = (P-1)/2, s_q = x_q + x_{P-q},
// d_q = x_q - x_{P-q}, p <= H:
//   A_p = x_0 + sum_q s_q cos(2 pi pq/P),  B_p = sum_q d_q sin(2 pi pq/P),
//   y_p = A_p + i SIGN B_p,  y_{P-p} = A_p - i SIGN B_p:
// two real GEMMs of H+1 outputs and as many terms over the real columns
// (ring, k1, re or im), a quarter of the P x P complex product.
//
// LDS holds a block's rings as rows n2 < P of nr R complex columns and one of
// padding (rows of neighbouring lanes start on different banks): s_q in row q
// and d_q in row P-q, then A_p in row p and B_p in row P-p.  For R = 2 and 4
// the load phase stores s and d directly; other R stage x_{n2} and run the
// R-point DFTs on the register passes first.  A wave takes one 16-column
// tile, one of the two GEMMs and up to five 16-row tiles; the table fragments
// come from global memory (L2, shared by all blocks) in operand order, three
// K steps ahead, the data fragments from LDS.
//
// Bluestein's convolution, which this replaces, does fewer operations (two
// FFTs of length >= 2N against 2 N P multiply-adds) but in some ten LDS passes
// with a barrier each.  Ring FFT, us, before -> now (forward / inverse): bw=23 x2048
// 202 -> 39 / 41, bw=46 x400 109 -> 31 / 34, bw=101 x100 139 -> 51 / 56, bw=263
// x32 320 -> 159 / 141, one field 27 -> 15, bw=437 x8 176 -> 82 / 91, bw=509
// x16 395 -> 378, 437 -> 373.  The gain shrinks with P and ends near the
// largest; no length up to 1024 lost.
//
// Bound (bw=263): the K loop runs at the FP64 MFMA rate by itself (8.2 of a
// block's 17 us), but the ring loads and stores of the other resident block
// add to it instead of hiding behind it.  Neither wave priorities, a start
// offset between the two blocks, fewer rings per block nor table loads a step
// ahead instead of three changed that.
#pragma once

#include "s2_complex.h"

namespace s2 {

constexpr int kPrimeMaxN = 1024;  // ring lengths up to it hold one prime factor above 19, and that once

typedef double pvec4 __attribute__((ext_vector_type(4)));

// div16 with its divisor and remainder (the reciprocals are per block)
struct DivF {
    int d;
    float r;  // 1/d
    __device__ __forceinline__ int quo(int x) const { return div16(x, r); }
    __device__ __forceinline__ int rem(int x, int q) const { return x - __mul24(q, d); }
    __device__ __forceinline__ int rem(int x) const { return rem(x, quo(x)); }
};
__device__ __forceinline__ DivF div_by(int d) { return {d, __builtin_amdgcn_rcpf((float)d)}; }

// Shape of the two GEMMs, at the head of the tables (a block's first loads;
// the integer divisions behind it took a block longer than its barriers).
struct PrimeDft {
    int P, R, H;
    int T;   // 16-row tiles of the H+1 outputs
    int KS;  // K steps of 4 terms, even (zero table entries past H)
    float rN, rP, rR, rH1;  // reciprocals of N, P, R, H+1
    int pad[7];
};
__host__ inline PrimeDft prime_dft(int N, int P) {
    const int H = (P - 1) / 2;
    return {P, N / P, H, (H + 16) / 16, 2 * ((H + 8) / 8), 1.0f / N, 1.0f / P, (float)P / N, 1.0f / (H + 1), {}};
}
// Tables: the PrimeDft, R twiddles exp(-2 pi i t/R), then [K step][cos, sin][tile][64]
// in MFMA operand order (lane = 16 (k mod 4) + row mod 16): cos(2 pi pq/P), q = k,
// and sin(2 pi p(k+1)/P), zero past p or q = H.
static_assert(sizeof(PrimeDft) == 64, "the twiddles follow at double2 4");
__host__ __device__ inline long prime_table_doubles(const PrimeDft& d) {
    return 8 + 2L * d.R + (long)d.KS * 2 * d.T * 64;
}
// log2 of the runs of row tiles per GEMM and column tile: at most five tiles
// per wave (40 VGPRs of sums; 16 tiles at most, P <= 509), and more runs while waves are idle.
inline int prime_runs_log2(const PrimeDft& d, int ct) {
    int lr = d.T <= 5 ? 0 : d.T <= 10 ? 1 : 2;
    while (lr < 2 && (4 << lr) * ct <= 8 && (2 << lr) <= d.T) ++lr;
    return lr;
}
__host__ __device__ inline size_t prime_lds_values(const PrimeDft& d, int nr) {
    return (size_t)d.P * (nr * d.R + 1) + d.R;
}

// One wave's G row tiles (from tile t0) of column tile c0: kind 0 the cosine
// GEMM over rows 0, 1, ..., kind 1 the sine GEMM over rows P-1, P-2, ....
// Every wave of a column tile reaches the barrier here between its reads and
// its writes.
template <int G>
__device__ __forceinline__ void prime_tiles(double* ld, int rs, int ncol, const PrimeDft& d, const double* tab, int kind,
                                            int t0, int c0) {
    const int lane = threadIdx.x & 63, x = lane & 15, kq = lane >> 4;
    const int col = c0 * 16 + x;
    const int cc = min(col, ncol - 1);
    const int kst = 2 * d.T * 64;
    const double* tp = tab + (kind * d.T + t0) * 64;
    // data row of K step ks: kq + 4 ks, or P-1 - (kq + 4 ks)
    const double* bp = ld + (kind ? d.P - 1 - kq : kq) * rs + cc;
    const int bst = kind ? -4 * rs : 4 * rs;
    pvec4 acc[G];
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = pvec4{0.0, 0.0, 0.0, 0.0};
    double a[4][G], b[4];
    auto load = [&](int u, int ks) __attribute__((always_inline)) {
        const double* t = tp + (long)ks * kst;
#pragma unroll
        for (int g = 0; g < G; ++g) a[u][g] = t[g * 64 + lane];
        b[u] = bp[ks * bst];
    };
    auto mul = [&](int u) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][g], b[u], acc[g], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // three steps ahead; KS is even, a last pair of steps after whole fours
#pragma unroll
    for (int u = 0; u < 4; ++u) load(u, min(u, d.KS - 1));
    const int k4 = d.KS & ~3;
    for (int ks = 0; ks < k4; ks += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            mul(u);
            load(u, min(ks + 4 + u, d.KS - 1));
        }
    }
    if (d.KS & 2) {
        mul(0);
        mul(1);
    }
    __syncthreads();
    if (col < ncol) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = (t0 + g) * 16 + 4 * r + kq;
                if (p <= d.H && t0 + g < d.T && (kind == 0 || p > 0)) ld[(kind ? d.P - p : p) * rs + col] = acc[g][r];
            }
    }
}

// i^(SIGN t) v
template <int SIGN>
__device__ __forceinline__ double2 rot90(double2 v, int t) {
    double2 r = (t & 1) ? make_double2(SIGN < 0 ? v.y : -v.y, SIGN < 0 ? -v.x : v.x) : v;
    return (t & 2) ? make_double2(-r.x, -r.y) : r;
}
// R-point DFT in registers, R = 2 or 4
template <int SIGN, int R>
__device__ __forceinline__ void dft_small(double2 (&v)[R]) {
    if constexpr (R == 2) {
        const double2 s = cadd(v[0], v[1]);
        v[1] = csub(v[0], v[1]);
        v[0] = s;
    } else {
        const double2 s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
        const double2 s13 = cadd(v[1], v[3]), d13 = rot90<SIGN>(csub(v[1], v[3]), 1);
        v[0] = cadd(s02, s13);
        v[2] = csub(s02, s13);
        v[1] = cadd(d02, d13);
        v[3] = csub(d02, d13);
    }
}
// The same over x_j = x[q + j P] (residue n1 = q + j P): outputs k1 are
// w^{k1 q} times the DFT over j at k1 P, w = exp(SIGN 2 pi i/R), P odd.
template <int SIGN, int R>
__device__ __forceinline__ void dft_stream(double2 (&v)[R], int q, int P) {
    dft_small<SIGN, R>(v);
    if constexpr (R == 2) {
        v[1] = rot90<SIGN>(v[1], (q & 1) * 2);
    } else {
        const bool sw = (P & 3) == 3;
        const double2 y1 = sw ? v[3] : v[1], y3 = sw ? v[1] : v[3];
        v[1] = rot90<SIGN>(y1, q);
        v[2] = rot90<SIGN>(v[2], 2 * q);
        v[3] = rot90<SIGN>(y3, 3 * q);
    }
}
// s_q and d_q of R columns from x (row q) and y (row P-q)
template <int R>
__device__ __forceinline__ void store_fold(double2* u, double2* w, const double2 (&x)[R], const double2 (&y)[R], bool two) {
#pragma unroll
    for (int e = 0; e < R; ++e) {
        u[e] = two ? cadd(x[e], y[e]) : x[e];
        if (two) w[e] = csub(x[e], y[e]);
    }
}
__device__ __forceinline__ int wrap(int x, int n) { return x >= n ? x - n : x; }

// R other than 2 and 4, rows x_{n2} in LDS (after a barrier): the R-point
// DFTs on the register passes, then s_q, d_q in place.
template <int SIGN>
__device__ __forceinline__ void prime_parts(double2* a, int nr, const PrimeDft& d, const double2* __restrict__ tw) {
    const int R = d.R, rs = nr * R + 1, nc = nr * R;
    double2* twl = a + d.P * rs;
    for (int i = threadIdx.x; i < R; i += kMrThreads) twl[i] = tw[4 + i];
    __syncthreads();
    const float mnr = magic16(nr);
    mr_reg_fft<double2, SIGN>(a, R, d.P * nr, twl, [=](int f) { return f * R + div16(f, mnr); });
    const DivF dc = div_by(nc);
    for (int i = threadIdx.x; i < d.H * nc; i += kMrThreads) {
        const int t = dc.quo(i), c = dc.rem(i, t), q = t + 1;
        double2* u = a + __mul24(q, rs) + c;
        double2* w = a + __mul24(d.P - q, rs) + c;
        const double2 x = *u, y = *w;
        *u = cadd(x, y);
        *w = csub(x, y);
    }
}

// The P-point DFTs in LDS, rows s, d in (after a barrier), rows A, B out.
__device__ __forceinline__ void prime_gemms(double2* a, int nr, int lr, const PrimeDft& d,
                                            const double2* __restrict__ tw) {
    const int rs = nr * d.R + 1, ncol = 2 * nr * d.R;
    const double* tab = reinterpret_cast<const double*>(tw + 4 + d.R);
    double* ld = reinterpret_cast<double*>(a);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ct = (ncol + 15) >> 4, runs = 1 << lr, G = (d.T + runs - 1) >> lr;
    // waves 2 runs per column tile, so 4 / runs column tiles per round
    const int ci = wave >> (lr + 1), kind = (wave >> lr) & 1;
    // a column tile's longer runs fall to other SIMDs than its neighbour's
    const int run = (wave ^ (wave >> 2)) & (runs - 1);
    const int t0 = run * G;
    for (int c = 0; c < ct; c += 4 >> lr) {
        switch (c + ci < ct ? min(G, d.T - t0) : 0) {
            case 1: prime_tiles<1>(ld, 2 * rs, ncol, d, tab, kind, t0, c + ci); break;
            case 2: prime_tiles<2>(ld, 2 * rs, ncol, d, tab, kind, t0, c + ci); break;
            case 3: prime_tiles<3>(ld, 2 * rs, ncol, d, tab, kind, t0, c + ci); break;
            case 4: prime_tiles<4>(ld, 2 * rs, ncol, d, tab, kind, t0, c + ci); break;
            case 5: prime_tiles<5>(ld, 2 * rs, ncol, d, tab, kind, t0, c + ci); break;
            default: __syncthreads(); break;  // no column tile or rows left for this wave
        }
    }
    __syncthreads();
}

// A +- i B
__device__ __forceinline__ double2 add_i(double2 A, double2 B) { return make_double2(A.x - B.y, A.y + B.x); }
__device__ __forceinline__ double2 sub_i(double2 A, double2 B) { return make_double2(A.x + B.y, A.y - B.x); }

// Forward load phase, RR = R = 2 or 4: a thread takes the samples of residues q
// and P-q (n = q + j P and P-q + j P, contiguous over q for each j) of a ring
// and stores its columns of rows q and P-q finished.
template <int RR>
__device__ __forceinline__ void prime_load_fwd(double2* a, const double* __restrict__ re, const double* __restrict__ im,
                                               int N, int n, int rs, const PrimeDft& d) {
    constexpr int U = 4 / RR;  // threads' steps whose loads are in flight together
    const DivF dh{d.H + 1, d.rH1};
    const int P = d.P, tot = n * (d.H + 1);
    for (int i0 = threadIdx.x; i0 < tot; i0 += U * kMrThreads) {
        double2 x[U][RR], y[U][RR];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * kMrThreads;
            if (i < tot) {
                const int jl = dh.quo(i), q = dh.rem(i, jl);
                const int o = __mul24(jl, N), ox = o + q, oy = o + (q ? P - q : 0);
#pragma unroll
                for (int j = 0; j < RR; ++j) {
                    x[u][j] = make_double2(re[(unsigned)(ox + j * P)], im[(unsigned)(ox + j * P)]);
                    y[u][j] = make_double2(re[(unsigned)(oy + j * P)], im[(unsigned)(oy + j * P)]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * kMrThreads;
            if (i < tot) {
                const int jl = dh.quo(i), q = dh.rem(i, jl);
                dft_stream<-1, RR>(x[u], q, P);
                dft_stream<-1, RR>(y[u], P - q, P);
                store_fold<RR>(a + __mul24(q, rs) + jl * RR, a + __mul24(P - q, rs) + jl * RR, x[u], y[u], q > 0);
            }
        }
    }
}
// Other R: the samples at (n2, n1), R-point DFTs and folding left to prime_parts.
template <>
__device__ __forceinline__ void prime_load_fwd<0>(double2* a, const double* __restrict__ re,
                                                  const double* __restrict__ im, int N, int n, int rs,
                                                  const PrimeDft& d) {
    // N = R P: a flat index and its ring's sample share their residues
    const DivF dN{N, d.rN}, dP{d.P, d.rP}, dR{d.R, d.rR};
    const int tot = n * N;
    for (int i0 = threadIdx.x; i0 < tot; i0 += 4 * kMrThreads) {
        double2 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * kMrThreads;
            if (i < tot) v[u] = make_double2(re[i], im[i]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * kMrThreads;
            if (i < tot) a[__mul24(dP.rem(i), rs) + __mul24(dN.quo(i), d.R) + dR.rem(i)] = v[u];
        }
    }
}

// Inverse load phase: rows k1 P +- q R of X.  REAL data: rows m < bw only, row
// N-r the conjugate of r, so x_{n1, P-q} the conjugate of x_{R-n1, q}.
template <int RR>
__device__ __forceinline__ void prime_load_inv(double2* a, const double2* __restrict__ X, int N, int B, int n, int rs,
                                               int real, const PrimeDft& d) {
    constexpr int U = 4 / RR;
    const DivF dn = div_by(n);
    const int P = d.P, tot = n * (d.H + 1);
    auto row = [&](int r, int jl) __attribute__((always_inline)) {
        const bool up = real && r > B;
        double2 v = X[(unsigned)(__mul24(up ? N - r : r, N) + jl)];
        if (up) v.y = -v.y;
        return r == B ? make_double2(0.0, 0.0) : v;
    };
    for (int i0 = threadIdx.x; i0 < tot; i0 += U * kMrThreads) {
        double2 x[U][RR], y[U][RR];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * kMrThreads;
            if (i < tot) {
                const int q = dn.quo(i), jl = dn.rem(i, q);
                int ra = q * RR, rb = q ? N - q * RR : 0;
#pragma unroll
                for (int e = 0; e < RR; ++e) {
                    x[u][e] = row(ra, jl);
                    if (!real) y[u][e] = row(rb, jl);
                    ra = wrap(ra + P, N);
                    rb = wrap(rb + P, N);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * kMrThreads;
            if (i < tot) {
                const int q = dn.quo(i), jl = dn.rem(i, q);
                if (real)
#pragma unroll
                    for (int e = 0; e < RR; ++e) y[u][e] = cconj(x[u][(RR - e) % RR]);
                dft_small<+1, RR>(x[u]);
                dft_small<+1, RR>(y[u]);
                store_fold<RR>(a + __mul24(q, rs) + jl * RR, a + __mul24(P - q, rs) + jl * RR, x[u], y[u], q > 0);
            }
        }
    }
}
template <>
__device__ __forceinline__ void prime_load_inv<0>(double2* a, const double2* __restrict__ X, int N, int B, int n,
                                                  int rs, int real, const PrimeDft& d) {
    const DivF dn = div_by(n), dR{d.R, d.rR};
    const int tot = n * N;
    for (int i0 = threadIdx.x; i0 < tot; i0 += 4 * kMrThreads) {
        double2 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * kMrThreads;
            if (i < tot) {
                const int t = dn.quo(i), jl = dn.rem(i, t), n2 = dR.quo(t);
                const int r = wrap(__mul24(dR.rem(t, n2), d.P) + __mul24(n2, d.R), N);
                const bool up = real && r > B;
                v[u] = X[(unsigned)(__mul24(up ? N - r : r, N) + jl)];
                if (up) v[u].y = -v[u].y;
                if (r == B) v[u] = make_double2(0.0, 0.0);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * kMrThreads;
            if (i < tot) {
                const int t = dn.quo(i), jl = dn.rem(i, t), n2 = dR.quo(t);
                a[__mul24(n2, rs) + __mul24(jl, d.R) + dR.rem(t, n2)] = v[u];
            }
        }
    }
}

// Forward store phase: rows k1 P +- p R of X (below `out`) from the row pair p.
template <int RR>
__device__ __forceinline__ void prime_store_fwd(const double2* a, double2* __restrict__ X, int N, int out, int n, int rs,
                                                const PrimeDft& d) {
    const DivF dn = div_by(n);
    constexpr int R = RR;
    const int P = d.P;
    for (int i = threadIdx.x; i < n * (d.H + 1); i += kMrThreads) {
        const int p = dn.quo(i), jl = dn.rem(i, p);
        const double2* u = a + __mul24(p, rs) + __mul24(jl, R);
        const double2* w = a + __mul24(p ? P - p : 0, rs) + __mul24(jl, R);
        int ka = __mul24(p, R), kb = N - ka;
#pragma unroll
        for (int k1 = 0; k1 < R; ++k1) {
            const double2 A = u[k1], Bv = p ? w[k1] : make_double2(0.0, 0.0);
            if (ka < out) X[(unsigned)(__mul24(ka, N) + jl)] = sub_i(A, Bv);
            if (p && kb < out) X[(unsigned)(__mul24(kb, N) + jl)] = add_i(A, Bv);
            ka = wrap(ka + P, N);
            kb = wrap(kb + P, N);
        }
    }
}

template <>
__device__ __forceinline__ void prime_store_fwd<0>(const double2* a, double2* __restrict__ X, int N, int out, int n,
                                                   int rs, const PrimeDft& d) {
    const DivF dn = div_by(n), dR{d.R, d.rR};
    for (int i = threadIdx.x; i < n * d.R * (d.H + 1); i += kMrThreads) {
        const int t = dn.quo(i), jl = dn.rem(i, t), p = dR.quo(t), k1 = dR.rem(t, p);
        const int c = __mul24(jl, d.R) + k1, o = __mul24(k1, d.P), pr = __mul24(p, d.R);
        const int ka = wrap(o + pr, N), kb = wrap(o + N - pr, N);
        const double2 A = a[__mul24(p, rs) + c], Bv = p ? a[__mul24(d.P - p, rs) + c] : make_double2(0.0, 0.0);
        if (ka < out) X[(unsigned)(__mul24(ka, N) + jl)] = sub_i(A, Bv);
        if (p && kb < out) X[(unsigned)(__mul24(kb, N) + jl)] = add_i(A, Bv);
    }
}

// Inverse store phase: samples q + j P and P-q + j P of a ring.
template <int RR>
__device__ __forceinline__ void prime_store_inv(const double2* a, double* __restrict__ re, double* __restrict__ im, int N,
                                                int n, int rs, const PrimeDft& d) {
    constexpr int R = RR;
    const DivF dh{d.H + 1, d.rH1};
    const int P = d.P, pm = P & (R - 1);
    for (int i = threadIdx.x; i < n * (d.H + 1); i += kMrThreads) {
        const int jl = dh.quo(i), q = dh.rem(i, jl);
        const double2* u = a + __mul24(q, rs) + __mul24(jl, R);
        const double2* w = a + __mul24(q ? P - q : 0, rs) + __mul24(jl, R);
        const int o = __mul24(jl, N), oy = o + (P - q);
        int c = q & (R - 1), e = (P - q) & (R - 1);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const double2 x = q ? add_i(u[c], w[c]) : u[c];
            re[(unsigned)(o + q + j * P)] = x.x;
            im[(unsigned)(o + q + j * P)] = x.y;
            if (q) {
                const double2 y = sub_i(u[e], w[e]);
                re[(unsigned)(oy + j * P)] = y.x;
                im[(unsigned)(oy + j * P)] = y.y;
            }
            c = (c + pm) & (R - 1);
            e = (e + pm) & (R - 1);
        }
    }
}

template <>
__device__ __forceinline__ void prime_store_inv<0>(const double2* a, double* __restrict__ re, double* __restrict__ im,
                                                   int N, int n, int rs, const PrimeDft& d) {
    const DivF dN{N, d.rN}, dP{d.P, d.rP}, dR{d.R, d.rR};
    for (int i = threadIdx.x; i < n * N; i += kMrThreads) {
        const int k = dP.rem(i), p = k > d.H ? d.P - k : k;
        const double2* u = a + __mul24(dN.quo(i), d.R) + dR.rem(i);
        const double2 A = u[__mul24(p, rs)], Bv = p ? u[__mul24(d.P - p, rs)] : make_double2(0.0, 0.0);
        const double2 v = k > d.H ? sub_i(A, Bv) : add_i(A, Bv);
        re[i] = v.x;
        im[i] = v.y;
    }
}

// One load per thread over an eighth of the tables' lines, issued with the ring
// loads: L2 starts cold, and the K loops would otherwise meet every line's
// first miss in turn.  Neighbouring blocks of an XCD take different eighths.
__device__ __forceinline__ double prime_warm(const double2* tw, const PrimeDft& d) {
    const int lines = (int)(prime_table_doubles(d) / 16);
    const int id = (int)((blockIdx.y * gridDim.x + blockIdx.x) >> 3);
    const int line = min((id & 7) * (lines >> 3) + (int)threadIdx.x, lines - 1);
    return reinterpret_cast<const double*>(tw)[line * 16];
}

__device__ __forceinline__ void prime_phi_fwd(const double* __restrict__ re, const double* __restrict__ im,
                                              double2* __restrict__ X, int N, int lr, int nr,
                                              const double2* __restrict__ tw, int real, unsigned char* smem) {
    double2* a = reinterpret_cast<double2*>(smem);
    const PrimeDft d = *reinterpret_cast<const PrimeDft*>(tw);
    const int rs = nr * d.R + 1;
    int bx = blockIdx.x, f = blockIdx.y;
    xcd_block(bx, f);
    const int j0 = bx * nr, n = min(nr, N - j0);
    const size_t base = ((size_t)f * N + j0) * N;
    const double warm = prime_warm(tw, d);
    if (d.R == 2) {
        prime_load_fwd<2>(a, re + base, im + base, N, n, rs, d);
    } else if (d.R == 4) {
        prime_load_fwd<4>(a, re + base, im + base, N, n, rs, d);
    } else {
        prime_load_fwd<0>(a, re + base, im + base, N, n, rs, d);
        prime_parts<-1>(a, nr, d, tw);
    }
    asm volatile("" ::"v"(warm));
    __syncthreads();
    prime_gemms(a, nr, lr, d, tw);
    X += (size_t)f * N * N + j0;
    const int out = real ? N >> 1 : N;  // REAL data: rows below bw (see k_fphi_fwd)
    if (d.R == 2) prime_store_fwd<2>(a, X, N, out, n, rs, d);
    else if (d.R == 4) prime_store_fwd<4>(a, X, N, out, n, rs, d);
    else prime_store_fwd<0>(a, X, N, out, n, rs, d);
}

__device__ __forceinline__ void prime_phi_inv(const double2* __restrict__ X, double* __restrict__ re,
                                              double* __restrict__ im, int N, int lr, int B, int nr,
                                              const double2* __restrict__ tw, int real, unsigned char* smem) {
    double2* a = reinterpret_cast<double2*>(smem);
    const PrimeDft d = *reinterpret_cast<const PrimeDft*>(tw);
    const int rs = nr * d.R + 1;
    int bx = blockIdx.x, f = blockIdx.y;
    xcd_block(bx, f);
    const int j0 = bx * nr, n = min(nr, N - j0);
    const double warm = prime_warm(tw, d);
    X += (size_t)f * N * N + j0;
    if (d.R == 2) {
        prime_load_inv<2>(a, X, N, B, n, rs, real, d);
    } else if (d.R == 4) {
        prime_load_inv<4>(a, X, N, B, n, rs, real, d);
    } else {
        prime_load_inv<0>(a, X, N, B, n, rs, real, d);
        prime_parts<+1>(a, nr, d, tw);
    }
    asm volatile("" ::"v"(warm));
    __syncthreads();
    prime_gemms(a, nr, lr, d, tw);
    const size_t base = ((size_t)f * N + j0) * N;
    if (d.R == 2) prime_store_inv<2>(a, re + base, im + base, N, n, rs, d);
    else if (d.R == 4) prime_store_inv<4>(a, re + base, im + base, N, n, rs, d);
    else prime_store_inv<0>(a, re + base, im + base, N, n, rs, d);
}

}  // namespace s2
