// K-chunked dense FP64 Legendre GEMMs (see s2_naive64.h) and their launches.
#pragma once

#include <algorithm>
#include <type_traits>

#include "s2_naive64.h"

namespace s2 {

// ---------------------------------------------------------------------------
// K-chunked: 16 CT columns per block, tables and data through LDS
// ---------------------------------------------------------------------------
// A block runs an order pair (m, bw-1-m) (about bw+1 degrees, so blocks are
// alike) for 64 data columns (CT = 4 column tiles), or 32 (CT = 2) for calls of
// fewer than 64 fields (above bw = 256, 16).  Table stages go global -> LDS by DMA, the data
// through registers (folded, in the forward) into LDS, both in MFMA operand
// order: every LDS read is 64 consecutive doubles.  An FP64 16x16x4 MFMA
// holds its SIMD's matrix core for 64 cycles and needs one 512-byte operand
// read, a quarter of the LDS rate with all four SIMDs busy, so the kernel is
// bound by the matrix cores once four waves per SIMD cover the stages'
// latency (bw=256 x 1024 forward: matrix cores busy 70% of 1.57 ms, 5.8 GB of HBM
// traffic at 3.7 TB/s; 44 TF/s, 49 with the padding, of 71.9 that a large library
// product reaches);
// hence 128 VGPRs, two stage buffers within 80 KiB of LDS and (CT = 4,
// bw <= 256) two blocks per CU.
//
// Data tiles are stored with the 16 columns of a K row permuted (the pair
// index, forward, or the column index, inverse, XOR a number from the K
// step and the row's high bit): the staging lanes of one LDS write cycle hold
// different K rows of the same columns, which would meet in the same banks.
__device__ __forceinline__ int n64_swz(int ks, int kq) { return (kq >> 1) + 2 * ks; }

// Forward.  Both orders of the pair run side by side, so that every stage of
// two K steps has the same work (order after order, the light order's stages
// have too few MFMAs to cover their loads).  Wave (c, p, h) owns column tile
// c, parity p and the h-th of H parts (two for bw > 256) of the pair's nt = NT H
// degree tiles: tiles below nh take the data of order m, the others of order
// bw-1-m.  Where that changes is fixed in each instance of the K loop
// (selected per tile and K step, it costs two VALU instructions a MFMA).
constexpr int n64_fwd_kd(int ct) { return 512 * ct; }  // doubles of a data stage: [2 K steps][2 orders][2 parities][CT][64]
constexpr int n64_fwd_tb(int nt) { return 2 * 2 * nt * 64; }  // of a table stage
constexpr int n64_fwd_lds(int nt, int ct) { return 2 * (n64_fwd_kd(ct) + n64_fwd_tb(nt)); }

template <int NT, int H, int CT>
__device__ __forceinline__ void naive64_fwd_kc(const double2* __restrict__ X, const double* __restrict__ NF,
                                               const GemmMeta& g, double* __restrict__ cre, double* __restrict__ cim,
                                               int m, int cb, int B, int F, int fmt, double* sm) {
    constexpr int NW = 2 * CT * H, KD = n64_fwd_kd(CT), nt = NT * H, TB = n64_fwd_tb(nt), LC = CT == 4 ? 2 : 1;
    static_assert(CT == 1 << LC, "CT is 2 or 4");
    const int N = 2 * B, nh = g.n0, ml = B - 1 - m;
    const int tid = threadIdx.x, lane = tid & 63, wave = n64_uniform(tid >> 6);
    const int c = wave & (CT - 1), p = (wave >> LC) & 1, t0 = (wave >> (LC + 1)) * NT;
    const int x16 = lane & 15, kq = lane >> 4;
    double* dat = sm;
    double* tab = sm + 2 * KD;
    const char* tsrc = reinterpret_cast<const char*>(NF + g.offF);
    auto stage = [&](int s, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < (2 * nt + NW - 1) / NW; ++k) {
            const int u = wave + NW * k;
            if ((k + 1) * NW <= 2 * nt || u < 2 * nt)
                n64_dma(tsrc + (size_t)s * (TB * 8) + u * 1024, lane * 16, tab + buf * TB + u * 128);
        }
    };
    // data staging: thread -> order o of the pair (waves CT .. 2 CT - 1 its second; further
    // waves repeat), complex row rr (columns 2rr, 2rr+1) and ring jj of an 8-ring stage;
    // offsets from the block's first field
    const int o = (wave >> LC) & 1, rr = (tid >> 3) & (8 * CT - 1), jj = tid & 7, nst = n64_bp(B) >> 3;
    const int mx = o ? ml : m, cpx = mix_cpf(mx, fmt), fb = min(cb * 16 * CT >> (cpx >> 1), F - 1);
    const char* xbase = reinterpret_cast<const char*>(X + (size_t)fb * N * N);
    unsigned oa, ob;
    {
        const int col = cb * 16 * CT + 2 * rr, k = col < F * cpx ? col : fb * cpx;
        const int f = k >> (cpx >> 1), rem = k & (cpx - 1);  // cpx is 2 or 4
        const unsigned row = (unsigned)((f - fb) * N + n64_row(rem, mx, N)) * N;
        oa = (row + jj) * 16u;
        ob = (row + N - 1 - jj) * 16u;
    }
    dvec2 va, vb;
    auto fetch = [&](int s) __attribute__((always_inline)) {
        va = n64_ld<dvec2>(xbase + s * 128, oa);
        vb = n64_ld<dvec2>(xbase - s * 128, ob);
    };
    double* dput = dat + (((jj >> 2) * 2 + o) * 2 * CT + (rr >> 3)) * 64 + (jj & 3) * 16 +
                   2 * ((rr & 7) ^ n64_swz(jj >> 2, jj & 3));
    auto put = [&](int buf) __attribute__((always_inline)) {
        if (H == 1 || wave < 2 * CT) {
            *reinterpret_cast<dvec2*>(dput + buf * KD) = va + vb;
            *reinterpret_cast<dvec2*>(dput + buf * KD + CT * 64) = va - vb;
        }
    };
    dvec4 acc[NT] = {};
    stage(0, 0);
    fetch(0);
    put(0);
    __builtin_amdgcn_s_waitcnt(0);  // this wave's LDS transfers have landed
    __syncthreads();
    const double* da = dat + (p * CT + c) * 64 + kq * 16 + (x16 & 1);
    const double* d0 = da + 2 * ((x16 >> 1) ^ n64_swz(0, kq));
    const double* d1 = da + 2 * ((x16 >> 1) ^ n64_swz(1, kq)) + 256 * CT;
    const double* ta = tab + (p * nt + t0) * 64 + lane;
    constexpr int G = NT <= 4 ? NT : (NT + 2) / 3, NG = (NT + G - 1) / G;  // tiles read one group ahead
    auto loop = [&](auto nhc) __attribute__((always_inline)) {
        constexpr int NH = decltype(nhc)::value;  // this wave's tiles of order m
        auto run = [&](int s, int buf, bool more) __attribute__((always_inline)) {  // stage s, in buffer buf
            if (more) {
                stage(s + 1, buf ^ 1);
                fetch(s + 1);
            }
            asm volatile("" ::: "memory");  // the loads stay ahead of the MFMAs
            const double* t = ta + buf * TB;
            double ah[2], al[2], b[2][G];
            if (NH > 0) ah[0] = d0[buf * KD], ah[1] = d1[buf * KD];
            if (NH < NT) al[0] = d0[buf * KD + 128 * CT], al[1] = d1[buf * KD + 128 * CT];
#pragma unroll
            for (int i = 0; i < G; ++i) b[0][i] = t[i * 64];
#pragma unroll
            for (int q = 0; q < 2 * NG; ++q) {
                const int k = q / NG, i0 = (q % NG) * G;
                if (q + 1 < 2 * NG) {
                    const int k1 = (q + 1) / NG, i1 = ((q + 1) % NG) * G;
#pragma unroll
                    for (int i = 0; i < G; ++i)
                        if (i1 + i < NT) b[(q + 1) & 1][i] = t[k1 * 2 * nt * 64 + (i1 + i) * 64];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < G; ++i)
                    if (i0 + i < NT)
                        acc[i0 + i] = Mma<double>::mma(i0 + i < NH ? ah[k] : al[k], b[q & 1][i], acc[i0 + i]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (more) put(buf ^ 1);
            __builtin_amdgcn_s_waitcnt(0);  // this wave's LDS transfers (stage s + 1) have landed
            __syncthreads();
        };
        for (int s = 0; s < nst; s += 2) {  // nst is even
            run(s, 0, true);
            run(s + 1, 1, s + 2 < nst);
        }
    };
    // a whole pair has at least as many tiles of the heavier order m, and one of the other
    constexpr int NH0 = H == 1 ? (NT + 1) / 2 : 0, NH1 = H == 1 ? NT - 1 : NT;
#define S2_N64_NH(n) \
    case n:          \
        if constexpr (n >= NH0 && n <= NH1) loop(std::integral_constant<int, n>{}); \
        break;
    switch (min(NT, nh - t0)) {
        S2_N64_NH(0)
        S2_N64_NH(1)
        S2_N64_NH(2)
        S2_N64_NH(3)
        S2_N64_NH(4)
        S2_N64_NH(5)
        S2_N64_NH(6)
        S2_N64_NH(7)
        S2_N64_NH(8)
        S2_N64_NH(9)
        default: break;
    }
#undef S2_N64_NH
    // the thread index through an empty asm: the store arithmetic stays after the K loop
    int tix = threadIdx.x;
    asm volatile("" : "+v"(tix));
    const int el = tix & 63, ew = n64_uniform(tix >> 6), et0 = (ew >> (LC + 1)) * NT, ep = (ew >> LC) & 1;
    for (int q = 0; q < 2; ++q) {
        const int mm = q ? ml : m, L = B - mm, tb = q ? nh : 0, te = q ? nh + mix_n0(ml, B) : nh;
        if (q && ml == m) break;  // odd bw: the middle order pairs with itself
        const int cpf = mix_cpf(mm, fmt), ncols = F * cpf;
        if (et0 >= te || et0 + NT <= tb) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int col = (cb * CT + (ew & (CT - 1))) * 16 + Mma<double>::row(el, r);
            if (col >= ncols) continue;
            const N64Out w = n64_out(col, mm, cpf, B, fmt, cre, cim);
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                const int t = et0 + i, d = 2 * (16 * (t - tb) + (el & 15)) + ep;
                if (t < tb || t >= te || d >= L) continue;
                w.o1[d] = w.s1 * acc[i][r];
                if (w.o2) w.o2[d] = w.s2 * acc[i][r];
            }
        }
    }
}

// Inverse: 128 CT threads, 2 JT of the ring tiles (from tile rz); wave (c, h)
// owns column tile c and JT ring tiles, both parities, so E +- O stay in
// its registers.  Stages of two K steps (8 degrees of each parity); the
// stages of the pair's two orders follow each other without a gap.
constexpr int n64_inv_tb(int jt) { return 8 * jt * 64; }  // doubles of a table stage: [2 K steps][2 parities][2 JT][64]
constexpr int n64_inv_kd(int ct) { return 256 * ct; }      // of a data stage: [2][2][CT][64]
constexpr int n64_inv_lds(int jt, int ct) { return 2 * (n64_inv_kd(ct) + n64_inv_tb(jt)); }

template <int JT, int CT>
__device__ __forceinline__ void naive64_inv_kc(const double* __restrict__ cre, const double* __restrict__ cim,
                                               const double* __restrict__ NI, const GemmMeta* __restrict__ meta,
                                               double2* __restrict__ X, int m, int cb, int rz, int B, int F, int fmt,
                                               double* sm) {
    constexpr int TB = n64_inv_tb(JT), KD = n64_inv_kd(CT), NW = 2 * CT, NK = (4 * JT + NW - 1) / NW, LC = CT == 4 ? 2 : 1;
    static_assert(CT == 1 << LC, "CT is 2 or 4");
    const int RT = n64_bp(B) >> 4, ml = B - 1 - m;
    const int n1 = meta[2 * m].ki >> 1, nst = ml == m ? n1 : n1 + (meta[2 * ml].ki >> 1);
    const char* ni1 = reinterpret_cast<const char*>(NI + meta[2 * m].offI);
    const char* ni2 = reinterpret_cast<const char*>(NI + meta[2 * ml].offI);
    const int tid = threadIdx.x, lane = tid & 63, wave = n64_uniform(tid >> 6);
    const int c = wave & (CT - 1), h = wave >> LC, x16 = lane & 15, kq = lane >> 4;
    double* dat = sm;
    double* tab = sm + 2 * KD;
    unsigned ot[NK];  // this lane's offsets in a table stage (two tiles per wave transfer)
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        const int u = min(wave + NW * k, 4 * JT - 1), q = u / JT, rt = min(rz + 2 * (u - q * JT) + (lane >> 5), RT - 1);
        ot[k] = (unsigned)((q * RT + rt) * 64 + (lane & 31) * 2) * 8u;
    }
    // data staging: thread -> column cc, degree offsets 16s + 2e, 16s + 2e + 1
    const int cc = tid >> 3, e = tid & 7;
    const double *cp1, *cp2;
    unsigned sg1, sg2;
    auto column = [&](int mm, const double*& cp, unsigned& sg) __attribute__((always_inline)) {
        const int cpf = mix_cpf(mm, fmt), col = cb * 16 * CT + cc, k = col < F * cpf ? col : 0;
        const int f = k >> (cpf >> 1), rem = k & (cpf - 1);
        cp = ((rem & 1) ? cim : cre) + (size_t)f * B * B + index_of_coeff((rem >> 1) ? -mm : mm, mm, B) + 2 * e;
        sg = ((rem >> 1) && (mm & 1)) ? 0x80000000u : 0u;  // rows -m carry (-1)^m
    };
    column(m, cp1, sg1);
    column(ml, cp2, sg2);
    auto stage = [&](int s, int buf) __attribute__((always_inline)) {
        const char* src = s < n1 ? ni1 + (size_t)s * (RT * 2048) : ni2 + (size_t)(s - n1) * (RT * 2048);
#pragma unroll
        for (int k = 0; k < NK; ++k)
            if ((k + 1) * NW <= 4 * JT || wave + NW * k < 4 * JT)
                n64_dma(src, ot[k], tab + buf * TB + (wave + NW * k) * 128);
    };
    dpair8 v;
    auto fetch = [&](int s) __attribute__((always_inline)) {
        const int sl = s < n1 ? s : s - n1, L = B - (s < n1 ? m : ml);
        const double* cp = s < n1 ? cp1 : cp2;
        if (16 * sl + 16 <= L) {
            v = *reinterpret_cast<const dpair8*>(cp + 16 * sl);
        } else {  // the run ends in this stage
            const int d = 16 * sl + 2 * e;
            v = *reinterpret_cast<const dpair8*>(cp + (min(d, L - 2) - 2 * e));  // clamped as in naive64_inv_direct
            v = dpair8{d + 1 < L ? v.x : d < L ? v.y : 0.0, d + 1 < L ? v.y : 0.0};
        }
    };
    double* dput = dat + ((e >> 2) * 2 * CT + (cc >> 4)) * 64 + (e & 3) * 16 +
                   ((((cc & 15) >> 2) + 4 * (cc & 3)) ^ n64_swz(e >> 2, e & 3));
    auto flip = [](double x, unsigned sg) __attribute__((always_inline)) {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
        return __builtin_bit_cast(double, b ^ ((unsigned long long)sg << 32));
    };
    auto put = [&](int s, int buf) __attribute__((always_inline)) {
        const unsigned sg = s < n1 ? sg1 : sg2;
        dput[buf * KD] = flip(v.x, sg);
        dput[buf * KD + CT * 64] = flip(v.y, sg);
    };
    stage(0, 0);
    fetch(0);
    put(0, 0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const double* d0 = dat + c * 64 + kq * 16 + (x16 ^ n64_swz(0, kq));
    const double* d1 = dat + c * 64 + kq * 16 + (x16 ^ n64_swz(1, kq)) + 128 * CT;
    const double* ta = tab + h * JT * 64 + lane;
    dvec4 acc[2][JT] = {};
    auto run = [&](int s, int buf) __attribute__((always_inline)) {  // stage s, in buffer buf
        if (s + 1 < nst) {
            stage(s + 1, buf ^ 1);
            fetch(s + 1);
        }
        asm volatile("" ::: "memory");  // the loads stay ahead of the MFMAs
        const double* t = ta + buf * TB;
        double a[4], b[2][JT];
        a[0] = d0[buf * KD];
        a[1] = d0[buf * KD + 64 * CT];
        a[2] = d1[buf * KD];
        a[3] = d1[buf * KD + 64 * CT];
#pragma unroll
        for (int i = 0; i < JT; ++i) b[0][i] = t[i * 64];
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // K step q/2, parity q%2; tiles read one group ahead
            if (q < 3)
#pragma unroll
                for (int i = 0; i < JT; ++i) b[(q + 1) & 1][i] = t[(q + 1) * 2 * JT * 64 + i * 64];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < JT; ++i) acc[q & 1][i] = Mma<double>::mma(a[q], b[q & 1][i], acc[q & 1][i]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (s + 1 < nst) put(s + 1, buf ^ 1);
        __builtin_amdgcn_s_waitcnt(0);  // this wave's LDS transfers (stage s + 1) have landed
        __syncthreads();
        if (s + 1 != n1 && s + 1 != nst) return;
        // the end of an order: its sums leave, the next one's start at zero
        const int mm = s + 1 == n1 ? m : ml, cpf = mix_cpf(mm, fmt);
        int tix = threadIdx.x;  // as in the forward epilogue
        asm volatile("" : "+v"(tix));
        const int el = tix & 63, ew = tix >> 6;
#pragma unroll
        for (int r2 = 0; r2 < 2; ++r2) {
            const int col = (cb * CT + (ew & (CT - 1))) * 16 + 4 * (el >> 4) + 2 * r2;
            if (col < F * cpf)
                n64_inv_store<JT>(acc[0], acc[1], X, mm, col, 2 * r2, 1.0, 16 * (rz + (ew >> LC) * JT) + (el & 15), B,
                                  cpf);
        }
#pragma unroll
        for (int i = 0; i < JT; ++i) acc[0][i] = acc[1][i] = dvec4{0.0, 0.0, 0.0, 0.0};
    };
    for (int s = 0;; s += 2) {
        run(s, 0);
        if (s + 1 == nst) break;
        run(s + 1, 1);
        if (s + 2 == nst) break;
    }
}

// ---------------------------------------------------------------------------
// kernels and launches
// ---------------------------------------------------------------------------
template <int H, int CT>
__device__ __forceinline__ void naive64_fwd_block(const double2* __restrict__ X, const double* __restrict__ NF,
                                                  const GemmMeta* __restrict__ meta, double* __restrict__ cre,
                                                  double* __restrict__ cim, int B, int F, int fmt, int nb, double* sm) {
    int m, cb;
    mix_pair(nb, m, cb);
    if (m >= mix_npairs(B)) return;
    const GemmMeta g = meta[2 * m];
    switch (g.Kf / H) {  // tiles per wave, bw in [128, 512]
        case 5: naive64_fwd_kc<5, H, CT>(X, NF, g, cre, cim, m, cb, B, F, fmt, sm); break;
        case 6: naive64_fwd_kc<6, H, CT>(X, NF, g, cre, cim, m, cb, B, F, fmt, sm); break;
        case 7: naive64_fwd_kc<7, H, CT>(X, NF, g, cre, cim, m, cb, B, F, fmt, sm); break;
        case 8: naive64_fwd_kc<8, H, CT>(X, NF, g, cre, cim, m, cb, B, F, fmt, sm); break;
        case 9: naive64_fwd_kc<9, H, CT>(X, NF, g, cre, cim, m, cb, B, F, fmt, sm); break;
        default: break;  // none (refused by n64_fwd_kc_launch)
    }
}

// 64 columns per block: 512 threads up to bw = 256, 1024 above
template <typename R, int NTH>
__global__ __launch_bounds__(NTH) __attribute__((amdgpu_waves_per_eu(4))) void k_gemm_fwd_kc(
    const double2* __restrict__ X, const R* __restrict__ NF, const GemmMeta* __restrict__ meta,
    double* __restrict__ cre, double* __restrict__ cim, int B, int F, int fmt, int nb) {
    extern __shared__ __align__(16) unsigned char smem[];
    naive64_fwd_block<NTH / 512, 4>(X, NF, meta, cre, cim, B, F, fmt, nb, reinterpret_cast<double*>(smem));
}

// A direct launch: grid (items / 4, orders rounded up to 8), an item per wave.
__device__ __forceinline__ bool n64_item(int B, int& m, int& item) {
    int bx;
    xcd_block_m(bx, m);
    item = bx * (kThreads / 64) + n64_uniform(threadIdx.x >> 6);
    return m < B;
}

// Fewer fields.  NTW > 0: direct, NTW degree tiles per wave.  NTW < 0:
// K-chunked with 32 columns per block, 256 threads up to bw = 256 (NTW = -1),
// 512 above (-2).
template <typename R, bool GEN, int CT, int NTW>
__global__ __launch_bounds__(NTW > 0 ? kThreads : 128 * CT * -NTW)
    __attribute__((amdgpu_waves_per_eu(NTW > 0 ? 1 : 4))) void k_gemm_fwd(
        const double2* __restrict__ X, const R* __restrict__ NF, const GemmMeta* __restrict__ meta,
        double* __restrict__ cre, double* __restrict__ cim, int B, int F, int fmt, int nb) {
    if constexpr (NTW > 0) {
        int m, item;
        if (n64_item(B, m, item)) naive64_fwd_direct<CT, NTW>(X, NF, meta, cre, cim, m, item, B, F, fmt);
    } else {
        extern __shared__ __align__(16) unsigned char smem[];
        naive64_fwd_block<-NTW, CT>(X, NF, meta, cre, cim, B, F, fmt, nb, reinterpret_cast<double*>(smem));
    }
}

template <int H, int CT>
void n64_fwd_kc_launch(const DevConsts& c, const GemmTables& g, const double2* X, double* cre, double* cim, int F,
                       Fmt fmt, hipStream_t s) {
    const int B = c.bw, nb = ((fmt == Fmt::Complex ? 4 : 2) * F + 16 * CT - 1) / (16 * CT);
    int nt = 0;
    for (int q = 0; q < mix_npairs(B); ++q) {
        const int n = n64_nt(q, B);
        // the instances of naive64_fwd_block: 5 to 9 tiles per wave (every bw in [128, 512])
        if (n < 5 * H || n > 9 * H) throw ArgError{"dense FP64 forward: no K-chunked kernel at this bandwidth"};
        nt = std::max(nt, n);
    }
    const dim3 grid(mix_npairs8(B) * nb);
    const size_t lds = sizeof(double) * n64_fwd_lds(nt, CT);
    const double* nf = (const double*)g.af;
    const GemmMeta* meta = g.meta;
    if constexpr (CT == 4)
        launch_lds(k_gemm_fwd_kc<double, 512 * H>, grid, 512 * H, lds, s, X, nf, meta, cre, cim, B, F, (int)fmt, nb);
    else
        launch_lds(k_gemm_fwd<double, false, CT, -H>, grid, 128 * CT * H, lds, s, X, nf, meta, cre, cim, B, F, (int)fmt,
                   nb);
}

}  // namespace s2
