// Dense FP64 Legendre GEMMs (s2_naive64.h): tables, the inverse and direct
// kernels, and the choice between them.
#include <cmath>

#include "s2_naive64_kc.h"

namespace s2 {

extern template void n64_fwd_kc_launch<1, 4>(const DevConsts&, const GemmTables&, const double2*, double*, double*, int,
                                             Fmt, hipStream_t);
extern template void n64_fwd_kc_launch<2, 4>(const DevConsts&, const GemmTables&, const double2*, double*, double*, int,
                                             Fmt, hipStream_t);
extern template void n64_fwd_kc_launch<1, 2>(const DevConsts&, const GemmTables&, const double2*, double*, double*, int,
                                             Fmt, hipStream_t);
extern template void n64_fwd_kc_launch<2, 2>(const DevConsts&, const GemmTables&, const double2*, double*, double*, int,
                                             Fmt, hipStream_t);

__global__ void k_naive64_pack(const double* __restrict__ w, const GemmMeta* __restrict__ meta,
                               double* __restrict__ NF, double* __restrict__ NI, int B) {
    const int m = blockIdx.x, N = 2 * B, RT = n64_bp(B) >> 4;
    const GemmMeta g = meta[2 * m];
    const int nt = g.Kf;
    const double cm = (m == 0) ? 0.0 : pmm_coeff(m);
    for (int j = threadIdx.x; j < B; j += blockDim.x) {
        const double th = (2.0 * j + 1.0) * M_PI / (2.0 * N);
        const double x = cos(th), wj = w[j];
        double cur = (m == 0) ? 0.70710678118654752440 : cm * pow(sin(th), (double)m);
        double prev = 0.0;
        double* nf = NF + g.offF + (size_t)(j >> 2) * 2 * nt * 64 + (j & 3) * 16;
        double* ni = NI + g.offI + (j >> 4) * 64 + (j & 15);
        for (int l = m; l < B; ++l) {
            const int p = (l - m) & 1, i = (l - m) >> 1;
            nf[(p * nt + (i >> 4)) * 64 + (i & 15)] = cur * wj;
            ni[((size_t)(i >> 2) * 2 + p) * RT * 64 + (i & 3) * 16] = cur * 0.39894228040143267794;
            if (l + 1 < B) {
                const double nx = l2_an(m, l) * (cur * x) + l2_cn(m, l) * prev;
                prev = cur;
                cur = nx;
            }
        }
    }
}

// Odd bw, seminaive orders: the reference's transposed tables drop the last
// entry of some cosine rows (Transpose_RowSize, cospml.c:270-288), so its
// synthesis of degree bw-1 is the cosine series without those terms.  That
// degree's table row is summed here from the transposed table, grid (cutoff).
__global__ void k_naive64_short_row(const double* __restrict__ TT, const long* __restrict__ toff,
                                    const GemmMeta* __restrict__ meta, double* __restrict__ NI, int B) {
    extern __shared__ __align__(16) unsigned char smem[];
    double* fc = reinterpret_cast<double*>(smem);
    const int m = blockIdx.x, N = 2 * B, RT = n64_bp(B) >> 4;
    const double* tt = TT + toff[m];
    const double s1 = 0.5 / sqrt((double)B);
    for (int c = threadIdx.x; c < B; c += blockDim.x) {
        long at = 0;
        for (int r = 0; r < c; ++r) at += transpose_row_size(r, m, B);
        const int d = B - 1 - (m + transpose_first(c, m)), rs = transpose_row_size(c, m, B);
        double v = 0.0;
        if (d >= 0 && !(d & 1) && (d >> 1) < rs) v = tt[at + (d >> 1)] * (c == 0 ? 1.0 / sqrt((double)N) : 2.0 * s1);
        fc[c] = v;
    }
    __syncthreads();
    const GemmMeta g = meta[2 * m];
    const int p = (B - 1 - m) & 1, i = (B - 1 - m) >> 1;
    for (int j = threadIdx.x; j < B; j += blockDim.x) {
        double v = 0.0;
        for (int c = 0; c < B; ++c) v += fc[c] * cospi((double)((long)c * (2 * j + 1) % (4 * N)) / (2.0 * N));
        if (m & 1) v *= sinpi((2.0 * j + 1.0) / (2.0 * N));
        NI[g.offI + (((size_t)(i >> 2) * 2 + p) * RT + (j >> 4)) * 64 + (i & 3) * 16 + (j & 15)] =
            v * 0.39894228040143267794;
    }
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
// direct: CT column tiles and RTW ring tiles per wave
template <typename R, bool GEN, int CT, int RTW>
__global__ __launch_bounds__(kThreads) void k_gemm_inv(const double* __restrict__ cre, const double* __restrict__ cim,
                                                       const R* __restrict__ NI, const GemmMeta* __restrict__ meta,
                                                       double2* __restrict__ X, int B, int F, int fmt) {
    int m, item;
    if (n64_item(B, m, item)) naive64_inv_direct<CT, RTW>(cre, cim, NI, meta, X, m, item, B, F, fmt);
}

template <int CT>
__device__ __forceinline__ void naive64_inv_block(const double* __restrict__ cre, const double* __restrict__ cim,
                                                  const double* __restrict__ NI, const GemmMeta* __restrict__ meta,
                                                  double2* __restrict__ X, int B, int F, int fmt, int nb, int nz, int jt,
                                                  double* sm) {
    int m, cz;
    mix_pair(nb * nz, m, cz);
    if (m >= mix_npairs(B)) return;
    const int cb = cz / nz, rz = (cz - cb * nz) * 2 * jt;
    switch (jt) {
        case 1: naive64_inv_kc<1, CT>(cre, cim, NI, meta, X, m, cb, rz, B, F, fmt, sm); break;
        case 2: naive64_inv_kc<2, CT>(cre, cim, NI, meta, X, m, cb, rz, B, F, fmt, sm); break;
        case 3: naive64_inv_kc<3, CT>(cre, cim, NI, meta, X, m, cb, rz, B, F, fmt, sm); break;
        default: naive64_inv_kc<4, CT>(cre, cim, NI, meta, X, m, cb, rz, B, F, fmt, sm); break;
    }
}
template <typename R, int NTH>
__global__ __launch_bounds__(NTH) __attribute__((amdgpu_waves_per_eu(4))) void k_gemm_inv_kc(
    const double* __restrict__ cre, const double* __restrict__ cim, const R* __restrict__ NI,
    const GemmMeta* __restrict__ meta, double2* __restrict__ X, int B, int F, int fmt, int nb, int nz, int jt) {
    extern __shared__ __align__(16) unsigned char smem[];
    naive64_inv_block<NTH / 128>(cre, cim, NI, meta, X, B, F, fmt, nb, nz, jt, reinterpret_cast<double*>(smem));
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// At bw = 512 the tables take 0.60 GB (forward) and 0.55 GB; at 1024 they would
// take over 4.3 GB each, which the few fields that fit beside them could not stream as fast
// as the seminaive tables' 1.4 GB.
bool n64_supported(int bw, int prec) { return prec == 0 && bw >= 16 && bw <= 512; }

// Fields per call (the plan's largest) from which the dense tables beat the
// seminaive ones (DCT included): always up to bw = 320; above, one to three
// fields are bound by the table stream, three times as long here (us per forward
// / inverse, dense against seminaive: bw=300 x1 35 / 24 against 38 / 36, bw=400 x2
// 77 / 69 against 63 / 64, x4 82 / 75 against 87 / 88, bw=512 x2 143 / 110
// against 104 / 98, x4 152 / 118 against 144 / 128, x8 173 / 131 against
// 217 / 210).  A plan holds one kind and runs its smaller calls on it as well
// (one field, dense against seminaive: bw=400 85 / 64 against 58 / 57, bw=512
// 147 / 124 against 72 / 80): with both, a field's last bits depended on its
// call's field count, and a plan held two table sets (bw=512 x8 2201 -> 1670 MB).
int n64_min_fields(int bw) { return bw <= 320 ? 1 : 4; }

void n64_tables_create(GemmTables& g, const DevTables& t, const DevConsts& c, hipStream_t s) {
    const int B = t.bw;
    g.bw = B;
    g.prec = 0;
    g.cut = 0;
    g.gen = !gemm_pow2(B);
    g.n64 = true;
    g.h_meta.assign(2 * B, GemmMeta{});
    long of = 0, oi = 0;
    for (int q = 0; q < mix_npairs(B); ++q) {
        const int nt = n64_nt(q, B);
        for (int o = 0; o < (2 * q == B - 1 ? 1 : 2); ++o) {
            const int m = o ? B - 1 - q : q;
            GemmMeta& e = g.h_meta[m * 2];  // both parities share an entry
            e.Lp = gm_lp(m, 0, B);
            e.Kf = nt;
            e.n0 = mix_n0(m, B);
            e.ki = n64_ki(m, B);
            e.offF = of + (o ? mix_n0(q, B) * 64 : 0);
            e.offI = oi;
            oi += (long)e.ki * 2 * (n64_bp(B) / 16) * 64;
        }
        of += (long)(n64_bp(B) / 4) * 2 * nt * 64;
    }
    g.nf = of;
    g.ni = oi;
    S2_HIP(hipMalloc(&g.meta, sizeof(GemmMeta) * 2 * B));
    S2_HIP(hipMalloc(&g.af, sizeof(double) * of));
    S2_HIP(hipMalloc(&g.ai, sizeof(double) * oi));
    S2_HIP(hipMemsetAsync(g.af, 0, sizeof(double) * of, s));
    S2_HIP(hipMemsetAsync(g.ai, 0, sizeof(double) * oi, s));
    S2_HIP(hipMemcpyAsync(g.meta, g.h_meta.data(), sizeof(GemmMeta) * 2 * B, hipMemcpyHostToDevice, s));
    k_naive64_pack<<<B, std::min(512, (B + 63) / 64 * 64), 0, s>>>(c.w_naive, g.meta, (double*)g.af, (double*)g.ai, B);
    S2_HIP(hipGetLastError());
    if ((B & 1) && t.cutoff > 0) {
        k_naive64_short_row<<<t.cutoff, 256, sizeof(double) * B, s>>>(t.inv, t.off, g.meta, (double*)g.ai, B);
        S2_HIP(hipGetLastError());
    }
    S2_HIP(hipStreamSynchronize(s));
}

int n64_cols(int F, Fmt fmt) { return (fmt == Fmt::Complex ? 4 : 2) * F; }

// Columns per block of the K-chunked kernels, 0: the direct ones.  Measured,
// us forward / inverse: direct against 32 columns bw=128 x16 16 / 14, 18 / 17,
// x32 26 / 19, 22 / 18; bw=256 x4 24 / 20, 34 / 23, x8 37 / 25, 38 / 24, x16
// 72 / 46, 45 / 39; bw=300 x4 46 / 32, 47 / 33; 32 against 64 columns bw=256 x8
// 38 / 24, 52 / 31, x32 63 / 65, 63 / 59; bw=512 x8 173 / 131, 185 / 168, x16
// 257 / 192, 233 / 187.  (bw = 100 x128 direct: 44 / 40.)  These are COMPLEX
// calls; REAL ones, of half the columns, follow the same lines in fields.
static int n64_kc_cols(int B, int F) {
    if (B < 128 || (long)F * B * B < 300000) return 0;
    return F >= 64 || (B > 256 && F >= 16) ? 64 : 32;
}
// A call of one column tile (at most 16 columns, whatever the format) fills half
// of a 32-column block: the direct kernels are faster, in the forward until the
// table stream outgrows them, by columns x bw^2, and in the inverse to bw = 480
// (whole calls, us, 32 columns / direct: forward, REAL, bw=256 x8 48.5 / 37.8,
// bw=320 x4 60.7 / 53.5, bw=340 x7 87.6 / 90.3, COMPLEX bw=300 x4 62.4 / 56.1,
// bw=352 x4 80.9 / 81.7; inverse, COMPLEX, bw=321 x4 73 / 62, bw=400 x4 117 / 105,
// bw=448 x4 136 / 133, bw=500 x4 171 / 175, bw=512 x4 181 / 196, REAL bw=400 x4
// 111 / 94).  Past bw = 384 the forward's table exceeds the 256 MB memory-side
// cache, and the direct kernel's waves keep too little of the HBM stream in
// flight (one field: bw=360 71 / 55, bw=400 85 / 129, bw=512 147 / 206).
static int n64_fwd_kc_cols(int B, int F, int cols) {
    if (B > 384) return std::max(32, n64_kc_cols(B, F));
    return cols <= 16 && (long)cols * B * B < 1600000 ? 0 : n64_kc_cols(B, F);
}
static int n64_inv_kc_cols(int B, int F, int cols) { return cols <= 16 && B < 480 ? 0 : n64_kc_cols(B, F); }

// Column tiles per wave of the direct kernels: the tuned ones for calls of as
// many data columns as they were timed at, else the rule (its figures beside
// the launches).
static int n64_fwd_ct(const GemmTables& g, int cols) {
    return g.t_cols == cols ? g.t_ct : g.bw > 32 && cols > 512 ? 2 : 1;
}
static int n64_inv_ct(const GemmTables& g, int cols) { return g.t_cols == cols ? g.t_ncb / 16 : cols > 256 ? 2 : 1; }

// Choices of a call: (16 x column tiles per wave of the inverse, column tiles
// of the forward) where a direct kernel serves it, the rule's first.  The
// K-chunked kernels have nothing to choose: their columns per block, one column
// tile per wave.
std::vector<std::pair<int, int>> n64_tile_choices(const GemmTables& g, int F, Fmt fmt) {
    const int cols = n64_cols(F, fmt), kf = n64_fwd_kc_cols(g.bw, F, cols), ki = n64_inv_kc_cols(g.bw, F, cols);
    if (kf && ki) return {{ki, 1}};
    GemmTables rule;
    rule.bw = g.bw;
    const int f0 = kf ? 1 : n64_fwd_ct(rule, cols), i0 = n64_inv_ct(rule, cols);
    std::vector<std::pair<int, int>> v;
    for (int i : {i0, 3 - i0})
        for (int f : {f0, 3 - f0})
            if ((f == f0 || !kf) && (i == i0 || !ki)) v.push_back({16 * i, f});
    return v;
}

template <int CT, int NTW>
static void n64_fwd_direct(const DevConsts& c, const GemmTables& g, const double2* X, double* cre, double* cim, int F,
                           Fmt fmt, hipStream_t s) {
    const int B = c.bw;
    const int items = (mix_n0(0, B) + NTW - 1) / NTW * ((n64_cols(F, fmt) + 16 * CT - 1) / (16 * CT));
    launch_lds(k_gemm_fwd<double, false, CT, NTW>, dim3((items + 3) / 4, (B + 7) & ~7), kThreads, 0, s, X,
               (const double*)g.af, (const GemmMeta*)g.meta, cre, cim, B, F, (int)fmt, 0);
}

template <int CT, int RTW>
static void n64_inv_direct(const DevConsts& c, const GemmTables& g, const double* cre, const double* cim, double2* X,
                           int F, Fmt fmt, hipStream_t s) {
    const int B = c.bw;
    const int items = (n64_bp(B) / 16 + RTW - 1) / RTW * ((n64_cols(F, fmt) + 16 * CT - 1) / (16 * CT));
    launch_lds(k_gemm_inv<double, false, CT, RTW>, dim3((items + 3) / 4, (B + 7) & ~7), kThreads, 0, s, cre, cim,
               (const double*)g.ai, (const GemmMeta*)g.meta, X, B, F, (int)fmt);
}

void n64_fwd_launch(const DevConsts& c, const GemmTables& g, const double2* X, double* cre, double* cim, int F, Fmt fmt,
                    hipStream_t s) {
    const int B = c.bw, cols = n64_cols(F, fmt), kc = n64_fwd_kc_cols(B, F, cols);
    if (kc == 64) return (B <= 256 ? n64_fwd_kc_launch<1, 4> : n64_fwd_kc_launch<2, 4>)(c, g, X, cre, cim, F, fmt, s);
    if (kc == 32) return (B <= 256 ? n64_fwd_kc_launch<1, 2> : n64_fwd_kc_launch<2, 2>)(c, g, X, cre, cim, F, fmt, s);
    // tiles per wave: more reuse each load more, fewer give more waves and a
    // shorter stream each (us, column x degree tiles: bw=64 x8 1x1 8.8, 1x2 9.2,
    // x64 13.9, 12.6, x1024 1x2 125, 2x1 114; bw=128 x8 12.0, 14.9; bw=256 x1
    // 23.6, 19.8; bw=300 x1 35, 41; bw=32, one degree tile, x1024 1x1 29, 2x1 32).
    // Few fields at bw 192 to 256: order 0's six to eight degree tiles in pairs fit
    // one block of four waves, from nine on they need a second, nearly empty one
    // (whole calls, one field, 1x1 / 1x2: bw=192 26.4 / 23.6, bw=200 28.7 / 26.6,
    // bw=256 29.4 / 25.8, bw=257 34 / 43, bw=272 34 / 43, bw=288 41 / 46)
    if (n64_fwd_ct(g, cols) == 2) n64_fwd_direct<2, 1>(c, g, X, cre, cim, F, fmt, s);
    else if (B > 32 && (F >= 16 || (B >= 192 && B <= 256))) n64_fwd_direct<1, 2>(c, g, X, cre, cim, F, fmt, s);
    else n64_fwd_direct<1, 1>(c, g, X, cre, cim, F, fmt, s);
}

// Ring tiles per wave and ring ranges of an inverse K-chunked block: the
// fewest tile slots, then the fewest ranges (coefficients are read once per range).
static void n64_inv_split(int B, int& jt, int& nz) {
    const int RT = n64_bp(B) / 16;
    int best = 1 << 30;
    for (int z = 1; z <= RT; ++z) {
        const int j = (RT + 2 * z - 1) / (2 * z);
        if (j <= 4 && j * z < best) best = j * z, jt = j, nz = z;
    }
}

void n64_inv_launch(const DevConsts& c, const GemmTables& g, const double* cre, const double* cim, double2* X, int F,
                    Fmt fmt, hipStream_t s) {
    const int B = c.bw, cols = n64_cols(F, fmt), kc = n64_inv_kc_cols(B, F, cols);
    if (kc) {
        const int nb = (cols + kc - 1) / kc;
        int jt = 1, nz = 1;
        n64_inv_split(B, jt, nz);
        launch_lds(kc == 64 ? k_gemm_inv_kc<double, 512> : k_gemm_inv_kc<double, 256>, dim3(mix_npairs8(B) * nb * nz),
                   8 * kc, sizeof(double) * n64_inv_lds(jt, kc / 16), s, cre, cim, (const double*)g.ai,
                   (const GemmMeta*)g.meta, X, B, F, (int)fmt, nb, nz, jt);
        return;
    }
    // as in the forward (us, column x ring tiles: bw=64 x8 1x1 7.9, 1x2 8.7, x64
    // 13.7, 11.4, x1024 1x2 115, 2x2 99; bw=128 x8 13.4, 10.6; bw=256 x1 18.3, 17.1)
    if (n64_inv_ct(g, cols) == 2) n64_inv_direct<2, 2>(c, g, cre, cim, X, F, fmt, s);
    else if (B >= 192 || F * B >= 1024) n64_inv_direct<1, 2>(c, g, cre, cim, X, F, fmt, s);
    else n64_inv_direct<1, 1>(c, g, cre, cim, X, F, fmt, s);
}

}  // namespace s2
