// fn_lines.hip -- line-by-line scans: grid column i from transmit row i (a focused or plane
// wave per line), das_pw.m's receive side.
//
// Only one transmit row meets a column, so there is no matrix product: each (voxel, bin,
// element) weight is used once, and the vector work of the weight (window cosine, phase sine
// and cosine) bounds the kernel.  One depth a lane: the column, the element and the spectra
// value are the same for the whole wave, so the spectra come by scalar loads (no LDS tile), an
// element's side of the voxel is a split of the loop instead of a select, and the phase words
// of consecutive bins are an addition apart.  On lateral positions symmetric about the array,
// voxel (-x, z) sees the elements in reverse order as (x, z) sees them: a lane's weights serve
// column i and column n_x - 1 - i.  128 lines x 512 depths, 128 elements: 3.01 -> 2.04 ms a
// frame, 0.75 of it the spectra (one M-tile of 16 rows staged in LDS per bin, four lane
// groups of elements per voxel and one voxel a weight before).
#include "fn_kernels.hip.h"

#include <hip/hip_runtime.h>

namespace fnk {

constexpr int LN_BINS = 4;  // bins a wave walks together: one phase word read and one element loop for all

// The spectra [n_f][MT][KI][64] by rows, [n_f][line][element]: a wave's scalar loads then take
// four elements of a line at once (in operand order each element's 8 bytes are a cache line of
// their own: 2.76 ms a frame of 128 x 512 against 2.13).  Values that are not finite are written
// as zeros: flag [MT][n_f] says whether the 16 lines of a tile hold any at a bin, and their
// elements are then noted in bad [n_f][line][KI / 8], one bit each.
__global__ __launch_bounds__(256) void lines_spectra_kernel(const float2 *__restrict__ X, float2 *__restrict__ out, int MT,
                                                            int KI, int n_x, int n_el, uint32_t *__restrict__ flag,
                                                            uint32_t *__restrict__ bad)
{
    __shared__ float2 t[32 * 66];  // one M-tile, element steps padded apart
    __shared__ uint32_t m[16 * 4];
    const int b = blockIdx.y, mt = blockIdx.x, KW = KI / 8;
    const float2 *src = X + ((size_t)b * MT + mt) * KI * 64;
    if (threadIdx.x < 64) m[threadIdx.x] = 0u;
    bool nf = false;
    for (int e = threadIdx.x; e < KI * 64; e += 256) {
        const float2 v = src[e];
        t[(e >> 6) * 66 + (e & 63)] = v;
        nf |= !(fabsf(v.x) < INFINITY && fabsf(v.y) < INFINITY);
    }
    const bool any = __syncthreads_or(nf);
    const int rows = min(16, n_x - 16 * mt);
    if (threadIdx.x == 0) flag[(size_t)mt * gridDim.y + b] = any;
    if (any) {
        for (int e = threadIdx.x; e < KI * 64; e += 256) {
            float2 &v = t[(e >> 6) * 66 + (e & 63)];
            if (fabsf(v.x) < INFINITY && fabsf(v.y) < INFINITY) continue;
            const int k = 4 * (e >> 6) + ((e & 63) >> 4);
            atomicOr(&m[(e & 15) * KW + (k >> 5)], 1u << (k & 31));
            v = make_float2(0.f, 0.f);
        }
        __syncthreads();
        if (threadIdx.x < rows * KW) bad[((size_t)b * n_x + 16 * mt) * KW + threadIdx.x] = m[threadIdx.x];
    }
    float2 *dst = out + ((size_t)b * n_x + 16 * mt) * n_el;
    for (int e = threadIdx.x; e < rows * n_el; e += 256) {
        const int r = e / n_el, k = e - r * n_el;
        dst[e] = t[(k >> 2) * 66 + (k & 3) * 16 + r];
    }
}

hipError_t launch_lines_spectra(const float2 *X, float2 *out, int n_f, int MT, int KI, int n_x, int n_el, uint32_t *flag,
                                uint32_t *bad, hipStream_t s)
{
    hipLaunchKernelGGL(lines_spectra_kernel, dim3((unsigned)MT, (unsigned)n_f), dim3(256), 0, s, X, out, MT, KI, n_x, n_el,
                       flag, bad);
    return hipGetLastError();
}

// Workgroup (depth tile of 64, bin chunk, column or column pair); its waves take blocks of
// LN_BINS bins in turn and add up through LDS in a fixed order.
template <int WCR, bool MIR>
__global__ __launch_bounds__(256) void lines_kernel(BeamArgs A, const float2 *__restrict__ X,
                                                    const uint32_t *__restrict__ flag, const uint32_t *__restrict__ bad, int KW)
{
    extern __shared__ uint32_t qs[];  // receive phase words [n_el][64]
    __shared__ float red[4][4][64];
    constexpr bool RTEST = WCR != WC_COS_ALL && WCR != WC_COS_RF;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = blockIdx.z, col2 = A.n_x - 1 - col;
    const int iz = blockIdx.x * 64 + lane, izc = min(iz, A.n_z - 1);
    const double x = A.px[col], z = A.pz[izc];
    const double xp = x / A.pitch, zp = z / (2.0 * A.pitch);
    const double clamp_z = sqrt(z / (2.88 * A.c0));  // das_pw.m:374
    const double zc = z / A.ctof;
    for (int k = wave; k < A.n_el; k += 4) {
        const double lat = (((double)k - A.M) * A.pitch - x) / A.ctof;
        qs[k * 64 + lane] = frac32(A.f_s * (sqrt(lat * lat + zc * zc) + A.delay[k]) / A.N);
    }
    const uint32_t Q1 = frac32(A.f_s * (pw_tx_time(A, col, x, z) + A.t0 / A.f_s) / A.N);
    const uint32_t Q2 = MIR ? frac32(A.f_s * (pw_tx_time(A, col2, A.px[col2], z) + A.t0 / A.f_s) / A.N) : 0u;
    const float dx0 = (float)(-A.M * A.pitch - x), pf = (float)A.pitch;
    const int k_mid = __builtin_amdgcn_readfirstlane((int)fmin(fmax(ceil(A.M + xp), 0.0), (double)A.n_el));
    __syncthreads();

    const int b_begin = blockIdx.y * A.bin_chunk, b_end = min(b_begin + A.bin_chunk, A.n_f);
    const size_t bstride = (size_t)A.n_x * A.n_el;
    const float2 *const row1 = X + (size_t)col * A.n_el;
    const float2 *const row2 = X + (size_t)col2 * A.n_el;
    float Ir = 0.f, Ii = 0.f, Ir2 = 0.f, Ii2 = 0.f;
    for (int b0 = b_begin + LN_BINS * wave; b0 < b_end; b0 += 4 * LN_BINS) {
        float iwl[LN_BINS], iwr[LN_BINS];
        int klo[LN_BINS], khi[LN_BINS];
        bool ok[LN_BINS];
        int lo = 0x7fff, hi = -1;
#pragma unroll
        for (int i = 0; i < LN_BINS; ++i) {
            const int b = min(b0 + i, b_end - 1);
            double Fr = A.Frx[b];
            if (A.clamp) Fr = fmin(Fr, A.sqrt_f[b] * clamp_z);  // das_pw.m:374-377
            const Aperture ap = make_aperture(x, xp, zp, Fr, A, A.support_rx);
            iwl[i] = ap.inv_wl;
            iwr[i] = ap.inv_wr;
            klo[i] = ap.klo;
            khi[i] = ap.khi;
            ok[i] = ap.valid && b0 + i < b_end;
            if (WCR == WC_COS_ALL) { lo = 0; hi = A.n_el - 1; }
            else if (ap.klo <= ap.khi) { lo = min(lo, ap.klo); hi = max(hi, ap.khi); }
        }
        lo = row_min16(lo);
        hi = row_max16(hi);
        const int u_lo = min(min(__builtin_amdgcn_readlane(lo, 0), __builtin_amdgcn_readlane(lo, 16)),
                             min(__builtin_amdgcn_readlane(lo, 32), __builtin_amdgcn_readlane(lo, 48)));
        const int u_hi = max(max(__builtin_amdgcn_readlane(hi, 0), __builtin_amdgcn_readlane(hi, 16)),
                             max(__builtin_amdgcn_readlane(hi, 32), __builtin_amdgcn_readlane(hi, 48)));
        float Lr[LN_BINS], Li[LN_BINS], Mr[LN_BINS], Mi[LN_BINS], as[LN_BINS];
#pragma unroll
        for (int i = 0; i < LN_BINS; ++i) Lr[i] = Li[i] = Mr[i] = Mi[i] = as[i] = 0.f;
        const float2 *x1[LN_BINS], *x2[LN_BINS];
#pragma unroll
        for (int i = 0; i < LN_BINS; ++i) {
            const size_t ob = (size_t)min(b0 + i, b_end - 1) * bstride;
            x1[i] = row1 + ob;
            x2[i] = row2 + ob;
        }
        // K elements from k on, on the side whose reciprocal half-widths are iw
        auto elements = [&](auto kc, const int k, const float *iw) __attribute__((always_inline)) {
            constexpr int K = decltype(kc)::value;
            typedef float values __attribute__((ext_vector_type(2 * K), aligned(8)));
            uint32_t Q[K], ph[K];
            float ad[K];
#pragma unroll
            for (int e = 0; e < K; ++e) {
                Q[e] = qs[(k + e) * 64 + lane];
                ph[e] = (uint32_t)(A.n_lb + b0) * Q[e];
                ad[e] = fabsf(fmaf((float)(k + e), pf, dx0));
            }
#pragma unroll
            for (int i = 0; i < LN_BINS; ++i) {
                const values X1 = *reinterpret_cast<const values *>(x1[i] + k);
                values X2{};  // the mirrored voxel's elements, in reverse order
                if (MIR) X2 = *reinterpret_cast<const values *>(x2[i] + (A.n_el - k - K));
#pragma unroll
                for (int e = 0; e < K; ++e) {
                    const float t = ad[e] * iw[i];
                    float a;
                    if (WCR == WC_COS_ALL)
                        a = fmaf(A.wrx.B, __builtin_amdgcn_cosf(__builtin_amdgcn_fractf(t * A.wrx.s_half)), A.wrx.A);
                    else
                        a = window_eval<WCR>(t, A.wrx);
                    if (RTEST) a = (k + e >= klo[i] && k + e <= khi[i]) ? a : 0.f;
                    const float rv = rev_of(ph[e]);
                    ph[e] += Q[e];
                    const float wr = a * __builtin_amdgcn_cosf(rv), wi = a * __builtin_amdgcn_sinf(rv);
                    as[i] += a;
                    const float xr = X1[2 * e], xi = X1[2 * e + 1];
                    Lr[i] = fmaf(wr, xr, fmaf(-wi, xi, Lr[i]));
                    Li[i] = fmaf(wr, xi, fmaf(wi, xr, Li[i]));
                    if (MIR) {
                        const float yr = X2[2 * (K - 1 - e)], yi = X2[2 * (K - 1 - e) + 1];
                        Mr[i] = fmaf(wr, yr, fmaf(-wi, yi, Mr[i]));
                        Mi[i] = fmaf(wr, yi, fmaf(wi, yr, Mi[i]));
                    }
                }
            }
        };
        auto sweep = [&](int k, const int k1, const float *iw) __attribute__((always_inline)) {
            for (; k + 4 <= k1; k += 4) elements(std::integral_constant<int, 4>{}, k, iw);
            for (; k < k1; ++k) elements(std::integral_constant<int, 1>{}, k, iw);
        };
        sweep(u_lo, min(k_mid, u_hi + 1), iwl);
        sweep(max(k_mid, u_lo), u_hi + 1, iwr);
#pragma unroll
        for (int i = 0; i < LN_BINS; ++i) {
            const uint32_t n = (uint32_t)(A.n_lb + b0 + i);
            if (ok[i]) {
                const float sc = A.norm_rx ? __builtin_amdgcn_rcpf(as[i]) : 1.0f;
                const float rv = rev_of(n * Q1), sn = __builtin_amdgcn_sinf(rv), cs = __builtin_amdgcn_cosf(rv);
                const float yr = Lr[i] * sc, yi = Li[i] * sc;
                Ir += cs * yr - sn * yi;
                Ii += cs * yi + sn * yr;
                if (MIR) {
                    const float rv2 = rev_of(n * Q2), sn2 = __builtin_amdgcn_sinf(rv2), cs2 = __builtin_amdgcn_cosf(rv2);
                    const float zr = Mr[i] * sc, zi = Mi[i] * sc;
                    Ir2 += cs2 * zr - sn2 * zi;
                    Ii2 += cs2 * zi + sn2 * zr;
                }
            }
            if (b0 + i == A.n_f - 1 && A.weights && iz < A.n_z) {
                const float w = ok[i] || WCR == WC_COS_ALL ? as[i] : 0.f;
                A.weights[(long)col * A.n_z + iz] = w;
                if (MIR) A.weights[(long)col2 * A.n_z + iz] = w;
            }
        }
    }
    // depths whose aperture holds an element that is not finite at a bin of this chunk (the bins'
    // flags alone are read where every value is finite)
    bool any = false;
    for (int b = b_begin + (int)threadIdx.x; b < b_end; b += 256)
        any |= flag[(size_t)(col >> 4) * A.n_f + b] || (MIR && flag[(size_t)(col2 >> 4) * A.n_f + b]);
    if (__syncthreads_or(any)) {
        for (int b = b_begin; b < b_end; ++b) {
            const bool f1 = flag[(size_t)(col >> 4) * A.n_f + b], f2 = MIR && flag[(size_t)(col2 >> 4) * A.n_f + b];
            if (!f1 && !f2) continue;
            double Fr = A.Frx[b];
            if (A.clamp) Fr = fmin(Fr, A.sqrt_f[b] * clamp_z);
            const Aperture ap = make_aperture(x, xp, zp, Fr, A, A.support_rx);
            if (!ap.valid) continue;
            if (f1 && mask_meets(bad + ((size_t)b * A.n_x + col) * KW, KW, ap.klo, ap.khi)) Ir = Ii = __builtin_nanf("");
            if (f2 && mask_meets(bad + ((size_t)b * A.n_x + col2) * KW, KW, A.n_el - 1 - ap.khi, A.n_el - 1 - ap.klo))
                Ir2 = Ii2 = __builtin_nanf("");
        }
    }
    red[wave][0][lane] = Ir;
    red[wave][1][lane] = Ii;
    red[wave][2][lane] = Ir2;
    red[wave][3][lane] = Ii2;
    __syncthreads();
    if (wave != 0 || iz >= A.n_z) return;
    for (int w = 1; w < 4; ++w) {
        Ir += red[w][0][lane];
        Ii += red[w][1][lane];
        Ir2 += red[w][2][lane];
        Ii2 += red[w][3][lane];
    }
    float2 *const out = A.partial ? A.partial + (long)blockIdx.y * A.n_x * A.n_z : A.image;
    out[(long)col * A.n_z + iz] =
        make_float2(A.out_scale * fmaf(-PHASE_BACK, Ii, Ir), A.out_scale * fmaf(PHASE_BACK, Ir, Ii));
    if (MIR && col2 != col)
        out[(long)col2 * A.n_z + iz] =
            make_float2(A.out_scale * fmaf(-PHASE_BACK, Ii2, Ir2), A.out_scale * fmaf(PHASE_BACK, Ir2, Ii2));
}

template <bool MIR>
static void launch(int wcr, dim3 grid, const BeamArgs &A, const float2 *X, const uint32_t *flag, const uint32_t *bad, int KW,
                   hipStream_t s)
{
    const size_t lds = (size_t)A.n_el * 64 * sizeof(uint32_t);  // 32 KiB at most
    switch (wcr) {
    case WC_RANGE: hipLaunchKernelGGL((lines_kernel<WC_RANGE, MIR>), grid, dim3(256), lds, s, A, X, flag, bad, KW); break;
    case WC_LINEAR: hipLaunchKernelGGL((lines_kernel<WC_LINEAR, MIR>), grid, dim3(256), lds, s, A, X, flag, bad, KW); break;
    case WC_COS_ALL: hipLaunchKernelGGL((lines_kernel<WC_COS_ALL, MIR>), grid, dim3(256), lds, s, A, X, flag, bad, KW); break;
    case WC_COS_RF: hipLaunchKernelGGL((lines_kernel<WC_COS_RF, MIR>), grid, dim3(256), lds, s, A, X, flag, bad, KW); break;
    default: hipLaunchKernelGGL((lines_kernel<WC_COS, MIR>), grid, dim3(256), lds, s, A, X, flag, bad, KW); break;
    }
}

// grid: (depth tiles of 64, bin chunks, columns, or pairs of mirrored columns)
hipError_t launch_lines(int wcr, bool mirror, int tiles, int splits, const BeamArgs &A, const float2 *X, const uint32_t *flag,
                        const uint32_t *bad, int KW, hipStream_t s)
{
    const dim3 grid((unsigned)tiles, (unsigned)splits, (unsigned)(mirror ? (A.n_x + 1) / 2 : A.n_x));
    if (mirror) launch<true>(wcr, grid, A, X, flag, bad, KW, s);
    else launch<false>(wcr, grid, A, X, flag, bad, KW, s);
    return hipGetLastError();
}

}  // namespace fnk
