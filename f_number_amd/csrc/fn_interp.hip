// fn_interp.hip -- plane-wave images of one F-number for every bin, by interpolation.
//
// With a receive aperture that does not change over the band (f_numbers.constant, no depth
// clamp at work: das_pw.m:374-377), the weights leave the sum over the bins:
//   I(v) = s / w(v) sum_k a_k(v) sum_a x_ak(tau_a(v) + tau_k(v)),
//   x_ak(t) = sum_n X_n(k,a) e^{j w_n t}   (das_pw.m:383-384, 462-467),
// a band-limited signal per channel evaluated at one time per (voxel, element, angle) instead
// of a product over every bin.  x is sampled once per execute on M >= 2.25 n_f points of the
// DFT period, demodulated to the band's centre bin n_c, and interpolated with 8 taps of a
// Kaiser-Bessel window (beta 19.25), whose Fourier transform psi the samples are divided by
// (non-uniform FFT of type 2; Dutt and Rokhlin 1993, Jackson et al. 1991):
//   g(m) = sum_n X_n / psi_n e^{j 2 pi (n - n_c) m / M},
//   x(t) = e^{j w_c t} sum_j phi(u - m_j) g(m_j),  u = M frac(f_s t / N).
// The interpolation's own error is 3.4e-8 (RMS over the band).
#include "fn_kernels.hip.h"

#include <hip/hip_runtime.h>

namespace fnk {

constexpr int IP_TAPS = 8, IP_LEAD = 3;  // taps at m = floor(u) - 3 .. floor(u) + 4
constexpr int IP_ANGLES = 32;            // transmit rows per workgroup

// twiddles e^{j 2 pi m / M} and 1 / psi per bin; psi(s) = exp(P(s^2)), s = (n - n_c) / M, from a
// fit of the taps' own transform (1.9e-12 for |s| <= 1 / 4.5)
__global__ void interp_tables_kernel(float2 *__restrict__ tw, float *__restrict__ ipsi, int M, int n_f)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M) {
        double sn, cs;
        sincospi(2.0 * (double)i / (double)M, &sn, &cs);
        tw[i] = make_float2((float)cs, (float)sn);
    }
    if (i < n_f) {
        const double s = (double)(i - n_f / 2) / (double)M, t = s * s;
        const double p = 8.1980521630112080e-01 +
                         t * (-1.5554323030750965e+01 +
                              t * (-6.2652098207127001e+00 +
                                   t * (-5.1333350962198327e+00 +
                                        t * (-5.2975760603106297e+00 +
                                             t * (-6.0015653919472696e+00 + t * -9.5853896600960731e+00)))));
        ipsi[i] = (float)exp(-p);
    }
}

// g of every channel: a complex product on v_mfma_f32_16x16x4f32 over K = (bin, part), as the
// adjoint's inverse DFT but with both output parts.  A block of 4 waves owns 64 table points
// and one operand group of the spectra (16 rows x 4 elements), a wave 16 points; the table
// row holds M points with IP_LEAD before and IP_TAPS - 1 - IP_LEAD after them (periodic).
// Bound by the matrix cores: 8 n_f M flop per channel.
__global__ __launch_bounds__(256) void interp_samples_kernel(const float2 *__restrict__ X, const float2 *__restrict__ tw,
                                                             const float *__restrict__ ipsi, float2 *__restrict__ G,
                                                             int M, int n_f, int MT, int KI, int n_tx, int n_el)
{
    extern __shared__ float2 tws[];  // [M], then 1 / psi [n_f]
    float *ps = reinterpret_cast<float *>(tws + M);
    for (int m = threadIdx.x; m < M; m += 256) tws[m] = tw[m];
    for (int b = threadIdx.x; b < n_f; b += 256) ps[b] = ipsi[b];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, q = lane >> 4;  // q = k within the step: bin q / 2, part q % 2
    const int part = q & 1, db = q >> 1;
    const int Mp = M + IP_TAPS - 1;
    const int p0 = blockIdx.x * 64 + wave * 16;
    const int mt = blockIdx.y / KI, K4 = blockIdx.y - mt * KI;
    int pt = p0 + r16 - IP_LEAD;  // this lane's point, in [0, M)
    pt = pt < 0 ? pt + M : pt % M;
    int m = (int)(((long)(db - n_f / 2 + (long)M * ((n_f / 2 + M - 1) / M)) * pt) % M);
    const int dm = (int)((2L * pt) % M);
    floatx4 aR[4], aI[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) aR[j] = aI[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const float *src = reinterpret_cast<const float *>(X) + ((size_t)mt * KI + K4) * 128 + 2 * r16 + part;
    const size_t bstride = (size_t)MT * KI * 128;
    auto load = [&](int b, float *v) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = b < n_f ? src[(size_t)b * bstride + 32 * j] : 0.f;
    };
    float nx[4];
    load(db, nx);
    for (int b0 = 0; b0 < n_f; b0 += 2) {
        float bv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) bv[j] = nx[j];
        load(b0 + 2 + db, nx);  // next step's spectra (zeros past the band)
        const float2 t = tws[m];
        const float f = b0 + db < n_f ? ps[b0 + db] : 0.f;
        m += dm;
        if (m >= M) m -= M;
        const float wr = f * (part ? -t.y : t.x), wi = f * (part ? t.x : t.y);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            aR[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wr, bv[j], aR[j], 0, 0, 0);
            aI[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wi, bv[j], aI[j], 0, 0, 0);
        }
    }
    // lane holds D[p0 + 4 q + r][row r16, element 4 K4 + j]
    const int a = 16 * mt + r16;
    if (a >= n_tx) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int k = 4 * K4 + j;
        if (k >= n_el) continue;
        float2 *dst = G + ((size_t)k * n_tx + a) * Mp + p0 + 4 * q;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (p0 + 4 * q + r < Mp) dst[r] = make_float2(aR[j][r], aI[j][r]);
    }
}

typedef float float4a8 __attribute__((ext_vector_type(4), aligned(8)));

// value at table position i0 + 1/2 + c of the samples at `row` (bytes): taps 2 j and 2 j + 1 of
// the pair (j, 7 - j) share even and odd polynomials in c
__device__ __forceinline__ void interp8(const char *row, uint32_t i0, float c, float &gr, float &gi)
{
    const char *p = row + 8u * i0;
    const float4a8 s0 = *reinterpret_cast<const float4a8 *>(p), s1 = *reinterpret_cast<const float4a8 *>(p + 16);
    const float4a8 s2 = *reinterpret_cast<const float4a8 *>(p + 32), s3 = *reinterpret_cast<const float4a8 *>(p + 48);
    const float d = c * c;
    const float e0 = fmaf(fmaf(fmaf(1.390039810e-03f, d, 4.946005845e-03f), d, 2.041528532e-03f), d, 7.047435852e-05f);
    const float o0 = fmaf(fmaf(fmaf(-2.858200068e-05f, d, -3.704311279e-03f), d, -4.049127416e-03f), d, -5.790473733e-04f);
    const float e1 = fmaf(fmaf(fmaf(-7.295899780e-03f, d, 2.271019865e-02f), d, 9.513245759e-02f), d, 1.661914457e-02f);
    const float o1 = fmaf(fmaf(fmaf(1.351819441e-03f, d, 6.533413863e-03f), d, -7.332735053e-02f), d, -6.186627072e-02f);
    const float e2 = fmaf(fmaf(fmaf(1.332373091e-02f, d, -9.772246291e-02f), d, 2.698575628e-01f), d, 2.550378280e-01f);
    const float o2 = fmaf(fmaf(fmaf(-5.154450362e-03f, d, 1.875588265e-02f), d, 4.505671124e-02f), d, -4.823773462e-01f);
    const float e3 = fmaf(fmaf(fmaf(-7.440250683e-03f, d, 7.007437570e-02f), d, -3.670323796e-01f), d, 8.633014061e-01f);
    const float o3 = fmaf(fmaf(fmaf(9.253488059e-03f, d, -6.311852839e-02f), d, 2.598245427e-01f), d, -5.095423420e-01f);
    const float w0 = fmaf(c, o0, e0), w7 = fmaf(-c, o0, e0), w1 = fmaf(c, o1, e1), w6 = fmaf(-c, o1, e1);
    const float w2 = fmaf(c, o2, e2), w5 = fmaf(-c, o2, e2), w3 = fmaf(c, o3, e3), w4 = fmaf(-c, o3, e3);
    gr = fmaf(w7, s3.z, fmaf(w6, s3.x, fmaf(w5, s2.z, fmaf(w4, s2.x, fmaf(w3, s1.z, fmaf(w2, s1.x, fmaf(w1, s0.z, w0 * s0.x)))))));
    gi = fmaf(w7, s3.w, fmaf(w6, s3.y, fmaf(w5, s2.w, fmaf(w4, s2.y, fmaf(w3, s1.w, fmaf(w2, s1.y, fmaf(w1, s0.w, w0 * s0.y)))))));
}

// One voxel a lane, 64 voxels a workgroup; its four waves take the elements of the union
// support in turn and add up through LDS.  The transmit phases and times of the group's
// angles sit in LDS, so the loop over the angles is an addition of phase words, four 16-byte
// gathers (neighbouring depths read neighbouring samples) and about 60 FMAs: bound by those
// and the L1 rate of the gathers.  An element's angles lie together, so the loop stays within
// one or two pages.  31 angles, boxcar, 512 x 384: 0.88 ms; 75 angles, 1024 x 512: 7 ms.
template <int WCR>
__global__ __launch_bounds__(256) void interp_beamform_kernel(InterpArgs S)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const BeamArgs &A = S.B;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a0 = blockIdx.y * IP_ANGLES, na = min(IP_ANGLES, A.n_tx - a0);
    float2 *ts = reinterpret_cast<float2 *>(smem);                          // [na][64] e^{j w_c tau_a}
    uint32_t *qs = reinterpret_cast<uint32_t *>(ts + (size_t)na * 64);      // [na][64] f_s tau_a / N
    __shared__ float red[3][4][64];
    const long n_vox = (long)A.n_x * A.n_z;
    const long v = (long)blockIdx.x * 64 + lane;
    const long vv = min(v, n_vox - 1);
    const int ix = (int)(vv / A.n_z), iz = (int)(vv - (long)ix * A.n_z);
    const double x = A.px[ix], z = A.pz[iz];
    for (int a = wave; a < na; a += 4) {
        const uint32_t Q = frac32(A.f_s * (pw_tx_time(A, a0 + a, x, z) + A.t0 / A.f_s) / A.N);
        const float rv = rev_of(S.n_c * Q);
        qs[a * 64 + lane] = Q;
        ts[a * 64 + lane] = make_float2(__builtin_amdgcn_cosf(rv), __builtin_amdgcn_sinf(rv));
    }
    const Aperture ap = make_aperture(x, x / A.pitch, z / (2.0 * A.pitch), A.Frx[0], A, A.support_rx);
    const bool ne = ap.klo <= ap.khi;
    const int lo = row_min16(ne ? ap.klo : 0x7fff), hi = row_max16(ne ? ap.khi : -1);
    const int u_lo = min(min(__builtin_amdgcn_readlane(lo, 0), __builtin_amdgcn_readlane(lo, 16)),
                         min(__builtin_amdgcn_readlane(lo, 32), __builtin_amdgcn_readlane(lo, 48)));
    const int u_hi = max(max(__builtin_amdgcn_readlane(hi, 0), __builtin_amdgcn_readlane(hi, 16)),
                         max(__builtin_amdgcn_readlane(hi, 32), __builtin_amdgcn_readlane(hi, 48)));
    __syncthreads();
    const double zc = z / A.ctof;
    const int Mp = S.M + IP_TAPS - 1;
    const size_t arow = (size_t)Mp * sizeof(float2);
    float Ir = 0.f, Ii = 0.f, asum = 0.f;
    for (int k = u_lo + wave; k <= u_hi; k += 4) {
        const double dk = ((double)k - A.M) * A.pitch - x;
        const float d = (float)dk;
        float a = window_eval<WCR>(fabsf(d) * (d < 0.f ? ap.inv_wl : ap.inv_wr), A.wrx);
        const bool own = k >= ap.klo && k <= ap.khi;
        a = own ? a : 0.f;
        asum += a;
        const double lat = dk / A.ctof;
        const uint32_t Qk = frac32(A.f_s * (sqrt(lat * lat + zc * zc) + A.delay[k]) / A.N);
        const char *row = reinterpret_cast<const char *>(S.G) + ((size_t)k * A.n_tx + a0) * Mp * sizeof(float2);
        float sr = 0.f, si = 0.f;
#pragma unroll 2
        for (int i = 0; i < na; ++i, row += arow) {
            const uint32_t Q = Qk + qs[i * 64 + lane];
            const float2 t = ts[i * 64 + lane];
            // table position M Q / 2^32: its integer part, and the fraction less 1/2
            const float c = (float)(int32_t)((Q * (uint32_t)S.M) ^ 0x80000000u) * (1.0f / 4294967296.0f);
            float gr, gi;
            interp8(row, __umulhi(Q, (uint32_t)S.M), c, gr, gi);
            sr = fmaf(t.x, gr, fmaf(-t.y, gi, sr));
            si = fmaf(t.x, gi, fmaf(t.y, gr, si));
        }
        const float rv = rev_of(S.n_c * Qk);
        const float er = a * __builtin_amdgcn_cosf(rv), ei = a * __builtin_amdgcn_sinf(rv);
        // (a channel whose samples are not finite stays with the voxels that hold its element)
        Ir = own ? fmaf(er, sr, fmaf(-ei, si, Ir)) : Ir;
        Ii = own ? fmaf(er, si, fmaf(ei, sr, Ii)) : Ii;
    }
    red[0][wave][lane] = Ir;
    red[1][wave][lane] = Ii;
    red[2][wave][lane] = asum;
    __syncthreads();
    if (wave != 0 || v >= n_vox) return;
    for (int w = 1; w < 4; ++w) {
        Ir += red[0][w][lane];
        Ii += red[1][w][lane];
        asum += red[2][w][lane];
    }
    const float sc = ap.valid ? A.out_scale * (A.norm_rx ? 1.0f / asum : 1.0f) : 0.f;
    // (an empty aperture contributes nothing, also where its weights are not finite)
    const float2 val = ap.valid ? make_float2(sc * fmaf(-PHASE_BACK, Ii, Ir), sc * fmaf(PHASE_BACK, Ir, Ii))
                                : make_float2(0.f, 0.f);
    if (A.partial) A.partial[(size_t)blockIdx.y * n_vox + v] = val;
    else A.image[v] = val;
    if (blockIdx.y == 0 && A.weights) A.weights[v] = ap.valid ? asum : S.empty_weight;
}

// at plan creation: the tables, and the largest dynamic LDS a plan may ask of the samples kernel
// (once for all sizes and here, so neither a capture nor another thread's launch meets it)
hipError_t launch_interp_tables(float2 *tw, float *ipsi, int M, int n_f, hipStream_t s)
{
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(interp_samples_kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, INTERP_LDS_MAX);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(interp_tables_kernel, dim3((unsigned)((std::max(M, n_f) + 255) / 256)), dim3(256), 0, s, tw, ipsi,
                       M, n_f);
    return hipGetLastError();
}

hipError_t launch_interp_samples(const float2 *X, const float2 *tw, const float *ipsi, float2 *G, int M, int n_f, int MT,
                                 int KI, int n_tx, int n_el, hipStream_t s)
{
    const size_t lds = (size_t)M * sizeof(float2) + (size_t)n_f * sizeof(float);
    hipLaunchKernelGGL(interp_samples_kernel, dim3((unsigned)((M + IP_TAPS - 1 + 63) / 64), (unsigned)(MT * KI)), dim3(256),
                       lds, s, X, tw, ipsi, G, M, n_f, MT, KI, n_tx, n_el);
    return hipGetLastError();
}

size_t interp_table_floats2(int M, int n_tx, int n_el) { return (size_t)n_tx * n_el * (M + IP_TAPS - 1); }
int interp_groups(int n_tx) { return (n_tx + IP_ANGLES - 1) / IP_ANGLES; }

hipError_t launch_interp_beamform(int wcr, const InterpArgs &S, hipStream_t s)
{
    const long n_vox = (long)S.B.n_x * S.B.n_z;
    const size_t lds = (size_t)std::min(IP_ANGLES, S.B.n_tx) * 64 * (sizeof(float2) + sizeof(uint32_t));
    const dim3 grid((unsigned)((n_vox + 63) / 64), (unsigned)interp_groups(S.B.n_tx));
    switch (wcr) {
    case WC_RANGE: hipLaunchKernelGGL(interp_beamform_kernel<WC_RANGE>, grid, dim3(256), lds, s, S); break;
    case WC_LINEAR: hipLaunchKernelGGL(interp_beamform_kernel<WC_LINEAR>, grid, dim3(256), lds, s, S); break;
    default: hipLaunchKernelGGL(interp_beamform_kernel<WC_COS>, grid, dim3(256), lds, s, S); break;
    }
    return hipGetLastError();
}

}  // namespace fnk
