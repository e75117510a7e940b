// fn_adjoint.hip -- adjoint (backprojection) of the plane-wave beamformer and the
// vector-Jacobian products of the differentiation form.
//
// The forward map (das_pw.m:383-467 with the time of flight of das_pw.m:336,
// 339-340, 427-428) is linear in the RF data x:
//   I(v) = s sum_n sum_a T_n(v,a) sum_k [a_nk(v) / w_n(v)] e^{j w_n tau_rx(v,k)} X_n(k,a),
//   X_n(k,a) = sum_t x[a][k][t] e^{-j 2 pi n t / N},
// with s the output scale (2 or 2/N), T_n = e^{j w_n tau_tx}, w_n(v) the
// normalising weight sum.  Its adjoint for the real inner product
// <u, y> = Re sum conj(u) y is
//   Z_n(k,a)      = s sum_v y(v) conj(T_n(v,a) a_nk(v) e^{j w_n tau_rx(v,k)}) / w_n(v)   (voxel contraction)
//   (A^H y)[a][k][t] = Re sum_n Z_n(k,a) e^{+j 2 pi n t / N}                          (band-limited inverse DFT)
//
// Voxel contraction on the matrix cores (fp16 hi + lo; the untruncated triangular window on
// v_mfma_f32_16x16x4f32 with Gauss's three multiplications): per bin, D[element][angle] += sum_v conj(B)[element][v] U[v][angle]
// with U = s y conj(T) / w.  The contraction index (voxels) is the MFMA K, so
// lane l holds the pairs (voxel 4s + l/16 of a 16-voxel group, element
// l%16 + 16 mt).  A block of 4 waves owns 4 consecutive bins (one per wave)
// and a voxel range: per 16-voxel group the block computes the phase words
// (FP64 time of flight reduced to 2^-32 revolutions) once into LDS, every wave
// contracts the group for its own bin and keeps its 16 x 128 x 16 result in
// registers across the whole range -- no atomics; one partial per (range, bin)
// is written at the end and reduced by a second kernel.  Apertures: each wave
// computes those of its bin for 64 voxels at once (one voxel per lane, from
// per-voxel FP64 terms precomputed with the phase words) every fourth group and
// keeps them in LDS for the four groups.
// Phase tiles are recomputed per bin, never stored.
//
// Vector-Jacobian products for a cotangent g (J real, dJ = sum Re(conj(g) dI)):
//   d J / d delay_k = sum_n w_n sum_a Im(conj(X_n(k,a)) Z_n(k,a))   with Z from y = g
//                   = sum_n w_n sum_a (Xr Zi - Xi Zr)
//   d J / d c_tof   = sum_v Re(conj(g(v)) dI(v)/dc)                 (dI/dc from the tangent kernel)
#include "fn_kernels.hip.h"

#include <hip/hip_runtime.h>

namespace fnk {

constexpr int ADJ_WAVES = 4;   // bins per block, one per wave (two blocks per CU)
constexpr int ADJ_ET = 8;      // element tiles of 16 (128 elements)
constexpr int ADJ_QS = 144;    // LDS words per voxel of the receive phase table ([mt][cidx] + pad: lanes
                               // 0-31 of a read meet 32 distinct banks)
constexpr int ADJ_GV = 32;     // voxels per LDS group (one barrier each): two 16-voxel contraction groups

// FULL: no per-element support test on a 128-element array (no padded
// elements).  Either the support is every element (the test reduces to the
// aperture's validity, which the voxel scale already carries), or it is the
// snapped aperture [lb, ub] of a window cut at t = 1 with pitch > width / 2: an
// element outside a valid snapped aperture then has t > 1 (with W the snapped
// half-width on its side, t - 1 >= (pitch - width/2) / (h + width/2)), so the
// window's own cut zeroes it.
template <int WCR, bool FULL>
__global__ __launch_bounds__(64 * ADJ_WAVES) __attribute__((amdgpu_waves_per_eu(2))) void adjoint_kernel(AdjArgs S)
{
    // group tables, double-buffered: the next group is loaded while this one is contracted
    __shared__ __align__(16) uint32_t q_rx[2][ADJ_GV * ADJ_QS];  // [voxel i][mt][cidx]: element cidx + 16 mt
    __shared__ uint32_t q_tx[2][ADJ_GV * 16];      // [voxel i][angle column]
    // cotangent times s / w_n(v) of each wave's bin for the group's voxels (0 outside the range)
    __shared__ float2 ys[2][ADJ_WAVES][ADJ_GV];
    // per wave, for 64 voxels: the window argument of element e on each side as e r1 / 16 + r0
    // and e l1 / 16 + l0 (r1, l1 the slopes of 16 elements; for WC_COS_RF with the window's
    // quarter-period scale and offset folded in), and the support klo | khi << 16
    __shared__ __align__(16) uint4 apx[ADJ_WAVES][64];
    __shared__ uint32_t akk[ADJ_WAVES][64];
    const BeamArgs &A = S.B;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cidx = lane & 15, q = lane >> 4;
    const long n_vox = (long)A.n_x * A.n_z;
    const int b = blockIdx.x * ADJ_WAVES + wave;
    const bool active = b < A.n_f;
    const int at = blockIdx.z;
    const long vr0 = (long)blockIdx.y * S.vox_per_range;
    const long vr1 = min(vr0 + S.vox_per_range, n_vox);
    const float c16 = (float)cidx * 0.0625f;  // element cidx in units of 16 elements
    const uint32_t n = (uint32_t)(A.n_lb + (active ? b : 0));
    double Fb = 0.0, sqf = 0.0;
    if (active) {
        Fb = A.Frx[b];
        sqf = A.sqrt_f[b];
    }

    floatx4 K1[ADJ_ET], K2[ADJ_ET], K3[ADJ_ET];
#pragma unroll
    for (int mt = 0; mt < ADJ_ET; ++mt) {
        K1[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
        K2[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
        K3[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

    const int qtx_stride = 16 * S.n_at;
    // the phase words and voxel data of the group at `base`: fetched into registers
    // at the top of the previous group's step and written to LDS buffer `buf` after
    // its contraction, so the global loads are in flight during that contraction
    static_assert(ADJ_WAVES == 4 && ADJ_GV % 16 == 0, "group loader assumes 256 threads");
    constexpr int RX4 = ADJ_GV * 32 / 256, TX1 = ADJ_GV * 16 / 256;  // uint4 / words per thread
    struct GroupRegs {
        uint4 rx[RX4];
        uint32_t tx[TX1];
        float2 ys;
    };
    static_assert(ADJ_WAVES * ADJ_GV <= 256, "one scale per thread");
    auto fetch_group = [&](long base) {
        GroupRegs r;
#pragma unroll
        for (int h = 0; h < RX4; ++h) {
            const int it = tid + 256 * h, i = it >> 5, j4 = it & 31;  // ADJ_GV voxels x 32 uint4
            const long u = base + i;
            r.rx[h] = make_uint4(0u, 0u, 0u, 0u);
            if (u < n_vox) r.rx[h] = reinterpret_cast<const uint4 *>(S.qrx + (size_t)u * 128)[j4];
        }
#pragma unroll
        for (int h = 0; h < TX1; ++h) {
            const int it = tid + 256 * h, iv = it >> 4, col = it & 15;  // ADJ_GV voxels x 16 angle columns
            const long uv = base + iv;
            r.tx[h] = uv < n_vox ? S.qtx[(size_t)uv * qtx_stride + 16 * at + col] : 0u;
        }
        r.ys = make_float2(0.f, 0.f);
        if (tid < ADJ_WAVES * ADJ_GV) {
            const int bs = blockIdx.x * ADJ_WAVES + tid / ADJ_GV;
            const long u3 = base + tid % ADJ_GV;
            if (bs < A.n_f && u3 < vr1) {
                const float sc = S.vsc[(size_t)bs * n_vox + u3];
                const float2 y = S.y[u3];
                r.ys = make_float2(sc * y.x, sc * y.y);
            }
        }
        return r;
    };
    auto store_group = [&](const GroupRegs &r, int buf) {
#pragma unroll
        for (int h = 0; h < RX4; ++h) {
            const int it = tid + 256 * h, i = it >> 5, j4 = it & 31;
            *reinterpret_cast<uint4 *>(&q_rx[buf][i * ADJ_QS + 4 * j4]) = r.rx[h];
        }
#pragma unroll
        for (int h = 0; h < TX1; ++h) q_tx[buf][tid + 256 * h] = r.tx[h];
        if (tid < ADJ_WAVES * ADJ_GV) ys[buf][tid / ADJ_GV][tid % ADJ_GV] = r.ys;
    };
    // per-voxel aperture terms of voxel `base + lane` (clamped into the grid)
    auto load_geo = [&](long base) {
        const double *g = S.vgeo + 4 * (size_t)min(base + lane, n_vox - 1);
        return make_double4(g[0], g[1], g[2], g[3]);
    };
    const bool a_ok = 16 * at + cidx < A.n_tx;
    const double x0 = -A.M * A.pitch;
    double4 geo = make_double4(0.0, 0.0, 0.0, 0.0);
    if (vr0 < vr1) {
        store_group(fetch_group(vr0), 0);
        if (active) geo = load_geo(vr0);
    }
    __syncthreads();
    int cur = 0;
    for (long gbase = vr0; gbase < vr1; gbase += ADJ_GV, cur ^= 1) {
        const bool more = gbase + ADJ_GV < vr1;
        GroupRegs next{};
        if (more) next = fetch_group(gbase + ADJ_GV);
#pragma unroll
        for (int hb = 0; hb < ADJ_GV / 16; ++hb) {
        const long base = gbase + 16 * hb;  // contraction group of 16 voxels
        const int o = 16 * hb;              // its offset in the LDS group
        const int gq = (int)((base - vr0) >> 4) & 3;           // group within the 64 voxels of apx
        if (active && base < vr1) {
            if (gq == 0) {
                // apertures of this wave's bin for voxels base .. base + 63, one per lane (forward formulas)
                double Fr = Fb;
                if (A.clamp) Fr = fmin(Fr, sqf * geo.w);  // das_pw.m:374-377
                const Aperture ap = make_aperture(geo.x, geo.y, geo.z, Fr, A, A.support_rx);
                // d = x_e - x = (x_0 - x) + e pitch; right side d / W_R, left side -d / W_L
                // (WC_COS_RF: times q_s, plus q_o)
                const double sl = WCR == WC_COS_RF ? (double)A.wrx.q_s : 1.0;
                const double qo = WCR == WC_COS_RF ? (double)A.wrx.q_o : 0.0;
                const double wr = (double)ap.inv_wr * sl, wl = (double)ap.inv_wl * sl, dx = x0 - geo.x;
                akk[wave][lane] = (uint32_t)ap.klo | ((uint32_t)ap.khi << 16);
                apx[wave][lane] = make_uint4(__float_as_uint((float)(16.0 * A.pitch * wr)),
                                             __float_as_uint((float)(-16.0 * A.pitch * wl)),
                                             __float_as_uint((float)(dx * wr + qo)), __float_as_uint((float)(qo - dx * wl)));
                if (base + 64 < vr1) geo = load_geo(base + 64);  // consumed four groups later
            }

            // element tiles [t_lo, t_hi] of 16 that meet the support of some voxel of the
            // group (wave-uniform): every other tile has zero window for all 16 voxels
            int t_lo, t_hi;
            {
                const uint32_t kk = akk[wave][16 * gq + cidx];
                const int kl = (int)(kk & 0xffffu), kh = (int)(kk >> 16);
                const int lo = row_min16(kl <= kh ? kl : 0x7fff), hi = row_max16(kl <= kh ? kh : -1);
                t_lo = __builtin_amdgcn_readfirstlane(lo) >> 4;
                t_hi = __builtin_amdgcn_readfirstlane(hi) >> 4;  // -1: no voxel of the group has elements
            }

            // Gauss: conj(B) U = (br - j bi)(ur + j ui):
            //   K1 = (br - bi) ur, K2 = br (ui - ur), K3 = bi (ur + ui); Re = K1 + K3, Im = K1 + K2
            // Per voxel step s (voxel 4 s + q of the group): U, and the window argument as
            // max(mt R1 + R0, mt L1 + L0) over the element tile mt (each side's term is the
            // larger exactly on its own side, so no per-element select)
            float Ur[4], U2[4], U3[4], R0[4], R1[4], L0[4], L1[4];
            int Klo[4], Khi[4];
            int qoff[4];
    #pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int i = 4 * s + q;  // voxel of this lane in step s
                const uint4 apv = apx[wave][16 * gq + i];  // written by this wave (LDS operations of a wave are ordered)
                if (!FULL) {
                    const uint32_t kk = akk[wave][16 * gq + i];
                    Klo[s] = (int)(kk & 0xffffu);
                    Khi[s] = (int)(kk >> 16);
                }
                R1[s] = __uint_as_float(apv.x);
                L1[s] = __uint_as_float(apv.y);
                R0[s] = fmaf(c16, R1[s], __uint_as_float(apv.z));  // element cidx of tile 0
                L0[s] = fmaf(c16, L1[s], __uint_as_float(apv.w));
                // U = s y conj(T) / w, s / w_n(v) from the per-plan table (0 outside a valid aperture)
                const float2 yv = a_ok ? ys[cur][wave][o + i] : make_float2(0.f, 0.f);
                const float rt = rev_of(n * q_tx[cur][(o + i) * 16 + cidx]);
                const float st = __builtin_amdgcn_sinf(rt), ct = __builtin_amdgcn_cosf(rt);
                const float ur = fmaf(yv.x, ct, yv.y * st);
                const float ui = fmaf(yv.y, ct, -(yv.x * st));
                Ur[s] = ur;
                U2[s] = ui - ur;
                U3[s] = ur + ui;
                qoff[s] = (o + i) * ADJ_QS + cidx;
            }
            // element tile outer, voxel step inner: four independent chains per tile
    #pragma unroll
            for (int mt = 0; mt < ADJ_ET; ++mt) {
                if (mt < t_lo || mt > t_hi) continue;
                const int e = cidx + 16 * mt;
    #pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const uint32_t Qv = q_rx[cur][qoff[s] + 16 * mt];
                    const float ta = mt == 0 ? R0[s] : fmaf((float)mt, R1[s], R0[s]);
                    const float tb = mt == 0 ? L0[s] : fmaf((float)mt, L1[s], L0[s]);
                    // max(ta, tb) as a signed-integer max of the bit patterns: fmaxf would
                    // first canonicalize both operands (two more instructions per weight),
                    // since they come from another basic block.  One of the two is >= 0 (each
                    // side's term is non-negative on its own side), and on non-negative floats
                    // the integer order is the float order, so the result is max(ta, tb)
                    const float tm = __int_as_float(max(__float_as_int(ta), __float_as_int(tb)));
                    float w;
                    if (WCR == WC_COS_RF) {
                        const float c = __builtin_amdgcn_cosf(__builtin_amdgcn_fmed3f(tm, 0.f, 0.25f));
                        w = c * c;
                    } else {
                        w = window_eval<WCR>(tm, A.wrx);
                    }
                    if (!FULL) w = (e >= Klo[s] && e <= Khi[s]) ? w : 0.f;
                    const float rv = rev_of(n * Qv);
                    const float sn = __builtin_amdgcn_sinf(rv), cs = __builtin_amdgcn_cosf(rv);
                    const float br = w * cs, bi = w * sn;
                    K1[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(br - bi, Ur[s], K1[mt], 0, 0, 0);
                    K2[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(br, U2[s], K2[mt], 0, 0, 0);
                    K3[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(bi, U3[s], K3[mt], 0, 0, 0);
                }
            }
        }  // active
        }  // hb
        // buffer cur ^ 1 was last read two groups ago (before the previous barrier)
        if (more) store_group(next, cur ^ 1);
        __syncthreads();  // group `gbase` consumed, group `gbase + ADJ_GV` stored
    }
    if (!active) return;
    // lane holds D[4q + r][cidx] = Z(element 16 mt + 4q + r, angle column cidx) of the range;
    // partial layout [range][bin][angle tile][plane][element 128][angle 16]
    const int per_bin = 2 * ADJ_ET * 256;
    float *dst = S.P + (((size_t)blockIdx.y * A.n_f + b) * S.n_at + at) * per_bin;
#pragma unroll
    for (int mt = 0; mt < ADJ_ET; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = (16 * mt + 4 * q + r) * 16 + cidx;
            dst[o] = K1[mt][r] + K3[mt][r];
            dst[ADJ_ET * 256 + o] = K1[mt][r] + K2[mt][r];
        }
}

// Units of the split contraction's cotangent operand: per bin and 64 consecutive voxels a power
// of two that brings their max |s y / w| into [2^7, 2^15), kept from one block to the next where
// it can be (each change costs the contraction 64 multiplications), or 0 where they are all
// zero; and whether any of them is far below that (UNIT_FAR) or not finite (UNIT_BAD: left out
// of the rest), which *rest then says.  A wave walks the blocks of one bin and voxel range.
// Bound by reading vsc once (4 bytes per bin and voxel).
constexpr uint32_t UNIT_FAR = 1u, UNIT_BAD = 2u;
constexpr int UNIT_DEPTH = 16;   // exponents below the unit that keep 22 bits in two fp16 halves
constexpr int UNIT_SPREAD = 64;  // the sums may be moved to a unit this far below the largest before it

// x = f 2^e, f in [0.5, 1), of the bits of x >= 0 (a subnormal's e is taken as 2^-100's: the
// factors below stay normal numbers)
__device__ __forceinline__ int exponent_of(int bits) { return max((bits >> 23) - 126, -100); }

__device__ __forceinline__ int wave_max(int v)
{
    v = row_max16(v);
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// 2^(14 - e), -100 <= e <= 128
__device__ __forceinline__ float unit_factor(int e) { return __int_as_float((127 + 14 - e) << 23); }

// a finite magnitude in its unit that keeps 22 bits there (NaN: no)
__device__ __forceinline__ bool near_unit(float m)
{
    const uint32_t least = (uint32_t)(127 + 14 - UNIT_DEPTH - 1) << 23;
    return __float_as_uint(m) - least < 0x7f800000u - least;
}

__device__ __forceinline__ bool finite2(float2 v) { return fabsf(v.x) < INFINITY && fabsf(v.y) < INFINITY; }

constexpr int UNIT_BINS = 4;  // bins a wave walks together (y read once)
__global__ __launch_bounds__(64) void adjoint_units_kernel(const float *__restrict__ vsc, const float2 *__restrict__ y,
                                                           long n_vox, int n_f, long vox_per_range, int n_blocks,
                                                           float *__restrict__ units, uint32_t *__restrict__ flags,
                                                           uint32_t *__restrict__ rest)
{
    const int lane = threadIdx.x, b0 = blockIdx.x * UNIT_BINS;
    const long v0 = (long)blockIdx.y * vox_per_range, v1 = min(v0 + vox_per_range, n_vox);
    int e_use[UNIT_BINS];
#pragma unroll
    for (int i = 0; i < UNIT_BINS; ++i) e_use[i] = -1000;
    float sc[UNIT_BINS];
    float2 q;
    auto load = [&](long base) {
        const long u = min(base + lane, n_vox - 1);
        q = y[u];
#pragma unroll
        for (int i = 0; i < UNIT_BINS; ++i) sc[i] = vsc[(size_t)min(b0 + i, n_f - 1) * n_vox + u];
    };
    load(v0);
    for (long at = v0; at < v1; at += 64) {
        float2 v[UNIT_BINS];
#pragma unroll
        for (int i = 0; i < UNIT_BINS; ++i) v[i] = at + lane < v1 ? make_float2(sc[i] * q.x, sc[i] * q.y) : make_float2(0.f, 0.f);
        load(at + 64);  // the next block, while this one is looked at
#pragma unroll
        for (int i = 0; i < UNIT_BINS; ++i) {
            const bool ok = finite2(v[i]);
            const int bits = ok ? __float_as_int(fmaxf(fabsf(v[i].x), fabsf(v[i].y))) : 0;  // (floats >= 0 in integer order)
            const int hi = wave_max(bits), lo = -wave_max(bits ? -bits : -0x7f800000);
            uint32_t w = __ballot(!ok) ? UNIT_BAD : 0u;
            float us = 0.f;
            if (hi) {
                const int e = exponent_of(hi);
                const float least = __int_as_float(lo);
                if (e > e_use[i] + 1 || e < e_use[i] - 6 ||
                    (!near_unit(least * unit_factor(e_use[i])) && near_unit(least * unit_factor(e))))
                    e_use[i] = e;
                us = unit_factor(e_use[i]);
                w |= near_unit(least * us) ? 0u : UNIT_FAR;
            }
            if (lane == 0 && b0 + i < n_f) {
                const size_t o = (size_t)(b0 + i) * n_blocks + (at >> 6);
                units[o] = us;
                flags[o] = w;
                if (w) atomicOr(rest, 1u);
            }
        }
    }
}

// The voxel contraction on v_mfma_f32_16x16x32_f16 with both operands split into fp16 high
// and low halves (as the forward kernels' fp16x3 form): Re Z = sum br ur + bi ui, Im Z =
// sum br ui - bi ur, three products each.  Same blocks, tables and double buffer as the FP32
// kernel above; a group of 32 voxels is one MFMA K, lane group q holding its voxels 4 s + q.
// Per element tile and 32 voxels: 12 matrix-core instructions of 16 cycles against 24 of 32,
// beside 8 weights a lane; bound by the vector work of the weights.
// The cotangent operand is in the unit of its 64 voxels (adjoint_units_kernel); the FP32 sums
// move to the next block's unit by 64 multiplications where it differs (neighbouring depths
// seldom need it), so elements that meet no loud voxel keep their bits.
// REST: what that leaves, added to its partials.  Voxels far below their unit, band by band in
// units of their own; blocks 2^64 below an earlier one, which the sums' exponents have no room
// for; and NaN for the elements of a voxel that is not finite.  A launch without such a
// block ends at once (*rest, which the reduction of the partials clears again).
template <int WCR, bool FULL, bool REST>
__global__ __launch_bounds__(64 * ADJ_WAVES) __attribute__((amdgpu_waves_per_eu(REST ? 1 : 2))) void
adjoint_split_kernel(AdjArgs S)
{
    static_assert(ADJ_GV == 32, "a group is one MFMA K");
    __shared__ __align__(16) uint32_t q_rx[2][ADJ_GV * ADJ_QS];  // [voxel i][mt][cidx]: element cidx + 16 mt
    __shared__ uint32_t q_tx[2][ADJ_GV * 16];                    // [voxel i][angle column]
    __shared__ float2 ys[2][ADJ_WAVES][ADJ_GV];                  // scaled cotangent times s / w_n(v) per wave's bin
    // as in the FP32 kernel: window arguments and supports of 64 voxels per wave
    __shared__ __align__(16) uint4 apx[ADJ_WAVES][64];
    __shared__ uint32_t akk[ADJ_WAVES][64];
    const BeamArgs &A = S.B;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cidx = lane & 15, q = lane >> 4;
    const long n_vox = (long)A.n_x * A.n_z;
    const int b = blockIdx.x * ADJ_WAVES + wave;
    const bool active = b < A.n_f;
    const int at = blockIdx.z;
    long vr0 = (long)blockIdx.y * S.vox_per_range;
    long vr1 = min(vr0 + S.vox_per_range, n_vox);
    const int n_blocks = (int)((n_vox + 63) >> 6);
    // (the factors' bits: biased exponents, 0 where there is none)
    const uint32_t *const units = reinterpret_cast<const uint32_t *>(S.units) + (size_t)(active ? b : 0) * n_blocks;
    const float c16 = (float)cidx * 0.0625f;  // element cidx in units of 16 elements
    const uint32_t n = (uint32_t)(A.n_lb + (active ? b : 0));
    const double Fb = active ? A.Frx[b] : 0.0, sqf = active ? A.sqrt_f[b] : 0.0;

    floatx4 ZR[ADJ_ET], ZI[ADJ_ET];
#pragma unroll
    for (int mt = 0; mt < ADJ_ET; ++mt) ZR[mt] = ZI[mt] = floatx4{0.f, 0.f, 0.f, 0.f};

    const int qtx_stride = 16 * S.n_at;
    constexpr int RX4 = ADJ_GV * 32 / 256, TX1 = ADJ_GV * 16 / 256;  // uint4 / words per thread
    struct GroupRegs {
        uint4 rx[RX4];
        uint32_t tx[TX1];
        float2 ys;
        float us;
    };
    const int bs = blockIdx.x * ADJ_WAVES + tid / ADJ_GV;  // (threads below ADJ_WAVES x ADJ_GV)
    const uint32_t us_row = (uint32_t)bs * (uint32_t)n_blocks;  // (n_f n_vox / 64 words: vsc holds n_f n_vox floats)
    auto fetch_group = [&](long base) {
        GroupRegs r;
#pragma unroll
        for (int h = 0; h < RX4; ++h) {
            const int it = tid + 256 * h, i = it >> 5, j4 = it & 31;  // ADJ_GV voxels x 32 uint4
            const long u = base + i;
            r.rx[h] = make_uint4(0u, 0u, 0u, 0u);
            if (u < n_vox) r.rx[h] = reinterpret_cast<const uint4 *>(S.qrx + (size_t)u * 128)[j4];
        }
#pragma unroll
        for (int h = 0; h < TX1; ++h) {
            const int it = tid + 256 * h, iv = it >> 4, col = it & 15;  // ADJ_GV voxels x 16 angle columns
            const long uv = base + iv;
            r.tx[h] = uv < n_vox ? S.qtx[(size_t)uv * qtx_stride + 16 * at + col] : 0u;
        }
        r.ys = make_float2(0.f, 0.f);
        r.us = 0.f;
        if (tid < ADJ_WAVES * ADJ_GV) {
            const long u3 = base + tid % ADJ_GV;
            if (bs < A.n_f && u3 < vr1) {
                const float sc = S.vsc[(size_t)bs * n_vox + u3];
                const float2 y = S.y[u3];
                r.ys = make_float2(sc * y.x, sc * y.y);
                if (!REST) r.us = S.units[us_row + (uint32_t)(base >> 6)];
            }
        }
        return r;
    };
    auto store_group = [&](const GroupRegs &r, int buf) {
#pragma unroll
        for (int h = 0; h < RX4; ++h) {
            const int it = tid + 256 * h, i = it >> 5, j4 = it & 31;
            *reinterpret_cast<uint4 *>(&q_rx[buf][i * ADJ_QS + 4 * j4]) = r.rx[h];
        }
#pragma unroll
        for (int h = 0; h < TX1; ++h) q_tx[buf][tid + 256 * h] = r.tx[h];
        if (tid < ADJ_WAVES * ADJ_GV) {
            float2 v = r.ys;
            if (!REST) {
                v = make_float2(v.x * r.us, v.y * r.us);
                if (!near_unit(fabsf(v.x) + fabsf(v.y))) v = make_float2(0.f, 0.f);  // left to REST, or zero
            }
            ys[buf][tid / ADJ_GV][tid % ADJ_GV] = v;
        }
    };
    // per-voxel aperture terms of voxel `base + lane` (clamped into the grid)
    auto load_geo = [&](long base) {
        const double *g = S.vgeo + 4 * (size_t)min(base + lane, n_vox - 1);
        return make_double4(g[0], g[1], g[2], g[3]);
    };
    const bool a_ok = 16 * at + cidx < A.n_tx;
    const double x0 = -A.M * A.pitch;
    // apertures of this wave's bin for the 64 voxels of `geo`, one per lane (forward formulas)
    auto apertures = [&](const double4 geo) __attribute__((always_inline)) {
        double Fr = Fb;
        if (A.clamp) Fr = fmin(Fr, sqf * geo.w);  // das_pw.m:374-377
        const Aperture ap = make_aperture(geo.x, geo.y, geo.z, Fr, A, A.support_rx);
        // d = x_e - x = (x_0 - x) + e pitch; right side d / W_R, left side -d / W_L, times
        // the window's argument scale, plus its offset
        const double sl = WCR == WC_COS_RF ? (double)A.wrx.q_s : WCR == WC_COS_ALL ? (double)A.wrx.s_half : 1.0;
        const double qo = WCR == WC_COS_RF ? (double)A.wrx.q_o : 0.0;
        const double wr = (double)ap.inv_wr * sl, wl = (double)ap.inv_wl * sl, dx = x0 - geo.x;
        akk[wave][lane] = (uint32_t)ap.klo | ((uint32_t)ap.khi << 16);
        apx[wave][lane] = make_uint4(__float_as_uint((float)(16.0 * A.pitch * wr)),
                                     __float_as_uint((float)(-16.0 * A.pitch * wl)),
                                     __float_as_uint((float)(dx * wr + qo)), __float_as_uint((float)(qo - dx * wl)));
    };
    // the group of 32 voxels in buffer `cur`, half gh of apx
    auto contract = [&](const int cur, const int gh) __attribute__((always_inline)) {
        // element tiles [t_lo, t_hi] of 16 that meet the support of some voxel of the
        // group (wave-uniform): every other tile has zero window for all 32 voxels
        int t_lo, t_hi;
        {
            const uint32_t kk = akk[wave][32 * gh + (lane & 31)];
            const int kl = (int)(kk & 0xffffu), kh = (int)(kk >> 16);
            const int lo = row_min16(kl <= kh ? kl : 0x7fff), hi = row_max16(kl <= kh ? kh : -1);
            t_lo = min(__builtin_amdgcn_readlane(lo, 0), __builtin_amdgcn_readlane(lo, 16)) >> 4;
            t_hi = max(__builtin_amdgcn_readlane(hi, 0), __builtin_amdgcn_readlane(hi, 16)) >> 4;  // -1: none
        }
        // per voxel step s (voxel 4 s + q): the window argument as max(mt R1 + R0, mt L1 + L0)
        // over the element tile mt, and the cotangent operand U = s y conj(T) / w
        float R0[8], R1[8], L0[8], L1[8];
        uint32_t kk[8];
        u32x4 urh, url, uih, uil;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            float ur[2], ui[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int sv = 2 * p + h, i = 4 * sv + q;
                const uint4 apv = apx[wave][32 * gh + i];  // written by this wave (LDS operations of a wave are ordered)
                if (!FULL) kk[sv] = akk[wave][32 * gh + i];
                R1[sv] = __uint_as_float(apv.x);
                L1[sv] = __uint_as_float(apv.y);
                R0[sv] = fmaf(c16, R1[sv], __uint_as_float(apv.z));  // element cidx of tile 0
                L0[sv] = fmaf(c16, L1[sv], __uint_as_float(apv.w));
                const float2 yv = a_ok ? ys[cur][wave][i] : make_float2(0.f, 0.f);
                const float rt = rev_of(n * q_tx[cur][i * 16 + cidx]);
                const float st = __builtin_amdgcn_sinf(rt), ct = __builtin_amdgcn_cosf(rt);
                ur[h] = fmaf(yv.x, ct, yv.y * st);
                ui[h] = fmaf(yv.y, ct, -(yv.x * st));
            }
            uint32_t hi, lo;
            pack2<PREC_FP16X3>(ur[0], 1.f, ur[1], 1.f, hi, lo);
            urh[p] = hi;
            url[p] = lo;
            pack2<PREC_FP16X3>(ui[0], 1.f, ui[1], 1.f, hi, lo);
            uih[p] = hi;
            uil[p] = lo;
        }
        const u32x4 nurh = neg16(urh), nurl = neg16(url);
#pragma unroll
        for (int mt = 0; mt < ADJ_ET; ++mt) {
            if (mt < t_lo || mt > t_hi) continue;
            const int e = cidx + 16 * mt;
            u32x4 brh, brl, bih, bil;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                float w[2], sn[2], cs[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int sv = 2 * p + h;
                    const uint32_t Qv = q_rx[cur][(4 * sv + q) * ADJ_QS + cidx + 16 * mt];
                    const float ta = mt == 0 ? R0[sv] : fmaf((float)mt, R1[sv], R0[sv]);
                    const float tb = mt == 0 ? L0[sv] : fmaf((float)mt, L1[sv], L0[sv]);
                    // max(ta, tb) as an integer max of the bit patterns (one of the two is >= 0,
                    // where the integer order is the float order; fmaxf would canonicalize both)
                    const float tm = __int_as_float(max(__float_as_int(ta), __float_as_int(tb)));
                    if (WCR == WC_COS_RF) {
                        const float c = __builtin_amdgcn_cosf(__builtin_amdgcn_fmed3f(tm, 0.f, 0.25f));
                        w[h] = SPLIT_PEAK * c * c;
                    } else if (WCR == WC_COS_ALL) {
                        w[h] = fmaf(A.wrx.B, __builtin_amdgcn_cosf(__builtin_amdgcn_fractf(tm)), A.wrx.A);
                    } else {
                        w[h] = window_eval<WCR>(tm, A.wrx);
                    }
                    if (!FULL) w[h] = (e >= (int)(kk[sv] & 0xffffu) && e <= (int)(kk[sv] >> 16)) ? w[h] : 0.f;
                    const float rv = rev_of(n * Qv);
                    sn[h] = __builtin_amdgcn_sinf(rv);
                    cs[h] = __builtin_amdgcn_cosf(rv);
                }
                uint32_t hi, lo;
                pack2<PREC_FP16X3>(w[0], cs[0], w[1], cs[1], hi, lo);
                brh[p] = hi;
                brl[p] = lo;
                pack2<PREC_FP16X3>(w[0], sn[0], w[1], sn[1], hi, lo);
                bih[p] = hi;
                bil[p] = lo;
            }
            ZR[mt] = mfma16<PREC_FP16X3>(brh, urh, ZR[mt]);
            ZI[mt] = mfma16<PREC_FP16X3>(brh, uih, ZI[mt]);
            ZR[mt] = mfma16<PREC_FP16X3>(bih, uih, ZR[mt]);
            ZI[mt] = mfma16<PREC_FP16X3>(bih, nurh, ZI[mt]);
            ZR[mt] = mfma16<PREC_FP16X3>(brh, url, ZR[mt]);
            ZI[mt] = mfma16<PREC_FP16X3>(brh, uil, ZI[mt]);
            ZR[mt] = mfma16<PREC_FP16X3>(bih, uil, ZR[mt]);
            ZI[mt] = mfma16<PREC_FP16X3>(bih, nurl, ZI[mt]);
            ZR[mt] = mfma16<PREC_FP16X3>(brl, urh, ZR[mt]);
            ZI[mt] = mfma16<PREC_FP16X3>(brl, uih, ZI[mt]);
            ZR[mt] = mfma16<PREC_FP16X3>(bil, uih, ZR[mt]);
            ZI[mt] = mfma16<PREC_FP16X3>(bil, nurh, ZI[mt]);
        }
    };
    const int per_bin = 2 * ADJ_ET * 256;
    // lane holds D[4q + r][cidx] = Z(element 16 mt + 4q + r, angle column cidx) of the range
    auto partial = [&](int range) { return S.P + (((size_t)range * A.n_f + b) * S.n_at + at) * per_bin; };
    if constexpr (REST) {
        if (!*S.rest) return;
        for (int range = blockIdx.y; range < S.n_vr; range += gridDim.y) {
            vr0 = (long)range * S.vox_per_range;
            vr1 = min(vr0 + S.vox_per_range, n_vox);
            const int k0 = (int)(vr0 >> 6), k1 = (int)((vr1 + 63) >> 6);
            int e_min = 0x7fff;  // as the other form walks the units
            for (int k = k0; k < k1; ++k) {
                const int eu = active ? (int)(units[k] >> 23) : 0;
                e_min = eu ? min(e_min, eu) : e_min;
                const bool skipped = eu > e_min + UNIT_SPREAD;
                const uint32_t w = active ? S.flags[(size_t)b * n_blocks + k] : 0u;
                if (!__syncthreads_or(w != 0u || skipped)) continue;
                for (int gh = 0; gh < 2; ++gh) {
                    const long base = 64L * k + 32 * gh;
                    if (base >= vr1) break;
                    __syncthreads();  // buffer 0 is free
                    store_group(fetch_group(base), 0);
                    __syncthreads();
                    if (!active) continue;
                    if (gh == 0) apertures(load_geo(base));
                    float *const dst = partial(range);
                    float2 v = make_float2(0.f, 0.f);  // what is left of voxel base + lane
                    if (lane < ADJ_GV) v = ys[0][wave][lane];
                    uint64_t nf = __ballot(!finite2(v));
                    if (!finite2(v)) v = make_float2(0.f, 0.f);
                    for (; nf; nf &= nf - 1) {
                        const uint32_t k2 = akk[wave][32 * gh + __builtin_ctzll(nf)];
                        for (int i = 0; i < 4 * ADJ_ET; ++i) {  // (the elements whose sums this lane holds)
                            const int e = 16 * (i >> 2) + 4 * q + (i & 3), o = e * 16 + cidx;
                            if (e >= (int)(k2 & 0xffffu) && e <= (int)(k2 >> 16))
                                dst[o] = dst[ADJ_ET * 256 + o] = __builtin_nanf("");
                        }
                    }
                    const float us0 = __uint_as_float((uint32_t)eu << 23);
                    if (!skipped && near_unit(fabsf(v.x * us0) + fabsf(v.y * us0))) v = make_float2(0.f, 0.f);  // the other form's
                    int bits = __float_as_int(fmaxf(fabsf(v.x), fabsf(v.y)));
                    for (;;) {
                        const int m = wave_max(bits);
                        if (m == 0) break;
                        const int e = exponent_of(m);
                        const bool in = exponent_of(bits) >= e - UNIT_DEPTH;
                        const float us = unit_factor(e);
                        if (lane < ADJ_GV) ys[0][wave][lane] = in ? make_float2(v.x * us, v.y * us) : make_float2(0.f, 0.f);
                        bits = in ? 0 : bits;
#pragma unroll
                        for (int mt = 0; mt < ADJ_ET; ++mt) ZR[mt] = ZI[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
                        contract(0, gh);
                        const float inv = ldexpf(A.wrx.inv_peak, e - 14);
#pragma unroll
                        for (int mt = 0; mt < ADJ_ET; ++mt)
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const int o = (16 * mt + 4 * q + r) * 16 + cidx;
                                dst[o] += ZR[mt][r] * inv;
                                dst[ADJ_ET * 256 + o] += ZI[mt][r] * inv;
                            }
                    }
                }
            }
        }
        return;
    }
    double4 geo = make_double4(0.0, 0.0, 0.0, 0.0);
    if (vr0 < vr1) {
        store_group(fetch_group(vr0), 0);
        if (active) geo = load_geo(vr0);
    }
    __syncthreads();
    int cur = 0;
    // biased exponents of the sums' factor and of the smallest so far (the largest unit); 0: none
    int e_acc = 0, e_min = 0x7fff;
    uint32_t w_next = vr0 < vr1 ? units[vr0 >> 6] : 0u;
    bool skip = false;
    for (long base = vr0; base < vr1; base += ADJ_GV, cur ^= 1) {
        const bool more = base + ADJ_GV < vr1;
        GroupRegs next{};
        if (more) next = fetch_group(base + ADJ_GV);
        const int gh = (int)((base - vr0) >> 5) & 1;  // half of the 64 voxels of apx
        if (gh == 0) {
            const int eu = (int)(__builtin_amdgcn_readfirstlane(w_next) >> 23);
            e_min = eu ? min(e_min, eu) : e_min;
            skip = eu == 0 || eu > e_min + UNIT_SPREAD;
            if (skip && eu && lane == 0) atomicOr(const_cast<uint32_t *>(S.rest), 1u);
            if (!skip && eu != e_acc) {
                const float f = ldexpf(1.0f, e_acc ? max(eu - e_acc, -126) : 0);
#pragma unroll
                for (int mt = 0; mt < ADJ_ET; ++mt) {
                    ZR[mt] *= f;
                    ZI[mt] *= f;
                }
                e_acc = eu;
            }
            if (base + 64 < vr1) w_next = units[(base + 64) >> 6];
        }
        if (active) {
            if (gh == 0) {
                apertures(geo);
                if (base + 64 < vr1) geo = load_geo(base + 64);  // consumed two groups later
            }
            if (!skip) contract(cur, gh);
        }  // active
        // buffer cur ^ 1 was last read two groups ago (before the previous barrier)
        if (more) store_group(next, cur ^ 1);
        __syncthreads();  // group `base` consumed, group `base + ADJ_GV` stored
    }
    if (!active) return;
    const float inv = e_acc ? ldexpf(A.wrx.inv_peak, 127 - e_acc) : 0.f;
    float *dst = partial(blockIdx.y);
#pragma unroll
    for (int mt = 0; mt < ADJ_ET; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = (16 * mt + 4 * q + r) * 16 + cidx;
            dst[o] = ZR[mt][r] * inv;
            dst[ADJ_ET * 256 + o] = ZI[mt][r] * inv;
        }
}

// Phase words of every voxel for the voxel contraction: FP64 time of flight
// (das_pw.m:336, 339-340, 427-428 with c_tof and the delay offsets) reduced to
// frac(f_s tau / N) in units of 2^-32.  qrx[v][e] holds element e (zero-padded
// to 128 elements), qtx[v][a] angle a (16 n_at columns).
__global__ __launch_bounds__(256) void adjoint_tables_kernel(BeamArgs A, uint32_t *__restrict__ qrx,
                                                             uint32_t *__restrict__ qtx, double *__restrict__ vgeo,
                                                             int n_at)
{
    const long n_vox = (long)A.n_x * A.n_z;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    const int n_cols = 128 + 16 * n_at + 1;
    if (i >= n_vox * n_cols) return;
    const long v = i / n_cols;
    const int col = (int)(i - v * n_cols);
    const int ix = (int)(v / A.n_z), iz = (int)(v - (long)ix * A.n_z);
    const double x = A.px[ix], z = A.pz[iz];
    if (col == 128 + 16 * n_at) {
        // aperture terms, the same expressions as the forward kernel's prologue
        vgeo[4 * v] = x;
        vgeo[4 * v + 1] = x / A.pitch;
        vgeo[4 * v + 2] = z / (2.0 * A.pitch);
        vgeo[4 * v + 3] = sqrt(z / (2.88 * A.c0));
    } else if (col < 128) {
        const int e = col;
        const double lat = (((double)e - A.M) * A.pitch - x) / A.ctof, zc = z / A.ctof;
        const double tau = sqrt(lat * lat + zc * zc) + (e < A.n_el ? A.delay[e] : 0.0);
        qrx[v * 128 + e] = frac32(A.f_s * tau / A.N);
    } else {
        const int a = col - 128;
        double tau = 0.0;
        if (a < A.n_tx) tau = pw_tx_time(A, a, x, z) + A.t0 / A.f_s;
        qtx[v * 16 * n_at + a] = frac32(A.f_s * tau / A.N);
    }
}

// Z[b][a][k] = sum over voxel ranges of the partials; one thread per (bin, angle
// tile, element, angle column), the column fastest so the partial reads coalesce.  delay:
// per-element delay offsets d_k that the phase words leave out, taken in here as e^{-j w_n d_k}
// (null: none), with the rounding of the spectra planes that hold them in the forward kernels
__global__ __launch_bounds__(256) void adjoint_reduce_kernel(const float *__restrict__ P, float2 *__restrict__ Z,
                                                             int n_vr, int n_f, int n_at, int n_tx, int n_el,
                                                             const double *__restrict__ delay, double fs_over_N, int n_lb,
                                                             uint32_t *__restrict__ rest)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *rest = 0u;  // for the next contraction
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    const long total = (long)n_f * n_at * 16 * ADJ_ET * 16;
    if (i >= total) return;
    const int col = (int)(i & 15), k = (int)((i >> 4) % (16 * ADJ_ET));
    const long bat = i / (16 * 16 * ADJ_ET);  // b n_at + at
    const int at = (int)(bat % n_at), b = (int)(bat / n_at);
    const int a = 16 * at + col;
    if (a >= n_tx || k >= n_el) return;
    const int per_bin = 2 * ADJ_ET * 256;
    const size_t off_re = (size_t)k * 16 + col, off_im = (size_t)ADJ_ET * 256 + off_re;
    float re = 0.f, im = 0.f;
    for (int r = 0; r < n_vr; ++r) {
        const size_t base = (((size_t)r * n_f + b) * n_at + at) * per_bin;
        re += P[base + off_re];
        im += P[base + off_im];
    }
    if (delay) {
        const uint32_t Q = (uint32_t)(n_lb + b) * frac32(fs_over_N * delay[k]);
        float sn, cs;
        sincospif((float)(int32_t)Q * (1.0f / 2147483648.0f), &sn, &cs);
        const float t = re;
        re = re * cs + im * sn;
        im = im * cs - t * sn;
    }
    // the truncated phases' mean rotation, conjugate to the forward kernels' (PHASE_BACK)
    Z[((size_t)b * n_tx + a) * n_el + k] = make_float2(fmaf(PHASE_BACK, im, re), fmaf(-PHASE_BACK, re, im));
}

// (A^H y)[ch][t] = Re sum_b Z[b][ch] e^{+j 2 pi (n_lb + b) t / N}, ch = a n_el + k, as a
// real product on the matrix cores: D[t][ch] += sum_k A[t][k] B[k][ch] over k = (bin, part),
//   A[t][(b, 0)] = Re w,  A[t][(b, 1)] = -Im w,  w = e^{+j 2 pi m / N}, m = (n_lb + b) t mod N,
//   B[(b, 0)][ch] = Re Z[b][ch],  B[(b, 1)][ch] = Im Z[b][ch].
// v_mfma_f32_16x16x4f32: lane l supplies A[t0 + l % 16][k0 + l / 16] and
// B[k0 + l / 16][c0 + l % 16], so one K step of 4 covers two bins.  A block of 4 waves
// owns 64 samples x 64 channels; a wave 16 samples (1 tile) x 64 channels (4 tiles), with
// the next step's spectra loaded while the current step's products run.
// Twiddles in LDS; each lane advances its index m by 2t mod N per step in integers.
constexpr int IDFT_WT = 1, IDFT_WC = 4;

__global__ __launch_bounds__(256) void adjoint_idft_kernel(const float2 *__restrict__ Z, const float2 *__restrict__ tw,
                                                           float *__restrict__ out, int n_t, int n_ch, int N, int n_lb,
                                                           int n_f)
{
    extern __shared__ float2 tws[];
    for (int m = threadIdx.x; m < N; m += 256) tws[m] = tw[m];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, q = lane >> 4;  // q = k within the step: bin q / 2, part q % 2
    const int part = q & 1, db = q >> 1;
    const int t0 = blockIdx.x * (64 * IDFT_WT) + wave * (16 * IDFT_WT);
    const int c0 = blockIdx.y * 64;
    int m[IDFT_WT], dm[IDFT_WT];
    bool tok[IDFT_WT];
#pragma unroll
    for (int i = 0; i < IDFT_WT; ++i) {
        const int t = t0 + 16 * i + r16;
        tok[i] = t < n_t;
        m[i] = (int)(((long)(n_lb + db) * t) % N);
        dm[i] = (int)((2L * t) % N);
    }
    int ch[IDFT_WC];
#pragma unroll
    for (int j = 0; j < IDFT_WC; ++j) ch[j] = c0 + 16 * j + r16;
    floatx4 acc[IDFT_WT][IDFT_WC];
#pragma unroll
    for (int i = 0; i < IDFT_WT; ++i)
#pragma unroll
        for (int j = 0; j < IDFT_WC; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto load_z = [&](int b, float *bv) {
#pragma unroll
        for (int j = 0; j < IDFT_WC; ++j) {
            float2 z = make_float2(0.f, 0.f);
            if (b < n_f && ch[j] < n_ch) z = Z[(size_t)b * n_ch + ch[j]];
            bv[j] = part ? z.y : z.x;
        }
    };
    float bn[IDFT_WC];
    load_z(db, bn);
    for (int b0 = 0; b0 < n_f; b0 += 2) {
        float a[IDFT_WT], bv[IDFT_WC];
#pragma unroll
        for (int j = 0; j < IDFT_WC; ++j) bv[j] = bn[j];
        load_z(b0 + 2 + db, bn);  // next step's spectra (zeros past the band)
#pragma unroll
        for (int i = 0; i < IDFT_WT; ++i) {
            const float2 w = tws[m[i]];
            a[i] = tok[i] ? (part ? -w.y : w.x) : 0.f;
            m[i] += dm[i];
            if (m[i] >= N) m[i] -= N;
        }
#pragma unroll
        for (int i = 0; i < IDFT_WT; ++i)
#pragma unroll
            for (int j = 0; j < IDFT_WC; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], bv[j], acc[i][j], 0, 0, 0);
    }
    // lane holds D[t0 + 16 i + 4 q + r][ch[j]], r = 0..3: four consecutive samples of one channel
    const bool vec = (n_t & 3) == 0;
#pragma unroll
    for (int i = 0; i < IDFT_WT; ++i)
#pragma unroll
        for (int j = 0; j < IDFT_WC; ++j) {
            const int t = t0 + 16 * i + 4 * q;
            if (ch[j] >= n_ch || t >= n_t) continue;
            float *dst = out + (size_t)ch[j] * n_t + t;
            if (vec) {  // t + 3 < n_t and 16-byte aligned
                *reinterpret_cast<float4 *>(dst) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (t + r < n_t) dst[r] = acc[i][j][r];
            }
        }
}

// d J / d delay_k = sum_b w_b sum_a (Xr Zi - Xi Zr); one block per element, FP64 sums.
// X in the operand order of the spectra: (((b MT + a/16) KI + k/4) 64 + (a & 15) + 16 (k & 3)).
__global__ __launch_bounds__(256) void vjp_delay_kernel(const float2 *__restrict__ X, const float2 *__restrict__ Z,
                                                        double *__restrict__ out, int n_f, int n_tx, int n_el, int MT,
                                                        int KI, int n_lb, double w_unit)
{
    __shared__ double red[256];
    const int k = blockIdx.x;
    double acc = 0.0;
    for (long i = threadIdx.x; i < (long)n_f * n_tx; i += 256) {
        const int b = (int)(i / n_tx), a = (int)(i - (long)b * n_tx);
        const float2 x = X[(((size_t)b * MT + (a >> 4)) * KI + (k >> 2)) * 64 + (a & 15) + 16 * (k & 3)];
        const float2 z = Z[((size_t)b * n_tx + a) * n_el + k];
        acc += w_unit * (double)(n_lb + b) * ((double)x.x * z.y - (double)x.y * z.x);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[k] = red[0];
}

// sum_v Re(conj(g) d): stage 1 per-block partials, stage 2 one block (deterministic)
__global__ __launch_bounds__(256) void dot_re_partial_kernel(const float2 *__restrict__ g, const float2 *__restrict__ d,
                                                             double *__restrict__ part, long n)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const float2 a = g[i], b = d[i];
        acc += (double)a.x * b.x + (double)a.y * b.y;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void sum_partials_kernel(const double *__restrict__ part, int n, double *__restrict__ out)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) acc += part[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// Normalization of the voxel contraction per (bin, voxel): s / w_n(v) for a valid
// receive aperture, 0 otherwise, with w_n(v) the sum of the apodization weights over
// the array (das_pw.m:400-410, normalizations.on; s alone for off).  It depends on
// the geometry, the F-numbers and the window only -- not on the time of flight --
// and is computed once per plan, with the contraction kernel's aperture and element
// arithmetic (elements cidx + 16 mt, FULL as there).
template <int WCR, bool FULL>
__global__ __launch_bounds__(256) void adjoint_scale_kernel(BeamArgs A, float *__restrict__ vsc)
{
    const long n_vox = (long)A.n_x * A.n_z;
    const long v = (long)blockIdx.x * 256 + threadIdx.x;
    const int b = blockIdx.y;
    if (v >= n_vox) return;
    const int ix = (int)(v / A.n_z), iz = (int)(v - (long)ix * A.n_z);
    const double x = A.px[ix], z = A.pz[iz];
    double Fr = A.Frx[b];
    if (A.clamp) Fr = fmin(Fr, A.sqrt_f[b] * sqrt(z / (2.88 * A.c0)));  // das_pw.m:374-377
    const Aperture ap = make_aperture(x, x / A.pitch, z / (2.0 * A.pitch), Fr, A, A.support_rx);
    float sc = 0.f;
    if (ap.klo <= ap.khi) {
        const float pf = (float)A.pitch;
        const float x0f = (float)(-A.M * A.pitch - x);
        const float sl = WCR == WC_COS_RF ? A.wrx.q_s : 1.0f;
        const float iwl = ap.inv_wl * sl, iwr = ap.inv_wr * sl;
        float asum = 0.f;
        const int e_end = FULL ? A.n_el : 16 * ADJ_ET;
        for (int e = 0; e < e_end; ++e) {
            const int cidx = e & 15, mt = e >> 4;
            const float d = fmaf((float)(16 * mt), pf, fmaf((float)cidx, pf, x0f));
            float w;
            if (WCR == WC_COS_RF) {
                w = window_rf(fabsf(d), d < 0.f ? iwl : iwr, A.wrx.q_o);
            } else if (WCR == WC_COS_ALL) {
                w = window_eval<WC_COS>(fabsf(d) * (d < 0.f ? iwl : iwr), A.wrx);
            } else {
                w = window_eval<WCR>(fabsf(d) * (d < 0.f ? iwl : iwr), A.wrx);
            }
            if (!FULL) w = (e >= ap.klo && e <= ap.khi) ? w : 0.f;
            asum += w;
        }
        sc = A.out_scale * (A.norm_rx ? 1.0f / asum : 1.0f);
    }
    vsc[(size_t)b * n_vox + v] = sc;
}

// split: the fp16 contraction, its window arguments scaled by SPLIT_PEAK (S.B) beside the
// normalization's (B, as they are)
template <int WCR, bool FULL>
static void launch_adjoint_class(bool scale, bool split, dim3 grid, hipStream_t s, const AdjArgs &S, const BeamArgs &B)
{
    const long n_vox = (long)B.n_x * B.n_z;
    if (scale) {
        hipLaunchKernelGGL((adjoint_scale_kernel<WCR, FULL>), dim3((unsigned)((n_vox + 255) / 256), (unsigned)B.n_f),
                           dim3(256), 0, s, B, const_cast<float *>(S.vsc));
    }
    if constexpr (WCR == WC_LINEAR) {
        if (!split) {
            hipLaunchKernelGGL((adjoint_kernel<WCR, FULL>), grid, dim3(64 * ADJ_WAVES), 0, s, S);
            return;
        }
    }
    const int n_blocks = (int)((n_vox + 63) / 64);
    hipLaunchKernelGGL(adjoint_units_kernel, dim3((unsigned)((B.n_f + UNIT_BINS - 1) / UNIT_BINS), grid.y), dim3(64), 0, s, S.vsc, S.y,
                       n_vox, B.n_f,
                       S.vox_per_range, n_blocks, const_cast<float *>(S.units), const_cast<uint32_t *>(S.flags),
                       const_cast<uint32_t *>(S.rest));
    hipLaunchKernelGGL((adjoint_split_kernel<WCR, FULL, false>), grid, dim3(64 * ADJ_WAVES), 0, s, S);
    hipLaunchKernelGGL((adjoint_split_kernel<WCR, FULL, true>), dim3(grid.x, std::min(grid.y, 8u), grid.z),
                       dim3(64 * ADJ_WAVES), 0, s, S);
}

// The contraction runs on the fp16 split, but for the untruncated triangular window, whose
// weights have no bound (11 angles, 384 x 384, 542 bins, whole adjoint: 6.6 ms against 9.3 in FP32; Hann 8.6 against 15.1).
hipError_t launch_adjoint(int wcr, bool tables, bool scale, dim3 grid, hipStream_t s, const AdjArgs &S0)
{
    AdjArgs S = S0;
    const long n_vox = (long)S.B.n_x * S.B.n_z;
    const long n_tab = n_vox * (128 + 16 * S.n_at + 1);
    if (tables)
        hipLaunchKernelGGL(adjoint_tables_kernel, dim3((unsigned)((n_tab + 255) / 256)), dim3(256), 0, s, S.B,
                           const_cast<uint32_t *>(S.qrx), const_cast<uint32_t *>(S.qtx), const_cast<double *>(S.vgeo),
                           S.n_at);
    // no support test: whole element tiles of 16 (tiles past the last element meet no support)
    const bool full = range_free(S.B, S.B.n_el % 16 == 0 ? S.B.n_el : 16 * ADJ_ET);
    const bool split = !(wcr == WC_LINEAR && std::isinf(S.B.wrx.t_cut));
    const BeamArgs B = S.B;
    if (split) {
        S.B.wrx.A *= SPLIT_PEAK;
        S.B.wrx.B *= SPLIT_PEAK;
        S.B.wrx.C *= SPLIT_PEAK;
        S.B.wrx.peak = SPLIT_PEAK;
        S.B.wrx.inv_peak = 1.0f / SPLIT_PEAK;
    }
    // the forward's element-loop classes hold where the support test is free here too
    if ((wcr == WC_COS_RF || wcr == WC_COS_ALL) && !full) wcr = WC_COS;
    switch (wcr) {
    case WC_COS_RF: launch_adjoint_class<WC_COS_RF, true>(scale, split, grid, s, S, B); break;
    case WC_COS_ALL: launch_adjoint_class<WC_COS_ALL, true>(scale, split, grid, s, S, B); break;
    case WC_RANGE:
        if (full) launch_adjoint_class<WC_RANGE, true>(scale, split, grid, s, S, B);
        else launch_adjoint_class<WC_RANGE, false>(scale, split, grid, s, S, B);
        break;
    case WC_LINEAR:
        if (full) launch_adjoint_class<WC_LINEAR, true>(scale, split, grid, s, S, B);
        else launch_adjoint_class<WC_LINEAR, false>(scale, split, grid, s, S, B);
        break;
    default:
        if (full) launch_adjoint_class<WC_COS, true>(scale, split, grid, s, S, B);
        else launch_adjoint_class<WC_COS, false>(scale, split, grid, s, S, B);
        break;
    }
    return hipGetLastError();
}

hipError_t launch_adjoint_reduce(const float *P, float2 *Z, int n_vr, int n_f, int n_at, int n_tx, int n_el,
                                 const double *delay, double fs_over_N, int n_lb, uint32_t *rest, hipStream_t s)
{
    const long total = (long)n_f * n_at * 16 * ADJ_ET * 16;
    hipLaunchKernelGGL(adjoint_reduce_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, P, Z, n_vr, n_f,
                       n_at, n_tx, n_el, delay, fs_over_N, n_lb, rest);
    return hipGetLastError();
}

hipError_t launch_adjoint_idft(const float2 *Z, const float2 *tw, float *out, int n_t, int n_ch, int N, int n_lb,
                               int n_f, hipStream_t s)
{
    const size_t lds = (size_t)N * sizeof(float2);
    static size_t lds_done = 0;  // raised once per process and size (graph capture issues no attribute calls)
    if (lds > 65536 && lds > lds_done) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(adjoint_idft_kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        lds_done = lds;
    }
    hipLaunchKernelGGL(adjoint_idft_kernel, dim3((unsigned)((n_t + 64 * IDFT_WT - 1) / (64 * IDFT_WT)), (unsigned)((n_ch + 63) / 64)),
                       dim3(256), lds, s, Z, tw, out, n_t, n_ch, N, n_lb, n_f);
    return hipGetLastError();
}

hipError_t launch_vjp_delay(const float2 *X, const float2 *Z, double *out, int n_f, int n_tx, int n_el, int MT, int KI,
                            int n_lb, double w_unit, hipStream_t s)
{
    hipLaunchKernelGGL(vjp_delay_kernel, dim3((unsigned)n_el), dim3(256), 0, s, X, Z, out, n_f, n_tx, n_el, MT, KI,
                       n_lb, w_unit);
    return hipGetLastError();
}

hipError_t launch_dot_re(const float2 *g, const float2 *d, long n, double *part, int n_part, double *out, hipStream_t s)
{
    hipLaunchKernelGGL(dot_re_partial_kernel, dim3((unsigned)n_part), dim3(256), 0, s, g, d, part, n);
    hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(256), 0, s, part, n_part, out);
    return hipGetLastError();
}

}  // namespace fnk
