// fn_core.hip -- plans, kernel dispatch and the GPU entry points of the C ABI
// (fn_das_pw / fn_das_sa / fn_plan_*).  Replaces the orchestration of
// gpu_bf_das_pw_rf.cu:700-1122 and gpu_bf_saft_rf.cu:800-1292: device
// buffers, spectra, per-frequency beamforming and the output scale.
#include "fn_internal.h"
#include "fn_kernels.hip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cstdarg>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace fnk {
#define FN_DECL_LAUNCHERS(m, k)                                                                      \
    hipError_t launch_beamform_m##m##_k##k##_p0(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &); \
    hipError_t launch_beamform_m##m##_k##k##_p1(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &); \
    hipError_t launch_beamform_m##m##_k##k##_p2(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &); \
    hipError_t launch_beamform_m##m##_k##k##_p3(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &);
FN_DECL_LAUNCHERS(0, 8)
FN_DECL_LAUNCHERS(0, 16)
FN_DECL_LAUNCHERS(0, 32)
FN_DECL_LAUNCHERS(1, 8)
FN_DECL_LAUNCHERS(1, 16)
FN_DECL_LAUNCHERS(1, 32)
FN_DECL_LAUNCHERS(0, 48)
FN_DECL_LAUNCHERS(0, 64)
FN_DECL_LAUNCHERS(1, 48)
FN_DECL_LAUNCHERS(1, 64)
#undef FN_DECL_LAUNCHERS
#define FN_DECL_ENS(k)                                                                                  \
    hipError_t launch_beamform_ens_k##k##_p0(int, int, dim3, size_t, hipStream_t, const BeamArgs &, int); \
    hipError_t launch_beamform_ens_k##k##_p1(int, int, dim3, size_t, hipStream_t, const BeamArgs &, int); \
    hipError_t launch_beamform_ens_k##k##_p2(int, int, dim3, size_t, hipStream_t, const BeamArgs &, int); \
    hipError_t launch_beamform_ens_k##k##_p3(int, int, dim3, size_t, hipStream_t, const BeamArgs &, int);
FN_DECL_ENS(8)
FN_DECL_ENS(16)
FN_DECL_ENS(32)
#undef FN_DECL_ENS
// mirrored voxels (the fp16 split) [KI = 8 .. 48]
hipError_t launch_beamform_mir_k8(int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_mir_k16(int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_mir_k32(int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_mir_k48(int, int, dim3, size_t, hipStream_t, const BeamArgs &);
typedef hipError_t (*MirLauncher)(int, int, dim3, size_t, hipStream_t, const BeamArgs &);
static const MirLauncher kMirLaunchers[4] = {launch_beamform_mir_k8, launch_beamform_mir_k16, launch_beamform_mir_k32,
                                             launch_beamform_mir_k48};
// the last argument: 1 for a row stack (per-row transmit phases), 0 for an ensemble
typedef hipError_t (*EnsLauncher)(int, int, dim3, size_t, hipStream_t, const BeamArgs &, int);
// [KI = 8, 16, 32][form of the contraction] (FP32: the windows the fp16 split is not for)
static const EnsLauncher kEnsLaunchers[3][4] = {
    {launch_beamform_ens_k8_p0, launch_beamform_ens_k8_p1, launch_beamform_ens_k8_p2, launch_beamform_ens_k8_p3},
    {launch_beamform_ens_k16_p0, launch_beamform_ens_k16_p1, launch_beamform_ens_k16_p2, launch_beamform_ens_k16_p3},
    {launch_beamform_ens_k32_p0, launch_beamform_ens_k32_p1, launch_beamform_ens_k32_p2, launch_beamform_ens_k32_p3}};
hipError_t launch_beamform_nw_m0_k8(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_nw_m0_k16(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_nw_m0_k32(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_nw_m1_k8(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_nw_m1_k16(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_nw_m1_k32(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &);
#define FN_DECL_PERSIST(m, k)                                                                                \
    hipError_t launch_beamform_persistent_m##m##_k##k##_p0(int, int, int, int, size_t, hipStream_t,               \
                                                           const BeamArgs *, const int4 *, int, int *, int *);    \
    hipError_t launch_beamform_persistent_m##m##_k##k##_p1(int, int, int, int, size_t, hipStream_t,               \
                                                           const BeamArgs *, const int4 *, int, int *, int *);    \
    hipError_t launch_beamform_persistent_m##m##_k##k##_p2(int, int, int, int, size_t, hipStream_t,               \
                                                           const BeamArgs *, const int4 *, int, int *, int *);    \
    hipError_t launch_beamform_persistent_m##m##_k##k##_p3(int, int, int, int, size_t, hipStream_t,               \
                                                           const BeamArgs *, const int4 *, int, int *, int *);
FN_DECL_PERSIST(0, 8) FN_DECL_PERSIST(0, 16) FN_DECL_PERSIST(0, 32)
FN_DECL_PERSIST(1, 8) FN_DECL_PERSIST(1, 16) FN_DECL_PERSIST(1, 32)
typedef hipError_t (*PersistLauncher)(int, int, int, int, size_t, hipStream_t, const BeamArgs *, const int4 *, int,
                                      int *, int *);
#define FN_PERSIST_ROW(m, k)                                                                                 \
    {launch_beamform_persistent_m##m##_k##k##_p0, launch_beamform_persistent_m##m##_k##k##_p1,                 \
     launch_beamform_persistent_m##m##_k##k##_p2, launch_beamform_persistent_m##m##_k##k##_p3}
static const PersistLauncher kPersistLaunchers[2][3][4] = {
    {FN_PERSIST_ROW(0, 8), FN_PERSIST_ROW(0, 16), FN_PERSIST_ROW(0, 32)},
    {FN_PERSIST_ROW(1, 8), FN_PERSIST_ROW(1, 16), FN_PERSIST_ROW(1, 32)}};
hipError_t launch_windowed_rows(const BeamArgs &A, int mode, int win_rx, double par_rx, float *h_rx, int win_tx,
                                double par_tx, float *h_tx, hipStream_t s);
hipError_t launch_focused_signal(const BeamArgs &A, int mode, int wcr, int wct, int MT_all, int KI, int nw, int ix,
                                 int iz, float2 *F, const float2 *tw, float2 *out, hipStream_t s);
hipError_t launch_beamform_tan_k8(int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_tan_k16(int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_tan_k32(int, int, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_tan_k8_p2(int, int, bool, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_tan_k16_p2(int, int, bool, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_beamform_tan_k32_p2(int, int, bool, dim3, size_t, hipStream_t, const BeamArgs &);
hipError_t launch_adjoint(int wcr, bool tables, bool scale, dim3 grid, hipStream_t s, const AdjArgs &S);
hipError_t launch_adjoint_reduce(const float *P, float2 *Z, int n_vr, int n_f, int n_at, int n_tx, int n_el,
                                 const double *delay, double fs_over_N, int n_lb, uint32_t *rest, hipStream_t s);
hipError_t launch_adjoint_idft(const float2 *Z, const float2 *tw, float *out, int n_t, int n_ch, int N, int n_lb,
                               int n_f, hipStream_t s);
hipError_t launch_lines(int wcr, bool mirror, int tiles, int splits, const BeamArgs &A, const float2 *X, const uint32_t *flag,
                        const uint32_t *bad, int KW, hipStream_t s);
hipError_t launch_lines_spectra(const float2 *X, float2 *out, int n_f, int MT, int KI, int n_x, int n_el, uint32_t *flag,
                                uint32_t *bad, hipStream_t s);
hipError_t launch_interp_tables(float2 *tw, float *ipsi, int M, int n_f, hipStream_t s);
hipError_t launch_interp_samples(const float2 *X, const float2 *tw, const float *ipsi, float2 *G, int M, int n_f, int MT,
                                 int KI, int n_tx, int n_el, hipStream_t s);
hipError_t launch_interp_beamform(int wcr, const InterpArgs &S, hipStream_t s);
size_t interp_table_floats2(int M, int n_tx, int n_el);
int interp_groups(int n_tx);
hipError_t launch_vjp_delay(const float2 *X, const float2 *Z, double *out, int n_f, int n_tx, int n_el, int MT, int KI,
                            int n_lb, double w_unit, hipStream_t s);
hipError_t launch_dot_re(const float2 *g, const float2 *d, long n, double *part, int n_part, double *out, hipStream_t s);
typedef hipError_t (*BeamLauncher)(int, int, int, dim3, size_t, hipStream_t, const BeamArgs &);
// [mode][KI = 8, 16, 32] (windowed normalization; [mode][KI = 8 .. 64][precision] below)
static const BeamLauncher kNwLaunchers[2][3] = {
    {launch_beamform_nw_m0_k8, launch_beamform_nw_m0_k16, launch_beamform_nw_m0_k32},
    {launch_beamform_nw_m1_k8, launch_beamform_nw_m1_k16, launch_beamform_nw_m1_k32}};
#define FN_BEAM_ROW(m, k) \
    {launch_beamform_m##m##_k##k##_p0, launch_beamform_m##m##_k##k##_p1, launch_beamform_m##m##_k##k##_p2, \
     launch_beamform_m##m##_k##k##_p3}
static const BeamLauncher kBeamLaunchers[2][5][4] = {
    {FN_BEAM_ROW(0, 8), FN_BEAM_ROW(0, 16), FN_BEAM_ROW(0, 32), FN_BEAM_ROW(0, 48), FN_BEAM_ROW(0, 64)},
    {FN_BEAM_ROW(1, 8), FN_BEAM_ROW(1, 16), FN_BEAM_ROW(1, 32), FN_BEAM_ROW(1, 48), FN_BEAM_ROW(1, 64)}};
#undef FN_BEAM_ROW
// One thread per voxel of the left half and chunk of bins; bound by a division and eight roundings
// in FP64 per voxel and bin (128 x 96, 240 bins: 7 us).
constexpr int MIRROR_BINS = 8;
__global__ __launch_bounds__(256) void mirror_check_kernel(MirrorArgs m)
{
    const long v = (long)blockIdx.x * 256 + threadIdx.x;
    if (v >= (long)(m.n_x / 2) * m.n_z) return;
    const int b0 = blockIdx.y * MIRROR_BINS, b1 = min(b0 + MIRROR_BINS, m.n_f);
    bool off = false;
    for (int b = b0; b < b1; ++b) off |= mirror_off(m, v, b);
    if (off) *m.tie = 1u;
}

// image (and weights, where given) of n_z depths per column into the first depths of columns of NZ
__global__ void paste_depths_kernel(const float2 *img, const float *w, long n, int n_z, int NZ, float2 *out, float *w_out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long o = i / n_z * NZ + i % n_z;
    out[o] = img[i];
    if (w) w_out[o] = w[i];
}

// zero fill used instead of hipMemsetAsync so the launch sequence stays
// capturable into a graph
__global__ void fill_zero_kernel(float *p, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}
}  // namespace fnk

using fnh::fail;

namespace {

constexpr size_t kMaxLds = 160 * 1024;  // gfx950 LDS per workgroup

struct Run {
    hipEvent_t e0, e1, e2;
};

}  // namespace

// room for 16-bit planes: of a plan's own tiling and the tangent's (others: ensure_planes), of its
// own, of its own without the zero tiles of a last group, or none (an FP32 call then runs the
// FP32 kernels)
enum class Planes { plan, own, bare, none };

struct fn_plan {
    int mode = 0;  // 0: plane waves, 1: synthetic aperture
    int device = 0;
    fnh::Grid g;
    int n_x = 0, n_z = 0, n_t = 0, n_el = 0, n_tx = 0;
    long n_vox = 0;
    int KI = 0, MT_all = 0, MT_tmpl = 0, n_groups = 1, bin_split = 1;
    int n_frames = 1;  // ensemble frames (transmit rows = frames x angles)
    int ens_angles = 0;  // ensemble: angles per frame
    int wcr = 0, wct = 0;
    int nw = 0;                 // windowed normalization (CPU semantics): taper kernels, one bin chunk
    int lbl = 0;                // line scan: grid column i from transmit row i (groups = columns)
    float *d_nw = nullptr;      // L / 2 per (voxel, element): receive, then (SA) transmit
    int executed = 0;           // spectra of an execute are in d_X (focused signal)
    float2 *d_sigF = nullptr;   // focused spectrum of the signal voxel [n_f]
    std::vector<double> h_px, h_pz, h_Frx, h_Ftx, h_sqf;  // host copies (signal voxel search)
    std::vector<double> h_delay;                          // delay offsets of the last set_tof (empty: zeros)
    int precision = FN_PRECISION_FP32;  // as asked for
    int kprec = FN_PRECISION_FP32;      // form of the forward contraction (kernel_precision)
    Planes planes = Planes::plan;
    int mirror = 0;         // lateral positions symmetric: planes hold the reversed elements too
    int line_mirror = 0;    // line scan on symmetric lateral positions: two columns share their weights
    uint32_t *d_tie = nullptr;  // plans that may mirror: the check's answer (mirror_off)
    int tie_later = 0;          // a one-shot call's plan: its own kernels look (Mirror::later)
    int delays_even = 1;    // delay offsets symmetric about the array's centre
    int interp_M = 0;       // > 0: the forward image by interpolation of M samples per channel
    float2 *d_Xrow = nullptr;  // line scan: the spectra by rows [n_f][line][element]
    uint32_t *d_lflag = nullptr;  // its tiles' flags and masks of elements that are not finite (fn_lines.hip)
    float2 *d_ip = nullptr; // its channel samples, twiddles [M] and 1 / psi [n_f]
    // interpolated plans with depths where the F-number clamp is at work: a plan of those
    // leading depths (on this plan's spectra), its image and weights, pasted over the first rows
    fn_plan *shallow = nullptr;
    float2 *d_simg = nullptr;
    float *d_sw = nullptr;
    int verbosity = 0;
    fnk::BeamArgs args{};
    fnk::SpecArgs sargs{};
    size_t lds_beam = 0, lds_spec = 0;
    unsigned char *d_block = nullptr;  // one allocation: the tables, the delay offsets, spectra, planes and scales
    double *d_px = nullptr, *d_pz = nullptr, *d_Frx = nullptr, *d_Ftx = nullptr, *d_txp = nullptr, *d_sqf = nullptr;
    float2 *d_tw = nullptr, *d_X = nullptr;
    void *d_Xlp = nullptr;    // 16-bit spectra planes (mixed precision)
    float *d_xscale = nullptr;
    uint32_t *d_bad = nullptr;    // elements that are not finite, beside the planes
    float *d_rowscale = nullptr;  // ensembles: scales of the rows and the peaks behind them (row_scales)
    double *d_delay = nullptr;  // per-element delay offsets (zeros unless set)
    double *d_zeros = nullptr;  // zeros in their place
    // adjoint / vector-Jacobian workspace (allocated on first use)
    float *d_P = nullptr;       // voxel-range partials of the voxel contraction
    float2 *d_Z = nullptr;      // reduced contraction [n_f][n_tx][n_el]
    uint32_t *d_qtab = nullptr; // per-voxel phase words of the contraction
    double *d_part = nullptr;   // reduction partials
    int adj_vr = 0, adj_at = 0;
    long tof_serial = 1;                // bumped by every set_tof
    long tiling_serial = 1;             // bumped by every set_tiling (whose buffers may be others)
    long adj_tab_serial = 0;            // tof_serial the phase tables were built for
    hipStream_t adj_tab_stream = nullptr;  // stream that built them (reuse is ordered only there)
    float *d_vsc = nullptr;                // adjoint normalization s / w_n(v) [n_f][n_vox]
    bool adj_sc_built = false;
    hipStream_t adj_sc_stream = nullptr;
    long adj_vpr = 0;
    size_t x_bytes = 0, xlp_bytes = 0;
    int xlp_tiles = 0;          // tiles that d_Xlp has room for
    void *d_xlp_own = nullptr;  // planes beyond those of the block (ensure_planes)
    float2 *d_pimg = nullptr;   // partial images [slot][n_vox] (several workgroups per voxel)
    size_t pimg_cap = 0;        // float2 capacity of d_pimg
    float2 *d_ptan = nullptr;   // tangent partials: image slots, then dI/dc slots
    size_t ptan_cap = 0;
    hipStream_t stream = nullptr;
    int profiling = 0;
    std::vector<Run> pending, spare;
    double spec_ms = 0.0, beam_ms = 0.0;
    int runs = 0;
    double flops = 0.0;
    // useful_flops: counted on the first fn_plan_info_get (n_f x up to 64 x 64 apertures, 15 ms
    // at 250 bins), which executing a plan does not need
    mutable std::once_flag useful_once;
    mutable double useful_flops = 0.0;
};

namespace {

// the forward kernel whose lanes stand for a voxel and its mirror image (beamform_tile, MIR)
bool use_mirror(const fn_plan *P) { return P->mirror && P->n_groups == 1 && !P->interp_M; }

// M-tiles of the 16-bit planes: the transmit tiles and their mirrored ones, or whole groups, which
// the kernels at 65-128 elements copy ahead of their products (the others fill in a last group's
// zero tiles themselves: synthetic aperture of 224 elements, bf16x3, 14 tiles in groups of 4: 83.1
// ms with zero tiles to read, 77.3 without); a no-allocation call short of room leaves them out too
int plane_tiles(const fn_plan *P)
{
    if (use_mirror(P)) return 2 * P->MT_all;
    return P->KI != 32 || P->planes == Planes::bare ? P->MT_all : P->n_groups * P->MT_tmpl;
}

// the tangent with mirrored voxels (mirrored plans run the fp16 split): one tile of rows
bool tangent_mirror(const fn_plan *P) { return P->mirror && P->MT_all == 1; }

// delay offsets of mirrored plans: taken into the planes unless they are symmetric
const double *plane_delay(const fn_plan *P, bool mirror) { return mirror && !P->delays_even ? P->d_delay : nullptr; }

// voxel tiles of 64 per beamforming group: the whole grid, half its columns (mirrored
// voxels), or (line scan) one column
long beam_tiles(const fn_plan *P)
{
    if (P->lbl) return (P->n_z + 63) / 64;
    return ((use_mirror(P) ? (long)((P->n_x + 1) / 2) * P->n_z : P->n_vox) + 63) / 64;
}

// workgroups that share a voxel: bin chunks times transmit groups (a line scan's
// groups are its columns, one per voxel); ensembles add their frames' rows atomically
int beam_slots(const fn_plan *P)
{
    if (P->interp_M) return fnk::interp_groups(P->n_tx);
    return P->n_frames > 1 ? 1 : P->bin_split * (P->lbl ? 1 : P->n_groups);
}

int hip_fail(hipError_t e, const char *what)
{
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();  // reported here, not by the next launch
        return fail(FN_ERR_OUT_OF_MEMORY, "%s: out of device memory", what);
    }
    return fail(FN_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

#define HIP_CHECK(call, what)                          \
    do {                                               \
        hipError_t e_ = (call);                        \
        if (e_ != hipSuccess) return hip_fail(e_, what); \
    } while (0)

// partial-image buffer of the plan's tiling (grown, never shrunk; freed with the plan); where
// there is no memory for a larger one the old one stays
int ensure_partials(fn_plan *P)
{
    const int slots = beam_slots(P);
    const size_t need = slots > 1 ? (size_t)slots * P->n_vox : 0;
    if (need <= P->pimg_cap) return FN_OK;
    HIP_CHECK(hipSetDevice(P->device), "hipSetDevice");
    float2 *grown = nullptr;
    HIP_CHECK(hipMalloc(&grown, need * sizeof(float2)), "partial images");
    hipFree(P->d_pimg);  // synchronizes: no launch still reads it
    P->d_pimg = grown;
    P->pimg_cap = need;
    return FN_OK;
}

int select_device(int index)
{
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count < 1) return fail(FN_ERR_NO_DEVICES, "Could not find any HIP devices!");
    // gpu_bf_das_pw_rf.cu:460 tests (index >= 0 || index < count), which always
    // passes; the intended check is applied here.
    if (index < 0 || index >= count) return fail(FN_ERR_DEVICE, "Selected device does not exist!");
    HIP_CHECK(hipSetDevice(index), "hipSetDevice");
    return FN_OK;
}

// window -> (class, coefficients, support); see fn_kernels.hip.h for the forms
int setup_window(const fn_window &w, int semantics, fnk::WinCoef *c, int *wc, int *support)
{
    const bool cpu = semantics == FN_SEMANTICS_CPU;
    *c = fnk::WinCoef{-1.f, INFINITY, 0.f, 1.f, 0.f, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f};
    switch (w.id) {
    case FN_WINDOW_BOXCAR:
        *wc = fnk::WC_RANGE;
        *support = cpu ? fnk::SUPPORT_OPEN_H : fnk::SUPPORT_SNAPPED;
        return FN_OK;
    case FN_WINDOW_TUKEY:
        *wc = fnk::WC_COS;
        c->t_flat = c->t_off = (float)(1.0 - w.parameter);
        c->t_cut = 1.f;
        c->A = c->B = 0.5f;
        c->s_half = (float)(0.5 / w.parameter);
        c->q_s = (float)(0.25 / w.parameter);
        c->q_o = (float)(-(1.0 - w.parameter) * 0.25 / w.parameter);
        *support = fnk::SUPPORT_SNAPPED;  // the window is zero beyond the snapped aperture
        return FN_OK;
    case FN_WINDOW_HANN:
        *wc = fnk::WC_COS;
        c->t_cut = cpu ? INFINITY : 1.f;
        c->A = c->B = 0.5f;
        c->s_half = 0.5f;
        c->q_s = 0.25f;
        *support = cpu ? fnk::SUPPORT_ALL : fnk::SUPPORT_SNAPPED;
        return FN_OK;
    case FN_WINDOW_TRIANGULAR:
        *wc = fnk::WC_LINEAR;
        c->t_cut = cpu ? INFINITY : 1.f;
        c->A = 1.f;
        c->C = -1.f;
        *support = cpu ? fnk::SUPPORT_ALL : fnk::SUPPORT_SNAPPED;
        return FN_OK;
    default:
        // id 3 (cosine) has no windows.* class (gpu_bf_helper_functions.cu:56-97 never yields it)
        return fail(FN_ERR_WINDOW, "window id %d is not reachable from any windows.* class", (int)w.id);
    }
}

// taper of the windowed normalization in CPU semantics as window_any()
// coefficients (|t|: flat part, A + C t + B cos(2 pi (t - t_off) s_half), cut)
int taper_coef(const fn_window &w, fnk::WinCoef *c)
{
    *c = fnk::WinCoef{-1.f, INFINITY, 0.f, 1.f, 0.f, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f};
    switch (w.id) {
    case FN_WINDOW_BOXCAR: c->t_cut = 1.f; return FN_OK;                       // |t| < 1
    case FN_WINDOW_HANN: c->A = c->B = 0.5f; c->s_half = 0.5f; return FN_OK;   // untruncated
    case FN_WINDOW_TUKEY:
        c->t_flat = c->t_off = (float)(1.0 - w.parameter);
        c->t_cut = 1.f;
        c->A = c->B = 0.5f;
        c->s_half = (float)(0.5 / w.parameter);
        return FN_OK;
    case FN_WINDOW_TRIANGULAR: c->A = 1.f; c->C = -1.f; return FN_OK;          // 1 - |t|, untruncated
    default: return fail(FN_ERR_WINDOW, "window id %d is not reachable from any windows.* class", (int)w.id);
    }
}

// windowed normalization: L / 2 per (voxel, element) from the FP64 row pass,
// once per plan (geometry and F-number tables only)
int setup_windowed(fn_plan *P, bool rx, const fn_window &wrx, const fn_window &nwin_rx, bool tx, const fn_window &wtx,
                   const fn_window &nwin_tx)
{
    if (P->precision != FN_PRECISION_FP32)
        return fail(FN_ERR_UNSUPPORTED, "normalizations.windowed runs in FP32 only");
    if (P->n_frames > 1) return fail(FN_ERR_UNSUPPORTED, "normalizations.windowed: single-frame plans only");
    const size_t n = (size_t)P->n_vox * P->n_el;
    HIP_CHECK(hipMalloc(&P->d_nw, n * (rx + tx) * sizeof(float)), "windowed normalization rows");
    float *h_rx = rx ? P->d_nw : nullptr, *h_tx = tx ? P->d_nw + (rx ? n : 0) : nullptr;
    int s;
    if (rx && (s = taper_coef(nwin_rx, &P->args.wn_rx))) return s;
    if (tx && (s = taper_coef(nwin_tx, &P->args.wn_tx))) return s;
    hipError_t e = fnk::launch_windowed_rows(P->args, P->mode, wrx.id, wrx.parameter, h_rx, wtx.id, wtx.parameter, h_tx,
                                             P->stream);
    if (e != hipSuccess) return hip_fail(e, "windowed_rows_kernel");
    HIP_CHECK(hipStreamSynchronize(P->stream), "windowed_rows_kernel");
    P->args.nw_rx = h_rx;
    P->args.nw_tx = h_tx;
    return FN_OK;
}

// forward element loops without per-element support tests: the raised cosine
// over every element of a full array (CPU Hann) takes WC_COS_ALL, a cosine
// window whose cut implies the support takes WC_COS_RF.  The tangent and the adjoint have
// instances of both on the fp16 split; a tangent on FP32 instructions runs the general class
void use_cos_all(fn_plan *P)
{
    if (P->nw) return;
    const fnk::WinCoef &w = P->args.wrx;
    // elements the kernel's loop runs over: the 16-bit forms run whole chunks of 32 elements
    // that meet a support (some kernels of a plan skip finer steps), so 96 or 160 elements
    // need no support test either, while their padding would be a part of a chunk otherwise
    const bool lp = P->kprec != FN_PRECISION_FP32;
    const int n_run = lp && P->n_el % 32 == 0 ? P->n_el : 4 * P->KI;
    if (P->wcr == fnk::WC_COS) {
        if (P->args.support_rx == fnk::SUPPORT_ALL && P->n_el == n_run &&
            w.t_off == 0.f && w.t_flat < 0.f && std::isinf(w.t_cut))
            P->wcr = fnk::WC_COS_ALL;
        else if (fnk::cos_rf_window(P->args, P->args.support_rx, w, n_run))
            P->wcr = fnk::WC_COS_RF;
    }
    // the synthetic aperture's transmit side: the same cut-window class for its
    // transmitters (the SA kernels launch it; every other SA path evaluates the window
    // with its support test, which WC_COS_RF maps to)
    // whole tiles of 16 transmitters: the padding tiles get no weight
    const fnk::WinCoef &t = P->args.wtx;
    const int n_tx = P->n_el % 16 == 0 ? P->n_el : 4 * P->KI;
    if (P->mode == 1 && P->wct == fnk::WC_COS) {
        if (P->args.support_tx == fnk::SUPPORT_ALL && P->n_el == n_tx && t.t_off == 0.f && t.t_flat < 0.f &&
            std::isinf(t.t_cut))
            P->wct = fnk::WC_COS_ALL;
        else if (fnk::cos_rf_window(P->args, P->args.support_tx, t, n_tx))
            P->wct = fnk::WC_COS_RF;
    }
}

int wcr_general(int wcr) { return (wcr == fnk::WC_COS_ALL || wcr == fnk::WC_COS_RF) ? fnk::WC_COS : wcr; }

// default transmit tiles per plane-wave workgroup that fit the register file:
// ensembles hold per-row image accumulators, so 4; FP32 and fp16 at 128 elements 5
int tile_cap(int n_frames, int precision, int KI)
{
    if (n_frames <= 1) return 5;
    if ((precision == FN_PRECISION_FP16 || precision == FN_PRECISION_FP32) && KI == 32) return 5;
    return 4;
}

// transmit tiles per group of a row stack (its own kernel instances, per-row phases)
int stack_tile_cap(int precision, int KI) { return (precision == FN_PRECISION_FP16 && KI == 32) ? 5 : 4; }

// a receive window without a cut and not a cosine: its weights grow with the element distance
bool unbounded_window(int wcr, const fnk::WinCoef &w) { return wcr == fnk::WC_LINEAR && std::isinf(w.t_cut); }

// Form of the forward contraction.  FP32 plans run the fp16 hi + lo split: its operands
// carry 22-23 bits and its products accumulate in FP32, so its error against 64 bits is that
// of the FP32 products (11 angles, Tukey: 4.9e-7 both; 75 angles, Hann: 2.3e-7 and 2.2e-7;
// synthetic aperture: 5.7e-7 and 5.6e-7), and it takes 12 matrix-core instructions of 16
// cycles per 32 elements and tile against 24 of 32 (75 angles at 1024 x 512: 174.6 ms
// against 422.5; 11 angles at 256 x 256: 3.1 against 4.5; synthetic aperture at 512 x 512:
// 94 against 168).  The synthetic aperture beyond 128 elements keeps the FP32 kernel, which
// is the faster there (192 elements, 128 x 256: 54 ms against 65); the windowed
// normalization and line scans (no matrix product) have FP32 kernels only.
int kernel_precision(const fn_plan *P, int precision)
{
    if (precision == FN_PRECISION_FP32 && !P->nw && !P->lbl && (P->KI <= 32 || P->mode == 0) &&
        !unbounded_window(P->wcr, P->args.wrx))
        return FN_PRECISION_FP16X3;
    return precision;
}

int form_planes(int kprec) { return kprec == FN_PRECISION_FP16 ? 2 : 4; }

// staged spectra bytes per M-tile and element step: FP32 interleaved complex, or 16-bit
// planes (Xr, Xi and, for the split forms, their residuals)
size_t form_step_bytes(int kprec) { return kprec == FN_PRECISION_FP32 ? 64 * sizeof(float2) : (size_t)form_planes(kprec) * 64 * 2; }

// scales of MT tiles of transmit rows: [2][16 MT], and room for their peaks per chunk of bins
constexpr int ROW_PEAK_CHUNKS = 64;
size_t row_scale_bytes(int MT) { return (size_t)(2 + ROW_PEAK_CHUNKS) * 16 * MT * sizeof(float); }
// (bf16 has the exponents of FP32; one-pass fp16, which is asked for, shares its bins' scale among
// the rows of a launch: 100 frames and 10 jobs 49.9 ms with rows' own scales, 49.5 without)
bool has_row_scales(int kprec) { return kprec == FN_PRECISION_FP16X3; }

size_t plane_bytes(const fn_plan *P, int tiles) { return (size_t)P->g.n_f * form_planes(P->kprec) * tiles * P->KI * 64 * 2; }

// words of a mask of 4 KI elements, and bytes of the masks beside n_f bins of planes (each of
// `rows` operand rows has its own where they are other frames or jobs)
int bad_words(int KI) { return KI / 8; }
size_t bad_bytes(int n_f, int rows, int KI) { return (size_t)n_f * rows * bad_words(KI) * sizeof(uint32_t); }

// words of a line scan's flags, before its masks
size_t lines_flags(const fn_plan *P) { return (size_t)P->MT_all * P->g.n_f; }

// element steps per lane: 4 KI >= n_el elements in four lane groups
int ki_of(int n_el)
{
    if (n_el <= 32) return 8;
    if (n_el <= 64) return 16;
    if (n_el <= 128) return 32;
    if (n_el <= 192) return 48;
    if (n_el <= 256) return 64;
    return 0;
}

// index of a KI in the launcher tables
int ki_index(int KI) { return KI == 8 ? 0 : KI == 16 ? 1 : KI == 32 ? 2 : KI == 48 ? 3 : 4; }

// transmit tiles per synthetic-aperture group: every transmitter up to 128
// elements, groups of 4 tiles beyond (the staged tile within 128 KiB)
int sa_mt(int KI) { return KI <= 32 ? KI / 4 : 4; }

// transmit tiles per plane-wave group beyond 128 elements: the staged FP32 tile
// (MT x KI x 512 bytes) within 80 KiB
int pw_mt_wide(int KI) { return KI <= 32 ? 5 : 81920 / (KI * 512); }

struct Common {
    const double *px, *pz;
    int n_x, n_z, n_t, n_el, n_tx;
    double f_s, width, pitch, c0, t0;
    int semantics, precision, scale, index_gpu, verbosity;
};

void destroy(fn_plan *p)
{
    if (!p) return;
    destroy(p->shallow);
    hipFree(p->d_block); hipFree(p->d_xlp_own); hipFree(p->d_ip); hipFree(p->d_simg); hipFree(p->d_sw); hipFree(p->d_P); hipFree(p->d_Z); hipFree(p->d_part); hipFree(p->d_qtab); hipFree(p->d_vsc); hipFree(p->d_nw);
    hipFree(p->d_sigF); hipFree(p->d_pimg); hipFree(p->d_ptan);
    for (auto &r : p->pending) { hipEventDestroy(r.e0); hipEventDestroy(r.e1); hipEventDestroy(r.e2); }
    for (auto &r : p->spare) { hipEventDestroy(r.e0); hipEventDestroy(r.e1); hipEventDestroy(r.e2); }
    if (p->stream) hipStreamDestroy(p->stream);
    delete p;
}

// sub-allocation of a device block: 256-byte aligned pieces
struct Carve {
    size_t used = 0;
    size_t take(size_t bytes)
    {
        const size_t at = used;
        used += (bytes + 255) & ~(size_t)255;
        return at;
    }
};

// transmit tiles per group the autotuner may try: the default cap, and for fp16
// ensembles at 128 elements up to 8 (one wave per SIMD; each weight serves 128 rows)
int max_tiles(const fn_plan *P)
{
    if (P->mode == 1) return sa_mt(P->KI);
    if (P->lbl) return 1;
    if (P->nw) return std::min(P->MT_all, 2);
    if (P->n_frames > 1 && P->kprec == FN_PRECISION_FP16 && P->KI == 32) return std::min(P->MT_all, 8);
    return std::min(P->MT_all, std::min(tile_cap(P->n_frames, P->precision, P->KI), pw_mt_wide(P->KI)));
}

#ifndef FN_FEW_ROWS_BLOCKS
#define FN_FEW_ROWS_BLOCKS 8192L
#endif
static bool few_rows_pw(const fn_plan *P)
{
    return P->mode == 0 && P->n_frames == 1 && !P->lbl && P->MT_tmpl <= 2;
}

// lateral positions symmetric about the array to 1e-12 pitches (create_common then looks at
// every aperture: mirror_check_kernel).  Not the boxcar window at one F-number for every bin, whose
// images of some size are interpolated; what is left of them is small.
bool mirrored_positions(const fn_plan *P, const Common &c, const double *Frx, int n_f)
{
    if (!Frx || c.n_x < 2) return false;
    if (P->wcr == fnk::WC_RANGE && std::all_of(Frx, Frx + n_f, [&](double F) { return F == Frx[0]; })) return false;
    for (int i = 0; i < (c.n_x + 1) / 2; ++i)
        if (!(std::fabs(c.px[i] + c.px[c.n_x - 1 - i]) <= 1e-12 * c.pitch)) return false;
    return true;
}

// Plans whose lanes may stand for two mirrored voxels: single-frame plane waves in the fp16
// split whose transmit rows fill one or two tiles (one at 129-192 elements), where the vector
// work of the weights bounds the kernel, on symmetric lateral positions.  In
// ms without / with (256 x 256): 11 angles 3.12 / 2.42, 31 angles 4.00 / 3.28, 192 elements
// 5.96 / 4.42; from three tiles on the products bound it and twice the tiles have no room in
// registers and LDS; 256 elements 7.27 / 9.59.  The one-pass fp16 form, whose operands' rounding
// shows in the image, keeps one voxel a lane, so that a plan's image does not depend on whether
// it runs alone or in a batch.
bool mirror_plan(const fn_plan *P, const Common &c, const double *Frx, int n_f)
{
    if (P->mode != 0 || P->n_frames > 1 || P->lbl || P->nw || P->kprec != FN_PRECISION_FP16X3) return false;
    if (P->KI > 48 || P->MT_all > (P->KI <= 32 ? 2 : 1)) return false;
    return mirrored_positions(P, c, Frx, n_f);
}

// Plans that may mirror: look at the apertures on the device and wait for the answer; leave the
// look to the planes kernel of a one-shot call, which finds the answer in its image and runs
// again in the rare case (one more launch or copy there is 20 to 70 us of 750); or one voxel a
// lane.
enum class Mirror { check, later, no };

// shared configuration of plan creation: tiling, launch shape and the scalar
// arguments of the kernels; no device work and no allocation (the
// no-allocation entry point runs it on a plan held on the stack)
int configure_common(fn_plan *P, const Common &c, const fnh::Grid &g, const double *Frx, bool mirror = true,
                     Planes planes = Planes::plan)
{
    if (c.precision < FN_PRECISION_FP32 || c.precision > FN_PRECISION_FP16)
        return fail(FN_ERR_ARGUMENT, "unknown precision %d", c.precision);
    P->device = c.index_gpu;
    P->g = g;
    P->n_x = c.n_x; P->n_z = c.n_z; P->n_t = c.n_t; P->n_el = c.n_el; P->n_tx = c.n_tx;
    P->n_vox = (long)c.n_x * c.n_z;
    P->verbosity = c.verbosity;
    P->precision = c.precision;
    P->KI = ki_of(c.n_el);
    P->planes = planes;
    P->kprec = planes == Planes::none ? c.precision : kernel_precision(P, c.precision);
    if (!P->KI) return fail(FN_ERR_UNSUPPORTED, "at most 256 array elements are supported (got %d)", c.n_el);
    if (P->KI > 32) {
        // beyond 128 elements: the one-launch forward kernel of single-frame plans
        if (P->n_frames > 1) return fail(FN_ERR_UNSUPPORTED, "ensembles: at most 128 elements (got %d)", c.n_el);
        if (P->lbl) return fail(FN_ERR_UNSUPPORTED, "line scans: at most 128 elements (got %d)", c.n_el);
        if (P->nw)
            return fail(FN_ERR_UNSUPPORTED, "normalizations.windowed (CPU semantics): at most 128 elements (got %d)",
                        c.n_el);
    }
    // operand rows: an ensemble's angles x frame slots (frames rounded up to a multiple
    // of 4, angle-major), otherwise the transmit rows
    const int op_rows = P->n_frames > 1 ? P->ens_angles * P->args.ens_slots : c.n_tx;
    P->MT_all = (op_rows + 15) / 16;
    if (P->lbl) {
        // line scan: one group per grid column (fn_lines.hip)
        P->MT_tmpl = 1;
        P->n_groups = c.n_x;
    } else if (P->mode == 0) {
        // at most 5 transmit tiles per group keep the LDS tile within 80 KiB
        // (ensembles: 4-5, for the per-row image accumulators)
        const int max_tiles = P->nw ? 2 : std::min(tile_cap(P->n_frames, P->precision, P->KI), pw_mt_wide(P->KI));
        const int groups = (P->MT_all + max_tiles - 1) / max_tiles;
        P->MT_tmpl = (P->MT_all + groups - 1) / groups;
        P->n_groups = (P->MT_all + P->MT_tmpl - 1) / P->MT_tmpl;
    } else {
        P->MT_tmpl = sa_mt(P->KI);
        P->n_groups = (P->MT_all + P->MT_tmpl - 1) / P->MT_tmpl;
    }
    P->mirror = mirror && mirror_plan(P, c, Frx, g.n_f);
    P->line_mirror = mirror && P->lbl && mirrored_positions(P, c, Frx, g.n_f);
    const size_t step_bytes = form_step_bytes(P->kprec);
    P->lds_beam = (size_t)P->MT_tmpl * P->KI * step_bytes;
    P->lds_spec = (size_t)g.N * sizeof(float2) + 64 * 65 * sizeof(float);
    if (P->lds_beam > kMaxLds) return fail(FN_ERR_UNSUPPORTED, "transmit tile exceeds LDS");
    if (P->lds_spec > kMaxLds) return fail(FN_ERR_UNSUPPORTED, "DFT order %d too large for the LDS twiddle table", g.N);

    // bin split: enough workgroups to fill 256 CUs several times over
    const long tiles = beam_tiles(P);
    const long blocks = tiles * P->n_groups;
    int split = 1;  // windowed normalization: every block walks all bins (valid-row counts)
    if (P->lbl) {
        // line scans: about 3072 workgroups (two rounds of the 1280 that fit and some; mirrored
        // columns share one), at most 12 chunks.  ms at 1 / 6 / 12 chunks: 128 lines x 512 depths
        // 2.46 / 2.04 / 2.05, 64 x 256 1.71 / 0.81 / 0.84, 101 x 300 1.78 / 1.25 / 1.17; 256 x 1024
        // at 1 / 2 / 12 7.46 / 7.23 / 7.70
        const long wg = tiles * (P->line_mirror ? (c.n_x + 1) / 2 : c.n_x);
        split = (int)std::min<long>({(3072 + wg - 1) / wg, 12L, (long)std::max(1, g.n_f / 16)});
    } else if (!P->nw && blocks < (few_rows_pw(P) ? FN_FEW_ROWS_BLOCKS : 2048L)) {
        // single-frame plane waves of one or two transmit tiles per group (vector-ALU
        // bound element loops): about FN_FEW_ROWS_BLOCKS blocks, otherwise about 2048
        const long target = few_rows_pw(P) ? FN_FEW_ROWS_BLOCKS : 2048L;
        split = (int)std::min<long>((target + blocks - 1) / blocks, std::max(1, g.n_f / 8));
    } else if (P->mode == 0 && !P->nw && P->n_frames == 1) {
        // a group's band spectra beyond 32 MiB (many transmit tiles, a long band): about 4 MiB
        // (an XCD's L2) to a chunk of bins, at most 16.  The kernels on FP32 instructions, whose
        // workgroups kept in step, fetched half as much beyond L2 with it.  The present ones drift
        // apart within a chunk and the count hardly matters; it stays, with the sums' order, where it
        // was.  ms at 1 / 2 / 4 / 8 / 16 / 32 chunks: 75 angles x 1455 bins 179.0 / 178.4 / 179.1 /
        // 179.7 / 179.9 / 177.9, bf16x3 x 542 bins 32.1 / 31.9 / 31.9 / 32.2 / 32.9 / 34.3
        const double set = (double)g.n_f * (double)P->lds_beam;
        if (set > 32.0 * 1048576.0)
            split = (int)std::min<double>({16.0, std::ceil(set / (4.0 * 1048576.0)), (double)std::max(1, g.n_f / 8)});
    }
    int chunk = (g.n_f + split - 1) / split;
    if (P->lbl) chunk = (chunk + 15) / 16 * 16;  // whole rounds of its four waves, four bins each
    P->bin_split = (g.n_f + chunk - 1) / chunk;
    P->x_bytes = (size_t)g.n_f * P->MT_all * P->KI * 64 * sizeof(float2);
    P->xlp_tiles = 0;
    if (P->kprec != FN_PRECISION_FP32 && !P->lbl) {
        P->xlp_tiles = P->mirror ? 2 * P->MT_all : plane_tiles(P);
        // (the tangent runs pairs of tiles)
        if (P->planes == Planes::plan && P->mode == 0 && P->n_frames == 1 && P->KI <= 32 && P->precision == FN_PRECISION_FP32)
            P->xlp_tiles = std::max(P->xlp_tiles, P->MT_all > 1 ? (P->MT_all + 1) / 2 * 2 : 1);
    }
    P->xlp_bytes = plane_bytes(P, P->xlp_tiles);

    fnk::BeamArgs &A = P->args;
    A.ctof = c.c0;
    A.dimage = nullptr;
    A.n_x = c.n_x; A.n_z = c.n_z; A.n_el = c.n_el; A.n_tx = op_rows;
    A.n_f = g.n_f; A.n_lb = g.n_lb; A.N = g.N;
    A.bin_chunk = chunk;
    A.tx_group = P->MT_tmpl;
    A.M = (c.n_el - 1) / 2.0;
    A.pitch = c.pitch; A.width = c.width; A.c0 = c.c0; A.f_s = c.f_s; A.t0 = c.t0;
    // das_pw.m:384,467 (CPU: 2 * sum) vs gpu_bf_das_pw_rf.cu:1118-1119 (MEX: 2 / N * sum)
    A.out_scale = (c.scale == FN_SCALE_CPU) ? 2.0f : (float)(2.0 / g.N);

    fnk::SpecArgs &S = P->sargs;
    S.n_t = c.n_t; S.n_ch = c.n_el * c.n_tx; S.N = g.N; S.n_lb = g.n_lb; S.n_f = g.n_f;
    S.n_el = c.n_el; S.n_tx = op_rows; S.MT = P->MT_all; S.KI = P->KI;
    S.row0 = 0; S.MT_out = P->MT_all; S.write_pad = 1;
    S.ens_slots = P->args.ens_slots;
    S.ens_frames = P->args.ens_frames;
    S.ens_angles = P->n_frames > 1 ? P->ens_angles : 0;

    P->flops = 8.0 * g.n_f * (double)P->n_vox * c.n_el * (P->lbl ? 1 : c.n_tx);
    return FN_OK;
}

fnk::MirrorArgs mirror_args(const fn_plan *P)
{
    const fnk::BeamArgs &A = P->args;
    return {P->d_tie, A.px, A.pz, A.Frx, A.sqrt_f, A.M, A.pitch, A.c0, A.n_x, A.n_z, A.n_el, A.n_f, A.clamp};
}

int interp_points(const fn_plan *P);

// planes of `tiles` tiles and more: of every tiling a plan may be given, once, beside those of its
// block (which a captured graph may still read)
int ensure_planes(fn_plan *P, int tiles)
{
    if (P->kprec == FN_PRECISION_FP32 || P->lbl || tiles <= P->xlp_tiles) return FN_OK;
    const int most = std::max(tiles, P->MT_all + std::max(P->MT_tmpl, max_tiles(P)) - 1);
    HIP_CHECK(hipSetDevice(P->device), "hipSetDevice");
    HIP_CHECK(hipMalloc(&P->d_xlp_own, plane_bytes(P, most)), "16-bit spectra planes");
    P->xlp_tiles = most;
    P->xlp_bytes += plane_bytes(P, most);
    P->d_Xlp = P->d_xlp_own;
    P->args.Xlp = P->d_Xlp;
    return FN_OK;
}

// shared part of plan creation, after configure_common: the device tables and workspace.
// One allocation and one copy: the tables (positions, F-numbers, sqrt(f_n), transmit rows
// txp, twiddles, zero delay offsets) are laid out on the host first.  Every slot of the
// spectra and their planes is written by each execute, padding as zeros.
int create_common(fn_plan *P, const Common &c, const fnh::Grid &g, const double *Frx, const double *Ftx,
                  const std::vector<double> &txp, const fn_plan *spectra_of = nullptr, Mirror how = Mirror::check)
{
    int s;
    if ((s = select_device(c.index_gpu))) return s;

    HIP_CHECK(hipStreamCreateWithFlags(&P->stream, hipStreamNonBlocking), "hipStreamCreate");
    P->h_px.assign(c.px, c.px + c.n_x);
    P->h_pz.assign(c.pz, c.pz + c.n_z);
    P->h_Frx.assign(Frx, Frx + g.n_f);
    if (Ftx) P->h_Ftx.assign(Ftx, Ftx + g.n_f);
    // sqrt(f_n) per bin for the depth clamp of the F-number
    P->h_sqf.resize(g.n_f);
    for (int b = 0; b < g.n_f; ++b) P->h_sqf[b] = std::sqrt(c.f_s * (double)(g.n_lb + b) / g.N);
    // twiddles e^{+j 2 pi m / N} rounded once from long double (conjugated in the kernel);
    // those of N - m are the conjugates
    std::vector<float2> tw(g.N);
    for (int m = 0; m <= g.N / 2; ++m) {
        const long double ang = 2.0L * 3.141592653589793238462643383279502884L * (long double)m / (long double)g.N;
        long double sn, cs;
        sincosl(ang, &sn, &cs);
        tw[m] = make_float2((float)cs, (float)sn);
        if (m) tw[g.N - m] = make_float2((float)cs, -(float)sn);
    }
    Carve cv;
    const size_t o_px = cv.take(c.n_x * sizeof(double)), o_pz = cv.take(c.n_z * sizeof(double));
    const size_t o_F = cv.take(g.n_f * sizeof(double)), o_Ft = cv.take(Ftx ? g.n_f * sizeof(double) : 0);
    const size_t o_sqf = cv.take(g.n_f * sizeof(double)), o_txp = cv.take(txp.size() * sizeof(double));
    const size_t o_tw = cv.take(tw.size() * sizeof(float2)), o_dl = cv.take(c.n_el * sizeof(double));
    const size_t o_zr = cv.take(c.n_el * sizeof(double));
    const size_t o_tie = cv.take(sizeof(uint32_t));
    const size_t tables = cv.used;
    // (an interpolated image takes no planes: only its plan's tangent does)
    const bool lp = P->xlp_tiles > 0;
    if (!spectra_of && interp_points(P)) P->xlp_tiles = 0;
    P->xlp_bytes = plane_bytes(P, P->xlp_tiles);
    const size_t o_X = cv.take(spectra_of ? 0 : P->x_bytes), o_Xlp = cv.take(P->xlp_bytes);
    const size_t o_xs = cv.take(lp ? g.n_f * sizeof(float) : 0);
    P->args.bad_rows = P->n_frames > 1 ? 16 * P->MT_all : 1;
    P->args.bad_words = bad_words(P->KI);
    const size_t o_bad = cv.take(lp ? bad_bytes(g.n_f, P->args.bad_rows, P->KI) : 0);
    const size_t o_rs = cv.take(P->n_frames > 1 && has_row_scales(P->kprec) ? row_scale_bytes(P->MT_all) : 0);
    const size_t o_xr = cv.take(P->lbl ? (size_t)g.n_f * c.n_x * c.n_el * sizeof(float2) : 0);
    const size_t o_lf = cv.take(P->lbl ? lines_flags(P) * sizeof(uint32_t) + bad_bytes(g.n_f, c.n_x, P->KI) : 0);
    std::vector<unsigned char> h(tables, 0);
    auto put = [&](size_t at, const void *src, size_t bytes) { if (bytes) std::memcpy(h.data() + at, src, bytes); };
    put(o_px, c.px, c.n_x * sizeof(double));
    put(o_pz, c.pz, c.n_z * sizeof(double));
    put(o_F, Frx, g.n_f * sizeof(double));
    if (Ftx) put(o_Ft, Ftx, g.n_f * sizeof(double));
    put(o_sqf, P->h_sqf.data(), g.n_f * sizeof(double));
    put(o_txp, txp.data(), txp.size() * sizeof(double));
    put(o_tw, tw.data(), tw.size() * sizeof(float2));
    HIP_CHECK(hipMalloc(&P->d_block, cv.used), "plan tables and spectra workspace");
    HIP_CHECK(hipMemcpy(P->d_block, h.data(), tables, hipMemcpyHostToDevice), "plan tables");
    auto at = [&](size_t o) { return reinterpret_cast<double *>(P->d_block + o); };
    P->d_px = at(o_px);
    P->d_pz = at(o_pz);
    P->d_Frx = at(o_F);
    P->d_Ftx = Ftx ? at(o_Ft) : nullptr;
    P->d_sqf = at(o_sqf);
    P->d_txp = txp.empty() ? nullptr : at(o_txp);
    P->d_tw = reinterpret_cast<float2 *>(at(o_tw));
    P->d_delay = at(o_dl);
    P->d_zeros = at(o_zr);
    P->d_X = spectra_of ? spectra_of->d_X : reinterpret_cast<float2 *>(at(o_X));
    P->d_Xlp = P->xlp_bytes ? at(o_Xlp) : nullptr;
    P->d_bad = lp ? reinterpret_cast<uint32_t *>(at(o_bad)) : nullptr;
    P->d_rowscale = P->n_frames > 1 && has_row_scales(P->kprec) ? reinterpret_cast<float *>(at(o_rs)) : nullptr;
    P->d_Xrow = P->lbl ? reinterpret_cast<float2 *>(at(o_xr)) : nullptr;
    P->d_lflag = P->lbl ? reinterpret_cast<uint32_t *>(at(o_lf)) : nullptr;
    P->d_xscale = lp ? reinterpret_cast<float *>(at(o_xs)) : nullptr;

    fnk::BeamArgs &A = P->args;
    A.X = P->d_X;
    A.delay = P->d_delay;
    A.Xlp = P->d_Xlp;
    A.xscale = P->d_xscale;
    A.bad = P->d_bad;
    A.row_scale = P->d_rowscale;
    A.px = P->d_px; A.pz = P->d_pz; A.Frx = P->d_Frx; A.Ftx = P->d_Ftx; A.txp = P->d_txp; A.sqrt_f = P->d_sqf;
    if (P->mirror || P->line_mirror) {
        P->d_tie = reinterpret_cast<uint32_t *>(P->d_block + o_tie);
        P->tie_later = how == Mirror::later && !P->lbl;  // (line scans have no planes)
        if (!P->tie_later) {
            uint32_t tie = 0;
            const dim3 grid((unsigned)(((long)(c.n_x / 2) * c.n_z + 255) / 256),
                            (unsigned)((g.n_f + fnk::MIRROR_BINS - 1) / fnk::MIRROR_BINS));
            hipLaunchKernelGGL(fnk::mirror_check_kernel, grid, dim3(256), 0, P->stream, mirror_args(P));
            HIP_CHECK(hipGetLastError(), "mirror_check_kernel");
            HIP_CHECK(hipMemcpyAsync(&tie, P->d_tie, sizeof(tie), hipMemcpyDeviceToHost, P->stream), "mirror_check_kernel");
            HIP_CHECK(hipStreamSynchronize(P->stream), "mirror_check_kernel");
            // one voxel a lane: the planes of either tiling fit the mirrored ones' room
            const int tiles = P->xlp_tiles;
            if (tie && (s = configure_common(P, c, g, Frx, false))) return s;
            P->xlp_tiles = tiles;
            P->xlp_bytes = plane_bytes(P, tiles);
        }
    }
    return ensure_partials(P);
}

// Elements whose weight can be nonzero for one voxel and bin: the aperture of
// das_pw.m:387-411 (das_sa.m:384-400) -- the open boxcar support (CPU), the snapped
// [lb, ub] of a window that vanishes beyond it, or every element of an untruncated
// window (CPU Hann and triangular) on a non-empty aperture; 0 where the aperture is
// empty (the bin is skipped).
int active_elements(double x, double z, double F, int support, double pitch, int n_el)
{
    const double M = (n_el - 1) / 2.0;
    const double hp = z / (2.0 * pitch * F);  // h / pitch (F = 0: the whole array)
    const double ua = M + (x / pitch - hp), ub = M + (x / pitch + hp);
    const double lb = std::fmax(std::ceil(ua), 0.0), ubd = std::fmin(std::floor(ub), n_el - 1.0);
    if (lb > ubd) return 0;
    if (support == fnk::SUPPORT_OPEN_H) {
        const double lo = std::fmax(std::floor(ua) + 1.0, 0.0), hi = std::fmin(std::ceil(ub) - 1.0, n_el - 1.0);
        return hi >= lo ? (int)(hi - lo) + 1 : 0;
    }
    if (support == fnk::SUPPORT_ALL) return n_el;
    return (int)(ubd - lb) + 1;
}

// Useful complex multiply-adds per frame for the roofline (8 flop each): the sum over
// voxels and bins of the active receive elements times the transmit rows (plane
// waves), or times the active transmitters (synthetic aperture), from a sample of
// about 64 x 64 voxels and every bin, scaled to the grid.
double useful_macs(const fn_plan *P)
{
    const int nx = P->n_x, nz = P->n_z;
    const double *px = P->h_px.data(), *pz = P->h_pz.data(), *Frx = P->h_Frx.data(), *Ftx = P->h_Ftx.data();
    const double f_s = P->args.f_s, c0 = P->args.c0, pitch = P->args.pitch;
    const fnh::Grid &g = P->g;
    const int sx = std::max(1, nx / 64), sz = std::max(1, nz / 64);
    double sum = 0.0;
    long n = 0;
    for (int ix = 0; ix < nx; ix += sx)
        for (int iz = 0; iz < nz; iz += sz, ++n)
            for (int b = 0; b < g.n_f; ++b) {
                double Fr = Frx[b];
                if (P->args.clamp) {
                    const double fn = f_s * (double)(g.n_lb + b) / g.N;
                    Fr = std::fmin(Fr, std::sqrt(fn * pz[iz] / (2.88 * c0)));  // das_pw.m:374-377
                }
                const int k = active_elements(px[ix], pz[iz], Fr, P->args.support_rx, pitch, P->n_el);
                if (!k) continue;
                if (P->mode == 1) {
                    const int t = active_elements(px[ix], pz[iz], Ftx[b], P->args.support_tx, pitch, P->n_el);
                    sum += (double)k * t;
                } else {
                    sum += (double)k * (P->lbl ? 1 : P->n_tx);  // a line scan's voxel meets one row
                }
            }
    return n ? sum / n * (double)P->n_vox : 0.0;
}

// interpolated plans: the two tables behind the channel samples
size_t interp_samples(const fn_plan *P) { return fnk::interp_table_floats2(P->interp_M, P->n_tx, P->n_el); }
float2 *interp_tw(const fn_plan *P) { return P->d_ip + interp_samples(P); }
float *interp_ipsi(const fn_plan *P) { return reinterpret_cast<float *>(interp_tw(P) + P->interp_M); }

// leading depths up to the last one where the clamp min(F, sqrt(f z / (2.88 c))) of the first
// F-number bites at the lowest frequency (das_pw.m:374-377)
int clamped_depths(const fn_plan *P)
{
    int n = 0;
    for (int i = 0; P->args.clamp && i < P->n_z; ++i)
        if (!(P->h_sqf[0] * std::sqrt(P->h_pz[i] / (2.88 * P->args.c0)) >= P->h_Frx[0])) n = i + 1;
    return n;
}

// Estimated seconds of the two forms of an image: the sum over the bins of MT transmit tiles
// (0.9 us + 0.35 us per tile for 16 voxels and a bin) and the interpolation of M samples per
// channel (8 n_f M flop per padded channel at 100 TFLOP/s, then 75 ns per 64 voxels, element and
// angle), each over 1024 SIMDs.
double sum_seconds(const fn_plan *P, int MT)
{
    return P->n_vox / 16.0 * P->g.n_f * (0.9 + 0.35 * MT) * (P->KI / 32.0) * 1e-6 / 1024.0;
}
double interp_seconds(const fn_plan *P, long M)
{
    return 8.0 * P->g.n_f * M * (16.0 * P->MT_all) * (4.0 * P->KI) / 1e14 +
           P->n_vox / 64.0 * P->n_el * P->n_tx * 75e-9 / 1024.0;
}

// Samples per channel of a plan whose image can be interpolated (fn_interp.hip), 0 otherwise:
// FP32 plane waves of one frame with one F-number for every bin; the depths where its clamp is
// at work, at most half of them, have a plan of their own.  31 angles, boxcar, 512 x 384 (432
// bins): 0.9 ms against 7.2 for the sum over the bins, and 0.23 for the samples; 75 angles,
// 1024 x 512 (1455 bins, 14 % of the depths clamped): 27 ms against 118.  The samples cost the
// same for any image, so the line is where both forms' estimated times cross (100 x 77 voxels,
// 11 angles, 542 bins: 0.39 ms against 0.45; a quarter of these voxels: about even).  The samples
// stay within 2 GiB (a hundredth of the card's memory) and their twiddles within LDS.
int interp_points(const fn_plan *P)
{
    const int n_f = P->g.n_f;
    if (P->mode != 0 || P->n_frames > 1 || P->lbl || P->nw || P->precision != FN_PRECISION_FP32) return 0;
    const double F = P->h_Frx[0];
    if (!std::all_of(P->h_Frx.begin(), P->h_Frx.end(), [&](double f) { return f == F; })) return 0;
    if (2 * clamped_depths(P) > P->n_z) return 0;
    const long M = ((9L * n_f + 3) / 4 + 15) / 16 * 16;
    if (M * 8 + (long)n_f * 4 > fnk::INTERP_LDS_MAX) return 0;
    if (fnk::interp_table_floats2((int)M, P->n_tx, P->n_el) * sizeof(float2) > ((size_t)2 << 30)) return 0;
    return interp_seconds(P, M) > sum_seconds(P, P->MT_all) ? 0 : (int)M;
}

int pw_plan(const fn_pw_params *p, fn_plan **out, const fn_plan *spectra_of = nullptr, Mirror how = Mirror::check);

// the interpolated form's buffers (and the plan of its clamped depths); a plan without room for
// them, or whose clamped depths have another DFT, keeps the sum over the bins
int setup_interp(fn_plan *P, const fn_pw_params *p)
{
    P->interp_M = interp_points(P);
    if (!P->interp_M) return FN_OK;
    auto keep_sum = [&]() {
        destroy(P->shallow);
        hipFree(P->d_simg); hipFree(P->d_sw); hipFree(P->d_ip);
        P->shallow = nullptr;
        P->d_simg = P->d_ip = nullptr;
        P->d_sw = nullptr;
        P->interp_M = 0;
        (void)hipGetLastError();
        fnh::clear_error();
        return ensure_planes(P, plane_tiles(P));
    };
    const int nz = clamped_depths(P);
    if (nz > 0) {
        fn_pw_params q = *p;
        q.n_z = nz;
        if (pw_plan(&q, &P->shallow, P) != FN_OK) return keep_sum();
        const fnh::Grid &a = P->g, &b = P->shallow->g;
        if (a.N != b.N || a.n_lb != b.n_lb || a.n_f != b.n_f) return keep_sum();
        if (hipMalloc(&P->d_simg, (size_t)P->n_x * nz * sizeof(float2)) != hipSuccess ||
            hipMalloc(&P->d_sw, (size_t)P->n_x * nz * sizeof(float)) != hipSuccess)
            return keep_sum();
    }
    const size_t bytes = (interp_samples(P) + P->interp_M) * sizeof(float2) + P->g.n_f * sizeof(float);
    if (hipMalloc(&P->d_ip, bytes) != hipSuccess) return keep_sum();
    if (ensure_partials(P) != FN_OK) {
        if (int s = keep_sum()) return s;
        return ensure_partials(P);
    }
    const hipError_t e = fnk::launch_interp_tables(interp_tw(P), interp_ipsi(P), P->interp_M, P->g.n_f, P->stream);
    if (e != hipSuccess) return hip_fail(e, "interp_tables_kernel");
    HIP_CHECK(hipStreamSynchronize(P->stream), "interp_tables_kernel");
    return FN_OK;
}

// device bytes of interpolated channel samples, their tables and the plan of the clamped depths
size_t interp_bytes(const fn_plan *P)
{
    if (!P->interp_M) return 0;
    size_t n = (interp_samples(P) + P->interp_M) * sizeof(float2) + P->g.n_f * sizeof(float);
    if (P->shallow) n += P->shallow->xlp_bytes + (size_t)P->shallow->n_vox * (sizeof(float2) + sizeof(float));
    return n;
}

// device bytes of a line scan's spectra by rows
size_t row_bytes(const fn_plan *P) { return P->lbl ? (size_t)P->g.n_f * P->n_x * P->n_el * sizeof(float2) : 0; }

// the spectra and everything that is laid out from them
size_t workspace_bytes(const fn_plan *P) { return P->x_bytes + P->xlp_bytes + interp_bytes(P) + row_bytes(P); }

hipError_t launch_beam(const fn_plan *P, dim3 grid, const fnk::BeamArgs &A, hipStream_t s)
{
    if (P->interp_M) {
        fnk::InterpArgs S{};
        S.B = A;
        S.B.wrx = P->args.wrx;  // FP32 weights
        S.G = P->d_ip;
        S.M = P->interp_M;
        S.n_c = (uint32_t)(P->g.n_lb + P->g.n_f / 2);
        S.empty_weight = P->wcr == fnk::WC_COS_ALL ? (float)P->n_el : 0.f;  // as the full-array class reports it
        return fnk::launch_interp_beamform(wcr_general(P->wcr), S, s);
    }
    const int kidx = ki_index(P->KI);  // ensembles, line scans and windowed plans stop at KI = 32
    if (P->lbl)
        return fnk::launch_lines(P->wcr, P->line_mirror && P->delays_even, (int)grid.x, (int)grid.y, A, P->d_Xrow,
                                 P->d_lflag, P->d_lflag + lines_flags(P), bad_words(P->KI), s);
    if (use_mirror(P)) return fnk::kMirLaunchers[kidx](P->MT_tmpl, P->wcr, grid, P->lds_beam, s, A);
    if (P->nw) return fnk::kNwLaunchers[P->mode][kidx](P->MT_tmpl, P->wcr, P->wct, grid, P->lds_beam, s, A);
    if (P->n_frames > 1) return fnk::kEnsLaunchers[kidx][P->kprec](P->MT_tmpl, P->wcr, grid, P->lds_beam, s, A, 0);
    return fnk::kBeamLaunchers[P->mode][kidx][P->kprec](P->MT_tmpl, P->wcr, P->wct, grid, P->lds_beam, s, A);
}

// raise a kernel's dynamic-LDS limit once per process and size (no attribute
// calls inside captured launch sequences)
hipError_t lds_limit(const void *kern, size_t lds, size_t &done)
{
    if (lds <= 65536 || lds <= done) return hipSuccess;
    hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e == hipSuccess) done = lds;
    return e;
}

// the band spectra of RF d_rf into the operand layout X described by S
int launch_spectra_into(const fn_plan *P, const void *d_rf, int dtype, hipStream_t s, float2 *X,
                        const fnk::SpecArgs &S)
{
    // 64 bins x one operand group (16 rows x 4 elements) per block
    dim3 sg((unsigned)((S.n_f + 63) / 64), (unsigned)(S.MT * S.KI));
    static size_t done_f = 0, done_d = 0;
    HIP_CHECK(dtype == FN_DTYPE_F32
                  ? lds_limit(reinterpret_cast<const void *>(fnk::spectra_kernel<float>), P->lds_spec, done_f)
                  : lds_limit(reinterpret_cast<const void *>(fnk::spectra_kernel<double>), P->lds_spec, done_d),
              "spectra LDS limit");
    if (dtype == FN_DTYPE_F32) {
        hipLaunchKernelGGL(fnk::spectra_kernel<float>, sg, dim3(256), P->lds_spec, s,
                           reinterpret_cast<const float *>(d_rf), P->d_tw, X, S);
    } else {
        hipLaunchKernelGGL(fnk::spectra_kernel<double>, sg, dim3(256), P->lds_spec, s,
                           reinterpret_cast<const double *>(d_rf), P->d_tw, X, S);
    }
    HIP_CHECK(hipGetLastError(), "spectra_kernel");
    return FN_OK;
}

int launch_spectra(fn_plan *P, const void *d_rf, int dtype, hipStream_t s)
{
    P->executed = 1;
    return launch_spectra_into(P, d_rf, dtype, s, P->d_X, P->sargs);
}

// the arguments of the forward kernels: the fp16 split evaluates a bounded receive window
// times an exact factor (SPLIT_PEAK)
fnk::BeamArgs forward_args(const fn_plan *P)
{
    fnk::BeamArgs A = P->args;
    A.xlp_tiles = plane_tiles(P);
    if (P->kprec == FN_PRECISION_FP16X3 && !unbounded_window(P->wcr, A.wrx)) {
        A.wrx.A *= fnk::SPLIT_PEAK;
        A.wrx.B *= fnk::SPLIT_PEAK;
        A.wrx.C *= fnk::SPLIT_PEAK;
        A.wrx.peak = fnk::SPLIT_PEAK;
        A.wrx.inv_peak = 1.0f / fnk::SPLIT_PEAK;
    }
    return A;
}

// the beamforming arguments of one execute (image and weight buffers)
fnk::BeamArgs beam_args(const fn_plan *P, float *d_image, float *d_w, float *d_w_rx)
{
    fnk::BeamArgs A = forward_args(P);
    if (P->interp_M || P->lbl) A.bad = nullptr;               // no planes
    A.tie = P->tie_later && use_mirror(P) ? P->d_tie : nullptr;
    if (plane_delay(P, use_mirror(P))) A.delay = P->d_zeros;  // in the planes already
    A.image = reinterpret_cast<float2 *>(d_image);
    A.n_slots = beam_slots(P);
    A.slot_z = P->lbl ? 1 : P->n_groups;
    A.partial = A.n_slots > 1 ? P->d_pimg : nullptr;
    if (P->mode == 0) {
        A.weights = d_w;
        A.weights_tx = nullptr;
    } else {
        A.weights = d_w_rx;
        A.weights_tx = d_w;
    }
    return A;
}

int launch_row_scales(const float2 *X, float *scale, int MT, int KI, int n_f, hipStream_t s)
{
    const int rows = 16 * MT, chunk = (n_f + ROW_PEAK_CHUNKS - 1) / ROW_PEAK_CHUNKS, n = (n_f + chunk - 1) / chunk;
    hipLaunchKernelGGL(fnk::row_peak_kernel, dim3((unsigned)MT, (unsigned)n), dim3(256), 0, s, X, scale + 2 * rows, MT, KI,
                       n_f, chunk);
    HIP_CHECK(hipGetLastError(), "row_peak_kernel");
    hipLaunchKernelGGL(fnk::row_scale_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s, scale + 2 * rows, scale,
                       rows, n);
    HIP_CHECK(hipGetLastError(), "row_scale_kernel");
    return FN_OK;
}

// the 16-bit operand planes (and per-bin scales) of FP32 spectra X of MT tiles (MT_out,
// mirror_el, delay, bad: see lowp_planes_kernel; rowscale: launch_row_scales, null: none); nothing
// for FP32 kernels
int launch_lowp_planes(const fn_plan *P, const float2 *X, void *Xlp, float *xscale, uint32_t *bad, int bad_rows, int MT,
                       int MT_out, int mirror_el, const double *delay, hipStream_t s, float *rowscale = nullptr)
{
    const float *row_inv = rowscale ? rowscale + 16 * MT : nullptr;
    const fnk::MirrorArgs look = P->tie_later && use_mirror(P) ? mirror_args(P) : fnk::MirrorArgs{};
    if (rowscale)
        if (int st = launch_row_scales(X, rowscale, MT, P->KI, P->g.n_f, s)) return st;
    // a block per bin, and where the grid's mirror is looked at here, one more for each 2048 pairs of voxels
    const long pairs = look.tie ? (long)(look.n_x / 2) * look.n_z : 0;
    const dim3 cg((unsigned)P->g.n_f, 1 + (unsigned)std::min<long>(16, (pairs + 2047) / 2048)), cb(256);
    const double fs_over_N = P->args.f_s / P->g.N;
    switch (P->kprec) {
    case FN_PRECISION_FP32: return FN_OK;
    case FN_PRECISION_BF16X3:
        hipLaunchKernelGGL(fnk::lowp_planes_kernel<fnk::PREC_BF16X3>, cg, cb, 0, s, X, Xlp, xscale, MT, P->KI, MT_out,
                           mirror_el, delay, fs_over_N, P->g.n_lb, P->n_el, row_inv, bad, bad_rows, bad_words(P->KI), look);
        break;
    case FN_PRECISION_FP16X3:
        hipLaunchKernelGGL(fnk::lowp_planes_kernel<fnk::PREC_FP16X3>, cg, cb, 0, s, X, Xlp, xscale, MT, P->KI, MT_out,
                           mirror_el, delay, fs_over_N, P->g.n_lb, P->n_el, row_inv, bad, bad_rows, bad_words(P->KI), look);
        break;
    default:
        hipLaunchKernelGGL(fnk::lowp_planes_kernel<fnk::PREC_FP16>, cg, cb, 0, s, X, Xlp, xscale, MT, P->KI, MT_out,
                           mirror_el, delay, fs_over_N, P->g.n_lb, P->n_el, row_inv, bad, bad_rows, bad_words(P->KI), look);
        break;
    }
    HIP_CHECK(hipGetLastError(), "lowp_planes_kernel");
    return FN_OK;
}

int finish_beam(const fn_plan *P, const fnk::BeamArgs &A, hipStream_t s, float2 *dimage = nullptr);

// the clamped depths of an interpolated plan, from its spectra, pasted into its image
int run_shallow(const fn_plan *P, const fnk::BeamArgs &A, hipStream_t s)
{
    const fn_plan *C = P->shallow;
    if (int st = launch_lowp_planes(C, C->d_X, C->d_Xlp, C->d_xscale, C->d_bad, 1, C->MT_all, plane_tiles(C), use_mirror(C) ? C->n_el : 0,
                                    plane_delay(C, use_mirror(C)), s))
        return st;
    const fnk::BeamArgs B = beam_args(C, reinterpret_cast<float *>(P->d_simg), A.weights ? P->d_sw : nullptr, nullptr);
    const hipError_t e = launch_beam(C, dim3((unsigned)beam_tiles(C), (unsigned)C->bin_split, (unsigned)C->n_groups), B, s);
    if (e != hipSuccess) return hip_fail(e, "beamform_kernel");
    if (int st = finish_beam(C, B, s)) return st;
    hipLaunchKernelGGL(fnk::paste_depths_kernel, dim3((unsigned)((C->n_vox + 255) / 256)), dim3(256), 0, s, P->d_simg,
                       A.weights ? P->d_sw : nullptr, C->n_vox, C->n_z, P->n_z, A.image, A.weights);
    HIP_CHECK(hipGetLastError(), "paste_depths_kernel");
    return FN_OK;
}

// after the beamforming launch: the partial images of a voxel's workgroups summed
// in slot order into the image (none when one workgroup owns each voxel), the voxels that meet
// values that are not finite (16-bit forms), and the clamped depths of an interpolated plan
int finish_beam(const fn_plan *P, const fnk::BeamArgs &A, hipStream_t s, float2 *dimage)
{
    if (A.partial) {
        hipLaunchKernelGGL(fnk::reduce_partials_kernel, dim3((unsigned)((P->n_vox + 255) / 256)), dim3(256), 0, s, A, A.image,
                           dimage);
        HIP_CHECK(hipGetLastError(), "reduce_partials_kernel");
    } else if (A.bad) {
        hipLaunchKernelGGL(fnk::nonfinite_kernel, dim3((unsigned)((P->n_vox + 255) / 256)), dim3(256), 0, s, A);
        HIP_CHECK(hipGetLastError(), "nonfinite_kernel");
    }
    return P->shallow && !dimage ? run_shallow(P, A, s) : FN_OK;
}

// everything of an execute before the beamforming launch: the zeroed images of an
// ensemble (its frames' rows are added atomically), the band spectra and (16-bit
// forms) their planes
int prepare(fn_plan *P, const void *d_rf, int dtype, float *d_image, hipStream_t s)
{
    if (P->n_frames > 1) {
        const long n = 2 * P->n_vox * P->n_frames;
        hipLaunchKernelGGL(fnk::fill_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d_image, n);
        HIP_CHECK(hipGetLastError(), "fill_zero_kernel");
    }
    const fnk::SpecArgs &S = P->sargs;
    if (int st = launch_spectra(P, d_rf, dtype, s)) return st;
    if (P->lbl) {
        const hipError_t e = fnk::launch_lines_spectra(P->d_X, P->d_Xrow, S.n_f, S.MT, S.KI, P->n_x, P->n_el, P->d_lflag,
                                                       P->d_lflag + lines_flags(P), s);
        return e == hipSuccess ? FN_OK : hip_fail(e, "lines_spectra_kernel");
    }
    if (P->interp_M) {
        const hipError_t e = fnk::launch_interp_samples(P->d_X, interp_tw(P), interp_ipsi(P), P->d_ip, P->interp_M, S.n_f,
                                                        S.MT, S.KI, P->n_tx, P->n_el, s);
        return e == hipSuccess ? FN_OK : hip_fail(e, "interp_samples_kernel");
    }
    return launch_lowp_planes(P, P->d_X, P->d_Xlp, P->d_xscale, P->d_bad, P->args.bad_rows, S.MT, plane_tiles(P),
                              use_mirror(P) ? P->n_el : 0, plane_delay(P, use_mirror(P)), s, P->d_rowscale);
}

int execute(fn_plan *P, const void *d_rf, int dtype, float *d_image, float *d_w, float *d_w_rx, hipStream_t user)
{
    if (!P || !d_rf || !d_image) return fail(FN_ERR_ARGUMENT, "null argument");
    if (dtype != FN_DTYPE_F32 && dtype != FN_DTYPE_F64) return fail(FN_ERR_RF_DATA, "RF data must be float32 or float64");
    HIP_CHECK(hipSetDevice(P->device), "hipSetDevice");
    hipStream_t s = user;  // NULL: the default stream
    const fnk::BeamArgs A = beam_args(P, d_image, d_w, d_w_rx);
    Run run{};
    if (P->profiling) {
        if (!P->spare.empty()) {
            run = P->spare.back();
            P->spare.pop_back();
        } else {
            HIP_CHECK(hipEventCreate(&run.e0), "hipEventCreate");
            HIP_CHECK(hipEventCreate(&run.e1), "hipEventCreate");
            HIP_CHECK(hipEventCreate(&run.e2), "hipEventCreate");
        }
    }
    if (P->profiling) HIP_CHECK(hipEventRecord(run.e0, s), "hipEventRecord");
    if (int st = prepare(P, d_rf, dtype, d_image, s)) return st;
    if (P->profiling) HIP_CHECK(hipEventRecord(run.e1, s), "hipEventRecord");
    const long tiles = beam_tiles(P);
    hipError_t e = launch_beam(P, dim3((unsigned)tiles, (unsigned)P->bin_split, (unsigned)P->n_groups), A, s);
    if (e != hipSuccess) return hip_fail(e, "beamform_kernel");
    if (int st = finish_beam(P, A, s)) return st;
    if (P->profiling) {
        HIP_CHECK(hipEventRecord(run.e2, s), "hipEventRecord");
        P->pending.push_back(run);
    }
    return FN_OK;
}

int collect_profile(fn_plan *P)
{
    for (auto &r : P->pending) {
        HIP_CHECK(hipEventSynchronize(r.e2), "hipEventSynchronize");
        float a = 0.f, b = 0.f;
        HIP_CHECK(hipEventElapsedTime(&a, r.e0, r.e1), "hipEventElapsedTime");
        HIP_CHECK(hipEventElapsedTime(&b, r.e1, r.e2), "hipEventElapsedTime");
        P->spec_ms += a;
        P->beam_ms += b;
        P->runs += 1;
        P->spare.push_back(r);
    }
    P->pending.clear();
    return FN_OK;
}

// plane-wave configuration shared by plan creation and the no-allocation entry
// point: receive window, normalization, transmit rows (no device work)
int configure_pw(fn_plan *P, const fn_pw_params *p, Common *c)
{
    P->mode = 0;
    P->n_frames = std::max(1, p->n_frames);
    P->lbl = p->line_scan != 0;
    // windowed normalization: the CPU path tapers (windowed.m:81-86); the
    // reference MEX reads the window and normalizes as "on" (gpu_bf_das_pw_rf.cu:421-427)
    P->nw = p->normalization == FN_NORMALIZATION_WINDOWED && p->semantics == FN_SEMANTICS_CPU;
    int wsup = 0;
    if (int s = setup_window(p->window, p->semantics, &P->args.wrx, &P->wcr, &wsup)) return s;
    P->args.support_rx = wsup;
    P->args.norm_rx = p->normalization != FN_NORMALIZATION_OFF;
    P->args.clamp = p->semantics == FN_SEMANTICS_CPU;
    // transmit rows: every angle of every frame.  An ensemble's operand rows are
    // angle-major over frame slots (row = angle * slots + slot, slots = frames rounded up
    // to a multiple of 4), so that the four rows a lane holds per M-tile share one angle
    const int n_rows = p->n_angles * P->n_frames;
    P->args.ens_frames = P->n_frames > 1 ? P->n_frames : 0;
    P->args.ens_slots = P->n_frames > 1 ? (P->n_frames + 3) / 4 * 4 : 0;
    P->ens_angles = p->n_angles;
    P->args.tx_kind = p->virtual_sources ? fnk::TX_VIRTUAL : fnk::TX_PLANE;
    *c = Common{p->positions_x, p->positions_z, p->n_x, p->n_z, p->n_samples, p->n_elements, n_rows,
                p->f_s, p->element_width, p->element_pitch, p->c_0, p->index_t0,
                p->semantics, p->precision, p->output_scale, p->index_gpu, p->verbosity};
    return FN_OK;
}

// spectra_of: a plan of the same acquisition whose spectra this one reads (its clamped depths)
int pw_plan(const fn_pw_params *p, fn_plan **out, const fn_plan *spectra_of, Mirror how)
{
    fnh::Grid g;
    int s = fnh::validate_pw(p, &g);
    if (s) return s;
    fn_plan *P = new (std::nothrow) fn_plan();
    if (!P) return fail(FN_ERR_OUT_OF_MEMORY, "host allocation");
    Common c{};
    if ((s = configure_pw(P, p, &c))) { destroy(P); return s; }
    if ((s = configure_common(P, c, g, p->f_number_values, how != Mirror::no))) { destroy(P); return s; }
    const int n_rows = P->args.n_tx;  // operand rows (ensembles: frame slots)
    // steering geometry in FP64: das_pw.m:323-327 (x_ref = sign(e_x) x_0), or the
    // virtual sources (x_vs, z_vs, |r_vs|)
    std::vector<double> txp(3 * (size_t)n_rows);
    const double M = (p->n_elements - 1) / 2.0;
    for (int row = 0; row < n_rows; ++row) {
        const int a = P->n_frames > 1 ? row / P->args.ens_slots : row;  // angle-major ensemble rows
        if (p->virtual_sources) {
            const double xv = p->virtual_sources[2 * a], zv = p->virtual_sources[2 * a + 1];
            txp[3 * row] = xv;
            txp[3 * row + 1] = zv;
            txp[3 * row + 2] = std::sqrt(xv * xv + zv * zv);
            continue;
        }
        const double th = p->steering_angles[a];
        const double ex = -std::sin(th), ez = std::cos(th);
        const double sg = (ex > 0) - (ex < 0);
        txp[3 * row] = ex;
        txp[3 * row + 1] = ez;
        txp[3 * row + 2] = sg * ((0 - M) * p->element_pitch);
    }
    if ((s = create_common(P, c, g, p->f_number_values, nullptr, txp, spectra_of, how))) { destroy(P); return s; }
    if (P->nw && (s = setup_windowed(P, true, p->window, p->normalization_window, false, p->window,
                                     p->normalization_window))) { destroy(P); return s; }
    use_cos_all(P);
    if (!spectra_of && (s = setup_interp(P, p))) { destroy(P); return s; }
    *out = P;
    return FN_OK;
}

int sa_plan(const fn_sa_params *p, fn_plan **out)
{
    fnh::Grid g;
    int s = fnh::validate_sa(p, &g);
    if (s) return s;
    fn_plan *P = new (std::nothrow) fn_plan();
    if (!P) return fail(FN_ERR_OUT_OF_MEMORY, "host allocation");
    P->mode = 1;
    const bool cpu = p->semantics == FN_SEMANTICS_CPU;
    const bool nw_rx = cpu && p->normalization_rx == FN_NORMALIZATION_WINDOWED;
    const bool nw_tx = cpu && p->normalization_tx == FN_NORMALIZATION_WINDOWED;
    P->nw = nw_rx || nw_tx;
    int sup = 0;
    if ((s = setup_window(p->window_rx, p->semantics, &P->args.wrx, &P->wcr, &sup))) { destroy(P); return s; }
    P->args.support_rx = sup;
    if ((s = setup_window(p->window_tx, p->semantics, &P->args.wtx, &P->wct, &sup))) { destroy(P); return s; }
    P->args.support_tx = sup;
    P->args.norm_rx = p->normalization_rx != FN_NORMALIZATION_OFF;
    P->args.norm_tx = p->normalization_tx != FN_NORMALIZATION_OFF;
    P->args.clamp = 0;  // das_sa.m:354-358: no depth clamp
    Common c{p->positions_x, p->positions_z, p->n_x, p->n_z, p->n_samples, p->n_elements, p->n_elements,
             p->f_s, p->element_width, p->element_pitch, p->c_0, p->index_t0,
             p->semantics, p->precision, p->output_scale, p->index_gpu, p->verbosity};
    if ((s = configure_common(P, c, g, p->f_number_rx_values))) { destroy(P); return s; }
    if ((s = create_common(P, c, g, p->f_number_rx_values, p->f_number_tx_values, {}))) { destroy(P); return s; }
    if (P->nw && (s = setup_windowed(P, nw_rx, p->window_rx, p->normalization_window_rx, nw_tx, p->window_tx,
                                     p->normalization_window_tx))) { destroy(P); return s; }
    use_cos_all(P);
    *out = P;
    return FN_OK;
}

size_t dtype_size(int dtype) { return dtype == FN_DTYPE_F64 ? 8 : 4; }

// ---- tiling and autotuning ---------------------------------------------

int set_tiling(fn_plan *P, int mt, int split)
{
    if (!P) return fail(FN_ERR_ARGUMENT, "null plan");
    if (P->mode == 1) {
        if (mt != sa_mt(P->KI)) return fail(FN_ERR_ARGUMENT, "synthetic-aperture plans use %d transmit tiles", sa_mt(P->KI));
    } else if (mt < 1 || mt > max_tiles(P)) {
        return fail(FN_ERR_ARGUMENT, "m_tiles must be in 1..%d", max_tiles(P));
    }
    const int n_f = P->g.n_f;
    if (split < 1 || split > n_f) return fail(FN_ERR_ARGUMENT, "bin_split must be in 1..%d", n_f);
    if (P->nw && split != 1) return fail(FN_ERR_ARGUMENT, "windowed normalization runs with bin_split 1");
    if ((size_t)mt * P->KI * form_step_bytes(P->kprec) > kMaxLds) return fail(FN_ERR_ARGUMENT, "transmit tile exceeds LDS");
    const int chunk0 = P->args.bin_chunk, mt0 = P->MT_tmpl;
    auto apply = [P, n_f](int tiles, int chunk) {
        P->MT_tmpl = tiles;
        P->n_groups = P->lbl ? P->n_x : (P->MT_all + tiles - 1) / tiles;
        P->bin_split = (n_f + chunk - 1) / chunk;
        P->lds_beam = (size_t)tiles * P->KI * form_step_bytes(P->kprec);
        P->args.tx_group = tiles;
        P->args.bin_chunk = chunk;
        ++P->tiling_serial;
    };
    apply(mt, (n_f + split - 1) / split);
    int st = P->interp_M ? FN_OK : ensure_planes(P, plane_tiles(P));
    if (st == FN_OK) st = ensure_partials(P);
    if (st != FN_OK) apply(mt0, chunk0);  // no memory: the tiling before, whose buffers are there
    return st;
}

int autotune(fn_plan *P, const void *d_rf, int dtype, float *d_image, int reps, fn_tune_result *res, hipStream_t s)
{
    if (!P || !d_rf || !d_image || !res) return fail(FN_ERR_ARGUMENT, "null argument");
    reps = std::max(1, reps);
    const int mt0 = P->MT_tmpl, split0 = P->bin_split;
    std::vector<std::pair<int, int>> cand;
    const int n_f = P->g.n_f;
    const int mt_lo = P->mode == 1 ? sa_mt(P->KI) : 1, mt_hi = max_tiles(P);
    if (P->interp_M) cand.emplace_back(mt0, split0);  // (an interpolated image has no tiling)
    for (int mt = mt_lo; mt <= mt_hi && !P->interp_M; ++mt) {
        // distinct group counts only: the tile count of a balanced split
        if (P->mode == 0) {
            const int groups = (P->MT_all + mt - 1) / mt;
            if ((P->MT_all + groups - 1) / groups != mt) continue;
        }
        for (int split : {1, 2, 4, 8, 16, split0})
            if (split <= n_f && (!P->nw || split == 1) &&
                std::find(cand.begin(), cand.end(), std::make_pair(mt, split)) == cand.end())
                cand.emplace_back(mt, split);
    }
    hipEvent_t e0, e1;
    HIP_CHECK(hipEventCreate(&e0), "hipEventCreate");
    HIP_CHECK(hipEventCreate(&e1), "hipEventCreate");
    const int prof = P->profiling;
    P->profiling = 0;
    double best = 1e300, dflt = -1.0;
    int best_mt = mt0, best_split = split0, st = FN_OK;
    for (auto &c : cand) {
        if ((st = set_tiling(P, c.first, c.second))) break;
        if ((st = execute(P, d_rf, dtype, d_image, nullptr, nullptr, s))) break;  // warm-up
        hipEventRecord(e0, s);
        for (int r = 0; r < reps && !st; ++r) st = execute(P, d_rf, dtype, d_image, nullptr, nullptr, s);
        hipEventRecord(e1, s);
        if (st) break;
        hipError_t e = hipEventSynchronize(e1);
        float ms = 0.f;
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
        if (e != hipSuccess) { st = hip_fail(e, "autotune timing"); break; }
        const double per = ms / reps;
        if (c.first == mt0 && c.second == split0) dflt = per;
        if (per < best) { best = per; best_mt = c.first; best_split = c.second; }
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    P->profiling = prof;
    if (st) { set_tiling(P, mt0, split0); return st; }
    if ((st = set_tiling(P, best_mt, best_split))) return st;
    res->best_ms = best;
    res->default_ms = dflt;
    res->m_tiles = P->MT_tmpl;
    res->bin_split = P->bin_split;
    res->n_candidates = (int32_t)cand.size();
    return FN_OK;
}

// ---- differentiation form ----------------------------------------------

int set_tof(fn_plan *P, double c_tof, const double *delays)
{
    if (!P) return fail(FN_ERR_ARGUMENT, "null plan");
    if (!(c_tof == c_tof) || c_tof > DBL_MAX) return fail(FN_ERR_ARGUMENT, "c_tof must be finite");
    std::vector<double> d(P->n_el, 0.0);
    if (delays)
        for (int k = 0; k < P->n_el; ++k) {
            if (!(std::fabs(delays[k]) <= 1.0)) return fail(FN_ERR_ARGUMENT, "delay offset %d must be finite and |d| <= 1 s", k);
            d[k] = delays[k];
        }
    HIP_CHECK(hipSetDevice(P->device), "hipSetDevice");
    // kernels of earlier calls on any stream may still read the delay offsets
    HIP_CHECK(hipDeviceSynchronize(), "hipDeviceSynchronize");
    HIP_CHECK(hipMemcpy(P->d_delay, d.data(), d.size() * sizeof(double), hipMemcpyHostToDevice), "delay offsets");
    P->h_delay = d;
    P->delays_even = std::equal(d.begin(), d.end(), d.rbegin());
    P->args.ctof = c_tof > 0 ? c_tof : P->args.c0;
    ++P->tof_serial;
    return P->shallow ? set_tof(P->shallow, c_tof, delays) : FN_OK;
}

int check_pw_fp32(const fn_plan *P, const char *what)
{
    if (!P) return fail(FN_ERR_ARGUMENT, "null plan");
    if (P->mode != 0) return fail(FN_ERR_UNSUPPORTED, "%s: plane-wave plans only", what);
    if (P->n_frames > 1) return fail(FN_ERR_UNSUPPORTED, "%s: single-frame plans only", what);
    if (P->n_el > 128) return fail(FN_ERR_UNSUPPORTED, "%s: at most 128 elements", what);
    if (P->nw) return fail(FN_ERR_UNSUPPORTED, "%s: normalizations.windowed is not differentiated", what);
    if (P->lbl) return fail(FN_ERR_UNSUPPORTED, "%s: line-scan plans are forward only", what);
    return FN_OK;
}

int execute_tangent(fn_plan *P, const void *d_rf, int dtype, float *d_image, float *d_dimage, float *d_w,
                    hipStream_t user)
{
    if (int st = check_pw_fp32(P, "tangent")) return st;
    if (!d_rf || !d_image || !d_dimage) return fail(FN_ERR_ARGUMENT, "null argument");
    if (dtype != FN_DTYPE_F32 && dtype != FN_DTYPE_F64) return fail(FN_ERR_RF_DATA, "RF data must be float32 or float64");
    HIP_CHECK(hipSetDevice(P->device), "hipSetDevice");
    hipStream_t s = user;  // NULL: the default stream
    if (int st = launch_spectra(P, d_rf, dtype, s)) return st;
    // groups of at most two transmit tiles keep the tangent accumulators in registers
    const int mt = std::min(P->MT_all, 2);
    const int groups = (P->MT_all + mt - 1) / mt;
    // plans whose forward runs the fp16 split contract the tangent on it too (11 angles, 384 x
    // 384, 542 bins: 14.7 ms in FP32, 9.7 split, 6.8 mirrored), with mirrored voxels where one tile holds every row (four tiles of both
    // accumulators would spill)
    const bool split_form = P->kprec == FN_PRECISION_FP16X3;
    const bool mirror = tangent_mirror(P);
    if (split_form) {
        if (int st = ensure_planes(P, mirror ? 2 * P->MT_all : groups * mt)) return st;
        if (int st = launch_lowp_planes(P, P->d_X, P->d_Xlp, P->d_xscale, P->d_bad, 1, P->MT_all, mirror ? 2 * P->MT_all : groups * mt,
                                        mirror ? P->n_el : 0, plane_delay(P, mirror), s))
            return st;
    }
    fnk::BeamArgs A = split_form ? forward_args(P) : P->args;
    if (!split_form) A.bad = nullptr;  // no planes in this call
    if (plane_delay(P, mirror)) A.delay = P->d_zeros;
    A.xlp_tiles = mirror ? 2 * P->MT_all : groups * mt;
    A.image = reinterpret_cast<float2 *>(d_image);
    A.dimage = d_dimage;
    A.weights = d_w;
    A.weights_tx = nullptr;
    A.tx_group = mt;
    // bin chunks: at least the plan's, and about 8192 workgroups (at most 8 chunks) when
    // the grid is smaller -- 11 angles, 384 x 384, 542 bins: 17.5 ms in one chunk,
    // 15.7-15.8 ms in 4 or 8
    const long tiles = ((mirror ? (long)((P->n_x + 1) / 2) * P->n_z : P->n_vox) + 63) / 64;
    int split = P->bin_split;
    if (tiles * groups * split < 8192)
        split = std::max(split, (int)std::min<long>({(8192 + tiles * groups - 1) / (tiles * groups), 8L,
                                                    (long)std::max(1, P->g.n_f / 8)}));
    const int chunk = (P->g.n_f + split - 1) / split;
    split = (P->g.n_f + chunk - 1) / chunk;
    A.bin_chunk = chunk;
    // partial images and tangents of the workgroups that share a voxel, summed in slot order
    A.n_slots = split * groups;
    A.slot_z = groups;
    A.partial = nullptr;
    if (A.n_slots > 1) {
        const size_t need = 2 * (size_t)A.n_slots * P->n_vox;
        if (need > P->ptan_cap) {
            if (P->d_ptan) HIP_CHECK(hipFree(P->d_ptan), "hipFree");
            P->d_ptan = nullptr;
            P->ptan_cap = 0;
            HIP_CHECK(hipMalloc(&P->d_ptan, need * sizeof(float2)), "tangent partial images");
            P->ptan_cap = need;
        }
        A.partial = P->d_ptan;
    }
    const size_t lds = (size_t)mt * P->KI * 64 * sizeof(float2);  // the split's planes are as large
    const dim3 grid((unsigned)tiles, (unsigned)split, (unsigned)groups);
    hipError_t e;
    if (split_form) {
        e = P->KI == 8    ? fnk::launch_beamform_tan_k8_p2(mt, P->wcr, mirror, grid, lds, s, A)
            : P->KI == 16 ? fnk::launch_beamform_tan_k16_p2(mt, P->wcr, mirror, grid, lds, s, A)
                          : fnk::launch_beamform_tan_k32_p2(mt, P->wcr, mirror, grid, lds, s, A);
    } else {
        const int wcr = wcr_general(P->wcr);
        e = P->KI == 8    ? fnk::launch_beamform_tan_k8(mt, wcr, grid, lds, s, A)
            : P->KI == 16 ? fnk::launch_beamform_tan_k16(mt, wcr, grid, lds, s, A)
                          : fnk::launch_beamform_tan_k32(mt, wcr, grid, lds, s, A);
    }
    if (e != hipSuccess) return hip_fail(e, "beamform tangent kernel");
    return finish_beam(P, A, s, reinterpret_cast<float2 *>(d_dimage));
}

// voxel contraction Z_n(k,a) = s sum_v y conj(T B) / w into P->d_Z
#ifndef FN_ADJ_BLOCKS
// target workgroups of the adjoint voxel contraction: about sixteen rounds of two blocks
// per CU (11 angles, 384 x 384, 542 bins: 10.2 ms at 2048, 9.8 at 4096, 9.6 at 8192,
// 10.8 at 1024; more ranges enlarge the partials the reduction reads, 0.5 GB there)
#define FN_ADJ_BLOCKS 8192L
#endif

int contract_adjoint(fn_plan *P, const float *d_y, hipStream_t s)
{
    const int n_f = P->g.n_f;
    const int n_chunks = (n_f + 3) / 4;  // bins per block of the contraction kernel (one per wave)
    if (!P->d_Z) {
        P->adj_at = (P->n_tx + 15) / 16;
        const long groups64 = (P->n_vox + 63) / 64;  // ranges are whole 64-voxel aperture blocks
        // FN_ADJ_BLOCKS workgroups (rounded down so the last round is not a short
        // tail), bounded by the voxel blocks
        long vr = FN_ADJ_BLOCKS / ((long)n_chunks * P->adj_at);
        vr = std::max(1L, std::min(vr, groups64));
        const long blocks_per_range = (groups64 + vr - 1) / vr;
        P->adj_vpr = blocks_per_range * 64;
        P->adj_vr = (int)((groups64 + blocks_per_range - 1) / blocks_per_range);
        const size_t p_floats = (size_t)P->adj_vr * n_f * P->adj_at * 2 * 128 * 16;
        HIP_CHECK(hipMalloc(&P->d_P, p_floats * sizeof(float)), "adjoint partials");
        HIP_CHECK(hipMalloc(&P->d_Z, (size_t)n_f * P->n_tx * P->n_el * sizeof(float2)), "adjoint contraction");
        HIP_CHECK(hipMalloc(&P->d_part, 1024 * sizeof(double)), "reduction partials");
        // phase words (128 + 16 n_at per voxel) followed by 4 doubles of aperture terms per voxel
        HIP_CHECK(hipMalloc(&P->d_qtab, (size_t)P->n_vox * (128 + 16 * P->adj_at + 8) * sizeof(uint32_t)),
                  "phase tables");
        // s / w_n(v) per bin and voxel, then the cotangent's units and flags per bin and 64 voxels, and a flag for all
        const size_t vsc_bytes = ((size_t)n_f * (P->n_vox + 2 * groups64) + 1) * sizeof(float);
        HIP_CHECK(hipMalloc(&P->d_vsc, vsc_bytes), "adjoint normalization");
        hipLaunchKernelGGL(fnk::fill_zero_kernel, dim3(1), dim3(256), 0, s, P->d_vsc + vsc_bytes / sizeof(float) - 1, 1L);
        HIP_CHECK(hipGetLastError(), "fill_zero_kernel");
    }
    fnk::AdjArgs S{};
    S.B = P->args;
    // the delay offsets where the tangent has them: a gradient's real parts dwarf its imaginary
    // ones, and cancel only between phases rounded alike (64 elements, 3 angles: d J / d delay
    // 2.9e-6 from 64 bits with the offsets in the tangent's planes and the adjoint's words)
    const double *delay = plane_delay(P, tangent_mirror(P));
    if (delay) S.B.delay = P->d_zeros;
    S.y = reinterpret_cast<const float2 *>(d_y);
    S.P = P->d_P;
    S.qrx = P->d_qtab;
    S.qtx = P->d_qtab + (size_t)P->n_vox * 128;
    S.vgeo = reinterpret_cast<const double *>(P->d_qtab + (size_t)P->n_vox * (128 + 16 * P->adj_at));
    S.vsc = P->d_vsc;
    S.units = P->d_vsc + (size_t)n_f * P->n_vox;
    S.flags = reinterpret_cast<const uint32_t *>(S.units + (size_t)n_f * ((P->n_vox + 63) / 64));
    S.rest = S.flags + (size_t)n_f * ((P->n_vox + 63) / 64);
    S.n_vr = P->adj_vr;
    S.vox_per_range = P->adj_vpr;
    S.n_at = P->adj_at;
    // bin quads fastest: the workgroups dispatched together share a voxel range, whose
    // phase-word tables then stay in L2
    const dim3 grid((unsigned)n_chunks, (unsigned)P->adj_vr, (unsigned)P->adj_at);
    // the phase tables depend on the geometry and the time of flight only: rebuilt
    // after set_tof, or when this call's stream is not the one that built them; the
    // normalization table on the geometry only: built once per stream
    const bool tables = P->adj_tab_serial != P->tof_serial || P->adj_tab_stream != s;
    const bool scale = !P->adj_sc_built || P->adj_sc_stream != s;
    hipError_t e = fnk::launch_adjoint(P->wcr, tables, scale, grid, s, S);
    if (e == hipSuccess && tables) {
        P->adj_tab_serial = P->tof_serial;
        P->adj_tab_stream = s;
    }
    if (e == hipSuccess && scale) {
        P->adj_sc_built = true;
        P->adj_sc_stream = s;
    }
    if (e != hipSuccess) return hip_fail(e, "adjoint_kernel");
    e = fnk::launch_adjoint_reduce(P->d_P, P->d_Z, P->adj_vr, n_f, P->adj_at, P->n_tx, P->n_el, delay,
                                   P->args.f_s / P->g.N, P->g.n_lb, const_cast<uint32_t *>(S.rest), s);
    if (e != hipSuccess) return hip_fail(e, "adjoint_reduce_kernel");
    return FN_OK;
}

int adjoint(fn_plan *P, const float *d_y, float *d_rf_adj, hipStream_t user)
{
    if (int st = check_pw_fp32(P, "adjoint")) return st;
    if (!d_y || !d_rf_adj) return fail(FN_ERR_ARGUMENT, "null argument");
    HIP_CHECK(hipSetDevice(P->device), "hipSetDevice");
    hipStream_t s = user;  // NULL: the default stream
    if (int st = contract_adjoint(P, d_y, s)) return st;
    hipError_t e = fnk::launch_adjoint_idft(P->d_Z, P->d_tw, d_rf_adj, P->n_t, P->n_tx * P->n_el, P->g.N, P->g.n_lb,
                                            P->g.n_f, s);
    if (e != hipSuccess) return hip_fail(e, "adjoint_idft_kernel");
    return FN_OK;
}

int vjp(fn_plan *P, const void *d_rf, int dtype, const float *d_g, const float *d_dimage, double *d_vjp_delay,
        double *d_vjp_c, hipStream_t user)
{
    if (int st = check_pw_fp32(P, "vjp")) return st;
    if (!d_rf || !d_g || !d_vjp_delay) return fail(FN_ERR_ARGUMENT, "null argument");
    if (dtype != FN_DTYPE_F32 && dtype != FN_DTYPE_F64) return fail(FN_ERR_RF_DATA, "RF data must be float32 or float64");
    HIP_CHECK(hipSetDevice(P->device), "hipSetDevice");
    hipStream_t s = user;  // NULL: the default stream
    if (int st = launch_spectra(P, d_rf, dtype, s)) return st;
    if (int st = contract_adjoint(P, d_g, s)) return st;
    const double w_unit = 2.0 * 3.14159265358979323846 * P->args.f_s / P->g.N;
    hipError_t e = fnk::launch_vjp_delay(P->d_X, P->d_Z, d_vjp_delay, P->g.n_f, P->n_tx, P->n_el, P->MT_all, P->KI,
                                         P->g.n_lb, w_unit, s);
    if (e != hipSuccess) return hip_fail(e, "vjp_delay_kernel");
    if (d_dimage && d_vjp_c) {
        const int n_part = (int)std::min<long>(1024, (P->n_vox + 255) / 256);
        e = fnk::launch_dot_re(reinterpret_cast<const float2 *>(d_g), reinterpret_cast<const float2 *>(d_dimage),
                               P->n_vox, P->d_part, n_part, d_vjp_c, s);
        if (e != hipSuccess) return hip_fail(e, "dot_re_kernel");
    }
    return FN_OK;
}

// a bin of voxel (ix, iz) with non-empty aperture(s): the FP64 bounds of
// make_aperture (das_pw.m:399-414, das_sa.m:384-414)
bool bin_valid(const fn_plan *P, int ix, int iz, int b)
{
    const fnk::BeamArgs &A = P->args;
    const double x = P->h_px[ix], z = P->h_pz[iz];
    const double xp = x / A.pitch, zp = z / (2.0 * A.pitch);
    auto ok = [&](double F) {
        const double hp = zp / F;
        const double ua = A.M + (xp - hp), ub = A.M + (xp + hp);
        return std::fmax(std::ceil(ua), 0.0) <= std::fmin(std::floor(ub), (double)(A.n_el - 1));
    };
    double Fr = P->h_Frx[b];
    if (A.clamp) Fr = std::fmin(Fr, P->h_sqf[b] * std::sqrt(z / (2.88 * A.c0)));  // das_pw.m:374-377
    bool v = ok(Fr);
    if (P->mode == 1) v = v && ok(P->h_Ftx[b]);
    return v;
}

// focused RF signal of the last voxel the CPU loop processes (das_pw.m:477-481,
// das_sa.m:501-505) from the spectra of the plan's last execute: complex [N_dft]
int focused_signal(fn_plan *P, float *d_signal, hipStream_t s)
{
    if (!P || !d_signal) return fail(FN_ERR_ARGUMENT, "null argument");
    if (P->n_frames > 1) return fail(FN_ERR_UNSUPPORTED, "focused signal: single-frame plans only");
    if (P->lbl) return fail(FN_ERR_UNSUPPORTED, "focused signal: not available for line-scan plans");
    if (P->n_el > 128) return fail(FN_ERR_UNSUPPORTED, "focused signal: at most 128 elements");
    if (!P->executed) return fail(FN_ERR_ARGUMENT, "focused signal: execute the plan first");
    int vx = -1, vz = -1;  // last lateral position with a valid bin, its last such depth
    for (int ix = P->n_x - 1; ix >= 0 && vx < 0; --ix)
        for (int iz = P->n_z - 1; iz >= 0 && vx < 0; --iz)
            for (int b = 0; b < P->g.n_f; ++b)
                if (bin_valid(P, ix, iz, b)) {
                    vx = ix;
                    vz = iz;
                    break;
                }
    if (vx < 0) return fail(FN_ERR_ARGUMENT, "focused signal: no voxel has a non-empty aperture");
    HIP_CHECK(hipSetDevice(P->device), "hipSetDevice");
    if (!P->d_sigF) HIP_CHECK(hipMalloc(&P->d_sigF, (size_t)P->g.n_f * sizeof(float2)), "signal spectrum");
    hipError_t e = fnk::launch_focused_signal(P->args, P->mode, P->wcr, P->wct, P->MT_all, P->KI, P->nw, vx, vz,
                                              P->d_sigF, P->d_tw, reinterpret_cast<float2 *>(d_signal), s);
    if (e != hipSuccess) return hip_fail(e, "focused_spectrum_kernel");
    return FN_OK;
}

// run-time report of the last one-shot call of this thread with verbosity >= 1:
// the device, the launch parameters, the memory in use and per-stage times (the
// sections gpu_bf_das_pw_rf.cu:664-689, 875-903, 1128-1144 print); the gateways
// print it after their own status section
thread_local std::string t_report;

void report_line(std::string &r, const char *fmt, ...)
{
    char buf[256];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    r += buf;
}

const char *kRule = " --------------------------------------------------------------------------------\n";

void report_bytes(std::string &r, const char *what, double bytes, double total)
{
    report_line(r, "     %-31s: %12.2f KiByte (%6.2f %%)\n", what, bytes / 1024.0, total > 0 ? 100.0 * bytes / total : 0.0);
}

void report_time(std::string &r, const char *what, double ms, double total)
{
    report_line(r, "     %-34s: %10.3f ms (%6.2f %%)\n", what, ms, total > 0 ? 100.0 * ms / total : 0.0);
}

void compose_report(const fn_plan *P, size_t rf_bytes, size_t img_bytes, size_t w_bytes, int n_w, const float *ms)
{
    std::string &r = t_report;
    r.clear();
    hipDeviceProp_t prop{};
    int count = 0, drv = 0, rt = 0;
    size_t mem_free = 0, mem_total = 0;
    hipGetDeviceProperties(&prop, P->device);
    hipGetDeviceCount(&count);
    hipDriverGetVersion(&drv);
    hipRuntimeGetVersion(&rt);
    hipMemGetInfo(&mem_free, &mem_total);
    static const char *kPrec[] = {"fp32", "bf16x3", "fp16x3", "fp16"};
    static const char *kWin[] = {"range", "linear", "cosine", "cosine, full array", "cosine, cut at the aperture"};
    r += kRule;
    report_line(r, " Selected device %d of %d: %s (%s)\n", P->device, count, prop.name, prop.gcnArchName);
    r += kRule;
    report_line(r, "  %-20s: %-18d %-22s: %d\n", "compute units", prop.multiProcessorCount, "wavefront size", prop.warpSize);
    report_line(r, "  %-20s: %-11.2f MiByte %-22s: %.2f KiByte\n", "total global memory",
                (double)prop.totalGlobalMem / 1048576.0, "LDS per compute unit",
                (double)prop.maxSharedMemoryPerMultiProcessor / 1024.0);
    report_line(r, "  %-20s: %-18d %-22s: %d.%d / %d.%d\n", "registers per block", prop.regsPerBlock,
                "driver / runtime", drv / 10000000, (drv / 100000) % 100, rt / 10000000, (rt / 100000) % 100);
    std::string form = kPrec[P->precision];
    if (P->interp_M) form += ", interpolated";
    else if (P->lbl ? P->line_mirror && P->delays_even : use_mirror(P)) form += P->lbl ? ", mirrored columns" : ", mirrored voxels";
    report_line(r, "  %-20s: %-22s %-22s: %s\n", "contraction", form.c_str(), "mode",
                P->lbl         ? "line scan"
                : P->mode == 1 ? "synthetic aperture"
                : P->n_frames > 1 ? "plane waves, ensemble" : "plane waves");
    r += kRule;
    r += " launch parameters\n";
    r += kRule;
    const long tiles = P->interp_M ? (P->n_vox + 63) / 64 : beam_tiles(P);
    if (P->interp_M) {
        report_line(r, "  %-20s: %-6ld x 64 voxels %-11s %-22s: %d of up to 32 angles\n", "voxel tiles", tiles, "",
                    "transmit groups", beam_slots(P));
        report_line(r, "  %-20s: %-18d %-22s: %d of %d\n", "samples per channel", P->interp_M, "clamped depths (summed)",
                    P->shallow ? P->shallow->n_z : 0, P->n_z);
        report_line(r, "  %-20s: %-18ld %-22s: %s\n", "workgroups", tiles * beam_slots(P), "receive window class",
                    kWin[wcr_general(P->wcr)]);
    } else if (P->lbl) {
        const int cols = P->line_mirror && P->delays_even ? (P->n_x + 1) / 2 : P->n_x;
        report_line(r, "  %-20s: %-6ld x 64 depths %-11s %-22s: %d of %d lines\n", "depth tiles", tiles, "", "column groups", cols,
                    P->n_x);
        report_line(r, "  %-20s: %-3d of %-5d bins\n", "bin chunks", P->bin_split, P->args.bin_chunk);
        report_line(r, "  %-20s: %-18ld %-22s: %s\n", "workgroups", tiles * P->bin_split * cols, "receive window class",
                    kWin[P->wcr]);
    } else {
        report_line(r, "  %-20s: %-6ld x 64 voxels %-11s %-22s: %d x %d of 16 rows\n", "voxel tiles", tiles, "",
                    "transmit groups x tiles", P->n_groups, P->MT_tmpl);
        report_line(r, "  %-20s: %-3d of %-5d bins %-8s %-22s: %d (4 elements each)\n", "bin chunks", P->bin_split,
                    P->args.bin_chunk, "", "element steps / lane", P->KI);
        report_line(r, "  %-20s: %-18ld %-22s: %s\n", "workgroups", tiles * P->bin_split * P->n_groups,
                    "receive window class", kWin[P->wcr]);
    }
    const double b_pos = 8.0 * (P->n_x + P->n_z);
    const double b_tab = 8.0 * P->g.n_f * (P->d_Ftx ? 3 : 2) + (P->d_txp ? 24.0 * P->n_tx : 0.0) + 8.0 * P->g.N +
                         8.0 * P->n_el;
    const double b_spec = (double)workspace_bytes(P) + (P->d_xscale ? 4.0 * P->g.n_f : 0.0);
    const double b_part = 8.0 * (double)P->pimg_cap;
    const double b_tot = b_pos + b_tab + rf_bytes + b_spec + b_part + img_bytes + (double)w_bytes * n_w;
    r += kRule;
    report_line(r, " memory consumption (available global memory: %.2f MiByte (%.2f %%))\n", mem_free / 1048576.0,
                mem_total ? 100.0 * mem_free / mem_total : 0.0);
    r += kRule;
    report_bytes(r, "voxel positions", b_pos, b_tot);
    report_bytes(r, "F-numbers, steering, twiddles", b_tab, b_tot);
    report_bytes(r, "RF signals", (double)rf_bytes, b_tot);
    report_bytes(r, "band spectra (workspace)", b_spec, b_tot);
    if (b_part > 0) report_bytes(r, "partial images", b_part, b_tot);
    report_bytes(r, "DAS image", (double)img_bytes, b_tot);
    if (n_w) report_bytes(r, "weights", (double)w_bytes * n_w, b_tot);
    report_line(r, "     %-31s  %s\n", "-------------------------------", "----------------------------");
    report_bytes(r, "total", b_tot, b_tot);
    const double t_tot = ms[0] + ms[1] + ms[2] + ms[3];
    r += kRule;
    r += " performance statistics:\n";
    r += kRule;
    report_time(r, "memory transfer: host to device", ms[0], t_tot);
    report_time(r, "band-limited DFT (spectra)", ms[1], t_tot);
    report_time(r, "beamforming kernel", ms[2], t_tot);
    report_time(r, "memory transfer: device to host", ms[3], t_tot);
    report_line(r, "     %-34s  %s\n", "----------------------------------", "------------------------");
    report_time(r, "total", t_tot, t_tot);
}

// one-shot: H2D, execute, D2H (gpu_bf_das_pw_rf.cu:730-1122); with verbosity >= 1
// the stages are timed with HIP events and reported.  *unmirror: the image is not to be used, a
// plan of Mirror::no is
int one_shot(fn_plan *P, const void *rf, int dtype, float *image, float *w0, float *w1, bool *unmirror = nullptr)
{
    const size_t rf_bytes = (size_t)P->n_t * P->n_el * P->n_tx * dtype_size(dtype);
    const size_t img_bytes = (size_t)P->n_vox * 2 * sizeof(float) * P->n_frames;
    const size_t w_bytes = (size_t)P->n_vox * sizeof(float);
    const bool rep = P->verbosity > 0;
    void *d_rf = nullptr;
    float *d_img = nullptr, *d_w0 = nullptr, *d_w1 = nullptr;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    int s = FN_OK;
    hipError_t e = hipMalloc(&d_rf, rf_bytes);
    if (e == hipSuccess) e = hipMalloc(&d_img, img_bytes);
    if (e == hipSuccess && w0) e = hipMalloc(&d_w0, w_bytes);
    if (e == hipSuccess && w1) e = hipMalloc(&d_w1, w_bytes);
    for (int i = 0; i < 4 && rep && e == hipSuccess; ++i) e = hipEventCreate(&ev[i]);
    if (rep) P->profiling = 1;
    if (e == hipSuccess && rep) e = hipEventRecord(ev[0], P->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(d_rf, rf, rf_bytes, hipMemcpyHostToDevice, P->stream);
    if (e == hipSuccess && rep) e = hipEventRecord(ev[1], P->stream);
    if (e != hipSuccess) s = hip_fail(e, "one-shot buffers");
    if (!s) s = execute(P, d_rf, dtype, d_img, d_w0, d_w1, P->stream);
    if (!s) {
        e = rep ? hipEventRecord(ev[2], P->stream) : hipSuccess;
        if (e == hipSuccess) e = hipMemcpyAsync(image, d_img, img_bytes, hipMemcpyDeviceToHost, P->stream);
        if (e == hipSuccess && w0) e = hipMemcpyAsync(w0, d_w0, w_bytes, hipMemcpyDeviceToHost, P->stream);
        if (e == hipSuccess && w1) e = hipMemcpyAsync(w1, d_w1, w_bytes, hipMemcpyDeviceToHost, P->stream);
        if (e == hipSuccess && rep) e = hipEventRecord(ev[3], P->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(P->stream);
        if (e != hipSuccess) s = hip_fail(e, "one-shot results");
    }
    if (!s && rep) {
        float ms[4] = {0.f, 0.f, 0.f, 0.f};
        hipEventElapsedTime(&ms[0], ev[0], ev[1]);
        hipEventElapsedTime(&ms[3], ev[2], ev[3]);
        collect_profile(P);
        ms[1] = (float)P->spec_ms;
        ms[2] = (float)P->beam_ms;
        compose_report(P, rf_bytes, img_bytes, w_bytes, (w0 ? 1 : 0) + (w1 ? 1 : 0), ms);
    }
    for (auto &x : ev)
        if (x) hipEventDestroy(x);
    hipFree(d_rf); hipFree(d_img); hipFree(d_w0); hipFree(d_w1);
    if (unmirror) *unmirror = !s && std::memcmp(image, &fnk::TIE_MARK, sizeof(fnk::TIE_MARK)) == 0;
    return s;
}

}  // namespace

// ---- the no-allocation entry point (fn_das_pw_noalloc) ---------------------
// Every device table and the spectra workspace of one call live in `scratch`, a
// file-scope array of this code object: each device holds its own copy at its
// own address, which host code obtains once per device with hipGetSymbolAddress
// and then uses exclusively (the array's name in host code is only a stand-in).
// Calls on one device share the array and race if they overlap.
namespace {
constexpr size_t kScratchBytes = ((size_t)32 << 20) + ((size_t)64 << 10);  // (the masks take 32 KiB at most)
constexpr int kMaxDevices = 64;
}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace fnk {
// host arrays reach the scratch as kernel arguments (captured at launch, so the
// caller's arrays are free to change once the call returns): 448 doubles a launch
struct UploadChunk {
    double v[448];
};

__global__ void upload_chunk_kernel(double *dst, UploadChunk c, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) dst[i] = c.v[i];
}

// the tables pw_plan computes on the host, computed here from the raw inputs:
// twiddles e^{+j 2 pi m / N}, sqrt(f_n) per bin, the steering rows
// (das_pw.m:323-327: e_x = -sin, e_z = cos, x_ref = sign(e_x) x_0; or the
// virtual sources (x_vs, z_vs, |r_vs|)) and zero delay offsets
__global__ void noalloc_tables_kernel(float2 *tw, int N, double *sqf, int n_f, int n_lb, double f_s, double *txp,
                                      const double *raw_tx, int n_tx, int virt, double M, double pitch, double *delay,
                                      int n_el)
{
    const int n = max(max(N, n_f), max(n_tx, n_el));
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if (i < N) {
            double sn, cs;
            sincospi(2.0 * (double)i / (double)N, &sn, &cs);
            tw[i] = make_float2((float)cs, (float)sn);
        }
        if (i < n_f) sqf[i] = sqrt(f_s * (double)(n_lb + i) / N);
        if (i < n_tx) {
            if (virt) {
                const double xv = raw_tx[2 * i], zv = raw_tx[2 * i + 1];
                txp[3 * i] = xv;
                txp[3 * i + 1] = zv;
                txp[3 * i + 2] = sqrt(xv * xv + zv * zv);
            } else {
                const double th = raw_tx[i];
                const double ex = -sin(th), ez = cos(th);
                const double sg = (ex > 0) - (ex < 0);
                txp[3 * i] = ex;
                txp[3 * i + 1] = ez;
                txp[3 * i + 2] = sg * ((0 - M) * pitch);
            }
        }
        if (i < n_el) delay[i] = 0.0;
    }
}
}  // namespace fnk

namespace {

std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};

// the device address of `scratch` on `device`, looked up on the first call on that
// device (which is current: select_device ran) and kept
int scratch_on_device(int device, unsigned char **out)
{
    if (device < 0 || device >= kMaxDevices) return fail(FN_ERR_DEVICE, "device index %d beyond %d", device, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        void *ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (!ptr) return fail(FN_ERR_HIP, "hipGetSymbolAddress(scratch) returned a null address");
        g_scratch_ptr[device] = ptr;
    }
    *out = static_cast<unsigned char *>(g_scratch_ptr[device]);
    return FN_OK;
}

int upload_chunked(double *dst, const double *src, long n, hipStream_t s)
{
    fnk::UploadChunk c;
    for (long i0 = 0; i0 < n; i0 += 448) {
        const int m = (int)std::min<long>(448, n - i0);
        std::memcpy(c.v, src + i0, (size_t)m * sizeof(double));
        hipLaunchKernelGGL(fnk::upload_chunk_kernel, dim3(1), dim3(256), 0, s, dst + i0, c, m);
        HIP_CHECK(hipGetLastError(), "upload_chunk_kernel");
    }
    return FN_OK;
}

int das_pw_noalloc(const fn_pw_params *p, const void *d_rf, int dtype, float *d_image, float *d_w, hipStream_t s)
{
    fnh::Grid g;
    int st = fnh::validate_pw(p, &g);
    if (st) return st;
    if (!d_rf) return fail(FN_ERR_RF_DATA, "RF data missing");
    if (!d_image) return fail(FN_ERR_ARGUMENT, "image buffer missing");
    if (dtype != FN_DTYPE_F32 && dtype != FN_DTYPE_F64) return fail(FN_ERR_RF_DATA, "RF data must be float32 or float64");
    if (p->n_frames > 1) return fail(FN_ERR_UNSUPPORTED, "fn_das_pw_noalloc: one frame per call (use a plan for ensembles)");
    if (p->line_scan) return fail(FN_ERR_UNSUPPORTED, "fn_das_pw_noalloc: line scans need a plan");
    if (p->normalization == FN_NORMALIZATION_WINDOWED && p->semantics == FN_SEMANTICS_CPU)
        return fail(FN_ERR_UNSUPPORTED, "fn_das_pw_noalloc: normalizations.windowed (CPU semantics) needs a plan");
    // the configuration of fn_plan_pw_create on a plan held on the stack: the same
    // tiling and kernels, with every device pointer in the scratch
    fn_plan P;
    Common c{};
    if ((st = configure_pw(&P, p, &c))) return st;
    const int n_f = g.n_f, n_tx = c.n_tx, raw_per_tx = p->virtual_sources ? 2 : 1;
    Carve cv;
    size_t o_X = 0, o_Xlp = 0, o_xs = 0, o_px = 0, o_pz = 0, o_F = 0, o_sqf = 0, o_raw = 0, o_txp = 0, o_tw = 0, o_dl = 0,
           o_pi = 0, o_bad = 0;
    int slots = 1;
    // one voxel a lane: whether the grid's apertures mirror is only known after a look at them on
    // the device, which this call may not wait for.  A call whose planes do not fit beside its
    // spectra leaves out their zero tiles, then an FP32 call runs the FP32 kernels.
    for (const Planes room : {Planes::own, Planes::bare, Planes::none}) {
        if (room == Planes::none && p->precision != FN_PRECISION_FP32) break;
        if ((st = configure_common(&P, c, g, p->f_number_values, false, room))) return st;
        cv = Carve{};
        o_X = cv.take(P.x_bytes);
        o_Xlp = cv.take(P.xlp_bytes);
        o_xs = cv.take(P.kprec != FN_PRECISION_FP32 ? (size_t)n_f * sizeof(float) : 0);
        o_bad = cv.take(P.kprec != FN_PRECISION_FP32 ? bad_bytes(n_f, 1, P.KI) : 0);
        o_px = cv.take((size_t)c.n_x * sizeof(double));
        o_pz = cv.take((size_t)c.n_z * sizeof(double));
        o_F = cv.take((size_t)n_f * sizeof(double));
        o_sqf = cv.take((size_t)n_f * sizeof(double));
        o_raw = cv.take((size_t)n_tx * raw_per_tx * sizeof(double));
        o_txp = cv.take((size_t)n_tx * 3 * sizeof(double));
        o_tw = cv.take((size_t)g.N * sizeof(float2));
        o_dl = cv.take((size_t)c.n_el * sizeof(double));
        slots = beam_slots(&P);
        o_pi = cv.take(slots > 1 ? (size_t)slots * P.n_vox * sizeof(float2) : 0);
        if (cv.used <= kScratchBytes) break;
    }
    if (cv.used > kScratchBytes)
        return fail(FN_ERR_UNSUPPORTED,
                    "fn_das_pw_noalloc: this call needs %zu bytes of device scratch, the entry point holds %zu "
                    "(spectra workspace %zu bytes); use a plan",
                    cv.used, kScratchBytes, P.x_bytes + P.xlp_bytes);
    use_cos_all(&P);
    if ((st = select_device(p->index_gpu))) return st;
    unsigned char *base = nullptr;
    if ((st = scratch_on_device(p->index_gpu, &base))) return st;
    P.d_X = reinterpret_cast<float2 *>(base + o_X);
    P.d_Xlp = P.xlp_bytes ? base + o_Xlp : nullptr;
    P.d_xscale = P.xlp_bytes ? reinterpret_cast<float *>(base + o_xs) : nullptr;
    P.d_bad = P.xlp_bytes ? reinterpret_cast<uint32_t *>(base + o_bad) : nullptr;
    P.args.bad_rows = 1;
    P.args.bad_words = bad_words(P.KI);
    P.d_px = reinterpret_cast<double *>(base + o_px);
    P.d_pz = reinterpret_cast<double *>(base + o_pz);
    P.d_Frx = reinterpret_cast<double *>(base + o_F);
    P.d_sqf = reinterpret_cast<double *>(base + o_sqf);
    P.d_txp = reinterpret_cast<double *>(base + o_txp);
    P.d_tw = reinterpret_cast<float2 *>(base + o_tw);
    P.d_delay = reinterpret_cast<double *>(base + o_dl);
    P.d_pimg = slots > 1 ? reinterpret_cast<float2 *>(base + o_pi) : nullptr;
    double *raw = reinterpret_cast<double *>(base + o_raw);
    if ((st = upload_chunked(P.d_px, p->positions_x, c.n_x, s))) return st;
    if ((st = upload_chunked(P.d_pz, p->positions_z, c.n_z, s))) return st;
    if ((st = upload_chunked(P.d_Frx, p->f_number_values, n_f, s))) return st;
    if ((st = upload_chunked(raw, p->virtual_sources ? p->virtual_sources : p->steering_angles, (long)n_tx * raw_per_tx,
                             s)))
        return st;
    const int n_tab = std::max(std::max(g.N, n_f), std::max(n_tx, c.n_el));
    hipLaunchKernelGGL(fnk::noalloc_tables_kernel, dim3((unsigned)((n_tab + 255) / 256)), dim3(256), 0, s, P.d_tw,
                       g.N, P.d_sqf, n_f, g.n_lb, c.f_s, P.d_txp, raw, n_tx, p->virtual_sources ? 1 : 0,
                       (p->n_elements - 1) / 2.0, p->element_pitch, P.d_delay, c.n_el);
    HIP_CHECK(hipGetLastError(), "noalloc_tables_kernel");
    fnk::BeamArgs &A = P.args;
    A.X = P.d_X;
    A.Xlp = P.d_Xlp;
    A.xscale = P.d_xscale;
    A.bad = P.d_bad;
    A.px = P.d_px; A.pz = P.d_pz; A.Frx = P.d_Frx; A.Ftx = nullptr; A.txp = P.d_txp; A.sqrt_f = P.d_sqf;
    A.delay = P.d_delay;
    // spectra (every operand slot of the workspace is written, padding as zeros) and
    // the 16-bit planes, the beamformer, and the sum of the partial images
    if ((st = prepare(&P, d_rf, dtype, d_image, s))) return st;
    const fnk::BeamArgs B = beam_args(&P, d_image, d_w, nullptr);
    hipError_t e = launch_beam(&P, dim3((unsigned)beam_tiles(&P), (unsigned)P.bin_split, (unsigned)P.n_groups), B, s);
    if (e != hipSuccess) return hip_fail(e, "beamform_kernel");
    return finish_beam(&P, B, s);
}

}  // namespace

extern "C" {

int32_t fn_das_pw_noalloc(const fn_pw_params *p, const void *d_rf, int32_t rf_dtype, float *d_image, float *d_weights,
                          void *stream)
{
    fnh::clear_error();
    return das_pw_noalloc(p, d_rf, rf_dtype, d_image, d_weights, static_cast<hipStream_t>(stream));
}

int32_t fn_device_count(int32_t *count)
{
    if (!count) return fail(FN_ERR_ARGUMENT, "null argument");
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    *count = (e == hipSuccess) ? c : 0;
    return FN_OK;
}

int32_t fn_plan_pw_create(const fn_pw_params *p, fn_plan **plan)
{
    if (!plan) return fail(FN_ERR_ARGUMENT, "null plan pointer");
    *plan = nullptr;
    return pw_plan(p, plan);
}

int32_t fn_plan_sa_create(const fn_sa_params *p, fn_plan **plan)
{
    if (!plan) return fail(FN_ERR_ARGUMENT, "null plan pointer");
    *plan = nullptr;
    return sa_plan(p, plan);
}

int32_t fn_plan_info_get(const fn_plan *P, fn_plan_info *info)
{
    if (!P || !info) return fail(FN_ERR_ARGUMENT, "null argument");
    info->N_dft = P->g.N;
    info->n_lb = P->g.n_lb;
    info->n_ub = P->g.n_ub;
    info->n_f = P->g.n_f;
    info->n_tx = P->n_tx;
    info->n_voxels = P->n_vox;
    info->workspace_bytes = (int64_t)workspace_bytes(P);
    info->flops_per_frame = P->flops;
    std::call_once(P->useful_once, [P] { P->useful_flops = 8.0 * useful_macs(P); });
    info->useful_flops_per_frame = P->useful_flops;
    info->tile_voxels = 64;
    info->bin_split = P->bin_split;
    info->m_tiles = P->MT_tmpl;
    info->k_steps = P->KI;
    return FN_OK;
}

int32_t fn_plan_execute(fn_plan *P, const void *d_rf, int32_t dtype, float *d_image, float *d_w, float *d_w_rx,
                        void *stream)
{
    fnh::clear_error();
    return execute(P, d_rf, dtype, d_image, d_w, d_w_rx, reinterpret_cast<hipStream_t>(stream));
}

int32_t fn_plan_autotune(fn_plan *P, const void *d_rf, int32_t dtype, float *d_image, int32_t repetitions,
                         fn_tune_result *result, void *stream)
{
    fnh::clear_error();
    return autotune(P, d_rf, dtype, d_image, repetitions, result, reinterpret_cast<hipStream_t>(stream));
}

int32_t fn_plan_set_tiling(fn_plan *P, int32_t m_tiles, int32_t bin_split)
{
    fnh::clear_error();
    return set_tiling(P, m_tiles, bin_split);
}

int32_t fn_plan_set_tof(fn_plan *P, double c_tof, const double *delay_offsets)
{
    fnh::clear_error();
    return set_tof(P, c_tof, delay_offsets);
}

int32_t fn_plan_execute_tangent(fn_plan *P, const void *d_rf, int32_t dtype, float *d_image, float *d_dimage_dc,
                                float *d_w, void *stream)
{
    fnh::clear_error();
    return execute_tangent(P, d_rf, dtype, d_image, d_dimage_dc, d_w, reinterpret_cast<hipStream_t>(stream));
}

int32_t fn_plan_focused_signal(fn_plan *P, float *d_signal, void *stream)
{
    fnh::clear_error();
    return focused_signal(P, d_signal, reinterpret_cast<hipStream_t>(stream));
}

int32_t fn_plan_adjoint(fn_plan *P, const float *d_y, float *d_rf_adj, void *stream)
{
    fnh::clear_error();
    return adjoint(P, d_y, d_rf_adj, reinterpret_cast<hipStream_t>(stream));
}

int32_t fn_plan_vjp(fn_plan *P, const void *d_rf, int32_t dtype, const float *d_g, const float *d_dimage_dc,
                    double *d_vjp_delay, double *d_vjp_c, void *stream)
{
    fnh::clear_error();
    return vjp(P, d_rf, dtype, d_g, d_dimage_dc, d_vjp_delay, d_vjp_c, reinterpret_cast<hipStream_t>(stream));
}

int32_t fn_plan_set_profiling(fn_plan *P, int32_t enable)
{
    if (!P) return fail(FN_ERR_ARGUMENT, "null plan");
    P->profiling = enable ? 1 : 0;
    return FN_OK;
}

int32_t fn_plan_get_profile(fn_plan *P, double *spectra_ms, double *beamform_ms, int32_t *n_runs)
{
    if (!P) return fail(FN_ERR_ARGUMENT, "null plan");
    int s = collect_profile(P);
    if (s) return s;
    if (spectra_ms) *spectra_ms = P->spec_ms;
    if (beamform_ms) *beamform_ms = P->beam_ms;
    if (n_runs) *n_runs = P->runs;
    P->spec_ms = P->beam_ms = 0.0;
    P->runs = 0;
    return FN_OK;
}

int32_t fn_plan_destroy(fn_plan *P)
{
    if (P) {
        hipSetDevice(P->device);
        hipStreamSynchronize(P->stream);
    }
    destroy(P);
    return FN_OK;
}

const char *fn_last_report(void) { return t_report.c_str(); }

int32_t fn_das_pw(const fn_pw_params *p, const void *data_rf, int32_t rf_dtype, float *image, float *weights)
{
    fnh::clear_error();
    t_report.clear();
    if (!data_rf) return fail(FN_ERR_RF_DATA, "RF data missing");
    if (!image) return fail(FN_ERR_ARGUMENT, "image buffer missing");
    if (rf_dtype != FN_DTYPE_F32 && rf_dtype != FN_DTYPE_F64) return fail(FN_ERR_RF_DATA, "RF data must be float32 or float64");
    fn_plan *P = nullptr;
    int s = pw_plan(p, &P, nullptr, Mirror::later);
    if (s) return s;
    bool unmirror = false;
    s = one_shot(P, data_rf, rf_dtype, image, weights, nullptr, &unmirror);
    destroy(P);
    if (s || !unmirror) return s;
    if ((s = pw_plan(p, &P, nullptr, Mirror::no))) return s;
    s = one_shot(P, data_rf, rf_dtype, image, weights, nullptr);
    destroy(P);
    return s;
}

int32_t fn_das_pw_adjoint(const fn_pw_params *p, double c_tof, const double *delay_offsets, const float *image_y,
                          float *rf_adj)
{
    fnh::clear_error();
    if (!image_y || !rf_adj) return fail(FN_ERR_ARGUMENT, "image and output buffers are required");
    fn_plan *P = nullptr;
    int s = pw_plan(p, &P);
    if (s) return s;
    s = set_tof(P, c_tof, delay_offsets);
    const size_t img_bytes = (size_t)P->n_vox * 2 * sizeof(float);
    const size_t rf_bytes = (size_t)P->n_t * P->n_el * P->n_tx * sizeof(float);
    float *d_y = nullptr, *d_rf = nullptr;
    if (!s) {
        hipError_t e = hipMalloc(&d_y, img_bytes);
        if (e == hipSuccess) e = hipMalloc(&d_rf, rf_bytes);
        if (e == hipSuccess) e = hipMemcpyAsync(d_y, image_y, img_bytes, hipMemcpyHostToDevice, P->stream);
        if (e != hipSuccess) s = hip_fail(e, "adjoint buffers");
    }
    if (!s) s = adjoint(P, d_y, d_rf, P->stream);
    if (!s) {
        hipError_t e = hipMemcpyAsync(rf_adj, d_rf, rf_bytes, hipMemcpyDeviceToHost, P->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(P->stream);
        if (e != hipSuccess) s = hip_fail(e, "adjoint result");
    }
    hipFree(d_y);
    hipFree(d_rf);
    destroy(P);
    return s;
}

int32_t fn_das_sa(const fn_sa_params *p, const void *data_rf, int32_t rf_dtype, float *image, float *weights_tx,
                  float *weights_rx)
{
    fnh::clear_error();
    t_report.clear();
    if (!data_rf) return fail(FN_ERR_RF_DATA, "RF data missing");
    if (!image) return fail(FN_ERR_ARGUMENT, "image buffer missing");
    if (rf_dtype != FN_DTYPE_F32 && rf_dtype != FN_DTYPE_F64) return fail(FN_ERR_RF_DATA, "RF data must be float32 or float64");
    fn_plan *P = nullptr;
    int s = sa_plan(p, &P);
    if (s) return s;
    s = one_shot(P, data_rf, rf_dtype, image, weights_tx, weights_rx);
    destroy(P);
    return s;
}

// ---- batches: many plans captured into one graph ----------------------

// plans of one kernel class (mode, element steps, transmit tiles, window classes,
// precision) beamformed by one persistent launch over their work items
struct BatchClass {
    std::vector<int> plans;
    fnk::BeamArgs *d_jobs = nullptr;  // one BeamArgs per plan (its buffers)
    int4 *d_items = nullptr;          // (job, voxel tile, bin chunk, transmit group), longest chunks first
    int *d_counter = nullptr;
    int n_items = 0, grid = 0;
};

// Row stack: plane-wave plans of a batch that differ only in their transmit rows
// (steering angles) and RF share every receive-side quantity -- voxel grid,
// frequency grid, F-numbers, window, normalization, element geometry and delays.
// Their rows are stacked into one operand (16 rows per matrix-core tile, a plan's
// rows need not start a tile) and beamformed by one ensemble launch whose epilogue
// adds every row to its own plan's image.  The apodization x phase values, one per
// (voxel, bin, element) generated on the vector ALUs, then serve all stacked rows
// of a transmit group (up to 64) instead of the few rows of one plan.
struct RowStack {
    std::vector<int> plans;  // members (batch indices), stacked in this order
    std::vector<int> row0;   // first stacked row of each member
    int rows = 0, MT_all = 0, MT_tmpl = 0, n_groups = 0, bin_split = 1, chunk = 0;
    size_t lds_beam = 0;
    float2 *d_X = nullptr;
    void *d_Xlp = nullptr;
    float *d_xscale = nullptr, *d_rowscale = nullptr;
    uint32_t *d_bad = nullptr;
    double *d_txp = nullptr;
    int *d_row_frame = nullptr;
    float2 **d_frame_image = nullptr;
};

struct fn_batch {
    std::vector<fn_plan *> plans;
    int device = 0;
    int persistent = 0;                // plans sharing a kernel class run as one persistent launch
    int stacking = 1;                  // row stacks of plans that share their receive side
    std::vector<RowStack> stacks;
    std::vector<BatchClass> classes;
    std::vector<int> singles;          // plans launched on their own
    hipStream_t pstream = nullptr;     // stream of the persistent launches inside the capture
    std::vector<hipStream_t> streams;  // forked worker streams (default priority)
    hipStream_t capture = nullptr;
    std::vector<hipEvent_t> joins;
    hipEvent_t fork = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<const void *> rf;
    std::vector<int32_t> dtypes;
    std::vector<float *> images;
    std::vector<std::pair<long, long>> serials;  // every plan's tof_serial and tiling_serial when the graph was captured
    int captures = 0;
    int64_t n_nodes = 0;
};

static void batch_release_graph(fn_batch *b)
{
    if (b->exec) hipGraphExecDestroy(b->exec);
    if (b->graph) hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    for (auto &c : b->classes) {
        hipFree(c.d_jobs);
        hipFree(c.d_items);
        hipFree(c.d_counter);
    }
    for (auto &r : b->stacks) {
        hipFree(r.d_X);
        hipFree(r.d_Xlp);
        hipFree(r.d_xscale);
        hipFree(r.d_rowscale);
        hipFree(r.d_bad);
        hipFree(r.d_txp);
        hipFree(r.d_row_frame);
        hipFree(r.d_frame_image);
    }
    b->stacks.clear();
    b->classes.clear();
    b->singles.clear();
}

// plans whose rows can share one beamforming launch: everything but the transmit
// rows and the RF is equal (single-frame plane-wave plans up to 128 elements)
static bool row_stackable(const fn_plan *P)
{
    // beyond three tiles of rows a plan fills its own transmit groups (the ensemble
    // kernel holds at most four tiles per group against five of the plain kernel)
    return P->mode == 0 && P->n_frames == 1 && !P->lbl && !P->nw && P->KI <= 32 && P->n_tx <= 48;
}

// Interpolated plans join a stack where its one sum over the bins is estimated below their
// images: 0.12 ms for a stack and 0.03 ms a plan beside the two estimates.  ms stacked / apart
// (128 elements, 367 bins): 16 plans of 1 angle at 64 x 64 1.64 / 2.46, 128 x 128 2.03 / 2.49,
// 256 x 256 3.50 / 2.58; 4 at 64 x 64 0.60 / 0.70, 128 x 128 0.97 / 0.70; 16 of 3 angles at 128 x
// 128 2.54 / 2.55; 4 of 11 at 256 x 256 4.00 / 0.97.
static bool stack_interpolated(const fn_batch *b, const std::vector<int> &plans)
{
    int rows = 0;
    double apart = 0.0;
    for (int i : plans) {
        const fn_plan *P = b->plans[i];
        rows += P->n_tx;
        apart += (P->interp_M ? interp_seconds(P, P->interp_M) : sum_seconds(P, P->MT_all)) + 30e-6;
    }
    return sum_seconds(b->plans[plans[0]], (rows + 15) / 16) + 120e-6 < apart;
}

static bool same_receive_side(const fn_plan *a, const fn_plan *b)
{
    const fnk::BeamArgs &x = a->args, &y = b->args;
    auto zeros = [](const std::vector<double> &v) { return std::all_of(v.begin(), v.end(), [](double d) { return d == 0.0; }); };
    const bool delays = (a->h_delay.empty() || zeros(a->h_delay)) && (b->h_delay.empty() || zeros(b->h_delay))
                            ? true
                            : a->h_delay == b->h_delay;
    return a->device == b->device && a->precision == b->precision && a->n_x == b->n_x && a->n_z == b->n_z &&
           a->n_t == b->n_t && a->n_el == b->n_el && a->KI == b->KI && a->g.N == b->g.N && a->g.n_lb == b->g.n_lb &&
           a->g.n_f == b->g.n_f && a->wcr == b->wcr && a->h_px == b->h_px && a->h_pz == b->h_pz &&
           a->h_Frx == b->h_Frx && delays && std::memcmp(&x.wrx, &y.wrx, sizeof(x.wrx)) == 0 &&
           x.support_rx == y.support_rx && x.norm_rx == y.norm_rx && x.clamp == y.clamp &&
           x.out_scale == y.out_scale && x.tx_kind == y.tx_kind && x.pitch == y.pitch && x.width == y.width &&
           x.c0 == y.c0 && x.ctof == y.ctof && x.f_s == y.f_s && x.t0 == y.t0 && x.M == y.M;
}

// group the stackable plans (two or more per stack), size each stack's tiling and
// build its tables: stacked steering rows, row -> plan, plan -> image; outside any capture
static int batch_plan_stacks(fn_batch *b, float *const *d_images, std::vector<char> &taken)
{
    const int n = (int)b->plans.size();
    for (int i = 0; i < n; ++i) {
        if (taken[i] || !row_stackable(b->plans[i])) continue;
        RowStack r;
        for (int j = i; j < n; ++j)
            if (!taken[j] && row_stackable(b->plans[j]) && same_receive_side(b->plans[i], b->plans[j]))
                r.plans.push_back(j);
        auto interpolated = [&](int j) { return b->plans[j]->interp_M > 0; };
        if (std::any_of(r.plans.begin(), r.plans.end(), interpolated) && !stack_interpolated(b, r.plans))
            r.plans.erase(std::remove_if(r.plans.begin(), r.plans.end(), interpolated), r.plans.end());
        if (r.plans.size() < 2) continue;
        for (int j : r.plans) {
            r.row0.push_back(r.rows);
            r.rows += b->plans[j]->n_tx;
            taken[j] = 1;
        }
        const fn_plan *P0 = b->plans[r.plans[0]];
        r.MT_all = (r.rows + 15) / 16;
        const int max_tiles = stack_tile_cap(P0->kprec, P0->KI);  // the stack kernel's register budget
        const int groups = (r.MT_all + max_tiles - 1) / max_tiles;
        r.MT_tmpl = (r.MT_all + groups - 1) / groups;
        r.n_groups = (r.MT_all + r.MT_tmpl - 1) / r.MT_tmpl;
        r.lds_beam = (size_t)r.MT_tmpl * P0->KI * form_step_bytes(P0->kprec);
        // bin chunks: enough workgroups to fill the GPU several times over
        const long blocks = (P0->n_vox + 63) / 64 * r.n_groups;  // one voxel a lane
        int split = 1;
        if (blocks < 2048) split = (int)std::min<long>((2048 + blocks - 1) / blocks, std::max(1, P0->g.n_f / 8));
        r.chunk = (P0->g.n_f + split - 1) / split;
        r.bin_split = (P0->g.n_f + r.chunk - 1) / r.chunk;
        b->stacks.push_back(r);  // freed with the graph, also on failure
        RowStack &R = b->stacks.back();
        const size_t n_f = (size_t)P0->g.n_f;
        const size_t x_bytes = n_f * R.MT_all * P0->KI * 64 * sizeof(float2);
        std::vector<int> rf(16 * (size_t)R.MT_all, -1);
        std::vector<float2 *> imgs;
        for (size_t m = 0; m < R.plans.size(); ++m) {
            for (int a = 0; a < b->plans[R.plans[m]]->n_tx; ++a) rf[R.row0[m] + a] = (int)m;
            imgs.push_back(reinterpret_cast<float2 *>(d_images[R.plans[m]]));
        }
        hipError_t e = hipMalloc(&R.d_X, x_bytes);
        if (e == hipSuccess) e = hipMemset(R.d_X, 0, x_bytes);  // rows past the last plan stay zero
        if (e == hipSuccess && P0->kprec != FN_PRECISION_FP32) {
            e = hipMalloc(&R.d_Xlp, n_f * form_planes(P0->kprec) * R.n_groups * R.MT_tmpl * P0->KI * 64 * 2);
            if (e == hipSuccess) e = hipMalloc(&R.d_xscale, n_f * sizeof(float));
            if (e == hipSuccess) e = hipMalloc(&R.d_bad, bad_bytes((int)n_f, 16 * R.MT_all, P0->KI));
            if (e == hipSuccess && has_row_scales(P0->kprec)) e = hipMalloc(&R.d_rowscale, row_scale_bytes(R.MT_all));
        }
        if (e == hipSuccess) e = hipMalloc(&R.d_txp, 3 * sizeof(double) * R.rows);
        for (size_t m = 0; m < R.plans.size() && e == hipSuccess; ++m) {
            const fn_plan *P = b->plans[R.plans[m]];
            e = hipMemcpy(R.d_txp + 3 * (size_t)R.row0[m], P->d_txp, 3 * sizeof(double) * P->n_tx, hipMemcpyDeviceToDevice);
        }
        if (e == hipSuccess) e = hipMalloc(&R.d_row_frame, rf.size() * sizeof(int));
        if (e == hipSuccess) e = hipMemcpy(R.d_row_frame, rf.data(), rf.size() * sizeof(int), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMalloc(&R.d_frame_image, imgs.size() * sizeof(float2 *));
        if (e == hipSuccess)
            e = hipMemcpy(R.d_frame_image, imgs.data(), imgs.size() * sizeof(float2 *), hipMemcpyHostToDevice);
        if (e != hipSuccess) return hip_fail(e, "row stack tables");
    }
    return FN_OK;
}

// one stack on stream s: the members' images zeroed, their spectra into the stacked
// operand (each at its first row), the 16-bit planes, one ensemble launch
static int batch_run_stack(fn_batch *b, const RowStack &R, const void *const *d_rf, const int32_t *dtypes,
                           float *const *d_images, hipStream_t s)
{
    const fn_plan *P0 = b->plans[R.plans[0]];
    for (size_t m = 0; m < R.plans.size(); ++m) {
        fn_plan *P = b->plans[R.plans[m]];
        const long nz = 2 * P->n_vox;
        hipLaunchKernelGGL(fnk::fill_zero_kernel, dim3((unsigned)((nz + 255) / 256)), dim3(256), 0, s,
                           d_images[R.plans[m]], nz);
        HIP_CHECK(hipGetLastError(), "fill_zero_kernel");
        fnk::SpecArgs S = P->sargs;
        S.row0 = R.row0[m];
        S.MT_out = R.MT_all;
        S.write_pad = 0;
        if (int st = launch_spectra_into(P, d_rf[R.plans[m]], dtypes[R.plans[m]], s, R.d_X, S)) return st;
    }
    if (int st = launch_lowp_planes(P0, R.d_X, R.d_Xlp, R.d_xscale, R.d_bad, 16 * R.MT_all, R.MT_all, R.n_groups * R.MT_tmpl, 0, nullptr, s,
                                    R.d_rowscale))
        return st;
    fnk::BeamArgs A = forward_args(P0);
    A.X = R.d_X;
    A.Xlp = R.d_Xlp;
    A.xscale = R.d_xscale;
    A.row_scale = R.d_rowscale;
    A.bad = R.d_bad;
    A.bad_rows = 16 * R.MT_all;
    A.txp = R.d_txp;
    A.n_tx = R.rows;
    A.tx_group = R.MT_tmpl;
    A.xlp_tiles = R.n_groups * R.MT_tmpl;
    A.bin_chunk = R.chunk;
    A.ens_frames = 0;
    A.ens_slots = 0;
    A.row_frame = R.d_row_frame;
    A.frame_image = R.d_frame_image;
    A.image = nullptr;
    A.weights = nullptr;
    A.weights_tx = nullptr;
    A.partial = nullptr;
    A.n_slots = 1;
    A.slot_z = R.n_groups;
    const dim3 grid((unsigned)((P0->n_vox + 63) / 64), (unsigned)R.bin_split, (unsigned)R.n_groups);
    hipError_t e = fnk::kEnsLaunchers[ki_index(P0->KI)][P0->kprec](R.MT_tmpl, P0->wcr, grid, R.lds_beam, s, A, 1);
    if (e != hipSuccess) return hip_fail(e, "beamform_kernel (row stack)");
    if (!A.bad) return FN_OK;
    hipLaunchKernelGGL(fnk::nonfinite_kernel, dim3((unsigned)((P0->n_vox + 255) / 256)), dim3(256), 0, s, A);
    HIP_CHECK(hipGetLastError(), "nonfinite_kernel (row stack)");
    return FN_OK;
}

// kernel class of a plan for the persistent launches; -1: launched on its own
// (ensembles, windowed normalization)
static long batch_class_key(const fn_plan *P)
{
    if (P->n_frames > 1 || P->nw || P->lbl || P->interp_M || P->KI > 32) return -1;  // persistent kernels up to 128 elements
    return ((((long)P->mode * 64 + P->KI) * 16 + P->MT_tmpl) * 8 + P->wcr) * 8 * 4 + P->wct * 4 + P->kprec;
}

// group the plans into classes, upload each class's job and work-item tables and
// size its grid (resident workgroups x CUs); outside any capture
static int batch_plan_classes(fn_batch *b, float *const *d_images)
{
    std::vector<char> taken(b->plans.size(), 0);
    if (b->stacking)
        if (int st = batch_plan_stacks(b, d_images, taken)) return st;
    std::vector<std::pair<long, std::vector<int>>> groups;
    for (int i = 0; i < (int)b->plans.size(); ++i) {
        if (taken[i]) continue;
        const long key = b->persistent ? batch_class_key(b->plans[i]) : -1;
        if (key < 0) { b->singles.push_back(i); continue; }
        auto it = std::find_if(groups.begin(), groups.end(), [&](const auto &g) { return g.first == key; });
        if (it == groups.end()) groups.push_back({key, {i}});
        else it->second.push_back(i);
    }
    // a class launch waits for the spectra of all its plans: classes are cut into
    // launches of at most kPersistPlans plans, so that one launch beamforms while
    // the worker streams prepare the next
    constexpr size_t kPersistPlans = 8;
    std::vector<std::vector<int>> launches;
    for (auto &g : groups) {
        if (g.second.size() < 2) { b->singles.push_back(g.second[0]); continue; }
        const size_t n_l = (g.second.size() + kPersistPlans - 1) / kPersistPlans;
        for (size_t l = 0; l < n_l; ++l) {
            const size_t lo = g.second.size() * l / n_l, hi = g.second.size() * (l + 1) / n_l;
            launches.emplace_back(g.second.begin() + lo, g.second.begin() + hi);
        }
    }
    int n_cu = 256;
    hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, b->device);
    for (auto &plans : launches) {
        BatchClass c;
        c.plans = plans;
        std::vector<fnk::BeamArgs> jobs;
        std::vector<std::pair<int, int4>> items;  // (bins of the chunk, item)
        for (int j = 0; j < (int)c.plans.size(); ++j) {
            const fn_plan *P = b->plans[c.plans[j]];
            jobs.push_back(beam_args(P, d_images[c.plans[j]], nullptr, nullptr));
            const int tiles = (int)((P->n_vox + 63) / 64), chunk = P->args.bin_chunk;
            for (int bz = 0; bz < P->n_groups; ++bz)
                for (int by = 0; by < P->bin_split; ++by) {
                    const int bins = std::min(chunk, P->g.n_f - by * chunk);
                    for (int bx = 0; bx < tiles; ++bx) items.push_back({bins, make_int4(j, bx, by, bz)});
                }
        }
        std::stable_sort(items.begin(), items.end(), [](const auto &a, const auto &b2) { return a.first > b2.first; });
        std::vector<int4> it4(items.size());
        for (size_t q = 0; q < items.size(); ++q) it4[q] = items[q].second;
        c.n_items = (int)it4.size();
        const fn_plan *P0 = b->plans[c.plans[0]];
        const int kidx = P0->KI == 8 ? 0 : (P0->KI == 16 ? 1 : 2);
        int occ = 0;
        hipError_t e = fnk::kPersistLaunchers[P0->mode][kidx][P0->kprec](P0->MT_tmpl, P0->wcr, P0->wct, 0,
                                                                            P0->lds_beam, nullptr, nullptr, nullptr, 0,
                                                                            nullptr, &occ);
        if (e != hipSuccess) return hip_fail(e, "persistent kernel occupancy");
        c.grid = std::max(1, std::min(c.n_items, std::max(1, occ) * n_cu));
        e = hipMalloc(&c.d_jobs, jobs.size() * sizeof(fnk::BeamArgs));
        if (e == hipSuccess) e = hipMalloc(&c.d_items, it4.size() * sizeof(int4));
        if (e == hipSuccess) e = hipMalloc(&c.d_counter, sizeof(int));
        if (e == hipSuccess) e = hipMemcpy(c.d_jobs, jobs.data(), jobs.size() * sizeof(fnk::BeamArgs), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(c.d_items, it4.data(), it4.size() * sizeof(int4), hipMemcpyHostToDevice);
        b->classes.push_back(c);  // freed with the graph, also on failure
        if (e != hipSuccess) return hip_fail(e, "persistent batch tables");
    }
    return FN_OK;
}

int32_t fn_batch_create(fn_plan *const *plans, int32_t n_plans, int32_t n_streams, fn_batch **out)
{
    fnh::clear_error();
    if (!plans || !out || n_plans < 1) return fail(FN_ERR_ARGUMENT, "plans and batch pointer required");
    *out = nullptr;
    n_streams = std::max(1, std::min(n_streams, 16));
    auto *b = new (std::nothrow) fn_batch();
    if (!b) return fail(FN_ERR_OUT_OF_MEMORY, "host allocation");
    b->device = plans[0] ? plans[0]->device : 0;
    for (int i = 0; i < n_plans; ++i) {
        if (!plans[i]) { delete b; return fail(FN_ERR_ARGUMENT, "plan %d is null", i); }
        if (plans[i]->device != b->device) { delete b; return fail(FN_ERR_ARGUMENT, "plans must share one device"); }
        b->plans.push_back(plans[i]);
    }
    int st = FN_OK;
    hipError_t e = hipSetDevice(b->device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->capture, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->pstream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&b->fork, hipEventDisableTiming);
    for (int i = 0; i < n_streams && e == hipSuccess; ++i) {
        hipStream_t w = nullptr;
        hipEvent_t j = nullptr;
        e = hipStreamCreateWithFlags(&w, hipStreamNonBlocking);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&j, hipEventDisableTiming);
        if (w) b->streams.push_back(w);
        if (j) b->joins.push_back(j);
    }
    if (e != hipSuccess) st = hip_fail(e, "batch streams");
    if (st) { fn_batch_destroy(b); return st; }
    *out = b;
    return FN_OK;
}

int32_t fn_batch_execute(fn_batch *b, const void *const *d_rf, const int32_t *dtypes, float *const *d_images,
                         void *stream)
{
    fnh::clear_error();
    if (!b || !d_rf || !dtypes || !d_images) return fail(FN_ERR_ARGUMENT, "null argument");
    const size_t n = b->plans.size();
    for (size_t i = 0; i < n; ++i)
        if (!d_rf[i] || !d_images[i]) return fail(FN_ERR_ARGUMENT, "buffers of plan %d missing", (int)i);
    HIP_CHECK(hipSetDevice(b->device), "hipSetDevice");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const bool same = b->exec && b->rf.size() == n &&
                      std::equal(b->rf.begin(), b->rf.end(), d_rf) &&
                      std::equal(b->dtypes.begin(), b->dtypes.end(), dtypes) &&
                      std::equal(b->images.begin(), b->images.end(), d_images) &&
                      std::equal(b->plans.begin(), b->plans.end(), b->serials.begin(), [](const fn_plan *P, auto &t) {
                          return P->tof_serial == t.first && P->tiling_serial == t.second;
                      });
    if (!same) {
        batch_release_graph(b);
        // eager pass: validates every job and raises kernel LDS limits outside the capture
        for (size_t i = 0; i < n; ++i) {
            const int prof = b->plans[i]->profiling;
            b->plans[i]->profiling = 0;
            int st = execute(b->plans[i], d_rf[i], dtypes[i], d_images[i], nullptr, nullptr, s);
            b->plans[i]->profiling = prof;
            if (st) return st;
        }
        HIP_CHECK(hipStreamSynchronize(s), "batch warm-up");
        if (int st = batch_plan_classes(b, d_images)) { batch_release_graph(b); return st; }
        // the row stacks once outside the capture (raises their kernels' LDS limits)
        for (const RowStack &R : b->stacks)
            if (int st = batch_run_stack(b, R, d_rf, dtypes, d_images, s)) { batch_release_graph(b); return st; }
        if (!b->stacks.empty()) HIP_CHECK(hipStreamSynchronize(s), "row stack warm-up");
        HIP_CHECK(hipStreamBeginCapture(b->capture, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
        int st = FN_OK;
        const size_t W = b->streams.size();
        hipError_t e = hipEventRecord(b->fork, b->capture);
        for (size_t w = 0; w < W && e == hipSuccess; ++w) e = hipStreamWaitEvent(b->streams[w], b->fork, 0);
        // row stacks and plans on their own (ensembles and the like, usually the longest)
        // first, one worker each; the persistent classes' spectra on the other workers
        const size_t n_single = b->stacks.size() + b->singles.size();
        size_t slot = 0;
        for (const RowStack &R : b->stacks) {
            if (e != hipSuccess || st) break;
            st = batch_run_stack(b, R, d_rf, dtypes, d_images, b->streams[slot++ % W]);
        }
        for (int i : b->singles) {
            if (e != hipSuccess || st) break;
            fn_plan *P = b->plans[i];
            hipStream_t ws = b->streams[slot++ % W];
            st = prepare(P, d_rf[i], dtypes[i], d_images[i], ws);
            const long tiles = beam_tiles(P);
            const fnk::BeamArgs A = beam_args(P, d_images[i], nullptr, nullptr);
            if (!st) e = launch_beam(P, dim3((unsigned)tiles, (unsigned)P->bin_split, (unsigned)P->n_groups), A, ws);
            if (!st && e == hipSuccess) st = finish_beam(P, A, ws);
        }
        const size_t w0 = n_single < W ? n_single : 0, n_w = n_single < W ? W - n_single : W;
        slot = 0;
        for (auto &c : b->classes) {
            if (e != hipSuccess || st) break;
            std::vector<char> used(W, 0);
            for (int i : c.plans) {
                if (st) break;
                const size_t w = w0 + slot++ % n_w;
                st = prepare(b->plans[i], d_rf[i], dtypes[i], d_images[i], b->streams[w]);
                used[w] = 1;
            }
            // the class's launch waits for exactly its own plans' spectra
            for (size_t w = 0; w < W && e == hipSuccess && !st; ++w) {
                if (!used[w]) continue;
                e = hipEventRecord(b->joins[w], b->streams[w]);
                if (e == hipSuccess) e = hipStreamWaitEvent(b->pstream, b->joins[w], 0);
            }
            if (e != hipSuccess || st) break;
            const fn_plan *P0 = b->plans[c.plans[0]];
            const int kidx = P0->KI == 8 ? 0 : (P0->KI == 16 ? 1 : 2);
            e = fnk::kPersistLaunchers[P0->mode][kidx][P0->kprec](P0->MT_tmpl, P0->wcr, P0->wct, c.grid,
                                                                     P0->lds_beam, b->pstream, c.d_jobs, c.d_items,
                                                                     c.n_items, c.d_counter, nullptr);
            for (int i : c.plans) {
                if (e != hipSuccess || st) break;
                st = finish_beam(b->plans[i], beam_args(b->plans[i], d_images[i], nullptr, nullptr), b->pstream);
            }
        }
        for (size_t w = 0; w < W && e == hipSuccess && !st; ++w) {
            e = hipEventRecord(b->joins[w], b->streams[w]);
            if (e == hipSuccess) e = hipStreamWaitEvent(b->capture, b->joins[w], 0);
        }
        if (!b->classes.empty() && e == hipSuccess && !st) {
            e = hipEventRecord(b->fork, b->pstream);
            if (e == hipSuccess) e = hipStreamWaitEvent(b->capture, b->fork, 0);
        }
        hipGraph_t g = nullptr;
        hipError_t e2 = hipStreamEndCapture(b->capture, &g);
        if (e == hipSuccess) e = e2;
        if (st) { if (g) hipGraphDestroy(g); return st; }
        if (e != hipSuccess) { if (g) hipGraphDestroy(g); return hip_fail(e, "batch capture"); }
        b->graph = g;
        e = hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0);
        if (e != hipSuccess) { batch_release_graph(b); return hip_fail(e, "hipGraphInstantiate"); }
        size_t nodes = 0;
        if (hipGraphGetNodes(g, nullptr, &nodes) == hipSuccess) b->n_nodes = (int64_t)nodes;
        b->rf.assign(d_rf, d_rf + n);
        b->dtypes.assign(dtypes, dtypes + n);
        b->images.assign(d_images, d_images + n);
        b->serials.clear();
        for (const fn_plan *P : b->plans) b->serials.push_back({P->tof_serial, P->tiling_serial});
        b->captures += 1;
    }
    HIP_CHECK(hipGraphLaunch(b->exec, s), "hipGraphLaunch");
    return FN_OK;
}

int32_t fn_batch_info(const fn_batch *b, int64_t *n_nodes, int32_t *n_captures)
{
    if (!b) return fail(FN_ERR_ARGUMENT, "null batch");
    if (n_nodes) *n_nodes = b->n_nodes;
    if (n_captures) *n_captures = b->captures;
    return FN_OK;
}

int32_t fn_batch_destroy(fn_batch *b)
{
    if (!b) return FN_OK;
    hipSetDevice(b->device);
    for (hipStream_t w : b->streams) hipStreamSynchronize(w);
    if (b->capture) hipStreamSynchronize(b->capture);
    if (b->pstream) hipStreamSynchronize(b->pstream);
    batch_release_graph(b);
    for (hipStream_t w : b->streams) hipStreamDestroy(w);
    for (hipEvent_t j : b->joins) hipEventDestroy(j);
    if (b->fork) hipEventDestroy(b->fork);
    if (b->capture) hipStreamDestroy(b->capture);
    if (b->pstream) hipStreamDestroy(b->pstream);
    delete b;
    return FN_OK;
}

int32_t fn_batch_set_stacking(fn_batch *b, int32_t enable)
{
    fnh::clear_error();
    if (!b) return fail(FN_ERR_ARGUMENT, "null batch");
    if (b->stacking != (enable != 0)) {
        hipSetDevice(b->device);
        batch_release_graph(b);  // captured again at the next execute
    }
    b->stacking = enable != 0;
    return FN_OK;
}

int32_t fn_batch_stacks(const fn_batch *b, int32_t *n_stacks, int32_t *n_stacked_plans)
{
    if (!b) return fail(FN_ERR_ARGUMENT, "null batch");
    int32_t k = 0;
    for (const RowStack &r : b->stacks) k += (int32_t)r.plans.size();
    if (n_stacks) *n_stacks = (int32_t)b->stacks.size();
    if (n_stacked_plans) *n_stacked_plans = k;
    return FN_OK;
}

int32_t fn_batch_set_persistent(fn_batch *b, int32_t enable)
{
    fnh::clear_error();
    if (!b) return fail(FN_ERR_ARGUMENT, "null batch");
    if (b->persistent != (enable != 0)) {
        hipSetDevice(b->device);
        batch_release_graph(b);  // captured again at the next execute
    }
    b->persistent = enable != 0;
    return FN_OK;
}

}  // extern "C"
