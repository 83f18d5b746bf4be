// pyramid.hip -- CDNA4 (gfx950) multiscale pyramid of the reference's
// multiscale denoising (multiscaler/multiscaler.cpp, decompose.cpp,
// recompose.cpp, merge_coarse.cpp; src/utils/VBM3Ddenoising_multiscale.sh)
// and its C-ABI entry points.
//
// Images are planar float [c][rows][cols] in HBM.  The DCT pyramid takes
// the full-frame 2D DCT as two matrix products per channel -- T = X A_C^T
// along the rows, Y = A_R T down the columns, A_N the REDFT10 (or
// REDFT01) matrix -- in FP64 through rocBLAS's strided-batched DGEMM on
// the matrix cores, then one rounding to float: the transform's exact
// value to within double rounding (the reference's FFTW float transform
// differs from it in the last bits).  The matrices are formed on the GPU
// and the planes of many frames go through each product together.  The
// Gaussian and Lanczos pyramids
// are separable convolutions, one thread per output sample, in the
// reference's float order: bit for bit its results.
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>

#include <cmath>
#include <cstdint>
#include <string>
#include <vector>

#include "vbm3d_hip.h"

#pragma clang fp contract(off)

struct vbm3d_ctx;

namespace vb {
hipStream_t ctx_stream(vbm3d_ctx* c);
int ctx_device(vbm3d_ctx* c);
hipError_t ctx_pyr_workspace(vbm3d_ctx* c, size_t bytes, void** p);
hipError_t ctx_multiscale_buffer(vbm3d_ctx* c, size_t bytes, void** p);
void ctx_multiscale_trim(vbm3d_ctx* c, size_t keep);
size_t ctx_pyr_held(const vbm3d_ctx* c);
rocblas_handle ctx_blas(vbm3d_ctx* c);
int ctx_fail(int code, const std::string& msg);
}  // namespace vb

namespace vb {
namespace {

constexpr int BX = 64, BY = 4;
constexpr int kMaxPyrTaps = 32;
constexpr size_t kPyrBatchBytes = (size_t)1 << 30;  // workspace bound of a batch of frames
// Bytes of multiscale denoising's buffers (about 4.7 clips and the batch's
// workspace) that a context keeps for its next call; larger ones are freed at
// the call's end, where allocating them again is small beside the call (20 RGB
// frames 1280x720: 96.7 -> 97.4 ms; 30 grey frames 640x480, 0.57 GB, would take
// 17.8 ms instead of 16.9).
constexpr size_t kMultiscaleKeep = (size_t)1 << 30;

struct PTaps {
    float k[kMaxPyrTaps];
    int n;
    float offset;
};

dim3 g2(int cols, int rows, int ch) {
    return dim3((unsigned)((cols + BX - 1) / BX), (unsigned)((rows + BY - 1) / BY), (unsigned)ch);
}

// ---- element kernels
// The top-left rows x cols block of each sr x sc plane, as doubles
// (decompose.cpp:44-52 where the block is smaller than the plane)
__global__ void k_to_double(const float* __restrict__ in, int sr, int sc, double* out, int rows, int cols) {
    const int q = blockIdx.x * BX + threadIdx.x, r = blockIdx.y * BY + threadIdx.y;
    const size_t c = blockIdx.z;
    if (q >= cols || r >= rows) return;
    out[(c * rows + r) * cols + q] = (double)in[(c * sr + r) * sc + q];
}

// float(Y) / (4 rows cols) for the forward DCT (multiscaler.cpp:52-56),
// float(Y) for the inverse, of the top-left h x w block of rows x cols
// planes, into dr x dc planes (recompose.cpp:50-56 where these are larger)
__global__ void k_from_double(const double* __restrict__ in, int rows, int cols, float* out, int dr, int dc, int h,
                              int w, float div, int apply) {
    const int q = blockIdx.x * BX + threadIdx.x, r = blockIdx.y * BY + threadIdx.y;
    const size_t c = blockIdx.z;
    if (q >= w || r >= h) return;
    const float v = (float)in[(c * rows + r) * cols + q];
    out[(c * dr + r) * dc + q] = apply ? v / div : v;
}

// REDFT10 (inverse = 0: 2 cos(pi k (2n+1) / 2N)) or REDFT01 (1 for n = 0,
// else 2 cos(pi n (2k+1) / 2N)) as a row-major N x N table [k][n].  The
// argument is reduced in integers, so that cospi sees it in [0, 2).
// Filled here, a table takes microseconds; the host's cosines took most of
// a call (4 RGB frames 640x360 in 3 levels: 86.9 ms per call, 4.3 ms of
// them in kernels).
__global__ void k_dct_table(double* a, int N, int inverse) {
    const int n = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + threadIdx.y;
    if (n >= N || k >= N) return;
    const unsigned long long m = inverse ? (unsigned long long)n * (2u * (unsigned)k + 1u)
                                         : (unsigned long long)k * (2u * (unsigned)n + 1u);
    const double c = cospi((double)(m % (4ull * (unsigned)N)) / (2.0 * N));
    a[(size_t)k * N + n] = inverse && n == 0 ? 1.0 : 2.0 * c;
}

__global__ void k_fill_zero(float* p, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = 0.f;
}

__global__ void k_axpy(float* a, const float* __restrict__ b, long n, float sign) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        a[i] = sign > 0 ? a[i] + b[i] : a[i] - b[i];
}

// ---- separable convolution with clamped, rounded tap positions
// (multiscaler.cpp:136-185): pass 0 along the rows index, pass 1 along
// the columns, float sums in tap order
__global__ void k_conv_clamped(const float* __restrict__ in, float* out, int rows, int cols, PTaps t, int pass) {
    const int q = blockIdx.x * BX + threadIdx.x, r = blockIdx.y * BY + threadIdx.y, c = blockIdx.z;
    if (q >= cols || r >= rows) return;
    const float* p = in + (size_t)c * rows * cols;
    float val = 0.0f;
    for (int i = 0; i < t.n; i++) {
        if (pass == 0) {
            int j = (int)roundf((float)r - t.offset + (float)i);
            j = min(max(j, 0), rows - 1);
            val += p[(size_t)j * cols + q] * t.k[i];
        } else {
            int j = (int)roundf((float)q - t.offset + (float)i);
            j = min(max(j, 0), cols - 1);
            val += p[(size_t)r * cols + j] * t.k[i];
        }
    }
    out[((size_t)c * rows + r) * cols + q] = val;
}

// ---- one-direction convolution, symmetric boundary, truncated tap
// positions (multiscaler.cpp:190-247); dir 0 along the rows index
__global__ void k_conv_dir(const float* __restrict__ in, float* out, int rows, int cols, PTaps t, int dir) {
    const int q = blockIdx.x * BX + threadIdx.x, r = blockIdx.y * BY + threadIdx.y, c = blockIdx.z;
    if (q >= cols || r >= rows) return;
    const float* p = in + (size_t)c * rows * cols;
    const int X = dir == 0 ? rows : cols, X2 = 2 * X, x = dir == 0 ? r : q;
    float val = 0.0f;
    for (int i = 0; i < t.n; i++) {
        int j = (int)((float)x - t.offset + (float)i);
        while (j < 0) j += X2;
        while (j >= X2) j -= X2;
        if (j >= X) j = X2 - 1 - j;
        val += p[dir == 0 ? (size_t)j * cols + q : (size_t)r * cols + j] * t.k[i];
    }
    out[((size_t)c * rows + r) * cols + q] = val;
}

// out[2r][2q] = in[r][q] of a (rows x cols) -> (rows/2 x cols/2) subsample
__global__ void k_subsample(const float* __restrict__ in, float* out, int rows, int cols) {
    const int r2 = rows / 2, c2 = cols / 2;
    const int q = blockIdx.x * BX + threadIdx.x, r = blockIdx.y * BY + threadIdx.y, c = blockIdx.z;
    if (q >= c2 || r >= r2) return;
    out[((size_t)c * r2 + r) * c2 + q] = in[((size_t)c * rows + 2 * r) * cols + 2 * q];
}

// one phase of the 2x upsampling (multiscaler.cpp:337-398): out[2j + rp]
// [2k + cp] = t[j][k]; for an uneven target the last row / column copies
// the phase's last row / column where the reference does
__global__ void k_up_phase(const float* __restrict__ t, float* out, int rows, int cols, int sx, int sy, int rp,
                           int cp) {
    const int q = blockIdx.x * BX + threadIdx.x, r = blockIdx.y * BY + threadIdx.y, c = blockIdx.z;
    if (q >= cols || r >= rows) return;
    const float v = t[((size_t)c * rows + r) * cols + q];
    float* o = out + (size_t)c * sx * sy;
    o[(size_t)(2 * r + rp) * sy + 2 * q + cp] = v;
    // (rp, cp) = (0, 1): last column, rows 2j; (1, 0): last row, columns
    // 2k; (1, 1): last row, columns 2k+1, last column, rows 2j+1, corner
    const bool oddx = sx % 2 == 1, oddy = sy % 2 == 1;
    if (rp == 0 && cp == 1 && oddy && q == cols - 1) o[(size_t)(2 * r) * sy + sy - 1] = v;
    if (rp == 1 && cp == 0 && oddx && r == rows - 1) o[(size_t)(sx - 1) * sy + 2 * q] = v;
    if (rp == 1 && cp == 1) {
        if (oddx && r == rows - 1) o[(size_t)(sx - 1) * sy + 2 * q + 1] = v;
        if (oddy && q == cols - 1) o[(size_t)(2 * r + 1) * sy + sy - 1] = v;
        if (oddx && oddy && r == rows - 1 && q == cols - 1) o[(size_t)(sx - 1) * sy + sy - 1] = v;
    }
}

// ---- host-side taps (multiscaler.cpp:261-276, 392-418, 279-304)
PTaps gaussian_taps(int n, float sigma, float mean) {
    PTaps t{};
    t.n = n;
    t.offset = mean;
    double sum = 0.;
    for (int i = 0; i < n; i++) {
        const int val = (int)((i - mean) / sigma);
        t.k[i] = (float)std::exp(-0.5 * val * val);
        sum += t.k[i];
    }
    if (sum > 0.)
        for (int i = 0; i < n; i++) t.k[i] = (float)(t.k[i] / sum);
    return t;
}

float lanczos3(float x) {
    if (std::abs(x) >= 3) return 0.f;
    if (x == 0.) return 1.f;
    return (float)(std::sin(M_PI * x) / (M_PI * x) * std::sin(M_PI * x / 3.) / (M_PI * x / 3.));
}

PTaps lanczos_taps(int n, float offset) {
    PTaps t{};
    t.n = n;
    t.offset = offset;
    double sum = 0.;
    for (int i = 0; i < n; i++) {
        t.k[i] = (float)(lanczos3((float)((i - offset) / 2.)) / 2.);
        sum += t.k[i];
    }
    if (sum > 0.)
        for (int i = 0; i < n; i++) t.k[i] = (float)(t.k[i] / sum);
    return t;
}

PTaps down_taps(bool lanczos) {
    if (lanczos) return lanczos_taps(12, 5.5f);
    const float sigma = 1.39f, prec = 3.0f;
    const float offset = (float)(std::ceil(sigma * std::sqrt(2.0 * prec * std::log(10.0))) + 0.5);
    return gaussian_taps((int)(1 + 2 * offset), sigma, offset);
}

#define PYR_TRY(expr)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess) return ctx_fail(VBM3D_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)
#define BLAS_TRY(expr)                                                                       \
    do {                                                                                     \
        rocblas_status s_ = (expr);                                                          \
        if (s_ != rocblas_status_success)                                                    \
            return ctx_fail(VBM3D_ERR_HIP, std::string(#expr) + ": " + rocblas_status_to_string(s_)); \
    } while (0)

// The device work of the pyramid entries: a context, its stream, and an arena
// in the context's workspace (planes, and the DCT matrices of the call at
// hand, which every dct2 forms anew).
struct Pyr {
    vbm3d_ctx* ctx;
    hipStream_t s;
    char* base = nullptr;
    size_t cap = 0, used = 0;

    template <class T>
    T* take(size_t n) {
        const size_t at = (used + 255) & ~(size_t)255;
        if (at + n * sizeof(T) > cap) return nullptr;
        used = at + n * sizeof(T);
        return (T*)(base + at);
    }
};

// 2D DCT (REDFT10, / 4 rows cols) or inverse (REDFT01) of the top-left
// rows x cols block of `np` planes of sr x sc (multiscaler.cpp:21-98) with
// two strided-batched DGEMMs; the top-left h x w block of the result goes
// into planes of dr x dc.  src and dst may be the same planes.
// Column-major view: a row-major rows x cols plane is the cols x rows
// matrix P^T; T^T = A_C P^T, then Y^T = T^T A_R^T.
int dct2(Pyr& P, const float* src, int sr, int sc, float* dst, int dr, int dc, int h, int w, int rows, int cols, int np,
         bool inverse) {
    const size_t n = (size_t)np * rows * cols;
    const size_t mark = P.used;
    double* x = P.take<double>(n);
    double* t = P.take<double>(n);
    double* ar = P.take<double>((size_t)rows * rows);
    double* ac = P.take<double>((size_t)cols * cols);
    if (!x || !t || !ar || !ac) return ctx_fail(VBM3D_ERR_NOMEM, "pyramid workspace too small");
    const dim3 b(BX, BY);
    hipLaunchKernelGGL(k_dct_table, g2(rows, rows, 1), b, 0, P.s, ar, rows, inverse ? 1 : 0);
    hipLaunchKernelGGL(k_dct_table, g2(cols, cols, 1), b, 0, P.s, ac, cols, inverse ? 1 : 0);
    hipLaunchKernelGGL(k_to_double, g2(cols, rows, np), b, 0, P.s, src, sr, sc, x, rows, cols);
    PYR_TRY(hipGetLastError());
    rocblas_handle hd = ctx_blas(P.ctx);
    const double one = 1.0, zero = 0.0;
    const rocblas_stride st = (rocblas_stride)rows * cols;
    // T^T (cols x rows) = A_C (row-major table = col-major A_C^T, transposed) * P^T
    BLAS_TRY(rocblas_dgemm_strided_batched(hd, rocblas_operation_transpose, rocblas_operation_none, cols, rows, cols,
                                           &one, ac, cols, 0, x, cols, st, &zero, t, cols, st, np));
    // Y^T (cols x rows) = T^T * A_R^T (the row-major table read column-major)
    BLAS_TRY(rocblas_dgemm_strided_batched(hd, rocblas_operation_none, rocblas_operation_none, cols, rows, rows, &one,
                                           t, cols, st, ar, rows, 0, &zero, x, cols, st, np));
    hipLaunchKernelGGL(k_from_double, g2(w, h, np), b, 0, P.s, x, rows, cols, dst, dr, dc, h, w,
                       (float)(4 * rows * cols), inverse ? 0 : 1);
    PYR_TRY(hipGetLastError());
    P.used = mark;
    return VBM3D_OK;
}

// The whole planes, in place.
int dct2(Pyr& P, float* img, int rows, int cols, int np, bool inverse) {
    return dct2(P, img, rows, cols, img, rows, cols, rows, cols, rows, cols, np, inverse);
}

int conv_clamped(Pyr& P, float* img, float* tmp, int rows, int cols, int ch, const PTaps& t) {
    hipLaunchKernelGGL(k_conv_clamped, g2(cols, rows, ch), dim3(BX, BY), 0, P.s, img, tmp, rows, cols, t, 0);
    hipLaunchKernelGGL(k_conv_clamped, g2(cols, rows, ch), dim3(BX, BY), 0, P.s, tmp, img, rows, cols, t, 1);
    PYR_TRY(hipGetLastError());
    return VBM3D_OK;
}

// gdown / ldown (multiscaler.cpp:281-331, 421-443): blur a copy, keep
// every other sample; out is (rows/2) x (cols/2)
int down(Pyr& P, const float* img, float* out, int rows, int cols, int ch, bool lanczos) {
    const size_t n = (size_t)ch * rows * cols, mark = P.used;
    float* b = P.take<float>(n);
    float* tmp = P.take<float>(n);
    if (!b || !tmp) return ctx_fail(VBM3D_ERR_NOMEM, "pyramid workspace too small");
    PYR_TRY(hipMemcpyAsync(b, img, n * 4, hipMemcpyDeviceToDevice, P.s));
    int rc = conv_clamped(P, b, tmp, rows, cols, ch, down_taps(lanczos));
    if (rc) return rc;
    hipLaunchKernelGGL(k_subsample, g2(cols / 2, rows / 2, ch), dim3(BX, BY), 0, P.s, b, out, rows, cols);
    PYR_TRY(hipGetLastError());
    P.used = mark;
    return VBM3D_OK;
}

// gup / lup (multiscaler.cpp:337-398, 448-509): rows x cols -> sx x sy
int up(Pyr& P, const float* img, float* out, int rows, int cols, int ch, int sx, int sy, bool lanczos) {
    const size_t n = (size_t)ch * rows * cols, mark = P.used;
    float* t1 = P.take<float>(n);
    float* t2 = P.take<float>(n);
    if (!t1 || !t2) return ctx_fail(VBM3D_ERR_NOMEM, "pyramid workspace too small");
    const PTaps k1 = lanczos ? lanczos_taps(6, 2.25f) : gaussian_taps(5, 0.5f, 2.f);
    const PTaps k2 = lanczos ? lanczos_taps(6, 2.75f) : gaussian_taps(5, 0.5f, 1.5f);
    const dim3 g = g2(cols, rows, ch), b(BX, BY);
    hipLaunchKernelGGL(k_fill_zero, dim3(1024), dim3(256), 0, P.s, out, (long)ch * sx * sy);
    hipLaunchKernelGGL(k_conv_dir, g, b, 0, P.s, img, t1, rows, cols, k1, 0);
    hipLaunchKernelGGL(k_conv_dir, g, b, 0, P.s, t1, t2, rows, cols, k1, 1);
    hipLaunchKernelGGL(k_up_phase, g, b, 0, P.s, t2, out, rows, cols, sx, sy, 0, 0);
    hipLaunchKernelGGL(k_conv_dir, g, b, 0, P.s, t1, t2, rows, cols, k2, 1);
    hipLaunchKernelGGL(k_up_phase, g, b, 0, P.s, t2, out, rows, cols, sx, sy, 0, 1);
    hipLaunchKernelGGL(k_conv_dir, g, b, 0, P.s, img, t1, rows, cols, k2, 0);
    hipLaunchKernelGGL(k_conv_dir, g, b, 0, P.s, t1, t2, rows, cols, k1, 1);
    hipLaunchKernelGGL(k_up_phase, g, b, 0, P.s, t2, out, rows, cols, sx, sy, 1, 0);
    hipLaunchKernelGGL(k_conv_dir, g, b, 0, P.s, t1, t2, rows, cols, k2, 1);
    hipLaunchKernelGGL(k_up_phase, g, b, 0, P.s, t2, out, rows, cols, sx, sy, 1, 1);
    PYR_TRY(hipGetLastError());
    P.used = mark;
    return VBM3D_OK;
}

// Level sizes: each level halves the previous one (integer division).
void level_sizes(int rows, int cols, int levels, std::vector<int>& lr, std::vector<int>& lc) {
    lr.resize(levels);
    lc.resize(levels);
    for (int i = 0; i < levels; i++) {
        lr[i] = rows;
        lc[i] = cols;
        rows /= 2;
        cols /= 2;
    }
}

size_t level_words(int rows, int cols, int ch, int levels) {
    std::vector<int> lr, lc;
    level_sizes(rows, cols, levels, lr, lc);
    size_t n = 0;
    for (int i = 0; i < levels; i++) n += (size_t)ch * lr[i] * lc[i];
    return n;
}

// Workspace bytes of one image's pyramid operations: the DCT's two
// double planes and matrices, or the convolutions' float planes, and a
// full-size float plane for recomposition.
size_t pyr_bytes(int rows, int cols, int ch) {
    const size_t n = (size_t)ch * rows * cols;
    return n * 8 * 2 + ((size_t)rows * rows + (size_t)cols * cols) * 8 + n * 4 * 6 + 16 * 256;
}

int check_image(int rows, int cols, int ch, int levels, int type) {
    if (rows < 1 || cols < 1 || (ch != 1 && ch != 3) || (long)rows * cols > (1L << 28))
        return ctx_fail(VBM3D_ERR_ARG, "image: 1 or 3 channels, at most 2^28 pixels");
    if (levels < 1 || (type != 0 && type != 1 && type != 2))
        return ctx_fail(VBM3D_ERR_ARG, "levels >= 1 and type 0 (DCT), 1 (Gaussian) or 2 (Lanczos)");
    std::vector<int> lr, lc;
    level_sizes(rows, cols, levels, lr, lc);
    if (lr[levels - 1] < 1 || lc[levels - 1] < 1) return ctx_fail(VBM3D_ERR_ARG, "too many levels for the image size");
    return VBM3D_OK;
}

// The levels' planes, stored one level after the other: level i of `np`
// planes in total, of which `at` come before the ones at hand.
template <class T>
std::vector<T*> level_ptrs(T* base, int rows, int cols, int np, int levels, int at) {
    std::vector<int> lr, lc;
    level_sizes(rows, cols, levels, lr, lc);
    std::vector<T*> p(levels);
    for (int i = 0; i < levels; i++) {
        const size_t sz = (size_t)lr[i] * lc[i];
        p[i] = base + sz * at;
        base += sz * np;
    }
    return p;
}

// decompose.cpp:17-106 on `ch` device planes (the channels of one or more
// frames); out[i]: the planes of level i.
int decompose_dev(Pyr& P, const float* img, int rows, int cols, int ch, int levels, int type,
                  const std::vector<float*>& out) {
    std::vector<int> lr, lc;
    level_sizes(rows, cols, levels, lr, lc);
    const size_t n = (size_t)ch * rows * cols, mark = P.used;
    int rc;
    if (type == 0) {
        float* d = P.take<float>(n);
        if (!d) return ctx_fail(VBM3D_ERR_NOMEM, "pyramid workspace too small");
        if ((rc = dct2(P, img, rows, cols, d, rows, cols, rows, cols, rows, cols, ch, false))) return rc;
        for (int i = 0; i < levels; i++)
            if ((rc = dct2(P, d, rows, cols, out[i], lr[i], lc[i], lr[i], lc[i], lr[i], lc[i], ch, true))) return rc;
        P.used = mark;
        return VBM3D_OK;
    }
    PYR_TRY(hipMemcpyAsync(out[0], img, n * 4, hipMemcpyDeviceToDevice, P.s));
    for (int i = 1; i < levels; i++)
        if ((rc = down(P, out[i - 1], out[i], lr[i - 1], lc[i - 1], ch, type == 2))) return rc;
    return VBM3D_OK;
}

// recompose.cpp:17-125 on `ch` device planes; lev[i]: the planes of level i.
int recompose_dev(Pyr& P, const std::vector<const float*>& lev, int rows, int cols, int ch, int levels, int type,
                  float factor, float* out) {
    std::vector<int> lr, lc;
    level_sizes(rows, cols, levels, lr, lc);
    const size_t mark = P.used;
    int rc;
    if (type == 0) {
        if ((rc = dct2(P, lev[0], rows, cols, out, rows, cols, rows, cols, rows, cols, ch, false))) return rc;
        for (int i = 1; i < levels; i++) {
            const int h = lr[i], w = lc[i];
            // the copied block: j < h * factor, k < w * factor (float bounds)
            int bh = 0, bw = 0;
            while (bh < h && (float)bh < h * factor) bh++;
            while (bw < w && (float)bw < w * factor) bw++;
            if (bh > 0 && bw > 0 && (rc = dct2(P, lev[i], h, w, out, rows, cols, bh, bw, h, w, ch, false))) return rc;
        }
        if ((rc = dct2(P, out, rows, cols, ch, true))) return rc;
        P.used = mark;
        return VBM3D_OK;
    }
    const bool lz = type == 2;
    float* cur = P.take<float>((size_t)ch * rows * cols);
    float* nxt = P.take<float>((size_t)ch * rows * cols);
    float* small = P.take<float>((size_t)ch * rows * cols);
    if (!cur || !nxt || !small) return ctx_fail(VBM3D_ERR_NOMEM, "pyramid workspace too small");
    PYR_TRY(hipMemcpyAsync(cur, lev[levels - 1], (size_t)ch * lr[levels - 1] * lc[levels - 1] * 4,
                           hipMemcpyDeviceToDevice, P.s));
    for (int i = levels - 2; i >= 0; --i) {
        const int h = lr[i], w = lc[i], h2 = lr[i + 1], w2 = lc[i + 1];
        const float* image = lev[i];
        if ((rc = down(P, image, small, h, w, ch, lz))) return rc;
        const long n2 = (long)ch * h2 * w2;
        hipLaunchKernelGGL(k_axpy, dim3(256), dim3(256), 0, P.s, cur, small, n2, -1.f);
        PYR_TRY(hipGetLastError());
        // gblur(current, factor) (:279-304): skipped below 0.41
        if (!(factor < 0.41)) {
            const float prec = 3.0f;
            const float offset = (float)((int)std::ceil(factor * std::sqrt(2.0 * prec * std::log(10.0)))) - 0.5f;
            const int nt = (int)(2 * offset);
            if (nt > kMaxPyrTaps) return ctx_fail(VBM3D_ERR_UNSUPPORTED, "recomposition blur too wide");
            if ((rc = conv_clamped(P, cur, small, h2, w2, ch, gaussian_taps(nt, factor, offset)))) return rc;
        }
        if ((rc = up(P, cur, nxt, h2, w2, ch, h, w, lz))) return rc;
        hipLaunchKernelGGL(k_axpy, dim3(256), dim3(256), 0, P.s, nxt, image, (long)ch * h * w, 1.f);
        PYR_TRY(hipGetLastError());
        std::swap(cur, nxt);
    }
    PYR_TRY(hipMemcpyAsync(out, cur, (size_t)ch * rows * cols * 4, hipMemcpyDeviceToDevice, P.s));
    P.used = mark;
    return VBM3D_OK;
}

int pyr_open(vbm3d_ctx* ctx, Pyr& P, size_t bytes) {
    if (!ctx) return ctx_fail(VBM3D_ERR_ARG, "null context");
    if (hipSetDevice(ctx_device(ctx)) != hipSuccess) return ctx_fail(VBM3D_ERR_HIP, "hipSetDevice failed");
    P.ctx = ctx;
    P.s = ctx_stream(ctx);
    void* b = nullptr;
    if (ctx_pyr_workspace(ctx, bytes, &b) != hipSuccess)
        return ctx_fail(VBM3D_ERR_NOMEM, "device allocation of the pyramid workspace failed");
    P.base = (char*)b;
    P.cap = bytes;
    P.used = 0;
    if (!ctx_blas(ctx)) return ctx_fail(VBM3D_ERR_HIP, "rocblas_create_handle failed");
    return VBM3D_OK;
}

// Device copies of host inputs, released on every return.
struct Dev {
    std::vector<void*> p;
    ~Dev() {
        for (void* q : p) (void)hipFree(q);
    }
    float* get(size_t n) {
        void* q = nullptr;
        if (hipMalloc(&q, n * 4 > 0 ? n * 4 : 4) != hipSuccess) return nullptr;
        p.push_back(q);
        return (float*)q;
    }
};

// Multiscale denoising on the context's buffers (vbm3d_multiscale_denoise).
int multiscale_denoise(vbm3d_ctx* ctx, float sigma, const float* noisy, unsigned W, unsigned H, unsigned F,
                       unsigned C, const vbm3d_params* p1, const vbm3d_params* p2, int levels, int type,
                       float factor, int color_space, int ref_grid_nb, float* denoised, float* noisy_levels,
                       float* denoised_levels) {
    int rc = check_image((int)H, (int)W, (int)C, levels, type);
    if (rc) return rc;
    if (!noisy || !denoised || F == 0) return ctx_fail(VBM3D_ERR_ARG, "null buffer or empty video");
    if (!(sigma > 0.f)) return ctx_fail(VBM3D_ERR_ARG, "sigma must be positive");
    if (!ctx) return ctx_fail(VBM3D_ERR_ARG, "null context");
    if (hipSetDevice(ctx_device(ctx)) != hipSuccess) return ctx_fail(VBM3D_ERR_HIP, "hipSetDevice failed");
    std::vector<int> lr, lc;
    level_sizes((int)H, (int)W, levels, lr, lc);
    const size_t fw = (size_t)C * H * W, flev = level_words((int)H, (int)W, (int)C, levels);
    // the video, its levels (noisy and denoised: per level [F][C][h][w],
    // level after level) and a basic estimate
    void* base = nullptr;
    if (ctx_multiscale_buffer(ctx, (2 * fw + 2 * flev) * F * 4, &base) != hipSuccess)
        return ctx_fail(VBM3D_ERR_NOMEM, "device allocation failed");
    float *dn = (float*)base, *dbas = dn + fw * F, *dlev = dbas + fw * F, *dden = dlev + flev * F;
    // frames that go through the pyramid together: as many as a workspace of
    // kPyrBatchBytes holds, or of 1/64 of the free memory (the denoiser's
    // rings come out of the same), and fewer if it cannot be had, down to one
    // (planes are a grid dimension: at most 65535).  The free memory is asked
    // for only where the context's workspace is too small.
    const size_t frame_bytes = pyr_bytes((int)H, (int)W, (int)C);
    auto frames_in = [&](size_t room) {
        return (int)std::max<size_t>(1, std::min<size_t>(std::min<size_t>(F, 65535 / C), room / frame_bytes));
    };
    int batch = frames_in(kPyrBatchBytes);
    if (pyr_bytes((int)H, (int)W, (int)C * batch) > ctx_pyr_held(ctx)) {
        size_t room = 0, total = 0;
        if (hipMemGetInfo(&room, &total) != hipSuccess) room = 0;
        batch = frames_in(std::min(kPyrBatchBytes, std::max(room / 64, ctx_pyr_held(ctx))));
    }
    Pyr P;
    while ((rc = pyr_open(ctx, P, pyr_bytes((int)H, (int)W, (int)C * batch))) == VBM3D_ERR_NOMEM && batch > 1) {
        batch = (batch + 1) / 2;
        (void)hipGetLastError();  // the failed allocation's
    }
    if (rc) return rc;
    std::vector<size_t> loff(levels);
    size_t o = 0;
    for (int i = 0; i < levels; i++) {
        loff[i] = o;
        o += (size_t)C * lr[i] * lc[i] * F;
    }
    PYR_TRY(hipMemcpyAsync(dn, noisy, fw * F * 4, hipMemcpyHostToDevice, P.s));
    // 1. every frame into its levels
    for (unsigned t = 0; t < F; t += (unsigned)batch) {
        const int nf = (int)std::min<unsigned>((unsigned)batch, F - t);
        if ((rc = decompose_dev(P, dn + fw * t, (int)H, (int)W, (int)C * nf, levels, type,
                                level_ptrs(dlev, (int)H, (int)W, (int)(C * F), levels, (int)(C * t)))))
            return rc;
    }
    if (noisy_levels) {
        PYR_TRY(hipMemcpyAsync(noisy_levels, dlev, flev * F * 4, hipMemcpyDeviceToHost, P.s));
    }
    PYR_TRY(hipStreamSynchronize(P.s));
    // 2. each level denoised as a video with sigma / 2^level, truncated to
    //    two decimals as the multiscale shell script's `bc` computes it
    //    (src/utils/VBM3Ddenoising_multiscale.sh:52-58)
    for (int i = 0; i < levels; i++) {
        const double sl_exact = (double)sigma / std::ldexp(1.0, i);
        const float sl = (float)(std::floor(sl_exact * 100.0 + 1e-9) / 100.0);
        vbm3d_params q1, q2;
        if (p1) q1 = *p1;
        else vbm3d_default_params_1(&q1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1.f, -1.f, (unsigned)-1, (unsigned)-1, sl);
        if (p2) q2 = *p2;
        else vbm3d_default_params_2(&q2, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1.f, (unsigned)-1, (unsigned)-1, sl);
        if ((rc = vbm3d_run_device(ctx, sl, dlev + loff[i], nullptr, nullptr, (unsigned)lc[i], (unsigned)lr[i], F, C, &q1,
                                   &q2, color_space, ref_grid_nb, dbas, dden + loff[i], nullptr)))
            return rc;
    }
    if (denoised_levels) {
        PYR_TRY(hipMemcpyAsync(denoised_levels, dden, flev * F * 4, hipMemcpyDeviceToHost, P.s));
    }
    // 3. every frame recomposed from its denoised levels
    for (unsigned t = 0; t < F; t += (unsigned)batch) {
        const int nf = (int)std::min<unsigned>((unsigned)batch, F - t);
        if ((rc = recompose_dev(P, level_ptrs((const float*)dden, (int)H, (int)W, (int)(C * F), levels, (int)(C * t)),
                                (int)H, (int)W, (int)C * nf, levels, type, factor, dn + fw * t)))
            return rc;
    }
    PYR_TRY(hipMemcpyAsync(denoised, dn, fw * F * 4, hipMemcpyDeviceToHost, P.s));
    PYR_TRY(hipStreamSynchronize(P.s));
    return VBM3D_OK;
}

}  // namespace
}  // namespace vb

using namespace vb;

extern "C" {

int vbm3d_pyr_levels(int rows, int cols, int levels, int* lrows, int* lcols) {
    if (rows < 1 || cols < 1 || levels < 1 || !lrows || !lcols) return ctx_fail(VBM3D_ERR_ARG, "invalid arguments");
    std::vector<int> lr, lc;
    level_sizes(rows, cols, levels, lr, lc);
    for (int i = 0; i < levels; i++) {
        lrows[i] = lr[i];
        lcols[i] = lc[i];
    }
    return VBM3D_OK;
}

int vbm3d_pyr_decompose(vbm3d_ctx* ctx, const float* img, int rows, int cols, int ch, int levels, int type, float* out) {
    int rc = check_image(rows, cols, ch, levels, type);
    if (rc) return rc;
    if (!img || !out) return ctx_fail(VBM3D_ERR_ARG, "null buffer");
    Pyr P;
    if ((rc = pyr_open(ctx, P, pyr_bytes(rows, cols, ch)))) return rc;
    const size_t n = (size_t)ch * rows * cols, nl = level_words(rows, cols, ch, levels);
    Dev D;
    float* di = D.get(n);
    float* dout = D.get(nl);
    if (!di || !dout) return ctx_fail(VBM3D_ERR_NOMEM, "device allocation failed");
    PYR_TRY(hipMemcpyAsync(di, img, n * 4, hipMemcpyHostToDevice, P.s));
    if ((rc = decompose_dev(P, di, rows, cols, ch, levels, type, level_ptrs(dout, rows, cols, ch, levels, 0)))) return rc;
    PYR_TRY(hipMemcpyAsync(out, dout, nl * 4, hipMemcpyDeviceToHost, P.s));
    PYR_TRY(hipStreamSynchronize(P.s));
    return VBM3D_OK;
}

int vbm3d_pyr_recompose(vbm3d_ctx* ctx, const float* levels_in, int rows, int cols, int ch, int levels, int type,
                        float factor, float* out) {
    int rc = check_image(rows, cols, ch, levels, type);
    if (rc) return rc;
    if (!levels_in || !out) return ctx_fail(VBM3D_ERR_ARG, "null buffer");
    Pyr P;
    if ((rc = pyr_open(ctx, P, pyr_bytes(rows, cols, ch)))) return rc;
    const size_t n = (size_t)ch * rows * cols, nl = level_words(rows, cols, ch, levels);
    Dev D;
    float* dl = D.get(nl);
    float* dout = D.get(n);
    if (!dl || !dout) return ctx_fail(VBM3D_ERR_NOMEM, "device allocation failed");
    PYR_TRY(hipMemcpyAsync(dl, levels_in, nl * 4, hipMemcpyHostToDevice, P.s));
    if ((rc = recompose_dev(P, level_ptrs((const float*)dl, rows, cols, ch, levels, 0), rows, cols, ch, levels, type,
                           factor, dout))) return rc;
    PYR_TRY(hipMemcpyAsync(out, dout, n * 4, hipMemcpyDeviceToHost, P.s));
    PYR_TRY(hipStreamSynchronize(P.s));
    return VBM3D_OK;
}

int vbm3d_pyr_merge_coarse(vbm3d_ctx* ctx, const float* fine, int rows, int cols, const float* coarse, int crows,
                           int ccols, int ch, float factor, float* out) {
    int rc = check_image(rows, cols, ch, 1, 0);
    if (rc) return rc;
    if ((rc = check_image(crows, ccols, ch, 1, 0))) return rc;
    if (!fine || !coarse || !out) return ctx_fail(VBM3D_ERR_ARG, "null buffer");
    // the copied block must lie inside both images (merge_coarse.cpp:39-45)
    int bh = 0, bw = 0;
    while ((float)bh < crows * factor) bh++;
    while ((float)bw < ccols * factor) bw++;
    if (bh > crows || bw > ccols || bh > rows || bw > cols)
        return ctx_fail(VBM3D_ERR_ARG, "the coarse image's block does not fit (factor too large)");
    Pyr P;
    if ((rc = pyr_open(ctx, P, pyr_bytes(rows, cols, ch) + pyr_bytes(crows, ccols, ch)))) return rc;
    const size_t n = (size_t)ch * rows * cols, nc = (size_t)ch * crows * ccols;
    Dev D;
    float* df = D.get(n);
    float* dc = D.get(nc);
    if (!df || !dc) return ctx_fail(VBM3D_ERR_NOMEM, "device allocation failed");
    PYR_TRY(hipMemcpyAsync(df, fine, n * 4, hipMemcpyHostToDevice, P.s));
    PYR_TRY(hipMemcpyAsync(dc, coarse, nc * 4, hipMemcpyHostToDevice, P.s));
    if ((rc = dct2(P, df, rows, cols, ch, false))) return rc;
    if (bh > 0 && bw > 0 &&
        (rc = dct2(P, dc, crows, ccols, df, rows, cols, bh, bw, crows, ccols, ch, false)))
        return rc;
    if ((rc = dct2(P, df, rows, cols, ch, true))) return rc;
    PYR_TRY(hipMemcpyAsync(out, df, n * 4, hipMemcpyDeviceToHost, P.s));
    PYR_TRY(hipStreamSynchronize(P.s));
    return VBM3D_OK;
}

int vbm3d_multiscale_denoise(vbm3d_ctx* ctx, float sigma, const float* noisy, unsigned W, unsigned H, unsigned F,
                             unsigned C, const vbm3d_params* p1, const vbm3d_params* p2, int levels, int type,
                             float factor, int color_space, int ref_grid_nb, float* denoised, float* noisy_levels,
                             float* denoised_levels) {
    const int rc = multiscale_denoise(ctx, sigma, noisy, W, H, F, C, p1, p2, levels, type, factor, color_space, ref_grid_nb,
                                      denoised, noisy_levels, denoised_levels);
    // a call that failed midway leaves no copy on the caller's buffers behind
    if (rc && ctx) (void)hipStreamSynchronize(ctx_stream(ctx));
    if (ctx) ctx_multiscale_trim(ctx, kMultiscaleKeep);
    return rc;
}

}  // extern "C"
