// flow.hip -- CDNA4 (gfx950) TV-L1 optical flow, the reference's flow
// companion (tvl1flow/tvl1flow_lib.c; Zach, Pock and Bischof 2007 with
// Chambolle's dual projection), and its C-ABI entry points.
//
// The pyramid runs as element-wise and stencil kernels over [ny][nx] float
// planes in HBM, one thread per pixel; the primal-dual iterations run
// several per launch on regions held in registers and LDS.  Every kernel
// evaluates the reference's expressions in its order and precision -- float
// where it stores float, double where its expressions promote (Gaussian taps
// and sums, bicubic cells, the normalisation, 1.0 + taut * |grad|) -- with no
// FMA contraction and IEEE-correct division and square root, so each pixel's
// value is the reference's sequential value.  The one reduction, the mean squared
// change that stops the iterations, is summed in double in a fixed order;
// the reference sums it in float, which can only move the stopping
// iteration when the two sums straddle epsilon^2.
//
// The iterations never return to the host one by one: a control word in
// device memory says where a level stands, every launch reads it, does what
// comes next and leaves the word for the launch after it, and the host
// enqueues launches and looks at the word now and then.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <type_traits>
#include <vector>

#include "vbm3d_hip.h"

#pragma clang fp contract(off)

struct vbm3d_ctx;

namespace vb {
// context access, defined in capi.hip
hipStream_t ctx_stream(vbm3d_ctx* c);
int ctx_device(vbm3d_ctx* c);
hipError_t ctx_flow_workspace(vbm3d_ctx* c, size_t bytes, void** p);
int ctx_fail(int code, const std::string& msg);
}  // namespace vb

namespace vb {
namespace {

constexpr int kMaxIter = 300;     // MAX_ITERATIONS (tvl1flow_lib.c:22)
constexpr int kMaxTaps = 64;      // Gaussian half-window bound of this implementation
constexpr int BX = 64, BY = 4;    // pixel blocks: one wavefront per row segment

struct Taps {
    double b[kMaxTaps];
    int size;
};

// The flow's state planes of one side of the ping-pong.
struct FlowState {
    float *u1, *u2, *p11, *p12, *p21, *p22;
};

// Where a level stands; every launch of k_level_step reads one word and
// leaves the next launch's.
enum { kWarp, kStart, kRun, kDone };
struct FlowCtl {
    int phase;  // kWarp: set up `warp`; kStart: its first iterations; kRun: test
                // the last launch's iterations, then go on; kDone: level solved
    int warp;   // warp at hand
    int iter;   // its iterations so far (those not yet tested included)
    int steps;  // kRun: iterations of the last launch
    int cur;    // which state holds the flow and the dual field
    int stop;   // large levels: k_level_test's result for those iterations
};

__device__ __forceinline__ int clampi(int x, int n, bool& out) {
    if (x < 0) {
        out = true;
        return 0;
    }
    if (x >= n) {
        out = true;
        return n - 1;
    }
    return x;
}

// Catmull-Rom cell (tvl1flow/bicubic_interpolation.c:120-131), double.
__device__ __forceinline__ double cell(double v0, double v1, double v2, double v3, double x) {
    const double c3 = 3.0 * (v1 - v2) + v3 - v0;
    const double c2 = 2.0 * v0 - 5.0 * v1 + 4.0 * v2 - v3 + x * c3;
    return v1 + 0.5 * x * (v2 - v0 + x * c2);
}

// The 4x4 neighbourhood of (uu, vv) with Neumann clamping; the row below
// the sample is clamped with the x direction's sign, as the reference
// does (bicubic_interpolation.c:156-232).  Returns false when a clamp
// happened (the sample lies outside).
struct Nbhd {
    int cx[4], cy[4];
    double fx, fy;
};
__device__ __forceinline__ bool nbhd(float uu, float vv, int nx, int ny, Nbhd& n) {
    const int sx = uu < 0 ? -1 : 1, sy = vv < 0 ? -1 : 1;
    bool out = false;
    const int iu = (int)uu, iv = (int)vv;
    const int x = clampi(iu, nx, out), y = clampi(iv, ny, out);
    n.cx[0] = clampi(iu - sx, nx, out);
    n.cy[0] = clampi(iv - sx, ny, out);
    n.cx[1] = x;
    n.cy[1] = y;
    n.cx[2] = clampi(iu + sx, nx, out);
    n.cy[2] = clampi(iv + sy, ny, out);
    n.cx[3] = clampi(iu + 2 * sx, nx, out);
    n.cy[3] = clampi(iv + 2 * sy, ny, out);
    n.fx = (double)(uu - (float)x);
    n.fy = (double)(vv - (float)y);
    return !out;
}

__device__ __forceinline__ float interp(const float* __restrict__ in, int nx, const Nbhd& n) {
    double col[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        col[c] = cell(in[n.cx[c] + nx * n.cy[0]], in[n.cx[c] + nx * n.cy[1]], in[n.cx[c] + nx * n.cy[2]],
                      in[n.cx[c] + nx * n.cy[3]], n.fy);
    return (float)cell(col[0], col[1], col[2], col[3], n.fx);
}

// ---- normalisation to [0, 255] by the joint range (tvl1flow_lib.c:341-376)
__global__ void k_minmax(const float* __restrict__ a, const float* __restrict__ b, long n, float* part) {
    float mn0 = INFINITY, mx0 = -INFINITY, mn1 = INFINITY, mx1 = -INFINITY;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        mn0 = fminf(mn0, a[i]);
        mx0 = fmaxf(mx0, a[i]);
        mn1 = fminf(mn1, b[i]);
        mx1 = fmaxf(mx1, b[i]);
    }
    for (int o = 32; o >= 1; o >>= 1) {
        mn0 = fminf(mn0, __shfl_xor(mn0, o, 64));
        mx0 = fmaxf(mx0, __shfl_xor(mx0, o, 64));
        mn1 = fminf(mn1, __shfl_xor(mn1, o, 64));
        mx1 = fmaxf(mx1, __shfl_xor(mx1, o, 64));
    }
    __shared__ float s[4][4];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s[w][0] = mn0;
        s[w][1] = mx0;
        s[w][2] = mn1;
        s[w][3] = mx1;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < (int)(blockDim.x >> 6); q++) {
            s[0][0] = fminf(s[0][0], s[q][0]);
            s[0][1] = fmaxf(s[0][1], s[q][1]);
            s[0][2] = fminf(s[0][2], s[q][2]);
            s[0][3] = fmaxf(s[0][3], s[q][3]);
        }
        for (int k = 0; k < 4; k++) part[blockIdx.x * 4 + k] = s[0][k];
    }
}

__global__ void k_normalize(const float* __restrict__ a, const float* __restrict__ b, float* oa, float* ob, long n,
                            const float* __restrict__ part, int nparts) {
    float mn = INFINITY, mx = -INFINITY;
    for (int q = 0; q < nparts; q++) {
        mn = fminf(mn, fminf(part[4 * q], part[4 * q + 2]));
        mx = fmaxf(mx, fmaxf(part[4 * q + 1], part[4 * q + 3]));
    }
    const float den = mx - mn;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        if (den > 0) {
            oa[i] = (float)(255.0 * (a[i] - mn) / den);
            ob[i] = (float)(255.0 * (b[i] - mn) / den);
        } else {
            oa[i] = a[i];
            ob[i] = b[i];
        }
    }
}

// ---- separable Gaussian, reflecting edges, double taps and sums
// (tvl1flow/mask.c:234-337): a line of n samples extended by `size` on
// each side, the left mirror excluding the edge sample, the right one
// including it.
__device__ __forceinline__ int reflect(int e, int n) { return e < 0 ? -e : (e >= n ? 2 * n - e - 1 : e); }

__global__ void k_gauss_rows(const float* __restrict__ in, float* out, int nx, int ny, Taps t) {
    const int j = blockIdx.x * BX + threadIdx.x, i = blockIdx.y * BY + threadIdx.y;
    if (j >= nx || i >= ny) return;
    const float* row = in + (size_t)i * nx;
    double sum = t.b[0] * (double)row[j];
    for (int k = 1; k < t.size; k++) sum += t.b[k] * ((double)row[reflect(j - k, nx)] + (double)row[reflect(j + k, nx)]);
    out[(size_t)i * nx + j] = (float)sum;
}

__global__ void k_gauss_cols(const float* __restrict__ in, float* out, int nx, int ny, Taps t) {
    const int j = blockIdx.x * BX + threadIdx.x, i = blockIdx.y * BY + threadIdx.y;
    if (j >= nx || i >= ny) return;
    double sum = t.b[0] * (double)in[(size_t)i * nx + j];
    for (int k = 1; k < t.size; k++)
        sum += t.b[k] * ((double)in[(size_t)reflect(i - k, ny) * nx + j] + (double)in[(size_t)reflect(i + k, ny) * nx + j]);
    out[(size_t)i * nx + j] = (float)sum;
}

// ---- bicubic resampling of a level (zoom.c:44-117): output (j1, i1)
// samples the input at (j1 / fx, i1 / fy); k_upsample then multiplies a flow
// by the 1 / zfactor of tvl1flow_lib.c:453-457.
__global__ void k_resample(const float* __restrict__ in, float* out, int nx, int ny, int nxx, int nyy, float fx,
                           float fy) {
    const int j1 = blockIdx.x * BX + threadIdx.x, i1 = blockIdx.y * BY + threadIdx.y;
    if (j1 >= nxx || i1 >= nyy) return;
    const float i2 = (float)i1 / fy, j2 = (float)j1 / fx;
    Nbhd n;
    (void)nbhd(j2, i2, nx, ny, n);
    out[(size_t)i1 * nxx + j1] = interp(in, nx, n);
}

// Both components of a flow, multiplied by `scale`: from state s0 or, at a
// solved level (ctl not null), from the state that holds it
__global__ void k_upsample(const FlowCtl* __restrict__ ctl, FlowState s0, FlowState s1, float* o1, float* o2, int nx,
                           int ny, int nxx, int nyy, float fx, float fy, float scale) {
    const int j1 = blockIdx.x * BX + threadIdx.x, i1 = blockIdx.y * BY + threadIdx.y;
    if (j1 >= nxx || i1 >= nyy) return;
    const FlowState& s = ctl && ctl->cur ? s1 : s0;
    const float i2 = (float)i1 / fy, j2 = (float)j1 / fx;
    Nbhd n;
    (void)nbhd(j2, i2, nx, ny, n);
    o1[(size_t)i1 * nxx + j1] = interp(s.u1, nx, n) * scale;
    o2[(size_t)i1 * nxx + j1] = interp(s.u2, nx, n) * scale;
}

// The solved flow of the finest level
__global__ void k_flow_out(const FlowCtl* __restrict__ ctl, FlowState s0, FlowState s1, float* u, float* v, long n) {
    const FlowState& s = ctl->cur ? s1 : s0;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        u[i] = s.u1[i];
        v[i] = s.u2[i];
    }
}

// ---- centred gradient with one-sided edges (mask.c:144-214)
// and the control word of a new level
__global__ void k_cgrad(const float* __restrict__ in, float* dx, float* dy, int nx, int ny, FlowCtl* ctl) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && threadIdx.y == 0) *ctl = FlowCtl{kWarp, 0, 0, 0, 0, 0};
    const int j = blockIdx.x * BX + threadIdx.x, i = blockIdx.y * BY + threadIdx.y;
    if (j >= nx || i >= ny) return;
    const size_t k = (size_t)i * nx + j;
    const size_t jl = j > 0 ? k - 1 : k, jr = j < nx - 1 ? k + 1 : k;
    const size_t iu = i > 0 ? k - nx : k, id = i < ny - 1 ? k + nx : k;
    dx[k] = (float)(0.5 * (double)(in[jr] - in[jl]));
    dy[k] = (float)(0.5 * (double)(in[id] - in[iu]));
}

// ---- one warp's set-up at a pixel (tvl1flow_lib.c:150-166): the target image and
// its derivatives at the flow-displaced positions (zero outside), |grad|^2
// and the constant part of the linearised residual.
__device__ __forceinline__ void warp_px(const float* __restrict__ I0, const float* __restrict__ I1,
                                        const float* __restrict__ I1x, const float* __restrict__ I1y, float u1,
                                        float u2, float* wx, float* wy, float* grad, float* rho_c, int i, int j,
                                        int nx, int ny) {
    const size_t p = (size_t)i * nx + j;
    const float uu = (float)j + u1, vv = (float)i + u2;
    Nbhd n;
    float w = 0.f, gx = 0.f, gy = 0.f;
    if (nbhd(uu, vv, nx, ny, n)) {
        w = interp(I1, nx, n);
        gx = interp(I1x, nx, n);
        gy = interp(I1y, nx, n);
    }
    const float Ix2 = gx * gx, Iy2 = gy * gy;
    wx[p] = gx;
    wy[p] = gy;
    grad[p] = Ix2 + Iy2;
    rho_c[p] = w - gx * u1 - gy * u2 - I0[p];
}

// ---- the primal-dual iterations (tvl1flow_lib.c:168-252)
//
// What one iteration does at a pixel is a stencil of radius 1 on the flow
// (u1, u2) and the dual field (p11, p12, p21, p22): the primal step needs
// the dual field at the left and upper neighbours, the dual step the new
// flow at the right and lower ones.  Run one launch per step, an iteration
// was three launches and 88 bytes of traffic per pixel.  Here a workgroup
// takes an RX x RY region into LDS and runs T iterations on it; the outer
// T pixels of the region go stale, one ring per iteration, and only the
// inside is written, to the other state of a ping-pong.  The stopping test
// needs the mean squared change of every iteration: each launch leaves its
// iterations' sums per workgroup, the next launch adds them up (every
// workgroup the same sums in the same order) and knows whether the warp
// had converged inside the last launch.  If it had, and not at its last
// iteration, that launch ran too far: the iterations up to the stopping
// one are run again from the state it started from, which the ping-pong
// still holds.  So the flow and the iteration counts are those of the
// one-by-one form.  What bounds it: instruction issue on large levels (two
// double-precision roots and five divisions per pixel and iteration),
// the latency of the chain load, test, iterations, store on small ones.
// Measured: a 1920x1080 pair 18.6 -> 7.5 ms, a 317x241 pair 8.7 -> 2.7 ms.

// Backward-difference divergence with the reference's edge cases
// (mask.c:39-90) at a pixel that is first / last in its row (L, R) and
// column (T, B), from the two components, the left neighbour of the first
// and the upper neighbour of the second.
template <bool EDGE>
__device__ __forceinline__ float div_px(float v1, float v1l, float v2, float v2u, unsigned edge) {
    if (!EDGE || edge == 0) return (v1 - v1l) + (v2 - v2u);
    const bool L = edge & 1, R = edge & 2, T = edge & 4, B = edge & 8;
    const float h = L ? v1 : (R ? -v1l : v1 - v1l);
    if (T) return h + v2;
    if (B) return h - v2u;
    return h + v2 - v2u;
}

// Thresholding towards the data term (tvl1flow_lib.c:170-212): the
// auxiliary flow at a pixel.
__device__ __forceinline__ void threshold_px(float a, float b, float gx, float gy, float g, float rc, float l_t,
                                             float& v1, float& v2) {
    const float rho = rc + (gx * a + gy * b);
    float d1, d2;
    if (rho < -l_t * g) {
        d1 = l_t * gx;
        d2 = l_t * gy;
    } else if (rho > l_t * g) {
        d1 = -l_t * gx;
        d2 = -l_t * gy;
    } else if ((double)g < 1E-10) {
        d1 = d2 = 0.f;
    } else {
        const float fi = -rho / g;
        d1 = fi * gx;
        d2 = fi * gy;
    }
    v1 = a + d1;
    v2 = b + d2;
}

// The projected dual update of one flow component (tvl1flow_lib.c:233-252)
// from its forward gradient.  |grad| is taken in double: the squares of
// floats are exact, so one rounding of their sum and one of the root; as a
// float this is the C library's hypot.  The sum 1.0 + taut |grad| in double,
// rounded to float, is the float sum: it is exact in double wherever it
// differs from 1.
__device__ __forceinline__ void dual_px(float& pa, float& pb, float ux, float uy, float taut) {
    const float g = (float)sqrt(__builtin_fma((double)ux, (double)ux, (double)uy * (double)uy));
    const float ng = 1.0f + taut * g;
    pa = (pa + taut * ux) / ng;
    pb = (pb + taut * uy) / ng;
}

// Sum over a wavefront in a fixed order on the DPP network (quad swaps,
// half-row and row mirrors, the row-15 and lane-31 broadcasts): lane 63
// holds it.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xF, false);
    return v + __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_sum(double v) {
    v = dpp_add<0xB1, 0xF>(v);
    v = dpp_add<0x4E, 0xF>(v);
    v = dpp_add<0x141, 0xF>(v);
    v = dpp_add<0x140, 0xF>(v);
    v = dpp_add<0x142, 0xA>(v);
    return dpp_add<0x143, 0xC>(v);
}

struct LevelArgs {
    FlowCtl* ctl;     // [2], by launch parity
    double* part;     // [2][T][blocks] sums of squared changes
    FlowState st[2];
    const float *I0, *I1, *I1x, *I1y;
    const float *u1, *u2;  // the level's initial flow
    float *wx, *wy, *grad, *rho;
    int nx, ny, nwarps;
    float l_t, theta, taut, size, eps2;
    int* counts;  // iterations of each warp
};

// Whether `steps` <= T iterations ending at iteration `iter`, with sums in
// part [step][nblk], hold the warp's last one: its index, or -1.  The
// wavefronts of a workgroup of NT threads share the steps; each sum is
// formed in a fixed order.  s: NT / 64 doubles.  Every thread gets it.
template <int NT, int T>
__device__ int stop_step(const LevelArgs& a, const double* __restrict__ part, int nblk, int steps, int iter, double* s) {
    constexpr int WPS = NT / 64 / T;  // wavefronts per step
    static_assert(WPS >= 1, "a wavefront per step");
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, k = w / WPS;
    double acc = 0.0;
    if (k < steps)
        for (int q = (w - k * WPS) * 64 + lane; q < nblk; q += WPS * 64) acc += part[(size_t)k * nblk + q];
    acc = wave_sum(acc);
    if (lane == 63) s[w] = acc;
    __syncthreads();
    for (int q = 0; q < steps; q++) {
        double t = 0.0;
        for (int r = 0; r < WPS; r++) t += s[q * WPS + r];
        float err = (float)t;
        err /= a.size;
        if (!(err > a.eps2) || iter - steps + q + 1 >= kMaxIter) return q;
    }
    return -1;
}

// The test as a launch of its own, for levels of more than kTestBlocks
// workgroups: there every workgroup of the next launch adding up all sums
// reads more than the level itself (3,672 workgroups at 1920x1080: 323 MB a
// launch).
constexpr int kTestBlocks = 256;
template <int T>
__global__ __launch_bounds__(1024) void k_level_test(LevelArgs a, int par, int nblk) {
    __shared__ double s_sum[16];
    const FlowCtl c = a.ctl[par];
    if (c.phase != kRun) return;
    const int k = stop_step<1024, T>(a, a.part + (size_t)(par ^ 1) * T * nblk, nblk, c.steps, c.iter, s_sum);
    if (threadIdx.x == 0) a.ctl[par].stop = k;
}

template <int RX, int RY, int NT, int T>
__global__ __launch_bounds__(NT) void k_level_step(LevelArgs a, int par) {
    constexpr int PX = RX * RY / NT, UX = RX - 2 * T, UY = RY - 2 * T;
    static_assert(RX * RY % NT == 0 && UX > 0 && UY > 0, "whole pixels per thread");
    __shared__ float s_u1[RX * RY], s_u2[RX * RY], s_p11[RX * RY], s_p12[RX * RY], s_p21[RX * RY], s_p22[RX * RY];
    __shared__ double s_sum[NT / 64], s_err[T][NT / 64];
    const int t = threadIdx.x;
    const int nblk = gridDim.x * gridDim.y, blk = blockIdx.y * gridDim.x + blockIdx.x;
    const FlowCtl c = a.ctl[par];
    FlowCtl next = c;
    int steps = 0, src = c.cur;  // iterations to run, from state src into the other
    bool setup = false;          // or set the warp up
    if (c.phase == kWarp) {
        setup = true;
        next.phase = kStart;
    } else if (c.phase == kRun) {
        const int k = nblk > kTestBlocks
                          ? c.stop
                          : stop_step<NT, T>(a, a.part + (size_t)(par ^ 1) * T * nblk, nblk, c.steps, c.iter, s_sum);
        if (k >= 0) {
            if (blk == 0 && t == 0) a.counts[c.warp] = c.iter - c.steps + k + 1;
            next.warp = c.warp + 1;
            next.phase = next.warp == a.nwarps ? kDone : kWarp;
            if (k + 1 < c.steps) {
                steps = k + 1;  // again, up to the stopping iteration
                src = c.cur ^ 1;
            } else if (next.phase == kWarp) {
                setup = true;
                next.phase = kStart;
            }
        }
    }
    if (c.phase == kStart || next.phase == kRun) {
        next.iter = c.phase == kStart ? 0 : c.iter;
        next.steps = steps = min(T, kMaxIter - next.iter);
        next.iter += steps;
        next.phase = kRun;
        next.cur = src ^ 1;
    }
    if (blk == 0 && t == 0) a.ctl[par ^ 1] = next;
    const int nx = a.nx, ny = a.ny;
    const int x0 = (int)blockIdx.x * UX - T, y0 = (int)blockIdx.y * UY - T;  // the region's corner
    if (setup) {
        // the flow displaces from state `cur`; the level's first warp takes
        // its initial flow and a zero dual field into state 0
        const FlowState& st = a.st[c.cur];
        const bool first = next.warp == 0;
        for (int q = t; q < UX * UY; q += NT) {
            const int j = x0 + T + q % UX, i = y0 + T + q / UX;
            if (j >= nx || i >= ny) continue;
            const size_t p = (size_t)i * nx + j;
            const float u = first ? a.u1[p] : st.u1[p], v = first ? a.u2[p] : st.u2[p];
            if (first) {
                st.u1[p] = u;
                st.u2[p] = v;
                st.p11[p] = st.p12[p] = st.p21[p] = st.p22[p] = 0.f;
            }
            warp_px(a.I0, a.I1, a.I1x, a.I1y, u, v, a.wx, a.wy, a.grad, a.rho, i, j, nx, ny);
        }
        return;
    }
    if (steps == 0) return;  // done
    const FlowState& in = a.st[src];
    const FlowState& out = a.st[src ^ 1];
    const bool test = next.phase == kRun;
    float u1[PX], u2[PX], p11[PX], p12[PX], p21[PX], p22[PX], gx[PX], gy[PX], g[PX], rc[PX];
    unsigned flags[PX];  // edge bits, 16: in the image, 32: written
#pragma unroll
    for (int q = 0; q < PX; q++) {
        const int li = t + q * NT, lx = li % RX, ly = li / RX, j = x0 + lx, i = y0 + ly;
        flags[q] = 0;
        u1[q] = u2[q] = p11[q] = p12[q] = p21[q] = p22[q] = gx[q] = gy[q] = g[q] = rc[q] = 0.f;
        if (j >= 0 && i >= 0 && j < nx && i < ny) {
            const size_t p = (size_t)i * nx + j;
            u1[q] = in.u1[p];
            u2[q] = in.u2[p];
            p11[q] = in.p11[p];
            p12[q] = in.p12[p];
            p21[q] = in.p21[p];
            p22[q] = in.p22[p];
            gx[q] = a.wx[p];
            gy[q] = a.wy[p];
            g[q] = a.grad[p];
            rc[q] = a.rho[p];
            flags[q] = 16u | (j == 0 ? 1u : 0u) | (j == nx - 1 ? 2u : 0u) | (i == 0 ? 4u : 0u) | (i == ny - 1 ? 8u : 0u);
            if (lx >= T && lx < RX - T && ly >= T && ly < RY - T) flags[q] |= 32u;
        }
        s_p11[li] = p11[q];
        s_p12[li] = p12[q];
        s_p21[li] = p21[q];
        s_p22[li] = p22[q];
    }
    __syncthreads();
    double es[T] = {};  // this thread's squared changes per iteration
    auto iterate = [&](auto edge_t) {
        constexpr bool EDGE = decltype(edge_t)::value;
#pragma unroll 1
        for (int k = 0; k < steps; k++) {
            double e = 0.0;
#pragma unroll
            for (int q = 0; q < PX; q++) {
                const int li = t + q * NT, ll = max(li - 1, 0), lu = li < RX ? li : li - RX;
                float v1, v2;
                threshold_px(u1[q], u2[q], gx[q], gy[q], g[q], rc[q], a.l_t, v1, v2);
                const float n1 = v1 + a.theta * div_px<EDGE>(p11[q], s_p11[ll], p12[q], s_p12[lu], flags[q] & 15u);
                const float n2 = v2 + a.theta * div_px<EDGE>(p21[q], s_p21[ll], p22[q], s_p22[lu], flags[q] & 15u);
                if (flags[q] & 32u)
                    e += (double)((n1 - u1[q]) * (n1 - u1[q]) + (n2 - u2[q]) * (n2 - u2[q]));
                u1[q] = n1;
                u2[q] = n2;
                s_u1[li] = n1;
                s_u2[li] = n2;
            }
#pragma unroll
            for (int r = 0; r < T; r++) es[r] = k == r ? e : es[r];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < PX; q++) {
                const int li = t + q * NT, lr = min(li + 1, RX * RY - 1), ld = li >= RX * (RY - 1) ? li : li + RX;
                const bool nr = EDGE && (flags[q] & 2u), nd = EDGE && (flags[q] & 8u);
                dual_px(p11[q], p12[q], nr ? 0.f : s_u1[lr] - u1[q], nd ? 0.f : s_u1[ld] - u1[q], a.taut);
                dual_px(p21[q], p22[q], nr ? 0.f : s_u2[lr] - u2[q], nd ? 0.f : s_u2[ld] - u2[q], a.taut);
                s_p11[li] = p11[q];
                s_p12[li] = p12[q];
                s_p21[li] = p21[q];
                s_p22[li] = p22[q];
            }
            __syncthreads();
        }
    };
    if (x0 > 0 && y0 > 0 && x0 + RX < nx && y0 + RY < ny) iterate(std::false_type{});
    else iterate(std::true_type{});
    if (test) {
#pragma unroll
        for (int k = 0; k < T; k++) {
            const double e = wave_sum(es[k]);
            if ((t & 63) == 63) s_err[k][t >> 6] = e;
        }
        __syncthreads();
    }
    if (test && t < steps) {
        double acc = 0.0;
        for (int q = 0; q < NT / 64; q++) acc += s_err[t][q];
        a.part[((size_t)par * T + t) * nblk + blk] = acc;
    }
#pragma unroll
    for (int q = 0; q < PX; q++) {
        if (!(flags[q] & 32u)) continue;
        const int li = t + q * NT;
        const size_t p = (size_t)(y0 + li / RX) * nx + x0 + li % RX;
        out.u1[p] = u1[q];
        out.u2[p] = u2[q];
        out.p11[p] = p11[q];
        out.p12[p] = p12[q];
        out.p21[p] = p21[q];
        out.p22[p] = p22[q];
    }
}

__global__ void k_fill(float* p, long n, float v) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

// Gaussian taps (mask.c:246-264), on the host with the C library's exp.
Taps make_taps(double sigma) {
    Taps t{};
    const double den = 2 * sigma * sigma;
    t.size = (int)(5 * sigma) + 1;
    if (t.size > kMaxTaps) return t;
    for (int i = 0; i < t.size; i++) t.b[i] = 1 / (sigma * std::sqrt(2.0 * 3.1415926)) * std::exp(-i * i / den);
    double norm = 0;
    for (int i = 0; i < t.size; i++) norm += t.b[i];
    norm *= 2;
    norm -= t.b[0];
    for (int i = 0; i < t.size; i++) t.b[i] /= norm;
    return t;
}

dim3 grid2(int nx, int ny) { return dim3((unsigned)((nx + BX - 1) / BX), (unsigned)((ny + BY - 1) / BY)); }

// The region and iterations per launch of k_level_step, 512 threads.  A level
// whose 32 x 16 regions fit a round of the chip (kTestBlocks workgroups) is
// bound by the latency of an iteration: one pixel per thread, about 2.3 us an
// iteration with the launch (32 x 32 regions, 4 iterations: 3.1).  A larger
// one is bound by instruction issue and the halo's share: two pixels per
// thread of a 32 x 32 region, 4 iterations, 93 us a launch at 1920x1080
// (the small form 77 for 3; 64 x 32 regions 116, 64 x 48 97, 64 x 64 101).
struct StepShape {
    int rx, ry, t;
};
constexpr int kStepNT = 512;
constexpr StepShape kSmallStep = {32, 16, 3}, kLargeStep = {32, 32, 4};
dim3 step_grid(const StepShape& sh, int nx, int ny) {
    const int ux = sh.rx - 2 * sh.t, uy = sh.ry - 2 * sh.t;
    return dim3((unsigned)((nx + ux - 1) / ux), (unsigned)((ny + uy - 1) / uy));
}
bool small_step(int nx, int ny) {
    const dim3 g = step_grid(kSmallStep, nx, ny);
    return (size_t)g.x * g.y <= (size_t)kTestBlocks;
}
// doubles of the sums of a level (two parities)
size_t step_sums(int nx, int ny) {
    const StepShape& sh = small_step(nx, ny) ? kSmallStep : kLargeStep;
    const dim3 g = step_grid(sh, nx, ny);
    return 2 * (size_t)sh.t * g.x * g.y;
}

hipError_t launch_step(const LevelArgs& a, int par, hipStream_t s) {
    if (small_step(a.nx, a.ny)) {
        constexpr StepShape S = kSmallStep;
        hipLaunchKernelGGL((k_level_step<S.rx, S.ry, kStepNT, S.t>), step_grid(S, a.nx, a.ny), dim3(kStepNT), 0, s, a,
                           par);
    } else {
        constexpr StepShape S = kLargeStep;
        const dim3 g = step_grid(S, a.nx, a.ny);
        if (g.x * g.y > (unsigned)kTestBlocks)
            hipLaunchKernelGGL((k_level_test<S.t>), dim3(1), dim3(1024), 0, s, a, par, (int)(g.x * g.y));
        hipLaunchKernelGGL((k_level_step<S.rx, S.ry, kStepNT, S.t>), g, dim3(kStepNT), 0, s, a, par);
    }
    return hipGetLastError();
}

struct Level {
    int nx, ny;
    float *I0, *I1, *u1, *u2;
};

#define FLOW_TRY(expr)                                                                       \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess) return ctx_fail(VBM3D_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

int gauss(float* img, float* tmp, int nx, int ny, double sigma, hipStream_t s) {
    const Taps t = make_taps(sigma);
    if (t.size > kMaxTaps) return ctx_fail(VBM3D_ERR_UNSUPPORTED, "Gaussian window too large");
    if (t.size >= nx || t.size >= ny)
        return ctx_fail(VBM3D_ERR_ARG, "image too small for its Gaussian window (" + std::to_string(nx) + "x" +
                                           std::to_string(ny) + ", half-width " + std::to_string(t.size) + ")");
    hipLaunchKernelGGL(k_gauss_rows, grid2(nx, ny), dim3(BX, BY), 0, s, img, tmp, nx, ny, t);
    hipLaunchKernelGGL(k_gauss_cols, grid2(nx, ny), dim3(BX, BY), 0, s, tmp, img, nx, ny, t);
    FLOW_TRY(hipGetLastError());
    return VBM3D_OK;
}

void zoom_size(int nx, int ny, int* nxx, int* nyy, float factor) {
    *nxx = (int)((float)nx * factor + 0.5);
    *nyy = (int)((float)ny * factor + 0.5);
}

}  // namespace

// The whole multiscale flow on device buffers (tvl1flow_lib.c:384-485).
int tvl1_device(vbm3d_ctx* ctx, const float* I0, const float* I1, float* u, float* v, int nx, int ny,
                const vbm3d_tvl1_params* prm, int* iters) {
    const float tau = prm->tau, lambda = prm->lambda, theta = prm->theta, zf = prm->zfactor, eps = prm->epsilon;
    const int nscales = prm->nscales, fscale = prm->fscale, warps = prm->nwarps;
    if (nx < 2 || ny < 2) return ctx_fail(VBM3D_ERR_ARG, "images must be at least 2x2");
    if (nscales < 1 || fscale < 0 || fscale >= nscales || warps < 1 || !(zf > 0.f && zf < 1.f) || !(theta > 0.f) ||
        !(tau > 0.f))
        return ctx_fail(VBM3D_ERR_ARG, "invalid TV-L1 parameters");
    if ((long)nx * ny > (1L << 30)) return ctx_fail(VBM3D_ERR_ARG, "image too large");
    hipStream_t s = ctx_stream(ctx);
    // level sizes and workspace: levels 0..nscales-1 (images; flows of
    // levels >= 1), then the per-level work planes at the finest size
    std::vector<Level> L(nscales);
    L[0].nx = nx;
    L[0].ny = ny;
    for (int k = 1; k < nscales; k++) {
        zoom_size(L[k - 1].nx, L[k - 1].ny, &L[k].nx, &L[k].ny, zf);
        if (L[k].nx < 2 || L[k].ny < 2) return ctx_fail(VBM3D_ERR_ARG, "too many scales for the image size");
    }
    const size_t n0 = (size_t)nx * ny;
    size_t words = 0;
    for (int k = 0; k < nscales; k++) words += (size_t)L[k].nx * L[k].ny * (k == 0 ? 2 : 4);
    // the step launches' sums
    size_t nparts = 0;
    for (int k = fscale; k < nscales; k++) nparts = std::max(nparts, step_sums(L[k].nx, L[k].ny));
    const size_t work_planes = 19;  // I1x I1y wx wy grad rho_c tmp, two states of six planes
    // planes, then the iterations' sums, the min/max partials, the control
    // words and the iteration counts, each 256-byte aligned
    const size_t bytes = (words + work_planes * n0) * 4 + nparts * 8 + 256 * 4 + 4096 + (size_t)nscales * warps * 4;
    void* base = nullptr;
    if (ctx_flow_workspace(ctx, bytes, &base) != hipSuccess)
        return ctx_fail(VBM3D_ERR_NOMEM, "device allocation of the flow workspace failed");
    float* f = (float*)base;
    for (int k = 0; k < nscales; k++) {
        const size_t sz = (size_t)L[k].nx * L[k].ny;
        L[k].I0 = f;
        f += sz;
        L[k].I1 = f;
        f += sz;
        if (k == 0) {
            L[k].u1 = u;
            L[k].u2 = v;
        } else {
            L[k].u1 = f;
            f += sz;
            L[k].u2 = f;
            f += sz;
        }
    }
    float *I1x = f, *I1y = f + n0, *wx = f + 2 * n0, *wy = f + 3 * n0, *grad = f + 4 * n0, *rho = f + 5 * n0;
    float* tmp = f + 6 * n0;
    FlowState st[2];
    for (int q = 0; q < 2; q++) {
        float* b = f + (7 + 6 * q) * n0;
        st[q] = FlowState{b, b + n0, b + 2 * n0, b + 3 * n0, b + 4 * n0, b + 5 * n0};
    }
    f += work_planes * n0;
    double* part = (double*)(((uintptr_t)f + 255) & ~(uintptr_t)255);
    float* mm = (float*)(part + nparts);  // 64 workgroups x 4 min/max partials
    FlowCtl* ctl = (FlowCtl*)(((uintptr_t)(mm + 256) + 255) & ~(uintptr_t)255);
    int* counts = (int*)(ctl + 2);  // iterations, [level][warp]

    // normalisation and 0.8-sigma pre-smoothing (tvl1flow_lib.c:416-421)
    hipLaunchKernelGGL(k_minmax, dim3(64), dim3(256), 0, s, I0, I1, (long)n0, mm);
    hipLaunchKernelGGL(k_normalize, dim3(1024), dim3(256), 0, s, I0, I1, L[0].I0, L[0].I1, (long)n0, mm, 64);
    FLOW_TRY(hipGetLastError());
    int rc;
    if ((rc = gauss(L[0].I0, tmp, nx, ny, 0.8, s)) != VBM3D_OK) return rc;
    if ((rc = gauss(L[0].I1, tmp, nx, ny, 0.8, s)) != VBM3D_OK) return rc;
    // the pyramid (zoom.c:44-83): smooth a copy, resample
    const double zsig = (float)(0.6 * std::sqrt(1.0 / (zf * zf) - 1.0));
    for (int k = 1; k < nscales; k++) {
        const size_t sz = (size_t)L[k - 1].nx * L[k - 1].ny;
        for (int img = 0; img < 2; img++) {
            float* src = img ? L[k - 1].I1 : L[k - 1].I0;
            float* dst = img ? L[k].I1 : L[k].I0;
            FLOW_TRY(hipMemcpyAsync(wx, src, sz * 4, hipMemcpyDeviceToDevice, s));
            if ((rc = gauss(wx, tmp, L[k - 1].nx, L[k - 1].ny, zsig, s)) != VBM3D_OK) return rc;
            hipLaunchKernelGGL(k_resample, grid2(L[k].nx, L[k].ny), dim3(BX, BY), 0, s, wx, dst, L[k - 1].nx,
                               L[k - 1].ny, L[k].nx, L[k].ny, zf, zf);
        }
    }
    const long ncoarse = (long)L[nscales - 1].nx * L[nscales - 1].ny;
    hipLaunchKernelGGL(k_fill, dim3(256), dim3(256), 0, s, L[nscales - 1].u1, ncoarse, 0.f);
    hipLaunchKernelGGL(k_fill, dim3(256), dim3(256), 0, s, L[nscales - 1].u2, ncoarse, 0.f);
    FLOW_TRY(hipGetLastError());

    const float inv = (float)1.0 / zf, l_t = lambda * theta, taut = tau / theta, eps2 = eps * eps;
    auto upsample = [&](int k, bool solved) -> int {
        const float fx = (float)L[k - 1].nx / L[k].nx, fy = (float)L[k - 1].ny / L[k].ny;
        const FlowState plain{L[k].u1, L[k].u2, nullptr, nullptr, nullptr, nullptr};
        hipLaunchKernelGGL(k_upsample, grid2(L[k - 1].nx, L[k - 1].ny), dim3(BX, BY), 0, s, solved ? ctl : nullptr,
                           solved ? st[0] : plain, st[1], L[k - 1].u1, L[k - 1].u2, L[k].nx, L[k].ny, L[k - 1].nx,
                           L[k - 1].ny, fx, fy, inv);
        FLOW_TRY(hipGetLastError());
        return VBM3D_OK;
    };
    int level = 0;
    for (int k = nscales - 1; k >= fscale; k--, level++) {
        const int lx = L[k].nx, ly = L[k].ny;
        const long sz = (long)lx * ly;
        // one level (tvl1flow_lib.c:96-305)
        hipLaunchKernelGGL(k_cgrad, grid2(lx, ly), dim3(BX, BY), 0, s, L[k].I1, I1x, I1y, lx, ly, ctl);
        FLOW_TRY(hipGetLastError());
        const LevelArgs la{ctl, part, {st[0], st[1]}, L[k].I0, L[k].I1, I1x, I1y, L[k].u1, L[k].u2, wx, wy, grad, rho,
                           lx, ly, warps, l_t, theta, taut, (float)sz, eps2, counts + (size_t)level * warps};
        // The launches follow one another without the host; it looks at the
        // control word now and then and stops once the level is solved
        // (launches past that end at once).  The first batch covers a set-up
        // and about five step launches per warp.
        FlowCtl host_ctl{};
        int par = 0;
        for (int batch = 7 * warps;; batch = 16) {
            batch = (batch + 1) & ~1;  // the word read below is ctl[0]
            for (int it = 0; it < batch; it++, par ^= 1) FLOW_TRY(launch_step(la, par, s));
            FLOW_TRY(hipMemcpyAsync(&host_ctl, ctl, sizeof(FlowCtl), hipMemcpyDeviceToHost, s));
            FLOW_TRY(hipStreamSynchronize(s));
            if (host_ctl.phase == kDone) break;
        }
        if (k == 0) {
            hipLaunchKernelGGL(k_flow_out, dim3(1024), dim3(256), 0, s, ctl, st[0], st[1], u, v, (long)n0);
            FLOW_TRY(hipGetLastError());
            break;
        }
        if ((rc = upsample(k, true)) != VBM3D_OK) return rc;
    }
    for (int k = fscale - 1; k >= 1; k--)
        if ((rc = upsample(k, false)) != VBM3D_OK) return rc;
    if (iters)
        FLOW_TRY(hipMemcpyAsync(iters, counts, (size_t)(nscales - fscale) * warps * 4, hipMemcpyDeviceToHost, s));
    FLOW_TRY(hipStreamSynchronize(s));
    return VBM3D_OK;
}

}  // namespace vb

extern "C" {

void vbm3d_tvl1_default_params(vbm3d_tvl1_params* p) {
    // tvl1flow/main.c:20-30
    p->tau = 0.25f;
    p->lambda = 0.15f;
    p->theta = 0.3f;
    p->nscales = 100;
    p->fscale = 0;
    p->zfactor = 0.5f;
    p->nwarps = 5;
    p->epsilon = 0.01f;
}

int vbm3d_tvl1_nscales(int nx, int ny, float zfactor, int nscales) {
    // tvl1flow/main.c:139-146
    const float N = (float)(1 + std::log(std::hypot((double)nx, (double)ny) / 16.0) / std::log((double)(1 / zfactor)));
    if (N < nscales) nscales = (int)N;
    return nscales;
}

int vbm3d_tvl1_flow_device(vbm3d_ctx* ctx, const float* d_I0, const float* d_I1, float* d_u, float* d_v, int nx,
                           int ny, const vbm3d_tvl1_params* prm, int* iters) {
    if (!ctx || !d_I0 || !d_I1 || !d_u || !d_v || !prm) return vb::ctx_fail(VBM3D_ERR_ARG, "null argument");
    if (hipSetDevice(vb::ctx_device(ctx)) != hipSuccess) return vb::ctx_fail(VBM3D_ERR_HIP, "hipSetDevice failed");
    return vb::tvl1_device(ctx, d_I0, d_I1, d_u, d_v, nx, ny, prm, iters);
}

int vbm3d_tvl1_flow(vbm3d_ctx* ctx, const float* I0, const float* I1, float* u, float* v, int nx, int ny,
                    const vbm3d_tvl1_params* prm, int* iters) {
    if (!ctx || !I0 || !I1 || !u || !v || !prm) return vb::ctx_fail(VBM3D_ERR_ARG, "null argument");
    if (nx < 2 || ny < 2 || (long)nx * ny > (1L << 30)) return vb::ctx_fail(VBM3D_ERR_ARG, "invalid image size");
    if (hipSetDevice(vb::ctx_device(ctx)) != hipSuccess) return vb::ctx_fail(VBM3D_ERR_HIP, "hipSetDevice failed");
    const size_t n = (size_t)nx * ny;
    float* d = nullptr;
    if (hipMalloc(&d, n * 4 * 4) != hipSuccess) return vb::ctx_fail(VBM3D_ERR_NOMEM, "device allocation failed");
    hipStream_t s = vb::ctx_stream(ctx);
    int rc = VBM3D_OK;
    if (hipMemcpyAsync(d, I0, n * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(d + n, I1, n * 4, hipMemcpyHostToDevice, s) != hipSuccess)
        rc = vb::ctx_fail(VBM3D_ERR_HIP, "upload failed");
    if (rc == VBM3D_OK) rc = vb::tvl1_device(ctx, d, d + n, d + 2 * n, d + 3 * n, nx, ny, prm, iters);
    if (rc == VBM3D_OK &&
        (hipMemcpyAsync(u, d + 2 * n, n * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
         hipMemcpyAsync(v, d + 3 * n, n * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
         hipStreamSynchronize(s) != hipSuccess))
        rc = vb::ctx_fail(VBM3D_ERR_HIP, "download failed");
    (void)hipStreamSynchronize(s);
    (void)hipFree(d);
    return rc;
}

}  // extern "C"
