// kernels_filter.hip -- CDNA4 (gfx950) group filtering of the VBM3D
// collaborative filter (2D transforms, transform along the group,
// shrinkage, inverse transforms) and its step-2 adjoint: one wavefront per
// reference patch; lane = coefficient position, the group dimension lives
// in registers.
//
// Every kernel reproduces the reference's FP32 operation order so that the
// GPU result is bit-identical to the sequential CPU restatement:
//   * no FMA contraction (file-wide pragma + -ffp-contract=off);
//   * float sums accumulated sequentially in the reference's index order;
//   * IEEE-correct float division (hipcc's default);
//   * the Haar butterflies multiply a float sum by a double constant and
//     round once to float, as src/lib_transforms.cpp:468-469 does.
#include "kernels_common.h"

#pragma clang fp contract(off)

namespace vb {
namespace {

// ---------------------------------------------------------------------
// Group filtering.
// ---------------------------------------------------------------------
// Column of (member n, coefficient kk) in row kk of the Wiener v^2 buffer:
// n rotated by kk / (64 / NS), so that the 64 lanes' stores of one n fall
// in 64 distinct banks while each row stays contiguous.
template <int NS>
__host__ __device__ constexpr int v2_col(int kk, int n) {
    return (n + (kk >> (NS == 1 ? 6 : NS == 2 ? 5 : NS == 4 ? 4 : NS == 8 ? 3 : 2))) & (NS - 1);
}

// 1D transform along the group and shrinkage for one channel
// (ht_filtering_haar/_hadamard src/vbm3d.cpp:1405-1521,
// wiener_filtering_haar/_hadamard :1539-1666).  Lane kk holds coefficient
// kk of every group member: zg/eg are [n][64].  Step 1 returns the
// aggregation weight (valid in every lane); step 2 stores value^2 of
// (n, kk) in row kk of v2, at column v2_col for the weight sum done
// afterwards in the reference's flat order n + kk*nSx (wiener_sum).
template <int K, int NS, int STEP>
__device__ float shrink(float* zg, float* eg, float* v2, int lane, bool had, float lambda,
                        float sig) {
    constexpr int K2 = K * K;
    const bool act = lane < K2;
    float z[NS], e[NS];
#pragma unroll
    for (int n = 0; n < NS; n++) {
        z[n] = act ? zg[n * K2 + lane] : 0.f;
        if (STEP == 2) e[n] = act ? eg[n * K2 + lane] : 0.f;
    }
    float weight = 0.f;
    if (STEP == 1) {
        t3_fwd<NS>(z, had);
        const float thr = had ? lambda * sig * sqrtf((float)NS) : lambda * sig;
        int cnt = 0;
#pragma unroll
        for (int n = 0; n < NS; n++) {
            const bool keep = act && ((n == 0 && lane == 0) || fabsf(z[n]) > thr);
            if (keep) cnt++;
            else z[n] = 0.f;
        }
        cnt = wave_sum_i32(cnt);
        t3_inv<NS>(z, had);
        if (had) {
            const float coef = 1.0f / (float)NS;
#pragma unroll
            for (int n = 0; n < NS; n++) z[n] *= coef;
        }
        weight = 1.f / (sig * sig * (float)cnt);
#pragma unroll
        for (int n = 0; n < NS; n++)
            if (act) zg[n * K2 + lane] = z[n];
    } else {
        t3_fwd<NS>(z, had);
        t3_fwd<NS>(e, had);
        const float s2 = sig * sig;
        const float coef = 1.0f / (float)NS;
#pragma unroll
        for (int n = 0; n < NS; n++) {
            float value = e[n] * e[n];
            if (had) value = value * coef;
            value /= (value + s2);
            e[n] = had ? z[n] * value * coef : z[n] * value;
            if (act) v2[lane * NS + v2_col<NS>(lane, n)] = value * value;
        }
        t3_inv<NS>(e, had);
#pragma unroll
        for (int n = 0; n < NS; n++)
            if (act) eg[n * K2 + lane] = e[n];
    }
    return weight;
}

// Sequential float sum of channel c's v^2 over the flat index
// f = n + kk*nSx (src/vbm3d.cpp:1651).  Rows are NS words, read 16 bytes
// at a time; the rotation undone here is v2_col's.
template <int K, int NS>
__device__ __forceinline__ float wiener_sum(const float* vc) {
    constexpr int K2 = K * K;
    float acc = 0.f;
#pragma unroll
    for (int kk = 0; kk < K2; kk++) {
        float x[NS];
        if constexpr (NS >= 4) {
#pragma unroll
            for (int j = 0; j < NS / 4; j++) {
                const float4 q = *(const float4*)(vc + kk * NS + 4 * j);
                x[4 * j] = q.x;
                x[4 * j + 1] = q.y;
                x[4 * j + 2] = q.z;
                x[4 * j + 3] = q.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < NS; j++) x[j] = vc[kk * NS + j];
        }
#pragma unroll
        for (int n = 0; n < NS; n++) acc = acc + x[v2_col<NS>(kk, n)];
    }
    return acc;
}

// Per-wavefront LDS layout of k_filter (4-byte words): transposes, zg,
// eg, then one v^2 buffer per channel, each region 16-byte aligned.
__host__ __device__ constexpr int round4(int v) { return (v + 3) & ~3; }
// Whether the filtered members of a group leave through one staged copy
// (filter_one): three channels whose planes are not whole cache lines.
__host__ __device__ constexpr bool stage_est(int K, int C, int step) { return step == 2 && C == 3 && (K * K) % 32 != 0; }
// Words from one staged member to the next: the padded member, and 4 more
// so that the members' stores fall in different LDS banks.
__host__ __device__ constexpr int stage_pitch(int K, int C) { return (C * K * K + 31) / 32 * 32 + 4; }
// Words before the v^2 buffers: transposes, zg and eg, over which the
// staged members go.
__host__ __device__ constexpr int filter_front(int K, int C, int N, int step) {
    const int w = round4((64 / K) * xstride(K)) + (step == 2 ? 2 : 1) * round4(N * K * K);
    const int st = stage_est(K, C, step) ? (N < 64 / K ? N : 64 / K) * stage_pitch(K, C) : 0;
    return w > st ? w : st;
}
__host__ __device__ inline int filter_lds_words(int K, int C, int N, int step) {
    return filter_front(K, C, N, step) + (step == 2 ? C * round4(K * K * N) : 0);
}

// Channel sigma without a dynamically indexed array (a private array
// would live in scratch memory).
template <class A>
__device__ __forceinline__ float sig_of(const A& a, int c) {
    return c == 0 ? a.sig[0] : (c == 1 ? a.sig[1] : a.sig[2]);
}

template <int K, int C, int STEP, class A>
__device__ __forceinline__ void filter_one(const A& a, const long r, float* X, const int lane) {
    constexpr int K2 = K * K;
    constexpr int PB = 64 / K;           // patches per lane batch
    constexpr int XS = xstride(K), XP = K + 1;
    // X: [PB][XS] transposes, then the group buffers
    const int gw = round4(a.N * K2);               // group buffer words
    float* zg = X + round4(PB * XS);               // [N][K2]
    float* eg = zg + gw;                           // [N][K2] (step 2)
    float* v2 = X + filter_front(K, C, a.N, STEP);  // [C][gw] (step 2)
    const unsigned t = (unsigned)(r / a.nrf), i = (unsigned)(r - (long)t * a.nrf);
    const unsigned slot = __builtin_amdgcn_readfirstlane((t % a.ring) * a.nrf + i);
    const unsigned W = a.W, wh = a.wh, whc = a.whc;
    const int nsx = (int)__builtin_amdgcn_readfirstlane(a.nsx[slot]);
    const bool bior = a.T2D == 1;
    const bool had = a.T3D == 2;
    const uint32_t* mem = a.idx + (size_t)slot * a.N;
    const Div32 dW = {a.dW.m, a.dW.s1, a.dW.s2}, dWHC = {a.dWHC.m, a.dWHC.s1, a.dWHC.s2};
    typedef const __attribute__((address_space(4))) float cfloat;
    const cfloat* TF = (const cfloat*)(bior ? a.tabs->biorF : a.tabs->dctF);
    const cfloat* TI = (const cfloat*)(bior ? a.tabs->biorI : a.tabs->dctI);
    const cfloat* NRM = (const cfloat*)a.tabs->nrm;
    const cfloat* INV = (const cfloat*)a.tabs->inv;
    const float dct_out = a.tabs->dct_out;
    const int nl = lane / K, rr = lane - nl * K;    // batch patch, row / column index
    const bool lact = lane < PB * K;
    // Staged members: the outputs of channels 0 and 1 stay in registers until
    // the group's members go out together, each padded to whole cache lines
    // (a member in one lane batch; the unpadded ring of the scratch array
    // takes the plain stores).
    constexpr bool STG = stage_est(K, C, STEP);
    const bool stg = STG && nsx <= PB && a.ms == stage_pitch(K, C) - 4;
    float held[STG ? C - 1 : 1][K];
    float wsel = 0.f;  // step 1: lane c ends with channel c's weight
    // mb0: offset of row rr of member nl, the lane's row in the first lane
    // batch (its index is read whether or not the member exists, so that
    // the load does not wait for the group size; every slot holds N
    // entries).  The first batch's row of each (channel, source) pair is
    // fetched one pair ahead of its use.
    auto decode = [&](unsigned mi) {
        const unsigned pt = div32(mi, dWHC);
        const unsigned py = div32(mi - pt * whc, dW), px = mi - pt * whc - py * W;
        return pt * whc + (py + rr) * W + px;
    };
    const unsigned mb0 = decode(mem[min(nl, a.N - 1)]);
    const bool act0 = lact && nl < nsx;
    float xn[K];
    auto fetch = [&](int c, int g) {
        if (act0) {
            const float* row = (g == 0 ? a.noisy : a.basic) + mb0 + c * wh;
#pragma unroll
            for (int q = 0; q < K; q++) xn[q] = row[q];
        }
    };
    fetch(0, 0);

    for (int c = 0; c < C; c++) {
        // ---- forward 2D transforms of all members (bior_2d_forward
        //      src/lib_transforms.cpp:125-181; DCT src/vbm3d.cpp:1245-1302)
        for (int g = 0; g < (STEP == 2 ? 2 : 1); g++) {
            const float* src = g == 0 ? a.noisy : a.basic;
            float* dst = g == 0 ? zg : eg;
            for (int nb0 = 0; nb0 < nsx; nb0 += PB) {
                const int n = nb0 + nl;
                const bool act = lact && n < nsx;
                if (act) {
                    float x[K];
                    if (nb0 == 0) {
                        // the first batch's row was fetched ahead; fetch the
                        // next (channel, source) row while this one is used
#pragma unroll
                        for (int q = 0; q < K; q++) x[q] = xn[q];
                        if (STEP == 2 && g == 0) fetch(c, 1);
                        else if (c + 1 < C) fetch(c + 1, 0);
                    } else {
                        const float* row = src + decode(mem[n]) + c * wh;
#pragma unroll
                        for (int q = 0; q < K; q++) x[q] = row[q];
                    }
                    // pass 1 along the row: t[v] = sum_q x[q] M[v][q]
                    if (bior) {
#pragma unroll
                        for (int v = 0; v < K; v++) {
                            float m = 0.f;
#pragma unroll
                            for (int q = 0; q < K; q++) m = m + x[q] * TF[v * K + q];
                            X[nl * XS + v * XP + rr] = m;  // stored transposed
                        }
                    } else {
                        float y[K];
                        dct_fwd_pass<K>(x, y, TF);
#pragma unroll
                        for (int v = 0; v < K; v++) X[nl * XS + v * XP + rr] = y[v];
                    }
                }
                wave_sync();
                if (act) {
                    // pass 2 down column rr of t
                    float col[K];
#pragma unroll
                    for (int p = 0; p < K; p++) col[p] = X[nl * XS + rr * XP + p];
                    // BIOR keeps out[i*8+j] = (column i, output j); the DCT
                    // writes out[u*K+v] scaled by coef_norm
                    if (bior) {
#pragma unroll
                        for (int u = 0; u < K; u++) {
                            float m = 0.f;
#pragma unroll
                            for (int p = 0; p < K; p++) m = m + col[p] * TF[u * K + p];
                            dst[n * K2 + rr * 8 + u] = m;
                        }
                    } else {
                        float y[K];
                        dct_fwd_pass<K>(col, y, TF);
#pragma unroll
                        for (int u = 0; u < K; u++) dst[n * K2 + u * K + rr] = y[u] * NRM[u * K + rr];
                    }
                }
                wave_sync();
            }
        }
        // ---- 1D transform along the group, shrinkage, inverse
        float* v2c = v2 + c * gw;
        const float sgc = sig_of(a, c);
        float wc;
        switch (nsx) {
            case 1: wc = shrink<K, 1, STEP>(zg, eg, v2c, lane, had, a.lambda, sgc); break;
            case 2: wc = shrink<K, 2, STEP>(zg, eg, v2c, lane, had, a.lambda, sgc); break;
            case 4: wc = shrink<K, 4, STEP>(zg, eg, v2c, lane, had, a.lambda, sgc); break;
            case 8: wc = shrink<K, 8, STEP>(zg, eg, v2c, lane, had, a.lambda, sgc); break;
            default: wc = shrink<K, 16, STEP>(zg, eg, v2c, lane, had, a.lambda, sgc); break;
        }
        if (lane == c) wsel = wc;
        wave_sync();
        // ---- inverse 2D transforms (bior_2d_inverse src/lib_transforms.cpp:
        //      270-321; dct_2d_inv src/vbm3d.cpp:1678-1713), store [n][pixel].
        //      A member's outputs replace its coefficients in LDS (pass 1
        //      of its batch has read them all), and the group's planes then
        //      leave in contiguous 256-byte stores.
        //      Three channels of 7x7 planes are not whole cache lines: there
        //      the members are staged (held, stage_est) and leave in 16-byte
        //      stores of whole lines, so that the aggregation reads 5 lines
        //      per member instead of the 7.5 of separate planes.
        float* est = STEP == 2 ? eg : zg;
        float* dstg = a.est + (size_t)slot * (unsigned)(a.N * a.ms) + c * K2;
        for (int nb0 = 0; nb0 < nsx; nb0 += PB) {
            const int n = nb0 + nl;
            const bool act = lact && n < nsx;
            if (act) {
                float x[K];
#pragma unroll
                for (int s2 = 0; s2 < K; s2++)
                    x[s2] = bior ? est[n * K2 + s2 * 8 + rr] : est[n * K2 + rr * K + s2] * INV[rr * K + s2];
                if (bior) {
#pragma unroll
                    for (int v = 0; v < K; v++) {
                        float m = 0.f;
#pragma unroll
                        for (int q = 0; q < K; q++) m = m + x[q] * TI[v * K + q];
                        X[nl * XS + v * XP + rr] = m;
                    }
                } else {
                    float y[K];
                    dct_inv_pass<K>(x, y, TI);
#pragma unroll
                    for (int v = 0; v < K; v++) X[nl * XS + v * XP + rr] = y[v];
                }
            }
            wave_sync();
            if (act) {
                float col[K];
#pragma unroll
                for (int p = 0; p < K; p++) col[p] = X[nl * XS + rr * XP + p];
                // BIOR: pixel (row u, column rr); DCT: pixel (row u, column
                // rr) after the 1/(2k) factor
                if (bior) {
#pragma unroll
                    for (int u = 0; u < K; u++) {
                        float m = 0.f;
#pragma unroll
                        for (int p = 0; p < K; p++) m = m + col[p] * TI[u * K + p];
                        est[n * K2 + u * K + rr] = m;
                    }
                } else {
                    float y[K];
                    dct_inv_pass<K>(col, y, TI);
                    if (stg) {
                        if (c == C - 1) {
                            // X and the group buffers are no longer read
                            // (one lane batch: col is in registers)
                            wave_sync();
#pragma unroll
                            for (int u = 0; u < K; u++) {
                                float* m = X + n * stage_pitch(K, C) + u * K + rr;
#pragma unroll
                                for (int h = 0; h < C - 1; h++) m[h * K2] = held[STG ? h : 0][u];
                                m[(C - 1) * K2] = dct_out * y[u];
                            }
                        } else {
#pragma unroll
                            for (int u = 0; u < K; u++) {
                                const float o = dct_out * y[u];
                                if (c == 0) held[0][u] = o;
                                else held[STG ? 1 : 0][u] = o;
                            }
                        }
                    } else {
#pragma unroll
                        for (int u = 0; u < K; u++) est[n * K2 + u * K + rr] = dct_out * y[u];
                    }
                }
            }
            wave_sync();
        }
        if (stg) {
            if (c < C - 1) continue;
            constexpr int M4 = (stage_pitch(K, C) - 4) / 4;  // 16-byte pieces of a member
            float4* g4 = (float4*)(a.est + (size_t)slot * (unsigned)(a.N * a.ms));
            for (int j = lane; j < nsx * M4; j += 64) {
                const int n = j / M4;
                g4[j] = *(const float4*)(X + n * stage_pitch(K, C) + 4 * (j - n * M4));
            }
            continue;
        }
        for (int j = lane; j < nsx * K2; j += 64) {
            const int n = j / K2;
            dstg[n * a.ms + (j - n * K2)] = est[j];
        }
        wave_sync();  // read before the next channel's transforms refill it
    }
    if (STEP == 2) {
        // Wiener weights: sequential float sums over the flat index
        // (src/vbm3d.cpp:1651), one lane per channel
        wave_sync();
        if (lane < C) {
            const float* vc = v2 + lane * gw;
            float acc;
            switch (nsx) {
                case 1: acc = wiener_sum<K, 1>(vc); break;
                case 2: acc = wiener_sum<K, 2>(vc); break;
                case 4: acc = wiener_sum<K, 4>(vc); break;
                case 8: acc = wiener_sum<K, 8>(vc); break;
                default: acc = wiener_sum<K, 16>(vc); break;
            }
            const float sg = sig_of(a, lane), s2 = sg * sg;
            float wgt;
            if (had) wgt = acc > 0.0f ? 1.0f / (s2 * acc) : 1.0f;
            else wgt = 1.f / (s2 * acc);
            a.wgt[(size_t)slot * C + lane] = wgt;
        }
    } else if (lane < C) {
        a.wgt[(size_t)slot * C + lane] = wsel;
    }
}

template <int K, int C, int STEP>
__global__ __launch_bounds__(256) void k_filter(FArgs a) {
    extern __shared__ float smem[];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
    const long r = a.r_begin + (long)xcd_order(blockIdx.x, gridDim.x) * nw + w;
    if (r >= a.r_end) return;
    filter_one<K, C, STEP>(a, r, smem + (size_t)w * filter_lds_words(K, C, a.N, STEP), lane);
}

// One item per wave over a batch: global wave g takes item g, so the
// hardware's workgroup dispatch order is the queue.
template <int K, int C, int STEP>
__global__ __launch_bounds__(256) void k_filter_multi(const FArgs* __restrict__ jobs, WorkQueue q, int words) {
    extern __shared__ float smem[];
    const int lane = threadIdx.x & 63;
    const long g = uniform_long((long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if (g >= q.total) return;
    const int j = queue_job(q, g);
    typedef const __attribute__((address_space(4))) FArgs cFA;
    cFA& a = ((cFA*)jobs)[j];
    filter_one<K, C, STEP>(a, a.r_begin + (g - uniform_long(q.item_begin[j])),
                           smem + (size_t)(threadIdx.x >> 6) * words, lane);
}

template <int K, int C, int STEP>
__global__ __launch_bounds__(256) void k_filter_queue(const FArgs* __restrict__ jobs, WorkQueue q, int words) {
    extern __shared__ float smem[];
    const int lane = threadIdx.x & 63;
    float* X = smem + (size_t)(threadIdx.x >> 6) * words;
    typedef const __attribute__((address_space(4))) FArgs cFA;
    int j = 0;
    long jb = 0, je = 0;
    long it0 = queue_take(q, lane);
    while (it0 < q.total) {
        const unsigned long long nxt = queue_issue(q, lane);
        const long it1 = min(q.total, it0 + (long)q.grab);
        for (long it = it0; it < it1; it++) {
            queue_seek(q, it, j, jb, je);
            cFA& a = ((cFA*)jobs)[j];  // scalar loads of the job
            filter_one<K, C, STEP>(a, a.r_begin + (it - jb), X, lane);
        }
        it0 = queue_value(nxt);
    }
}

// ---------------------------------------------------------------------
// Group filtering of temporal patches (kt > 1 slices at one position in
// consecutive frames; src/vbm3d.cpp:573-575, 589, 816-831, 1866-1956): the
// row-parallel form of filter_one over the (member, slice) pairs, with the
// temporal DCT of each coefficient's slices between the 2D transforms and
// the transform along the group, in the operation order of k_filter_gen.
// Bound by instruction issue and by the LDS of the Wiener weights' terms
// (17.7 KB per wavefront at k 7, kt 2, N 8, three channels).  8 RGB frames
// 320x240 at kt 2, against k_filter_gen, one lane per coefficient and a
// member slice at a time: step 2 6.38 -> 1.95 ms, step 1 0.34 -> 0.14.
// ---------------------------------------------------------------------
// Words of a v^2 row of ns members: one more, so that the lanes' rows start
// in different banks.
__host__ __device__ constexpr int kt_row(int ns) { return ns + 1; }
__host__ __device__ inline int filter_kt_words(int K, int C, int kt, int N, int step) {
    const int g = round4(N * K * K * kt);
    return round4((64 / K) * xstride(K)) + (step == 2 ? 2 : 1) * g +
           (step == 2 ? C * round4(K * K * kt * kt_row(N)) : 0) + round4(N * kt);
}

// shrink over K2t coefficients, several per lane; zg, eg are [n][K2t].
// Returns the number of kept coefficients (step 1).
template <int NS, int STEP>
__device__ int shrink_kt(float* zg, float* eg, float* v2, int K2t, int lane, bool had, float lambda, float sig) {
    const float coef = 1.0f / (float)NS;
    int cnt = 0;
    for (int kk = lane; kk < K2t; kk += 64) {
        float z[NS], e[NS];
#pragma unroll
        for (int n = 0; n < NS; n++) {
            z[n] = zg[n * K2t + kk];
            if (STEP == 2) e[n] = eg[n * K2t + kk];
        }
        t3_fwd<NS>(z, had);
        if (STEP == 1) {
            const float thr = had ? lambda * sig * sqrtf((float)NS) : lambda * sig;
#pragma unroll
            for (int n = 0; n < NS; n++) {
                if ((n == 0 && kk == 0) || fabsf(z[n]) > thr) cnt++;
                else z[n] = 0.f;
            }
            t3_inv<NS>(z, had);
#pragma unroll
            for (int n = 0; n < NS; n++) zg[n * K2t + kk] = had ? z[n] * coef : z[n];
        } else {
            t3_fwd<NS>(e, had);
            const float s2 = sig * sig;
#pragma unroll
            for (int n = 0; n < NS; n++) {
                float value = e[n] * e[n];
                if (had) value = value * coef;
                value /= (value + s2);
                e[n] = had ? z[n] * value * coef : z[n] * value;
                v2[kk * kt_row(NS) + n] = value * value;
            }
            t3_inv<NS>(e, had);
#pragma unroll
            for (int n = 0; n < NS; n++) eg[n * K2t + kk] = e[n];
        }
    }
    return STEP == 1 ? wave_sum_i32(cnt) : 0;
}

// Sequential sum of a channel's v^2 in the flat order n + kk * NS.
template <int NS>
__device__ float wiener_sum_kt(const float* v, int K2t) {
    float acc = 0.f;
#pragma unroll 4
    for (int kk = 0; kk < K2t; kk++)
#pragma unroll
        for (int n = 0; n < NS; n++) acc = acc + v[kk * kt_row(NS) + n];
    return acc;
}

template <int K, int C, int STEP>
__global__ __launch_bounds__(256) void k_filter_kt(FArgs a) {
    constexpr int K2 = K * K, PB = 64 / K, XS = xstride(K), XP = K + 1;
    extern __shared__ float smem[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long r = a.r_begin + (long)xcd_order(blockIdx.x, gridDim.x) * (blockDim.x >> 6) + w;
    if (r >= a.r_end) return;
    const int kt = a.kt, K2t = K2 * kt;
    float* X = smem + (size_t)w * filter_kt_words(K, C, kt, a.N, STEP);
    const int gw = round4(a.N * K2t), vw = round4(K2t * kt_row(a.N));
    float* zg = X + round4(PB * XS);     // [n][kt][K2]
    float* eg = zg + gw;                 // the same (step 2)
    float* v2 = eg + gw;                 // [C][vw] (step 2)
    unsigned* s_pos = (unsigned*)(STEP == 2 ? v2 + C * vw : zg + gw);  // [N * kt]
    const unsigned t = (unsigned)(r / a.nrf), i = (unsigned)(r - (long)t * a.nrf);
    const unsigned slot = __builtin_amdgcn_readfirstlane((t % a.ring) * a.nrf + i);
    const unsigned W = a.W, wh = a.wh, whc = a.whc;
    const int nsx = (int)__builtin_amdgcn_readfirstlane(a.nsx[slot]);
    const int npair = nsx * kt;  // pair = n * kt + slice
    const bool bior = a.T2D == 1, had = a.T3D == 2, temporal = !bior;
    const uint32_t* mem = a.idx + (size_t)slot * a.N;
    typedef const __attribute__((address_space(4))) float cfloat;
    const cfloat* TF = (const cfloat*)(bior ? a.tabs->biorF : a.tabs->dctF);
    const cfloat* TI = (const cfloat*)(bior ? a.tabs->biorI : a.tabs->dctI);
    const cfloat* NRM = (const cfloat*)a.tabs->nrm;
    const cfloat* INV = (const cfloat*)a.tabs->inv;
    const cfloat* tF = (const cfloat*)a.tabsg->tF;
    const cfloat* tI = (const cfloat*)a.tabsg->tI;
    const float tnorm = a.tabsg->tnorm, dct_out = a.tabs->dct_out;
    const Div32 dWHC = {a.dWHC.m, a.dWHC.s1, a.dWHC.s2};
    const int nl = lane / K, rr = lane - nl * K;
    const bool lact = lane < PB * K;
    float wsel = 0.f;
    // the pairs' corners, so that a batch's rows wait for no index load
    for (int pi = lane; pi < npair; pi += 64) {
        const int n = small_div(pi, kt);
        const unsigned mi = mem[n], pt = div32(mi, dWHC);
        s_pos[pi] = (pt + (unsigned)(pi - n * kt)) * whc + (mi - pt * whc);
    }
    wave_sync();
    for (int c = 0; c < C; c++) {
        for (int pb0 = 0; pb0 < npair; pb0 += PB) {
            const int pi = pb0 + nl;
            const bool act = lact && pi < npair;
            // both sources' rows are loaded before the first is used
            float x[STEP][K];
            if (act) {
                const size_t o = (size_t)s_pos[pi] + (size_t)c * wh + (size_t)rr * W;
#pragma unroll
                for (int g = 0; g < STEP; g++)
#pragma unroll
                    for (int q = 0; q < K; q++) x[g][q] = (g == 0 ? a.noisy : a.basic)[o + q];
            }
#pragma unroll
            for (int g = 0; g < STEP; g++) {
                float* dst = g == 0 ? zg : eg;
                if (act) {
                    if (bior) {
#pragma unroll
                        for (int v = 0; v < K; v++) {
                            float m = 0.f;
#pragma unroll
                            for (int q = 0; q < K; q++) m = m + x[g][q] * TF[v * K + q];
                            X[nl * XS + v * XP + rr] = m;
                        }
                    } else {
                        float y[K];
                        dct_fwd_pass<K>(x[g], y, TF);
#pragma unroll
                        for (int v = 0; v < K; v++) X[nl * XS + v * XP + rr] = y[v];
                    }
                }
                wave_sync();
                if (act) {
                    float col[K];
#pragma unroll
                    for (int p = 0; p < K; p++) col[p] = X[nl * XS + rr * XP + p];
                    if (bior) {
#pragma unroll
                        for (int u = 0; u < K; u++) {
                            float m = 0.f;
#pragma unroll
                            for (int p = 0; p < K; p++) m = m + col[p] * TF[u * K + p];
                            dst[pi * K2 + rr * 8 + u] = m;
                        }
                    } else {
                        float y[K];
                        dct_fwd_pass<K>(col, y, TF);
#pragma unroll
                        for (int u = 0; u < K; u++) dst[pi * K2 + u * K + rr] = y[u] * NRM[u * K + rr];
                    }
                }
                wave_sync();
            }
        }
        for (int g = 0; g < STEP; g++) {
            float* dst = g == 0 ? zg : eg;
            if (temporal) {  // along each coefficient's slices
                for (int e = lane; e < K2 * nsx; e += 64) {
                    const int n = e / K2;
                    float* x = dst + n * K2t + (e - n * K2);
                    float v[kGenMaxKt];
#pragma unroll
                    for (int q = 0; q < kGenMaxKt; q++) v[q] = q < kt ? x[q * K2] : 0.f;
#pragma unroll
                    for (int u = 0; u < kGenMaxKt; u++)
                        if (u < kt) {
                            float m = 0.f;
#pragma unroll
                            for (int q = 0; q < kGenMaxKt; q++)
                                if (q < kt) m = m + v[q] * tF[u * kt + q];
                            x[u * K2] = u == 0 ? (float)((double)(m * tnorm) * 0.7071067811865475) : m * tnorm;
                        }
                }
                wave_sync();
            }
        }
        float* v2c = v2 + c * vw;
        const float sg = sig_of(a, c);
        int cnt;
        switch (nsx) {
            case 1: cnt = shrink_kt<1, STEP>(zg, eg, v2c, K2t, lane, had, a.lambda, sg); break;
            case 2: cnt = shrink_kt<2, STEP>(zg, eg, v2c, K2t, lane, had, a.lambda, sg); break;
            case 4: cnt = shrink_kt<4, STEP>(zg, eg, v2c, K2t, lane, had, a.lambda, sg); break;
            case 8: cnt = shrink_kt<8, STEP>(zg, eg, v2c, K2t, lane, had, a.lambda, sg); break;
            default: cnt = shrink_kt<16, STEP>(zg, eg, v2c, K2t, lane, had, a.lambda, sg); break;
        }
        if (STEP == 1 && lane == c) wsel = 1.f / (sg * sg * (float)cnt);
        wave_sync();
        float* est = STEP == 2 ? eg : zg;
        if (temporal) {
            for (int e = lane; e < K2 * nsx; e += 64) {
                const int n = e / K2;
                float* x = est + n * K2t + (e - n * K2);
                float z[kGenMaxKt];
#pragma unroll
                for (int u = 0; u < kGenMaxKt; u++) z[u] = u < kt ? x[u * K2] : 0.f;
                z[0] = (float)((double)z[0] * 1.414213562373095);
#pragma unroll
                for (int q = 0; q < kGenMaxKt; q++)
                    if (q < kt) {
                        float m = 0.f;
#pragma unroll
                        for (int u = 0; u < kGenMaxKt; u++)
                            if (u < kt) m = m + z[u] * tI[q * kt + u];
                        x[q * K2] = m * tnorm;
                    }
            }
            wave_sync();
        }
        for (int pb0 = 0; pb0 < npair; pb0 += PB) {
            const int pi = pb0 + nl;
            const bool act = lact && pi < npair;
            if (act) {
                float x[K];
#pragma unroll
                for (int q = 0; q < K; q++)
                    x[q] = bior ? est[pi * K2 + q * 8 + rr] : est[pi * K2 + rr * K + q] * INV[rr * K + q];
                if (bior) {
#pragma unroll
                    for (int v = 0; v < K; v++) {
                        float m = 0.f;
#pragma unroll
                        for (int q = 0; q < K; q++) m = m + x[q] * TI[v * K + q];
                        X[nl * XS + v * XP + rr] = m;
                    }
                } else {
                    float y[K];
                    dct_inv_pass<K>(x, y, TI);
#pragma unroll
                    for (int v = 0; v < K; v++) X[nl * XS + v * XP + rr] = y[v];
                }
            }
            wave_sync();
            if (act) {
                float col[K];
#pragma unroll
                for (int p = 0; p < K; p++) col[p] = X[nl * XS + rr * XP + p];
                if (bior) {
#pragma unroll
                    for (int u = 0; u < K; u++) {
                        float m = 0.f;
#pragma unroll
                        for (int p = 0; p < K; p++) m = m + col[p] * TI[u * K + p];
                        est[pi * K2 + u * K + rr] = m;
                    }
                } else {
                    float y[K];
                    dct_inv_pass<K>(col, y, TI);
#pragma unroll
                    for (int u = 0; u < K; u++) est[pi * K2 + u * K + rr] = dct_out * y[u];
                }
            }
            wave_sync();
        }
        // est[slot][n][c][slice][pixel]
        float* dstg = a.est + (size_t)slot * (unsigned)(a.N * a.ms) + c * K2t;
        for (int n = 0; n < nsx; n++)
            for (int q = lane; q < K2t; q += 64) dstg[n * a.ms + q] = est[n * K2t + q];
        wave_sync();
    }
    if (STEP == 2) {
        if (lane < C) {
            const float* vc = v2 + lane * vw;
            float acc;
            switch (nsx) {
                case 1: acc = wiener_sum_kt<1>(vc, K2t); break;
                case 2: acc = wiener_sum_kt<2>(vc, K2t); break;
                case 4: acc = wiener_sum_kt<4>(vc, K2t); break;
                case 8: acc = wiener_sum_kt<8>(vc, K2t); break;
                default: acc = wiener_sum_kt<16>(vc, K2t); break;
            }
            const float sg = sig_of(a, lane), s2 = sg * sg;
            a.wgt[(size_t)slot * C + lane] = had ? (acc > 0.0f ? 1.0f / (s2 * acc) : 1.0f) : 1.f / (s2 * acc);
        }
    } else if (lane < C) {
        a.wgt[(size_t)slot * C + lane] = wsel;
    }
}

// ---------------------------------------------------------------------
// Adjoint of step 2 with the groups, Wiener gains and weights frozen by
// the basic estimate.  Step 2 is then linear in the noisy video:
//   final = D^-1 sum_g Agg_g (kaiser w_g) G T3^-1 V_g T3 F Gather_g z,
// so its transpose gathers u = grad / den, applies the transposes of the
// inverse 2D transform G, of the group operator (T3^-1 V T3)^T, which is
// T3^-1 V T3 again for the orthonormal Haar and for the symmetric
// Hadamard, and of the forward 2D transform F, scaled by w_g.  The
// per-member results go to `est`; the aggregation kernel in raw mode then
// sums them over every member patch covering a pixel.  These are plain
// FP32 evaluations of the transposed operators, not bit-replays of a
// reference computation.
//
// The 2D transforms run row-parallel like filter_one's: lane = (member,
// row), a pass along the row, a transpose through LDS, a pass down the
// column.  (One lane per coefficient, every member after the other, took
// 6.08 ms on 32 grey frames 640x360, the forward filter 1.67; this form
// takes 2.5.)  The aggregation weights are the forward pass's: read from
// its ring where that still holds the clip (a.wgt_kept), else summed again.
// ---------------------------------------------------------------------
// Group operator of one channel, transposed: Wiener gains from the basic
// coefficients eg, then T3^-1 V T3 applied to zg in place; v^2 to v2 (unless
// null) as shrink stores it.
template <int K, int NS>
__device__ void adj_group(float* zg, const float* eg, float* v2, int lane, bool had, float sig) {
    constexpr int K2 = K * K;
    const bool act = lane < K2;
    float z[NS], e[NS];
#pragma unroll
    for (int n = 0; n < NS; n++) {
        z[n] = act ? zg[n * K2 + lane] : 0.f;
        e[n] = act ? eg[n * K2 + lane] : 0.f;
    }
    t3_fwd<NS>(e, had);
    t3_fwd<NS>(z, had);
    const float s2 = sig * sig;
    const float coef = 1.0f / (float)NS;
#pragma unroll
    for (int n = 0; n < NS; n++) {
        float value = e[n] * e[n];
        if (had) value = value * coef;
        value /= (value + s2);
        z[n] = had ? z[n] * value * coef : z[n] * value;
        if (v2 && act) v2[lane * NS + v2_col<NS>(lane, n)] = value * value;
    }
    t3_inv<NS>(z, had);
#pragma unroll
    for (int n = 0; n < NS; n++)
        if (act) zg[n * K2 + lane] = z[n];
}

__host__ __device__ inline int adjoint_lds_words(int K, int N) {
    return round4((64 / K) * xstride(K)) + 3 * round4(N * K * K);
}

template <int K, int C>
__global__ __launch_bounds__(256) void k_filter_adjoint(FArgs a) {
    constexpr int K2 = K * K, PB = 64 / K, XS = xstride(K), XP = K + 1;
    extern __shared__ float smem[];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
    const long r = a.r_begin + (long)xcd_order(blockIdx.x, gridDim.x) * nw + w;
    if (r >= a.r_end) return;
    float* X = smem + (size_t)w * adjoint_lds_words(K, a.N);  // [PB][XS] transposes
    const int gw = round4(a.N * K2);
    float* zg = X + round4(PB * XS);  // [N][K2]
    float* eg = zg + gw;              // [N][K2]
    float* v2 = eg + gw;              // [K2*N]
    const unsigned t = (unsigned)(r / a.nrf), i = (unsigned)(r - (long)t * a.nrf);
    const unsigned slot = __builtin_amdgcn_readfirstlane((t % a.ring) * a.nrf + i);
    const unsigned W = a.W, wh = a.wh, whc = a.whc;
    const int nsx = (int)__builtin_amdgcn_readfirstlane(a.nsx[slot]);
    const bool bior = a.T2D == 1, had = a.T3D == 2;
    const uint32_t* mem = a.idx + (size_t)slot * a.N;
    const Div32 dW = {a.dW.m, a.dW.s1, a.dW.s2}, dWHC = {a.dWHC.m, a.dWHC.s1, a.dWHC.s2};
    typedef const __attribute__((address_space(4))) float cfloat;
    const cfloat* TF = (const cfloat*)(bior ? a.tabs->biorF : a.tabs->dctF);
    const cfloat* TI = (const cfloat*)(bior ? a.tabs->biorI : a.tabs->dctI);
    const cfloat* NRM = (const cfloat*)a.tabs->nrm;
    const cfloat* INV = (const cfloat*)a.tabs->inv;
    const cfloat* KAI = (const cfloat*)a.tabs->kaiser;
    const float dct_out = a.tabs->dct_out;
    const int nl = lane / K, rr = lane - nl * K;
    const bool lact = lane < PB * K;
    // t[v] = sum_q x[q] T[q][v] of a row, stored transposed; then its
    // column rr of the lane's member
    auto pass_T = [&](const float (&x)[K], const cfloat* T, float (&col)[K], bool act) {
        if (act)
#pragma unroll
            for (int v = 0; v < K; v++) {
                float m = 0.f;
#pragma unroll
                for (int q = 0; q < K; q++) m = m + x[q] * T[q * K + v];
                X[nl * XS + v * XP + rr] = m;
            }
        wave_sync();
        if (act)
#pragma unroll
            for (int p = 0; p < K; p++) col[p] = X[nl * XS + rr * XP + p];
        wave_sync();
    };
    for (int c = 0; c < C; c++) {
        for (int nb0 = 0; nb0 < nsx; nb0 += PB) {
            const int n = nb0 + nl;
            const bool act = lact && n < nsx;
            float x[K], u[K], col[K];
            if (act) {
                const unsigned mi = mem[n], pt = div32(mi, dWHC);
                const unsigned py = div32(mi - pt * whc, dW), px = mi - pt * whc - py * W;
                const size_t o = (size_t)pt * whc + (size_t)c * wh + (size_t)(py + rr) * W + px;
#pragma unroll
                for (int q = 0; q < K; q++) x[q] = a.basic[o + q];
#pragma unroll
                for (int q = 0; q < K; q++) {
                    const float dn = a.den[o + q];
                    u[q] = KAI[rr * K + q] * (dn != 0.f ? a.gy[o + q] / dn : 0.f);
                }
                // the basic patch's coefficients as the forward pass forms
                // them (filter_one), so that the gains are its bits
                if (bior) {
#pragma unroll
                    for (int v = 0; v < K; v++) {
                        float m = 0.f;
#pragma unroll
                        for (int q = 0; q < K; q++) m = m + x[q] * TF[v * K + q];
                        X[nl * XS + v * XP + rr] = m;
                    }
                } else {
                    float y[K];
                    dct_fwd_pass<K>(x, y, TF);
#pragma unroll
                    for (int v = 0; v < K; v++) X[nl * XS + v * XP + rr] = y[v];
                }
            }
            wave_sync();
            if (act) {
#pragma unroll
                for (int p = 0; p < K; p++) col[p] = X[nl * XS + rr * XP + p];
                if (bior) {
#pragma unroll
                    for (int v = 0; v < K; v++) {
                        float m = 0.f;
#pragma unroll
                        for (int p = 0; p < K; p++) m = m + col[p] * TF[v * K + p];
                        eg[n * K2 + rr * 8 + v] = m;
                    }
                } else {
                    float y[K];
                    dct_fwd_pass<K>(col, y, TF);
#pragma unroll
                    for (int v = 0; v < K; v++) eg[n * K2 + v * K + rr] = y[v] * NRM[v * K + rr];
                }
            }
            wave_sync();
            // Transpose of the inverse 2D transform.  DCT: G(c) = dct_out M
            // (c o inv) M^T with M[x][y] = dctI[x*K+y], so G^T(r) = inv o
            // dct_out (M^T r M).  BIOR: G(c)[u][m] = sum S[u][p] c[q][p]
            // S[m][q] with S = biorI, so G^T(r)[q][p] = sum r[u][m] S[u][p]
            // S[m][q].
            pass_T(u, TI, col, act);
            if (act)
#pragma unroll
                for (int v = 0; v < K; v++) {
                    float o = 0.f;
#pragma unroll
                    for (int p = 0; p < K; p++) o = o + TI[p * K + v] * col[p];
                    if (bior) zg[n * K2 + rr * 8 + v] = o;
                    else zg[n * K2 + v * K + rr] = INV[v * K + rr] * dct_out * o;
                }
            wave_sync();
        }
        const float sg = sig_of(a, c);
        float* v2c = a.wgt_kept ? nullptr : v2;
        switch (nsx) {
            case 1: adj_group<K, 1>(zg, eg, v2c, lane, had, sg); break;
            case 2: adj_group<K, 2>(zg, eg, v2c, lane, had, sg); break;
            case 4: adj_group<K, 4>(zg, eg, v2c, lane, had, sg); break;
            case 8: adj_group<K, 8>(zg, eg, v2c, lane, had, sg); break;
            default: adj_group<K, 16>(zg, eg, v2c, lane, had, sg); break;
        }
        wave_sync();
        float wg;
        if (a.wgt_kept) {
            wg = a.wgt[(size_t)slot * C + c];
        } else {
            // the group's weight, summed in the forward pass's order
            float acc = 0.f;
            if (lane == 0) switch (nsx) {
                    case 1: acc = wiener_sum<K, 1>(v2); break;
                    case 2: acc = wiener_sum<K, 2>(v2); break;
                    case 4: acc = wiener_sum<K, 4>(v2); break;
                    case 8: acc = wiener_sum<K, 8>(v2); break;
                    default: acc = wiener_sum<K, 16>(v2); break;
                }
            acc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(acc), 0));
            const float s2 = sg * sg;
            wg = had ? (acc > 0.0f ? 1.0f / (s2 * acc) : 1.0f) : 1.f / (s2 * acc);
        }
        // Transpose of the forward 2D transform.  DCT: F(x) = nrm o (A x
        // A^T), A = dctF, so F^T(c) = A^T (nrm o c) A.  BIOR: F(x) = B x^T
        // B^T, B = biorF, so F^T(c)[s][q] = sum c[i][j] B[j][s] B[i][q].
        float* dst = a.est + (size_t)slot * (unsigned)(a.N * a.ms) + c * K2;
        for (int nb0 = 0; nb0 < nsx; nb0 += PB) {
            const int n = nb0 + nl;
            const bool act = lact && n < nsx;
            float x[K], col[K];
            if (act)
#pragma unroll
                for (int q = 0; q < K; q++)
                    x[q] = bior ? zg[n * K2 + rr * K + q] : NRM[rr * K + q] * zg[n * K2 + rr * K + q];
            pass_T(x, TF, col, act);
            if (act)
#pragma unroll
                for (int p = 0; p < K; p++) {
                    float o = 0.f;
#pragma unroll
                    for (int q = 0; q < K; q++) o = o + TF[q * K + p] * col[q];
                    // DCT: col is column rr of t, o = y[p][rr]; BIOR: col is
                    // t[.][rr], o = y[rr][p]
                    zg[n * K2 + (bior ? rr * K + p : p * K + rr)] = wg * o;
                }
            wave_sync();
        }
        for (int q = lane; q < nsx * K2; q += 64) {
            const int n = q / K2;
            dst[n * a.ms + (q - n * K2)] = zg[q];
        }
        wave_sync();
    }
}

__global__ void k_adjoint_fallback(float* gz, const float* gy, const float* den, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && den[i] == 0.f) gz[i] = gz[i] + gy[i];
}

}  // namespace

// ---------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------
template <int K, int C, int STEP>
static hipError_t filter_k(const FArgs& a, hipStream_t s) {
    const long n = a.r_end - a.r_begin;
    if (n <= 0) return hipSuccess;
    const size_t per_wave = (size_t)filter_lds_words(K, C, a.N, STEP) * 4;
    int waves = 4;
    while (waves > 1 && per_wave * waves > 64 * 1024) waves--;
    if (per_wave > 64 * 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_filter<K, C, STEP>), dim3((unsigned)((n + waves - 1) / waves)),
                       dim3(64 * waves), per_wave * waves, s, a);
    return hipGetLastError();
}

template <int K>
static hipError_t filter_kc(int step, const FArgs& a, hipStream_t s) {
    if (a.C == 1) return step == 1 ? filter_k<K, 1, 1>(a, s) : filter_k<K, 1, 2>(a, s);
    return step == 1 ? filter_k<K, 3, 1>(a, s) : filter_k<K, 3, 2>(a, s);
}

hipError_t launch_filter(int K, int step, const FArgs& a, hipStream_t s) {
    switch (K) {
        case 4: return filter_kc<4>(step, a, s);
        case 5: return filter_kc<5>(step, a, s);
        case 6: return filter_kc<6>(step, a, s);
        case 7: return filter_kc<7>(step, a, s);
        case 8: return filter_kc<8>(step, a, s);
        default: return hipErrorInvalidValue;
    }
}

template <int K, int C, int STEP>
static hipError_t filter_kt_k(const FArgs& a, hipStream_t s) {
    const long n = a.r_end - a.r_begin;
    if (n <= 0) return hipSuccess;
    const size_t per_wave = (size_t)filter_kt_words(K, C, a.kt, a.N, STEP) * 4;
    if (per_wave > 64 * 1024) return hipErrorInvalidValue;
    // the workgroup that leaves most wavefronts on a CU's 160 KB of LDS
    int waves = 1, best = 0;
    for (int v = 1; v <= 4 && per_wave * v <= 64 * 1024; v++) {
        const int on = (int)(160 * 1024 / (per_wave * v)) * v;
        if (on >= best) best = on, waves = v;
    }
    hipLaunchKernelGGL((k_filter_kt<K, C, STEP>), dim3((unsigned)((n + waves - 1) / waves)), dim3(64 * waves),
                       per_wave * waves, s, a);
    return hipGetLastError();
}

template <int K>
static hipError_t filter_kt_kc(int step, const FArgs& a, hipStream_t s) {
    if (a.C == 1) return step == 1 ? filter_kt_k<K, 1, 1>(a, s) : filter_kt_k<K, 1, 2>(a, s);
    return step == 1 ? filter_kt_k<K, 3, 1>(a, s) : filter_kt_k<K, 3, 2>(a, s);
}

hipError_t launch_filter_kt(int K, int step, const FArgs& a, hipStream_t s) {
    switch (K) {
        case 4: return filter_kt_kc<4>(step, a, s);
        case 5: return filter_kt_kc<5>(step, a, s);
        case 6: return filter_kt_kc<6>(step, a, s);
        case 7: return filter_kt_kc<7>(step, a, s);
        case 8: return filter_kt_kc<8>(step, a, s);
        default: return hipErrorInvalidValue;
    }
}

int filter_kt_lds_words(int K, int C, int kt, int N, int step) { return filter_kt_words(K, C, kt, N, step); }

template <int K>
static hipError_t filter_adj_k(const FArgs& a, hipStream_t s) {
    const long n = a.r_end - a.r_begin;
    if (n <= 0) return hipSuccess;
    const size_t per_wave = (size_t)adjoint_lds_words(K, a.N) * 4;
    int waves = 4;
    while (waves > 1 && per_wave * waves > 64 * 1024) waves--;
    if (per_wave > 64 * 1024) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((n + waves - 1) / waves)), block(64 * waves);
    if (a.C == 1) hipLaunchKernelGGL((k_filter_adjoint<K, 1>), grid, block, per_wave * waves, s, a);
    else hipLaunchKernelGGL((k_filter_adjoint<K, 3>), grid, block, per_wave * waves, s, a);
    return hipGetLastError();
}

hipError_t launch_filter_adjoint(int K, const FArgs& a, hipStream_t s) {
    switch (K) {
        case 4: return filter_adj_k<4>(a, s);
        case 5: return filter_adj_k<5>(a, s);
        case 6: return filter_adj_k<6>(a, s);
        case 7: return filter_adj_k<7>(a, s);
        case 8: return filter_adj_k<8>(a, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_adjoint_fallback(float* gz, const float* gy, const float* den, size_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_adjoint_fallback, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, gz, gy, den, n);
    return hipGetLastError();
}

template <int K, int C, int STEP>
static hipError_t filter_queue_k(const FArgs* jobs, const WorkQueue& q, int words, int waves, int blocks,
                                 hipStream_t s) {
    hipLaunchKernelGGL((k_filter_queue<K, C, STEP>), dim3(blocks), dim3(64 * waves), (size_t)words * 4 * waves, s,
                       jobs, q, words);
    return hipGetLastError();
}

template <int K>
static hipError_t filter_queue_kc(int C, int step, const FArgs* jobs, const WorkQueue& q, int words, int waves,
                                  int blocks, hipStream_t s) {
    if (C == 1)
        return step == 1 ? filter_queue_k<K, 1, 1>(jobs, q, words, waves, blocks, s)
                         : filter_queue_k<K, 1, 2>(jobs, q, words, waves, blocks, s);
    return step == 1 ? filter_queue_k<K, 3, 1>(jobs, q, words, waves, blocks, s)
                     : filter_queue_k<K, 3, 2>(jobs, q, words, waves, blocks, s);
}

template <int K, int C, int STEP>
static hipError_t filter_multi_k(const FArgs* jobs, const WorkQueue& q, int words, int waves, hipStream_t s) {
    const long blocks = (q.total + waves - 1) / waves;
    hipLaunchKernelGGL((k_filter_multi<K, C, STEP>), dim3((unsigned)blocks), dim3(64 * waves),
                       (size_t)words * 4 * waves, s, jobs, q, words);
    return hipGetLastError();
}

template <int K>
static hipError_t filter_multi_kc(int C, int step, const FArgs* jobs, const WorkQueue& q, int words, int waves,
                                  hipStream_t s) {
    if (C == 1)
        return step == 1 ? filter_multi_k<K, 1, 1>(jobs, q, words, waves, s)
                         : filter_multi_k<K, 1, 2>(jobs, q, words, waves, s);
    return step == 1 ? filter_multi_k<K, 3, 1>(jobs, q, words, waves, s)
                     : filter_multi_k<K, 3, 2>(jobs, q, words, waves, s);
}

hipError_t launch_filter_multi(int K, int C, int step, const FArgs* jobs, const WorkQueue& q, int words,
                               int waves, hipStream_t s) {
    if (q.total <= 0) return hipSuccess;
    if ((size_t)words * 4 * waves > 64 * 1024 || waves < 1 || waves > 4) return hipErrorInvalidValue;
    switch (K) {
        case 4: return filter_multi_kc<4>(C, step, jobs, q, words, waves, s);
        case 5: return filter_multi_kc<5>(C, step, jobs, q, words, waves, s);
        case 6: return filter_multi_kc<6>(C, step, jobs, q, words, waves, s);
        case 7: return filter_multi_kc<7>(C, step, jobs, q, words, waves, s);
        case 8: return filter_multi_kc<8>(C, step, jobs, q, words, waves, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_filter_queue(int K, int C, int step, const FArgs* jobs, const WorkQueue& q, int words,
                               int waves, int blocks, hipStream_t s) {
    if (q.total <= 0 || blocks <= 0) return hipSuccess;
    if ((size_t)words * 4 * waves > 64 * 1024 || waves < 1 || waves > 4) return hipErrorInvalidValue;
    switch (K) {
        case 4: return filter_queue_kc<4>(C, step, jobs, q, words, waves, blocks, s);
        case 5: return filter_queue_kc<5>(C, step, jobs, q, words, waves, blocks, s);
        case 6: return filter_queue_kc<6>(C, step, jobs, q, words, waves, blocks, s);
        case 7: return filter_queue_kc<7>(C, step, jobs, q, words, waves, blocks, s);
        case 8: return filter_queue_kc<8>(C, step, jobs, q, words, waves, blocks, s);
        default: return hipErrorInvalidValue;
    }
}

int filter_words(int K, int C, int N, int step) { return filter_lds_words(K, C, N, step); }

}  // namespace vb
