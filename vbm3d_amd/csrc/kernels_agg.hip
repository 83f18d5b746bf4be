// kernels_agg.hip -- CDNA4 (gfx950) ordered aggregation of the VBM3D
// collaborative filter: one 32x16 output tile per workgroup; contributions
// are gathered in the reference's (crop, frame, row, column, n) order, so
// every pixel's sum is formed in the same order as the CPU and no atomics
// are used.  Also the colour transform and the small utility kernels.
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
// Aggregation (src/vbm3d.cpp:612-650, 860-924) with the division and the
// den == 0 fallback (:168-170, :198-202, :267-280, :333-346).
// ---------------------------------------------------------------------
// One 32x16 output tile of one frame per workgroup (eight wavefronts).
// The reference patches whose groups can reach the tile are scanned in
// processing order (crop, frame, row, column), one per thread at a time;
// the group members that overlap the tile are compacted into an ordered
// list, and each wavefront then accumulates, for its 8x8 block, the
// members that overlap the block in list order: every output sample sees
// its contributions in exactly the reference's order.
//
// What bounds it: with three channels the cache lines of `est` its gathers
// touch, with one channel instruction issue.  An entry used to be decoded
// on the scalar unit, 27 scalar and 28 vector instructions; decoded by one
// lane for 64 entries at once and taken through readlane it costs about 10
// and 23 (14 with one channel).  Scanning a tile's chunks into one list
// before any sum leaves the scan's registers out of the sums and one
// barrier per chunk.  Measured, step 2 and step 1: 30 RGB frames 960x540
// 3.67 -> 2.94 and 1.10 -> 1.00 ms (the first with the padded members of
// est_words, 3.59 without); 10 grey frames 176x144 97 -> 57 and 34 -> 23
// us; 32 grey frames 640x360 1.52 -> 1.00 ms.  With three channels 3, 6 or
// 8 entries in flight are slower than 4 (3.07, 3.41, 3.04 ms), with one
// channel 12 or 16 within noise of 8.
// ONE: the grid is a single crop (nb = 1); the per-crop sums are then the
// totals, and no crop-order merge is kept live across the scan.
// KT: members of a.kt > 1 slices, one per frame from the member's on; the
// output frame takes the slice that lies in it (8 RGB frames 320x240 at kt 2,
// against k_aggregate_gen: 1.75 -> 0.29 and 0.39 -> 0.07 ms).
template <int C, bool RAW, int NM, bool ONE, bool KT, class A>
__device__ __forceinline__ void agg_tile(const A& a, const int bx, const int by, const unsigned bz, const int nl) {
    constexpr int TX = kAggTileX, TY = kAggTileY, NT = kAggThreads;
    constexpr int QS = 8;             // a wavefront's block edge
    constexpr int NWV = NT / 64, WX = TX / QS;
    constexpr int U = C == 1 ? 8 : 4;  // entries whose loads are in flight together
    static_assert(TX % QS == 0 && TY % QS == 0 && NT % 64 == 0, "tile of 8x8 blocks");
    static_assert(TX + kMaxK - 1 <= 64 && TY + kMaxK - 1 <= 32 && NT * kMaxN <= 65536, "list entry fields");
    // the ordered list of members that overlap the tile: {member n (4
    // bits), its column + K - 1 and row + K - 1 in the tile (6, 5 bits), its
    // slice (KT); slot}.  It holds what one NT-patch chunk can bring (nl >= N members
    // each), in practice the whole tile's members.
    extern __shared__ uint2 agg_lists[];
    uint2* L_e = agg_lists;
    const int cap = NT * nl;
    __shared__ uint16_t s_pick[NWV][128];  // per wavefront: entries overlapping its block, not yet summed
    __shared__ float s_kai[kMaxWin * kMaxWin * 4];
    __shared__ int s_w[2][NWV];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = tid >> 6;
    const int x0 = bx * TX, y0 = by * TY;
    const unsigned to = a.t_begin + bz;
    const int qx0 = (wv % WX) * QS, qy0 = (wv / WX) * QS;  // this wave's block in the tile
    const int px = x0 + qx0 + (lane & (QS - 1)), py = y0 + qy0 + lane / QS;
    const bool inside = px < (int)a.W && py < (int)a.H;
    const int K = a.K, K2 = K * K, N = a.N;
    const unsigned W = a.W, wh = a.wh, whc = a.whc;
    for (int i = tid; i < K2; i += NT) s_kai[i] = a.tabs->kaiser[i];
    float tn[C], td[C];
#pragma unroll
    for (int c = 0; c < C; c++) tn[c] = td[c] = 0.f;
    // a member at q = to*whc + y*W + x overlaps the tile's rows iff
    // q - to*whc lies in [ylo*W, yhi*W)
    const unsigned tbase = to * whc;
    const int kt = KT ? a.kt : 1;
    const int trlo = max(0, (int)to - a.Nf - (kt - 1)), trhi = min((int)a.Fr - 1, (int)to + a.Nf);
    const int nfr = trhi - trlo + 1;
    // the largest frame distance of a member that reaches this frame from a
    // patch in frame tr (its frame lies in [to - kt + 1, to])
    auto far = [&](int tr) {
        const int k = abs(tr - (int)to);
        return KT ? min(max(k, abs(tr - ((int)to - kt + 1))), a.Nf) : k;
    };
    // the position of member mi in this frame, less tbase (and its slice)
    auto in_frame = [&](uint32_t mi, unsigned* ht) {
        unsigned r = mi - tbase;
        if (KT) {
            *ht = 0;
            for (int q = 1; q < kt && r >= whc; q++) {
                r += whc;
                *ht = q;
            }
        }
        return r;
    };
    const Div32 dW = {a.divW.m, a.divW.s1, a.divW.s2};
    const unsigned rmin = (unsigned)max(0, y0 - K + 1) * W, rmax = (unsigned)min((int)a.H, y0 + TY) * W;
    // packed pairs of 16 bits (x low, y high): the lane's pixel in list
    // entry coordinates, the patch's last sample, and the bytes of a
    // sample's column and row
    typedef short short2v __attribute__((ext_vector_type(2)));
    typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));
    const short2v lpos = {(short)(qx0 + (lane & (QS - 1)) + K - 1), (short)(qy0 + lane / QS + K - 1)};
    const short2v kmax = {(short)(K - 1), (short)(K - 1)}, zero = {0, 0};
    typedef const __attribute__((address_space(1))) char gchar;
    typedef const __attribute__((address_space(1))) float gfloat;
    const ushort2v kstr = {4, (unsigned short)(4 * K)};

    // per frame of a crop's box: {first index, columns, first row, first
    // column} of the grid patches whose members can reach the tile, and the
    // division by the column count
    constexpr int MF = 2 * kGenMaxNf + (KT ? kGenMaxKt : 1);  // frames of patches
    static_assert(MF <= 32, "one scan of 32 lanes");
    __shared__ int4 s_box[MF];
    __shared__ int s_bnd[6 * MF];
    __shared__ Div32 s_div[MF];
    __shared__ int s_total;

    // The crops that hold a patch whose members can reach the tile, from
    // the widest box (frame distance Nf): a tile meets one crop, at the
    // seams up to four, and a crop without patches adds nothing.  (16 grey
    // frames 1280x720 on 16 crops, visiting only these: step 2 and step 1
    // 2.52 -> 1.54 and 1.65 -> 0.98 ms with the rest of this kernel.)
    uint32_t crops = 1u;
    if (!ONE) {
        __shared__ int s_any[2 * kMaxCrops];
        for (int q = tid; q < 2 * a.ncrop; q += NT) {
            const int ci = q >> 1, col = q & 1;
            const int4 v = a.boxtab[((size_t)ci * (a.nty + a.ntx) + (col ? a.nty + bx : by)) * (a.Nf + 1) + a.Nf];
            s_any[q] = v.y > v.x;
        }
        __syncthreads();
        crops = (uint32_t)__ballot(lane < a.ncrop && s_any[2 * (lane & (kMaxCrops - 1))] && s_any[2 * (lane & (kMaxCrops - 1)) + 1]);
    }

    for (; crops; crops &= crops - 1) {
        const int ci = ONE ? 0 : __builtin_ctz(crops);
        const int* meta = a.crop_meta + ci * 5;
        const int off = meta[0], ncols = meta[2];
        // A member k frames away from its reference patch lies within
        // min(R, R0 + k Rs) of it, so the box narrows towards the output
        // frame.  The frames' boxes are concatenated in frame order: the
        // scan below still visits the patches in processing order (crop,
        // frame, row, column).
        __syncthreads();  // the previous crop's table is no longer read
        // the host's table of the bounds: one load per bound, the columns'
        // division with them.  (Searched here, they are a chain of dependent
        // loads ahead of everything else a tile does: a batch of 64 mixed
        // clips 576 -> 567 ms without it.)
        if (tid < 2 * nfr) {
            const int q = tid >> 1, col = tid & 1;
            const int k = far(trlo + q);
            const size_t tl = (size_t)ci * (a.nty + a.ntx) + (col ? a.nty + bx : by);
            const int4 v = a.boxtab[tl * (a.Nf + 1) + k];
            s_bnd[6 * q + 2 * col] = v.x;
            s_bnd[6 * q + 2 * col + 1] = v.y;
            if (col) {
                s_bnd[6 * q + 4] = v.z;
                s_bnd[6 * q + 5] = v.w;
            }
        }
        __syncthreads();
        // wavefront 0: lane q < nfr assembles frame q's box; the boxes'
        // first indices are an exclusive scan of their patch counts
        if (wv == 0) {
            int cnt = 0, nc = 0, ia = 0, ja = 0;
            if (lane < nfr) {
                ia = s_bnd[6 * lane];
                ja = s_bnd[6 * lane + 2];
                const int nr = max(s_bnd[6 * lane + 1] - ia, 0);
                nc = max(s_bnd[6 * lane + 3] - ja, 0);
                cnt = nr * nc;
                const unsigned sh = (unsigned)s_bnd[6 * lane + 5];
                s_div[lane] = Div32{(uint32_t)s_bnd[6 * lane + 4], sh & 0xFFu, sh >> 8};
            }
            int incl = cnt;
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) {
                const int y = __shfl_up(incl, o, 64);
                if (lane >= o) incl += y;
            }
            if (lane < nfr) s_box[lane] = make_int4(incl - cnt, nc, ia, ja);
            if (lane == nfr - 1) s_total = incl;
        }
        __syncthreads();
        const long total = s_total;
        float pn[C], pd[C];
#pragma unroll
        for (int c = 0; c < C; c++) pn[c] = pd[c] = 0.f;

        // The scan data of a chunk: slot, group size, member indices (up to
        // NM >= N of them).
        uint32_t slot = 0, mi[NM];
        int ns = 0;
        auto fetch = [&](long cb) {
            const unsigned e = (unsigned)(cb + tid);
            slot = 0;
            ns = 0;
#pragma unroll
            for (int n = 0; n < NM; n++) mi[n] = 0u;
            if (e < total) {
                // the frame whose box holds index e: the last one starting
                // at or before it (empty boxes start where the next does)
                int q = 0;
#pragma unroll
                for (int st = 16; st >= 1; st >>= 1)
                    if (q + st < nfr && (int)e >= s_box[q + st].x) q += st;
                const int4 bx = s_box[q];
                const Div32 dq = s_div[q];
                const unsigned rest = e - (unsigned)bx.x;
                const unsigned ii = div32(rest, dq), jj = rest - ii * (unsigned)bx.y;
                const unsigned tr = trlo + q;
                slot = (tr % a.ring) * a.nrf + off + (bx.z + ii) * ncols + (bx.w + jj);
                ns = (int)a.nsx[slot];
                const uint32_t* mem = a.idx + (size_t)slot * N;
#pragma unroll
                for (int n = 0; n < NM; n++) mi[n] = n < N ? mem[n] : 0u;
            }
        };
        // Sums the first `cnt` <= 64 entries of this wavefront's pick list,
        // in order.  Lane q decodes entry q -- position, est address,
        // weights -- for all of them at once; the entries then go one after
        // the other through readlane into scalar registers, so that an
        // entry costs neither scalar decoding nor a dependent load.
        const uint64_t cstr = (uint64_t)(unsigned)(K2 * kt * 4);  // bytes from one channel's plane to the next
        auto sum_picks = [&](int cnt) {
            const uint2 ent = L_e[s_pick[wv][lane < cnt ? lane : 0]];
            float ew[RAW ? 1 : C];
            if (!RAW)
#pragma unroll
                for (int c = 0; c < C; c++) ew[c] = a.wgt[(size_t)ent.y * C + c];
            const uint32_t epos = ((ent.x >> 4) & 63u) | ((KT ? (ent.x >> 10) & 31u : ent.x >> 10) << 16);
            // the member index slot * N + n fits 32 bits (the host refuses
            // larger rings)
            const uint32_t pl = ent.y * (unsigned)N + (ent.x & 15u);
            const uint64_t eb = (uint64_t)a.est + (uint64_t)pl * (unsigned)(a.ms * 4) +
                                (KT ? (ent.x >> 15) * (unsigned)(K2 * 4) : 0u);
            const uint32_t elo = (uint32_t)eb, ehi = (uint32_t)(eb >> 32);
            for (int j0 = 0; j0 < cnt; j0 += U) {
                // U entries at a time: every load is issued before the first
                // sum.  Straight-line loads: an absent entry repeats the
                // last one, a lane outside a patch reads the patch's sample
                // nearest to it (within the rows and columns the patch's own
                // lanes read, so no extra cache line); only the sums below
                // are masked
                float ev[U][C], kai[U];
                bool on[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int j = min(j0 + u, cnt - 1);
                    const uint32_t pos = __builtin_amdgcn_readlane(epos, j);
                    const uint64_t b = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(elo, j) |
                                       ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(ehi, j) << 32);
                    const short2v d = lpos - __builtin_bit_cast(short2v, pos);
                    const short2v cl = __builtin_elementwise_min(__builtin_elementwise_max(d, zero), kmax);
                    on[u] = (j0 + u < cnt) & (__builtin_bit_cast(uint32_t, d) == __builtin_bit_cast(uint32_t, cl));
                    const uint32_t ko = __builtin_amdgcn_udot2(__builtin_bit_cast(ushort2v, cl), kstr, 0u, false);
                    kai[u] = *(const float*)((const char*)s_kai + ko);
#pragma unroll
                    for (int c = 0; c < C; c++) ev[u][c] = *(const gfloat*)((const gchar*)(b + c * cstr) + ko);
                }
                // keeps the loads above from being sunk to their sums
                asm volatile("" ::: "memory");
#pragma unroll
                for (int u = 0; u < U; u++) {
                    float w[RAW ? 1 : C];
                    if (!RAW)
#pragma unroll
                        for (int c = 0; c < C; c++)
                            w[c] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ew[c]), min(j0 + u, cnt - 1)));
                    if (!on[u]) continue;
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        if (RAW) {
                            pn[c] = pn[c] + ev[u][c];
                        } else {
                            const float kw = kai[u] * w[c];
                            pn[c] = pn[c] + kw * ev[u][c];
                            pd[c] = pd[c] + kw;
                        }
                    }
                }
            }
        };
        long cb = 0;
        while (cb < total) {
            // Scan: chunks are appended to the list until they are all in
            // or the next one does not fit (it is scanned again after the
            // sums below; an empty list takes any chunk).  The loads of
            // chunk cb + NT fly while chunk cb is listed.
            int len = 0;
            fetch(cb);
            while (cb < total) {
                uint32_t hits = 0;
#pragma unroll
                for (int n = 0; n < NM; n++) {
                    if (n >= ns) break;
                    unsigned ht;
                    const unsigned r = in_frame(mi[n], &ht);
                    if (r < rmin || r >= rmax) continue;
                    const int qy = (int)div32(r, dW), qx = (int)(r - (unsigned)qy * W);
                    if (qx <= x0 + TX - 1 && qx + K - 1 >= x0) hits |= 1u << n;
                }
                // ordered compaction: exclusive block scan of the hit counts
                const int cnt = __popc(hits);
                int x = cnt;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int y = __shfl_up(x, o, 64);
                    if (lane >= o) x += y;
                }
                const int par = (int)(cb / NT) & 1;  // alternate, so that one barrier a chunk is enough
                if (lane == 63) s_w[par][wv] = x;
                __syncthreads();
                int base = 0, tot = 0;
#pragma unroll 1
                for (int q = 0; q < NWV; q++) {
                    const int sq = s_w[par][q];
                    base += q < wv ? sq : 0;
                    tot += sq;
                }
                if (len + tot > cap) break;  // workgroup-uniform
                const uint32_t sl = slot;
                uint32_t m2[NM];
#pragma unroll
                for (int n = 0; n < NM; n++) m2[n] = mi[n];
                cb += NT;
                if (cb < total) fetch(cb);
                int o = len + base + x - cnt;
#pragma unroll
                for (int n = 0; n < NM; n++)
                    if ((hits >> n) & 1u) {
                        unsigned ht = 0;
                        const unsigned r = in_frame(m2[n], &ht);
                        const unsigned qy = div32(r, dW), qx = r - qy * W;
                        L_e[o] = make_uint2((unsigned)n | ((qx + K - 1 - x0) << 4) | ((qy + K - 1 - y0) << 10) |
                                                (KT ? ht << 15 : 0u),
                                            sl);
                        o++;
                    }
                len += tot;
            }
            __syncthreads();
            // Sums: this wave takes the list entries overlapping its 8x8
            // block, in order, 64 at a time.
            int np = 0, j0 = 0;
            for (;;) {
                while (np < 64 && j0 < len) {
                    bool ov = false;
                    if (j0 + lane < len) {
                        const uint32_t ent = L_e[j0 + lane].x;
                        // block-relative corner + K - 1 in [0, QS + K - 2]
                        const unsigned ex = ((ent >> 4) & 63u) - (unsigned)qx0;
                        const unsigned ey = (KT ? (ent >> 10) & 31u : ent >> 10) - (unsigned)qy0;
                        ov = ex <= (unsigned)(QS + K - 2) && ey <= (unsigned)(QS + K - 2);
                    }
                    const uint64_t m = __ballot(ov);
                    if (ov) s_pick[wv][np + lanes_below(m, lane)] = (uint16_t)(j0 + lane);
                    np += __popcll(m);
                    j0 += 64;
                }
                if (np == 0) break;
                wave_sync();
                sum_picks(min(np, 64));
                if (np > 64) s_pick[wv][lane] = s_pick[wv][64 + lane];
                np = max(np - 64, 0);
                wave_sync();
            }
            __syncthreads();
        }
#pragma unroll
        for (int c = 0; c < C; c++) {
            if (ONE) {
                tn[c] = pn[c];
                td[c] = pd[c];
            } else {
                tn[c] = tn[c] + pn[c];
                td[c] = td[c] + pd[c];
            }
        }
    }
    if (inside) {
#pragma unroll
        for (int c = 0; c < C; c++) {
            const size_t o = (size_t)to * whc + (size_t)c * wh + (size_t)py * W + px;
            if (a.num_out) a.num_out[o] = tn[c];
            if (a.den_out) a.den_out[o] = td[c];
            if (a.out) a.out[o] = td[c] == 0.f ? a.fallback[o] : tn[c] / td[c];
        }
    }
}

// Occupancy floor by the members the scan holds.  Up to 8: 8 waves per SIMD
// (64 registers), the kernel waits on memory more than it computes (6 waves
// with twice the entries in flight: 3.04 against 2.94 ms).  Above 8 the list
// takes up to 64 KB, which leaves two workgroups to a CU (4 waves per SIMD),
// and 64 registers spilled up to 280 bytes a lane for waves that could not
// run: 5.  (N 16, step 2 at floor 8 / 6 / 5 / 4: 8 grey frames 640x360 0.564 /
// 0.476 / 0.500 / 0.501 ms, on 16 crops 0.999 / 0.908 / 0.874 / 0.895, 8 RGB
// frames 320x240 0.287 / 0.246 / 0.244 / 0.255; a batch of 12 RGB clips
// 200x150x6, whole call, 5.54 / 5.04 / 4.81 / 4.80.)
constexpr int agg_waves_floor(int NM) { return NM > 8 ? 5 : 8; }

template <int C, bool RAW, int NM, bool ONE, bool KT>
__global__ __launch_bounds__(kAggThreads) __attribute__((amdgpu_waves_per_eu(agg_waves_floor(NM)))) void k_aggregate(
    AArgs a) {
    agg_tile<C, RAW, NM, ONE, KT>(a, blockIdx.x, blockIdx.y, blockIdx.z, a.N);
}

// Batched form with one workgroup per tile: workgroup b takes item b, so
// the hardware's dispatch order is the queue; item -> (job, frame, tile
// row, tile column).  The same occupancy floor as k_aggregate.
template <int C, int NM>
__global__ __launch_bounds__(kAggThreads) __attribute__((amdgpu_waves_per_eu(agg_waves_floor(NM)))) void k_aggregate_multi(
    const AArgs* __restrict__ jobs, WorkQueue q, int nl) {
    const long it = (long)blockIdx.x;
    if (it >= q.total) return;  // workgroup-uniform
    const int j = queue_job(q, it);
    typedef const __attribute__((address_space(4))) AArgs cAA;
    cAA& a = ((cAA*)jobs)[j];  // scalar loads of the job
    const long local = it - uniform_long(q.item_begin[j]);
    const long tx = (a.W + kAggTileX - 1) / kAggTileX, ty = (a.H + kAggTileY - 1) / kAggTileY;
    const long bz = local / (tx * ty), rem = local - bz * tx * ty;
    if (a.ncrop == 1) agg_tile<C, false, NM, true, false>(a, (int)(rem % tx), (int)(rem / tx), (unsigned)bz, nl);
    else agg_tile<C, false, NM, false, false>(a, (int)(rem % tx), (int)(rem / tx), (unsigned)bz, nl);
}

// Persistent form: one tile per take (the workgroup is the unit); item ->
// (job, frame, tile row, tile column).
template <int C, int NM>
__global__ __launch_bounds__(kAggThreads) void k_aggregate_queue(const AArgs* __restrict__ jobs, WorkQueue q, int nl) {
    __shared__ long s_item;
    for (;;) {
        __syncthreads();  // every thread has read the previous item
        if (threadIdx.x == 0) s_item = (long)atomicAdd(q.counter, 1ull);
        __syncthreads();
        const long it = s_item;
        if (it >= q.total) break;
        const int j = queue_job(q, it);
        typedef const __attribute__((address_space(4))) AArgs cAA;
        cAA& a = ((cAA*)jobs)[j];  // scalar loads of the job
        const long local = it - q.item_begin[j];
        const long tx = (a.W + kAggTileX - 1) / kAggTileX, ty = (a.H + kAggTileY - 1) / kAggTileY;
        const long bz = local / (tx * ty), rem = local - bz * tx * ty;
        if (a.ncrop == 1) agg_tile<C, false, NM, true, false>(a, (int)(rem % tx), (int)(rem / tx), (unsigned)bz, nl);
        else agg_tile<C, false, NM, false, false>(a, (int)(rem % tx), (int)(rem / tx), (unsigned)bz, nl);
    }
}

// ---------------------------------------------------------------------
// Colour transform, 3 channels (src/Utilities/LibVideoT.hpp:777-887).
// ---------------------------------------------------------------------
__global__ void k_color(float* v, unsigned wh, unsigned F, int forward) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)wh * F) return;
    const size_t f = i / wh, k = i - f * wh;
    float* r = v + f * 3 * wh;
    const float R = r[k], G = r[wh + k], B = r[2 * wh + k];
    float o0, o1, o2;
    if (forward) {
        o0 = 0.299f * R + 0.587f * G + 0.114f * B;
        o1 = -0.14713f * R - 0.28886f * G + 0.436f * B;
        o2 = 0.615f * R - 0.51498f * G - 0.10001f * B;
    } else {
        o0 = R + 1.13983f * B;
        o1 = R - 0.39465f * G - 0.5806f * B;
        o2 = R + 2.03211f * G;
    }
    r[k] = o0;
    r[wh + k] = o1;
    r[2 * wh + k] = o2;
}

// Clears the work-queue counters of a batch (a kernel rather than a
// memset, so that it can sit inside a captured graph).
__global__ void k_zero_u64(unsigned long long* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

// Work counters of one block-matching launch: stats[0] += candidates,
// stats[1] += group members (one atomic per block).
__global__ void k_sum_counts(const uint32_t* cnt, long n, unsigned long long* stats) {
    __shared__ unsigned long long part[2][4];
    unsigned long long c0 = 0, c1 = 0;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        c0 += cnt[2 * i];
        c1 += cnt[2 * i + 1];
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        c0 += (unsigned long long)__shfl_xor((long long)c0, o, 64);
        c1 += (unsigned long long)__shfl_xor((long long)c1, o, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { part[0][w] = c0; part[1][w] = c1; }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long s0 = 0, s1 = 0;
        for (int k = 0; k < (int)(blockDim.x >> 6); k++) { s0 += part[0][k]; s1 += part[1][k]; }
        atomicAdd(&stats[0], s0);
        atomicAdd(&stats[1], s1);
    }
}

// Largest rounded magnitude of the flows given, in one launch with one
// atomic per workgroup and eight loads in flight: a launch per flow with an
// atomic per wavefront took 112 us for both flows of 12 frames 637x357, this
// takes 30.
__global__ __launch_bounds__(256) void k_flow_absmax(const float* __restrict__ ff, const float* __restrict__ bf, size_t n,
                                                     unsigned* out) {
    unsigned m = 0;
    const float* fl[2] = {ff, bf};
#pragma unroll
    for (int d = 0; d < 2; d++) {
        if (!fl[d]) continue;
        for (size_t i0 = (size_t)blockIdx.x * 2048 + threadIdx.x; i0 < n; i0 += (size_t)gridDim.x * 2048) {
            float v[8];  // in flight together
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = i0 + q * 256 < n ? fl[d][i0 + q * 256] : 0.f;
#pragma unroll
            for (int q = 0; q < 8; q++) m = max(m, (unsigned)fminf(fabsf(roundf(v[q])), 65535.f));  // NaN, huge: 65535
        }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
    __shared__ unsigned s[4];
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = max(max(s[0], s[1]), max(s[2], s[3]));
        if (m) atomicMax(out, m);
    }
}

}  // namespace

// ---------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------
hipError_t launch_aggregate_multi(int C, const AArgs* jobs, const WorkQueue& q, int maxN, hipStream_t s) {
    if (q.total <= 0) return hipSuccess;
    if (maxN < 1 || maxN > kMaxN || q.total > 0x7FFFFFFFL) return hipErrorInvalidValue;
    const size_t lds = (size_t)kAggThreads * maxN * sizeof(uint2);
    const dim3 grid((unsigned)q.total), blk(kAggThreads);
    if (maxN <= 8) {
        if (C == 1) hipLaunchKernelGGL((k_aggregate_multi<1, 8>), grid, blk, lds, s, jobs, q, maxN);
        else hipLaunchKernelGGL((k_aggregate_multi<3, 8>), grid, blk, lds, s, jobs, q, maxN);
    } else {
        if (C == 1) hipLaunchKernelGGL((k_aggregate_multi<1, 16>), grid, blk, lds, s, jobs, q, maxN);
        else hipLaunchKernelGGL((k_aggregate_multi<3, 16>), grid, blk, lds, s, jobs, q, maxN);
    }
    return hipGetLastError();
}

hipError_t launch_aggregate_queue(int C, const AArgs* jobs, const WorkQueue& q, int blocks, int maxN, hipStream_t s) {
    if (q.total <= 0 || blocks <= 0) return hipSuccess;
    if (maxN < 1 || maxN > kMaxN) return hipErrorInvalidValue;
    const size_t lds = (size_t)kAggThreads * maxN * sizeof(uint2);
    const dim3 blk(kAggThreads);
    // members held in registers by the scan: 8, or 16 when some job has N = 16
    if (maxN <= 8) {
        if (C == 1) hipLaunchKernelGGL((k_aggregate_queue<1, 8>), dim3(blocks), blk, lds, s, jobs, q, maxN);
        else hipLaunchKernelGGL((k_aggregate_queue<3, 8>), dim3(blocks), blk, lds, s, jobs, q, maxN);
    } else {
        if (C == 1) hipLaunchKernelGGL((k_aggregate_queue<1, 16>), dim3(blocks), blk, lds, s, jobs, q, maxN);
        else hipLaunchKernelGGL((k_aggregate_queue<3, 16>), dim3(blocks), blk, lds, s, jobs, q, maxN);
    }
    return hipGetLastError();
}

hipError_t launch_zero_u64(unsigned long long* p, int n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_zero_u64, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

hipError_t launch_aggregate(int C, const AArgs& a, unsigned frames, hipStream_t s) {
    if (frames == 0) return hipSuccess;
    dim3 grid((a.W + kAggTileX - 1) / kAggTileX, (a.H + kAggTileY - 1) / kAggTileY, frames);
    if (a.N < 1 || a.N > kMaxN) return hipErrorInvalidValue;
    const size_t lds = (size_t)kAggThreads * a.N * sizeof(uint2);  // the tile's ordered list
    const dim3 blk(kAggThreads);
    // members held in registers by the scan: 8, or 16 for N = 16
#define VB_AGG2(NM, ONE, RAW, KT)                                                          \
    {                                                                                      \
        if (C == 1) hipLaunchKernelGGL((k_aggregate<1, RAW, NM, ONE, KT>), grid, blk, lds, s, a); \
        else hipLaunchKernelGGL((k_aggregate<3, RAW, NM, ONE, KT>), grid, blk, lds, s, a); \
    }
#define VB_AGG1(NM, ONE)                          \
    if (a.raw) VB_AGG2(NM, ONE, true, false)      \
    else if (a.kt > 1) VB_AGG2(NM, ONE, false, true) \
    else VB_AGG2(NM, ONE, false, false)
#define VB_AGG(NM)               \
    if (a.ncrop == 1) {          \
        VB_AGG1(NM, true)        \
    } else {                     \
        VB_AGG1(NM, false)       \
    }
    if (a.N <= 8) {
        VB_AGG(8)
    } else {
        VB_AGG(16)
    }
#undef VB_AGG
#undef VB_AGG1
#undef VB_AGG2
    return hipGetLastError();
}

hipError_t launch_color(float* v, unsigned W, unsigned H, unsigned F, bool forward,
                        hipStream_t s) {
    const size_t n = (size_t)W * H * F;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_color, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, v,
                       W * H, F, forward ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_sum_counts(const uint32_t* counts, long n, unsigned long long* stats, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sum_counts, dim3(256), dim3(256), 0, s, counts, n, stats);
    return hipGetLastError();
}

hipError_t launch_flow_absmax(const float* ff, const float* bf, size_t n, unsigned* out, hipStream_t s) {
    if (n == 0 || (!ff && !bf)) return hipSuccess;
    const size_t blocks = (n + 2047) / 2048;
    hipLaunchKernelGGL(k_flow_absmax, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0, s, ff, bf, n, out);
    return hipGetLastError();
}

}  // namespace vb
