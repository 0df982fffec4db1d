// kq_vq_quant.hip -- the VQ quantiser (gfx950): from a dense weight matrix to
// the indices, codebooks and scales kq_vq_gemv reads.
//
// Reference: quantize_matrix / _kmeans, vq-gemv/quant/pq_quantize.py:28-83
// (there an offline MLX script). Steps (4 + 2 * iters launches; the full scan
// 3 + 2 * iters):
//
// 1. vq_scale_k: per (row, scale group) the abs-max scale (fp32), stored as
//    fp16; the pairs are normalised by the fp32 scale, 1 where it is 0
//    (pq_quantize.py:59-62).
// 2. vq_sample_k: per codebook block (rows_per_cb rows; the reference has one
//    per matrix) the k-means sample -- every pair of the block if there are
//    at most `sample`, else `sample` pairs drawn with replacement
//    (pq_quantize.py:38-39) -- and 256 initial centroids drawn from the
//    sample (pq_quantize.py:40). Draws are splitmix64 of (seed, block, draw
//    number), so a run is reproducible.
// 3. per Lloyd iteration (pq_quantize.py:41-48): each sample point goes to
//    argmax_c fmaf(p.x, c.x, fmaf(p.y, c.y, -|c|^2/2)) (the reference's
//    argmax of p.c - |c|^2/2; ties to the lowest c); the points are summed
//    per centroid in 2^-40 fixed point (integer sums, so the result does not
//    depend on their order) and each centroid moves to its mean (empty
//    clusters stay).
// 4. every pair of every row goes to its block's nearest fp32 centroid
//    (pq_quantize.py:66-73); the codebook is stored as fp16, rounded from the
//    means (a centroid that never moved: from its sample point).
//
// The nearest-centroid searches are all of the work: 256 scores for each of
// 25 x 200,000 sample points a block and then for every pair. Points lie in
// the square [-1, 1]^2 (a weight over its group's abs-max), so the square is
// cut into cells and vq_cells_k lists, per cell, the few centroids that can
// win anywhere in it (2-4 of 256 on average); vq_lloyd_k and vq_label_k score
// only those, in ascending order, and so pick what the full scan picks, bit
// for bit. Shapes whose buffers have no room for the lists run the full scan
// (vq_km_assign_k, vq_km_update_k, vq_assign_k).
#include "kq_device.h"
#include "kq_internal.h"

namespace kq {

namespace {

constexpr uint32_t kCB = 256;   // codewords
constexpr uint32_t kQT = 256;   // threads per workgroup
constexpr uint32_t kPPT = 4;    // pairs per thread in the assignment passes
constexpr uint32_t kInitDraw = 0x80000000u;  // draw numbers of the initial centroids

struct QWs {
    size_t sc, pts, cent, acc, total;
    uint32_t ns;  // sample points per block (the stride of pts)
};

QWs qws_layout(uint32_t M, uint32_t K, uint32_t G, uint32_t R, uint32_t sample) {
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const uint32_t nblk = (M + R - 1) / R;
    const uint64_t nmax = (uint64_t)(R < M ? R : M) * (K / 2);
    QWs L;
    L.ns = (uint32_t)(nmax < sample ? nmax : sample);
    L.sc = 0;
    L.pts = al(4ull * M * (K / G));
    L.cent = L.pts + al(8ull * nblk * L.ns);
    L.acc = L.cent + al(8ull * nblk * kCB);
    L.total = L.acc + al(24ull * nblk * kCB);
    return L;
}

struct VqAcc {
    unsigned long long x, y, n;  // fixed-point sums (two's complement) and the count
};

template <int DT>
__device__ __forceinline__ float wload(const void* W, size_t i) {
    if constexpr (DT == KQ_F32) return reinterpret_cast<const float*>(W)[i];
    else if constexpr (DT == KQ_BF16) return bf2f(reinterpret_cast<const uint16_t*>(W)[i]);
    else return h2f(reinterpret_cast<const uint16_t*>(W)[i]);
}

__device__ __forceinline__ uint64_t vq_hash(uint64_t seed, uint32_t blk, uint32_t j) {
    uint64_t x = seed + 0x9E3779B97F4A7C15ull * ((((uint64_t)blk) << 32) + (uint64_t)j + 1ull);
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// uniform index in [0, n) from draw j of block blk
__device__ __forceinline__ uint32_t vq_draw(uint64_t seed, uint32_t blk, uint32_t j, uint32_t n) {
    return (uint32_t)(((vq_hash(seed, blk, j) >> 32) * (uint64_t)n) >> 32);
}

__device__ __forceinline__ float vq_hc(float cx, float cy) { return -0.5f * fmaf(cx, cx, cy * cy); }

// The normalised pair i of row m.
template <int DT>
__device__ __forceinline__ float2 vq_pair(const void* W, const float* sc, uint32_t K, uint32_t G,
                                          uint32_t m, uint32_t i) {
    const float s = sc[(size_t)m * (K / G) + (2u * i) / G];
    const size_t o = (size_t)m * K + 2u * i;
    return make_float2(wload<DT>(W, o) / s, wload<DT>(W, o + 1) / s);
}

// Sample point j of block b (every pair when the block has at most `sample`).
template <int DT>
__device__ __forceinline__ float2 vq_sample_point(const void* W, const float* sc, uint32_t K,
                                                  uint32_t G, uint32_t r0, uint32_t N,
                                                  uint32_t sample, uint64_t seed, uint32_t b,
                                                  uint32_t j) {
    const uint32_t p = N <= sample ? j : vq_draw(seed, b, j, N);
    return vq_pair<DT>(W, sc, K, G, r0 + p / (K / 2), p % (K / 2));
}

// Nearest centroid: strictly greater score wins, ascending c.
__device__ __forceinline__ uint32_t vq_nearest(float px, float py, const float4* cs) {
    uint32_t best = 0;
    float bs = -INFINITY;
    for (uint32_t c = 0; c < kCB; ++c) {
        const float4 q = cs[c];
        const float s = fmaf(px, q.x, fmaf(py, q.y, q.z));
        if (s > bs || c == 0) {
            bs = s;
            best = c;
        }
    }
    return best;
}

// Centroids of block b into LDS as (x, y, -|c|^2/2, 0).
__device__ __forceinline__ void vq_load_cent(const float2* cent, uint32_t b, float4* cs) {
    for (uint32_t c = threadIdx.x; c < kCB; c += blockDim.x) {
        const float2 v = cent[(size_t)b * kCB + c];
        cs[c] = make_float4(v.x, v.y, vq_hc(v.x, v.y), 0.0f);
    }
}

// One workgroup per row: the maxima of the row's 32-element chunks (thread
// per chunk) into LDS, then per scale group the maximum of its chunks.
template <int DT>
__global__ __launch_bounds__(kQT) void vq_scale_k(const void* __restrict__ W, uint32_t K,
                                                  uint32_t G, uint16_t* __restrict__ S,
                                                  float* __restrict__ sc) {
    extern __shared__ float cm[];  // [K / 32]
    const uint32_t m = blockIdx.x, nck = K / 32, gpr = K / G;
    const size_t row = (size_t)m * K;
    for (uint32_t c = threadIdx.x; c < nck; c += kQT) {
        float a = 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < 32; ++k) a = fmaxf(a, fabsf(wload<DT>(W, row + c * 32 + k)));
        cm[c] = a;
    }
    __syncthreads();
    const uint32_t cpg = G / 32;
    for (uint32_t g = threadIdx.x; g < gpr; g += kQT) {
        float a = 0.0f;
        for (uint32_t c = 0; c < cpg; ++c) a = fmaxf(a, cm[g * cpg + c]);
        S[(size_t)m * gpr + g] = f2h(a);
        sc[(size_t)m * gpr + g] = a > 0.0f ? a : 1.0f;
    }
}

template <int DT>
__global__ __launch_bounds__(kQT) void vq_sample_k(const void* __restrict__ W, uint32_t M,
                                                   uint32_t K, uint32_t G, uint32_t R,
                                                   uint32_t sample, uint32_t ns_stride,
                                                   uint32_t nblk, uint32_t xcd,
                                                   uint64_t seed, const float* __restrict__ sc,
                                                   float2* __restrict__ pts,
                                                   float2* __restrict__ cent,
                                                   uint16_t* __restrict__ Cb,
                                                   VqAcc* __restrict__ acc) {
    // xcd: all of a block's workgroups run on one XCD (workgroups go to the 8
    // XCDs in turn), so a block's rows are gathered through one L2
    uint32_t b = blockIdx.y, wg = blockIdx.x;
    if (xcd) {
        const uint32_t l = blockIdx.y * gridDim.x + blockIdx.x;
        b = (l / 8 / gridDim.x) * 8 + l % 8;
        wg = l / 8 % gridDim.x;
    }
    if (b >= nblk) return;
    const uint32_t r0 = b * R, rows = min(R, M - r0);
    const uint32_t N = rows * (K / 2), ns = min(N, sample);
    const uint32_t j = wg * kQT + threadIdx.x;
    if (j < ns)
        pts[(size_t)b * ns_stride + j] =
            vq_sample_point<DT>(W, sc, K, G, r0, N, sample, seed, b, j);
    if (wg == 0) {
        for (uint32_t c = threadIdx.x; c < kCB; c += kQT) {
            const uint32_t jj = vq_draw(seed, b, kInitDraw + c, ns);
            const float2 v = vq_sample_point<DT>(W, sc, K, G, r0, N, sample, seed, b, jj);
            cent[(size_t)b * kCB + c] = v;
            Cb[((size_t)b * kCB + c) * 2] = f2h(v.x);
            Cb[((size_t)b * kCB + c) * 2 + 1] = f2h(v.y);
            acc[(size_t)b * kCB + c] = VqAcc{0, 0, 0};
        }
    }
}

__global__ __launch_bounds__(kQT) void vq_km_assign_k(const float2* __restrict__ pts,
                                                      uint32_t ns_stride, uint32_t M, uint32_t K,
                                                      uint32_t R, uint32_t sample,
                                                      const float2* __restrict__ cent,
                                                      VqAcc* __restrict__ acc) {
    __shared__ float4 cs[kCB];
    __shared__ unsigned long long sx[kCB], sy[kCB], sn[kCB];
    const uint32_t b = blockIdx.y, rows = min(R, M - b * R);
    const uint32_t ns = min(rows * (K / 2), sample);
    const uint32_t j0 = blockIdx.x * kQT * kPPT;
    if (j0 >= ns) return;  // uniform
    vq_load_cent(cent, b, cs);
    for (uint32_t c = threadIdx.x; c < kCB; c += kQT) sx[c] = sy[c] = sn[c] = 0;
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < kPPT; ++u) {
        const uint32_t j = j0 + u * kQT + threadIdx.x;
        if (j < ns) {
            const float2 p = pts[(size_t)b * ns_stride + j];
            const uint32_t a = vq_nearest(p.x, p.y, cs);
            atomicAdd(&sx[a], (unsigned long long)__float2ll_rz(p.x * 0x1p40f));
            atomicAdd(&sy[a], (unsigned long long)__float2ll_rz(p.y * 0x1p40f));
            atomicAdd(&sn[a], 1ull);
        }
    }
    __syncthreads();
    for (uint32_t c = threadIdx.x; c < kCB; c += kQT) {
        if (sn[c] == 0) continue;
        VqAcc* q = acc + (size_t)b * kCB + c;
        atomicAdd(&q->x, sx[c]);
        atomicAdd(&q->y, sy[c]);
        atomicAdd(&q->n, sn[c]);
    }
}

// A moved centroid: fp32 for the next searches, and its codeword, rounded to fp16
// once from the mean itself (through the fp32 centroid, ties of that rounding's
// making would round twice).
__device__ __forceinline__ void vq_store_mean(double x, double y, size_t i, float2* cent,
                                              uint16_t* Cb) {
    cent[i] = make_float2((float)x, (float)y);
    Cb[2 * i] = __builtin_bit_cast(uint16_t, (_Float16)x);
    Cb[2 * i + 1] = __builtin_bit_cast(uint16_t, (_Float16)y);
}

__global__ __launch_bounds__(kQT) void vq_km_update_k(VqAcc* __restrict__ acc,
                                                      float2* __restrict__ cent,
                                                      uint16_t* __restrict__ Cb) {
    const size_t i = (size_t)blockIdx.x * kCB + threadIdx.x;
    const VqAcc q = acc[i];
    if (q.n != 0) {
        vq_store_mean((double)(long long)q.x * 0x1p-40 / (double)q.n,
                      (double)(long long)q.y * 0x1p-40 / (double)q.n, i, cent, Cb);
    }
    acc[i] = VqAcc{0, 0, 0};
}

// One workgroup per (row, kQT * kPPT pairs) (grid x = rows); thread t takes pairs 4t .. 4t+3
// of the workgroup's range and writes their 4 index bytes as one word.
template <int DT>
__global__ __launch_bounds__(kQT) void vq_assign_k(const void* __restrict__ W, uint32_t K,
                                                   uint32_t G, uint32_t R,
                                                   const float* __restrict__ sc,
                                                   const float2* __restrict__ cent,
                                                   uint8_t* __restrict__ IDX) {
    __shared__ float4 cs[kCB];
    const uint32_t m = blockIdx.x, half = K / 2;
    vq_load_cent(cent, m / R, cs);
    __syncthreads();
    const uint32_t i0 = (blockIdx.y * kQT + threadIdx.x) * kPPT;
    if (i0 >= half) return;
    uint32_t word = 0;
#pragma unroll
    for (uint32_t u = 0; u < kPPT; ++u) {
        const float2 p = vq_pair<DT>(W, sc, K, G, m, i0 + u);
        word |= vq_nearest(p.x, p.y, cs) << (8 * u);
    }
    *reinterpret_cast<uint32_t*>(IDX + (size_t)m * half + i0) = word;
}

// ---- the cell lists -------------------------------------------------------
// [-1, 1]^2 in 2^LG x 2^LG cells; a cell's list is 16 bytes: the count, then
// up to kCellCap centroid indices in ascending order, then zeros (scoring
// centroid 0 where it is no candidate changes nothing: it loses); count
// kCellFull: more than fit, score all 256.
//
// Which centroids a list must hold: let c* have the greatest score at the
// cell's centre m. The score difference to any other c is affine in p, so over
// the cell (half width h) it is at most
//     score_c(m) - score_c*(m) + h * (|c.x - c*.x| + |c.y - c*.y|),
// and c is left out if that is below -kCellEps: c* then beats it at every
// point. The margin covers the roundings. Points, centroids and -|c|^2/2 are
// within [-1, 1], so a computed score is within 2 roundings of values below 3
// (3.6e-7) of the exact one, at p and at m alike (4 x 3.6e-7); a point's cell
// is computed with a rounding of 2 * 2^-24 (covered by kCellSlack in h).
// A centroid equal to c* with a higher index never wins either (equal scores
// go to the lowest index). NaN points score NaN against everything and get
// index 0 from the full scan and from a list alike; a NaN centroid never wins
// unless it is centroid 0, which then keeps every point (empty list = 0).
constexpr float kCellEps = 8e-6f, kCellSlack = 2e-6f;
constexpr uint32_t kCellCap = 15, kCellFull = 255;
constexpr uint32_t kCellT = 1024;      // threads of vq_cells_k: 16 x 16 cells a workgroup
constexpr uint32_t kSlotB = 5 * 1024;  // partial sums of one workgroup: x, y (u64), n (u32)
constexpr uint32_t kPT = 1024;       // threads of the point kernels

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
// Maximum over the wave (from lane 63: rows merged as in wave_sum).
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_f<0xB1>(v));
    v = fmaxf(v, dpp_f<0x4E>(v));
    v = fmaxf(v, dpp_f<0x124>(v));
    v = fmaxf(v, dpp_f<0x128>(v));
    v = fmaxf(v, dpp_f<0x142, 0xA>(v));
    v = fmaxf(v, dpp_f<0x143, 0xC>(v));
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

template <int LG>
constexpr uint32_t cells_bytes() {
    return 16u << (2 * LG);
}

// Centroids of a block from the partial sums of its nslot workgroups (0: as
// they are in cent), stored by the block's first workgroup, and the lists of
// the workgroup's 16 x 16 cells. Bound by its serial steps, so 16 waves share
// them: a quarter of the partial sums each thread (all its loads in flight
// together), then a wave per 4 x 4 cells -- one wave-wide search for the
// candidates of all 16, from which each cell's 4 lanes pick its own.
template <int LG>
__global__ __launch_bounds__(kCellT) void vq_cells_k(const uint8_t* __restrict__ slots,
                                                     uint32_t nslot, uint32_t ntile,
                                                     float2* __restrict__ cent,
                                                     uint16_t* __restrict__ Cb,
                                                     u32x4* __restrict__ lists) {
    constexpr uint32_t kTiles = 1u << (LG - 4);  // 16-cell tiles per axis
    constexpr float kW = 2.0f / (1 << LG);       // cell width
    __shared__ float2 cs[kCB];
    __shared__ float hs[kCB];
    __shared__ unsigned long long px[4][kCB], py[4][kCB];
    __shared__ uint32_t pn[4][kCB];
    __shared__ uint8_t coarse[16][kCB];
    const uint32_t b = blockIdx.y, t = threadIdx.x, lane = t & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const size_t ci = (size_t)b * kCB + (t & (kCB - 1));
    if (nslot != 0) {
        const uint32_t c = t & (kCB - 1), part = t / kCB;
        const uint8_t* p0 = slots + (size_t)b * nslot * kSlotB;
        unsigned long long x = 0, y = 0;
        uint32_t n = 0;
#pragma unroll 4
        for (uint32_t k = part; k < nslot; k += 4) {
            const uint8_t* p = p0 + (size_t)k * kSlotB;
            x += reinterpret_cast<const unsigned long long*>(p)[c];
            y += reinterpret_cast<const unsigned long long*>(p + 2048)[c];
            n += reinterpret_cast<const uint32_t*>(p + 4096)[c];
        }
        px[part][c] = x;
        py[part][c] = y;
        pn[part][c] = n;
        __syncthreads();
    }
    if (t < kCB) {
        float2 v = cent[ci];
        if (nslot != 0) {
            const unsigned long long x = px[0][t] + px[1][t] + px[2][t] + px[3][t];
            const unsigned long long y = py[0][t] + py[1][t] + py[2][t] + py[3][t];
            const uint32_t n = pn[0][t] + pn[1][t] + pn[2][t] + pn[3][t];
            if (n != 0) {
                const double ax = (double)(long long)x * 0x1p-40 / (double)n;
                const double ay = (double)(long long)y * 0x1p-40 / (double)n;
                v = make_float2((float)ax, (float)ay);
                // the other workgroups use cent[ci] only where n is 0
                if (blockIdx.x == 0) vq_store_mean(ax, ay, ci, cent, Cb);
            }
        }
        cs[t] = v;
        hs[t] = vq_hc(v.x, v.y);
    }
    __syncthreads();

    const uint32_t tile0 = blockIdx.x * ntile, tile1 = min(tile0 + ntile, kTiles * kTiles);
    for (uint32_t tile = tile0; tile < tile1; ++tile) {
        if (tile != tile0) __syncthreads();  // coarse[] is read
        // coarse cell (wave % 4, wave / 4) of the tile: 4 x 4 cells
        const uint32_t tx = tile & (kTiles - 1), ty = tile / kTiles;
        const float x0 = -1.0f + (float)(tx * 16 + (wave & 3) * 4) * kW;
        const float y0 = -1.0f + (float)(ty * 16 + (wave >> 2) * 4) * kW;
        uint32_t nc = 0;
        {
            const float mx = x0 + 2.0f * kW, my = y0 + 2.0f * kW;
            float2 q[4];
            float sj[4], best = -INFINITY;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                q[j] = cs[lane + 64 * j];
                sj[j] = fmaf(mx, q[j].x, fmaf(my, q[j].y, hs[lane + 64 * j]));
                best = fmaxf(best, sj[j]);  // NaN: the other operand
            }
            best = wave_max(best);
            uint32_t w = 0;
            bool have = false;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const unsigned long long eq = __ballot(sj[j] == best);
                if (!have && eq != 0) {
                    have = true;
                    w = 64 * j + (uint32_t)__builtin_ctzll(eq);
                }
            }
            const float wx = cs[w].x, wy = cs[w].y, h = 2.0f * kW + kCellSlack;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t c = lane + 64 * j;
                const float dx = q[j].x - wx, dy = q[j].y - wy;
                const bool in = have && (sj[j] - best) + h * (fabsf(dx) + fabsf(dy)) >= -kCellEps &&
                                !(dx == 0.0f && dy == 0.0f && c > w);
                const unsigned long long m = __ballot(in);
                if (in) coarse[wave][nc + (uint32_t)__popcll(m & ((1ull << lane) - 1))] = (uint8_t)c;
                nc += (uint32_t)__popcll(m);
            }
        }
        __syncthreads();

        // cell (u % 4, u / 4) of the coarse cell: lanes 4u .. 4u + 3, lane sub
        // takes candidates sub, sub + 4, ...
        const uint32_t u = lane >> 2, sub = lane & 3;
        const float mx = x0 + ((float)(u & 3) + 0.5f) * kW, my = y0 + ((float)(u >> 2) + 0.5f) * kW;
        float best = -INFINITY;
        uint32_t w = 0;
        for (uint32_t i = sub; i < nc; i += 4) {
            const uint32_t c = coarse[wave][i];
            const float2 q = cs[c];
            const float s = fmaf(mx, q.x, fmaf(my, q.y, hs[c]));
            if (s > best) {
                best = s;
                w = c;
            }
        }
        auto merge = [&](float ob, uint32_t ow) __attribute__((always_inline)) {
            if (ob > best || (ob == best && ow < w)) {
                best = ob;
                w = ow;
            }
        };
        merge(dpp_f<0xB1>(best), dpp_u<0xB1>(w));  // the quad's greatest score, its lowest index
        merge(dpp_f<0x4E>(best), dpp_u<0x4E>(w));
        const float wx = cs[w].x, wy = cs[w].y, h = 0.5f * kW + kCellSlack;
        uint32_t l[4] = {0, 0, 0, 0}, n = 0;
        for (uint32_t i0 = 0; i0 < nc; i0 += 4) {  // uniform
            const uint32_t i = i0 + sub, c = coarse[wave][i < nc ? i : nc - 1];
            const float2 q = cs[c];
            const float s = fmaf(mx, q.x, fmaf(my, q.y, hs[c])), dx = q.x - wx, dy = q.y - wy;
            const bool in = i < nc && (s - best) + h * (fabsf(dx) + fabsf(dy)) >= -kCellEps &&
                            !(dx == 0.0f && dy == 0.0f && c > w);
            const uint32_t m = (uint32_t)(__ballot(in) >> (lane & 60)) & 15u;  // this quad's
            const uint32_t at = n + 1 + (uint32_t)__popc(m & ((1u << sub) - 1));
            const uint32_t v = in ? c << (8 * (at & 3)) : 0u;
#pragma unroll
            for (int k = 0; k < 4; ++k) l[k] |= (at >> 2) == (uint32_t)k ? v : 0u;
            n += (uint32_t)__popc(m);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            l[k] |= dpp_u<0xB1>(l[k]);
            l[k] |= dpp_u<0x4E>(l[k]);
        }
        const float2 q0 = cs[0];
        if (q0.x != q0.x || q0.y != q0.y) l[0] = n = 0;
        l[0] |= n > kCellCap ? kCellFull : n;
        const uint32_t cy = ty * 16 + (wave >> 2) * 4 + (u >> 2), cx = tx * 16 + (wave & 3) * 4 + (u & 3);
        if (sub == 0)
            lists[((size_t)b << (2 * LG)) + (cy << LG) + cx] =
                u32x4{l[0], l[1], l[2], l[3]};
    }
}

// A block's lists and centroids into LDS.
template <int LG>
__device__ __forceinline__ void vq_load_cells(const u32x4* lists, const float2* cent, uint32_t b,
                                              u32x4* lc, float2* cs) {
    const u32x4* src = lists + ((size_t)b << (2 * LG));
    for (uint32_t i = threadIdx.x; i < (1u << (2 * LG)); i += blockDim.x) lc[i] = src[i];
    for (uint32_t c = threadIdx.x; c < kCB; c += blockDim.x) cs[c] = cent[(size_t)b * kCB + c];
}

// vq_nearest from the point's cell list.
// The random LDS reads bound the passes: -|c|^2/2 read from LDS instead of three
// VALU operations a score took a whole quantisation from 1501 to 1661 us
// (14336x4096, codebook per 256 rows).
template <int LG>
__device__ __forceinline__ uint32_t vq_nearest_cell(float px, float py, const uint32_t* lc,
                                                    const float2* cs) {
    constexpr float kHalf = (float)(1 << (LG - 1)), kLast = (float)((1 << LG) - 1);
    const uint32_t ix = (uint32_t)fminf(fmaxf(fmaf(px, kHalf, kHalf), 0.0f), kLast);
    const uint32_t iy = (uint32_t)fminf(fmaxf(fmaf(py, kHalf, kHalf), 0.0f), kLast);
    const uint32_t* l = lc + ((iy << LG) + ix) * 4;
    float bs = -INFINITY;
    uint32_t best = 0;
    auto score = [&](uint32_t c) __attribute__((always_inline)) {
        const float2 q = cs[c];
        const float s = fmaf(px, q.x, fmaf(py, q.y, vq_hc(q.x, q.y)));
        if (s > bs) {
            bs = s;
            best = c;
        }
    };
    const uint32_t w0 = l[0], n = w0 & 0xFF;
    score((w0 >> 8) & 0xFF);
    score((w0 >> 16) & 0xFF);
    score(w0 >> 24);
    if (n > 3) {
        if (n == kCellFull) {
            bs = -INFINITY;
            for (uint32_t c = 0; c < kCB; ++c) score(c);
            return best;
        }
#pragma unroll 1
        for (uint32_t k = 1; k < 4 && n >= 4 * k; ++k) {
            const uint32_t w = l[k];
            score(w & 0xFF);
            score((w >> 8) & 0xFF);
            score((w >> 16) & 0xFF);
            score(w >> 24);
        }
    }
    return best;
}

// A coordinate in 2^-40 fixed point (towards zero, NaN 0: __float2ll_rz of p *
// 2^40), plus the bits of kFixOne: an integer of at most 41 bits lies in the low
// bits of its sum with 1.5 * 2^52. The compiler's 64-bit conversion takes about
// three times the instructions of this one (14336x4096, codebook per 256
// rows, a whole quantisation: 1535 -> 1506 us).
constexpr unsigned long long kFixOne = 0x4338000000000000ull;
__device__ __forceinline__ unsigned long long vq_fix(float p) {
    const float v = fabsf(p) <= 2.0f ? __builtin_truncf(p * 0x1p40f) : 0.0f;
    return __builtin_bit_cast(unsigned long long, (double)v + 0x1.8p52);
}

// One Lloyd assignment: the sums of a workgroup's points (a contiguous share
// of the block's sample) per centroid, to the workgroup's own slot.
template <int LG>
__global__ __launch_bounds__(kPT) void vq_lloyd_k(const float2* __restrict__ pts,
                                                  uint32_t ns_stride, uint32_t M, uint32_t K,
                                                  uint32_t R, uint32_t sample,
                                                  const float2* __restrict__ cent,
                                                  const u32x4* __restrict__ lists,
                                                  uint8_t* __restrict__ slots) {
    extern __shared__ __align__(16) unsigned char smem[];
    u32x4* lc = reinterpret_cast<u32x4*>(smem);
    float2* cs = reinterpret_cast<float2*>(smem + cells_bytes<LG>());
    unsigned long long* sx = reinterpret_cast<unsigned long long*>(cs + kCB);
    unsigned long long* sy = sx + kCB;
    uint32_t* sn = reinterpret_cast<uint32_t*>(sy + kCB);
    const uint32_t b = blockIdx.y, rows = min(R, M - b * R), t = threadIdx.x;
    const uint32_t ns = min(rows * (K / 2), sample);
    vq_load_cells<LG>(lists, cent, b, lc, cs);
    for (uint32_t c = t; c < kCB; c += kPT) {
        sx[c] = sy[c] = 0;
        sn[c] = 0;
    }
    __syncthreads();
    const uint32_t per = (ns + gridDim.x - 1) / gridDim.x;
    const uint32_t j0 = min(blockIdx.x * per, ns), j1 = min(j0 + per, ns);
    const float2* P = pts + (size_t)b * ns_stride;
    constexpr int U = 4;  // points in flight a thread
    for (uint32_t j = j0 + t; j < j1; j += U * kPT) {
        float2 p[U];
#pragma unroll
        for (int u = 0; u < U; ++u) p[u] = P[min(j + u * kPT, j1 - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (j + u * kPT < j1) {
                const uint32_t a =
                    vq_nearest_cell<LG>(p[u].x, p[u].y, reinterpret_cast<const uint32_t*>(lc), cs);
                atomicAdd(&sx[a], vq_fix(p[u].x));
                atomicAdd(&sy[a], vq_fix(p[u].y));
                atomicAdd(&sn[a], 1u);
            }
        }
    }
    __syncthreads();
    uint8_t* slot = slots + ((size_t)b * gridDim.x + blockIdx.x) * kSlotB;
    for (uint32_t c = t; c < kCB; c += kPT) {
        const unsigned long long ones = kFixOne * sn[c];  // modulo 2^64, as the sums
        reinterpret_cast<unsigned long long*>(slot)[c] = sx[c] - ones;
        reinterpret_cast<unsigned long long*>(slot + 2048)[c] = sy[c] - ones;
        reinterpret_cast<uint32_t*>(slot + 4096)[c] = sn[c];
    }
}

// The indices of a workgroup's share of its block: thread by thread 4 pairs
// (one index word) of one row.
template <int LG, int DT>
__global__ __launch_bounds__(kPT) void vq_label_k(const void* __restrict__ W, uint32_t M,
                                                  uint32_t K, uint32_t G, uint32_t R,
                                                  const float* __restrict__ sc,
                                                  const float2* __restrict__ cent,
                                                  const u32x4* __restrict__ lists,
                                                  uint8_t* __restrict__ IDX) {
    extern __shared__ __align__(16) unsigned char smem[];
    u32x4* lc = reinterpret_cast<u32x4*>(smem);
    float2* cs = reinterpret_cast<float2*>(smem + cells_bytes<LG>());
    const uint32_t b = blockIdx.y, r0 = b * R, rows = min(R, M - r0), t = threadIdx.x;
    vq_load_cells<LG>(lists, cent, b, lc, cs);
    __syncthreads();
    const uint32_t wpr = K / 8, nw = rows * wpr;  // index words per row, of the block
    const uint32_t per = (nw + gridDim.x - 1) / gridDim.x;
    const uint32_t j0 = min(blockIdx.x * per, nw), j1 = min(j0 + per, nw);
    uint32_t* out = reinterpret_cast<uint32_t*>(IDX) + (size_t)r0 * wpr;
    for (uint32_t j = j0 + t; j < j1; j += kPT) {
        const uint32_t r = j / wpr, i0 = (j - r * wpr) * 4;
        uint32_t word = 0;
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const float2 p = vq_pair<DT>(W, sc, K, G, r0 + r, i0 + u);
            word |= vq_nearest_cell<LG>(p.x, p.y, reinterpret_cast<const uint32_t*>(lc), cs)
                    << (8 * u);
        }
        out[j] = word;
    }
}

// Where the lists fit: those of the iterations and the partial sums lie in
// IDX (only the last pass writes it), those of the last pass in the sample,
// which no one reads any more by then.
struct CellPlan {
    int lg;           // 6 or 5; 0: no room, full scan
    uint32_t nslot;   // workgroups (and partial sums) per block of vq_lloyd_k
};
CellPlan cell_plan(uint32_t M, uint32_t K, uint32_t R, uint32_t ns) {
    const uint64_t nblk = (M + R - 1) / R, idx = (uint64_t)M * (K / 2), cu = cu_count();
    for (int lg = 6; lg >= 5; --lg) {
        const uint64_t lb = 16ull << (2 * lg);
        if (lb > 8ull * ns || nblk * (lb + kSlotB) + 16 > idx) continue;
        // two workgroups a CU fit, in one round (rounded up, 56 blocks took 560
        // workgroups and a second round for 48 of them); at least 4096 points
        // each, and at most 48 a block: every workgroup of vq_cells_k reads
        // all partial sums
        uint64_t n = nblk < 2 * cu ? 2 * cu / nblk : 1, most = (ns + 4095) / 4096;
        if (n > most) n = most;
        if (n > 48) n = 48;
        const uint64_t fit = ((idx - 16) / nblk - lb) / kSlotB;
        if (n > fit) n = fit;
        return CellPlan{lg, (uint32_t)n};
    }
    return CellPlan{0, 0};
}

template <int LG, int DT>
hipError_t vq_cells_go(const void* W, uint32_t M, uint32_t K, uint32_t G, uint32_t R,
                       uint32_t iters, uint32_t sample, uint32_t ns, uint32_t nslot, uint8_t* IDX,
                       uint16_t* Cb, const float* sc, float2* pts, float2* cent, hipStream_t s) {
    const uint32_t nblk = (M + R - 1) / R;
    u32x4* lists = reinterpret_cast<u32x4*>(((uintptr_t)IDX + 15) & ~(uintptr_t)15);
    uint8_t* slots = reinterpret_cast<uint8_t*>(lists) + (size_t)nblk * cells_bytes<LG>();
    u32x4* last = reinterpret_cast<u32x4*>(pts);
    const size_t lds_label = cells_bytes<LG>() + kCB * 8, lds_lloyd = lds_label + kSlotB;
    hipError_t e = hipSuccess;
    if (lds_lloyd > 64 * 1024) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(vq_lloyd_k<LG>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_lloyd);
        if (e != hipSuccess) return e;
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(vq_label_k<LG, DT>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_label);
        if (e != hipSuccess) return e;
    }
    // tiles of 16 x 16 cells a workgroup: one, or as many as leave one round of
    // two workgroups a CU (56 blocks: 16 us at one tile and two rounds)
    const uint32_t tiles = (1u << (2 * LG)) / 256, cu2 = 2 * cu_count();
    uint32_t ntile = ((uint64_t)tiles * nblk + cu2 - 1) / cu2;
    if (ntile > tiles) ntile = tiles;
    const dim3 gc((tiles + ntile - 1) / ntile, nblk);
    for (uint32_t it = 0; it <= iters; ++it) {
        vq_cells_k<LG><<<gc, kCellT, 0, s>>>(slots, it == 0 ? 0 : nslot, ntile, cent, Cb,
                                             it == iters ? last : lists);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (it == iters) break;
        vq_lloyd_k<LG><<<dim3(nslot, nblk), kPT, lds_lloyd, s>>>(pts, ns, M, K, R, sample, cent,
                                                                 lists, slots);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    const uint32_t words = (R < M ? R : M) * (K / 8);
    uint32_t gx = nblk < cu2 ? cu2 / nblk : 1;  // one round, as vq_lloyd_k
    if (gx > (words + kPT - 1) / kPT) gx = (words + kPT - 1) / kPT;
    vq_label_k<LG, DT><<<dim3(gx, nblk), kPT, lds_label, s>>>(W, M, K, G, R, sc, cent, last, IDX);
    return hipGetLastError();
}

template <int DT>
hipError_t vq_quant_go(const void* W, uint32_t M, uint32_t K, uint32_t G, uint32_t R,
                       uint32_t iters, uint32_t sample, uint64_t seed, uint8_t* IDX, uint16_t* Cb,
                       uint16_t* S, uint8_t* ws, hipStream_t s) {
    const QWs L = qws_layout(M, K, G, R, sample);
    float* sc = reinterpret_cast<float*>(ws + L.sc);
    float2* pts = reinterpret_cast<float2*>(ws + L.pts);
    float2* cent = reinterpret_cast<float2*>(ws + L.cent);
    VqAcc* acc = reinterpret_cast<VqAcc*>(ws + L.acc);
    const uint32_t nblk = (M + R - 1) / R;
    vq_scale_k<DT><<<M, kQT, (K / 32) * sizeof(float), s>>>(W, K, G, S, sc);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // an XCD a block: 106 -> 61 us at 56 blocks of 256 x 4096; with few blocks
    // XCDs would idle, and from 8192 the grid would pass its limits
    const uint32_t xcd = nblk >= 16 && nblk <= 8192;
    vq_sample_k<DT><<<dim3((L.ns + kQT - 1) / kQT, xcd ? (nblk + 7) / 8 * 8 : nblk), kQT, 0, s>>>(
        W, M, K, G, R, sample, L.ns, nblk, xcd, seed, sc, pts, cent, Cb, acc);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const CellPlan cp = cell_plan(M, K, R, L.ns);
    if (cp.lg == 6)
        return vq_cells_go<6, DT>(W, M, K, G, R, iters, sample, L.ns, cp.nslot, IDX, Cb, sc, pts,
                                  cent, s);
    if (cp.lg == 5)
        return vq_cells_go<5, DT>(W, M, K, G, R, iters, sample, L.ns, cp.nslot, IDX, Cb, sc, pts,
                                  cent, s);
    const dim3 ga((L.ns + kQT * kPPT - 1) / (kQT * kPPT), nblk);
    for (uint32_t it = 0; it < iters; ++it) {
        vq_km_assign_k<<<ga, kQT, 0, s>>>(pts, L.ns, M, K, R, sample, cent, acc);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        vq_km_update_k<<<nblk, kCB, 0, s>>>(acc, cent, Cb);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    const dim3 gf(M, (K / 2 + kQT * kPPT - 1) / (kQT * kPPT));
    vq_assign_k<DT><<<gf, kQT, 0, s>>>(W, K, G, R, sc, cent, IDX);
    return hipGetLastError();
}

}  // namespace

size_t vq_quant_ws_bytes(uint32_t M, uint32_t K, uint32_t scale_group, uint32_t rows_per_cb,
                         uint32_t sample) {
    return qws_layout(M, K, scale_group, rows_per_cb, sample).total;
}

hipError_t launch_vq_quantize(const void* W, int w_dtype, uint32_t M, uint32_t K,
                              uint32_t rows_per_cb, uint32_t scale_group, uint32_t iters,
                              uint32_t sample, uint64_t seed, uint8_t* IDX, uint16_t* Cb,
                              uint16_t* S, void* ws, hipStream_t s) {
    uint8_t* w = reinterpret_cast<uint8_t*>(ws);
    if (w_dtype == KQ_F32)
        return vq_quant_go<KQ_F32>(W, M, K, scale_group, rows_per_cb, iters, sample, seed, IDX, Cb,
                                   S, w, s);
    if (w_dtype == KQ_BF16)
        return vq_quant_go<KQ_BF16>(W, M, K, scale_group, rows_per_cb, iters, sample, seed, IDX,
                                    Cb, S, w, s);
    return vq_quant_go<KQ_F16>(W, M, K, scale_group, rows_per_cb, iters, sample, seed, IDX, Cb, S,
                               w, s);
}

}  // namespace kq
