// kq_skinny_kernel.h -- skinny GEMM (2 to 16 tokens in one pass) on the gfx950
// matrix cores for both weight formats: int4 group-affine (KIND 0) and
// codebook pairs (KIND 1). Instantiated in kq_skinny_*.hip.
//
//   y[t,m] = sum_g S[m,g] * (w[m,g,:] . x[t,g,:]) (+ B[m,g] * sum(x[t,g,:]))
//
// One v_mfma_f32_16x16x32_f16 takes 32 k of a 16-row tile and all tokens
// (A = x, rows = tokens; B = weights, columns = rows; lane L holds row L%16,
// 8 k of group L/16; D lane L: tokens 4(L/16)+r of row L%16). Both formats
// store 8 weights of a row in one 32-bit word (8 nibbles, or 4 one-byte
// indices of weight pairs), so the memory side is the same code:
//
//   * a step is a pair of 128-k spans, 128 bytes a row. A load instruction
//     reads whole 128-byte lines of 8 rows (64 bytes of 16 rows, the operand
//     layout, streams ~20% slower): lane (n, kg) loads chunk 4 (n/8) + kg of
//     row 8h + n%8, and one DPP move per register (row_ror:8 into half of
//     each row) turns the two loads h = 0, 1 into row n's chunks kg and
//     4 + kg. No LDS stage stands between memory and the matrix cores.
//   * x: a load instruction reads 512 bytes of 2 tokens (64 bytes of 16
//     tokens, the operand layout, cost 2-5 us more a call at 16 tokens: it is
//     the rows an instruction touches that count) and goes through a stage of
//     the wave's own in LDS, swizzled by the token. (Up to 8 tokens, X8, rows
//     of D past the tokens hold other tokens' products; nothing reads them.)
//   * v_permlane swaps bring the 32 k of an MFMA into one scale group, and x
//     is read back in that order.
//   * int4 words become 64 + q (AND-OR), and per group acc += S * D with
//     D = sum (64 + q) x; sum_g (B - 64 S) * sum(x) of four groups is one
//     fp32 MFMA, its sum(x) operand from MFMAs of x against constant rows.
//     (With 1024 + q in half the words, two instructions fewer a word pair
//     need five, the fp32 sums are ten times as far off.)
//   * codebook words are 4 LDS lookups, one of 64 interleaved copies per lane
//     (kq_vq.hip), the address one v_perm_b32.
//   * interleaved scales and biases: lane (n, kg) loads those of group kg of
//     row n, which is the bias MFMA's operand, and ds_bpermute hands a scale to
//     every lane of its row. Separate arrays (and codebook scales) have half
//     the bytes a row and load: they are loaded once per window of 4 steps
//     (28672 x 8192, 16 tokens, bf16: 46 -> 39 us; interleaved ones are faster
//     per step, 40 against 43 us at 8 tokens, as the window's copies spill).
//     Two-byte scales may start at any of them: gfx950 buffer loads take
//     unaligned words, and no word reaches past its row.
//   * the last pair of a row ends at K (it overlaps the pair before unless
//     256 divides K, with the k already taken zeroed in x), so every load of
//     weights and scales lies inside its row for any K >= 256. (An infinite
//     codeword or scale would meet those zeros and give NaN.)
//
// Work split: a workgroup of P x Q waves owns tiles_wg row tiles; wave (p, q)
// takes K part p (J pairs) of tiles (round * Q + q) * T ..., T at a time, and
// the parts of a round are summed in LDS in a fixed order. What bounds it: the
// weight stream plus the first loads' latency; issue takes ~16 VALU per MFMA.
#pragma once
#include "kq_int4_mfma_kernel.h"

namespace kq {
namespace skinny {

constexpr uint32_t kPair = 256;      // k of a step
constexpr uint32_t kWin = 4;         // steps of a scale window
// Waves a workgroup: one tile a wave and up to 8 tokens leave room for 16 waves (4 a
// SIMD, 128 VGPRs: 106-128 in use, 7 spilled with 64-wide groups' separate scales).
__host__ __device__ constexpr uint32_t max_waves(uint32_t T, bool x8) { return T == 1 && x8 ? 16 : 8; }

struct Args {
    const uint8_t* W;    // nibbles or indices, K / 2 bytes a row
    const uint16_t* S;   // interleaved (scale, bias) pairs, or scales
    const uint16_t* B;   // biases (separate layout only)
    const uint16_t* C;   // codebooks (KIND 1)
    const uint16_t* X;
    void* Y;
    uint32_t M, K, ntok, y_f32;
    uint32_t gpr;        // scale groups per row
    uint32_t gshift;     // KIND 1, groups of 128 or more: log2 of the group
    uint32_t P, Q, J, NP;  // K parts, row lanes, pairs per part, pairs per row
    uint32_t tiles_wg, rounds;
    uint32_t rpc, cb_lds;  // KIND 1: rows per codebook (multiple of 16), LDS bytes of the copies
    uint32_t part_lds;     // LDS bytes of the K-part sums (the x stages follow)
};

// Ring depth in steps. Two everywhere: a K part has 2-14 steps, and the loads a
// deeper ring issues past a short part's end cost more than they hide.
constexpr int kDepth = 2;

// One step's registers. m, int4 interleaved: lane (n, kg) holds (scale, bias)
// of groups 4h + kg of row n. Else (steps that begin a window): lane (n, kg)
// holds the scales of row n for the window's step kg, two a dword, then the
// biases.
template <int T, bool X8, int MR>
struct Slot {
    u32x4 w[T][2];
    u32x4 x[X8 ? 4 : 8];
    uint32_t m[T][MR ? MR : 1];
};

template <int BANK>
__device__ __forceinline__ u32x4 ror8_into(u32x4 old, u32x4 src) {
    u32x4 r;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        r[k] = (uint32_t)__builtin_amdgcn_update_dpp((int)old[k], (int)src[k], 0x128, 0xF, BANK, false);
    return r;
}

// 64 + nibble of a word's nibbles (all four pairs in bits 4-7 of a half: 64 is
// the least that an exponent can carry there), in dequant order.
__device__ __forceinline__ f16x8 dq64(uint32_t w, const DequantConsts& k) {
    return __builtin_bit_cast(f16x8, u32x4{and_or(w << 4, k.hi, k.e64), and_or(w, k.hi, k.e64),
                                           and_or(w >> 4, k.hi, k.e64), and_or(w >> 8, k.hi, k.e64)});
}

// x pairs in the order the weights' dequantisation gives them.
template <int KIND>
__device__ __forceinline__ u32x4 xorder(u32x4 v) {
    return KIND == 0 ? __builtin_bit_cast(u32x4, mfma::xperm(v)) : v;
}

__device__ __forceinline__ uint32_t lds_word(uint32_t addr) {
    return *(const __attribute__((address_space(3))) uint32_t*)(uintptr_t)addr;
}
// The codewords of a word's 4 indices, from the lane's copies (lane4 = lane << 2).
__device__ __forceinline__ f16x8 codewords(uint32_t w, uint32_t lane4) {
    const u32x4 v{lds_word(__builtin_amdgcn_perm(w, lane4, 0x0C0C0400u)),
                  lds_word(__builtin_amdgcn_perm(w, lane4, 0x0C0C0500u)),
                  lds_word(__builtin_amdgcn_perm(w, lane4, 0x0C0C0600u)),
                  lds_word(__builtin_amdgcn_perm(w, lane4, 0x0C0C0700u))};
    return __builtin_bit_cast(f16x8, v);
}

// KIND 0: int4, GM the quant group. KIND 1: codebook, GM 32 or 64 the scale
// group, 128 a group of 128 or more (power of two), 0 one scale per row.
template <int KIND, int GM, bool SB, bool BF, int T, bool X8>
__global__ __launch_bounds__(64 * max_waves(T, X8)) void skinny_k(Args A) {
    constexpr int NGP = GM ? 256 / GM : 1;   // groups per pair (GM 0: one chain)
    constexpr int NG = GM ? 128 / GM : 1;    // groups per span
    constexpr int PER = GM ? 4 / NG : 4;     // MFMAs per group and span
    constexpr int NC = KIND == 1 && NG < 2 ? 2 : NG, PERC = 4 / NC;  // chains a span, MFMAs a chain
    constexpr int NH = (NGP + 3) / 4;        // quads of groups (bias MFMAs) per pair
    constexpr int GR = GM ? GM : 128;        // regroup / x order
    constexpr int D = kDepth, NX = X8 ? 4 : 8;
    constexpr bool kFar = KIND == 1 && GM == 128;          // a group may be longer than a span
    constexpr int MA = SB ? NH : kFar ? 2 : NGP / 2;       // dwords of one array
    constexpr int MR = GM == 0 ? 0 : KIND == 0 && !SB ? 2 * MA : MA;
    constexpr uint32_t MB = SB ? 4 : 2;      // meta bytes per group (per array)

    extern __shared__ __align__(16) unsigned char smem[];
    float* part = reinterpret_cast<float*>(smem + A.cb_lds);

    const uint32_t K = A.K, M = A.M;
    const uint32_t tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t q = wave / A.P, p = wave - q * A.P;
    const uint32_t n = lane & 15, kg = lane >> 4;
    const uint32_t row0 = blockIdx.x * A.tiles_wg * 16;
    const uint32_t rows = min(A.tiles_wg * 16, M - row0);
    const uint32_t rowb = K >> 1, srowb = A.gpr * MB;
    constexpr uint32_t kOOB = 0x80000000u;

    // descriptors from the workgroup's first row: rows past M load zeros
    const uint8_t* Wp = A.W + (size_t)row0 * rowb;
    const uint32_t wbytes = rows * rowb;
    const rsrc_t rS = make_rsrc(reinterpret_cast<const uint8_t*>(A.S) + (size_t)row0 * srowb, rows * srowb);
    const rsrc_t rB = make_rsrc(reinterpret_cast<const uint8_t*>(KIND == 0 && !SB ? A.B : A.S) +
                                    (size_t)row0 * srowb, rows * srowb);

    // the codebook of the workgroup's rows
    u32x4 cbq{0, 0, 0, 0};
    if constexpr (KIND == 1)
        cbq = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(A.C + (size_t)(row0 / A.rpc) * 512, 1024),
                                                    lane * 16, 0, 0);

    // lane parts of the addresses
    // x load j: the pair's 256 k of tokens 2j, 2j + 1 (512 bytes each)
    uint32_t xvo[NX], xk[NX];  // byte offset, k within the pair
#pragma unroll
    for (int j = 0; j < NX; ++j) {
        const uint32_t t = 2 * j + (lane >> 5);
        xk[j] = (lane & 31) * 8;
        xvo[j] = (t < A.ntok ? t : A.ntok - 1) * K * 2 + xk[j] * 2;
    }
    // the wave's x stage: 512 bytes a token, its 16-byte chunks swizzled by the token
    unsigned char* xst = smem + A.cb_lds + A.part_lds + wave * (uint32_t)(X8 ? 4096 : 8192);
    uint32_t xwo[NX], xro[4];
#pragma unroll
    for (int j = 0; j < NX; ++j) {
        const uint32_t t = 2 * j + (lane >> 5);
        xwo[j] = t * 512 + (((lane & 31) ^ t) * 16);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // span 0; span 1 is 256 bytes on (bit 4 of the chunk)
        const uint32_t t = X8 ? n & 7 : n;
        xro[j] = t * 512 + ((mfma::xword<GR>(j, kg) ^ t) * 16);
    }
    const uint32_t wlane = (n & 7) * rowb + (4 * (n >> 3) + kg) * 16, wtile = 16 * rowb, w8 = 8 * rowb;

    struct Cur {
        uint32_t j, round;
    };
    const uint32_t jn = A.NP > p * A.J ? min(A.J, A.NP - p * A.J) : 0u;
    auto advance = [&](Cur& c) __attribute__((always_inline)) {
        if (++c.j == A.J) {
            c.j = 0;
            ++c.round;
        }
    };
    auto tile_of = [&](uint32_t round) __attribute__((always_inline)) {  // within the workgroup
        return (round * A.Q + q) * T;
    };
    Slot<T, X8, MR> ring[D];
    uint32_t mw[T][MR ? MR : 1];  // the current window's scales (not interleaved)

    auto issue = [&](Slot<T, X8, MR>& e, Cur c) __attribute__((always_inline)) {
        const bool ok = c.round < A.rounds && c.j < jn;  // uniform
        const uint32_t pr = p * A.J + (ok ? c.j : 0u);
        const uint32_t k0 = __builtin_amdgcn_readfirstlane(min(pr * kPair, K - kPair));
        const uint32_t tile = __builtin_amdgcn_readfirstlane(tile_of(c.round < A.rounds ? c.round : 0u));
        const uint32_t off = ok ? 0u : kOOB;
        // a step past the end loads zeros, without traffic
        const rsrc_t rW = make_rsrc(Wp, ok ? wbytes : 0u), rX = make_rsrc(A.X, ok ? A.ntok * K * 2 : 0u);
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                e.w[i][h] = __builtin_amdgcn_raw_buffer_load_b128(
                    rW, wlane + (tile + i) * wtile + h * w8, k0 >> 1, kNT);
        if constexpr (MR > 0 && SB) {
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const uint32_t go = NGP >= 4 || kg < 2 ? off + (k0 / (GM ? GM : 1) + 4 * h + kg) * MB : kOOB;
#pragma unroll
                for (int i = 0; i < T; ++i)
                    e.m[i][h] = __builtin_amdgcn_raw_buffer_load_b32(
                        rS, ((tile + i) * 16 + n) * srowb + go, 0, 0);
            }
        }
        if constexpr (MR > 0 && !SB) {
            if (c.j % kWin == 0) {  // uniform
                // lane (n, kg): the window's step kg (past the part's end: its last)
                const uint32_t pm = p * A.J + min(c.j + kg, max(jn, 1u) - 1);
                const uint32_t km = min(pm * kPair, K - kPair);
#pragma unroll
                for (int i = 0; i < T; ++i) {
                    const uint32_t ro = off + ((tile + i) * 16 + n) * srowb;
                    if constexpr (kFar) {
                        e.m[i][0] = __builtin_amdgcn_raw_buffer_load_b16(rS, ro + (km >> A.gshift) * 2, 0, 0);
                        e.m[i][1] = __builtin_amdgcn_raw_buffer_load_b16(rS, ro + ((km + 128) >> A.gshift) * 2, 0, 0);
                    } else {
                        const uint32_t vo = ro + km / (GM ? GM : 1) * MB;
#pragma unroll
                        for (int a = 0; a < MR / MA; ++a) {
                            const rsrc_t r = a ? rB : rS;
                            uint32_t* d = &e.m[i][a * MA];
                            if constexpr (MA == 1) d[0] = __builtin_amdgcn_raw_buffer_load_b32(r, vo, 0, 0);
                            else if constexpr (MA == 2) {
                                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, vo, 0, 0);
                                d[0] = v.x;
                                d[1] = v.y;
                            } else {
#pragma unroll
                                for (int z = 0; z < MA / 4; ++z) {
                                    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, vo + 16 * z, 0, 0);
#pragma unroll
                                    for (int y = 0; y < 4; ++y) d[4 * z + y] = v[y];
                                }
                            }
                        }
                    }
                }
            }
        }
        const uint32_t lo = pr * kPair - k0;  // k of the pair that the pair before took
#pragma unroll
        for (int j = 0; j < NX; ++j)
            e.x[j] = __builtin_amdgcn_raw_buffer_load_b128(rX, xk[j] >= lo ? xvo[j] : kOOB, k0 * 2, 0);
    };

    Cur ci{0, 0};
    mfma::static_for<D>([&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        issue(ring[k], ci);
        advance(ci);
        __builtin_amdgcn_sched_barrier(0);
    });

    if constexpr (KIND == 1) {
        // 64 copies of every entry, entry e at e << 8: wave w stores copy groups
        // (w' + lane) % 16, w' = w, w + waves, ..., of the lane's 4 entries
        // (conflict-free)
        unsigned char* eb = smem + lane * 1024;
        for (uint32_t w2 = wave; w2 < 16; w2 += nthr >> 6) {
            const uint32_t g = (w2 + lane) & 15;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                *reinterpret_cast<u32x4*>(eb + k * 256 + g * 16) = u32x4{cbq[k], cbq[k], cbq[k], cbq[k]};
        }
        __syncthreads();
    }

    const DequantConsts kc;
    // ac[g]: ones in row 4g, the operand of the x sums
    f16x8 ac[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const uint32_t o = n == 4u * g ? 0x3C003C00u : 0u;
        ac[g] = __builtin_bit_cast(f16x8, u32x4{o, o, o, o});
    }
    const f32x4 zero{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[T];
#pragma unroll
    for (int i = 0; i < T; ++i) acc[i] = zero;

    auto store = [&](uint32_t row, uint32_t t, float v) __attribute__((always_inline)) {
        if (t < A.ntok && row < rows) {
            const size_t o = (size_t)t * M + row0 + row;
            if (A.y_f32) reinterpret_cast<float*>(A.Y)[o] = v;
            else reinterpret_cast<uint16_t*>(A.Y)[o] = f2h(v);
        }
    };
    auto finish = [&](uint32_t round) __attribute__((always_inline)) {
        if constexpr (KIND == 1 && GM == 0) {  // one scale per row
#pragma unroll
            for (int i = 0; i < T; ++i) {
                const uint32_t row = (tile_of(round) + i) * 16 + n;
                const float s = h2f((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rS, row * 2, 0, 0));
                acc[i] *= s;
            }
        }
        if (A.P == 1) {
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) store((tile_of(round) + i) * 16 + n, 4 * kg + r, acc[i][r]);
        } else {
            float* buf = part + (size_t)(A.rounds > 1 ? round & 1 : 0) * (A.P * A.Q) * T * 256;
            float* pw = buf + (size_t)wave * T * 256;
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) pw[(i * 4 + r) * 64 + lane] = acc[i][r];
            __syncthreads();
            const uint32_t nout = A.Q * T * 16 * A.ntok;
            for (uint32_t o = tid; o < nout; o += nthr) {
                const uint32_t nn = o & 15, rest = o >> 4, ti = rest % (A.Q * T), t = rest / (A.Q * T);
                const uint32_t qq = ti / T, i = ti % T;
                const float* pr = buf + ((size_t)(qq * A.P * T + i) * 4 + (t & 3)) * 64 + 16 * (t >> 2) + nn;
                float v = 0.0f;
                for (uint32_t pp = 0; pp < A.P; ++pp) v += pr[(size_t)pp * T * 256];
                store((round * A.Q * T + ti) * 16 + nn, t, v);
            }
        }
#pragma unroll
        for (int i = 0; i < T; ++i) acc[i] = zero;
    };

    auto step = [&](const Slot<T, X8, MR>& e, Cur c) __attribute__((always_inline)) {
        if constexpr (MR > 0 && !SB) {
            if (c.j % kWin == 0) {  // uniform
#pragma unroll
                for (int i = 0; i < T; ++i)
#pragma unroll
                    for (int z = 0; z < MR; ++z) mw[i][z] = e.m[i][z];
            }
        }
        if (c.j < jn) {  // uniform
            // x to the wave's LDS (chunk c of token t at c ^ t), back as operands
#pragma unroll
            for (int j = 0; j < NX; ++j) *reinterpret_cast<u32x4*>(xst + xwo[j]) = xorder<KIND>(e.x[j]);
            uint32_t m[T][MR ? MR : 1];
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int z = 0; z < MR && !SB; ++z)
                    m[i][z] = mfma::bperm(4 * (n + 16 * (c.j % kWin)), mw[i][z]);
            // KIND 1: products of at most 64 k in a chain, and the step's sums
            // apart from the running ones: the vector path's error, 1e-7 (one
            // chain of all of a wave's k: 4.1e-7 at K = 28672)
            f32x4 st[T];
#pragma unroll
            for (int i = 0; i < T; ++i) st[i] = zero;
            // sum(x) of groups 4h + kg for token n, in lane (n, kg)
            f32x4 xs[NH];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                f16x8 xa[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) xa[j] = *reinterpret_cast<const f16x8*>(xst + xro[j] + s * 256);
                if constexpr (KIND == 0) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int g = s * NG + j / PER;
                        xs[g / 4] = mfma::mma16(ac[g % 4], xa[j], (4 * s + j) % (4 * PER) == 0 ? zero : xs[g / 4]);
                    }
                }
#pragma unroll
                for (int i = 0; i < T; ++i) {
                    const u32x4 r = s == 0 ? ror8_into<0xC>(e.w[i][0], e.w[i][1])
                                           : ror8_into<0x3>(e.w[i][1], e.w[i][0]);
                    uint32_t w[4] = {r.x, r.y, r.z, r.w};
                    mfma::regroup<GR>(w);
                    f32x4 dg[NC];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f16x8 b = KIND == 0 ? dq64(w[j], kc) : codewords(w[j], lane << 2);
                        dg[j / PERC] = mfma::mma16(xa[j], b, j % PERC == 0 ? zero : dg[j / PERC]);
                    }
#pragma unroll
                    for (int ch = 0; ch < NC; ++ch) {
                        if constexpr (GM == 0) st[i] += dg[ch];
                        else {
                            const int g = s * NG + ch * NG / NC;
                            uint32_t sr;
                            if constexpr (SB) sr = mfma::bperm(4 * (n + 16 * (g & 3)), e.m[i][g / 4]);
                            else if constexpr (kFar) sr = m[i][g];
                            else sr = m[i][(g >> 1) % MA] >> (16 * (g & 1));
                            const float sc = mfma::lo16f<BF>(sr);
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                if constexpr (KIND == 0) acc[i][k] = fmaf(sc, dg[ch][k], acc[i][k]);
                                else st[i][k] = fmaf(sc, dg[ch][k], st[i][k]);
                            }
                        }
                    }
                }
            }
            if constexpr (KIND == 1) {
#pragma unroll
                for (int i = 0; i < T; ++i) acc[i] += st[i];
            }
            if constexpr (KIND == 0) {
#pragma unroll
                for (int i = 0; i < T; ++i)
#pragma unroll
                    for (int h = 0; h < NH; ++h) {
                        // this lane's group 4h + kg (G 128: lanes kg >= 2 have none)
                        uint32_t sr, br;
                        if constexpr (SB) {
                            sr = e.m[i][h];
                            br = sr >> 16;
                        } else {
                            const bool lo2 = MA == 1 || kg < 2;
                            const uint32_t sh = 16 * (kg & 1);
                            sr = (lo2 ? m[i][2 * h % MA] : m[i][(2 * h + 1) % MA]) >> sh;
                            br = (lo2 ? m[i][MA + 2 * h % MA] : m[i][MA + (2 * h + 1) % MA]) >> sh;
                        }
                        float bi = fmaf(-64.0f, mfma::lo16f<BF>(sr), mfma::lo16f<BF>(br));
                        if constexpr (NGP < 4) bi = kg < 2 ? bi : 0.0f;
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[h][0], bi, acc[i], 0, 0, 0);
                    }
            }
        }
        if (c.j == A.J - 1) finish(c.round);
    };

    // every wave runs rounds * J steps (uniform), the last D apart: they issue
    // nothing past the end
    Cur cc{0, 0};
    const uint32_t total = A.rounds * A.J;
    uint32_t ns = 0;
    for (; ns + D < total; ns += D) {
        mfma::static_for<D>([&](auto dd) __attribute__((always_inline)) {
            constexpr int d = decltype(dd)::value;
            step(ring[d], cc);
            advance(cc);
            issue(ring[d], ci);
            advance(ci);
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    mfma::static_for<D>([&](auto dd) __attribute__((always_inline)) {
        constexpr int d = decltype(dd)::value;
        if (ns + d < total) step(ring[d], cc);
        advance(cc);
    });
}

template <int KIND, int GM, bool SB, bool BF, int T, bool X8>
hipError_t go(const Args& a, const Plan& pl, hipStream_t s) {
    auto kern = skinny_k<KIND, GM, SB, BF, T, X8>;
    const size_t lds = a.cb_lds + pl.part_lds + pl.x_lds;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    kern<<<pl.nwg, pl.P * pl.Q * 64, lds, s>>>(a);
    return hipGetLastError();
}

// Variants with room for their registers: no four tiles with 8 groups a step, nor
// with 4 groups' separate scales above 8 tokens (26-58 VGPRs spilled), and no
// separate scales of 8 groups up to 8 tokens (one tile spills 39-49).
template <int KIND, int GM, bool SB, bool BF>
hipError_t dispatch(const Args& a, const Plan& pl, hipStream_t s) {
    const bool x8 = a.ntok <= 8;
    if constexpr (KIND == 0 && GM == 32 && !SB) {
        if (x8 || pl.T > 2) return hipErrorInvalidValue;
        return pl.T == 1 ? go<KIND, GM, SB, BF, 1, false>(a, pl, s) : go<KIND, GM, SB, BF, 2, false>(a, pl, s);
    }
    if (pl.T == 1) return x8 ? go<KIND, GM, SB, BF, 1, true>(a, pl, s) : go<KIND, GM, SB, BF, 1, false>(a, pl, s);
    if (pl.T == 2) return x8 ? go<KIND, GM, SB, BF, 2, true>(a, pl, s) : go<KIND, GM, SB, BF, 2, false>(a, pl, s);
    if constexpr (KIND == 0 && GM == 64 && !SB) {
        if (x8) return go<KIND, GM, SB, BF, 4, true>(a, pl, s);
    } else if constexpr (GM != 32)
        return x8 ? go<KIND, GM, SB, BF, 4, true>(a, pl, s) : go<KIND, GM, SB, BF, 4, false>(a, pl, s);
    return hipErrorInvalidValue;
}

}  // namespace skinny
}  // namespace kq
