// kq_skinny.hip -- launch planning of the skinny matrix-core kernels
// (kq_skinny_kernel.h, instantiated in kq_skinny_i4_g*.hip and
// kq_skinny_vq.hip).
#include "kq_skinny_kernel.h"

namespace kq {

hipError_t launch_skinny_i4_g32(const skinny::Args& a, const skinny::Plan& pl, bool sb, bool bf, hipStream_t s);
hipError_t launch_skinny_i4_g64(const skinny::Args& a, const skinny::Plan& pl, bool sb, bool bf, hipStream_t s);
hipError_t launch_skinny_i4_g128(const skinny::Args& a, const skinny::Plan& pl, bool sb, bool bf, hipStream_t s);
bool skinny_vq_usable(int gm);
hipError_t launch_skinny_vq_gm(const skinny::Args& a, const skinny::Plan& pl, int gm, hipStream_t s);

namespace {

constexpr size_t kLdsMax = 160 * 1024;

// What orders a shape's plans: a launch with its first loads and the K-part sums,
// then a wave's steps at 8 waves a CU (a step: T tiles and the x of 256 k) --
// 1.25 / 2.0 / 4.3 us at T = 1 / 2 / 4 up to 8 tokens, 2.05 / 2.7 / 4.9 us above
// -- and 1 us a further round. Fewer tiles a step pay for x again, more leave
// fewer waves to hide a step's serial chain.
double plan_us(const skinny::Plan& pl, uint32_t batch) {
    const int t = pl.T == 1 ? 0 : pl.T == 2 ? 1 : 2;
    static constexpr double kStep[2][3] = {{1.25, 2.0, 4.3}, {2.05, 2.7, 4.9}};
    const uint32_t waves = pl.P * pl.Q;
    return 3.6 + (double)pl.rounds * pl.J * (waves > 8 ? waves / 8.0 : 1.0) * kStep[batch > 8][t] +
           1.0 * (pl.rounds - 1);
}

// Tiles spread over every CU (a workgroup a CU, in rounds of T x Q tiles); the
// T and K parts P of the shortest duration. per: tiles a workgroup, cb: LDS
// bytes of codebooks.
bool make_plan(uint32_t M, uint32_t K, uint32_t batch, uint32_t tmax, uint32_t per, size_t cb,
               skinny::Plan& out) {
    if (K < skinny::kPair || K % 32 || K > (1u << 24) || M == 0) return false;
    const uint32_t ntiles = (M + 15) / 16;
    const uint32_t NP = (K + skinny::kPair - 1) / skinny::kPair;
    // 32-bit offsets in a workgroup, its last round's empty tiles included
    if (((uint64_t)per + 64) * 16 * (K / 2) >= (1ull << 31)) return false;
    bool found = false;
    double best = 0.0;
    for (uint32_t T : {1u, 2u, 4u}) {
        if (T > tmax) continue;
        const uint32_t wmax = skinny::max_waves(T, batch <= 8);
        for (uint32_t P = 1; P <= wmax && P <= NP; ++P) {
            const uint32_t want = (per + T - 1) / T, Q = want < wmax / P ? want : wmax / P;
            const uint32_t rounds = (per + T * Q - 1) / (T * Q);
            const size_t lds = P > 1 ? (size_t)(rounds > 1 ? 2 : 1) * P * Q * T * 1024 : 0;
            const size_t xl = (size_t)P * Q * (batch <= 8 ? 4096 : 8192);
            if (lds + xl + cb > kLdsMax) continue;
            const skinny::Plan pl{T, P, Q, (NP + P - 1) / P, NP, rounds, per, (ntiles + per - 1) / per, lds, xl};
            const double cost = plan_us(pl, batch);
            if (!found || cost < best) {
                found = true;
                best = cost;
                out = pl;
            }
        }
    }
    return found;
}

skinny::Args make_args(const skinny::Plan& pl, uint32_t M, uint32_t K, uint32_t ntok, bool y_f32) {
    skinny::Args a{};
    a.M = M;
    a.K = K;
    a.ntok = ntok;
    a.y_f32 = y_f32 ? 1 : 0;
    a.P = pl.P;
    a.Q = pl.Q;
    a.J = pl.J;
    a.NP = pl.NP;
    a.tiles_wg = pl.tiles_wg;
    a.rounds = pl.rounds;
    a.part_lds = (uint32_t)pl.part_lds;
    return a;
}

// Four tiles of 64-wide groups' separate scales spill above 8 tokens: two instead
// take 0.68-1.10 times as long, 0.84 on average of 150 calls (10888x2048, 10 tokens:
// 11.9 -> 8.1 us).
uint32_t int4_tmax(uint32_t G, uint32_t batch, bool inter) {
    return G == 32 || (G == 64 && !inter && batch > 8) ? 2 : 4;
}

// Tiles a workgroup: every CU's share.
uint32_t even_share(uint32_t M) {
    const uint32_t cu = cu_count();
    return ((M + 15) / 16 + cu - 1) / cu;
}

// A workgroup's rows lie in one codebook block (64 KiB of copies): tiles a
// workgroup, the smallest share that divides a block's tiles (0: blocks end
// inside a tile, or are smaller than the share).
uint32_t vq_share(uint32_t M, uint32_t rpc) {
    uint32_t per = even_share(M);
    if (rpc >= M) return per;
    if (rpc % 16) return 0;
    const uint32_t blk = rpc / 16;
    while (per < blk && blk % per) ++per;
    return blk % per ? 0 : per;
}
constexpr size_t kCbLds = 65536;

int vq_gm(uint32_t K, uint32_t scale_group) {
    if (scale_group == K) return 0;
    return scale_group >= 128 ? 128 : (int)scale_group;
}

}  // namespace

// Modelled duration of a plan, which the choice between paths goes by: a launch,
// then a wave's steps, one part fixed and one that grows with the waves a CU and
// a little with the CUs in use. form: a step's cost by scale layout (fitted
// together over both formats: 250-28672 rows, K 512-28672, 3000 calls, nineteen in
// twenty within 15%).
static double skinny_us(const skinny::Plan& pl, uint32_t batch, double form) {
    static constexpr double kStep[2][3] = {{0.0, 0.1, 0.0}, {0.2, 1.6, 4.74}},
                            kWaves[2][3] = {{1.37, 2.14, 4.06}, {1.7, 1.25, 0.0}};
    const int t = pl.T == 1 ? 0 : pl.T == 2 ? 1 : 2, b = batch > 8;
    const double fill = pl.P * pl.Q / 8.0 * (0.8 + 0.2 * pl.nwg / cu_count());
    return 3.2 + (double)pl.rounds * pl.J * (kStep[b][t] + kWaves[b][t] * fill) * form;
}

// A step's cost by int4 layout (medians of 14000 calls, nine in ten within 15%): 8
// groups a pair take more work for scales.
double int4_skinny_us(const skinny::Plan& pl, uint32_t G, uint32_t batch, bool inter) {
    const bool two8 = inter && pl.T == 2 && batch <= 8;
    double form = two8 ? 0.98 : 0.92;
    if (G == 64) form = pl.T == 4 ? 1.1 : two8 ? 1.07 : 1.03;
    if (G == 32) form = !inter ? 1.08 : two8 ? 1.45 : 1.22;
    return skinny_us(pl, batch, form) + (pl.T > 1 ? 0.3 : 0.0);
}

bool int4_skinny_plan(uint32_t M, uint32_t K, uint32_t G, uint32_t batch, bool inter, skinny::Plan& pl) {
    if (batch < 1 || batch > 16 || !(G == 32 || G == 64 || G == 128) || K % G) return false;
    // not in use: one tile's windows spill there, two tiles alone are unmeasured
    if (!inter && G == 32 && batch <= 8) return false;
    return make_plan(M, K, batch, int4_tmax(G, batch, inter), even_share(M), 0, pl);
}

hipError_t launch_int4_skinny(const uint32_t* W, const uint16_t* S, const uint16_t* B, int meta_kind,
                              bool interleaved, const uint16_t* X, void* Y, bool y_f32, uint32_t M,
                              uint32_t K, uint32_t G, uint32_t batch, const skinny::Plan& pl,
                              hipStream_t s) {
    skinny::Args a = make_args(pl, M, K, batch, y_f32);
    a.W = reinterpret_cast<const uint8_t*>(W);
    a.S = S;
    a.B = B;
    a.X = X;
    a.Y = Y;
    a.gpr = K / G;
    const bool bf = meta_kind == 1;
    if (G == 32) return launch_skinny_i4_g32(a, pl, interleaved, bf, s);
    if (G == 64) return launch_skinny_i4_g64(a, pl, interleaved, bf, s);
    return launch_skinny_i4_g128(a, pl, interleaved, bf, s);
}

bool vq_skinny_plan(uint32_t M, uint32_t K, uint32_t rows_per_cb, uint32_t scale_group, uint32_t batch,
                    skinny::Plan& pl) {
    if (batch < 1 || batch > 16) return false;
    const int gm = vq_gm(K, scale_group);
    const uint32_t per = vq_share(M, rows_per_cb);
    return per != 0 && make_plan(M, K, batch, gm == 32 ? 2 : 4, per, kCbLds, pl);
}

double vq_skinny_us(const skinny::Plan& pl, uint32_t K, uint32_t scale_group, uint32_t batch) {
    const int gm = vq_gm(K, scale_group);
    return skinny_us(pl, batch, gm == 32 ? 1.1 : gm == 64 ? 1.02 : 1.0);
}

bool vq_skinny_usable(uint32_t K, uint32_t scale_group) { return skinny_vq_usable(vq_gm(K, scale_group)); }

hipError_t launch_vq_skinny(const uint8_t* IDX, const uint16_t* C, const uint16_t* S, const uint16_t* X,
                            void* Y, bool y_f32, uint32_t M, uint32_t K, uint32_t rows_per_cb,
                            uint32_t scale_group, uint32_t batch, const skinny::Plan& pl, hipStream_t s) {
    const int gm = vq_gm(K, scale_group);
    skinny::Args a = make_args(pl, M, K, batch, y_f32);
    a.W = IDX;
    a.C = C;
    a.S = S;
    a.X = X;
    a.Y = Y;
    a.gpr = gm == 0 ? 1 : K / scale_group;
    while ((1u << a.gshift) < scale_group) ++a.gshift;
    a.rpc = rows_per_cb < M ? rows_per_cb : (M + 15) / 16 * 16;
    a.cb_lds = (uint32_t)kCbLds;
    return launch_skinny_vq_gm(a, pl, gm, s);
}

}  // namespace kq
