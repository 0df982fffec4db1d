// kq_internal.h -- host-side launchers shared between the kernel files and the
// C ABI shim (kq_api.cpp). Launchers assume validated arguments.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "kq.h"

namespace kq {

struct Int4Cfg {
    int rows;    // VALU: rows per wave item; MFMA: K parts per workgroup
    int unroll;  // VALU: ring depth; MFMA: ring depth D, or 10 * tiles per wave + D
};

// Compute units of the current device (queried once; 256 if the query fails).
uint32_t cu_count();

// Launch plan of one pass of the vector path (kq_int4.hip, make_vplan).
struct VPlan {
    uint32_t R, P, Q, J, rounds, groups_wg, nwg, nreal, nsteps, D, xw;
    size_t lds;
};
// The passes of a call: `times` of `nb` tokens on one plan each, in order.
struct Int4Passes {
    struct {
        uint32_t nb, times;
        VPlan pl;
    } p[4];
    uint32_t n;  // 0: no plan
};
Int4Passes int4_valu_passes(uint32_t M, uint32_t K, uint32_t batch, Int4Cfg cfg);
// The passes in batch-1-pass units x 100 (AUTO's crossover).
uint32_t int4_valu_cost(const Int4Passes& ps);
// Their modelled duration (us; AUTO's crossovers, with int4_mfma and with the
// skinny kernels).
double int4_valu_us(const Int4Passes& ps, uint32_t M, uint32_t K, uint32_t G);
double int4_valu_pass_us(const Int4Passes& ps, uint32_t M, uint32_t K, uint32_t G);

// gsel (device pointer, may be null): the kernel reads the matrix index
// gsel[0] and moves W, S and B by gsel[0] * gstride bytes -- one matrix of a
// pool chosen by an earlier launch, with no host round trip. Gathered calls
// take one token and split bf16 S and B (the MoE expert layout).
hipError_t launch_int4_valu(const uint32_t* W, const uint16_t* S, const uint16_t* B, int meta_kind,
                            bool interleaved, const uint16_t* X, void* Y, bool y_f32, uint32_t M,
                            uint32_t K, uint32_t G, uint32_t batch, const Int4Passes& ps,
                            hipStream_t s, const uint32_t* gsel = nullptr, uint64_t gstride = 0);
bool int4_valu_supported(uint32_t K, Int4Cfg cfg);

// Launch plan of the matrix-core path (kq_int4_mfma.hip); false: a shape or a
// forced cfg it does not take.
namespace mfma {
struct Plan {
    uint32_t T, P, Q, J, J8, rounds, groups_wg, nwg, nsteps, waves;
    size_t lds;
};
}  // namespace mfma
bool int4_mfma_plan(uint32_t M, uint32_t K, uint32_t G, uint32_t batch, Int4Cfg cfg, mfma::Plan& pl);
hipError_t launch_int4_mfma(const uint32_t* W, const uint16_t* S, const uint16_t* B, int meta_kind,
                            bool interleaved, const uint16_t* X, void* Y, bool y_f32, uint32_t M,
                            uint32_t K, uint32_t G, uint32_t batch, const mfma::Plan& pl,
                            hipStream_t s);
// Modelled duration (us) of a matrix-core pass, of all tokens (AUTO's
// crossovers, with the vector path and with the skinny kernels).
double int4_mfma_us(const mfma::Plan& pl, uint32_t batch);
double int4_mfma_pass_us(const mfma::Plan& pl, uint32_t G, uint32_t batch);

// Skinny matrix-core kernels (kq_skinny.hip), 1-16 tokens in one pass: the
// launch plan (false: a shape they don't take) and its modelled duration.
namespace skinny {
struct Plan {
    uint32_t T, P, Q, J, NP, rounds, tiles_wg, nwg;
    size_t part_lds, x_lds;  // the K-part sums, the waves' x stages
};
}  // namespace skinny
bool int4_skinny_plan(uint32_t M, uint32_t K, uint32_t G, uint32_t batch, bool inter, skinny::Plan& pl);
double int4_skinny_us(const skinny::Plan& pl, uint32_t G, uint32_t batch, bool inter);
hipError_t launch_int4_skinny(const uint32_t* W, const uint16_t* S, const uint16_t* B, int meta_kind,
                              bool interleaved, const uint16_t* X, void* Y, bool y_f32, uint32_t M,
                              uint32_t K, uint32_t G, uint32_t batch, const skinny::Plan& pl,
                              hipStream_t s);
bool vq_skinny_plan(uint32_t M, uint32_t K, uint32_t rows_per_cb, uint32_t scale_group, uint32_t batch,
                    skinny::Plan& pl);
double vq_skinny_us(const skinny::Plan& pl, uint32_t K, uint32_t scale_group, uint32_t batch);
bool vq_skinny_usable(uint32_t K, uint32_t scale_group);  // as loaded on this device
// Whether a call takes them (kq_vq.hip), were they usable.
bool vq_takes_skinny(uint32_t M, uint32_t K, uint32_t rows_per_cb, uint32_t scale_group, uint32_t batch);
hipError_t launch_vq_skinny(const uint8_t* IDX, const uint16_t* C, const uint16_t* S, const uint16_t* X,
                            void* Y, bool y_f32, uint32_t M, uint32_t K, uint32_t rows_per_cb,
                            uint32_t scale_group, uint32_t batch, const skinny::Plan& pl, hipStream_t s);

// The path an int4 call takes (forced: a launch shape, or null): KQ_PATH_*, or
// kPathSkinny (its plan to sp, if given), KQ_PATH_AUTO where it is refused. meta8:
// scales and biases start at multiples of 8 bytes.
constexpr int kPathSkinny = 4;
int int4_route(uint32_t M, uint32_t K, uint32_t G, uint32_t batch, bool inter, bool meta8, int path,
               skinny::Plan* sp, const Int4Cfg* forced);

// Debug scalar path: one thread per (row, token), plain chunk loop (v0).
hipError_t launch_int4_scalar(const uint32_t* W, const uint16_t* S, const uint16_t* B,
                              int meta_kind, bool interleaved, const uint16_t* X, void* Y,
                              bool y_f32, uint32_t M, uint32_t K, uint32_t G, uint32_t batch,
                              hipStream_t s);
hipError_t launch_xsum32(const uint16_t* X, float* xs, uint32_t K, uint32_t batch, hipStream_t s);
// unroll 0 and threads 0: the default shape (U = 1, 2048 x 256 threads)
hipError_t launch_stream_read(const void* src, size_t bytes, uint32_t* sink, uint32_t unroll,
                              uint32_t threads, hipStream_t s, uint16_t* out = nullptr,
                              uint32_t nout = 0);

bool vq_supported(uint32_t M, uint32_t K, uint32_t rows_per_cb);
hipError_t launch_vq(const uint8_t* IDX, const uint16_t* C, const uint16_t* S, const uint16_t* X,
                     void* Y, bool y_f32, uint32_t M, uint32_t K, uint32_t rows_per_cb,
                     uint32_t scale_group, uint32_t batch, hipStream_t s);

// VQ quantiser (kq_vq_quant.hip)
size_t vq_quant_ws_bytes(uint32_t M, uint32_t K, uint32_t scale_group, uint32_t rows_per_cb,
                         uint32_t sample);
hipError_t launch_vq_quantize(const void* W, int w_dtype, uint32_t M, uint32_t K,
                              uint32_t rows_per_cb, uint32_t scale_group, uint32_t iters,
                              uint32_t sample, uint64_t seed, uint8_t* IDX, uint16_t* Cb,
                              uint16_t* S, void* ws, hipStream_t s);

// MoE
size_t moe_ws_bytes(const kq_moe_desc& d, uint32_t batch);
hipError_t launch_ws_zero(void* ws, size_t bytes, hipStream_t s);
hipError_t launch_moe_router(const void* R, bool r_f32, const void* X, bool x_f32, uint32_t batch,
                             const kq_moe_desc& d, uint32_t* idx, float* wgt, uint16_t* xh,
                             void* ws, hipStream_t s);
hipError_t launch_moe_gate_up(const uint8_t* pool, const kq_moe_desc& d, const uint32_t* idx,
                              const uint16_t* xh, uint16_t* H, uint32_t batch, hipStream_t s);
// Whether it runs the expert-partitioned kernel.
bool moe_gate_up_partitions(const kq_moe_desc& d, uint32_t batch);
hipError_t launch_moe_down(const uint8_t* pool, const kq_moe_desc& d, const uint32_t* idx,
                           const float* wgt, const uint16_t* H, void* Y, bool y_f32,
                           uint32_t batch, void* ws, hipStream_t s);  // ws: workspace or null
// Router logits only (float [batch][n_experts] to lg; xh = half(X) if X is fp32).
hipError_t launch_moe_logits(const void* R, bool r_f32, const void* X, bool x_f32, uint32_t batch,
                             const kq_moe_desc& d, uint16_t* xh, float* lg, hipStream_t s);
// One operation per launch, batch 1 (see kq_moe_unfused.hip).
size_t moe_unfused_ws_bytes(const kq_moe_desc& d);
uint32_t moe_unfused_launches(const kq_moe_desc& d);
hipError_t launch_moe_unfused(const uint8_t* pool, const kq_moe_desc& d, const void* R, bool r_f32,
                              const void* X, bool x_f32, uint32_t* idx, float* wgt, uint16_t* xh,
                              uint16_t* H, void* Y, bool y_f32, void* ws, hipStream_t s);
// kq_moe_block on the per-device static workspace (no allocation).
hipError_t launch_moe_block_noalloc(const uint8_t* pool, const kq_moe_desc& d, const void* R,
                                    bool r_f32, const void* X, bool x_f32, uint32_t batch,
                                    uint32_t* idx, float* wgt, uint16_t* xh, uint16_t* H, void* Y,
                                    bool y_f32, hipStream_t s);
// path: KQ_MOE_PATH_* (KQ_MOE_PATH_ONE only where moe_one_supported holds)
hipError_t launch_moe_block(const uint8_t* pool, const kq_moe_desc& d, const void* R, bool r_f32,
                            const void* X, bool x_f32, uint32_t batch, uint32_t* idx, float* wgt,
                            uint16_t* xh, uint16_t* H, void* Y, bool y_f32, void* ws,
                            hipStream_t s, int path);
// The one-launch block's limits (shape, and every workgroup resident at once).
bool moe_one_supported(const kq_moe_desc& d, uint32_t batch);
// The atomic sum(h) block's limits (the streaming gate/up and down).
bool moe_atomic_supported(const kq_moe_desc& d, uint32_t batch);

}  // namespace kq
