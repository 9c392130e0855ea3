// On-device MoE routing and the MoE output epilogue.
//
// The reference routes a Qwen-MoE token on the host side of a sync: router
// logits by F.linear on the fp16 router matrix, torch.topk, a float32 softmax
// of the k logits cast back to fp16, then .tolist() of the picks
// (runtime/qwen_moe.py:386-416); after the experts it adds the shared expert
// scaled by sigmoid(shared_expert_gate . x) and clamps to the fp16 range
// (runtime/qwen_moe.py:496-513).  These kernels keep all of it on the device:
//  * gemv_f16: y = fp16(sum_k w[r][k] * x[k]) for fp16 weights (the router
//    and the shared-expert gate; the converter stores unquantized tensors as
//    fp16, tools/convert_qwen_moe.py:177-189), fp32 accumulation, each row in
//    the fixed four-part order of f16_row_dot (common.h);
//  * route_topk: the k largest logits per token in descending order (ties:
//    lower expert index first; NaN above every number, as torch.topk), and
//    fp16(softmax_fp32(those logits));
//  * moe_combine: y = clamp(expert_out + fp16(fp16(sigmoid(gate)) * shared_out))
//    with torch's fp16 elementwise semantics (each op in fp32, rounded to fp16).

#include <algorithm>

#include "common.h"
#include "topk.h"

namespace gdsllm {
namespace {

constexpr int kF16Waves = 4;      // waves per workgroup of the fp16 GEMV
constexpr int kMaxBatch = 8;
constexpr int kMaxExperts = 4096;  // 64 pick words per lane
constexpr int kMaxTopK = 64;       // one pick per lane

// Vector path (K % 8 == 0, rows and x 16-byte aligned): a 4-wave workgroup
// per row, rows dealt round-robin over the grid; wave w computes part w of
// the row (chunks w, w+4, ... of 512 columns: all its NJ loads in flight
// before the first dot product), the four wave sums meet in LDS and wave 0
// adds them in part order.  The sums are f16_row_dot's, bit for bit.
template <int NJ>
__device__ __forceinline__ void f16_row_parts(const uint16_t* __restrict__ wr, const uint16_t* __restrict__ X, int K,
                                              int nb, int64_t ldx, int wave, int lane, float (*part)[kMaxBatch]) {
    if constexpr (NJ == 0) {  // rows past 16 chunks: a loop over the part's chunks
        float acc[kMaxBatch];
#pragma unroll
        for (int b = 0; b < kMaxBatch; ++b) acc[b] = 0.f;
        for (int c = 8 * lane + 512 * wave; c < K; c += 2048) {
            const uint4 w = load_nt16(wr + c);
#pragma unroll
            for (int b = 0; b < kMaxBatch; ++b) {
                if (b < nb) {
                    const uint4 xv = *reinterpret_cast<const uint4*>(X + b * ldx + c);
                    acc[b] = dot2(w.x, xv.x, acc[b]);
                    acc[b] = dot2(w.y, xv.y, acc[b]);
                    acc[b] = dot2(w.z, xv.z, acc[b]);
                    acc[b] = dot2(w.w, xv.w, acc[b]);
                }
            }
        }
#pragma unroll
        for (int b = 0; b < kMaxBatch; ++b) {
            if (b < nb) {
                const float s = group_sum<64>(acc[b]);
                if (lane == 0) part[wave][b] = s;
            }
        }
        return;
    }
    constexpr int NW = NJ > 0 ? NJ : 1;
    uint4 w[NW];
#pragma unroll
    for (int j = 0; j < NW; ++j) {
        const int c = 8 * lane + 512 * (wave + 4 * j);
        w[j] = c < K ? load_nt16(wr + c) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int b = 0; b < kMaxBatch; ++b) {
        if (b < nb) {
            float acc = 0.f;
#pragma unroll
            for (int j = 0; j < NW; ++j) {
                const int c = 8 * lane + 512 * (wave + 4 * j);
                if (c < K) {
                    const uint4 xv = *reinterpret_cast<const uint4*>(X + b * ldx + c);
                    acc = dot2(w[j].x, xv.x, acc);
                    acc = dot2(w[j].y, xv.y, acc);
                    acc = dot2(w[j].z, xv.z, acc);
                    acc = dot2(w[j].w, xv.w, acc);
                }
            }
            const float s = group_sum<64>(acc);
            if (lane == 0) part[wave][b] = s;
        }
    }
}

// Rows blockIdx.x, += gridDim.x of x rows nb*blockIdx.y .. +nb-1 (fewer past
// T): y[b][r] = fp16(((p0 + p1) + p2) + p3).
template <int NJ>
__global__ __launch_bounds__(kF16Waves * 64) void gemv_f16(const uint16_t* __restrict__ W,
                                                           const uint16_t* __restrict__ X, uint16_t* __restrict__ Y,
                                                           int M, int K, int nb, int64_t T, int64_t ldx, int64_t ldy) {
    __shared__ float part[4][kMaxBatch];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t t0 = static_cast<int64_t>(blockIdx.y) * nb;
    X += t0 * ldx;
    Y += t0 * ldy;
    nb = static_cast<int>(min(static_cast<int64_t>(nb), T - t0));
    for (int r = blockIdx.x; r < M; r += gridDim.x) {
        f16_row_parts<NJ>(W + static_cast<int64_t>(r) * K, X, K, nb, ldx, wave, lane, part);
        __syncthreads();
        if (wave == 0 && lane < nb)
            Y[lane * ldy + r] = f2h_bits(((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane]);
        __syncthreads();
    }
}

// Scalar path (rows or x off the 16-byte grid, or K % 8 != 0): one wave per
// row, one element per lane per 64 columns.
__global__ __launch_bounds__(kF16Waves * 64) void gemv_f16_scalar(const uint16_t* __restrict__ W,
                                                                  const uint16_t* __restrict__ X,
                                                                  uint16_t* __restrict__ Y, int M, int K, int nb,
                                                                  int64_t T, int64_t ldx, int64_t ldy) {
    const int64_t t0 = static_cast<int64_t>(blockIdx.y) * nb;
    X += t0 * ldx;
    Y += t0 * ldy;
    nb = static_cast<int>(min(static_cast<int64_t>(nb), T - t0));
    const int lane = threadIdx.x & 63;
    const int wpb = static_cast<int>(blockDim.x) >> 6;
    const int nwaves = static_cast<int>(gridDim.x) * wpb;
    for (int r = static_cast<int>(blockIdx.x) * wpb + (threadIdx.x >> 6); r < M; r += nwaves) {
        const uint16_t* wr = W + static_cast<int64_t>(r) * K;
        float acc[kMaxBatch];
#pragma unroll
        for (int b = 0; b < kMaxBatch; ++b) acc[b] = 0.f;
        for (int c = lane; c < K; c += 64) {
            const float w = h2f(wr[c]);
#pragma unroll
            for (int b = 0; b < kMaxBatch; ++b)
                if (b < nb) acc[b] = fmaf(w, h2f(X[b * ldx + c]), acc[b]);
        }
#pragma unroll
        for (int b = 0; b < kMaxBatch; ++b) {
            if (b < nb) {
                const float s = group_sum<64>(acc[b]);
                if (lane == 0) Y[b * ldy + r] = f2h_bits(s);
            }
        }
    }
}

// Top-k of one token by one wave.  NPL pick words per lane live in registers
// (logit lane + 64*j), NPL * 64 >= E (topk.h).
template <int NPL>
__device__ __forceinline__ void topk_wave(const uint16_t* __restrict__ L, int E, int k, int32_t* __restrict__ idx,
                                          uint16_t* __restrict__ wts, int lane) {
    // all loads first (unconditional, past E re-reading logit 0): a load under
    // a branch would be waited for before the next one is issued
    uint32_t h[NPL], word[NPL];
#pragma unroll
    for (int j = 0; j < NPL; ++j) h[j] = L[lane + 64 * j < E ? lane + 64 * j : 0];
#pragma unroll
    for (int j = 0; j < NPL; ++j) word[j] = lane + 64 * j < E ? pick_word(h[j], lane + 64 * j) : 0u;
    int my_idx;
    uint32_t my_key, top_key;
    topk_select<NPL>(word, k, lane, my_idx, my_key, top_key);
    const uint16_t w = topk_weight(my_key, top_key, k, lane);
    if (lane < k) {
        idx[lane] = my_idx;
        wts[lane] = w;
    }
}

// One wave per token.
template <int NPL>
__global__ __launch_bounds__(64) void route_topk(const uint16_t* __restrict__ logits, int E, int64_t ld, int k,
                                                int32_t* __restrict__ idx, uint16_t* __restrict__ wts) {
    const int64_t t = blockIdx.x;
    topk_wave<NPL>(logits + t * ld, E, k, idx + t * k, wts + t * k, static_cast<int>(threadIdx.x));
}

// h = fp16(fp16(silu(g)) * u), 8 elements per thread (VEC: every pointer on the
// 16-byte grid; the last thread takes the remainder one by one).  Bound by
// memory: 2048 x 11008 is 135 MB, where torch's SiLU and product in two passes
// move 225 MB (24.5 + 21.7 us); at decode size it saves a launch (2 x 4.6 us).
template <bool VEC>
__global__ __launch_bounds__(256) void silu_mul(const uint16_t* g, const uint16_t* u, uint16_t* h, int64_t n) {
    const int64_t i0 = 8 * (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x);
    if (i0 >= n) return;
    if (VEC && i0 + 8 <= n) {
        const uint4 gv = *reinterpret_cast<const uint4*>(g + i0), uv = *reinterpret_cast<const uint4*>(u + i0);
        auto two = [](uint32_t a, uint32_t b) {
            return static_cast<uint32_t>(silu_mul_h(h2f(a & 0xFFFFu), h2f(b & 0xFFFFu))) |
                   (static_cast<uint32_t>(silu_mul_h(h2f(a >> 16), h2f(b >> 16))) << 16);
        };
        *reinterpret_cast<uint4*>(h + i0) = make_uint4(two(gv.x, uv.x), two(gv.y, uv.y), two(gv.z, uv.z), two(gv.w, uv.w));
    } else {
        for (int64_t i = i0; i < i0 + 8 && i < n; ++i) h[i] = silu_mul_h(h2f(g[i]), h2f(u[i]));
    }
}

// y = clamp(e + fp16(fp16(sigmoid(g)) * s), -65504, 65504) elementwise, g per token.
__global__ __launch_bounds__(256) void moe_combine(const uint16_t* __restrict__ eo, const uint16_t* __restrict__ so,
                                                   const uint16_t* __restrict__ gl, uint16_t* __restrict__ y,
                                                   int64_t H, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const float g = h2f(gl[i / H]);
    const float sw = h2f(f2h_bits(fp32_rounded(1.0f / fp32_rounded(1.0f + expf(-g)))));
    const float s = h2f(f2h_bits(fp32_rounded(sw * h2f(so[i]))));
    float r = h2f(f2h_bits(fp32_rounded(h2f(eo[i]) + s)));
    if (r > 65504.0f) r = 65504.0f;   // NaN compares false both ways and stays NaN
    if (r < -65504.0f) r = -65504.0f;
    y[i] = f2h_bits(r);
}

}  // namespace
}  // namespace gdsllm

using namespace gdsllm;

namespace {
// y[t][r] for T rows of x, nb of them per workgroup (grid.y).
int gemv_f16_run(const void* weight, const void* x, void* y, int64_t out_dim, int64_t in_dim, int64_t T, int nb,
                 int64_t ldx, int64_t ldy, void* stream) {
    const int M = static_cast<int>(out_dim), K = static_cast<int>(in_dim);
    const bool vec = K % 8 == 0 && reinterpret_cast<uintptr_t>(weight) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(x) % 16 == 0 && (T == 1 || ldx % 8 == 0);
    const auto* w = static_cast<const uint16_t*>(weight);
    const hipStream_t st = as_stream(stream);
    const int64_t most = int64_t(65535) * nb;  // x rows of one launch: grid.y is 16 bits
    for (int64_t t = 0; t < T; t += most) {
        const int64_t n = std::min(most, T - t);
        const auto* xp = static_cast<const uint16_t*>(x) + t * ldx;
        auto* yp = static_cast<uint16_t*>(y) + t * ldy;
        const unsigned gy = static_cast<unsigned>((n + nb - 1) / nb);
        if (vec) {
            // a 4-wave workgroup per row (one row each while the grid fits)
            const int grid = std::min(M, 16 * cu_count());
            const int nj = ((K + 511) / 512 + 3) / 4;
            auto launch = [&](auto kern) {
                hipLaunchKernelGGL(kern, dim3(grid, gy), dim3(kF16Waves * 64), 0, st, w, xp, yp, M, K, nb, n, ldx, ldy);
            };
            if (nj <= 1) launch(gemv_f16<1>);
            else if (nj <= 2) launch(gemv_f16<2>);
            else if (nj <= 4) launch(gemv_f16<4>);
            else launch(gemv_f16<0>);
        } else {
            const int grid = std::min((M + kF16Waves - 1) / kF16Waves, 8 * cu_count());
            hipLaunchKernelGGL(gemv_f16_scalar, dim3(grid, gy), dim3(kF16Waves * 64), 0, st, w, xp, yp, M, K, nb, n,
                               ldx, ldy);
        }
        if (int rc = check_hip(hipGetLastError(), "gemv_f16 launch")) return rc;
    }
    return ok();
}

int check_gemv_f16(const std::string& n, const void* weight, const void* x, const void* y, int64_t out_dim,
                   int64_t in_dim, int64_t T, int64_t ldx, int64_t ldy, bool& empty) {
    empty = false;
    if (out_dim > (int64_t(1) << 30) || in_dim > (int64_t(1) << 24))
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": dimension too large");
    if (out_dim == 0 || in_dim == 0 || T == 0) {
        empty = true;
        return GDSLLM_OK;
    }
    if (!weight || !x || !y) return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": null pointer");
    if (T > 1 && (ldx < in_dim || ldy < out_dim))
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": ldx/ldy smaller than the row length");
    if (reinterpret_cast<uintptr_t>(weight) % 2 || reinterpret_cast<uintptr_t>(x) % 2 ||
        reinterpret_cast<uintptr_t>(y) % 2)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": weight, x and y must be 2-byte aligned");
    return GDSLLM_OK;
}
}  // namespace

extern "C" int gdsllm_gemv_f16(const void* weight, const void* x, void* y, int64_t out_dim, int64_t in_dim,
                               int64_t batch, int64_t ldx, int64_t ldy, void* stream) {
    const std::string n = "gemv_f16";
    if (out_dim < 0 || in_dim < 0) return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": negative dimension");
    if (batch < 1 || batch > kMaxBatch)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": batch must be in [1, 8], got " + std::to_string(batch));
    bool empty;
    if (int rc = check_gemv_f16(n, weight, x, y, out_dim, in_dim, batch, ldx, ldy, empty)) return rc;
    if (empty) return ok();
    return gemv_f16_run(weight, x, y, out_dim, in_dim, batch, static_cast<int>(batch), ldx, ldy, stream);
}

extern "C" int gdsllm_gemv_f16_tokens(const void* weight, const void* x, void* y, int64_t out_dim, int64_t in_dim,
                                      int64_t tokens, int64_t ldx, int64_t ldy, void* stream) {
    const std::string n = "gemv_f16_tokens";
    if (out_dim < 0 || in_dim < 0 || tokens < 0)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": negative dimension");
    bool empty;
    if (int rc = check_gemv_f16(n, weight, x, y, out_dim, in_dim, tokens, ldx, ldy, empty)) return rc;
    if (empty) return ok();
    // Up to 8 x rows share a workgroup's weight row; fewer where that would
    // leave less than two workgroups per CU.  Each output is one wave-ordered
    // sum over its own rows of W and x, so nb does not change its bits.  The
    // 1 x 4096 shared-expert gate over 512 tokens: 64 launches of 8 tokens
    // took 478 us (kernel trace sum), this one launch, one token per workgroup, 5.3.
    const int64_t per = out_dim * std::min<int64_t>(tokens, int64_t(1) << 20) / (2 * static_cast<int64_t>(cu_count()));
    const int nb = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(kMaxBatch, per)));
    return gemv_f16_run(weight, x, y, out_dim, in_dim, tokens, nb, ldx, ldy, stream);
}

extern "C" int gdsllm_moe_route_topk(const void* logits, int64_t num_experts, int64_t n_tok, int64_t ld_logits,
                                     int64_t top_k, int32_t* idx, void* weights, void* stream) {
    const std::string n = "moe_route_topk";
    if (num_experts < 1 || num_experts > kMaxExperts)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT,
                         n + ": num_experts must be in [1, 4096], got " + std::to_string(num_experts));
    if (top_k < 1 || top_k > kMaxTopK || top_k > num_experts)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT,
                         n + ": top_k must be in [1, min(64, num_experts)], got " + std::to_string(top_k));
    if (n_tok < 0 || n_tok > (int64_t(1) << 31) - 1)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": bad token count");
    if (n_tok == 0) return ok();
    if (ld_logits < num_experts) return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": ld_logits < num_experts");
    if (!logits || !idx || !weights) return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": null pointer");
    if (reinterpret_cast<uintptr_t>(logits) % 2 || reinterpret_cast<uintptr_t>(weights) % 2 ||
        reinterpret_cast<uintptr_t>(idx) % 4)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": misaligned pointer");
    const auto* l = static_cast<const uint16_t*>(logits);
    auto* w = static_cast<uint16_t*>(weights);
    const int E = static_cast<int>(num_experts), k = static_cast<int>(top_k);
    const dim3 grid(static_cast<unsigned>(n_tok)), block(64);
    const hipStream_t s = as_stream(stream);
    if (E <= 128) hipLaunchKernelGGL(route_topk<2>, grid, block, 0, s, l, E, ld_logits, k, idx, w);
    else if (E <= 512) hipLaunchKernelGGL(route_topk<8>, grid, block, 0, s, l, E, ld_logits, k, idx, w);
    else if (E <= 1024) hipLaunchKernelGGL(route_topk<16>, grid, block, 0, s, l, E, ld_logits, k, idx, w);
    else hipLaunchKernelGGL(route_topk<64>, grid, block, 0, s, l, E, ld_logits, k, idx, w);
    if (int rc = check_hip(hipGetLastError(), "moe_route_topk launch")) return rc;
    return ok();
}

extern "C" int gdsllm_moe_combine(const void* expert_out, const void* shared_out, const void* shared_gate_logit,
                                  void* y, int64_t hidden, int64_t n_tok, void* stream) {
    const std::string n = "moe_combine";
    if (hidden < 0 || n_tok < 0) return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": negative dimension");
    if (hidden > (int64_t(1) << 24) || n_tok > (int64_t(1) << 24))
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": dimension too large");
    if (hidden == 0 || n_tok == 0) return ok();
    if (!expert_out || !shared_out || !shared_gate_logit || !y)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": null pointer");
    if ((reinterpret_cast<uintptr_t>(expert_out) | reinterpret_cast<uintptr_t>(shared_out) |
         reinterpret_cast<uintptr_t>(shared_gate_logit) | reinterpret_cast<uintptr_t>(y)) % 2)
        return set_error(GDSLLM_ERR_INVALID_ARGUMENT, n + ": pointers must be 2-byte aligned");
    const int64_t total = hidden * n_tok;
    hipLaunchKernelGGL(moe_combine, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, as_stream(stream),
                       static_cast<const uint16_t*>(expert_out), static_cast<const uint16_t*>(shared_out),
                       static_cast<const uint16_t*>(shared_gate_logit), static_cast<uint16_t*>(y), hidden, total);
    if (int rc = check_hip(hipGetLastError(), "moe_combine launch")) return rc;
    return ok();
}

extern "C" int gdsllm_silu_mul(const void* gate, const void* up, void* h, int64_t n, void* stream) {
    const std::string nm = "silu_mul";
    if (n < 0 || n > (int64_t(1) << 40)) return set_error(GDSLLM_ERR_INVALID_ARGUMENT, nm + ": n out of range");
    if (n == 0) return ok();
    if (!gate || !up || !h) return set_error(GDSLLM_ERR_INVALID_ARGUMENT, nm + ": null pointer");
    const uintptr_t bits = reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) | reinterpret_cast<uintptr_t>(h);
    if (bits % 2) return set_error(GDSLLM_ERR_INVALID_ARGUMENT, nm + ": pointers must be 2-byte aligned");
    const auto *g = static_cast<const uint16_t*>(gate), *u = static_cast<const uint16_t*>(up);
    auto* hp = static_cast<uint16_t*>(h);
    const int64_t most = int64_t(1) << 34;  // elements of one launch: 2^31 threads, of fewer than 2^32
    for (int64_t i = 0; i < n; i += most) {
        const int64_t c = std::min(most, n - i);
        const dim3 grid(static_cast<unsigned>((c + 2047) / 2048));
        if (bits % 16 == 0) hipLaunchKernelGGL(silu_mul<true>, grid, dim3(256), 0, as_stream(stream), g + i, u + i, hp + i, c);
        else hipLaunchKernelGGL(silu_mul<false>, grid, dim3(256), 0, as_stream(stream), g + i, u + i, hp + i, c);
        if (int rc = check_hip(hipGetLastError(), "silu_mul launch")) return rc;
    }
    return ok();
}
