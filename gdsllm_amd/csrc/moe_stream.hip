// Grouped expert GEMM of the MoE prefill for experts with few tokens
// (runtime/qwen_moe.py:475-492): affine-Q4 weights streamed from HBM straight
// into registers.
//
// What bounds it: with ~10 tokens per expert a chunk reads the whole expert
// pool for about 20 flop per weight, so the stream of the pool (3.6 GB of 512
// experts of 1024 x 4096) is the floor.  The split-K tiles of prefill.hip
// meet at a barrier every 128 columns and refill their pipeline for each
// 128-row tile; that skeleton alone took longer than the stream.  Here:
//  * A workgroup (8 waves) keeps the x rows of 16 tokens over all of K in LDS
//    (32 K bytes) and runs a range of the expert's rows against them: one
//    barrier per 16 tokens, no reduction across waves.
//  * A wave owns two fragments of 16 weight rows (gate and up rows of the same
//    outputs, or 32 down rows) over all of K and streams them through
//    registers, one unit of UC 128-column chunks ahead of the products and
//    across row tiles.  A load takes whole 128-byte lines of 8 rows: 16-byte
//    pieces of 16 rows, the fragment order, kept 35 cache lookups and as many
//    half-used lines in flight per load (697 us for the gate/up launch of 512
//    tokens over 512 experts of 1024 x 4096, 572 with whole lines).
//  * The wave turns a chunk pair into fragment order in 2 KiB of LDS of its
//    own: lane (r = l % 16, j = l / 16) reads columns 32j .. +31 of row r, whose
//    four words are the A operands of four v_mfma_f32_16x16x32_f16 with the
//    same columns of 16 tokens as B.  Scales and biases come for SU units at a
//    time (64 consecutive bytes of a row where K allows), held in registers.
//  * Dequantization: a nibble alone in a byte is an fp8 (e4m3) code of exactly
//    q / 512, so two masks and a shift per word and one
//    v_cvt_scalef32_pk_f16_fp8 per pair give q, and a packed fma with (s, b)
//    the fp16 weight, the same bits as prefill.hip's: 11 instructions per 8
//    weights, three of them half as long as the rest, against 13.  x is stored
//    in the order the pairs come out in.
// Measured (512 tokens, top 10 of 512 experts, hidden 4096, ffn 1024, g 64): the
// chunk 1109 -> 822 us, gate/up 726 -> 531 us and down 425 -> 281 us by
// kernel trace (4.6 and 4.3 TB/s).  No change from other row ranges per job,
// from twice the waves per compute unit in the down launch, or from waves that
// start at different columns.
// Each pass over an expert's rows is jobs of its own: a job of both passes of a
// 17-32 token tile was the tail of the launch (20 tokens, top 6, one expert at
// 18: 135 us against 82), and an XCD that drew the loaded experts held up the
// rest.  prefill.hip's moe_sort gives the streams only chunks that suit them.

#include <algorithm>

#include "moe_stream.h"

namespace gdsllm {
namespace {

constexpr int kWaves = 8;
constexpr int kTok = kStreamTokens;
constexpr int kLdsMax = 163840;

typedef uint32_t u32x4a4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2a4_t __attribute__((ext_vector_type(2), aligned(4)));

// NB bytes (4, 8 or a multiple of 16; 4-byte aligned) into dwords.
template <int NB>
__device__ __forceinline__ void load_dwords(const uint8_t* p, uint32_t (&d)[NB / 4]) {
    if constexpr (NB >= 16) {
#pragma unroll
        for (int i = 0; i < NB / 16; ++i) {
            const u32x4a4_t v = *reinterpret_cast<const u32x4a4_t*>(p + 16 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) d[4 * i + e] = v[e];
        }
    } else if constexpr (NB == 8) {
        const u32x2a4_t v = *reinterpret_cast<const u32x2a4_t*>(p);
        d[0] = v[0];
        d[1] = v[1];
    } else {
        d[0] = *reinterpret_cast<const uint32_t*>(p);
    }
}

template <int G, int UC, int SU, bool DUAL>
__global__ __launch_bounds__(kWaves * 64) void moe_stream_kernel(MoeStreamArgs a, int rows_per_job, int jobs_per_pass) {
    constexpr int SBU = UC * 256 / G;  // scale bytes of one row per unit
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r16 = lane & 15, j = lane >> 4;

    // The grid covers the worst case; the first passes * jobs_per_pass
    // workgroups take a job, an XCD a contiguous range of them (one expert's
    // x rows come into one L2, and so do its weights for both passes of a tile).
    const int jobs = __builtin_amdgcn_readfirstlane(a.passes[0]) * jobs_per_pass, bid = blockIdx.x;
    if (bid >= jobs) return;  // uniform
    const int per = jobs >> 3, rem = jobs & 7, xcd = bid & 7;
    const int q = xcd * per + (xcd < rem ? xcd : rem) + (bid >> 3);
    const int pass = q / jobs_per_pass, two = __builtin_amdgcn_readfirstlane(a.passes[1]);
    const int4 td = a.tiles[pass < 2 * two ? pass >> 1 : pass - two];
    const int64_t e = __builtin_amdgcn_readfirstlane(td.x);
    const int t0 = pass < 2 * two ? kTok * (pass & 1) : 0;
    const int p0 = __builtin_amdgcn_readfirstlane(td.y) + t0, nt = __builtin_amdgcn_readfirstlane(td.z) - t0;
    const int m0 = (q % jobs_per_pass) * rows_per_job, K = a.K;
    constexpr int kTileRows = DUAL ? 16 : 32;  // output rows of a wave's tile
    const int nwt = min(rows_per_job, a.M - m0) / kTileRows;
    const int cnt = nwt > wave ? (nwt - wave + kWaves - 1) / kWaves : 0;  // tiles of this wave: wave, wave + 8, ..
    const int upt = K / (128 * UC);                                       // units per tile

    const int64_t rb_w = K / 2, rb_s = 2 * (K / G);
    // fragment f of the tile at output row m: rows m .. +15 of gate / up, or m + 16f .. of the one matrix
    const uint8_t* wbase[2];
#pragma unroll
    for (int f = 0; f < 2; ++f)
        wbase[f] = (DUAL && f ? a.w2 : a.w) + e * a.estride_w + (m0 + (DUAL ? 0 : 16 * f)) * rb_w;
    // words: a load takes 128 bytes (256 columns, a whole cache line) of each
    // of 8 rows, lane 8r + p piece p ^ r of row r: read back in fragment
    // order, the rows of a piece lie in distinct banks
    const uint32_t vw = static_cast<uint32_t>((lane >> 3) * rb_w + 16 * ((lane & 7) ^ (lane >> 3)));
    const int rd0 = 128 * r16 + 16 * (j ^ (r16 & 7)), rd1 = rd0 ^ 64;
    // scales and biases of SU units at a time: load q takes matrices 4q / SU ..
    // of (gate scales, gate biases, up scales, up biases; fragment 0, then 1),
    // lane (matrix, row, unit): SBU bytes each
    const uint8_t* sb[SU];
#pragma unroll
    for (int q4 = 0; q4 < SU; ++q4) {
        const int mat = (64 * q4 + lane) / (16 * SU), row = (lane / SU) & 15;
        sb[q4] = (mat & 1 ? (DUAL && mat > 1 ? a.b2 : a.b) + e * a.estride_b
                          : (DUAL && mat > 1 ? a.s2 : a.s) + e * a.estride_s) +
                 (m0 + (DUAL ? 0 : 16 * (mat >> 1)) + row) * rb_s + SBU * (lane % SU);
    }
    uint8_t* const wst = lds + 2 * kTok * K + wave * (2048 + 64 * SBU);  // this wave's staging: words, then scales
    uint8_t* const sst = wst + 2048;

    struct Unit {
        u32x4_t w[2][UC];
    };
    struct Scales {
        uint32_t v[SU][SBU / 4];
    };
    Unit buf[2];
    Scales scur, snxt;
    // selects this lane's fp16 of a dword of two groups, twice
    const uint32_t sel = (G == 64 ? j >> 1 : j & 1) ? 0x03020302u : 0x01000100u;

    const int n = min(kTok, nt);
    int lt = 0, lk = 0;  // tile and unit of the next load
    auto load_unit = [&](Unit& u) {
        const int64_t row = static_cast<int64_t>(wave + kWaves * lt) * kTileRows;
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int c = 0; c < UC; ++c)  // c / 2: the 256 columns, c % 2: rows 0-7 or 8-15
                u.w[f][c] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(
                    wbase[f] + (row + 8 * (c & 1)) * rb_w + lk * (64 * UC) + vw + 128 * (c >> 1)));
        // past the wave's last unit the loads repeat it
        if (lk + 1 < upt) ++lk;
        else if (lt + 1 < cnt) {
            lk = 0;
            ++lt;
        }
    };
    int st = 0, sk = 0;  // tile and unit of the next scales
    auto load_scales = [&](Scales& u) {
        const int64_t row = static_cast<int64_t>(wave + kWaves * st) * kTileRows;
#pragma unroll
        for (int q4 = 0; q4 < SU; ++q4) load_dwords<SBU>(sb[q4] + row * rb_s + sk * SBU, u.v[q4]);
        if (sk + SU < upt) sk += SU;
        else if (st + 1 < cnt) {
            sk = 0;
            ++st;
        }
    };
    const int pos = p0 + min(r16, n - 1);
    const int64_t xrow = a.tok ? a.tok[pos] : pos;
    if (cnt > 0) {
        load_scales(scur);
        load_unit(buf[0]);
    }

    // x of the 16 tokens: 16-byte block (m, i) of columns 32m + 8i .. +7
    // goes where lane 16(m % 4) + t reads B operand i of chunk m / 4, its
    // values in the order 0 2 4 6 1 3 5 7.  Rows past n keep what is there:
    // they feed only outputs that are not stored.
    if (r16 < n) {
        const uint16_t* xr = a.x + xrow * a.ldx + 8 * j;
        const int nm = K / (32 * kWaves);  // blocks of this wave: m = wave, wave + 8, ..
        for (int mb = 0; mb < nm; mb += 8) {
            u32x4_t v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                v[i] = *reinterpret_cast<const u32x4_t*>(xr + 32 * (wave + kWaves * min(mb + i, nm - 1)));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int m = wave + kWaves * min(mb + i, nm - 1);
                u32x4_t o;
                o[0] = __builtin_amdgcn_perm(v[i][1], v[i][0], 0x05040100u);
                o[1] = __builtin_amdgcn_perm(v[i][3], v[i][2], 0x05040100u);
                o[2] = __builtin_amdgcn_perm(v[i][1], v[i][0], 0x07060302u);
                o[3] = __builtin_amdgcn_perm(v[i][3], v[i][2], 0x07060302u);
                *reinterpret_cast<u32x4_t*>(lds + 1024 * (4 * (m >> 2) + j) + 256 * (m & 3) + 16 * r16) = o;
            }
        }
    }
    lds_barrier();

    float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    int ct = 0, ck = 0;  // tile and unit of the next product
    auto compute = [&](const Unit& u, int su) {  // unit su of the loaded scales
        const uint8_t* xs = lds + ck * (4096 * UC) + 16 * lane;
        // through LDS into fragment order; one wave's LDS accesses keep
        // their order, so the staging area is reused without waiting
        uint32_t sc[2][SBU / 4], bi[2][SBU / 4];
        u32x4_t wf[2][2][2];  // [256 columns, alternating][fragment][chunk]
        auto stage = [&](int p) {
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                *reinterpret_cast<u32x4_t*>(wst + 16 * lane) = u.w[f][2 * p];
                *reinterpret_cast<u32x4_t*>(wst + 1024 + 16 * lane) = u.w[f][2 * p + 1];
                asm volatile("" ::: "memory");
                wf[p & 1][f][0] = *reinterpret_cast<const u32x4_t*>(wst + rd0);
                wf[p & 1][f][1] = *reinterpret_cast<const u32x4_t*>(wst + rd1);
                asm volatile("" ::: "memory");
            }
        };
        if (lane % SU == su) {
#pragma unroll
            for (int q4 = 0; q4 < SU; ++q4)
#pragma unroll
                for (int d = 0; d < SBU / 4; ++d)
                    reinterpret_cast<uint32_t*>(sst + SBU * ((64 * q4 + lane) / SU))[d] = scur.v[q4][d];
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int d = 0; d < SBU / 4; ++d) {
                sc[f][d] = reinterpret_cast<const uint32_t*>(sst + SBU * (32 * f + r16))[d];
                bi[f][d] = reinterpret_cast<const uint32_t*>(sst + SBU * (32 * f + 16 + r16))[d];
            }
        stage(0);
#pragma unroll
        for (int c = 0; c < UC; ++c) {
            half8_t xf[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) xf[i] = *reinterpret_cast<const half8_t*>(xs + 1024 * (4 * c + i));
            if (c % 2 == 1 && c + 1 < UC) stage((c + 1) / 2);
            half2_t ss[2], bb[2];
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                uint32_t s, b;
                if constexpr (G == 32) {
                    s = j >> 1 ? sc[f][2 * c + 1] : sc[f][2 * c];
                    b = j >> 1 ? bi[f][2 * c + 1] : bi[f][2 * c];
                } else if constexpr (G == 64) {
                    s = sc[f][c];
                    b = bi[f][c];
                } else {
                    s = sc[f][c / 2];
                    b = bi[f][c / 2];
                }
                const uint32_t sl = G == 128 ? (c & 1 ? 0x03020302u : 0x01000100u) : sel;
                ss[f] = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, s, sl));
                bb[f] = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, b, sl));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    const uint32_t w = wf[(c >> 1) & 1][f][c & 1][i];
                    const uint32_t even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
                    const half2_t p[4] = {__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(even, 512.0f, false),
                                          __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(even, 512.0f, true),
                                          __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(odd, 512.0f, false),
                                          __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(odd, 512.0f, true)};
                    u32x4_t o;
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        o[v] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(p[v], ss[f], bb[f]));
                    acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, o), xf[i], acc[f], 0, 0, 0);
                }
            }
        }
        if (++ck < upt) return;
        // the tile is done: lane (t = r16, j) holds rows 4j .. +3 of token t
        const int row = m0 + (wave + kWaves * ct) * kTileRows + 4 * j;
        if (r16 < n) {
            uint16_t* yp = a.y + static_cast<int64_t>(p0 + r16) * a.ldy + row;
#pragma unroll
            for (int f = 0; f < (DUAL ? 1 : 2); ++f) {
                uint32_t h[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) h[i] = DUAL ? silu_mul_h(acc[0][i], acc[1][i]) : f2h_bits(acc[f][i]);
                *reinterpret_cast<uint2*>(yp + 16 * f) = uint2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
            }
        }
        acc[0] = acc[1] = float4_t{0.f, 0.f, 0.f, 0.f};
        ck = 0;
        ++ct;
    };
    const int units = cnt * upt;
    constexpr int kBody = SU > 1 ? SU : 2;  // units per pass of the loop: whole scale loads, both buffers
    int u = 0;
    for (; u + kBody <= units; u += kBody) {
#pragma unroll
        for (int i = 0; i < kBody; ++i) {
            load_unit(buf[(i + 1) & 1]);
            if (i % SU == 0) load_scales(snxt);
            __builtin_amdgcn_sched_barrier(0);  // the loads go out ahead of the products
            compute(buf[i & 1], i % SU);
            if (i % SU == SU - 1) scur = snxt;
        }
    }
    if constexpr (SU == 1)
        if (u < units) compute(buf[0], 0);
}

// Row range of a job: 256 gate/up outputs (two tiles a wave) or 1024 down
// rows (four), so that a job streams about a megabyte against one fill of x.
constexpr int job_rows(bool dual) { return dual ? 256 : 1024; }

template <int G, int UC, int SU, bool DUAL>
int launch(const MoeStreamArgs& a, int64_t max_passes, hipStream_t stream) {
    const int rpj = std::min(a.M, job_rows(DUAL)), jpp = moe_stream_jobs(a.M, DUAL);
    const size_t lds = static_cast<size_t>(2 * kTok) * a.K + kWaves * (2048 + 64 * UC * 256 / G);
    const void* fn = reinterpret_cast<const void*>(&moe_stream_kernel<G, UC, SU, DUAL>);
    if (int rc = prepare_lds(fn, lds)) return rc;
    hipLaunchKernelGGL((moe_stream_kernel<G, UC, SU, DUAL>), dim3(static_cast<unsigned>(max_passes * jpp)),
                       dim3(kWaves * 64), lds, stream, a, rpj, jpp);
    return check_hip(hipGetLastError(), "moe_stream launch");
}

// Units of 512 columns (256 for g = 32, whose scales are twice as many, and
// where 512 does not divide K), scales of four, two or one units per load.
template <int G, bool DUAL>
int pick(const MoeStreamArgs& a, int64_t max_passes, hipStream_t stream) {
    constexpr int UC = G == 32 ? 2 : 4;
    if (a.K % (128 * UC) != 0) return launch<G, 2, 1, DUAL>(a, max_passes, stream);
    if (a.K % (512 * UC) == 0) return launch<G, UC, 4, DUAL>(a, max_passes, stream);
    if (a.K % (256 * UC) == 0) return launch<G, UC, 2, DUAL>(a, max_passes, stream);
    return launch<G, UC, 1, DUAL>(a, max_passes, stream);
}

template <int G>
int pick(const MoeStreamArgs& a, bool dual, int64_t max_passes, hipStream_t stream) {
    return dual ? pick<G, true>(a, max_passes, stream) : pick<G, false>(a, max_passes, stream);
}

}  // namespace

bool moe_stream_fits(int64_t M, int64_t K) {
    return K % 256 == 0 && M % 256 == 0 && 2 * kTok * K + kWaves * 3072 <= kLdsMax;
}

int moe_stream_jobs(int64_t M, bool dual) {
    return static_cast<int>((M + job_rows(dual) - 1) / job_rows(dual));
}

int moe_stream(const MoeStreamArgs& a, int group_size, bool dual, int64_t max_passes, hipStream_t stream) {
    switch (group_size) {
        case 32: return pick<32>(a, dual, max_passes, stream);
        case 64: return pick<64>(a, dual, max_passes, stream);
        default: return pick<128>(a, dual, max_passes, stream);
    }
}

}  // namespace gdsllm
