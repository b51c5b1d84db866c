// produce.hip - the step before attention on the session path: per-head
// RMSNorm of Q and K, rotary position embedding, rounding to the cache dtype,
// and the K/V append into head-major rows, in one launch.
//
// Order and arithmetic follow Model::run (src/model/mod.rs:611-662):
//  * rmsnorm (src/cpu/reductions.rs:8-49): squares and their sum in FP64,
//    denominator sqrt(sum / D + eps) in FP64, value = f32(x * (1 / den) * w) in
//    FP64 (the reference divides by den; the reciprocal form can move the FP64
//    value by an ulp, which changes the FP32 result only at a rounding tie);
//  * rotary (src/cpu/attention.rs:10-64): frequency theta^(-2j/D), angle =
//    position * frequency and sine/cosine in FP64, rounded to FP32; rotation
//    a*c - b*s, b*c + a*s in FP32 with separate roundings (no contraction);
//  * proportional rotary (src/cpu/proportional_rotary.rs:32-91): inverse
//    frequency base^(-2j/D) / factor for pairs j < rotated_dims / 2, other
//    features copied;
//  * Llama 3 rotary (src/cpu/llama3_rotary.rs:44-61, 87-146): the ordinary
//    frequency theta^(-2j/D) kept for wavelengths below original/high, divided
//    by factor above original/low, blended linearly in original/wavelength in
//    between, all in FP64; angle and rotation as for split-half;
//  * LayerKv::append (src/model/cache.rs:64-85): token-major new rows into
//    head-major cache rows, here rounded once to the cache dtype.
// The FP64 sum runs in a different order than the reference's sequential one;
// the denominator can differ in its last FP64 bit, which reaches an FP32
// result only at a rounding tie.
//
// Non-finite inputs or results set the device status word (the reference
// returns Error::NonFinite).
#include <cstddef>
#include <type_traits>

#include "device.hpp"

namespace tkh {


namespace {

__host__ __device__ __forceinline__ int rotary_pairs(int kind, int D, int rotated_dims) {
    return (kind == 1 || kind == 3) ? D / 2 : (kind == 2 ? rotated_dims / 2 : 0);
}

// Inverse frequency of pair j in FP64: theta^(-2j/D), divided by factor for
// the proportional form (src/cpu/proportional_rotary.rs:68-70), or scaled by
// wavelength band for Llama 3 (Llama3Scaling::inverse_frequency,
// src/cpu/llama3_rotary.rs:44-61; 6.283185307179586 is 2*pi rounded to FP64).
__device__ __forceinline__ double inverse_frequency(const RotarySpec &r, int D, int j) {
#pragma clang fp contract(off)
    const double ordinary = pow((double)r.theta, -(2.0 * (double)j) / (double)D);
    if (r.kind == 2) return ordinary / (double)r.factor;
    if (r.kind != 3) return ordinary;
    const double factor = r.factor, low = r.low, high = r.high;
    const double wavelength = 6.283185307179586 / ordinary;
    if (factor == 1.0 || wavelength < r.original / high) return ordinary;
    if (wavelength > r.original / low) return ordinary / factor;
    const double smooth = (r.original / wavelength - low) / (high - low);
    return (1.0 - smooth) * ordinary / factor + smooth * ordinary;
}

// Rotation of pair j at absolute position pos: angle and sine/cosine in FP64,
// rounded once to FP32 (src/cpu/attention.rs:41-46,
// src/cpu/proportional_rotary.rs:68-74, src/cpu/llama3_rotary.rs:126-128).
__device__ __forceinline__ float rotary_part(const RotarySpec &r, int D, int64_t pos, int j, bool sine) {
#pragma clang fp contract(off)
    const double angle = (double)pos * inverse_frequency(r, D, j);
    return sine ? (float)sin(angle) : (float)cos(angle);
}

template <int DT> __device__ __forceinline__ void store_out(void *base, int64_t i, float x);
template <> __device__ __forceinline__ void store_out<F32>(void *base, int64_t i, float x) {
    reinterpret_cast<float *>(base)[i] = x;
}
template <> __device__ __forceinline__ void store_out<F16>(void *base, int64_t i, float x) {
    reinterpret_cast<_Float16 *>(base)[i] = (_Float16)x;
}
template <> __device__ __forceinline__ void store_out<BF16>(void *base, int64_t i, float x) {
    reinterpret_cast<__bf16 *>(base)[i] = (__bf16)x;  // round to nearest even
}


}  // namespace

// One workgroup covers `rows` head slots of one token: slots [0, Hq) are query
// heads, [Hq, Hq + Hkv) key heads, the rest value heads; a wave takes slots wave,
// wave + waves, ..., RG of them at a time, so their loads and their FP64 chains
// overlap.  Lane l holds elements l, l + 64, ... of a row (K of them, D <= 64 K).
//
// The token's (cos, sin) are the same for every head.  TABLE: each wave reads
// them from p->rope once.  Without it a wave per 64 pairs and function evaluates
// the FP64 pow and sine or cosine and the others read the result from LDS, so the host gives a workgroup every slot of its token:
// evaluating them in each of 32 slots' waves made 128 tokens of 16/8/128 take
// 9.3 us, this 7.6 (4,096 tokens 169 and 49 us).
template <int DT, int K, bool TABLE>
__device__ __forceinline__ void produce_rows(const_ptr<ProduceParams> p, const ProduceLayer io, int hkv, int64_t t,
                                             int first, int rows) {
#pragma clang fp contract(off)
    constexpr int RG = K <= 1 ? 2 : (K == 2 ? 4 : (K == 4 ? 2 : 1));
    constexpr int KP = (K + 1) / 2;               // rotary pairs per lane
    constexpr int WAVES = TABLE ? 4 : 8;
    __shared__ float rowbuf[WAVES][RG][64 * K];
    __shared__ f32x2 rot[TABLE ? 1 : 64 * KP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int D = p->d, hq = p->hq, half = D / 2;
    const RotarySpec spec{p->rot.kind, p->rot.rotated_dims, p->rot.theta, p->rot.factor, p->rot.low, p->rot.high, p->rot.original};
    const int pairs = rotary_pairs(spec.kind, D, spec.rotated_dims);
    const int64_t position = p->position + t;
    const int end = first + rows < hq + 2 * hkv ? first + rows : hq + 2 * hkv;

    float x[RG][K] = {}, wq[K], wk[K];
    f32x2 cs[KP];
    auto source = [&](int slot) {
        return slot < hq ? io.q + (t * hq + slot) * D
                         : (slot < hq + hkv ? io.k + (t * hkv + slot - hq) * D : io.v + (t * hkv + slot - hq - hkv) * D);
    };
    auto load = [&](int slot0) {
#pragma unroll
        for (int i = 0; i < RG; ++i) {
            const int slot = slot0 + i * waves;
            if (slot < end) {
                const float *src = source(slot);
                for (int k = 0; k < K; ++k) x[i][k] = lane + 64 * k < D ? src[lane + 64 * k] : 0.0f;
            }
        }
    };
    // Every load first (rows, norm weights, rotary pairs), then the arithmetic.
    load(first + wave);
    for (int k = 0; k < K; ++k) {
        const int i = lane + 64 * k;
        wq[k] = io.q_norm && i < D ? io.q_norm[i] : 0.0f;
        wk[k] = io.k_norm && i < D ? io.k_norm[i] : 0.0f;
    }
    for (int k = 0; k < KP; ++k) {
        const int j = lane + 64 * k;
        cs[k] = f32x2{1.0f, 0.0f};
        if constexpr (TABLE) {
            if (j < pairs) cs[k] = *gload_ptr<f32x2>(p->rope + 2 * ((position - p->rope_pos0) * pairs + j));
        }
    }
    if constexpr (!TABLE) {
        if (pairs > 0) {
            // The lower half of the workgroup takes the cosines, the upper the
            // sines: each wave's chain holds one of them.
            const int j = threadIdx.x & 255;
            const bool sine = wave >= WAVES / 2;
            if (j < pairs) rot[j][sine ? 1 : 0] = rotary_part(spec, D, position, j, sine);
            __syncthreads();
            for (int k = 0; k < KP; ++k)
                if (lane + 64 * k < pairs) cs[k] = rot[lane + 64 * k];
        }
    }

    bool bad = false;
    for (int slot0 = first + wave; slot0 < end; slot0 += RG * waves) {
        if (slot0 != first + wave) load(slot0);
        // The norm of every row of the group before any is stored.
#pragma unroll
        for (int i = 0; i < RG; ++i) {
            const int slot = slot0 + i * waves;
            if (slot >= end) continue;
            for (int k = 0; k < K; ++k) bad |= lane + 64 * k < D && !is_finite_f(x[i][k]);
            const bool is_q = slot < hq;
            if (slot >= hq + hkv || !(is_q ? io.q_norm : io.k_norm)) continue;
            double ss = 0.0;
            for (int k = 0; k < K; ++k)
                if (lane + 64 * k < D) {
                    const double v = (double)x[i][k];
                    ss += v * v;
                }
            ss = wave_sum_f64(ss);
            const double inv = 1.0 / sqrt(ss / (double)D + (double)p->eps);
            for (int k = 0; k < K; ++k) {
                const float w = is_q ? wq[k] : wk[k];
                const float y = (float)((double)x[i][k] * inv * (double)w);
                bad |= lane + 64 * k < D && (!is_finite_f(y) || !is_finite_f(w));
                x[i][k] = y;
            }
        }
        // The rotary pairs elements j and j + D/2, which may sit in other lanes:
        // through LDS (the wave's own rows).
#pragma unroll
        for (int i = 0; i < RG; ++i)
            for (int k = 0; k < K; ++k) rowbuf[wave][i][lane + 64 * k] = x[i][k];
        wave_lds_order();
#pragma unroll
        for (int i = 0; i < RG; ++i) {
            const int slot = slot0 + i * waves;
            if (slot >= end) continue;
            if (slot >= hq + hkv) {
                const int64_t dst = (int64_t)(slot - hq - hkv) * io.out_head_stride + t * D;
                for (int k = 0; k < K; ++k)
                    if (lane + 64 * k < D) store_out<DT>(io.v_out, dst + lane + 64 * k, x[i][k]);
                continue;
            }
            const bool is_q = slot < hq;
            void *out = is_q ? io.q_out : io.k_out;
            const int64_t dst = is_q ? (t * hq + slot) * D : (int64_t)(slot - hq) * io.out_head_stride + t * D;
            const float *row = rowbuf[wave][i];
            for (int k = 0; k < KP; ++k) {
                const int j = lane + 64 * k;
                if (j >= half) continue;
                float a = row[j], b = row[j + half];
                if (j < pairs) {
                    const float c = cs[k][0], sn = cs[k][1];
                    const float ac = a * c, bs = b * sn, bc = b * c, as = a * sn;
                    a = ac - bs;
                    b = bc + as;
                    bad |= !is_finite_f(a) || !is_finite_f(b);
                }
                store_out<DT>(out, dst + j, a);
                store_out<DT>(out, dst + j + half, b);
            }
        }
        wave_lds_order();  // the next group's rows take their place
    }
    raise_status(p->status, bad, ST_NONFINITE_INPUT);
}

// blocks_per_token workgroups of `rows` slots per token.
template <int DT, int K, bool TABLE>
__global__ __launch_bounds__(TABLE ? 256 : 512) void produce_qkv(ProduceParams args, int rows, int blocks_per_token) {
    // Its fields arrive through dependent scalar loads: their lines (and the
    // hidden arguments' start) first, in one round trip.
    const_ptr<ProduceParams> p = warm_kernarg_ptr<ProduceParams, (sizeof(ProduceParams) + 8 + 63) / 64, 0>();
    const uint32_t bpt = (uint32_t)blocks_per_token;
    const ProduceLayer io{p->q, p->k, p->v, p->q_norm, p->k_norm, p->q_out, p->k_out, p->v_out, p->out_head_stride};
    produce_rows<DT, K, TABLE>(p, io, p->hkv, blockIdx.x / bpt, (int)(blockIdx.x % bpt) * rows, rows);
}

// The chunk of several session layers, one after the other in the grid (the
// rotary table is the session's).  A layer without K/V of its own has k_out
// null: only its Q rows are made.
template <int DT, int K>
__global__ __launch_bounds__(256) void produce_qkv_layers(ProduceLayersArgs args, int rows, int blocks_per_token) {
    const_ptr<ProduceLayersArgs> a = warm_kernarg_ptr<ProduceLayersArgs, 11, offsetof(ProduceLayersArgs, e) + DECODE_LAYERS_MAX * sizeof(ProduceLayer) - 4>();
    const uint32_t bpt = (uint32_t)blocks_per_token, per = bpt * (uint32_t)a->p.tokens;
    const uint32_t layer = blockIdx.x / per, b = blockIdx.x % per;
    const_ptr<ProduceLayer> e = &a->e[layer];
    const ProduceLayer io{e->q, e->k, e->v, e->q_norm, e->k_norm, e->q_out, e->k_out, e->v_out, e->out_head_stride};
    produce_rows<DT, K, true>(&a->p, io, io.k_out ? a->p.hkv : 0, b / bpt, (int)(b % bpt) * rows, rows);
}

// (cos, sin) of every (position, pair) for rows [pos0, pos0 + rows): the
// producer's table, filled once per session with the same FP64 formulas.
__global__ __launch_bounds__(256) void rotary_table(float *out, int64_t pos0, int64_t rows,
                                                    int pairs, RotarySpec rot, int D) {
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * pairs) return;
    const int64_t r = i / pairs;
    const int j = (int)(i % pairs);
    out[2 * i] = rotary_part(rot, D, pos0 + r, j, false);
    out[2 * i + 1] = rotary_part(rot, D, pos0 + r, j, true);
}

}  // namespace tkh

extern "C" int tkh_rotary_pairs(int rotary, int head_dim, int rotated_dims) {
    return tkh::rotary_pairs(rotary, head_dim, rotated_dims);
}

extern "C" hipError_t tkh_launch_rotary_table(float *out, int64_t pos0, int64_t rows,
                                              const tkh::RotarySpec *rot, int head_dim,
                                              hipStream_t stream) {
    using namespace tkh;
    const int pairs = rotary_pairs(rot->kind, head_dim, rot->rotated_dims);
    const int64_t n = rows * pairs;
    if (n <= 0) return hipSuccess;
    dim3 grid((unsigned)((n + 255) / 256)), block(256);
    hipLaunchKernelGGL(rotary_table, grid, block, 0, stream, out, pos0, rows, pairs, *rot,
                       head_dim);
    return hipGetLastError();
}

// Slots per workgroup.  With a rotary table: two for each of its four waves.
// Without one each workgroup evaluates its token's rotation, so it takes up to 32
// slots (four for each of eight waves), unless the card is mostly idle anyway
// (one round of one slot per wave on 256 CUs: 1 token of 32/8/128 6.3 us
// against 8.1 with all 48), and all of them from 1,024 tokens on, where the FP64
// work decides (48 slots: 128 tokens 6.5 us in two workgroups, 8.6 in one; 4,096
// tokens 80 and 66).
static int produce_slots(int64_t tokens, int slots, bool table) {
    if (table || tokens * ((slots + 7) / 8) <= 256) return 8;
    const int blocks = tokens >= 1024 ? 1 : (slots + 31) / 32;
    return ((slots + blocks - 1) / blocks + 7) / 8 * 8;
}

template <int DT, int K>
static hipError_t launch_produce(const tkh::ProduceParams *p, hipStream_t stream) {
    using namespace tkh;
    const bool table = p->rope != nullptr || rotary_pairs(p->rot.kind, p->d, p->rot.rotated_dims) == 0;
    const int slots = p->hq + 2 * p->hkv, rows = produce_slots(p->tokens, slots, table), bpt = (slots + rows - 1) / rows;
    const dim3 grid((unsigned)(p->tokens * bpt));
    if (table) hipLaunchKernelGGL((produce_qkv<DT, K, true>), grid, dim3(256), 0, stream, *p, rows, bpt);
    else hipLaunchKernelGGL((produce_qkv<DT, K, false>), grid, dim3(512), 0, stream, *p, rows, bpt);
    return hipGetLastError();
}

// f(type tag, elements-per-lane tag) for a dtype and head size.
template <class F> static hipError_t produce_build(int dtype, int d, F f) {
    using namespace tkh;
    auto of = [&](auto dt) {
        if (d <= 64) return f(dt, std::integral_constant<int, 1>{});
        if (d <= 128) return f(dt, std::integral_constant<int, 2>{});
        if (d <= 256) return f(dt, std::integral_constant<int, 4>{});
        return f(dt, std::integral_constant<int, 8>{});
    };
    if (dtype == F32) return of(std::integral_constant<int, F32>{});
    if (dtype == F16) return of(std::integral_constant<int, F16>{});
    if (dtype == BF16) return of(std::integral_constant<int, BF16>{});
    return hipErrorInvalidValue;
}

extern "C" hipError_t tkh_launch_produce(const tkh::ProduceParams *p, int dtype, hipStream_t stream) {
    if (p->tokens <= 0 || p->hq + 2 * p->hkv <= 0 || p->d > 512 || p->d % 2) return hipErrorInvalidValue;
    return produce_build(dtype, p->d, [&](auto dt, auto k) {
        return launch_produce<decltype(dt)::value, decltype(k)::value>(p, stream);
    });
}

// The layers' chunk; the rows have a rotary table, or no rotary.
extern "C" hipError_t tkh_launch_produce_layers(const tkh::ProduceLayersArgs *a, int dtype, hipStream_t stream) {
    using namespace tkh;
    const int slots = a->p.hq + 2 * a->p.hkv, rows = produce_slots(a->p.tokens, slots, true), bpt = (slots + rows - 1) / rows;
    const dim3 grid((unsigned)(a->count * a->p.tokens * bpt)), block(256);
    if (a->p.tokens <= 0 || a->count <= 0 || a->p.d > 512 || a->p.d % 2) return hipErrorInvalidValue;
    return produce_build(dtype, a->p.d, [&](auto dt, auto k) {
        hipLaunchKernelGGL((produce_qkv_layers<decltype(dt)::value, decltype(k)::value>), grid, block, 0, stream, *a, rows, bpt);
        return hipGetLastError();
    });
}
