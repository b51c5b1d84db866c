// attention.hip - attention in FP32 arithmetic on the matrix cores: FP32
// storage, head sizes outside 64/128/256, and the optional score/probability
// diagnostics the reference operators can return.  bf16/f16 chunks and decode
// at head_dim 64/128/256 take the MFMA prefill and streaming decode kernels
// instead.
//
//  * attn_split<DT, DP>: any head_dim D <= DP on the 16-bit matrix cores, FP32
//    values as 16-bit planes.  A workgroup is four waves (eight: split_waves) over 16
//    packed rows each (query x head of the GQA group) of one (problem, KV head),
//    optionally one key split of it.
//  * attn_tile<DP>: the same on the FP32 matrix cores, for FP32 storage above 128.
//  * attn_tile_merge: combines split-K partials (max, mass, unnormalised
//    context) and writes the context; makes the diagnostics' probabilities from
//    the stored scores and each row's merged (max, mass).
//
// Weights are powers of two (v_exp_f32) of score differences times log2 e.
// Masked keys contribute exactly zero.
#include "device.hpp"

namespace tkh {

namespace {

// attn_tile's keys per staged tile: K and V tiles of FP32 rows in about 66 KiB of LDS
// (two workgroups per CU).
__host__ __device__ constexpr int tile_keys(int DP) { return DP <= 256 ? 32 : 16; }

// Its waves that share a row group's features: a wave holds the Q and context of 128,
// which fits two waves per SIMD without spills.
__host__ __device__ constexpr int tile_feature_waves(int DP) { return DP / 128; }

// Four consecutive stored elements.
template <int DT> struct Raw4 { using T = uint32_t __attribute__((ext_vector_type(2))); };
template <> struct Raw4<F32> { using T = u32x4; };

template <int DT> __device__ __forceinline__ f32x4 widen4(typename Raw4<DT>::T w) {
    static_assert(DT == F32 || DT == F16, "bf16 is its own plane");
    if constexpr (DT == F32) {
        return __builtin_bit_cast(f32x4, w);
    } else {
        f32x4 x;
        for (int e = 0; e < 2; ++e) {
            const uint32_t u = w[e];
            const f16x2 h = __builtin_bit_cast(f16x2, u);
            x[2 * e] = (float)h[0];
            x[2 * e + 1] = (float)h[1];
        }
        return x;
    }
}

// Elements [off, off + 4) of a row of which the first n exist.  VEC (every row
// starts on a whole chunk and ends with one): one vector load, the caller
// keeps `off` inside the row.  Otherwise one by one, the rest zeros.
template <int DT, bool VEC, class Off>
__device__ __forceinline__ typename Raw4<DT>::T load4(const void *base, Off off, int n) {
    using T = typename Raw4<DT>::T;
    if constexpr (VEC) {
        return *gload_ptr<T>(reinterpret_cast<const uint8_t *>(base) + off * ElemSize<DT>::value);
    }
    T w{};
    for (int e = 0; e < 4; ++e)
        if (e < n) {
            if constexpr (DT == F32) w[e] = *gload_ptr<uint32_t>(reinterpret_cast<const uint32_t *>(base) + off + e);
            else w[e >> 1] |= (uint32_t)*gload_ptr<uint16_t>(reinterpret_cast<const uint16_t *>(base) + off + e) << (16 * (e & 1));
        }
    return w;
}

// Four floats at any 4-byte aligned address.
using f32x4u = float __attribute__((ext_vector_type(4), aligned(4)));

// Over the four lanes j, j + 16, j + 32, j + 48 of a query row.
__device__ __forceinline__ float row4_sum(float x) { return xor_sum(xor_sum(x, 16), 32); }
__device__ __forceinline__ float row4_max(float x) { return xor_max(xor_max(x, 16), 32); }

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// What a workgroup and one of its waves cover.
struct TileWork {
    int kvh, split, splits;      // KV head, key split and splits of the problem
    int m_kv, prow, ks;          // packed rows of the KV head, this lane's, and the wave's share of the keys
    int t_row, h_row;            // its token and query head (a valid row's)
    bool active, rvalid;         // the wave has rows; the lane's row exists
    int64_t lo;                  // first logical key of the workgroup's range
    int n;                       // its keys; relative to `lo` from here on:
    int rlo, rhi;                // keys the lane's row sees
    int wlo, whi;                // ... some row of the wave sees
    int flo, fhi;                // ... every row of the wave sees
    int vlo, vhi;                // ... some row of the workgroup sees
};

// Wave group `wg` (of the rw x kw that share the workgroup) and lane row j.
__device__ __forceinline__ TileWork tile_work(const TileArgs &a, int wg, int j, const_ptr<Problem> *problem) {
    const Params &p = a.p;
    TileWork w;
    const int G = p.group;
    const bool full_diag = p.diag_mode == 1;
    // XCD-major tile order (dispatch slot b runs on XCD b % 8): the row blocks
    // of one KV head, which read the same keys, share an XCD's L2.
    int64_t tile;
    {
        const uint32_t nb = gridDim.x, per = (nb + 7) / 8;
        const uint32_t x = blockIdx.x % 8, k = blockIdx.x / 8;
        const uint32_t full = nb % 8 == 0 ? 8 : nb % 8;
        tile = (int64_t)(x < full ? x * per + k : full * per + (x - full) * (per - 1) + k);
    }
    const_ptr<Problem> pr = problem_ptr(p, tile);
    *problem = pr;
    const uint32_t local = (uint32_t)(tile - pr->tile_base), nrb = (uint32_t)pr->row_blocks;
    const uint32_t ns = (uint32_t)pr->splits;
    const int rb = (int)(local % nrb);
    w.split = (int)(local / nrb % ns);
    w.splits = (int)ns;
    w.kvh = (int)(local / (nrb * ns));
    const int64_t k_pos0 = pr->k_pos0, keys = pr->keys, q_pos0 = pr->q_pos0;
    const int m_kv = w.m_kv = pr->queries * G;
    const int rw = a.rw, rg = wg % rw;
    w.ks = wg / rw;
    const int row0 = (rb * rw + rg) * 16;    // the wave's first packed row
    w.active = w.ks < a.kw && row0 < m_kv;
    w.prow = row0 + j;
    w.rvalid = w.ks < a.kw && w.prow < m_kv;
    const int rrow = w.prow < m_kv ? w.prow : m_kv - 1;
    w.t_row = (int)((uint32_t)rrow / (uint32_t)G);
    w.h_row = w.kvh * G + (int)((uint32_t)rrow % (uint32_t)G);

    // The split's keys; the workgroup's rows see [v_lo, v_hi) of them.  The
    // full diagnostics score every key, so they walk the whole split.
    const int64_t base_lo = full_diag ? 0 : pr->vis_lo, base_hi = full_diag ? keys : pr->vis_hi;
    const int64_t s_lo = base_lo + (int64_t)w.split * pr->split_keys;
    const int64_t s_hi = s_lo + pr->split_keys < base_hi ? s_lo + pr->split_keys : base_hi;
    int64_t r_lo, r_hi, v_lo, v_hi, w_lo, w_hi, f_lo, f_hi, tmp;
    visible_range(p, k_pos0, keys, q_pos0 + w.t_row, &r_lo, &r_hi);
    const int wg_first = rb * rw * 16, wg_last = min(wg_first + rw * 16, m_kv) - 1;
    visible_range(p, k_pos0, keys, q_pos0 + (uint32_t)wg_first / (uint32_t)G, &v_lo, &tmp);
    visible_range(p, k_pos0, keys, q_pos0 + (uint32_t)wg_last / (uint32_t)G, &tmp, &v_hi);
    v_lo = v_lo > s_lo ? v_lo : s_lo;
    v_hi = v_hi < s_hi ? v_hi : s_hi;
    const int wv_first = min(row0, m_kv - 1), wv_last = min(row0 + 15, m_kv - 1);
    visible_range(p, k_pos0, keys, q_pos0 + (uint32_t)wv_first / (uint32_t)G, &w_lo, &f_hi);
    visible_range(p, k_pos0, keys, q_pos0 + (uint32_t)wv_last / (uint32_t)G, &f_lo, &w_hi);
    const int64_t lo = full_diag ? s_lo : v_lo, hi = full_diag ? s_hi : v_hi;
    const int n = hi > lo ? (int)(hi - lo) : 0;
    auto rel = [&](int64_t x) { return (int)(x < lo ? 0 : (x > lo + n ? n : x - lo)); };
    w.lo = lo;
    w.n = n;
    w.rlo = w.rvalid ? rel(r_lo) : 0;
    w.rhi = w.rvalid ? rel(r_hi) : 0;
    w.wlo = rel(w_lo);
    w.whi = w.active ? rel(w_hi) : 0;
    w.flo = rel(f_lo);
    w.fhi = rel(f_hi);
    w.vlo = rel(v_lo);
    w.vhi = rel(v_hi);
    return w;
}

// A row's weights are 2^((y - m) mul), where y is the raw dot product (mul = scale *
// log2 e) or, where scores_scaled, the scaled, capped or stored score (mul =
// log2 e), and m the row's maximum y.  The difference comes first, so that the
// maximum weighs exactly 1 however large the scores are.  (One fma against m * mul
// rounded beforehand saves an instruction, 0.1 us of the FP32 chunk's 22.9 and
// nothing of the other calls, but weighs the maximum 2^d with d up to half an ulp of
// m * mul: past FP32's exponents from scores of 1e9 on.)  Raw dots are taken where mul is an ordinary number; where their difference
// overflows, the smaller one has no weight.
__device__ __forceinline__ bool scores_scaled(const Params &p) {
    return p.softcap != 0.0f || p.diag_mode != 0 || !(p.scale >= 0x1p-100f && p.scale <= 0x1p100f);
}
__device__ __forceinline__ float exp_mul(const Params &p) { return scores_scaled(p) ? LOG2E : p.scale * LOG2E; }
// The weight of y against m (0 for y at -inf; m is finite: 0 in place of -inf).
__device__ __forceinline__ float weight(float y, float m, float mul) { return __builtin_amdgcn_exp2f((y - m) * mul); }
__device__ __forceinline__ float finite_max(float m) { return m == NEG_INF ? 0.0f : m; }

// The dots of a staged tile's blocks as y values with masked keys at -inf: lane
// row j against keys 16 b + 4 g + r (relative, t0 on).  Stores the diagnostics'
// scores in the waves that have `store`.  Blocks that every row of the
// wave sees need no comparison (a row past the last has the last row's dots, which
// nothing stores).  Returns the lane's maximum; amax
// collects the largest |y|, NaN included (finite_scores).
template <int NB>
__device__ __forceinline__ float finish_scores(const Params &p, const TileWork &w, const_ptr<Problem> pr, int t0, int g,
                                               bool store, const bool (&scored)[NB], f32x4 (&st)[NB], float &amax) {
    const float scale = p.scale, cap = p.softcap;
    const bool full_diag = p.diag_mode == 1, scaled = scores_scaled(p);
    const bool last_row = w.h_row == p.query_heads - 1 && w.t_row == pr->queries - 1;
    const bool diag = p.diag_mode != 0 && store && w.rvalid && (full_diag || last_row);
    float *const xs = p.scores ? p.scores : p.probs;  // raw scores (attn_tile_merge turns them into probabilities)
    float tmax = NEG_INF;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (!scored[b]) {
            st[b] = f32x4{NEG_INF, NEG_INF, NEG_INF, NEG_INF};
            continue;
        }
        if (scaled)
            for (int r = 0; r < 4; ++r) st[b][r] *= scale;
        if (cap != 0.0f)
            for (int r = 0; r < 4; ++r) st[b][r] = softcap_f(st[b][r], cap);
        const int k0 = t0 + 16 * b, key = k0 + 4 * g;
        if (diag) {
            const f32x4 x = st[b];
            const int first = full_diag ? 0 : w.rlo, end = full_diag ? w.n : w.rhi;
            float *xr = xs + (full_diag ? ((int64_t)w.h_row * pr->queries + w.t_row) * pr->keys : 0) + w.lo + key;
            if (key >= first && key + 4 <= end) *reinterpret_cast<f32x4u *>(xr) = x;
            else
                for (int r = 0; r < 4; ++r)
                    if (key + r >= first && key + r < end) xr[r] = x[r];
        }
        if (k0 >= w.flo && k0 + 16 <= w.fhi) {
            for (int r = 0; r < 4; ++r) amax = __builtin_elementwise_maximum(amax, __builtin_fabsf(st[b][r]));
        } else {
            for (int r = 0; r < 4; ++r) {
                const bool vis = key + r >= w.rlo && key + r < w.rhi;
                amax = __builtin_elementwise_maximum(amax, vis ? __builtin_fabsf(st[b][r]) : 0.0f);
                st[b][r] = vis ? st[b][r] : NEG_INF;
            }
        }
        for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, st[b][r]);
    }
    return tmax;
}

// Whether every score a lane saw is finite: the scaled one, also where y is the raw
// dot (rounding keeps the order, so the largest tells).
__device__ __forceinline__ bool finite_scores(const Params &p, float amax) {
    return is_finite_f(scores_scaled(p) ? amax : amax * p.scale);
}

// Where a lane's row of unnormalised context goes: divided by its mass into the
// output, or into its partial with (max, mass) beside it.  `lead`: this lane
// stores the row's (max, mass).
struct TileOut {
    bool direct, write;
    bool bad_mass = false, bad_out = false;
    float inv;
    float *row;
    int D;
    __device__ __forceinline__ TileOut(const TileArgs &a, const TileWork &w, const_ptr<Problem> pr, int dp, bool lead, float m,
                                       float l) {
        const Params &p = a.p;
        const int S = w.splits * a.kw;
        const int64_t part = pr->slot_base + ((int64_t)w.kvh * w.m_kv + w.prow) * S + w.split * a.kw + w.ks;
        D = p.head_dim;
        direct = S == 1;
        write = direct || m != NEG_INF;  // a partial whose split shows the row no key is never read
        inv = direct ? 1.0f / l : 1.0f;
        row = direct ? pr->out + ((int64_t)w.t_row * p.query_heads + w.h_row) * D : p.part_o + part * dp;
        if (!w.rvalid) return;
        bad_mass = direct && (!(l > 0.0f) || !is_finite_f(l));
        if (lead && (!direct || p.diag_mode != 0)) {
            const f32x2 ml = {m, l};
            *gstore_ptr<f32x2>(p.part_ml + 2 * part) = ml;
        }
    }
    __device__ __forceinline__ void emit(int d, f32x4 o, bool &bad) {
        for (int e = 0; e < 4; ++e) {
            bad |= d + e < D && !is_finite_f(o[e]);
            o[e] *= inv;
            bad_out |= d + e < D && !is_finite_f(o[e]);
        }
        if (!write) return;
        if (d + 4 <= D) *reinterpret_cast<f32x4u *>(row + d) = o;
        else
            for (int e = 0; e < 4; ++e)
                if (d + e < D) row[d + e] = o[e];
    }
    __device__ __forceinline__ void report(const Params &p, bool bad) const {
        raise_status(p, bad, ST_NONFINITE_INPUT);
        raise_status(p, bad_mass, ST_BAD_MASS);
        raise_status(p, direct && bad_out, ST_NONFINITE_OUTPUT);
    }
};

}  // namespace

// What bounds it: v_mfma_f32_16x16x4 (32 cycles for 2,048 FLOP, 157 TFLOP/s
// over the card) on long ranges, launches and memory round trips on short
// ones.  Every product and sum stays FP32, as storage and reference have it.
//
// Lane (j, g) = (lane % 16, lane / 16) of a wave holds query row j:
//  * S^T = K Q^T per 16-key block: A = K (key j, features 16 c + 4 g + e in
//    step (c, e)), B = Q^T (row j, the same features), so both operands are
//    read four features at a time; the result holds row j, keys 4 g + r.
//  * O^T = V^T P^T: step r takes keys 4 g + r, where the scores already sit,
//    so P needs no exchange; A = V at key 4 g + r, feature 64 fb + 4 j + e of
//    MFMA (fb, e), again four features per LDS read.  The lane ends with
//    features 64 fb + 16 g .. + 15 of its row.
// K rows are padded by four floats in LDS, so the 16 rows of a read fall on
// distinct banks.  A tile's global loads are in flight while the one before
// it is multiplied.
//
// A workgroup takes a.rw row groups; with fewer than four the other waves
// share the groups' keys (a.kw of them, 16-key blocks in turn), each writing
// a partial of its own, so short row blocks keep every SIMD busy.
//
// It replaced one wave per (query, head) on the vector unit, whose lanes each read a
// key row of their own.  Calls back to back, FP32: 128 queries over 1025 keys at
// 8/1/512 2419 -> 53 us, over 1920 keys at 8/4/256 1807 -> 43 us, 300 tokens of
// 8/4/256 with both diagnostics 285 -> 29 us.  (Each chunk's load under a branch of
// its own made the compiler wait for one before the next, and 512-wide rows held by
// one wave spilled 390 registers.)
template <int DP, bool VEC>
__global__ __launch_bounds__(256, 2) void attn_tile(TileArgs a) {
    warm_kernarg<(sizeof(TileArgs) + 63) / 64, 0>();
    constexpr int KT = tile_keys(DP), NB = KT / 16, FS = tile_feature_waves(DP);
    constexpr int DW = DP / FS, FC = DW / 16, FB = DW / 64;  // a wave's features
    constexpr int KS = DP + 4;               // staged K row stride
    constexpr int NCH = KT * DP / 4 / 256;   // 4-element chunks per thread and tile
    __shared__ __attribute__((aligned(16))) float kt[KT * KS];
    __shared__ __attribute__((aligned(16))) float vt[KT * DP];
    __shared__ __attribute__((aligned(16))) f32x4 dots[4 * NB * 64];  // partial scores
    using Raw = typename Raw4<F32>::T;
    const Params &p = a.p;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int j = lane & 15, g = lane >> 4;
    const int G = p.group, Hq = p.query_heads, D = p.head_dim;
    const bool full_diag = p.diag_mode == 1;

    const_ptr<Problem> pr;
    const TileWork w = tile_work(a, wave / FS, j, &pr);
    const int kw = a.kw, ks = w.ks, kvh = w.kvh, m_kv = w.m_kv, nseg = pr->nseg, n = w.n;
    const int fs = wave % FS, f0 = fs * DW;  // the wave's features start at f0
    const bool active = w.active, rvalid = w.rvalid;
    const int t_row = w.t_row, h_row = w.h_row, rlo = w.rlo, rhi = w.rhi, wlo = w.wlo, whi = w.whi;
    const int vlo = w.vlo, vhi = w.vhi;
    const int64_t lo = w.lo, keys = pr->keys;

    // Features past the head are zeros in Q, K and V.  A vector load of one
    // reads the row's last chunk instead, so that no load is under a branch: the
    // loads of a tile stay in flight together.
    const int last = D - 4;  // first feature of a row's last whole chunk
    auto feature = [&](int d) { return VEC ? min(d, last) : d; };
    f32x4 q[FC];
    for (int c = 0; c < FC; ++c) {
        const int d = f0 + 16 * c + 4 * g;
        const int64_t at = (int64_t)t_row * pr->q_row_stride + (int64_t)h_row * D;
        q[c] = widen4<F32>(load4<F32, VEC>(pr->q, at + feature(d), D - d));
    }
    if constexpr (VEC)
        for (int c = 0; c < FC; ++c)
            if (f0 + 16 * c + 4 * g > last) q[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // A thread's chunk m of a tile: row i / (DP / 4), features 4 (i % (DP / 4)).
    // Rows past the range read its last row (K: masked; V: zeroed on staging,
    // so a stored non-finite value outside the visible keys never meets a zero
    // probability).
    constexpr int CPR = DP / 4;
    Raw kreg[NCH], vreg[NCH];
    auto fetch = [&](int t0) {
        if (nseg == 1) {
            const void *kb = pr->seg[0].k, *vb = pr->seg[0].v;
            const int64_t rs = pr->seg[0].row_stride, at = (int64_t)kvh * pr->seg[0].head_stride + lo * rs;
#pragma unroll
            for (int m = 0; m < NCH; ++m) {
                const int i = tid + 256 * m, d = 4 * (i % CPR);
                const int64_t off = at + min(t0 + i / CPR, n - 1) * rs + feature(d);
                kreg[m] = load4<F32, VEC>(kb, off, D - d);
                vreg[m] = load4<F32, VEC>(vb, off, D - d);
            }
        } else {
#pragma unroll
            for (int m = 0; m < NCH; ++m) {
                const int i = tid + 256 * m, d = 4 * (i % CPR);
                const void *kb, *vb;
                const int64_t off = seg_select(pr, lo + min(t0 + i / CPR, n - 1), kvh, &kb, &vb) + feature(d);
                kreg[m] = load4<F32, VEC>(kb, off, D - d);
                vreg[m] = load4<F32, VEC>(vb, off, D - d);
            }
        }
    };
    auto stage = [&](int t0) {
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < NCH; ++m) {
            const int i = tid + 256 * m, r = i / CPR, d = 4 * (i % CPR);
            const bool head = !VEC || d <= last, in = t0 + r >= vlo && t0 + r < vhi;
            *reinterpret_cast<f32x4 *>(kt + r * KS + d) = head ? widen4<F32>(kreg[m]) : zero;
            *reinterpret_cast<f32x4 *>(vt + r * DP + d) = head && in ? widen4<F32>(vreg[m]) : zero;
        }
    };

    f32x4 acc[FB][4];
    for (int fb = 0; fb < FB; ++fb)
        for (int e = 0; e < 4; ++e) acc[fb][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const float mul = exp_mul(p);
    float m_run = NEG_INF, l_run = 0.0f, amax = 0.0f;  // m_run: the row's maximum y

    if (n > 0) fetch(0);
    for (int t0 = 0; t0 < n; t0 += KT) {
        __syncthreads();
        stage(t0);
        __syncthreads();
        if (t0 + KT < n) fetch(t0 + KT);
        // Scores of the wave's blocks: dots over its features, then the sum of the
        // dots of the waves that share them (the same order in each).
        f32x4 st[NB];
        bool seen[NB], scored[NB];  // some row of the wave sees a key of the block; its scores are wanted
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int k0 = t0 + 16 * b;
            const bool mine = active && b % kw == ks;
            seen[b] = mine && k0 < whi && k0 + 16 > wlo;
            scored[b] = seen[b] || (full_diag && mine && k0 < n);
            f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;  // two chains
            if (scored[b]) {
                const float *kr = kt + (16 * b + j) * KS + f0 + 4 * g;
#pragma unroll
                for (int c = 0; c < FC; c += 2) {
                    const f32x4 k0v = *reinterpret_cast<const f32x4 *>(kr + 16 * c);
                    const f32x4 k1v = *reinterpret_cast<const f32x4 *>(kr + 16 * c + 16);
                    for (int e = 0; e < 4; ++e) {
                        s0 = mfma4(k0v[e], q[c][e], s0);
                        s1 = mfma4(k1v[e], q[c + 1][e], s1);
                    }
                }
            }
            for (int r = 0; r < 4; ++r) st[b][r] = s0[r] + s1[r];
            dots[(wave * NB + b) * 64 + lane] = st[b];
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const f32x4 *d = dots + (wave - fs) * NB * 64 + b * 64 + lane;
            st[b] = d[0];
            for (int w = 1; w < FS; ++w)
                for (int r = 0; r < 4; ++r) st[b][r] += d[w * NB * 64][r];
        }
        float tmax = finish_scores<NB>(p, w, pr, t0, g, fs == 0, scored, st, amax);
        // The tile's maximum over the row's four lanes; O and l move with it.
        tmax = row4_max(tmax);
        const float m_new = fmaxf(m_run, tmax);
        if (__ballot(m_new > m_run) != 0) {
            const float corr = weight(m_run, finite_max(m_new), mul);
            l_run *= corr;
            for (int fb = 0; fb < FB; ++fb)
                for (int e = 0; e < 4; ++e)
                    for (int r = 0; r < 4; ++r) acc[fb][e][r] *= corr;
            m_run = m_new;
        }
        const float m_ref = finite_max(m_run);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (!seen[b]) continue;
            for (int r = 0; r < 4; ++r) {
                const float e = weight(st[b][r], m_ref, mul);
                st[b][r] = e;
                l_run += e;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float *vr = vt + (16 * b + 4 * g + r) * DP + f0 + 4 * j;
                for (int fb = 0; fb < FB; ++fb) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(vr + 64 * fb);
                    for (int e = 0; e < 4; ++e) acc[fb][e] = mfma4(v[e], st[b][r], acc[fb][e]);
                }
            }
        }
    }

    l_run = row4_sum(l_run);
    bool bad = !finite_scores(p, amax);
    TileOut out(a, w, pr, DP, g == 0 && fs == 0, m_run, l_run);
    if (rvalid)
        for (int fb = 0; fb < FB; ++fb)
            for (int r = 0; r < 4; ++r)
                out.emit(f0 + 64 * fb + 16 * g + 4 * r, f32x4{acc[fb][0][r], acc[fb][1][r], acc[fb][2][r], acc[fb][3][r]}, bad);
    out.report(p, bad);
}

// ---------------------------------------------------------------------------
// attn_split: the same walk on the 16-bit matrix cores (v_mfma_f32_16x16x32,
// sixteen times the FP32 rate), with FP32 values as 16-bit planes, in which a product
// is known to 2^-25 of itself and sums are FP32's.  Launches and memory round trips
// bound it at the sizes below, the staging through registers on long ranges.
//
//  * Probabilities are three bf16 planes, each the rounding of what the last left:
//    their sum is the FP32 value.
//  * bf16 storage: Q, K and V are planes as they are.
//  * f16 storage: Q and K are, on the f16 form of the MFMA; V's 11 bits are two bf16
//    planes, exactly, and the product left out is below 2^-26 of the whole.  (Two
//    f16 planes of 2^11 P, two MFMAs where these take five, kept 22 bits of a weight
//    of 1 and none of one of 2^-36: 69 keys e^-25 as heavy as one whose V is zero
//    summed to 23% of their context.  They took 23.2 us for 128 queries over 2048
//    keys at 12/4/96, 24.2 for 300 tokens of 16/8/128 with diagnostics and 40.5 for
//    128 queries over 1025 keys at 8/1/512; these 26.1, 25.8 and 37.3.)
//  * F32 storage: Q, K and V are three bf16 planes each, and a product of two
//    values is the six plane products down to 2^-18 of it; the three left out are
//    below 2^-25 of it together, half of FP32's own rounding.
//
// Planes end at bf16's smallest number, 2^-133, so an element (or weight) below
// 2^-109 keeps fewer bits than FP32 has: contexts of V about 1e-33 are off by 2e-7 as
// all others, of 1e-36 by 3e-5, where FP32 products gave 4e-7.  Planes scaled apart
// would hold them at the price of a sum each (the sums apart below took FP32 1.5%
// longer), for values that no activation has.
//
// Against one wave per (query, head) on the vector unit, per call with the wait or
// the append where the call has one: a 128-token FP32 chunk at offset 1920 (14/2/64)
// 1017 -> 23.0 us, a 512-token FP32 prompt 313 -> 35.6 us, 300 tokens of 16/8/128 bf16
// with both diagnostics 243 -> 37.1 us, 128 queries over 1025 keys at 8/1/512 bf16
// 2240 -> 55 us; errors against 64 bits a quarter to 0.6 of its.
//
// Lane (j, g) holds query row j.  Q.K: A = K plane (key j of a 16-key block,
// features 32 s + 8 g .. + 7), B = Q.  P.V over 32 keys: the MFMA's k index
// 8 g + 4 b + r stands for key 16 b + 4 g + r, where the scores already sit, so P
// needs no exchange; A = V transposed, feature 16 fb + j, staged with its keys in
// that order.  A thread transposes four keys by four features in registers on the
// way to LDS.  The 16 rows of an operand read fall on distinct banks: K rows are
// padded by 16 bytes, V rows (whose size decides whether two workgroups of
// 512-wide heads fit a CU) have their 16-byte chunks XOR-swizzled by row.
__host__ __device__ constexpr int split_keys(int DP) { return DP <= 64 ? 64 : 32; }
__host__ __device__ constexpr int split_feature_waves(int DP) { return DP <= 256 ? 1 : 2; }
// Waves of a workgroup.  Four, and two workgroups per CU; but 512-wide f16 tiles (V in
// two planes: 113 KiB with the dots) leave room for one, which takes eight (with four,
// 128 queries over 1025 keys at 8/1/512 took 44.0 us and 256 over 2300 at 8/2/512 107,
// with eight 37.3 and 63; a wave then holds the next tile without spills, too).
__host__ __device__ constexpr int split_waves(int DT, int DP) { return DT == F16 && DP == 512 ? 8 : 4; }

namespace {

// Planes of Q and K, of V, and of a probability.
constexpr int PROB_PLANES = 3;
template <int DT> struct Planes { static constexpr int qk = 1, v = 1; };
template <> struct Planes<F32> { static constexpr int qk = 3, v = 3; };
template <> struct Planes<F16> { static constexpr int qk = 1, v = 2; };

template <int DT> __device__ __forceinline__ f32x4 mfma32k(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (DT == F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Two floats rounded to bf16 and packed; they keep what the rounding left.  (Cut
// off instead, values either side of a power of two have leading planes 0.4%
// apart, and sums that cancel in FP32 no longer do plane by plane.)  LIMIT: a
// value that would round to infinity takes the largest bf16 first.
template <bool LIMIT> __device__ __forceinline__ uint32_t plane2(float &a, float &b) {
    constexpr float top = 0x1.fep127f;
    const f32x2 v = {LIMIT ? __builtin_amdgcn_fmed3f(a, -top, top) : a, LIMIT ? __builtin_amdgcn_fmed3f(b, -top, top) : b};
    const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
    a -= __builtin_bit_cast(float, w << 16);
    b -= __builtin_bit_cast(float, w & 0xffff0000u);
    return w;
}

// Eight stored elements as planes of an MFMA operand.
template <int DT>
__device__ __forceinline__ void planes8(typename Raw4<DT>::T lo, typename Raw4<DT>::T hi, u32x4 (&out)[Planes<DT>::qk]) {
    if constexpr (DT == F32) {
        const f32x4 x = widen4<DT>(lo), y = widen4<DT>(hi);
        float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
        for (int e = 0; e < 4; ++e) {
            out[0][e] = plane2<true>(v[2 * e], v[2 * e + 1]);
            out[1][e] = plane2<false>(v[2 * e], v[2 * e + 1]);
            out[2][e] = plane2<false>(v[2 * e], v[2 * e + 1]);
        }
    } else {
        out[0] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
}

// A lane's probabilities of 32 keys (two score blocks) as planes.
__device__ __forceinline__ void prob_planes(const f32x4 &x, const f32x4 &y, u32x4 (&out)[PROB_PLANES]) {
    float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    for (int pl = 0; pl < PROB_PLANES; ++pl)
        for (int e = 0; e < 4; ++e) out[pl][e] = plane2<false>(v[2 * e], v[2 * e + 1]);
}

}  // namespace

// VE: elements that start and end every row in whole vectors (1: element loads).
template <int DT, int DP, int VE>
__global__ __launch_bounds__(64 * split_waves(DT, DP), 2) void attn_split(TileArgs a) {
    warm_kernarg<(sizeof(TileArgs) + 63) / 64, 0>();
    constexpr int KT = split_keys(DP), NB = KT / 16, NG = KT / 32, FS = split_feature_waves(DP);
    constexpr int NW = split_waves(DT, DP), NT = 64 * NW;     // waves and threads
    constexpr int DW = DP / FS, QS = DW / 32, FB = DW / 16;   // a wave's features, Q.K steps, P.V blocks
    constexpr int SP = Planes<DT>::qk, VP = Planes<DT>::v;
    constexpr int KROW = DP * 2 + 16, VROW = KT * 2;          // staged row bytes: K per key, V per feature
    constexpr int KPL = KT * KROW, VPL = DP * VROW;           // bytes per plane
    constexpr bool VEC = VE > 1;
    // A thread's K chunks of eight features and V blocks of four keys by VF
    // features.  Rows of whole 16-byte vectors of 16-bit elements load eight at a time
    // (K and Q: 300 tokens of 16/8/128 with diagnostics 39.7 -> 37.1 us a call); a wide
    // tile's V blocks take eight as well (with K and Q, 128 queries of 8/1/512 59.7 ->
    // 57.1), where narrower tiles have too few blocks for every thread.
    constexpr int VF = VE == 8 && DP >= 256 ? 8 : 4;
    constexpr int NK = KT * DP / 8 / NT, NV = KT * DP / (4 * VF) / NT;
    static_assert(NK >= 1 && NV >= 1, "staging covers the tile");
    __shared__ __attribute__((aligned(16))) uint8_t kt[SP * KPL];
    __shared__ __attribute__((aligned(16))) uint8_t vt[VP * VPL];
    __shared__ __attribute__((aligned(16))) f32x4 dots[FS > 1 ? NW * NB * 64 : 1];  // partial scores
    using Raw = typename Raw4<DT>::T;
    const Params &p = a.p;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int j = lane & 15, g = lane >> 4;
    const int D = p.head_dim;
    const bool full_diag = p.diag_mode == 1;
    const_ptr<Problem> pr;
    const TileWork w = tile_work(a, wave / FS, j, &pr);
    const int fs = wave % FS, f0 = fs * DW;  // the wave's features start at f0
    const int nseg = pr->nseg, n = w.n;
    // Byte offset of 16-byte chunk c of V row f.
    auto v_at = [](int f, int c) { return f * VROW + ((c ^ (KT == 32 ? f >> 2 & 3 : f >> 1 & 7)) << 4); };

    // Features past the head are zeros in Q, K and V (attn_tile's loads).
    const Raw none{};
    auto whole = [&](int d, int width) { return VE == 1 || d + width <= D; };
    auto load_four = [&](const void *base, auto off, int d) {
        return load4<DT, VEC>(base, off + (VEC ? min(d, D - 4) : d), D - d);
    };
    auto load_eight = [&](const void *base, auto off, int d, Raw (&to)[2]) {
        if constexpr (VE == 8) {
            const u32x4 x = *gload_ptr<u32x4>(reinterpret_cast<const uint8_t *>(base) + (off + min(d, D - 8)) * 2);
            to[0] = Raw{x[0], x[1]};
            to[1] = Raw{x[2], x[3]};
        } else {
            to[0] = load_four(base, off, d);
            to[1] = load_four(base, off, d + 4);
        }
    };
    Raw qraw[QS][2];
    {
        const int64_t at = (int64_t)w.t_row * pr->q_row_stride + (int64_t)w.h_row * D;
        for (int s = 0; s < QS; ++s) load_eight(pr->q, at, f0 + 32 * s + 8 * g, qraw[s]);
    }

    // K chunk m of a thread: row i / (DP / 8), features 8 (i % (DP / 8)).  V block
    // m: key quad i % 8 of its 32-key group, features VF (i / 8 % (DP / VF)).
    constexpr int CPR = DP / 8, FPR = DP / VF;
    Raw kreg[NK][2], vreg[NV][4][VF / 4];
    // at(row) -> (K, V) addresses of the tile's row, whose elements follow.
    auto fetch_rows = [&](auto at) {
#pragma unroll
        for (int m = 0; m < NK; ++m) {
            const int i = tid + NT * m, d = 8 * (i % CPR);
            const void *kb, *vb;
            const auto off = at(i / CPR, &kb, &vb);
            load_eight(kb, off, d, kreg[m]);
        }
#pragma unroll
        for (int m = 0; m < NV; ++m) {
            const int i = tid + NT * m, d = VF * (i / 8 % FPR), k0 = i / (8 * FPR) * 32 + 4 * (i % 8);
            for (int r = 0; r < 4; ++r) {
                const void *kb, *vb;
                const auto off = at(k0 + r, &kb, &vb);
                if constexpr (VF == 8) load_eight(vb, off, d, vreg[m][r]);
                else vreg[m][r][0] = load_four(vb, off, d);
            }
        }
    };
    constexpr int ES = ElemSize<DT>::value;
    auto fetch = [&](int t0) {
        const int left = n - 1 - t0;  // rows past the last repeat it
        if (VEC && nseg == 1) {
            // A tile's rows span less than 2 GiB (launch_tile): a uniform base and
            // 32-bit offsets.
            const int64_t first = ((int64_t)w.kvh * pr->seg[0].head_stride + (w.lo + t0) * pr->seg[0].row_stride) * ES;
            const uint8_t *kb = reinterpret_cast<const uint8_t *>(pr->seg[0].k) + first;
            const uint8_t *vb = reinterpret_cast<const uint8_t *>(pr->seg[0].v) + first;
            const uint32_t rs = (uint32_t)pr->seg[0].row_stride;
            auto rows = [&](auto row_of) {
                fetch_rows([&](int r, const void **k, const void **v) {
                    *k = kb;
                    *v = vb;
                    return row_of(r) * rs;
                });
            };
            if (left >= KT - 1) rows([](int r) { return (uint32_t)r; });
            else rows([&](int r) { return (uint32_t)min(r, left); });
        } else {
            fetch_rows([&](int r, const void **k, const void **v) { return seg_select(pr, w.lo + t0 + min(r, left), w.kvh, k, v); });
        }
    };
    // The first tile is on its way before Q is waited for.
    if (n > 0) fetch(0);
    u32x4 q[QS][SP];
    for (int s = 0; s < QS; ++s) {
        const int d = f0 + 32 * s + 8 * g;
        planes8<DT>(whole(d, 4) ? qraw[s][0] : none, whole(d + 4, 4) ? qraw[s][1] : none, q[s]);
    }
    auto stage = [&](int t0) {
#pragma unroll
        for (int m = 0; m < NK; ++m) {
            const int i = tid + NT * m, d = 8 * (i % CPR);
            u32x4 pl[SP];
            planes8<DT>(whole(d, 4) ? kreg[m][0] : none, whole(d + 4, 4) ? kreg[m][1] : none, pl);
            for (int s = 0; s < SP; ++s) *reinterpret_cast<u32x4 *>(kt + s * KPL + i / CPR * KROW + 2 * d) = pl[s];
        }
#pragma unroll
        for (int m = 0; m < NV; ++m) {
            const int i = tid + NT * m, qd = i % 8, d0 = VF * (i / 8 % FPR), t = i / (8 * FPR);
            const int k0 = t0 + 32 * t + 4 * qd;
            for (int half = 0; half < VF / 4; ++half) {
                const int d = d0 + 4 * half;
                Raw x[4];
                for (int r = 0; r < 4; ++r)
                    x[r] = whole(d, 4) && k0 + r >= w.vlo && k0 + r < w.vhi ? vreg[m][r][half] : none;
                // Row f holds the group's keys as 8-byte pieces: g = qd % 4 first, then b = qd / 4.
                auto to = [&](int e) { return vt + v_at(d + e, 4 * t + (qd & 3)) + 8 * (qd >> 2); };
                if constexpr (VP > 1) {
                    f32x4 y[4];
                    for (int r = 0; r < 4; ++r) y[r] = widen4<DT>(x[r]);
                    for (int e = 0; e < 4; ++e) {
                        float v[4] = {y[0][e], y[1][e], y[2][e], y[3][e]};
                        for (int s = 0; s < VP; ++s) {
                            using Quad = typename Raw4<F16>::T;
                            constexpr bool LIMIT = DT == F32;
                            const Quad o = s == 0 ? Quad{plane2<LIMIT>(v[0], v[1]), plane2<LIMIT>(v[2], v[3])}
                                                  : Quad{plane2<false>(v[0], v[1]), plane2<false>(v[2], v[3])};
                            *reinterpret_cast<Quad *>(to(e) + s * VPL) = o;
                        }
                    }
                } else {
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t pick = e & 1 ? 0x07060302u : 0x05040100u;
                        const uint32_t o0 = __builtin_amdgcn_perm(x[1][e >> 1], x[0][e >> 1], pick);
                        const uint32_t o1 = __builtin_amdgcn_perm(x[3][e >> 1], x[2][e >> 1], pick);
                        *reinterpret_cast<Raw *>(to(e)) = Raw{o0, o1};
                    }
                }
            }
        }
    };

    f32x4 acc[FB];
    for (int fb = 0; fb < FB; ++fb) acc[fb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const float mul = exp_mul(p);
    float m_run = NEG_INF, l_run = 0.0f, amax = 0.0f;  // m_run: the row's maximum y

    for (int t0 = 0; t0 < n; t0 += KT) {
        __syncthreads();
        stage(t0);
        __syncthreads();
        if (t0 + KT < n) fetch(t0 + KT);
        f32x4 st[NB];
        bool seen[NB], scored[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int k0 = t0 + 16 * b;
            seen[b] = w.active && k0 < w.whi && k0 + 16 > w.wlo;
            scored[b] = seen[b] || (full_diag && w.active && k0 < n);
            f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;  // the leading planes, the rest (or two chains)
            if (scored[b]) {
                const uint8_t *kr = kt + (16 * b + j) * KROW + 2 * f0 + 16 * g;
#pragma unroll
                for (int s = 0; s < QS; ++s) {
                    u32x4 k[SP];
                    for (int pl = 0; pl < SP; ++pl) k[pl] = *reinterpret_cast<const u32x4 *>(kr + pl * KPL + 64 * s);
                    if constexpr (SP == 3) {
                        s0 = mfma32k<DT>(k[0], q[s][0], s0);
                        s1 = mfma32k<DT>(k[2], q[s][0], s1);
                        s1 = mfma32k<DT>(k[0], q[s][2], s1);
                        s1 = mfma32k<DT>(k[1], q[s][1], s1);
                        s1 = mfma32k<DT>(k[1], q[s][0], s1);
                        s1 = mfma32k<DT>(k[0], q[s][1], s1);
                    } else if (s % 2 == 0) {
                        s0 = mfma32k<DT>(k[0], q[s][0], s0);
                    } else {
                        s1 = mfma32k<DT>(k[0], q[s][0], s1);
                    }
                }
            }
            for (int r = 0; r < 4; ++r) st[b][r] = s0[r] + s1[r];
            if constexpr (FS > 1) dots[(wave * NB + b) * 64 + lane] = st[b];
        }
        if constexpr (FS > 1) {
            __syncthreads();
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const f32x4 *d = dots + (wave - fs) * NB * 64 + b * 64 + lane;
                st[b] = d[0];
                for (int x = 1; x < FS; ++x)
                    for (int r = 0; r < 4; ++r) st[b][r] += d[x * NB * 64][r];
            }
        }
        float tmax = finish_scores<NB>(p, w, pr, t0, g, fs == 0, scored, st, amax);
        tmax = row4_max(tmax);
        const float m_new = fmaxf(m_run, tmax);
        if (__ballot(m_new > m_run) != 0) {
            const float corr = weight(m_run, finite_max(m_new), mul);
            l_run *= corr;
            for (int fb = 0; fb < FB; ++fb)
                for (int r = 0; r < 4; ++r) acc[fb][r] *= corr;
            m_run = m_new;
        }
        const float m_ref = finite_max(m_run);
#pragma unroll
        for (int t = 0; t < NG; ++t) {
            if (!seen[2 * t] && !seen[2 * t + 1]) continue;
            for (int b = 2 * t; b < 2 * t + 2; ++b)
                for (int r = 0; r < 4; ++r) {
                    st[b][r] = weight(st[b][r], m_ref, mul);
                    l_run += st[b][r];
                }
            u32x4 pb[PROB_PLANES];
            prob_planes(st[2 * t], st[2 * t + 1], pb);
            const uint8_t *vr = vt + v_at(f0 + j, 4 * t + g);  // the swizzle repeats every 16 rows
#pragma unroll
            for (int fb = 0; fb < FB; ++fb) {
                u32x4 v[VP];
                for (int pl = 0; pl < VP; ++pl) v[pl] = *reinterpret_cast<const u32x4 *>(vr + pl * VPL + 16 * fb * VROW);
                // The smallest products first.  f16's five are summed before they join
                // the context: rounded once, as its error against 64 bits asks for
                // (2.88e-7 -> 2.09e-7 for 256 queries over 2300 keys at 8/2/512, and
                // 2.38e-7 from planes of 22 bits).
                constexpr bool APART = DT == F16;
                f32x4 o = APART ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : acc[fb];
                if constexpr (VP == 3) o = mfma32k<BF16>(v[2], pb[0], o);
                o = mfma32k<BF16>(v[0], pb[2], o);
                if constexpr (VP > 1) {
                    o = mfma32k<BF16>(v[1], pb[1], o);
                    o = mfma32k<BF16>(v[1], pb[0], o);
                }
                o = mfma32k<BF16>(v[0], pb[1], o);
                o = mfma32k<BF16>(v[0], pb[0], o);
                if constexpr (APART)
                    for (int r = 0; r < 4; ++r) acc[fb][r] += o[r];
                else acc[fb] = o;
            }
        }
    }

    l_run = row4_sum(l_run);
    bool bad = !finite_scores(p, amax);
    TileOut out(a, w, pr, DP, g == 0 && fs == 0, m_run, l_run);
    if (w.rvalid)
        for (int fb = 0; fb < FB; ++fb) out.emit(f0 + 16 * fb + 4 * g, acc[fb], bad);
    out.report(p, bad);
}

// The probabilities of one diagnostics row by one wave, from the scores the
// attention kernel stored (in the probability buffer itself when the caller asked
// for no scores): masked keys are exactly +0.  The row's partials are merged by the
// lanes (at most 64 of them).
__device__ __forceinline__ void probs_row(const TileArgs &a, int64_t row_index) {
    const Params &p = a.p;
    const Problem &pr = p.single;  // diagnostics are single-problem calls
    const int G = p.group, Hq = p.query_heads, lane = threadIdx.x & 63;
    const bool full = p.diag_mode == 1;
    const int64_t hr = full ? row_index : (int64_t)Hq * pr.queries - 1;
    const int h = (int)(hr / pr.queries), t = (int)(hr % pr.queries);
    const int m_kv = pr.queries * G, S = pr.splits * a.kw;
    const int64_t local = (int64_t)(h / G) * m_kv + (int64_t)t * G + h % G;
    const float *ml = p.part_ml + 2 * (pr.slot_base + local * S);
    f32x2 mine = {NEG_INF, 0.0f};
    if (lane < S) mine = *gload_ptr<f32x2>(ml + 2 * lane);
    int64_t lo, hi;
    visible_range(p, pr, pr.q_pos0 + t, &lo, &hi);
    const int64_t row = full ? hr * pr.keys : 0, end = full ? pr.keys : hi;
    const float *xs = (p.scores ? p.scores : p.probs) + row;
    const float mul = exp_mul(p), M = finite_max(wave_max(mine[0]));
    const float L = wave_sum(weight(mine[0], M, mul) * mine[1]);
    const float inv = 1.0f / L;
#pragma unroll 4
    for (int64_t key = (full ? 0 : lo) + lane; key < end; key += 64) {
        const float x = xs[key];
        p.probs[row + key] = key >= lo && key < hi ? weight(x, M, mul) * inv : 0.0f;
    }
}

__device__ __forceinline__ int find_row_problem(const Params &p, int64_t row) {
    int lo = 0, hi = p.nproblems - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (p.problems[mid].part_base <= row) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Split-K combine, in the first merge_blocks workgroups: one thread per four
// features of a row, so a launch has rows x D / 4 threads and a thread's partials
// (16 splits at a time) are all in flight together; the time is one memory round
// trip.  The workgroups after those make the diagnostics' probabilities, a wave per
// row: 300 tokens of 16/8/128 took 5 us and, as a launch of its own whose threads
// each went through a row's partials one by one, 11 us; together they take 9.6.
__global__ __launch_bounds__(256) void attn_tile_merge(TileArgs a, int64_t total_rows, int dp, uint32_t merge_blocks) {
    const Params &p = a.p;
    if (blockIdx.x >= merge_blocks) {
        const int64_t r = (int64_t)(blockIdx.x - merge_blocks) * 4 + (threadIdx.x >> 6);
        if (r < (p.diag_mode == 1 ? (int64_t)p.query_heads * p.single.queries : 1)) probs_row(a, r);
        return;
    }
    const int D = p.head_dim, Hq = p.query_heads, G = p.group;
    const uint32_t per = (uint32_t)(D + 3) / 4;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = i / per;
    if (row >= total_rows) return;
    const int d = 4 * (int)(i - row * per);
    const Problem &pr = p.nproblems == 1 ? p.single : p.problems[find_row_problem(p, row)];
    const int m_kv = pr.queries * G, S = pr.splits * a.kw;
    const int64_t local = row - pr.part_base;
    const int kvh = (int)(local / m_kv), prow = (int)(local % m_kv);
    const int64_t part = pr.slot_base + local * S;
    const float *ml = p.part_ml + 2 * part, *po = p.part_o + part * dp + d;
    constexpr int W = 16;
    const float mul = exp_mul(p);
    float M = NEG_INF, L = 0.0f;
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < S; s0 += W) {
        f32x2 mv[W];
        f32x4 ov[W];
        float M1 = M;
#pragma unroll
        for (int s = 0; s < W; ++s)
            if (s0 + s < S) {
                mv[s] = *gload_ptr<f32x2>(ml + 2 * (s0 + s));
                ov[s] = *gload_ptr<f32x4>(po + (int64_t)(s0 + s) * dp);
            }
#pragma unroll
        for (int s = 0; s < W; ++s)
            if (s0 + s < S) M1 = fmaxf(M1, mv[s][0]);
        const float base = finite_max(M1), corr = weight(M, base, mul);
        L *= corr;
        for (int e = 0; e < 4; ++e) o[e] *= corr;
#pragma unroll
        for (int s = 0; s < W; ++s)
            if (s0 + s < S && mv[s][0] != NEG_INF) {
                const float w = weight(mv[s][0], base, mul);
                L = __builtin_fmaf(w, mv[s][1], L);
                for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(w, ov[s][e], o[e]);
            }
        M = M1;
    }
    const bool bad_mass = !(L > 0.0f) || !is_finite_f(L);
    const float inv = 1.0f / L;
    bool bad_out = false;
    float *out = pr.out + ((int64_t)(prow / G) * Hq + kvh * G + prow % G) * D + d;
    for (int e = 0; e < 4; ++e) {
        o[e] *= inv;
        bad_out |= d + e < D && !is_finite_f(o[e]);
    }
    if (d + 4 <= D) *reinterpret_cast<f32x4u *>(out) = o;
    else
        for (int e = 0; e < 4; ++e)
            if (d + e < D) out[e] = o[e];
    raise_status(p, bad_mass, ST_BAD_MASS);
    raise_status(p, bad_out, ST_NONFINITE_OUTPUT);
}

}  // namespace tkh

// Head sizes the kernels are built for (the smallest that holds `head_dim`).
extern "C" int tkh_tile_head(int head_dim) {
    return head_dim <= 64 ? 64 : (head_dim <= 128 ? 128 : (head_dim <= 256 ? 256 : 512));
}
// attn_split takes every 16-bit launch and FP32 ones up to 128, whose six plane
// products cost 6/16 of FP32 MFMAs; three planes of wider FP32 tiles do not leave
// room for two workgroups in LDS, and those stay on attn_tile.
static bool tile_splits(int dtype, int head_dim) { return dtype != tkh::F32 || tkh_tile_head(head_dim) <= 128; }
// Waves of a workgroup, and workgroups a CU holds.
static int tile_waves(int dtype, int head_dim) {
    return tile_splits(dtype, head_dim) ? tkh::split_waves(dtype, tkh_tile_head(head_dim)) : 4;
}
extern "C" int tkh_tile_resident(int dtype, int head_dim) { return tile_waves(dtype, head_dim) > 4 ? 1 : 2; }
// Keys of a staged tile, row groups a workgroup has waves for, and how many of
// its waves may share a row group's keys.
extern "C" int tkh_tile_keys(int dtype, int head_dim) {
    const int dp = tkh_tile_head(head_dim);
    return tile_splits(dtype, head_dim) ? tkh::split_keys(dp) : tkh::tile_keys(dp);
}
extern "C" int tkh_tile_row_waves(int dtype, int head_dim) {
    const int dp = tkh_tile_head(head_dim);
    return tile_waves(dtype, head_dim) / (tile_splits(dtype, head_dim) ? tkh::split_feature_waves(dp) : tkh::tile_feature_waves(dp));
}
extern "C" int tkh_tile_share(int dtype, int head_dim) {
    return tile_splits(dtype, head_dim) ? 1 : tkh_tile_keys(dtype, head_dim) / 16;
}

// start/stop, when not null, are recorded around the kernel by the dispatch
// itself (hipExtLaunchKernelGGL), so profiled durations exclude the host gap
// that separate hipEventRecord calls would add.
extern "C" hipError_t tkh_launch_tile(const tkh::TileArgs *a, int dtype, hipStream_t stream,
                                      hipEvent_t start, hipEvent_t stop) {
    using namespace tkh;
    const int dp = tkh_tile_head(a->p.head_dim);
    dim3 grid((unsigned)a->p.total_tiles), block((unsigned)(64 * tile_waves(dtype, a->p.head_dim)));
#define TKH_LAUNCH(...) hipExtLaunchKernelGGL((__VA_ARGS__), grid, block, 0, stream, start, stop, 0, *a)
#define TKH_TILE(DP)                                                                    \
    if (dtype == F32 && dp == DP) {                                                     \
        if (a->vec >= 4) TKH_LAUNCH(attn_tile<DP, true>);                               \
        else TKH_LAUNCH(attn_tile<DP, false>);                                          \
        return hipGetLastError();                                                       \
    }
#define TKH_SPLIT(DT, DP)                                                               \
    if (dtype == DT && dp == DP) {                                                      \
        if (DT != F32 && a->vec >= 8) TKH_LAUNCH(attn_split<DT, DP, DT != F32 ? 8 : 4>); \
        else if (a->vec >= 4) TKH_LAUNCH(attn_split<DT, DP, 4>);                        \
        else TKH_LAUNCH(attn_split<DT, DP, 1>);                                         \
        return hipGetLastError();                                                       \
    }
    TKH_SPLIT(F32, 64) TKH_SPLIT(F32, 128) TKH_TILE(256) TKH_TILE(512)
    TKH_SPLIT(F16, 64) TKH_SPLIT(F16, 128) TKH_SPLIT(F16, 256) TKH_SPLIT(F16, 512)
    TKH_SPLIT(BF16, 64) TKH_SPLIT(BF16, 128) TKH_SPLIT(BF16, 256) TKH_SPLIT(BF16, 512)
#undef TKH_SPLIT
#undef TKH_TILE
#undef TKH_LAUNCH
    return hipErrorInvalidValue;
}

// The combine of `total_rows` rows (0: the keys were not split) and the
// probabilities, when the call asks for them.
extern "C" hipError_t tkh_launch_tile_merge(const tkh::TileArgs *a, int64_t total_rows, hipStream_t stream,
                                            hipEvent_t start, hipEvent_t stop) {
    using namespace tkh;
    const int64_t merge = (total_rows * ((a->p.head_dim + 3) / 4) + 255) / 256;
    const int64_t rows = !a->p.probs ? 0 : (a->p.diag_mode == 1 ? (int64_t)a->p.query_heads * a->p.single.queries : 1);
    dim3 grid((unsigned)(merge + (rows + 3) / 4)), block(256);
    hipExtLaunchKernelGGL(attn_tile_merge, grid, block, 0, stream, start, stop, 0, *a, total_rows,
                          tkh_tile_head(a->p.head_dim), (uint32_t)merge);
    return hipGetLastError();
}
