// MoE routing, grouping, merge and argmax kernels (integer/bandwidth work, no MFMA).
#include "dih_device.h"
#include "dih_internal.h"

namespace dih {

// ------------------------------------------------------------------------------ top-8

// One wave per token (prefill_top8 gpu_prefill.mm:151-161 / SelectExperts
// Qwen36Model.cs:246-262): eight rounds of wave max with ties to the lowest expert id,
// then softmax over the eight chosen logits (largest subtracted, summed in slot order).
// A non-finite logit sets *status = 1, the token's ids to 0 and its probabilities to NaN: the
// merge then leaves that token's residual (and normed row) unchanged, where the reference's
// host path throws before writing (SelectExperts, Qwen36Model.cs:252).
__global__ __launch_bounds__(256) void top8_kernel(const void *logits, int logits_bf16, int tokens,
                                                   int experts, uint32_t *ids, float *probs,
                                                   uint32_t *status, float *logits_copy,
                                                   uint32_t *zero_word) {
    if (zero_word && blockIdx.x == 0 && threadIdx.x == 0) *zero_word = 0u;
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= tokens) return;
    float cand[4];
    bool bad = false;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int e = lane + 64 * j;
        float v = -INFINITY;
        if (e < experts) {
            const size_t at = (size_t)t * experts + e;
            v = logits_bf16 ? bf16_to_f32(static_cast<const uint16_t *>(logits)[at])
                            : static_cast<const float *>(logits)[at];
            if (!isfinite(v)) bad = true;
            if (logits_copy) logits_copy[at] = v;
        }
        cand[j] = v;
    }
    const bool any_bad = __any(bad);
    float chosen[8];
    uint32_t picked[8];
#pragma unroll
    for (int n = 0; n < 8; n++) {
        float best = cand[0];
        uint32_t id = (uint32_t)lane;
#pragma unroll
        for (int j = 1; j < 4; j++)
            if (cand[j] > best) { best = cand[j]; id = (uint32_t)(lane + 64 * j); }
        const float m = wave_max(best);
        const uint32_t sel = wave_min_u32(best == m ? id : 0xffffffffu);
        chosen[n] = m;
        picked[n] = sel;
#pragma unroll
        for (int j = 0; j < 4; j++)
            if ((uint32_t)(lane + 64 * j) == sel) cand[j] = -INFINITY;
    }
    if (lane == 0) {
        float p[8], total = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) { p[i] = __expf(chosen[i] - chosen[0]); total += p[i]; }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            ids[(size_t)t * 8 + i] = any_bad ? 0u : picked[i];
            probs[(size_t)t * 8 + i] = any_bad ? __builtin_nanf("") : p[i] / total;
        }
        if (any_bad && status) *status = 1u;
    }
}

bool launch_top8(const void *logits, int logits_bf16, int tokens, int experts, uint32_t *ids,
                 float *probs, uint32_t *status, float *logits_copy, uint32_t *zero_word,
                 hipStream_t s, char *error, int capacity) {
    DIH_LAUNCH(top8_kernel, dim3((tokens + 3) / 4), dim3(256), 0, s, logits, logits_bf16,
                       tokens, experts, ids, probs, status, logits_copy, zero_word);
    return hip_ok(hipGetLastError(), error, capacity, "top8 launch");
}

// ------------------------------------------------------------------------- grouping

// Block e lists the routes r (= token*8 + slot) with ids[r] == e in ascending order
// (prefill_build_groups prefill_moe.mm:8-17 uses a SIMD prefix sum per 32 routes). Here a
// thread takes 64 consecutive routes a pass (16 K routes per pass of 256 threads, all its
// loads issued together), counts its matches and places them after an add-scan of the
// block's counts: one barrier per pass. Block `experts` (when with_shared) lists the
// shared expert's routes T*8 + t for every token. Blocks do not communicate: the GEMM
// derives its chunks from the counts (in expert order, so the order is deterministic where
// the reference's atomic tile append, prefill_moe.mm:15, is not).
__global__ __launch_bounds__(256) void group_kernel(const uint32_t *ids, int tokens, int experts,
                                                    int with_shared, uint32_t *counts,
                                                    uint32_t *routes) {
    constexpr int kPer = 64;   // routes per thread and pass
    __shared__ uint32_t wave_tot[2][4];
    const int e = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int T8 = tokens * 8;
    uint32_t *out = routes + (size_t)e * tokens;
    if (e == experts) {
        for (int t = tid; t < tokens; t += 256) out[t] = (uint32_t)(T8 + t);
        if (tid == 0) counts[e] = (uint32_t)tokens;
        return;
    }
    uint32_t total = 0;
    int buf = 0;
    for (int base = 0; base < T8; base += 256 * kPer, buf ^= 1) {
        const int r0 = base + kPer * tid;
        // 16-byte loads at clamped offsets (T8 is a multiple of 8), masked past the routes
        uint4 v[kPer / 4];
#pragma unroll
        for (int k4 = 0; k4 < kPer / 4; k4++)
            v[k4] = *reinterpret_cast<const uint4 *>(ids + min(r0 + 4 * k4, T8 - 4));
        uint64_t hit = 0;
#pragma unroll
        for (int k4 = 0; k4 < kPer / 4; k4++) {
            if (r0 + 4 * k4 >= T8) continue;
            const uint64_t h = (uint64_t)(v[k4].x == (uint32_t)e) | (uint64_t)(v[k4].y == (uint32_t)e) << 1 |
                               (uint64_t)(v[k4].z == (uint32_t)e) << 2 | (uint64_t)(v[k4].w == (uint32_t)e) << 3;
            hit |= h << (4 * k4);
        }
        const uint32_t cnt = (uint32_t)__popcll(hit);
        uint32_t incl = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(incl, d, 64);
            if (lane >= d) incl += y;
        }
        if (lane == 63) wave_tot[buf][wave] = incl;
        __syncthreads();
        uint32_t off = total + incl - cnt;
        for (int w = 0; w < wave; w++) off += wave_tot[buf][w];
        // A token lists an expert at most once, so count <= tokens; ids that repeat an
        // expert within a token are truncated here instead of overrunning the list.
        while (hit) {
            const int k = __builtin_ctzll(hit);
            hit &= hit - 1;
            if (off < (uint32_t)tokens) out[off] = (uint32_t)(r0 + k);
            off++;
        }
        total += wave_tot[buf][0] + wave_tot[buf][1] + wave_tot[buf][2] + wave_tot[buf][3];
    }
    if (tid == 0) counts[e] = min(total, (uint32_t)tokens);
}

bool launch_build_groups(const uint32_t *ids, int tokens, int experts, int with_shared,
                         uint32_t *counts, uint32_t *routes, hipStream_t s, char *error, int capacity) {
    DIH_LAUNCH(group_kernel, dim3(experts + with_shared), dim3(256), 0, s, ids, tokens, experts,
               with_shared, counts, routes);
    return hip_ok(hipGetLastError(), error, capacity, "grouping launch");
}

// ---------------------------------------------------------------------------- merge

// One block per token (prefill_merge gpu_prefill.mm:140-150): gate = sigmoid(shared_route .
// x[t]); y = gate*out[T*8+t] + sum_{slot 0..7} p*out[t*8+slot]; residual[t] += y (f32 or
// bf16 storage); with norm_w, normed[t] = r * rsqrt(mean(r^2) + eps) * norm_w over the
// stored r.
//
// Bound by latency for short chunks and by the route outputs (9*H*4 bytes a token) for long
// ones. A thread owns VEC consecutive columns of each 256*VEC, two such pieces at a time: the
// nine route rows, the residual and the norm weights of the first two pieces (all of a
// 2048-wide row) are requested before the shared-expert gate's dot product, whose wait and
// barrier they then cover, and a row of up to kMergeHold pieces keeps its stored r in
// registers for the norm. VEC 4 needs every row 16-byte aligned (8-byte for bf16), VEC 1
// takes any other caller buffers. Against one column a thread at a time behind the gate: a
// 77-token 5-bit layer with norm 143.2 -> 138.6 us, 2048 tokens 349.9 -> 343.6 us; a 512-token
// 8-bit one within the runs' spread.
constexpr int kMergeHold = 2;

// VEC consecutive elements of an f32 or bf16 row.
template <int VEC>
DIH_DEV void row_load(float (&v)[VEC], const void *p, int f32, size_t at) {
    if constexpr (VEC == 4) {
        if (f32) {
            const dih_f32x4 q = *reinterpret_cast<const dih_f32x4 *>(static_cast<const float *>(p) + at);
            v[0] = q[0]; v[1] = q[1]; v[2] = q[2]; v[3] = q[3];
        } else {
            const uint2 q = *reinterpret_cast<const uint2 *>(static_cast<const uint16_t *>(p) + at);
            v[0] = __uint_as_float(q.x << 16); v[1] = __uint_as_float(q.x & 0xffff0000u);
            v[2] = __uint_as_float(q.y << 16); v[3] = __uint_as_float(q.y & 0xffff0000u);
        }
    } else {
        v[0] = residual_load(p, f32, at);
    }
}

// Stores them; v becomes what was stored (rounded to bf16).
template <int VEC>
DIH_DEV void row_store(float (&v)[VEC], void *p, int f32, size_t at) {
    if constexpr (VEC == 4) {
        if (f32) {
            *reinterpret_cast<dih_f32x4 *>(static_cast<float *>(p) + at) = dih_f32x4{v[0], v[1], v[2], v[3]};
        } else {
            const uint2 q = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(p) + at) = q;
            v[0] = __uint_as_float(q.x << 16); v[1] = __uint_as_float(q.x & 0xffff0000u);
            v[2] = __uint_as_float(q.y << 16); v[3] = __uint_as_float(q.y & 0xffff0000u);
        }
    } else {
        v[0] = residual_store(p, f32, at, v[0]);
    }
}

template <int BITS, int VEC>
__global__ __launch_bounds__(256) void merge_kernel(const uint32_t *sr_packed,
                                                    const uint16_t *sr_scales,
                                                    const uint16_t *sr_biases,
                                                    const uint16_t *x, int tokens, int H,
                                                    const float *route_out, const float *probs,
                                                    void *residual, MergeOut mo) {
    __shared__ float part[4];
    __shared__ float sq[4];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nchunk = H >> 5;
    const int np = H / VEC;   // pieces of a row (H is a multiple of 64)
    const float *sh = route_out + ((size_t)tokens * 8 + t) * H;
    const float *ro = route_out + (size_t)t * 8 * H;
    const size_t row = (size_t)t * H;
    // this thread's pieces p0 and p0 + 256 (clamped in bounds; pieces past the row are not
    // stored): shared row, eight route rows, residual
    float in[2][9][VEC], res[2][VEC], nw[2][VEC];
    auto load = [&](int p0) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int c = VEC * min(p0 + 256 * k, np - 1);
            row_load<VEC>(in[k][8], sh, 1, c);
#pragma unroll
            for (int s = 0; s < 8; s++) row_load<VEC>(in[k][s], ro + (size_t)s * H, 1, c);
            row_load<VEC>(res[k], residual, mo.residual_f32, row + c);
        }
    };
    float p[8];
#pragma unroll
    for (int s = 0; s < 8; s++) p[s] = probs[(size_t)t * 8 + s];
    // the gate's operands first: its wait then leaves the rows in flight
    Chunk<BITS> c0;
    float xr[32];
    uint32_t sc0 = 0, bi0 = 0;
    if (tid < nchunk) {
        load_chunk<BITS>(c0, sr_packed, tid);
        sc0 = sr_scales[tid >> 1];
        bi0 = sr_biases[tid >> 1];
        load_x32(xr, x + row, 1, tid * 32);
    }
    load(tid);
    if (mo.norm_w) {
#pragma unroll
        for (int k = 0; k < 2; k++) row_load<VEC>(nw[k], mo.norm_w, 1, VEC * min(tid + 256 * k, np - 1));
    }
    // (a row has at most 256 chunks: one a thread)
    float d = 0.f;
    if (tid < nchunk) {
        float xs = 0.f;
#pragma unroll
        for (int i = 0; i < 32; i++) xs += xr[i];
        d = bf16_to_f32(sc0) * chunk_dot<BITS>(c0, xr) + bf16_to_f32(bi0) * xs;
    }
    d = wave_sum(d);
    if (lane == 0) part[wave] = d;
    __syncthreads();
    const float gate = sigmoidf_((part[0] + part[1]) + (part[2] + part[3]));
    // a token whose router logits were not finite (NaN probabilities) keeps its residual
    // and normed row unchanged (uniform over the block: one token)
    if (__builtin_isnan(p[0])) return;
    float ss = 0.f;
    for (int p0 = tid; p0 < np; p0 += 512) {
        if (p0 != tid) load(p0);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            if (p0 + 256 * k >= np) continue;
#pragma unroll
            for (int j = 0; j < VEC; j++) {
                float y = in[k][8][j] * gate;
#pragma unroll
                for (int s = 0; s < 8; s++) y += in[k][s][j] * p[s];
                res[k][j] += y;
            }
            row_store<VEC>(res[k], residual, mo.residual_f32, row + VEC * (p0 + 256 * k));
#pragma unroll
            for (int j = 0; j < VEC; j++) ss += res[k][j] * res[k][j];
        }
    }
    if (!mo.norm_w) return;  // uniform over the launch
    ss = wave_sum(ss);
    if (lane == 0) sq[wave] = ss;
    __syncthreads();
    const float scale = rsqrtf(((sq[0] + sq[1]) + (sq[2] + sq[3])) / (float)H + mo.eps);
    const bool held = np <= 256 * kMergeHold;
    for (int p0 = tid; p0 < np; p0 += 512) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int pc = p0 + 256 * k;
            if (pc >= np) continue;
            if (!held) {   // (each thread re-reads only the elements it wrote)
                row_load<VEC>(res[k], residual, mo.residual_f32, row + VEC * pc);
                row_load<VEC>(nw[k], mo.norm_w, 1, VEC * pc);
            }
            float v[VEC];
#pragma unroll
            for (int j = 0; j < VEC; j++) v[j] = res[k][j] * scale * nw[k][j];
            row_store<VEC>(v, mo.normed, mo.normed_f32, row + VEC * pc);
        }
    }
}

// Whether rows of `H` elements (a multiple of 64) from p can be read four elements at a time.
static bool rows_by_four(const void *p, int f32) {
    return (reinterpret_cast<uintptr_t>(p) & (f32 ? 15 : 7)) == 0;
}

bool launch_moe_merge(const Matrix *shared_route, const uint16_t *x, int tokens, int hidden,
                      const float *route_out, const float *probs, void *residual,
                      const MergeOut &mo, hipStream_t s, char *error, int capacity) {
    const bool four = rows_by_four(route_out, 1) && rows_by_four(residual, mo.residual_f32) &&
                      (!mo.norm_w || (rows_by_four(mo.norm_w, 1) && rows_by_four(mo.normed, mo.normed_f32)));
#define DIH_MERGE_CASE(B, V)                                                                                  \
    if (shared_route->bits == B && four == (V == 4))                                                          \
        DIH_LAUNCH((merge_kernel<B, V>), dim3(tokens), dim3(256), 0, s, shared_route->packed(),               \
                   shared_route->scales(), shared_route->biases(), x, tokens, hidden, route_out, probs,       \
                   residual, mo);
    DIH_MERGE_CASE(8, 4) DIH_MERGE_CASE(8, 1) DIH_MERGE_CASE(5, 4) DIH_MERGE_CASE(5, 1)
#undef DIH_MERGE_CASE
    return hip_ok(hipGetLastError(), error, capacity, "merge launch");
}

// ---------------------------------------------------------------------------- norm

// One block per token: normed[t] = r[t] * rsqrt(sum(r[t]^2)/H + eps) * w (the norm of
// graph_merge_norm / prefill_add_norm, gpu_graph.mm:40-61). Bound by latency (one block for
// the decode token): each of 1024 threads requests its N residual and N weight elements at
// once, one memory round trip, and keeps them (N = 2 up to 2048 columns, 8 up to 8192). The
// decode step with norm went 19.7 -> 17.1 us (8-bit) and 19.0 -> 16.7 us (5-bit) against 256
// threads reading eight elements each, twice.
template <int N>
__global__ __launch_bounds__(1024) void rmsnorm_kernel(const void *r, int r_f32, int H, const float *w,
                                                       float eps, void *out, int out_f32, const float *probs) {
    __shared__ float sq[16];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float p0 = probs ? probs[(size_t)t * 8] : 0.f;
    float v[N], wv[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int c = min(tid + 1024 * k, H - 1);
        v[k] = residual_load(r, r_f32, (size_t)t * H + c);
        wv[k] = w[c];
    }
    // the token's merge was skipped (non-finite router logits): its normed row stays as it was
    if (__builtin_isnan(p0)) return;
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < N; k++) ss += tid + 1024 * k < H ? v[k] * v[k] : 0.f;
    ss = wave_sum(ss);
    if (lane == 0) sq[wave] = ss;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int k = 0; k < 16; k++) total += sq[k];
    const float scale = rsqrtf(total / (float)H + eps);
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int c = tid + 1024 * k;
        if (c >= H) continue;
        const size_t at = (size_t)t * H + c;
        const float o = v[k] * scale * wv[k];
        if (out_f32) static_cast<float *>(out)[at] = o;
        else static_cast<uint16_t *>(out)[at] = f32_to_bf16(o);
    }
}

bool launch_rmsnorm(const void *r, int r_f32, int tokens, int hidden, const float *w, float eps,
                    void *out, int out_f32, const float *probs, hipStream_t s, char *error, int capacity) {
    if (hidden <= 2048)
        DIH_LAUNCH((rmsnorm_kernel<2>), dim3(tokens), dim3(1024), 0, s, r, r_f32, hidden, w, eps, out, out_f32, probs);
    else if (hidden <= 8192)
        DIH_LAUNCH((rmsnorm_kernel<8>), dim3(tokens), dim3(1024), 0, s, r, r_f32, hidden, w, eps, out, out_f32, probs);
    else {
        set_error(error, capacity, "Norm rows wider than 8192 are not supported");
        return false;
    }
    return hip_ok(hipGetLastError(), error, capacity, "norm launch");
}

// --------------------------------------------------------------------------- argmax

// Two levels, two launches (graph_argmax_blocks/final gpu_graph.mm:160-175): each block of
// the first reduces 1024 values to (max, lowest index), flagging non-finite values (one
// 16-byte load a thread, so the pass is one memory round trip over 243 blocks for the
// 248,320 logits; 4096 values a block, 61 blocks, took 5.6 us); one block of the second
// reduces the partials. Result 0xffffffff when any value is not finite. (One
// launch with a last-block ticket measured 10.7-12 us: the ticket's release fence and
// device-scope atomic from every block cost more than the second launch.)

// (max, lowest index) of a block's candidates; pairs whose index is 0xfffffffe mark a
// non-finite value, and 0xffffffff marks "no candidate". Thread 0 gets the result.
DIH_DEV void argmax_block(float best, uint32_t id, bool bad, float *wv, uint32_t *wi,
                          float &bm, uint32_t &bi) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool any_bad_w = __any(bad);
    const float m = wave_max(best);
    const uint32_t sel = wave_min_u32(best == m ? id : 0xffffffffu);
    if (lane == 0) { wv[wave] = m; wi[wave] = any_bad_w ? 0xfffffffeu : sel; }
    __syncthreads();
    bm = -INFINITY;
    bi = 0xffffffffu;
    if (tid == 0) {
        bool invalid = false;
        for (int w = 0; w < 4; w++) {
            if (wi[w] == 0xfffffffeu) { invalid = true; continue; }
            if (wi[w] != 0xffffffffu && (wv[w] > bm || (wv[w] == bm && wi[w] < bi))) { bm = wv[w]; bi = wi[w]; }
        }
        if (invalid) bi = 0xfffffffeu;
    }
}

__global__ __launch_bounds__(256) void argmax_blocks_kernel(const float *v, int n, float *pval,
                                                            uint32_t *pidx) {
    __shared__ float wv[4];
    __shared__ uint32_t wi[4];
    const int tid = threadIdx.x;
    const int base = blockIdx.x * kArgmaxPer;
    float x[4];
    // a coalesced 16-byte load a thread when the block is whole and aligned, else scalar
    if (base + kArgmaxPer <= n && (reinterpret_cast<uintptr_t>(v) & 15) == 0) {
        const float4 q = *reinterpret_cast<const float4 *>(v + base + 4 * tid);
        x[0] = q.x; x[1] = q.y; x[2] = q.z; x[3] = q.w;
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int at = base + 4 * tid + k;
            x[k] = at < n ? v[at] : -INFINITY;
        }
    }
    float best = -INFINITY;
    uint32_t id = 0xffffffffu;
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int at = base + 4 * tid + k;
        if (at < n) {
            if (!isfinite(x[k])) bad = true;
            else if (x[k] > best || (x[k] == best && (uint32_t)at < id)) { best = x[k]; id = (uint32_t)at; }
        }
    }
    float bm;
    uint32_t bi;
    argmax_block(best, id, bad, wv, wi, bm, bi);
    if (tid == 0) { pval[blockIdx.x] = bm; pidx[blockIdx.x] = bi; }
}

__global__ __launch_bounds__(256) void argmax_final_kernel(const float *pval, const uint32_t *pidx,
                                                           int nparts, uint32_t *next) {
    __shared__ float wv[4];
    __shared__ uint32_t wi[4];
    float best = -INFINITY;
    uint32_t id = 0xffffffffu;
    bool bad = false;
    for (int k = threadIdx.x; k < nparts; k += 256) {
        const uint32_t pi = pidx[k];
        const float pv = pval[k];
        if (pi == 0xfffffffeu) bad = true;
        else if (pi != 0xffffffffu && (pv > best || (pv == best && pi < id))) { best = pv; id = pi; }
    }
    float bm;
    uint32_t bi;
    argmax_block(best, id, bad, wv, wi, bm, bi);
    if (threadIdx.x == 0) *next = bi == 0xfffffffeu ? 0xffffffffu : bi;
}

bool launch_argmax(const float *values, int n, float *part_val, uint32_t *part_idx,
                   uint32_t *next, hipStream_t s, char *error, int capacity) {
    static_assert(kArgmaxPer == 4 * 256, "4 values a thread");
    const int blocks = (n + kArgmaxPer - 1) / kArgmaxPer;
    DIH_LAUNCH(argmax_blocks_kernel, dim3(blocks), dim3(256), 0, s, values, n, part_val, part_idx);
    if (!hip_ok(hipGetLastError(), error, capacity, "argmax launch")) return false;
    DIH_LAUNCH(argmax_final_kernel, dim3(1), dim3(256), 0, s, part_val, part_idx, blocks, next);
    return hip_ok(hipGetLastError(), error, capacity, "argmax launch");
}

}  // namespace dih
