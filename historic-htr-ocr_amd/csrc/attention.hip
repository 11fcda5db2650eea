// Attention for gfx950: the decode step's q/k post-processing and split-K GQA decode attention, and the prefill's
// per-head norm + RoPE + KV store and causal flash attention.
//
// Reference semantics: qkv_post.wgsl:31-83, attn_decode.wgsl:34-100 + attn_merge.wgsl:22-39 (text.rs:639-641),
// rms_norm.wgsl / rope_neox.wgsl / kv_store.wgsl / attention_causal.wgsl (text.rs:484-499). Head dim 128.
//
// KV cache layout (this library's): f16, head-major per layer, [n_kv][n_ctx][128] — one KV head's keys are
// contiguous, so a workgroup working on (kv head, key chunk) reads one contiguous range (256 bytes per key).
#include <type_traits>

#include "htr_internal.h"
#include "wave.h"

namespace {

constexpr int D = 128;

// one head's 128 values held as (lane, lane + 64) by a 64-lane wave: RMS norm with w, then RoPE NEOX with (c, s)
__device__ __forceinline__ void norm_rope(float &x0, float &x1, const float *w, const float *rope_row, int lane,
                                          float eps) {
    const float ss = wave_sum(x0 * x0 + x1 * x1, lane);
    const float scale = 1.0f / sqrtf(ss / (float)D + eps);
    const float y0 = (x0 * scale) * w[lane], y1 = (x1 * scale) * w[lane + 64];
    const float c = rope_row[2 * lane], s = rope_row[2 * lane + 1];
    x0 = y0 * c - y1 * s;
    x1 = y0 * s + y1 * c;
}

// qkv_post: block h < n_head: q head (norm, rope, in place); < n_head + n_kv: k head (norm, rope, f16 cache);
// else v head (f16 cache). One wave per head.
__global__ __launch_bounds__(64) void k_qkv_post(float *qkv, const float *qn, const float *kn, const float *rope,
                                                 int n_head, int n_kv, const int *pos_dev, int pos_arg, int n_ctx,
                                                 float eps, _Float16 *kc, _Float16 *vc) {
    const int h = blockIdx.x, lane = threadIdx.x;
    const int pos = pos_dev ? *pos_dev : pos_arg;
    if (pos < 0 || pos >= n_ctx) return;  // the cache has no such row (the host checks positions first)
    float *x = qkv + (size_t)h * D;
    float x0 = x[lane], x1 = x[lane + 64];
    if (h >= n_head + n_kv) {
        _Float16 *o = vc + ((size_t)(h - n_head - n_kv) * n_ctx + pos) * D;
        o[lane] = (_Float16)x0;
        o[lane + 64] = (_Float16)x1;
        return;
    }
    norm_rope(x0, x1, h < n_head ? qn : kn, rope + (size_t)pos * D, lane, eps);
    if (h < n_head) {
        x[lane] = x0;
        x[lane + 64] = x1;
    } else {
        _Float16 *o = kc + ((size_t)(h - n_head) * n_ctx + pos) * D;
        o[lane] = (_Float16)x0;
        o[lane + 64] = (_Float16)x1;
    }
}

// ---- split-K decode attention -----------------------------------------------------------------------------------------
//
// grid chunks · n_kv, 256 threads. A workgroup takes C = 16·NI keys of one KV head and both of its q heads (GQA
// group 2), so every K / V byte is read once. Thread t owns the 16-byte slice j = t & 15 (dims 8j … 8j+7) of the keys
// kk + 16·i (kk = t >> 4, i < NI): one wave-wide load reads 4 keys (1 KiB), and every K and V load of the chunk is
// issued before the first use.
//   1. scores s[h][key] = (q_h·scale)·k: 8 products per slice, summed over the 16 slices of a key by an
//      exchange-and-halve butterfly over all 2·NI (key, head) values at once → LDS (barrier)
//   2. every wave: m = max s, p = exp(s − m), l = Σ p for both heads → its own LDS copy of p (no barrier)
//   3. o[h][·] = Σ p·v from the V registers, summed over the 16 key positions (lane bits 5, 4, then the 4 waves in
//      LDS: barrier)
//   4. the chunk's (m, l, o) → partials [h][c][130]; the last workgroup of the KV head (atomic ticket) merges:
//      M = max m_c, w_c = e^(m_c − M), O = Σ o_c·w_c / Σ l_c·w_c — each wave one (head, 64 dims), its loads of all
//      chunks issued at once, no workgroup barrier. A single-chunk call writes O = o / l directly.
// Cross-lane moves are DPP / permlane VALU moves (wave.h). Cross-workgroup traffic is the partials' stores and loads
// plus the ticket atomic (one 128-byte line per KV head), with no release fence (one per workgroup would write back
// the L2 each time): with 8 KV heads, on a device whose launches put workgroup b on XCD b mod 8 and whose L2 shows a
// workgroup-scope store to the other workgroups of its XCD (both checked at open), every workgroup of a KV head shares
// one XCD, and the stores and the ticket stay in its L2 (workgroup scope); otherwise they go through the coherence
// point (agent scope, sc1).
constexpr int AW = 256;
constexpr int MAX_CHUNK_KEYS = 256;  // C ≤ 256 (NI ≤ 16)
constexpr int MAX_CHUNKS = 256;      // chunks per KV head: n_ctx ≤ 65536
constexpr int MERGE_FAST = 32;       // chunks merged by the branch-free path (each merging thread holds their o
                                     // partials in registers; n_ctx ≤ 8192 stays within it)
static_assert(MAX_CHUNKS % MERGE_FAST == 0, "the merge's weight groups fit s_w");
constexpr int CNT_STRIDE = 32;       // ticket counters 128 bytes apart: the KV heads' atomics do not share a line

// the KV cache stream: non-temporal loads (each key / value is read once a step)
typedef int gint4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int4 aload16(const void *p) {
    const gint4 v = __builtin_nontemporal_load((const __attribute__((address_space(1))) gint4 *)(uintptr_t)p);
    return make_int4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ void unpack8(const int4 w, float (&f)[8]) {
    const uint32_t u[4] = {(uint32_t)w.x, (uint32_t)w.y, (uint32_t)w.z, (uint32_t)w.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        _Float16 lo, hi;
        const uint16_t a = (uint16_t)(u[i] & 0xffff), b = (uint16_t)(u[i] >> 16);
        __builtin_memcpy(&lo, &a, 2);
        __builtin_memcpy(&hi, &b, 2);
        f[2 * i] = (float)lo;
        f[2 * i + 1] = (float)hi;
    }
}

__device__ __forceinline__ float ld_dev(const float *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// XL: every workgroup of a KV head runs on one XCD — the partials and the ticket are handed over in that XCD's L2
// (workgroup-scope stores and atomic, read by agent-scope loads that find the L2's lines); else through the coherence
// point (agent scope)
__device__ __forceinline__ void st_part(float *p, float v, bool xl) {
    if (xl) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int4 pack8(const float (&f)[8]) {
    uint32_t u[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const _Float16 lo = (_Float16)f[2 * i], hi = (_Float16)f[2 * i + 1];
        uint16_t a, b;
        __builtin_memcpy(&a, &lo, 2);
        __builtin_memcpy(&b, &hi, 2);
        u[i] = (uint32_t)a | ((uint32_t)b << 16);
    }
    return make_int4((int)u[0], (int)u[1], (int)u[2], (int)u[3]);
}

// qkv_post.wgsl's per-head RMS norm and RoPE NEOX (pairs (i, i + 64)) at one position, for the 8 dims 8j … 8j + 7
// of one head's raw row: the 16 lanes j = 0 … 15 of a lane row hold the head together (Σx² over them); the lane also
// holds the partner dims (slice j ^ 8). Loads first (post_load), the arithmetic later (post_apply), so that the
// loads go out before the K / V loads and the arithmetic waits for these alone.
struct PostIn {
    float4 a[2], b[2], wa[2], wb[2];
};
__device__ __forceinline__ void post_load(PostIn &p, const float *x, const float *w, int j) {
    const int jp = j ^ 8;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        p.a[h] = *reinterpret_cast<const float4 *>(x + 8 * j + 4 * h);
        p.b[h] = *reinterpret_cast<const float4 *>(x + 8 * jp + 4 * h);
        p.wa[h] = *reinterpret_cast<const float4 *>(w + 8 * j + 4 * h);
        p.wb[h] = *reinterpret_cast<const float4 *>(w + 8 * jp + 4 * h);
    }
}
__device__ __forceinline__ void unpack4x2(const float4 (&v)[2], float (&f)[8]) {
    f[0] = v[0].x, f[1] = v[0].y, f[2] = v[0].z, f[3] = v[0].w, f[4] = v[1].x, f[5] = v[1].y, f[6] = v[1].z, f[7] = v[1].w;
}
// cs: the (c, s) pairs of rope indices 8(j % 8) … + 7
__device__ __forceinline__ void post_apply(const PostIn &p, const float (&cs)[16], int j, int lane, float eps,
                                           float (&out)[8]) {
    float a[8], b[8], wa[8], wb[8];
    unpack4x2(p.a, a);
    unpack4x2(p.b, b);
    unpack4x2(p.wa, wa);
    unpack4x2(p.wb, wb);
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) ss = fmaf(a[e], a[e], ss);
    ss = group_sum<8>(ss, lane);
    const float scale = 1.0f / sqrtf(ss / (float)D + eps);
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float ya = (a[e] * scale) * wa[e], yb = (b[e] * scale) * wb[e];
        const float c = cs[2 * e], s = cs[2 * e + 1];
        out[e] = j < 8 ? ya * c - yb * s : yb * s + ya * c;
    }
}

// prefill rows: k heads (norm, RoPE → f16 cache rows pos0 + t) and v heads (→ f16 cache), 16 lanes × 8 dims a head row
// (the q heads are normed and turned where the causal attention reads them)
__global__ __launch_bounds__(256) void k_kv_rows(const float *k, const float *v, const float *kn, const float *rope,
                                                 int n_rows, int n_kv, int pos0, int n_ctx, float eps, _Float16 *kc,
                                                 _Float16 *vc) {
    const int lane = threadIdx.x & 63, j = lane & 15, id = blockIdx.x * 16 + (threadIdx.x >> 4);
    const int row = min(id, n_rows - 1), t = row / (2 * n_kv), h = row % (2 * n_kv), pos = pos0 + t;
    const bool isv = h >= n_kv;
    const int kvh = isv ? h - n_kv : h;
    PostIn in;
    post_load(in, (isv ? v : k) + ((size_t)t * n_kv + kvh) * D, kn, j);
    float cs[16], y[8], raw[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float4 r = *reinterpret_cast<const float4 *>(rope + (size_t)pos * D + 16 * (j & 7) + 4 * i);
        cs[4 * i] = r.x, cs[4 * i + 1] = r.y, cs[4 * i + 2] = r.z, cs[4 * i + 3] = r.w;
    }
    post_apply(in, cs, j, lane, eps, y);
    unpack4x2(in.a, raw);
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = isv ? raw[e] : y[e];
    if (id < n_rows)
        *reinterpret_cast<int4 *>((isv ? vc : kc) + ((size_t)kvh * n_ctx + pos) * D + 8 * j) = pack8(y);
}

// FUSED: q is the raw [q | k | v] row of the qkv matvec and the kernel does qkv_post's work itself: each workgroup
// norms and ropes its two q heads; the new key / value (position n_keys − 1) are made from the raw row, rounded to
// f16 as the cache holds them, used in place of the cache row by the workgroup whose chunk holds them, and stored
// into the cache by that workgroup (no other workgroup reads that row)
template <int NI, bool FUSED>
__global__ __launch_bounds__(AW) void k_attn_decode(const float *q, const _Float16 *kc, const _Float16 *vc, int n_kv,
                                                    int n_ctx, const int *pos_dev, int n_keys_arg, int max_chunk,
                                                    float scale, float post, float *part, uint32_t *counters,
                                                    float *out, AttnFuse fz, int xl) {
    constexpr int C = 16 * NI;
    constexpr int N = 2 * NI;              // (key, head) values per thread
    constexpr int KL = C >= 64 ? C / 64 : 1;  // keys per lane in the softmax
    __shared__ float s_sc[2][C];
    __shared__ float s_pw[4][2][C];  // each wave's copy of p
    __shared__ float s_lw[2];
    __shared__ float s_o[4][2][D];
    __shared__ float s_w[4][MAX_CHUNKS];
    __shared__ int s_last;
    // a 1D grid of the KV heads' chunks; with 8 KV heads workgroup b runs on XCD b mod 8 (a launch spreads its
    // workgroups round-robin), so a KV head's chunks and its merge's loads of their partials share one XCD's L2: at
    // 512 keys 5.52 → 5.25 µs a graph node (the same at 2048 and 8192 keys)
    const int nb = gridDim.x / n_kv;
    const int c = n_kv == 8 ? (int)blockIdx.x >> 3 : (int)blockIdx.x % nb;
    const int kvh = n_kv == 8 ? (int)blockIdx.x & 7 : (int)blockIdx.x / nb;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = tid & 15, kk = tid >> 4;
    // keys beyond the cache are never read (the host checks positions first; a bad one yields no output)
    const int n_keys = min(pos_dev ? *pos_dev + 1 : n_keys_arg, n_ctx);
    if (FUSED && pos_dev && *pos_dev >= n_ctx) return;  // the cache has no such row (the host checks positions first)
    const int n_chunk = (n_keys + C - 1) / C;
    if (c >= n_chunk || n_chunk > max_chunk) return;  // uniform per workgroup
    const int k0 = c * C;
    const int h0 = 2 * kvh;

    // FUSED: the raw q / k / v slices, norm weights and rope row go out first (they come from L2, the keys from HBM)
    const int pos = n_keys - 1;
    PostIn pin[3];
    float4 vraw[2], rope4[4];
    if constexpr (FUSED) {
        post_load(pin[0], q + (size_t)h0 * D, fz.qn, j);
        post_load(pin[1], q + (size_t)(h0 + 1) * D, fz.qn, j);
        post_load(pin[2], q + (size_t)(fz.n_head + kvh) * D, fz.kn, j);
        const float *vr0 = q + (size_t)(fz.n_head + n_kv + kvh) * D + 8 * j;
        vraw[0] = *reinterpret_cast<const float4 *>(vr0);
        vraw[1] = *reinterpret_cast<const float4 *>(vr0 + 4);
        const float *rr = fz.rope + (size_t)pos * D + 16 * (j & 7);
#pragma unroll
        for (int i = 0; i < 4; i++) rope4[i] = *reinterpret_cast<const float4 *>(rr + 4 * i);
        __builtin_amdgcn_sched_barrier(0);
    }

    // 0. every K and V load of the chunk (keys past n_keys read the last key and are masked)
    const _Float16 *kb = kc + (size_t)kvh * n_ctx * D, *vb = vc + (size_t)kvh * n_ctx * D;
    int4 kr[NI], vr[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int key = min(k0 + kk + 16 * i, n_keys - 1);
        kr[i] = aload16(kb + (size_t)key * D + 8 * j);
    }
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int key = min(k0 + kk + 16 * i, n_keys - 1);
        vr[i] = aload16(vb + (size_t)key * D + 8 * j);
    }
    if constexpr (FUSED) __builtin_amdgcn_sched_barrier(0);  // the K / V loads are out before the arithmetic
    float qa[8], qb[8];
    int4 knew = make_int4(0, 0, 0, 0), vnew = make_int4(0, 0, 0, 0);
    if constexpr (FUSED) {
        float cs[16];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            cs[4 * i] = rope4[i].x, cs[4 * i + 1] = rope4[i].y, cs[4 * i + 2] = rope4[i].z, cs[4 * i + 3] = rope4[i].w;
        }
        float ta[8], tb[8], kn8[8], v8[8];
        post_apply(pin[0], cs, j, lane, fz.eps, ta);
        post_apply(pin[1], cs, j, lane, fz.eps, tb);
        post_apply(pin[2], cs, j, lane, fz.eps, kn8);
        unpack4x2(vraw, v8);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            qa[e] = ta[e] * scale;
            qb[e] = tb[e] * scale;
        }
        knew = pack8(kn8);
        vnew = pack8(v8);
        if (c == n_chunk - 1 && kk == 0) {
            *reinterpret_cast<int4 *>(fz.kc + ((size_t)kvh * n_ctx + pos) * D + 8 * j) = knew;
            *reinterpret_cast<int4 *>(fz.vc + ((size_t)kvh * n_ctx + pos) * D + 8 * j) = vnew;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            qa[e] = q[h0 * D + 8 * j + e] * scale;
            qb[e] = q[(h0 + 1) * D + 8 * j + e] * scale;
        }
    }

    // 1. scores. FUSED: every key at or past pos takes the new row (keys past pos were clamped onto row pos, whose
    // cache contents are stale — a rewound session's old row — and being rewritten by this workgroup): masked keys
    // then multiply finite values by 0 below, whatever the cache held
    float v[N];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        float kf[8];
        unpack8(FUSED && k0 + kk + 16 * i >= pos ? knew : kr[i], kf);
        float da = 0.0f, db = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            da = fmaf(qa[e], kf[e], da);
            db = fmaf(qb[e], kf[e], db);
        }
        v[2 * i] = da;
        v[2 * i + 1] = db;
    }
    if constexpr (N >= 16) {
        halve<N, 8, 4>(v, lane);  // lane j keeps values (N/16)·j + r
#pragma unroll
        for (int r = 0; r < N / 16; r++) {
            const int idx = (N / 16) * j + r, i = idx >> 1, h = idx & 1;
            const int key = kk + 16 * i;
            s_sc[h][key] = k0 + key < n_keys ? v[r] * post : -INFINITY;
        }
    } else {
        constexpr int S = N == 2 ? 1 : N == 4 ? 2 : 3;  // log2 N
        halve<N, 8, S>(v, lane);                         // lane j keeps value j >> (4 − S)
        const float t = group_sum<(8 >> S)>(v[0], lane);
        if ((j & ((16 >> S) - 1)) == 0) {
            const int idx = j >> (4 - S), i = idx >> 1, h = idx & 1;
            const int key = kk + 16 * i;
            s_sc[h][key] = k0 + key < n_keys ? t * post : -INFINITY;
        }
    }
    __syncthreads();

    // 2. softmax statistics, every wave for both heads into its own copy of p
    float l_h[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        float sv[KL], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < KL; i++) {
            const int key = lane + 64 * i;
            sv[i] = key < C ? s_sc[h][key] : -INFINITY;
            mx = fmaxf(mx, sv[i]);
        }
        mx = wave_max(mx, lane);
        float l = 0.0f;
#pragma unroll
        for (int i = 0; i < KL; i++) {
            const int key = lane + 64 * i;
            const float p = expf(sv[i] - mx);  // masked keys: exp(−inf) = 0
            if (key < C) s_pw[wave][h][key] = p;
            l += p;
        }
        l_h[h] = wave_sum(l, lane);
        if (h == 0 && wave == 0 && lane == 0) s_lw[0] = mx;
        if (h == 1 && wave == 0 && lane == 0) s_lw[1] = mx;
    }
    __builtin_amdgcn_wave_barrier();

    // 3. values
    float o[16];  // [h][e]
#pragma unroll
    for (int e = 0; e < 16; e++) o[e] = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; i++) {
        float vf[8];
        unpack8(FUSED && k0 + kk + 16 * i >= pos ? vnew : vr[i], vf);
        const float pa = s_pw[wave][0][kk + 16 * i], pb = s_pw[wave][1][kk + 16 * i];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            o[e] = fmaf(pa, vf[e], o[e]);
            o[8 + e] = fmaf(pb, vf[e], o[8 + e]);
        }
    }
    halve<16, 32, 2>(o, lane);  // over lane bits 5, 4: lane keeps values 8·b5 + 4·b4 + r
    {
        const int base = 8 * ((lane >> 5) & 1) + 4 * ((lane >> 4) & 1);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int idx = base + r, h = idx >> 3, e = idx & 7;
            s_o[wave][h][8 * j + e] = o[r];
        }
    }
    __syncthreads();
    const int hh = tid >> 7, d = tid & 127;  // 256 threads = 2 heads × 128 dims
    const float oc = (s_o[0][hh][d] + s_o[1][hh][d]) + (s_o[2][hh][d] + s_o[3][hh][d]);
    const float lc = l_h[hh];  // every wave holds both heads' sums
    const int h = h0 + hh;
    if (n_chunk == 1) {
        out[h * D + d] = oc / lc;
        return;
    }

    // 4. partials, then the last workgroup of the KV head merges
    float *pc = part + ((size_t)h * max_chunk + c) * (D + 2);  // [h][c][m, l, o[128]]
    st_part(pc + 2 + d, oc, xl);
    if (d == 0) st_part(pc, s_lw[hh], xl);
    if (d == 1) st_part(pc + 1, lc, xl);
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's stores are performed
    __syncthreads();
    uint32_t *ticket = counters + (size_t)kvh * CNT_STRIDE;
    if (tid == 0)
        s_last = (xl ? __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)
                     : __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ==
                 (uint32_t)(n_chunk - 1);
    __syncthreads();
    if (!s_last) return;
    // the merge: wave w → head h0 + (w >> 1), dims (w & 1)·64 + lane
    const int mh = h0 + (wave >> 1), md = (wave & 1) * 64 + lane;
    const float *ph = part + (size_t)mh * max_chunk * (D + 2);
    float O = 0.0f, L;
    if (n_chunk <= MERGE_FAST) {
        // every load at once, branch-free (chunk indexes clamped; what lies past n_chunk gets weight 0): lane ℓ's
        // chunk statistics (m, l of chunk ℓ) and this thread's dim of every chunk's o; the weights are worked out
        // while the o loads are in flight
        const int cl = min(lane, n_chunk - 1);
        float mv = ld_dev(ph + (size_t)cl * (D + 2)), lv = ld_dev(ph + (size_t)cl * (D + 2) + 1);
        float ov[MERGE_FAST];
#pragma unroll
        for (int i = 0; i < MERGE_FAST; i++) ov[i] = ld_dev(ph + (size_t)min(i, n_chunk - 1) * (D + 2) + 2 + md);
        if (lane >= n_chunk) mv = -INFINITY, lv = 0.0f;
        const float mx = wave_max(mv, lane);
        const float w = expf(mv - mx);  // lanes past n_chunk: e^(−inf) = 0
        L = wave_sum(lv * w, lane);
        // the weights straight from the lanes that hold them (a scalar operand of the fma)
#pragma unroll
        for (int i = 0; i < MERGE_FAST; i++)
            O = fmaf(ov[i], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), i)), O);
    } else {
        // long contexts: the weights through LDS (zero past n_chunk up to a whole group), the o partials in groups of
        // MERGE_FAST chunks, each group's loads at once
        float mx = -INFINITY;
        for (int cc = lane; cc < n_chunk; cc += 64) mx = fmaxf(mx, ld_dev(ph + (size_t)cc * (D + 2)));
        mx = wave_max(mx, lane);
        const int n_up = (n_chunk + MERGE_FAST - 1) / MERGE_FAST * MERGE_FAST;
        float l = 0.0f;
        for (int cc = lane; cc < n_up; cc += 64) {
            const int cl = min(cc, n_chunk - 1);
            const float mc = ld_dev(ph + (size_t)cl * (D + 2)), lc = ld_dev(ph + (size_t)cl * (D + 2) + 1);
            const float w = cc < n_chunk ? expf(mc - mx) : 0.0f;
            s_w[wave][cc] = w;
            l = fmaf(lc, w, l);
        }
        L = wave_sum(l, lane);
        __builtin_amdgcn_wave_barrier();
        for (int c0 = 0; c0 < n_chunk; c0 += MERGE_FAST) {
            float ov[MERGE_FAST];
#pragma unroll
            for (int i = 0; i < MERGE_FAST; i++)
                ov[i] = ld_dev(ph + (size_t)min(c0 + i, n_chunk - 1) * (D + 2) + 2 + md);
#pragma unroll
            for (int i = 0; i < MERGE_FAST; i++) O = fmaf(ov[i], s_w[wave][c0 + i], O);
        }
    }
    out[mh * D + md] = O / L;
    if (tid == 0) {  // for the next launch
        if (xl) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---- prefill causal attention ----------------------------------------------------------------------------------------
//
// attention_causal.wgsl's arithmetic (text.rs:484-499; the same on every compute path): q·scale in f32, scores as
// f32 dot products with the f16 keys, an online softmax in f32 over the keys each query sees (0 … its position),
// out = acc · (1 / l). Here on the f16 matrix cores (v_mfma_f32_32x32x16_f16) with f32-grade operands: q·scale =
// qh + ql and 2^3·p = ph + pl, each half rounded to f16 (K and V are f16 already), so every product of what is held is
// exact and every sum f32; the 2^3 (exact) drops out with l, which carries it too. The p pair holds 22 bits of p down to
// 2^-5 of a query's largest, and is within 2^-28 of that largest below (pl is subnormal there). The q pair holds 22 bits,
// except that qh is rounded from the f32 product and ql is the rest beside the product rounded to f16 in one step (that
// is how the compiler takes x·scale where both are wanted): where the f32 product is a tie the two f16 values differ, and
// the pair is an f16 ulp off (5e-5 of random elements, none with a power of two as scale; the outputs' error against 64
// bits is 4.8e-6 for it, 3e-7 without). Holding the product to one value would cost nothing, but moves single outputs by
// up to 1e-3 of their size.
//
//   work     a workgroup takes 32 queries of both q heads of a KV head: 4 waves = 2 heads × the even / odd key blocks,
//            the two parts merged through LDS at the end. A stage is 2 blocks of 32 keys (32 KB), K and V each
//            double-buffered, K a stage ahead of V: the score MFMAs of the next stage run under the softmax of this one.
//            Two workgroups a CU; the first half of the grid takes the query blocks longest first, the second half
//            shortest first, so the two that a CU holds have complementary lengths;
//   blocks   K [32 keys][128 dims] with row r's 16-byte chunk c at 16r + (c ^ r%16), then V [32 keys][128 dims] with
//            chunk c at 16r + (c ^ 2(r%8)), straight from the cache rows by direct-to-LDS loads (a wave's instruction
//            is 4 whole rows): 16 lanes' fragment reads of K (16 rows, one chunk) and of V (4 rows, two chunks) fall
//            on different bank groups. Keys past the last read the last key and are masked;
//   scores   Sᵀ (32 keys × 32 queries) = K·(qh + ql)ᵀ: lane ℓ = 32h + c holds query c's scores of keys
//            8(i / 4) + 4h + i % 4 (i < 16); the max over a query's keys is one swap across lane bit 5;
//   softmax  p = 2^(s·log2 e + nm), nm = 3 − log2 e · (the max when it was last moved): one fma and one v_exp_f32 a
//            score, and nm is the only state, so its rounding cancels between p, l and O. nm moves (and O and l are
//            rescaled) only when some p would pass 2^8, so most blocks skip the 64-register rescale. An exponent is
//            rounded at its own size, which is why the shift is small (10, and 15 for the top: 2.3e-7 against 64 bits
//            for 64 queries, 2.9e-7 for 1925; 1.9e-7 and 2.4e-7 so, as e^(s − max) gave), and l is summed a block at a
//            time, for the same reason. nm holds scores of 2^26 to within 4, so p keeps to f16's range; a wave with a
//            query whose scores could be larger (Σ |q·scale| of a half row from 512 on, against f16 keys of 65504 at
//            most) keeps the max itself and takes s − max first;
//   values   Oᵀ (128 dims × 32 queries) += Vᵀ·(ph + pl)ᵀ: the Vᵀ operand by ds_read_b64_tr_b16 (16 lanes read 4 key
//            rows × 16 dims and each gets one dim's 4 keys), the P operand straight from the lane's score registers.
//
// Bound: the score MFMAs with the softmax between them (a 32x32x16 MFMA takes 17 ns a SIMD here; with its 5 VALU
// instructions and exponential about 23), then the stage's loads (20 %: a timing copy without them ran 34 µs for 40) and
// a stage's barrier. Measured against 16 queries a workgroup on 16x16x32 MFMAs, O rescaled at every block and the keys
// copied into blocks by a launch before it (n_q from position 0, 16 / 8 heads, median µs of a kernel trace): 1925 queries
// 75.2 + 8.0 → 42.9 (39.6 a call among others: 383 TFLOP/s of q·k and p·v); with the q heads' norm and RoPE, which a third
// launch did (5.2 and 9.4 with the K / V rows, now 4.8 and 5.1): 333 11.4 + 4.9 → 13.1, 1023 25.9 + 5.5 → 24.4.
// Eight waves and four key parts, one workgroup a CU: 20 % slower at 1925 queries (its merge is twice the LDS traffic and
// its waves run in step); only 32 queries on 2000 earlier keys gained, 31.4 → 29.7.
constexpr int CQ = 32, CK = 32, CB_CHUNKS = 1024;  // queries a workgroup, keys a block, 16-byte chunks a key block
constexpr int CKS = 2, CW = 64 * 2 * CKS;          // key parts; threads
constexpr float P_SHIFT = 3.0f, P_TOP = 8.0f;      // log2 of the largest p when nm moves, and before it must
constexpr float LOG2E = 1.4426950408889634f;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef __fp16 fp16x4 __attribute__((ext_vector_type(4)));

// p − (float)h for the low (0) or high (1) half of h: one mixed-precision fma
template <int HI> __device__ __forceinline__ float minus_half(float p, uint32_t h) {
    float r;
    if constexpr (HI) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(p));
    else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(p));
    return r;
}

// OT: the output's type — f32, or f16 (rounded to nearest even: the value the f16 path's o-projection tile holds).
// POST: q holds the raw rows of the q projection; the head's RMS norm (weights qn) and RoPE are applied as they are read
template <typename OT, bool POST>
__global__ __launch_bounds__(CW) void k_attn_causal(const float *q, const _Float16 *kc, const _Float16 *vc, int n_q,
                                                    int pos0, int n_head, int n_kv, int n_ctx, float scale,
                                                    const float *qn, const float *rope, float eps, OT *out) {
    __shared__ __attribute__((aligned(16))) int4 s_kv[2][CKS][CB_CHUNKS];  // [buffer][part][chunk]
    __shared__ float s_ml[2 * CKS][2][CQ];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hf = lane >> 5, c = lane & 31;
    const int n_qb = (n_q + CQ - 1) / CQ;
    const int kvh = blockIdx.x % n_kv, rank = blockIdx.x / n_kv;
    const int half = (n_qb + 1) / 2, qb = rank < half ? n_qb - 1 - rank : rank - half;
    const int hh = wave & 1, kp = wave >> 1, h = 2 * kvh + hh;
    const int q_first = CQ * qb, q_last = min(q_first + CQ - 1, n_q - 1);
    const int qi = min(q_first + c, n_q - 1), qpos = pos0 + qi;
    const int n_keys = pos0 + q_last + 1;                  // keys the last query of the block sees
    const int nkb = (n_keys + CK - 1) / CK, n_stage = (nkb + CKS - 1) / CKS;
    const int n_full = (pos0 + q_first + 1) / CK / CKS;     // stages whose keys every query sees
    const _Float16 *kh = kc + (size_t)kvh * n_ctx * D, *vh = vc + (size_t)kvh * n_ctx * D;

    // a stage's K or V → buffer st % 2: 4 direct loads a wave, each of the 4 waves 4 rows of 16 (keys past the last: the last)
    const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int4 *)&s_kv[0][0][64 * wave];
    const int lrow = 4 * wave + (lane >> 4), lc = lane & 15;
    const uint32_t koff = 16 * (lc ^ (lrow & 15)), voff = 16 * (lc ^ (2 * (lrow & 7)));  // the same for row lrow + 16
    auto issue = [&](int st, bool isv) {
        const int s0 = CK * CKS * st;  // the stage's first key
        const char *base = (const char *)(isv ? vh : kh) + (size_t)s0 * (2 * D);
        const uint32_t off = isv ? voff : koff, last = 2 * D * min(n_keys - 1 - s0, CK * CKS - 1) + off;  // the last key's
#pragma unroll
        for (int i = 0; i < 2 * CKS; i++)  // rows 16i + lrow of the stage: half a block
            lds_load16(base, min(2 * D * (16 * i + lrow) + off, last),
                       lds + (uint32_t)sizeof(int4) * (((st & 1) * CKS + i / 2) * CB_CHUNKS + (isv ? 512 : 0) + 256 * (i % 2)));
    };
    issue(0, false);
    issue(0, true);
    if (n_stage > 1) issue(1, false);

    // q·scale as f16 pairs: B operand of step ks = dims 16ks + 8hf … + 7 of query c
    half8 qh[8], ql[8];
    bool far;
    {
        const float *qrow = q + ((size_t)qi * n_head + h) * D + 8 * hf;
        float x[8][8];
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            const float4 a0 = *reinterpret_cast<const float4 *>(qrow + 16 * ks);
            const float4 a1 = *reinterpret_cast<const float4 *>(qrow + 16 * ks + 4);
            x[ks][0] = a0.x, x[ks][1] = a0.y, x[ks][2] = a0.z, x[ks][3] = a0.w;
            x[ks][4] = a1.x, x[ks][5] = a1.y, x[ks][6] = a1.z, x[ks][7] = a1.w;
        }
        if constexpr (POST) {
            float ss = 0.0f;
#pragma unroll
            for (int ks = 0; ks < 8; ks++)
#pragma unroll
                for (int e = 0; e < 8; e++) ss = fmaf(x[ks][e], x[ks][e], ss);
            const float inv = 1.0f / sqrtf(pair_sum<32>(ss) / (float)D + eps);
            // the pairs (i, i + 64) are steps ks and ks + 4 of the same lane
            const float *cs = rope + (size_t)qpos * D + 16 * hf;
#pragma unroll
            for (int ks = 0; ks < 4; ks++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float2 t = *reinterpret_cast<const float2 *>(cs + 32 * ks + 2 * e);
                    const float y0 = (x[ks][e] * inv) * qn[16 * ks + 8 * hf + e];
                    const float y1 = (x[ks + 4][e] * inv) * qn[64 + 16 * ks + 8 * hf + e];
                    x[ks][e] = y0 * t.x - y1 * t.y;
                    x[ks + 4][e] = y0 * t.y + y1 * t.x;
                }
        }
        float size = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 8; ks++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float qs = x[ks][e] * scale;
                const _Float16 hi = (_Float16)qs;
                qh[ks][e] = hi;
                ql[ks][e] = (_Float16)(qs - (float)hi);
                size += fabsf(qs);
            }
        far = __builtin_amdgcn_ballot_w64(!(size < 512.0f)) != 0;
    }
    // the lane's fragment slots in a block: K step ks (key c, dims 16ks + 8hf …); V tile t (16-lane group: dims
    // 32t + 16(ℓ/16 % 2) …, keys 4hf + (ℓ%16)/4 of each 8-key group)
    int ka[8], va[4];
#pragma unroll
    for (int ks = 0; ks < 8; ks++) ka[ks] = 16 * c + ((2 * ks + hf) ^ (c & 15));
    const int vrow = 4 * hf + ((lane & 15) >> 2);
#pragma unroll
    for (int t = 0; t < 4; t++)
        va[t] = 16 * (512 + 16 * vrow + ((4 * t + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ (2 * vrow))) + 8 * (lane & 1);

    f32x16 o[4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[t][i] = 0.0f;
    float nm = 3.0e38f, l = 0.0f;  // far: nm is −max

    auto scores = [&](f32x16 &s, int st) {
        const int4 *blk = s_kv[st & 1][kp];
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            const half8 a = *reinterpret_cast<const half8 *>(blk + ka[ks]);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qh[ks], ks ? s : f32x16{}, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ql[ks], s, 0, 0, 0);
        }
    };
    // stage st in buffer b: its scores are in s; the next stage's are computed into sn under the softmax's VALU work
    auto step = [&](int st, int b, f32x16 &s, f32x16 &sn, auto mask, auto is_far) {
        constexpr bool MASK = decltype(mask)::value, FAR = decltype(is_far)::value;
        // this wave's loads of K stage st + 1 and V stage st are in, its reads of K stage st and V stage st − 1 have
        // their values (their MFMAs may stand behind the barrier); behind it everyone's, and the two buffers are free
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (st + 2 < n_stage) issue(st + 2, false);
        if (st + 1 < n_stage) issue(st + 1, true);
        const int k0 = CK * (CKS * st + kp);
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if (MASK && k0 + 8 * (i >> 2) + 4 * hf + (i & 3) > qpos) s[i] = -INFINITY;  // keys after the query
            mx = fmaxf(mx, s[i]);
        }
        mx = pair_max<32>(mx);
        if (__builtin_amdgcn_ballot_w64(FAR ? mx + nm > 0.0f : fmaf(mx, LOG2E, nm) > P_TOP)) {
            const float to = fminf(nm, FAR ? -mx : fmaf(-mx, LOG2E, P_SHIFT));
            const float corr = __builtin_amdgcn_exp2f(FAR ? (to - nm) * LOG2E : to - nm);
            nm = to;
            l *= corr;
#pragma unroll
            for (int t = 0; t < 4; t++) o[t] *= corr;
        }
        if (FAR) {
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] += nm;
        }
        const float add = FAR ? P_SHIFT : nm;
        // the order pinned: behind each score MFMA of the next stage its share of this stage's softmax (left to itself
        // the compiler issues the MFMAs back to back and the softmax behind them)
        // (past the last stage: scores of what the buffer holds, not used)
        const int4 *kb = s_kv[b ^ 1][kp];
        const auto *vb = (const __attribute__((address_space(3))) char *)s_kv[b][kp];
        // V tile t, step ss: slots 8hf … + 7 are keys 16ss + 4hf … + 3, then 16ss + 8 + 4hf … + 3 — the scores 8ss …
        // that the lane holds
        auto vread = [&](int t, int ss) {
            const auto *p = vb + va[t] + 256 * 16 * ss;
            const fp16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) fp16x4 *)p);
            const fp16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) fp16x4 *)(p + 256 * 8));
            half8 v;
            __builtin_memcpy(&v, &lo, 8);
            __builtin_memcpy((char *)&v + 8, &hi, 8);
            return v;
        };
        uint32_t ph[8], pl[8];
        float ls;
        half8 a[8], v[4];
#pragma unroll
        for (int ks = 0; ks < 3; ks++) a[ks] = *reinterpret_cast<const half8 *>(kb + ka[ks]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            sn = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks], qh[ks], ks ? sn : f32x16{}, 0, 0, 0);
            if (ks + 3 < 8) a[ks + 3] = *reinterpret_cast<const half8 *>(kb + ka[ks + 3]);
            else v[ks - 5] = vread(ks - 5, 0);
            const float2_t p = {__builtin_amdgcn_exp2f(fmaf(s[2 * ks], LOG2E, add)),
                                __builtin_amdgcn_exp2f(fmaf(s[2 * ks + 1], LOG2E, add))};  // masked: 2^(−inf) = 0
            const half2_t hi = __builtin_convertvector(p, half2_t);
            __builtin_memcpy(&ph[ks], &hi, 4);
            asm volatile("" : "+v"(ph[ks]));  // holds the conversion here
            __builtin_amdgcn_sched_barrier(0);
            sn = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks], ql[ks], sn, 0, 0, 0);
            ls = ks ? ls + p[0] : p[0];
            ls += p[1];
            const half2_t lo = __builtin_convertvector((float2_t{minus_half<0>(p[0], ph[ks]), minus_half<1>(p[1], ph[ks])}), half2_t);
            __builtin_memcpy(&pl[ks], &lo, 4);
            asm volatile("" : "+v"(pl[ks]));
            __builtin_amdgcn_sched_barrier(0);
        }
        v[3] = vread(3, 0);
        l += ls;
#pragma unroll
        for (int ss = 0; ss < 2; ss++) {
            half8 h8, l8;
            __builtin_memcpy(&h8, &ph[4 * ss], 16);
            __builtin_memcpy(&l8, &pl[4 * ss], 16);
            half8 vn[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[t], h8, o[t], 0, 0, 0);
                if (ss == 0) vn[t] = vread(t, 1);
            }
#pragma unroll
            for (int t = 0; t < 4; t++) {
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[t], l8, o[t], 0, 0, 0);
                if (ss == 0) v[t] = vn[t];
            }
        }
    };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // K and V stage 0, K stage 1
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    f32x16 s0, s1;
    scores(s0, 0);
    int st = 0;
    // (the two kinds of wave pass the same barriers, one a stage)
    if (far) {
        for (; st < n_stage; st++) {
            step(st, st & 1, s0, s1, std::true_type{}, std::true_type{});
            s0 = s1;
        }
    }
    for (; st + 1 < n_full; st += 2) {
        step(st, 0, s0, s1, std::false_type{}, std::false_type{});
        step(st + 1, 1, s1, s0, std::false_type{}, std::false_type{});
    }
    for (; st < n_stage; st++) {
        step(st, st & 1, s0, s1, std::true_type{}, std::false_type{});
        s0 = s1;
    }
    l = pair_sum<32>(l);
    // merge the key parts of each head through LDS (the stage buffers, once every wave is done with them): every wave
    // leaves its sums as its lanes hold them, then wave (head, part) finishes its share of the
    // head's dims
    __syncthreads();
    float *s_o = reinterpret_cast<float *>(&s_kv[0][0][0]);  // [wave][tile][register][lane]
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) s_o[((wave * 4 + t) * 16 + i) * 64 + lane] = o[t][i];
    if (hf == 0) s_ml[wave][0][c] = nm, s_ml[wave][1][c] = l;
    __syncthreads();
    if (q_first + c >= n_q) return;
    float w[CKS], lsum = 0.0f, top = 3.0e38f;
#pragma unroll
    for (int p = 0; p < CKS; p++) top = fminf(top, s_ml[2 * p + hh][0][c]);
#pragma unroll
    for (int p = 0; p < CKS; p++) {  // (both parts of a head hold the same queries: far or not alike)
        w[p] = __builtin_amdgcn_exp2f((top - s_ml[2 * p + hh][0][c]) * (far ? LOG2E : 1.0f));  // a part without keys: 0
        lsum = fmaf(s_ml[2 * p + hh][1][c], w[p], lsum);
    }
    const float inv = 1.0f / lsum;
    OT *orow = out + ((size_t)(q_first + c) * n_head + h) * D + 4 * hf;
#pragma unroll
    for (int u = 0; u < 16 / CKS; u++) {
        const int t = kp * (4 / CKS) + (u >> 2), r = u & 3;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] = 0.0f;
#pragma unroll
            for (int p = 0; p < CKS; p++) v[e] = fmaf(s_o[(((2 * p + hh) * 4 + t) * 16 + 4 * r + e) * 64 + lane], w[p], v[e]);
            v[e] *= inv;
        }
        if constexpr (sizeof(OT) == 4) {
            *reinterpret_cast<float4 *>(orow + 32 * t + 8 * r) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
            *reinterpret_cast<half4 *>(orow + 32 * t + 8 * r) =
                half4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
        }
    }
}

// caches that are not 16-byte aligned, copied so that the direct loads can read them: [K, V][n_kv][n_keys][128]
__global__ __launch_bounds__(256) void k_kv_align(const _Float16 *kc, const _Float16 *vc, int n_kv, int n_ctx,
                                                  int n_keys, _Float16 *out) {
    const size_t half = (size_t)n_kv * n_keys * D;
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < 2 * half; i += (size_t)gridDim.x * 256) {
        const size_t j = i < half ? i : i - half, head = j / ((size_t)n_keys * D), r = j % ((size_t)n_keys * D);
        out[i] = (i < half ? kc : vc)[head * n_ctx * D + r];
    }
}

}  // namespace

int attn_chunk_for(int n_ctx) {
    // 16 keys per workgroup, doubled while a KV head would need more than 32 chunks (at most 32 partials per head are
    // merged for n_ctx ≤ 8192), up to 256 keys. Measured on one MI355X at 1536 keys: 24 chunks of 64 keys 6.95 µs a
    // launch, 48 of 32 8.2 µs, 96 of 16 12.3 µs, 12 of 128 7.15 µs (the merge and the ticket grow with the chunk
    // count, the workgroup's own load phase with its keys). At most 16 or 8 chunks a KV head instead (graph nodes,
    // µs at 512 / 2048 / 8192 keys): 5.26 / 6.19 / 10.19 with 32, 5.25 / 6.48 / 10.15 with 16, 5.22 / 8.24 / 10.19
    // with 8 — 512 keys sit at the launch's floor whatever the split
    int chunk = 16;
    while ((n_ctx + chunk - 1) / chunk > 32 && chunk < MAX_CHUNK_KEYS) chunk *= 2;
    return chunk;
}

size_t attn_part_bytes(int n_head, int max_chunk) { return (size_t)n_head * max_chunk * (D + 2) * 4; }

size_t attn_counter_bytes(int n_kv) { return (size_t)n_kv * CNT_STRIDE * 4; }

int launch_qkv_post(htr_device *dev, hipStream_t st, float *qkv, const float *qn, const float *kn, const float *rope,
                    int n_head, int n_kv, const int *pos_dev, int pos, int n_ctx, float eps, uint16_t *kc,
                    uint16_t *vc) {
    hipLaunchKernelGGL(k_qkv_post, dim3(n_head + 2 * n_kv), dim3(64), 0, st, qkv, qn, kn, rope, n_head, n_kv, pos_dev,
                       pos, n_ctx, eps, (_Float16 *)kc, (_Float16 *)vc);
    return htr_launched(dev, "k_qkv_post");
}

int launch_attn_decode(htr_device *dev, hipStream_t st, const float *q, const uint16_t *kc, const uint16_t *vc,
                       int n_head, int n_kv, int n_ctx, const int *pos_dev, int n_keys, float scale,
                       const AttnScratch &sc, float *out, const AttnFuse *fuse, bool scale_after) {
    if (n_head != 2 * n_kv) return htr_fail("decode attention: %d q heads on %d kv heads (groups of 2)", n_head, n_kv);
    if (sc.chunk < 16 || sc.chunk > MAX_CHUNK_KEYS || (sc.chunk & (sc.chunk - 1)))
        return htr_fail("decode attention: chunk %d (a power of two, 16 … %d)", sc.chunk, MAX_CHUNK_KEYS);
    if (!pos_dev && (n_keys < 1 || n_keys > n_ctx)) return htr_fail("decode attention: %d keys, cache %d", n_keys, n_ctx);
    if ((size_t)sc.max_chunk * sc.chunk < (size_t)n_ctx || sc.max_chunk > MAX_CHUNKS)
        return htr_fail("decode attention: %d chunks of %d keys for a %d-row cache (at most %d chunks)", sc.max_chunk,
                        sc.chunk, n_ctx, MAX_CHUNKS);
    const int grid_x = pos_dev ? sc.max_chunk : (n_keys + sc.chunk - 1) / sc.chunk;
    const dim3 grid(grid_x * n_kv);
    const AttnFuse fz = fuse ? *fuse : AttnFuse{};
    if (fuse && (fz.n_head != n_head || !fz.qn || !fz.kn || !fz.rope || !fz.kc || !fz.vc))
        return htr_fail("decode attention: incomplete qkv_post arguments");
    // the F32 path scales each score after its dot product (attn_scores.wgsl:38); the f16 paths scale q first
    // (attn_decode.wgsl:40). A scale of exactly 1 on the other side leaves the values as they are.
    if (scale_after && fuse) return htr_fail("decode attention: the fused step pre-scales q");
    const float pre = scale_after ? 1.0f : scale, post = scale_after ? scale : 1.0f;
    // 8 KV heads: workgroup b takes KV head b mod 8 and runs on XCD b mod 8, so a head's chunks share one XCD's L2
    // where the device's placement and XCD-local visibility were checked at open (token_step_xcds): 512 / 2048 / 8192
    // keys 5.25 → 4.93, 6.17 → 5.82, 10.2 → 9.83 µs a graph node (A/B twice on one box, outputs bit-identical)
    const int xl = n_kv == 8 && dev->xcd_round_robin == 1;
#define HTR_ATTN(NI)                                                                                                   \
    if (fuse)                                                                                                          \
        hipLaunchKernelGGL((k_attn_decode<NI, true>), grid, dim3(AW), 0, st, q, (const _Float16 *)kc,                  \
                           (const _Float16 *)vc, n_kv, n_ctx, pos_dev, n_keys, sc.max_chunk, pre, post, sc.part,       \
                           sc.counters, out, fz, xl);                                                                  \
    else                                                                                                               \
        hipLaunchKernelGGL((k_attn_decode<NI, false>), grid, dim3(AW), 0, st, q, (const _Float16 *)kc,                 \
                           (const _Float16 *)vc, n_kv, n_ctx, pos_dev, n_keys, sc.max_chunk, pre, post, sc.part,       \
                           sc.counters, out, fz, xl)
    switch (sc.chunk / 16) {
    case 1: HTR_ATTN(1); break;
    case 2: HTR_ATTN(2); break;
    case 4: HTR_ATTN(4); break;
    case 8: HTR_ATTN(8); break;
    default: HTR_ATTN(16); break;
    }
#undef HTR_ATTN
    return htr_launched(dev, "k_attn_decode");
}

int launch_kv_rows(htr_device *dev, hipStream_t st, const float *k, const float *v, const float *kn, const float *rope,
                   int n_tok, int n_kv, int pos0, int n_ctx, float eps, uint16_t *kc, uint16_t *vc) {
    const int n_rows = 2 * n_tok * n_kv;
    hipLaunchKernelGGL(k_kv_rows, dim3((n_rows + 15) / 16), dim3(256), 0, st, k, v, kn, rope, n_rows, n_kv, pos0, n_ctx,
                       eps, (_Float16 *)kc, (_Float16 *)vc);
    return htr_launched(dev, "k_kv_rows");
}

int launch_attn_causal(htr_device *dev, hipStream_t st, const float *q, const uint16_t *kc, const uint16_t *vc,
                       int n_q, int pos0, int n_head, int n_kv, int n_ctx, float scale, const CausalPost *post,
                       float *out, _Float16 *out16) {
    if (n_head != 2 * n_kv) return htr_fail("causal attention: %d q heads on %d kv heads (groups of 2)", n_head, n_kv);
    if (n_q < 1 || pos0 < 0 || pos0 + n_q > n_ctx)
        return htr_fail("causal attention: %d queries from position %d in a %d-row cache", n_q, pos0, n_ctx);
    if (!out == !out16) return htr_fail("causal attention: one output, f32 or f16");
    if (((uintptr_t)kc | (uintptr_t)vc) & 15) return htr_fail("causal attention: the caches must be 16-byte aligned");
    const dim3 grid(((n_q + CQ - 1) / CQ) * n_kv);
    const CausalPost p = post ? *post : CausalPost{};
#define HTR_CAUSAL(OT, POST, O)                                                                                        \
    hipLaunchKernelGGL((k_attn_causal<OT, POST>), grid, dim3(CW), 0, st, q, (const _Float16 *)kc, (const _Float16 *)vc, \
                       n_q, pos0, n_head, n_kv, n_ctx, scale, p.qn, p.rope, p.eps, O)
    if (out && post) HTR_CAUSAL(float, true, out);
    else if (out) HTR_CAUSAL(float, false, out);
    else if (post) HTR_CAUSAL(_Float16, true, out16);
    else HTR_CAUSAL(_Float16, false, out16);
#undef HTR_CAUSAL
    return htr_launched(dev, out ? "k_attn_causal" : "k_attn_causal<f16>");
}

// ---- the allocation-free decode attention ----------------------------------------------------------------------------
//
// htr_decode_attention_static keeps its split-K partials and ticket counters in one file-scope device array instead
// of device memory the library allocates. Every GPU the library runs on holds its own copy (STATIC_SCRATCH_BYTES,
// until the process ends); its address on a device is looked up once, when the device is opened
// (attn_static_scratch_init), and kept in the device object — host code passes that address, never the array's name
// (which on the host is a stand-in, not a device address). Layout: the tickets of up to STATIC_MAX_KV KV heads (one
// 128-byte line each), then the partials [n_head][max_chunk][130] f32. Every call clears the tickets it uses with a
// fill kernel first; calls that overlap on one GPU share the array and race.
namespace {

constexpr size_t STATIC_SCRATCH_BYTES = 4u << 20;
constexpr int STATIC_MAX_KV = 64;
constexpr size_t STATIC_CNT_BYTES = (size_t)STATIC_MAX_KV * CNT_STRIDE * 4;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

__global__ __launch_bounds__(256) void k_zero_u32(uint32_t *p, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0u;
}

}  // namespace

int attn_static_scratch_init(htr_device *dev) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return htr_fail("hipGetSymbolAddress of the static attention scratch on device %d: %s", dev->ordinal,
                        hipGetErrorString(e));
    dev->static_scratch = p;
    return 0;
}

// ---- ABI ------------------------------------------------------------------------------------------------------------

extern "C" int htr_qkv_post(htr_device *dev, float *d_qkv, const float *d_q_norm, const float *d_k_norm,
                            const float *d_rope, int n_head, int n_kv, int pos, int n_ctx, float eps, uint16_t *d_k,
                            uint16_t *d_v) {
    HTR_TRY(htr_check_alive(dev));
    if (!d_qkv || !d_q_norm || !d_k_norm || !d_rope || !d_k || !d_v) return htr_fail("htr_qkv_post: null argument");
    if (pos < 0 || pos >= n_ctx || n_head <= 0 || n_kv <= 0)
        return htr_fail("htr_qkv_post: position %d of a %d-row cache, %d / %d heads", pos, n_ctx, n_head, n_kv);
    return launch_qkv_post(dev, dev->stream, d_qkv, d_q_norm, d_k_norm, d_rope, n_head, n_kv, nullptr, pos, n_ctx, eps,
                           d_k, d_v);
}

extern "C" int htr_causal_attention(htr_device *dev, const float *d_q, const uint16_t *d_k, const uint16_t *d_v,
                                    int n_q, int pos0, int n_head, int n_kv, int n_ctx, float scale, float *d_out) {
    HTR_TRY(htr_check_alive(dev));
    if (!d_q || !d_k || !d_v || !d_out) return htr_fail("htr_causal_attention: null argument");
    if (n_q < 1 || pos0 < 0 || n_ctx < 1 || pos0 > n_ctx - n_q)
        return htr_fail("htr_causal_attention: %d queries from position %d in a %d-row cache", n_q, pos0, n_ctx);
    if (n_head != 2 * n_kv) return htr_fail("causal attention: %d q heads on %d kv heads (groups of 2)", n_head, n_kv);
    if (((uintptr_t)d_k | (uintptr_t)d_v) & 15) {
        const int n_keys = pos0 + n_q;
        const size_t half = (size_t)n_kv * n_keys * D;
        void *copy;
        HTR_TRY(htr_scratch(dev, SCR_CAUSAL_KV, 2 * half * sizeof(_Float16), &copy));
        hipLaunchKernelGGL(k_kv_align, dim3(dev->n_cu * 8), dim3(256), 0, dev->stream, (const _Float16 *)d_k,
                           (const _Float16 *)d_v, n_kv, n_ctx, n_keys, (_Float16 *)copy);
        HTR_TRY(htr_launched(dev, "k_kv_align"));
        d_k = (const uint16_t *)copy;
        d_v = d_k + half;
        n_ctx = n_keys;
    }
    return launch_attn_causal(dev, dev->stream, d_q, d_k, d_v, n_q, pos0, n_head, n_kv, n_ctx, scale, nullptr, d_out);
}

extern "C" int htr_decode_attention(htr_device *dev, const float *d_q, const uint16_t *d_k, const uint16_t *d_v,
                                    int n_head, int n_kv, int n_ctx, int n_keys, float scale, float *d_out) {
    HTR_TRY(htr_check_alive(dev));
    if (!d_q || !d_k || !d_v || !d_out) return htr_fail("htr_decode_attention: null argument");
    if (n_keys < 1 || n_keys > n_ctx) return htr_fail("htr_decode_attention: %d keys in a %d-row cache", n_keys, n_ctx);
    if (n_ctx > MAX_CHUNKS * MAX_CHUNK_KEYS)
        return htr_fail("htr_decode_attention: a %d-row cache (at most %d)", n_ctx, MAX_CHUNKS * MAX_CHUNK_KEYS);
    AttnScratch sc{};
    sc.chunk = attn_chunk_for(n_ctx);
    sc.max_chunk = (n_ctx + sc.chunk - 1) / sc.chunk;
    HTR_TRY(htr_scratch(dev, SCR_ATTN_PART, attn_part_bytes(n_head, sc.max_chunk), (void **)&sc.part));
    HTR_TRY(htr_scratch(dev, SCR_ATTN_CNT, attn_counter_bytes(n_kv), (void **)&sc.counters));
    return launch_attn_decode(dev, dev->stream, d_q, d_k, d_v, n_head, n_kv, n_ctx, nullptr, n_keys, scale, sc, d_out);
}

extern "C" int htr_decode_attention_static(htr_device *dev, const float *d_q, const uint16_t *d_k, const uint16_t *d_v,
                                           int n_head, int n_kv, int n_ctx, int n_keys, float scale, float *d_out) {
    HTR_TRY(htr_check_alive(dev));
    if (!d_q || !d_k || !d_v || !d_out) return htr_fail("htr_decode_attention_static: null argument");
    if (n_keys < 1 || n_keys > n_ctx)
        return htr_fail("htr_decode_attention_static: %d keys in a %d-row cache", n_keys, n_ctx);
    if (n_ctx > MAX_CHUNKS * MAX_CHUNK_KEYS)
        return htr_fail("htr_decode_attention_static: a %d-row cache (at most %d)", n_ctx, MAX_CHUNKS * MAX_CHUNK_KEYS);
    if (n_kv < 1 || n_kv > STATIC_MAX_KV)
        return htr_fail("htr_decode_attention_static: %d KV heads (the static scratch has tickets for %d)", n_kv,
                        STATIC_MAX_KV);
    if (!dev->static_scratch) return htr_fail("htr_decode_attention_static: the device has no static scratch address");
    AttnScratch sc{};
    sc.chunk = attn_chunk_for(n_ctx);
    sc.max_chunk = (n_ctx + sc.chunk - 1) / sc.chunk;
    const size_t part = attn_part_bytes(n_head, sc.max_chunk);
    if (part > STATIC_SCRATCH_BYTES - STATIC_CNT_BYTES)
        return htr_fail("htr_decode_attention_static: %d heads x %d chunks need %zu bytes of partials, the static scratch "
                        "holds %zu",
                        n_head, sc.max_chunk, part, STATIC_SCRATCH_BYTES - STATIC_CNT_BYTES);
    unsigned char *base = (unsigned char *)dev->static_scratch;
    sc.counters = (uint32_t *)base;
    sc.part = (float *)(base + STATIC_CNT_BYTES);
    const int n_cnt = n_kv * CNT_STRIDE;
    hipLaunchKernelGGL(k_zero_u32, dim3((n_cnt + 255) / 256), dim3(256), 0, dev->stream, sc.counters, n_cnt);
    HTR_TRY(htr_launched(dev, "k_zero_u32"));
    return launch_attn_decode(dev, dev->stream, d_q, d_k, d_v, n_head, n_kv, n_ctx, nullptr, n_keys, scale, sc, d_out);
}
