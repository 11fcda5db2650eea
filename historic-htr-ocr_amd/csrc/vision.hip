// The vision encoder's non-GEMM kernels for gfx950, and the f16 pieces of the f32 operands that its patch embedding
// and projector multiply on the matrix cores.
//
// Reference semantics (the f16 compute path, vision.rs:328-423): patchify.wgsl (normalise + im2col), rms_norm.wgsl /
// rms_norm_h (gpu.rs:268-275), rope2d.wgsl (+ vision.rs:159-175; applied as K and q are read), heads_f16.wgsl,
// attention_coop.wgsl (flash attention with q·scale, K, V and P rounded to f16, f32 sums, the output rounded to f16),
// unfold2x2.wgsl, gelu.wgsl; the f32 matmuls of the patch embedding (K = 588) and the projector (f32 activations,
// f16-valued weights) run as f16 GEMMs over split operands (k_split_f16).
#include <cmath>
#include <type_traits>

#include "htr_internal.h"
#include "wave.h"

namespace {

constexpr int VW = 256;

__device__ __forceinline__ size_t gsize() { return (size_t)gridDim.x * VW; }
__device__ __forceinline__ size_t gid() { return blockIdx.x * (size_t)VW + threadIdx.x; }

// x as f16 pieces: hi = f16(x), lo = f16(x − hi)
__device__ __forceinline__ void split_hi_lo(float v, _Float16 &hi, _Float16 &lo) {
    hi = (_Float16)v;
    lo = (_Float16)(v - (float)hi);
}

// patchify.wgsl, P[t][c·p·p + ky·p + kx] = lut[c·256 + rgb[((ty·p + ky)·w + tx·p + kx)·3 + c]], straight into the pieces
// [hi | hi | lo] that the patch embedding multiplies (k_split_f16's layout, segments of kp): a patch a workgroup. The
// bytes of a patch and its 3·kp halves are all that moves; patches written as f32 and split by a second kernel took
// 24 + 20 µs for 8580 of them, this 21 µs
__global__ __launch_bounds__(VW) void k_patchify_split(const uint8_t *rgb, const float *lut, int w, int px, int side, int kp,
                                                       _Float16 *out) {
    const int t = blockIdx.x, pp = side * side;
    const uint8_t *src = rgb + ((size_t)(t / px) * side * w + (size_t)(t % px) * side) * 3;
    _Float16 *dst = out + (size_t)t * 3 * kp;
    for (int r = threadIdx.x; r < kp; r += VW) {
        const int c = r / pp, i = r % pp;
        const float v = r < 3 * pp ? lut[c * 256 + src[((size_t)(i / side) * w + i % side) * 3 + c]] : 0.0f;
        _Float16 hi, lo;
        split_hi_lo(v, hi, lo);
        dst[r] = hi;
        dst[kp + r] = hi;
        dst[2 * kp + r] = lo;
    }
}

// one workgroup per row: y = x·1/sqrt(mean(x²) + eps)·w, as f32 or rounded to f16
template <typename T>
__global__ __launch_bounds__(VW) void k_rms_norm_rows(const float *x, const float *w, T *y, int dim, float eps) {
    __shared__ float red[VW / 64];
    const size_t base = (size_t)blockIdx.x * dim;
    const int tid = threadIdx.x, lane = tid & 63;
    float s = 0.0f;
    for (int i = tid; i < dim; i += VW) s = fmaf(x[base + i], x[base + i], s);
    s = wave_sum(s, lane);
    if (lane == 0) red[tid >> 6] = s;
    __syncthreads();
    const float scale = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)dim + eps);
    for (int i = tid; i < dim; i += VW) y[base + i] = (T)((x[base + i] * scale) * w[i]);
}

// the same for dim = 1024·NV: a thread holds NV float4 of the row, so x is read once, in 16-byte loads
template <typename T, int NV>
__global__ __launch_bounds__(VW) void k_rms_norm_rows4(const float *x, const float *w, T *y, int dim, float eps) {
    __shared__ float red[VW / 64];
    const float4 *xr = reinterpret_cast<const float4 *>(x + (size_t)blockIdx.x * dim);
    const int tid = threadIdx.x, lane = tid & 63;
    float4 v[NV];
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; j++) {
        v[j] = xr[tid + VW * j];
        s = fmaf(v[j].x, v[j].x, s);
        s = fmaf(v[j].y, v[j].y, s);
        s = fmaf(v[j].z, v[j].z, s);
        s = fmaf(v[j].w, v[j].w, s);
    }
    s = wave_sum(s, lane);
    if (lane == 0) red[tid >> 6] = s;
    __syncthreads();
    const float scale = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)dim + eps);
    const float4 *w4 = reinterpret_cast<const float4 *>(w);
    typedef T t4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const float4 ww = w4[tid + VW * j];
        const t4 o = {(T)((v[j].x * scale) * ww.x), (T)((v[j].y * scale) * ww.y), (T)((v[j].z * scale) * ww.z),
                      (T)((v[j].w * scale) * ww.w)};
        *reinterpret_cast<t4 *>(y + (size_t)blockIdx.x * dim + 4 * (tid + VW * j)) = o;
    }
}

// rope2d.wgsl on 8 consecutive dims d0 … d0 + 7 of a head (d0 a multiple of 8, head dim 64), in registers: the
// pairs (2k, 2k + 1) of each 32-dim half, half 0 turned by the row t / px, half 1 by the column t % px;
// cs = [half][pos][k] × (cos, sin), 16 pairs a half
__device__ __forceinline__ void rope8(float (&x)[8], const float *cs, int t, int px, int max_pos, int d0) {
    const int half = d0 >> 5, k0 = (d0 & 31) >> 1, pos = half == 0 ? t / px : t % px;
    const float4 *c4 = reinterpret_cast<const float4 *>(cs + 2 * (((size_t)half * max_pos + pos) * 16 + k0));
    const float4 a = c4[0], b = c4[1];
    const float c[4] = {a.x, a.z, b.x, b.z}, sn[4] = {a.y, a.w, b.y, b.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float x0 = x[2 * e], x1 = x[2 * e + 1];
        x[2 * e] = x0 * c[e] - x1 * sn[e];
        x[2 * e + 1] = x0 * sn[e] + x1 * c[e];
    }
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

// Key order of the transposed values inside a block of 32 keys: stored slot 16s + 8h + j (s, h < 2, j < 8) holds key
// 16s + 8(j / 4) + 4h + j % 4. These are the keys whose scores lane half h holds in registers 8s … 8s + 7 after the
// 32x32 score MFMAs below, so P·V step s takes its P operand straight from those registers.
__device__ __forceinline__ int vt_key(int slot) {
    const int st = slot >> 4, hf = (slot >> 3) & 1, j = slot & 7;
    return 16 * st + 8 * (j >> 2) + 4 * hf + (j & 3);
}

// K / V of one head in blocks of 32 keys, 8 KB a block: K [32 keys][64 dims] then Vᵀ [64 dims][32 slots], f16, in
// 16-byte chunks placed so that the attention's fragment reads from LDS hit 16 different 16-byte bank groups in every
// 16 lanes (gfx950's LDS serves 16 lanes of a 16-byte read a cycle across 256 bytes): K row r, chunk j (dims 8j …) at
// chunk r·8 + (j ^ (r/2 % 8)); Vᵀ row d, chunk q (slots 8q …) at 256 + d·4 + (q ^ (d/4 % 4))
constexpr int KVB = 8192;
__device__ __forceinline__ int kv_kchunk(int r, int j) { return r * 8 + (j ^ ((r >> 1) & 7)); }
__device__ __forceinline__ int kv_vchunk(int d, int q) { return 256 + d * 4 + (q ^ ((d >> 2) & 3)); }

// rope2d.wgsl on K, then heads_f16.wgsl's rounding: K, V f32 [n][H·64] → f16 blocks as above, keys n … ⌈n/32⌉·32 − 1
// zero. grid (blocks, H), one block of one head per workgroup; V goes through LDS for the transposition.
__global__ __launch_bounds__(VW) void k_heads_f16(const float *K, const float *V, _Float16 *KV, int n_tok, int n_head,
                                                  int n_blk, const float *cs, int px, int max_pos) {
    __shared__ _Float16 s_v[32][64 + 2];
    const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int r = tid >> 3, j8 = tid & 7, t = 32 * b + r;
    float kv[8] = {}, vv[8] = {};
    if (t < n_tok) {
        const float4 *ks = reinterpret_cast<const float4 *>(K + (size_t)t * n_head * 64 + h * 64 + 8 * j8);
        const float4 *vs = reinterpret_cast<const float4 *>(V + (size_t)t * n_head * 64 + h * 64 + 8 * j8);
        const float4 k0 = ks[0], k1 = ks[1], v0 = vs[0], v1 = vs[1];
        kv[0] = k0.x, kv[1] = k0.y, kv[2] = k0.z, kv[3] = k0.w, kv[4] = k1.x, kv[5] = k1.y, kv[6] = k1.z, kv[7] = k1.w;
        vv[0] = v0.x, vv[1] = v0.y, vv[2] = v0.z, vv[3] = v0.w, vv[4] = v1.x, vv[5] = v1.y, vv[6] = v1.z, vv[7] = v1.w;
        rope8(kv, cs, t, px, max_pos, 8 * j8);
    }
    half8 kh;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        kh[j] = (_Float16)kv[j];
        s_v[r][8 * j8 + j] = (_Float16)vv[j];
    }
    half8 *blk = reinterpret_cast<half8 *>(KV + ((size_t)h * n_blk + b) * (KVB / 2));
    blk[kv_kchunk(r, j8)] = kh;
    __syncthreads();
    const int d = tid >> 2, q = tid & 3;
    half8 vt;
#pragma unroll
    for (int j = 0; j < 8; j++) vt[j] = s_v[vt_key(8 * q + j)][d];
    blk[kv_vchunk(d, q)] = vt;
}

// attention_coop.wgsl's arithmetic on the f16 MFMAs: O[t][h] = softmax(q16·K16ᵀ)·V16 with q16 = f16(q·scale), keys in
// blocks of 32 with the running max (start −3e38), P = f16(e^(S − max)), l = l·corr + Σ P, O = O·corr + P·V (f32
// accumulation in the matrix unit, as the reference's cooperative matrices accumulate); O / l → f16.
// A wave takes QG groups of 32 queries of one head. Per key block and group, Sᵀ (32 keys × 32 queries) = K·q16ᵀ is 4
// MFMAs 32x32x16: lane ℓ = 32h + c then holds query c's scores of keys 8(i / 4) + 4h + i % 4 (i < 16), the other 16
// in lane ℓ ^ 32. Oᵀ (64 dims × 32 queries) += Vᵀ·Pᵀ is 4 more, lane ℓ accumulating dims 32t + 8(i / 4) + 4h + i % 4
// of query c, so the rescale by the query's corr stays in the lane.
// The 4 waves of a workgroup (128·QG queries) share the key blocks: stages of AST blocks are copied from memory to LDS by
// direct loads, the next stage's in flight while the current one is in use, and each wave reads its fragments from there.
// Work: a page makes n_head · ⌈n / (128·QG)⌉ tiles, a workgroup is one of two on every CU (`workers` a group), and an
// uneven last round would cost as much as a full one. So each worker takes whole tiles while the rounds are full, and the
// tiles that are left are cut along their keys into equal shares, one a worker, whose sums go to memory and are joined by
// k_attn_vision_merge. The workers of a group (with H a multiple of 8: an XCD, workgroup b runs on XCD b % 8) share its
// heads, so a head's keys stay in one XCD's L2.
constexpr int FQ = 32, FB = 32, FWAVES = VW / 64, AST = 2;
// p = 2^(s·log2 e + nm), nm = 10 − log2 e · (the max when it was last moved): nm moves, and O and l are rescaled, only
// when some p would pass 2^15 (f16 holds 65504), so most blocks skip the rescale; nm is the only state, its rounding
// cancels between p, l and O. That rounding is up to 4 at 2^26 and doubles with the max: from there on the shift is left
// out, so p stays in f16's range up to 2^28, as far as e^(s − max) taken as 2^(s·log2 e − max·log2 e) did
constexpr float P_SHIFT = 10.0f, P_TOP = 15.0f, LOG2E = 1.4426950408889634f;
constexpr int RING = 3;      // stages in LDS: the one in use, the next one (its first K block), one loading
constexpr int CUT_COST = 8;  // stages that a cut has to save: the partial sums' way through memory and the merge's launch

struct VSplit {
    int groups, workers;      // groups of heads; workers a group
    int tiles, full;          // tiles a group; the first `full` of them are taken whole
    int n_qt, n_stage;        // tiles a head; stages of AST key blocks
    __host__ __device__ int slots() const { return workers + tiles - full - 1; }  // a group's
    __host__ __device__ int first(int i) const {  // the first of worker i's stages of the tiles that are cut
        return (int)((long long)(tiles - full) * n_stage * i / workers);
    }
};
// a worker's sums of a part of a tile: [wave][query group][dim tile][16] registers, then nm and l, × 64 lanes. Worker i's
// part of cut tile t is the group's slot i + t (along the keys i or t grows from one part to the next)
template <int QG> constexpr int PART = FWAVES * QG * 34 * 64;

// QG groups of 32 queries a wave: the groups share every K / V fragment read from LDS and give the wave QG
// independent chains (Sᵀ MFMAs → max → exp → P·V) to interleave
template <int QG>
__global__ __launch_bounds__(VW) void k_attn_vision(const float *Q, const _Float16 *KV, _Float16 *O, int n_tok,
                                                    int n_head, int n_blk, VSplit sp, float scale, const float *cs,
                                                    int px, int max_pos, float *part) {
    __shared__ __attribute__((aligned(16))) half8 s_kv[RING][AST * KVB / 16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hf = lane >> 5, c = lane & 31;
    const int grp = blockIdx.x % sp.groups, wk = blockIdx.x / sp.groups, row = n_head * 64;
    const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) half8 *)&s_kv[0][64 * wave];
    // the lane's fragment chunks within a block: K step ks (key c, dims 16ks + 8h …), Vᵀ tile t step st (dim 32t + c,
    // slots 16st + 8h …)
    int kc[4], vc[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) kc[ks] = kv_kchunk(c, 2 * ks + hf);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int st = 0; st < 2; st++) vc[2 * t + st] = kv_vchunk(32 * t + c, 2 * st + hf);
    // stages 0 … n_full − 1 hold keys < n_tok only
    const int n_full = n_tok / (AST * FB);

    // stages st0 … st1 − 1 of a tile; slot: where the sums go, −1: the tile is whole
    auto run = [&](int tile, int st0, int st1, int slot) {
        const int h = grp * (n_head / sp.groups) + tile / sp.n_qt, q0 = ((tile % sp.n_qt) * FWAVES + wave) * FQ * QG;
        const char *gkv = (const char *)KV + (size_t)h * n_blk * KVB;
        // a stage is 16 KB: 4 direct loads a wave (blocks past the last repeat it: in bounds)
        auto issue = [&](int st) {
#pragma unroll
            for (int i = 0; i < 2 * AST; i++)
                lds_load16(gkv + (size_t)min(st * AST + i / 2, n_blk - 1) * KVB + (i % 2) * (VW * 16), 16 * tid,
                           lds + (st % RING) * (AST * KVB) + i * (VW * 16));
        };
        issue(st0);
        if (st0 + 1 < st1) issue(st0 + 1);
        half8 qf[QG][4];  // B operand of step ks: q16[query c][dims 16ks + 8h … + 7], q turned by rope2d first
#pragma unroll
        for (int g = 0; g < QG; g++) {
            const int qi = min(q0 + FQ * g + c, n_tok - 1);
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const float4 *src = reinterpret_cast<const float4 *>(Q + (size_t)qi * row + h * 64 + 16 * ks + 8 * hf);
                const float4 x0 = src[0], x1 = src[1];
                float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
                rope8(x, cs, qi, px, max_pos, 16 * ks + 8 * hf);
#pragma unroll
                for (int e = 0; e < 8; e++) qf[g][ks][e] = (_Float16)(x[e] * scale);
            }
        }
        f32x16 o[QG][2];
        float nm[QG], l[QG];
#pragma unroll
        for (int g = 0; g < QG; g++) {
            nm[g] = 3.0e38f;
            l[g] = 0.0f;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[g][t][i] = 0.0f;
        }
        // the two groups take turns: while the VALU does group X's softmax of block j, the matrix pipe does group Y's next
        // scores and its P·V of the block before. Phase 0: X = 0, Y = 1 with the scores of block j, P·V of j − 1, and K of
        // block j + 1 read behind them; phase 1: X = 1, Y = 0 with the scores of block j + 1, V of block j read, then P·V
        // of j. The order is pinned: behind each MFMA two scores' share of the softmax
        f32x16 sc[QG];
        half8 kf[4], vf[4] = {};
        uint32_t pb[QG][8] = {};
        auto kread = [&](const half8 *blk, int ks) { kf[ks] = blk[kc[ks]]; };
        auto pv = [&](int g, int i) {
            const int t = i & 1, st = i >> 1;
            half8 p;
            __builtin_memcpy(&p, &pb[g][4 * st], 16);
            o[g][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[2 * t + st], p, o[g][t], 0, 0, 0);
        };
        auto score = [&](int g, int ks) {
            sc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ks], qf[g][ks], ks ? sc[g] : f32x16{}, 0, 0, 0);
        };
        // blk: block j; nxt: block j + 1 (past the last one: whatever the buffer holds; its scores are not used); k0: the
        // block's first key; MASK: keys ≥ n_tok score −inf
        auto step = [&](const half8 *blk, const half8 *nxt, int k0, auto mask) {
            constexpr bool MASK = decltype(mask)::value;
#pragma unroll
            for (int X = 0; X < QG; X++) {
                const int Y = X ^ 1;
                float mx = -INFINITY;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    if (MASK && k0 + 8 * (i >> 2) + 4 * hf + (i & 3) >= n_tok) sc[X][i] = -INFINITY;
                    mx = fmaxf(mx, sc[X][i]);
                }
                mx = pair_max<32>(mx);
                if (__builtin_amdgcn_ballot_w64(fmaf(mx, LOG2E, nm[X]) > P_TOP)) {
                    const float to = fminf(nm[X], fmaf(-mx, LOG2E, fabsf(mx) < 0x1p26f ? P_SHIFT : 0.0f));
                    const float corr = __builtin_amdgcn_exp2f(to - nm[X]);
                    nm[X] = to;
                    l[X] *= corr;
#pragma unroll
                    for (int t = 0; t < 2; t++) o[X][t] *= corr;
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (i < 4) score(Y, i);
                    else pv(Y, i - 4);
                    if (X == 0 && i >= 4) kread(nxt, i - 4);
                    if (X == 1 && i < 4) vf[i] = blk[vc[i]];
                    // P rounded to f16 in pairs (v_cvt_pk_f16_f32, round to nearest even), summed as f32 by v_dot2 against (1, 1)
                    const half2_t p2 = __builtin_convertvector(
                        (float2_t{__builtin_amdgcn_exp2f(fmaf(sc[X][2 * i], LOG2E, nm[X])),
                                  __builtin_amdgcn_exp2f(fmaf(sc[X][2 * i + 1], LOG2E, nm[X]))}),
                        half2_t);
                    __builtin_memcpy(&pb[X][i], &p2, 4);
                    l[X] = __builtin_amdgcn_fdot2(p2, half2_t{(_Float16)1.0f, (_Float16)1.0f}, l[X], false);
                    asm volatile("" : "+v"(pb[X][i]), "+v"(l[X]));  // holds the two here
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        static_assert(QG == 2 && AST == 2, "the turns of two groups, two blocks a stage");
        auto turn = [&](int st) {
            // this wave's loads of stage st + 1 are in and its reads of stage st − 1 have their values, wherever their
            // MFMAs stand; behind the barrier everyone's
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (st + 2 < st1) issue(st + 2);
        };
        auto at = [&](int st, int j) { return s_kv[st % RING] + j * (KVB / 16); };
        // the loop body has one path, so O stays in the same registers through every iteration
        const int to = min(st1, n_full);
        turn(st0);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) kread(at(st0, 0), ks);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) score(0, ks);
        for (int st = st0; st < to; st++) {
            if (st > st0) turn(st);
            step(at(st, 0), at(st, 1), 0, std::false_type{});
            step(at(st, 1), at(st + 1, 0), 0, std::false_type{});
        }
        if (to < st1) {  // the last stage, with keys ≥ n_tok
            const int st = st1 - 1, k0 = st * AST * FB;
            if (st > st0) turn(st);
            step(at(st, 0), at(st, 1), k0, std::true_type{});
            if (k0 + FB < n_tok) step(at(st, 1), at(st, 1), k0 + FB, std::true_type{});
        }
#pragma unroll
        for (int i = 0; i < 4; i++) pv(1, i);
        // the next tile's first stage overwrites a buffer that another wave may still read
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int g = 0; g < QG; g++) {
            l[g] = pair_sum<32>(l[g]);
            if (slot >= 0) {
                float *p = part + (size_t)slot * PART<QG> + (size_t)(wave * QG + g) * 34 * 64 + lane;
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int i = 0; i < 16; i++) p[(16 * t + i) * 64] = o[g][t][i];
                p[32 * 64] = nm[g];
                p[33 * 64] = l[g];
            } else if (q0 + FQ * g + c < n_tok) {
                typedef _Float16 half4 __attribute__((ext_vector_type(4)));
                const float inv = 1.0f / l[g];
                _Float16 *dst = O + (size_t)(q0 + FQ * g + c) * row + h * 64 + 4 * hf;
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        *reinterpret_cast<half4 *>(dst + 32 * t + 8 * r) =
                            half4{(_Float16)(o[g][t][4 * r] * inv), (_Float16)(o[g][t][4 * r + 1] * inv),
                                  (_Float16)(o[g][t][4 * r + 2] * inv), (_Float16)(o[g][t][4 * r + 3] * inv)};
            }
        }
    };
    // the worker's share of the cut tiles (it touches two at most), then its whole ones
    const int a = sp.first(wk), b = sp.first(wk + 1), t0 = a / sp.n_stage, cut = b > a ? (b - 1) / sp.n_stage - t0 + 1 : 0;
    const int whole = wk < sp.full ? (sp.full - 1 - wk) / sp.workers + 1 : 0;
    for (int u = 0; u < cut + whole; u++) {
        const int base = (t0 + u) * sp.n_stage;
        const bool part_of = u < cut;
        run(part_of ? sp.full + t0 + u : wk + (u - cut) * sp.workers, part_of ? max(a - base, 0) : 0,
            part_of ? min(b - base, sp.n_stage) : sp.n_stage, part_of ? grp * sp.slots() + wk + t0 + u : -1);
    }
}

// the cut tiles: the sums of the workers that share one, joined. grid (groups · cut tiles, 16·QG): a wave takes 8 of the
// 32 registers of one (wave, query group) of the tile
template <int QG>
__global__ __launch_bounds__(64) void k_attn_vision_merge(const float *part, _Float16 *O, int n_tok, int n_head, VSplit sp) {
    const int lane = threadIdx.x, hf = lane >> 5, c = lane & 31;
    const int grp = blockIdx.x % sp.groups, t = blockIdx.x / sp.groups;
    const int wg = blockIdx.y >> 2, r0 = 8 * (blockIdx.y & 3);  // (wave, group); the first register
    // the workers whose shares meet stages [base, base + n_stage) of the cut tiles
    const int base = t * sp.n_stage;
    int w0 = (int)((long long)base * sp.workers / ((long long)(sp.tiles - sp.full) * sp.n_stage));
    while (w0 > 0 && sp.first(w0) > base) w0--;
    while (sp.first(w0 + 1) <= base) w0++;
    float nm = 3.0e38f, l = 0.0f, o[8] = {};
    for (int w = w0; w < sp.workers && sp.first(w) < base + sp.n_stage; w++) {
        if (sp.first(w + 1) == sp.first(w)) continue;
        const float *p = part + (size_t)(grp * sp.slots() + w + t) * PART<QG> + (size_t)wg * 34 * 64 + lane;
        const float pn = p[32 * 64], pl = p[33 * 64];
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = p[(r0 + e) * 64];
        const float top = fminf(nm, pn), a = __builtin_amdgcn_exp2f(top - nm), b = __builtin_amdgcn_exp2f(top - pn);
        nm = top;
        l = l * a + pl * b;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = o[e] * a + v[e] * b;
    }
    const int tile = sp.full + t, h = grp * (n_head / sp.groups) + tile / sp.n_qt;
    const int q = (tile % sp.n_qt) * (FWAVES * FQ * QG) + wg * FQ + c;
    if (q >= n_tok) return;
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    const float inv = 1.0f / l;
    // register 16t + i is dim 32t + 8(i / 4) + 4h + i % 4
    _Float16 *dst = O + (size_t)q * n_head * 64 + h * 64 + 32 * (r0 >> 4) + 8 * ((r0 & 15) >> 2) + 4 * hf;
#pragma unroll
    for (int r = 0; r < 2; r++)
        *reinterpret_cast<half4 *>(dst + 8 * r) = half4{(_Float16)(o[4 * r] * inv), (_Float16)(o[4 * r + 1] * inv),
                                                        (_Float16)(o[4 * r + 2] * inv), (_Float16)(o[4 * r + 3] * inv)};
}

// the projector's input: rows normed (y = x·1/sqrt(mean(x²) + eps)·w), unfold2x2.wgsl, Z[o][c·4 + ky·2 + kx] =
// Y[(2·oy + ky)·px + 2·ox + kx][c], as the pieces [hi | lo] (k_split_f16's layout): an output row a workgroup, which reads
// its four patches twice (the second time from the caches) and writes 8 bytes a channel and piece. Norm, unfold and split
// as three kernels took 18 + 29 + 26 µs for 8580 rows of 1024, this 19 µs
__global__ __launch_bounds__(VW) void k_norm_unfold_split(const float *X, const float *w, int px, int dim, float eps,
                                                          _Float16 *out) {
    __shared__ float red[4][VW / 64];
    const int o = blockIdx.x, tid = threadIdx.x, lane = tid & 63, ox = o % (px / 2), oy = o / (px / 2);
    const float *x[4];
    float s[4] = {}, scale[4];
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = X + ((size_t)(2 * oy + (j >> 1)) * px + 2 * ox + (j & 1)) * dim;
    for (int c = tid; c < dim; c += VW)
#pragma unroll
        for (int j = 0; j < 4; j++) s[j] = fmaf(x[j][c], x[j][c], s[j]);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        s[j] = wave_sum(s[j], lane);
        if (lane == 0) red[j][tid >> 6] = s[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++)
        scale[j] = 1.0f / sqrtf(((red[j][0] + red[j][1]) + (red[j][2] + red[j][3])) / (float)dim + eps);
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    half4 *hi = reinterpret_cast<half4 *>(out + (size_t)o * 8 * dim), *lo = hi + dim;
    for (int c = tid; c < dim; c += VW) {
        half4 h, l;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float v = (x[j][c] * scale[j]) * w[c];
            asm volatile("" : "+v"(v));  // one f32 value for both pieces
            _Float16 a, b;
            split_hi_lo(v, a, b);
            h[j] = a, l[j] = b;
        }
        hi[c] = h;
        lo[c] = l;
    }
}

// gelu.wgsl (tanh form, argument clamped to ±15)
__device__ __forceinline__ float gelu(float x) {
    const float t = fminf(fmaxf(0.7978845608028654f * x * (1.0f + 0.044715f * x * x), -15.0f), 15.0f);
    return 0.5f * x * (1.0f + tanhf(t));
}

// f32 values as f16 pieces for f32-grade products on the f16 matrix cores: x [m][k] → rows of nseg segments of kp
// values (kp ≥ k, a multiple of 32, the values past k zero); segment s holds hi = f16(x), or lo = f16(x − hi) where bit
// s of lo_mask is set. x − hi is exact in f32 and hi + lo is x within 2^-22·|x| (|x| < 65504). With X as [hi, hi, lo]
// and W as [hi, lo, hi] one f16 GEMM over 3·kp sums xh·wh + xh·wl + xl·wh in f32; f16-valued W: X [hi, lo], W [w, w].
// GELU: of gelu(x)
template <bool GELU>
__global__ __launch_bounds__(VW) void k_split_f16(const float *x, int m, int k, int kp, int nseg, int lo_mask,
                                                  _Float16 *out) {
    const size_t total = (size_t)m * kp;
    for (size_t i = gid(); i < total; i += gsize()) {
        const int c = (int)(i % kp);
        const size_t r = i / kp;
        float v = c < k ? x[r * k + c] : 0.0f;
        if (GELU) {
            v = gelu(v);
            asm volatile("" : "+v"(v));  // one f32 value for both pieces
        }
        _Float16 hi, lo;
        split_hi_lo(v, hi, lo);
        for (int s = 0; s < nseg; s++) out[(r * nseg + s) * kp + c] = (lo_mask >> s) & 1 ? lo : hi;
    }
}

int grid_for(size_t total) { return (int)std::max<size_t>(1, std::min<size_t>((total + VW - 1) / VW, 65536)); }

}  // namespace

int launch_patchify_split(htr_device *dev, hipStream_t st, const uint8_t *rgb, const float *lut, int w, int px, int n,
                          int side, int kp, _Float16 *out) {
    if (n < 1 || kp < 3 * side * side) return htr_fail("patchify: %d patches of side %d in segments of %d", n, side, kp);
    hipLaunchKernelGGL(k_patchify_split, dim3(n), dim3(VW), 0, st, rgb, lut, w, px, side, kp, out);
    return htr_launched(dev, "k_patchify_split");
}

int launch_rms_norm_f16(htr_device *dev, hipStream_t st, const float *x, const float *w, _Float16 *y, int rows, int dim,
                        float eps) {
    switch (dim % (4 * VW) ? 0 : dim / (4 * VW)) {
    case 1: hipLaunchKernelGGL((k_rms_norm_rows4<_Float16, 1>), dim3(rows), dim3(VW), 0, st, x, w, y, dim, eps); break;
    case 2: hipLaunchKernelGGL((k_rms_norm_rows4<_Float16, 2>), dim3(rows), dim3(VW), 0, st, x, w, y, dim, eps); break;
    case 4: hipLaunchKernelGGL((k_rms_norm_rows4<_Float16, 4>), dim3(rows), dim3(VW), 0, st, x, w, y, dim, eps); break;
    default: hipLaunchKernelGGL(k_rms_norm_rows<_Float16>, dim3(rows), dim3(VW), 0, st, x, w, y, dim, eps); break;
    }
    return htr_launched(dev, "k_rms_norm_rows<f16>");
}

int launch_heads_f16(htr_device *dev, hipStream_t st, const float *k, const float *v, _Float16 *kv, int n_tok,
                     int n_head, const float *cs, int px, int max_pos) {
    if (px < 1 || (n_tok + px - 1) / px > max_pos || px > max_pos)
        return htr_fail("vision heads: %d tokens on %d columns, rope table of %d positions", n_tok, px, max_pos);
    const int n_blk = (n_tok + FB - 1) / FB;
    hipLaunchKernelGGL(k_heads_f16, dim3(n_blk, n_head), dim3(VW), 0, st, k, v, kv, n_tok, n_head, n_blk, cs, px,
                       max_pos);
    return htr_launched(dev, "k_heads_f16");
}

size_t vision_kv_bytes(int n_tok, int n_head) { return (size_t)n_head * ((n_tok + FB - 1) / FB) * KVB; }

// two query groups a wave: 0.69 ms a layer at 12100 patches against 0.79 ms with one (223 VGPRs, 2 waves a SIMD; forcing 3
// spills 111 of them)
constexpr int VQG = 2;

static VSplit vision_split(const htr_device *dev, int n_tok, int n_head) {
    VSplit sp{};
    sp.groups = n_head % 8 == 0 ? 8 : 1;
    sp.workers = 2 * dev->n_cu / sp.groups;
    sp.n_qt = (n_tok + VQG * FQ * FWAVES - 1) / (VQG * FQ * FWAVES);
    sp.n_stage = ((n_tok + FB - 1) / FB + AST - 1) / AST;
    sp.tiles = n_head / sp.groups * sp.n_qt;
    sp.full = sp.tiles;
    // the tiles past the full rounds are cut where that shortens the last round by more than the merge costs
    const int left = sp.tiles % sp.workers;
    if (left && (left * sp.n_stage + sp.workers - 1) / sp.workers + CUT_COST < sp.n_stage) sp.full -= left;
    return sp;
}

size_t vision_part_bytes(const htr_device *dev, int n_tok, int n_head) {
    const VSplit sp = vision_split(dev, n_tok, n_head);
    return sp.full == sp.tiles ? 0 : (size_t)sp.groups * sp.slots() * PART<VQG> * sizeof(float);
}

int launch_attn_vision(htr_device *dev, hipStream_t st, const float *q, const _Float16 *kv, _Float16 *o, int n_tok,
                       int n_head, float scale, const float *cs, int px, int max_pos, float *part) {
    if (n_tok < 1) return htr_fail("vision attention: %d tokens", n_tok);
    if (px < 1 || (n_tok + px - 1) / px > max_pos || px > max_pos)
        return htr_fail("vision attention: %d tokens on %d columns, rope table of %d positions", n_tok, px, max_pos);
    const VSplit sp = vision_split(dev, n_tok, n_head);
    hipLaunchKernelGGL(k_attn_vision<VQG>, dim3(sp.groups * sp.workers), dim3(VW), 0, st, q, kv, o, n_tok, n_head,
                       (n_tok + FB - 1) / FB, sp, scale, cs, px, max_pos, part);
    HTR_TRY(htr_launched(dev, "k_attn_vision"));
    if (sp.full == sp.tiles) return 0;
    hipLaunchKernelGGL(k_attn_vision_merge<VQG>, dim3(sp.groups * (sp.tiles - sp.full), 16 * VQG), dim3(64), 0, st, part, o,
                       n_tok, n_head, sp);
    return htr_launched(dev, "k_attn_vision_merge");
}

int launch_norm_unfold_split(htr_device *dev, hipStream_t st, const float *x, const float *w, int px, int py, int dim,
                             float eps, _Float16 *out) {
    hipLaunchKernelGGL(k_norm_unfold_split, dim3((px / 2) * (py / 2)), dim3(VW), 0, st, x, w, px, dim, eps, out);
    return htr_launched(dev, "k_norm_unfold_split");
}

int launch_split_f16(htr_device *dev, hipStream_t st, const float *x, int m, int k, int kp, int nseg, int lo_mask,
                     _Float16 *out, bool of_gelu) {
    if (m < 1 || k < 1 || kp < k || kp % 32 || nseg < 1 || nseg > 3)
        return htr_fail("split_f16: [%d x %d] into %d segments of %d", m, k, nseg, kp);
    const dim3 grid(grid_for((size_t)m * kp));
    if (of_gelu) hipLaunchKernelGGL(k_split_f16<true>, grid, dim3(VW), 0, st, x, m, k, kp, nseg, lo_mask, out);
    else hipLaunchKernelGGL(k_split_f16<false>, grid, dim3(VW), 0, st, x, m, k, kp, nseg, lo_mask, out);
    return htr_launched(dev, "k_split_f16");
}
