// Dense kernels of the prefill for gfx950: Y[M,N] (+)= X[M,K]·Wᵀ with q8_0 weights, RMS norm over rows, SwiGLU.
//
// Reference semantics: matmul.wgsl:47-91 (F32 path: W dequantised exactly — q·d is exact in f32 — and f32
// accumulation; acc = 1 adds onto Y, the residual stream), matmul_coop_q8_0 / matmul128h_q8_0 (gpu.rs:1976-1995, the
// f16 path: X and the dequantised W rounded to f16 where they enter the tiles, f32 accumulation), rms_norm.wgsl:21-41,
// swiglu.wgsl:18-24 (text.rs:484-518). The prefill's GEMMs on f16 planes made at load are in mfma_gemm.hip.
#include <algorithm>

#include "htr_internal.h"

namespace {

// one workgroup per row: y = x · 1/sqrt(mean(x²) + eps) · w
__global__ __launch_bounds__(256) void k_rms_norm(const float *x, const float *w, float *y, int dim, float eps) {
    __shared__ float red[4];
    const size_t base = (size_t)blockIdx.x * dim;
    const int tid = threadIdx.x;
    float s = 0.0f;
    for (int i = tid; i < dim; i += 256) s = fmaf(x[base + i], x[base + i], s);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    const float scale = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)dim + eps);
    for (int i = tid; i < dim; i += 256) y[base + i] = (x[base + i] * scale) * w[i];
}

__global__ __launch_bounds__(256) void k_swiglu(float *g, const float *u, size_t n) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const float v = g[i];
        g[i] = (v / (1.0f + expf(-v))) * u[i];
    }
}


// ---- GEMMs on q8_0 weights -------------------------------------------------------------------------------------------
//
// One kernel for both compute paths and any shape, on the 16-bit matrix cores:
//   f16 path  X and f16(q·d) rounded to nearest even as they enter LDS, v_mfma_f32_32x32x16_f16, f32 sums;
//   F32 path  every product of the exact q8_0 value with the f32 X. A quant is a bf16 value (7 bits) and X is the sum
//             of three (EX: its top 8 bits, the next 8, the last 8, each truncated, so x = b1 + b2 + b3 exactly), so
//             three bf16 MFMAs add a block's Σ q·x in f32 with every product exact, and one f32 fma per output and
//             block adds d·Σ q·x: three 16-bit MFMAs stand for what takes f32 ones sixteen times as long. That holds for
//             a tile without |x| from 2^115 on (a block's sum of q·x may overflow where the scaled one does not), without
//             bits of an x under bf16's smallest and without an infinite scale; one that meets them is done again by
//             wide_blocks. Looking for them costs nothing measurable; splitting and scaling every tile that way instead
//             12 % (1023 × 1024 × 3072 onto the residual 36.1 → 40.6 µs).
// Work: a workgroup owns 64T × 64T outputs; KG groups of 4 waves (2 × 2, 32T × 32T outputs a wave) take the K stages in
// turn, each through its own pair of LDS buffers, and their sums are added in group order through LDS at the end: a
// prompt of some hundred rows makes few tiles, and the groups give such a CU four waves a SIMD to hide the loads'
// latency without a second launch for the sum. A stage is KB blocks of 32 k (f16: 2, EX: 1); its loads go to registers
// R stages ahead and are converted as they are stored to LDS (16-byte chunks of 8 k, XOR-placed so that the 16 lanes of
// a fragment read fall on 16 bank groups). K past the last block is zeros, rows past M and columns past N are read clamped
// and not stored.
// Bound: the 128 × 128 tile's MFMAs and conversions about even; the 64 × 64 ones by the stages' load latency. Measured
// against the kernels before it (f32 FMA tiles on the f16 path, v_mfma_f32_32x32x2_f32 on the F32 path), a call: f16
// 48 × 1024 × 2048 230 → 13.2 µs, 1925 × 3072 × 1024 422 → 29.8 µs (406 TFLOP/s); F32 1023 × 1024 × 3072 onto the
// residual 111 → 35 µs (182 TFLOP/s, past the f32 MFMA's 157 peak). Error against 64 bits 5.6e-7 … 9.8e-7 → 1.2e-7 …
// 2.0e-7: a block's 96 products are summed inside the matrix unit before the one f32 fma that scales them.
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

// the slot of chunk c of row r in rows of CPR chunks; the XOR is its own inverse
template <int CPR> __device__ __forceinline__ int q8_slot(int r, int c) {
    return CPR * r + (c ^ (CPR == 4 ? (r >> 2) & 3 : (r >> 1) & 7));
}

// the high halves of two words as one: (hi16(a), hi16(b)), a in the low half
__device__ __forceinline__ uint32_t hi_pair(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

__device__ __forceinline__ int8_t q_byte(int2 v, int e) { return (int8_t)((uint32_t)(e < 4 ? v.x : v.y) >> (8 * (e & 3))); }

__device__ __forceinline__ int4 hi_halves(const uint32_t (&b)[8]) {
    return make_int4((int)hi_pair(b[0], b[1]), (int)hi_pair(b[2], b[3]), (int)hi_pair(b[4], b[5]), (int)hi_pair(b[6], b[7]));
}

// what a tile has met of X and of the scales: the largest magnitude that is not a NaN, and what the third pieces left over
struct Q8Seen {
    float top = 0.0f;
    uint32_t rest = 0;
    __device__ __forceinline__ void add(float a, float b) {
        asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(top) : "v"(a), "v"(b));
    }
    __device__ __forceinline__ bool wide() const { return !(top < 0x1p115f) || (rest & 0xffffu); }
};

// 8 values as three bf16 pieces, x = b1 + b2 + b3: each piece the top 16 bits of what is left (no rounding: 24 = 3 · 8
// bits). Nothing is left over from |x| = 2^-110 on (bf16 ends at 2^-133). NaN: a NaN, at least in the second piece
__device__ __forceinline__ void split3(const float (&x)[8], int4 (&out)[3], Q8Seen &seen) {
    uint32_t b[3][8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        b[0][e] = __float_as_uint(x[e]);
        const float r1 = x[e] - __uint_as_float(b[0][e] & 0xffff0000u);
        b[1][e] = __float_as_uint(r1);
        b[2][e] = __float_as_uint(r1 - __uint_as_float(b[1][e] & 0xffff0000u));
        seen.rest |= b[2][e];
        if (e & 1) seen.add(x[e - 1], x[e]);
    }
#pragma unroll
    for (int s = 0; s < 3; s++) out[s] = hi_halves(b[s]);
}

// 32 × 32J outputs of a wave over the blocks b0, b0 + step, … below b1, each product exact for all of f32 and a block's sum
// finite where the scaled one is: x = b1 + 2^-8·b2 + 2^-16·b3, what is left scaled up each time (it is under 2^-7·|x|), so
// that nothing is lost at the lower end, against the quants with 2^0, 2^-8 and 2^-16; and d = 2^e · m, with 2^e on the
// quants (q · 2^e is a bf16 value) and m = 1 … 2, with d's sign, on the block's sum. ±inf, NaN, d = ±inf and NaN as the
// products q·d·x give them. (The matrix unit keeps subnormal bf16 operands and f32 sums.) The products and their order are
// those of the caller's own pass (q, d: the J weight rows; ko, kh: where the lane's first 8 k of a block start, and its
// other 8), so a row's results do not depend on the other rows. Straight from memory, a block at a time: 1023 × 1024 × 3072
// with a subnormal value (a SwiGLU output, say) in one row 35 → 105 µs, in every row 110
template <int J>
__device__ __forceinline__ void wide_blocks(const float *x, const int8_t *const (&q)[J], const _Float16 *const (&d)[J],
                                            int b0, int b1, int step, int ko, int kh, int al, f32x16 (&c)[J]) {
    typedef uint16_t ushort8 __attribute__((ext_vector_type(8)));
    struct Regs {
        float4 a[2][2];
        int2 q[J][2];
        _Float16 d[J];
    };
    auto gload = [&](int b) {
        Regs r;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int at = 32 * b + ko + h * kh;
            const float *xs = x + at;
            if (al) {
                r.a[h][0] = reinterpret_cast<const float4 *>(xs)[0];
                r.a[h][1] = reinterpret_cast<const float4 *>(xs)[1];
            } else {
                r.a[h][0] = make_float4(xs[0], xs[1], xs[2], xs[3]);
                r.a[h][1] = make_float4(xs[4], xs[5], xs[6], xs[7]);
            }
#pragma unroll
            for (int j = 0; j < J; j++) r.q[j][h] = *reinterpret_cast<const int2 *>(q[j] + at);
        }
#pragma unroll
        for (int j = 0; j < J; j++) r.d[j] = d[j][b];
        return r;
    };
#pragma unroll
    for (int j = 0; j < J; j++) c[j] = f32x16{};
#pragma unroll 1
    for (int b = b0; b < b1; b += step) {
        const Regs r = gload(b);
        f32x16 p[J] = {};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float4 u = r.a[h][0], v = r.a[h][1];
            const float xv[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
            uint32_t f[3][8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                f[0][e] = __float_as_uint(xv[e]);
                const float r1 = (xv[e] - __uint_as_float(f[0][e] & 0xffff0000u)) * 256.0f;
                const float r2 = (r1 - __uint_as_float(__float_as_uint(r1) & 0xffff0000u)) * 256.0f;
                const bool inf = fabsf(xv[e]) == INFINITY;  // inf − inf would make NaN of it
                f[1][e] = inf ? 0u : __float_as_uint(r1);
                f[2][e] = inf ? 0u : __float_as_uint(r2);
            }
#pragma unroll
            for (int j = 0; j < J; j++) {
                // 2^e of d (of 0: the smallest, m is 0)
                const float pow2 = fmaxf(__uint_as_float(__float_as_uint((float)r.d[j]) & 0x7f800000u), 0x1p-24f);
                uint32_t w[8];
#pragma unroll
                for (int e = 0; e < 8; e++) w[e] = __float_as_uint((float)q_byte(r.q[j][h], e) * pow2);
                const int4 w4 = hi_halves(w);
                ushort8 wb;
                __builtin_memcpy(&wb, &w4, 16);
#pragma unroll
                for (int pl = 0; pl < 3; pl++) {
                    // 8 off each exponent; a zero stays
                    if (pl) wb = __builtin_elementwise_sub_sat(wb, (ushort8)(uint16_t)(8 << 7));
                    const int4 a4 = hi_halves(f[pl]);
                    bf16x8 a, wp;
                    __builtin_memcpy(&a, &a4, 16);
                    __builtin_memcpy(&wp, &wb, 16);
                    p[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, wp, p[j], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < J; j++) {
            const float ds = (float)r.d[j];
            const float m = ds == 0.0f || ds != ds ? ds : __uint_as_float((__float_as_uint(ds) & 0x807fffffu) | 0x3f800000u);
#pragma unroll
            for (int i = 0; i < 16; i++) c[j][i] = fmaf(p[j][i], m, c[j][i]);
        }
    }
}

template <bool EX, int T, int KG> struct Q8Tile {
    static constexpr int BT = 64 * T, KB = EX ? 1 : 2, CPR = 4 * KB, PL = EX ? 3 : 1, R = 2;
    static constexpr int UN = T * KB;                                  // chunks a thread stages of X, and of W
    static constexpr int ACH = PL * BT * CPR, BUF = ACH + BT * CPR;    // 16-byte chunks: X's planes, a buffer
    static constexpr int LDS = 2 * KG * BUF;
    static_assert(KG == 1 || 2 * BUF * 16 >= BT * BT * 4, "a group's sums fit its buffers");
};

// al: X may be read in 16-byte units
template <bool EX, int T, int KG>
__global__ __launch_bounds__(256 * KG) void k_gemm_q8_0(const float *x, const int8_t *wq, const _Float16 *wd, float *y,
                                                        int m, int n, int k, int acc, int al, int tiles_m, int tiles_n) {
    using C = Q8Tile<EX, T, KG>;
    constexpr int KB = C::KB, CPR = C::CPR, R = C::R, UN = C::UN;
    __shared__ __attribute__((aligned(16))) int4 s_t[C::LDS];
    __shared__ float s_d[EX ? KG : 1][2][EX ? C::BT : 1];
    __shared__ int s_wide;
    const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8), tid = threadIdx.x & 255, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
    // workgroup b runs on XCD b mod 8: each XCD takes a contiguous band of tiles, walked 4 tile rows at a time, so the
    // workgroups of an XCD share X and W rows in its L2
    int tm, tn;
    {
        const int total = tiles_m * tiles_n, xcd = (int)blockIdx.x % 8, i = (int)blockIdx.x / 8;
        const int t = xcd * (total / 8) + min(xcd, total % 8) + i, gsz = 4 * tiles_n, g = t / gsz, gr = t % gsz;
        const int gm = min(4, tiles_m - 4 * g);
        tm = 4 * g + gr % gm;
        tn = gr / gm;
    }
    const int row0 = tm * C::BT, col0 = tn * C::BT, nb = k / 32, nst = (nb + KB - 1) / KB;
    int4 *buf0 = s_t + grp * 2 * C::BUF;

    // staging: chunk u = tid + 256·i of the stage is row u / CPR, k 8·(u % CPR) … + 7, of the X tile and of the W tile
    struct Regs {
        float4 a[UN][2];
        int2 q[UN];
        _Float16 d[UN];
    } ring[R];
    auto gload = [&](Regs &r, int st) {
#pragma unroll
        for (int i = 0; i < UN; i++) {
            const int u = tid + 256 * i, rr = u / CPR, c = u % CPR, b = min(st * KB + c / 4, nb - 1);
            const float *xs = x + (size_t)min(row0 + rr, m - 1) * k + 32 * b + 8 * (c & 3);
            if (al) {
                r.a[i][0] = reinterpret_cast<const float4 *>(xs)[0];
                r.a[i][1] = reinterpret_cast<const float4 *>(xs)[1];
            } else {
                r.a[i][0] = make_float4(xs[0], xs[1], xs[2], xs[3]);
                r.a[i][1] = make_float4(xs[4], xs[5], xs[6], xs[7]);
            }
            const size_t wr = min(col0 + rr, n - 1);
            r.q[i] = *reinterpret_cast<const int2 *>(wq + wr * k + 32 * b + 8 * (c & 3));
            r.d[i] = wd[wr * nb + b];
        }
    };
    Q8Seen seen;
    auto lstore = [&](const Regs &r, int st, int buf) {
        int4 *s = buf0 + buf * C::BUF;
#pragma unroll
        for (int i = 0; i < UN; i++) {
            const int u = tid + 256 * i, rr = u / CPR, c = u % CPR, at = q8_slot<CPR>(rr, c);
            const float4 a0 = r.a[i][0], a1 = r.a[i][1];
            float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
            float d = (float)r.d[i];
            if ((st + 1) * KB > nb) {  // only a stage that runs past the last block pays for the zeros
                const bool in = st * KB + c / 4 < nb;
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = in ? v[e] : 0.0f;
                d = in ? d : 0.0f;
            }
            if constexpr (EX) {
                int4 p[3];
                split3(v, p, seen);
                seen.add(d, 0.0f);
#pragma unroll
                for (int t = 0; t < 3; t++) s[t * C::BT * CPR + at] = p[t];
                uint32_t f[8];
#pragma unroll
                for (int e = 0; e < 8; e++) f[e] = __float_as_uint((float)q_byte(r.q[i], e));
                s[C::ACH + at] = hi_halves(f);
                if (c == 0) s_d[grp][buf][rr] = d;
            } else {
                half2_t hx[4], hw[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    hx[e] = __builtin_convertvector((float2_t{v[2 * e], v[2 * e + 1]}), half2_t);
                    hw[e] = __builtin_convertvector(
                        (float2_t{(float)q_byte(r.q[i], 2 * e) * d, (float)q_byte(r.q[i], 2 * e + 1) * d}), half2_t);
                }
                int4 px, pw;
                __builtin_memcpy(&px, hx, 16);
                __builtin_memcpy(&pw, hw, 16);
                s[at] = px;
                s[C::ACH + at] = pw;
            }
        }
    };
    f32x16 c[T][T];
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
        for (int j = 0; j < T; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) c[i][j][r] = 0.0f;
    const int fa = 32 * T * wm + (lane & 31), fb = 32 * T * wn + (lane & 31), hk = lane >> 5;
    auto compute = [&](int buf) {
        const int4 *s = buf0 + buf * C::BUF;
        if constexpr (EX) {
            f32x16 p[T][T];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                bf16x8 b[T];
#pragma unroll
                for (int j = 0; j < T; j++)
                    b[j] = *reinterpret_cast<const bf16x8 *>(s + C::ACH + q8_slot<CPR>(fb + 32 * j, 2 * h + hk));
#pragma unroll
                for (int pl = 0; pl < 3; pl++) {
                    bf16x8 a[T];
#pragma unroll
                    for (int i = 0; i < T; i++)
                        a[i] = *reinterpret_cast<const bf16x8 *>(s + pl * C::BT * CPR + q8_slot<CPR>(fa + 32 * i, 2 * h + hk));
#pragma unroll
                    for (int i = 0; i < T; i++)
#pragma unroll
                        for (int j = 0; j < T; j++)
                            p[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], h + pl ? p[i][j] : f32x16{}, 0, 0, 0);
                }
            }
#pragma unroll
            for (int j = 0; j < T; j++) {
                const float d = s_d[grp][buf][fb + 32 * j];
#pragma unroll
                for (int i = 0; i < T; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) c[i][j][r] = fmaf(p[i][j][r], d, c[i][j][r]);
            }
        } else {
#pragma unroll
            for (int h = 0; h < 2 * KB; h++) {
                half8 a[T], b[T];
#pragma unroll
                for (int i = 0; i < T; i++) a[i] = *reinterpret_cast<const half8 *>(s + q8_slot<CPR>(fa + 32 * i, 2 * h + hk));
#pragma unroll
                for (int j = 0; j < T; j++)
                    b[j] = *reinterpret_cast<const half8 *>(s + C::ACH + q8_slot<CPR>(fb + 32 * j, 2 * h + hk));
#pragma unroll
                for (int i = 0; i < T; i++)
#pragma unroll
                    for (int j = 0; j < T; j++) c[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], c[i][j], 0, 0, 0);
            }
        }
    };
    // the barrier between a buffer's stores and its reads: LDS accesses done, the register loads left in flight
    auto lds_barrier = [&] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // group grp's stage i is grp + KG·i; every group runs the same count (a stage past the last is zeros). Step i reads
    // buffer i % 2 while stage i + 1 is stored to the other, which step i − 1 read before the barrier that ended it
    const int steps = (nst + KG - 1) / KG;
    if (EX && threadIdx.x == 0) s_wide = 0;  // before the first barrier
#pragma unroll
    for (int r = 0; r < R; r++) gload(ring[r], grp + KG * r);
    lstore(ring[0], grp, 0);
    gload(ring[0], grp + KG * R);
    lds_barrier();
    for (int i0 = 0; i0 < steps; i0 += R) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i = i0 + r;
            if (i < steps) {
                compute(i & 1);
                if (i + 1 < steps) lstore(ring[(r + 1) % R], grp + KG * (i + 1), (i + 1) & 1);
                gload(ring[(r + 1) % R], grp + KG * (i + 1 + R));
                lds_barrier();
            }
        }
    }
    if constexpr (EX) {
        if (__builtin_amdgcn_ballot_w64(seen.wide()) && lane == 0) s_wide = 1;
        __syncthreads();
        if (__builtin_expect(s_wide, 0)) {
            const int8_t *qs[T];
            const _Float16 *ds[T];
#pragma unroll
            for (int j = 0; j < T; j++) {
                const size_t wr = min(col0 + fb + 32 * j, n - 1);
                qs[j] = wq + wr * k, ds[j] = wd + wr * nb;
            }
#pragma unroll
            for (int i = 0; i < T; i++)
                wide_blocks<T>(x + (size_t)min(row0 + fa + 32 * i, m - 1) * k, qs, ds, grp, nb, KG, 8 * hk, 16, al, c[i]);
        }
    }
    // lane ℓ, register r: row 8(r/4) + 4(ℓ/32) + r%4, column ℓ%32 of each 32 × 32 tile
    if constexpr (KG == 1) {
#pragma unroll
        for (int j = 0; j < T; j++) {
            const int col = col0 + fb + 32 * j;
#pragma unroll
            for (int i = 0; i < T; i++) {
                const int rbase = row0 + 32 * T * wm + 32 * i + 4 * hk;
                float old[16];
                if (acc) {  // every load before the first store, which may alias them
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        old[r] = y[(size_t)min(rbase + 8 * (r >> 2) + (r & 3), m - 1) * n + min(col, n - 1)];
                }
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int row = rbase + 8 * (r >> 2) + (r & 3);
                    if (row < m && col < n) y[(size_t)row * n + col] = acc ? old[r] + c[i][j][r] : c[i][j][r];
                }
            }
        }
    } else {
        // the groups' sums through their own (idle) buffers, added in group order
        constexpr int BT = C::BT, GS = 2 * C::BUF * 4;  // floats from a group's buffers to the next's
        float *s_o = reinterpret_cast<float *>(s_t);
#pragma unroll
        for (int i = 0; i < T; i++)
#pragma unroll
            for (int j = 0; j < T; j++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    s_o[grp * GS + (32 * T * wm + 32 * i + 8 * (r >> 2) + 4 * hk + (r & 3)) * BT + fb + 32 * j] = c[i][j][r];
        __syncthreads();
        constexpr int NE = BT * BT / (256 * KG);
        float old[NE];
        if (acc) {  // every load before the first store, which may alias them
#pragma unroll
            for (int e = 0; e < NE; e++) {
                const int o = threadIdx.x + 256 * KG * e;
                old[e] = y[(size_t)min(row0 + o / BT, m - 1) * n + min(col0 + o % BT, n - 1)];
            }
        }
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const int o = threadIdx.x + 256 * KG * e, row = row0 + o / BT, col = col0 + o % BT;
            float v = s_o[o];
#pragma unroll
            for (int g = 1; g < KG; g++) v += s_o[g * GS + o];
            if (row < m && col < n) y[(size_t)row * n + col] = acc ? old[e] + v : v;
        }
    }
}

// ---- few rows ----------------------------------------------------------------------------------------------------------
//
// The same products for at most 32 rows. The tiles above make a call of that size a chain of conversions and stage
// latencies on a handful of CUs (a 64 × 64 tile converts mostly rows that are not there); here a workgroup owns 32 columns
// and its 8 waves split K: each takes a contiguous run of q8_0 blocks straight from memory into MFMA fragments (no LDS, no
// barrier; 3 blocks of loads in flight), and the waves' sums are added in order through LDS. Inside a block lane half h
// takes k 16h … 16h + 15 for both MFMA steps (any order of k serves that X and W share), so a lane's quants are one 16-byte
// load and its X values one 64-byte run: 32 rows are 64 lines a load, which is what bounds it and why it stops at 32.
constexpr int FEW_WAVES = 8, FEW_R = 3;

template <bool EX>
__global__ __launch_bounds__(64 * FEW_WAVES) void k_gemm_q8_0_few(const float *x, const int8_t *wq, const _Float16 *wd,
                                                                  float *y, int m, int n, int k, int acc, int al) {
    __shared__ float s_o[FEW_WAVES][32][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col0 = blockIdx.x * 32, r32 = lane & 31, hk = lane >> 5, nb = k / 32;
    const int per = (nb + FEW_WAVES - 1) / FEW_WAVES, b0 = min(per * wave, nb), b1 = min(b0 + per, nb);
    const size_t wr = min(col0 + r32, n - 1);
    const int8_t *q = wq + wr * k + 16 * hk;
    const _Float16 *d = wd + wr * nb;
    const float *xr = x + (size_t)min(r32, m - 1) * k + 16 * hk;
    struct Regs {
        float4 a[4];
        int4 q;
        _Float16 d;
    } ring[FEW_R];
    auto gload = [&](Regs &r, int b) {
        b = max(min(b, b1 - 1), 0);
        const float *xs = xr + 32 * b;
#pragma unroll
        for (int i = 0; i < 4; i++)
            r.a[i] = al ? reinterpret_cast<const float4 *>(xs)[i]
                        : make_float4(xs[4 * i], xs[4 * i + 1], xs[4 * i + 2], xs[4 * i + 3]);
        r.q = *reinterpret_cast<const int4 *>(q + 32 * b);
        r.d = d[b];
    };
    f32x16 c = {};
    Q8Seen seen;
    auto use = [&](const Regs &r) {
        const int2 qs[2] = {make_int2(r.q.x, r.q.y), make_int2(r.q.z, r.q.w)};
        if constexpr (EX) {
            bf16x8 b[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                uint32_t f[8];
#pragma unroll
                for (int e = 0; e < 8; e++) f[e] = __float_as_uint((float)q_byte(qs[h], e));
                const int4 v = hi_halves(f);
                __builtin_memcpy(&b[h], &v, 16);
            }
            f32x16 p;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float4 u = r.a[2 * h], v = r.a[2 * h + 1];
                const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
                int4 a[3];
                split3(f, a, seen);
#pragma unroll
                for (int pl = 0; pl < 3; pl++) {
                    bf16x8 av;
                    __builtin_memcpy(&av, &a[pl], 16);
                    p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, b[h], h + pl ? p : f32x16{}, 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < 16; i++) c[i] = fmaf(p[i], (float)r.d, c[i]);
            seen.add((float)r.d, 0.0f);
        } else {
            const float ds = (float)r.d;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                half2_t w[4];
#pragma unroll
                for (int e = 0; e < 4; e++)
                    w[e] = __builtin_convertvector(
                        (float2_t{(float)q_byte(qs[h], 2 * e) * ds, (float)q_byte(qs[h], 2 * e + 1) * ds}), half2_t);
                half8 b;
                __builtin_memcpy(&b, w, 16);
                const float4 u = r.a[2 * h], v = r.a[2 * h + 1];
                const half2_t a4[4] = {__builtin_convertvector((float2_t{u.x, u.y}), half2_t),
                                       __builtin_convertvector((float2_t{u.z, u.w}), half2_t),
                                       __builtin_convertvector((float2_t{v.x, v.y}), half2_t),
                                       __builtin_convertvector((float2_t{v.z, v.w}), half2_t)};
                half8 a;
                __builtin_memcpy(&a, a4, 16);
                c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
            }
        }
    };
#pragma unroll
    for (int i = 0; i < FEW_R; i++) gload(ring[i], b0 + i);
    for (int i0 = b0; i0 < b1; i0 += FEW_R) {
#pragma unroll
        for (int i = 0; i < FEW_R; i++)
            if (i0 + i < b1) {
                use(ring[i]);
                gload(ring[i], i0 + i + FEW_R);
            }
    }
    if (EX && __builtin_expect(__builtin_amdgcn_ballot_w64(seen.wide()) != 0, 0)) {
        const int8_t *const qs[1] = {q};
        const _Float16 *const ds[1] = {d};
        f32x16 wide[1];
        wide_blocks<1>(xr, qs, ds, b0, b1, 1, 0, 8, al, wide);  // (xr and q start at the lane's half of a block)
        c = wide[0];
    }
    // lane ℓ, register r: row 8(r/4) + 4(ℓ/32) + r%4, column ℓ%32
#pragma unroll
    for (int i = 0; i < 16; i++) s_o[wave][8 * (i >> 2) + 4 * hk + (i & 3)][r32] = c[i];
    __syncthreads();
    constexpr int NE = 32 * 32 / (64 * FEW_WAVES);
    float old[NE];
    if (acc) {  // every load before the first store, which may alias them
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const int o = tid + 64 * FEW_WAVES * e;
            old[e] = y[(size_t)min(o / 32, m - 1) * n + min(col0 + o % 32, n - 1)];
        }
    }
#pragma unroll
    for (int e = 0; e < NE; e++) {
        const int o = tid + 64 * FEW_WAVES * e, row = o / 32, col = col0 + o % 32;
        float v = s_o[0][o / 32][o % 32];
#pragma unroll
        for (int g = 1; g < FEW_WAVES; g++) v += s_o[g][o / 32][o % 32];
        if (row < m && col < n) y[(size_t)row * n + col] = acc ? old[e] + v : v;
    }
}

// ---- the F32 path's K and V projections --------------------------------------------------------------------------------
//
// Y = X·Wᵀ with every output one chain of f32 fmas over k in order (matmul.wgsl:47-91), bit for bit: v_mfma_f32_16x16x4_f32
// adds its four products one after another, each rounded. K and V are rounded to f16 into the cache, where a last-bit
// difference of the f32 sum can move a value by an f16 ulp, which then stays in every later layer: with these two products
// in the reference's order the logits of a 1023-token prompt through 28 layers are 4.6e-5 from the f32 oracle's, with the
// exact block sums of k_gemm_q8_0 (which no order of f32 sums equals) 1.16e-4.
// A workgroup owns 32 × 64 outputs of one of the two matrices (grid z), 4 waves of 16 × 32; K in stages of two q8_0
// blocks, double-buffered in LDS as f32, their loads two stages ahead. A row's 32 values lie by k mod 4, then k / 4, so a
// lane's operands of the 8 MFMAs (k = 4s + its quarter) are two 16-byte chunks, placed at chunk ^ (row/2 % 8). Bound: the
// stages' latency at prompt sizes (333 × 2 · 1024 × 1024 28.7 µs a launch, 49 TFLOP/s; one block a stage 33.5 µs).
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct KvGemm {
    const int8_t *q[2];
    const _Float16 *d[2];
    float *y[2];
};

__global__ __launch_bounds__(256) void k_gemm_q8_0_chain(const float *x, const KvGemm w, int m, int n, int k) {
    constexpr int KB = 2;  // blocks a stage; a last odd one is followed by zeros (0·0 + c = c)
    __shared__ __attribute__((aligned(16))) float s_a[2][KB][32 * 32], s_b[2][KB][64 * 32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, row0 = blockIdx.y * 32, col0 = blockIdx.x * 64, nb = k / 32;
    // staging: k 8·lq … + 7 of both blocks of W row lr, and of one block (the thread's half) of X row lr % 32
    const int lr = tid >> 2, lq = tid & 3, ab = tid >> 7, ar = lr & 31;
    const float *xr = x + (size_t)min(row0 + ar, m - 1) * k + 8 * lq;
    const int8_t *wq = w.q[blockIdx.z] + (size_t)(col0 + lr) * k + 8 * lq;
    const _Float16 *wd = w.d[blockIdx.z] + (size_t)(col0 + lr) * nb;
    struct Regs {
        float4 a0, a1;
        int2 q[KB];
        _Float16 d[KB];
    };
    auto gload = [&](Regs &r, int st) {
        const float4 *xs = reinterpret_cast<const float4 *>(xr + 32 * min(KB * st + ab, nb - 1));
        r.a0 = xs[0];
        r.a1 = xs[1];
#pragma unroll
        for (int i = 0; i < KB; i++) {
            const int kb = min(KB * st + i, nb - 1);
            r.q[i] = *reinterpret_cast<const int2 *>(wq + 32 * kb);
            r.d[i] = wd[kb];
        }
    };
    // the float slot of (row r, quarter k mod 4 = t, k / 4 = 2·lq): the pair (2·lq, 2·lq + 1) is contiguous
    auto slot = [](int r, int t, int l) { return 32 * r + 4 * ((2 * t + (l >> 1)) ^ ((r >> 1) & 7)) + 2 * (l & 1); };
    auto lstore = [&](const Regs &r, int st) {
        const float a[8] = {r.a0.x, r.a0.y, r.a0.z, r.a0.w, r.a1.x, r.a1.y, r.a1.z, r.a1.w};
        const bool in = KB * st + ab < nb;
#pragma unroll
        for (int t = 0; t < 4; t++)
            *reinterpret_cast<float2 *>(&s_a[st & 1][ab][slot(ar, t, lq)]) = in ? make_float2(a[t], a[4 + t]) : make_float2(0.0f, 0.0f);
#pragma unroll
        for (int i = 0; i < KB; i++) {
            const float d = KB * st + i < nb ? (float)r.d[i] : 0.0f;
#pragma unroll
            for (int t = 0; t < 4; t++)
                *reinterpret_cast<float2 *>(&s_b[st & 1][i][slot(lr, t, lq)]) =
                    make_float2((float)q_byte(r.q[i], t) * d, (float)q_byte(r.q[i], 4 + t) * d);
        }
    };
    f32x4 c[2] = {f32x4{}, f32x4{}};
    const int fa = 16 * wm + (lane & 15), fb = 32 * wn + (lane & 15), t = lane >> 4;
    auto frag = [&](const float *s, int r, float (&f)[8]) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float4 v = *reinterpret_cast<const float4 *>(s + slot(r, t, 2 * h));
            f[4 * h] = v.x, f[4 * h + 1] = v.y, f[4 * h + 2] = v.z, f[4 * h + 3] = v.w;
        }
    };
    // LDS accesses done at the barrier, the next stages' register loads left in flight
    auto lds_barrier = [] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const int nst = (nb + KB - 1) / KB;
    Regs ring[2];
    gload(ring[0], 0);
    gload(ring[1], 1);
    lstore(ring[0], 0);
    gload(ring[0], 2);
    lds_barrier();
    for (int s0 = 0; s0 < nst; s0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int st = s0 + u;
            if (st >= nst) break;
            float a[KB][8], b[KB][2][8];
#pragma unroll
            for (int i = 0; i < KB; i++) {
                frag(s_a[u][i], fa, a[i]);
                frag(s_b[u][i], fb, b[i][0]);
                frag(s_b[u][i], fb + 16, b[i][1]);
            }
#pragma unroll
            for (int i = 0; i < KB; i++)
#pragma unroll
                for (int s = 0; s < 8; s++)
#pragma unroll
                    for (int j = 0; j < 2; j++) c[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][s], b[i][j][s], c[j], 0, 0, 0);
            if (st + 1 < nst) lstore(ring[u ^ 1], st + 1);
            gload(ring[u ^ 1], st + 3);
            lds_barrier();
        }
    }
    // lane ℓ, register r: row 4(ℓ/16) + r, column ℓ%16
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = row0 + 16 * wm + 4 * t + r;
            if (row < m) w.y[blockIdx.z][(size_t)row * n + col0 + 32 * wn + 16 * j + (lane & 15)] = c[j][r];
        }
}

// the f16 plane of a q8_0 weight: h = f16(q · d) (round to nearest even), 8 values a thread
__global__ __launch_bounds__(256) void k_q8_to_f16(const int8_t *q, const _Float16 *d, _Float16 *h, size_t n8,
                                                    int cols) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n8; i += (size_t)gridDim.x * 256) {
        const size_t e = 8 * i, r = e / cols, c = e % cols;
        const float s = (float)d[r * (cols / 32) + c / 32];
        const int2 v = *reinterpret_cast<const int2 *>(q + e);
        const uint32_t u[2] = {(uint32_t)v.x, (uint32_t)v.y};
        _Float16 o[8];
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] = (_Float16)((float)(int8_t)(u[j / 4] >> (8 * (j % 4))) * s);
        int4 out;
        __builtin_memcpy(&out, o, 16);
        *reinterpret_cast<int4 *>(h + e) = out;
    }
}

}  // namespace

int weight_attach_f16(htr_device *dev, hipStream_t st, htr_weight *w) {
    if (w->h) return 0;
    if (!w->q) return htr_fail("weight_attach_f16: the weight has no q8_0 planes");
    HTR_TRY(htr_dev_alloc(dev, w->rows * w->cols * 2, HTR_MEM_WEIGHTS, (void **)&w->h));
    const size_t n8 = w->rows * w->cols / 8;  // cols is a multiple of 32
    const int grid = (int)std::min<size_t>((n8 + 255) / 256, (size_t)dev->n_cu * 16);
    hipLaunchKernelGGL(k_q8_to_f16, dim3(grid), dim3(256), 0, st, w->q, w->d, w->h, n8, (int)w->cols);
    return htr_launched(dev, "k_q8_to_f16");
}

namespace {

template <bool EX, int T, int KG>
int launch_q8(htr_device *dev, hipStream_t st, const float *x, const htr_weight *w, float *y, int m, int acc) {
    const int n = (int)w->rows, bt = 64 * T, tm = (m + bt - 1) / bt, tn = (n + bt - 1) / bt;
    hipLaunchKernelGGL((k_gemm_q8_0<EX, T, KG>), dim3(tm * tn), dim3(256 * KG), 0, st, x, w->q, w->d, y, m, n,
                       (int)w->cols, acc, (int)((uintptr_t)x % 16 == 0), tm, tn);
    return 0;
}

template <bool EX> int gemm_q8(htr_device *dev, hipStream_t st, const float *x, const htr_weight *w, float *y, int m, int acc) {
    if (!w->q) return htr_fail("gemm: weight has no q8_0 planes");
    const int n = (int)w->rows;
    const long t128 = (long)((m + 127) / 128) * ((n + 127) / 128), t64 = (long)((m + 63) / 64) * ((n + 63) / 64);
    // few rows on one round of workgroups (µs a call, tiles → few; f16: 1 × 1024 × 1024 8.6 → 6.2, 8 × 1024 × 3072 17.4 →
    // 14.0, 12 × 1024 × 1024 8.7 → 8.0, 16 rows even, 24 8.7 → 9.8; F32: 1 × 1024 × 1024 11.3 → 6.4, 8 × 1024 × 3072 27.4 →
    // 14.6, 32 × 1024 × 2048 19.7 → 16.2; 16 × 16384 × 1024, two rounds: 9.7 → 16.2 and 13.1 → 16.4)
    if (m <= (EX ? 32 : 12) && (n + 31) / 32 <= dev->n_cu) {
        hipLaunchKernelGGL(k_gemm_q8_0_few<EX>, dim3((n + 31) / 32), dim3(64 * FEW_WAVES), 0, st, x, w->q, w->d, y, m, n,
                           (int)w->cols, acc, (int)((uintptr_t)x % 16 == 0));
        return htr_launched(dev, EX ? "k_gemm_q8_0_few<f32>" : "k_gemm_q8_0_few<f16>");
    }
    // 128 × 128 tiles from one a CU on; of the 64 × 64 ones, 4 K groups while every CU has a tile at most, else 2, whose
    // workgroups go two to a CU (288 tiles, 333 × 3072 × 1024: f16 18.5 → 14.2 µs, F32 24.1 → 21.8); 2 for a short K too,
    // where a group has a stage or two and the sum of four costs more than they save (4 → 2 groups, 100 × 1024: F32
    // K = 64 5.0 → 4.3, 256 6.1 → 6.0, 384 7.1 → 7.2; f16 K = 64 6.0 → 4.5, 512 6.9 → 6.3)
    if (t128 >= dev->n_cu) launch_q8<EX, 2, 1>(dev, st, x, w, y, m, acc);
    else if (t64 > dev->n_cu || w->cols <= (EX ? 256 : 512)) launch_q8<EX, 1, 2>(dev, st, x, w, y, m, acc);
    else launch_q8<EX, 1, 4>(dev, st, x, w, y, m, acc);
    return htr_launched(dev, EX ? "k_gemm_q8_0<f32>" : "k_gemm_q8_0<f16>");
}

}  // namespace

int launch_gemm_q8_0_f32(htr_device *dev, hipStream_t st, const float *x, const htr_weight *w, float *y, int m,
                         int acc) {
    return gemm_q8<true>(dev, st, x, w, y, m, acc);
}

int launch_gemm_q8_0_r16(htr_device *dev, hipStream_t st, const float *x, const htr_weight *w, float *y, int m,
                         int acc) {
    return gemm_q8<false>(dev, st, x, w, y, m, acc);
}

int launch_gemm_q8_0_kv(htr_device *dev, hipStream_t st, const float *x, const htr_weight *wk, const htr_weight *wv,
                        float *k, float *v, int m) {
    const int n = (int)wk->rows, cols = (int)wk->cols;
    if (!wk->q || !wv->q || wv->rows != wk->rows || wv->cols != wk->cols || n % 64 || cols % 32)
        return htr_fail("gemm_kv: K [%zu x %zu], V [%zu x %zu]: equal, rows a multiple of 64", wk->rows, wk->cols, wv->rows,
                        wv->cols);
    const KvGemm w = {{wk->q, wv->q}, {wk->d, wv->d}, {k, v}};
    hipLaunchKernelGGL(k_gemm_q8_0_chain, dim3(n / 64, (m + 31) / 32, 2), dim3(256), 0, st, x, w, m, n, cols);
    return htr_launched(dev, "k_gemm_q8_0_chain");
}

int launch_rms_norm(htr_device *dev, hipStream_t st, const float *x, const float *w, float *y, int rows, int dim,
                    float eps) {
    hipLaunchKernelGGL(k_rms_norm, dim3(rows), dim3(256), 0, st, x, w, y, dim, eps);
    return htr_launched(dev, "k_rms_norm");
}

int launch_swiglu(htr_device *dev, hipStream_t st, float *g, const float *u, size_t n) {
    const int grid = (int)std::min<size_t>((n + 255) / 256, 16384);
    hipLaunchKernelGGL(k_swiglu, dim3(grid), dim3(256), 0, st, g, u, n);
    return htr_launched(dev, "k_swiglu");
}

// ---- ABI ------------------------------------------------------------------------------------------------------------

extern "C" int htr_matmul_q8_0(htr_device *dev, const float *d_x, size_t m, const htr_weight *w, float *d_y, int acc) {
    HTR_TRY(htr_check_alive(dev));
    if (!d_x || !d_y || !w) return htr_fail("htr_matmul_q8_0: null argument");
    if (m == 0) return 0;
    if (m > (size_t)INT32_MAX / 2) return htr_fail("htr_matmul_q8_0: %zu rows", m);
    return dev->compute == HTR_COMPUTE_F32 ? launch_gemm_q8_0_f32(dev, dev->stream, d_x, w, d_y, (int)m, acc)
                                           : launch_gemm_q8_0_r16(dev, dev->stream, d_x, w, d_y, (int)m, acc);
}
