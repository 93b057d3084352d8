// Factored linear EMA (mathbrain/factored_ema.py:22-146) on gfx950, fp32-accurate.
//
// Per sequence b and head h the reference runs a per-step state recurrence
// (S_n <- rho_n S_n; o_t = sum_n (q_t ⊙ W_n)^T S_n; S_n += e_k[x_t] ⊗ e_v[x_t]), which is
// O(L N hd^2) and keeps an [N, hd, hd] state per (b, h).  Here the same output is split
// into two exact parts:
//
//   token part   o_t += sum_{s<t} A[t,s] e_v[x_s],  A[t,s] = sum_i q_t[i] e_k[x_s][i] G[t-s][i],
//                G[d] = sum_n rho_n^d W_n  (a [L+1, D] table, one small GEMM on the host side)
//                -> O(L^2 hd) pair work with no state at all (L < N hd at the model's shapes);
//   c_base part  o_t += sum_n rho_n^(t+1) sum_i q_t[i] W_n[i] S_n[i,:],
//                S_n = sum_k c_base[k,n] e_k[u_k] ⊗ e_v[u_k]  (the reference's initial state).
//
// The kernels: fac_outer (scaled outer-product accumulation, builds S_n and the backward's
// M_n = sum_t rho_n^(t+1) q_t ⊗ dO_t), fac_apply (contracts such a state with rows: the
// c_base part of o, of dQ and of the slot gradients), and the token-pair kernels: fac_tok_pair
// (o, and the token gradients of e_v), fac_tok_gate (dQ, and the token gradients of e_k) and
// fac_tok_dist (dG[d], from which dW_pe = P dG with P[n,d] = rho_n^d).
#include "flash_common.h"

namespace mb {
namespace {

__device__ inline int64_t clamp_row(const int64_t* idx, int64_t e, int64_t nrows) {
    int64_t r = idx ? idx[e] : e;
    r = r < 0 ? 0 : r;
    return r < nrows ? r : -1;
}

// out[b,h,n,i,j] = sum_r alpha[b,r,n] X[row_x(b,r), h*HD+i] Y[row_y(b,r), h*HD+j].
// Block (n block, h, b); thread (n, i) with 256/HD rates per block; the Y row of each r is
// the same for the whole block.
template <int HD>
__global__ void __launch_bounds__(256)
fac_outer_kernel(const float* __restrict__ X, const int64_t* __restrict__ xrow,
                 const float* __restrict__ Y, const int64_t* __restrict__ yrow, int64_t ld,
                 int64_t nrows, const float* __restrict__ alpha, int64_t as_b, int64_t as_r,
                 int64_t as_n, int R, int H, int N, float* __restrict__ out) {
    constexpr int NB = 256 / HD;
    const int b = blockIdx.z, h = blockIdx.y;
    const int n = blockIdx.x * NB + threadIdx.x / HD;
    const int i = threadIdx.x % HD;
    const bool nok = n < N;
    float acc[HD];
#pragma unroll
    for (int j = 0; j < HD; ++j) acc[j] = 0.0f;
    for (int r = 0; r < R; ++r) {
        const float a = nok ? alpha[b * as_b + r * as_r + n * as_n] : 0.0f;
        if (a == 0.0f) continue;
        const int64_t e = (int64_t)b * R + r;
        const int64_t rx = clamp_row(xrow, e, nrows), ry = clamp_row(yrow, e, nrows);
        if (rx < 0 || ry < 0) continue;
        const float av = a * X[rx * ld + h * HD + i];
        const float* yr = Y + ry * ld + h * HD;
#pragma unroll
        for (int j = 0; j < HD; ++j) acc[j] = __builtin_fmaf(av, yr[j], acc[j]);
    }
    if (nok) {
        float* o = out + ((((int64_t)b * H + h) * N + n) * HD + i) * HD;
#pragma unroll
        for (int j = 0; j < HD; ++j) o[j] = acc[j];
    }
}

// TRANS = false: out[b,r,h,i] (+)= sum_n alpha[b,r,n] sum_j w[n,i] M[b,h,n,i,j] Y[row(b,r),h,j]
// TRANS = true:  out[b,r,h,j] (+)= sum_n alpha[b,r,n] sum_i w[n,i] M[b,h,n,i,j] Y[row(b,r),h,i]
// (w NULL: 1).  A register-tiled GEMM per rate: block (kApplyRows rows, h, b), 16 x 16 threads
// each owning kApplyRows/16 rows x HD/16 outputs; the Y rows and the rows' alphas are staged
// once, the (scaled, oriented) M_n tile once per rate, with the next rate's tile loaded into
// registers while the current one is used.
constexpr int kApplyRows = 128;

template <int HD, bool TRANS>
__global__ void __launch_bounds__(256)
fac_apply_kernel(const float* __restrict__ M, const float* __restrict__ w, int64_t ldw,
                 const float* __restrict__ Y, const int64_t* __restrict__ yrow, int64_t ld,
                 int64_t nrows, const float* __restrict__ alpha, int64_t as_b, int64_t as_r,
                 int64_t as_n, int R, int H, int N, float* __restrict__ out, int64_t ldo,
                 int accumulate) {
    constexpr int RS = HD + 4;              // LDS row stride (floats)
    constexpr int CO = HD / 16;             // outputs per thread
    constexpr int RO = kApplyRows / 16;     // rows per thread
    constexpr int AN = 16;                  // rates whose alphas are staged at a time
    constexpr int ME = HD * HD / 256;       // M_n elements per thread
    __shared__ __align__(16) float Ys[kApplyRows * RS];
    __shared__ __align__(16) float Mt[HD * RS];
    __shared__ float As[kApplyRows * AN];
    const int b = blockIdx.z, h = blockIdx.y;
    const int r0 = blockIdx.x * kApplyRows;
    const int tid = threadIdx.x;
    const int tr = tid / 16, to = tid % 16;
    for (int e = tid; e < kApplyRows * (HD / 4); e += 256) {
        const int rr = e / (HD / 4), c = e % (HD / 4);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r0 + rr < R) {
            const int64_t ry = clamp_row(yrow, (int64_t)b * R + r0 + rr, nrows);
            if (ry >= 0) v = *reinterpret_cast<const float4*>(Y + ry * ld + h * HD + 4 * c);
        }
        *reinterpret_cast<float4*>(Ys + rr * RS + 4 * c) = v;
    }
    const float* Mb = M + ((int64_t)b * H + h) * N * HD * HD;
    float mreg[ME];
    auto load_m = [&](int n) {
#pragma unroll
        for (int q = 0; q < ME; ++q) {
            const int e = tid + 256 * q;
            float v = Mb[(int64_t)n * HD * HD + e];
            if (w) v *= w[n * ldw + h * HD + e / HD];
            mreg[q] = v;
        }
    };
    load_m(0);
    float acc[RO][CO];
#pragma unroll
    for (int a = 0; a < RO; ++a)
#pragma unroll
        for (int c = 0; c < CO; ++c) acc[a][c] = 0.0f;
    for (int n = 0; n < N; ++n) {
        __syncthreads();
        if (n % AN == 0) {
            for (int e = tid; e < kApplyRows * AN; e += 256) {
                const int rr = e / AN, nn = n + e % AN;
                As[e] = (r0 + rr < R && nn < N)
                            ? alpha[b * as_b + (int64_t)(r0 + rr) * as_r + nn * as_n] : 0.0f;
            }
        }
#pragma unroll
        for (int q = 0; q < ME; ++q) {
            const int e = tid + 256 * q;
            const int i = e / HD, j = e % HD;
            if (TRANS) Mt[j * RS + i] = mreg[q];
            else Mt[i * RS + j] = mreg[q];
        }
        __syncthreads();
        if (n + 1 < N) load_m(n + 1);
        float sacc[RO][CO];
#pragma unroll
        for (int a = 0; a < RO; ++a)
#pragma unroll
            for (int c = 0; c < CO; ++c) sacc[a][c] = 0.0f;
#pragma unroll 2
        for (int k0 = 0; k0 < HD; k0 += 4) {
            float4 mv[CO];
#pragma unroll
            for (int c = 0; c < CO; ++c) mv[c] = *reinterpret_cast<const float4*>(Mt + (to * CO + c) * RS + k0);
#pragma unroll
            for (int a = 0; a < RO; ++a) {
                const float4 yv = *reinterpret_cast<const float4*>(Ys + (tr * RO + a) * RS + k0);
#pragma unroll
                for (int c = 0; c < CO; ++c) {
                    float t = sacc[a][c];
                    t = __builtin_fmaf(yv.x, mv[c].x, t);
                    t = __builtin_fmaf(yv.y, mv[c].y, t);
                    t = __builtin_fmaf(yv.z, mv[c].z, t);
                    t = __builtin_fmaf(yv.w, mv[c].w, t);
                    sacc[a][c] = t;
                }
            }
        }
#pragma unroll
        for (int a = 0; a < RO; ++a) {
            const float al = As[(tr * RO + a) * AN + n % AN];
#pragma unroll
            for (int c = 0; c < CO; ++c) acc[a][c] = __builtin_fmaf(al, sacc[a][c], acc[a][c]);
        }
    }
#pragma unroll
    for (int a = 0; a < RO; ++a) {
        const int r = r0 + tr * RO + a;
        if (r >= R) continue;
        float* dst = out + ((int64_t)b * R + r) * ldo + h * HD + to * CO;
#pragma unroll
        for (int c = 0; c < CO; ++c) dst[c] = accumulate ? dst[c] + acc[a][c] : acc[a][c];
    }
}

// ---- MFMA forms of the state kernels (hd = 64) ------------------------------------------
//
// The state contractions are plain GEMMs per rate.  These forms run them on the bf16 matrix
// cores with every fp32 operand split into bf16 hi + lo parts and three products
// (hi*hi + hi*lo + lo*hi, fp32 accumulation), which keeps about 2^-16 relative error per
// product.  Operand layout of v_mfma_f32_16x16x32_bf16: A[row = lane%16][k = 8 (lane/16) + e],
// B[k = 8 (lane/16) + e][col = lane%16], D[row = 4 (lane/16) + i][col = lane%16].
// Bound: the matrix cores, provided that an operand is split once per workgroup and not once per
// wave, and that the loads run a tile ahead.  B56 T512 H8 N64 with a history of 4 096 tokens,
// forward + backward: fac_outer 3.00 -> 1.70 ms, fac_apply 5.34 -> 3.17 ms against four waves
// that each split their own tiles, unprefetched, for the half-rate 16x16x16 form.

constexpr int kStateDim = 64;
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ inline void split_bf16x8(const float (&v)[8], bf16x8& hi, bf16x8& lo) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const __bf16 t = (__bf16)v[e];
        hi[e] = t;
        lo[e] = (__bf16)(v[e] - (float)t);
    }
}

__device__ inline f32x4 mfma3(bf16x8 ah, bf16x8 al, bf16x8 bh, bf16x8 bl, f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, c, 0, 0, 0);
}

// Workgroup id -> (block r < nr, head bh = b H + h).  The nr blocks of a head read the same
// tiles: where the heads divide among the 8 XCDs (ids go to them round-robin), they share one
// XCD's L2.
struct HeadBlock {
    int r, bh;
};
__device__ inline HeadBlock head_block(int id, int nr, int heads) {
    if (heads % 8) return HeadBlock{id % nr, id / nr};
    const int k = id >> 3;
    return HeadBlock{k % nr, (k / nr) * 8 + (id & 7)};
}

// fac_apply_kernel for hd = 64: 128 rows of a head, 8 waves of 32 rows x 32 outputs.  The Y rows
// are split once; a rate's scaled and oriented M_n is split once for the workgroup, into one of
// two LDS buffers, while the next rate's is on its way.
constexpr int kStateRows = 128;

template <bool TRANS>
__global__ void __launch_bounds__(512, 4)
fac_apply_mfma_kernel(const float* __restrict__ M, const float* __restrict__ w, int64_t ldw,
                      const float* __restrict__ Y, const int64_t* __restrict__ yrow, int64_t ld,
                      int64_t nrows, const float* __restrict__ alpha, int64_t as_b, int64_t as_r,
                      int64_t as_n, int B, int R, int H, int N, float* __restrict__ out, int64_t ldo,
                      int accumulate) {
    constexpr int HD = kStateDim;
    constexpr int AN = 64;               // rates whose alphas are staged at once
    constexpr int AS = kStateRows + 4;   // floats per rate
    constexpr int MS = HD + 8;           // bf16 per output column: 16-byte reads on all banks
    __shared__ __align__(16) float As[AN * AS];
    __shared__ __align__(16) __bf16 Mt[2][2][HD * MS];  // [buffer][hi, lo][output][k]
    const int nr = (R + kStateRows - 1) / kStateRows;
    const HeadBlock hb = head_block(blockIdx.x, nr, B * H);
    const int b = hb.bh / H, h = hb.bh % H;
    const int r0 = hb.r * kStateRows;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c16 = lane & 15, g = lane >> 4;
    const int rw = 32 * (wave & 3), cw = 32 * (wave >> 2);
    bf16x8 ahi[2][2], alo[2][2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const int r = r0 + rw + 16 * rt + c16;
        const int64_t ry = r < R ? clamp_row(yrow, (int64_t)b * R + r, nrows) : -1;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (ry >= 0) {
                const float* p = Y + ry * ld + h * HD + 32 * ks + 8 * g;
                const f32x4u q0 = *reinterpret_cast<const f32x4u*>(p), q1 = *reinterpret_cast<const f32x4u*>(p + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) { v[e] = q0[e]; v[4 + e] = q1[e]; }
            }
            split_bf16x8(v, ahi[rt][ks], alo[rt][ks]);
        }
    }
    // this thread's part of a tile: output column mo, k = mk .. mk + 7
    const int mo = TRANS ? lane : tid >> 3, mk = 8 * (TRANS ? wave : tid & 7);
    const float* Mb = M + (int64_t)hb.bh * N * HD * HD;
    const float* wh = w ? w + h * HD : nullptr;
    float m[8], ms[8];
    auto load_tile = [&](int n) {
        const float* Mn = Mb + (int64_t)n * HD * HD;
        if (!TRANS) {  // B[k][o] = w[n, o] M_n[o][k]
            const f32x4 q0 = *reinterpret_cast<const f32x4*>(Mn + mo * HD + mk);
            const f32x4 q1 = *reinterpret_cast<const f32x4*>(Mn + mo * HD + mk + 4);
            ms[0] = wh ? wh[n * ldw + mo] : 1.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) { m[e] = q0[e]; m[4 + e] = q1[e]; }
        } else {       // B[k][o] = w[n, k] M_n[k][o]
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                m[e] = Mn[(mk + e) * HD + mo];
                ms[e] = wh ? wh[n * ldw + mk + e] : 1.0f;
            }
        }
    };
    f32x4 acc[2][2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) acc[rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    load_tile(0);
    for (int n = 0; n < N; ++n) {
        if (n % AN == 0) {
            __syncthreads();
            for (int e = tid; e < kStateRows * AN; e += 512) {
                const int rr = e / AN, nn = e % AN;
                As[nn * AS + rr] = (r0 + rr < R && n + nn < N)
                                       ? alpha[b * as_b + (int64_t)(r0 + rr) * as_r + (n + nn) * as_n] : 0.0f;
            }
        }
        __bf16* buf = Mt[n & 1][0];
        {
            float v[8];
            bf16x8 hi, lo;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = m[e] * ms[TRANS ? e : 0];
            split_bf16x8(v, hi, lo);
            *reinterpret_cast<bf16x8*>(buf + mo * MS + mk) = hi;
            *reinterpret_cast<bf16x8*>(buf + HD * MS + mo * MS + mk) = lo;
        }
        if (n + 1 < N) load_tile(n + 1);
        __syncthreads();
        f32x4 s[2][2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) s[rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const __bf16* p = buf + (cw + 16 * ct + c16) * MS + 32 * ks + 8 * g;
                const bf16x8 bh = *reinterpret_cast<const bf16x8*>(p);
                const bf16x8 bl = *reinterpret_cast<const bf16x8*>(p + HD * MS);
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) s[rt][ct] = mfma3(ahi[rt][ks], alo[rt][ks], bh, bl, s[rt][ct]);
            }
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const f32x4 al = *reinterpret_cast<const f32x4*>(As + (n % AN) * AS + rw + 16 * rt + 4 * g);
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[rt][ct][i] = __builtin_fmaf(al[i], s[rt][ct][i], acc[rt][ct][i]);
        }
    }
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + rw + 16 * rt + 4 * g + i;
            if (r >= R) continue;
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
                float* dst = out + ((int64_t)b * R + r) * ldo + h * HD + cw + 16 * ct + c16;
                *dst = accumulate ? *dst + acc[rt][ct][i] : acc[rt][ct][i];
            }
        }
}

// fac_outer_kernel for hd = 64: 8 rates of a head, two per wave, each the whole 64 x 64 output of
// its rate in 16 tiles.  The walked rows come in blocks of 32 (one MFMA k step), staged with the
// row as the fast index: X in fp32 (each rate weights it before the split), Y split.  Two rates
// to a wave halve the LDS reads per product (one rate: 18 of 16 bytes per 48; two: 20 per 96).
constexpr int kOuterRows = 32;
constexpr int kOuterRates = 8;

__global__ void __launch_bounds__(256, 2)
fac_outer_mfma_kernel(const float* __restrict__ X, const int64_t* __restrict__ xrow,
                      const float* __restrict__ Y, const int64_t* __restrict__ yrow, int64_t ld,
                      int64_t nrows, const float* __restrict__ alpha, int64_t as_b, int64_t as_r,
                      int64_t as_n, int B, int R, int H, int N, float* __restrict__ out) {
    constexpr int HD = kStateDim;
    constexpr int XS = kOuterRows + 4;  // floats per dimension
    constexpr int YS = kOuterRows + 8;  // bf16 per dimension
    __shared__ __align__(16) float Xs[2][HD * XS], As[2][kOuterRates * XS];
    __shared__ __align__(16) __bf16 Ys[2][2][HD * YS];  // [buffer][hi, lo]
    const int nr = (N + kOuterRates - 1) / kOuterRates;
    const HeadBlock hb = head_block(blockIdx.x, nr, B * H);
    const int b = hb.bh / H, h = hb.bh % H;
    const int n0 = hb.r * kOuterRates;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c16 = lane & 15, g = lane >> 4;
    // staged by this thread: rows 2 sp, 2 sp + 1 of dimensions sc .. sc + 3, and one alpha
    const int sp = (tid >> 2) & 15, sc = 4 * ((tid & 3) + 4 * wave);
    const int an = tid & (kOuterRates - 1), ar = tid / kOuterRates;
    int64_t rx[2], ry[2];
    f32x4 vx[2], vy[2];
    float va;
    auto load_ids = [&](int k0) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int r = k0 + 2 * sp + e;
            const int64_t ex = (int64_t)b * R + r;
            rx[e] = r < R ? clamp_row(xrow, ex, nrows) : -1;
            ry[e] = r < R ? clamp_row(yrow, ex, nrows) : -1;
        }
    };
    auto load_rows = [&](int k0) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const bool ok = rx[e] >= 0 && ry[e] >= 0;
            vx[e] = ok ? f32x4(*reinterpret_cast<const f32x4u*>(X + rx[e] * ld + h * HD + sc)) : f32x4{0.f, 0.f, 0.f, 0.f};
            vy[e] = ok ? f32x4(*reinterpret_cast<const f32x4u*>(Y + ry[e] * ld + h * HD + sc)) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const int r = k0 + ar, n = n0 + an;
        va = r < R && n < N ? alpha[b * as_b + (int64_t)r * as_r + n * as_n] : 0.0f;
    };
    f32x4 acc[2][4][4];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int it = 0; it < 4; ++it)
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) acc[q][it][jt] = f32x4{0.f, 0.f, 0.f, 0.f};
    load_ids(0);
    load_rows(0);
    load_ids(kOuterRows);
    for (int k0 = 0, buf = 0; k0 < R; k0 += kOuterRows, buf ^= 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            *reinterpret_cast<float2*>(Xs[buf] + (sc + e) * XS + 2 * sp) = make_float2(vx[0][e], vx[1][e]);
            __bf16 hi[2], lo[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                hi[q] = (__bf16)vy[q][e];
                lo[q] = (__bf16)(vy[q][e] - (float)hi[q]);
            }
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            *reinterpret_cast<bf16x2*>(Ys[buf][0] + (sc + e) * YS + 2 * sp) = bf16x2{hi[0], hi[1]};
            *reinterpret_cast<bf16x2*>(Ys[buf][1] + (sc + e) * YS + 2 * sp) = bf16x2{lo[0], lo[1]};
        }
        As[buf][an * XS + ar] = va;
        if (k0 + kOuterRows < R) {
            load_rows(k0 + kOuterRows);
            load_ids(k0 + 2 * kOuterRows);
        }
        __syncthreads();
        float al[2][8];
        bool any = false;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float* p = As[buf] + (2 * wave + q) * XS + 8 * g;
            const f32x4 t0 = *reinterpret_cast<const f32x4*>(p), t1 = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                al[q][e] = t0[e];
                al[q][4 + e] = t1[e];
                any = any || t0[e] != 0.0f || t1[e] != 0.0f;
            }
        }
        if (!__any(any)) continue;
        bf16x8 bh[4], bl[4];
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) {
            bh[jt] = *reinterpret_cast<const bf16x8*>(Ys[buf][0] + (16 * jt + c16) * YS + 8 * g);
            bl[jt] = *reinterpret_cast<const bf16x8*>(Ys[buf][1] + (16 * jt + c16) * YS + 8 * g);
        }
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const float* p = Xs[buf] + (16 * it + c16) * XS + 8 * g;
            const f32x4 t0 = *reinterpret_cast<const f32x4*>(p), t1 = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float v[8];
                bf16x8 ah, alo;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = al[q][e] * t0[e];
                    v[4 + e] = al[q][4 + e] * t1[e];
                }
                split_bf16x8(v, ah, alo);
#pragma unroll
                for (int jt = 0; jt < 4; ++jt) acc[q][it][jt] = mfma3(ah, alo, bh[jt], bl[jt], acc[q][it][jt]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int n = n0 + 2 * wave + q;
        if (n >= N) continue;
        float* o = out + ((int64_t)hb.bh * N + n) * HD * HD;
#pragma unroll
        for (int it = 0; it < 4; ++it)
#pragma unroll
            for (int jt = 0; jt < 4; ++jt)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[(16 * it + 4 * g + i) * HD + 16 * jt + c16] = acc[q][it][jt][i];
    }
}

__device__ inline bool tok_ok(int64_t v, int64_t V) { return v >= 0 && v < V; }

// ---- token pairs ---------------------------------------------------------------------------
//
// A block of 4 waves covers 64 steps (the "rows") of one (b, h) and walks the 64-step blocks of
// the other index (the "walked" steps); wave w has rows 16 w .. 16 w + 15.  What a 64 x 64 tile
// of pairs needs is one of two forms:
//
//   sums over the dimensions of a product of three rows, A[t,s] = sum_i q_t[i] e_k[x_s][i]
//   G[t-s][i]: a thread takes 4 x 4 pairs and walks the dimensions, whose rows are staged with
//   the dimension as the slow index; the 4 x 4 pairs have 7 distances, 8 consecutive floats;
//
//   sums over the walked steps of dA[r,w] y_w ⊙ G[d]: a thread takes 4 rows x 4 dimensions (2 x 4
//   at head_dim 32) and walks the steps; its rows' distances move by one per step, so a step
//   reads one new row of G.
//
// The products without G (A e_v, dO e_v^T, A^T dO) go to the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32: A[row = lane % 16][k = lane / 16], B[k = lane / 16][col = lane % 16],
// D[row = 4 (lane / 16) + i][col = lane % 16]).  Bound: VALU issue, two operations per pair and
// dimension (A in the forward and for dE_v, dQ, dE_k and dG: 10 in all), and next to it the LDS
// reads, 3 or 4 of 16 bytes per 32 operations.  Lanes as steps with whole rows in registers
// instead read G from LDS for every pair and dimension, and the other rows once per wave.
// B56 T512 H8 head_dim 64, forward + backward: 9.4 -> 3.5 ms (o 0.73, dE_v 0.64, dQ 0.63,
// dE_k 0.66, dG 0.84); B5 T253 H4 head_dim 32, the whole call: 1.76 -> 1.60 ms.

constexpr int kTokB = 64;  // steps per block

// Rows of one head: of a [L, D] slice (ids NULL), or E[x[r]] of a table; rows outside [0, L) and
// ids outside [0, V) read as zeros.  Their address is another row's and the zeros are selected
// after the load: a load under a condition is issued alone, and its id before it (the kernels of
// a forward and backward at B56 T512 took 4.34 ms so, 3.91 with a tile's loads in flight together).
struct TokRows {
    const float* p;
    const int64_t* ids;
    int64_t V, D;
    int L;
    __device__ inline int64_t id(int r) const {
        const int64_t v = min(max(r, 0), L - 1);
        return ids ? ids[v] : v;
    }
    __device__ inline const float* at(int64_t v, int r, bool& ok) const {  // v = id(r)
        ok = r >= 0 && r < L;
        if (ids) {
            ok = ok && tok_ok(v, V);
            v = tok_ok(v, V) ? v : 0;
        }
        return p + v * D;
    }
    __device__ inline const float* row(int r, bool& ok) const { return at(id(r), r, ok); }
};

__device__ inline f32x4 load4(const float* p, int c, bool ok) {
    const f32x4 v = *reinterpret_cast<const f32x4u*>(p + c);
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = ok ? v[e] : 0.f;
    return o;
}

// A thread's part of dimensions k0 .. k0 + KC - 1 of rows lo .. lo + ROWS - 1, stored to dst[k][r] (RS
// floats per dimension).  Four lanes on 64 bytes of a row and 16 rows per wave: the transposed
// writes use every bank twice.
template <int ROWS, int KC, int RS>
struct DimPiece {
    static constexpr int RT = ROWS / 16, NV = RT * (KC / 16) / 4;
    f32x4 v[NV];
    __device__ static inline int row(int q) {
        return ((4 * q + (threadIdx.x >> 6)) % RT) * 16 + ((threadIdx.x >> 2) & 15);
    }
    __device__ static inline int dim(int q) {
        return ((4 * q + (threadIdx.x >> 6)) / RT) * 16 + 4 * (threadIdx.x & 3);
    }
    __device__ inline void load(const TokRows& src, int lo, int k0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            bool ok;
            const float* p = src.row(lo + row(q), ok);
            v[q] = load4(p, k0 + dim(q), ok);
        }
    }
    __device__ inline void store(float* dst) const {
#pragma unroll
        for (int q = 0; q < NV; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) dst[(dim(q) + e) * RS + row(q)] = v[q][e];
    }
};

// A thread's part of rows lo .. lo + ROWS - 1: their ids, the loads, and the store to dst[r][i] (RS
// floats per row).  The three are apart so that a tile's ids and rows are on their way while the
// tile before it is computed (3.9 -> 3.5 ms).
template <int ROWS, int HD, int RS>
struct RowPiece {
    static constexpr int C4 = HD / 4, NV = ROWS * C4 / 256, STEP = 256 / C4;
    int64_t id[NV];
    f32x4 v[NV];
    __device__ inline void ids(const TokRows& src, int lo) {
#pragma unroll
        for (int q = 0; q < NV; ++q) id[q] = src.id(lo + threadIdx.x / C4 + q * STEP);
    }
    __device__ inline void load(const TokRows& src, int lo) {
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            bool ok;
            const float* p = src.at(id[q], lo + threadIdx.x / C4 + q * STEP, ok);
            v[q] = load4(p, 4 * (threadIdx.x % C4), ok);
        }
    }
    __device__ inline void store(float* dst) const {
#pragma unroll
        for (int q = 0; q < NV; ++q)
            *reinterpret_cast<f32x4*>(dst + (threadIdx.x / C4 + q * STEP) * RS + 4 * (threadIdx.x % C4)) = v[q];
    }
};

// out[r] = sum_w A(r, w) Z[w], A(r, w) = sum_i X[r][i] Y[w][i] G[d][i].  FWD: rows are steps t
// and the walked ones s < t (O); otherwise rows are steps s and the walked ones t > s (dE_v).
template <int HD, bool FWD>
__global__ void __launch_bounds__(256, 2)
fac_tok_pair_kernel(const float* __restrict__ Q, const float* __restrict__ dO, const int64_t* __restrict__ x,
                    int64_t V, const float* __restrict__ Ek, const float* __restrict__ Ev,
                    const float* __restrict__ G, int L, int H, float* __restrict__ out) {
    constexpr int KC = 32;        // dimensions per staged piece of Y and G
    constexpr int RS = kTokB + 4;   // floats per dimension of 64 rows, and of an A row
    constexpr int GS = 2 * kTokB + 4;
    constexpr int ZS = HD + 16;   // the four k groups of an operand read on different banks
    __shared__ __align__(16) float Xs[HD * RS], Ys[KC * RS], Gs[KC * GS], As[kTokB * RS], Zs[kTokB * ZS];
    const int64_t D = (int64_t)H * HD;
    const int b = blockIdx.z, h = blockIdx.y, nb = gridDim.x;
    const int rb = FWD ? nb - 1 - (int)blockIdx.x : (int)blockIdx.x;  // most walked blocks first
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ty = tid >> 4, tx = tid & 15;
    const int c16 = lane & 15, g = lane >> 4;
    const int64_t* xb = x + (int64_t)b * L;
    const int64_t slice = (int64_t)b * L * D + h * HD;
    const TokRows q{Q + slice, nullptr, 0, D, L}, ek{Ek + h * HD, xb, V, D, L};
    const TokRows z = FWD ? TokRows{Ev + h * HD, xb, V, D, L} : TokRows{dO + slice, nullptr, 0, D, L};
    const TokRows gt{G + h * HD, nullptr, 0, D, L + 1};
    const TokRows xr = FWD ? q : ek, yr = FWD ? ek : q;
    f32x4 acc[HD / 16];
#pragma unroll
    for (int j = 0; j < HD / 16; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    {
        DimPiece<kTokB, HD, RS> px;
        px.load(xr, rb * kTokB, 0);
        px.store(Xs);
    }
    const float* gbase = Gs + (FWD ? 4 * (ty - tx) : 4 * (tx - ty)) + 60;
    const int w_lo = FWD ? 0 : rb, w_hi = FWD ? rb : nb - 1;
    DimPiece<kTokB, KC, RS> py;
    DimPiece<2 * kTokB, KC, GS> pg;
    RowPiece<kTokB, HD, ZS> pz;
    auto load = [&](int wb, int kc) {
        py.load(yr, wb * kTokB, kc);
        pg.load(gt, (FWD ? rb - wb : wb - rb) * kTokB - (kTokB - 1), kc);
        if (kc == 0) {
            pz.ids(z, wb * kTokB);
            pz.load(z, wb * kTokB);
        }
    };
    load(w_lo, 0);
    for (int wb = w_lo; wb <= w_hi; ++wb) {
        float a[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) a[i][j] = 0.f;
#pragma unroll
        for (int kc = 0; kc < HD; kc += KC) {
            __syncthreads();
            py.store(Ys);
            pg.store(Gs);
            if (kc == 0) pz.store(Zs);
            if (kc + KC < HD) load(wb, kc + KC);
            else load(min(wb + 1, w_hi), 0);
            __syncthreads();
#pragma unroll 4
            for (int k = 0; k < KC; ++k) {
                const f32x4 xv = *reinterpret_cast<const f32x4*>(Xs + (kc + k) * RS + 4 * ty);
                const f32x4 yv = *reinterpret_cast<const f32x4*>(Ys + k * RS + 4 * tx);
                const f32x4 g0 = *reinterpret_cast<const f32x4*>(gbase + k * GS);
                const f32x4 g1 = *reinterpret_cast<const f32x4*>(gbase + k * GS + 4);
                const float gg[8] = {g0[0], g0[1], g0[2], g0[3], g1[0], g1[1], g1[2], g1[3]};
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        a[i][j] = __builtin_fmaf(xv[i] * yv[j], gg[(FWD ? i - j : j - i) + 3], a[i][j]);
            }
        }
        if (wb == rb || wb == nb - 1) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = rb * kTokB + 4 * ty + i, w = wb * kTokB + 4 * tx + j;
                    a[i][j] = (FWD ? r > w : w > r) && w < L ? a[i][j] : 0.f;
                }
        }
        // the wave's 16 rows of A, written and read by the same wave
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<f32x4*>(As + (4 * ty + i) * RS + 4 * tx) = f32x4{a[i][0], a[i][1], a[i][2], a[i][3]};
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll 4
        for (int k = 0; k < kTokB / 4; ++k) {
            const float av = As[(16 * wave + c16) * RS + 4 * k + g];
#pragma unroll
            for (int j = 0; j < HD / 16; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, Zs[(4 * k + g) * ZS + 16 * j + c16], acc[j], 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = rb * kTokB + 16 * wave + 4 * g + i;
        if (r >= L) continue;
        bool ok = true;
        if (!FWD) ek.row(r, ok);
#pragma unroll
        for (int j = 0; j < HD / 16; ++j) out[slice + (int64_t)r * D + 16 * j + c16] = ok ? acc[j][i] : 0.f;
    }
}

// The A or B operands of a product over the dimensions of row r: lane group g holds dimensions
// 16 q + 4 g + e of step 4 q + e (the sum over k takes them in any order).
template <int HD>
__device__ inline void dim_operand(const TokRows& src, int64_t id, int r, int g, float (&v)[HD / 4]) {
    bool ok;
    const float* p = src.at(id, r, ok);
#pragma unroll
    for (int q = 0; q < HD / 16; ++q) {
        const f32x4 t = load4(p, 16 * q + 4 * g, ok);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * q + e] = t[e];
    }
}

// acc[a][:] += sum_w da[w][a] y_w ⊙ g_{w,a} for the thread's TT rows and 4 dimensions: da in LDS
// (WS floats per walked step), the rows y_w of Y from ig on, and g_{w,a} = row (first + DIR w -+ a) of
// G: a step moves every row's distance by one.
template <int HD, int DIR, int WS>
__device__ inline void gate_rows(const float* da, const float* Y, const float* G, int first, int ig,
                                 f32x4 (&acc)[HD / 16]) {
    constexpr int TT = HD / 16;
    f32x4 g[TT];
#pragma unroll
    for (int a = 1; a < TT; ++a) g[a - 1] = *reinterpret_cast<const f32x4*>(G + (first - DIR * a) * HD + ig);
    const float* gp = G + first * HD + ig;
#pragma unroll 4
    for (int w = 0; w < kTokB; ++w) {
#pragma unroll
        for (int a = TT - 1; a > 0; --a) g[a] = g[a - 1];
        g[0] = *reinterpret_cast<const f32x4*>(gp + DIR * w * HD);
        const f32x4 y = *reinterpret_cast<const f32x4*>(Y + w * HD + ig);
        float d[TT];
        if constexpr (TT == 4) {
            const f32x4 t = *reinterpret_cast<const f32x4*>(da + w * WS);
#pragma unroll
            for (int a = 0; a < TT; ++a) d[a] = t[a];
        } else {
            const float2 t = *reinterpret_cast<const float2*>(da + w * WS);
            d[0] = t.x; d[1] = t.y;
        }
#pragma unroll
        for (int a = 0; a < TT; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[a][e] = __builtin_fmaf(d[a] * y[e], g[a][e], acc[a][e]);
    }
}

// out[r] = sum_w dA(r, w) Y[w] ⊙ G[d], dA(r, w) = X[r] . Z[w].  ROWT: rows are steps t and the
// walked ones s < t (dQ: X = dO, Z = e_v, Y = e_k); otherwise rows are steps s and the walked
// ones t > s (dE_k: X = e_v, Z = dO, Y = q).
template <int HD, bool ROWT>
__global__ void __launch_bounds__(256, 2)
fac_tok_gate_kernel(const float* __restrict__ Q, const float* __restrict__ dO, const int64_t* __restrict__ x,
                    int64_t V, const float* __restrict__ Ek, const float* __restrict__ Ev,
                    const float* __restrict__ G, int L, int H, float* __restrict__ out) {
    constexpr int TT = HD / 16;
    constexpr int WS = 16 + 4;  // floats per walked step of a wave's 16 rows
    __shared__ __align__(16) float Ys[kTokB * HD], Gs[2 * kTokB * HD], dAs[4 * kTokB * WS];
    const int64_t D = (int64_t)H * HD;
    const int b = blockIdx.z, h = blockIdx.y, nb = gridDim.x;
    const int rb = ROWT ? nb - 1 - (int)blockIdx.x : (int)blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c16 = lane & 15, g = lane >> 4;
    const int64_t* xb = x + (int64_t)b * L;
    const int64_t slice = (int64_t)b * L * D + h * HD;
    const TokRows go{dO + slice, nullptr, 0, D, L}, ev{Ev + h * HD, xb, V, D, L};
    const TokRows yr = ROWT ? TokRows{Ek + h * HD, xb, V, D, L} : TokRows{Q + slice, nullptr, 0, D, L};
    const TokRows gt{G + h * HD, nullptr, 0, D, L + 1};
    const TokRows xr = ROWT ? go : ev, zr = ROWT ? ev : go;
    float* da = dAs + wave * kTokB * WS;
    const int ig = 4 * (lane % (HD / 4)), rg = TT * (lane / (HD / 4));  // 4 dimensions; TT rows of the wave
    f32x4 acc[TT];
#pragma unroll
    for (int a = 0; a < TT; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    float xv[HD / 4];
    {
        const int r = rb * kTokB + 16 * wave + c16;
        dim_operand<HD>(xr, xr.id(r), r, g, xv);
    }
    const int w_lo = ROWT ? 0 : rb, w_hi = ROWT ? rb : nb - 1;
    RowPiece<kTokB, HD, HD> py;
    RowPiece<2 * kTokB, HD, HD> pg;
    int64_t zid[4];
    float zv[4][HD / 4];
    auto ids = [&](int wb) {
        py.ids(yr, wb * kTokB);
#pragma unroll
        for (int j = 0; j < 4; ++j) zid[j] = zr.id(wb * kTokB + 16 * j + c16);
    };
    auto load = [&](int wb) {
        const int dlo = (ROWT ? rb - wb : wb - rb) * kTokB - (kTokB - 1);
        pg.ids(gt, dlo);
        pg.load(gt, dlo);
        py.load(yr, wb * kTokB);
#pragma unroll
        for (int j = 0; j < 4; ++j) dim_operand<HD>(zr, zid[j], wb * kTokB + 16 * j + c16, g, zv[j]);
    };
    ids(w_lo);
    load(w_lo);
    for (int wb = w_lo; wb <= w_hi; ++wb) {
        ids(min(wb + 1, w_hi));
        __syncthreads();
        py.store(Ys);
        pg.store(Gs);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < HD / 4; ++k) d = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[k], zv[j][k], d, 0, 0, 0);
            if (wb == rb || wb == nb - 1) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = rb * kTokB + 16 * wave + 4 * g + i, w = wb * kTokB + 16 * j + c16;
                    d[i] = (ROWT ? r > w : w > r) && w < L ? d[i] : 0.f;
                }
            }
            *reinterpret_cast<f32x4*>(da + (16 * j + c16) * WS + 4 * g) = d;
        }
        load(min(wb + 1, w_hi));
        __syncthreads();
        // distance of row r and walked step w: row r - w + 63 of the staged ones (ROWT), w - r + 63
        const int r0 = 16 * wave + rg;
        if (ROWT) gate_rows<HD, -1, WS>(da + rg, Ys, Gs, r0 + kTokB - 1, ig, acc);
        else gate_rows<HD, 1, WS>(da + rg, Ys, Gs, kTokB - 1 - r0, ig, acc);
    }
#pragma unroll
    for (int a = 0; a < TT; ++a) {
        const int r = rb * kTokB + 16 * wave + rg + a;
        if (r >= L) continue;
        bool ok = true;
        if (!ROWT) ev.row(r, ok);
        *reinterpret_cast<f32x4u*>(out + slice + (int64_t)r * D + ig) = ok ? acc[a] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
}

// Rows are distances d, walked steps t: dGb[b,d,h,:] = sum_t (dO_t . e_v[x_{t-d}]) q_t ⊙
// e_k[x_{t-d}] for d in [1, L); row 0 is zero.  The steps s = t - d of a tile span 127 rows; the
// products dO_t . e_v[x_s] of a wave's 16 steps t fall on 79 of them, five column tiles.
template <int HD>
__global__ void __launch_bounds__(256, 2)
fac_tok_dist_kernel(const float* __restrict__ Q, const float* __restrict__ dO, const int64_t* __restrict__ x,
                    int64_t V, const float* __restrict__ Ek, const float* __restrict__ Ev, int L, int H,
                    float* __restrict__ dGb) {
    constexpr int TT = HD / 16;
    constexpr int WS = kTokB + 4;
    __shared__ __align__(16) float Qs[kTokB * HD], Es[2 * kTokB * HD], dAs[kTokB * WS];
    const int64_t D = (int64_t)H * HD;
    const int b = blockIdx.z, h = blockIdx.y, nb = gridDim.x, db = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c16 = lane & 15, g = lane >> 4;
    const int64_t* xb = x + (int64_t)b * L;
    const int64_t slice = (int64_t)b * L * D + h * HD;
    const TokRows qr{Q + slice, nullptr, 0, D, L}, go{dO + slice, nullptr, 0, D, L};
    const TokRows ek{Ek + h * HD, xb, V, D, L}, ev{Ev + h * HD, xb, V, D, L};
    const int ig = 4 * (lane % (HD / 4)), rg = TT * (lane / (HD / 4));
    f32x4 acc[TT];
#pragma unroll
    for (int a = 0; a < TT; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    RowPiece<kTokB, HD, HD> pq;
    RowPiece<2 * kTokB, HD, HD> pe;
    int64_t zid[5];
    auto ids = [&](int tb) {
        const int slo = (tb - db) * kTokB - (kTokB - 1);
        pe.ids(ek, slo);
#pragma unroll
        for (int j = 0; j < 5; ++j) zid[j] = ev.id(slo + 16 * (wave + j) + c16);
    };
    auto load = [&](int tb) {
        pq.ids(qr, tb * kTokB);
        pq.load(qr, tb * kTokB);
        pe.load(ek, (tb - db) * kTokB - (kTokB - 1));
    };
    ids(db);
    load(db);
    for (int tb = db; tb < nb; ++tb) {
        const int slo = (tb - db) * kTokB - (kTokB - 1);
        const int next = min(tb + 1, nb - 1);
        float xv[HD / 4], zv[5][HD / 4];
        dim_operand<HD>(go, go.id(tb * kTokB + 16 * wave + c16), tb * kTokB + 16 * wave + c16, g, xv);
#pragma unroll
        for (int j = 0; j < 5; ++j) dim_operand<HD>(ev, zid[j], slo + 16 * (wave + j) + c16, g, zv[j]);
        __syncthreads();
        pq.store(Qs);
        pe.store(Es);
        ids(next);
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < HD / 4; ++k) v = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[k], zv[j][k], v, 0, 0, 0);
            const int si = 16 * (wave + j) + c16;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = 16 * wave + 4 * g + i, d = t + kTokB - 1 - si;
                if (d >= 0 && d < kTokB) dAs[t * WS + d] = slo + si >= 0 && db + d > 0 && tb * kTokB + t < L ? v[i] : 0.f;
            }
        }
        load(next);
        __syncthreads();
        const int d0 = 16 * wave + rg;
        gate_rows<HD, 1, WS>(dAs + d0, Qs, Es, kTokB - 1 - d0, ig, acc);
    }
#pragma unroll
    for (int a = 0; a < TT; ++a) {
        const int d = db * kTokB + 16 * wave + rg + a;
        if (d < L) *reinterpret_cast<f32x4u*>(dGb + slice + (int64_t)d * D + ig) = acc[a];
    }
}

int check_hd(int hd, const char* what) {
    if (hd != 32 && hd != 64)
        return fail(MB_ERR_UNSUPPORTED, "%s: head_dim=%d (supported: 32, 64)", what, hd);
    return MB_OK;
}

}  // namespace
}  // namespace mb

using namespace mb;

extern "C" int mb_factored_outer(const float* X, const int64_t* xrow, const float* Y,
                                 const int64_t* yrow, int64_t ld, int64_t nrows, const float* alpha,
                                 int64_t as_b, int64_t as_r, int64_t as_n, int B, int R, int H,
                                 int N, int hd, float* out, void* stream) {
    MB_REQUIRE(B >= 0 && R >= 0 && H >= 1 && N >= 1 && nrows >= 0,
               "mb_factored_outer: bad sizes B=%d R=%d H=%d N=%d", B, R, H, N);
    if (int rc = check_hd(hd, "mb_factored_outer")) return rc;
    MB_REQUIRE(ld >= (int64_t)H * hd, "mb_factored_outer: row stride %lld < H*hd", (long long)ld);
    if (B == 0) return MB_OK;
    MB_REQUIRE(X && Y && alpha && out, "mb_factored_outer: null pointer argument");
    hipStream_t st = (hipStream_t)stream;
    const dim3 blk(256);
    if (hd == 64) {
        const int64_t grid = (int64_t)B * H * ((N + kOuterRates - 1) / kOuterRates);
        MB_REQUIRE(grid <= INT32_MAX, "mb_factored_outer: B=%d H=%d N=%d too large", B, H, N);
        hipLaunchKernelGGL(fac_outer_mfma_kernel, dim3((unsigned)grid), blk, 0, st, X, xrow, Y, yrow, ld, nrows,
                           alpha, as_b, as_r, as_n, B, R, H, N, out);
    } else {
        hipLaunchKernelGGL(fac_outer_kernel<32>, dim3((N + 7) / 8, H, B), blk, 0, st, X, xrow, Y,
                           yrow, ld, nrows, alpha, as_b, as_r, as_n, R, H, N, out);
    }
    return check_launch("mb_factored_outer");
}

extern "C" int mb_factored_apply(const float* M, const float* w, int64_t ldw, const float* Y,
                                 const int64_t* yrow, int64_t ld, int64_t nrows, const float* alpha,
                                 int64_t as_b, int64_t as_r, int64_t as_n, int B, int R, int H,
                                 int N, int hd, int transpose, float* out, int64_t ldo,
                                 int accumulate, void* stream) {
    MB_REQUIRE(B >= 0 && R >= 0 && H >= 1 && N >= 1 && nrows >= 0,
               "mb_factored_apply: bad sizes B=%d R=%d H=%d N=%d", B, R, H, N);
    if (int rc = check_hd(hd, "mb_factored_apply")) return rc;
    MB_REQUIRE(ld >= (int64_t)H * hd && ldo >= (int64_t)H * hd,
               "mb_factored_apply: row strides must be >= H*hd");
    if (B == 0 || R == 0) return MB_OK;
    MB_REQUIRE(M && Y && alpha && out, "mb_factored_apply: null pointer argument");
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((R + kApplyRows - 1) / kApplyRows, H, B), blk(256);
#define MB_FAC_APPLY(HDV, TR)                                                                     \
    hipLaunchKernelGGL((fac_apply_kernel<HDV, TR>), grid, blk, 0, st, M, w, ldw, Y, yrow, ld, nrows, \
                       alpha, as_b, as_r, as_n, R, H, N, out, ldo, accumulate)
    if (hd == 64) {
        const int64_t g64 = (int64_t)B * H * ((R + kStateRows - 1) / kStateRows);
        MB_REQUIRE(g64 <= INT32_MAX, "mb_factored_apply: B=%d H=%d R=%d too large", B, H, R);
        if (transpose)
            hipLaunchKernelGGL(fac_apply_mfma_kernel<true>, dim3((unsigned)g64), dim3(512), 0, st, M, w, ldw, Y, yrow,
                               ld, nrows, alpha, as_b, as_r, as_n, B, R, H, N, out, ldo, accumulate);
        else
            hipLaunchKernelGGL(fac_apply_mfma_kernel<false>, dim3((unsigned)g64), dim3(512), 0, st, M, w, ldw, Y, yrow,
                               ld, nrows, alpha, as_b, as_r, as_n, B, R, H, N, out, ldo, accumulate);
    } else {
        if (transpose) MB_FAC_APPLY(32, true); else MB_FAC_APPLY(32, false);
    }
#undef MB_FAC_APPLY
    return check_launch("mb_factored_apply");
}

extern "C" int mb_factored_tok_fwd(const float* Q, const int64_t* x, int64_t V, const float* E_k,
                                   const float* E_v, const float* G, int B, int L, int H, int hd,
                                   float* O, void* stream) {
    MB_REQUIRE(B >= 0 && L >= 0 && H >= 1 && V >= 1, "mb_factored_tok_fwd: bad sizes");
    if (int rc = check_hd(hd, "mb_factored_tok_fwd")) return rc;
    if (B == 0 || L == 0) return MB_OK;
    MB_REQUIRE(Q && x && E_k && E_v && G && O, "mb_factored_tok_fwd: null pointer argument");
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((L + kTokB - 1) / kTokB, H, B), blk(256);
    if (hd == 64)
        hipLaunchKernelGGL((fac_tok_pair_kernel<64, true>), grid, blk, 0, st, Q, nullptr, x, V, E_k, E_v, G, L, H, O);
    else
        hipLaunchKernelGGL((fac_tok_pair_kernel<32, true>), grid, blk, 0, st, Q, nullptr, x, V, E_k, E_v, G, L, H, O);
    return check_launch("mb_factored_tok_fwd");
}

extern "C" int mb_factored_tok_bwd(const float* Q, const float* dO, const int64_t* x, int64_t V,
                                   const float* E_k, const float* E_v, const float* G, int B, int L,
                                   int H, int hd, float* dQ, float* dEk_tok, float* dEv_tok,
                                   float* dG_b, void* stream) {
    MB_REQUIRE(B >= 0 && L >= 0 && H >= 1 && V >= 1, "mb_factored_tok_bwd: bad sizes");
    if (int rc = check_hd(hd, "mb_factored_tok_bwd")) return rc;
    if (B == 0 || L == 0) return MB_OK;
    MB_REQUIRE(Q && dO && x && E_k && E_v && G && dQ && dEk_tok && dEv_tok && dG_b,
               "mb_factored_tok_bwd: null pointer argument");
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((L + kTokB - 1) / kTokB, H, B), blk(256);
#define MB_FAC_BWD(HDV)                                                                            \
    do {                                                                                           \
        hipLaunchKernelGGL((fac_tok_gate_kernel<HDV, true>), grid, blk, 0, st, Q, dO, x, V, E_k, E_v, G, L, H, \
                           dQ);                                                                    \
        hipLaunchKernelGGL((fac_tok_gate_kernel<HDV, false>), grid, blk, 0, st, Q, dO, x, V, E_k, E_v, G, L, H, \
                           dEk_tok);                                                               \
        hipLaunchKernelGGL((fac_tok_pair_kernel<HDV, false>), grid, blk, 0, st, Q, dO, x, V, E_k, E_v, G, L, H, \
                           dEv_tok);                                                               \
        hipLaunchKernelGGL(fac_tok_dist_kernel<HDV>, grid, blk, 0, st, Q, dO, x, V, E_k, E_v, L, H, dG_b); \
    } while (0)
    if (hd == 64) MB_FAC_BWD(64);
    else MB_FAC_BWD(32);
#undef MB_FAC_BWD
    return check_launch("mb_factored_tok_bwd");
}
