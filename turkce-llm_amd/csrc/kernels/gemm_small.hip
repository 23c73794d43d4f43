// gemm_small.hip -- fp32 GEMMs with few output tiles: one 32x32 tile of C per
// workgroup, its four waves sharing out k.
//
// A product of a few hundred rows (a short prompt, a decode batch, a small
// model's layer) gives the 64x64 tiles a few dozen workgroups; each walks its
// whole k through LDS, two barriers per 32 k, and most CUs idle.  Here a CU's
// four SIMDs work on different k of one small tile: wave w takes the 32-deep
// blocks w, w + 4, ... straight from global memory in the operand layout of
// v_mfma_f32_32x32x2f32 (no LDS, no barrier), the next block's loads in
// flight while the current one is multiplied, and the four sums meet in LDS
// once, added in wave order.  No second launch for a split-K reduction, and
// the RoPE and SwiGLU epilogues, which need whole sums, get the split too.
// Bound by the latency of two or three dependent load batches: 64x1152x384
// 8.0 -> 5.8 us, 128x2048x384 9.9 -> 6.1, 512x384x384 11.9 -> 6.0; sixteen
// waves spilled, and where they did not (NT) were no faster.
#include "common.h"

template <int TA, int TB, bool AL, bool GLU>
__device__ __forceinline__ void gemm_small_body(const GemmParams& p) {
    constexpr int W = 4;     // waves
    constexpr int LD = 36;   // floats per row of a wave's sums: 16-byte rows, conflict-free quads
    __shared__ __attribute__((aligned(16))) float lds[W * 32 * LD];
    __shared__ float lcs[2 * W * 32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane & 31, hf = lane >> 5;
    const int tm = (int)blockIdx.x % p.tiles_m, tn = (int)blockIdx.x / p.tiles_m;
    const int row = min(tm * 32 + l, p.M - 1);
    // SwiGLU: 16 gate columns and the matching 16 up columns
    const int col = GLU ? (l < 16 ? 0 : p.glu_F - 16) + 16 * tn + l : min(tn * 32 + l, p.N - 1);
    const float* a = p.A + (TA ? row : (long long)row * p.lda);
    const float* b = p.B + (TB ? (long long)col * p.ldb : col);

    // the lane's four k of each of a block's four 8-k groups: 8j + 4 hf + s
    auto load = [&](const float* x, int ld, bool kmajor, int k0, f32x4 (&f)[4]) {
        const bool whole = k0 + 32 <= p.K;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = k0 + 8 * j + 4 * hf;
            if (whole) {
                if (kmajor && AL) f[j] = *(const f32x4*)(x + k);
                else {
#pragma unroll
                    for (int s = 0; s < 4; s++) f[j][s] = kmajor ? x[k + s] : x[(long long)(k + s) * ld];
                }
            } else {
#pragma unroll
                for (int s = 0; s < 4; s++)
                    f[j][s] = k + s < p.K ? (kmajor ? x[k + s] : x[(long long)(k + s) * ld]) : 0.f;
            }
        }
    };
    f32x16 acc, acc2;   // two sums of alternate 8-k groups: half as many roundings in a row
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = acc2[r] = 0.f;
    float cs = 0.f;
    const bool cs_on = TB == 0 && p.csum != nullptr && tm == 0;
    f32x4 fa[2][4], fb[2][4];
    const int k1 = 32 * wave;
    if (k1 < p.K) {
        load(a, p.lda, TA == 0, k1, fa[0]);
        load(b, p.ldb, TB == 1, k1, fb[0]);
    }
    auto block = [&](int k0, f32x4 (&xa)[4], f32x4 (&xb)[4], f32x4 (&na)[4], f32x4 (&nb)[4]) {
        if (k0 + 32 * W < p.K) {
            load(a, p.lda, TA == 0, k0 + 32 * W, na);
            load(b, p.ldb, TB == 1, k0 + 32 * W, nb);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (TB == 0) cs += (xb[j][0] + xb[j][1]) + (xb[j][2] + xb[j][3]);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                f32x16& c = (j & 1) ? acc2 : acc;
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(xb[j][s], xa[j][s], c, 0, 0, 0);
            }
        }
    };
    for (int k0 = k1; k0 < p.K; k0 += 64 * W) {
        block(k0, fa[0], fb[0], fa[1], fb[1]);
        if (k0 + 32 * W < p.K) block(k0 + 32 * W, fa[1], fb[1], fa[0], fb[0]);
    }
    acc += acc2;
    // lane: row l of the tile, columns 8g + 4 hf + q
    float* lw = lds + wave * 32 * LD;
#pragma unroll
    for (int g = 0; g < 4; g++)
        *(f32x4*)(lw + l * LD + 8 * g + 4 * hf) = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    if (cs_on) lcs[(2 * wave + hf) * 32 + l] = cs;
    __syncthreads();
    auto sum_waves = [&](int m, int n) {
        f32x4 t = *(const f32x4*)(lds + m * LD + n);
#pragma unroll
        for (int w = 1; w < W; w++) t += *(const f32x4*)(lds + (32 * w + m) * LD + n);
        return t;
    };
    if (cs_on && threadIdx.x < 32 && tn * 32 + (int)threadIdx.x < p.N) {
        float t = lcs[threadIdx.x];
#pragma unroll
        for (int w = 1; w < 2 * W; w++) t += lcs[w * 32 + threadIdx.x];
        p.csum[tn * 32 + threadIdx.x] = t;
    }
    if constexpr (GLU) {
        if (threadIdx.x < 128) {
            const int rl = threadIdx.x >> 2, m = tm * 32 + rl, n = 4 * (threadIdx.x & 3), c = 16 * tn + n;
            if (m < p.M) {
                f32x4 gv = sum_waves(rl, n) * p.alpha, uv = sum_waves(rl, 16 + n) * p.alpha, o;
                if (p.bias) {
                    gv += *(const f32x4*)(p.bias + c);
                    uv += *(const f32x4*)(p.bias + p.glu_F + c);
                }
                float* dst = p.C + (long long)m * p.ldc + c;
                *(f32x4*)dst = gv;
                *(f32x4*)(dst + p.glu_F) = uv;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float sg = 1.0f / (1.0f + expf(-gv[q]));
                    o[q] = (gv[q] * sg) * uv[q];
                }
                *(f32x4*)(p.glu_h + (long long)m * p.glu_F + c) = o;
            }
        }
    } else {
        const int rl = threadIdx.x >> 3, m = tm * 32 + rl, nl = 4 * (threadIdx.x & 7), n = tn * 32 + nl;
        if (m >= p.M || n >= p.N) return;
        const f32x4 s = sum_waves(rl, nl);
        float* dst = p.C + (long long)m * p.ldc + n;
        const float* res = p.resid + (long long)m * p.ldr + n;
        const bool vec = n + 3 < p.N && ((p.ldc | (p.resid ? p.ldr : 0)) & 3) == 0 &&
                         ((reinterpret_cast<uintptr_t>(p.C) | reinterpret_cast<uintptr_t>(p.resid) |
                           reinterpret_cast<uintptr_t>(p.bias)) & 15) == 0;
        f32x4 cv = {0.f, 0.f, 0.f, 0.f}, bv = cv, rv = cv, v;
        if (vec) {
            if (p.beta != 0.f) cv = *(const f32x4*)dst;
            if (p.bias) bv = *(const f32x4*)(p.bias + n);
            if (p.resid) rv = *(const f32x4*)res;
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const bool in = n + q < p.N;
                if (in && p.beta != 0.f) cv[q] = dst[q];
                if (in && p.bias) bv[q] = p.bias[n + q];
                if (in && p.resid) rv[q] = res[q];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float x = p.alpha * s[q];
            if (p.beta != 0.f) x = x + p.beta * cv[q];
            if (p.bias) x = x + bv[q];
            if (p.resid) x = rv[q] + x;
            v[q] = x;
        }
        if (p.rope_cos && n < p.rope_cols) rope4(p, m, n, v);
        if (vec) *(f32x4*)dst = v;
        else {
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (n + q < p.N) dst[q] = v[q];
        }
    }
}

#define GEMM_SMALL(NAME, TA, TB, AL, GLU)                                             \
    extern "C" __global__ void __launch_bounds__(256) NAME(GemmParams p) {             \
        gemm_small_body<TA, TB, AL, GLU>(p);                                           \
    }
GEMM_SMALL(k_smallgemm_nn, 0, 0, true, false)
GEMM_SMALL(k_smallgemm_nt, 0, 1, true, false)
GEMM_SMALL(k_smallgemm_tn, 1, 0, true, false)
GEMM_SMALL(k_smallgemm_nn_u, 0, 0, false, false)
GEMM_SMALL(k_smallgemm_nt_u, 0, 1, false, false)
GEMM_SMALL(k_smallgemm_tn_u, 1, 0, false, false)
GEMM_SMALL(k_smallgemm_nn_glu, 0, 0, true, true)
