// gemm_split.hip -- fp32 GEMMs on the bf16 matrix cores, without loss of
// precision: every fp32 operand, times 2^24, is split into three bf16 parts
// that add up to it exactly, and the products that matter are formed on
// v_mfma_f32_32x32x16_bf16 with fp32 accumulation.
//
//   2^24 x = h + m + l,  h = bf16(2^24 x), m = bf16(2^24 x - h), l = the rest (exact)
//   2^48 a*b ~ al*bh + ah*bl + am*bm + am*bh + ah*bm + ah*bh
//
// The factor is there for the smallest operands: the lowest bit of any fp32
// (2^-149) becomes 2^-125, so no part is ever subnormal.  Without it the
// split held 24 bits only from 2^-110 on and 8 at 2^-126.  Sums are scaled
// back by 2^-48.  Operands near 2^104 and sums near 2^80 and beyond overflow
// and take the recomputation on the fp32 matrix cores that an infinity takes.
// It costs one multiplication per value of B (A's replaces its sign change):
// QKV 8192x1152x384 58.3 -> 59.0 us, the LM head unchanged; the same bits.
//
// Sums of products of bf16 parts: Henry, Tang and Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019.
//
// The three products left out are below 2^-24 of |a*b|, and a product of two
// bf16 has 16 significant bits, so it enters the sum unrounded: what is
// rounded is the running sum, as with the fp32 matrix cores, and less often
// (6 times per 16 k instead of 8).  Error against 64 bits, N(0,1) x
// N(0,0.02): K = 384 2.9e-7 (fp32 MFMA 3.5e-7), K = 8192 in one sum 1.4e-6
// (1.6e-6).
//
// Serves raw GEMMs, the matmul node and the decoder's prefill; the trainer
// keeps the fp32 tiles (trlm_gemm_keep_fp32), and with them the row statistics
// and column sums that only it asks for: the host gives no such product here.
//
// Why: the fp32 matrix cores (157 TFLOP/s) were 79-86 % busy, so large GEMMs
// could only gain from another unit.  Six bf16
// products at the 2.0 PFLOP/s that the matrix cores sustain on random data
// are worth 333 TFLOP/s.  Measured before -> after: LM head forward
// 8192x31769x384 1526 -> 1050 us, gate/up 8192x2048x384 105 -> 75 us,
// its dW 106 -> 83 us.  What bounds it now is the power limit: the LM head
// runs at 1.8 GHz (2.4 GHz with a zero operand, 758 us), whatever the
// schedule: double-buffered 16-deep steps with the split interleaved between
// the MFMAs, a second fragment set and 256x128 tiles were all within 5 %.
//
// Layout: 256 threads = 4 waves in 2x2, one LDS buffer of 32 k, the next
// step's values loaded into registers while the current one is multiplied;
// three (128x128) to six (64x64) workgroups per CU overlap one's split with
// another's MFMAs.  The parts lie as 16-byte chunks of 8 k of one row, which
// is a lane's operand of one MFMA, so every fragment is one conflict-free
// ds_read_b128.  An operand that is contiguous along m / n is loaded two rows
// per thread; its even and odd rows go to separate 32-row blocks (as
// GemmIlv's), so that the stores are conflict-free too.
#include "common.h"

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// The three bf16 parts of eight floats times scale (a power of two, of either
// sign), two to a register.
__device__ __forceinline__ void split8(const float (&x)[8], float scale, u32x4& h, u32x4& m, u32x4& l) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float x0 = x[2 * i] * scale, x1 = x[2 * i + 1] * scale;
        const unsigned hu = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){x0, x1}, bf16x2));
        const float r0 = x0 - __builtin_bit_cast(float, hu << 16);
        const float r1 = x1 - __builtin_bit_cast(float, hu & 0xffff0000u);
        const unsigned mu = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){r0, r1}, bf16x2));
        const float s0 = r0 - __builtin_bit_cast(float, mu << 16);
        const float s1 = r1 - __builtin_bit_cast(float, mu & 0xffff0000u);
        h[i] = hu;
        m[i] = mu;
        l[i] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){s0, s1}, bf16x2));
    }
}

constexpr int X3_BK = 32;     // k per step
constexpr int X3_FLIP = 4;    // steps between changes of the sum's sign
constexpr float X3_SCALE = 0x1p24f, X3_UNSCALE = 0x1p-48f;   // of an operand, of a sum

// One operand's part of a k step: R rows (of m or n) by 32 k.
// LDS: [plane h/m/l][chunk c of 8 k][slot], 16 bytes each; chunk c holds
// k = 4c..4c+3 and 16+4c..16+4c+3 (the same for both operands).
// AL: rows 16-byte aligned (ld a multiple of 4), so that four k or two rows are one
// load; without it every value is loaded by itself.
template <int R, bool KM, bool AL>
struct X3Tile {
    static constexpr int W = (!KM && R >= 128) ? 2 : 1;     // rows per thread and id
    static constexpr int NI = R * 4 / 256 / W;              // ids per thread
    static constexpr int COL = R + 2;                       // 16-byte units per chunk column (2 of padding)
    static constexpr int UNITS = 12 * COL;
    static constexpr bool ILV = W == 2;
    float x[NI * W][8];
    const float* ptr[NI];
    int second[NI];          // unaligned: the second row's offset (0 where it would be past the edge)
    long long step, ld;

    __device__ __forceinline__ static int slot(int r) { return ILV ? (r & ~63) + ((r & 63) >> 1) + 32 * (r & 1) : r; }

    __device__ __forceinline__ void init(const float* base, int ld_, int r0, int rlim, int k0, int glu_F = 0) {
        ld = ld_;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int id = threadIdx.x + 256 * i;
            if constexpr (KM) {
                int gr = r0 + id / 4;
                if (gr >= rlim) gr = rlim - 1;
                ptr[i] = base + (long long)gr * ld + k0 + 4 * (id % 4);
            } else {
                const int r = W * (id % (R / W));
                int gr = r0 + r;
                if (glu_F) gr = (r < R / 2 ? 0 : glu_F - R / 2) + (r0 >> 1) + r;
                if (gr >= rlim) gr = 0;
                second[i] = AL || gr + 1 < rlim;
                ptr[i] = base + (long long)(k0 + 4 * (id / (R / W))) * ld + gr;
            }
        }
        step = KM ? X3_BK : (long long)X3_BK * ld;
    }
    // the 32 k from k0, all inside the matrix
    __device__ __forceinline__ void load() {
#pragma unroll
        for (int i = 0; i < NI; i++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if constexpr (KM && !AL) {
#pragma unroll
                    for (int e = 0; e < 4; e++) x[i][4 * j + e] = ptr[i][16 * j + e];
                } else if constexpr (KM) {
                    const f32x4 v = *(const f32x4*)(ptr[i] + 16 * j);
#pragma unroll
                    for (int e = 0; e < 4; e++) x[i][4 * j + e] = v[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float* src = ptr[i] + (16 * j + e) * ld;
                        if constexpr (W == 2 && !AL) {
                            x[2 * i][4 * j + e] = src[0];
                            x[2 * i + 1][4 * j + e] = src[second[i]];
                        } else if constexpr (W == 2) {
                            const f32x2 v = *(const f32x2*)src;
                            x[2 * i][4 * j + e] = v[0];
                            x[2 * i + 1][4 * j + e] = v[1];
                        } else {
                            x[i][4 * j + e] = *src;
                        }
                    }
                }
            }
            ptr[i] += step;
        }
    }
    // the rem < 32 k from `off` on (a whole number of steps past the pointers),
    // the rest of the step taken as zero; the pointers stay
    __device__ __forceinline__ void load_part(int off, int rem) {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int id = threadIdx.x + 256 * i;
            const int k0 = KM ? 4 * (id % 4) : 4 * (id / (R / W));
            const float* src = ptr[i] + (KM ? off : off * ld);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int kk = (j < 4 ? j : 12 + j);
                const bool in = k0 + kk < rem;
#pragma unroll
                for (int w = 0; w < W; w++)
                    x[W * i + w][j] = in ? (KM ? src[kk] : src[kk * ld + (w ? second[i] : 0)]) : 0.f;
            }
        }
    }
    __device__ __forceinline__ void store(u32x4* lds, float scale) const {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int id = threadIdx.x + 256 * i;
            const int c = KM ? id % 4 : id / (R / W);
            const int r = KM ? id / 4 : W * (id % (R / W));
#pragma unroll
            for (int w = 0; w < W; w++) {
                u32x4 h, m, l;
                split8(x[W * i + w], scale, h, m, l);
                u32x4* d = lds + c * COL + slot(r + w);
                d[0] = h;
                d[4 * COL] = m;
                d[8 * COL] = l;
            }
        }
    }
    template <int NF>
    __device__ __forceinline__ static void frags(const u32x4* lds, int rb0, int kk, int lane, bf16x8 (&f)[3][NF]) {
        const u32x4* s = lds + (2 * kk + (lane >> 5)) * COL + rb0 + (lane & 31);
#pragma unroll
        for (int pl = 0; pl < 3; pl++)
#pragma unroll
            for (int i = 0; i < NF; i++) f[pl][i] = __builtin_bit_cast(bf16x8, s[pl * 4 * COL + 32 * i]);
    }
};

// SwiGLU epilogue of 128-column tiles: columns 0..63 of the tile are gate
// columns 64 tn .., 64..127 the matching up columns.  32 rows of every wave
// block at a time go through LDS, so that C leaves in whole row segments and
// the two waves of a row block share the h = (g * sigmoid(g)) * u of its rows.
template <int BM, bool ILA>
__device__ __forceinline__ void gemm_epilogue_glu2(const GemmParams& p, const f32x16 (&acc)[BM / 64][2], int r0, int tn,
                                                   int wave, int lane, float* lds) {
    constexpr int FM = BM / 64;
    static_assert(!ILA, "NN: A is K-contiguous");
    const int wn = wave & 1, half = lane >> 5, ml = lane & 31;
    const int ch = lane & 15, rl = lane >> 4;
    const int cb = (wn == 0 ? 0 : p.glu_F) + 64 * tn + 4 * ch;
    float* lw = lds + wave * 32 * 64;
    const float* lg = lds + (wave & ~1) * 32 * 64;
    const f32x4 b = p.bias ? *(const f32x4*)(p.bias + cb) : f32x4{0.f, 0.f, 0.f, 0.f};
    const f32x4 bg = p.bias ? *(const f32x4*)(p.bias + 64 * tn + 4 * ch) : f32x4{0.f, 0.f, 0.f, 0.f};
    const f32x4 bu = p.bias ? *(const f32x4*)(p.bias + p.glu_F + 64 * tn + 4 * ch) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < FM; i++) {
        __syncthreads();   // the main loop's, or the last pass's, reads are done
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int qp = 0; qp < 4; qp += 2) {
                const f32x4 v = {p.alpha * acc[i][0][4 * g + qp], p.alpha * acc[i][1][4 * g + qp],
                                 p.alpha * acc[i][0][4 * g + qp + 1], p.alpha * acc[i][1][4 * g + qp + 1]};
                *(f32x4*)(lw + ml * 64 + 4 * ((4 * g + 2 * half + qp / 2) ^ (ml & 7))) = v;
            }
        __syncthreads();
        f32x4 v[8];
#pragma unroll
        for (int it = 0; it < 8; it++) {
            const int rr = it * 4 + rl;
            v[it] = *(const f32x4*)(lw + rr * 64 + 4 * (ch ^ (rr & 7))) + b;
        }
#pragma unroll
        for (int it = 0; it < 8; it++) {
            const int row = r0 + 32 * i + it * 4 + rl;
            if (row < p.M) *(f32x4*)(p.C + (long long)row * p.ldc + cb) = v[it];
        }
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int rr = wn * 16 + it * 4 + rl, row = r0 + 32 * i + rr;
            const f32x4 gv = *(const f32x4*)(lg + rr * 64 + 4 * (ch ^ (rr & 7))) + bg;
            const f32x4 uv = *(const f32x4*)(lg + 32 * 64 + rr * 64 + 4 * (ch ^ (rr & 7))) + bu;
            f32x4 o;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float sg = 1.0f / (1.0f + expf(-gv[q]));
                o[q] = (gv[q] * sg) * uv[q];
            }
            if (row < p.M) *(f32x4*)(p.glu_h + (long long)row * p.glu_F + 64 * tn + 4 * ch) = o;
        }
    }
}

// A wave block recomputed on the fp32 matrix cores, straight from global
// memory.  Only for a block with an infinity or NaN in it: an operand that is
// infinite (or is once scaled, or rounds to infinity in bf16) has no split,
// and its products must come out as fp32 gives them.
template <int TA, int TB, int FM, int FN, bool ILA, bool ILB, class ColB>
__device__ __forceinline__ void gemm_wave_f32(const GemmParams& p, const float* A, const float* B, int r0,
                                              ColB col, int kb, int ke, int lane, f32x16 (&acc)[FM][FN]) {
    const int l = lane & 31, hf = lane >> 5;
    long long oa[FM], ob[FN];
#pragma unroll
    for (int i = 0; i < FM; i++) {
        int r = r0 + (ILA ? 64 * (i >> 1) + 2 * l + (i & 1) : 32 * i + l);
        if (r >= p.M) r = p.M - 1;
        oa[i] = TA ? r : (long long)r * p.lda;
    }
#pragma unroll
    for (int j = 0; j < FN; j++) {
        int c = col(ILB ? 64 * (j >> 1) + 2 * l + (j & 1) : 32 * j + l);
        if (c >= p.N) c = p.N - 1;
        ob[j] = TB ? (long long)c * p.ldb : c;
    }
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    for (int k0 = kb; k0 < ke; k0 += 2) {
        const int k = k0 + hf;
        float fa[FM], fb[FN];
#pragma unroll
        for (int i = 0; i < FM; i++) fa[i] = k < ke ? A[oa[i] + (TA ? (long long)k * p.lda : k)] : 0.f;
#pragma unroll
        for (int j = 0; j < FN; j++) fb[j] = k < ke ? B[ob[j] + (TB ? k : (long long)k * p.ldb)] : 0.f;
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
}

template <int TA, int TB, int BM, int BN, bool AL = true, bool GLU = false>
__device__ __forceinline__ void gemm_x3_body(const GemmParams& p) {
    constexpr int FM = BM / 64, FN = BN / 64;
    using TileA = X3Tile<BM, TA == 0, AL>;
    using TileB = X3Tile<BN, TB == 1, AL>;
    __shared__ u32x4 lds[TileA::UNITS + TileB::UNITS];
    u32x4* la = lds;
    u32x4* lb = lds + TileA::UNITS;

    int tm, tn, split;
    gemm_tile_coords(p, tm, tn, split);
    const int batch = p.splits > 1 ? 0 : (int)blockIdx.z;
    const float* A = p.A + batch * p.sA;
    const float* B = p.B + batch * p.sB;
    float* C = p.C + batch * p.sC + split * p.sW;
    const int m0 = tm * BM, n0 = tn * BN;
    const int kb = split * p.kchunk;
    int ke = kb + p.kchunk;
    if (ke > p.K) ke = p.K;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm0 = (wave >> 1) * (BM / 2), wn0 = (wave & 1) * (BN / 2);

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    TileA ta;
    TileB tb;
    ta.init(A, p.lda, m0, p.M, kb);
    tb.init(B, p.ldb, n0, p.N, kb, GLU ? p.glu_F : 0);
    // the partial k step (the last k) comes first, so the loop's loads need no checks
    const int rem = (ke - kb) % X3_BK, nk = (ke - kb) / X3_BK + (rem ? 1 : 0);
    if (rem) {
        ta.load_part(ke - kb - rem, rem);
        tb.load_part(ke - kb - rem, rem);
    } else if (nk) {
        ta.load();
        tb.load();
    }
    // The bf16 MFMA rounds its sum down by some 0.003 ulp on average, whatever
    // the sign.  That is nothing in one element, but it has the same sign in
    // all of them and would show in sums over C's rows (a bias gradient's), so
    // the sum is formed negated for every other four steps: two steps
    // positive, four negative, four positive, ...
    float scale = X3_SCALE;
    auto times = [&](float f) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] *= f;
    };
    for (int t = 0; t < nk; t++) {
        if (t % X3_FLIP == X3_FLIP / 2) {
            asm volatile("");   // a branch, not a select per element in every step
            scale = -scale;
            times(-1.f);
        }
        ta.store(la, scale);
        tb.store(lb, X3_SCALE);
        if (t + 1 < nk) {
            ta.load();
            tb.load();
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            bf16x8 fa[3][FM], fb[3][FN];
            TileA::template frags<FM>(la, wm0, kk, lane, fa);
            TileB::template frags<FN>(lb, wn0, kk, lane, fb);
            // small products first
            constexpr int PA[6] = { 2, 0, 1, 1, 0, 0 }, PB[6] = { 0, 2, 1, 0, 1, 0 };
#pragma unroll
            for (int t = 0; t < 6; t++)
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[PB[t]][j], fa[PA[t]][i], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    times(scale > 0.f ? X3_UNSCALE : -X3_UNSCALE);
    // the largest magnitude (as bits) among the block's elements of C; what
    // an edge tile holds past M or N comes from padding and is left out
    unsigned top = 0;
    auto magnitude = [&](auto edge) {
#pragma unroll
        for (int i = 0; i < FM; i++) {
            const int row = m0 + wm0 + (TileA::ILV ? 2 * (lane & 31) + i : 32 * i + (lane & 31));
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int n = 8 * (r / 4) + 4 * (lane >> 5) + r % 4;
                    const int col = n0 + wn0 + (TileB::ILV ? 2 * n + j : 32 * j + n);
                    const float v = acc[i][j][r];   // a copy: bit_cast of a vector's element reads element 0
                    unsigned u = __builtin_bit_cast(unsigned, v) & 0x7fffffffu;
                    if constexpr (decltype(edge)::value) u = row < p.M && col < p.N ? u : 0u;
                    top = max(top, u);
                }
        }
    };
    if (m0 + BM <= p.M && n0 + BN <= p.N) magnitude(std::false_type{});
    else magnitude(std::true_type{});
    if (__any(top >= 0x7f800000u)) {
        if constexpr (GLU) {
            const int c0 = (wn0 == 0 ? 0 : p.glu_F) + (n0 >> 1);
            gemm_wave_f32<TA, TB, FM, FN, TileA::ILV, TileB::ILV>(p, A, B, m0 + wm0, [=](int c) { return c0 + c; }, kb,
                                                                  ke, lane, acc);
        } else {
            gemm_wave_f32<TA, TB, FM, FN, TileA::ILV, TileB::ILV>(p, A, B, m0 + wm0,
                                                                  [=](int c) { return n0 + wn0 + c; }, kb, ke, lane,
                                                                  acc);
        }
    }
    if constexpr (GLU && BN == 64) {
        gemm_epilogue_glu(p, acc[0][0], m0 + wm0, tn, wave >> 1, wave & 1, lane, (float*)lds);
    } else if constexpr (GLU) {
        gemm_epilogue_glu2<BM, TileA::ILV>(p, acc, m0 + wm0, tn, wave, lane, (float*)lds);
    } else {
        constexpr bool LDS_STORE = 4 * 32 * (BN / 2) <= 4 * (TileA::UNITS + TileB::UNITS);
        gemm_epilogue<BM, BN, LDS_STORE, TileA::ILV, TileB::ILV, false>(p, C, acc, m0 + wm0, n0 + wn0, lane,
                                                                 (float*)lds + wave * 32 * (BN / 2));
    }
}

#define GEMM_X3(NAME, TA, TB, BM, BN, WPE)                                                        \
    extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE)))   \
    NAME(GemmParams p) {                                                                           \
        gemm_x3_body<TA, TB, BM, BN>(p);                                                           \
    }
#define GEMM_X3_LAYOUTS(TILE, BM, BN, WPE)              \
    GEMM_X3(k_xgemm_nn_##TILE, 0, 0, BM, BN, WPE)        \
    GEMM_X3(k_xgemm_nt_##TILE, 0, 1, BM, BN, WPE)        \
    GEMM_X3(k_xgemm_tn_##TILE, 1, 0, BM, BN, WPE)
GEMM_X3_LAYOUTS(128x128, 128, 128, 3)
GEMM_X3_LAYOUTS(64x128_k32, 64, 128, 4)
GEMM_X3_LAYOUTS(64x64_k32, 64, 64, 5)
// unaligned operands
#define GEMM_X3_U(NAME, TA, TB, BM, BN, WPE)                                                      \
    extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE)))   \
    NAME(GemmParams p) {                                                                           \
        gemm_x3_body<TA, TB, BM, BN, false>(p);                                                    \
    }
GEMM_X3_U(k_xgemm_nn_64x64_u, 0, 0, 64, 64, 5)
GEMM_X3_U(k_xgemm_nt_64x64_u, 0, 1, 64, 64, 5)
GEMM_X3_U(k_xgemm_tn_64x64_u, 1, 0, 64, 64, 5)
GEMM_X3_U(k_xgemm_tt_64x64_u, 1, 1, 64, 64, 5)
GEMM_X3_U(k_xgemm_nn_128x128_u, 0, 0, 128, 128, 3)
GEMM_X3_U(k_xgemm_nt_128x128_u, 0, 1, 128, 128, 3)
GEMM_X3_U(k_xgemm_tn_128x128_u, 1, 0, 128, 128, 3)
// the gate/up projection with the SwiGLU epilogue (host: K % 32 == 0, N = 2F, F a multiple of half the tile)
#define GEMM_X3_GLU(NAME, BM, BN, WPE)                                                            \
    extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE)))   \
    NAME(GemmParams p) {                                                                           \
        gemm_x3_body<0, 0, BM, BN, true, true>(p);                                                       \
    }
GEMM_X3_GLU(k_xgemm_nn_64x64_k32_glu, 64, 64, 5)
GEMM_X3_GLU(k_xgemm_nn_128x128_glu, 128, 128, 3)
