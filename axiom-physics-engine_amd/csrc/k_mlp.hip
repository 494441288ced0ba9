// Warm-start MLP kernels for gfx950: BF16 MFMA forward and backward with fp32
// accumulation, a fixed-order reduction of per-block gradients, and Adam.
//
// MFMA shape: gfx950's v_mfma_f32_16x16x32_bf16 (one wave computes a 16x16 fp32 tile
// from a 16x32 bf16 A and a 32x16 bf16 B tile).  Lane l (r = l % 16, q = l / 16) holds
//   A[r][8q + i], B[8q + i][r] (i = 0..7) and D[4q + i][r] (i = 0..3).
// Hidden activations are staged through LDS between layers (bf16).
// The same rounding points as the CPU oracle's bf16 emulation: inputs and
// weights rounded to bf16 (nearest even), hidden activations rounded after the
// ReLU, propagated hidden gradients rounded before they feed an MFMA.
#include "k_mlp.hpp"

namespace axm {

typedef short bf16x8 __attribute__((ext_vector_type(8)));   // bf16 bit patterns
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t f2bf(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t relu_bf(float v) { return f2bf(v > 0.0f ? v : 0.0f); }

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, a), __builtin_bit_cast(bf16x8v, b), c, 0,
                                                   0, 0);
}
// eight consecutive bf16 (16-byte aligned)
__device__ __forceinline__ bf16x8 ld8(const uint16_t* p) { return *(const bf16x8*)p; }
__device__ __forceinline__ f32x4 splat(float v) {
    f32x4 r;
    r.x = r.y = r.z = r.w = v;
    return r;
}
__device__ __forceinline__ f32x4 ldf4(const float* p) { return *(const f32x4*)p; }
// ReLU and bf16 of one lane's four accumulators (8-byte aligned)
__device__ __forceinline__ void store_relu4(uint16_t* p, f32x4 v) {
    bf16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (short)relu_bf(v[i]);
    *(bf16x4*)p = o;
}

// ---------------------------------------------------------------- casts
__global__ void k_mlp_cast(const float* __restrict__ prm, MlpWeights W) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (uint32_t)(MLP_H * MLP_INP)) {
        const uint32_t o = i / MLP_INP, k = i % MLP_INP;
        W.w1[i] = k < (uint32_t)MLP_IN ? f2bf(prm[MLP_OFF_W1 + o * MLP_IN + k]) : (uint16_t)0;
    }
    if (i < (uint32_t)(MLP_H * MLP_H)) {
        W.w2[i] = f2bf(prm[MLP_OFF_W2 + i]);
        W.w2t[(i % MLP_H) * MLP_H + i / MLP_H] = f2bf(prm[MLP_OFF_W2 + i]);
    }
    if (i < (uint32_t)(MLP_OUTP * MLP_H)) {
        const uint32_t o = i / MLP_H, k = i % MLP_H;
        W.w3[i] = o < (uint32_t)MLP_OUT ? f2bf(prm[MLP_OFF_W3 + o * MLP_H + k]) : (uint16_t)0;
    }
}

// The bf16 inputs of a row as the operand of the one 32-wide k step (k >= 24 padded with 0): lane
// (r, q) reads the row's inputs 8q .. 8q+7.
__device__ __forceinline__ void load_x(const float* __restrict__ X, uint32_t n, uint32_t row, int q, f32x4 x[2]) {
    x[0] = x[1] = splat(0.0f);
    if (row < n && q < MLP_IN / 8) {
        const float* p = X + (size_t)row * MLP_IN + 8 * q;  // 32-byte aligned
        x[0] = ldf4(p);
        x[1] = ldf4(p + 4);
    }
}
__device__ __forceinline__ bf16x8 cast_x(const f32x4 x[2]) {
    bf16x8 a;
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = (short)f2bf(x[i >> 2][i & 3]);
    return a;
}

// ---------------------------------------------------------------- forward
// Every product is taken as weights x activations, so a lane's four accumulators are four
// consecutive units of one row: 8-byte stores into row-major activations.  LDS rows are padded by
// 8 units: the 16 rows of an operand read start in different banks (unpadded, all of them in one).
// A wave takes 32 rows at a time, so each weight it reads from LDS feeds two products, and waves
// share nothing after the weights: no barrier in the loop, the next rows' inputs on the way.
// LDS-bound (per 32 rows 45 KB of weights and 35 KB of activations per wave).
// 4M rows: 0.28 ms; with unpadded rows, 16 rows a wave and a barrier between the layers 1.23 ms.
constexpr int F_W1 = MLP_INP + 8, F_H = MLP_H + 8;  // padded LDS rows (units)
constexpr int F_WAVES = 8, F_TILE = 32;             // waves of a block, rows of a wave at a time
constexpr size_t F_OFF_W2 = 2 * MLP_H * F_W1, F_OFF_W3 = F_OFF_W2 + 2 * MLP_H * F_H,
                 F_OFF_B = F_OFF_W3 + 2 * MLP_OUTP * F_H, F_OFF_ACT = F_OFF_B + 4 * (2 * MLP_H + 4),
                 F_LDS = F_OFF_ACT + 2 * F_WAVES * F_TILE * F_H;

__global__ void __launch_bounds__(64 * F_WAVES) k_mlp_forward(MlpDev P, const float* __restrict__ X, uint32_t n_cap,
                                                              const uint32_t* __restrict__ n_dev, uint32_t n_mul,
                                                              float* __restrict__ Y) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint16_t* sW1 = (uint16_t*)smem;
    uint16_t* sW2 = (uint16_t*)(smem + F_OFF_W2);
    uint16_t* sW3 = (uint16_t*)(smem + F_OFF_W3);
    float* sB = (float*)(smem + F_OFF_B);
    uint32_t n = n_cap;
    if (n_dev) {
        const uint64_t v = (uint64_t)(*n_dev) * n_mul;
        n = v < n_cap ? (uint32_t)v : n_cap;
    }
    const uint32_t tiles = n / F_TILE + (n % F_TILE ? 1u : 0u);
    if (blockIdx.x >= tiles) return;  // uniform per block
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    uint32_t t = blockIdx.x + gridDim.x * wave;  // tiles go to the blocks in turn, then to their waves
    f32x4 x[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) load_x(X, t < tiles ? n : 0u, F_TILE * t + 16 * h + r, q, x[h]);
    for (uint32_t i = threadIdx.x; i < (uint32_t)(MLP_H * MLP_INP / 8); i += blockDim.x)
        *(bf16x8*)&sW1[i / (MLP_INP / 8) * F_W1 + i % (MLP_INP / 8) * 8] = ld8(P.w1 + 8 * i);
    for (uint32_t i = threadIdx.x; i < (uint32_t)(MLP_H * MLP_H / 8); i += blockDim.x)
        *(bf16x8*)&sW2[i / (MLP_H / 8) * F_H + i % (MLP_H / 8) * 8] = ld8(P.w2 + 8 * i);
    for (uint32_t i = threadIdx.x; i < (uint32_t)(MLP_OUTP * MLP_H / 8); i += blockDim.x)
        *(bf16x8*)&sW3[i / (MLP_H / 8) * F_H + i % (MLP_H / 8) * 8] = ld8(P.w3 + 8 * i);
    if (threadIdx.x < (uint32_t)MLP_H) {
        sB[threadIdx.x] = P.prm[MLP_OFF_B1 + threadIdx.x];
        sB[MLP_H + threadIdx.x] = P.prm[MLP_OFF_B2 + threadIdx.x];
    }
    if (threadIdx.x < 4u) sB[2 * MLP_H + threadIdx.x] = threadIdx.x < (uint32_t)MLP_OUT ? P.prm[MLP_OFF_B3 + threadIdx.x] : 0.0f;
    __syncthreads();
    uint16_t* act = (uint16_t*)(smem + F_OFF_ACT) + wave * F_TILE * F_H;
    // a wave's own LDS accesses complete in order; this keeps the compiler from moving them
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    for (; t < tiles; t += gridDim.x * F_WAVES) {
        const bf16x8 a0 = cast_x(x[0]), a1 = cast_x(x[1]);
        const uint32_t tn = tiles - t > gridDim.x * F_WAVES ? t + gridDim.x * F_WAVES : 0u;
#pragma unroll
        for (int h = 0; h < 2; ++h) load_x(X, tn ? n : 0u, F_TILE * tn + 16 * h + r, q, x[h]);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bf16x8 w = ld8(&sW1[(16 * j + r) * F_W1 + 8 * q]);
            const f32x4 b = ldf4(&sB[16 * j + 4 * q]);
            store_relu4(&act[r * F_H + 16 * j + 4 * q], mfma32(w, a0, b));
            store_relu4(&act[(16 + r) * F_H + 16 * j + 4 * q], mfma32(w, a1, b));
        }
        wave_sync();
        f32x4 acc[2][8];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[0][j] = acc[1][j] = ldf4(&sB[MLP_H + 16 * j + 4 * q]);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const bf16x8 h0 = ld8(&act[r * F_H + 32 * kk + 8 * q]), h1 = ld8(&act[(16 + r) * F_H + 32 * kk + 8 * q]);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const bf16x8 w = ld8(&sW2[(16 * j + r) * F_H + 32 * kk + 8 * q]);
                acc[0][j] = mfma32(w, h0, acc[0][j]);
                acc[1][j] = mfma32(w, h1, acc[1][j]);
            }
        }
        wave_sync();
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            store_relu4(&act[r * F_H + 16 * j + 4 * q], acc[0][j]);
            store_relu4(&act[(16 + r) * F_H + 16 * j + 4 * q], acc[1][j]);
        }
        wave_sync();
        const f32x4 b3 = q == 0 ? ldf4(&sB[2 * MLP_H]) : splat(0.0f);
        f32x4 y[2] = {b3, b3};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const bf16x8 w = ld8(&sW3[r * F_H + 32 * kk + 8 * q]);
            y[0] = mfma32(w, ld8(&act[r * F_H + 32 * kk + 8 * q]), y[0]);
            y[1] = mfma32(w, ld8(&act[(16 + r) * F_H + 32 * kk + 8 * q]), y[1]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t row = F_TILE * t + 16 * h + r;
            if (q == 0 && row < n) {
                float* o = Y + (size_t)row * MLP_OUT;
                o[0] = y[h][0];
                o[1] = y[h][1];
                o[2] = y[h][2];
            }
        }
        wave_sync();
    }
}

// ---------------------------------------------------------------- backward
// One block of 16 waves takes 64 rows at a time; a wave owns unit tile j = wave % 8 and half of the
// row tiles (forward, d1) or of the input tiles (dW), so its weights stay in registers, read
// straight from memory.  The backward products contract over rows and need the activations with
// rows consecutive: each forward tile is computed both ways round (the products are too few to
// matter: a lane's four accumulators are four rows one way and four units the other), so every
// store is 8 bytes and every operand read 16, from rows padded by 8 against bank conflicts.
// A pass of 64 rows takes 9 us, most of it waits at the seven barriers and the two serial sums; a
// batch of 4096 rows (64 blocks) 14.7 us.  With 4 waves, weights staged in LDS and operands
// gathered two bytes at a time a batch, its update included, took 58 us, now 19.
constexpr int G_THREADS = 1024;
constexpr int G_ROW = MLP_H + 8, G_COL = MLP_ROWS_PER_BLOCK + 8;  // padded rows: [row][unit], [unit][row]
constexpr size_t G_SZ_ROW = 2 * MLP_ROWS_PER_BLOCK * G_ROW, G_SZ_COL = 2 * MLP_H * G_COL;
constexpr size_t G_OFF_H1T = G_SZ_ROW, G_OFF_H2 = G_OFF_H1T + G_SZ_COL, G_OFF_H2T = G_OFF_H2 + G_SZ_ROW,
                 G_OFF_D2T = G_OFF_H2T + G_SZ_COL, G_OFF_D1T = G_OFF_D2T + G_SZ_COL, G_OFF_XT = G_OFF_D1T + G_SZ_COL,
                 G_OFF_DY = G_OFF_XT + 2 * MLP_INP * G_COL, G_OFF_W3F = G_OFF_DY + 4 * MLP_OUT * MLP_ROWS_PER_BLOCK,
                 G_OFF_LOSS = G_OFF_W3F + 4 * MLP_OUT * MLP_H, G_LDS = G_OFF_LOSS + 8 * 4;

// Sum of a unit's 64 rows, in row order, added to s.
__device__ __forceinline__ float add_rows(float s, const uint16_t* p) {
#pragma unroll 4
    for (int c = 0; c < MLP_ROWS_PER_BLOCK; c += 8) {
        const bf16x8 v = ld8(p + c);
#pragma unroll
        for (int i = 0; i < 8; ++i) s += bf2f((uint16_t)v[i]);
    }
    return s;
}
// relu'(h) * bf16(sum_o w[o] dy[o])
__device__ __forceinline__ uint16_t back3(uint16_t h, float w0, float w1, float w2, float e0, float e1, float e2) {
    float s = 0.0f;
    s += w0 * e0;
    s += w1 * e1;
    s += w2 * e2;
    return bf2f(h) > 0.0f ? f2bf(s) : (uint16_t)0;
}

__global__ void __launch_bounds__(G_THREADS) k_mlp_grad(MlpDev P, const float* __restrict__ X,
                                                        const float* __restrict__ Yt, uint32_t n, float scale,
                                                        float* __restrict__ partial, double* __restrict__ loss_partial) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint16_t* sH1 = (uint16_t*)smem;
    uint16_t* sH1T = (uint16_t*)(smem + G_OFF_H1T);
    uint16_t* sH2 = (uint16_t*)(smem + G_OFF_H2);  // h2, then d2
    uint16_t* sH2T = (uint16_t*)(smem + G_OFF_H2T);
    uint16_t* sD2T = (uint16_t*)(smem + G_OFF_D2T);
    uint16_t* sD1T = (uint16_t*)(smem + G_OFF_D1T);
    uint16_t* sXT = (uint16_t*)(smem + G_OFF_XT);
    float* sdy = (float*)(smem + G_OFF_DY);    // [3][64]
    float* sW3f = (float*)(smem + G_OFF_W3F);  // [3][128]
    double* sLoss = (double*)(smem + G_OFF_LOSS);
    constexpr int ROWS = MLP_ROWS_PER_BLOCK;
    int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    int r = lane & 15, q = lane >> 4;
    const int j = wave & 7, half = wave >> 3;
    if (tid < MLP_OUT * MLP_H) sW3f[tid] = bf2f(P.w3[tid]);
    // biases of the wave's tile, of unit r and of units 4q .. 4q+3
    const float b1 = P.prm[MLP_OFF_B1 + 16 * j + r], b2 = P.prm[MLP_OFF_B2 + 16 * j + r];
    const float b3 = r < MLP_OUT ? P.prm[MLP_OFF_B3 + r] : 0.0f;
    f32x4 b1v, b2v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        b1v[i] = P.prm[MLP_OFF_B1 + 16 * j + 4 * q + i];
        b2v[i] = P.prm[MLP_OFF_B2 + 16 * j + 4 * q + i];
    }
    f32x4 gW2[4], gW1 = splat(0.0f);
#pragma unroll
    for (int b = 0; b < 4; ++b) gW2[b] = splat(0.0f);
    float g3 = 0.0f, gb = 0.0f;  // dW3 (waves 10-15); db2 (waves 8, 9), db1 (waves 0, 1) or db3 (wave 2)
    double lossacc = 0.0;
    for (uint32_t base = blockIdx.x * ROWS; base < n; base += gridDim.x * ROWS) {
        // Weights are loaded in each pass, well before their use, and addresses formed anew: held over the
        // passes they would spill (the empty asm keeps them in the loop).
        const uint16_t *pw1 = P.w1, *pw2 = P.w2, *pw2t = P.w2t, *pw3 = P.w3;
        asm volatile("" : "+s"(pw1), "+s"(pw2), "+s"(pw2t), "+s"(pw3), "+v"(r), "+v"(q), "+v"(tid));
        const bf16x8 w1 = ld8(pw1 + (16 * j + r) * MLP_INP + 8 * q);
        bf16x8 w2[4], w2t[4], w3[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) w2[kk] = ld8(pw2 + (16 * j + r) * MLP_H + 32 * kk + 8 * q);
        // ---- forward
        float yt[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (wave < 4 && r < MLP_OUT) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t row = base + 16 * wave + 4 * q + i;
                if (row < n) yt[i] = Yt[(size_t)row * MLP_OUT + r];
            }
        }
        f32x4 x[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) load_x(X, n, base + 16 * (2 * half + h) + r, q, x[h]);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = 16 * (2 * half + h);
            const bf16x8 a = cast_x(x[h]);
            if (j == 0) {
#pragma unroll
                for (int i = 0; i < 8; ++i) sXT[(8 * q + i) * G_COL + row + r] = (uint16_t)a[i];
            }
            store_relu4(&sH1T[(16 * j + r) * G_COL + row + 4 * q], mfma32(a, w1, splat(b1)));
            store_relu4(&sH1[(row + r) * G_ROW + 16 * j + 4 * q], mfma32(w1, a, b1v));
        }
        if (wave < 4) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) w3[kk] = ld8(pw3 + r * MLP_H + 32 * kk + 8 * q);
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) w2t[kk] = ld8(pw2t + (16 * j + r) * MLP_H + 32 * kk + 8 * q);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = 16 * (2 * half + h);
            f32x4 acc = splat(b2), accv = b2v;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const bf16x8 a = ld8(&sH1[(row + r) * G_ROW + 32 * kk + 8 * q]);
                acc = mfma32(a, w2[kk], acc);
                accv = mfma32(w2[kk], a, accv);
            }
            store_relu4(&sH2T[(16 * j + r) * G_COL + row + 4 * q], acc);
            store_relu4(&sH2[(row + r) * G_ROW + 16 * j + 4 * q], accv);
        }
        __syncthreads();
        if (wave < 4) {
            f32x4 y = splat(b3);
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) y = mfma32(ld8(&sH2[(16 * wave + r) * G_ROW + 32 * kk + 8 * q]), w3[kk], y);
            if (r < MLP_OUT) {
                f32x4 d = splat(0.0f);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (base + 16 * wave + 4 * q + i < n) {
                        const float e = y[i] - yt[i];
                        lossacc += (double)e * (double)e;
                        d[i] = e * scale;
                    }
                }
                *(f32x4*)&sdy[r * ROWS + 16 * wave + 4 * q] = d;
            }
        }
        __syncthreads();
        // ---- d2 = relu'(h2) * bf16(W3^T dy), both ways round: 8 units of a row (in place of h2) and
        // 8 rows of a unit for each thread
        {
            const int row = tid >> 4, k = (tid & 15) * 8;
            bf16x8 h = ld8(&sH2[row * G_ROW + k]);
            const float e0 = sdy[row], e1 = sdy[ROWS + row], e2 = sdy[2 * ROWS + row];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const f32x4 v0 = ldf4(&sW3f[k + 4 * p]), v1 = ldf4(&sW3f[MLP_H + k + 4 * p]),
                            v2 = ldf4(&sW3f[2 * MLP_H + k + 4 * p]);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    h[4 * p + i] = (short)back3((uint16_t)h[4 * p + i], v0[i], v1[i], v2[i], e0, e1, e2);
            }
            *(bf16x8*)&sH2[row * G_ROW + k] = h;
        }
        {
            const int k = tid >> 3, row = (tid & 7) * 8;
            bf16x8 h = ld8(&sH2T[k * G_COL + row]);
            const float v0 = sW3f[k], v1 = sW3f[MLP_H + k], v2 = sW3f[2 * MLP_H + k];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const f32x4 e0 = ldf4(&sdy[row + 4 * p]), e1 = ldf4(&sdy[ROWS + row + 4 * p]),
                            e2 = ldf4(&sdy[2 * ROWS + row + 4 * p]);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    h[4 * p + i] = (short)back3((uint16_t)h[4 * p + i], v0, v1, v2, e0[i], e1[i], e2[i]);
            }
            *(bf16x8*)&sD2T[k * G_COL + row] = h;
        }
        __syncthreads();
        // ---- d1 = relu'(h1) * bf16(d2 W2), units by rows
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = 16 * (2 * half + h);
            f32x4 d = splat(0.0f);
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) d = mfma32(ld8(&sH2[(row + r) * G_ROW + 32 * kk + 8 * q]), w2t[kk], d);
            bf16x4 v = *(const bf16x4*)&sH1T[(16 * j + r) * G_COL + row + 4 * q];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = (short)(bf2f((uint16_t)v[i]) > 0.0f ? f2bf(d[i]) : (uint16_t)0);
            *(bf16x4*)&sD1T[(16 * j + r) * G_COL + row + 4 * q] = v;
        }
        // ---- layer 2: dW2[o][k] += sum_r d2[r][o] h1[r][k]
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const bf16x8 a = ld8(&sD2T[(16 * j + r) * G_COL + 32 * c + 8 * q]);
#pragma unroll
            for (int b = 0; b < 4; ++b)
                gW2[b] = mfma32(a, ld8(&sH1T[(16 * (4 * half + b) + r) * G_COL + 32 * c + 8 * q]), gW2[b]);
        }
        // ---- layer 3: dW3 += dy^T h2, db3 += dy, db2 += d2, rows in order
        if (wave >= 10) {
            const int o = (wave - 10) >> 1, k = (tid - 640) & (MLP_H - 1);
#pragma unroll 2
            for (int c = 0; c < ROWS; c += 8) {
                const bf16x8 v = ld8(&sH2T[k * G_COL + c]);
                const f32x4 e0 = ldf4(&sdy[o * ROWS + c]), e1 = ldf4(&sdy[o * ROWS + c + 4]);
#pragma unroll
                for (int i = 0; i < 8; ++i) g3 += (i < 4 ? e0[i & 3] : e1[i & 3]) * bf2f((uint16_t)v[i]);
            }
        } else if (wave >= 8) {
            gb = add_rows(gb, &sD2T[(tid - 512) * G_COL]);
        } else if (wave == 2 && lane < MLP_OUT) {
#pragma unroll 4
            for (int rr = 0; rr < ROWS; rr += 4) {
                const f32x4 e = ldf4(&sdy[lane * ROWS + rr]);
#pragma unroll
                for (int i = 0; i < 4; ++i) gb += e[i];
            }
        }
        __syncthreads();
        // ---- layer 1: dW1[o][k] += sum_r d1[r][o] x[r][k], db1 += d1
#pragma unroll
        for (int c = 0; c < 2; ++c)
            gW1 = mfma32(ld8(&sD1T[(16 * j + r) * G_COL + 32 * c + 8 * q]),
                         ld8(&sXT[(16 * half + r) * G_COL + 32 * c + 8 * q]), gW1);
        if (wave < 2) gb += add_rows(0.0f, &sD1T[tid * G_COL]);
        __syncthreads();
    }
    // ---- per-block partials
    float* out = partial + (size_t)blockIdx.x * MLP_NPARAM;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            out[MLP_OFF_W2 + (16 * j + 4 * q + i) * MLP_H + 16 * (4 * half + b) + r] = gW2[b][i];
    if (16 * half + r < MLP_IN) {
#pragma unroll
        for (int i = 0; i < 4; ++i) out[MLP_OFF_W1 + (16 * j + 4 * q + i) * MLP_IN + 16 * half + r] = gW1[i];
    }
    if (wave < 2) out[MLP_OFF_B1 + tid] = gb;
    else if (wave == 2 && lane < MLP_OUT) out[MLP_OFF_B3 + lane] = gb;
    else if (wave == 8 || wave == 9) out[MLP_OFF_B2 + tid - 512] = gb;
    else if (wave >= 10) out[MLP_OFF_W3 + tid - 640] = g3;
    // block sum of the loss (fixed order)
    if (wave < 4) {
        for (int o = 32; o >= 1; o >>= 1) lossacc += __shfl_xor(lossacc, o, 64);
        if (lane == 0) sLoss[wave] = lossacc;
    }
    __syncthreads();
    if (tid == 0) loss_partial[blockIdx.x] = ((sLoss[0] + sLoss[1]) + sLoss[2]) + sLoss[3];
}

// The update of one parameter per thread: the gradient, either the blocks' partials summed in block
// order (kept in grad) or as given, then with ADAM the step of the fp32 parameter and its bf16 copies.
// One wave per block spreads the 20,099 chains of loads over the chip; sixteen loads are in
// flight in each.  The last block sums the blocks' losses.
// 4.2 us for 64 partials (5.1 MB); as a reduction, a step and a cast in three launches 12.
template <bool REDUCE, bool ADAM>
__global__ void __launch_bounds__(64) k_mlp_update(const float* __restrict__ partial, uint32_t blocks,
                                                   const double* __restrict__ loss_partial, double inv_count,
                                                   float* __restrict__ grad, double* __restrict__ loss,
                                                   float* __restrict__ prm, float* __restrict__ m, float* __restrict__ v,
                                                   MlpWeights W, MlpAdam A) {
    const uint32_t i = blockIdx.x * 64u + threadIdx.x;
    if (REDUCE && blockIdx.x + 1u == gridDim.x) {
        double s = 0.0;
        for (uint32_t b = threadIdx.x; b < blocks; b += 64u) s += loss_partial[b];
        for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
        if (threadIdx.x == 0u) *loss = s * inv_count;
        return;
    }
    if (i >= (uint32_t)MLP_NPARAM) return;
    float p0 = 0.0f, m0 = 0.0f, v0 = 0.0f;
    if (ADAM) {
        p0 = prm[i];
        m0 = m[i];
        v0 = v[i];
    }
    float gi = 0.0f;
    if (REDUCE) {
        const float* p = partial + i;
        uint32_t b = 0;
        for (; b + 16u <= blocks; b += 16u) {
            float t[16];
#pragma unroll
            for (uint32_t k = 0; k < 16u; ++k) t[k] = p[(size_t)(b + k) * MLP_NPARAM];
#pragma unroll
            for (uint32_t k = 0; k < 16u; ++k) gi += t[k];
        }
        for (; b < blocks; ++b) gi += p[(size_t)b * MLP_NPARAM];
        grad[i] = gi;
    } else {
        gi = grad[i];
    }
    if (!ADAM) return;
    const float mi = A.b1 * m0 + (1.0f - A.b1) * gi;
    const float vi = A.b2 * v0 + (1.0f - A.b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / A.c1;
    const float vh = vi / A.c2;
    const float pi = p0 - A.lr * mh / (sqrtf(vh) + A.eps);
    prm[i] = pi;
    const uint16_t h = f2bf(pi);
    if (i < (uint32_t)MLP_OFF_B1) {
        W.w1[i / MLP_IN * MLP_INP + i % MLP_IN] = h;
    } else if (i >= (uint32_t)MLP_OFF_W2 && i < (uint32_t)MLP_OFF_B2) {
        const uint32_t e = i - MLP_OFF_W2;
        W.w2[e] = h;
        W.w2t[e % MLP_H * MLP_H + e / MLP_H] = h;
    } else if (i >= (uint32_t)MLP_OFF_W3 && i < (uint32_t)MLP_OFF_B3) {
        W.w3[i - MLP_OFF_W3] = h;
    }
}

// ---------------------------------------------------------------- launchers
void launch_mlp_cast(const float* prm, const MlpWeights& W, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_cast, dim3((MLP_H * MLP_H + 255) / 256), dim3(256), 0, s, prm, W);
}

void launch_mlp_forward(const MlpDev& P, const float* X, uint32_t n_cap, const uint32_t* n_dev, uint32_t n_mul,
                        float* Y, uint32_t blocks, hipStream_t s) {
    if (n_cap == 0) return;
    const uint32_t need = n_cap / F_TILE + (n_cap % F_TILE ? 1u : 0u);
    const uint32_t g = blocks < need ? blocks : need;
    hipLaunchKernelGGL(k_mlp_forward, dim3(g ? g : 1), dim3(64 * F_WAVES), F_LDS, s, P, X, n_cap, n_dev, n_mul, Y);
}

size_t mlp_grad_partial_floats(uint32_t blocks) { return (size_t)blocks * MLP_NPARAM; }

hipError_t mlp_prepare_device() {
    const hipError_t e =
        hipFuncSetAttribute((const void*)k_mlp_forward, hipFuncAttributeMaxDynamicSharedMemorySize, (int)F_LDS);
    if (e != hipSuccess) return e;
    return hipFuncSetAttribute((const void*)k_mlp_grad, hipFuncAttributeMaxDynamicSharedMemorySize, (int)G_LDS);
}

void launch_mlp_grad(const MlpTrain& T, const float* X, const float* Y, uint32_t n, double* loss, const MlpAdam* adam,
                     hipStream_t s) {
    const uint32_t need = n / MLP_ROWS_PER_BLOCK + (n % MLP_ROWS_PER_BLOCK ? 1u : 0u);
    const uint32_t g = T.blocks < need ? T.blocks : need;
    const float scale = 2.0f / (float)((double)n * MLP_OUT);
    const double inv = 1.0 / ((double)n * MLP_OUT);
    const dim3 u((MLP_NPARAM + 63) / 64 + 1);
    hipLaunchKernelGGL(k_mlp_grad, dim3(g), dim3(G_THREADS), G_LDS, s, MlpDev{T.prm, T.W.w1, T.W.w2, T.W.w2t, T.W.w3}, X, Y,
                       n, scale, T.partial, T.loss_partial);
    if (adam)
        hipLaunchKernelGGL((k_mlp_update<true, true>), u, dim3(64), 0, s, T.partial, g, T.loss_partial, inv, T.grad, loss,
                           T.prm, T.m, T.v, T.W, *adam);
    else
        hipLaunchKernelGGL((k_mlp_update<true, false>), u, dim3(64), 0, s, T.partial, g, T.loss_partial, inv, T.grad, loss,
                           T.prm, T.m, T.v, T.W, MlpAdam{});
}

void launch_mlp_adam(const MlpTrain& T, const MlpAdam& adam, hipStream_t s) {
    hipLaunchKernelGGL((k_mlp_update<false, true>), dim3((MLP_NPARAM + 63) / 64), dim3(64), 0, s, T.partial, 0u,
                       T.loss_partial, 0.0, T.grad, (double*)nullptr, T.prm, T.m, T.v, T.W, adam);
}

}  // namespace axm
