// mlp_hip.hip — learned front-end: a syndrome -> logical-class MLP with
// hand-written HIP training and inference kernels for gfx950.
//
// Network: x (n_in bits, zero-padded to a multiple of 32) -> 3 hidden layers
// (ReLU) -> n_out logits.  Weights are kept in FP32 (master copy, Adam) and
// in BF16 (the copy every GEMM reads); activations are BF16; every product is
// accumulated in FP32 by v_mfma_f32_32x32x16_bf16.  Training minimises the
// soft cross-entropy against class posteriors produced by the tensor-network
// decoder.  A confidence gate accepts the network's class when its posterior
// reaches a threshold and queues the other syndromes for the TN path.
//
// This component has no counterpart in the reference (TensorQEC.jl has no
// learned decoder); it sits in front of the TNMMAP path
// (src/decoding/tndecoder.jl:160-165) and falls back to it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "tqec_hip.h"

namespace tqec {
int set_error_shared(int code, const std::string &msg);
}

namespace {

int fail(int code, const std::string &m) { return tqec::set_error_shared(code, m); }

#define TQM_HIP(call)                                                                                     \
    do {                                                                                                  \
        hipError_t e_ = (call);                                                                           \
        if (e_ != hipSuccess) return fail(TQEC_EDEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

typedef uint16_t bf16;
typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

__device__ __forceinline__ float bf2f(bf16 h) { return __uint_as_float(((uint32_t)h) << 16); }
// Round to nearest even, one v_cvt_pk_bf16_f32 for two values (rounding in
// integer arithmetic, five instructions a value, made the fused forward kernel
// 73.6 us instead of 67.5 at 65,536 rows of 48 inputs).
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bfx2;
__device__ __forceinline__ uint32_t f2bf2(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bfx2));
}
__device__ __forceinline__ bf16 f2bf(float f) { return (bf16)f2bf2(f, 0.f); }

// ---------------------------------------------------------------------------
// Backward GEMM of the layer-by-layer path: C[M][N] = A[M][K] * B^T (B[n*ldb +
// k]) where mask > 0, BF16 in and out, FP32 accumulate.  Block tile 128x128, K
// step 32, 4 waves each owning 64x64 = 2x2 MFMA tiles of 32x32.  Tiles are
// staged in LDS as [row][k] (k contiguous) so each lane reads its 8
// consecutive k values with one 16-byte LDS load.  Rows beyond M/N are
// zero-filled on load and skipped on store; K must be a multiple of 32.
// ---------------------------------------------------------------------------

struct GemmArgs {
    const bf16 *A;
    const bf16 *B;
    int M, N, K, lda, ldb, ldc;
    const bf16 *mask;
    bf16 *outb;
};

constexpr int BM = 128, BN = 128, BK = 32, LDSK = BK + 8;

// S[r][k] for r in [0,128), k in [0,32) of G[r*ld + k]: 512 chunks of 8
__device__ __forceinline__ void load_tile(bf16 *S, const bf16 *G, int rows0, int R, int k0, int ld, int tid) {
    for (int c = tid; c < 512; c += 256) {
        const int r = c >> 2, kc = (c & 3) * 8;
        const int gr = rows0 + r;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (gr < R) v = *reinterpret_cast<const uint4 *>(G + (size_t)gr * ld + k0 + kc);
        *reinterpret_cast<uint4 *>(S + r * LDSK + kc) = v;
    }
}

__global__ void __launch_bounds__(256) gemm_bf16_kernel(GemmArgs g) {
    __shared__ __align__(16) bf16 As[BM * LDSK];
    __shared__ __align__(16) bf16 Bs[BN * LDSK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    f32x16 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    for (int k0 = 0; k0 < g.K; k0 += BK) {
        load_tile(As, g.A, m0, g.M, k0, g.lda, tid);
        load_tile(Bs, g.B, n0, g.N, k0, g.ldb, tid);
        __syncthreads();
        for (int kk = 0; kk < BK; kk += 16) {
            bf16x8 a[2], b[2];
            for (int i = 0; i < 2; ++i)
                a[i] = *reinterpret_cast<const bf16x8 *>(As + (wm + i * 32 + (lane & 31)) * LDSK + kk + 8 * (lane >> 5));
            for (int j = 0; j < 2; ++j)
                b[j] = *reinterpret_cast<const bf16x8 *>(Bs + (wn + j * 32 + (lane & 31)) * LDSK + kk + 8 * (lane >> 5));
            for (int i = 0; i < 2; ++i)
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // D layout of the 32x32 tile: lane l holds column l%32, value v is row
    // 8*(v/4) + 4*(l/32) + v%4.
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) {
            const int col = n0 + wn + j * 32 + (lane & 31);
            if (col >= g.N) continue;
            for (int v = 0; v < 16; ++v) {
                const int row = m0 + wm + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (row >= g.M) continue;
                const size_t o = (size_t)row * g.ldc + col;
                g.outb[o] = bf2f(g.mask[o]) > 0.f ? f2bf(acc[i][j][v]) : (bf16)0;
            }
        }
}

// Forward GEMM of a hidden layer: H[M][N] = relu(A[M][K] * W + bias) with
// the weights given transposed, Wt[N][K], so both tiles are rows of 16-byte
// k-chunks.  Block tile 128 x 128, K step KS (64, or 32 when K is not a
// multiple of 64), 4 waves in a 2 x 2 grid each owning 64 x 64 = 2 x 2 MFMA
// tiles (64 x 128 were slower: one wave per SIMD); the next K step's tiles are
// loaded into registers while the current one is multiplied out of LDS.  Same
// MFMA sequence (k ascending in steps of 16) as gemm_bf16_kernel, so the
// results are identical.  The biases are loaded in front of the K loop and the
// outputs rounded in front of the branches around their stores: a bias waited
// for after a store is a wait for that store, too (loads and stores share a
// counter).  Forward pass of 65,536 rows of 48 inputs, width 512: 189 us, 254
// with each output biased, rounded and stored in a branch of its own (width
// 1024: 691 and 823, width 256: 130 and 165).
template <int KS>
__global__ void __launch_bounds__(256) gemm_fwd_kernel(const bf16 *__restrict__ A, const bf16 *__restrict__ Wt,
                                                       int M, int N, int K, const float *__restrict__ bias,
                                                       bf16 *__restrict__ out) {
    constexpr int NW = 2, TN = 64 * NW;        // MFMA tiles per wave, block tile columns
    constexpr int LK = KS + 8;                 // padded LDS row (bf16)
    constexpr int PA = 128 * KS / 8 / 256;     // 16-byte chunks per thread: A tile
    constexpr int PB = TN * KS / 8 / 256;      //                             B tile
    __shared__ __align__(16) bf16 As[128 * LK];
    __shared__ __align__(16) bf16 Bs[TN * LK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * 128, n0 = blockIdx.x * TN;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * (32 * NW);
    uint4 ra[PA], rb[PB];
    auto fetch = [&](int k0) {
        for (int j = 0; j < PA; ++j) {
            const int c = tid + j * 256;
            const int r = c / (KS / 8), kc = (c % (KS / 8)) * 8;
            const int gm = m0 + r;
            ra[j] = gm < M ? *reinterpret_cast<const uint4 *>(A + (size_t)gm * K + k0 + kc) : make_uint4(0, 0, 0, 0);
        }
        for (int j = 0; j < PB; ++j) {
            const int c = tid + j * 256;
            const int r = c / (KS / 8), kc = (c % (KS / 8)) * 8;
            const int gn = n0 + r;
            rb[j] = gn < N ? *reinterpret_cast<const uint4 *>(Wt + (size_t)gn * K + k0 + kc) : make_uint4(0, 0, 0, 0);
        }
    };
    auto stash = [&]() {
        for (int j = 0; j < PA; ++j) {
            const int c = tid + j * 256;
            *reinterpret_cast<uint4 *>(As + (c / (KS / 8)) * LK + (c % (KS / 8)) * 8) = ra[j];
        }
        for (int j = 0; j < PB; ++j) {
            const int c = tid + j * 256;
            *reinterpret_cast<uint4 *>(Bs + (c / (KS / 8)) * LK + (c % (KS / 8)) * 8) = rb[j];
        }
    };
    f32x16 acc[2][NW];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < NW; ++j)
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    float bc[NW];
    for (int j = 0; j < NW; ++j) bc[j] = bias[min(n0 + wn + j * 32 + (lane & 31), N - 1)];
    fetch(0);
    stash();
    __syncthreads();
    for (int k0 = 0; k0 < K; k0 += KS) {
        const bool more = k0 + KS < K;
        if (more) fetch(k0 + KS);
        for (int kk = 0; kk < KS; kk += 16) {
            bf16x8 a[2], b[NW];
            for (int i = 0; i < 2; ++i)
                a[i] = *reinterpret_cast<const bf16x8 *>(As + (wm + i * 32 + (lane & 31)) * LK + kk + 8 * (lane >> 5));
            for (int j = 0; j < NW; ++j)
                b[j] = *reinterpret_cast<const bf16x8 *>(Bs + (wn + j * 32 + (lane & 31)) * LK + kk + 8 * (lane >> 5));
            for (int i = 0; i < 2; ++i)
                for (int j = 0; j < NW; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
        if (more) {
            stash();
            __syncthreads();
        }
    }
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < NW; ++j) {
            const int col = n0 + wn + j * 32 + (lane & 31);
            // in pairs, and before the branches around the stores
            uint32_t u[8];
#pragma unroll
            for (int v = 0; v < 8; ++v)
                u[v] = f2bf2(fmaxf(acc[i][j][2 * v] + bc[j], 0.f), fmaxf(acc[i][j][2 * v + 1] + bc[j], 0.f));
            if (col >= N) continue;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = m0 + wm + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (row < M) out[(size_t)row * N + col] = (bf16)(u[v >> 1] >> (16 * (v & 1)));
            }
        }
}

// ---------------------------------------------------------------------------
// Fused inference: the whole network for a tile of 128 syndromes in one
// workgroup, hidden width 512.  The tile's activations stay in LDS
// (128 x 512 BF16 = 128 KB, rows of 64 16-byte chunks, chunk c of row m
// stored at c ^ (m & 15) so that the 16 lanes of a ds_read_b128 pass hit
// distinct banks) and each layer overwrites them in place after a barrier.
// Every product runs on v_mfma_f32_32x32x16_bf16 with the operands swapped
// (D = W^T * act^T): wave w owns output columns [w * 512 / NW, ...) for all
// 128 rows, so no two waves read the same weights and each wave streams its
// weight fragments straight from global memory (L2-resident, 1.1 MB for the
// d=7 network) in the fragment order laid out once by pack_fused_kernel,
// two k-steps ahead; only the activations are shared, with no barrier inside
// a layer.  A lane of a D tile holds 4 consecutive output columns of one
// row, written back as one 8-byte LDS store per group.  Biases seed the
// accumulators.  The output layer (N <= 32, padded) runs the same way with
// one wave per 32 rows.  FP32 accumulation, BF16 activations, as the
// layer-by-layer kernels (same roundings; the bias enters before the
// products instead of after them).
// ---------------------------------------------------------------------------

constexpr int kFusedRows = 128, kFusedHid = 512;

__device__ __forceinline__ int act_off(int m, int chunk) { return m * (kFusedHid * 2) + ((chunk ^ (m & 15)) << 4); }

// Fragment-ordered weights, all of them in one launch.  Forward (wf), hidden
// layer l (K x 512): for each 16-row k-step s and 32-column tile t, 64 lanes x
// 8 BF16: lane L holds W[16 s + 8 (L >> 5) + e][32 t + (L & 31)], e = 0..7;
// output layer: one 32-column tile, columns >= nout zero.  Backward (wk, the
// two inner hidden layers), contracting over the columns: lane L holds
// W[32 t + (L & 31)][16 s + 8 (L >> 5) + e].  Last, the output layer's rows
// padded with zeros to 4 or 16 classes.
constexpr int kPacks = 7;
struct PackArgs {
    const bf16 *W[kPacks];
    bf16 *out[kPacks];
    int64_t end[kPacks];   // running totals of the outputs' elements
    int N[kPacks];         // columns of W
    int tiles[kPacks];     // 32-wide tiles of the output index (padded rows: their length)
    int kind[kPacks];      // 0 forward, 1 backward, 2 padded rows
};

__global__ void pack_fused_kernel(PackArgs a) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.end[kPacks - 1]) return;
    int g = 0;
    while (i >= a.end[g]) ++g;
    if (g) i -= a.end[g - 1];
    if (a.kind[g] == 2) {
        const int64_t k = i / a.tiles[g];
        const int n = (int)(i - k * a.tiles[g]);
        a.out[g][i] = n < a.N[g] ? a.W[g][k * a.N[g] + n] : (bf16)0;
        return;
    }
    const int e = (int)(i & 7), L = (int)((i >> 3) & 63);
    const int64_t q = i >> 9;   // (s, t)
    const int t = (int)(q % a.tiles[g]), s = (int)(q / a.tiles[g]);
    const int k = 16 * s + 8 * (L >> 5) + e, n = 32 * t + (L & 31);
    if (a.kind[g] == 1) a.out[g][i] = a.W[g][(int64_t)n * a.N[g] + k];
    else a.out[g][i] = n < a.N[g] ? a.W[g][(int64_t)k * a.N[g] + n] : (bf16)0;
}

template <int NW>
__global__ void __launch_bounds__(64 * NW) mlp_fused_fwd_kernel(const uint8_t *__restrict__ syn, int64_t B, int n_in,
                                                                 int kin, const bf16 *__restrict__ wf1,
                                                                 const bf16 *__restrict__ wf2,
                                                                 const bf16 *__restrict__ wf3,
                                                                 const float *__restrict__ b1,
                                                                 const float *__restrict__ b2,
                                                                 const float *__restrict__ b3,
                                                                 const bf16 *__restrict__ wf4,
                                                                 const float *__restrict__ b4, int nout,
                                                                 float *__restrict__ z) {
    extern __shared__ __align__(16) unsigned char act[];
    constexpr int NT = 16 / NW;                  // 32-column tiles per wave
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m32 = lane & 31, h = lane >> 5;
    const int64_t row0 = (int64_t)blockIdx.x * kFusedRows;
    // syndrome bits -> BF16 0/1 features in columns [0, kin)
    const int cpr = kin >> 3;
    for (int q = tid; q < kFusedRows * cpr; q += 64 * NW) {
        const int m = q / cpr, c = q - m * cpr;
        const int64_t r = row0 + m;
        uint16_t v[8];
        for (int e = 0; e < 8; ++e) {
            const int f = 8 * c + e;
            v[e] = (r < B && f < n_in && (syn[r * n_in + f] & 1)) ? (uint16_t)0x3f80 : (uint16_t)0;
        }
        uint4 u;
        memcpy(&u, v, 16);
        *reinterpret_cast<uint4 *>(act + act_off(m, c)) = u;
    }
    __syncthreads();
    for (int l = 0; l < 3; ++l) {
        const int K = l == 0 ? kin : kFusedHid;
        const int steps = K >> 4;   // even: K is a multiple of 32
        const bf16 *W = l == 0 ? wf1 : (l == 1 ? wf2 : wf3);
        const float *bias = l == 0 ? b1 : (l == 1 ? b2 : b3);
        f32x16 acc[NT][4];
        for (int t = 0; t < NT; ++t) {
            // lane holds columns 32 T + 8 g + 4 h + r for v = 4 g + r
            const int n0 = 32 * (wave * NT + t) + 4 * h;
            for (int g = 0; g < 4; ++g) {
                const float4 bb = *reinterpret_cast<const float4 *>(bias + n0 + 8 * g);
                for (int mt = 0; mt < 4; ++mt) {
                    acc[t][mt][4 * g + 0] = bb.x;
                    acc[t][mt][4 * g + 1] = bb.y;
                    acc[t][mt][4 * g + 2] = bb.z;
                    acc[t][mt][4 * g + 3] = bb.w;
                }
            }
        }
        // weight fragments of k-steps s and s + 1 in flight (two register
        // sets, the loop unrolled by two so that every index is static)
        bf16x8 wa0[NT], wa1[NT];
        auto wload = [&](int s, bf16x8 *dst) {
            for (int t = 0; t < NT; ++t)
                dst[t] = *reinterpret_cast<const bf16x8 *>(W + ((((int64_t)s * 16 + wave * NT + t) << 6) + lane) * 8);
        };
        auto kstep = [&](int s, bf16x8 *wa) {
            bf16x8 xb[4], cur[NT];
            for (int mt = 0; mt < 4; ++mt)
                xb[mt] = *reinterpret_cast<const bf16x8 *>(act + act_off(32 * mt + m32, 2 * s + h));
            for (int t = 0; t < NT; ++t) cur[t] = wa[t];
            if (s + 2 < steps) wload(s + 2, wa);
            for (int t = 0; t < NT; ++t)
                for (int mt = 0; mt < 4; ++mt)
                    acc[t][mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[t], xb[mt], acc[t][mt], 0, 0, 0);
        };
        wload(0, wa0);
        wload(1, wa1);
        for (int s = 0; s < steps; s += 2) {
            kstep(s, wa0);
            kstep(s + 1, wa1);
        }
        __syncthreads();   // every wave is done reading this layer's input
        for (int t = 0; t < NT; ++t)
            for (int mt = 0; mt < 4; ++mt) {
                const int m = 32 * mt + m32;
                for (int g = 0; g < 4; ++g) {
                    const int n0 = 32 * (wave * NT + t) + 8 * g + 4 * h;
                    uint2 u;
                    u.x = f2bf2(fmaxf(acc[t][mt][4 * g], 0.f), fmaxf(acc[t][mt][4 * g + 1], 0.f));
                    u.y = f2bf2(fmaxf(acc[t][mt][4 * g + 2], 0.f), fmaxf(acc[t][mt][4 * g + 3], 0.f));
                    *reinterpret_cast<uint2 *>(act + act_off(m, n0 >> 3) + ((n0 & 7) << 1)) = u;
                }
            }
        __syncthreads();
    }
    // output layer: wave w -> rows [32 w, 32 w + 32) of the tile, all (padded) 32 columns
    for (int mt = wave; mt < 4; mt += NW) {
        f32x16 acc;
        for (int v = 0; v < 16; ++v) {
            const int n = 8 * (v >> 2) + 4 * h + (v & 3);
            acc[v] = n < nout ? b4[n] : 0.f;
        }
        for (int s = 0; s < kFusedHid / 16; ++s) {
            const bf16x8 w = *reinterpret_cast<const bf16x8 *>(wf4 + (((int64_t)s << 6) + lane) * 8);
            const bf16x8 x = *reinterpret_cast<const bf16x8 *>(act + act_off(32 * mt + m32, 2 * s + h));
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, acc, 0, 0, 0);
        }
        const int64_t r = row0 + 32 * mt + m32;
        if (r < B)
            for (int v = 0; v < 16; ++v) {
                const int n = 8 * (v >> 2) + 4 * h + (v & 3);
                if (n < nout) z[r * nout + n] = acc[v];
            }
    }
}

// ---------------------------------------------------------------------------
// Training, hidden width 512: everything that is local to a row in one launch.
// A workgroup of 8 waves takes 32 rows through the forward pass, the loss, and
// the backward pass down to the first layer's pre-activations; all activations
// of the tile stay in LDS (X, H1, H2, H3: 4 x 32 KB, laid out by act_off) and
// each gradient overwrites the activations it is masked with.  What the weight
// gradients contract over the batch goes to global memory once: X, H1, H2 and
// dA1..dA3 (BF16); the output layer's gradient and the bias gradients leave as
// one partial sum per tile.  32 rows, so that the trainer's 8,192 rows give
// one workgroup to each of the 256 CUs; the bound is then the weights'
// stream from L2 (2.1 MB per workgroup against 64 B per clock and CU), kept
// six k-steps ahead in registers.  Products, roundings to BF16 and FP32
// accumulation are those of the layer-by-layer kernels.  Measured at 48 inputs,
// 8,192 rows: 36.2 us with up to 4 classes, 54.1 with up to 16 (whose output
// weights take 64 registers; two of the 256 spill); the layers one by one took
// 75 us forward and down to dA1, and sums over the batch by one thread per
// parameter 8.3 ms more.  A training step also packs the changed weights (7.2
// us) and runs Adam (5.3).
// ---------------------------------------------------------------------------

constexpr int kTrainRows = 32, kTrainMaxOut = 16;
constexpr int kTrainBuf = kTrainRows * kFusedHid * 2;   // bytes of one tile of activations
// buffers, logit partials of the 8 waves, dz
constexpr int kTrainLds = 4 * kTrainBuf + 8 * kTrainRows * kTrainMaxOut * 4 + kTrainRows * kTrainMaxOut * 4;

struct TrainArgs {
    const uint8_t *syn;
    const float *q;
    int64_t B;
    int n_in, kin, nout;
    const bf16 *wf[4];      // forward fragments
    const bf16 *wk[2];      // backward fragments of layers 2 and 3
    const bf16 *w4;         // output layer, [512][NP]
    const float *bias[4];
    bf16 *X, *H1, *H2, *dA1, *dA2, *dA3;
    float *part;            // per tile: dW4 [512][nout] | db4 [nout] | db1 | db2 | db3
    int64_t part_len;
    float *loss_parts;
};

// acc[t] += W^T x src^T for this wave's two 32-column tiles, weights six
// k-steps and activations two steps ahead.  start() issues the first six
// steps' weights; it is called before the epilogue and the barrier in front of
// the product.  Left to itself the compiler moves every load down to its use
// (a layer then takes 20 us), so the steps are kept apart by scheduling
// barriers.
struct TrainGemm {
    static constexpr int DEP = 6, XD = 2, STEPS = kFusedHid / 16;
    bf16x8 wb[DEP][2];
    const bf16 *base;
    const unsigned char *src;
    int m32, h;

    __device__ __forceinline__ void wload(int slot, int s) {
#pragma unroll
        for (int t = 0; t < 2; ++t) wb[slot][t] = *reinterpret_cast<const bf16x8 *>(base + ((s * 16 + t) << 9));
    }
    __device__ __forceinline__ bf16x8 xload(int s) const {
        return *reinterpret_cast<const bf16x8 *>(src + act_off(m32, 2 * s + h));
    }
    __device__ __forceinline__ void start(const bf16 *__restrict__ W, const unsigned char *from, int steps, int wave,
                                          int lane) {
        base = W + (wave << 10) + lane * 8;
        src = from;
        m32 = lane & 31;
        h = lane >> 5;
#pragma unroll
        for (int s = 0; s < DEP; ++s) wload(s, min(s, steps - 1));
        __builtin_amdgcn_sched_barrier(0);
    }
    // K = 512
    __device__ __forceinline__ void run(f32x16 acc[2]) {
        bf16x8 x[XD];
#pragma unroll
        for (int s = 0; s < XD; ++s) x[s] = xload(s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wb[s % DEP][t], x[s % XD], acc[t], 0, 0, 0);
            if (s + DEP < STEPS) wload(s % DEP, s + DEP);
            if (s + XD < STEPS) x[s % XD] = xload(s + XD);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // any number of steps (the input layer): those beyond the first six as they come
    __device__ __forceinline__ void run(f32x16 acc[2], int steps) {
#pragma unroll
        for (int s = 0; s < DEP; ++s)
            if (s < steps) {
                const bf16x8 x = xload(s);
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wb[s][t], x, acc[t], 0, 0, 0);
            }
        for (int s = DEP; s < steps; ++s) {
            const bf16x8 x = xload(s);
            wload(0, s);
#pragma unroll
            for (int t = 0; t < 2; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wb[0][t], x, acc[t], 0, 0, 0);
        }
    }
};

// The pair of gradients (a, b) as BF16 where the activations in `h` are positive.
__device__ __forceinline__ uint32_t masked_pair(uint32_t h, float a, float b) {
    const uint32_t m = (bf2f((bf16)h) > 0.f ? 0xffffu : 0u) | (__uint_as_float(h & 0xffff0000u) > 0.f ? 0xffff0000u : 0u);
    return f2bf2(a, b) & m;
}

// A tile of activations or gradients out to rows row0.. of `out`.
__device__ __forceinline__ void train_store(const unsigned char *buf, bf16 *__restrict__ out, int64_t row0, int tid) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int m = (tid >> 6) + 8 * j, c = tid & 63;
        *reinterpret_cast<uint4 *>(out + (row0 + m) * kFusedHid + 8 * c) =
            *reinterpret_cast<const uint4 *>(buf + act_off(m, c));
    }
}

// Sum over the tile's rows of column tid.
__device__ __forceinline__ float train_colsum(const unsigned char *buf, int tid) {
    float s = 0.f;
#pragma unroll
    for (int m = 0; m < kTrainRows; ++m)
        s += bf2f(*reinterpret_cast<const bf16 *>(buf + act_off(m, tid >> 3) + ((tid & 7) << 1)));
    return s;
}

// NP: classes, padded to 4 or 16 (dz and w4 hold zeros beyond nout).
template <int NP>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) mlp_train_rows_kernel(TrainArgs a) {
    extern __shared__ __align__(16) unsigned char act[];
    unsigned char *bx = act, *b1 = act + kTrainBuf, *b2 = act + 2 * kTrainBuf, *b3 = act + 3 * kTrainBuf;
    float *zp = reinterpret_cast<float *>(act + 4 * kTrainBuf);           // [8][32][NP]
    float *dz = zp + 8 * kTrainRows * kTrainMaxOut;                        // [32][NP]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m32 = lane & 31, h = lane >> 5;
    const int64_t row0 = (int64_t)blockIdx.x * kTrainRows;
    TrainGemm gm;
    gm.start(a.wf[0], bx, a.kin >> 4, wave, lane);
    // syndrome bits -> BF16 0/1 features in columns [0, kin)
    const int cpr = a.kin >> 3;
    for (int q = tid; q < kTrainRows * cpr; q += 512) {
        const int m = q / cpr, c = q - m * cpr;
        const uint8_t *row = a.syn + (row0 + m) * a.n_in;
        uint16_t v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int f = 8 * c + e;
            const uint8_t bit = row[min(f, a.n_in - 1)];
            v[e] = (f < a.n_in && (bit & 1)) ? (uint16_t)0x3f80 : (uint16_t)0;
        }
        uint4 u;
        memcpy(&u, v, 16);
        *reinterpret_cast<uint4 *>(bx + act_off(m, c)) = u;
        *reinterpret_cast<uint4 *>(a.X + (row0 + m) * a.kin + 8 * c) = u;
    }
    __syncthreads();
    // forward: lane holds row m32, columns 64 wave + 32 t + 8 g + 4 h + r for v = 4 g + r
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        unsigned char *dst = l == 0 ? b1 : (l == 1 ? b2 : b3);
        f32x16 acc[2];
        for (int t = 0; t < 2; ++t)
            for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
        float4 bias[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                bias[t][g] = *reinterpret_cast<const float4 *>(a.bias[l] + 64 * wave + 32 * t + 8 * g + 4 * h);
        if (l == 0) gm.run(acc, a.kin >> 4);
        else gm.run(acc);
        if (l < 2) gm.start(a.wf[l + 1], dst, TrainGemm::STEPS, wave, lane);
        else if (NP == 4) gm.start(a.wk[1], b3, TrainGemm::STEPS, wave, lane);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n0 = 64 * wave + 32 * t + 8 * g + 4 * h;
                uint2 u;
                u.x = f2bf2(fmaxf(acc[t][4 * g] + bias[t][g].x, 0.f), fmaxf(acc[t][4 * g + 1] + bias[t][g].y, 0.f));
                u.y = f2bf2(fmaxf(acc[t][4 * g + 2] + bias[t][g].z, 0.f), fmaxf(acc[t][4 * g + 3] + bias[t][g].w, 0.f));
                *reinterpret_cast<uint2 *>(dst + act_off(m32, n0 >> 3) + ((n0 & 7) << 1)) = u;
            }
        __syncthreads();
        if (l < 2) train_store(dst, l == 0 ? a.H1 : a.H2, row0, tid);
    }
    // output weights of this thread's 8 columns of dA3, on their way early
    bf16x8 w4[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) w4[i] = *reinterpret_cast<const bf16x8 *>(a.w4 + ((tid & 63) * NP + i) * 8);
    // and row tid's targets
    float q[NP];
#pragma unroll
    for (int c = 0; c < NP; ++c)
        if (tid < kTrainRows && c < a.nout) q[c] = a.q[(row0 + tid) * a.nout + c];
    // logits: wave w sums hidden units [64 w, 64 w + 64)
    {
        f32x16 acc;
        for (int v = 0; v < 16; ++v) acc[v] = 0.f;
        for (int s = 4 * wave; s < 4 * wave + 4; ++s) {
            const bf16x8 w = *reinterpret_cast<const bf16x8 *>(a.wf[3] + (((int64_t)s << 6) + lane) * 8);
            const bf16x8 x = *reinterpret_cast<const bf16x8 *>(b3 + act_off(m32, 2 * s + h));
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, acc, 0, 0, 0);
        }
        for (int v = 0; v < 8; ++v) {
            const int n = 8 * (v >> 2) + 4 * h + (v & 3);
            if (n < NP) zp[(wave * kTrainRows + m32) * NP + n] = acc[v];
        }
    }
    __syncthreads();
    if (tid < kTrainRows * NP) {
        const int m = tid / NP, c = tid % NP;
        float s = c < a.nout ? a.bias[3][c] : 0.f;
        for (int w = 0; w < 8; ++w) s += zp[(w * kTrainRows + m) * NP + c];
        dz[tid] = s;
    }
    __syncthreads();
    if (tid < 64) {
        // softmax cross-entropy of row tid, and its gradient in place of its logits
        float l = 0.f;
        if (tid < kTrainRows) {
            float *z = dz + tid * NP;
            float m = -INFINITY;
            for (int c = 0; c < a.nout; ++c) m = fmaxf(m, z[c]);
            float s = 0.f;
            for (int c = 0; c < a.nout; ++c) s += expf(z[c] - m);
            const float ls = logf(s);
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                if (c < a.nout) {
                    const float lp = z[c] - m - ls;
                    const float qc = q[c];
                    l -= qc * lp;
                    z[c] = (expf(lp) - qc) / (float)a.B;
                } else {
                    z[c] = 0.f;
                }
            }
        }
        for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
        if (tid == 0) a.loss_parts[blockIdx.x] = l;
    }
    __syncthreads();
    float *part = a.part + (int64_t)blockIdx.x * a.part_len;
    float *db = part + (int64_t)kFusedHid * a.nout + a.nout;
    {
        // output layer's gradients: this thread's hidden unit against every class
        float w[NP];
#pragma unroll
        for (int c = 0; c < NP; ++c) w[c] = 0.f;
#pragma unroll 8
        for (int m = 0; m < kTrainRows; ++m) {
            const float x = bf2f(*reinterpret_cast<const bf16 *>(b3 + act_off(m, tid >> 3) + ((tid & 7) << 1)));
#pragma unroll
            for (int c = 0; c < NP; ++c) w[c] += x * dz[m * NP + c];
        }
#pragma unroll
        for (int c = 0; c < NP; ++c)
            if (c < a.nout) part[tid * a.nout + c] = w[c];
        if (tid < a.nout) {
            float s = 0.f;
            for (int m = 0; m < kTrainRows; ++m) s += dz[m * NP + tid];
            part[(int64_t)kFusedHid * a.nout + tid] = s;
        }
    }
    __syncthreads();
    // dA3 = (dz W4^T) where H3 > 0, in place: 8 columns of 4 rows per thread
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int m = wave + 8 * j;
        float d[NP];
#pragma unroll
        for (int c = 0; c < NP; ++c) d[c] = dz[m * NP + c];
        uint4 *p = reinterpret_cast<uint4 *>(b3 + act_off(m, tid & 63));
        float s[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            s[e] = 0.f;
#pragma unroll
            for (int c = 0; c < NP; ++c) s[e] += d[c] * bf2f((bf16)w4[(e * NP + c) >> 3][(e * NP + c) & 7]);
        }
        uint4 u = *p;
        u.x = masked_pair(u.x, s[0], s[1]);
        u.y = masked_pair(u.y, s[2], s[3]);
        u.z = masked_pair(u.z, s[4], s[5]);
        u.w = masked_pair(u.w, s[6], s[7]);
        *p = u;
    }
    __syncthreads();
    train_store(b3, a.dA3, row0, tid);
    if (NP != 4) gm.start(a.wk[1], b3, TrainGemm::STEPS, wave, lane);
    db[2 * kFusedHid + tid] = train_colsum(b3, tid);
    // dA2, dA1
#pragma unroll
    for (int l = 1; l >= 0; --l) {
        unsigned char *dst = l == 1 ? b2 : b1;
        f32x16 acc[2];
        for (int t = 0; t < 2; ++t)
            for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
        gm.run(acc);
        if (l == 1) gm.start(a.wk[0], b2, TrainGemm::STEPS, wave, lane);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n0 = 64 * wave + 32 * t + 8 * g + 4 * h;
                uint2 *p = reinterpret_cast<uint2 *>(dst + act_off(m32, n0 >> 3) + ((n0 & 7) << 1));
                uint2 u = *p;
                u.x = masked_pair(u.x, acc[t][4 * g], acc[t][4 * g + 1]);
                u.y = masked_pair(u.y, acc[t][4 * g + 2], acc[t][4 * g + 3]);
                *p = u;
            }
        __syncthreads();
        train_store(dst, l == 1 ? a.dA2 : a.dA1, row0, tid);
        db[l * kFusedHid + tid] = train_colsum(dst, tid);
    }
}

// Weight gradients of the three hidden layers, dW_l [K_l][N] = in_l^T dA_l
// summed over the batch, in one launch.  Both operands lie with the contracted
// index (the batch row) outermost, so the tiles are copied to LDS as they are
// and ds_read_b64_tr_b16 hands each lane its column's consecutive rows: for
// each 16 lanes, lane i receives element i % 4 of the 8 bytes that lanes
// i / 4, i / 4 + 4, .. addressed.  Rows of 320 B (256 + 64) put the four rows
// that 32 lanes read on disjoint banks.  128 x 128 tiles, 64 rows per step,
// two LDS buffers and two steps more in registers (a step's 16 MFMAs per wave
// are far shorter than a load).  A batch has far more
// rows than the gradients have tiles (36 at 64 inputs), so the rows are split
// to fill the CUs and each split writes its own partial sum.  The split runs
// fastest in blockIdx.x: workgroups go round the 8 XCDs, so with 8 splits each
// XCD reads one eighth of the rows into its L2, once for all tiles.
struct DwArgs {
    const bf16 *in[3];
    const bf16 *d[3];
    int K[3];          // columns of in_l
    int tile0[4];      // first tile of each layer, total
    int64_t off[3];    // of dW_l in a partial sum
    int N;
    int nsplit;
    int64_t B, rows;   // rows per split (a multiple of 32)
    float *part;
    int64_t part_len;
};

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short bf16x4;
constexpr int kDwStep = 64, kDwLd = 160;

__device__ __forceinline__ bf16x8 tr_fragment(const bf16 *tile, int kk, int col, int lane) {
    const int g = lane >> 4, i = lane & 15;
    const bf16 *p = tile + (kk + 8 * (g >> 1) + (i >> 2)) * kDwLd + col + 16 * (g & 1) + 4 * (i & 3);
    typedef __attribute__((address_space(3))) bf16x4 lds4;
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)p);
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)(p + 4 * kDwLd));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

__global__ void __launch_bounds__(256) mlp_dw_kernel(DwArgs a) {
    __shared__ __align__(16) bf16 As[2][kDwStep * kDwLd];
    __shared__ __align__(16) bf16 Bs[2][kDwStep * kDwLd];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int split = blockIdx.x % a.nsplit, tile = blockIdx.x / a.nsplit;
    // selected, not indexed: an indexed argument would be copied to scratch
    const bool l2 = tile >= a.tile0[2], l1 = tile >= a.tile0[1];
    const int t = tile - (l2 ? a.tile0[2] : l1 ? a.tile0[1] : 0), nt = a.N / 128;
    const int m0 = (t / nt) * 128, n0 = (t % nt) * 128;
    const int K = l2 ? a.K[2] : l1 ? a.K[1] : a.K[0];
    const int N = a.N;
    const bf16 *in = l2 ? a.in[2] : l1 ? a.in[1] : a.in[0], *d = l2 ? a.d[2] : l1 ? a.d[1] : a.d[0];
    const int64_t r0 = (int64_t)split * a.rows;
    const int rows = (int)(min(a.B, r0 + a.rows) - r0);
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    // this thread's chunks: rows tr + 16 j of a step, columns tx .. tx + 7 (K is
    // a multiple of 32, so a chunk is inside or outside as a whole); rows and
    // columns outside are read at a valid place and stored as zeros
    const int tr = tid >> 4, tx = (tid & 15) * 8;
    const bool inside = m0 + tx < K;
    const bf16 *pa = in + r0 * K + (inside ? m0 + tx : 0), *pb = d + r0 * N + n0 + tx;
    struct Step {
        uint4 a[4], b[4];
    };
    auto fetch = [&](Step &s, int k0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = min(k0 + tr + 16 * j, rows - 1);
            s.a[j] = *reinterpret_cast<const uint4 *>(pa + (int64_t)r * K);
            s.b[j] = *reinterpret_cast<const uint4 *>(pb + (int64_t)r * N);
        }
    };
    auto stash = [&](const Step &s, int k0, int buf) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool row = k0 + tr + 16 * j < rows;
            const uint32_t ma = row && inside ? ~0u : 0u, mb = row ? ~0u : 0u;
            bf16 *o = &As[buf][(tr + 16 * j) * kDwLd + tx], *q = &Bs[buf][(tr + 16 * j) * kDwLd + tx];
            *reinterpret_cast<uint4 *>(o) = make_uint4(s.a[j].x & ma, s.a[j].y & ma, s.a[j].z & ma, s.a[j].w & ma);
            *reinterpret_cast<uint4 *>(q) = make_uint4(s.b[j].x & mb, s.b[j].y & mb, s.b[j].z & mb, s.b[j].w & mb);
        }
    };
    f32x16 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    auto multiply = [&](int buf) {
#pragma unroll
        for (int kk = 0; kk < kDwStep; kk += 16) {
            bf16x8 x[2], y[2];
            for (int i = 0; i < 2; ++i) x[i] = tr_fragment(As[buf], kk, wm + 32 * i, lane);
            for (int j = 0; j < 2; ++j) y[j] = tr_fragment(Bs[buf], kk, wn + 32 * j, lane);
            for (int i = 0; i < 2; ++i)
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[i], y[j], acc[i][j], 0, 0, 0);
        }
    };
    // step k in LDS buffer k / 64 % 2, the two after it in registers or on their way
    Step s0, s1;
    // (the scheduling barriers keep the loads in this order: mixed, a wait for
    // the older step is a wait for all of them)
    fetch(s0, 0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(s1, kDwStep);
    __builtin_amdgcn_sched_barrier(0);
    stash(s0, 0, 0);
    fetch(s0, 2 * kDwStep);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    for (int k0 = 0; k0 < rows; k0 += 2 * kDwStep) {
        stash(s1, k0 + kDwStep, 1);
        fetch(s1, k0 + 3 * kDwStep);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0);
        __syncthreads();
        stash(s0, k0 + 2 * kDwStep, 0);
        fetch(s0, k0 + 4 * kDwStep);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1);
        __syncthreads();
    }
    float *out = a.part + (int64_t)split * a.part_len + (l2 ? a.off[2] : l1 ? a.off[1] : a.off[0]);
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) {
            const int col = n0 + wn + j * 32 + (lane & 31);
            for (int v = 0; v < 16; ++v) {
                const int row = m0 + wm + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (row < K) out[(int64_t)row * N + col] = acc[i][j][v];
            }
        }
}

// Sums the partial gradients, always in the same order: the hidden layers'
// weights over the row splits (one thread per parameter), the rest over the
// row tiles (32 parameters x 8 groups of tiles per workgroup).
struct GradSumArgs {
    const float *wpart, *rpart;
    int64_t wlen, rlen;         // parameters in a partial sum of each kind
    int nsplit, ntile;
    int64_t woff[3], wend[3];   // of each hidden layer's weights in `grad`, and running totals in a partial sum
    int64_t roff[5], rend[5];   // of W4, b4, b1, b2, b3
    unsigned wblocks;
    float *grad;
};

__global__ void __launch_bounds__(256) mlp_grad_sum_kernel(GradSumArgs a) {
    if (blockIdx.x < a.wblocks) {
        const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (i >= a.wlen) return;
        float s = 0.f;
#pragma unroll 4
        for (int k = 0; k < a.nsplit; ++k) s += a.wpart[(int64_t)k * a.wlen + i];
        int g = 0;
        while (i >= a.wend[g]) ++g;
        a.grad[a.woff[g] + i - (g ? a.wend[g - 1] : 0)] = s;
        return;
    }
    __shared__ float red[8][32];
    const int64_t i = (int64_t)(blockIdx.x - a.wblocks) * 32 + (threadIdx.x & 31);
    const int grp = threadIdx.x >> 5;
    float s = 0.f;
    if (i < a.rlen)
#pragma unroll 8
        for (int k = grp; k < a.ntile; k += 8) s += a.rpart[(int64_t)k * a.rlen + i];
    red[grp][threadIdx.x & 31] = s;
    __syncthreads();
    if (grp || i >= a.rlen) return;
    s = 0.f;
    for (int k = 0; k < 8; ++k) s += red[k][threadIdx.x & 31];
    int g = 0;
    while (i >= a.rend[g]) ++g;
    a.grad[a.roff[g] + i - (g ? a.rend[g - 1] : 0)] = s;
}

// Wt[n][k] = W[k][n] for the three hidden-layer weight matrices.
__global__ void transpose_bf16_kernel(const bf16 *__restrict__ W, int K, int N, bf16 *__restrict__ Wt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)K * N) return;
    const int n = (int)(i / K), k = (int)(i - (int64_t)n * K);
    Wt[i] = W[(int64_t)k * N + n];
}

// ---------------------------------------------------------------------------
// Small kernels
// ---------------------------------------------------------------------------

// Syndrome bytes [B][n_in] -> BF16 0/1 features [B][kin] (zero padded).
__global__ void embed_kernel(const uint8_t *__restrict__ syn, int64_t B, int n_in, int kin, bf16 *__restrict__ X) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B * kin) return;
    const int64_t b = i / kin;
    const int f = (int)(i - b * kin);
    X[i] = (f < n_in && (syn[b * n_in + f] & 1)) ? (bf16)0x3f80 : (bf16)0;
}

// Output layer for hid = 512, nout <= 4: each lane keeps W[8*lane .. 8*lane+7][0..nout)
// in registers and reads its 8 hidden values of a row with one 16-byte load;
// waves stride over the rows.  Each lane sums its 8 products, then an
// xor-shuffle tree adds the lanes (FP32 throughout).
template <int NOUT>
__global__ void __launch_bounds__(256) out_fwd512_kernel(const bf16 *__restrict__ H, int64_t B,
                                                         const bf16 *__restrict__ W, const float *__restrict__ bias,
                                                         float *__restrict__ z) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    float w[8][NOUT];
    for (int j = 0; j < 8; ++j)
        for (int c = 0; c < NOUT; ++c) w[j][c] = bf2f(W[(8 * lane + j) * NOUT + c]);
    for (int64_t b = wave; b < B; b += nwaves) {
        const uint4 u = *reinterpret_cast<const uint4 *>(H + b * 512 + 8 * lane);
        bf16 h[8];
        memcpy(h, &u, 16);
        float part[NOUT];
        for (int c = 0; c < NOUT; ++c) part[c] = 0.f;
        for (int j = 0; j < 8; ++j) {
            const float x = bf2f(h[j]);
            for (int c = 0; c < NOUT; ++c) part[c] += x * w[j][c];
        }
        for (int c = 0; c < NOUT; ++c) {
            float s = part[c];
            for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
            if (lane == 0) z[b * NOUT + c] = s + bias[c];
        }
    }
}

// Output layer: z[b][c] = sum_k H[b][k] W[k][c] + bias[c]; one wave per row.
__global__ void out_fwd_kernel(const bf16 *__restrict__ H, int64_t B, int hid, const bf16 *__restrict__ W,
                               const float *__restrict__ bias, int nout, float *__restrict__ z) {
    const int64_t b = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (b >= B) return;
    float part[16];
    for (int c = 0; c < nout; ++c) part[c] = 0.f;
    for (int k = lane; k < hid; k += 64) {
        const float h = bf2f(H[b * hid + k]);
        for (int c = 0; c < nout; ++c) part[c] += h * bf2f(W[k * nout + c]);
    }
    for (int c = 0; c < nout; ++c) {
        float s = part[c];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) z[b * nout + c] = s + bias[c];
    }
}

// Softmax + soft cross-entropy: dz = (softmax(z) - q) / B (FP32), loss summed
// per block into loss_parts.
__global__ void xent_kernel(const float *__restrict__ z, const float *__restrict__ q, int64_t B, int nout,
                            float *__restrict__ dz, float *__restrict__ loss_parts) {
    __shared__ float red[256];
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.f;
    if (b < B) {
        float m = -INFINITY;
        for (int c = 0; c < nout; ++c) m = fmaxf(m, z[b * nout + c]);
        float s = 0.f;
        for (int c = 0; c < nout; ++c) s += expf(z[b * nout + c] - m);
        const float ls = logf(s);
        for (int c = 0; c < nout; ++c) {
            const float lp = z[b * nout + c] - m - ls;
            const float qc = q[b * nout + c];
            l -= qc * lp;
            dz[b * nout + c] = (expf(lp) - qc) / (float)B;
        }
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_parts[blockIdx.x] = red[0];
}

// dA[b][k] = (sum_c dz[b][c] W[k][c]) masked by H[b][k] > 0, as BF16.
__global__ void out_bwd_dx_kernel(const float *__restrict__ dz, const bf16 *__restrict__ W, const bf16 *__restrict__ H,
                                  int64_t B, int hid, int nout, bf16 *__restrict__ dA) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B * hid) return;
    const int64_t b = i / hid;
    const int k = (int)(i - b * hid);
    float s = 0.f;
    for (int c = 0; c < nout; ++c) s += dz[b * nout + c] * bf2f(W[k * nout + c]);
    dA[i] = bf2f(H[i]) > 0.f ? f2bf(s) : (bf16)0;
}

// Partial sums over a tile of kSumRows rows, as mlp_train_rows_kernel leaves
// them: the output layer's gradients dW4[k][c] = sum_b H[b][k] dz[b][c] and
// db4[c], and the column sums of a hidden layer's dA.
constexpr int kSumRows = 32;

__global__ void out_bwd_dw_kernel(const bf16 *__restrict__ H, const float *__restrict__ dz, int64_t B, int hid,
                                  int nout, float *__restrict__ part, int64_t part_len) {
    const int64_t r0 = (int64_t)blockIdx.x * kSumRows, r1 = min(B, r0 + kSumRows);
    const int i = blockIdx.y * blockDim.x + threadIdx.x;
    if (i >= (hid + 1) * nout) return;
    const int k = i / nout, c = i - k * nout;
    float s = 0.f;
    for (int64_t b = r0; b < r1; ++b) s += (k < hid ? bf2f(H[b * hid + k]) : 1.f) * dz[b * nout + c];
    part[blockIdx.x * part_len + i] = s;
}

__global__ void colsum_kernel(const bf16 *__restrict__ D, int64_t B, int n, float *__restrict__ part,
                              int64_t part_len) {
    const int64_t r0 = (int64_t)blockIdx.x * kSumRows, r1 = min(B, r0 + kSumRows);
    const int c = blockIdx.y * blockDim.x + threadIdx.x;
    if (c >= n) return;
    float s = 0.f;
    for (int64_t b = r0; b < r1; ++b) s += bf2f(D[b * n + c]);
    part[blockIdx.x * part_len + c] = s;
}

// Adam on the FP32 master parameters; refreshes the BF16 copy.
__global__ void adam_kernel(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, bf16 *__restrict__ wb, int64_t n, float lr, float b1, float b2,
                            float eps, float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    wb[i] = f2bf(wi);
}

__global__ void to_bf16_kernel(const float *__restrict__ w, bf16 *__restrict__ wb, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) wb[i] = f2bf(w[i]);
}

// Confidence gate: the class is accepted when the largest posterior is at
// least `threshold`; otherwise the syndrome id is appended to `reject`.
__global__ void gate_kernel(const float *__restrict__ z, int64_t B, int nout, float threshold,
                            int32_t *__restrict__ classes, float *__restrict__ conf, int32_t *__restrict__ reject,
                            int32_t *__restrict__ reject_count) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    float m = -INFINITY;
    int bi = 0;
    for (int c = 0; c < nout; ++c) {
        const float x = z[b * nout + c];
        if (x > m) {
            m = x;
            bi = c;
        }
    }
    float s = 0.f;
    for (int c = 0; c < nout; ++c) s += expf(z[b * nout + c] - m);
    const float pmax = 1.f / s;
    if (conf) conf[b] = pmax;
    if (classes) classes[b] = bi;
    if (pmax < threshold && reject) {
        const int32_t slot = atomicAdd(reject_count, 1);
        reject[slot] = (int32_t)b;
    }
}

__global__ void zero_count_kernel(int32_t *p) { *p = 0; }

// Class posteriors from TN marginals: q[b][c] = mar[b][c] / sum_c mar[b][c].
__global__ void normalize_kernel(const double *__restrict__ mar, int64_t B, int nout, float *__restrict__ q) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    double s = 0;
    for (int c = 0; c < nout; ++c) s += mar[b * nout + c];
    for (int c = 0; c < nout; ++c) q[b * nout + c] = s > 0 ? (float)(mar[b * nout + c] / s) : 1.f / nout;
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

struct tqec_mlp {
    int n_in = 0, kin = 0, hid = 0, nout = 0;
    int64_t nparams = 0;
    int64_t off[8] = {0};          // W1 b1 W2 b2 W3 b3 W4 b4 in the flat parameter vector
    float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    bf16 *wb = nullptr;
    bf16 *wt[3] = {nullptr, nullptr, nullptr};   // transposed BF16 weights of the hidden layers (inference GEMM)
    bool wt_stale = true;
    // fused inference (hidden width 512): fragment-ordered BF16 weights of the
    // four layers, rebuilt after every weight change
    bf16 *wf[4] = {nullptr, nullptr, nullptr, nullptr};
    bf16 *wk[2] = {nullptr, nullptr};   // of the two inner hidden layers, for the backward pass
    bf16 *w4 = nullptr;                 // output layer's rows, padded
    bool wf_stale = true;
    bool fused = true;             // forward, gate and training on the fused kernels where they apply
    int64_t zcap = 0;              // rows the logits buffer z holds
    bool fused_attr = false;
    int64_t step = 0;
    // activations / scratch for up to `cap` rows
    int64_t cap = 0;
    bf16 *X = nullptr, *H1 = nullptr, *H2 = nullptr, *H3 = nullptr, *dA = nullptr, *dB = nullptr;
    float *z = nullptr, *dz = nullptr, *loss_parts = nullptr;
    int64_t loss_cap = 0;
    // partial gradients: hidden weights per row split, the rest per row tile
    float *wpart = nullptr, *rpart = nullptr;
    size_t wpart_cap = 0, rpart_cap = 0;
    bool train_attr = false;
};

namespace {

int64_t param_count(int kin, int hid, int nout, int64_t off[8]) {
    int64_t o = 0;
    const int64_t sizes[8] = {(int64_t)kin * hid, hid, (int64_t)hid * hid, hid, (int64_t)hid * hid, hid,
                              (int64_t)hid * nout, nout};
    for (int i = 0; i < 8; ++i) {
        off[i] = o;
        o += sizes[i];
    }
    return o;
}

bool fused_ok(const tqec_mlp *p) { return p->hid == kFusedHid && p->nout <= 32 && p->kin <= kFusedHid; }
bool use_fused(const tqec_mlp *p) { return p->fused && fused_ok(p); }

// Partial sums of the loss that a training pass over B rows leaves.
int64_t loss_blocks(const tqec_mlp *p, int64_t B) {
    return use_fused(p) ? B / kTrainRows : (B + 255) / 256;
}

int ensure_cap(tqec_mlp *p, int64_t B) {
    if (p->cap >= B) return TQEC_OK;
    bf16 **bufs[6] = {&p->X, &p->H1, &p->H2, &p->H3, &p->dA, &p->dB};
    for (auto b : bufs)
        if (*b) (void)hipFree(*b);
    if (p->z) (void)hipFree(p->z);
    if (p->dz) (void)hipFree(p->dz);
    p->z = nullptr;
    p->zcap = 0;
    p->cap = 0;
    TQM_HIP(hipMalloc((void **)&p->X, (size_t)B * p->kin * sizeof(bf16)));
    for (int i = 1; i < 6; ++i) TQM_HIP(hipMalloc((void **)bufs[i], (size_t)B * p->hid * sizeof(bf16)));
    TQM_HIP(hipMalloc((void **)&p->z, (size_t)B * p->nout * sizeof(float)));
    p->zcap = B;
    TQM_HIP(hipMalloc((void **)&p->dz, (size_t)B * p->nout * sizeof(float)));
    const int64_t nb = (B + kTrainRows - 1) / kTrainRows;   // enough for either kind of pass
    if (p->loss_cap < nb) {
        if (p->loss_parts) (void)hipFree(p->loss_parts);
        TQM_HIP(hipMalloc((void **)&p->loss_parts, (size_t)nb * sizeof(float)));
        p->loss_cap = nb;
    }
    p->cap = B;
    return TQEC_OK;
}

void gemm(const GemmArgs &a, hipStream_t st) {
    dim3 grid((a.N + BN - 1) / BN, (a.M + BM - 1) / BM);
    hipLaunchKernelGGL(gemm_bf16_kernel, grid, dim3(256), 0, st, a);
}

int padded_classes(const tqec_mlp *p) { return p->nout <= 4 ? 4 : kTrainMaxOut; }

// Fragment-ordered weights of the fused kernels, rebuilt after a weight change.
int pack_weights(tqec_mlp *p, hipStream_t st) {
    if (!p->wf_stale && p->wf[0]) return TQEC_OK;
    const int kdim[4] = {p->kin, p->hid, p->hid, p->hid};
    PackArgs a{};
    int64_t end = 0;
    for (int g = 0; g < 6; ++g) {
        const int l = g < 4 ? g : g - 3;   // layers 1..4 forward, then 2 and 3 backward
        const int npad = l < 3 ? p->hid : 32;
        const int64_t n = (int64_t)kdim[l] * npad;
        bf16 **dst = g < 4 ? &p->wf[g] : &p->wk[g - 4];
        if (!*dst) TQM_HIP(hipMalloc((void **)dst, (size_t)n * sizeof(bf16)));
        a.W[g] = p->wb + p->off[2 * l];
        a.out[g] = *dst;
        a.end[g] = end += n;
        a.N[g] = l < 3 ? p->hid : p->nout;
        a.tiles[g] = npad / 32;
        a.kind[g] = g >= 4;
    }
    const int np = padded_classes(p);
    if (!p->w4) TQM_HIP(hipMalloc((void **)&p->w4, (size_t)p->hid * np * sizeof(bf16)));
    a.W[6] = p->wb + p->off[6];
    a.out[6] = p->w4;
    a.end[6] = end += (int64_t)p->hid * np;
    a.N[6] = p->nout;
    a.tiles[6] = np;
    a.kind[6] = 2;
    hipLaunchKernelGGL(pack_fused_kernel, dim3((unsigned)((end + 255) / 256)), dim3(256), 0, st, a);
    TQM_HIP(hipGetLastError());
    p->wf_stale = false;
    return TQEC_OK;
}

// Logits only (no activations kept): the fused kernel, one workgroup per 128 rows.
int forward_fused(tqec_mlp *p, const uint8_t *d_syn, int64_t B, hipStream_t st) {
    if (p->zcap < B) {
        // logits only; the activation buffers are allocated for training
        if (p->z) (void)hipFree(p->z);
        p->z = nullptr;
        p->zcap = 0;
        TQM_HIP(hipMalloc((void **)&p->z, (size_t)B * p->nout * sizeof(float)));
        p->zcap = B;
    }
    const size_t lds = (size_t)kFusedRows * kFusedHid * 2;
    if (!p->fused_attr) {
        TQM_HIP(hipFuncSetAttribute((const void *)mlp_fused_fwd_kernel<8>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)lds));
        p->fused_attr = true;
    }
    int rc;
    if ((rc = pack_weights(p, st))) return rc;
    const unsigned grid = (unsigned)((B + kFusedRows - 1) / kFusedRows);
    const float *b[4] = {p->w + p->off[1], p->w + p->off[3], p->w + p->off[5], p->w + p->off[7]};
    hipLaunchKernelGGL(mlp_fused_fwd_kernel<8>, dim3(grid), dim3(512), lds, st, d_syn, B, p->n_in, p->kin, p->wf[0],
                       p->wf[1], p->wf[2], b[0], b[1], b[2], p->wf[3], b[3], p->nout, p->z);
    TQM_HIP(hipGetLastError());
    return TQEC_OK;
}

int forward(tqec_mlp *p, const uint8_t *d_syn, int64_t B, hipStream_t st, bool keep = true) {
    int rc;
    if (!keep && use_fused(p)) return forward_fused(p, d_syn, B, st);
    if ((rc = ensure_cap(p, B))) return rc;
    const int64_t nx = B * p->kin;
    hipLaunchKernelGGL(embed_kernel, dim3((unsigned)((nx + 255) / 256)), dim3(256), 0, st, d_syn, B, p->n_in, p->kin,
                       p->X);
    const bf16 *in[3] = {p->X, p->H1, p->H2};
    bf16 *out[3] = {p->H1, p->H2, p->H3};
    const int kdim[3] = {p->kin, p->hid, p->hid};
    if (p->wt_stale) {
        for (int l = 0; l < 3; ++l) {
            const int64_t n = (int64_t)kdim[l] * p->hid;
            hipLaunchKernelGGL(transpose_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                               p->wb + p->off[2 * l], kdim[l], p->hid, p->wt[l]);
        }
        p->wt_stale = false;
    }
    for (int l = 0; l < 3; ++l) {
        const dim3 grid((unsigned)(p->hid / 128), (unsigned)((B + 127) / 128));
        const float *bias = p->w + p->off[2 * l + 1];
        if (kdim[l] % 64 == 0)
            hipLaunchKernelGGL(gemm_fwd_kernel<64>, grid, dim3(256), 0, st, in[l], p->wt[l], (int)B, p->hid, kdim[l],
                               bias, out[l]);
        else
            hipLaunchKernelGGL(gemm_fwd_kernel<32>, grid, dim3(256), 0, st, in[l], p->wt[l], (int)B, p->hid, kdim[l],
                               bias, out[l]);
    }
    const unsigned rows_per_block = 4;
    if (p->hid == 512 && p->nout <= 4) {
        const unsigned blocks = (unsigned)std::min<int64_t>((B + 3) / 4, 4096);
        if (p->nout == 4)
            hipLaunchKernelGGL(out_fwd512_kernel<4>, dim3(blocks), dim3(256), 0, st, p->H3, B, p->wb + p->off[6],
                               p->w + p->off[7], p->z);
        else if (p->nout == 2)
            hipLaunchKernelGGL(out_fwd512_kernel<2>, dim3(blocks), dim3(256), 0, st, p->H3, B, p->wb + p->off[6],
                               p->w + p->off[7], p->z);
        else
            hipLaunchKernelGGL(out_fwd_kernel, dim3((unsigned)((B + rows_per_block - 1) / rows_per_block)), dim3(256),
                               0, st, p->H3, B, p->hid, p->wb + p->off[6], p->w + p->off[7], p->nout, p->z);
    } else {
        hipLaunchKernelGGL(out_fwd_kernel, dim3((unsigned)((B + rows_per_block - 1) / rows_per_block)), dim3(256), 0,
                           st, p->H3, B, p->hid, p->wb + p->off[6], p->w + p->off[7], p->nout, p->z);
    }
    TQM_HIP(hipGetLastError());
    return TQEC_OK;
}

int grow(float **buf, size_t *cap, size_t need) {
    if (*cap >= need) return TQEC_OK;
    if (*buf) TQM_HIP(hipFree(*buf));
    *buf = nullptr;
    *cap = 0;
    TQM_HIP(hipMalloc((void **)buf, need * sizeof(float)));
    *cap = need;
    return TQEC_OK;
}

int64_t row_part_len(const tqec_mlp *p) { return (int64_t)(p->hid + 1) * p->nout + 3 * (int64_t)p->hid; }

// Weight gradients of the hidden layers from their inputs and dA1..dA3 (d[l]
// the gradient at layer l + 1's pre-activation), then all partial sums into
// `grad`.
int weight_gradients(tqec_mlp *p, const bf16 *const d[3], int64_t B, int ntile, float *grad, hipStream_t st) {
    DwArgs w{};
    const bf16 *in[3] = {p->X, p->H1, p->H2};
    const int kdim[3] = {p->kin, p->hid, p->hid};
    GradSumArgs g{};
    int tiles = 0;
    int64_t len = 0;
    for (int l = 0; l < 3; ++l) {
        w.in[l] = in[l];
        w.d[l] = d[l];
        w.K[l] = kdim[l];
        w.tile0[l] = tiles;
        w.off[l] = len;
        tiles += (kdim[l] + 127) / 128 * (p->hid / 128);
        len += (int64_t)kdim[l] * p->hid;
        g.woff[l] = p->off[2 * l];
        g.wend[l] = len;
    }
    w.tile0[3] = tiles;
    w.N = p->hid;
    w.B = B;
    w.part_len = len;
    // one split per XCD, at least four steps of rows in each
    int64_t split = std::max<int64_t>(1, std::min<int64_t>(8, B / (4 * kDwStep)));
    w.rows = ((B + split - 1) / split + 31) / 32 * 32;
    split = (B + w.rows - 1) / w.rows;
    int rc;
    if ((rc = grow(&p->wpart, &p->wpart_cap, (size_t)(split * len)))) return rc;
    w.part = p->wpart;
    w.nsplit = (int)split;
    hipLaunchKernelGGL(mlp_dw_kernel, dim3((unsigned)(tiles * split)), dim3(256), 0, st, w);
    g.wpart = p->wpart;
    g.rpart = p->rpart;
    g.wlen = len;
    g.rlen = row_part_len(p);
    g.nsplit = (int)split;
    g.ntile = ntile;
    const int64_t rn[5] = {(int64_t)p->hid * p->nout, p->nout, p->hid, p->hid, p->hid};
    const int ri[5] = {6, 7, 1, 3, 5};
    int64_t end = 0;
    for (int i = 0; i < 5; ++i) {
        g.roff[i] = p->off[ri[i]];
        g.rend[i] = end += rn[i];
    }
    g.wblocks = (unsigned)((len + 255) / 256);
    g.grad = grad;
    hipLaunchKernelGGL(mlp_grad_sum_kernel, dim3(g.wblocks + (unsigned)((g.rlen + 31) / 32)), dim3(256), 0, st, g);
    TQM_HIP(hipGetLastError());
    return TQEC_OK;
}

// Forward and backward pass of a network that the fused kernels cover.
int train_fused(tqec_mlp *p, const uint8_t *d_syn, const float *d_q, int64_t B, float *grad, hipStream_t st) {
    int rc;
    if ((rc = ensure_cap(p, B))) return rc;
    if ((rc = pack_weights(p, st))) return rc;
    const int64_t tiles = B / kTrainRows;
    if ((rc = grow(&p->rpart, &p->rpart_cap, (size_t)(tiles * row_part_len(p))))) return rc;
    if (!p->train_attr) {
        TQM_HIP(hipFuncSetAttribute((const void *)mlp_train_rows_kernel<4>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    kTrainLds));
        TQM_HIP(hipFuncSetAttribute((const void *)mlp_train_rows_kernel<kTrainMaxOut>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kTrainLds));
        p->train_attr = true;
    }
    TrainArgs a{};
    a.syn = d_syn;
    a.q = d_q;
    a.B = B;
    a.n_in = p->n_in;
    a.kin = p->kin;
    a.nout = p->nout;
    for (int l = 0; l < 4; ++l) {
        a.wf[l] = p->wf[l];
        a.bias[l] = p->w + p->off[2 * l + 1];
    }
    a.wk[0] = p->wk[0];
    a.wk[1] = p->wk[1];
    a.w4 = p->w4;
    a.X = p->X;
    a.H1 = p->H1;
    a.H2 = p->H2;
    a.dA1 = p->H3;   // H3 itself never leaves the tile
    a.dA2 = p->dB;
    a.dA3 = p->dA;
    a.part = p->rpart;
    a.part_len = row_part_len(p);
    a.loss_parts = p->loss_parts;
    if (p->nout <= 4)
        hipLaunchKernelGGL(mlp_train_rows_kernel<4>, dim3((unsigned)tiles), dim3(512), kTrainLds, st, a);
    else
        hipLaunchKernelGGL(mlp_train_rows_kernel<kTrainMaxOut>, dim3((unsigned)tiles), dim3(512), kTrainLds, st, a);
    const bf16 *d[3] = {a.dA1, a.dA2, a.dA3};
    return weight_gradients(p, d, B, (int)tiles, grad, st);
}

// Gradients of the mean soft cross-entropy into `grad` (FP32, flat layout),
// layer by layer after forward().
int backward(tqec_mlp *p, const float *d_q, int64_t B, float *grad, hipStream_t st) {
    const int64_t nb = (B + 255) / 256;
    const int64_t tiles = (B + kSumRows - 1) / kSumRows, plen = row_part_len(p);
    int rc;
    if ((rc = grow(&p->rpart, &p->rpart_cap, (size_t)(tiles * plen)))) return rc;
    hipLaunchKernelGGL(xent_kernel, dim3((unsigned)nb), dim3(256), 0, st, p->z, d_q, B, p->nout, p->dz, p->loss_parts);
    // output layer
    const int64_t no = (int64_t)(p->hid + 1) * p->nout;
    hipLaunchKernelGGL(out_bwd_dw_kernel, dim3((unsigned)tiles, (unsigned)((no + 255) / 256)), dim3(256), 0, st, p->H3,
                       p->dz, B, p->hid, p->nout, p->rpart, plen);
    const int64_t nh = B * p->hid;
    hipLaunchKernelGGL(out_bwd_dx_kernel, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, st, p->dz,
                       p->wb + p->off[6], p->H3, B, p->hid, p->nout, p->dA);
    // hidden layers 3, 2, 1: d[l] holds dL/d(pre-activation) of layer l + 1;
    // H3 has been read when dA1 takes its place
    const bf16 *hin[3] = {p->X, p->H1, p->H2};
    bf16 *d[3] = {p->H3, p->dB, p->dA};
    for (int l = 2; l >= 0; --l) {
        hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)tiles, (unsigned)((p->hid + 255) / 256)), dim3(256), 0, st, d[l],
                           B, p->hid, p->rpart + no + (int64_t)l * p->hid, plen);
        if (l > 0) {
            // d in_l [B][K] = dA [B][N] * W_l^T (W_l stored [K][N]), masked by in_l > 0
            GemmArgs x{};
            x.A = d[l];
            x.B = p->wb + p->off[2 * l];
            x.M = (int)B;
            x.N = p->hid;
            x.K = p->hid;
            x.lda = p->hid;
            x.ldb = p->hid;
            x.ldc = p->hid;
            x.mask = hin[l];
            x.outb = d[l - 1];
            gemm(x, st);
        }
    }
    TQM_HIP(hipGetLastError());
    const bf16 *dc[3] = {d[0], d[1], d[2]};
    return weight_gradients(p, dc, B, (int)tiles, grad, st);
}

// Training takes tiles of 32 rows (mlp_train_rows_kernel has no ragged one, and
// the layer-by-layer pass keeps its rule); inference takes any batch size.
int check_batch(tqec_mlp *p, int64_t B, bool training) {
    if (!p) return fail(TQEC_ENULL, "null network");
    if (B <= 0 || B > (int64_t(1) << 30)) return fail(TQEC_EINVAL, "batch size out of range");
    if (training && B % 32 != 0) return fail(TQEC_EINVAL, "training batch size must be a multiple of 32");
    return TQEC_OK;
}

}  // namespace

extern "C" {

int tqec_mlp_create(int32_t n_in, int32_t hidden, int32_t n_out, tqec_mlp **out) {
    if (!out) return fail(TQEC_ENULL, "null output handle");
    *out = nullptr;
    if (n_in <= 0 || n_in > 4096 || hidden <= 0 || hidden % 128 != 0 || n_out <= 0 || n_out > 16)
        return fail(TQEC_EINVAL, "n_in in [1, 4096], hidden a multiple of 128, n_out in [1, 16]");
    auto *p = new (std::nothrow) tqec_mlp();
    if (!p) return fail(TQEC_ENOMEM, "out of host memory");
    p->n_in = n_in;
    p->kin = (n_in + 31) / 32 * 32;
    p->hid = hidden;
    p->nout = n_out;
    p->nparams = param_count(p->kin, hidden, n_out, p->off);
    const size_t nb = (size_t)p->nparams;
    hipError_t e = hipMalloc((void **)&p->w, nb * 4);
    if (e == hipSuccess) e = hipMalloc((void **)&p->g, nb * 4);
    if (e == hipSuccess) e = hipMalloc((void **)&p->m, nb * 4);
    if (e == hipSuccess) e = hipMalloc((void **)&p->v, nb * 4);
    if (e == hipSuccess) e = hipMalloc((void **)&p->wb, nb * 2);
    for (int l = 0; l < 3 && e == hipSuccess; ++l)
        e = hipMalloc((void **)&p->wt[l], (size_t)(l == 0 ? p->kin : p->hid) * p->hid * 2);
    if (e == hipSuccess) e = hipMemset(p->w, 0, nb * 4);
    if (e == hipSuccess) e = hipMemset(p->m, 0, nb * 4);
    if (e == hipSuccess) e = hipMemset(p->v, 0, nb * 4);
    if (e == hipSuccess) e = hipMemset(p->wb, 0, nb * 2);
    if (e != hipSuccess) {
        tqec_mlp_destroy(p);
        return fail(TQEC_EDEVICE, hipGetErrorString(e));
    }
    *out = p;
    return TQEC_OK;
}

int64_t tqec_mlp_num_params(const tqec_mlp *p) { return p ? p->nparams : -1; }

int tqec_mlp_set_params(tqec_mlp *p, const float *host) {
    if (!p || !host) return fail(TQEC_ENULL, "null argument");
    // padded input rows of W1 (k >= n_in) must stay zero
    std::vector<float> w(host, host + p->nparams);
    for (int k = p->n_in; k < p->kin; ++k)
        for (int c = 0; c < p->hid; ++c) w[p->off[0] + (int64_t)k * p->hid + c] = 0.f;
    TQM_HIP(hipMemcpy(p->w, w.data(), (size_t)p->nparams * 4, hipMemcpyHostToDevice));
    TQM_HIP(hipMemset(p->m, 0, (size_t)p->nparams * 4));
    TQM_HIP(hipMemset(p->v, 0, (size_t)p->nparams * 4));
    hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((p->nparams + 255) / 256)), dim3(256), 0, 0, p->w, p->wb,
                       p->nparams);
    TQM_HIP(hipDeviceSynchronize());
    p->step = 0;
    p->wt_stale = true;
    p->wf_stale = true;
    return TQEC_OK;
}

int tqec_mlp_get_params(tqec_mlp *p, float *host) {
    if (!p || !host) return fail(TQEC_ENULL, "null argument");
    TQM_HIP(hipDeviceSynchronize());
    TQM_HIP(hipMemcpy(host, p->w, (size_t)p->nparams * 4, hipMemcpyDeviceToHost));
    return TQEC_OK;
}

int tqec_mlp_forward(tqec_mlp *p, const uint8_t *d_syn, int64_t B, float *d_logits, void *stream) {
    int rc;
    if ((rc = check_batch(p, B, false))) return rc;
    if (!d_syn || !d_logits) return fail(TQEC_ENULL, "null device pointer");
    hipStream_t st = (hipStream_t)stream;
    if ((rc = forward(p, d_syn, B, st, false))) return rc;
    TQM_HIP(hipMemcpyAsync(d_logits, p->z, (size_t)B * p->nout * 4, hipMemcpyDeviceToDevice, st));
    return TQEC_OK;
}

int tqec_mlp_gradients(tqec_mlp *p, const uint8_t *d_syn, const float *d_targets, int64_t B, float *d_grad,
                       float *h_loss, void *stream) {
    int rc;
    if ((rc = check_batch(p, B, true))) return rc;
    if (!d_syn || !d_targets) return fail(TQEC_ENULL, "null device pointer");
    hipStream_t st = (hipStream_t)stream;
    float *grad = d_grad ? d_grad : p->g;
    if (use_fused(p)) {
        if ((rc = train_fused(p, d_syn, d_targets, B, grad, st))) return rc;
    } else {
        if ((rc = forward(p, d_syn, B, st))) return rc;
        if ((rc = backward(p, d_targets, B, grad, st))) return rc;
    }
    if (h_loss) {
        const int64_t nb = loss_blocks(p, B);
        std::vector<float> parts(nb);
        TQM_HIP(hipMemcpyAsync(parts.data(), p->loss_parts, nb * 4, hipMemcpyDeviceToHost, st));
        TQM_HIP(hipStreamSynchronize(st));
        double s = 0;
        for (float x : parts) s += x;
        *h_loss = (float)(s / (double)B);
    }
    return TQEC_OK;
}

int tqec_mlp_train_step(tqec_mlp *p, const uint8_t *d_syn, const float *d_targets, int64_t B, float lr,
                        float *h_loss, void *stream) {
    int rc;
    if ((rc = tqec_mlp_gradients(p, d_syn, d_targets, B, nullptr, h_loss, stream))) return rc;
    hipStream_t st = (hipStream_t)stream;
    p->step += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)p->step), c2 = 1.f - std::pow(b2, (float)p->step);
    hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((p->nparams + 255) / 256)), dim3(256), 0, st, p->w, p->g, p->m,
                       p->v, p->wb, p->nparams, lr, b1, b2, 1e-8f, c1, c2);
    p->wt_stale = true;
    p->wf_stale = true;
    // padded rows of W1 get zero gradient (zero inputs) and so stay zero
    TQM_HIP(hipGetLastError());
    return TQEC_OK;
}

int tqec_mlp_gate(tqec_mlp *p, const uint8_t *d_syn, int64_t B, float threshold, int32_t *d_classes,
                  float *d_confidence, int32_t *d_reject, int32_t *d_reject_count, void *stream) {
    int rc;
    if ((rc = check_batch(p, B, false))) return rc;
    if (!d_syn || (d_reject && !d_reject_count)) return fail(TQEC_ENULL, "null device pointer");
    hipStream_t st = (hipStream_t)stream;
    if ((rc = forward(p, d_syn, B, st, false))) return rc;
    if (d_reject_count) hipLaunchKernelGGL(zero_count_kernel, dim3(1), dim3(1), 0, st, d_reject_count);
    hipLaunchKernelGGL(gate_kernel, dim3((unsigned)((B + 255) / 256)), dim3(256), 0, st, p->z, B, p->nout, threshold,
                       d_classes, d_confidence, d_reject, d_reject_count);
    TQM_HIP(hipGetLastError());
    return TQEC_OK;
}

int tqec_posteriors_from_marginals(const double *d_marginals, int64_t n, int32_t n_classes, float *d_q,
                                   void *stream) {
    if (n < 0 || n_classes <= 0) return fail(TQEC_EINVAL, "bad sizes");
    if (n > 0 && (!d_marginals || !d_q)) return fail(TQEC_ENULL, "null device pointer");
    if (n == 0) return TQEC_OK;
    hipLaunchKernelGGL(normalize_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       d_marginals, n, n_classes, d_q);
    TQM_HIP(hipGetLastError());
    return TQEC_OK;
}

int tqec_mlp_set_inference(tqec_mlp *p, int32_t kernel) {
    if (!p) return fail(TQEC_ENULL, "null network");
    if (kernel != 0 && kernel != 1) return fail(TQEC_EINVAL, "inference kernel must be 0 (layer by layer) or 1 (fused)");
    if (kernel == 1 && !fused_ok(p))
        return fail(TQEC_EUNSUPPORTED, "the fused kernel needs hidden width 512, n_out <= 32 and n_in <= 512");
    p->fused = kernel == 1;
    return TQEC_OK;
}

int tqec_mlp_inference(const tqec_mlp *p, int32_t *kernel) {
    if (!p || !kernel) return fail(TQEC_ENULL, "null argument");
    *kernel = use_fused(p) ? 1 : 0;
    return TQEC_OK;
}

void tqec_mlp_destroy(tqec_mlp *p) {
    if (!p) return;
    void *bufs[] = {p->w,  p->g,  p->m,  p->v,  p->wb, p->X,  p->H1,         p->H2,    p->H3,
                    p->dA, p->dB, p->z,  p->dz, p->loss_parts, p->wt[0], p->wt[1], p->wt[2],
                    p->wf[0], p->wf[1], p->wf[2], p->wf[3], p->wk[0], p->wk[1], p->w4, p->wpart, p->rpart};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    delete p;
}

}  // extern "C"
