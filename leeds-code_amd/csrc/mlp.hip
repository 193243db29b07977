// Small multilayer perceptron for the learned closure: training and
// inference on the GPU.  Three dense layers (n_in -> W -> W -> n_out) with
// GELU between them; BF16 weights and activations on the matrix cores
// (v_mfma_f32_16x16x32_bf16) with FP32 accumulation, FP32 master weights
// updated by Adam.
//
// Up to 256 inputs and a width of 256 (FUSE_MAX) a pass is one kernel: a
// workgroup takes 32 rows through all layers, with their activations as the
// next layer's BF16 operand in LDS and the weights packed beforehand in
// operand order (k_mlp_fwd, k_mlp_bwd); the weight and bias gradients of all
// layers are one launch (k_mlp_dw).  Larger networks run a GEMM per layer
// (k_gemm_bf16: operands in FP32 memory with arbitrary strides, rounded to
// BF16 through LDS, workgroup tile 64 x 64 by 4 waves, K in steps of 32).
// Both sum K in the same steps of 32 and the biases' gradients row by row, so
// a network's results do not depend on which of them runs.
// MFMA operand layout (16x16x32 bf16): lane l holds A[i = l%16][k = 8(l/16)
// .. 8(l/16)+7] and B[k = 8(l/16) ..][j = l%16]; the result lane holds
// C[4(l/16) + r][l%16], r = 0..3.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/lsd.h"
#include "lsd_internal.h"

namespace lsd {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

struct GemmArgs {
    int M, N, K;
    const float* A;
    long sam, sak;  // A(i,k) = A[i*sam + k*sak]
    const float* B;
    long sbk, sbn;  // B(k,j) = B[k*sbk + j*sbn]
    float* C;
    long ldc;       // C(i,j) = C[i*ldc + j]
    const float* bias;  // [N] or null
    int accumulate;     // C += result
    int act;            // 0 none, 1 GELU (Z keeps the pre-activation)
    float* Z;           // [M][ldc] pre-activation when act = 1
};

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

constexpr int GT = 64;   // tile edge
constexpr int GK = 32;   // K step
constexpr int GKP = 40;  // padded LDS row (bf16) against bank conflicts

__global__ void __launch_bounds__(256) k_gemm_bf16(GemmArgs g) {
    __shared__ __bf16 As[GT][GKP];
    __shared__ __bf16 Bs[GT][GKP];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int l16 = lane & 15, q = lane >> 4;
    const int i0 = blockIdx.y * GT, j0 = blockIdx.x * GT;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    v4f acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < g.K; k0 += GK) {
        // stage: 64 x 32 of A and of B^T, 8 elements per thread each
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int idx = t + 256 * e;  // 0 .. 2047
            const int r = idx >> 5, kk = idx & 31;
            const int i = i0 + r, k = k0 + kk, j = j0 + r;
            const float av = (i < g.M && k < g.K) ? g.A[(long)i * g.sam + (long)k * g.sak] : 0.f;
            const float bv = (j < g.N && k < g.K) ? g.B[(long)k * g.sbk + (long)j * g.sbn] : 0.f;
            As[r][kk] = (__bf16)av;
            Bs[r][kk] = (__bf16)bv;
        }
        __syncthreads();
        bf16x8 af[2], bfr[2];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int v = 0; v < 8; v++) af[a][v] = As[wi + 16 * a + l16][8 * q + v];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int v = 0; v < 8; v++) bfr[b][v] = Bs[wj + 16 * b + l16][8 * q + v];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bfr[b], acc[a][b], 0, 0, 0);
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = i0 + wi + 16 * a + 4 * q + r;
                const int j = j0 + wj + 16 * b + l16;
                if (i >= g.M || j >= g.N) continue;
                float v = acc[a][b][r];
                if (g.bias) v += g.bias[j];
                float* c = g.C + (long)i * g.ldc + j;
                if (g.accumulate) v += *c;
                if (g.act == 1) {
                    g.Z[(long)i * g.ldc + j] = v;
                    v = gelu(v);
                }
                *c = v;
            }
}

static int gemm(hipStream_t st, GemmArgs g) {
    dim3 grid((g.N + GT - 1) / GT, (g.M + GT - 1) / GT);
    hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(256), 0, st, g);
    LSD_HIP(hipGetLastError());
    return LSD_OK;
}

// d = d * gelu'(Z), elementwise (dH on entry, dZ on exit)
__global__ void k_gelu_back(long n, const float* __restrict__ Z, float* __restrict__ d) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = d[i] * gelu_grad(Z[i]);
}

// Column sums of dY [rows][ld], cols of each row, into db (bias gradients), row
// by row.  COLSUM_AHEAD rows are loaded before they are added: with one load at
// a time the sum is a chain of memory latencies, which moved by up to 14 % with
// the rows' stride and place.
constexpr int COLSUM_AHEAD = 8;
__global__ void k_colsum(int rows, int cols, int ld, const float* __restrict__ dY, float* __restrict__ db) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= cols) return;
    float s = 0.f;
    int i = 0;
    for (; i + COLSUM_AHEAD <= rows; i += COLSUM_AHEAD) {
        float v[COLSUM_AHEAD];
#pragma unroll
        for (int e = 0; e < COLSUM_AHEAD; e++) v[e] = dY[(long)(i + e) * ld + j];
#pragma unroll
        for (int e = 0; e < COLSUM_AHEAD; e++) s += v[e];
    }
    for (; i < rows; i++) s += dY[(long)i * ld + j];
    db[j] = s;
}

// ------------------------------------------------------------ fused passes

constexpr int FUSE_MAX = 256;           // inputs and width of the fused passes
constexpr int MF_ROWS = 32;             // rows per workgroup; its four waves share the columns
constexpr int MF_WAVES = 4;
constexpr int MF_AHEAD = 4;             // K steps of weights in flight
constexpr int MF_LD = FUSE_MAX + 8;     // LDS row (BF16): 16 rows in distinct banks
// 16-column tiles of a hidden layer: the width rounded up to 64, 128 or 256
// (compile-time, so the accumulators stay in registers)
static int mf_tiles(int width) { return width <= 64 ? 4 : width <= 128 ? 8 : 16; }

// Weights in operand order, [k step][column tile][lane][8]: lane l of tile t
// in step s holds B(k = 32 s + 8 (l / 16) + v, j = 16 t + l % 16), zero past
// the edges.  B(k, j) = w[k sk + j sj].
struct PackJob {
    const float* w;
    __bf16* out;
    int K, N, nt, ks;
    long sk, sj;
};
constexpr int NPACK = 5;  // W1, W2, W3 forward; W3, W2 backward
struct PackArgs {
    PackJob j[NPACK];
};

__global__ void __launch_bounds__(256) k_mlp_pack(PackArgs a) {
    const PackJob p = a.j[blockIdx.y];
    const int i = blockIdx.x * 256 + threadIdx.x;  // (step, tile, lane)
    if (i >= p.ks * p.nt * 64) return;
    const int lane = i & 63, t = (i >> 6) % p.nt, s = (i >> 6) / p.nt;
    const int j = 16 * t + (lane & 15);
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int k = 32 * s + 8 * (lane >> 4) + e;
        v[e] = (__bf16)((k < p.K && j < p.N) ? p.w[k * p.sk + j * p.sj] : 0.f);
    }
    reinterpret_cast<bf16x8*>(p.out)[i] = v;
}

struct MlpArgs {
    long rows;
    int nin, width, nout;
    int nto;              // column tiles of the output
    int ks1, kso;         // K steps over the inputs and the outputs
    const float* x;       // [rows][nin]
    const float *b1, *b2, *b3;
    const __bf16 *w1, *w2, *w3;  // packed, forward
    const __bf16 *w3t, *w2t;     // packed, backward
    float *Z1, *H1, *Z2, *H2, *Y;
    const float* dY;      // [rows][ldy]
    int ldy;
    float *dZ1, *dZ2;     // [rows][width]
};

// Rows row0 .. row0 + 31 of a [rows][n] matrix into LDS as BF16 (8 rows per
// wave), zero in columns n .. 32 ks - 1; rows past the end repeat the last.
__device__ __forceinline__ void mf_stage(__bf16* S, const float* __restrict__ x, long rows, long row0, int n, int ld,
                                         int ks) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int c = lane; c < 32 * ks; c += 64) {
        const bool in = c < n;
        const int cc = in ? c : n - 1;
        float v[8];
#pragma unroll
        for (int r = 0; r < 8; r++) v[r] = x[min(row0 + 8 * wave + r, rows - 1) * ld + cc];
#pragma unroll
        for (int r = 0; r < 8; r++) S[(8 * wave + r) * MF_LD + c] = (__bf16)(in ? v[r] : 0.f);
    }
    __syncthreads();
}

// acc = S (32 rows x 32 ks) times this wave's tiles t = wave + 4 u < nt of the
// packed weights, loaded MF_AHEAD K steps ahead (steps past the end repeat the
// last one and are not multiplied).
template <int NW>
__device__ __forceinline__ void mf_layer(const __bf16* S, const __bf16* __restrict__ w, int ks, int nt,
                                         v4f (&acc)[2][NW]) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int u = 0; u < NW; u++) acc[a][u] = v4f{0.f, 0.f, 0.f, 0.f};
    bf16x8 b[MF_AHEAD][NW];
    auto load = [&](bf16x8 (&d)[NW], int s) {
        const bf16x8* wf = reinterpret_cast<const bf16x8*>(w) + (size_t)min(s, ks - 1) * nt * 64 + lane;
#pragma unroll
        for (int u = 0; u < NW; u++) d[u] = wf[min(wave + MF_WAVES * u, nt - 1) * 64];
    };
#pragma unroll
    for (int e = 0; e < MF_AHEAD; e++) load(b[e], e);
    for (int s0 = 0; s0 < ks; s0 += MF_AHEAD) {
#pragma unroll
        for (int e = 0; e < MF_AHEAD; e++) {
            const int s = s0 + e;
            if (s < ks) {
#pragma unroll
                for (int a = 0; a < 2; a++) {
                    const bf16x8 af = *reinterpret_cast<const bf16x8*>(S + (16 * a + l16) * MF_LD + 32 * s + 8 * q);
#pragma unroll
                    for (int u = 0; u < NW; u++)
                        acc[a][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, b[e][u], acc[a][u], 0, 0, 0);
                }
            }
            load(b[e], s + MF_AHEAD);
        }
    }
}

// Forward pass; TRAIN keeps the pre-activations and activations for the
// backward pass.  A workgroup holds 32 rows, its waves the column tiles, so
// the erf of GELU (40 instructions) and the weights' operand loads from L2,
// which bound it, spread over 4 waves per 32 rows (one wave per 32 rows: 92 us
// for the 8192 rows of a minibatch, 110 us for 57792 rows of inference, where
// three GEMM launches took 258 us).
template <int NT, bool TRAIN>
__global__ void __launch_bounds__(64 * MF_WAVES) k_mlp_fwd(MlpArgs g) {
    constexpr int NW = NT / MF_WAVES;
    __shared__ __attribute__((aligned(16))) __bf16 S[2][MF_ROWS * MF_LD];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
    const long row0 = (long)blockIdx.x * MF_ROWS;
    const int left = (int)min(g.rows - row0, (long)MF_ROWS);  // rows of this workgroup
    v4f acc[2][NW];
    mf_stage(S[0], g.x, g.rows, row0, g.nin, g.nin, g.ks1);
#pragma unroll 1
    for (int layer = 0; layer < 2; layer++) {
        mf_layer(S[layer], layer ? g.w2 : g.w1, layer ? NT / 2 : g.ks1, NT, acc);
        const float* bias = layer ? g.b2 : g.b1;
        float* Z = (layer ? g.Z2 : g.Z1) + row0 * g.width;
        float* H = (layer ? g.H2 : g.H1) + row0 * g.width;
        __bf16* So = S[1 - layer];
#pragma unroll
        for (int u = 0; u < NW; u++) {
            const int j = 16 * (wave + MF_WAVES * u) + l16;
            const bool in = j < g.width;
            const float bj = in ? bias[j] : 0.f;
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = 16 * a + 4 * q + r;
                    const float z = acc[a][u][r] + bj;
                    const float h = gelu(z);
                    if (TRAIN && in && row < left) {
                        Z[row * g.width + j] = z;
                        H[row * g.width + j] = h;
                    }
                    // zero past the width, also where the row holds an
                    // infinity: it would meet the zero weights there as NaN
                    So[row * MF_LD + j] = (__bf16)(in ? h : 0.f);
                }
        }
        __syncthreads();
    }
    // (layer 1 read S[1] and wrote S[0])
    mf_layer(S[0], g.w3, NT / 2, g.nto, acc);
#pragma unroll
    for (int u = 0; u < NW; u++) {
        const int t = wave + MF_WAVES * u, j = 16 * t + l16;
        if (t >= g.nto || j >= g.nout) continue;
        const float bj = g.b3[j];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 16 * a + 4 * q + r;
                if (row < left) g.Y[(row0 + row) * g.nout + j] = acc[a][u][r] + bj;
            }
    }
}

// Backward pass through the layers: dZ2 = (dY W3) gelu'(Z2), dZ1 = (dZ2 W2)
// gelu'(Z1).
template <int NT>
__global__ void __launch_bounds__(64 * MF_WAVES) k_mlp_bwd(MlpArgs g) {
    constexpr int NW = NT / MF_WAVES;
    __shared__ __attribute__((aligned(16))) __bf16 S[2][MF_ROWS * MF_LD];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
    const long row0 = (long)blockIdx.x * MF_ROWS;
    const int left = (int)min(g.rows - row0, (long)MF_ROWS);
    v4f acc[2][NW];
    mf_stage(S[0], g.dY, g.rows, row0, g.nout, g.ldy, g.kso);
#pragma unroll 1
    for (int layer = 0; layer < 2; layer++) {
        const float* Z = (layer ? g.Z1 : g.Z2) + row0 * g.width;
        float* dZ = (layer ? g.dZ1 : g.dZ2) + row0 * g.width;
        float z[NW][2][4];  // loaded ahead of the products
#pragma unroll
        for (int u = 0; u < NW; u++) {
            const int jc = min(16 * (wave + MF_WAVES * u) + l16, g.width - 1);
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int r = 0; r < 4; r++) z[u][a][r] = Z[min(16 * a + 4 * q + r, left - 1) * g.width + jc];
        }
        mf_layer(S[layer], layer ? g.w2t : g.w3t, layer ? NT / 2 : g.kso, NT, acc);
#pragma unroll
        for (int u = 0; u < NW; u++) {
            const int j = 16 * (wave + MF_WAVES * u) + l16;
            const bool in = j < g.width;
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = 16 * a + 4 * q + r;
                    const float d = acc[a][u][r] * gelu_grad(z[u][a][r]);
                    if (in && row < left) dZ[row * g.width + j] = d;
                    if (layer == 0) S[1][row * MF_LD + j] = (__bf16)(in ? d : 0.f);
                }
        }
        __syncthreads();
    }
}

// Weight and bias gradients: C[M][N] = A^T B over all rows (A [rows][M],
// B [rows][N]) and db[M] = column sums of A, for the three layers at once.
struct DwJob {
    const float *A, *B;
    float *C, *db;
    int M, N, ti, tj;  // tiles of 32 rows and columns
    int lda, ldb;
};
struct DwArgs {
    DwJob j[3];
    int rows;
    int tile0[4];  // first tile of each job; tile0[3]: all
    int col0[4];   // first bias block of each job; col0[3]: all
};
constexpr int DW_K = 128;      // rows per chunk of a product
constexpr int DW_AHEAD = 3;    // chunks in flight
constexpr int DW_LD = DW_K + 8;
constexpr int DW_COLS = 16;    // columns of a bias block
constexpr int DW_CHUNK = 512;  // rows per LDS chunk of a bias block

// Every sum runs over the rows in order (steps of 32 in the products, one by
// one in the biases), as a GEMM and a column sum per layer do, so it cannot be
// split: it is bound by the latency of the row loads over the rows in flight.
// A workgroup takes a 32 x 32 tile and keeps DW_AHEAD chunks of 128 rows in
// flight, each thread 8 rows x 4 columns, which it turns into the BF16
// operands' order on the way to LDS; or 16 bias columns, whose four waves load
// ahead for the lanes that add.  8192 rows of 92-256-256-10: 6.3 ms for the
// six launches before (16 workgroups with uncoalesced loads, one work-item per
// bias column), 91 us with a 16 x 16 tile per wave (63 loads in flight per wave
// are 4 steps), 53 us so (the biases alone 44 us: their adds are one chain).
template <bool VEC>
__global__ void __launch_bounds__(256) k_mlp_dw(DwArgs g) {
    union Lds {
        float bias[2][DW_COLS][DW_CHUNK + 4];
        __bf16 op[2][2][32][DW_LD];  // [buffer][A, B][column][row of the chunk]
    };
    __shared__ __attribute__((aligned(16))) Lds lds;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
    const int rows = g.rows;
    if ((int)blockIdx.x < g.col0[3]) {
        const int b = blockIdx.x, k = b < g.col0[1] ? 0 : b < g.col0[2] ? 1 : 2;
        const DwJob J = g.j[k];
        const int j = (b - g.col0[k]) * DW_COLS + l16, jc = min(j, J.M - 1);
        // wave w loads rows 128 w + 32 q .. + 31 of a chunk, one column per lane
        float v[32];
        auto load = [&](int c) {
            const int r0 = c * DW_CHUNK + 128 * wave + 32 * q;
#pragma unroll
            for (int i = 0; i < 32; i++) v[i] = J.A[(size_t)min(r0 + i, rows - 1) * J.lda + jc];
        };
        const int nc = (rows + DW_CHUNK - 1) / DW_CHUNK;
        float s = 0.f;
        load(0);
        for (int c = 0; c < nc; c++) {
            float(*d)[DW_CHUNK + 4] = lds.bias[c & 1];
#pragma unroll
            for (int i = 0; i < 32; i += 4)
                *reinterpret_cast<float4*>(&d[l16][128 * wave + 32 * q + i]) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
            __syncthreads();  // the other buffer's adds ended before the barrier of the last chunk
            if (c + 1 < nc) load(c + 1);
            if (threadIdx.x < DW_COLS) {
                const int n = min(DW_CHUNK, rows - c * DW_CHUNK);
                const float4* col = reinterpret_cast<const float4*>(d[l16]);
                if (n == DW_CHUNK) {
                    // 32 rows at a time, the next 32 read while these are added
                    float4 t[2][8];
#pragma unroll
                    for (int e = 0; e < 8; e++) t[0][e] = col[e];
#pragma unroll 1
                    for (int r = 0; r < DW_CHUNK / 4; r += 16) {
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const float4* nx = col + min(r + 8 * h + 8, DW_CHUNK / 4 - 8);
#pragma unroll
                            for (int e = 0; e < 8; e++) t[1 - h][e] = nx[e];
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int e = 0; e < 8; e++) {
                                s += t[h][e].x;
                                s += t[h][e].y;
                                s += t[h][e].z;
                                s += t[h][e].w;
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                } else {
                    for (int r = 0; r < n; r++) s += d[l16][r];
                }
            }
        }
        if (threadIdx.x < DW_COLS && j < J.M) J.db[j] = s;
        return;
    }
    const int tile = blockIdx.x - g.col0[3];
    const int k = tile < g.tile0[1] ? 0 : tile < g.tile0[2] ? 1 : 2;
    const DwJob J = g.j[k];
    const int ti = (tile - g.tile0[k]) / J.tj, tj = (tile - g.tile0[k]) % J.tj;
    // this thread's columns 4 cq .. 4 cq + 3 of A (half 0) or B and rows
    // 8 oc .. 8 oc + 7 of a chunk
    const int half = threadIdx.x >> 7, cq = threadIdx.x & 7, oc = (threadIdx.x >> 3) & 15;
    const float* src = half ? J.B : J.A;
    const int ld = half ? J.ldb : J.lda, c0 = 32 * (half ? tj : ti) + 4 * cq;
    float v[DW_AHEAD][8][4];
    auto load = [&](int u, int c) {
        if constexpr (VEC) {
            const float* p = src + min(c0, ld - 4);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float4 x = *reinterpret_cast<const float4*>(p + (size_t)min(DW_K * c + 8 * oc + e, rows - 1) * ld);
                v[u][e][0] = x.x;
                v[u][e][1] = x.y;
                v[u][e][2] = x.z;
                v[u][e][3] = x.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
#pragma unroll
                for (int f = 0; f < 4; f++)
                    v[u][e][f] = src[(size_t)min(DW_K * c + 8 * oc + e, rows - 1) * ld + min(c0 + f, ld - 1)];
        }
    };
    const int nc = (rows + DW_K - 1) / DW_K;
#pragma unroll
    for (int u = 0; u < DW_AHEAD; u++) load(u, u);
    const int wi = 16 * (wave >> 1), wj = 16 * (wave & 1);
    v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
    int b = 0;
    for (int c1 = 0; c1 < nc; c1 += DW_AHEAD) {
#pragma unroll
        for (int u = 0; u < DW_AHEAD; u++) {
            // chunks past the last are zeros (no early exit: the loads of the
            // ring would be waited for at its join)
            const int c = c1 + u;
#pragma unroll
            for (int f = 0; f < 4; f++) {
                bf16x8 o;
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = (__bf16)(DW_K * c + 8 * oc + e < rows ? v[u][e][f] : 0.f);
                *reinterpret_cast<bf16x8*>(&lds.op[b][half][4 * cq + f][8 * oc]) = o;
            }
            __syncthreads();  // the other buffer's reads ended before the last chunk's barrier
            load(u, c + DW_AHEAD);
#pragma unroll
            for (int s = 0; s < DW_K / 32; s++) {
                const bf16x8 af = *reinterpret_cast<const bf16x8*>(&lds.op[b][0][wi + l16][32 * s + 8 * q]);
                const bf16x8 bf = *reinterpret_cast<const bf16x8*>(&lds.op[b][1][wj + l16][32 * s + 8 * q]);
                if (c < nc) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, acc, 0, 0, 0);
            }
            b ^= 1;
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int i = 32 * ti + wi + 4 * q + r, j = 32 * tj + wj + l16;
        if (i < J.M && j < J.N) J.C[(size_t)i * J.N + j] = acc[r];
    }
}

// dY = 2 (Y - T) / (rows * cols); per-block partial sums of squared error.
// dY has rows of ldy values, of which nout are written.
__global__ void k_mse(long n, int nout, int ldy, const float* __restrict__ Y, const float* __restrict__ T, float scale,
                      float* __restrict__ dY, float* __restrict__ part) {
    __shared__ float red[256];
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    float e = 0.f;
    if (i < n) {
        const float d = Y[i] - T[i];
        dY[i / nout * ldy + i % nout] = 2.f * d * scale;
        e = d * d;
    }
    red[threadIdx.x] = e;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Adam on the FP32 master parameters.
__global__ void k_adam(long n, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                       float* __restrict__ m2, float lr, float b1, float b2, float eps, float c1, float c2) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.f - b1) * gi;
    const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    p[i] = p[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
}

}  // namespace lsd

using namespace lsd;

// Parameter block (FP32, contiguous): W1[W][in] b1[W] W2[W][W] b2[W] W3[out][W] b3[out]
struct lsd_mlp {
    int nin, width, nout;
    long np;
    hipStream_t stream = nullptr;
    lsd::HostStage stage;  // copies to and from the caller's arrays
    float* p = nullptr;   // parameters
    float* g = nullptr;   // gradients
    float* m1 = nullptr;  // Adam moments
    float* m2 = nullptr;
    long step = 0;
    // inputs and outputs (capacity io_cap rows), activations and gradients of
    // a training pass (capacity rows cap), training set of lsd_mlp_train
    long io_cap = 0, cap = 0, set_cap = 0;
    float *X = nullptr, *Z1 = nullptr, *H1 = nullptr, *Z2 = nullptr, *H2 = nullptr, *Y = nullptr, *T = nullptr;
    float *dY = nullptr, *dZ1 = nullptr, *dZ2 = nullptr, *part = nullptr;
    float *sx = nullptr, *st = nullptr;
    float* h_part = nullptr;
    int slots = 0;  // steps whose loss partials fit part and h_part
    // packed weights of the fused passes
    __bf16* pk = nullptr;
    bool fused() const { return nin <= FUSE_MAX && width <= FUSE_MAX && nto() <= mf_tiles(width); }
    int nt() const { return mf_tiles(width); }
    int nto() const { return (nout + 15) / 16; }
    int ks1() const { return (nin + 31) / 32; }
    int ks2() const { return nt() / 2; }
    int kso() const { return (nout + 31) / 32; }
    // sizes of the packed operands in NPACK order
    long pk_n(int k) const {
        const int s[NPACK] = {ks1() * nt(), ks2() * nt(), ks2() * nto(), kso() * nt(), ks2() * nt()};
        return (long)s[k] * 512;
    }
    __bf16* pk_at(int k) const {
        long o = 0;
        for (int i = 0; i < k; i++) o += pk_n(i);
        return pk + o;
    }
    int ldy() const { return (nout + 3) / 4 * 4; }          // row length of dY
    long nb_cap() const { return (cap * nout + 255) / 256; }  // loss partials per slot
    long o_w1() const { return 0; }
    long o_b1() const { return (long)width * nin; }
    long o_w2() const { return o_b1() + width; }
    long o_b2() const { return o_w2() + (long)width * width; }
    long o_w3() const { return o_b2() + width; }
    long o_b3() const { return o_w3() + (long)nout * width; }
};

// Losses of so many steps stay on the device before they are copied to the
// host together: 256, or as many as LOSS_BYTES hold partials of (one at least).
constexpr int LOSS_STEPS = 256;
constexpr long LOSS_BYTES = 4L << 20;
static int loss_slots(long nb) { return (int)std::max(1L, std::min((long)LOSS_STEPS, LOSS_BYTES / (long)sizeof(float) / nb)); }

static void mlp_free_rows(lsd_mlp* m) {
    float** bufs[] = {&m->Z1, &m->H1, &m->Z2, &m->H2, &m->T, &m->dY, &m->dZ1, &m->dZ2, &m->part};
    for (float** b : bufs) {
        if (*b) (void)hipFree(*b);
        *b = nullptr;
    }
    if (m->h_part) (void)hipHostFree(m->h_part);
    m->h_part = nullptr;
    m->cap = 0;
}
static void mlp_free_io(lsd_mlp* m) {
    if (m->X) (void)hipFree(m->X);
    if (m->Y) (void)hipFree(m->Y);
    m->X = m->Y = nullptr;
    m->io_cap = 0;
}
static void mlp_free_set(lsd_mlp* m) {
    if (m->sx) (void)hipFree(m->sx);
    if (m->st) (void)hipFree(m->st);
    m->sx = m->st = nullptr;
    m->set_cap = 0;
}

// room for `rows` inputs and outputs
static int mlp_io(lsd_mlp* m, long rows) {
    if (rows <= m->io_cap) return LSD_OK;
    mlp_free_io(m);
    LSD_HIP(hipMalloc((void**)&m->X, sizeof(float) * rows * m->nin));
    LSD_HIP(hipMalloc((void**)&m->Y, sizeof(float) * rows * m->nout));
    m->io_cap = rows;
    return LSD_OK;
}

// room for a training pass over `rows` rows (and for a forward pass of a GEMM
// per layer)
static int mlp_rows(lsd_mlp* m, long rows) {
    int rc = mlp_io(m, rows);
    if (rc || rows <= m->cap) return rc;
    mlp_free_rows(m);
    const long W = m->width;
    const long nb = (rows * m->nout + 255) / 256;
    float** hid[] = {&m->Z1, &m->H1, &m->Z2, &m->H2, &m->dZ1, &m->dZ2};
    for (float** b : hid) LSD_HIP(hipMalloc((void**)b, sizeof(float) * rows * W));
    LSD_HIP(hipMalloc((void**)&m->T, sizeof(float) * rows * m->nout));
    LSD_HIP(hipMalloc((void**)&m->dY, sizeof(float) * rows * m->ldy()));
    m->slots = loss_slots(nb);
    LSD_HIP(hipMalloc((void**)&m->part, sizeof(float) * nb * m->slots));
    LSD_HIP(hipHostMalloc((void**)&m->h_part, sizeof(float) * nb * m->slots, hipHostMallocDefault));
    m->cap = rows;
    return LSD_OK;
}

static MlpArgs mlp_args(const lsd_mlp* m, long rows, const float* x) {
    MlpArgs g{};
    g.rows = rows;
    g.nin = m->nin;
    g.width = m->width;
    g.nout = m->nout;
    g.nto = m->nto();
    g.ks1 = m->ks1();
    g.kso = m->kso();
    g.x = x;
    g.b1 = m->p + m->o_b1();
    g.b2 = m->p + m->o_b2();
    g.b3 = m->p + m->o_b3();
    g.w1 = m->pk_at(0);
    g.w2 = m->pk_at(1);
    g.w3 = m->pk_at(2);
    g.w3t = m->pk_at(3);
    g.w2t = m->pk_at(4);
    g.Z1 = m->Z1;
    g.H1 = m->H1;
    g.Z2 = m->Z2;
    g.H2 = m->H2;
    g.Y = m->Y;
    g.dY = m->dY;
    g.ldy = m->ldy();
    g.dZ1 = m->dZ1;
    g.dZ2 = m->dZ2;
    return g;
}

// packs the present weights for the fused passes
static int mlp_pack(lsd_mlp* m) {
    const long W = m->width;
    const float *w1 = m->p + m->o_w1(), *w2 = m->p + m->o_w2(), *w3 = m->p + m->o_w3();
    PackArgs a;
    a.j[0] = PackJob{w1, m->pk_at(0), m->nin, (int)W, m->nt(), m->ks1(), 1, m->nin};
    a.j[1] = PackJob{w2, m->pk_at(1), (int)W, (int)W, m->nt(), m->ks2(), 1, W};
    a.j[2] = PackJob{w3, m->pk_at(2), (int)W, m->nout, m->nto(), m->ks2(), 1, W};
    a.j[3] = PackJob{w3, m->pk_at(3), m->nout, (int)W, m->nt(), m->kso(), W, 1};
    a.j[4] = PackJob{w2, m->pk_at(4), (int)W, (int)W, m->nt(), m->ks2(), W, 1};
    long most = 0;
    for (int k = 0; k < NPACK; k++) most = std::max(most, m->pk_n(k) / 8);
    hipLaunchKernelGGL(k_mlp_pack, dim3((unsigned)((most + 255) / 256), NPACK), dim3(256), 0, m->stream, a);
    LSD_HIP(hipGetLastError());
    return LSD_OK;
}

template <class F>
static void by_tiles(int nt, F&& f) {
    if (nt == 4) f(std::integral_constant<int, 4>{});
    else if (nt == 8) f(std::integral_constant<int, 8>{});
    else f(std::integral_constant<int, 16>{});
}

// forward over rows at x (device) into m->Y; train: keep the activations
static int mlp_forward_dev(lsd_mlp* m, long rows, const float* x, bool train) {
    const int W = m->width;
    if (m->fused()) {
        int rc = mlp_pack(m);
        if (rc) return rc;
        const MlpArgs a = mlp_args(m, rows, x);
        const dim3 grid((unsigned)((rows + MF_ROWS - 1) / MF_ROWS));
        const auto run = [&](auto nt) {
            constexpr int NT = decltype(nt)::value;
            if (train) hipLaunchKernelGGL((k_mlp_fwd<NT, true>), grid, dim3(64 * MF_WAVES), 0, m->stream, a);
            else hipLaunchKernelGGL((k_mlp_fwd<NT, false>), grid, dim3(64 * MF_WAVES), 0, m->stream, a);
        };
        by_tiles(m->nt(), run);
        LSD_HIP(hipGetLastError());
        return LSD_OK;
    }
    GemmArgs g{};
    g.M = (int)rows;
    // layer 1: Z1 = X W1^T + b1, H1 = gelu(Z1)
    g.N = W; g.K = m->nin;
    g.A = x; g.sam = m->nin; g.sak = 1;
    g.B = m->p + m->o_w1(); g.sbk = 1; g.sbn = m->nin;
    g.C = m->H1; g.ldc = W; g.bias = m->p + m->o_b1(); g.act = 1; g.Z = m->Z1;
    int rc = gemm(m->stream, g);
    if (rc) return rc;
    // layer 2
    g.N = W; g.K = W;
    g.A = m->H1; g.sam = W; g.sak = 1;
    g.B = m->p + m->o_w2(); g.sbk = 1; g.sbn = W;
    g.C = m->H2; g.ldc = W; g.bias = m->p + m->o_b2(); g.act = 1; g.Z = m->Z2;
    if ((rc = gemm(m->stream, g))) return rc;
    // layer 3 (linear)
    g.N = m->nout; g.K = W;
    g.A = m->H2; g.sam = W; g.sak = 1;
    g.B = m->p + m->o_w3(); g.sbk = 1; g.sbn = W;
    g.C = m->Y; g.ldc = m->nout; g.bias = m->p + m->o_b3(); g.act = 0; g.Z = nullptr;
    return gemm(m->stream, g);
}

// loss partials (slot `slot` of m->part) and gradients for the forward pass of
// x against the targets t, both on the device
static int mlp_backward_dev(lsd_mlp* m, long rows, const float* x, const float* t, int slot) {
    const int W = m->width;
    const long ny = rows * m->nout;
    const long nb = (ny + 255) / 256;
    hipLaunchKernelGGL(k_mse, dim3((unsigned)nb), dim3(256), 0, m->stream, ny, m->nout, m->ldy(), m->Y, t, 1.0f / (float)ny, m->dY,
                       m->part + slot * m->nb_cap());
    if (m->fused()) {
        const MlpArgs a = mlp_args(m, rows, x);
        by_tiles(m->nt(), [&](auto nt) {
            hipLaunchKernelGGL(k_mlp_bwd<decltype(nt)::value>, dim3((unsigned)((rows + MF_ROWS - 1) / MF_ROWS)),
                               dim3(64 * MF_WAVES), 0, m->stream, a);
        });
        DwArgs d;
        d.rows = (int)rows;
        const int wt = (W + 31) / 32;

        d.j[0] = DwJob{m->dZ2, m->H1, m->g + m->o_w2(), m->g + m->o_b2(), W, W, wt, wt, W, W};
        d.j[1] = DwJob{m->dZ1, x, m->g + m->o_w1(), m->g + m->o_b1(), W, m->nin, wt, (m->nin + 31) / 32, W, m->nin};
        d.j[2] = DwJob{m->dY, m->H2, m->g + m->o_w3(), m->g + m->o_b3(), m->nout, W, (m->nout + 31) / 32, wt,
                       m->ldy(), W};
        d.tile0[0] = d.col0[0] = 0;
        for (int k = 0; k < 3; k++) {
            d.tile0[k + 1] = d.tile0[k] + d.j[k].ti * d.j[k].tj;
            d.col0[k + 1] = d.col0[k] + (d.j[k].M + DW_COLS - 1) / DW_COLS;
        }
        // 16-byte loads where all rows are aligned (dY's are padded to it; the
        // batch x may start at any row of the training set)
        const dim3 dg((unsigned)(d.col0[3] + d.tile0[3]));
        if (m->nin % 4 == 0 && W % 4 == 0) hipLaunchKernelGGL(k_mlp_dw<true>, dg, dim3(256), 0, m->stream, d);
        else hipLaunchKernelGGL(k_mlp_dw<false>, dg, dim3(256), 0, m->stream, d);
        LSD_HIP(hipGetLastError());
        return LSD_OK;
    }
    GemmArgs g{};
    int rc;
    // dW3 = dY^T H2  [nout x W],  db3 = colsum dY
    g.M = m->nout; g.N = W; g.K = (int)rows;
    g.A = m->dY; g.sam = 1; g.sak = m->ldy();
    g.B = m->H2; g.sbk = W; g.sbn = 1;
    g.C = m->g + m->o_w3(); g.ldc = W;
    if ((rc = gemm(m->stream, g))) return rc;
    hipLaunchKernelGGL(k_colsum, dim3((m->nout + 255) / 256), dim3(256), 0, m->stream, (int)rows, m->nout, m->ldy(), m->dY,
                       m->g + m->o_b3());
    // dH2 = dY W3  [rows x W];  dZ2 = dH2 gelu'(Z2)
    g = GemmArgs{};
    g.M = (int)rows; g.N = W; g.K = m->nout;
    g.A = m->dY; g.sam = m->ldy(); g.sak = 1;
    g.B = m->p + m->o_w3(); g.sbk = W; g.sbn = 1;
    g.C = m->dZ2; g.ldc = W;
    if ((rc = gemm(m->stream, g))) return rc;
    const long nw = rows * W;
    hipLaunchKernelGGL(k_gelu_back, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, m->stream, nw, m->Z2, m->dZ2);
    // dW2 = dZ2^T H1, db2
    g = GemmArgs{};
    g.M = W; g.N = W; g.K = (int)rows;
    g.A = m->dZ2; g.sam = 1; g.sak = W;
    g.B = m->H1; g.sbk = W; g.sbn = 1;
    g.C = m->g + m->o_w2(); g.ldc = W;
    if ((rc = gemm(m->stream, g))) return rc;
    hipLaunchKernelGGL(k_colsum, dim3((W + 255) / 256), dim3(256), 0, m->stream, (int)rows, W, W, m->dZ2,
                       m->g + m->o_b2());
    // dH1 = dZ2 W2, dZ1 = dH1 gelu'(Z1)
    g = GemmArgs{};
    g.M = (int)rows; g.N = W; g.K = W;
    g.A = m->dZ2; g.sam = W; g.sak = 1;
    g.B = m->p + m->o_w2(); g.sbk = W; g.sbn = 1;
    g.C = m->dZ1; g.ldc = W;
    if ((rc = gemm(m->stream, g))) return rc;
    hipLaunchKernelGGL(k_gelu_back, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, m->stream, nw, m->Z1, m->dZ1);
    // dW1 = dZ1^T X, db1
    g = GemmArgs{};
    g.M = W; g.N = m->nin; g.K = (int)rows;
    g.A = m->dZ1; g.sam = 1; g.sak = W;
    g.B = x; g.sbk = m->nin; g.sbn = 1;
    g.C = m->g + m->o_w1(); g.ldc = m->nin;
    if ((rc = gemm(m->stream, g))) return rc;
    hipLaunchKernelGGL(k_colsum, dim3((W + 255) / 256), dim3(256), 0, m->stream, (int)rows, W, W, m->dZ1,
                       m->g + m->o_b1());
    LSD_HIP(hipGetLastError());
    return LSD_OK;
}

// The losses of the first n slots of m->part, to the host: the partials of
// each are added in order.
static int mlp_losses(lsd_mlp* m, int n, const long* rows, float* loss) {
    const long nbc = m->nb_cap();
    LSD_HIP(hipMemcpyAsync(m->h_part, m->part, sizeof(float) * n * nbc, hipMemcpyDeviceToHost, m->stream));
    LSD_HIP(hipStreamSynchronize(m->stream));
    for (int k = 0; k < n; k++) {
        const long ny = rows[k] * m->nout, nb = (ny + 255) / 256;
        double s = 0.0;
        for (long b = 0; b < nb; b++) s += m->h_part[k * nbc + b];
        loss[k] = (float)(s / (double)ny);
    }
    return LSD_OK;
}

extern "C" {

int lsd_mlp_create(int n_in, int width, int n_out, unsigned long long seed, lsd_mlp** out) {
    if (!out || n_in < 1 || width < 1 || n_out < 1) {
        lsd::set_error("lsd_mlp_create: bad sizes");
        return LSD_E_ARG;
    }
    *out = nullptr;
    lsd_mlp* m = new lsd_mlp();
    m->nin = n_in;
    m->width = width;
    m->nout = n_out;
    m->np = m->o_b3() + n_out;
    auto fail = [&](void) {
        if (m->pk) (void)hipFree(m->pk);
        if (m->p) (void)hipFree(m->p);
        if (m->g) (void)hipFree(m->g);
        if (m->m1) (void)hipFree(m->m1);
        if (m->m2) (void)hipFree(m->m2);
        if (m->stream) (void)hipStreamDestroy(m->stream);
        delete m;
        return LSD_E_HIP;
    };
    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess ||
        hipMalloc((void**)&m->p, sizeof(float) * m->np) != hipSuccess ||
        hipMalloc((void**)&m->g, sizeof(float) * m->np) != hipSuccess ||
        hipMalloc((void**)&m->m1, sizeof(float) * m->np) != hipSuccess ||
        hipMalloc((void**)&m->m2, sizeof(float) * m->np) != hipSuccess ||
        (m->fused() && hipMalloc((void**)&m->pk, (size_t)((char*)m->pk_at(NPACK) - (char*)m->pk)) != hipSuccess)) {
        lsd::set_error("lsd_mlp_create: allocation failed");
        return fail();
    }
    // He-style initial weights from a 64-bit LCG (host), zero biases
    std::vector<float> h(m->np, 0.0f);
    unsigned long long s = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    auto uni = [&]() {
        s = s * 6364136223846793005ULL + 1442695040888963407ULL;
        return (double)(s >> 11) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](long off, long n, int fan_in) {
        const double a = std::sqrt(6.0 / fan_in);
        for (long i = 0; i < n; i++) h[off + i] = (float)((2.0 * uni() - 1.0) * a);
    };
    fill(m->o_w1(), (long)width * n_in, n_in);
    fill(m->o_w2(), (long)width * width, width);
    fill(m->o_w3(), (long)n_out * width, width);
    if (hipMemcpy(m->p, h.data(), sizeof(float) * m->np, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(m->m1, 0, sizeof(float) * m->np) != hipSuccess ||
        hipMemset(m->m2, 0, sizeof(float) * m->np) != hipSuccess) {
        lsd::set_error("lsd_mlp_create: initialisation failed");
        return fail();
    }
    *out = m;
    return LSD_OK;
}

void lsd_mlp_destroy(lsd_mlp* m) {
    if (!m) return;
    mlp_free_rows(m);
    mlp_free_io(m);
    mlp_free_set(m);
    if (m->pk) (void)hipFree(m->pk);
    (void)hipFree(m->p);
    (void)hipFree(m->g);
    (void)hipFree(m->m1);
    (void)hipFree(m->m2);
    m->stage.release();
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

long lsd_mlp_num_params(const lsd_mlp* m) { return m ? m->np : 0; }

int lsd_mlp_get_params(lsd_mlp* m, float* out) {
    if (!m || !out) { lsd::set_error("lsd_mlp_get_params: null"); return LSD_E_ARG; }
    LSD_HIP(hipMemcpy(out, m->p, sizeof(float) * m->np, hipMemcpyDeviceToHost));
    return LSD_OK;
}

int lsd_mlp_set_params(lsd_mlp* m, const float* in) {
    if (!m || !in) { lsd::set_error("lsd_mlp_set_params: null"); return LSD_E_ARG; }
    LSD_HIP(hipMemcpy(m->p, in, sizeof(float) * m->np, hipMemcpyHostToDevice));
    return LSD_OK;
}

int lsd_mlp_forward(lsd_mlp* m, long rows, const float* x, float* y) {
    if (!m || !x || !y || rows < 1) { lsd::set_error("lsd_mlp_forward: bad arguments"); return LSD_E_ARG; }
    int rc = m->fused() ? mlp_io(m, rows) : mlp_rows(m, rows);
    if (rc) return rc;
    const lsd::HostPart in = {const_cast<float*>(x), m->X, sizeof(float) * rows * m->nin};
    const lsd::HostPart out = {y, m->Y, sizeof(float) * rows * m->nout};
    lsd::CopyGuard guard(m->stream);
    // from 16 MiB on the chunks: rows kept from call to call take 920 us that
    // way at 21 MB and 780 directly, new rows with new results 990 and 1140
    if ((rc = lsd::host_copy(m->stage, m->stream, &in, 1, false, size_t(16) << 20))) return rc;
    if ((rc = mlp_forward_dev(m, rows, m->X, false))) return rc;
    return guard.pass(lsd::host_copy(m->stage, m->stream, &out, 1, true));
}

int lsd_mlp_grad(lsd_mlp* m, long rows, const float* x, const float* target, float* loss, float* grad) {
    if (!m || !x || !target || rows < 1) { lsd::set_error("lsd_mlp_grad: bad arguments"); return LSD_E_ARG; }
    int rc = mlp_rows(m, rows);
    if (rc) return rc;
    lsd::CopyGuard guard(m->stream);
    LSD_HIP(hipMemcpyAsync(m->X, x, sizeof(float) * rows * m->nin, hipMemcpyHostToDevice, m->stream));
    LSD_HIP(hipMemcpyAsync(m->T, target, sizeof(float) * rows * m->nout, hipMemcpyHostToDevice, m->stream));
    if ((rc = mlp_forward_dev(m, rows, m->X, true))) return rc;
    if ((rc = mlp_backward_dev(m, rows, m->X, m->T, 0))) return rc;
    if (loss && (rc = mlp_losses(m, 1, &rows, loss))) return rc;
    if (grad) LSD_HIP(hipMemcpyAsync(grad, m->g, sizeof(float) * m->np, hipMemcpyDeviceToHost, m->stream));
    LSD_HIP(hipStreamSynchronize(m->stream));
    return guard.pass(LSD_OK);
}

// Adam steps on minibatches drawn in order from (x, target) [rows x n],
// batch rows each (the last batch of a pass may be shorter); the data are
// copied to the device once per call.  loss[steps] receives the minibatch
// losses (may be null).
int lsd_mlp_train(lsd_mlp* m, long rows, const float* x, const float* target, long batch, int steps, float lr,
                  float* loss) {
    if (!m || !x || !target || rows < 1 || batch < 1 || steps < 0) {
        lsd::set_error("lsd_mlp_train: bad arguments");
        return LSD_E_ARG;
    }
    if (batch > rows) batch = rows;
    if (rows > m->set_cap) {
        mlp_free_set(m);
        LSD_HIP(hipMalloc((void**)&m->sx, sizeof(float) * rows * m->nin));
        LSD_HIP(hipMalloc((void**)&m->st, sizeof(float) * rows * m->nout));
        m->set_cap = rows;
    }
    int rc = mlp_rows(m, batch);
    if (rc) return rc;
    lsd::CopyGuard guard(m->stream);
    LSD_HIP(hipMemcpyAsync(m->sx, x, sizeof(float) * rows * m->nin, hipMemcpyHostToDevice, m->stream));
    LSD_HIP(hipMemcpyAsync(m->st, target, sizeof(float) * rows * m->nout, hipMemcpyHostToDevice, m->stream));
    long pos = 0;
    long nrows[LOSS_STEPS];  // of the steps whose losses are still on the device
    int nl = 0;
    for (int s = 0; s < steps; s++) {
        const long nrow = std::min(batch, rows - pos);
        const float* xs = m->sx + pos * m->nin;
        pos = (pos + nrow) % rows;
        if ((rc = mlp_forward_dev(m, nrow, xs, true))) break;
        if ((rc = mlp_backward_dev(m, nrow, xs, m->st + (xs - m->sx) / m->nin * m->nout, nl))) break;
        m->step++;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.f - powf(b1, (float)m->step), c2 = 1.f - powf(b2, (float)m->step);
        hipLaunchKernelGGL(k_adam, dim3((unsigned)((m->np + 255) / 256)), dim3(256), 0, m->stream, m->np, m->p, m->g,
                           m->m1, m->m2, lr, b1, b2, 1e-8f, c1, c2);
        LSD_HIP(hipGetLastError());
        if (!loss) continue;
        nrows[nl++] = nrow;
        if (nl == m->slots || s + 1 == steps) {
            if ((rc = mlp_losses(m, nl, nrows, loss + s + 1 - nl))) break;
            nl = 0;
        }
    }
    LSD_HIP(hipStreamSynchronize(m->stream));
    return guard.pass(rc);
}

}  // extern "C"
