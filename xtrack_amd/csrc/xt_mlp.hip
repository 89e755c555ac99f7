// xt_mlp.hip -- BF16 matrix products with FP32 accumulation on the CDNA4
// matrix cores, for the survival-turn surrogate network (training and
// inference).  No counterpart in the reference.
//
// C[M x N] = op(A)[M x K] . op(B)[K x N] (+ bias[n]) (ReLU), where op(A)(m, k)
// = A[m * sam + k * sak] and op(B)(k, n) = B[k * sbk + n * sbn]: strides
// select plain or transposed operands, which is all the forward pass
// (X W), the input gradient (dZ W^T) and the weight gradient (X^T dZ)
// need.  The result is written in FP32 and, optionally, rounded to BF16
// (round to nearest even) for the next product.
//
// Each 256-thread block computes a 64 x 64 tile of C over a range of k: the
// four waves stage 64 x 32 tiles of op(A) and op(B) in LDS (k contiguous
// per row, so that a lane's fragment is one 16-byte LDS read; 16-byte
// global loads where the operand allows, the next k step's tiles loaded
// into registers while this step's products run), then each wave
// multiplies its 32 x 32 quarter as 2 x 2 tiles of gfx950's
// v_mfma_f32_16x16x32_bf16.  The result tile goes back through LDS so
// that each thread writes 16 consecutive columns of one row with vector
// stores (FP32, and the BF16 copy).  Block ids map to tiles so that the
// column tiles of one row tile run on one XCD (shared op(A) rows in one L2).  Operand layout of that instruction (64 lanes,
// lane l): A holds row l % 16 and the eight consecutive k = 8 (l / 16) + j;
// B holds column l % 16 and the same k; the accumulator holds column l % 16
// and rows 4 (l / 16) + j, j < 4.
//
// Products with few output tiles and a long k (the weight gradient X^T dZ
// over a batch) split k over up to 256 / tiles blocks (grid z); each block
// writes its partial tile to a workspace and a second kernel sums the
// partials in split order (deterministic) and applies bias, ReLU and the
// BF16 rounding.  The workspace is at most GEMM_WS_FLOATS floats: the
// library allocates it once per device for xtm_gemm_bf16;
// xtm_gemm_bf16_noalloc uses a file-scope device array instead.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>

#include "../../include/xtrack_amd.h"

int32_t xt_report_error(int32_t code, const char *msg);   // xt_kernel.hip

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

constexpr int TM = 64, TN = 64, TK = 32;
constexpr int LDK = TK + 8;     // LDS row: 40 bf16 = 80 bytes (16-byte aligned fragments)
constexpr int CLD = TN + 4;     // LDS row of the result tile: 68 floats (16-byte aligned)
constexpr int64_t GEMM_WS_FLOATS = 1 << 20;   // split partials: splits x M x N <= 256 x 64 x 64

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu))   // NaN: keep it quiet
        return (uint16_t)((u >> 16) | 0x0040u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

/* A thread's share of the op(X) tile rows r0.., k k0.. (bf16 bits, zero
   outside [0, R) x [0, Kend)); X(r, k) = X[r * sr + k * sk].  256 threads,
   8 elements each: with k contiguous (sk == 1) 8 consecutive k of one row,
   with rows contiguous (sr == 1) 8 consecutive rows of one k, else 8
   elements 256 apart in the tile.  Contiguous elements inside the operand
   that start on a 16-byte boundary are one 16-byte load. */
__device__ __forceinline__ u16x8 load_tile(const uint16_t *__restrict__ X, int64_t sr,
                                           int64_t sk, int64_t r0, int64_t k0, int64_t R,
                                           int64_t Kend, int tid) {
    const bool base16 = ((uintptr_t)X & 15) == 0;
    u16x8 v;
    if (sk == 1) {
        const int r = tid >> 2, c = (tid & 3) * 8;
        const int64_t row = r0 + r, k = k0 + c, off = row * sr + k;
        if (base16 && row < R && k + 8 <= Kend && (off & 7) == 0)
            return *reinterpret_cast<const u16x8 *>(&X[off]);
        for (int j = 0; j < 8; j++) v[j] = (row < R && k + j < Kend) ? X[off + j] : (uint16_t)0;
    } else if (sr == 1) {
        const int kk = tid >> 3, r = (tid & 7) * 8;
        const int64_t k = k0 + kk, row = r0 + r, off = row + k * sk;
        if (base16 && k < Kend && row + 8 <= R && (off & 7) == 0)
            return *reinterpret_cast<const u16x8 *>(&X[off]);
        for (int j = 0; j < 8; j++) v[j] = (row + j < R && k < Kend) ? X[off + j] : (uint16_t)0;
    } else {
        for (int j = 0; j < 8; j++) {
            const int e = tid + 256 * j, r = e / TK, c = e % TK;
            const int64_t row = r0 + r, k = k0 + c;
            v[j] = (row < R && k < Kend) ? X[row * sr + k * sk] : (uint16_t)0;
        }
    }
    return v;
}

/* The thread's share (load_tile) into the LDS tile S[row][k]. */
__device__ __forceinline__ void store_tile(uint16_t *S, const u16x8 v, int64_t sr, int64_t sk,
                                           int tid) {
    if (sk == 1) {
        const int r = tid >> 2, c = (tid & 3) * 8;
        *reinterpret_cast<u16x8 *>(&S[r * LDK + c]) = v;
    } else if (sr == 1) {
        const int kk = tid >> 3, r = (tid & 7) * 8;
        for (int j = 0; j < 8; j++) S[(r + j) * LDK + kk] = v[j];
    } else {
        for (int j = 0; j < 8; j++) {
            const int e = tid + 256 * j;
            S[(e / TK) * LDK + e % TK] = v[j];
        }
    }
}

/* Block (x, y, z): C tile rows 64 y.., columns 64 x.., k range
   [z kc, min(K, (z + 1) kc)).  With ws == nullptr the tile gets the
   epilogue and goes to C/Cb; else the raw partial goes to ws[z][m][n].
   MASK: the result is zeroed where mask is not positive (a code of its own:
   the test alone costs the other products 3 to 5 % of 65,536 rows). */
template <bool MASK>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(
    const uint16_t *__restrict__ A, int64_t sam, int64_t sak, const uint16_t *__restrict__ B,
    int64_t sbk, int64_t sbn, float *__restrict__ C, int64_t ldc, uint16_t *__restrict__ Cb,
    const float *__restrict__ bias, int32_t relu, const float *__restrict__ mask, int64_t M,
    int64_t N, int64_t K, int64_t kc, float *__restrict__ ws) {
    // operand tiles during the k loop, the result tile after it
    __shared__ __align__(16) unsigned char smem[TM * CLD * 4];
    uint16_t *As = reinterpret_cast<uint16_t *>(smem);
    uint16_t *Bs = As + TM * LDK;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // Workgroups go to the eight XCDs round-robin by linear id, and each XCD
    // has its own L2: map the ids so that the column tiles of one row tile
    // (which read the same op(A) rows) run on one XCD.  Row tile t goes to
    // XCD t % 8; a bijection when the row-tile count is a multiple of 8.
    int64_t ty = blockIdx.y, tx = blockIdx.x;
    if ((gridDim.y & 7) == 0) {
        const int64_t lin = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
        const int64_t xcd = lin & 7, local = lin >> 3;
        tx = local % gridDim.x;
        ty = xcd + 8 * (local / gridDim.x);
    }
    const int64_t m0 = ty * TM, n0 = tx * TN;
    const int wm = 32 * (w >> 1), wn = 32 * (w & 1);
    const int r16 = lane & 15, kq = (lane >> 4) * 8;
    const int64_t kbeg = (int64_t)blockIdx.z * kc;
    const int64_t kend = kbeg + kc < K ? kbeg + kc : K;
    f32x4 acc[2][2];
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // op(B)(k, n): rows of the staged tile are n, its k stride sbk.  The
    // next k step's tiles are loaded into registers while this one's
    // products run.
    u16x8 va, vb;
    if (kbeg < kend) {
        va = load_tile(A, sam, sak, m0, kbeg, M, kend, tid);
        vb = load_tile(B, sbn, sbk, n0, kbeg, N, kend, tid);
    }
    for (int64_t k0 = kbeg; k0 < kend; k0 += TK) {
        store_tile(As, va, sam, sak, tid);
        store_tile(Bs, vb, sbn, sbk, tid);
        __syncthreads();
        if (k0 + TK < kend) {
            va = load_tile(A, sam, sak, m0, k0 + TK, M, kend, tid);
            vb = load_tile(B, sbn, sbk, n0, k0 + TK, N, kend, tid);
        }
        bf16x8 a[2], b[2];
        for (int i = 0; i < 2; i++) {
            a[i] = *reinterpret_cast<const bf16x8 *>(&As[(wm + 16 * i + r16) * LDK + kq]);
            b[i] = *reinterpret_cast<const bf16x8 *>(&Bs[(wn + 16 * i + r16) * LDK + kq]);
        }
        for (int i = 0; i < 2; i++)
            for (int j = 0; j < 2; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        __syncthreads();
    }
    // the tile through LDS, so that each thread writes 16 consecutive
    // columns of one row (vector stores where the row lies inside C)
    float *Cs = reinterpret_cast<float *>(smem);
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++)
            for (int q = 0; q < 4; q++)
                Cs[(wm + 16 * i + 4 * (lane >> 4) + q) * CLD + wn + 16 * j + r16] = acc[i][j][q];
    __syncthreads();
    const int row = tid >> 2, c0 = (tid & 3) * 16;
    const int64_t m = m0 + row;
    if (m >= M) return;
    float *out = ws ? ws + ((int64_t)blockIdx.z * M + m) * N : C + m * ldc;
    const bool vec = (((uintptr_t)out & 15) == 0) && (ws || !Cb || ((uintptr_t)(Cb + m * ldc) & 7) == 0);
    for (int c = c0; c < c0 + 16; c += 4) {
        const int64_t n = n0 + c;
        if (n >= N) break;
        f32x4 v = *reinterpret_cast<const f32x4 *>(&Cs[row * CLD + c]);
        if (!ws) {
            for (int e = 0; e < 4; e++) {
                if (bias && n + e < N) v[e] += bias[n + e];
                if (relu && !(v[e] > 0.f)) v[e] = 0.f;
                if (MASK && n + e < N) v[e] *= mask[m * ldc + n + e] > 0.f ? 1.f : 0.f;
            }
        }
        if (vec && n + 4 <= N) {
            *reinterpret_cast<f32x4 *>(&out[n]) = v;
            if (!ws && Cb) {
                uint16_t b4[4] = {f32_to_bf16_rne(v[0]), f32_to_bf16_rne(v[1]),
                                  f32_to_bf16_rne(v[2]), f32_to_bf16_rne(v[3])};
                uint64_t packed;
                __builtin_memcpy(&packed, b4, 8);
                *reinterpret_cast<uint64_t *>(&Cb[m * ldc + n]) = packed;
            }
        } else {
            for (int e = 0; e < 4 && n + e < N; e++) {
                out[n + e] = v[e];
                if (!ws && Cb) Cb[m * ldc + n + e] = f32_to_bf16_rne(v[e]);
            }
        }
    }
}

/* Sum of the `splits` partial tiles in split order, then the epilogue. */
__global__ __launch_bounds__(256) void gemm_reduce_kernel(
    const float *__restrict__ ws, int64_t splits, float *__restrict__ C, int64_t ldc,
    uint16_t *__restrict__ Cb, const float *__restrict__ bias, int32_t relu,
    const float *__restrict__ mask, int64_t M, int64_t N) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= M * N) return;
    const int64_t m = e / N, n = e % N;
    float v = 0.f;
    for (int64_t s = 0; s < splits; s++) v += ws[s * M * N + e];
    if (bias) v += bias[n];
    if (relu && !(v > 0.f)) v = 0.f;
    if (mask) v *= mask[m * ldc + n] > 0.f ? 1.f : 0.f;
    C[m * ldc + n] = v;
    if (Cb) Cb[m * ldc + n] = f32_to_bf16_rne(v);
}

/* k split: more blocks for products with few output tiles and a long k */
int64_t gemm_splits(int64_t M, int64_t N, int64_t K, int64_t *kc) {
    const int64_t tiles = ((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    int64_t s = 1;
    if (tiles < 128 && K > 8 * TK) {
        s = (K + 8 * TK - 1) / (8 * TK);          // at least 8 k-steps per block
        const int64_t cap = 256 / tiles > 1 ? 256 / tiles : 1;
        if (s > cap) s = cap;
    }
    int64_t c = (K + s - 1) / s;
    c = (c + TK - 1) / TK * TK;
    *kc = c > 0 ? c : TK;
    return (K + *kc - 1) / *kc > 0 ? (K + *kc - 1) / *kc : 1;
}

int32_t gemm_launch(const uint16_t *A, int64_t sam, int64_t sak, const uint16_t *B,
                    int64_t sbk, int64_t sbn, float *C, int64_t ldc, uint16_t *Cb,
                    const float *bias, int32_t relu, int64_t M, int64_t N, int64_t K,
                    hipStream_t stream, float *ws, int64_t ws_floats, int64_t splits,
                    int64_t kc, const float *mask = nullptr) {
    const int64_t gy = (M + TM - 1) / TM, gx = (N + TN - 1) / TN;
    const auto product = mask ? gemm_bf16_kernel<true> : gemm_bf16_kernel<false>;
    if (splits > 1) {
        if (!ws || splits * M * N > ws_floats)
            return xt_report_error(XTM_ERR_ARG, "xtm_gemm_bf16: split partials exceed the "
                                                "workspace");
        hipLaunchKernelGGL(product, dim3((unsigned)gx, (unsigned)gy, (unsigned)splits),
                           dim3(256), 0, stream, A, sam, sak, B, sbk, sbn, C, ldc, Cb, bias,
                           relu, mask, M, N, K, kc, ws);
        if (hipGetLastError() != hipSuccess)
            return xt_report_error(XTM_ERR_HIP, "xtm_gemm_bf16: kernel launch failed");
        const int64_t nb = (M * N + 255) / 256;
        hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)nb), dim3(256), 0, stream, ws,
                           splits, C, ldc, Cb, bias, relu, mask, M, N);
    } else {
        hipLaunchKernelGGL(product, dim3((unsigned)gx, (unsigned)gy, 1), dim3(256), 0, stream,
                            A, sam, sak, B, sbk, sbn, C, ldc, Cb, bias, relu, mask, M, N,
                           K, K > 0 ? K : 1, (float *)nullptr);
    }
    return hipGetLastError() == hipSuccess
               ? XTM_OK
               : xt_report_error(XTM_ERR_HIP, "xtm_gemm_bf16: kernel launch failed");
}

int32_t gemm_check(const uint16_t *A, const uint16_t *B, const float *C, int64_t ldc,
                   int64_t M, int64_t N, int64_t K) {
    if (!A || !B || !C || M < 0 || N < 0 || K < 0 || ldc < N)
        return xt_report_error(XTM_ERR_ARG, "xtm_gemm_bf16: null operand, negative size or "
                                            "ldc < N");
    const int64_t gy = (M + TM - 1) / TM, gx = (N + TN - 1) / TN;
    if (gy > 65535 || gx > 0x7fffffff)
        return xt_report_error(XTM_ERR_ARG, "xtm_gemm_bf16: M above 65535 * 64 rows");
    return XTM_OK;
}

/* ---- the 16-256-256-256-1 network in one kernel ------------------------------
 *
 * Layer by layer through xtm_gemm_bf16 a prediction moves every activation
 * through HBM in FP32 and BF16: 262,147 rows took 0.99 ms.  Here the
 * activations stay in registers from the input to the output: 0.076 ms, 940
 * TFLOP/s (a large BF16 library product on this card: 1230).
 *
 * The products run transposed, Z^T = W^T H^T: weights are the A operand (rows:
 * output features), activations the B operand (columns: batch rows), so that a
 * lane's results belong to its own batch column.  The accumulator of a
 * 16-feature tile holds features 4 (l / 16) + j of column l % 16 in lane l; the
 * next layer's B operand wants features 8 (l / 16) + j, j < 8, of a 32-feature
 * step.  Two tiles a, b of one step become that operand by swapping the lower
 * half of b with the upper half of a and then the odd rows of 16 lanes of one
 * with the even rows of the other: 2 swaps per 32-bit word, no LDS.  Every
 * k step multiplies the same 32 features in the same places as
 * gemm_bf16_kernel, steps in order, so the results are the same bits.
 *
 * A wave carries MLP_CT = 3 column tiles (48 batch rows): with 4 tiles the two
 * layers' operands alone are 256 registers; with 3 a wave stays within 256 and
 * two blocks share a CU.  A weight fragment (1 KB) read from LDS serves 3
 * products of 16 cycles: 85 bytes per clock and CU, of 128.  Weights come
 * packed in fragment order and pass through LDS in chunks of 64 features (32
 * KB), the next chunk copied by global_load_lds while this one multiplies. */
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int MLP_H = 256;                       // hidden width
constexpr int MLP_IN = 16;
constexpr int MLP_CT = 3;                        // column tiles per wave
constexpr int MLP_ROWS = 4 * 16 * MLP_CT;        // batch rows per block
constexpr int MLP_FRAG = 1024;                   // bytes of one 16 x 32 fragment
constexpr int MLP_CHUNK = 32 * MLP_FRAG;         // 64 features x 256 inputs
// packed weights in bytes: layer 1 (16 tiles x 1 step), 2 and 3 (16 x 8),
// 4 (1 x 8), then the biases (3 x 256 + 1 floats)
constexpr int MLP_P1 = 0, MLP_P2 = 16 * MLP_FRAG, MLP_P3 = MLP_P2 + 128 * MLP_FRAG,
              MLP_P4 = MLP_P3 + 128 * MLP_FRAG, MLP_PB = MLP_P4 + 8 * MLP_FRAG,
              MLP_PACKED = MLP_PB + (3 * MLP_H + 4) * 4;

struct MlpWeights {
    const float *w[4];   // [in][out] row-major
    const float *b[4];
};

/* Packed fragments: fragment (tile t, step s) of a layer holds, for lane l and
   j < 8, W[k = 32 s + 8 (l / 16) + j][n = 16 t + l % 16] in BF16 (zero outside
   the layer).  One thread per lane and fragment; 280 fragments. */
__global__ __launch_bounds__(256) void mlp_pack_kernel(MlpWeights W, unsigned char *out) {
    const int idx = blockIdx.x * 256 + threadIdx.x;
    const int f = idx >> 6, lane = idx & 63;
    if (f < 280) {
        int layer, t, st;
        if (f < 16) { layer = 0; t = f; st = 0; }
        else if (f < 144) { layer = 1; t = (f - 16) >> 3; st = (f - 16) & 7; }
        else if (f < 272) { layer = 2; t = (f - 144) >> 3; st = (f - 144) & 7; }
        else { layer = 3; t = 0; st = f - 272; }
        const int K = layer == 0 ? MLP_IN : MLP_H, N = layer == 3 ? 1 : MLP_H;
        const int n = 16 * t + (lane & 15), k0 = 32 * st + 8 * (lane >> 4);
        u16x8 v;
        for (int j = 0; j < 8; j++)
            v[j] = (k0 + j < K && n < N)
                       ? f32_to_bf16_rne(W.w[layer][(int64_t)(k0 + j) * N + n])
                       : (uint16_t)0;
        *reinterpret_cast<u16x8 *>(out + (int64_t)f * MLP_FRAG + lane * 16) = v;
    } else {
        const int k = idx - 280 * 64;
        float *bo = reinterpret_cast<float *>(out + MLP_PB);
        if (k < 3 * MLP_H) bo[k] = W.b[k >> 8][k & 255];
        else if (k == 3 * MLP_H) bo[k] = W.b[3][0];
    }
}

/* `bytes` (a multiple of 4096) from global memory into LDS, 16 bytes a lane,
   asynchronous: complete after the next s_waitcnt vmcnt(0) and barrier */
__device__ __forceinline__ void copy_to_lds(const unsigned char *src, unsigned char *dst,
                                            int bytes) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int o = wave * 1024; o < bytes; o += 4096)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void *)(src + o + lane * 16),
            (__attribute__((address_space(3))) void *)(dst + o), 16, 0, 0);
}

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    bf16x2 v;
    v[0] = (__bf16)a;
    v[1] = (__bf16)b;
    uint32_t u;
    __builtin_memcpy(&u, &v, 4);
    return u;
}

__device__ __forceinline__ void swap_tiles(uint32_t &a, uint32_t &b) {
    u32x2 r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    r = __builtin_amdgcn_permlane16_swap(r[0], r[1], false, false);
    a = r[0];
    b = r[1];
}

/* One 32-feature step p of a hidden layer (tiles 2p, 2p + 1): products over
   STEPS k steps, bias, ReLU, BF16, and the next layer's operand of the step. */
template <int STEPS>
__device__ __forceinline__ void mlp_step(const unsigned char *frag, const float *bias,
                                         const bf16x8 (&in)[STEPS][MLP_CT],
                                         bf16x8 (&out)[MLP_CT], int lane) {
    f32x4 acc[2][MLP_CT];
    for (int t = 0; t < 2; t++)
        for (int c = 0; c < MLP_CT; c++) acc[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < STEPS; s++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const bf16x8 w = *reinterpret_cast<const bf16x8 *>(
                frag + (t * STEPS + s) * MLP_FRAG + lane * 16);
#pragma unroll
            for (int c = 0; c < MLP_CT; c++)
                acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, in[s][c], acc[t][c], 0, 0, 0);
        }
    uint32_t h[2][MLP_CT][2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(&bias[16 * t + 4 * (lane >> 4)]);
#pragma unroll
        for (int c = 0; c < MLP_CT; c++) {
            float v[4];
            for (int j = 0; j < 4; j++) {
                v[j] = acc[t][c][j] + b[j];
                if (!(v[j] > 0.f)) v[j] = 0.f;
            }
            h[t][c][0] = pack_bf16(v[0], v[1]);
            h[t][c][1] = pack_bf16(v[2], v[3]);
        }
    }
#pragma unroll
    for (int c = 0; c < MLP_CT; c++) {
        swap_tiles(h[0][c][0], h[1][c][0]);
        swap_tiles(h[0][c][1], h[1][c][1]);
        const u32x4 u = {h[0][c][0], h[0][c][1], h[1][c][0], h[1][c][1]};
        __builtin_memcpy(&out[c], &u, 16);
    }
}

/* out[r] = network((x[r] - mean) / std) * y_std + y_mean for r < M (mean
   nullptr: x as it is; scale 0: without y_std and y_mean) */
__global__ __launch_bounds__(256, 2) void mlp_forward_kernel(
    const float *__restrict__ x, const float *__restrict__ mean, const float *__restrict__ std,
    const unsigned char *__restrict__ packed, float *__restrict__ out, int64_t M, int32_t scale,
    float y_std, float y_mean) {
    __shared__ __align__(16) unsigned char wbuf[2][MLP_CHUNK];
    __shared__ __align__(16) float bias[3 * MLP_H + 4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, g = lane >> 4;
    const int64_t row0 = (int64_t)blockIdx.x * MLP_ROWS + wave * 16 * MLP_CT + col;
    copy_to_lds(packed + MLP_P1, wbuf[0], 16 * MLP_FRAG);
    for (int k = threadIdx.x; k < 3 * MLP_H + 1; k += 256)
        bias[k] = reinterpret_cast<const float *>(packed + MLP_PB)[k];
    // the input operand: features 8 g + j of batch row row0 + 16 c, one step,
    // zero from feature 16 on
    bf16x8 x0[1][MLP_CT];
#pragma unroll
    for (int c = 0; c < MLP_CT; c++) {
        const int64_t row = row0 + 16 * c;
        float v[8];
        for (int j = 0; j < 8; j++) v[j] = 0.f;
        if (g < 2 && row < M) {
            const f32x4 a = *reinterpret_cast<const f32x4 *>(&x[row * MLP_IN + 8 * g]);
            const f32x4 b = *reinterpret_cast<const f32x4 *>(&x[row * MLP_IN + 8 * g + 4]);
            for (int j = 0; j < 4; j++) {
                v[j] = a[j];
                v[j + 4] = b[j];
            }
            if (mean)
                for (int j = 0; j < 8; j++) v[j] = (v[j] - mean[8 * g + j]) / std[8 * g + j];
        }
        for (int j = 0; j < 8; j++) x0[0][c][j] = (__bf16)v[j];
    }
    bf16x8 h1[8][MLP_CT], h2[8][MLP_CT];
    int buf = 0;
    auto next = [&](const unsigned char *src, int bytes) {
        // the chunk copied last is complete, and the other buffer is free
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (bytes) copy_to_lds(src, wbuf[buf ^ 1], bytes);
    };
    next(packed + MLP_P2, MLP_CHUNK);
#pragma unroll
    for (int p = 0; p < 8; p++)
        mlp_step<1>(wbuf[buf] + 2 * p * MLP_FRAG, bias + 32 * p, x0, h1[p], lane);
    buf ^= 1;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        next(q < 3 ? packed + MLP_P2 + (q + 1) * MLP_CHUNK : packed + MLP_P3, MLP_CHUNK);
#pragma unroll
        for (int p = 0; p < 2; p++)
            mlp_step<8>(wbuf[buf] + 16 * p * MLP_FRAG, bias + MLP_H + 64 * q + 32 * p, h1,
                        h2[2 * q + p], lane);
        buf ^= 1;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        next(q < 3 ? packed + MLP_P3 + (q + 1) * MLP_CHUNK : packed + MLP_P4,
             q < 3 ? MLP_CHUNK : 8 * MLP_FRAG);
#pragma unroll
        for (int p = 0; p < 2; p++)
            mlp_step<8>(wbuf[buf] + 16 * p * MLP_FRAG, bias + 2 * MLP_H + 64 * q + 32 * p, h2,
                        h1[2 * q + p], lane);
        buf ^= 1;
    }
    next(nullptr, 0);
    f32x4 acc[MLP_CT];
    for (int c = 0; c < MLP_CT; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const bf16x8 w =
            *reinterpret_cast<const bf16x8 *>(wbuf[buf] + s * MLP_FRAG + lane * 16);
#pragma unroll
        for (int c = 0; c < MLP_CT; c++)
            acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, h1[s][c], acc[c], 0, 0, 0);
    }
    // feature 0 of every column lies in the first 16 lanes
    if (g == 0)
        for (int c = 0; c < MLP_CT; c++) {
            const int64_t row = row0 + 16 * c;
            float v = acc[c][0] + bias[3 * MLP_H];
            if (scale) v = v * y_std + y_mean;
            if (row < M) out[row] = v;
        }
}

/* ---- the training step's elementwise work -----------------------------------
 * A step on 1,024 rows holds 30 MFLOP of elementwise work on 140,000 weights;
 * as some 150 tensor operations it took 0.84 ms, all of it launches.  Each
 * kernel here does one kind of it for every layer at once. */
constexpr int MLP_MAX = 8;   // layers

struct ConvertList {
    const float *src[MLP_MAX + 1];
    uint16_t *dst[MLP_MAX + 1];
    int64_t end[MLP_MAX + 1];   // running element counts
    int32_t n;
};

__global__ __launch_bounds__(256) void convert_kernel(ConvertList L) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int t = 0;
    while (t < L.n && e >= L.end[t]) t++;
    if (t == L.n) return;
    const int64_t k = e - (t ? L.end[t - 1] : 0);
    L.dst[t][k] = f32_to_bf16_rne(L.src[t][k]);
}

struct SumList {
    const float *a[MLP_MAX];
    float *out[MLP_MAX];
    int64_t cols[MLP_MAX], block_end[MLP_MAX];
    int32_t n;
};

/* Column sums of row-major (rows x cols) arrays: 16 columns per block, 16
   threads per column over the block's rows, their partial sums in double.
   A thread's additions are a chain of loads: with SUM_ROWS rows per block
   and eight loads in flight the chain stays short whatever the batch, and
   blockIdx.y cuts larger batches, whose partial sums (part: one row of all
   columns per cut) column_sum_finish adds in order.  Bound by reading the
   rows once.  Backward pass of the default network, us, one chain over all
   rows against this: 1,024 rows 150 / 131, 65,536 rows 2669 / 978. */
constexpr int64_t SUM_ROWS = 1024;

__global__ __launch_bounds__(256) void column_sum_kernel(SumList L, int64_t rows,
                                                         double *__restrict__ part_out,
                                                         int64_t all_cols) {
    __shared__ double part[16][17];
    int t = 0;
    int64_t c0 = 0;
    while (t + 1 < L.n && (int64_t)blockIdx.x >= L.block_end[t]) c0 += L.cols[t++];
    const int64_t b0 = t ? L.block_end[t - 1] : 0;
    const int c = threadIdx.x & 15, r = threadIdx.x >> 4;
    const int64_t col = 16 * ((int64_t)blockIdx.x - b0) + c, n = L.cols[t];
    const int64_t first = (int64_t)blockIdx.y * SUM_ROWS;
    const int64_t end = first + SUM_ROWS < rows ? first + SUM_ROWS : rows;
    double s = 0.0;
    if (col < n) {
        const float *a = L.a[t] + col;
        int64_t k = first + r;
        for (; k + 16 * 7 < end; k += 16 * 8) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = a[(k + 16 * j) * n];
#pragma unroll
            for (int j = 0; j < 8; j++) s += (double)v[j];
        }
        for (; k < end; k += 16) s += (double)a[k * n];
    }
    part[r][c] = s;
    __syncthreads();
    if (r == 0 && col < n) {
        for (int k = 1; k < 16; k++) s += part[k][c];
        if (part_out)
            part_out[(int64_t)blockIdx.y * all_cols + c0 + col] = s;
        else
            L.out[t][col] = (float)s;
    }
}

__global__ __launch_bounds__(256) void column_sum_finish(SumList L,
                                                         const double *__restrict__ part,
                                                         int64_t all_cols, int32_t cuts) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= all_cols) return;
    int t = 0;
    int64_t c0 = 0;
    while (e >= c0 + L.cols[t]) c0 += L.cols[t++];
    double s = part[e];
    for (int32_t k = 1; k < cuts; k++) s += part[k * all_cols + e];
    L.out[t][e - c0] = (float)s;
}

struct AdamList {
    float *p[2 * MLP_MAX], *m[2 * MLP_MAX], *v[2 * MLP_MAX];
    const float *g[2 * MLP_MAX];
    int64_t end[2 * MLP_MAX];
    int32_t n;
};

/* One Adam update of every weight and bias; *t is the step count, this step
   included.  Bound by the 28 bytes per weight it moves: 140,000 weights in
   one launch against 94 tensor operations. */
__global__ __launch_bounds__(256) void adam_kernel(AdamList L, const float *__restrict__ t,
                                                   float lr, float beta1, float alpha1,
                                                   float beta2, float alpha2, float eps) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int k = 0;
    while (k < L.n && e >= L.end[k]) k++;
    if (k == L.n) return;
    const int64_t i = e - (k ? L.end[k - 1] : 0);
    const float bc1 = 1.f - powf(beta1, *t), bc2 = 1.f - powf(beta2, *t);
    const float g = L.g[k][i];
    const float m = fmaf(alpha1, g, L.m[k][i] * beta1);
    const float v = fmaf(alpha2 * g, g, L.v[k][i] * beta2);
    L.m[k][i] = m;
    L.v[k][i] = v;
    L.p[k][i] -= lr * (m / bc1) / (sqrtf(v / bc2) + eps);
}

/* workspace of xtm_gemm_bf16: allocated once per device on first need */
constexpr int kMaxDevices = 64;
std::mutex g_ws_mutex;
float *g_ws[kMaxDevices] = {};

/* Scratch of xtm_gemm_bf16_noalloc: one copy per GPU, held until the
   process ends.  In host code `scratch` names a host-side stand-in, not a
   device address: its device address is taken with hipGetSymbolAddress
   once per device, with that device current, and only that pointer
   (g_scratch[device]) is handed to the kernels.  Every call on a GPU
   shares the array; split partials are written before they are read, so
   nothing needs clearing between calls, and calls that overlap on one GPU
   race. */
__device__ __align__(256) float scratch[GEMM_WS_FLOATS];
float *g_scratch[kMaxDevices] = {};

}  // namespace

namespace {

int32_t gemm_with_workspace(const uint16_t *A, int64_t sam, int64_t sak, const uint16_t *B,
                            int64_t sbk, int64_t sbn, float *C, int64_t ldc, uint16_t *Cb,
                            const float *bias, int32_t relu, const float *mask, int64_t M,
                            int64_t N, int64_t K, hipStream_t stream) {
    int32_t st = gemm_check(A, B, C, ldc, M, N, K);
    if (st != XTM_OK || M == 0 || N == 0) return st;
    int64_t kc;
    const int64_t splits = gemm_splits(M, N, K, &kc);
    float *ws = nullptr;
    if (splits > 1) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
            return xt_report_error(XTM_ERR_HIP, "xtm_gemm_bf16: no current device");
        std::lock_guard<std::mutex> lock(g_ws_mutex);
        if (!g_ws[dev] && hipMalloc(&g_ws[dev], GEMM_WS_FLOATS * sizeof(float)) != hipSuccess) {
            g_ws[dev] = nullptr;
            return xt_report_error(XTM_ERR_HIP, "xtm_gemm_bf16: workspace allocation failed");
        }
        ws = g_ws[dev];
    }
    return gemm_launch(A, sam, sak, B, sbk, sbn, C, ldc, Cb, bias, relu, M, N, K, stream, ws,
                       GEMM_WS_FLOATS, splits, kc, mask);
}

int32_t launched(const char *what) {
    return hipGetLastError() == hipSuccess ? XTM_OK : xt_report_error(XTM_ERR_HIP, what);
}

/* FP32 -> BF16 of the weights of layers [first, n), into their place in the
   concatenation of all layers, and of `more` (n_more values) when not null */
int32_t convert_weights(int32_t first, int32_t n, const int64_t *sizes, const float *const *w,
                        uint16_t *wb, const float *more, uint16_t *more_b, int64_t n_more,
                        hipStream_t stream) {
    ConvertList L;
    L.n = 0;
    int64_t total = 0, off = 0;
    for (int32_t l = 0; l < n; l++) {
        const int64_t c = sizes[l] * sizes[l + 1];
        if (l >= first) {
            L.src[L.n] = w[l];
            L.dst[L.n] = wb + off;
            L.end[L.n++] = total += c;
        }
        off += c;
    }
    if (more) {
        L.src[L.n] = more;
        L.dst[L.n] = more_b;
        L.end[L.n++] = total += n_more;
    }
    hipLaunchKernelGGL(convert_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       stream, L);
    return launched("xtm_mlp_train: kernel launch failed");
}

bool train_args_ok(int32_t n, const int64_t *sizes, int64_t B) {
    if (n < 1 || n > MLP_MAX || !sizes || B < 1 || sizes[n] != 1) return false;
    int64_t total = 0;
    for (int32_t l = 0; l <= n; l++) {
        if (sizes[l] < 1 || sizes[l] > 1 << 20) return false;
        if (l) total += sizes[l - 1] * sizes[l];
    }
    return total < (int64_t)1 << 38 && B < (int64_t)1 << 31;
}

}  // namespace

extern "C" {

int32_t xtm_mlp_train_forward(int32_t n, const int64_t *sizes, const uint16_t *xb,
                              const float *const *w, const float *const *b, uint16_t *wb,
                              float *z, uint16_t *h, float *out, int64_t B, void *stream) {
    if (!train_args_ok(n, sizes, B) || !xb || !w || !b || !wb || !out || (n > 1 && (!z || !h)))
        return xt_report_error(XTM_ERR_ARG, "xtm_mlp_train_forward: invalid arguments");
    const hipStream_t s = (hipStream_t)stream;
    int32_t st = convert_weights(0, n, sizes, w, wb, nullptr, nullptr, 0, s);
    const uint16_t *in = xb;
    for (int32_t l = 0; l < n && st == XTM_OK; l++) {
        const int64_t K = sizes[l], N = sizes[l + 1];
        const bool last = l == n - 1;
        st = gemm_with_workspace(in, K, 1, wb, N, 1, last ? out : z, N, last ? nullptr : h, b[l],
                                 last ? 0 : 1, nullptr, B, N, K, s);
        in = h;
        wb += K * N;
        if (!last) {
            z += B * N;
            h += B * N;
        }
    }
    return st;
}

int32_t xtm_mlp_train_backward(int32_t n, const int64_t *sizes, const uint16_t *xb,
                               const uint16_t *h, const float *z, const float *const *w,
                               const float *dout, uint16_t *wb, float *dz, uint16_t *dzb,
                               float *const *gw, float *const *gb, int64_t B, void *stream) {
    if (!train_args_ok(n, sizes, B) || !xb || !w || !dout || !wb || !dzb || !gw || !gb ||
        (n > 1 && (!h || !z || !dz)))
        return xt_report_error(XTM_ERR_ARG, "xtm_mlp_train_backward: invalid arguments");
    const hipStream_t s = (hipStream_t)stream;
    // hidden layer l: z, dz (its first n - 1 layers) and h at off[l]; dzb also
    // holds the output layer's, at off[n - 1]
    int64_t off[MLP_MAX + 1] = {0}, woff[MLP_MAX + 1] = {0};
    for (int32_t l = 0; l < n; l++) {
        off[l + 1] = off[l] + B * sizes[l + 1];
        woff[l + 1] = woff[l] + sizes[l] * sizes[l + 1];
    }
    int32_t st = convert_weights(1, n, sizes, w, wb, dout, dzb + off[n - 1], B, s);
    SumList S;
    S.n = n;
    int64_t blocks = 0, cols = 0;
    for (int32_t l = n - 1; l >= 0 && st == XTM_OK; l--) {
        const int64_t K = sizes[l], N = sizes[l + 1];
        const uint16_t *d = dzb + off[l], *in = l ? h + off[l - 1] : xb;
        // h^T dz
        st = gemm_with_workspace(in, 1, K, d, N, 1, gw[l], N, nullptr, nullptr, 0, nullptr, K, N,
                                 B, s);
        if (l > 0 && st == XTM_OK)   // dz W^T where the layer below is active
            st = gemm_with_workspace(d, N, 1, wb + woff[l], 1, N, dz + off[l - 1], K,
                                     dzb + off[l - 1], nullptr, 0, z + off[l - 1], B, K, N, s);
    }
    if (st != XTM_OK) return st;
    for (int32_t l = 0; l < n; l++) {
        S.a[l] = l == n - 1 ? dout : dz + off[l];
        S.out[l] = gb[l];
        S.cols[l] = sizes[l + 1];
        S.block_end[l] = blocks += (sizes[l + 1] + 15) / 16;
        cols += sizes[l + 1];
    }
    // partial sums in dzb, which the products are done with: cuts x cols
    // doubles are at most a quarter of its B x cols BF16 values
    const int64_t cuts = (B + SUM_ROWS - 1) / SUM_ROWS;
    double *part = cuts > 1 ? reinterpret_cast<double *>(((uintptr_t)dzb + 7) & ~(uintptr_t)7)
                            : nullptr;
    hipLaunchKernelGGL(column_sum_kernel, dim3((unsigned)blocks, (unsigned)cuts), dim3(256), 0, s,
                       S, B, part, cols);
    if (part)
        hipLaunchKernelGGL(column_sum_finish, dim3((unsigned)((cols + 255) / 256)), dim3(256), 0,
                           s, S, (const double *)part, cols, (int32_t)cuts);
    return launched("xtm_mlp_train_backward: kernel launch failed");
}

int32_t xtm_adam_step(int32_t n, float *const *p, const float *const *g, float *const *m,
                      float *const *v, const int64_t *count, const float *t, float lr,
                      float beta1, float alpha1, float beta2, float alpha2, float eps,
                      void *stream) {
    if (n < 1 || n > 2 * MLP_MAX || !p || !g || !m || !v || !count || !t)
        return xt_report_error(XTM_ERR_ARG, "xtm_adam_step: invalid arguments");
    AdamList L;
    int64_t total = 0;
    L.n = n;
    for (int32_t k = 0; k < n; k++) {
        if (!p[k] || !g[k] || !m[k] || !v[k] || count[k] < 0)
            return xt_report_error(XTM_ERR_ARG, "xtm_adam_step: null array");
        L.p[k] = p[k];
        L.g[k] = g[k];
        L.m[k] = m[k];
        L.v[k] = v[k];
        L.end[k] = total += count[k];
    }
    if (total == 0) return XTM_OK;
    if (total > (int64_t)1 << 38)
        return xt_report_error(XTM_ERR_ARG, "xtm_adam_step: too many values");
    hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, L, t, lr, beta1, alpha1, beta2, alpha2, eps);
    return launched("xtm_adam_step: kernel launch failed");
}

int32_t xtm_gemm_bf16(const uint16_t *A, int64_t sam, int64_t sak, const uint16_t *B,
                      int64_t sbk, int64_t sbn, float *C, int64_t ldc, uint16_t *Cb,
                      const float *bias, int32_t relu, int64_t M, int64_t N, int64_t K,
                      void *stream) {
    return gemm_with_workspace(A, sam, sak, B, sbk, sbn, C, ldc, Cb, bias, relu, nullptr, M, N,
                               K, (hipStream_t)stream);
}

int32_t xtm_gemm_bf16_noalloc(const uint16_t *A, int64_t sam, int64_t sak, const uint16_t *B,
                              int64_t sbk, int64_t sbn, float *C, int64_t ldc, uint16_t *Cb,
                              const float *bias, int32_t relu, int64_t M, int64_t N, int64_t K,
                              void *stream) {
    int32_t st = gemm_check(A, B, C, ldc, M, N, K);
    if (st != XTM_OK || M == 0 || N == 0) return st;
    int64_t kc;
    const int64_t splits = gemm_splits(M, N, K, &kc);
    float *ws = nullptr;
    if (splits > 1) {
        if (splits * M * N > GEMM_WS_FLOATS)
            return xt_report_error(XTM_ERR_ARG, "xtm_gemm_bf16_noalloc: split partials exceed "
                                                "the scratch array (2^20 floats)");
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
            return xt_report_error(XTM_ERR_HIP, "xtm_gemm_bf16_noalloc: no current device");
        std::lock_guard<std::mutex> lock(g_ws_mutex);
        if (!g_scratch[dev]) {
            void *p = nullptr;
            const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !p)
                return xt_report_error(XTM_ERR_HIP, "xtm_gemm_bf16_noalloc: "
                                                    "hipGetSymbolAddress(scratch) failed");
            g_scratch[dev] = static_cast<float *>(p);
        }
        ws = g_scratch[dev];
    }
    return gemm_launch(A, sam, sak, B, sbk, sbn, C, ldc, Cb, bias, relu, M, N, K,
                       (hipStream_t)stream, ws, GEMM_WS_FLOATS, splits, kc);
}

int64_t xtm_gemm_bf16_scratch_floats(void) { return GEMM_WS_FLOATS; }

int64_t xtm_mlp_workspace_bytes(void) { return MLP_PACKED; }

int32_t xtm_mlp_forward(const float *x, const float *mean, const float *std,
                        const float *const *w, const float *const *b, void *workspace,
                        float *out, int64_t M, int32_t scale, float y_std, float y_mean,
                        void *stream) {
    if (!x || !w || !b || !workspace || !out || M < 0 || (mean && !std) ||
        ((uintptr_t)x & 15) || ((uintptr_t)workspace & 15))
        return xt_report_error(XTM_ERR_ARG, "xtm_mlp_forward: null or misaligned argument");
    MlpWeights W;
    for (int k = 0; k < 4; k++) {
        if (!w[k] || !b[k])
            return xt_report_error(XTM_ERR_ARG, "xtm_mlp_forward: null weights");
        W.w[k] = w[k];
        W.b[k] = b[k];
    }
    if (M == 0) return XTM_OK;
    const int64_t nb = (M + MLP_ROWS - 1) / MLP_ROWS;
    if (nb > 0x7fffffff) return xt_report_error(XTM_ERR_ARG, "xtm_mlp_forward: too many rows");
    unsigned char *packed = static_cast<unsigned char *>(workspace);
    const int threads = 280 * 64 + 3 * MLP_H + 1;
    hipLaunchKernelGGL(mlp_pack_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, W, packed);
    if (hipGetLastError() != hipSuccess)
        return xt_report_error(XTM_ERR_HIP, "xtm_mlp_forward: kernel launch failed");
    hipLaunchKernelGGL(mlp_forward_kernel, dim3((unsigned)nb), dim3(256), 0,
                       (hipStream_t)stream, x, mean, std, packed, out, M, scale, y_std, y_mean);
    return hipGetLastError() == hipSuccess
               ? XTM_OK
               : xt_report_error(XTM_ERR_HIP, "xtm_mlp_forward: kernel launch failed");
}

}  // extern "C"
