// Surrogate MLP kernels for CDNA4 (gfx950): BF16 x BF16 -> FP32 GEMMs on the
// matrix cores (v_mfma_f32_32x32x16_bf16) with fused bias / SiLU / SiLU'
// epilogues, batch gather, MSE loss gradient, bias column sums and Adam.
//
// GEMM tiling: a 256-thread block owns a 64 x 64 tile of C, each of its four
// wavefronts a 32 x 32 sub-tile accumulated in 16 FP32 registers per lane.
// The block's operands pass through LDS in chunks of TK k, both with k
// contiguous; the next chunk's loads (16 bytes per lane) are in flight under
// the current chunk's matrix instructions.  Per MFMA step a lane supplies 8
// consecutive k of row (l mod 32) of opA and the same 8 k of column (l mod 32)
// of opB, k = k0 + 8 (l / 32) + i; the product sums over all 16 k of the step
// whatever order the unit pairs them in, as long as A and B slots agree.  The
// 32 x 32 result sits in lane l, register r at column l mod 32, row
// 8 (r / 4) + 4 (l / 32) + r mod 4.  Out-of-range k, m, n read as 0.
// Loading fragments element by element from global memory bound the former
// kernel: 4096 rows through a 256 x 256 layer of five members took 150 us, now
// 18 us (the same steps in the same order: the same bits).
#include "device_common.hpp"
#include "mlp.hpp"

namespace sbe {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float dsilu(float z)
{
    const float s = 1.0f / (1.0f + __expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

constexpr int TK = 64;       // k per LDS chunk (128: 21 us where 64 takes 16, twice the LDS per block)
constexpr int TV = TK / 32;  // vectors per thread and operand of a chunk
constexpr int TS = TK + 8;   // LDS row stride: rows stay 16-byte aligned, banks spread

// Elements (r, k) of a chunk operand, r = r0 .. r0 + 63, k = k0 .. k0 + TK - 1, TV
// vectors of 8 per thread.  RC 0: P[r ld + k], a vector runs along k; RC 1:
// P[k ld + r], a vector runs along r.  vec: every vector inside the matrix is
// aligned and whole (decided on the host).
template <int RC>
__device__ __forceinline__ void chunk_load(const bf16 *P, long ld, int rows, int K, int r0, int k0, int vec, v8bf (&v)[TV])
{
    const bf16 zero = (bf16)0.0f;
#pragma unroll
    for (int i = 0; i < TV; i++) {
        const int e = threadIdx.x + 256 * i;
        const int r = r0 + (RC ? (e & 7) * 8 : e / (TK / 8)), k = k0 + (RC ? e >> 3 : (e % (TK / 8)) * 8);
        const bool in = r < rows && k < K;
#pragma unroll
        for (int j = 0; j < 8; j++) v[i][j] = zero;
        if (!in) continue;
        const bf16 *q = P + (RC ? (long)k * ld + r : (long)r * ld + k);
        if (vec) {
            v[i] = *reinterpret_cast<const v8bf *>(q);
        } else {
            const int left = RC ? rows - r : K - k;
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (j < left) v[i][j] = q[j];
        }
    }
}

// the same vectors into the LDS chunk [r][k]
template <int RC>
__device__ __forceinline__ void chunk_store(bf16 *L, const v8bf (&v)[TV])
{
#pragma unroll
    for (int i = 0; i < TV; i++) {
        const int e = threadIdx.x + 256 * i;
        if (RC) {
            const int r = (e & 7) * 8, k = e >> 3;
#pragma unroll
            for (int j = 0; j < 8; j++) L[(r + j) * TS + k] = v[i][j];
        } else {
            *reinterpret_cast<v8bf *>(L + e / (TK / 8) * TS + e % (TK / 8) * 8) = v[i];
        }
    }
}

template <int TA, int TB>
__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs g)
{
    __shared__ __align__(16) bf16 As[64 * TS], Bs[64 * TS];
    const int e = blockIdx.z;
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int mb = blockIdx.y * 64, nb = blockIdx.x * 64;
    const int m0 = mb + (w >> 1) * 32, n0 = nb + (w & 1) * 32;
    const bf16 *A = g.A + e * g.strideA, *B = g.B + e * g.strideB;
    const int col = n0 + (l & 31);
    const bf16 *fa = As + ((w >> 1) * 32 + (l & 31)) * TS + 8 * (l >> 5);
    const bf16 *fb = Bs + ((w & 1) * 32 + (l & 31)) * TS + 8 * (l >> 5);
    const bool sums = g.rowsum && blockIdx.x == 0;
    float rs = 0.0f;
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    v8bf va[TV], vb[TV];
    chunk_load<TA>(A, g.lda, g.M, g.K, mb, 0, g.vecA, va);
    chunk_load<!TB>(B, g.ldb, g.N, g.K, nb, 0, g.vecB, vb);
    for (int k0 = 0; k0 < g.K; k0 += TK) {
        if (k0) __syncthreads();
        chunk_store<TA>(As, va);
        chunk_store<!TB>(Bs, vb);
        __syncthreads();
        if (k0 + TK < g.K) {
            chunk_load<TA>(A, g.lda, g.M, g.K, mb, k0 + TK, g.vecA, va);
            chunk_load<!TB>(B, g.ldb, g.N, g.K, nb, k0 + TK, g.vecB, vb);
        }
#pragma unroll
        for (int s = 0; s < TK / 16; s++)
            if (k0 + 16 * s < g.K)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const v8bf *>(fa + 16 * s),
                                                              *reinterpret_cast<const v8bf *>(fb + 16 * s), acc, 0, 0, 0);
        if (sums) {
            // four threads per row of opA, a quarter of the chunk each
            const bf16 *q = As + (threadIdx.x >> 2) * TS + (threadIdx.x & 3) * (TK / 4);
#pragma unroll
            for (int j = 0; j < TK / 4; j++) rs += (float)q[j];
        }
    }
    if (sums) {
        rs += __shfl_xor(rs, 1);
        rs += __shfl_xor(rs, 2);
        const int m = mb + (threadIdx.x >> 2);
        if ((threadIdx.x & 3) == 0 && m < g.M) g.rowsum[e * g.strideRow + m] = rs;
    }
    const int n = col;
    if (n >= g.N) return;
    const float bias = (g.mode == 1 || g.mode == 2) ? g.bias[e * g.strideBias + n] : 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int m = m0 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3);
        if (m >= g.M) continue;
        const float v = acc[r];
        if (g.mode == 0) {
            g.C[e * g.strideC + (long)m * g.ldc + n] = v;
        } else if (g.mode == 1) {
            const float z = v + bias;
            g.C[e * g.strideC + (long)m * g.ldc + n] = z;
            g.H[e * g.strideH + (long)m * g.ldh + n] = (bf16)silu(z);
        } else if (g.mode == 2) {
            g.C[e * g.strideC + (long)m * g.ldc + n] = v + bias;
        } else {
            const float z = g.Zin[e * g.strideZ + (long)m * g.ldz + n];
            g.H[e * g.strideH + (long)m * g.ldh + n] = (bf16)(v * dsilu(z));
        }
    }
}

hipError_t launch_gemm(const GemmArgs &g0, int ta, int tb, int members, hipStream_t s)
{
    // 16-byte loads: the vectors of 8 along an operand's contiguous index are
    // whole (its extent and every row and member start are multiples of 8)
    GemmArgs g = g0;
    auto whole = [](const bf16 *p, long extent, long ld, long stride) {
        return ((reinterpret_cast<unsigned long long>(p) & 15) | ((extent | ld | stride) & 7)) == 0;
    };
    g.vecA = whole(g.A, ta ? g.M : g.K, g.lda, members > 1 ? g.strideA : 0);
    g.vecB = whole(g.B, tb ? g.K : g.N, g.ldb, members > 1 ? g.strideB : 0);
    dim3 grid((unsigned)((g.N + 63) / 64), (unsigned)((g.M + 63) / 64), (unsigned)members), blk(256);
    switch (ta * 2 + tb) {
    case 0: hipLaunchKernelGGL((gemm_kernel<0, 0>), grid, blk, 0, s, g); break;
    case 1: hipLaunchKernelGGL((gemm_kernel<0, 1>), grid, blk, 0, s, g); break;
    case 2: hipLaunchKernelGGL((gemm_kernel<1, 0>), grid, blk, 0, s, g); break;
    default: hipLaunchKernelGGL((gemm_kernel<1, 1>), grid, blk, 0, s, g); break;
    }
    return hipGetLastError();
}

// grid (batch, members), block 64
__global__ void gather_kernel(const float *Xall, const float *Tall, int din, int dout, const int *perm, long n_perm,
                              const int *counter, int spe, int batch, int cap, bf16 *X, float *T)
{
    const int b = blockIdx.x, e = blockIdx.y;
    const long idx = perm ? perm[e * n_perm + (long)(*counter % spe) * batch + b] : b;
    const long row = (long)e * cap + b;
    for (int i = threadIdx.x; i < din; i += 64) X[row * din + i] = (bf16)Xall[idx * din + i];
    for (int i = threadIdx.x; i < dout; i += 64) T[row * dout + i] = Tall[idx * dout + i];
}

hipError_t launch_gather(const float *Xall, const float *Tall, int din, int dout, const int *perm, long n_perm,
                         const int *counter, int spe, int batch, int cap, int members, bf16 *X, float *T,
                         hipStream_t s)
{
    hipLaunchKernelGGL(gather_kernel, dim3((unsigned)batch, (unsigned)members), dim3(64), 0, s, Xall, Tall, din, dout,
                       perm, n_perm, counter, spe, batch, cap, X, T);
    return hipGetLastError();
}

// one block per member, fixed summation order
constexpr int LOSS_T = 1024;
__global__ __launch_bounds__(LOSS_T) void loss_grad_kernel(const float *Y, const float *T, int batch, int cap, int dout,
                                                           bf16 *dY, float *loss, int loss_stride, const int *counter)
{
    __shared__ float red[LOSS_T / 64];
    const int e = blockIdx.x;
    const long cnt = (long)batch * dout, off = (long)e * cap * dout;
    const float sc = 2.0f / (float)cnt;
    float acc = 0.0f;
#pragma unroll 4
    for (long i = threadIdx.x; i < cnt; i += LOSS_T) {
        const float d = Y[off + i] - T[off + i];
        dY[off + i] = (bf16)(sc * d);
        acc += d * d;
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) acc += __shfl_xor(acc, m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0 && loss) {
        float t = 0.0f;
        for (int w = 0; w < LOSS_T / 64; w++) t += red[w];
        loss[(long)e * loss_stride + (counter ? *counter : 0)] = t / (float)cnt;
    }
}

hipError_t launch_loss_grad(const float *Y, const float *T, int batch, int cap, int dout, int members, bf16 *dY,
                            float *loss, int loss_stride, const int *counter, hipStream_t s)
{
    hipLaunchKernelGGL(loss_grad_kernel, dim3((unsigned)members), dim3(LOSS_T), 0, s, Y, T, batch, cap, dout, dY, loss,
                       loss_stride, counter);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void adam_kernel(float *p, bf16 *pb, float *m, float *v, const float *g, long count,
                                                   float lr, float b1, float b2, float eps, long total,
                                                   const int *counter)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const int t = *counter + 1;
    const float frac = fminf((float)(t - 1) / (float)total, 1.0f);
    const float lr_t = lr * 0.5f * (1.0f + cospif(frac));
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / (1.0f - powf(b1, (float)t)), vh = vi / (1.0f - powf(b2, (float)t));
    const float pi = p[i] - lr_t * mh / (sqrtf(vh) + eps);
    p[i] = pi;
    pb[i] = (bf16)pi;
}

hipError_t launch_adam(float *p, bf16 *pb, float *m, float *v, const float *g, long count, float lr, float b1,
                       float b2, float eps, long total, const int *counter, hipStream_t s)
{
    hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, p, pb, m, v, g, count, lr,
                       b1, b2, eps, total, counter);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void to_bf16_kernel(const float *p, bf16 *pb, long count)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < count) pb[i] = (bf16)p[i];
}

hipError_t launch_to_bf16(const float *p, bf16 *pb, long count, hipStream_t s)
{
    hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, p, pb, count);
    return hipGetLastError();
}

__global__ void increment_kernel(int *counter) { *counter += 1; }

hipError_t launch_increment(int *counter, hipStream_t s)
{
    hipLaunchKernelGGL(increment_kernel, dim3(1), dim3(1), 0, s, counter);
    return hipGetLastError();
}

}  // namespace sbe
