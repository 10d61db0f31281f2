// Observer kernels.
//
// Current expectation value at an output time (default k-space region, w_k = 1):
//   j_d = (1/N_k) sum_k Re sum_ab [ i D_d(k)_ab T_ba - dH0/dk_d(k)_ab rho_ba ],
//   T = H0(k) rho - rho H0(k),
// with H0, D_d, dH0/dk_d evaluated at k + A (code/src/ObserverCPU.cpp:188-210,
// normalisation :293-308).  The operators come from a partial phase sum whose
// last axis is contracted here.  Two passes, fixed summation order
// (deterministic).
#include "device_common.hpp"
#include "kernels.hpp"
#include "observer_device.hpp"
#include "stage_device.hpp"

namespace sbe {

// The per-k current for 16 bands: KB consecutive k-points per wavefront, in the
// accumulator layout.  Lane entry (a, b) of a k-point's matrices holds T_ba and
// rho_ba, and the sum over (a, b) goes before the one over the last axis' cells r,
//   j_d = Re sum_r tw_r sum_ab [ i D_d(r)_ab T_ba - dH_d(r)_ab rho_ba ],
// so a phase-sum entry is loaded once for all k-points of its row and no operator
// is formed.  One k-point per wavefront read (1 + 2 dim) n n W_L entries from L2 and
// as many twiddles per k-point: 24^3 k 375 -> 125 us (KB 2; 3: 114, 4: 152 and two
// waves per SIMD).  Up to 8 bands keep a wavefront per k-point: the same with 8 or
// 2 k-points per wavefront took 49 us instead of 61 on 150 x 150 k, but 43 and 23
// instead of 11 on 15 x 15, the latency of one wavefront.
constexpr int JK_KB = 2;

__device__ __forceinline__ void jk_rows_body(const ObsArgs &a, const long blk)
{
    constexpr int N = 16, KB = JK_KB, EK = N * N / 64;
    const int n = a.n, nn = n * n, M = (1 + 2 * a.dim) * nn, WL = a.ph.WL;
    const int k0 = __builtin_amdgcn_readfirstlane((int)blk) * KB;
    int ent[EK];
    bool own[EK];
#pragma unroll
    for (int u = 0; u < EK; u++) {
        const int idx = threadIdx.x + 64 * u;
        own[u] = idx / N < n && idx % N < n;
        ent[u] = own[u] ? idx / N * n + idx % N : 0;
    }
    cd H[KB * EK];  // H0(k)
    if (!phase_rows<N, KB>(H, a.ph, a.nk, n, M, 0, k0)) {
#pragma unroll
        for (int kk = 0; kk < KB; kk++)
#pragma unroll
            for (int u = 0; u < EK; u++)
                H[kk * EK + u] = own[u] && k0 + kk < a.nk ? phase_last(a.ph, k0 + kk, M, ent[u]) : mk(0, 0);
    }
    cd R[KB * EK], T[KB * EK];
#pragma unroll
    for (int kk = 0; kk < KB; kk++)
#pragma unroll
        for (int u = 0; u < EK; u++) {
            const bool in = own[u] && k0 + kk < a.nk;
            const double2 v = reinterpret_cast<const double2 *>(a.x)[in ? 8 + (k0 + kk) * (long)a.P + ent[u] : 8];
            R[kk * EK + u] = in ? mk(v.x, v.y) : mk(0, 0);
        }
    // T = H0 rho - rho H0, then T and rho transposed
    __shared__ cd B0[Frag16::MS], B1[Frag16::MS];
    const AccPos pos = acc_pos<Frag16>();
#pragma unroll
    for (int kk = 0; kk < KB; kk++) {
        cd *h = H + kk * EK, *r = R + kk * EK, x[4], y[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            B0[pos.nat + Frag16::nat_step(j)] = h[j];
            B1[pos.nat + Frag16::nat_step(j)] = r[j];
        }
        wsync();
        CAcc t;
        cacc_zero(t);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            x[j] = B0[pos.tr + 4 * j];
            y[j] = B1[pos.tr + 4 * j];
        }
        mfma_cmul(x, r, t);
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = mk(-y[j].x, -y[j].y);
        mfma_cmul(x, h, t);
        wsync();
        acc_put<Frag16>(B0, pos, t);
        wsync();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            T[kk * EK + j] = B0[pos.tr + 4 * j];
            r[j] = y[j];
        }
        wsync();
    }
    int rest[KB];
    unsigned tp[KB];
    phase_map<KB>(a.ph, a.nk, k0, rest, tp);
    double jl[KB][3];
#pragma unroll
    for (int kk = 0; kk < KB; kk++)
#pragma unroll
        for (int d = 0; d < 3; d++) jl[kk][d] = 0;
    unsigned todo = (1u << KB) - 1;
    while (todo) {
        int row;
        const unsigned mine = next_row_group<KB>(todo, rest, row);
        const double2 *yr = reinterpret_cast<const double2 *>(a.ph.Y) + (long)row * M;
#pragma unroll 2
        for (int q = 0; q < WL; q++) {
            sd2 tw[KB];
#pragma unroll
            for (int kk = 0; kk < KB; kk++) tw[kk] = load_const<sd2>(reinterpret_cast<const sd2 *>(a.ph.twL) + tp[kk], q);
#pragma unroll
            for (int d = 0; d < 3; d++)
                if (d < a.dim) {
                    double2 yd[EK], yh[EK];
#pragma unroll
                    for (int u = 0; u < EK; u++) {
                        yd[u] = yr[(long)q * M + (1 + d) * nn + ent[u]];
                        yh[u] = yr[(long)q * M + (1 + a.dim + d) * nn + ent[u]];
                    }
#pragma unroll
                    for (int kk = 0; kk < KB; kk++)
                        if ((mine >> kk) & 1) {
                            asm volatile("");  // a branch over the products, not selects behind them
                            cd z = mk(0, 0), w = mk(0, 0);
#pragma unroll
                            for (int u = 0; u < EK; u++) {
                                z = cfma(mk(yd[u].x, yd[u].y), T[kk * EK + u], z);
                                w = cfma(mk(yh[u].x, yh[u].y), R[kk * EK + u], w);
                            }
                            // Re tw (i z - w)
                            jl[kk][d] += tw[kk].x * (-z.y - w.x) - tw[kk].y * (z.x - w.y);
                        }
                }
        }
    }
#pragma unroll
    for (int kk = 0; kk < KB; kk++)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double v = seg_sum<64>(jl[kk][d]);
            if (threadIdx.x == 0 && k0 + kk < a.nk) a.partial[(long)a.pstride * (k0 + kk) + d] = v;
        }
}

__global__ __launch_bounds__(64) void jk_rows_kernel(ObsArgs a)
{
    jk_rows_body(a, xcd_block(blockIdx.x, gridDim.x));
}

__global__ __launch_bounds__(64) void jk_kernel(ObsArgs a) { jk_body(a, blockIdx.x); }

// entry j owns blocks [block0[j], block0[j] + ceil(nk_j / observe_block_k))
__global__ __launch_bounds__(64) void jk_rows_batched_kernel(const ObsArgs *args, const long *block0, int m)
{
    const long gb = xcd_block(blockIdx.x, gridDim.x);
    const int j = find_entry_wave(block0, m, gb);
    jk_rows_body(args[j], gb - block0[j]);
}

__global__ __launch_bounds__(64) void jk_batched_kernel(const ObsArgs *args, const long *block0, int m)
{
    const long gb = blockIdx.x;
    const int j = find_entry_wave(block0, m, gb);
    const ObsArgs a = args[j];
    jk_body(a, gb - block0[j]);
}

int observe_block_k(int n) { return n > 8 ? JK_KB : 1; }

static hipError_t launch_jk(const ObsArgs &a, hipStream_t s)
{
    const int kb = observe_block_k(a.n);
    const dim3 grid((unsigned)((a.nk + kb - 1) / kb)), blk(64);
    if (a.n > 8) hipLaunchKernelGGL(jk_rows_kernel, grid, blk, 0, s, a);
    else hipLaunchKernelGGL(jk_kernel, grid, blk, 0, s, a);
    return hipGetLastError();
}

__device__ __forceinline__ void jreduce_body(const double *partial, long nk, double *j_out, int pstride)
{
    __shared__ double s[3][256];
    double acc[3] = {0, 0, 0};
    for (long k = threadIdx.x; k < nk; k += 256)
        for (int d = 0; d < 3; d++) acc[d] += partial[(long)pstride * k + d];
    for (int d = 0; d < 3; d++) s[d][threadIdx.x] = acc[d];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int d = 0; d < 3; d++) s[d][threadIdx.x] += s[d][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 3) j_out[threadIdx.x] = s[threadIdx.x][0] / (double)nk;
}

__global__ __launch_bounds__(256) void jreduce_kernel(const double *partial, long nk, double *j_out, int pstride)
{
    jreduce_body(partial, nk, j_out, pstride);
}

__global__ __launch_bounds__(256) void jreduce_batched_kernel(const ObsArgs *args)
{
    const ObsArgs &a = args[blockIdx.x];
    jreduce_body(a.partial, a.nk, a.j_out, a.pstride);
}

hipError_t launch_observe_j(const ObsArgs &a, hipStream_t s)
{
    if (a.n > OBS_MAXN) return hipErrorInvalidValue;
    hipError_t e = launch_jk(a, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(jreduce_kernel, dim3(1), dim3(256), 0, s, a.partial, a.nk, a.j_out, a.pstride);
    return hipGetLastError();
}

hipError_t launch_observe_jk(const ObsArgs &a, hipStream_t s)
{
    if (a.n > OBS_MAXN || a.pstride < 3) return hipErrorInvalidValue;
    return launch_jk(a, s);
}

// ---- k-space regions ------------------------------------------------------
// Weight of k-point k in region r (ObserverCPU::calcWeight,
// code/src/ObserverCPU.cpp:137-147; the position is getFFTfracShift,
// code/src/WhFourierTransform.cpp:163-174): p = grid(k)/Nk + shift + frac(A)
// (+ frac(-A) in the moving frame) - centre, w = prod_d exp(-c_d^2 inv),
// c_d = p_d - round(p_d).
__device__ __forceinline__ double region_w(const RegionArgs &a, const RegionDev &r, long k, const double off[3],
                                           const double negA[3])
{
    const KOrder ko{{a.ko.Nf[0], a.ko.Nf[1], a.ko.Nf[2]}, {a.ko.Nrep[0], a.ko.Nrep[1], a.ko.Nrep[2]}};
    int g[3];
    k_to_grid(ko, k, g[0], g[1], g[2]);
    double w = 1;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double pos = (double)g[d] / a.Nk[d] + off[d];
        if (r.moving) pos += negA[d];
        pos -= r.k[d];
        const double c = pos - rint(pos);
        w *= exp(-c * c * r.inv_sigma2);
    }
    return w;
}

// frac(shift + A) and frac(-A) from the state's special slots (the reference
// converts k_global_shift + A to fractional coordinates in one step,
// code/src/ObserverCPU.cpp:168-171)
__device__ __forceinline__ void region_offsets(const RegionArgs &a, double off[3], double negA[3])
{
    double A[3];
    for (int d = 0; d < 3; d++) A[d] = a.x[2 * d];
    for (int d = 0; d < 3; d++) {
        const double *ad = a.lat + 3 * d;
        off[d] = a.shift[d] + (A[0] * ad[0] + A[1] * ad[1] + A[2] * ad[2]) / (2 * M_PI);
        negA[d] = (-A[0] * ad[0] + -A[1] * ad[1] + -A[2] * ad[2]) / (2 * M_PI);
    }
}

// grid (R, chunks, ceil(Qtot / 64)), 256 threads: wavefront w of the block
// takes every fourth group of 64 k-points of the chunk; lane l evaluates the
// weight of k-point l of the group, then every lane accumulates its quantity
// q over the 64 k-points with the weights broadcast lane by lane, eight
// k-points' values in flight.  Block 0 of region 0 also keeps min / max over k
// of the smeared occupations.  With one load per trip and 4096 k-points per
// chunk a record of 24^3 k, 16 bands and two regions took 400 us, now 25 us with the density matrix and 9 without.
__device__ __forceinline__ double lane_value(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__global__ __launch_bounds__(256) void region_sum_kernel(RegionArgs a)
{
    constexpr int U = 8;
    const int r = blockIdx.x, ch = blockIdx.y;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int Qtot = a.Q + 1 + (a.density ? 2 * a.n * a.n : 0);
    const int q = blockIdx.z * 64 + lane;
    const RegionDev rg = a.reg[r];
    double off[3], negA[3];
    region_offsets(a, off, negA);
    const long k0 = (long)ch * a.chunk, k1 = min(a.nk, k0 + a.chunk);
    const bool mm = (r == 0 && blockIdx.z == 0 && q >= 3 && q < 3 + a.n);
    // the quantity of this lane over k: a row of X, 1, or an entry of rho
    const bool one = q == a.Q || q >= Qtot;
    const double *src = one || q < a.Q ? a.X + (one ? 0 : q) : a.x + 16 + (q - a.Q - 1);
    const long step = one || q < a.Q ? a.Q : 2 * (long)a.P;
    double acc = 0, mn = INFINITY, mx = -INFINITY;
    auto add = [&](double w, double v) {
        if (one) v = 1.0;
        acc += w * v;
        if (mm) {
            mn = fmin(mn, v);
            mx = fmax(mx, v);
        }
    };
    for (long g = k0 + 64 * wv; g < k1; g += 256) {
        const long kl = g + lane;
        const double wl = kl < k1 ? region_w(a, rg, kl, off, negA) : 0.0;
        const int cnt = (int)min((long)64, k1 - g);
        const double *p = src + g * step;
        int m = 0;
        for (; m + U <= cnt; m += U) {
            double v[U];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = p[(m + u) * step];
#pragma unroll
            for (int u = 0; u < U; u++) add(lane_value(wl, m + u), v[u]);
        }
        for (; m < cnt; m++) add(lane_value(wl, m), p[m * step]);
    }
    __shared__ double sh[3][256];
    sh[0][threadIdx.x] = acc;
    sh[1][threadIdx.x] = mn;
    sh[2][threadIdx.x] = mx;
    __syncthreads();
    if (wv == 0 && q < Qtot) {
        double t = sh[0][lane], lo = sh[1][lane], hi = sh[2][lane];
        for (int w2 = 1; w2 < 4; w2++) {
            t += sh[0][lane + 64 * w2];
            lo = fmin(lo, sh[1][lane + 64 * w2]);
            hi = fmax(hi, sh[2][lane + 64 * w2]);
        }
        a.part[((long)r * a.chunks + ch) * Qtot + q] = t;
        if (mm) {
            a.pmin[(long)ch * a.n + (q - 3)] = lo;
            a.pmax[(long)ch * a.n + (q - 3)] = hi;
        }
    }
}

// grid (R, ceil(Qtot / 64)), 256 threads: four wavefronts sum every fourth chunk of
// the block's quantities and of the weights, then divide by the weight sum
// (normalizeExpectationValues, code/src/ObserverCPU.cpp:293-308) and write the
// record; block 0 also writes A and the min / max over k
__global__ __launch_bounds__(256) void region_final_kernel(RegionArgs a)
{
    const int r = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int Qtot = a.Q + 1 + (a.density ? 2 * a.n * a.n : 0);
    const int q = blockIdx.y * 64 + lane, qs = q < Qtot ? q : a.Q;
    const double *part = a.part + (long)r * a.chunks * Qtot;
    double t = 0, ws = 0;
#pragma unroll 4
    for (int c = wv; c < a.chunks; c += 4) {
        t += part[(long)c * Qtot + qs];
        ws += part[(long)c * Qtot + a.Q];
    }
    __shared__ double sh[2][256];
    sh[0][threadIdx.x] = t;
    sh[1][threadIdx.x] = ws;
    __syncthreads();
    if (wv == 0 && q < Qtot) {
        for (int w2 = 1; w2 < 4; w2++) {
            t += sh[0][lane + 64 * w2];
            ws += sh[1][lane + 64 * w2];
        }
        a.rec[3 + (long)r * a.rstride + q] = (q == a.Q) ? t : t / ws;
    }
    if (r == 0 && blockIdx.y == 0) {
        if (threadIdx.x < 3) a.rec[threadIdx.x] = a.x[2 * threadIdx.x];
        double *mnmx = a.rec + 3 + (long)a.R * a.rstride;
        // min by the first wavefront, max by the second: lane = band + 16 x (every fourth chunk)
        const int b = lane & 15, c0 = lane >> 4;
        if (wv < 2 && b < a.n) {
            double v = wv ? -INFINITY : INFINITY;
            for (int c = c0; c < a.chunks; c += 4) {
                const double p = (wv ? a.pmax : a.pmin)[(long)c * a.n + b];
                v = wv ? fmax(v, p) : fmin(v, p);
            }
            for (int m = 16; m < 64; m <<= 1) {
                const double o = __shfl_xor(v, m);
                v = wv ? fmax(v, o) : fmin(v, o);
            }
            if (c0 == 0) mnmx[wv * a.n + b] = v;
        }
    }
}

hipError_t launch_region_sums(const RegionArgs &a, hipStream_t s)
{
    const int Qtot = a.Q + 1 + (a.density ? 2 * a.n * a.n : 0);
    if (a.R < 1 || a.chunks < 1 || a.nk < 1 || a.chunk * a.chunks < a.nk || a.rstride < Qtot)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(region_sum_kernel, dim3((unsigned)a.R, (unsigned)a.chunks, (unsigned)((Qtot + 63) / 64)),
                       dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(region_final_kernel, dim3((unsigned)a.R, (unsigned)((Qtot + 63) / 64)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_observe_j_batched(int n, const ObsArgs *d_args, const long *d_block0, int m, long blocks,
                                    hipStream_t s)
{
    if (m <= 0 || blocks <= 0) return hipSuccess;
    const dim3 grid((unsigned)blocks), blk(64);
    if (n > 8) hipLaunchKernelGGL(jk_rows_batched_kernel, grid, blk, 0, s, d_args, d_block0, m);
    else hipLaunchKernelGGL(jk_batched_kernel, grid, blk, 0, s, d_args, d_block0, m);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(jreduce_batched_kernel, dim3((unsigned)m), dim3(256), 0, s, d_args);
    return hipGetLastError();
}

}  // namespace sbe
