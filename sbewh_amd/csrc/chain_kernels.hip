// 1-D chains of two bands: four lanes per k-point, one matrix entry each,
// everything of a k-point in registers.
//
// Such an instance is small (256 k-points of 2 bands are 32 KB), and its time is
// launches and chains of dependent latencies, not arithmetic.  Lane (a, b) of a
// k-point's quad holds entry ab of every matrix; the other entries come through
// quad permutes.  A quad forms its own phase factor (dim = 1 has no contraction
// to share) and sums H0 and the position operator over the R cells, whose
// entries its lanes keep in registers; 2 x 2 is diagonalised by one rotation, with
// nothing to warm-start; x and the stage derivatives stay in registers.  So a
// whole Dormand-Prince attempt is one launch without a memory trip between its
// stages, its error norm included, and an output time (current and fresh
// derivative) is another.  Measured on 256 k, the general path first: an attempt
// 49 us in two launches, now 11 us in one; an output time 24 us in six launches,
// now 6 us; four right-hand sides 33.7 -> 14-17 us; a whole pulse with 1024 outputs
// 144-164 -> 55-71 ms, half of it the host's round trips.  (With a lane per k-point
// and its cells read through scalar loads an attempt takes 18 us.)
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace sbe {

// entry (S0, S1, S2, S3)[lane of the quad] of the quad's four values
template <int S0, int S1, int S2, int S3>
__device__ __forceinline__ double quad(double v)
{
    constexpr int CTRL = S0 | S1 << 2 | S2 << 4 | S3 << 6;
    const long long b = __double_as_longlong(v);
    const int lo = dpp_i<CTRL>((int)(b & 0xffffffffll)), hi = dpp_i<CTRL>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <int S0, int S1, int S2, int S3>
__device__ __forceinline__ cd quad(cd v)
{
    return mk(quad<S0, S1, S2, S3>(v.x), quad<S0, S1, S2, S3>(v.y));
}
// lane LANE's value in all four lanes
template <int LANE>
__device__ __forceinline__ cd quad_of(cd v)
{
    return quad<LANE, LANE, LANE, LANE>(v);
}
__device__ __forceinline__ cd quad_sum(cd v)
{
    v = cadd(v, quad<1, 0, 3, 2>(v));
    return cadd(v, quad<2, 3, 0, 1>(v));
}

// the wavefront's place in the chain; lanes beyond the last k-point repeat it
// (the quad permutes need every lane) and store nothing
struct Site {
    long k, at;  // k-point, state index of the lane's entry
    int e;       // entry: 2 a + b
    bool ok;
    double frac;  // i / Nk
};
__device__ __forceinline__ Site site(const ChainArgs &c)
{
    Site s;
    const long k = (long)blockIdx.x * 16 + (threadIdx.x >> 2);
    s.ok = k < c.nk;
    s.k = s.ok ? k : c.nk - 1;
    s.e = threadIdx.x & 3;
    s.at = 8 + s.k * c.P + s.e;
    s.frac = (double)(reinterpret_cast<const int2 *>(c.kphase)[s.k].y / c.W) / c.Nk;
    return s;
}

// The lane's entry of an operator in the cells -MW .. MW (zero outside the R box),
// or, MW = 0, read from memory for any box.
template <int MW>
struct Cells {
    cd v[2 * MW + 1];
};
template <int MW>
__device__ __forceinline__ void load_cells(const ChainArgs &c, const double *op, int e, Cells<MW> &o)
{
    if constexpr (MW > 0) {
#pragma unroll
        for (int m = -MW; m <= MW; m++) {
            const int r = m - c.rmin;
            const bool in = r >= 0 && r < c.W;
            const double2 t = reinterpret_cast<const double2 *>(op)[(in ? r : -c.rmin) * 4 + e];
            o.v[m + MW] = in ? mk(t.x, t.y) : mk(0, 0);
        }
    }
}

// (k + A) a_0 / 2 pi without k's own part: the phase offset of the vector potential A
__device__ __forceinline__ double phase_offset(const ChainArgs &c, double A)
{
    return ((c.kshift_au[0] + A) * c.a0[0] + c.kshift_au[1] * c.a0[1] + c.kshift_au[2] * c.a0[2]) / (2 * M_PI);
}

// The powers z^m0 .. z^(m0 + 3) of a quad's phase factor z, for the highest m0 first and
// then four lower at a time: each by its own argument, a lane one of them, rounded as the
// twiddles of the general path are,
struct DirectPowers {
    double arg;
    __device__ __forceinline__ void next(int m0, cd (&p)[4]) const
    {
        double s, co;
        sincospi(2 * (arg * (double)(m0 + (int)(threadIdx.x & 3))), &s, &co);
        const cd v = mk(co, s);
        p[0] = quad_of<0>(v);
        p[1] = quad_of<1>(v);
        p[2] = quad_of<2>(v);
        p[3] = quad_of<3>(v);
    }
    __device__ __forceinline__ void first(int m0, cd (&p)[4]) const { next(m0, p); }
};
// or, for an attempt's six stages, whose factors the lanes share out, as products
// (z^-4 is z^4's conjugate).
struct FactorPowers {
    cd z, low[4];
    __device__ __forceinline__ void first(int m0, cd (&p)[4])
    {
        low[0] = z;
        low[1] = cmul(z, z);
        low[2] = cmul(z, low[1]);
        low[3] = cmul(low[1], low[1]);
#pragma unroll
        for (int j = 0; j < 4; j++) p[j] = low[j];
        for (int m = 1; m < m0; m += 4)
#pragma unroll
            for (int j = 0; j < 4; j++) p[j] = cmul(p[j], low[3]);
    }
    __device__ __forceinline__ void next(int m0, cd (&p)[4]) const
    {
#pragma unroll
        for (int j = 0; j < 4; j++) p[j] = m0 == 1 ? low[j] : cmul(p[j], cconj(low[3]));
    }
};
// e^{i 2 pi (frac + off)}; what the sum's rounding loses (Knuth's two-sum) is put back to
// first order, since the powers multiply it
__device__ __forceinline__ cd phase_factor(const ChainArgs &c, double frac, double A)
{
    const double off = phase_offset(c, A), arg = frac + off, t = arg - frac;
    const double lost = 2 * M_PI * ((frac - (arg - t)) + (off - t));
    double s, co;
    sincospi(2 * arg, &s, &co);
    return mk(fma(-lost, s, co), fma(lost, co, s));
}

// sum_m z^m O_o(m), cells +m and -m sharing one power, from the far cells in: as a rule
// the blocks decay, cell 0 by far the largest, and each sum rounds at its own size.  Right-
// hand sides against long double, rms, the general path / cell 0 first / now: reach 4
// 3.6e-16 / 3.3e-16 / 3.5e-16, reach 12 4.4e-16 / 4.8e-16 / 3.9e-16, reach 40 6.2e-16 /
// 7.4e-16 / 4.5e-16.  In boxes read from memory four cells on each side are one trip:
// four right-hand sides on 10000 k, reach 12, 31.7 -> 22.2 us, a propagation on 512 k,
// reach 30, 4.87 -> 2.73 ms.
template <int MW, int NO, class P>
__device__ __forceinline__ void cell_sums(const ChainArgs &c, P pw, const Cells<MW> (&cell)[NO],
                                          const double *const (&op)[NO], int e, cd (&out)[NO])
{
    auto at = [&](int o, int r) {
        const double2 t = reinterpret_cast<const double2 *>(op[o])[r * 4 + e];
        return mk(t.x, t.y);
    };
    const int top = c.W - 1 + c.rmin, reach = MW > 0 ? MW : top > -c.rmin ? top : -c.rmin;
    const int most = 1 + (reach - 1) / 4 * 4;
    cd p[4];
#pragma unroll
    for (int o = 0; o < NO; o++) out[o] = mk(0, 0);
    if constexpr (MW > 0) {
        pw.first(1, p);
#pragma unroll
        for (int m = MW; m >= 1; m--)
#pragma unroll
            for (int o = 0; o < NO; o++) {
                out[o] = cfma(cell[o].v[MW + m], p[m - 1], out[o]);
                out[o] = cfma_jc(cell[o].v[MW - m], p[m - 1], out[o]);
            }
    } else {
        for (int m0 = most; m0 >= 1; m0 -= 4) {
            // a block's cells in one memory trip; outside the box cell 0, times 0
            cd u[4][NO], d[4][NO];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int o = 0; o < NO; o++) {
                    u[j][o] = at(o, (m0 + j <= top ? m0 + j : 0) - c.rmin);
                    d[j][o] = at(o, (m0 + j <= -c.rmin ? -(m0 + j) : 0) - c.rmin);
                }
            if (m0 == most) pw.first(m0, p);
            else pw.next(m0, p);
#pragma unroll
            for (int j = 3; j >= 0; j--) {
                const cd pu = m0 + j <= top ? p[j] : mk(0, 0), pd = m0 + j <= -c.rmin ? p[j] : mk(0, 0);
#pragma unroll
                for (int o = 0; o < NO; o++) {
                    out[o] = cfma(u[j][o], pu, out[o]);
                    out[o] = cfma_jc(d[j][o], pd, out[o]);
                }
            }
        }
    }
#pragma unroll
    for (int o = 0; o < NO; o++)
        if constexpr (MW > 0) out[o] = cadd(out[o], cell[o].v[MW]);
        else out[o] = cadd(out[o], at(o, -c.rmin));
}

// entry of X Y - Y X: dX = X_00 - X_11 multiplies the off-diagonal of Y and the
// reverse, and X_00 Y_00, the largest product and no part of the result, is not
// formed (with it the rounding error of a right-hand side, nine cells, was 4.3e-16, now 3.1e-16)
__device__ __forceinline__ cd commutator(cd X, cd Y)
{
    const int e = threadIdx.x & 3;
    const cd dX = csub(quad_of<0>(X), quad_of<3>(X)), dY = csub(quad_of<0>(Y), quad_of<3>(Y));
    // 00: X01 Y10 - Y01 X10, 01: dX Y01 - dY X01, 10: X10 dY - Y10 dX, 11: X10 Y01 - Y10 X01
    // (the permutes in all lanes, then the selects)
    const cd xu = quad<1, 1, 2, 2>(X), xl = quad<2, 1, 1, 1>(X), yu = quad<1, 1, 2, 2>(Y), yl = quad<2, 1, 1, 1>(Y);
    const cd p = e == 1 ? dX : xu, q = e == 2 ? dY : yl, r = e == 1 ? dY : yu, s = e == 2 ? dX : xl;
    return cfma(mk(-r.x, -r.y), s, cmul(p, q));
}

// entry of d rho/dt
__device__ __forceinline__ cd chain_rate(const ChainArgs &c, int e, cd H0, cd D, double E, cd rho)
{
    const cd t = commutator(mk(fma(E, D.x, H0.x), fma(E, D.y, H0.y)), rho);
    cd out = mk(t.y, -t.x);
    if (c.dephase) {
        // the rotation that diagonalises H0 (stage_device.hpp, jac_round), from the
        // identity: U = [[cs, sw], [-conj(sw), cs]], eigenvalue difference gap
        const cd h0 = quad_of<0>(H0), apq = quad_of<1>(H0), h1 = quad_of<3>(H0);
        const double d = h0.x - h1.x, m2 = fma(apq.x, apq.x, apq.y * apq.y);
        const double thr =
            1e-15 * (0.5 * (fabs(h0.x) + fabs(h0.y) + fabs(apq.x) + fabs(apq.y) + fabs(h1.x) + fabs(h1.y)));
        double cs = 1, gap = d;
        cd sw = mk(0, 0);
        if (m2 > thr * thr) {
            const double X = fma(d, d, 4 * m2), root = X * rsqrt_pos(X), Dq = fabs(d) + root;
            const double q = rsqrt_pos(fma(Dq, Dq, 4 * m2)), tq = copysign(2 * q, d);
            cs = Dq * q;
            sw = mk(tq * apq.x, tq * apq.y);
            gap = copysign(root, d);
        }
        double f = -c.F2;
        if (!(c.w < 0)) {
            const double dE = gap / c.w;
            f *= 1 - exp(-dE * dE);
        }
        const bool a = e & 2, b = e & 1;
        const cd u0a = a ? sw : mk(cs, 0), u0b = b ? sw : mk(cs, 0);
        const cd u1a = a ? mk(cs, 0) : mk(-sw.x, sw.y), u1b = b ? mk(cs, 0) : mk(-sw.x, sw.y);
        // (U rho U^dagger)_01 = sum_ab U_0a rho_ab conj(U_1b), _10 with 0 and 1 exchanged
        const cd h01 = cscale(quad_sum(cmul(cmul(u0a, rho), cconj(u1b))), f);
        const cd h10 = cscale(quad_sum(cmul(cmul(u1a, rho), cconj(u0b))), f);
        out = cfma_cj(u0a, cmul(h01, u1b), out);
        out = cfma_cj(u1a, cmul(h10, u0b), out);
    }
    return out;
}

__device__ __forceinline__ cd load_entry(const double *s, long at)
{
    const double2 v = reinterpret_cast<const double2 *>(s)[at];
    return mk(v.x, v.y);
}
// the lane's entry, and with pads the zeros between one matrix and the next
__device__ __forceinline__ void store_entry(double *s, const Site &p, int P, cd v, bool pads)
{
    if (!p.ok) return;
    reinterpret_cast<double2 *>(s)[p.at] = make_double2(v.x, v.y);
    if (pads)
        for (int q = 4; q + p.e < P; q += 4) reinterpret_cast<double2 *>(s)[p.at + q] = make_double2(0.0, 0.0);
}
// d/dt of special slot t: dA_0/dt = -E, the rest 0
__device__ __forceinline__ double2 special_rate(int t, double E) { return make_double2(t == 0 ? -E : 0.0, 0.0); }

// the special slots of dxdt; they are read as A by every block of
// chain_rhs_kernel, so with dxdt == x they are written behind it
__global__ void chain_specials_kernel(double *dxdt, double E)
{
    reinterpret_cast<double2 *>(dxdt)[threadIdx.x] = special_rate(threadIdx.x, E);
}

template <int MW>
__global__ __launch_bounds__(64) void chain_rhs_kernel(ChainArgs c, const double *x, double *dxdt, double E)
{
    const Site p = site(c);
    if (dxdt != x && blockIdx.x == 0 && threadIdx.x < 8)
        reinterpret_cast<double2 *>(dxdt)[threadIdx.x] = special_rate(threadIdx.x, E);
    const double *const op[2] = {c.Hb, c.Db};
    Cells<MW> cell[2];
    load_cells(c, c.Hb, p.e, cell[0]);
    load_cells(c, c.Db, p.e, cell[1]);
    const cd rho = load_entry(x, p.at);
    cd o[2];
    cell_sums(c, DirectPowers{p.frac + phase_offset(c, x[0])}, cell, op, p.e, o);
    store_entry(dxdt, p, c.P, chain_rate(c, p.e, o[0], o[1], E, rho), true);
}

// The block that takes the last ticket returns true in all its lanes (and has
// reset the counter); what every block stored before its ticket is visible.
__device__ __forceinline__ bool last_block(unsigned *ticket)
{
    unsigned t = 0;
    if (threadIdx.x == 0) t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    t = __shfl(t, 0);
    if (t + 1 != gridDim.x) return false;
    __threadfence();
    if (threadIdx.x == 0) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// j(t) of x into j[3] and, if k1, the derivative of x: the terms of jk_body per
// entry, one partial sum per block, added up by the last block in block order
template <int MW>
__global__ __launch_bounds__(64) void chain_output_kernel(ChainArgs c, const double *x, double *j, double *partial,
                                                          double *k1, double E, unsigned *ticket)
{
    const Site p = site(c);
    if (k1 && blockIdx.x == 0 && threadIdx.x < 8)
        reinterpret_cast<double2 *>(k1)[threadIdx.x] = special_rate(threadIdx.x, E);
    const double *const op[3] = {c.Hb, c.Db, c.dHb};
    Cells<MW> cell[3];
    load_cells(c, c.Hb, p.e, cell[0]);
    load_cells(c, c.Db, p.e, cell[1]);
    load_cells(c, c.dHb, p.e, cell[2]);
    const cd rho = load_entry(x, p.at);
    cd o[3];
    cell_sums(c, DirectPowers{p.frac + phase_offset(c, x[0])}, cell, op, p.e, o);
    // -Im D_ab T_ba - Re dH_ab rho_ba, T = H0 rho - rho H0
    const cd T = quad<0, 2, 1, 3>(commutator(o[0], rho)), rt = quad<0, 2, 1, 3>(rho);
    double jk = -cmul(o[1], T).y - cmul(o[2], rt).x;
    if (k1) store_entry(k1, p, c.P, chain_rate(c, p.e, o[0], o[1], E, rho), true);
    jk = seg_sum<64>(p.ok ? jk : 0.0);
    if (threadIdx.x == 0) partial[blockIdx.x] = jk;
    if (!last_block(ticket)) return;
    double v = 0;
    for (unsigned i = threadIdx.x; i < gridDim.x; i += 64)
        v += __hip_atomic_load(partial + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = seg_sum<64>(v);
    if (threadIdx.x < 3) j[threadIdx.x] = threadIdx.x == 0 ? v / (double)c.nk : 0.0;
}

// one attempt: x_new, k7 and the error norm (ChainAttempt)
template <int MW>
__global__ __launch_bounds__(64) void chain_attempt_kernel(ChainArgs c, ChainAttempt s)
{
    const Site p = site(c);
    const double *const op[2] = {c.Hb, c.Db};
    Cells<MW> cell[2];
    load_cells(c, c.Hb, p.e, cell[0]);
    load_cells(c, c.Db, p.e, cell[1]);
    const cd x = load_entry(s.x, p.at);
    cd kd[7];  // k_1 .. k_7
    kd[0] = load_entry(s.k1, p.at);
    // stage q reads k_1 .. k_{q+1}, the seventh k_1, k_3 .. k_6; the A slots of
    // its derivatives are k_1's and -E of the others' stages
    double A[6];
    {
        const double xA = s.x[0], kA = s.k1[0];
#pragma unroll
        for (int q = 0; q < 6; q++) {
            A[q] = xA;
#pragma unroll
            for (int j = 0; j < (q < 5 ? q + 1 : 5); j++) {
                const int kj = j == 0 || q < 5 ? j : j + 1;
                A[q] += s.c[q][j] * (kj == 0 ? kA : -s.E[kj - 1]);
            }
        }
    }
    // the quad's lanes form the phase factors of stages e and e + 4 (the last
    // two lanes' second one is not used)
    const int e = p.e;
    const cd za = phase_factor(c, p.frac, e == 0 ? A[0] : e == 1 ? A[1] : e == 2 ? A[2] : A[3]);
    const cd zb = phase_factor(c, p.frac, e & 1 ? A[5] : A[4]);
    const cd z[6] = {quad_of<0>(za), quad_of<1>(za), quad_of<2>(za), quad_of<3>(za), quad_of<0>(zb), quad_of<1>(zb)};
    cd in;
#pragma unroll
    for (int q = 0; q < 6; q++) {
        in = x;
#pragma unroll
        for (int j = 0; j < (q < 5 ? q + 1 : 5); j++) {
            const int kj = j == 0 || q < 5 ? j : j + 1;
            in.x += s.c[q][j] * kd[kj].x;
            in.y += s.c[q][j] * kd[kj].y;
        }
        cd o[2];
        cell_sums(c, FactorPowers{z[q], {}}, cell, op, e, o);
        kd[q + 1] = chain_rate(c, e, o[0], o[1], s.E[q], in);
    }
    store_entry(s.xn, p, c.P, in, true);
    store_entry(s.k7, p, c.P, kd[6], true);
    const int idx[6] = {0, 2, 3, 4, 5, 6};
    double2 kv[6];
#pragma unroll
    for (int j = 0; j < 6; j++) kv[j] = make_double2(kd[idx[j]].x, kd[idx[j]].y);
    ErrMax err;
    if (p.ok) err.add(err_entry(make_double2(x.x, x.y), kv, s.err_e, s.ea, s.er, s.dt));
    if (blockIdx.x == 0 && threadIdx.x < 8) {
        // the special slots
        const int t = threadIdx.x;
        const double2 xv = reinterpret_cast<const double2 *>(s.x)[t];
        kv[0] = reinterpret_cast<const double2 *>(s.k1)[t];
#pragma unroll
        for (int j = 1; j < 6; j++) kv[j] = special_rate(t, s.E[j]);
        double re = xv.x, im = xv.y;
#pragma unroll
        for (int j = 0; j < 5; j++) {
            re += s.c[5][j] * kv[j].x;
            im += s.c[5][j] * kv[j].y;
        }
        reinterpret_cast<double2 *>(s.xn)[t] = make_double2(re, im);
        reinterpret_cast<double2 *>(s.k7)[t] = kv[5];
        err.add(err_entry(xv, kv, s.err_e, s.ea, s.er, s.dt));
    }
    const double mine = err.wave();
    if (threadIdx.x == 0) s.partial[blockIdx.x] = mine;
    if (!last_block(s.ticket)) return;
    ErrMax all;
    for (unsigned b = threadIdx.x; b < gridDim.x; b += 64)
        all.add(__hip_atomic_load(s.partial + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    const double v = all.wave();
    if (threadIdx.x == 0) store_error(s.err_out, v);
}

// The cells a lane keeps: 4 VGPRs per cell and operator, so up to nine (the
// benchmark chain) fit beside the derivatives; wider boxes are read per stage.
template <class F>
static hipError_t by_extent(const ChainArgs &c, F &&launch)
{
    const int reach = -c.rmin > c.W - 1 + c.rmin ? -c.rmin : c.W - 1 + c.rmin;
    const dim3 grid((unsigned)((c.nk + 15) / 16)), blk(64);
    if (reach <= 2) launch(std::integral_constant<int, 2>{}, grid, blk);
    else if (reach <= 4) launch(std::integral_constant<int, 4>{}, grid, blk);
    else launch(std::integral_constant<int, 0>{}, grid, blk);
    return hipGetLastError();
}

hipError_t launch_chain_rhs(const ChainArgs &c, const double *x, double *dxdt, double E, hipStream_t s)
{
    const hipError_t e = by_extent(c, [&](auto mw, dim3 grid, dim3 blk) {
        hipLaunchKernelGGL(chain_rhs_kernel<decltype(mw)::value>, grid, blk, 0, s, c, x, dxdt, E);
    });
    if (e != hipSuccess || dxdt != x) return e;
    hipLaunchKernelGGL(chain_specials_kernel, dim3(1), dim3(8), 0, s, dxdt, E);
    return hipGetLastError();
}

hipError_t launch_chain_output(const ChainArgs &c, const double *x, double *j, double *partial, double *k1, double E,
                               unsigned *ticket, hipStream_t s)
{
    return by_extent(c, [&](auto mw, dim3 grid, dim3 blk) {
        hipLaunchKernelGGL(chain_output_kernel<decltype(mw)::value>, grid, blk, 0, s, c, x, j, partial, k1, E, ticket);
    });
}

hipError_t launch_chain_attempt(const ChainArgs &c, const ChainAttempt &a, hipStream_t s)
{
    return by_extent(c, [&](auto mw, dim3 grid, dim3 blk) {
        hipLaunchKernelGGL(chain_attempt_kernel<decltype(mw)::value>, grid, blk, 0, s, c, a);
    });
}

}  // namespace sbe
