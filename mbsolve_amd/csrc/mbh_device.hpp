/*
 * Per-cell density propagators of the gfx950 Maxwell-Bloch backend.
 *
 * Every update works on one grid cell whose state lives in registers and
 * reads its material constants through a wave-uniform pointer, so the
 * compiler turns the constant reads into scalar (s_load) loads.
 *
 * FP64 "mirror" forms follow the reference update expressions operand by
 * operand (dot products accumulate in ascending index order, starting
 * from the first product; no fused multiply-add), which makes them
 * bit-identical to a CPU implementation that uses the same order.
 */
#ifndef MBH_DEVICE_HPP
#define MBH_DEVICE_HPP

#include <hip/hip_runtime.h>
#include <type_traits>
#include <utility>
#include <stdint.h>

#include "../../include/mbsolve_hip.h"

namespace mbh {

/* Material constants are read through the constant address space: with a
 * wave-uniform address these become scalar (s_load) loads even though the
 * kernel stores to global memory. */
typedef const __attribute__((address_space(4))) double* cdp;

/* ---- complex helpers (naive formulas, the libstdc++ fast path) --------- */
struct cplx {
    double re, im;
};
typedef const __attribute__((address_space(4))) cplx* ccp;

__device__ __forceinline__ cplx cmul(cplx a, cplx b)
{
    return cplx{ a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re };
}
__device__ __forceinline__ cplx cadd(cplx a, cplx b)
{
    return cplx{ a.re + b.re, a.im + b.im };
}
__device__ __forceinline__ cplx csub(cplx a, cplx b)
{
    return cplx{ a.re - b.re, a.im - b.im };
}
/* 1 / z = conj(z) / |z|^2 */
__device__ __forceinline__ cplx cinv(cplx z)
{
    double s = z.re * z.re + z.im * z.im;
    return cplx{ z.re / s, -z.im / s };
}

/* Matrix product C = A B of N x N complex matrices (row-major). */
template<int N>
__device__ __forceinline__ void cmatmul(const cplx* A, const cplx* B, cplx* C)
{
#pragma unroll
    for (int i = 0; i < N; i++) {
#pragma unroll
        for (int j = 0; j < N; j++) {
            cplx acc = cmul(A[i * N], B[j]);
#pragma unroll
            for (int k = 1; k < N; k++) {
                acc = cadd(acc, cmul(A[i * N + k], B[k * N + j]));
            }
            C[i * N + j] = acc;
        }
    }
}

/* C = A B^dagger */
template<int N>
__device__ __forceinline__ void cmatmul_adj(const cplx* A, const cplx* B,
                                            cplx* C)
{
#pragma unroll
    for (int i = 0; i < N; i++) {
#pragma unroll
        for (int j = 0; j < N; j++) {
            cplx b0{ B[j * N].re, -B[j * N].im };
            cplx acc = cmul(A[i * N], b0);
#pragma unroll
            for (int k = 1; k < N; k++) {
                cplx bk{ B[j * N + k].re, -B[j * N + k].im };
                acc = cadd(acc, cmul(A[i * N + k], bk));
            }
            C[i * N + j] = acc;
        }
    }
}

/* Inverse of an N x N complex matrix: cofactor formula for N == 2,
 * Gauss-Jordan with partial pivoting (largest |a|^2) otherwise. */
template<int N>
__device__ __forceinline__ void cinverse(const cplx* A, cplx* R)
{
    if constexpr (N == 2) {
        cplx det = csub(cmul(A[0], A[3]), cmul(A[1], A[2]));
        cplx id = cinv(det);
        R[0] = cmul(A[3], id);
        R[1] = cmul(cplx{ -A[1].re, -A[1].im }, id);
        R[2] = cmul(cplx{ -A[2].re, -A[2].im }, id);
        R[3] = cmul(A[0], id);
    } else {
        cplx W[N * N];
#pragma unroll
        for (int i = 0; i < N * N; i++) {
            W[i] = A[i];
            R[i] = cplx{ (i / N == i % N) ? 1.0 : 0.0, 0.0 };
        }
#pragma unroll
        for (int col = 0; col < N; col++) {
            /* pivot search */
            int piv = col;
            double best = W[col * N + col].re * W[col * N + col].re +
                W[col * N + col].im * W[col * N + col].im;
#pragma unroll
            for (int r = col + 1; r < N; r++) {
                double v = W[r * N + col].re * W[r * N + col].re +
                    W[r * N + col].im * W[r * N + col].im;
                if (v > best) {
                    best = v;
                    piv = r;
                }
            }
            /* row swap (register-friendly: compare-select per row) */
#pragma unroll
            for (int r = col + 1; r < N; r++) {
                if (r == piv) {
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        cplx t = W[col * N + k];
                        W[col * N + k] = W[r * N + k];
                        W[r * N + k] = t;
                        t = R[col * N + k];
                        R[col * N + k] = R[r * N + k];
                        R[r * N + k] = t;
                    }
                }
            }
            cplx ip = cinv(W[col * N + col]);
#pragma unroll
            for (int k = 0; k < N; k++) {
                W[col * N + k] = cmul(W[col * N + k], ip);
                R[col * N + k] = cmul(R[col * N + k], ip);
            }
#pragma unroll
            for (int r = 0; r < N; r++) {
                if (r != col) {
                    cplx f = W[r * N + col];
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        W[r * N + k] = csub(W[r * N + k],
                                            cmul(f, W[col * N + k]));
                        R[r * N + k] = csub(R[r * N + k],
                                            cmul(f, R[col * N + k]));
                    }
                }
            }
        }
    }
}

/* NC constants of one material, the same for every lane, sixteen to a
 * register pair: lane l of each row of 16 lanes holds constants
 * 16 i + l % 16, and v_fmac_f64 with DPP row_newbcast multiplies by one of
 * them.  An FMA with such a constant then takes no load and no further
 * instruction, where scalar loads or LDS reads of some hundred constants
 * stall every step of a grid that leaves one wavefront on a SIMD.  (Measured
 * on one wavefront per SIMD: every VALU instruction issues 5 cycles after the
 * one before, a dependent FP64 FMA too, one with DPP after 6.)
 * All lanes must be active: an FMA reads the row's other lanes.
 * DPP reads a register no earlier than two wait states after its write.
 * The registers are written by loads before the steps; pin() at the start of
 * a step keeps those states where the compiler copies one there.  Elsewhere
 * only the register allocator could write one (a copy, a spill); the build
 * refuses a library whose code has such a write in the two wait states before
 * a read (isa_check.py). */
template<int NC>
struct row_consts {
    static constexpr int NR = (NC + 15) / 16;
    double r[NR];

    __device__ __forceinline__ void load(const double* p)
    {
        const int l = threadIdx.x & 15;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            r[i] = p[16 * i + l < NC ? 16 * i + l : NC - 1];
        }
    }
    __device__ __forceinline__ void pin()
    {
#pragma unroll
        for (int i = 0; i < NR; i++) {
            asm volatile("" : "+v"(r[i]));
        }
        asm volatile("s_nop 1" : "+v"(r[NR - 1]));
    }
    /* acc += constant I * x */
    template<int I>
    __device__ __forceinline__ void fmac(double& acc, double x) const
    {
        asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf "
            "bank_mask:0xf"
            : "+v"(acc)
            : "v"(r[I / 16]), "v"(x), "n"(I % 16));
    }
    /* constant I in every lane */
    template<int I>
    __device__ __forceinline__ double get() const
    {
        return __longlong_as_double(__builtin_amdgcn_update_dpp(
            0ll, __double_as_longlong(r[I / 16]), 0x150 + I % 16, 0xf, 0xf,
            true));
    }
};

/* calls f(std::integral_constant<int, i>()) for i = 0 .. N - 1 */
template<typename F, int... I>
__device__ __forceinline__ void static_for(F&& f,
                                           std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>()), ...);
}
template<int N, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for(f, std::make_integer_sequence<int, N>());
}

/* ======================================================================
 * lindblad_noop (algo_lindblad_noop.hpp:35-86): no density, p untouched.
 * ==================================================================== */
struct algo_noop {
    static constexpr int ROWC_WAVES = 1;
    static constexpr bool CONSTS = false;
    static constexpr bool ROWC = false;
    static constexpr int STAGE = 0;
    static constexpr bool SHIFT = false;
    static constexpr bool FAST_FDTD = false;
    static constexpr int DC = 0; /* stored density components */
    static constexpr int STATE = 1;
    struct state {
        double v[STATE];
    };
    __device__ static void update(cdp, state&, double, double&) {}
    template<int C>
    __device__ static void update_multi(cdp, state*, const double*, double*)
    {
    }
    __device__ static double inversion(cdp, const state&) { return 0.0; }
    __device__ static double population(cdp, const state&, int)
    {
        return 0.0;
    }
};

/* noop with the folded FDTD constants (FP32-storage form: not bound to the
 * reference's operation order) */
struct algo_noop_fast : algo_noop {
    static constexpr bool FAST_FDTD = true;
};
/* the same, for states whose cells with H held at zero start at zero: there
 * fc' = 0 keeps them at zero, so h' = h + fc' (e_c - e_l) needs no factor */
struct algo_noop_hz0 : algo_noop_fast {};

/* ======================================================================
 * lindblad_reg_cayley<N>::update (algo_lindblad_reg_cayley.hpp:228-257)
 *
 * Blob layout: see MBH_CAYLEY_STRIDE in mbsolve_hip.h.  State: the full
 * N x N complex density matrix, row-major, (re, im) interleaved, exactly
 * as the reference keeps it (no Hermitian symmetrisation).
 * ==================================================================== */
template<int N>
struct algo_cayley {
    static constexpr int ROWC_WAVES = 1;
    static constexpr bool CONSTS = false;
    static constexpr bool ROWC = false;
    static constexpr int STAGE = 0;
    static constexpr bool SHIFT = false;
    static constexpr bool FAST_FDTD = false;
    static constexpr int DC = 2 * N * N;
    static constexpr int STATE = 2 * N * N;
    struct state {
        double v[STATE];
    };

    static constexpr int OFF_H0 = 5;
    static constexpr int OFF_MU = OFF_H0 + 2 * N * N;
    static constexpr int OFF_d1 = OFF_MU + 2 * N * N;
    static constexpr int OFF_d2 = OFF_d1 + N * N;
    static constexpr int OFF_D1 = OFF_d2 + N * N;
    static constexpr int OFF_D2 = OFF_D1 + N * N;

    /* propagate_dissipation (algo_lindblad_reg_cayley.hpp:206-217):
     * coherences *= D2 (elementwise), diagonal <- D1 * diagonal. */
    __device__ static void dissipate(cdp q, const cplx* d, cplx* o)
    {
        cdp D1 = q + OFF_D1;
        cdp D2 = q + OFF_D2;
#pragma unroll
        for (int i = 0; i < N * N; i++) {
            o[i] = cplx{ D2[i] * d[i].re, D2[i] * d[i].im };
        }
#pragma unroll
        for (int i = 0; i < N; i++) {
            cplx acc{ D1[i * N] * d[0].re, D1[i * N] * d[0].im };
#pragma unroll
            for (int k = 1; k < N; k++) {
                acc.re = acc.re + D1[i * N + k] * d[k * N + k].re;
                acc.im = acc.im + D1[i * N + k] * d[k * N + k].im;
            }
            o[i * N + i] = acc;
        }
    }


    /* branch-free body; only for media with a density */
    __device__ static void update(cdp q, state& s, double e, double& p)
    {
        ccp H0 = (ccp)(q + OFF_H0);
        ccp mu = (ccp)(q + OFF_MU);
        const double prop_im = q[3];
        const double rhs_im = q[4];
        cplx* d = reinterpret_cast<cplx*>(s.v);

        /* H = H0 - e mu;  M = (-i/hbar dt) H */
        cplx A[N * N], B[N * N];
#pragma unroll
        for (int i = 0; i < N * N; i++) {
            cplx h{ H0[i].re - e * mu[i].re, H0[i].im - e * mu[i].im };
            cplx m{ -(prop_im * h.im), prop_im * h.re };
            double di = (i / N == i % N) ? 1.0 : 0.0;
            /* A = I - 0.5 M, B = I + 0.5 M */
            A[i] = cplx{ di - 0.5 * m.re, -(0.5 * m.im) };
            B[i] = cplx{ di + 0.5 * m.re, 0.5 * m.im };
        }
        /* Cayley propagator U2 = A^-1 B */
        cplx Ai[N * N], U2[N * N], Hm[N * N];
        cinverse<N>(A, Ai);
        cmatmul<N>(Ai, B, U2);
#pragma unroll
        for (int i = 0; i < N * N; i++) {
            Hm[i] = cplx{ H0[i].re, H0[i].im };
        }

        /* dissipation half step, unitary full step, dissipation half step */
        cplx d1[N * N], t[N * N];
        dissipate(q, d, d1);
        cmatmul<N>(U2, d1, t);
        cmatmul_adj<N>(t, U2, d1);
        dissipate(q, d1, d);

        /* polarization derivative: rhs = -i/hbar [H0, d] + D(d);
         * p = n Re tr(rhs mu) */
        cdp r1 = q + OFF_d1;
        cdp r2 = q + OFF_d2;
        cplx c1[N * N], c2[N * N];
        cmatmul<N>(Hm, d, c1);
        cmatmul<N>(d, Hm, c2);
        cplx rhs[N * N];
#pragma unroll
        for (int i = 0; i < N * N; i++) {
            cplx c = csub(c1[i], c2[i]);
            cplx g{ -(rhs_im * c.im), rhs_im * c.re };
            rhs[i] = cplx{ r2[i] * d[i].re, r2[i] * d[i].im };
            if (i / N == i % N) {
                int ii = i / N;
                cplx acc{ r1[ii * N] * d[0].re, r1[ii * N] * d[0].im };
#pragma unroll
                for (int k = 1; k < N; k++) {
                    acc.re = acc.re + r1[ii * N + k] * d[k * N + k].re;
                    acc.im = acc.im + r1[ii * N + k] * d[k * N + k].im;
                }
                rhs[i] = acc;
            }
            rhs[i] = cadd(g, rhs[i]);
        }
        double tr = 0.0;
#pragma unroll
        for (int i = 0; i < N; i++) {
            double di = rhs[i * N].re * mu[i].re - rhs[i * N].im * mu[i].im;
#pragma unroll
            for (int k = 1; k < N; k++) {
                di = di +
                    (rhs[i * N + k].re * mu[k * N + i].re -
                     rhs[i * N + k].im * mu[k * N + i].im);
            }
            tr = (i == 0) ? di : tr + di;
        }
        p = q[1] * tr;
    }

    template<int C>
    __device__ static void update_multi(cdp q, state* s, const double* e,
                                        double* p)
    {
#pragma unroll
        for (int c = 0; c < C; c++) {
            update(q, s[c], e[c], p[c]);
        }
    }

    /* calc_inversion / calc_population (algo_lindblad_reg_cayley.hpp:259-267) */
    __device__ static double inversion(cdp, const state& s)
    {
        return s.v[2 * (N + 1)] - s.v[0];
    }
    __device__ static double population(cdp, const state& s, int m)
    {
        double r = 0.0;
#pragma unroll
        for (int i = 0; i < N; i++) {
            if (i == m) {
                r = s.v[2 * (i * N + i)];
            }
        }
        return r;
    }
};

/* ======================================================================
 * algo_cayley<2> for media with a diagonal real Hamiltonian and a real,
 * purely off-diagonal symmetric dipole (what qm_desc_2lvl builds,
 * qm_description.hpp:338-432): the same operations in the same order without
 * those whose operand is an exact zero or one, so the results are bit for
 * bit those of the general form (up to the sign of zeros).  With
 * H = diag(a, b) - e u sigma_x, alpha = prop_im a / 2, beta = prop_im b / 2
 * and gamma = -prop_im e u / 2 the factors are
 *   I - M/2 = ((1, -alpha), (0, -gamma); (0, -gamma), (1, -beta)),
 * their determinant is (1 - alpha beta + gamma^2, -alpha - beta), and p needs
 * the two coherences of rhs only: about 215 FP64 instructions per cell
 * instead of 430.  The two divisions by |det|^2 share one reciprocal (the
 * quotients come from the hardware division's own sequence without its
 * scaling, which is the identity in the range checked here; outside it the
 * step runs the general update).
 * ==================================================================== */
struct algo_cayley2r : algo_cayley<2> {
    static constexpr bool CONSTS = true;
    struct consts {
        double alpha, beta, c0, nc1, c11, hp, u;
        double D2a, D2b, D1[4], r2a, r2b, a, b, rhs_im, carrier;
        const double* q; /* the blob (general update) */
    };
    template<typename P>
    __device__ static consts load(P q)
    {
        consts k;
        const double prop_im = q[3];
        k.rhs_im = q[4];
        k.carrier = q[1];
        k.a = q[OFF_H0];
        k.b = q[OFF_H0 + 6];
        k.u = q[OFF_MU + 2];
        k.alpha = 0.5 * (prop_im * k.a);
        k.beta = 0.5 * (prop_im * k.b);
        k.c0 = 1.0 - k.alpha * k.beta;
        const double c1 = -k.beta - k.alpha;
        k.nc1 = -c1;
        k.c11 = c1 * c1;
        k.hp = 0.5 * prop_im;
        k.D2a = q[OFF_D2 + 1];
        k.D2b = q[OFF_D2 + 2];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            k.D1[i] = q[OFF_D1 + i];
        }
        k.r2a = q[OFF_d2 + 1];
        k.r2b = q[OFF_d2 + 2];
        k.q = (const double*)q;
        return k;
    }
    /* a medium without a density: the state stays, p is zero */
    __device__ static consts one()
    {
        consts k{};
        k.c0 = k.D2a = k.D2b = k.D1[0] = k.D1[3] = 1.0;
        return k;
    }

    __device__ static void dissipate2(const consts& k, double* d)
    {
        const double* D1 = k.D1;
        d[2] = k.D2a * d[2];
        d[3] = k.D2a * d[3];
        d[4] = k.D2b * d[4];
        d[5] = k.D2b * d[5];
        const double r0 = D1[0] * d[0] + D1[1] * d[6];
        const double i0 = D1[0] * d[1] + D1[1] * d[7];
        const double r1 = D1[2] * d[0] + D1[3] * d[6];
        const double i1 = D1[2] * d[1] + D1[3] * d[7];
        d[0] = r0;
        d[1] = i0;
        d[6] = r1;
        d[7] = i1;
    }

    template<int C>
    __device__ static void apply(const consts& k, state* s, const double* e,
                                 double* p)
    {
        double gam[C], dr[C], s2[C];
        bool ok = true;
#pragma unroll
        for (int c = 0; c < C; c++) {
            gam[c] = k.hp * (-(e[c] * k.u));
            dr[c] = k.c0 + gam[c] * gam[c];
            s2[c] = dr[c] * dr[c] + k.c11;
            ok = ok && s2[c] >= 0x1p-200 && s2[c] <= 0x1p+200;
        }
        if (!__all(ok)) {
#pragma unroll
            for (int c = 0; c < C; c++) {
                if (k.q != nullptr) {
                    algo_cayley<2>::update((cdp)k.q, s[c], e[c], p[c]);
                }
            }
            return;
        }
#pragma unroll
        for (int c = 0; c < C; c++) {
            double* v = s[c].v;
            const double g = gam[c], al = k.alpha, be = k.beta;
            /* 1 / det = (x, y) */
            double r = __builtin_amdgcn_rcp(s2[c]);
            double t = fma(-s2[c], r, 1.0);
            r = fma(r, t, r);
            t = fma(-s2[c], r, 1.0);
            r = fma(r, t, r);
            double x = dr[c] * r;
            x = fma(fma(-s2[c], x, dr[c]), r, x);
            double y = k.nc1 * r;
            y = fma(fma(-s2[c], y, k.nc1), r, y);
            /* inverse of I - M/2 */
            const cplx R0{ x + be * y, y - be * x };
            const cplx R1{ -(g * y), g * x };
            const cplx R3{ x + al * y, y - al * x };
            /* U = R (I + M/2) */
            const double g1r = R1.re * g, g1i = R1.im * g;
            const cplx U0{ (R0.re - R0.im * al) - g1i,
                           (R0.re * al + R0.im) + g1r };
            const cplx U1{ -(R0.im * g) + (R1.re - R1.im * be),
                           R0.re * g + (R1.re * be + R1.im) };
            const cplx U2{ (R1.re - R1.im * al) - R3.im * g,
                           (R1.re * al + R1.im) + R3.re * g };
            const cplx U3{ -g1i + (R3.re - R3.im * be),
                           g1r + (R3.re * be + R3.im) };
            const cplx U[4] = { U0, U1, U2, U3 };
            dissipate2(k, v);
            cplx d[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                d[i] = cplx{ v[2 * i], v[2 * i + 1] };
            }
            cmatmul<2>(U, d, w);
            cmatmul_adj<2>(w, U, d);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v[2 * i] = d[i].re;
                v[2 * i + 1] = d[i].im;
            }
            dissipate2(k, v);
            /* the coherences of rhs = -i/hbar [H0, d] + D(d) */
            const double q1 =
                -(k.rhs_im * (k.a * v[3] - v[3] * k.b)) + k.r2a * v[2];
            const double q2 =
                -(k.rhs_im * (k.b * v[5] - v[5] * k.a)) + k.r2b * v[4];
            p[c] = k.carrier * (q1 * k.u + q2 * k.u);
        }
    }

    __device__ static void update(cdp q, state& s, double e, double& p)
    {
        apply<1>(load(q), &s, &e, &p);
    }
};

/* ======================================================================
 * Two-level regularized Cayley in closed Bloch form.  Mathematically the
 * update of algo_cayley<2> (algo_lindblad_reg_cayley.hpp:206-257) for a
 * Hermitian state, rearranged.  With H = h0 I + h.sigma and
 * alpha = -(prop_im / 2) (h0, h_vec), the Cayley factor is proportional to
 *   W = s I - i beta.sigma,  beta = 2 alpha_vec,  s = 1 + alpha0^2 - |alpha|^2
 * so U rho U^+ rotates m = (Re rho01, -Im rho01, (rho00 - rho11) / 2) by
 *   m' = m + lambda (s beta x m + beta x (beta x m)),
 *   lambda = 2 / (s^2 + |beta|^2)
 * and keeps the trace tau.  The dissipation D scales the coherence by g and
 * maps the populations with D1.
 *
 * Carried state: sigma = the state between the unitary step and the second
 * dissipation half step, as (tau, m_x, m_y, m_z).  The reference state
 * after step n is rho_n = D(sigma_n), and the next step needs
 * D(rho_n) = D^2(sigma_n): one merged dissipation per step.  p and the
 * populations are fixed linear forms of sigma.
 *
 * Blob (BLOCH2_STRIDE doubles):
 *   [0] has_qm  [1..3] beta at e = 0  [4..6] d beta / d e
 *   [7] alpha0 at e = 0  [8] d alpha0 / d e  [9] g^2
 *   [10..13] F: D1^2 on (tau, m_z), row-major
 *   [14..17] p = P . (tau, m_x, m_y, m_z)
 *   [18..21] populations: rho00 = R00 tau + R01 m_z, rho11 = R10 tau + R11 m_z
 *   [22..25] D1 (row-major)  [26] g  [27] 1 + alpha0^2 at e = 0
 *   [28] (beta_z at e = 0)^2
 * ==================================================================== */
template<int KIND>
struct algo_bloch2_t {
    /* what is exactly zero in every medium, see apply */
    static constexpr bool REAL = KIND >= 1, DIAG = KIND == 2;
    static constexpr int ROWC_WAVES = 1;
    static constexpr int STAGE = 0;
    static constexpr bool SHIFT = false;
    static constexpr int DC = 4;
    static constexpr int STATE = 4;
    static constexpr bool FAST_FDTD = true;
    struct state {
        double v[STATE];
    };


    /* Constants of one material, loaded before the steps of a launch: from
     * a wave-uniform address they stay in SGPRs (read inside the step they
     * cost two scalar-load latencies per step), from a lane's own address
     * (one cell per lane) in VGPRs, so that every lane updates with its own
     * material's constants and no step has a branch on the material.
     * one(): a medium without a density, which leaves the state as it is
     * and p at zero. */
    static constexpr bool CONSTS = true;
    static constexpr bool ROWC = false;
    struct consts {
        double bcx, bcy, bcz, bex, bey, bez, a0c, a0e, g2;
        double F00, F01, F10, F11, P0, P1, P2, P3;
        double bz2, A0; /* DIAG: bcz^2; REAL: 1 + a0c^2 */
    };
    template<typename P>
    __device__ static consts load(P q)
    {
        consts k;
        k.bcx = q[1];
        k.bcy = q[2];
        k.bcz = q[3];
        k.bex = q[4];
        k.bey = q[5];
        k.bez = q[6];
        k.a0c = q[7];
        k.a0e = q[8];
        k.g2 = q[9];
        k.F00 = q[10];
        k.F01 = q[11];
        k.F10 = q[12];
        k.F11 = q[13];
        k.P0 = q[14];
        k.P1 = q[15];
        k.P2 = q[16];
        k.P3 = q[17];
        k.bz2 = q[28];
        k.A0 = q[27];
        return k;
    }
    __device__ static consts one()
    {
        consts k{};
        k.g2 = k.F00 = k.F11 = k.A0 = 1.0;
        return k;
    }

    /* 2 / n2 for n2 near 1: hardware reciprocal and one cubic step (with
     * t = 1 - n2 r of at most 2^-20, r (1 + t + t^2) is off by a relative
     * t^3) */
    __device__ static double two_over(double n2)
    {
        const double r = __builtin_amdgcn_rcp(n2);
        const double t = fma(-n2, r, 1.0);
        const double u = fma(r, fma(t, t, t), r);
        return u + u;
    }

    /* C cells of one material.  The rotation is written with
     * c = beta x m and u = lambda (s m + c):  m' = m + beta x u, whose y
     * component expands to m_y + lambda (s c_y + beta_y (beta.m) -
     * |beta|^2 m_y).
     * REAL: beta_y, d alpha0 / d e and the p coefficients of tau and m_z
     * are exactly zero (a real Hamiltonian, a real dipole and no dipole on
     * the diagonal to enter p).  DIAG: so are beta_x at e = 0 and
     * d beta_z / d e, and F00 = 1, F01 = 0 (a diagonal Hamiltonian and a
     * purely off-diagonal dipole, as qm_desc_2lvl builds them,
     * qm_description.hpp:338-432; the relaxation keeps the trace).  The
     * terms dropped are exact zeros and ones of the general form, so the
     * results are the same (up to the sign of zeros): 24 FP64 instructions
     * per cell (DIAG) and 30 (REAL) where the general form takes about 45.
     * 2^20 cells with an off-diagonal Hamiltonian, 1000 steps: 3.16 ms in
     * the general form, 2.32 ms. */
    template<int C>
    __device__ static void apply(const consts& k, state* s, const double* e,
                                 double* p)
    {
#pragma unroll
        for (int c = 0; c < C; c++) {
            double* v = s[c].v;
            /* second half step of the previous step and first half step
             * of this one */
            const double tr = DIAG ? v[0] : fma(k.F01, v[3], k.F00 * v[0]);
            const double mz = fma(k.F11, v[3], k.F10 * v[0]);
            const double mx = k.g2 * v[1];
            const double my = k.g2 * v[2];
            /* Cayley rotation at field e */
            const double bx =
                DIAG ? e[c] * k.bex : fma(e[c], k.bex, k.bcx);
            const double by = REAL ? 0.0 : fma(e[c], k.bey, k.bcy);
            const double bz = DIAG ? k.bcz : fma(e[c], k.bez, k.bcz);
            const double bz2 = DIAG ? k.bz2 : bz * bz;
            const double r2 =
                fma(bx, bx, REAL ? bz2 : fma(by, by, bz2));
            const double a0 = REAL ? 0.0 : fma(e[c], k.a0e, k.a0c);
            const double sc = fma(-0.25, r2, REAL ? k.A0 : fma(a0, a0, 1.0));
            const double lam = two_over(fma(sc, sc, r2));
            const double cy = fma(bz, mx, -(bx * mz));
            const double uy = lam * fma(sc, my, cy);
            v[0] = tr;
            if constexpr (REAL) {
                v[1] = fma(-bz, uy, mx);
                v[3] = fma(bx, uy, mz);
                v[2] = fma(lam, fma(sc, cy, -(r2 * my)), my);
                p[c] = fma(k.P2, v[2], k.P1 * v[1]);
            } else {
                const double cx = fma(by, mz, -(bz * my));
                const double cz = fma(bx, my, -(by * mx));
                const double ux = lam * fma(sc, mx, cx);
                const double uz = lam * fma(sc, mz, cz);
                const double bm = fma(bz, mz, fma(by, my, bx * mx));
                v[1] = fma(by, uz, fma(-bz, uy, mx));
                v[3] = fma(-by, ux, fma(bx, uy, mz));
                v[2] = fma(lam, fma(sc, cy, fma(by, bm, -(r2 * my))), my);
                p[c] = fma(k.P3, v[3],
                           fma(k.P2, v[2], fma(k.P1, v[1], k.P0 * tr)));
            }
        }
    }

    __device__ static void update(cdp q, state& s, double e, double& p)
    {
        apply<1>(load(q), &s, &e, &p);
    }

    __device__ static double population(cdp q, const state& s, int m)
    {
        if (m == 0) {
            return fma(q[19], s.v[3], q[18] * s.v[0]);
        }
        if (m == 1) {
            return fma(q[21], s.v[3], q[20] * s.v[0]);
        }
        return 0.0;
    }
    __device__ static double inversion(cdp q, const state& s)
    {
        return population(q, s, 1) - population(q, s, 0);
    }
};
using algo_bloch2 = algo_bloch2_t<0>;
using algo_bloch2s = algo_bloch2_t<1>;
using algo_bloch2r = algo_bloch2_t<2>;

/* ---- coherence-vector population readout ------------------------------
 * cv_representation::calc_population
 * (coherence_vector_representation.hpp:289-336). */
template<int N>
__device__ __forceinline__ double cv_population(const double* d, int m)
{
    if constexpr (N == 2) {
        return (m == 0) ? 0.5 - 0.5 * d[2] : 0.5 + 0.5 * d[2];
    } else if constexpr (N == 3) {
        const double s3 = sqrt(3.0);
        if (m == 0) {
            return 1.0 / 3 + 0.5 * (-1.0 * d[6] - 1.0 / s3 * d[7]);
        } else if (m == 1) {
            return 1.0 / 3 + 0.5 * (+1.0 * d[6] - 1.0 / s3 * d[7]);
        } else if (m == 2) {
            return 1.0 / 3 + 0.5 * (+2.0 / s3 * d[7]);
        }
        return 0.0;
    } else {
        double sum = 0.0;
#pragma unroll
        for (int i = 0; i < N - 1; i++) {
            /* -1, m or 0 over sqrt(k), folded: no division at run time */
            const double root = sqrt((double)(((i + 1) * (i + 2)) / 2));
            const double below = -1.0 / root, at = (double)(i + 1) / root;
            const double f = m < i + 1 ? below : (m == i + 1 ? at : 0.0);
            sum += f * d[N * (N - 1) + i];
        }
        return 1.0 / N + 0.5 * sum;
    }
}

/* ======================================================================
 * lindblad_cvr_rodr<N>::update (algo_lindblad_cvr_rodr.hpp:234-268),
 * reference form.  A2 is never materialised: row j of A2 is assembled
 * entry by entry in the reference's accumulation order and consumed
 * immediately, which yields the same floating-point values as building
 * the whole matrix first.
 * ==================================================================== */
template<int N>
struct algo_rodr {
    static constexpr int ROWC_WAVES = 1;
    static constexpr bool CONSTS = false;
    static constexpr bool ROWC = false;
    static constexpr int STAGE = 0;
    static constexpr bool SHIFT = false;
    static constexpr bool FAST_FDTD = false;
    static constexpr int K = N * N - 1;
    static constexpr int B = K / 2;
    static constexpr int DC = K;
    static constexpr int STATE = K;
    struct state {
        double v[STATE];
    };

    static constexpr int OFF_M = 5;
    static constexpr int OFF_U = OFF_M + K * K;
    static constexpr int OFF_U2 = OFF_U + K * K;
    static constexpr int OFF_A1 = OFF_U2 + K * K;
    static constexpr int OFF_V = OFF_A1 + K * K;
    static constexpr int OFF_DEQ = OFF_V + K;
    static constexpr int OFF_DIN = OFF_DEQ + K;
    static constexpr int OFF_TH = OFF_DIN + K;
    static constexpr int OFF_C1 = OFF_TH + B;
    static constexpr int OFF_C2 = OFF_C1 + B * K * K;


    /* only for media with a density */
    __device__ static void update(cdp q, state& s, double e, double& p)
    {
        const double M_CP = q[1];
        const double d_t = q[2];
        cdp M = q + OFF_M;
        cdp A1 = q + OFF_A1;
        cdp v = q + OFF_V;
        cdp d_eq = q + OFF_DEQ;
        cdp d_in = q + OFF_DIN;
        double* d = s.v;

        /* d1 = A1 (d + d_in) - d_in */
        double tmp[K], d1[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            tmp[k] = d[k] + d_in[k];
        }
#pragma unroll
        for (int i = 0; i < K; i++) {
            double acc = A1[i * K] * tmp[0];
#pragma unroll
            for (int k = 1; k < K; k++) {
                acc = acc + A1[i * K + k] * tmp[k];
            }
            d1[i] = acc - d_in[i];
        }

        /* d2 = A2 d1 */
        double d2[K];
        if constexpr (N == 2) {
            cdp U = q + OFF_U;
            cdp U2 = q + OFF_U2;
            const double th1 = q[3];
            double x = th1 * e * d_t;
            double sa = sin(x) / th1;
            double va = (1 - cos(x)) / (th1 * th1);
#pragma unroll
            for (int i = 0; i < K; i++) {
                double acc = 0.0;
#pragma unroll
                for (int k = 0; k < K; k++) {
                    double a2 = sa * U[i * K + k] + va * U2[i * K + k] +
                        ((i == k) ? 1.0 : 0.0);
                    acc = (k == 0) ? a2 * d1[0] : acc + a2 * d1[k];
                }
                d2[i] = acc;
            }
        } else {
            /* planes b >= n_theta have theta = 0 and zero C1, C2 in the
             * blob: their terms are exact zeros and leave A2 unchanged, so
             * every plane is evaluated without a data-dependent branch */
            cdp th = q + OFF_TH;
            double sv[B], vv[B];
#pragma unroll
            for (int b = 0; b < B; b++) {
                double x = th[b] * e * d_t;
                sv[b] = sin(x);
                vv[b] = 1 - cos(x);
            }
            cdp C1 = q + OFF_C1;
            cdp C2 = q + OFF_C2;
            /* rows: unrolled for small K; for large K one row per iteration
             * with the result routed through a compare-select chain so that
             * no register array is indexed dynamically */
            constexpr int ROW_UNROLL = (K <= 8) ? K : 1;
#pragma unroll ROW_UNROLL
            for (int i = 0; i < K; i++) {
                double acc = 0.0;
#pragma unroll
                for (int k = 0; k < K; k++) {
                    double a2 = (i == k) ? 1.0 : 0.0;
#pragma unroll
                    for (int b = 0; b < B; b++) {
                        a2 = a2 +
                            (sv[b] * C1[(b * K + i) * K + k] +
                             vv[b] * C2[(b * K + i) * K + k]);
                    }
                    acc = (k == 0) ? a2 * d1[0] : acc + a2 * d1[k];
                }
#pragma unroll
                for (int kk = 0; kk < K; kk++) {
                    if (kk == i) {
                        d2[kk] = acc;
                    }
                }
            }
        }

        /* d = A1 (d2 + d_in) - d_in */
#pragma unroll
        for (int k = 0; k < K; k++) {
            tmp[k] = d2[k] + d_in[k];
        }
#pragma unroll
        for (int i = 0; i < K; i++) {
            double acc = A1[i * K] * tmp[0];
#pragma unroll
            for (int k = 1; k < K; k++) {
                acc = acc + A1[i * K + k] * tmp[k];
            }
            d[i] = acc - d_in[i];
        }

        /* p = M_CP v^T (M d + d_eq) */
        double pacc = 0.0;
#pragma unroll
        for (int i = 0; i < K; i++) {
            double acc = M[i * K] * d[0];
#pragma unroll
            for (int k = 1; k < K; k++) {
                acc = acc + M[i * K + k] * d[k];
            }
            double w = acc + d_eq[i];
            double t = (M_CP * v[i]) * w;
            pacc = (i == 0) ? t : pacc + t;
        }
        p = pacc;
    }

    template<int C>
    __device__ static void update_multi(cdp q, state* s, const double* e,
                                        double* p)
    {
#pragma unroll
        for (int c = 0; c < C; c++) {
            update(q, s[c], e[c], p[c]);
        }
    }

    /* calc_inversion (algo_lindblad_cvr_rodr.hpp:274-277) */
    __device__ static double inversion(cdp, const state& s)
    {
        return s.v[N * (N - 1)];
    }
    __device__ static double population(cdp, const state& s, int m)
    {
        return cv_population<N>(s.v, m);
    }
};

/* ---- sin/cos for the rotated-basis form --------------------------------
 * Taylor series of sin (to x^13) and cos (to x^14) about 0 in Horner form
 * in x^2; for |x| <= 0.25 the truncation error is below 1e-21 relative. */
constexpr double TAYLOR_MAX = 0.25;

__device__ __forceinline__ void taylor_sincos(double x, double& s, double& c)
{
    const double x2 = x * x;
    double ps = 1.6059043836821614599e-10;        /* 1/13! */
    ps = fma(ps, x2, -2.5052108385441718775e-08); /* -1/11! */
    ps = fma(ps, x2, 2.7557319223985890653e-06);  /* 1/9! */
    ps = fma(ps, x2, -1.9841269841269841270e-04); /* -1/7! */
    ps = fma(ps, x2, 8.3333333333333333333e-03);  /* 1/5! */
    ps = fma(ps, x2, -1.6666666666666666667e-01); /* -1/3! */
    s = fma(ps * x2, x, x);
    double pc = -1.1470745597729724714e-11;       /* -1/14! */
    pc = fma(pc, x2, 2.0876756987868098979e-09);  /* 1/12! */
    pc = fma(pc, x2, -2.7557319223985890653e-07); /* -1/10! */
    pc = fma(pc, x2, 2.4801587301587301587e-05);  /* 1/8! */
    pc = fma(pc, x2, -1.3888888888888888889e-03); /* -1/6! */
    pc = fma(pc, x2, 4.1666666666666666667e-02);  /* 1/4! */
    pc = fma(pc, x2, -0.5);                       /* -1/2! */
    c = fma(pc, x2, 1.0);
}

/* the same coefficients, sin then cos (1/13! .. -1/3!, -1/14! .. 1/4!) */
static __constant__ const double TAYLOR_COEFF[12] = {
    1.6059043836821614599e-10,  -2.5052108385441718775e-08,
    2.7557319223985890653e-06,  -1.9841269841269841270e-04,
    8.3333333333333333333e-03,  -1.6666666666666666667e-01,
    -1.1470745597729724714e-11, 2.0876756987868098979e-09,
    -2.7557319223985890653e-07, 2.4801587301587301587e-05,
    -1.3888888888888888889e-03, 4.1666666666666666667e-02,
};

/* sin and cos of a small angle x, by wave-uniform tier of max |x|:
 * TIER 0: |x| <= 2^-13, x - x^3/6 and 1 - x^2/2 (relative truncation
 * error below 1e-17); TIER 1: |x| <= 2^-10, Taylor to x^5 / x^4 (below
 * 2e-21 / 3e-19); TIER 2: |x| <= 0.25, Taylor to x^13 / x^14; TIER 3:
 * library. */
template<int TIER>
__device__ __forceinline__ void tier_sincos(double x, double& s, double& c)
{
    if constexpr (TIER == 0) {
        const double x2 = x * x;
        s = fma(x * x2, -1.6666666666666666667e-01, x);
        c = fma(x2, -0.5, 1.0);
    } else if constexpr (TIER == 1) {
        const double x2 = x * x;
        s = fma(x * x2, fma(x2, 8.3333333333333333333e-03,
                            -1.6666666666666666667e-01), x);
        c = fma(x2, fma(x2, 4.1666666666666666667e-02, -0.5), 1.0);
    } else if constexpr (TIER == 4) {
        /* |x| <= 2^-5: to x^9 / x^8 (below 1e-22) */
        const double x2 = x * x;
        double ps = fma(x2, 2.7557319223985890653e-06,
                        -1.9841269841269841270e-04);
        ps = fma(ps, x2, 8.3333333333333333333e-03);
        ps = fma(ps, x2, -1.6666666666666666667e-01);
        s = fma(x * x2, ps, x);
        double pc = fma(x2, 2.4801587301587301587e-05,
                        -1.3888888888888888889e-03);
        pc = fma(pc, x2, 4.1666666666666666667e-02);
        pc = fma(pc, x2, -0.5);
        c = fma(pc, x2, 1.0);
    } else if constexpr (TIER == 2) {
        taylor_sincos(x, s, c);
    } else {
        sincos(x, &s, &c);
    }
}

/* ======================================================================
 * lindblad_cvr_rodr<N>::update with A2 applied to the vector instead of
 * assembled.  Each rotation plane b of the dipole Liouvillian is spanned by
 * two orthonormal vectors q1, q2 with C1_b = q2 q1^T - q1 q2^T and
 * C2_b = -(q1 q1^T + q2 q2^T), so with alpha = q1.d, beta = q2.d
 *   A2 d = d + sum_b q1 (-sin beta - (1 - cos) alpha)
 *                  + q2 ( sin alpha - (1 - cos) beta):
 * 4 K FMAs per plane where building A2 takes 4 K^2 operations per plane.
 * The host recovers the vectors from the blob's C1 and C2 and checks that
 * they reproduce both; a blob that is not of this form (and
 * MBH_OPT_GENERIC) takes algo_rodr, which accepts any C1, C2.
 * The half steps are A1 d + c with c = (A1 - I) d_in, and
 * p = pv.d + pb with pv = M_CP v^T M, pb = M_CP v.d_eq.  The basis stays
 * that of the coherence vector, so exact zeros of A1, pv and the planes
 * stay exact (a run that starts from noise has p = 0 until its coherences
 * grow, as in the reference form).  State: d, as algo_rodr.
 * Bound by the latency of one step's chain on grids that leave the SIMDs
 * one wavefront or none; with one wavefront per tile, whole runs, algo_rodr
 * -> algo_rodrp: six-level ladder, 8192 cells x 800 steps, 1702 -> 18.6 ms
 * (algo_rodr: 93 kflop and 10 KB of scratch per lane and step); five-level
 * comb, 8192 x 600, 239 -> 5.3 ms; three levels, 16384 x 8000, 112 -> 16.7
 * ms (11.2 from row registers); one cell, 10000 steps, 102 -> 34 ms.  Few
 * tiles, and six levels in the plain order always, take team_kernel with the
 * same arithmetic.
 *
 * Blob (STRIDE doubles): [0] has_qm  [1] number of planes  [2] pb
 *   [3] max theta dt   then c (K), pv (K), A1 (K^2),
 *   planes: B x { theta dt, q1 (K), q2 (K) }
 * ==================================================================== */
/* sin(x) and 1 - cos(x) of one cell's plane angles, by the cell's own range
 * (the results of a cell do not depend on its neighbours): SMALL |x| <=
 * 2^-5, Taylor to x^9 and x^8 (relative truncation below 1e-18); MEDIUM
 * |x| <= 0.25 (to x^13 / x^14); else the library. */
constexpr double PLANE_SMALL = 0.03125;

__device__ __forceinline__ void plane_small(double x, double& s, double& v)
{
    const double x2 = x * x;
    double ps = 2.7557319223985890653e-06;        /* 1/9! */
    ps = fma(ps, x2, -1.9841269841269841270e-04); /* -1/7! */
    ps = fma(ps, x2, 8.3333333333333333333e-03);  /* 1/5! */
    ps = fma(ps, x2, -1.6666666666666666667e-01); /* -1/3! */
    s = fma(ps * x2, x, x);
    double pc = -2.4801587301587301587e-05;       /* -1/8! */
    pc = fma(pc, x2, 1.3888888888888888889e-03);  /* 1/6! */
    pc = fma(pc, x2, -4.1666666666666666667e-02); /* -1/4! */
    pc = fma(pc, x2, 0.5);                        /* 1/2! */
    v = pc * x2;
}

__device__ __forceinline__ void plane_sincos(double x, bool small, bool medium,
                                             bool all_medium, double& s,
                                             double& v)
{
    plane_small(x, s, v);
    const double x2 = x * x;
    double qs = 1.6059043836821614599e-10;        /* 1/13! */
    qs = fma(qs, x2, -2.5052108385441718775e-08); /* -1/11! */
    qs = fma(qs, x2, 2.7557319223985890653e-06);
    qs = fma(qs, x2, -1.9841269841269841270e-04);
    qs = fma(qs, x2, 8.3333333333333333333e-03);
    qs = fma(qs, x2, -1.6666666666666666667e-01);
    double s2 = fma(qs * x2, x, x);
    double qc = 1.1470745597729724714e-11;        /* 1/14! */
    qc = fma(qc, x2, -2.0876756987868098979e-09); /* -1/12! */
    qc = fma(qc, x2, 2.7557319223985890653e-07);  /* 1/10! */
    qc = fma(qc, x2, -2.4801587301587301587e-05);
    qc = fma(qc, x2, 1.3888888888888888889e-03);
    qc = fma(qc, x2, -4.1666666666666666667e-02);
    qc = fma(qc, x2, 0.5);
    double v2 = qc * x2;
    if (!all_medium) {
        double sl, cl;
        sincos(x, &sl, &cl);
        s2 = medium ? s2 : sl;
        v2 = medium ? v2 : 1.0 - cl;
    }
    s = small ? s : s2;
    v = small ? v : v2;
}

template<int N>
struct algo_rodrp {
    static constexpr bool CONSTS = false;
    static constexpr bool SHIFT = false;
    static constexpr bool FAST_FDTD = false;
    static constexpr int K = N * N - 1;
    static constexpr int B = K / 2;
    static constexpr int DC = K;
    static constexpr int STATE = K;
    static constexpr int ROWC_WAVES = 2;
    struct state {
        double v[STATE];
    };

    static constexpr int OFF_C = 4;
    static constexpr int OFF_PV = OFF_C + K;
    static constexpr int OFF_A1 = OFF_PV + K;
    static constexpr int OFF_PL = OFF_A1 + K * K;
    static constexpr int PLANE = 1 + 2 * K;
    static constexpr int STRIDE = OFF_PL + B * PLANE;

    static constexpr int STAGE = 0;


    /* o = A1 d + c: every row accumulates in ascending order; RG rows side
     * by side hide the FMA latency (more would spill at K = 35) */
    template<int C, typename P>
    __device__ static void half_step(P q, const double (*d)[K],
                                     double (*o)[K])
    {
        const P c0 = q + OFF_C;
        const P A1 = q + OFF_A1;
        constexpr int RG = C != 1 ? 1 : (K <= 8 ? K : (K <= 24 ? 4 : 2));
#pragma unroll
        for (int i0 = 0; i0 < K; i0 += RG) {
            double acc[C][RG];
#pragma unroll
            for (int g = 0; g < RG; g++) {
                if (i0 + g < K) {
                    const double ci = c0[i0 + g];
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        acc[c][g] = ci;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < K; k++) {
#pragma unroll
                for (int g = 0; g < RG; g++) {
                    if (i0 + g < K) {
                        const double a = A1[(i0 + g) * K + k];
#pragma unroll
                        for (int c = 0; c < C; c++) {
                            acc[c][g] = fma(a, d[c][k], acc[c][g]);
                        }
                    }
                }
            }
#pragma unroll
            for (int g = 0; g < RG; g++) {
                if (i0 + g < K) {
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        o[c][i0 + g] = acc[c][g];
                    }
                }
            }
        }
    }

    template<int C, typename P>
    __device__ static void update_multi_p(P q, state* s, const double* e,
                                          double* p)
    {
        double d[C][K], r[C][K];
#pragma unroll
        for (int c = 0; c < C; c++) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                r[c][k] = s[c].v[k];
            }
        }
        bool small[C], medium[C];
        bool all_s = true, all_m = true;
#pragma unroll
        for (int c = 0; c < C; c++) {
            const double xm = q[3] * fabs(e[c]);
            small[c] = xm <= PLANE_SMALL;
            medium[c] = xm <= TAYLOR_MAX;
            all_s = all_s && small[c];
            all_m = all_m && medium[c];
        }
        all_s = __all(all_s);
        all_m = __all(all_m);
        const int np = (int)q[1];
        /* one copy of the half step in a loop of two; the offset that the
         * compiler cannot see through keeps A1's loads inside (kept for
         * the second half, A1 would spill) */
#pragma unroll 1
        for (int half = 0;; half++) {
            int off = 0;
            asm volatile("" : "+s"(off));
            half_step<C>(q + off, r, d);
            if (half == 1) {
                break;
            }
            /* the planes: r = A2 d */
#pragma unroll
            for (int c = 0; c < C; c++) {
#pragma unroll
                for (int k = 0; k < K; k++) {
                    r[c][k] = d[c][k];
                }
            }
            P pl = q + off + OFF_PL;
#pragma unroll 1
            for (int b = 0; b < np; b++, pl += PLANE) {
                const P q1 = pl + 1;
                const P q2 = pl + 1 + K;
                double u1[C], u2[C];
#pragma unroll
                for (int c = 0; c < C; c++) {
                    double al = 0.0, be = 0.0;
#pragma unroll
                    for (int k = 0; k < K; k++) {
                        al = fma(q1[k], d[c][k], al);
                        be = fma(q2[k], d[c][k], be);
                    }
                    double sn, vc;
                    if (all_s) {
                        plane_small(pl[0] * e[c], sn, vc);
                    } else {
                        plane_sincos(pl[0] * e[c], small[c], medium[c],
                                     all_m, sn, vc);
                    }
                    u1[c] = fma(-sn, be, -(vc * al));
                    u2[c] = fma(sn, al, -(vc * be));
                }
#pragma unroll
                for (int k = 0; k < K; k++) {
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        r[c][k] =
                            fma(q1[k], u1[c], fma(q2[k], u2[c], r[c][k]));
                    }
                }
            }
        }
        const P pv = q + OFF_PV;
#pragma unroll
        for (int c = 0; c < C; c++) {
            double acc = q[2];
#pragma unroll
            for (int k = 0; k < K; k++) {
                s[c].v[k] = d[c][k];
                acc = fma(pv[k], d[c][k], acc);
            }
            p[c] = acc;
        }
    }

    /* one cell per lane, three levels: the same step with the constants
     * from row registers (more levels would spill) */
    static constexpr bool ROWC = N == 3;
    static constexpr int NC = STRIDE - OFF_C;
    struct rowc {
        row_consts<NC> k;
        double th[B], thmax, pb;
        int np;
        cdp q;
        __device__ void load(cdp qs, const double* q)
        {
            this->q = qs;
            k.load(q + OFF_C);
#pragma unroll
            for (int b = 0; b < B; b++) {
                th[b] = q[OFF_PL + b * PLANE];
            }
            pb = q[2];
            thmax = q[3];
            np = (int)qs[1];
        }
    };
    __device__ __forceinline__ static void rows_half(const rowc& R, const double* d, double* o)
    {
        static_for<K>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            double acc = R.k.template get<i>();
            static_for<K>([&](auto k_) __attribute__((always_inline)) {
                constexpr int kk = decltype(k_)::value;
                R.k.template fmac<2 * K + i * K + kk>(acc, d[kk]);
            });
            o[i] = acc;
        });
    }
    __device__ __forceinline__ static void apply_rows(rowc& R, state& s, double e, double& p,
                                      bool mine)
    {
        R.k.pin();
        double d[K], r[K];
        rows_half(R, s.v, d);
        const double xm = R.thmax * fabs(e);
        const bool small = xm <= PLANE_SMALL, medium = xm <= TAYLOR_MAX;
        const bool all_s = __all(small || !mine);
        const bool all_m = __all(medium || !mine);
        /* the wide ranges of the angle in a rolled loop (one copy of the
         * library function; unrolled, its registers would halve the
         * wavefronts per SIMD) */
        double sn[B], vc[B];
        if (all_s) {
#pragma unroll
            for (int b = 0; b < B; b++) {
                plane_small(R.th[b] * e, sn[b], vc[b]);
            }
        } else {
            double ws[B], wv[B];
#pragma unroll 1
            for (int b = 0; b < B; b++) {
                plane_sincos(R.q[OFF_PL + b * PLANE] * e, small, medium,
                             all_m, ws[b], wv[b]);
            }
#pragma unroll
            for (int b = 0; b < B; b++) {
                sn[b] = ws[b];
                vc[b] = wv[b];
            }
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            r[k] = d[k];
        }
        static_for<B>([&](auto b_) __attribute__((always_inline)) {
            constexpr int b = decltype(b_)::value;
            constexpr int Q1 = 2 * K + K * K + b * PLANE + 1, Q2 = Q1 + K;
            if (b < R.np) {
                double al = 0.0, be = 0.0;
                static_for<K>([&](auto k_) __attribute__((always_inline)) {
                    constexpr int kk = decltype(k_)::value;
                    R.k.template fmac<Q1 + kk>(al, d[kk]);
                    R.k.template fmac<Q2 + kk>(be, d[kk]);
                });
                const double u1 = fma(-sn[b], be, -(vc[b] * al));
                const double u2 = fma(sn[b], al, -(vc[b] * be));
                static_for<K>([&](auto k_) __attribute__((always_inline)) {
                    constexpr int kk = decltype(k_)::value;
                    R.k.template fmac<Q2 + kk>(r[kk], u2);
                    R.k.template fmac<Q1 + kk>(r[kk], u1);
                });
            }
        });
        rows_half(R, r, s.v);
        double acc = R.pb;
        static_for<K>([&](auto k_) __attribute__((always_inline)) {
            constexpr int kk = decltype(k_)::value;
            R.k.template fmac<K + kk>(acc, s.v[kk]);
        });
        p = acc;
    }

    template<int C>
    __device__ static void update_multi(cdp q, state* s, const double* e,
                                        double* p)
    {
        update_multi_p<C>(q, s, e, p);
    }
    __device__ static void update(cdp q, state& s, double e, double& p)
    {
        update_multi<1>(q, &s, &e, &p);
    }

    __device__ static double inversion(cdp, const state& s)
    {
        return s.v[N * (N - 1)];
    }
    __device__ static double population(cdp, const state& s, int m)
    {
        return cv_population<N>(s.v, m);
    }
};

/* ======================================================================
 * Rodrigues in the rotated basis (z-form).  Mathematically identical to
 * algo_rodr (A2(e) = Q R(e) Q^T, Strang halves merged into W); see the
 * zform blob description in mbsolve_hip.h.  State: y (K values).
 * ==================================================================== */
template<int N>
struct algo_zform {
    static constexpr int ROWC_WAVES = N <= 3 ? 3 : 2;
    static constexpr bool CONSTS = false;
    static constexpr bool FAST_FDTD = true;
    static constexpr int K = N * N - 1;
    static constexpr int B = K / 2;
    static constexpr int DC = K;
    static constexpr int STATE = K;
    struct state {
        double v[STATE];
    };

    static constexpr int OFF_TH = 3;
    static constexpr int OFF_W = OFF_TH + B;
    static constexpr int OFF_C = OFF_W + K * K;
    static constexpr int OFF_A = OFF_C + K;
    static constexpr int OFF_P = OFF_A + K;
    static constexpr int OFF_O = OFF_P + K * K;
    static constexpr int OFF_QT = OFF_O + K;
    static constexpr int OFF_QTA1 = OFF_QT + K * K;
    static constexpr int OFF_DIN = OFF_QTA1 + K * K;
    /* appended to the device copy of the blob (not part of the C ABI
     * layout): y* = -Qt d_in, the fixed point of the step at zero field
     * (d = -d_in, the relaxation equilibrium).  FP32 storage holds
     * y - y*, so its rounding scales with the distance from equilibrium
     * instead of with |y*|. */
    static constexpr int OFF_YEQ = OFF_DIN + K;
    /* and, for the records, the populations as linear forms of y:
     * rho_mm = r_m . y + o_m, N rows of (r_m, o_m) */
    static constexpr int OFF_POP = OFF_YEQ + K;
    static constexpr int DEV_STRIDE = OFF_POP + N * (K + 1);
    static constexpr bool SHIFT = true;


    /* Small blobs (K <= 8) are staged in LDS by the tile kernel: W, c, a
     * and theta are then read from there every step instead of through
     * the scalar cache (their 600 bytes do not fit the SGPRs). */
    static constexpr int STAGE = (K <= 8) ? OFF_A + K : 0;

    template<int C>
    __device__ static void update_multi(cdp q, state* s, const double* e,
                                        double* p)
    {
        update_multi_p<C>(q, s, e, p);
    }

    /* C cells of one material: straight-line code with the cell index
     * innermost, so the independent chains interleave.  Planes beyond
     * n_theta have angle 0 (identity rotation, exact). */
    template<int C, typename P>
    __device__ static void update_multi_p(P q, state* s, const double* e,
                                          double* p)
    {
        const P th = q + OFF_TH;
        const P W = q + OFF_W;
        const P cv = q + OFF_C;
        const P a = q + OFF_A;

        double sn[C][B], cs[C][B];
        bool t0 = true, t1 = true, t2 = true;
#pragma unroll
        for (int c = 0; c < C; c++) {
#pragma unroll
            for (int b = 0; b < B; b++) {
                const double x = th[b] * e[c];
                const double ax = fabs(x);
                sn[c][b] = x;
                t0 = t0 && (ax <= 0x1p-13);
                t1 = t1 && (ax <= 0x1p-10);
                t2 = t2 && (ax <= TAYLOR_MAX);
            }
        }
        /* wave-uniform tier: the cheapest series accurate for every
         * angle of the wavefront */
        auto all_sincos = [&](auto tier) {
            constexpr int T = decltype(tier)::value;
#pragma unroll
            for (int c = 0; c < C; c++) {
#pragma unroll
                for (int b = 0; b < B; b++) {
                    tier_sincos<T>(sn[c][b], sn[c][b], cs[c][b]);
                }
            }
        };
        if (__all(t0)) {
            all_sincos(std::integral_constant<int, 0>());
        } else if (__all(t1)) {
            all_sincos(std::integral_constant<int, 1>());
        } else if (__all(t2)) {
            all_sincos(std::integral_constant<int, 2>());
        } else {
            all_sincos(std::integral_constant<int, 3>());
        }

        /* r = R(e) y */
        double r[C][K];
#pragma unroll
        for (int c = 0; c < C; c++) {
#pragma unroll
            for (int k = 2 * B; k < K; k++) {
                r[c][k] = s[c].v[k];
            }
#pragma unroll
            for (int b = 0; b < B; b++) {
                const double y0 = s[c].v[2 * b], y1 = s[c].v[2 * b + 1];
                r[c][2 * b] = fma(cs[c][b], y0, -(sn[c][b] * y1));
                r[c][2 * b + 1] = fma(sn[c][b], y0, cs[c][b] * y1);
            }
        }
        /* p = a . r + b, two interleaved partial sums */
        double pa[C], pb[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            pa[c] = q[2];
            pb[c] = 0.0;
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            const double ak = a[k];
#pragma unroll
            for (int c = 0; c < C; c++) {
                if (k & 1) {
                    pb[c] = fma(ak, r[c][k], pb[c]);
                } else {
                    pa[c] = fma(ak, r[c][k], pa[c]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < C; c++) {
            p[c] = pa[c] + pb[c];
        }
        /* y' = W r + c.  With one cell per lane and a small blob (K <= 8,
         * read from LDS) the rows are accumulated side by side (k outer):
         * K independent FMA chains instead of one chain per row after
         * another, at the price of holding W in VGPRs during the product.
         * Larger K (the 35 components of six levels) interleaves two rows:
         * half the chain latency without spilling to AGPRs (three rows
         * do).  Several cells per lane already interleave C chains. */
        constexpr int RG = C != 1 ? 1 : (K <= 8 ? K : 2);
#pragma unroll
        for (int i0 = 0; i0 < K; i0 += RG) {
            double acc[C][RG];
#pragma unroll
            for (int g = 0; g < RG; g++) {
                if (i0 + g < K) {
                    const double ci = cv[i0 + g];
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        acc[c][g] = ci;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < K; k++) {
#pragma unroll
                for (int g = 0; g < RG; g++) {
                    if (i0 + g < K) {
                        const double w = W[(i0 + g) * K + k];
#pragma unroll
                        for (int c = 0; c < C; c++) {
                            acc[c][g] = fma(w, r[c][k], acc[c][g]);
                        }
                    }
                }
            }
#pragma unroll
            for (int g = 0; g < RG; g++) {
                if (i0 + g < K) {
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        s[c].v[i0 + g] = acc[c][g];
                    }
                }
            }
        }
    }

    __device__ static void update(cdp q, state& s, double e, double& p)
    {
        update_multi<1>(q, &s, &e, &p);
    }

    /* one cell per lane, three and four levels: the same step with W, c and
     * a from row registers (five levels would spill at two wavefronts per
     * SIMD) */
    static constexpr bool ROWC = N == 3 || N == 4;
    static constexpr int NC = K * K + 2 * K;
    struct rowc {
        row_consts<NC> k; /* W, c, a */
        double th[B], thmax, b;
        cdp q;
        __device__ void load(cdp qs, const double* q)
        {
            this->q = qs;
            k.load(q + OFF_W);
            thmax = 0.0;
#pragma unroll
            for (int i = 0; i < B; i++) {
                th[i] = q[OFF_TH + i];
                thmax = fmax(thmax, fabs(th[i]));
            }
            b = q[2];
        }
    };
    __device__ __forceinline__ static void apply_rows(rowc& R, state& s, double e, double& p,
                                      bool mine)
    {
        R.k.pin();
        double sn[B], cs[B], r[K];
        /* wave-uniform tier, as in update_multi_p.  Up to 0.25 its series (on
         * a field of 0.12 per step, 262144 cells of three levels, 1000 steps,
         * 5.71 -> 3.37 ms against the library function); three levels take
         * it from 2^-10 on, a tier less in the chain of tests (16384 cells,
         * weak field, 4000 steps 3.13 -> 2.82 ms).  The library function in
         * a rolled loop (one copy; unrolled, its registers would halve the
         * wavefronts per SIMD). */
        const double xm = mine ? R.thmax * fabs(e) : 0.0;
        auto tier = [&](auto t) {
#pragma unroll
            for (int b = 0; b < B; b++) {
                tier_sincos<decltype(t)::value>(R.th[b] * e, sn[b], cs[b]);
            }
        };
        if (__all(xm <= 0x1p-13)) {
            tier(std::integral_constant<int, 0>());
        } else if (__all(xm <= 0x1p-10)) {
            tier(std::integral_constant<int, 1>());
        } else if (N > 3 && __all(xm <= 0x1p-5)) {
            tier(std::integral_constant<int, 4>());
        } else if (__all(xm <= TAYLOR_MAX)) {
            /* (coefficients from memory, by an address that the compiler
             * cannot see through: as literals they would be kept in
             * registers over the steps) */
            int off = 0;
            asm volatile("" : "+s"(off));
            cdp tc = (cdp)TAYLOR_COEFF + off;
#pragma unroll
            for (int b = 0; b < B; b++) {
                const double x = R.th[b] * e, x2 = x * x;
                double ps = tc[0], pc = tc[6];
#pragma unroll
                for (int i = 1; i < 6; i++) {
                    ps = fma(ps, x2, tc[i]);
                    pc = fma(pc, x2, tc[6 + i]);
                }
                pc = fma(pc, x2, -0.5);
                sn[b] = fma(ps * x2, x, x);
                cs[b] = fma(pc, x2, 1.0);
            }
        } else {
            double ws[B], wc[B];
#pragma unroll 1
            for (int b = 0; b < B; b++) {
                sincos(R.q[OFF_TH + b] * e, &ws[b], &wc[b]);
            }
#pragma unroll
            for (int b = 0; b < B; b++) {
                sn[b] = ws[b];
                cs[b] = wc[b];
            }
        }
#pragma unroll
        for (int k = 2 * B; k < K; k++) {
            r[k] = s.v[k];
        }
#pragma unroll
        for (int b = 0; b < B; b++) {
            const double y0 = s.v[2 * b], y1 = s.v[2 * b + 1];
            r[2 * b] = fma(cs[b], y0, -(sn[b] * y1));
            r[2 * b + 1] = fma(sn[b], y0, cs[b] * y1);
        }
        double pa = R.b, pb = 0.0;
        static_for<K>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            R.k.template fmac<K * K + K + i>(i & 1 ? pb : pa, r[i]);
        });
        p = pa + pb;
        static_for<K>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            s.v[i] = R.k.template get<K * K + i>();
        });
        static_for<K>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            static_for<K>([&](auto k_) __attribute__((always_inline)) {
                constexpr int kk = decltype(k_)::value;
                R.k.template fmac<i * K + kk>(s.v[i], r[kk]);
            });
        });
    }

    /* component k of the reference coherence vector after the step */
    __device__ static double dcomp(cdp q, const state& s, int k)
    {
        cdp P = q + OFF_P;
        cdp o = q + OFF_O;
        double acc = o[k];
#pragma unroll
        for (int j = 0; j < K; j++) {
            acc = fma(P[k * K + j], s.v[j], acc);
        }
        return acc;
    }
    __device__ static double inversion(cdp q, const state& s)
    {
        if (q[0] == 0.0) {
            return 0.0;
        }
        return dcomp(q, s, N * (N - 1));
    }
    __device__ static double population(cdp q, const state& s, int m)
    {
        cdp r = q + OFF_POP + (uint64_t)m * (K + 1);
        double acc = r[K];
#pragma unroll
        for (int j = 0; j < K; j++) {
            acc = fma(r[j], s.v[j], acc);
        }
        return acc;
    }
};

} /* namespace mbh */

#endif
