/*
 * FP64 Rodrigues by rotation planes (algo_rodrp) with the rows of a cell's
 * coherence vector split over the W wavefronts of a workgroup, for grids that
 * leave most of the chip idle with one wavefront per tile.
 *
 * All W wavefronts hold the same 64 cells, one per lane, and each updates E
 * and H of all of them (some twenty instructions).  Of a step's density update
 *   t = A1 d + c,  al_b = q1_b . t,  be_b = q2_b . t,
 *   r = t + sum_b (q1_b u1_b + q2_b u2_b),  d' = A1 r + c
 * wavefront w computes the rows [w R, (w + 1) R) of t, r and d' and the planes
 * w, w + W, ..; d, t, the u's and r pass through LDS, four barriers per step.
 * Every sum runs over the same operands in the same order as in algo_rodrp,
 * so the results are the same bit for bit and the choice between the two
 * kernels does not show.
 *
 * What bounds it: the FP64 instructions of one wavefront (K = 35: some 5600 in
 * algo_rodrp, 1650 here) and the four exchanges, some 200 cycles each.  A
 * wavefront's share of A1 and of the planes fits its registers, sixteen
 * constants to a register pair (row_consts), where algo_rodrp reads all of
 * them (K = 35: 19 KB, more than the scalar cache holds) in every step.  Each
 * wavefront writes every W-th record (with all in the first, one cell with
 * four records per step took 2.07 instead of 1.57 us per step).  Whole runs on
 * one tile per CU, one wavefront / team: K = 35, 800 steps 19.6 / 5.5 ms;
 * K = 24, 600 steps 5.3 / 2.2 ms; K = 8, one cell, 10000 steps 23.6 / 15.7 ms.
 */
#ifndef MBH_TEAM_HPP
#define MBH_TEAM_HPP

#include "mbh_tile.hpp"

namespace mbh {

/* Wavefronts per tile.  One tile per CU, us per step with 1 (algo_rodrp) and
 * with 2, 4 .. 8 wavefronts: K = 8 1.52, -, 1.17, 8: 1.2; K = 15 5.24, 4:
 * 3.25, 5: 3.34, 8: 3.16 (and 5.1 instead of 3.4 with two tiles per CU);
 * K = 24 8.8, 4: 4.40, 6: 4.33, 8: 4.33; K = 35 24.4, 4: 7.75, 7: 8.2, 8: 8.4
 * (four hold 128 registers of constants each and use one SIMD each). */
template<int N>
constexpr int team_waves()
{
    return N == 5 ? 6 : 4;
}

template<int N>
struct team_consts {
    typedef algo_rodrp<N> A;
    static constexpr int K = A::K, B = A::B, W = team_waves<N>();
    static constexpr int R = (K + W - 1) / W;  /* rows of a wavefront */
    static constexpr int PB = (B + W - 1) / W; /* planes of a wavefront */
    static constexpr int Q_ROWS = 0;                /* A1: [R][K] */
    static constexpr int Q_C = Q_ROWS + R * K;      /* c: [R] */
    static constexpr int Q_Q = Q_C + R;             /* q1, q2: [2 B][R] */
    static constexpr int Q_PLANE = Q_Q + 2 * B * R; /* [PB][1 + 2 K] */
    static constexpr int Q_PV = Q_PLANE + PB * A::PLANE; /* [K] */
    static constexpr int NC = Q_PV + K;

    row_consts<NC> k;
    double thmax, pb;
    int np;

    /* the wavefronts' constants follow the material's blob, 16 NR each */
    static constexpr int NW = 16 * row_consts<NC>::NR;
    static constexpr int STRIDE = A::STRIDE + W * NW;

    /* constant i of wavefront w in the blob of algo_rodrp (rows and planes
     * beyond the last repeat it; their results are not used) */
    static int at(int i, int w)
    {
        if (i >= Q_PV) {
            const int j = i - Q_PV;
            return A::OFF_PV + (j < K ? j : K - 1);
        }
        if (i >= Q_PLANE) {
            const int b = (i - Q_PLANE) / A::PLANE * W + w;
            return A::OFF_PL + (b < B ? b : B - 1) * A::PLANE +
                (i - Q_PLANE) % A::PLANE;
        }
        const bool q = i >= Q_Q, c = i >= Q_C;
        const int r = w * R + (q ? (i - Q_Q) % R : (c ? i - Q_C : i / K));
        const int row = r < K ? r : K - 1;
        if (q) {
            const int j = (i - Q_Q) / R;
            return A::OFF_PL + (j >> 1) * A::PLANE + 1 + (j & 1) * K + row;
        }
        return c ? A::OFF_C + row : A::OFF_A1 + row * K + i % K;
    }
    static void fill(double* o)
    {
        for (int w = 0; w < W; w++) {
            for (int i = 0; i < NW; i++) {
                o[A::STRIDE + w * NW + i] = o[at(i, w)];
            }
        }
    }
    __device__ __forceinline__ void load(cdp qs, const double* q, int w)
    {
        k.load(q + A::STRIDE + w * NW);
        pb = qs[2];
        thmax = qs[3];
        np = (int)qs[1];
    }
};

/* use(i, S[i][lane]) for i = 0 .. M - 1, eight LDS reads ahead of their use
 * (all of them ahead would take 2 M registers) */
template<int M, typename F>
__device__ __forceinline__ void team_pass(const double (*S)[64], int lane,
                                          F&& use)
{
    constexpr int CH = 8;
    double x[CH], y[CH];
#pragma unroll
    for (int i = 0; i < CH && i < M; i++) {
        x[i] = S[i][lane];
    }
    static_for<(M + CH - 1) / CH>([&](auto c_) __attribute__((always_inline)) {
        constexpr int i0 = decltype(c_)::value * CH;
#pragma unroll
        for (int i = 0; i < CH && i0 + CH + i < M; i++) {
            y[i] = S[i0 + CH + i][lane];
        }
        __builtin_amdgcn_sched_barrier(0);
        static_for<(M - i0 < CH ? M - i0 : CH)>(
            [&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value;
                use(std::integral_constant<int, i0 + i>(), x[i]);
            });
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < CH && i0 + CH + i < M; i++) {
            x[i] = y[i];
        }
    });
}

template<int N>
__global__ __launch_bounds__(64 * team_waves<N>()) void team_kernel(KArgs k)
{
    typedef algo_rodrp<N> A;
    typedef team_consts<N> T;
    constexpr int K = T::K, B = T::B, W = T::W, R = T::R, PB = T::PB;
    __shared__ tile_lds lds;
    __shared__ double s_d[K][64];     /* d */
    __shared__ double s_t[K][64];     /* t, then r */
    __shared__ double s_u[2 * B][64]; /* u1, u2 of every plane */

    const uint64_t t = k.tile_list ? k.tile_list[blockIdx.x] : blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int wv =
        __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int row0 = wv * R; /* rows of this wavefront: [row0, row0 + R) */
    const int64_t own_lo = (int64_t)(t * k.owned);
    const int64_t own_hi =
        ((own_lo + (int64_t)k.owned) < (int64_t)k.Gown) ? own_lo + k.owned
                                                         : (int64_t)k.Gown;
    const int64_t tile0 = own_lo - (int64_t)k.halo;
    const int64_t g = tile0 + lane;
    const uint64_t n0 = *as_const(k.n_base) + k.n_off;
    const uint32_t nsteps = k.nsteps;
    const tile_meta M{ as_const(k.tiles)[t].src_lo,
                       as_const(k.tiles)[t].src_hi,
                       as_const(k.tiles)[t].rec_lo,
                       as_const(k.tiles)[t].rec_hi };

    /* state, as in tile_body */
    const bool in = (g >= 0) && (g < (int64_t)k.G);
    const uint64_t gc = in ? (uint64_t)g : 0u;
    const int32_t mv = k.mat[gc];
    const uint8_t hv = k.hzero[gc];
    const double ev = ld<double>(k.e_in, gc);
    const double hv2 = ld<double>(k.h_in, gc);
    const double pv = ld<double>(k.p_in, gc);
    double d[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
        const int row = row0 + i < K ? row0 + i : K - 1;
        d[i] = ld<double>(k.d_in, (uint64_t)row * k.dstride + gc);
    }
    const int32_t m = in ? mat_of(mv) : -1;
    const int32_t ma = (in && mv >= 0 && (mv & MAT_QM) != 0) ? m : -1;
    const bool hz = in ? (hv != 0) : true;
    double e = in ? ev : 0.0;
    double h = (in && (g + 1 < (int64_t)k.G || n0 == 0)) ? hv2 : 0.0;
    double p = in ? pv : 0.0;
#pragma unroll
    for (int i = 0; i < R; i++) {
        d[i] = in ? d[i] : 0.0;
    }
    const dev_record rec_own = own_record(k, M, lane);
    const tile_sources srcs = stage_sources<true>(k, lds, lane, wv == 0,
                                                  M, tile0, n0, nsteps);
    const double* f = k.fdtd + (uint64_t)(m < 0 ? 0 : m) * FDTD_STRIDE;
    const double fa = f[0], fb = f[1], fg = f[3], fx = f[4];
    const double fc = m < 0 ? 0.0 : f[2];

    /* m1: the tile's first material with a density; others: lanes with
     * another one (the same in every wavefront) */
    const unsigned long long act = __ballot(ma >= 0);
    const int32_t m1 =
        act ? __builtin_amdgcn_readlane(ma, __builtin_ctzll(act)) : -1;
    const bool full1 = m1 >= 0 && __all(ma == m1);
    const unsigned long long others = __ballot(ma >= 0 && ma != m1);

    const uint64_t rec_steps = stage_records(
        k, lds.rec, rec_own, lane, wv == 0, M, own_lo, own_hi, n0, nsteps);

    T q;
    auto load_rows = [&](int32_t mm) __attribute__((always_inline)) {
        const uint64_t o = (uint64_t)(mm < 0 ? 0 : mm) * k.qstride;
        q.load((cdp)k.qm + o, (const double*)k.qm + o, wv);
    };
    load_rows(m1);

    double own[R]; /* this wavefront's rows of t */
    /* t = A1 d + c, and p from d if P */
    auto first_half = [&](auto with_p, bool mine)
        __attribute__((always_inline)) {
        constexpr bool P = decltype(with_p)::value;
        q.k.pin();
        double acc = q.pb;
        static_for<R>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            own[i] = q.k.template get<T::Q_C + i>();
        });
        team_pass<K>(s_d, lane, [&](auto k_, double x)
                                    __attribute__((always_inline)) {
            constexpr int kk = decltype(k_)::value;
            if constexpr (P) {
                q.k.template fmac<T::Q_PV + kk>(acc, x);
            }
            static_for<R>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value;
                q.k.template fmac<T::Q_ROWS + i * K + kk>(own[i], x);
            });
        });
        if constexpr (P) {
            p = mine ? acc : p;
        }
        static_for<R>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            if (row0 + i < K) {
                s_t[row0 + i][lane] = own[i];
            }
        });
    };
    auto planes = [&](bool mine) __attribute__((always_inline)) {
        q.k.pin();
        double al[PB], be[PB];
#pragma unroll
        for (int j = 0; j < PB; j++) {
            al[j] = be[j] = 0.0;
        }
        team_pass<K>(s_t, lane, [&](auto k_, double x)
                                    __attribute__((always_inline)) {
            constexpr int kk = decltype(k_)::value;
            static_for<PB>([&](auto j_) __attribute__((always_inline)) {
                constexpr int j = decltype(j_)::value;
                constexpr int Q1 = T::Q_PLANE + j * A::PLANE + 1;
                q.k.template fmac<Q1 + kk>(al[j], x);
                q.k.template fmac<Q1 + K + kk>(be[j], x);
            });
        });
        const double xm = q.thmax * fabs(e);
        const bool small = xm <= PLANE_SMALL, medium = xm <= TAYLOR_MAX;
        const bool all_s = __all(small || !mine);
        const bool all_m = __all(medium || !mine);
        double x[PB], sn[PB] = {}, vc[PB] = {};
        static_for<PB>([&](auto j_) __attribute__((always_inline)) {
            constexpr int j = decltype(j_)::value;
            x[j] = q.k.template get<T::Q_PLANE + j * A::PLANE>() * e;
        });
        if (all_s) {
#pragma unroll
            for (int j = 0; j < PB; j++) {
                plane_small(x[j], sn[j], vc[j]);
            }
        } else {
            /* (one copy, its constants not kept over the steps) */
#pragma unroll 1
            for (int j = 0; j < PB; j++) {
                double xj = x[0], sj, vj;
#pragma unroll
                for (int i = 1; i < PB; i++) {
                    xj = i == j ? x[i] : xj;
                }
                plane_sincos(xj, small, medium, all_m, sj, vj);
#pragma unroll
                for (int i = 0; i < PB; i++) {
                    sn[i] = i == j ? sj : sn[i];
                    vc[i] = i == j ? vj : vc[i];
                }
            }
        }
#pragma unroll
        for (int j = 0; j < PB; j++) {
            const int b = j * W + wv;
            if (b < q.np) {
                s_u[2 * b][lane] = fma(-sn[j], be[j], -(vc[j] * al[j]));
                s_u[2 * b + 1][lane] = fma(sn[j], al[j], -(vc[j] * be[j]));
            }
        }
    };
    /* r = A2 t, own rows (own: t, then r) */
    auto rotate = [&]() __attribute__((always_inline)) {
        q.k.pin();
        constexpr int CB = 4; /* planes per group of LDS reads */
        static_for<(B + CB - 1) / CB>([&](auto c_)
                                          __attribute__((always_inline)) {
            constexpr int b0 = decltype(c_)::value * CB;
            if (b0 < q.np) {
                double u[2 * CB];
#pragma unroll
                for (int i = 0; i < 2 * CB; i++) {
                    const int b = b0 + i / 2;
                    u[i] = b < B ? s_u[2 * b + (i & 1)][lane] : 0.0;
                }
                static_for<CB>([&](auto b_) __attribute__((always_inline)) {
                    constexpr int bi = decltype(b_)::value, b = b0 + bi;
                    if constexpr (b < B) {
                        if (b < q.np) {
                            static_for<R>([&](auto i_)
                                              __attribute__((always_inline)) {
                                constexpr int i = decltype(i_)::value;
                                q.k.template fmac<T::Q_Q + (2 * b + 1) * R +
                                                  i>(own[i], u[2 * bi + 1]);
                            });
                            static_for<R>([&](auto i_)
                                              __attribute__((always_inline)) {
                                constexpr int i = decltype(i_)::value;
                                q.k.template fmac<T::Q_Q + 2 * b * R + i>(
                                    own[i], u[2 * bi]);
                            });
                        }
                    }
                });
            }
        });
        static_for<R>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            if (row0 + i < K) {
                s_t[row0 + i][lane] = own[i];
            }
        });
    };
    /* d' = A1 r + c, own rows */
    auto second_half = [&](bool mine) __attribute__((always_inline)) {
        q.k.pin();
        static_for<R>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            own[i] = q.k.template get<T::Q_C + i>();
        });
        team_pass<K>(s_t, lane, [&](auto k_, double x)
                                    __attribute__((always_inline)) {
            constexpr int kk = decltype(k_)::value;
            static_for<R>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value;
                q.k.template fmac<T::Q_ROWS + i * K + kk>(own[i], x);
            });
        });
#pragma unroll
        for (int i = 0; i < R; i++) {
            d[i] = mine ? own[i] : d[i];
        }
    };
    auto share_d = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < R; i++) {
            if (row0 + i < K) {
                s_d[row0 + i][lane] = d[i];
            }
        }
        __syncthreads();
    };
    const std::true_type with_p;
    const std::false_type without_p;

    share_d();
    if (m1 >= 0 && others == 0ull) {
        first_half(without_p, true);
    }
    for (uint32_t s = 0; s < nsteps; s++) {
        /* E and H (every wavefront), as in tile_body */
        const double h_right = from_right(h);
        double en = (m >= 0) ? fa * e + fb * (-fg * p + (h_right - h) * fx)
                             : 0.0;
        for_sources<true>(k, lds, srcs, tile0, n0, s,
                          [&](int32_t at, bool hard, double v)
                              __attribute__((always_inline)) {
                              const double x = hard ? v : en + v;
                              en = at == lane ? x : en;
                          });
        const double e_left = from_left(en);
        h = hz ? 0.0 : h + fc * (en - e_left);
        e = en;
        if (m1 >= 0) {
            unsigned long long left = others;
            for (int32_t mm = m1;;) {
                const bool mine = full1 || ma == mm;
                if (others != 0ull) {
                    load_rows(mm);
                    first_half(without_p, mine);
                }
                __syncthreads();
                planes(mine);
                __syncthreads();
                rotate();
                __syncthreads();
                second_half(mine);
                if (left == 0ull) {
                    break;
                }
                /* the next material writes t where r is still read */
                __syncthreads();
                mm = __builtin_amdgcn_readlane(ma, __builtin_ctzll(left));
                left &= ~__ballot(ma == mm);
            }
            share_d();
            /* p, and the next step's t */
            if (others == 0ull) {
                first_half(with_p, full1 || ma == m1);
            } else {
                left = others;
                for (int32_t mm = m1;;) {
                    load_rows(mm);
                    first_half(with_p, ma == mm);
                    if (left == 0ull) {
                        break;
                    }
                    mm = __builtin_amdgcn_readlane(ma, __builtin_ctzll(left));
                    left &= ~__ballot(ma == mm);
                }
            }
        }
        if ((rec_steps >> s) & 1ull) {
            for_due_records<W>(
                k, lds.rec, lane, s, n0 + s,
                [&](record_ptr dst, int32_t lo, int32_t hi, uint32_t type,
                    uint32_t row) __attribute__((always_inline)) {
                    if (lane < lo || lane >= hi) {
                        return;
                    }
                    double v;
                    if (type == MBH_REC_ELECTRIC) {
                        v = e;
                    } else if (type == MBH_REC_MAGNETIC) {
                        v = h;
                    } else if (type < MBH_REC_DENSITY) {
                        v = p;
                    } else if (type == MBH_REC_INVERSION) {
                        v = s_d[N * (N - 1)][lane];
                    } else {
                        double x[K];
#pragma unroll
                        for (int i = 0; i < K; i++) {
                            x[i] = s_d[i][lane];
                        }
                        v = cv_population<N>(x, (int)row);
                    }
                    dst[lane] = v;
                },
                wv);
        }
    }

    if (g >= own_lo && g < own_hi) {
        if (wv == 0) {
            st<double>(k.e_out, g, e);
            st<double>(k.h_out, g, h);
            st<double>(k.p_out, g, p);
        }
#pragma unroll
        for (int i = 0; i < R; i++) {
            if (row0 + i < K) {
                st<double>(k.d_out, (uint64_t)(row0 + i) * k.dstride + g,
                           d[i]);
            }
        }
    }
}

template<int N>
hipError_t launch_team(const KArgs& k, uint64_t num_tiles, hipStream_t stream)
{
    hipLaunchKernelGGL((team_kernel<N>), dim3((unsigned)num_tiles),
                       dim3(64 * team_waves<N>()), 0, stream, k);
    return hipGetLastError();
}

} /* namespace mbh */

#endif
