/*
 * Temporally blocked FDTD + density tile kernel for gfx950.
 *
 * Geometry.  All runs of a context are laid out back to back in one
 * "super-grid" of G cells: run r occupies cells [base_r, base_r + N_r)
 * followed by one pseudo cell that holds the boundary value h[N_r] (always
 * zero).  A cell flagged `hzero` has its H forced to zero after every H
 * update (a run's first cell: h[0] = 0; the pseudo cell: h[N] = 0,
 * solver_cpu_fdtd.tpp:273-275), which decouples neighbouring runs exactly.
 *
 * One wavefront (64 lanes) owns one tile.  Lane l holds the C consecutive
 * cells g = g0 + l*C + c in registers, where g0 = t*owned - halo.  The
 * wavefront advances `nsteps <= halo` time steps without leaving the
 * registers; after s steps the outermost s cells at each tile edge are
 * stale, so only the `owned = 64*C - 2*halo` central cells are written
 * back.  Every cell's arithmetic is independent of the tiling, so results
 * do not depend on C or the temporal block.
 *
 * Step order inside the block is the plain one of solver_cpu_fdtd::run
 * (solver_cpu_fdtd.tpp:230-325): E update, sources, H update with
 * boundary condition, density update, record copy; with RED that of
 * solver_cpu_fdtd_red::run (solver_cpu_fdtd_red.tpp:451-549): density
 * update, E update, sources, H update with boundary condition, record copy.
 * Both orders have the same one-cell stencil reach per step, so the halo
 * rule above holds for either.
 */
#ifndef MBH_TILE_HPP
#define MBH_TILE_HPP

#include <type_traits>

#include "mbh_device.hpp"

namespace mbh {

constexpr int FDTD_STRIDE = 5; /* fac_a fac_b fac_c gamma dx_inv */
constexpr int BLOCH2_STRIDE = 29; /* two-level Cayley, Bloch form */

struct dev_source {
    uint64_t gx; /* super-grid cell */
    uint32_t type;
    uint32_t pad;
};

/* sources inside a tile's loaded span (halo included) and its records */
struct tile_meta {
    uint32_t src_lo, src_hi;
    uint32_t rec_lo, rec_hi;
};

struct dev_record {
    uint64_t gbegin; /* super-grid cell of position_idx */
    uint64_t cols;
    uint64_t rows;
    double ratio;
    double* dst; /* scratch + offset_real */
    uint32_t type;
    uint32_t row_idx;
    uint32_t col_idx;
    uint32_t pad;
};

struct KArgs {
    const void* e_in;
    const void* h_in;
    const void* p_in;
    const void* d_in;
    void* e_out;
    void* h_out;
    void* p_out;
    void* d_out;
    uint64_t G;       /* cells in the super-grid */
    uint64_t Gown;    /* cells owned by tiles: G minus the trailing pseudo
                         cell (its H is read at step 0 only) */
    uint64_t dstride; /* elements between density components */
    const int32_t* mat;   /* [G]: material, plus MAT_QM where it has a
                             density; -1: pseudo cell */
    const uint8_t* hzero; /* [G] */
    const double* fdtd;   /* [nmat][FDTD_STRIDE] */
    const double* qm;     /* [nmat][qstride] */
    uint64_t qstride;
    const tile_meta* tiles;   /* [num_tiles] */
    const dev_source* src;    /* sorted by gx */
    const double* src_data;   /* [sources][n_t], in the order of src */
    uint64_t n_t;
    const dev_record* tile_rec; /* the tiles' records, tile after tile */
    const uint64_t* n_base; /* device: first step = *n_base + n_off */
    uint64_t n_off;
    uint32_t nsteps;
    uint32_t halo;
    uint32_t owned;
    uint32_t yshift; /* FP32 z-form storage holds y - y* (VALU and MFMA) */
    const void* frag;     /* MFMA form: [nmat][frag_stride bytes] */
    uint64_t frag_stride;
    const uint32_t* tile_list; /* tiles of this launch (NULL: blockIdx) */
    /* MFMA form: the first n_mixed tiles of the list hold more than one
     * material; tile_mat[i] (i: position in the list) is the material of
     * a uniform tile, plus MAT_QM when it has a density (NULL: the
     * kernel reads the cells' materials) */
    const int32_t* tile_mat;
    uint32_t n_mixed;
};
constexpr int32_t MAT_QM = 0x40000000;
/* material of an entry of mat (-1: pseudo cell) */
__host__ __device__ constexpr int32_t mat_of(int32_t v)
{
    return v < 0 ? -1 : (v & ~MAT_QM);
}
/* kernel-table forms of the specialised kernels (internal, beside the
 * MBH_FORM_*): algo_noop_hz0, and algo_bloch2r with FP32 / FP64 state */
constexpr uint32_t KFORM_NOOP_HZ0 = 0x100;
constexpr uint32_t KFORM_BLOCH2R_MIXED = 0x101;
constexpr uint32_t KFORM_BLOCH2R_ZFORM64 = 0x102;
/* and algo_bloch2s */
constexpr uint32_t KFORM_BLOCH2S_MIXED = 0x106;
constexpr uint32_t KFORM_BLOCH2S_ZFORM64 = 0x107;
/* two-level Bloch kernels for lossless media with H held at zero */
template<class A>
constexpr bool bloch_real = std::is_same<A, algo_bloch2r>::value ||
    std::is_same<A, algo_bloch2s>::value;
/* algo_rodrp (FP64 Rodrigues by rotation planes), both step orders */
constexpr uint32_t KFORM_RODR_PLANES = 0x103;
/* algo_cayley2r (reference-order two-level Cayley without its exact zeros),
 * both step orders */
constexpr uint32_t KFORM_CAYLEY2R = 0x104;
/* algo_rodrp with a cell's rows split over the wavefronts of a workgroup
 * (team_kernel) */
constexpr uint32_t KFORM_RODR_TEAM = 0x105;

template<typename ST>
__device__ __forceinline__ double ld(const void* p, uint64_t i)
{
    return (double)(static_cast<const ST*>(p)[i]);
}
template<typename ST>
__device__ __forceinline__ void st(void* p, uint64_t i, double v)
{
    static_cast<ST*>(p)[i] = (ST)v;
}

/* read-only tables through the constant address space (scalar loads for
 * uniform indices) */
template<typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T*
as_const(const T* p)
{
    return (const __attribute__((address_space(4))) T*)p;
}

/* Whole-wavefront neighbour exchange with DPP: wave_shl:1 gives lane i the
 * value of lane i+1, wave_shr:1 the value of lane i-1 (the edge lane gets
 * 0; edge cells are halo cells).  Register-to-register, no LDS round trip. */
__device__ __forceinline__ double from_right(double x)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130,
                                               0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130,
                                               0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_left(double x)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138,
                                               0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138,
                                               0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

/* Runs `fn(material)` for every lane whose `m >= 0`, one distinct material
 * at a time; inside fn the material index is wave-uniform (SGPR), so
 * constant reads through it become scalar loads. */
template<typename F>
__device__ __forceinline__ void for_each_material(int32_t m, F&& fn)
{
    bool todo = m >= 0;
    for (;;) {
        unsigned long long mask = __ballot(todo);
        if (mask == 0ull) {
            break;
        }
        int leader = __builtin_ctzll(mask);
        int32_t mm = __builtin_amdgcn_readlane(m, leader);
        if (todo && m == mm) {
            fn(mm);
            todo = false;
        }
    }
}

/* copy_list_entry_dev::hasto_record (copy_list_entry.hpp:74-80) plus the
 * row bound */
__device__ __forceinline__ bool record_now(double ratio, uint64_t rows,
                                           uint64_t n)
{
    bool now = (n == 0);
    if (!now) {
        now = floor(ratio * (double)(n - 1)) != floor(ratio * (double)n);
    }
    return now && (uint64_t)floor(ratio * (double)n) < rows;
}

/* Records of a tile.  At the start of a launch the first REC_LANES of them
 * are evaluated for all steps of the block, one step per lane, and their
 * rows put in an LDS table (row minus the row at the block's first step;
 * REC_NOT: not due).  At a step with a due record lane r reads record r's
 * entry, and each due one is handed to the whole wavefront by readlane: one
 * LDS latency for all records of a step, where evaluating the row rule and
 * reading the descriptors cost some 700 cycles per record and step.  The
 * cells of a record at tile offsets [lo, hi) (clipped to the owned cells;
 * the tile's first cell, halo included, has offset 0) go to base + 8 offset
 * plus the row's offset.  Nothing but the table and the step mask stays live
 * over the steps.  Records beyond REC_LANES are read from memory at every
 * step that has one due. */
constexpr uint32_t REC_LANES = 16;
constexpr uint32_t REC_NOT = 0xffu;
constexpr uint32_t REC_STEPS = 64; /* largest temporal block */
struct rec_stage {
    uint64_t base[REC_LANES];
    uint64_t row_bytes[REC_LANES];
    uint32_t span[REC_LANES]; /* lo | hi << 16 */
    uint32_t what[REC_LANES]; /* type | level << 8 */
    uint32_t r_lo, nrec;
    uint32_t density; /* a population or the inversion may be among them */
    int64_t tile0, own_lo, own_hi;
    uint8_t row[REC_STEPS][REC_LANES];
};

/* coherences are not recorded */
__device__ __forceinline__ bool record_skipped(const dev_record& R)
{
    return R.type == MBH_REC_DENSITY && R.row_idx != R.col_idx;
}

__device__ __forceinline__ uint32_t lane_u32(uint32_t x, int i)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)x, i);
}
__device__ __forceinline__ uint64_t lane_u64(uint64_t x, int i)
{
    return ((uint64_t)lane_u32((uint32_t)(x >> 32), i) << 32) |
        lane_u32((uint32_t)x, i);
}
__device__ __forceinline__ double lane_f64(double x, int i)
{
    return __longlong_as_double(
        (long long)lane_u64((uint64_t)__double_as_longlong(x), i));
}

/* record i of the launch's list through scalar loads */
__device__ __forceinline__ dev_record scalar_record(const KArgs& k,
                                                    uint32_t i)
{
    const auto* r = as_const(k.tile_rec) + i;
    dev_record R;
    R.gbegin = r->gbegin;
    R.cols = r->cols;
    R.rows = r->rows;
    R.ratio = r->ratio;
    R.dst = r->dst;
    R.type = r->type;
    R.row_idx = r->row_idx;
    R.col_idx = r->col_idx;
    R.pad = 0;
    return R;
}

/* (global, not generic: a generic store holds up the next step's LDS reads
 * until it is done) */
typedef __attribute__((address_space(1))) double* record_ptr;

/* where record R goes at row `row`, and its span in the tile */
__device__ __forceinline__ uint64_t record_base(const dev_record& R,
                                                uint64_t row, int64_t tile0)
{
    return (uint64_t)(uintptr_t)R.dst + 8u * (row * R.cols) -
        8u * (uint64_t)((int64_t)R.gbegin - tile0);
}
__device__ __forceinline__ uint32_t record_span(const dev_record& R,
                                                int64_t tile0, int64_t own_lo,
                                                int64_t own_hi)
{
    const int64_t g0 = (int64_t)R.gbegin, g1 = g0 + (int64_t)R.cols;
    const uint32_t lo = (uint32_t)((g0 > own_lo ? g0 : own_lo) - tile0);
    const uint32_t hi = (uint32_t)((g1 < own_hi ? g1 : own_hi) - tile0);
    return lo | (hi << 16);
}

/* lane r's record r of the tile (r < REC_LANES) */
__device__ __forceinline__ dev_record own_record(const KArgs& k,
                                                 const tile_meta& M, int lane)
{
    dev_record R{};
    if ((uint32_t)lane < REC_LANES && (uint32_t)lane < M.rec_hi - M.rec_lo) {
        R = k.tile_rec[M.rec_lo + lane];
    }
    return R;
}

/* R: own_record.  Returns the steps of the block at which any of the tile's
 * records is due (one bit per step) and, if there are any, stages them. */
__device__ __forceinline__ uint64_t stage_records(
    const KArgs& k, rec_stage& S, const dev_record& R, int lane, bool writer,
    const tile_meta& M, int64_t own_lo, int64_t own_hi, uint64_t n0,
    uint32_t nsteps)
{
    static_assert(REC_STEPS == 64, "one lane and one mask bit per step");
    const uint32_t nrec = M.rec_hi - M.rec_lo;
    const uint32_t nlane = nrec < REC_LANES ? nrec : REC_LANES;
    const uint64_t n = n0 + (uint64_t)lane;
    const bool step = lane < (int)nsteps;
    uint64_t steps = 0;
    for (uint32_t i = 0; i < nrec; i++) {
        double ratio;
        uint64_t rows;
        bool skip;
        if (i < REC_LANES) {
            ratio = lane_f64(R.ratio, (int)i);
            rows = lane_u64(R.rows, (int)i);
            skip = lane_u32(record_skipped(R) ? 1u : 0u, (int)i) != 0u;
        } else {
            const dev_record Q = scalar_record(k, M.rec_lo + i);
            ratio = Q.ratio;
            rows = Q.rows;
            skip = record_skipped(Q);
        }
        const bool due = step && !skip && record_now(ratio, rows, n);
        if (i < REC_LANES && writer) {
            const uint64_t row = (uint64_t)floor(ratio * (double)n);
            const uint64_t row0 = (uint64_t)floor(ratio * (double)n0);
            S.row[lane][i] =
                due ? (uint8_t)(row - row0) : (uint8_t)REC_NOT;
        }
        steps |= __ballot(due);
    }
    if (steps != 0ull) {
        if (writer) {
            const int64_t tile0 = own_lo - (int64_t)k.halo;
            const bool dens = __any((uint32_t)lane < nlane &&
                                    !record_skipped(R) &&
                                    R.type >= MBH_REC_DENSITY) ||
                nrec > REC_LANES;
            if ((uint32_t)lane < nlane) {
                const uint64_t row0 =
                    (uint64_t)floor(R.ratio * (double)n0);
                S.base[lane] = record_base(R, row0, tile0);
                S.row_bytes[lane] = 8u * R.cols;
                S.span[lane] = record_span(R, tile0, own_lo, own_hi);
                S.what[lane] = R.type | (R.row_idx << 8);
            }
            if (lane == 0) {
                S.r_lo = M.rec_lo;
                S.nrec = nrec;
                S.density = dens ? 1u : 0u;
                S.tile0 = tile0;
                S.own_lo = own_lo;
                S.own_hi = own_hi;
            }
        }
        __syncthreads();
    }
    return steps;
}

/* Calls put(dst, lo, hi, type, level) for every record due at step s of the
 * block (step n of the run), all arguments wave-uniform: the cell at tile
 * offset o in [lo, hi) goes to dst[o].  Of W wavefronts with the same cells,
 * wavefront wv takes every W-th record. */
template<int W = 1, typename F>
__device__ __forceinline__ void for_due_records(const KArgs& k,
                                                const rec_stage& S, int lane,
                                                uint32_t s, uint64_t n,
                                                F&& put, int wv = 0)
{
    const uint32_t r = (uint32_t)lane & (REC_LANES - 1u);
    uint64_t base = S.base[r], row_bytes = S.row_bytes[r];
    uint32_t row = S.row[s][r], span = S.span[r], what = S.what[r];
    uint32_t n_all = S.nrec;
    /* (all reads ahead of the first use: one LDS latency) */
    asm volatile("" : "+v"(base), "+v"(row_bytes), "+v"(row), "+v"(span),
                      "+v"(what), "+v"(n_all));
    const uint32_t nrec = lane_u32(n_all, 0);
    const uint64_t dst = base + row_bytes * row;
    unsigned long long todo = __ballot((uint32_t)lane < REC_LANES &&
                                       (uint32_t)lane < nrec &&
                                       (W == 1 || lane % W == wv) &&
                                       row != REC_NOT);
    while (todo != 0ull) {
        const int i = __builtin_ctzll(todo);
        todo &= todo - 1;
        const uint32_t sp = lane_u32(span, i), w = lane_u32(what, i);
        put((record_ptr)(lane_u64(dst, i)),
            (int32_t)(sp & 0xffffu), (int32_t)(sp >> 16), w & 0xffu, w >> 8);
    }
    for (uint32_t i = REC_LANES; i < nrec; i++) {
        /* (the step number's conversions stay in here: hoisted, they would
         * hold registers over the steps) */
        asm volatile("" : "+s"(n));
        const dev_record R = scalar_record(k, lane_u32(S.r_lo, 0) + i);
        if ((W > 1 && (int)(i % (uint32_t)W) != wv) || record_skipped(R) ||
            !record_now(R.ratio, R.rows, n)) {
            continue;
        }
        const uint64_t at =
            lane_u64((uint64_t)floor(R.ratio * (double)n), 0);
        const int64_t tile0 = (int64_t)lane_u64((uint64_t)S.tile0, 0);
        const uint32_t sp = record_span(
            R, tile0, (int64_t)lane_u64((uint64_t)S.own_lo, 0),
            (int64_t)lane_u64((uint64_t)S.own_hi, 0));
        put((record_ptr)(record_base(R, at, tile0)),
            (int32_t)(sp & 0xffffu), (int32_t)(sp >> 16), R.type, R.row_idx);
    }
}

/* FP32 storage of the z-form holds y - y* (y* at OFF_YEQ of the material's
 * blob): v += sign * y* for a cell of material m with a density */
template<class A>
__device__ __forceinline__ void add_shift(const KArgs& k, int32_t m,
                                          double* v, double sign)
{
    /* loads from material 0's blob where m < 0 (every blob is there), so
     * that none waits in a branch of its own */
    const double* q =
        (const double*)k.qm + (uint64_t)(m < 0 ? 0 : m) * k.qstride;
    double y[A::DC];
#pragma unroll
    for (int j = 0; j < A::DC; j++) {
        y[j] = q[A::OFF_YEQ + j];
    }
    const bool on = (m >= 0) && (q[0] != 0.0);
#pragma unroll
    for (int j = 0; j < A::DC; j++) {
        v[j] = on ? fma(sign, y[j], v[j]) : v[j];
    }
}

constexpr uint32_t TILE_SOURCES = 7; /* of a tile, staged in LDS */
constexpr int MAX_BLOCK = 64;   /* largest temporal block */

/* LDS of a tile: the sources' values for the block's steps and their places,
 * the records */
struct tile_lds {
    double src[TILE_SOURCES][MAX_BLOCK];
    rec_stage rec;
    uint32_t where[TILE_SOURCES];
};
static_assert(sizeof(tile_lds) <= 4 * 1280, "see TILE_SOURCES");

/* Source values of a tile for the steps of the block: the first one's in a
 * register, one step per lane (REG: read by readlane; an LDS read in the
 * step's chain cost 165 of 410 cycles of the two-level Bloch step), the next
 * TILE_SOURCES in LDS, any more from memory.  Seven, so that tile_lds takes
 * four of the LDS's units of 1280 bytes: in five, a CU holds 25 instead of 32
 * tiles of the kernels that need 64 registers or fewer (noop, 2^26 cells, one
 * cell per lane: FP64 8.4 -> 7.6 ms, FP32 6.6 -> 6.0 ms per 96 steps).
 * where: offset of the source's cell in the tile (the tile's first cell, halo
 * included, has offset 0) and, in bit 0, its type. */
__device__ __forceinline__ uint32_t source_where(const KArgs& k, uint32_t i,
                                                 int64_t tile0)
{
    return ((uint32_t)((int64_t)as_const(k.src)[i].gx - tile0) << 1) |
        (as_const(k.src)[i].type == MBH_SRC_HARD ? 1u : 0u);
}
struct tile_sources {
    uint32_t lo, count;
    uint32_t where0;
    double v0;
};
__device__ __forceinline__ double source_load(const KArgs& k, uint32_t i,
                                              uint64_t n, bool in)
{
    /* (lanes beyond the block: the source's first value, not used) */
    return k.src_data[(uint64_t)i * k.n_t + (in ? n : 0u)];
}
template<bool REG>
__device__ __forceinline__ tile_sources stage_sources(
    const KArgs& k, tile_lds& S, int lane, bool writer, const tile_meta& M,
    int64_t tile0, uint64_t n0, uint32_t nsteps)
{
    tile_sources T{ M.src_lo, M.src_hi - M.src_lo, 0u, 0.0 };
    if (T.count > 0) {
        const bool in = lane < (int)nsteps;
        const uint64_t n = n0 + (uint64_t)lane;
        if constexpr (REG) {
            T.where0 = source_where(k, T.lo, tile0);
            T.v0 = source_load(k, T.lo, n, in);
        }
        constexpr uint32_t J0 = REG ? 1u : 0u;
        if (T.count > J0) {
            if (writer) {
                const uint32_t cnt = T.count - J0 < TILE_SOURCES
                    ? T.count - J0
                    : TILE_SOURCES;
                for (uint32_t j = 0; j < cnt; j++) {
                    S.src[j][lane] = source_load(k, T.lo + J0 + j, n, in);
                    if (lane == 0) {
                        S.where[j] = source_where(k, T.lo + J0 + j, tile0);
                    }
                }
            }
            __syncthreads();
        }
    }
    return T;
}
/* calls put(offset, hard, value) for every source of the tile, in list
 * order (solver_cpu_fdtd.tpp:247-255) */
template<bool REG, typename F>
__device__ __forceinline__ void for_sources(const KArgs& k,
                                            const tile_lds& S,
                                            const tile_sources& T,
                                            int64_t tile0, uint64_t n0,
                                            uint32_t s, F&& put)
{
    if (T.count == 0) {
        return;
    }
    if constexpr (REG) {
        put((int32_t)(T.where0 >> 1), (T.where0 & 1u) != 0u,
            lane_f64(T.v0, (int)s));
    }
    /* (rolled: unrolled over the staged ones, their places would be read
     * ahead of the steps into scalar registers) */
    constexpr uint32_t J0 = REG ? 1u : 0u;
#pragma unroll 1
    for (uint32_t j = J0; j < T.count; j++) {
        uint32_t w;
        double v;
        if (j < J0 + TILE_SOURCES) {
            w = S.where[j - J0];
            v = S.src[j - J0][s];
        } else {
            w = source_where(k, T.lo + j, tile0);
            v = as_const(k.src_data)[(uint64_t)(T.lo + j) * k.n_t + n0 + s];
        }
        put((int32_t)(w >> 1), (w & 1u) != 0u, v);
    }
}


/* One tile t: all steps of the temporal block for the tile's cells.
 * With W > 1 the tile spans W wavefronts of one workgroup, each holding a
 * contiguous run of 64 C cells; at the inner edges between them the
 * neighbour's boundary H (before the E update) and E (before the H
 * update) come through LDS every step, so only the tile's two outer edges
 * carry a halo (64 C W - 2 tb owned cells instead of 64 C - 2 tb). */
template<class A, int C, typename ST, bool RED = false, int W = 1>
__device__ __forceinline__ void tile_body(const KArgs& k, uint64_t t,
                                          tile_lds& lds)
{
    static_assert(W == 1 || !RED, "multi-wavefront tiles: plain order only");
    static_assert(W == 1 || A::STAGE == 0,
                  "multi-wavefront tiles: no per-wavefront LDS staging");
    /* boundary values of each wavefront's run for its neighbours */
    __shared__ double x_h[W > 1 ? W : 1]; /* H of the first cell */
    __shared__ double x_e[W > 1 ? W : 1]; /* E of the last cell */

    const int lane = threadIdx.x & 63;
    const int wv = (W > 1) ? (int)(threadIdx.x >> 6) : 0;
    const int64_t own_lo = (int64_t)(t * k.owned);
    const int64_t own_hi =
        ((own_lo + (int64_t)k.owned) < (int64_t)k.Gown) ? own_lo + k.owned
                                                         : (int64_t)k.Gown;
    const int64_t gl =
        own_lo - (int64_t)k.halo + (int64_t)(wv * 64 + lane) * C;
    const int64_t tile0 = own_lo - (int64_t)k.halo;
    const uint64_t n0 = *as_const(k.n_base) + k.n_off;
    const uint32_t nsteps = k.nsteps;
    const tile_meta M{ as_const(k.tiles)[t].src_lo,
                       as_const(k.tiles)[t].src_hi,
                       as_const(k.tiles)[t].rec_lo,
                       as_const(k.tiles)[t].rec_hi };

    /* When the tile's records are staged.  Before the state is loaded they
     * cost registers of their own only.  One cell per lane with constants in
     * registers (grids bound by the latency of a launch) has the descriptors
     * in flight together with the state and stages them after the constants
     * (two-level Bloch form, 8192 cells x 16000 steps: 3.73 ms, 3.90 with
     * the constants loaded after it); two-level Cayley without its zeros
     * stages them between the two (2^20 cells, 9.1 us per step, 9.3 before
     * the state).  Staged after the constants by every kernel, and with the
     * record code's addresses kept over the steps, the FP64 noop kernel
     * spilled (2^27 cells, tiles of 512 cells, blocks of 32 steps: 65 -> 72
     * us per step) and three-level Cayley fitted one wavefront per SIMD
     * instead of two (2^18 cells 14.8 -> 17.4 us per step, 14.3 here). */
    constexpr bool STAGE_LAST = C == 1 && (A::CONSTS || A::ROWC);
    constexpr bool STAGE_FIRST =
        !STAGE_LAST && !std::is_same<A, algo_cayley2r>::value;
    uint64_t rec_steps = 0; /* steps of this block with a due record */
    auto stage = [&](const dev_record& R) __attribute__((always_inline)) {
        if (M.rec_lo != M.rec_hi) {
            rec_steps = stage_records(k, lds.rec, R, lane, wv == 0, M, own_lo,
                                      own_hi, n0, nsteps);
        }
    };
    if constexpr (STAGE_FIRST) {
        stage(own_record(k, M, lane));
    }

    double e[C], h[C], p[C];
    double fa[C], fb[C], fc[C], fg[C], fx[C];
    typename A::state d[C];
    int32_t m[C];  /* material (-1: outside the grid) */
    int32_t ma[C]; /* the same where it has a density, else -1 */
    bool hz[C];

    /* The state loads of all cells first, each from a clamped address
     * (cell 0 where the cell lies outside the grid) and selected after,
     * then the loads that depend on the cells' materials: no load waits
     * in a branch of its own, and each group is in flight together. */
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int64_t g = gl + c;
        const bool in = (g >= 0) && (g < (int64_t)k.G);
        const uint64_t gc = in ? (uint64_t)g : 0u;
        const int32_t mv = k.mat[gc];
        const uint8_t hv = k.hzero[gc];
        const double ev = ld<ST>(k.e_in, gc);
        const double hv2 = ld<ST>(k.h_in, gc);
        const double pv = (A::DC > 0) ? ld<ST>(k.p_in, gc) : 0.0;
        double dv[A::DC > 0 ? A::DC : 1];
#pragma unroll
        for (int j = 0; j < A::DC; j++) {
            dv[j] = ld<ST>(k.d_in, (uint64_t)j * k.dstride + gc);
        }
        m[c] = in ? mat_of(mv) : -1;
        ma[c] = (A::DC > 0 && in && mv >= 0 && (mv & MAT_QM) != 0) ? m[c]
                                                                   : -1;
        hz[c] = in ? (hv != 0) : true;
        e[c] = in ? ev : 0.0;
        /* the trailing pseudo cell is never owned, so never written back:
         * its H is h[N] of the initial state at step 0 and zero after (the
         * boundary condition) */
        h[c] = (in && (g + 1 < (int64_t)k.G || n0 == 0)) ? hv2 : 0.0;
        /* no density: p keeps its initial zero (lindblad_noop) and is
         * neither read nor written */
        p[c] = (A::DC > 0 && in) ? pv : 0.0;
#pragma unroll
        for (int j = 0; j < A::DC; j++) {
            d[c].v[j] = in ? dv[j] : 0.0;
        }
    }
    dev_record rec_own{};
    if constexpr (!STAGE_FIRST) {
        rec_own = own_record(k, M, lane);
    }
    if constexpr (!STAGE_FIRST && !STAGE_LAST) {
        stage(rec_own);
    }
    /* the tile's sources, the first in a register; the larger z-forms and
     * four or more cells per lane with a density (but for the two-level
     * Bloch form of a real dipole) have no register pair to spare */
    constexpr bool SRC_REG = A::DC < 24 &&
        (C < 4 || A::DC == 0 || bloch_real<A>);
    const tile_sources srcs =
        stage_sources<SRC_REG>(k, lds, lane, wv == 0, M, tile0, n0,
                               nsteps);
#pragma unroll
    for (int c = 0; c < C; c++) {
        if constexpr (A::SHIFT && std::is_same<ST, float>::value) {
            if (k.yshift) {
                add_shift<A>(k, m[c], d[c].v, 1.0);
            }
        }
        /* material 0's row where the cell has none, then zeroed */
        const double* f =
            k.fdtd + (uint64_t)(m[c] < 0 ? 0 : m[c]) * FDTD_STRIDE;
        const double f0 = f[0], f1 = f[1], f2 = f[2], f3 = f[3], f4 = f[4];
        const bool known = m[c] >= 0;
        fa[c] = known ? f0 : 0.0;
        fb[c] = known ? f1 : 0.0;
        fc[c] = known ? f2 : 0.0;
        fg[c] = known ? f3 : 0.0;
        fx[c] = known ? f4 : 0.0;
        if constexpr (A::FAST_FDTD) {
            /* folded constants: e' = fa e + fg' p + fx' (h_r - h) with
             * fg' = -fb fg, fx' = fb fx (zero outside the grid, so those
             * cells stay zero); h' = hm h + fc' (e_c - e_l) with hm = 0,
             * fc' = 0 where H is held at zero */
            fg[c] = -(fb[c] * fg[c]);
            fx[c] = fb[c] * fx[c];
            fb[c] = hz[c] ? 0.0 : 1.0;
            fc[c] = hz[c] ? 0.0 : fc[c];
        }
    }

    /* material with a density, per cell (-1: vacuum or outside the grid),
     * and m1, the first of them in the tile. The lanes whose cells all have
     * m1 update with m1's constants as in a tile of one material (a tile
     * at an interface between m1 and vacuum is then as fast as one inside
     * the medium); the other lanes of the tile (a cell of another density
     * material, or one lane straddling the interface) take one update per
     * material. The arithmetic of a cell is the same either way. */
    int32_t first = -1;
#pragma unroll
    for (int c = C - 1; c >= 0; c--) {
        first = (ma[c] >= 0) ? ma[c] : first;
    }
    const unsigned long long act_lanes = __ballot(first >= 0);
    const int32_t m1 = act_lanes
        ? __builtin_amdgcn_readlane(first, __builtin_ctzll(act_lanes))
        : -1;
    bool all1 = true;
#pragma unroll
    for (int c = 0; c < C; c++) {
        all1 = all1 && (ma[c] == m1);
    }
    all1 = all1 && (m1 >= 0);
    const bool full1 = __all(all1);
    cdp q0 = (cdp)k.qm + (uint64_t)(m1 < 0 ? 0 : m1) * k.qstride;
    const bool q0_active = m1 >= 0;
    /* doubles of the material blob the algorithm wants staged in LDS */
    constexpr bool ROWS = A::ROWC && C == 1;
    constexpr int STAGE = ROWS ? 0 : A::STAGE;
    __shared__ double s_q[STAGE > 0 ? STAGE : 1];
    if constexpr (STAGE > 0) {
        if (q0_active) {
            for (int i = lane; i < STAGE; i += 64) {
                s_q[i] = q0[i];
            }
        }
        __syncthreads();
    }

    if constexpr (W > 1) {
        if (lane == 0) {
            x_h[wv] = h[0];
        }
        __syncthreads();
    }

    if constexpr (STAGE_LAST) {
        stage(rec_own);
    }

    /* material constants held over the steps: each lane's own with one cell
     * per lane, m1's otherwise */
    constexpr bool LANE = A::CONSTS && C == 1;
    auto consts = [&]() {
        if constexpr (LANE) {
            const auto q = A::load(
                (const double*)k.qm +
                (uint64_t)(ma[0] < 0 ? 0 : ma[0]) * k.qstride);
            return ma[0] >= 0 ? q : A::one();
        } else if constexpr (A::CONSTS) {
            return A::load(q0);
        } else {
            return 0;
        }
    }();

    /* or m1's, sixteen to a register pair; others: lanes of a tile with a
     * second density material */
    auto rows = [&]() {
        if constexpr (ROWS) {
            return typename A::rowc();
        } else {
            return 0;
        }
    }();
    auto load_rows = [&](int32_t mm) {
        if constexpr (ROWS) {
            const uint64_t at = (uint64_t)(mm < 0 ? 0 : mm) * k.qstride;
            rows.load((cdp)k.qm + at, (const double*)k.qm + at);
        }
    };
    load_rows(m1);
    const unsigned long long others =
        ROWS ? __ballot(ma[0] >= 0 && ma[0] != m1) : 0ull;

    /* density update of every cell from its current field
     * (solver_cpu_fdtd.tpp:278-285, solver_cpu_fdtd_red.tpp:451-457) */
    auto density_update = [&]() {
        if constexpr (LANE) {
            A::template apply<1>(consts, d, e, p);
        } else if constexpr (ROWS) {
            if (m1 >= 0) {
                /* Every lane computes with the constants of one material
                 * (the row registers need all lanes active), that
                 * material's cells keep the result; tiles with a second
                 * density material repeat it with that one's constants. */
                unsigned long long left = others;
                typename A::state old;
                double pold = 0.0;
                for (int32_t mm = m1;;) {
                    const bool mine = full1 || ma[0] == mm;
                    if (!full1) {
                        old = d[0];
                        pold = p[0];
                    }
                    A::apply_rows(rows, d[0], e[0], p[0], mine);
                    if (full1) {
                        break;
                    }
#pragma unroll
                    for (int j = 0; j < A::DC; j++) {
                        d[0].v[j] = mine ? d[0].v[j] : old.v[j];
                    }
                    p[0] = mine ? p[0] : pold;
                    if (others == 0ull) {
                        break;
                    }
                    mm = left != 0ull
                        ? __builtin_amdgcn_readlane(ma[0],
                                                    __builtin_ctzll(left))
                        : m1;
                    load_rows(mm);
                    if (left == 0ull) {
                        break;
                    }
                    left &= ~__ballot(ma[0] == mm);
                }
            }
        } else if constexpr (A::DC > 0) {
            auto update_m1 = [&]() {
                if constexpr (A::CONSTS) {
                    A::template apply<C>(consts, d, e, p);
                } else if constexpr (STAGE > 0) {
                    /* an offset the compiler cannot see through keeps the
                     * LDS reads inside the step (hoisted, the staged
                     * constants would occupy VGPRs for the whole loop) */
                    int off = 0;
                    asm volatile("" : "+s"(off));
                    A::template update_multi_p<C>((const double*)s_q + off,
                                                  d, e, p);
                } else {
                    A::template update_multi<C>(q0, d, e, p);
                }
            };
            /* small updates (two levels) get a second copy behind a
             * wave-uniform branch, so that tiles of one material run it
             * with full exec and no per-lane branch; for the large ones
             * the second copy costs more (instruction cache) than the
             * per-lane branch */
            constexpr bool TWO_COPIES = A::DC <= 4;
            if (TWO_COPIES && full1) {
                update_m1();
            } else if (all1) {
                update_m1();
            } else if (m1 >= 0) {
                /* lanes with a cell of another material: one update per
                 * material */
#pragma unroll
                for (int c = 0; c < C; c++) {
                    for_each_material(ma[c], [&](int32_t mm) {
                        A::update((cdp)k.qm + (uint64_t)mm * k.qstride, d[c],
                                  e[c], p[c]);
                    });
                }
            }
        }
    };

    auto step = [&](uint32_t s) __attribute__((always_inline)) {
        if constexpr (RED) {
            density_update();
        }

        /* E update (solver_cpu_fdtd.tpp:238-243) */
        double h_right = from_right(h[0]);
        if constexpr (W > 1) {
            /* the last lane's right neighbour is the next run's first
             * cell (beyond the tile's last run: halo, as with W = 1) */
            const double xr = (wv + 1 < W) ? x_h[wv + 1] : 0.0;
            h_right = (lane == 63) ? xr : h_right;
        }
        double en[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            const double hn = (c + 1 < C) ? h[(c + 1) % C] : h_right;
            if constexpr (A::FAST_FDTD && A::DC == 0) {
                en[c] = fma(fx[c], hn - h[c], fa[c] * e[c]); /* p = 0 */
            } else if constexpr (bloch_real<A>) {
                /* lossless (fa = 1 in the grid; cells outside it and the
                 * pseudo cells hold E = 0 with fg = fx = 0) */
                en[c] = fma(fx[c], hn - h[c], fma(fg[c], p[c], e[c]));
            } else if constexpr (A::FAST_FDTD) {
                en[c] = fma(fx[c], hn - h[c], fma(fg[c], p[c], fa[c] * e[c]));
            } else {
                en[c] = (m[c] >= 0)
                    ? fa[c] * e[c] +
                        fb[c] * (-fg[c] * p[c] + (hn - h[c]) * fx[c])
                    : 0.0;
            }
        }

        /* sources, in list order (solver_cpu_fdtd.tpp:247-255) */
        for_sources<SRC_REG>(k, lds, srcs, tile0, n0, s,
                    [&](int32_t at, bool hard, double v)
                        __attribute__((always_inline)) {
                        const int32_t off =
                            at - (int32_t)(wv * 64 + lane) * C;
#pragma unroll
                        for (int c = 0; c < C; c++) {
                            /* (selects: as branches the compiler makes an
                             * indexed store of them, en in scratch) */
                            const double x = hard ? v : en[c] + v;
                            en[c] = off == c ? x : en[c];
                        }
                    });

        /* H update and boundary condition (solver_cpu_fdtd.tpp:263-275) */
        double e_left = from_left(en[C - 1]);
        if constexpr (W > 1) {
            if (lane == 63) {
                x_e[wv] = en[C - 1];
            }
            __syncthreads();
            const double xl = (wv > 0) ? x_e[wv - 1] : 0.0;
            e_left = (lane == 0) ? xl : e_left;
        }
#pragma unroll
        for (int c = 0; c < C; c++) {
            const double ep = (c > 0) ? en[(c + C - 1) % C] : e_left;
            if constexpr (std::is_same<A, algo_noop_hz0>::value ||
                          bloch_real<A>) {
                /* every held cell starts at zero and its fc is zero */
                h[c] = fma(fc[c], en[c] - ep, h[c]);
            } else if constexpr (A::FAST_FDTD) {
                h[c] = fma(fc[c], en[c] - ep, fb[c] * h[c]);
            } else {
                h[c] = hz[c] ? 0.0 : h[c] + fc[c] * (en[c] - ep);
            }
        }
        if constexpr (W > 1) {
            /* the next step's E update reads it (every read of the old
             * value came before the barrier above) */
            if (lane == 0) {
                x_h[wv] = h[0];
            }
            __syncthreads();
        }

#pragma unroll
        for (int c = 0; c < C; c++) {
            e[c] = en[c];
        }
        if constexpr (!RED) {
            density_update();
        }
    };
    /* record copy (solver_cpu_fdtd.tpp:288-325) */
    auto record = [&](uint32_t s) __attribute__((always_inline)) {
            /* (a lane index the compiler cannot see through keeps the
             * addresses that depend on it out of the steps, where there is
             * no register to spare) */
            int ln = lane;
            if constexpr (A::DC > 0 || C >= 4) {
                asm volatile("" : "+v"(ln));
            }
            for_due_records(
                k, lds.rec, ln, s, n0 + s,
                [&](record_ptr dst, int32_t lo, int32_t hi, uint32_t type,
                    uint32_t row) __attribute__((always_inline)) {
                    const int32_t o0 = (int32_t)(wv * 64 + ln) * C;
                    if (type >= MBH_REC_DENSITY) {
                        /* density, inversion: the constants of one
                         * material at a time (scalar loads) */
#pragma unroll
                        for (int c = 0; c < C; c++) {
                            const bool mine = o0 + c >= lo && o0 + c < hi;
                            for_each_material(
                                mine ? m[c] : -1, [&](int32_t mm) {
                                    cdp q = (cdp)k.qm +
                                        (uint64_t)mm * k.qstride;
                                    dst[o0 + c] = k.qstride == 0 ? 0.0
                                        : (type == MBH_REC_INVERSION
                                               ? A::inversion(q, d[c])
                                               : A::population(q, d[c],
                                                               (int)row));
                                });
                        }
                        return;
                    }
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        if (o0 + c >= lo && o0 + c < hi) {
                            dst[o0 + c] = type == MBH_REC_ELECTRIC
                                ? e[c]
                                : (type == MBH_REC_MAGNETIC ? h[c] : p[c]);
                        }
                    }
                });
    };
    if constexpr (A::CONSTS || (A::DC == 0 && A::FAST_FDTD)) {
        /* short steps: those up to the next one with a due record in a loop
         * of their own, without a test for records in it (two-level Bloch
         * form, one cell per lane: 0.305 -> 0.270 us per step; with material
         * constants read inside the step the nest costs more, 1.35 -> 1.45
         * us for the reference-order Cayley step) */
        for (uint32_t s = 0; s < nsteps;) {
            const uint32_t end = rec_steps != 0ull
                ? (uint32_t)__builtin_ctzll(rec_steps) + 1u
                : nsteps;
            for (; s < end; s++) {
                step(s);
            }
            if (rec_steps != 0ull) {
                record(s - 1u);
                rec_steps &= rec_steps - 1ull;
            }
        }
    } else {
        for (uint32_t s = 0; s < nsteps; s++) {
            step(s);
            const bool due = ((rec_steps >> s) & 1ull) != 0ull;
            /* (unlikely: what spills, spills in the record code) */
            if (A::DC > 0 ? __builtin_expect(due, false) : due) {
                record(s);
            }
        }
    }

    /* write back the owned cells */
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int64_t g = gl + c;
        if constexpr (A::SHIFT && std::is_same<ST, float>::value) {
            if (k.yshift) {
                add_shift<A>(k, m[c], d[c].v, -1.0);
            }
        }
        if (g >= own_lo && g < own_hi) {
            st<ST>(k.e_out, g, e[c]);
            st<ST>(k.h_out, g, h[c]);
            if constexpr (A::DC > 0) {
                st<ST>(k.p_out, g, p[c]);
            }
#pragma unroll
            for (int j = 0; j < A::DC; j++) {
                st<ST>(k.d_out, (uint64_t)j * k.dstride + g, d[c].v[j]);
            }
        }
    }
}

/* wavefronts per SIMD the compiler is asked to fit (1: no request): the
 * two-level Bloch kernel at four cells per lane fits three without spills
 * in its step loop, against two unasked */
#ifndef MBH_BLOCH2R_WAVES
#define MBH_BLOCH2R_WAVES 3
#endif
template<class A, int C>
constexpr int tile_min_waves()
{
    if (bloch_real<A> && C == 4) {
        return MBH_BLOCH2R_WAVES;
    }
    if (std::is_same<A, algo_bloch2>::value && C == 4) {
        return 3;
    }
    /* (266 registers unasked; 2^20 cells 21.1 -> 18.0 us per step with
     * eleven of them spilled outside the step) */
    if (std::is_same<A, algo_cayley<2>>::value && C == 4) {
        return 2;
    }
    /* row registers: without a request the polynomial constants of the wide
     * sin / cos ranges, hoisted out of the steps, fill the file */
    return A::ROWC && C == 1 ? A::ROWC_WAVES : 1;
}

template<class A, int C, typename ST, bool RED = false>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(tile_min_waves<A, C>()))) void
tile_kernel(KArgs k)
{
    __shared__ tile_lds lds;
    tile_body<A, C, ST, RED>(
        k, k.tile_list ? k.tile_list[blockIdx.x] : blockIdx.x, lds);
}

/* tile of W wavefronts (64 W threads) */
template<class A, int C, int W, typename ST>
__global__ __launch_bounds__(64 * W)
__attribute__((amdgpu_waves_per_eu(tile_min_waves<A, C>()))) void
tile_kernel_mw(KArgs k)
{
    __shared__ tile_lds lds;
    tile_body<A, C, ST, false, W>(
        k, k.tile_list ? k.tile_list[blockIdx.x] : blockIdx.x, lds);
}

/* ---- launcher registry ------------------------------------------------- */
typedef hipError_t (*tile_launch_fn)(const KArgs& k, uint64_t num_tiles,
                                     hipStream_t stream);

struct kernel_entry {
    uint32_t algo;
    uint32_t levels;
    uint32_t form; /* MBH_FORM_* the kernel implements */
    uint32_t cells_per_lane;
    tile_launch_fn fn;
    uint32_t order; /* MBH_ORDER_* */
};

template<class A, int C, typename ST, bool RED = false>
hipError_t launch_tile(const KArgs& k, uint64_t num_tiles, hipStream_t stream)
{
    hipLaunchKernelGGL((tile_kernel<A, C, ST, RED>), dim3((unsigned)num_tiles),
                       dim3(64), 0, stream, k);
    return hipGetLastError();
}

/* multi-wavefront tiles: the tables list them with C W cells per lane of
 * the tile's first wavefront, so tile geometry (64 C W cells) needs no
 * other change on the host */
template<class A, int C, int W, typename ST>
hipError_t launch_tile_mw(const KArgs& k, uint64_t num_tiles,
                          hipStream_t stream)
{
    hipLaunchKernelGGL((tile_kernel_mw<A, C, W, ST>),
                       dim3((unsigned)num_tiles), dim3(64 * W), 0, stream, k);
    return hipGetLastError();
}

/* z-form state conversions (per cell, uniform material) */
struct ZArgs {
    const double* dref; /* reference coherence vectors, component-major */
    void* y;            /* z-form state (ST), component-major */
    uint64_t G;
    uint64_t dstride;
    const int32_t* mat;
    const double* zq;
    uint64_t zstride;
    uint32_t yshift; /* FP32 storage holds y - y* */
    uint64_t g0;     /* first super-grid cell converted */
    uint64_t count;  /* cells converted */
    double* out_cm;  /* y -> d only: if set, d of cell g0 + i goes to
                        out_cm[i * K + j] (cell-major) instead of dref */
};
typedef hipError_t (*zconv_fn)(const ZArgs& a, hipStream_t stream);

struct zconv_entry {
    uint32_t levels;
    uint32_t fp32;
    zconv_fn to_y;   /* dref -> y */
    zconv_fn from_y; /* y -> dref (written into dref) */
};

/* tables defined by the instantiation units */
extern const kernel_entry k_table_basic[];
extern const uint32_t k_table_basic_n;
extern const kernel_entry k_table_rodr[];
extern const uint32_t k_table_rodr_n;
extern const kernel_entry k_table_zform[];
extern const uint32_t k_table_zform_n;
extern const kernel_entry k_table_zm[];
extern const uint32_t k_table_zm_n;
extern const kernel_entry k_table_red[];
extern const uint32_t k_table_red_n;
extern const zconv_entry z_table[];
extern const uint32_t z_table_n;

} /* namespace mbh */

#endif
