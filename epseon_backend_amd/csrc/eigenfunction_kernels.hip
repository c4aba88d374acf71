// eigenfunction_kernels.hip -- gfx950 kernels for the normalised
// eigenfunctions of the refined levels and for the adjoint of the levels with
// respect to the tabulated potential.
//
// The reference has no eigenfunction or gradient code (its only algorithm,
// VibwaAlgorithm<FP>::run, cpp/gpu/include/epseon/gpu/algorithms/vibwa.hpp:
// 605-637, dispatches nothing); these kernels implement what its output
// buffer layout (task_configurator/algorithm_config.hpp:173-198) leaves room
// for.
//
// Discrete problem.  On the trimmed grid (Dirichlet points 0 and n-1) the
// Numerov recurrence with f_i = beta (E - V_i),
//   (1 + f_{i+1}) y_{i+1} = (2 - 10 f_i) y_i - (1 + f_{i-1}) y_{i-1},
// is A y + B diag(f) y = 0 with A = tridiag(1, -2, 1), B = tridiag(1, 10, 1).
// A and B commute, so diag(V) - B^-1 A / beta is symmetric with eigenpairs
// (E_v, y_v): the Hellmann-Feynman derivative of a level is
//   dE_v / dV_i = y_{v,i}^2 / sum_j y_{v,j}^2 = psi_{v,i}^2 h,
// psi normalised to sum_i psi_i^2 h = 1.
//
// Shots.  y is integrated in difference form (f carried at full relative
// precision, as in the refinement):
//   d_{i+1} = (d_i - (f_{i+1} + 10 f_i) y_i - f_{i-1} y_{i-1}) / (1 + f_{i+1}),
//   y_{i+1} = y_i + d_{i+1},
// once from each wall inward, both starting (y_0, y_1) = (0, 1), to the
// matching point m = argmin V (inside every level's classically allowed
// region, so both shots are stable and every lane of a wavefront walks the
// same points).  Each shot rescales by 2^-240 after every full 32 steps in
// which |y| reached 2^240.  The right shot is scaled by the least-squares
// factor c that fits it to the left one at points m and m+1.
//
// Segments.  Each side's shot is cut into segments of psi_seg_len steps.
// The normalisation runs every segment at once from two basis states
// (psi_segment_kernel: the segment's transfer map and the Gram sums of its
// columns), then chains the maps per level from the wall (normalize_kernel),
// which gives each segment's start state (a checkpoint), sum y^2 and the
// match.  The eigenfunction and adjoint passes resume every segment from its
// checkpoint in parallel.
//
// Lanes are levels of one potential; the potential table is wave-uniform and
// read with scalar loads, as in the scan.  Where the segment pass packs pairs
// of several segments into a wavefront, its lanes load their own values.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "records.hpp"

namespace epseon::hip {

namespace {

__device__ __forceinline__ double opaque(double x)
{
    asm volatile("" : "+v"(x));
    return x;
}

// 1/t for t = 1 + f in (1/2, 2): the hardware's approximation (within 2^-24)
// and a cubic step, r (1 + e + e^2) with e = 1 - t r.  The value before the
// last rounding is within 2^-72, so the result is nearly always the correctly
// rounded one (against the IEEE division, 4.3 10^9 values each: f uniform in
// (-1/2, 1/2) 12 of 10^9 differ, f log-uniform down to 2^-40 80, all by one
// unit in the last place).  The
// IEEE division spends twice the instructions on scaling and special cases
// that this range never meets: psi_segment_kernel 28 -> 21 vector instructions
// per point, 255 -> 60 registers.
__device__ __forceinline__ double reciprocal(const double t)
{
    const double r = __builtin_amdgcn_rcp(t);
    const double e = __builtin_fma(-t, r, 1.0);
    return __builtin_fma(__builtin_fma(e, e, e), r, r);
}

struct YShot {
    double y, ym, d, f, fm;
    int32_t k;

    __device__ __forceinline__ void init(const double e, const double u0, const double u1)
    {
        ym = 0.0;
        y = 1.0;
        d = 1.0;
        fm = e - u0;
        f = e - u1;
        k = 0;
    }

    __device__ __forceinline__ void step(const double u, const double e, const double c10)
    {
        const double fn = e - u;
        const double r = reciprocal(1.0 + fn);
        const double s = __builtin_fma(c10, f, fn);
        const double c = __builtin_fma(s, y, fm * ym);
        d = (d - c) * r;
        ym = y;
        y = y + d;
        fm = f;
        f = fn;
    }

    // Continue a shot from its checkpoint after j steps: u_prev and u_cur
    // are points j and j + 1 of the side's table.
    __device__ __forceinline__ void resume(const PsiCheckpoint& c, const double e, const double u_prev,
                                           const double u_cur)
    {
        y = c.y;
        ym = c.ym;
        d = c.d;
        k = c.k;
        fm = e - u_prev;
        f = e - u_cur;
    }

    // A level without a refined energy: every value stays zero.
    __device__ __forceinline__ void clear(const double e, const double u_prev, const double u_cur)
    {
        y = ym = d = 0.0;
        k = 0;
        fm = e - u_prev;
        f = e - u_cur;
    }

    // Returns the applied binary shift (0 or -240).
    __device__ __forceinline__ int32_t rescale()
    {
        const bool big = fmax(fabs(y), fabs(ym)) >= kPsiRescaleAt;
        const int32_t sh = big ? -kPsiRescaleLog2 : 0;
        y = __builtin_ldexp(y, sh);
        ym = __builtin_ldexp(ym, sh);
        d = __builtin_ldexp(d, sh);
        k += big ? kPsiRescaleLog2 : 0;
        return sh;
    }
};

// Wave-uniform table pointer in the constant address space (read-only for the
// whole launch): its loads are scalar loads.
using ConstTable = const __attribute__((address_space(4))) double*;

template <class Table>
__device__ __forceinline__ void load16(double (&buf)[16], const Table p)
{
#pragma unroll
    for (int q = 0; q < 16; ++q)
        buf[q] = p[q];
}

// 16 steps from a buffer, four at a time: their reciprocals overlap, and the
// scheduling fences keep the scheduler from computing all sixteen first (255
// registers, two wavefronts per SIMD, for no gain).
template <int Q0, class Body>
__device__ __forceinline__ void half_block(const double (&buf)[16], Body& body)
{
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        body.step(buf[q], Q0 + q);
        if (q % 4 == 3)
            __builtin_amdgcn_sched_barrier(0);
    }
}

// The last rem < 32 steps, from the two buffers.
template <int Q, class Body>
__device__ __forceinline__ void psi_tail(const double (&a)[16], const double (&b)[16], const int32_t rem, Body& body)
{
    if constexpr (Q < 31) {
        if (Q < rem) {
            body.step(Q < 16 ? a[Q % 16] : b[Q % 16], Q);
            psi_tail<Q + 1>(a, b, rem, body);
        }
    }
}

// Visit `steps` grid values p[0..steps): body.step(u, q) per value (q = index
// inside the current 32-step block), body.block_end(count, full) after each
// full block of 32 and after the tail.  Two 16-value buffers, each loaded one
// half-block ahead.  Reads up to 47 values past `steps` (tables are padded).
template <class Table, class Body>
__device__ __forceinline__ void psi_walk_from(Table p, const int32_t steps, Body& body)
{
    const int32_t nsb = steps >> 5;
    double a[16], b[16];
    load16(a, p);
    for (int32_t sb = 0; sb < nsb; ++sb) {
        load16(b, p + 16);
        half_block<0>(a, body);
        load16(a, p + 32);
        half_block<16>(b, body);
        body.block_end(32, true);
        p += 32;
    }
    const int32_t rem = steps - (nsb << 5);
    if (rem > 0) {
        load16(b, p + 16);
        psi_tail<0>(a, b, rem, body);
        body.block_end(rem, false);
    }
}

// The walk of a wavefront whose lanes share the segment.
template <class Body>
__device__ __forceinline__ void psi_walk(const double* __restrict__ table, const int32_t steps, Body& body)
{
    // Wave-uniform; stated, because a pointer whose parts were loaded after a
    // store sits in vector registers, and vector loads of the table would wait
    // in line behind the pass's own stores.
    const uint64_t at = reinterpret_cast<uint64_t>(table);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(at));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(at >> 32));
    ConstTable p = (ConstTable)((static_cast<uint64_t>(hi) << 32) | lo);
    psi_walk_from(p, steps, body);
}

// frexp exponent of m (0 for m = 0).
__device__ __forceinline__ int32_t binary_exponent(const double m)
{
    int e = 0;
    (void)__builtin_frexp(m, &e);
    return e;
}

// Pass 1, per segment: the shot's two basis solutions through the segment,
// started from (y, y_prev, d) = (1, 1, 0) and (0, -1, 1), so that a shot
// entering with (y, d) leaves with y times column a plus d times column b;
// and the Gram sums of their values at the visited points, from which the
// segment's sum of y^2 follows as a quadratic form in (y, d).  All values
// are renormalised by a power of two after every 32 steps and at the end;
// e is the accumulated exponent (the Gram sums carry it twice).
struct MatBody {
    double ay, aym, ad, by, bym, bd;
    double saa, sab, sbb;
    double f, fm, e, c10;
    int32_t ex;
    __device__ __forceinline__ void step(const double u, int)
    {
        saa = __builtin_fma(ay, ay, saa);
        sab = __builtin_fma(ay, by, sab);
        sbb = __builtin_fma(by, by, sbb);
        const double fn = e - u;
        const double r = reciprocal(1.0 + fn);
        const double sg = __builtin_fma(c10, f, fn);
        const double ca = __builtin_fma(sg, ay, fm * aym);
        const double cb = __builtin_fma(sg, by, fm * bym);
        ad = (ad - ca) * r;
        bd = (bd - cb) * r;
        aym = ay;
        bym = by;
        ay = ay + ad;
        by = by + bd;
        fm = f;
        f = fn;
    }
    __device__ __forceinline__ void renormalize()
    {
        const double mx = fmax(fmax(fmax(fabs(ay), fabs(aym)), fmax(fabs(ad), fabs(by))),
                               fmax(fabs(bym), fabs(bd)));
        const int32_t x = binary_exponent(mx);
        ay = __builtin_ldexp(ay, -x);
        aym = __builtin_ldexp(aym, -x);
        ad = __builtin_ldexp(ad, -x);
        by = __builtin_ldexp(by, -x);
        bym = __builtin_ldexp(bym, -x);
        bd = __builtin_ldexp(bd, -x);
        saa = __builtin_ldexp(saa, -2 * x);
        sab = __builtin_ldexp(sab, -2 * x);
        sbb = __builtin_ldexp(sbb, -2 * x);
        ex += x;
    }
    __device__ __forceinline__ void block_end(int32_t, const bool full)
    {
        if (full)
            renormalize();
    }
};

// Pass 2, eigenfunction output: psi_i = y_i * mult written to row[i0 + dir*j].
struct PsiBody {
    YShot s;
    double e, c10, a, mult;
    int32_t kf, i0, dir, base;
    // Staging: lane l's 32 values of a block go to tile[l], then the wave
    // writes them out, 16 lanes to a row and two values to a lane.
    double (*tile)[33];
    double* rows;  // row of the wave's first level, at the trimmed window's first point
    int64_t stride;
    int32_t nrows;
    __device__ __forceinline__ void step(const double u, const int q)
    {
        tile[threadIdx.x][q] = s.y * mult;
        s.step(u, e, c10);
    }
    __device__ __forceinline__ void block_end(const int32_t count, const bool full)
    {
        __syncthreads();
        const int32_t c = 2 * static_cast<int32_t>(threadIdx.x & 15);
        const int32_t h = static_cast<int32_t>(threadIdx.x >> 4);
        // Steps c and c + 1, in the order of their addresses.
        const int32_t lo = dir > 0 ? c : c + 1, hi = dir > 0 ? c + 1 : c;
        double* p = rows + static_cast<int64_t>(h) * stride + (i0 + dir * (base + lo));
        if (full && nrows == 64) {
#pragma unroll
            for (int32_t r = 0; r < 64; r += 4, p += 4 * stride) {
                typedef double pair __attribute__((ext_vector_type(2), aligned(8)));
                *reinterpret_cast<pair*>(p) = pair{tile[r + h][lo], tile[r + h][hi]};
            }
        } else {
            for (int32_t r = h; r < nrows; r += 4, p += 4 * stride) {
                if (lo < count)
                    p[0] = tile[r][lo];
                if (hi < count)
                    p[1] = tile[r][hi];
            }
        }
        __syncthreads();
        base += count;
        if (full) {
            (void)s.rescale();
            mult = __builtin_ldexp(a, s.k - kf);
        }
    }
};

// Pass 2, adjoint: lane contribution g h psi_i^2 = G y_i^2 staged in LDS and
// summed over the block's levels per point, 32 points at a time.
template <int W>
struct VjpBody {
    YShot s;
    double e, c10, g0, G;
    int32_t kf, i0, dir, base;
    bool accumulate;
    double (*sc)[32][65];  // [W][32][64 lanes + 1 pad]
    double (*sw)[32];      // [W][32]
    double* out;

    __device__ __forceinline__ void step(const double u, const int q)
    {
        const int32_t wv = static_cast<int32_t>(threadIdx.x >> 6);
        const int32_t ln = static_cast<int32_t>(threadIdx.x & 63);
        sc[wv][q][ln] = (G * s.y) * s.y;
        s.step(u, e, c10);
    }

    __device__ __forceinline__ void block_end(const int32_t count, const bool full)
    {
        const int32_t wv = static_cast<int32_t>(threadIdx.x >> 6);
        const int32_t ln = static_cast<int32_t>(threadIdx.x & 63);
        __syncthreads();
        const int32_t j = ln & 31;
        const int32_t h = (ln >> 5) * 32;
        double acc = 0.0;
#pragma unroll
        for (int t = 0; t < 32; ++t)
            acc += sc[wv][j][h + t];
        acc += __shfl_xor(acc, 32);
        if (ln < 32)
            sw[wv][j] = acc;
        __syncthreads();
        const int32_t t = static_cast<int32_t>(threadIdx.x);
        if (t < count) {
            double tot = sw[0][t];
#pragma unroll
            for (int w = 1; w < W; ++w)
                tot += sw[w][t];
            double* o = out + (i0 + dir * (base + t));
            *o = accumulate ? *o + tot : tot;
        }
        base += count;
        if (full) {
            (void)s.rescale();
            G = __builtin_ldexp(g0, 2 * (s.k - kf));
        }
    }
};

__device__ __forceinline__ bool level_active(const int32_t* __restrict__ status, const int64_t o)
{
    return status[o] == 0;
}

}  // namespace

// Shot segment of a PsiTask: the side's table, the first step j0 and the
// number of steps.
struct PsiSegment {
    const double* p;
    int32_t j0, steps;
};

__device__ __forceinline__ PsiSegment psi_segment(const PotentialRecord& P, const double* __restrict__ uv,
                                                  const double* __restrict__ uvr, const PsiTask& t)
{
    const int32_t total = t.side == 0 ? P.match : P.n_points - 2 - P.match;
    const int32_t last = (t.side == 0 ? P.psi_segs_left : P.psi_segs_right) - 1;
    const int32_t at = t.segment * P.psi_seg_len - psi_shift(P.first_point, P.n_points, t.side);
    const int32_t j0 = max(0, at), j1 = t.segment == last ? total : at + P.psi_seg_len;
    return PsiSegment{(t.side == 0 ? uv : uvr) + P.ut_offset, j0, j1 - j0};
}

__device__ __forceinline__ int64_t psi_slot(const PotentialRecord& P, const int32_t side, const int32_t segment,
                                            const int32_t l)
{
    return P.psi_ckpt + static_cast<int64_t>((side == 0 ? 0 : P.psi_segs_left) + segment) * P.level_count + l;
}

// Start a segment's shot: from the wall (segment 0), from the normalisation
// pass's checkpoint, or all zero for a level that did not converge.
__device__ __forceinline__ void psi_start(YShot& s, const PotentialRecord& P, const PsiTask& t,
                                          const PsiSegment& g, const PsiCheckpoint* __restrict__ ckpt,
                                          const int32_t l, const bool active, const double e)
{
    if (!active)
        s.clear(e, g.p[g.j0], g.p[g.j0 + 1]);
    else if (t.segment == 0)
        s.init(e, g.p[0], g.p[1]);
    else
        s.resume(ckpt[psi_slot(P, t.side, t.segment, l)], e, g.p[g.j0], g.p[g.j0 + 1]);
}

// Pass 1a: one wavefront per eigenfunction task (potential, 64 levels, side,
// segment): each converged level's segment matrix and Gram sums.
// kPacked: the wavefronts of a potential's tasks take its (segment, level)
// pairs in order, 64 each (a pair's number is its slot), and those past the
// last pair leave.  A lane then loads its own segment's values.
template <bool kPacked>
__global__ __launch_bounds__(64) void psi_segment_kernel(
    const double* __restrict__ uv, const double* __restrict__ uvr,
    const PotentialRecord* __restrict__ pots, const PsiTask* __restrict__ tasks,
    const double* __restrict__ levels, const int32_t* __restrict__ status,
    PsiSegMatrix* __restrict__ mats)
{
    PsiTask task = tasks[blockIdx.x];
    const PotentialRecord& P = pots[task.potential];
    int32_t l = task.first + static_cast<int32_t>(threadIdx.x);
    if (P.flags != 0)
        return;
    if constexpr (kPacked) {
        const int32_t segment = (task.side == 0 ? 0 : P.psi_segs_left) + task.segment;
        const int64_t pair =
            (static_cast<int64_t>(segment) * ((P.level_count + 63) / 64) + task.first / 64) * 64 + threadIdx.x;
        if (pair >= static_cast<int64_t>(P.psi_segs_left + P.psi_segs_right) * P.level_count)
            return;
        const int32_t at = static_cast<int32_t>(pair / P.level_count);
        l = static_cast<int32_t>(pair - static_cast<int64_t>(at) * P.level_count);
        task.side = at < P.psi_segs_left ? 0 : 1;
        task.segment = at - (task.side == 0 ? 0 : P.psi_segs_left);
    } else if (l >= P.level_count) {
        return;
    }
    const int64_t o = P.level_offset + l;
    if (!level_active(status, o))
        return;
    const double e = P.beta * levels[o];
    const PsiSegment g = psi_segment(P, uv, uvr, task);
    MatBody B{};
    B.ay = 1.0;
    B.aym = 1.0;
    B.ad = 0.0;
    B.by = 0.0;
    B.bym = -1.0;
    B.bd = 1.0;
    B.e = e;
    B.c10 = opaque(10.0);
    B.fm = e - g.p[g.j0];
    B.f = e - g.p[g.j0 + 1];
    if constexpr (kPacked)
        psi_walk_from(g.p + 2 + g.j0, g.steps, B);
    else
        psi_walk(g.p + 2 + g.j0, g.steps, B);
    B.renormalize();
    mats[psi_slot(P, task.side, task.segment, l)] =
        PsiSegMatrix{B.ay, B.aym, B.ad, B.by, B.bym, B.bd, B.saa, B.sab, B.sbb, B.ex, 0};
}

// End state of one side's chained shot.
struct SideEnd {
    double y, ym, sum;
    int32_t k;
};

// One side's shot, chained segment by segment.
struct SideChain {
    double y, ym, d, sum;
    int32_t k;
    __device__ __forceinline__ PsiCheckpoint state() const { return PsiCheckpoint{y, ym, d, k, 0}; }
    __device__ __forceinline__ void append(const PsiSegMatrix& M)
    {
        const double g = __builtin_fma(y * y, M.saa, __builtin_fma(2.0 * y * d, M.sab, d * d * M.sbb));
        const double yn = __builtin_fma(M.ay, y, M.by * d);
        const double ymn = __builtin_fma(M.aym, y, M.bym * d);
        const double dn = __builtin_fma(M.ad, y, M.bd * d);
        const int32_t x = binary_exponent(fmax(fmax(fabs(yn), fabs(ymn)), fabs(dn)));
        y = __builtin_ldexp(yn, -x);
        ym = __builtin_ldexp(ymn, -x);
        d = __builtin_ldexp(dn, -x);
        // y^2 sum relative to 2^(2k) of the new exponent k + e + x.
        sum = __builtin_ldexp(sum, -2 * (M.e + x)) + __builtin_ldexp(g, -2 * x);
        k += M.e + x;
    }
};

// Pass 1b: two wavefronts per 64 levels of one potential, one lane per level
// and side.  Chains the segment matrices of the side from its wall,
// (y, y_prev, d) = (1, 0, 1), renormalising by a power of two after each
// product, and writes the checkpoint (state and binary exponent) at each later
// segment start and the sum of y^2 as the segments' quadratic forms; then the
// sides meet at m and the first wavefront writes the levels' LevelNorm
// (exponents in bits).  Bound by the chain's latency: the matrices are loaded
// kAhead segments before their use, which leaves about 15 dependent FP64
// operations per segment.
__global__ __launch_bounds__(128) void normalize_kernel(
    const PotentialRecord* __restrict__ pots, const WaveTask* __restrict__ tasks, const int32_t n_tasks,
    const int32_t* __restrict__ status, const PsiSegMatrix* __restrict__ mats,
    PsiCheckpoint* __restrict__ ckpt, LevelNorm* __restrict__ norms)
{
    constexpr int32_t kAhead = 4;
    __shared__ SideEnd s_right[64];
    const int32_t tid = static_cast<int32_t>(blockIdx.x);
    if (tid >= n_tasks)
        return;
    const WaveTask task = tasks[tid];
    const PotentialRecord& P = pots[task.potential];
    const int32_t lane = static_cast<int32_t>(threadIdx.x & 63);
    const int32_t side = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(threadIdx.x >> 6));
    const int32_t l = task.first + lane;
    const int64_t o = P.level_offset + l;
    const bool valid = l < P.level_count;
    const bool active = valid && P.flags == 0 && level_active(status, o);
    SideEnd end{1.0, 0.0, 0.0, 0};
    if (active) {
        const int32_t segs = side == 0 ? P.psi_segs_left : P.psi_segs_right;
        const int64_t stride = P.level_count;
        const int64_t slot0 = psi_slot(P, side, 0, l);
        SideChain c{1.0, 0.0, 1.0, 0.0, 0};
        PsiSegMatrix next[kAhead];
#pragma unroll
        for (int32_t q = 0; q < kAhead; ++q)
            next[q] = mats[slot0 + min(q, segs - 1) * stride];
        int32_t sg = 0;
        // The first segment's checkpoint (the wall) is written like the
        // others and never read.
        for (; sg + kAhead <= segs; sg += kAhead) {
#pragma unroll
            for (int32_t q = 0; q < kAhead; ++q) {
                ckpt[slot0 + (sg + q) * stride] = c.state();
                c.append(next[q]);
                next[q] = mats[slot0 + min(sg + q + kAhead, segs - 1) * stride];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int32_t q = 0; q < kAhead - 1; ++q)
            if (sg + q < segs) {
                ckpt[slot0 + (sg + q) * stride] = c.state();
                c.append(next[q]);
            }
        end = SideEnd{c.y, c.ym, c.sum, c.k};
    }
    if (side == 1)
        s_right[lane] = end;
    __syncthreads();
    if (side == 1 || !valid)
        return;
    if (!active) {
        norms[o] = LevelNorm{0.0, 0.0, 0, 0};
        return;
    }
    const SideEnd right = s_right[lane];
    // Left: (y_m, y_{m+1}) = (ym, y); right (reversed): (y_{m+1}, y_m) = (ym, y);
    // the right shot scaled by c = cm 2^(k_left - k_right).
    const double num = __builtin_fma(end.ym, right.y, end.y * right.ym);
    const double den = __builtin_fma(right.y, right.y, right.ym * right.ym);
    const double cm = num / den;
    const double s = __builtin_fma(cm * cm, right.sum, end.sum);
    const double a = 1.0 / sqrt(s * P.h);
    norms[o] = LevelNorm{a, cm * a, end.k, right.k};
}

// Eigenfunctions: for each task (potential, first level, side, segment), the
// segment's points of rows first.. of that potential (full_points values per
// row at out[psi_offset - base + l * full_points]), re-run from the
// normalisation pass's checkpoints, staged in LDS and stored 32 contiguous
// values at a time (from the second segment on from the start of a 128-byte
// line where the rows have one: stores that straddled lines filled L2 with
// partly written ones, 2.2 TB/s against 4.0 on 8 x 200,000 points x 80 levels); the segment-0 tasks also zero the row outside the open
// trimmed window on their side (the whole row of an unresolved potential,
// whose only task is side 0, segment 0).  Zero for levels that did not
// converge.  One lane per level.
__global__ __launch_bounds__(64) void eigenfunction_kernel(
    const double* __restrict__ uv, const double* __restrict__ uvr,
    const PotentialRecord* __restrict__ pots, const PsiTask* __restrict__ tasks,
    const double* __restrict__ levels, const int32_t* __restrict__ status,
    const LevelNorm* __restrict__ norms, const PsiCheckpoint* __restrict__ ckpt, const int64_t base,
    double* __restrict__ out)
{
    __shared__ double s_tile[64][33];
    const PsiTask task = tasks[blockIdx.x];
    const PotentialRecord& P = pots[task.potential];
    const int32_t l = task.first + static_cast<int32_t>(threadIdx.x);
    const int32_t nrows = min(64, P.level_count - task.first);
    const bool valid = l < P.level_count;
    const int64_t N = P.full_points;
    double* row0 = out + (P.psi_offset - base) + static_cast<int64_t>(task.first) * N;
    double* row = row0 + static_cast<int64_t>(threadIdx.x) * N;
    const int64_t first = P.first_point;
    const int32_t n = P.n_points;
    const bool ok = P.flags == 0;
    if (task.segment == 0 && valid) {
        if (!ok) {
            for (int64_t i = 0; i < N; ++i)
                row[i] = 0.0;
        } else if (task.side == 0) {
            for (int64_t i = 0; i <= first; ++i)
                row[i] = 0.0;
        } else {
            for (int64_t i = first + n - 1; i < N; ++i)
                row[i] = 0.0;
        }
    }
    if (!ok)
        return;
    const int64_t o = P.level_offset + l;
    const bool active = valid && level_active(status, o);
    const LevelNorm nm = active ? norms[o] : LevelNorm{0.0, 0.0, 0, 0};
    const double e = P.beta * (active ? levels[o] : P.e_lo);
    const PsiSegment g = psi_segment(P, uv, uvr, task);

    PsiBody B{};
    B.e = e;
    B.c10 = opaque(10.0);
    B.a = task.side == 0 ? nm.a_left : nm.a_right;
    B.kf = task.side == 0 ? nm.k_left : nm.k_right;
    B.i0 = task.side == 0 ? 1 : n - 2;
    B.dir = task.side == 0 ? 1 : -1;
    B.base = g.j0;
    B.tile = s_tile;
    B.rows = row0 + first;
    B.stride = N;
    B.nrows = nrows;
    psi_start(B.s, P, task, g, ckpt, l, active, e);
    B.mult = __builtin_ldexp(B.a, B.s.k - B.kf);
    psi_walk(g.p + 2 + g.j0, g.steps, B);
}

// Adjoint: grad_v[user_offset + i] = sum_l grad_levels[l] psi_l(i)^2 h over
// the converged levels of the task's potential, zero elsewhere on the
// potential's full grid.  One block of W wavefronts per task (potential,
// side, segment): the segment's points, levels in groups of 64 W, the first
// group storing and later ones adding, so the sum order is fixed.  The
// segment-0 tasks also zero the points outside the open trimmed window on
// their side (all points of an unresolved potential, whose only task is side
// 0, segment 0).
template <int W>
__global__ __launch_bounds__(64 * W) void level_vjp_kernel(
    const double* __restrict__ uv, const double* __restrict__ uvr,
    const PotentialRecord* __restrict__ pots, const PsiTask* __restrict__ tasks,
    const double* __restrict__ levels, const int32_t* __restrict__ status,
    const LevelNorm* __restrict__ norms, const PsiCheckpoint* __restrict__ ckpt,
    const double* __restrict__ grad_levels, double* __restrict__ grad_v)
{
    __shared__ double s_c[W][32][65];
    __shared__ double s_w[W][32];
    const PsiTask task = tasks[blockIdx.x];
    const PotentialRecord& P = pots[task.potential];
    double* out = grad_v + P.user_offset;
    const int32_t N = P.full_points;
    const int32_t n = P.n_points;
    const int32_t first = static_cast<int32_t>(P.first_point);
    const bool ok = P.flags == 0;
    const int32_t t = static_cast<int32_t>(threadIdx.x);
    if (task.segment == 0) {
        if (!ok) {
            for (int32_t i = t; i < N; i += 64 * W)
                out[i] = 0.0;
            return;
        }
        if (task.side == 0)
            for (int32_t i = t; i <= first; i += 64 * W)
                out[i] = 0.0;
        else
            for (int32_t i = first + n - 1 + t; i < N; i += 64 * W)
                out[i] = 0.0;
    }
    if (!ok)
        return;
    const PsiSegment g = psi_segment(P, uv, uvr, task);
    const int32_t i0 = task.side == 0 ? 1 : n - 2;
    const int32_t dir = task.side == 0 ? 1 : -1;
    double* win = out + first;
    if (P.level_count == 0) {
        for (int32_t q = t; q < g.steps; q += 64 * W)
            win[i0 + dir * (g.j0 + q)] = 0.0;
        return;
    }
    const double c10 = opaque(10.0);
    for (int32_t g0 = 0; g0 < P.level_count; g0 += 64 * W) {
        const int32_t l = g0 + t;
        const int64_t o = P.level_offset + l;
        const bool active = l < P.level_count && level_active(status, o);
        const LevelNorm nm = active ? norms[o] : LevelNorm{0.0, 0.0, 0, 0};
        const double gl = active ? grad_levels[o] : 0.0;
        const double e = P.beta * (active ? levels[o] : P.e_lo);
        const double a = task.side == 0 ? nm.a_left : nm.a_right;

        VjpBody<W> B{};
        B.e = e;
        B.c10 = c10;
        B.g0 = gl * P.h * a * a;
        B.kf = task.side == 0 ? nm.k_left : nm.k_right;
        B.i0 = i0;
        B.dir = dir;
        B.base = g.j0;
        B.accumulate = g0 > 0;
        B.sc = s_c;
        B.sw = s_w;
        B.out = win;
        psi_start(B.s, P, task, g, ckpt, l, active, e);
        B.G = __builtin_ldexp(B.g0, 2 * (B.s.k - B.kf));
        psi_walk(g.p + 2 + g.j0, g.steps, B);
    }
}

// ---------------------------------------------------------------- launchers

hipError_t launch_normalize(hipStream_t stream, const double* uv, const double* uvr,
                            const PotentialRecord* pots, const PsiTask* psi_tasks, int32_t n_psi_tasks, bool packed,
                            const WaveTask* tasks, int32_t n_tasks, const double* levels,
                            const int32_t* status, PsiSegMatrix* mats, PsiCheckpoint* ckpt, LevelNorm* norms)
{
    if (n_psi_tasks > 0) {
        if (packed)
            hipLaunchKernelGGL(psi_segment_kernel<true>, dim3(static_cast<unsigned>(n_psi_tasks)), dim3(64), 0, stream,
                               uv, uvr, pots, psi_tasks, levels, status, mats);
        else
            hipLaunchKernelGGL(psi_segment_kernel<false>, dim3(static_cast<unsigned>(n_psi_tasks)), dim3(64), 0, stream,
                               uv, uvr, pots, psi_tasks, levels, status, mats);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess)
            return e;
    }
    if (n_tasks == 0)
        return hipSuccess;
    hipLaunchKernelGGL(normalize_kernel, dim3(static_cast<unsigned>(n_tasks)), dim3(128), 0, stream, pots, tasks,
                       n_tasks, status, mats, ckpt, norms);
    return hipGetLastError();
}

hipError_t launch_eigenfunctions(hipStream_t stream, const double* uv, const double* uvr,
                                 const PotentialRecord* pots, const PsiTask* tasks, int32_t n_tasks,
                                 const double* levels, const int32_t* status, const LevelNorm* norms,
                                 const PsiCheckpoint* ckpt, int64_t base, double* out)
{
    if (n_tasks == 0)
        return hipSuccess;
    hipLaunchKernelGGL(eigenfunction_kernel, dim3(static_cast<unsigned>(n_tasks)), dim3(64), 0, stream,
                       uv, uvr, pots, tasks, levels, status, norms, ckpt, base, out);
    return hipGetLastError();
}

hipError_t launch_level_vjp(hipStream_t stream, int32_t waves, const double* uv, const double* uvr,
                            const PotentialRecord* pots, const PsiTask* tasks, int32_t n_tasks,
                            const double* levels, const int32_t* status, const LevelNorm* norms,
                            const PsiCheckpoint* ckpt, const double* grad_levels, double* grad_v)
{
    if (n_tasks == 0)
        return hipSuccess;
    const dim3 grid(static_cast<unsigned>(n_tasks));
#define EPSEON_VJP(Wv)                                                                               \
    hipLaunchKernelGGL(level_vjp_kernel<Wv>, grid, dim3(64 * (Wv)), 0, stream, uv, uvr, pots, tasks, \
                       levels, status, norms, ckpt, grad_levels, grad_v)
    switch (waves) {
    case 1:
        EPSEON_VJP(1);
        break;
    case 2:
        EPSEON_VJP(2);
        break;
    case 3:
        EPSEON_VJP(3);
        break;
    case 4:
        EPSEON_VJP(4);
        break;
    default:
        return hipErrorInvalidValue;
    }
#undef EPSEON_VJP
    return hipGetLastError();
}

}  // namespace epseon::hip
