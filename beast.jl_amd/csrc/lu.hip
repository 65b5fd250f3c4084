// Dense complex LU with partial pivoting and the solves behind Z \ b.
//
// Reference: the reference factors its Matrix{ComplexF64} with LAPACK getrf and
// solves with getrs through LinearAlgebra (src/solvers/lusolver.jl:26-34,
// BEAST.lu in src/solvers/lu.jl:29-47).  Here the matrix stays in HBM, row-major
// interleaved complex, and is factored by a right-looking blocked LU
// (Golub & Van Loan, Matrix Computations, Alg. 3.4.x).
//
// FP64 factors (block depth 256) keep LAPACK's pivots exactly:
//   k_panel64       32-column panel, one row per thread in registers; per column the
//                   workgroups exchange pivot candidates through tagged words in
//                   device memory.  Pivot choice is LAPACK's: largest |Re|+|Im|,
//                   first row on ties.
//   k_apply64       the panel's row moves and its block row in the block's other
//                   columns; 32-row unit-lower solves of the wide block rows.
// FP32 factors (block depth 1024 while the trailing matrix is large, factored as
// two 512-column halves, then 512) pivot each 32-column panel by tournament
// (communication-avoiding LU, Grigori, Demmel & Xiang, SIAM J. Matrix Anal. Appl.
// 32 (2011)):
//   k_tslu_panel    one launch per panel: 512 rows per workgroup, two per thread
//                   in registers, reduced to 32 candidates by partial pivoting;
//                   the last workgroup of each group to finish merges the group one
//                   level up, and the last merge emits L11\U11, ipiv and the row
//                   moves.  Further workgroups carry the previous panel's update of
//                   the block.
//   k_tslu_apply    moves the rows in the block's other columns, solves the panel's
//                   block row, turns the panel rows into L21 = A21 U11^-1 and brings
//                   the next panel up to date.
// Shared by both:
//   The next block column is factored on a second stream while the trailing
//   update of the current one runs (look-ahead by one block).
//   k_swap_plan, k_laswp_apply  row interchanges: the sequential swaps replayed
//                   once on row indices, then each moved row moved once.
//   k_cgemm         C -= A B on MFMA (v_mfma_{f32,f64}_16x16x4): FP64 updates and
//                   the FP32 updates inside a block column.
//   k_cgemm_bf16x3  FP32 trailing update from split-bf16 planes (hi*hi + hi*lo +
//                   lo*hi on v_mfma_f32_16x16x32_bf16, FP32 accumulation).
// Solves: permutation gather, then one launch per triangle: for FP64 factors a
// substitution in 64-row blocks (k_trsv64), for FP32 factors 128-row blocks with
// inverted diagonal blocks and their couplings (k_trinv, k_blk_coupling,
// k_trsv_flag).  FP32 factors precondition flexible GMRES
// inside iterative refinement in FP64 (GMRES-IR, Carson & Higham, SIAM J. Sci.
// Comput. 40 (2018)), whose residuals use the resident FP64 matrix.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <mutex>
#include <climits>
#include <cmath>
#include <complex>
#include <cstring>
#include <limits>
#include <map>
#include <memory>
#include <vector>

#include "bh_device.h"
#include "bh_internal.h"
#include "bh_matrix.h"
#include "lu_rules.h"
#include "panel_gate.h"

namespace bh {

template <typename T>
struct CT;
template <>
struct CT<float> {
    using t = float2;
};
template <>
struct CT<double> {
    using t = double2;
};

template <typename V>
__device__ __forceinline__ V cmulv(V a, V b)
{
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}

template <typename V>
__device__ __forceinline__ V csubv(V a, V b)
{
    return {a.x - b.x, a.y - b.y};
}

// a b and a - b c with the contraction written out: the same bits wherever they are inlined
__device__ __forceinline__ float2 cmul_x(float2 a, float2 b)
{
    return {fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x)};
}

__device__ __forceinline__ float2 cfms_x(float2 a, float2 b, float2 c)
{
    return {fmaf(b.y, c.y, fmaf(-b.x, c.x, a.x)), fmaf(-b.y, c.x, fmaf(-b.x, c.y, a.y))};
}

__device__ __forceinline__ double2 cfma_x(double2 a, double2 b, double2 c)   // a + b c
{
    return {fma(-b.y, c.y, fma(b.x, c.x, a.x)), fma(b.y, c.x, fma(b.x, c.y, a.y))};
}

__device__ __forceinline__ double2 cfms_x(double2 a, double2 b, double2 c)
{
    return {fma(b.y, c.y, fma(-b.x, c.x, a.x)), fma(-b.y, c.x, fma(-b.x, c.y, a.y))};
}

// Maximum over a wave of unsigned keys (DPP: quad, half-row and row mirrors, then
// the row broadcasts of lanes 15 and 31), read from lane 63.
__device__ __forceinline__ unsigned wave_max_u32(unsigned v)
{
    int x = (int)v;
    x = (int)max((unsigned)x, (unsigned)__builtin_amdgcn_update_dpp(x, x, 0xB1, 0xF, 0xF, false));   // quad_perm 1,0,3,2
    x = (int)max((unsigned)x, (unsigned)__builtin_amdgcn_update_dpp(x, x, 0x4E, 0xF, 0xF, false));   // quad_perm 2,3,0,1
    x = (int)max((unsigned)x, (unsigned)__builtin_amdgcn_update_dpp(x, x, 0x141, 0xF, 0xF, false));  // row_half_mirror
    x = (int)max((unsigned)x, (unsigned)__builtin_amdgcn_update_dpp(x, x, 0x140, 0xF, 0xF, false));  // row_mirror
    x = (int)max((unsigned)x, (unsigned)__builtin_amdgcn_update_dpp(x, x, 0x142, 0xA, 0xF, false));  // row_bcast:15
    x = (int)max((unsigned)x, (unsigned)__builtin_amdgcn_update_dpp(x, x, 0x143, 0xC, 0xF, false));  // row_bcast:31
    return (unsigned)__builtin_amdgcn_readlane(x, 63);
}

// ---------------------------------------------------------------- FP64 panel
// A 32-column panel with LAPACK's partial pivoting.  Each thread holds one row of the panel
// in registers for the whole panel; rows do not move, each tracks the position that the
// interchanges give it and is stored there at the end.  Per column: every wave finds its
// best row (largest |Re|+|Im|, smallest position on ties) by DPP, puts that row into LDS,
// and after one barrier the workgroup knows its best.  One workgroup (the last rows) goes on
// from there.  Several exchange their candidates through slots in device memory: each
// publishes value, position and row as 64-bit words that carry the column's tag in their
// low bits, so a word is valid by itself and neither fences nor counters are needed; one
// wave of each workgroup reads all slots, takes the best and reads that row.  Slots
// alternate by column parity: a workgroup rewrites one only after every workgroup has
// published the next column, i.e. has read this one.
// Bound by latency: per column about one store and two dependent loads across the XCDs, and
// the rows' way through LDS.  Measured on the MI355X per panel of 32 columns, before (rows in
// LDS at a stride that put a wave's accesses on one bank, a grid barrier per column) and now:
// 17,406 rows 398 us alone -> 251 us beside the trailing products; 702 rows, three
// workgroups, 238 -> 123 us; up to 512 rows, one workgroup, 93 us.
// The columns run in four phases of eight.  In a phase the live columns shift down by one
// register per column and the finished multipliers enter at the end, so that the column
// being eliminated is always the phase's first register (a full unroll does not fit the
// instruction cache, a dynamic column index would put the row into scratch memory).
// Finished columns meet zeros in the pivot row.
constexpr int kP64Phase = 8;
constexpr int kP64T = 256;         // rows per workgroup beside the trailing products: the registers of half a CU,
                                   // as their workgroups, so that neither waits for a whole CU to drain
constexpr int kP64TOne = 512;      // rows of the panels that one workgroup takes
constexpr long long kP64WaitTicks = 2000000000LL;   // 20 s of the 100 MHz clock, then the panel reports an error

struct Panel64Slots {
    int stride;                // slots per parity: that of the largest panel, so that a slot keeps its place
    unsigned long long *key;   // [2][stride][2]: value bits 63..12 | tag 12; value bits 11..0, position 32, tag 20
    unsigned long long *row;   // [2][stride][4 kPW]: for each of the row's doubles its high and low half, each | tag 32
    int *info;                 // first zero pivot (1-based), 0 if none, -1: a wait ran out
    int *moves;                // [2 kPW]: row that ends at c + i; position where row c + i ends below the panel (-1: none)
};

__device__ __forceinline__ void put_word(unsigned long long *p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ unsigned long long get_word(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a candidate: value bits + 1 in (hi, lo) order, hi = 0 for none; smaller position on ties
struct Cand64 {
    unsigned hi, lo, pos;
};

__device__ __forceinline__ bool better(const Cand64 &a, const Cand64 &b)
{
    return a.hi != b.hi ? a.hi > b.hi : (a.lo != b.lo ? a.lo > b.lo : a.pos < b.pos);
}

// lane of the wave's best candidate (any lane if there is none)
__device__ __forceinline__ int best_lane(const Cand64 &k)
{
    const unsigned H = wave_max_u32(k.hi);
    unsigned long long m = __ballot(k.hi == H);
    if (m & (m - 1)) {
        const unsigned L = wave_max_u32(k.hi == H ? k.lo : 0u);
        m = __ballot(k.hi == H && k.lo == L);
        if (m & (m - 1)) {
            const unsigned Q = wave_max_u32(k.hi == H && k.lo == L ? ~k.pos : 0u);
            m = __ballot(k.hi == H && k.lo == L && ~k.pos == Q);
        }
    }
    return __ffsll((long long)m) - 1;
}

template <int NT>
struct Panel64Lds {
    double2 row[2][NT / 64][kPW];     // the waves' best rows
    Cand64 key[2][NT / 64];
    double2 u[kPW];                   // the pivot row (several workgroups)
    int pos;                          // its position
};

template <int NT, int C0>
__device__ __forceinline__ void panel64_phase(double2 (&v)[kPW], int &pos, bool &used, bool valid, int k0, int pw,
                                              long long *ipiv, const Panel64Slots &w, Panel64Lds<NT> &S)
{
    constexpr int W = kPW - C0, NW = NT / 64;
    constexpr bool kMany = NT == kP64T;   // several workgroups
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int G = gridDim.x, g = blockIdx.x;
#pragma unroll 1
    for (int t = 0; t < kP64Phase; ++t) {
        const int j = C0 + t, c = k0 + j, par = j & 1;
        if (j >= pw) {   // past the last column of a narrow panel: only the shift
            const double2 v0 = v[C0];
#pragma unroll
            for (int q = 1; q < W; ++q) v[C0 + q - 1] = v[C0 + q];
            v[kPW - 1] = v0;
            continue;
        }
        Cand64 k{0u, 0u, (unsigned)pos};
        if (valid && !used) {
            double mag = fabs(v[C0].x) + fabs(v[C0].y);
            if (!(mag >= 0.0)) mag = 0.0;   // a NaN ranks last
            const unsigned long long b = (unsigned long long)__double_as_longlong(mag);
            k.hi = (unsigned)(b >> 32) + 1u;
            k.lo = (unsigned)b;
        }
        const int wl = best_lane(k);
        if (lane == wl) {
            S.key[par][wid] = k;
#pragma unroll
            for (int q = 0; q < W; ++q) {
                double2 x = v[C0 + q];
                if (q > W - kP64Phase && q >= W - t) x = double2{0.0, 0.0};   // finished columns
                S.row[par][wid][q] = x;
            }
        }
        __syncthreads();
        Cand64 best = S.key[par][0];
        int wb = 0;
#pragma unroll
        for (int q = 1; q < NW; ++q) {
            const Cand64 kq = S.key[par][q];
            if (better(kq, best)) { best = kq; wb = q; }
        }
        const double2 *u = S.row[par][wb];
        int p = best.hi ? (int)best.pos : c;
        if constexpr (kMany) {
            const unsigned tag = (unsigned)c + 1u;
            if (wid == 0) {   // publish: lane l writes double l of the row
                if (lane < 2 * W) {
                    const unsigned long long b = (unsigned long long)__double_as_longlong(((const double *)u)[lane]);
                    unsigned long long *o = w.row + ((size_t)par * w.stride + g) * 4 * kPW + 2 * lane;
                    put_word(o, (b & 0xffffffff00000000ull) | tag);
                    put_word(o + 1, (b << 32) | tag);
                }
                if (lane == 0) {
                    const unsigned long long b = best.hi ? ((unsigned long long)best.hi << 32) | best.lo : 0ull;
                    unsigned long long *o = w.key + ((size_t)par * w.stride + g) * 2;
                    put_word(o, (b & ~0xfffull) | (tag & 0xfffu));
                    put_word(o + 1, (b << 52) | ((unsigned long long)(unsigned)best.pos << 20) | (tag & 0xfffffu));
                }
            }
            if (wid == NW - 1) {
                Cand64 mine{0u, 0u, 0u};
                int mg = 0;
                const long long t0 = wall_clock64();
                bool late = false;
                int spins = 0;
                for (int q0 = 0; q0 < G; q0 += 64) {
                    const int q = q0 + lane;
                    const unsigned long long *o = w.key + ((size_t)par * w.stride + min(q, G - 1)) * 2;
                    unsigned long long a, b;
                    for (;;) {
                        a = get_word(o);
                        b = get_word(o + 1);
                        const bool ok = (a & 0xfffu) == (tag & 0xfffu) && (b & 0xfffffu) == (tag & 0xfffffu);
                        if (__all(ok)) break;
                        // a wait that has run out ends the others too
                        if ((++spins & 1023) == 0 &&
                            (wall_clock64() - t0 > kP64WaitTicks ||
                             __hip_atomic_load(w.info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < 0)) {
                            late = true;
                            break;
                        }
                    }
                    const unsigned long long b64 = (a & ~0xfffull) | (b >> 52);
                    const Cand64 kq{(unsigned)(b64 >> 32), (unsigned)b64, (unsigned)(b >> 20)};
                    if (q < G && better(kq, mine)) { mine = kq; mg = q; }
                }
                const int bl = best_lane(mine);
                const int gb = __builtin_amdgcn_readlane(mg, bl);
                const unsigned bhi = (unsigned)__builtin_amdgcn_readlane((int)mine.hi, bl);
                const int bp = __builtin_amdgcn_readlane((int)mine.pos, bl);
                const unsigned long long *o = w.row + ((size_t)par * w.stride + gb) * 4 * kPW + 2 * min(lane, 2 * W - 1);
                unsigned long long a, b;
                for (;;) {
                    a = get_word(o);
                    b = get_word(o + 1);
                    if (late || __all((unsigned)a == tag && (unsigned)b == tag)) break;
                    if ((++spins & 1023) == 0 && wall_clock64() - t0 > kP64WaitTicks) late = true;
                }
                if (late && lane == 0) __hip_atomic_store(w.info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (lane < 2 * W)
                    ((double *)S.u)[lane] = __longlong_as_double((long long)((a & 0xffffffff00000000ull) | (b >> 32)));
                if (lane == 0) S.pos = panel64_pivot(late, bhi != 0, bp, c);
            }
            __syncthreads();
            u = S.u;
            p = S.pos;
        }
        const double2 piv = u[0];
        const bool nz = piv.x != 0.0 || piv.y != 0.0;
        if (g == 0 && tid == 0) {
            ipiv[c] = p;
            if (!nz) atomicCAS(w.info, 0, c + 1);   // a wait that ran out keeps its mark
        }
        if (valid && !used) panel64_move(pos, used, c, p);
        const double den = piv.x * piv.x + piv.y * piv.y;
        const double2 inv{piv.x / den, -piv.y / den};
        const double2 v0 = v[C0];
        const bool elim = valid && !used && nz;
        double2 l = cmulv(v0, inv);
        if (!elim) l = double2{0.0, 0.0};
#pragma unroll
        for (int q = 1; q < W; ++q) v[C0 + q - 1] = csubv(v[C0 + q], cmulv(l, u[q]));
        v[kPW - 1] = elim ? l : v0;
    }
    // the live columns are now first, the finished ones last: put them in order
    double2 f[kP64Phase];
#pragma unroll
    for (int q = 0; q < kP64Phase; ++q) f[q] = v[kPW - kP64Phase + q];
#pragma unroll
    for (int q = kPW - 1; q >= C0 + kP64Phase; --q) v[q] = v[q - kP64Phase];
#pragma unroll
    for (int q = 0; q < kP64Phase; ++q) v[C0 + q] = f[q];
}

template <int NT>
__global__ __launch_bounds__(NT, 2) void k_panel64(double2 *A, long long lda, int n, int k0, int pw, long long *ipiv,
                                                   Panel64Slots w)
{
    __shared__ Panel64Lds<NT> S;
    const int row = k0 + blockIdx.x * NT + threadIdx.x;
    const bool valid = row < n;
    double2 v[kPW];
    // each thread its own row, as it lies (turning whole-line loads through LDS is slower)
#pragma unroll
    for (int q = 0; q < kPW; ++q) v[q] = double2{0.0, 0.0};
    if (valid) {
        const double2 *src = A + (long long)row * lda + k0;
#pragma unroll
        for (int q = 0; q < kPW; ++q)
            if (q < pw) v[q] = src[q];
    }
    int pos = valid ? row : -1;
    bool used = false;
    panel64_phase<NT, 0>(v, pos, used, valid, k0, pw, ipiv, w, S);
    panel64_phase<NT, 8>(v, pos, used, valid, k0, pw, ipiv, w, S);
    panel64_phase<NT, 16>(v, pos, used, valid, k0, pw, ipiv, w, S);
    panel64_phase<NT, 24>(v, pos, used, valid, k0, pw, ipiv, w, S);
    // every workgroup has read its rows before any gets here: it published columns formed from them
    if (valid) {
        double2 *dst = A + (long long)pos * lda + k0;
#pragma unroll
        for (int q = 0; q < kPW; ++q)
            if (q < pw) dst[q] = v[q];
    }
    if (valid && pos < k0 + pw) w.moves[pos - k0] = row;
    if (valid && row < k0 + pw) w.moves[kPW + row - k0] = pos >= k0 + pw ? pos : -1;
}

// Columns beside a panel [c, c + pw), 16 per workgroup out of [a0, a1) and [b0, b1): the
// panel's row moves (moves: row that goes to c + i; position where row c + i goes below the
// panel, -1: none; NULL: no moves), and in the columns of [b0, b1) the panel's block row,
// B := L^-1 B on the rows c .. c + pw with L the unit lower triangle of Lp (stride ldl).
// Four columns to a wave, 16 lanes to a column, each with two rows: the solved entry goes
// to the column's lanes by a row broadcast.  (One thread per column took 23 us in FP64, a
// chain of 528 complex multiplications; 224 columns take 7 us this way.)
template <int K>
__device__ __forceinline__ float row_bcast(float x)   // lane K of each 16
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + K, 0xF, 0xF, true));
}

template <int K>
__device__ __forceinline__ double row_bcast(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x150 + K, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + K, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <int I, typename V>
__device__ __forceinline__ void unit_solve_step(V &x0, V &x1, const V (*L)[kPW + 1], int r)
{
    if constexpr (I < kPW - 1) {
        const V xs = I < 16 ? x0 : x1;
        const V xi{row_bcast<I & 15>(xs.x), row_bcast<I & 15>(xs.y)};
        if constexpr (I < 15) {
            const V u = cfms_x(x0, L[r][I], xi);
            if (r > I) x0 = u;
        }
        const V u = cfms_x(x1, L[r + 16][I], xi);
        if (r + 16 > I) x1 = u;
        unit_solve_step<I + 1>(x0, x1, L, r);
    }
}

template <typename T>
__device__ __forceinline__ void apply_strip(typename CT<T>::t *A, long long lda, int c, const typename CT<T>::t *Lp,
                                            long long ldl, int pw, const int *moves, int a0, int a1, int b0, int b1,
                                            int bid)
{
    using V = typename CT<T>::t;
    __shared__ V s_buf[2 * kPW][17];
    __shared__ V L[kPW][kPW + 1];
    __shared__ int s_src[2 * kPW], s_dst[2 * kPW];
    const int tid = threadIdx.x, w1 = a1 - a0;
    const bool solve = bid * 16 + 16 > w1 && b1 > b0;   // some of its columns are right of the panel
    if (tid < 2 * kPW) {
        const int i = tid & (kPW - 1);
        int src = -1, dst = -1;
        if (i < pw) {
            if (tid < kPW) { src = moves ? moves[i] : c + i; dst = c + i; }
            else if (moves) { src = c + i; dst = moves[kPW + i]; }
        }
        s_src[tid] = src;
        s_dst[tid] = dst;
    }
    if (solve)
        for (int e = tid; e < kPW * kPW; e += 256) {
            const int i = e / kPW, q = e % kPW;
            L[i][q] = i < pw && q < pw ? Lp[i * ldl + q] : V{0, 0};
        }
    __syncthreads();
    const int cl = tid & 15, t = bid * 16 + cl;
    const int col = t < w1 ? a0 + t : (t < w1 + (b1 - b0) ? b0 + (t - w1) : -1);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int e = (tid >> 4) + 16 * k;
        s_buf[e][cl] = col >= 0 && s_dst[e] >= 0 ? A[(long long)s_src[e] * lda + col] : V{0, 0};
    }
    __syncthreads();
    if (solve) {
        const int sc = tid >> 4, r = tid & 15;
        V x0 = s_buf[r][sc], x1 = s_buf[r + 16][sc];
        unit_solve_step<0>(x0, x1, L, r);
        if (bid * 16 + sc >= w1) {
            s_buf[r][sc] = x0;
            s_buf[r + 16][sc] = x1;
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int e = (tid >> 4) + 16 * k;
        if (col >= 0 && s_dst[e] >= 0 && (t >= w1 || s_src[e] != s_dst[e])) A[(long long)s_dst[e] * lda + col] = s_buf[e][cl];
    }
}

__global__ __launch_bounds__(256) void k_apply64(double2 *A, long long lda, int c, int lc, int pw, const int *moves,
                                                 int a0, int a1, int b0, int b1)
{
    apply_strip<double>(A, lda, c, A + (long long)c * lda + lc, lda, pw, moves, a0, a1, b0, b1, blockIdx.x);
}

// ---------------------------------------------------------------- tournament pivoting
// Panel factorisation with tournament pivoting (TSLU, the panel step of CALU:
// Grigori, Demmel & Xiang, SIAM J. Matrix Anal. Appl. 32 (2011)), used by the
// FP32 factorisations that GMRES-IR refines.  Partial pivoting needs one
// grid-wide exchange per column; here the pw <= 32 pivot rows of a panel are chosen
//   1. per workgroup of kTsluRows rows: partial pivoting selects <= pw candidates,
//   2. by a reduction tree: a workgroup stacks up to kTsluFan candidate sets (their
//      rows as they entered the panel) and keeps the rows partial pivoting selects,
// until one set remains.  Partial pivoting on the final stack picks its
// pivots among the winners in order, and eliminating with winners only leaves
// the winners' rows exactly as partial pivoting on the winners alone would
// (no loser is ever a pivot row), so the final workgroup also emits
// L11 \ U11, LAPACK-style sequential interchanges and the row moves.
// The panel's entries lie in an array of their own, P[n][kPW], which the launches of a panel
// only read: a set is therefore its row numbers alone, whoever merges it takes the rows
// from P, and nothing but those numbers and a counter passes between workgroups.
// k_tslu_apply then moves the rows, forms L21 = P U11^-1 and writes the next panel's P.
// Bound by latency, the chain of 32 columns per level.  Two rows per thread halve the
// levels (512 rows to a set: two levels up to 8192 rows, three up to 131,072) for half as
// many more instructions per column.  Measured on the MI355X per 32-column panel, before
// (256 rows a workgroup, the previous panel's update in front of it) -> now: tournament
// 107 -> 75 us at 4050 unknowns, 122 -> 87 us at 9003; apply 27 -> 14 and 27 -> 17 us.

// rows per workgroup of k_tslu_apply
__host__ __device__ inline int tslu_apply_row_count(int rows) { return rows <= 8192 ? 32 : 64; }

// Partial pivoting over R kTsluT rows held in registers, R = 1 or 2 per thread (v: the rows'
// kPW entries; rows with used set never pivot; slot: a row's number in the workgroup).
// piv[j] (LDS) receives the slot whose row pivots column j (-1 if none is left), j_of[h]
// the column that a row pivots.
// Pivot choice: largest |Re|+|Im| at 2^-13 relative resolution (key = value bits with the
// low 10 mantissa bits replaced by 1023 - slot), smaller slot on ties.  Two barriers per
// column: after the first every wave knows the others' best keys (found by DPP), and the
// winning lane stores its row; after the second every wave reads that row, one entry per
// lane, and takes its entries from there into scalar registers, with which it eliminates.
// (One barrier, with every wave's best row stored before it, costs 620 cycles of LDS
// writes per column; a broadcast read of the row by every wave would fill the LDS pipe.)
// The next column's own update, key and reduction go first, and the rest of the update
// runs between the next barrier and the use of the keys read behind it.  In each of four
// phases of eight columns the live columns shift down by one register per column and the
// multipliers enter at the end, so that the column in hand is always the phase's first
// register; finished columns meet zeros in the pivot row.  The elimination has no branch
// (rows that take no part subtract a zero multiple).
struct __align__(16) GeppLds {
    unsigned key[2][4];
    float2 row[2][kPW];
    int piv[kPW];
    int zero;   // first column whose pivot is exactly zero (INT_MAX: none)
};

__device__ __forceinline__ unsigned pivot_key(float2 x, bool used, int slot)
{
    const float mag = fabsf(x.x) + fabsf(x.y);
    return used ? 0u : ((__float_as_uint(mag) & ~1023u) | (unsigned)(1023 - slot));
}

__device__ __forceinline__ float lane_f(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// the waves' best keys of one column, and the best of this thread's rows
template <int R>
__device__ __forceinline__ void gepp_keys(const float2 (&v)[2][kPW], int c, const bool (&used)[2], const int (&slot)[2],
                                          int par, GeppLds &S, unsigned (&key)[2])
{
    unsigned kb = 0;
#pragma unroll
    for (int h = 0; h < R; ++h) {
        key[h] = pivot_key(v[h][c], used[h], slot[h]);
        kb = max(kb, key[h]);
    }
    const unsigned wmax = wave_max_u32(kb);
    if ((threadIdx.x & 63) == 0) S.key[par][threadIdx.x >> 6] = wmax;
}

template <int R, int C0>
__device__ __forceinline__ void gepp_phase(float2 (&v)[2][kPW], bool (&used)[2], const int (&slot)[2], int (&j_of)[2],
                                           int pw, GeppLds &S, unsigned (&key)[2], unsigned &kmax)
{
    constexpr int W = kPW - C0, kPhase = 8;
    static_assert(kTsluT / 64 == 4, "one key per wave");
    const int tid = threadIdx.x, lane = tid & 63;
#pragma unroll 1
    for (int t = 0; t < kPhase; ++t) {
        const int j = C0 + t, par = j & 1;
        if (j >= pw) {   // past the last column of a narrow panel: only the shift
#pragma unroll
            for (int h = 0; h < R; ++h) {
                const float2 v0 = v[h][C0];
#pragma unroll
                for (int q = 1; q < W; ++q) v[h][C0 + q - 1] = v[h][C0 + q];
                v[h][kPW - 1] = v0;
            }
            continue;
        }
        // kmax: column j's best key; key: those of this thread's rows
        const int p = kmax ? 1023 - (int)(kmax & 1023u) : -1;
#pragma unroll
        for (int h = 0; h < R; ++h)
            if (key[h] == kmax && kmax != 0u) {
#pragma unroll
                for (int q = 0; q < W; ++q) S.row[par][q] = v[h][C0 + q];
            }
        __syncthreads();
        float2 pl = S.row[par][min(lane, W - 1)];        // the pivot row, entry q in lane q
        if (p < 0 || lane >= W - t) pl = float2{0, 0};   // no pivot, finished columns
        const float2 d{lane_f(pl.x, 0), lane_f(pl.y, 0)};
        if (tid == 0) {
            S.piv[j] = p;
            if (d.x == 0.f && d.y == 0.f) S.zero = min(S.zero, j);
        }
        const float den = fmaf(d.x, d.x, d.y * d.y);
        const float rd = den != 0.f ? __builtin_amdgcn_rcpf(den) : 0.f;
        float2 l[R], last[R];
        const float ux1 = lane_f(pl.x, 1), uy1 = lane_f(pl.y, 1);
#pragma unroll
        for (int h = 0; h < R; ++h) {
            if (slot[h] == p) {
                used[h] = true;
                j_of[h] = j;
            }
            const float2 v0 = v[h][C0];
            const bool elim = !used[h] && den != 0.f;
            // multiplier v0 / d through the hardware reciprocal of |d|^2 (zero for rows
            // that take no part)
            const float rden = elim ? rd : 0.f;
            l[h] = float2{fmaf(v0.x, d.x, v0.y * d.y) * rden, fmaf(v0.y, d.x, -v0.x * d.y) * rden};
            last[h] = float2{elim ? l[h].x : v0.x, elim ? l[h].y : v0.y};
            v[h][C0] = float2{fmaf(l[h].y, uy1, fmaf(-l[h].x, ux1, v[h][C0 + 1].x)),
                              fmaf(-l[h].y, ux1, fmaf(-l[h].x, uy1, v[h][C0 + 1].y))};
        }
        // the next column's keys (after the last column nothing reads them)
        gepp_keys<R>(v, C0, used, slot, par ^ 1, S, key);
        __syncthreads();
        const uint4 kq = *(const uint4 *)S.key[par ^ 1];
#pragma unroll
        for (int q = 2; q < W; ++q) {
            const float ux = lane_f(pl.x, q), uy = lane_f(pl.y, q);
#pragma unroll
            for (int h = 0; h < R; ++h)
                v[h][C0 + q - 1] = float2{fmaf(l[h].y, uy, fmaf(-l[h].x, ux, v[h][C0 + q].x)),
                                          fmaf(-l[h].y, ux, fmaf(-l[h].x, uy, v[h][C0 + q].y))};
        }
#pragma unroll
        for (int h = 0; h < R; ++h) v[h][kPW - 1] = last[h];
        kmax = max(max(kq.x, kq.y), max(kq.z, kq.w));
    }
    // the live columns are now first, the finished ones last: put them in order
#pragma unroll
    for (int h = 0; h < R; ++h) {
        float2 f[kPhase];
#pragma unroll
        for (int q = 0; q < kPhase; ++q) f[q] = v[h][kPW - kPhase + q];
#pragma unroll
        for (int q = kPW - 1; q >= C0 + kPhase; --q) v[h][q] = v[h][q - kPhase];
#pragma unroll
        for (int q = 0; q < kPhase; ++q) v[h][C0 + q] = f[q];
    }
}

template <int R>
__device__ __forceinline__ void block_gepp(float2 (&v)[2][kPW], bool (&used)[2], const int (&slot)[2], int (&j_of)[2],
                                           int pw, GeppLds &S)
{
    unsigned key[2];
    j_of[0] = j_of[1] = -1;
    if (threadIdx.x == 0) S.zero = INT_MAX;
    gepp_keys<R>(v, 0, used, slot, 0, S, key);
    __syncthreads();
    const uint4 kq = *(const uint4 *)S.key[0];
    unsigned kmax = max(max(kq.x, kq.y), max(kq.z, kq.w));
    gepp_phase<R, 0>(v, used, slot, j_of, pw, S, key, kmax);
    gepp_phase<R, 8>(v, used, slot, j_of, pw, S, key, kmax);
    gepp_phase<R, 16>(v, used, slot, j_of, pw, S, key, kmax);
    gepp_phase<R, 24>(v, used, slot, j_of, pw, S, key, kmax);
    __syncthreads();
}

// x := x U^-1 for one row x on the 16 lanes of a row group, lane r with the entries r and
// r + 16, U upper triangular (LDS); i0, i1: the reciprocals of U's diagonal entries r, r + 16.
template <int I>
__device__ __forceinline__ void right_solve_step(float2 &x0, float2 &x1, const float2 (*U)[kPW + 1], int r, float2 i0,
                                                 float2 i1)
{
    if constexpr (I < kPW) {
        const float2 y = I < 16 ? cmul_x(x0, i0) : cmul_x(x1, i1);
        const float2 xi{row_bcast<I & 15>(y.x), row_bcast<I & 15>(y.y)};
        if constexpr (I < 16) {
            const float2 u = cfms_x(x0, xi, U[I][r]);
            x0.x = r > I ? u.x : (r == I ? y.x : x0.x);
            x0.y = r > I ? u.y : (r == I ? y.y : x0.y);
            x1 = cfms_x(x1, xi, U[I][r + 16]);
        } else {
            const float2 u = cfms_x(x1, xi, U[I][r + 16]);
            x1.x = r + 16 > I ? u.x : (r + 16 == I ? y.x : x1.x);
            x1.y = r + 16 > I ? u.y : (r + 16 == I ? y.y : x1.y);
        }
        right_solve_step<I + 1>(x0, x1, U, r, i0, i1);
    }
}

// What the tournament leaves: sequential interchanges, the factored winners, the row moves.
struct TsluFinal {
    long long *ipiv;   // rows c .. c+pw receive the sequential interchanges
    float2 *top;       // [kPW][kPW] L11 \ U11, row j = the row that goes to c + j
    int *moves;        // [2 kPW]: row that goes to c + i; position where row c + i goes below the panel (-1: none)
    int *info;         // first zero pivot (1-based), 0 if none
};

template <typename T, int TM, int TN, bool M3>
__device__ __forceinline__ void cgemm_tile(int id, const typename CT<T>::t *__restrict__ Ap, long long lda,
                                           const typename CT<T>::t *__restrict__ Bp, long long ldb,
                                           typename CT<T>::t *Cp, long long ldc, int M, int N, int K);

// Counters and candidate sets of the tournament.  Level l holds n_l sets
// (n_0 = workgroups of the first stage, n_{l+1} = tslu_groups(n_l)); its sets start at set
// n_0 + ... + n_{l-1} and its group counters at n_1 + ... + n_l.
struct TsluWork {
    int *cnt;                  // arrivals per group; every counter is zero between panels
    unsigned long long *idx;   // [sets][kPW] candidate row numbers (-1: none) << 32 | tag of the panel
};

// The tournament of the panel [c, c + pw) with entries P as one launch, and the rest of the
// previous panel's update.
// Workgroups [0, nsets0) each take kTsluRows rows (r >= c) and select <= pw candidates by
// partial pivoting.  A workgroup publishes its set's row numbers, each with the panel's tag,
// and counts itself into its group; the last to arrive reads the group's numbers as their
// tags appear, takes the rows from P and merges them at the next level, and so on, so no
// workgroup waits for one that has not run.  The workgroup that partial-pivots the last
// single set writes L11 \ U11, ipiv and the row moves.
// Workgroup nsets0 (prev set) stores the previous panel's block row in this panel's columns
// (unext), and those behind it are the tiles of A[c:, c+kPW : c+kPW+upd_n) -= L21 U12 with
// the previous panel's L21 and U12 (this panel's columns had theirs from k_tslu_apply).
__device__ __forceinline__ void tslu_panel_body(float2 *A, long long lda, int n, int c, int pw, int nsets0, int prev,
                                                int upd_n, const float2 *P, const float2 *unext, const TsluWork &tw,
                                                const TsluFinal &fin, int bid)
{
    if (bid > nsets0) {
        cgemm_tile<float, 4, 2, true>(bid - nsets0 - 1, A + (long long)c * lda + c - kPW, lda,
                                      A + (long long)(c - kPW) * lda + c + kPW, lda, A + (long long)c * lda + c + kPW,
                                      lda, n - c, upd_n, kPW);
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    if (bid == nsets0) {
        for (int e = tid; e < kPW * kPW; e += kTsluT)
            if (e % kPW < pw) A[(long long)(c - kPW + e / kPW) * lda + c + e % kPW] = unext[e];
        return;
    }
    __shared__ GeppLds S;
    __shared__ int s_rowid[kTsluRows], s_next;
    const unsigned tag = (unsigned)c + 1u;
    int g = bid, nl = nsets0, off = 0, coff = 0;
    size_t first = 0;   // first set of the group being merged
    int nrows = -1;     // its rows (-1: the first stage)
    float2 v[2][kPW];
    bool used[2];
    int slot[2], j_of[2];   // j_of: the column the row pivots, -1 for none
    for (;;) {
        // each thread reads its rows as they lie (turning coalesced loads through LDS took 7 us
        // for 512 rows, these 3.5 us); a row that is none takes no part, whatever its registers hold
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            slot[h] = tid + h * kTsluT;
            used[h] = true;
            if (h == 1 && nrows >= 0 && nrows <= kTsluT) continue;
            int id = -1;
            if (nrows < 0) {
                const int row = c + g * kTsluRows + slot[h];
                id = row < n ? row : -1;
            } else if (slot[h] < nrows) {
                const unsigned long long *w = tw.idx + first * kPW + slot[h];
                unsigned long long x;
                // its workgroup stored it before it counted itself: on its way at most
                do x = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                while ((unsigned)x != tag);
                id = (int)(x >> 32);
            }
            const char *Pb = (const char *)P;
            const unsigned at = (unsigned)max(id, 0) * (unsigned)(kPW * sizeof(float2));
#pragma unroll
            for (int q = 0; q < kPW / 2; ++q) {
                const float4 x = *(const float4 *)(Pb + at + q * 16);
                v[h][2 * q] = float2{x.x, x.y};
                v[h][2 * q + 1] = float2{x.z, x.w};
            }
            s_rowid[slot[h]] = id;
            used[h] = id < 0;
        }
        // two rows per thread, or one where they suffice
        if (nrows >= 0 && nrows <= kTsluT) {
            block_gepp<1>(v, used, slot, j_of, pw, S);
        } else {
            block_gepp<2>(v, used, slot, j_of, pw, S);
        }
        if (nl == 1) break;
        if (tid < kPW) {
            const int p = tid < pw ? S.piv[tid] : -1;
            const int id = p >= 0 ? s_rowid[p] : -1;
            __hip_atomic_store(tw.idx + (size_t)(off + g) * kPW + tid, ((unsigned long long)(unsigned)id << 32) | tag,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const int fan = tslu_fan(nl), grp = g / fan, members = min(fan, nl - grp * fan);
        if (tid == 0) {
            const int arrived = __hip_atomic_fetch_add(tw.cnt + coff + grp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (arrived == members - 1)
                __hip_atomic_store(tw.cnt + coff + grp, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_next = arrived == members - 1;
        }
        __syncthreads();
        if (!s_next) return;
        // the last of its group: merge the group's sets one level up
        first = (size_t)off + (size_t)grp * fan;
        nrows = members * kPW;
        coff += tslu_groups(nl);
        off += nl;
        nl = tslu_groups(nl);
        g = grp;
    }
    // last stage: the owners of the pivot rows write L11 \ U11
#pragma unroll
    for (int h = 0; h < 2; ++h)
        if (j_of[h] >= 0) {   // (columns past pw are zero)
            float4 *o = (float4 *)(fin.top + j_of[h] * kPW);
#pragma unroll
            for (int q = 0; q < kPW / 2; ++q)
                o[q] = float4{v[h][2 * q].x, v[h][2 * q].y, v[h][2 * q + 1].x, v[h][2 * q + 1].y};
        }
    for (int e = tid; e < kPW * kPW; e += kTsluT)
        if (e / kPW >= pw) fin.top[e] = float2{0, 0};
    if (wid == 0) {
        // sequential interchanges bringing winner j to position c + j: lane t < pw follows the row
        // that began at c + t; a winner from further down has not moved before its own step
        const int pv = lane < pw ? S.piv[lane] : -1;
        const int win = pv >= 0 ? s_rowid[pv] : -1;
        int pos = c + lane, mine = c + lane;   // position of row c + lane; interchange of column lane
        for (int j = 0; j < pw; ++j) {
            const int here = c + j, w = __builtin_amdgcn_readlane(win, j);
            if (w < 0) continue;   // fewer candidates than columns: cannot happen for pw <= n - c
            const int own = w < c + pw ? w - c : -1;
            const int at = own >= 0 ? __builtin_amdgcn_readlane(pos, own) : w;
            if (lane == j) mine = at;
            if (lane == own) pos = here;
            else if (lane < pw && pos == here) pos = at;
        }
        if (lane < pw) fin.ipiv[c + lane] = mine;
        if (lane == 0 && S.zero != INT_MAX && *fin.info == 0) *fin.info = c + S.zero + 1;
        if (lane < kPW) {
            fin.moves[lane] = lane < pw && win >= 0 ? win : c + lane;
            fin.moves[kPW + lane] = lane < pw && pos >= c + pw ? pos : -1;
        }
    }
}

__global__ __launch_bounds__(kTsluT, 2) void k_tslu_panel(float2 *A, long long lda, int n, int c, int pw, int nsets0,
                                                          int prev, int upd_n, const float2 *P, const float2 *unext,
                                                          TsluWork tw, TsluFinal fin)
{
    tslu_panel_body(A, lda, n, c, pw, nsets0, prev, upd_n, P, unext, tw, fin, blockIdx.x);
}

// A block column's first panel: its entries into P.
__device__ __forceinline__ void tslu_load_body(const float2 *A, long long lda, int n, int c, int pw, float2 *P, int bid)
{
    const long long e = (long long)bid * 256 + threadIdx.x;
    const long long r = c + e / kPW;
    const int q = (int)(e % kPW);
    if (r < n) P[r * kPW + q] = q < pw ? A[r * lda + c + q] : float2{0, 0};
}

__global__ __launch_bounds__(256) void k_tslu_load(const float2 *A, long long lda, int n, int c, int pw, float2 *P)
{
    tslu_load_body(A, lda, n, c, pw, P, blockIdx.x);
}

// After a tournament.  Workgroups [0, nsw): the row moves and the panel's block row in the
// block's columns [a0, a1) left of the panel and [b0, b1) right of the next panel
// (apply_strip).  The others take ROWS panel rows r >= c each: rows c .. c+pw become
// L11 \ U11, every other row x (its entries in P, those of the panel row that moves here where
// one does) becomes L21 = x U11^-1, 16 lanes to a row; every workgroup forms the block row
// U12 in the next panel's nextw columns for itself; then the next panel's entries are
// Pn = (moved rows) - L21 U12.  In A the next panel's columns stay as they are (other
// workgroups read the rows that move); U12 goes to unext and from there into A with the next
// launch.  Bound by the chains of the two solves, 32 steps each; with 32 rows a workgroup
// they are halved while that still gives each CU one (8192 rows), beyond that 64 rows share
// a block row.
struct TsluApply {
    float2 *A;
    long long lda;
    int n, c, pw;
    const float2 *top;
    const int *moves;
    int a0, a1, b0, b1, nsw, nextw;
    const float2 *P;
    float2 *Pn, *unext;
};

template <int ROWS>
__device__ __forceinline__ void tslu_apply_rows(const TsluApply &a, int bid)
{
    constexpr int SETS = ROWS / 16, NC = kPW * ROWS / 256;   // rows per row group; next columns per thread
    __shared__ float2 U[kPW][kPW + 1];
    __shared__ __align__(16) float2 Un[kPW][kPW];
    __shared__ float2 xs[ROWS][kPW + 1];
    __shared__ int s_win[kPW], s_src[ROWS];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, r = lane & 15;
    const int c = a.c, pw = a.pw, n = a.n, nextw = a.nextw;
    const long long lda = a.lda;
    const int row0 = c + (bid - a.nsw) * ROWS;
    for (int i = tid; i < ROWS; i += 256) s_src[i] = row0 + i;
    if (tid < kPW) s_win[tid] = a.moves[tid];
    for (int e = tid; e < kPW * kPW; e += 256) U[e / kPW][e % kPW] = a.top[e];
    __syncthreads();
    if (tid < pw) {   // a panel row that moves into these rows
        const int to = a.moves[kPW + tid] - row0;
        if (to >= 0 && to < ROWS) s_src[to] = c + tid;
    }
    __syncthreads();
    // all loads first: the panel rows, the winners' and the moved rows' next columns
    float2 x0[SETS], x1[SETS], w0[2], w1[2], v[NC];
    int row[SETS];
#pragma unroll
    for (int k = 0; k < SETS; ++k) {
        const int i = (k * 4 + wid) * 4 + (lane >> 4);
        row[k] = row0 + i;
        const float2 *src = a.P + (size_t)min(s_src[i], n - 1) * kPW;
        x0[k] = src[r];
        x1[k] = src[r + 16];
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int col = k * 16 + wid * 4 + (lane >> 4);
        w0[k] = w1[k] = float2{0, 0};
        if (col < nextw) {
            w0[k] = a.A[(long long)s_win[r] * lda + c + kPW + col];
            w1[k] = a.A[(long long)s_win[r + 16] * lda + c + kPW + col];
        }
    }
    const int vi = tid % ROWS, vc = tid / ROWS * NC, vr = row0 + vi;
    const bool below = vr >= c + pw && vr < n;
    const long long vs = (long long)min(s_src[vi], n - 1) * lda + c + kPW + vc;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        v[q] = float2{0, 0};
        if (below && vc + q < nextw) v[q] = a.A[vs + q];
    }
    if (nextw > 0) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int col = k * 16 + wid * 4 + (lane >> 4);
            unit_solve_step<0>(w0[k], w1[k], U, r);
            Un[r][col] = w0[k];
            Un[r + 16][col] = w1[k];
        }
    }
    auto recip = [](float2 d) {
        const float den = fmaf(d.x, d.x, d.y * d.y), q = den != 0.f ? __builtin_amdgcn_rcpf(den) : 0.f;
        return float2{d.x * q, -d.y * q};
    };
    const float2 i0 = recip(U[r][r]), i1 = recip(U[r + 16][r + 16]);
#pragma unroll
    for (int k = 0; k < SETS; ++k) {
        right_solve_step<0>(x0[k], x1[k], U, r, i0, i1);
        const int at = row[k] - c;
        if (at < pw) {
            x0[k] = U[min(at, kPW - 1)][r];
            x1[k] = U[min(at, kPW - 1)][r + 16];
        }
        xs[row[k] - row0][r] = x0[k];
        xs[row[k] - row0][r + 16] = x1[k];
        if (row[k] < n) {
            float2 *o = a.A + (long long)row[k] * lda + c;
            if (r < pw) o[r] = x0[k];
            if (r + 16 < pw) o[r + 16] = x1[k];
        }
    }
    if (nextw <= 0) return;
    __syncthreads();
    if (bid == a.nsw)
        for (int e = tid; e < kPW * kPW; e += 256) a.unext[e] = Un[e / kPW][e % kPW];
    if (!below) return;
#pragma unroll 4
    for (int i = 0; i < kPW; ++i) {
        const float2 l = xs[vi][i];
        float2 u[NC];
#pragma unroll
        for (int q = 0; q < NC; ++q) u[q] = Un[i][vc + q];
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            v[q].x = fmaf(l.y, u[q].y, fmaf(-l.x, u[q].x, v[q].x));
            v[q].y = fmaf(-l.y, u[q].x, fmaf(-l.x, u[q].y, v[q].y));
        }
    }
    float4 *o = (float4 *)(a.Pn + (size_t)vr * kPW + vc);
#pragma unroll
    for (int q = 0; q < NC / 2; ++q) o[q] = float4{v[2 * q].x, v[2 * q].y, v[2 * q + 1].x, v[2 * q + 1].y};
}

__device__ __forceinline__ void tslu_apply_body(const TsluApply &a, int bid)
{
    if (bid < a.nsw)
        apply_strip<float>(a.A, a.lda, a.c, a.top, kPW, a.pw, a.moves, a.a0, a.a1, a.b0, a.b1, bid);
    else if (tslu_apply_row_count(a.n - a.c) == 32)
        tslu_apply_rows<32>(a, bid);
    else
        tslu_apply_rows<64>(a, bid);
}

__global__ __launch_bounds__(256) void k_tslu_apply(TsluApply a)
{
    tslu_apply_body(a, blockIdx.x);
}

// ---------------------------------------------------------------- row interchanges
// Sequential interchanges ipiv[k1..k2) (LAPACK laswp) on a set of columns.
// The same interchanges as one permutation of the touched rows.  Replaying
// them sequentially per column costs one dependent global round trip per
// interchange; instead k_swap_plan replays them once on row indices (LDS) and
// k_laswp_apply moves every touched row of every column in a single pass.
// Plan slots: [0, len) are rows k1 + i; [len, 2 len) the rows ipiv[k1 + i] >= k2
// (slot len + i for the first i naming that row).  plan[s] = the row whose
// content ends at slot s, plan[2 len + s] = the slot's row (-1: slot unused).
constexpr int kMaxSwaps = 256;
// FP32 LU block depth (trailing-update depth): while the trailing matrix is
// large the blocks are 1024 deep, factored as two halves of kNBInner one after
// the other on the block-column stream; that halves the C traffic of the
// trailing updates, which pays while the trailing update hides the longer
// block-column chain.  Smaller trailing matrices take 512-deep blocks.
constexpr int kNBFP32 = 1024, kNBFP32Small = 512, kNBDeepAbove = 24576;
constexpr int kNBInner = 512;
constexpr int kNBFP64 = 256;            // FP64 block depth
constexpr int kAheadFirstBelow = 20480;   // trailing width below which the next block column goes first

// The 1024-deep block columns join their 512-column halves with split-bf16 products,
// so the plain FP32 factorisation keeps 512 throughout.
inline int fp32_block_depth(int n, int k, bool split)
{
    return split && n - k > kNBDeepAbove ? kNBFP32 : kNBFP32Small;
}

__device__ __forceinline__ void swap_plan_body(const long long *ipiv, int k1, int k2, int *plan)
{
    __shared__ int s_piv[kMaxSwaps], s_partner[kMaxSwaps], s_src[2 * kMaxSwaps];
    const int len = k2 - k1, tid = threadIdx.x;
    for (int i = tid; i < len; i += 256) s_piv[i] = (int)ipiv[k1 + i];
    __syncthreads();
    for (int i = tid; i < len; i += 256) {
        const int p = s_piv[i];
        int partner = p - k1;
        if (p >= k2) {
            int first = i;
            for (int j = 0; j < i; ++j)
                if (s_piv[j] == p) { first = j; break; }
            partner = len + first;
        }
        s_partner[i] = partner;
        s_src[i] = k1 + i;
        const bool head = p >= k2 && partner == len + i;
        s_src[len + i] = head ? p : -1;
        plan[2 * len + i] = k1 + i;
        plan[3 * len + i] = head ? p : -1;
    }
    __syncthreads();
    if (tid == 0) {
        for (int i = 0; i < len; ++i) {
            const int q = s_partner[i];
            const int t = s_src[i];
            s_src[i] = s_src[q];
            s_src[q] = t;
        }
    }
    __syncthreads();
    for (int s = tid; s < 2 * len; s += 256) plan[s] = s_src[s];
}

__global__ __launch_bounds__(256) void k_swap_plan(const long long *ipiv, int k1, int k2, int *plan)
{
    swap_plan_body(ipiv, k1, k2, plan);
}

// Apply a swap plan of 2 len slots to columns [c0, c1) and [c2, c3): CW
// columns per workgroup (64 KiB of LDS at most), every moved row read into LDS
// before any is written.
template <typename T>
constexpr int laswp_cols() { return sizeof(T) == 4 ? 32 : 8; }

template <typename T>
__device__ __forceinline__ void laswp_apply_body(typename CT<T>::t *A, long long lda, const int *plan, int len, int c0,
                                                 int c1, int c2, int c3, int bid)
{
    using V = typename CT<T>::t;
    constexpr int CW = laswp_cols<T>(), RL = 256 / CW;
    extern __shared__ char smem_raw[];
    V *buf = (V *)smem_raw;   // [2 len][CW]
    const int tid = threadIdx.x, cl = tid % CW, rl = tid / CW;
    const int t = bid * CW + cl, w1 = c1 - c0;
    int col = -1;
    if (t < w1) col = c0 + t;
    else if (t < w1 + (c3 - c2)) col = c2 + (t - w1);
    const int *src = plan, *pos = plan + 2 * len;
    for (int s = rl; s < 2 * len; s += RL) {
        const int p = pos[s], q = src[s];
        if (col >= 0 && p >= 0 && p != q) buf[s * CW + cl] = A[(long long)q * lda + col];
    }
    __syncthreads();
    for (int s = rl; s < 2 * len; s += RL) {
        const int p = pos[s], q = src[s];
        if (col >= 0 && p >= 0 && p != q) A[(long long)p * lda + col] = buf[s * CW + cl];
    }
}

// FP32: a workgroup takes 32 columns, one per thread and eight slots at a time; every
// moved entry is held in registers (all its loads in flight at once, no LDS staging),
// then written after the barrier.
template <>
__device__ __forceinline__ void laswp_apply_body<float>(float2 *A, long long lda, const int *plan, int len, int c0,
                                                        int c1, int c2, int c3, int bid)
{
    constexpr int CW = laswp_cols<float>(), RL = 256 / CW, MAXK = 2 * kMaxSwaps / RL;
    __shared__ int s_src[2 * kMaxSwaps], s_pos[2 * kMaxSwaps];
    const int tid = threadIdx.x, cl = tid % CW, rl = tid / CW;
    for (int q = tid; q < 2 * len; q += 256) {
        s_src[q] = plan[q];
        s_pos[q] = plan[2 * len + q];
    }
    __syncthreads();
    const int t = bid * CW + cl, w1 = c1 - c0;
    int col = -1;
    if (t < w1) col = c0 + t;
    else if (t < w1 + (c3 - c2)) col = c2 + (t - w1);
    float2 v[MAXK];
#pragma unroll
    for (int k = 0; k < MAXK; ++k) {
        const int sl = rl + RL * k;
        if (sl < 2 * len && col >= 0) {
            const int p = s_pos[sl], q = s_src[sl];
            if (p >= 0 && p != q) v[k] = A[(long long)q * lda + col];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < MAXK; ++k) {
        const int sl = rl + RL * k;
        if (sl < 2 * len && col >= 0) {
            const int p = s_pos[sl], q = s_src[sl];
            if (p >= 0 && p != q) A[(long long)p * lda + col] = v[k];
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_laswp_apply(typename CT<T>::t *A, long long lda, const int *plan, int len,
                                                     int c0, int c1, int c2, int c3)
{
    laswp_apply_body<T>(A, lda, plan, len, c0, c1, c2, c3, blockIdx.x);
}

// ---------------------------------------------------------------- MFMA complex GEMM
// C[M x N] -= A[M x K] B[K x N], row-major complex, K a multiple of 16.
// Workgroup: 4 waves in 2 x 2, wave tile (16*TM) x (16*TN) complex.
template <typename T>
struct MfmaVec;
template <>
struct MfmaVec<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
};
template <>
struct MfmaVec<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
};

template <typename T>
__device__ __forceinline__ typename MfmaVec<T>::v4 mfma16(T a, T b, typename MfmaVec<T>::v4 c);

template <>
__device__ __forceinline__ MfmaVec<float>::v4 mfma16<float>(float a, float b, MfmaVec<float>::v4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <>
__device__ __forceinline__ MfmaVec<double>::v4 mfma16<double>(double a, double b, MfmaVec<double>::v4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

constexpr int kBK = 16;

// C[M x N] -= A[M x K] B[K x N], row-major complex, K a multiple of kBK.
// 256 threads = 2 x 2 waves, wave tile (16 TM) x (16 TN) complex, workgroup
// tile (32 TM) x (32 TN).  K advances in chunks of 16 through two LDS buffers:
// the next chunk is loaded into registers while the current one feeds the
// MFMAs, then stored to the other buffer (one barrier per chunk).
// M3 = false: four real products per complex product (Cr += ArBr - AiBi,
// Ci += ArBi + AiBr); M3 = true: three (T1 = ArBr, T2 = AiBi,
// T3 = (Ar+Ai)(Br+Bi), Cr = T1 - T2, Ci = T3 - T1 - T2), normwise stable and used
// for the FP32 factorisation that GMRES-IR refines.
// Tile of a GEMM launched as a 1-D grid of nbm x nbn tiles.  Workgroups are
// dispatched round-robin over the 8 XCDs (workgroup id mod 8), each with its
// own L2: the id is first remapped so every XCD owns a contiguous range of
// tiles, which is then walked in groups of kGroupM tile rows (column-major
// inside a group), so the workgroups an XCD runs at once share A row panels
// and B column panels in its L2.  Four tile rows per group (the 32 tiles an XCD
// runs at once: 4 x 8) measured 1% faster than 8, 2 or 16 on the C3 factorisation.
constexpr int kXcds = 8, kGroupM = 4;
__device__ __forceinline__ void gemm_tile(int id, int nbm, int nbn, int &tm, int &tn)
{
    const int total = nbm * nbn;
    const int q = total / kXcds, r = total % kXcds, x = id % kXcds;
    const int t = x * q + min(x, r) + id / kXcds;
    const int per_group = kGroupM * nbn;
    const int first = (t / per_group) * kGroupM;
    const int gm = min(kGroupM, nbm - first);
    const int in = t % per_group;
    tm = first + in % gm;
    tn = in / gm;
}

// One tile (linear index id, 256 threads) of the GEMM below.
template <typename T, int TM, int TN, bool M3>
__device__ __forceinline__ void cgemm_tile(int id, const typename CT<T>::t *__restrict__ Ap, long long lda,
                                           const typename CT<T>::t *__restrict__ Bp, long long ldb,
                                           typename CT<T>::t *Cp, long long ldc, int M, int N, int K)
{
    using V = typename CT<T>::t;
    using v4 = typename MfmaVec<T>::v4;
    constexpr int BM = 32 * TM, BN = 32 * TN;
    constexpr int APT = BM * kBK / 256;          // A elements per thread
    constexpr int BPT = kBK * BN / 256;          // B elements per thread
    constexpr int AROW = kBK / APT;              // threads per A row
    constexpr int BROW = BN / BPT;               // threads per B row
    constexpr int NACC = M3 ? 3 : 2;
    __shared__ V As[2][BM][kBK + 1];
    __shared__ V Bs[2][kBK][BN + 1];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wm = wv >> 1, wn = wv & 1;
    int tm, tn;
    gemm_tile(id, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
    const long long m0 = (long long)tm * BM, n0 = (long long)tn * BN;
    const int ar = tid / AROW, ac = (tid % AROW) * APT;
    const int br = tid / BROW, bc = (tid % BROW) * BPT;
    const bool arow_ok = m0 + ar < M;
    const V *ag = Ap + (m0 + ar) * lda + ac;
    const V *bg = Bp + (long long)br * ldb + n0 + bc;
    V ra[APT], rb[BPT];
    auto load = [&](int k0) {
#pragma unroll
        for (int j = 0; j < APT; ++j) ra[j] = arow_ok ? ag[k0 + j] : V{0, 0};
#pragma unroll
        for (int j = 0; j < BPT; ++j) rb[j] = (n0 + bc + j < N) ? bg[(long long)k0 * ldb + j] : V{0, 0};
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int j = 0; j < APT; ++j) As[buf][ar][ac + j] = ra[j];
#pragma unroll
        for (int j = 0; j < BPT; ++j) Bs[buf][br][bc + j] = rb[j];
    };
    v4 acc[NACC][TM][TN];
#pragma unroll
    for (int q = 0; q < NACC; ++q)
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b) acc[q][a][b] = v4{0, 0, 0, 0};
    const int li = lane & 15, lk = lane >> 4;
    load(0);
    store(0);
    __syncthreads();
    int cur = 0;
    for (int k0 = 0; k0 < K; k0 += kBK) {
        const bool more = k0 + kBK < K;
        if (more) load(k0 + kBK);
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 4) {
            V af[TM], bf[TN];
#pragma unroll
            for (int a = 0; a < TM; ++a) af[a] = As[cur][wm * 16 * TM + a * 16 + li][kk + lk];
#pragma unroll
            for (int b = 0; b < TN; ++b) bf[b] = Bs[cur][kk + lk][wn * 16 * TN + b * 16 + li];
            if constexpr (M3) {
                T as[TM], bs[TN];
#pragma unroll
                for (int a = 0; a < TM; ++a) as[a] = af[a].x + af[a].y;
#pragma unroll
                for (int b = 0; b < TN; ++b) bs[b] = bf[b].x + bf[b].y;
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) {
                        acc[0][a][b] = mfma16<T>(af[a].x, bf[b].x, acc[0][a][b]);
                        acc[1][a][b] = mfma16<T>(af[a].y, bf[b].y, acc[1][a][b]);
                        acc[2][a][b] = mfma16<T>(as[a], bs[b], acc[2][a][b]);
                    }
            } else {
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) {
                        acc[0][a][b] = mfma16<T>(af[a].x, bf[b].x, acc[0][a][b]);
                        acc[1][a][b] = mfma16<T>(af[a].x, bf[b].y, acc[1][a][b]);
                    }
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) {
                        acc[0][a][b] = mfma16<T>(-af[a].y, bf[b].y, acc[0][a][b]);
                        acc[1][a][b] = mfma16<T>(af[a].y, bf[b].x, acc[1][a][b]);
                    }
            }
        }
        if (more) store(cur ^ 1);
        __syncthreads();
        cur ^= 1;
    }
    // output row of register r in lane l (column l % 16): the f32 16x16x4 MFMA
    // keeps 4 consecutive rows per lane group (4 (l/16) + r), the f64 one
    // interleaves them (4 r + l/16)
    // all C reads are issued before any write, so they overlap (one memory
    // round trip per tile instead of one per element)
    V cv[TM][TN][4];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ri = sizeof(T) == 4 ? 4 * (lane >> 4) + r : 4 * r + (lane >> 4);
                const long long gi = m0 + wm * 16 * TM + a * 16 + ri;
                const long long gj = n0 + wn * 16 * TN + b * 16 + (lane & 15);
                cv[a][b][r] = (gi < M && gj < N) ? Cp[gi * ldc + gj] : V{0, 0};
            }
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ri = sizeof(T) == 4 ? 4 * (lane >> 4) + r : 4 * r + (lane >> 4);
                const long long gi = m0 + wm * 16 * TM + a * 16 + ri;
                const long long gj = n0 + wn * 16 * TN + b * 16 + (lane & 15);
                if (gi < M && gj < N) {
                    T re, im;
                    if constexpr (M3) {
                        re = acc[0][a][b][r] - acc[1][a][b][r];
                        im = acc[2][a][b][r] - acc[0][a][b][r] - acc[1][a][b][r];
                    } else {
                        re = acc[0][a][b][r];
                        im = acc[1][a][b][r];
                    }
                    V c = cv[a][b][r];
                    c.x -= re;
                    c.y -= im;
                    Cp[gi * ldc + gj] = c;
                }
            }
}

template <typename T, int TM, int TN, bool M3, int WPE>
__global__ __launch_bounds__(256, WPE) void k_cgemm(const typename CT<T>::t *__restrict__ Ap, long long lda,
                                                    const typename CT<T>::t *__restrict__ Bp, long long ldb,
                                                    typename CT<T>::t *Cp, long long ldc, int M, int N, int K)
{
    cgemm_tile<T, TM, TN, M3>(blockIdx.x, Ap, lda, Bp, ldb, Cp, ldc, M, N, K);
}

// ---------------------------------------------------------------- split-bf16 GEMM
// Mixed-path trailing update C -= A B with FP32 complex C.  Each FP32 value x is
// split into bf16 hi = bf16(x) and lo = bf16(x - hi); a real product is taken as
// hi*hi + hi*lo + lo*hi (the lo*lo term is below 2^-16 relative), i.e. three
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation, about 16 significant bits per
// product.  The FP32 LU that GMRES-IR refines tolerates this.  A and B are split
// once per panel step into planes (Re hi, Re lo, Im hi, Im lo), 32-deep k slices
// contiguous, so the GEMM streams bf16 through LDS and does no conversions.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
constexpr int kSplitBK = 32;
// LDS rows of a stage are unpadded (64 B); the 16-byte k group g of row r is stored at
// g ^ swz(r), which keeps both the staging writes (whole rows) and the fragment reads
// (16 rows, one k group) free of bank conflicts with 32 or 64 banks
__device__ __forceinline__ int split_swz(int r) { return ((r >> 1) ^ (r >> 2)) & 3; }

__device__ __forceinline__ void split_bf16(float x, __bf16 &hi, __bf16 &lo)
{
    hi = (__bf16)x;
    lo = (__bf16)(x - (float)hi);
}

// Plane layout: P[4][K / 32][rows][32], so that a k-step's 32-deep slice of a tile's rows
// is one contiguous run per plane (measured 1.3% faster products than P[4][rows][K]).
// A (rows x K, row-major complex, lda) -> P[4][K / 32][rows][32] bf16
__device__ __forceinline__ void split_rows_body(const float2 *__restrict__ A, long long lda, int rows, int K,
                                                __bf16 *__restrict__ P, long long idx)
{
    if (idx >= (long long)rows * K) return;
    const long long r = idx / K, k = idx % K;
    const float2 v = A[r * lda + k];
    const long long plane = (long long)rows * K;
    const long long o = ((k >> 5) * rows + r) * 32 + (k & 31);
    split_bf16(v.x, P[o], P[plane + o]);
    split_bf16(v.y, P[2 * plane + o], P[3 * plane + o]);
}

__global__ void k_split_rows(const float2 *__restrict__ A, long long lda, int rows, int K, __bf16 *__restrict__ P)
{
    split_rows_body(A, lda, rows, K, P, (long long)blockIdx.x * blockDim.x + threadIdx.x);
}

// B (K x cols, row-major complex, ldb) -> P[4][K / 32][cols][32] bf16 (transposed)
__device__ __forceinline__ void split_cols_body(const float2 *__restrict__ B, long long ldb, int K, int cols,
                                                __bf16 *__restrict__ P, int bx, int by)
{
    __shared__ float2 t[32][33];
    const int c0 = bx * 32, k0 = by * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
    for (int r = ty; r < 32; r += 8) {
        const int k = k0 + r, c = c0 + tx;
        t[r][tx] = (k < K && c < cols) ? B[(long long)k * ldb + c] : float2{0, 0};
    }
    __syncthreads();
    const long long plane = (long long)cols * K;
    for (int r = ty; r < 32; r += 8) {
        const int c = c0 + r, k = k0 + tx;
        if (c < cols && k < K) {
            const float2 v = t[tx][r];
            const long long o = ((long long)(k >> 5) * cols + c) * 32 + (k & 31);
            split_bf16(v.x, P[o], P[plane + o]);
            split_bf16(v.y, P[2 * plane + o], P[3 * plane + o]);
        }
    }
}

__global__ __launch_bounds__(256) void k_split_cols(const float2 *__restrict__ B, long long ldb, int K, int cols,
                                                    __bf16 *__restrict__ P)
{
    split_cols_body(B, ldb, K, cols, P, blockIdx.x, blockIdx.y);
}

// C is read and written once per tile with nontemporal accesses, so that the tile
// rows of C streaming through do not evict the A and B planes, which the other
// tiles of the launch re-read, from L2.
__device__ __forceinline__ float2 ntload2(const float2 *p)
{
    return float2{__builtin_nontemporal_load(&p->x), __builtin_nontemporal_load(&p->y)};
}

__device__ __forceinline__ void ntstore2(float2 *p, float2 v)
{
    __builtin_nontemporal_store(v.x, &p->x);
    __builtin_nontemporal_store(v.y, &p->y);
}

// C[M x N] -= A B from split planes PA[4][K/32][M][32], PB[4][K/32][N][32]; K a multiple of 32.
// WM x WN waves, wave tile (16 TM) x (16 TN) complex.  Two LDS stages (128 KB for the
// 128 x 128 tile, unpadded rows with swizzled k groups): the global loads of step k+1 are in flight while step k's products run
// from the other stage, one barrier per step; the first row block of the C tile is read
// during the last step's products.
template <int TM, int TN, int WM, int WN>
__device__ __forceinline__ void cgemm_bf16x3_body(const __bf16 *__restrict__ PA, const __bf16 *__restrict__ PB,
                                                  float2 *C, long long ldc, int M, int N, int K, int tile)
{
    constexpr int NT = 64 * WM * WN;
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN, BK = kSplitBK, RS = BK;
    __shared__ __align__(16) __bf16 As[2][4][BM][RS];
    __shared__ __align__(16) __bf16 Bs[2][4][BN][RS];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wm = wv / WN, wn = wv % WN;
    int tm, tn;
    gemm_tile(tile, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
    const long long m0 = (long long)tm * BM, n0 = (long long)tn * BN;
    const long long planeA = (long long)M * K, planeB = (long long)N * K;
    // 16-byte chunks (8 bf16) per chunk of K: A has 4 * BM * 4, B has 4 * BN * 4
    constexpr int ACH = 4 * BM * (BK / 8), BCH = 4 * BN * (BK / 8);
    constexpr int AP = (ACH + NT - 1) / NT, BP = (BCH + NT - 1) / NT;
    uint4 ra[AP], rb[BP];
    auto load = [&](int k0) {
#pragma unroll
        for (int q = 0; q < AP; ++q) {
            const int c = tid + NT * q;
            if (c < ACH) {
                const int p = c / (BM * 4), rem = c % (BM * 4), r = rem / 4, g = rem % 4;
                const long long row = m0 + r;
                ra[q] = row < M ? *(const uint4 *)(PA + p * planeA + ((long long)(k0 >> 5) * M + row) * 32 + 8 * g)
                                : uint4{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int q = 0; q < BP; ++q) {
            const int c = tid + NT * q;
            if (c < BCH) {
                const int p = c / (BN * 4), rem = c % (BN * 4), r = rem / 4, g = rem % 4;
                const long long col = n0 + r;
                rb[q] = col < N ? *(const uint4 *)(PB + p * planeB + ((long long)(k0 >> 5) * N + col) * 32 + 8 * g)
                                : uint4{0, 0, 0, 0};
            }
        }
    };
    auto store = [&](int st) {
#pragma unroll
        for (int q = 0; q < AP; ++q) {
            const int c = tid + NT * q;
            if (c < ACH) {
                const int p = c / (BM * 4), rem = c % (BM * 4), r = rem / 4, g = rem % 4;
                *(uint4 *)&As[st][p][r][8 * (g ^ split_swz(r))] = ra[q];
            }
        }
#pragma unroll
        for (int q = 0; q < BP; ++q) {
            const int c = tid + NT * q;
            if (c < BCH) {
                const int p = c / (BN * 4), rem = c % (BN * 4), r = rem / 4, g = rem % 4;
                *(uint4 *)&Bs[st][p][r][8 * (g ^ split_swz(r))] = rb[q];
            }
        }
    };
    // real and imaginary parts of the tile; the real part takes Re A Re B and
    // Im A (-Im B), the B fragments' imaginary planes negated by their sign bits
    f32x4 arr[TM][TN], ari[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            arr[a][b] = f32x4{0, 0, 0, 0};
            ari[a][b] = f32x4{0, 0, 0, 0};
        }
    const int li = lane & 15, lg = lane >> 4;   // row/col within a 16-block, k group of 8
    const int kofs = 8 * (lg ^ split_swz(li));    // the k group's place in LDS (rows start at multiples of 16)
    // products of one k-step from LDS stage st
    auto compute = [&](int st) {
        bf16x8 afr[TM][4];
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int p = 0; p < 4; ++p) afr[a][p] = *(const bf16x8 *)&As[st][p][wm * 16 * TM + a * 16 + li][kofs];
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            bf16x8 bfr[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) bfr[p] = *(const bf16x8 *)&Bs[st][p][wn * 16 * TN + b * 16 + li][kofs];
            const bf16x8 nb2 = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, bfr[2]) ^ 0x80008000u);
            const bf16x8 nb3 = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, bfr[3]) ^ 0x80008000u);
#pragma unroll
            for (int a = 0; a < TM; ++a) {
                arr[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][0], bfr[0], arr[a][b], 0, 0, 0);
                ari[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][0], bfr[2], ari[a][b], 0, 0, 0);
                arr[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][2], nb2, arr[a][b], 0, 0, 0);
                ari[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][2], bfr[0], ari[a][b], 0, 0, 0);
                arr[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][0], bfr[1], arr[a][b], 0, 0, 0);
                ari[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][0], bfr[3], ari[a][b], 0, 0, 0);
                arr[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][2], nb3, arr[a][b], 0, 0, 0);
                ari[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][2], bfr[1], ari[a][b], 0, 0, 0);
                arr[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][1], bfr[0], arr[a][b], 0, 0, 0);
                ari[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][1], bfr[2], ari[a][b], 0, 0, 0);
                arr[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][3], nb2, arr[a][b], 0, 0, 0);
                ari[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[a][3], bfr[0], ari[a][b], 0, 0, 0);
            }
        }
    };
    auto cidx = [&](int a, int b, int r, long long &gi, long long &gj) {
        gi = m0 + wm * 16 * TM + a * 16 + 4 * (lane >> 4) + r;
        gj = n0 + wn * 16 * TN + b * 16 + (lane & 15);
    };
    load(0);
    store(0);
    __syncthreads();
    int st = 0;
    for (int k0 = 0; k0 + BK < K; k0 += BK, st ^= 1) {
        load(k0 + BK);
        compute(st);
        store(st ^ 1);   // the other stage was last read before the previous barrier
        __syncthreads();
    }
    // last k-step: the first row block of this wave's C tile is read while its products run
    float2 c0[TN][4];
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            long long gi, gj;
            cidx(0, b, r, gi, gj);
            c0[b][r] = (gi < M && gj < N) ? ntload2(C + gi * ldc + gj) : float2{0, 0};
        }
    compute(st);
    float2 cv[TM][TN][4];
#pragma unroll
    for (int a = 1; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                long long gi, gj;
                cidx(a, b, r, gi, gj);
                cv[a][b][r] = (gi < M && gj < N) ? ntload2(C + gi * ldc + gj) : float2{0, 0};
            }
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) cv[0][b][r] = c0[b][r];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                long long gi, gj;
                cidx(a, b, r, gi, gj);
                if (gi < M && gj < N) {
                    float2 c = cv[a][b][r];
                    c.x -= arr[a][b][r];
                    c.y -= ari[a][b][r];
                    ntstore2(C + gi * ldc + gj, c);
                }
            }
}

template <int TM, int TN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_cgemm_bf16x3(const __bf16 *__restrict__ PA,
                                                                 const __bf16 *__restrict__ PB, float2 *C,
                                                                 long long ldc, int M, int N, int K)
{
    cgemm_bf16x3_body<TM, TN, WM, WN>(PA, PB, C, ldc, M, N, K, blockIdx.x);
}

// ---------------------------------------------------------------- conversions
template <typename T>
__global__ void k_to_work(const double2 *__restrict__ src, int n, typename CT<T>::t *dst, long long lda)
{
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)n * n) return;
    const long long i = idx / n, j = idx % n;
    const double2 v = src[idx];
    dst[i * lda + j] = {(T)v.x, (T)v.y};
}

// ---------------------------------------------------------------- solves
// X is n x nrhs row-major (rhs contiguous per row).
template <typename T>
__global__ void k_permute_in(const double2 *__restrict__ b, int n, int nrhs, const int *__restrict__ perm,
                             typename CT<T>::t *x)
{
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)n * nrhs) return;
    const int i = (int)(idx / nrhs), r = (int)(idx % nrhs);
    const double2 v = b[(long long)perm[i] * nrhs + r];
    x[idx] = {(T)v.x, (T)v.y};
}

constexpr int kTB = 64;   // triangular-solve block
constexpr int kMaxRhs = 8;

// The triangular solves run one launch per triangle, one workgroup per CU.  A workgroup takes
// a block in the order of a ticket counter, solves it and takes the next, until none is left
// (so a block never waits for a workgroup that has not started: every block it waits for has
// an earlier ticket, held by a running workgroup).  Tickets handed out per launch: the blocks
// plus one final ticket per workgroup.  Solved rows travel as 64-bit words, 32 bits of value
// over the launch's epoch: a word is valid by itself, so that neither fences nor flags are
// needed (the writeback and invalidation of two fences per block took longer than the block's
// products), and a block waits on the values themselves.  A wait that exceeds kTrsvSpin polls
// sets the error word and gives up, so every workgroup ends.
constexpr int kTrsvT = 512;                // threads of a workgroup
constexpr long long kTrsvSpin = 1LL << 24;
constexpr int kTrsvHead = 8;               // words before the values: [0] ticket counter and error flag

// the words tid, tid + kTrsvT, .. of the cnt words at src, as they are
template <int U>
__device__ __forceinline__ void words_fetch(const unsigned long long *src, int cnt, unsigned long long (&w)[U])
{
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = threadIdx.x + kTrsvT * u;
        w[u] = t < cnt ? get_word(src + t) : 0ull;
    }
}

// waits for them, all of a thread's in one round, and stores their values (zeros beyond cnt, up
// to total), that of word t at dst[place(t)]
template <int U, typename Place>
__device__ __forceinline__ void words_settle(const unsigned long long *src, int cnt, int total, int epoch,
                                             unsigned long long (&w)[U], unsigned *dst, const Place &place, int *err)
{
    long long it = 0;
    for (;;) {
        bool late = false;
#pragma unroll
        for (int u = 0; u < U; ++u) late = late || ((int)threadIdx.x + kTrsvT * u < cnt && (int)(unsigned)w[u] != epoch);
        if (!late) break;
        if (++it > kTrsvSpin) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        // once a wait has given up, the others do not wait out their own limits
        if ((it & 63) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
        __builtin_amdgcn_s_sleep(1);
        words_fetch<U>(src, cnt, w);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = threadIdx.x + kTrsvT * u;
        if (t < total) dst[place(t)] = t < cnt ? (unsigned)(w[u] >> 32) : 0u;
    }
}

// Sum over the eight lanes 8 m .. 8 m + 7 of a value, in each of them: DPP quad_perm 1,0,3,2
// and 2,3,0,1 make each quad uniform, then the half-row mirror adds the other quad.
template <int CTRL>
__device__ __forceinline__ float dpp_lane(float v)
{
    const int i = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, 0xF, 0xF, false));
}

template <int CTRL>
__device__ __forceinline__ double dpp_lane(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = (int)b, hi = (int)(b >> 32);
    const int l2 = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false);
    const int h2 = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false);
    return __longlong_as_double(((long long)h2 << 32) | (unsigned)l2);
}

template <typename T>
__device__ __forceinline__ T sum8_lanes(T v)
{
    v += dpp_lane<0xB1>(v);
    v += dpp_lane<0x4E>(v);
    v += dpp_lane<0x141>(v);
    return v;
}

__device__ __forceinline__ double lane_value(double v, int l)   // l uniform
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// FP64: blocks of 64 rows.  Thread (row t / 8, c8 = t % 8) holds of a 64 x 64 block the
// columns c8 + 8 j (j < 8); eight lanes read 128 bytes of a row at once.  Two blocks are in
// flight per workgroup, and the products with all solved blocks stay in the lanes until one
// sum over a row's eight at the end.  Then wave q substitutes column q in the diagonal block,
// a row per lane, the solved entry going round by readlane (no LDS and no division in the
// chain: the diagonal block lies in LDS by columns, U's reciprocals are formed before the wait).
// Bound by the chain of blocks, about 6 us each.  One triangle, before (a launch per block with
// a serial sweep through LDS) and now: 17,406 unknowns 12.6 -> 1.7 ms, 702 unknowns 420 -> 62 us.
constexpr int kBlk64Chunks = kTB / 8, kBlk64Ld = kTB + 1;
static_assert(kTrsvT == 8 * kTB, "a row of a block is eight threads");
static_assert(kMaxRhs <= kTrsvT / 64, "a wave per right-hand side");
using Blk64Regs = double2[kBlk64Chunks];

__device__ __forceinline__ void blk64_load(const double2 *Mx, long long ld, int rs, int cs, Blk64Regs &a)
{
    const int r = threadIdx.x >> 3, c8 = threadIdx.x & 7;
    const double2 *row = Mx + (long long)min(r, rs - 1) * ld;
#pragma unroll
    for (int j = 0; j < kBlk64Chunks; ++j) a[j] = c8 + 8 * j < cs ? row[c8 + 8 * j] : double2{0.0, 0.0};
}

// a + v into a, the rounding error added to e
__device__ __forceinline__ void add_two(double &a, double &e, double v)
{
    const double s = a + v, t = s - a;
    e += (a - (s - t)) + (v - t);
    a = s;
}

// acc[q] += this thread's part of its row times column q of x.  A block's part is summed by
// itself first (one sum over all of a row's blocks would round at its full size at every
// entry), and what the sum over the blocks rounds off is kept in low[q].
template <int NRHS>
__device__ __forceinline__ void blk64_acc(const Blk64Regs &a, const double2 *x, double2 (&acc)[NRHS], double2 (&low)[NRHS])
{
    const int c8 = threadIdx.x & 7;
#pragma unroll
    for (int q = 0; q < NRHS; ++q) {
        double2 v{0.0, 0.0};
#pragma unroll
        for (int j = 0; j < kBlk64Chunks; ++j) v = cfma_x(v, a[j], x[(c8 + 8 * j) * NRHS + q]);
        add_two(acc[q].x, low[q].x, v.x);
        add_two(acc[q].y, low[q].y, v.y);
        // else the sums sink below the loads that follow, all of x waits in registers, and they spill
        asm volatile("" : "+v"(acc[q].x), "+v"(acc[q].y)::"memory");
    }
}

template <bool LOWER, int NRHS>
__global__ __launch_bounds__(kTrsvT) void k_trsv64(const double2 *A, long long lda, int n, double2 *X,
                                                   unsigned long long *sync, int ticket0, int epoch)
{
    constexpr int kUnits = kTB * NRHS * 4, kU = (kUnits + kTrsvT - 1) / kTrsvT;
    __shared__ double2 D[kTB * kBlk64Ld];   // D[j kBlk64Ld + i]: row i, column j
    __shared__ double2 xs[kTB * NRHS];
    __shared__ double2 xb[2][kTB * NRHS];
    __shared__ int s_idx;
    int *counter = (int *)sync, *err = counter + 1;
    unsigned long long *xw = sync + kTrsvHead;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, nblk = (n + kTB - 1) / kTB;
    for (;;) {
        __syncthreads();   // the previous block's LDS reads are done
        if (tid == 0) s_idx = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - ticket0;
        __syncthreads();
        const int idx = s_idx;
        if (idx < 0 || idx >= nblk) return;   // no block left
        const int r0 = (LOWER ? idx : nblk - 1 - idx) * kTB, rs = min(kTB, n - r0);
        // dependency d < idx: the block solved d-th
        auto first = [&](int d) { return (LOWER ? d : nblk - 1 - d) * kTB; };
        auto load = [&](int d, Blk64Regs &a) { blk64_load(A + (long long)r0 * lda + first(d), lda, rs, min(kTB, n - first(d)), a); };
        unsigned long long w[kU];
        auto fetch = [&](int d) { words_fetch<kU>(xw + (size_t)first(d) * NRHS * 4, min(kTB, n - first(d)) * NRHS * 4, w); };
        Blk64Regs ra, rb;
        if (idx > 0) fetch(0);
        if (idx > 0) load(0, ra);
        if (idx > 1) load(1, rb);
        for (int e = tid; e < kTB * kTB; e += kTrsvT) {
            const int i = e / kTB, j = e % kTB;
            D[j * kBlk64Ld + i] = i < rs && j < rs ? A[(long long)(r0 + i) * lda + r0 + j] : double2{0.0, 0.0};
        }
        for (int t = tid; t < kTB * NRHS; t += kTrsvT) xs[t] = t < rs * NRHS ? X[(long long)r0 * NRHS + t] : double2{0.0, 0.0};
        __syncthreads();
        double2 rinv{1.0, 0.0};
        if (!LOWER && lane < rs) {
            const double2 d = D[lane * kBlk64Ld + lane];
            const double den = d.x * d.x + d.y * d.y;
            rinv = {d.x / den, -d.y / den};
        }
        double2 acc[NRHS], low[NRHS];
#pragma unroll
        for (int q = 0; q < NRHS; ++q) acc[q] = low[q] = {0.0, 0.0};
        auto one = [&](int d, Blk64Regs &a, double2 *x) {
            const int c0 = first(d), cnt = min(kTB, n - c0) * NRHS * 4;
            const unsigned long long *src = xw + (size_t)c0 * NRHS * 4;
            words_settle<kU>(src, cnt, kUnits, epoch, w, (unsigned *)x, [](int t) { return t; }, err);
            __syncthreads();
            if (d + 1 < idx) fetch(d + 1);
            blk64_acc<NRHS>(a, x, acc, low);
            if (d + 2 < idx) load(d + 2, a);
        };
        for (int d = 0; d < idx; d += 2) {
            one(d, ra, xb[0]);
            if (d + 1 < idx) one(d + 1, rb, xb[1]);
        }
        if (idx > 0) {
            const int r = tid >> 3, c8 = tid & 7;
#pragma unroll
            for (int q = 0; q < NRHS; ++q) {
                const double2 v{sum8_lanes(acc[q].x), sum8_lanes(acc[q].y)};
                const double2 w8{sum8_lanes(low[q].x), sum8_lanes(low[q].y)};
                if (c8 == q) {
                    xs[r * NRHS + q].x = (xs[r * NRHS + q].x - v.x) - w8.x;
                    xs[r * NRHS + q].y = (xs[r * NRHS + q].y - v.y) - w8.y;
                }
            }
            __syncthreads();
        }
        if (wid < NRHS) {
            // x: the solved entries, b - t before (t from zero: as in blk64_acc)
            const double2 b = xs[lane * NRHS + wid];
            double2 x = b, t{0.0, 0.0};
            if constexpr (LOWER) {
#pragma unroll 8
                for (int s = 0; s < rs - 1; ++s) {
                    t = cfma_x(t, D[s * kBlk64Ld + lane], double2{lane_value(x.x, s), lane_value(x.y, s)});
                    if (lane > s) x = csubv(b, t);
                }
            } else {
                x = double2{fma(b.x, rinv.x, -(b.y * rinv.y)), fma(b.x, rinv.y, b.y * rinv.x)};
#pragma unroll 8
                for (int s = rs - 1; s > 0; --s) {
                    t = cfma_x(t, D[s * kBlk64Ld + lane], double2{lane_value(x.x, s), lane_value(x.y, s)});
                    const double2 u = csubv(b, t);
                    if (lane < s) x = double2{fma(u.x, rinv.x, -(u.y * rinv.y)), fma(u.x, rinv.y, u.y * rinv.x)};
                }
            }
            if (lane < rs) {
                const size_t o = (size_t)(r0 + lane) * NRHS + wid;
                const unsigned long long bx = (unsigned long long)__double_as_longlong(x.x),
                                         by = (unsigned long long)__double_as_longlong(x.y), tag = (unsigned)epoch;
                put_word(xw + 4 * o, (bx << 32) | tag);
                put_word(xw + 4 * o + 1, (bx & 0xffffffff00000000ull) | tag);
                put_word(xw + 4 * o + 2, (by << 32) | tag);
                put_word(xw + 4 * o + 3, (by & 0xffffffff00000000ull) | tag);
                X[o] = x;
            }
        }
    }
}

// ---------------------------------------------------------------- FP32 solves with inverted diagonal blocks
// The FP32 factors only precondition GMRES-IR, so their triangular solves use
// explicit inverses of the 128 x 128 diagonal blocks (computed once per
// factorisation): each block step is then two small matrix-vector products with
// no serial sweep.
constexpr int kIB = 128;
constexpr int kTrinvParts = 4;   // lanes per column in k_trinv

// Inverse of the unit-lower 128 x 128 block held in S (LDS, zero above the diagonal,
// in place), by 32 x 32 blocks: the four diagonal blocks by forward substitution, a
// thread per column with the column in registers (no barrier); then block row I = 1..3
// as S_IJ = -S_II sum_{K=J..I-1} L_IK S_KJ (J < I), the sums first (into T, while
// L_IJ is still in place), then the products with S_II.  512 threads.
constexpr int kIB32 = 32;   // block of the blocked inverse
__device__ __forceinline__ void unit_lower_inverse_blocked(float2 *S, float2 (*T)[kIB32][kIB32])
{
    const int t = threadIdx.x;
    float2 x[kIB32];
    const int blk = t / kIB32, c = t % kIB32;
    if (t < kIB) {
        // column c of the inverse of diagonal block blk: x_r = [r == c] - sum_{k<r} L[r][k] x_k
        const float2 *L = S + (size_t)(kIB32 * blk) * kIB + kIB32 * blk;
#pragma unroll
        for (int r = 0; r < kIB32; ++r) {
            float2 acc{0, 0};
#pragma unroll
            for (int k = 0; k < r; ++k) {
                const float2 a = L[r * kIB + k];
                acc.x = fmaf(a.x, x[k].x, fmaf(-a.y, x[k].y, acc.x));
                acc.y = fmaf(a.x, x[k].y, fmaf(a.y, x[k].x, acc.y));
            }
            x[r] = r < c ? float2{0, 0} : (r == c ? float2{1, 0} : float2{-acc.x, -acc.y});
        }
    }
    __syncthreads();   // every diagonal block has been read
    if (t < kIB) {
        float2 *L = S + (size_t)(kIB32 * blk) * kIB + kIB32 * blk;
#pragma unroll
        for (int r = 0; r < kIB32; ++r) L[r * kIB + c] = x[r];
    }
    __syncthreads();
    for (int I = 1; I < kIB / kIB32; ++I) {
        const float2 *rowI = S + (size_t)(kIB32 * I) * kIB;
        for (int e = t; e < I * kIB32 * kIB32; e += kIB * kTrinvParts) {
            const int J = e / (kIB32 * kIB32), r = e / kIB32 % kIB32, cc = e % kIB32;
            float2 acc{0, 0};
#pragma unroll 16
            for (int k = kIB32 * J; k < kIB32 * I; ++k) {
                const float2 a = rowI[r * kIB + k], b = S[(size_t)k * kIB + kIB32 * J + cc];
                acc.x = fmaf(a.x, b.x, fmaf(-a.y, b.y, acc.x));
                acc.y = fmaf(a.x, b.y, fmaf(a.y, b.x, acc.y));
            }
            T[J][r][cc] = acc;
        }
        __syncthreads();
        for (int e = t; e < I * kIB32 * kIB32; e += kIB * kTrinvParts) {
            const int J = e / (kIB32 * kIB32), r = e / kIB32 % kIB32, cc = e % kIB32;
            float2 acc{0, 0};
#pragma unroll 8
            for (int k = 0; k <= r; ++k) {
                const float2 a = rowI[r * kIB + kIB32 * I + k], b = T[J][k][cc];
                acc.x = fmaf(a.x, b.x, fmaf(-a.y, b.y, acc.x));
                acc.y = fmaf(a.x, b.y, fmaf(a.y, b.x, acc.y));
            }
            S[(size_t)(kIB32 * I + r) * kIB + kIB32 * J + cc] = float2{-acc.x, -acc.y};
        }
        __syncthreads();
    }
}

// In-place inverse of diagonal block blockIdx.x of the unit-lower (LOWER) or
// upper factor in LDS; rows past the end of the matrix become identity rows.
// LOWER: blocked (unit_lower_inverse_blocked).  Upper: row by row,
// X[i][t] = ([i == t] - sum_k T[i][k] X[k][t]) / T[i][i] over the rows k already
// inverted (entries outside the triangle are zero), kTrinvParts threads per column
// sharing each row's dot product (partial sums combined through LDS).
template <bool LOWER>
__device__ __forceinline__ void trinv_body(const float2 *A, long long lda, int n, float2 *Dinv, int bid)
{
    __shared__ float2 S[kIB * kIB];
    const int t = threadIdx.x, col = t % kIB, part = t / kIB;
    const int b0 = bid * kIB, bs = min(kIB, n - b0);
    for (int idx = t; idx < kIB * kIB; idx += kIB * kTrinvParts) {
        const int i = idx / kIB, j = idx % kIB;
        float2 v{0, 0};
        if (i < bs && j < bs && (LOWER ? j < i : j >= i)) v = A[(long long)(b0 + i) * lda + b0 + j];
        if (i == j && (LOWER || i >= bs)) v = {1, 0};
        S[idx] = v;
    }
    __syncthreads();
    if constexpr (LOWER) {
        __shared__ float2 T[kIB / kIB32 - 1][kIB32][kIB32];
        unit_lower_inverse_blocked(S, T);
    } else {
        __shared__ float2 red[kTrinvParts][kIB];
        // part = t / kIB: the waves of a part read whole rows of S (consecutive columns,
        // no bank conflicts); part p sums the terms k = p mod kTrinvParts of each dot product
        for (int i = kIB - 1; i >= 0; --i) {
            float2 u{0, 0}, w{0, 0};   // two chains, so consecutive terms overlap
            int k = i + 1 + part;
            for (; k + kTrinvParts < kIB; k += 2 * kTrinvParts) {
                const float2 a = S[i * kIB + k], x = S[k * kIB + col];
                const float2 b = S[i * kIB + k + kTrinvParts], y = S[(k + kTrinvParts) * kIB + col];
                u.x += a.x * x.x - a.y * x.y;
                u.y += a.x * x.y + a.y * x.x;
                w.x += b.x * y.x - b.y * y.y;
                w.y += b.x * y.y + b.y * y.x;
            }
            if (k < kIB) {
                const float2 a = S[i * kIB + k], x = S[k * kIB + col];
                u.x += a.x * x.x - a.y * x.y;
                u.y += a.x * x.y + a.y * x.x;
            }
            red[part][col] = {u.x + w.x, u.y + w.y};
            const float2 d = S[i * kIB + i];
            __syncthreads();
            if (part == 0) {
                float2 acc = red[0][col];
#pragma unroll
                for (int p = 1; p < kTrinvParts; ++p) { acc.x += red[p][col].x; acc.y += red[p][col].y; }
                const float den = d.x * d.x + d.y * d.y;
                const float2 inv{d.x / den, -d.y / den};
                if (col > i) S[i * kIB + col] = {-(acc.x * inv.x - acc.y * inv.y), -(acc.x * inv.y + acc.y * inv.x)};
                else if (col == i) S[i * kIB + i] = inv;
            }
            __syncthreads();
        }
    }
    float2 *out = Dinv + (size_t)bid * kIB * kIB;
    for (int idx = t; idx < kIB * kIB; idx += kIB * kTrinvParts) out[idx] = S[idx];
}

template <bool LOWER>
__global__ __launch_bounds__(kIB * kTrinvParts) void k_trinv(const float2 *A, long long lda, int n, float2 *Dinv)
{
    trinv_body<LOWER>(A, lda, n, Dinv, blockIdx.x);
}

// The kTrsvT threads of a workgroup hold a 128 x 128 block in registers, loaded at once (one
// memory round trip per block instead of one per entry): thread t (wave w, lane l) takes the
// rows (kTrsvT / 8) p + 8 w + l / 8 (p < kBlkRows) and of each the 16-byte chunks
// l % 8 + 8 j (j < 8), i.e. the columns 2 (l % 8 + 8 j) and the one after.  Eight lanes read
// one 128-byte line of a row, so each load of a wave touches 8 cache lines (a layout with a
// row per lane touches 64, and the vector memory pipeline then takes four times as long over
// the block); the eight lanes of a row then sum their parts by DPP within the half-row.
constexpr int kBlkRowStep = kTrsvT / 8, kBlkRows = kIB / kBlkRowStep, kBlkChunks = 8;
static_assert(kBlkRows * kBlkRowStep == kIB, "rows of a block split evenly over the threads");
using BlkRegs = float4[kBlkRows][kBlkChunks];

// Rows r < rs and columns c < cs of Mx (1 <= rs, cs <= 128), zeros elsewhere.  Every load is
// issued, from rows and columns that are there (the last row again; the columns up to 64 or,
// with wide, 128: rows are padded to multiples of 64), so that nothing but an incomplete block
// waits for its values here.
__device__ __forceinline__ void blk_load(const float2 *Mx, long long ld, int rs, int cs, bool wide, BlkRegs &a)
{
    const int t = threadIdx.x, w = t >> 6, l = t & 63, rl = 8 * w + (l >> 3), c8 = l & 7;
    const float2 *M2 = Mx + (wide ? kIB / 2 : 0);
#pragma unroll
    for (int p = 0; p < kBlkRows; ++p) {
        const long long o = (long long)min(kBlkRowStep * p + rl, rs - 1) * ld + 2 * c8;   // 16-byte aligned
#pragma unroll
        for (int j = 0; j < kBlkChunks; ++j)
            a[p][j] = *(const float4 *)((j < kBlkChunks / 2 ? Mx : M2) + o + 16 * (j % (kBlkChunks / 2)));
    }
    if (rs < kIB || cs < kIB) {
#pragma unroll
        for (int p = 0; p < kBlkRows; ++p)
#pragma unroll
            for (int j = 0; j < kBlkChunks; ++j) {
                const int r = kBlkRowStep * p + rl, c = 2 * (c8 + 8 * j);
                if (r >= rs || c >= cs) a[p][j].x = a[p][j].y = 0.f;
                if (r >= rs || c + 1 >= cs) a[p][j].z = a[p][j].w = 0.f;
            }
    }
}

// acc[p][q] += (SUB: -=) this thread's part of row p times column q of xin (LDS, [NRHS][kIB]: a
// row pair in one 16-byte read, the eight lanes' reads on different banks);
// a: the thread's share of the block, in registers (stride 1) or in LDS (stride kTrsvT)
template <bool SUB, int NRHS>
__device__ __forceinline__ void blk_acc(const float4 *a, int stride, const float2 *xin, float2 (&acc)[kBlkRows][NRHS])
{
    const int c8 = threadIdx.x & 7;
#pragma unroll
    for (int q = 0; q < NRHS; ++q) {
        float2 v[kBlkRows];
#pragma unroll
        for (int p = 0; p < kBlkRows; ++p) v[p] = {0, 0};
#pragma unroll
        for (int j = 0; j < kBlkChunks; ++j) {
            const int c = 2 * (c8 + 8 * j);
            const float4 x01 = *(const float4 *)(xin + q * kIB + c);
            const float2 x0{x01.x, x01.y}, x1{x01.z, x01.w};
#pragma unroll
            for (int p = 0; p < kBlkRows; ++p) {   // explicit FMAs: the same bits for every NRHS
                const float4 m = a[(p * kBlkChunks + j) * stride];
                v[p].x = fmaf(-m.w, x1.y, fmaf(m.z, x1.x, fmaf(-m.y, x0.y, fmaf(m.x, x0.x, v[p].x))));
                v[p].y = fmaf(m.w, x1.x, fmaf(m.z, x1.y, fmaf(m.y, x0.x, fmaf(m.x, x0.y, v[p].y))));
            }
        }
#pragma unroll
        for (int p = 0; p < kBlkRows; ++p) {
            float2 &o = acc[p][q];
            o = SUB ? float2{o.x - v[p].x, o.y - v[p].y} : float2{o.x + v[p].x, o.y + v[p].y};
            // else the sums sink below the loads that follow, all of xin waits in registers, and they spill
            asm volatile("" : "+v"(o.x), "+v"(o.y)::"memory");
        }
    }
}

// G[i] = Dinv[i] M[i][i -/+ 1] for the blocks with a neighbour (LOWER: the
// block left of the diagonal of L, else the block right of the diagonal of U),
// so the solve step that waits for the neighbour is one product.  Workgroup
// (i, y) forms rows [16 y, 16 y + 16) of G[i]; thread t: row t / 16, columns
// 8 (t % 16) .. + 8.
template <bool LOWER>
__device__ __forceinline__ void blk_coupling_body(const float2 *A, long long lda, int n, const float2 *Dinv, float2 *G,
                                                  int bx, int by)
{
    __shared__ float2 Ds[16][kIB];
    __shared__ float2 Ms[32][kIB];
    const int nb = (n + kIB - 1) / kIB;
    const int i = bx, j = LOWER ? i - 1 : i + 1;
    if (j < 0 || j >= nb) return;   // uniform
    const int r0 = i * kIB, rs = min(kIB, n - r0), c0 = j * kIB, cs = min(kIB, n - c0);
    const int tid = threadIdx.x, rr = tid >> 4, cg = (tid & 15) * 8, y0 = by * 16;
    for (int idx = tid; idx < 16 * kIB; idx += 256) {
        const int r = idx / kIB, k = idx % kIB;
        Ds[r][k] = (y0 + r < rs && k < rs) ? Dinv[(size_t)i * kIB * kIB + (size_t)(y0 + r) * kIB + k] : float2{0, 0};
    }
    float2 acc[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] = {0, 0};
    for (int k0 = 0; k0 < kIB; k0 += 32) {
        __syncthreads();
        for (int idx = tid; idx < 32 * kIB; idx += 256) {
            const int k = idx / kIB, c = idx % kIB;
            Ms[k][c] = (k0 + k < rs && c < cs) ? A[(long long)(r0 + k0 + k) * lda + c0 + c] : float2{0, 0};
        }
        __syncthreads();
#pragma unroll 4
        for (int k = 0; k < 32; ++k) {
            const float2 d = Ds[rr][k0 + k];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const float2 m = Ms[k][cg + c];
                acc[c].x = fmaf(d.x, m.x, fmaf(-d.y, m.y, acc[c].x));
                acc[c].y = fmaf(d.x, m.y, fmaf(d.y, m.x, acc[c].y));
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) G[(size_t)i * kIB * kIB + (size_t)(y0 + rr) * kIB + cg + c] = acc[c];
}

template <bool LOWER>
__global__ __launch_bounds__(256) void k_blk_coupling(const float2 *A, long long lda, int n, const float2 *Dinv,
                                                      float2 *G)
{
    blk_coupling_body<LOWER>(A, lda, n, Dinv, G, blockIdx.x, blockIdx.y);
}

// FP32: blocks of 128 rows.  Block i subtracts the products with the blocks it depends on as
// their rows appear, two blocks of the factor in flight, the sums kept in the lanes until one
// sum over a row's eight; then x = Dinv b - G x_adjacent, with the coupling G to the adjacent
// block loaded and Dinv b formed before the adjacent rows are waited for, so that the chain
// from block to block is one exchange and one product.  Bound by that chain, and at 40,000
// unknowns by the reads of the factor.  One triangle, before (ready flags between fences) and
// now: 39,996 unknowns, one column 2.75 -> 1.42 ms (4.5 TB/s); 12,000, four columns 0.85 ->
// 0.51 ms; 4050, two columns 0.16 -> 0.12 ms.
template <bool LOWER, int NRHS>
__global__ __launch_bounds__(kTrsvT) void k_trsv_flag(const float2 *A, long long lda, int n, const float2 *Dinv,
                                                      const float2 *G, float2 *X, unsigned long long *sync,
                                                      int ticket0, int epoch)
{
    constexpr int kUnits = kIB * NRHS * 2, kU = (kUnits + kTrsvT - 1) / kTrsvT;
    __shared__ __align__(16) float2 xs[kIB * NRHS];   // [NRHS][kIB]
    __shared__ __align__(16) float2 xb[2][kIB * NRHS];
    // the inverted diagonal block, each thread's share at a place of its own (read back
    // by the thread that wrote it: no barrier, no bank conflicts)
    __shared__ float4 dsh[kBlkRows][kBlkChunks][kTrsvT];
    __shared__ int s_idx;
    int *counter = (int *)sync, *err = counter + 1;
    unsigned long long *xw = sync + kTrsvHead;
    const int tid = threadIdx.x, nblk = (n + kIB - 1) / kIB;
    const int rl = 8 * (tid >> 6) + ((tid & 63) >> 3), c8 = tid & 7;
    for (;;) {
        __syncthreads();   // the previous block's LDS reads are done
        if (tid == 0) s_idx = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - ticket0;
        __syncthreads();
        const int idx = s_idx;
        if (idx < 0 || idx >= nblk) return;   // no block left
        const int blk = LOWER ? idx : nblk - 1 - idx;
        const int r0 = blk * kIB, rs = min(kIB, n - r0);
        const int adj = idx - 1;   // dependency d: the block solved d-th; the last one is adjacent
        auto first = [&](int d) { return (LOWER ? d : nblk - 1 - d) * kIB; };
        auto load = [&](int d, BlkRegs &a) {
            const int c0 = first(d), cs = min(kIB, n - c0);
            const bool far = d < adj;
            if (d <= adj) blk_load(far ? A + (long long)r0 * lda + c0 : G + (size_t)blk * kIB * kIB, far ? lda : kIB, rs, cs,
                                   !far || c0 + kIB <= lda, a);
        };
        unsigned long long w[kU];
        auto fetch = [&](int d) { words_fetch<kU>(xw + (size_t)first(d) * NRHS * 2, min(kIB, n - first(d)) * NRHS * 2, w); };
        BlkRegs ra, rb;
        blk_load(Dinv + (size_t)blk * kIB * kIB, kIB, rs, rs, true, ra);
#pragma unroll
        for (int p = 0; p < kBlkRows; ++p)
#pragma unroll
            for (int j = 0; j < kBlkChunks; ++j) dsh[p][j][tid] = ra[p][j];
        if (idx > 0) fetch(0);
        load(0, ra);
        load(1, rb);
        for (int t = tid; t < kIB * NRHS; t += kTrsvT)
            xs[(t % NRHS) * kIB + t / NRHS] = t < rs * NRHS ? X[(long long)r0 * NRHS + t] : float2{0, 0};
        __syncthreads();
        float2 acc[kBlkRows][NRHS];
#pragma unroll
        for (int p = 0; p < kBlkRows; ++p)
#pragma unroll
            for (int q = 0; q < NRHS; ++q) acc[p][q] = {0, 0};
        auto settle = [&](int d, float2 *x) {
            words_settle<kU>(xw + (size_t)first(d) * NRHS * 2, min(kIB, n - first(d)) * NRHS * 2, kUnits, epoch, w, (unsigned *)x,
                             [](int t) { return ((t >> 1) % NRHS * kIB + (t >> 1) / NRHS) * 2 + (t & 1); }, err);
        };
        auto one = [&](int d, BlkRegs &a, float2 *x) {
            settle(d, x);
            __syncthreads();
            fetch(d + 1);
            blk_acc<false, NRHS>(&a[0][0], 1, x, acc);
            load(d + 2, a);
        };
        auto finish = [&](const BlkRegs &g, float2 *x) {   // the rest, with the coupling in g
            if (adj > 0) {
#pragma unroll
                for (int p = 0; p < kBlkRows; ++p)
#pragma unroll
                    for (int q = 0; q < NRHS; ++q) {
                        const float2 v{sum8_lanes(acc[p][q].x), sum8_lanes(acc[p][q].y)};
                        if (c8 == q) {   // rows from rs on: zeros
                            float2 &o = xs[q * kIB + kBlkRowStep * p + rl];
                            o = {o.x - v.x, o.y - v.y};
                        }
                        acc[p][q] = {0, 0};
                    }
                __syncthreads();
            }
            blk_acc<false, NRHS>(&dsh[0][0][tid], kTrsvT, xs, acc);
            if (adj >= 0) {
                settle(adj, x);
                __syncthreads();
                blk_acc<true, NRHS>(&g[0][0], 1, x, acc);
            }
#pragma unroll
            for (int p = 0; p < kBlkRows; ++p) {   // lane c8 of a row publishes column c8
                float2 v{0, 0};
#pragma unroll
                for (int q = 0; q < NRHS; ++q) {
                    const float2 u{sum8_lanes(acc[p][q].x), sum8_lanes(acc[p][q].y)};
                    if (c8 == q) v = u;
                }
                const int i = kBlkRowStep * p + rl;
                if (c8 < NRHS && i < rs) {
                    const size_t o = (size_t)(r0 + i) * NRHS + c8;
                    put_word(xw + 2 * o, ((unsigned long long)__float_as_uint(v.x) << 32) | (unsigned)epoch);
                    put_word(xw + 2 * o + 1, ((unsigned long long)__float_as_uint(v.y) << 32) | (unsigned)epoch);
                    X[o] = v;
                }
            }
        };
        int d = 0;
        for (; d + 1 < adj; d += 2) {
            one(d, ra, xb[0]);
            one(d + 1, rb, xb[1]);
        }
        if (d < adj) {
            one(d, ra, xb[0]);
            finish(rb, xb[1]);
        } else {
            finish(ra, xb[0]);
        }
    }
}

// r = b - A x (RESID) or r = A x in FP64 (A row-major n x n; x, b, r row-major n x NRHS).
// A workgroup takes kAxRows rows; its four waves take the 64-column pieces in turn, so an
// entry of x is loaded once for all the rows (with a wave per row, the 16 NRHS bytes of x per
// 16 bytes of A came from the caches for every row).  Bound by the one read of A: at 12,000
// unknowns and four columns 1.07 -> 0.50 ms (4.6 TB/s), at 39,996 and one 4.43 -> 4.11 ms
// (6.2 TB/s).  The waves' sums meet in LDS.  Explicit FMAs, the same for every NRHS:
// a column's bits do not depend on the others.
constexpr int kAxRows = 4;

template <bool RESID, int NRHS>
__global__ __launch_bounds__(256) void k_apply_a(const double2 *__restrict__ A, int n, const double2 *__restrict__ x,
                                                 const double2 *__restrict__ b, double2 *__restrict__ r)
{
    __shared__ double2 red[4][kAxRows][NRHS];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, row0 = blockIdx.x * kAxRows;
    const double2 *a[kAxRows];
#pragma unroll
    for (int k = 0; k < kAxRows; ++k) a[k] = A + (size_t)min(row0 + k, n - 1) * n;
    double2 acc[kAxRows][NRHS];
#pragma unroll
    for (int k = 0; k < kAxRows; ++k)
#pragma unroll
        for (int q = 0; q < NRHS; ++q) acc[k][q] = {0, 0};
    auto step = [&](const double2 (&av)[kAxRows], int c) {
#pragma unroll
        for (int q = 0; q < NRHS; ++q) {
            const double2 xv = x[(size_t)c * NRHS + q];
#pragma unroll
            for (int k = 0; k < kAxRows; ++k) {
                acc[k][q].x = fma(av[k].x, xv.x, fma(-av[k].y, xv.y, acc[k][q].x));
                acc[k][q].y = fma(av[k].x, xv.y, fma(av[k].y, xv.x, acc[k][q].y));
            }
        }
    };
    int c = 64 * wid + lane;
    // two pieces of every row in flight
    for (; c + 256 < n; c += 512) {
        double2 u[kAxRows], v[kAxRows];
#pragma unroll
        for (int k = 0; k < kAxRows; ++k) u[k] = a[k][c];
#pragma unroll
        for (int k = 0; k < kAxRows; ++k) v[k] = a[k][c + 256];
        step(u, c);
        step(v, c + 256);
    }
    if (c < n) {
        double2 u[kAxRows];
#pragma unroll
        for (int k = 0; k < kAxRows; ++k) u[k] = a[k][c];
        step(u, c);
    }
#pragma unroll
    for (int k = 0; k < kAxRows; ++k) {
#pragma unroll
        for (int q = 0; q < NRHS; ++q) {
            double sx = acc[k][q].x, sy = acc[k][q].y;
            for (int off = 32; off >= 1; off >>= 1) {
                sx += __shfl_xor(sx, off, 64);
                sy += __shfl_xor(sy, off, 64);
            }
            if (lane == 0) red[wid][k][q] = {sx, sy};
        }
    }
    __syncthreads();
    const int t = threadIdx.x;
    if (t < kAxRows * NRHS && row0 + t / NRHS < n) {
        const int k = t / NRHS, q = t % NRHS;
        const double sx = (red[0][k][q].x + red[1][k][q].x) + (red[2][k][q].x + red[3][k][q].x);
        const double sy = (red[0][k][q].y + red[1][k][q].y) + (red[2][k][q].y + red[3][k][q].y);
        const size_t o = (size_t)(row0 + k) * NRHS + q;
        if constexpr (RESID) r[o] = {b[o].x - sx, b[o].y - sy};
        else r[o] = {sx, sy};
    }
}

template <bool RESID>
void apply_a(hipStream_t s, const double2 *A, int n, const double2 *x, const double2 *b, double2 *r, int nrhs)
{
    const unsigned g = (unsigned)((n + kAxRows - 1) / kAxRows);
    switch (nrhs) {
    case 1: k_apply_a<RESID, 1><<<g, 256, 0, s>>>(A, n, x, b, r); break;
    case 2: k_apply_a<RESID, 2><<<g, 256, 0, s>>>(A, n, x, b, r); break;
    case 3: k_apply_a<RESID, 3><<<g, 256, 0, s>>>(A, n, x, b, r); break;
    case 4: k_apply_a<RESID, 4><<<g, 256, 0, s>>>(A, n, x, b, r); break;
    case 5: k_apply_a<RESID, 5><<<g, 256, 0, s>>>(A, n, x, b, r); break;
    case 6: k_apply_a<RESID, 6><<<g, 256, 0, s>>>(A, n, x, b, r); break;
    case 7: k_apply_a<RESID, 7><<<g, 256, 0, s>>>(A, n, x, b, r); break;
    case 8: k_apply_a<RESID, 8><<<g, 256, 0, s>>>(A, n, x, b, r); break;
    default: BH_FAIL(BH_ERR_INVALID, "nrhs %d out of range", nrhs);
    }
}

// GMRES vectors: q columns side by side (row-major n x q blocks), one Krylov space per
// column, all advanced by the same launches.
struct ColScale {
    double s[kMaxRhs];
};

__global__ void k_scale_cols(const double2 *__restrict__ src, int n, int q, ColScale sc, double2 *__restrict__ dst)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)n * q) return;
    const double f = sc.s[i % q];
    dst[i] = {src[i].x * f, src[i].y * f};
}

// out[block][j][c] = sum over the block's rows i of conj(V_j[i][c]) w[i][c], j < m, c < q
__global__ __launch_bounds__(256) void k_dots_cols(const double2 *__restrict__ Vb, int n, int m, int q,
                                                   const double2 *__restrict__ w, double2 *__restrict__ out)
{
    __shared__ double2 red[4][kMaxRhs];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int j = 0; j < m; ++j) {
        const double2 *v = Vb + (size_t)j * n * q;
        double ax[kMaxRhs], ay[kMaxRhs];
#pragma unroll
        for (int c = 0; c < kMaxRhs; ++c) ax[c] = ay[c] = 0;
        for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
#pragma unroll
            for (int c = 0; c < kMaxRhs; ++c) {
                if (c < q) {
                    const double2 a = v[(size_t)i * q + c], b = w[(size_t)i * q + c];
                    ax[c] += a.x * b.x + a.y * b.y;
                    ay[c] += a.x * b.y - a.y * b.x;
                }
            }
        }
#pragma unroll
        for (int c = 0; c < kMaxRhs; ++c) {
            if (c < q) {
                double sx = ax[c], sy = ay[c];
                for (int off = 32; off >= 1; off >>= 1) {
                    sx += __shfl_xor(sx, off, 64);
                    sy += __shfl_xor(sy, off, 64);
                }
                if (lane == 0) red[wid][c] = {sx, sy};
            }
        }
        __syncthreads();
        if ((int)threadIdx.x < q) {
            const int c = threadIdx.x;
            out[((size_t)blockIdx.x * m + j) * q + c] = {red[0][c].x + red[1][c].x + red[2][c].x + red[3][c].x,
                                                        red[0][c].y + red[1][c].y + red[2][c].y + red[3][c].y};
        }
        __syncthreads();
    }
}

// out[j][c] = sum of the 256 block parts of k_dots_cols, one wave each; 0 for columns not in mask
__global__ __launch_bounds__(64) void k_sum_parts(const double2 *__restrict__ part, int m, int q, unsigned mask,
                                                  double2 *__restrict__ out)
{
    const int jc = blockIdx.x, lane = threadIdx.x;
    double sx = 0, sy = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const double2 v = part[(size_t)(lane + 64 * b) * m * q + jc];
        sx += v.x;
        sy += v.y;
    }
    for (int off = 32; off >= 1; off >>= 1) {
        sx += __shfl_xor(sx, off, 64);
        sy += __shfl_xor(sy, off, 64);
    }
    if (lane == 0) out[jc] = (mask >> (jc % q)) & 1u ? double2{sx, sy} : double2{0.0, 0.0};
}

// w[i][c] -= sum_j h[j][c] V_j[i][c]
__global__ void k_axpys_cols(const double2 *__restrict__ Vb, int n, int m, int q, const double2 *__restrict__ h,
                             double2 *w)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)n * q) return;
    const int c = (int)(i % q);
    double2 acc = w[i];
    for (int j = 0; j < m; ++j) {
        const double2 v = Vb[(size_t)j * n * q + i], cf = h[(size_t)j * q + c];
        acc.x -= cf.x * v.x - cf.y * v.y;
        acc.y -= cf.x * v.y + cf.y * v.x;
    }
    w[i] = acc;
}

template <typename T>
__global__ void k_widen(const typename CT<T>::t *__restrict__ src, long long cnt, double2 *__restrict__ dst)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) dst[i] = {(double)src[i].x, (double)src[i].y};
}

// ---------------------------------------------------------------- host driver
void check(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) BH_FAIL(BH_ERR_HIP, "launch of %s failed: %s", what, hipGetErrorString(e));
}

template <typename T>
struct LUWork {
    DevBuf<unsigned long long> slots;      // FP64 panels: the workgroups' candidates
    DevBuf<int> moves;                     // row moves of the last panel
    DevBuf<int> info;
    DevBuf<int> plan;                      // row-interchange plan (k_swap_plan)
    DevBuf<int> tcnt;                      // tournament group counters (zero between panels)
    DevBuf<unsigned long long> tidx;       // tournament candidate sets (tagged row numbers), all levels
    DevBuf<float2> tpan;                   // the panels' entries, two arrays in turn
    DevBuf<float2> top, unext;             // factored winners; block row in the next panel's columns
    DevBuf<int> plan_side;                 // row-interchange plan of the block-column stream
    DevBuf<__bf16> pa_side, pb_side;       // split planes of the block-column stream
    DevBuf<__bf16> pa_u12;                 // split planes of L for the block row
    DevBuf<float2> eblk, eblk_side;        // I - inv(L_bb) of the 128-row diagonal blocks of a block row
                                           // (context stream, block-column stream)
    int eblk_of = -1, eblk_side_of = -1;   // first row of the block row whose inverses they hold
};

template <typename T, int TM, int TN, bool M3, int WPE>
void gemm_launch(Ctx &ctx, hipStream_t s, typename CT<T>::t *A, long long lda, int ar, int ac, int br, int bc, int cr,
                 int cc, int M, int N, int K)
{
    constexpr int BM = 32 * TM, BN = 32 * TN;
    const long long tiles = (long long)((N + BN - 1) / BN) * ((M + BM - 1) / BM);
    BH_REQUIRE(tiles < (1LL << 31), "gemm grid too large");
    const dim3 grid((unsigned)tiles);
    ProfScope prof(ctx, "k_cgemm", 8.0 * M * N * K, s);   // real flops of the complex update
    k_cgemm<T, TM, TN, M3, WPE><<<grid, 256, 0, s>>>(A + (long long)ar * lda + ac, lda,
                                                               A + (long long)br * lda + bc, lda,
                                                               A + (long long)cr * lda + cc, lda, M, N, K);
    check("k_cgemm");
}

// Tile shapes chosen by measurement on MI355X (N = 12288 LU): FP32 3M products,
// 128 x 64 complex tiles, two waves per SIMD; FP64 4M, 64 x 64, two waves per SIMD.
// FP32 products of one tile row (M <= 128, the block rows' updates) take 128 x 32
// tiles at three waves per SIMD: twice the tiles, so a 40k-wide row of them fills
// the device in whole rounds (C3 block rows: 46.5 -> 42.0 ms of FP32 products; each
// entry's sum over k runs in the same order as with 128 x 64 tiles).
template <typename T>
void gemm(Ctx &ctx, hipStream_t s, typename CT<T>::t *A, long long lda, int ar, int ac, int br, int bc, int cr, int cc,
          int M, int N, int K)
{
    if (M <= 0 || N <= 0 || K <= 0) return;
    BH_REQUIRE(K % kBK == 0, "gemm K=%d not a multiple of %d", K, kBK);
    if constexpr (sizeof(T) == 4) {
        if (M <= 128) gemm_launch<T, 4, 1, true, 3>(ctx, s, A, lda, ar, ac, br, bc, cr, cc, M, N, K);
        else gemm_launch<T, 4, 2, true, 2>(ctx, s, A, lda, ar, ac, br, bc, cr, cc, M, N, K);
    } else {
        gemm_launch<T, 2, 2, false, 2>(ctx, s, A, lda, ar, ac, br, bc, cr, cc, M, N, K);
    }
}

template <typename T>
void laswp(Ctx &ctx, hipStream_t s, typename CT<T>::t *A, long long lda, int k1, int k2, const long long *ipiv, int c0,
           int c1, int c2, int c3, int *plan)
{
    const int w = std::max(0, c1 - c0) + std::max(0, c3 - c2);
    const int len = k2 - k1;
    if (w <= 0 || len <= 0) return;
    ProfScope prof(ctx, "k_laswp", 2.0 * 2 * len * w * sizeof(typename CT<T>::t), s);   // upper bound: every slot moves
    BH_REQUIRE(len <= kMaxSwaps, "laswp: %d interchanges exceed %d", len, kMaxSwaps);
    k_swap_plan<<<1, 256, 0, s>>>(ipiv, k1, k2, plan);
    check("k_swap_plan");
    constexpr int CW = laswp_cols<T>();
    const size_t shm = sizeof(T) == 4 ? 0 : (size_t)2 * len * CW * sizeof(typename CT<T>::t);
    k_laswp_apply<T><<<(w + CW - 1) / CW, 256, shm, s>>>(A, lda, plan, len, c0, std::max(c0, c1), c2, std::max(c2, c3));
    check("k_laswp_apply");
}

// Rows [r, r + m) (m <= 32) of the columns [bc, bc + ncols) := L^-1 times them, L the unit lower
// triangle at (r, r).
void trsm64(hipStream_t s, double2 *A, long long lda, int r, int m, int bc, int ncols)
{
    if (ncols <= 0 || m <= 0) return;
    k_apply64<<<(ncols + 15) / 16, 256, 0, s>>>(A, lda, r, r, m, nullptr, bc, bc, bc, bc + ncols);
    check("k_apply64");
}

// FP64 panel [c, c + pw) of the block column [k, k + kb): the panel, then the row moves and the
// panel's block row in the block's other columns, then the update of the columns to its right.
void panel64(Ctx &ctx, hipStream_t s, LUWork<double> &W, double2 *A, long long lda, int n, int k, int kb, int c, int pw,
             long long *ipiv)
{
    const int rows = n - c;
    const int G = rows <= kP64TOne ? 1 : (rows + kP64T - 1) / kP64T;
    const int stride = (n + kP64T - 1) / kP64T;
    const Panel64Slots sl{stride, W.slots.p, W.slots.p + (size_t)4 * stride, W.info.p, W.moves.p};
    {
        ProfScope prof(ctx, "k_panel", (double)rows * pw * sizeof(double2) * 2, s);
        if (G == 1) {
            k_panel64<kP64TOne><<<1, kP64TOne, 0, s>>>(A, lda, n, c, pw, ipiv, sl);
        } else {
            k_panel64<kP64T><<<G, kP64T, 0, s>>>(A, lda, n, c, pw, ipiv, sl);
        }
        check("k_panel64");
    }
    const int cols = (c - k) + (k + kb - (c + pw));
    if (cols > 0) {
        k_apply64<<<(cols + 15) / 16, 256, 0, s>>>(A, lda, c, c, pw, W.moves.p, k, c, c + pw, k + kb);
        check("k_apply64");
    }
    if (c + pw < k + kb)
        gemm<double>(ctx, s, A, lda, c + pw, c, c, c + pw, c + pw, c + pw, n - (c + pw), k + kb - (c + pw), pw);
}

// One panel's launches, for the single and the batched schedule: the tournament's workgroups
// and k_tslu_apply's arguments and workgroups for the panel [c, c + pw) of the block column
// [k, k + kb).
struct TsluPanel {
    int nsets0, prev, upd_n, blocks, apply_blocks;
    const float2 *P;
    TsluApply ap;
};

TsluPanel tslu_plan(float2 *A, long long lda, int n, int k, int kb, int c, int pw, float2 *tpan, const float2 *top,
                    const int *moves, float2 *unext)
{
    TsluPanel t{};
    float2 *P[2] = {tpan, tpan + (size_t)n * kPW};
    const int turn = (c / kPW) & 1;
    t.P = P[turn];
    t.nsets0 = (n - c + kTsluRows - 1) / kTsluRows;
    t.prev = c > k ? 1 : 0;
    t.upd_n = t.prev ? std::max(0, k + kb - (c + kPW)) : 0;
    const long long tiles = t.upd_n > 0 ? (long long)((n - c + 127) / 128) * ((t.upd_n + 63) / 64) : 0;
    BH_REQUIRE(t.nsets0 + 1 + tiles < (1LL << 31), "tournament grid too large");
    t.blocks = (int)(t.nsets0 + t.prev + tiles);
    const int nextw = std::min(kPW, k + kb - (c + pw));
    const int b0 = std::min(c + pw + kPW, k + kb), w = (c - k) + (k + kb - b0), nsw = (w + 15) / 16;
    t.ap = TsluApply{A, lda, n, c, pw, top, moves, k, c, b0, k + kb, nsw, nextw, t.P, P[turn ^ 1], unext};
    const int ar = tslu_apply_row_count(n - c);
    t.apply_blocks = nsw + (n - c + ar - 1) / ar;
    return t;
}

// Panel of columns [c, c + pw) of the block column [k, k + kb) by tournament
// pivoting.  One launch runs the tournament, which writes ipiv[c .. c+pw), and applies the
// previous panel's update to the block's columns right of this panel; the apply launch
// moves the rows in the block's other columns, finishes the panel rows, forms the panel's
// block row and brings the next panel up to date.
void tslu_panel(Ctx &ctx, hipStream_t s, LUWork<float> &W, float2 *A, long long lda, int n, int k, int kb, int c,
                int pw, long long *ipiv)
{
    const TsluFinal fin{ipiv, W.top.p, W.moves.p, W.info.p};
    const TsluPanel t = tslu_plan(A, lda, n, k, kb, c, pw, W.tpan.p, W.top.p, W.moves.p, W.unext.p);
    {
        ProfScope prof(ctx, "k_tslu_panel", (double)(n - c) * pw * sizeof(float2), s);
        if (!t.prev) {
            k_tslu_load<<<(unsigned)(((long long)(n - c) * kPW + 255) / 256), 256, 0, s>>>(A, lda, n, c, pw, (float2 *)t.P);
            check("k_tslu_load");
        }
        k_tslu_panel<<<(unsigned)t.blocks, kTsluT, 0, s>>>(A, lda, n, c, pw, t.nsets0, t.prev, t.upd_n, t.P, W.unext.p,
                                                          TsluWork{W.tcnt.p, W.tidx.p}, fin);
        check("k_tslu_panel");
    }
    ProfScope prof(ctx, "k_tslu_apply", (double)(n - c) * pw * sizeof(float2) * (t.ap.nextw ? 4 : 2), s);
    k_tslu_apply<<<(unsigned)t.apply_blocks, 256, 0, s>>>(t.ap);
    check("k_tslu_apply");
}

// Trailing update C -= A B through split-bf16 planes (FP32 path only).
// With reuse_a, PA already holds the planes of the same A (same ar, ac, M, K).
void gemm_split(Ctx &ctx, hipStream_t s, float2 *A, long long lda, int ar, int ac, int br, int bc, int cr, int cc, int M,
                int N, int K, DevBuf<__bf16> &PA, DevBuf<__bf16> &PB, bool reuse_a = false)
{
    if (M <= 0 || N <= 0 || K <= 0) return;
    BH_REQUIRE(K % kSplitBK == 0, "split gemm K=%d not a multiple of %d", K, kSplitBK);
    BH_REQUIRE(!reuse_a || PA.n >= (size_t)4 * M * K, "split gemm: no planes to reuse");
    PA.ensure((size_t)4 * M * K);
    PB.ensure((size_t)4 * N * K);
    {
        ProfScope prof(ctx, "k_split", 8.0 * ((reuse_a ? 0.0 : (double)M) + N) * K * 2.0, s);
        const long long na = (long long)M * K;
        if (!reuse_a) {
            k_split_rows<<<(unsigned)((na + 255) / 256), 256, 0, s>>>(A + (long long)ar * lda + ac, lda, M, K, PA.p);
            check("k_split_rows");
        }
        dim3 g2((unsigned)((N + 31) / 32), (unsigned)((K + 31) / 32));
        k_split_cols<<<g2, 256, 0, s>>>(A + (long long)br * lda + bc, lda, K, N, PB.p);
        check("k_split_cols");
    }
    // work: bf16 MFMA flops executed (3 products per real product, 4 real per complex)
    ProfScope prof(ctx, "k_cgemm_bf16x3", 24.0 * M * N * K, s);
    // 128 x 128 complex tiles, 8 waves (4 x 2) of 32 x 64
    constexpr int TM = 2, TN = 4, WM = 4, WN = 2, BM = 16 * TM * WM, BN = 16 * TN * WN;
    const long long tiles = (long long)((N + BN - 1) / BN) * ((M + BM - 1) / BM);
    BH_REQUIRE(tiles < (1LL << 31), "gemm grid too large");
    k_cgemm_bf16x3<TM, TN, WM, WN><<<dim3((unsigned)tiles), 64 * WM * WN, 0, s>>>(
        PA.p, PB.p, A + (long long)cr * lda + cc, lda, M, N, K);
    check("k_cgemm_bf16x3");
}

// Block row of rows [k, k + kb): A[k:k+kb, c0:c1) := L11^-1 A[k:k+kb, c0:c1) (with PB,
// FP32 blocks deeper than kNBInner solve their halves and join them with one
// split-bf16 product through PB's planes).
template <typename T>
void block_row_u12(Ctx &ctx, hipStream_t s, LUWork<T> &W, typename CT<T>::t *A, long long lda, int n, int k, int kb,
                   int c0, int c1, DevBuf<__bf16> *PB = nullptr);

// Block column [k, k + kb): its 32-column panels and the updates inside the block.
template <typename T>
void factor_block(Ctx &ctx, hipStream_t s, LUWork<T> &W, typename CT<T>::t *A, long long lda, int n, int k, int kb,
                  long long *ipiv)
{
    if constexpr (sizeof(T) == 4) {
        if (kb > kNBInner) {
            // left half; its interchanges, block row and update reach the right half; right
            // half; its interchanges reach the left half
            const int h = kNBInner;
            factor_block<T>(ctx, s, W, A, lda, n, k, h, ipiv);
            for (int q = k; q < k + h; q += kMaxSwaps)
                laswp<T>(ctx, s, A, lda, q, std::min(q + kMaxSwaps, k + h), ipiv, k + h, k + kb, 0, 0, W.plan_side.p);
            block_row_u12<T>(ctx, s, W, A, lda, n, k, h, k + h, k + kb);
            gemm_split(ctx, s, A, lda, k + h, k, k, k + h, k + h, k + h, n - (k + h), kb - h, h, W.pa_side, W.pb_side);
            factor_block<T>(ctx, s, W, A, lda, n, k + h, kb - h, ipiv);
            for (int q = k + h; q < k + kb; q += kMaxSwaps)
                laswp<T>(ctx, s, A, lda, q, std::min(q + kMaxSwaps, k + kb), ipiv, k, k + h, 0, 0, W.plan_side.p);
            return;
        }
    }
    for (int sp = 0; sp < kb; sp += kPW) {
        const int c = k + sp, pw = std::min(kPW, kb - sp);
        if constexpr (sizeof(T) == 4) {
            tslu_panel(ctx, s, W, A, lda, n, k, kb, c, pw, ipiv);
        } else {
            panel64(ctx, s, W, A, lda, n, k, kb, c, pw, ipiv);
        }
    }
}

// E = I - S for kb/kIB blocks S = inv(L_bb) as k_trinv<true> leaves them (unit
// diagonal, zero above it): zero diagonal, negated strictly lower part.
__global__ void k_inv_to_e(float2 *E, int nblk)
{
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)nblk * kIB * kIB) return;
    const int i = (int)(idx / kIB % kIB), j = (int)(idx % kIB);
    const float2 v = E[idx];
    E[idx] = i == j ? float2{0, 0} : float2{-v.x, -v.y};
}

// Rows [r, r + kIB) of a block row, columns [c0, c1): C <- inv(L_bb) C, formed as
// C - E C with E = I - inv(L_bb).  The product has one tile row (M = kIB = BM), so
// each workgroup reads, as B, exactly the columns of C it writes, and reads all of
// them (main loop, then the epilogue's reads of C) before its first write.  128 x 32
// tiles, as for the other one-row products.
void blockrow_apply_inverse(Ctx &ctx, hipStream_t s, const float2 *E, float2 *A, long long lda, int r, int c0, int c1)
{
    const int N = c1 - c0;
    static_assert(32 * 4 == kIB, "one tile row of the FP32 product must cover the block");
    ProfScope prof(ctx, "k_cgemm", 8.0 * kIB * (double)N * kIB, s);
    float2 *C = A + (long long)r * lda + c0;
    k_cgemm<float, 4, 1, true, 3><<<(unsigned)((N + 31) / 32), 256, 0, s>>>(E, kIB, C, lda, C, lda, kIB, N, kIB);
    check("k_cgemm");
}

// U12 = L11^-1 A12 for block row [k, k + kb) over the columns [c0, n).
template <typename T>
void block_row_u12(Ctx &ctx, hipStream_t s, LUWork<T> &W, typename CT<T>::t *A, long long lda, int n, int k, int kb,
                   int c0, int c1, DevBuf<__bf16> *PB)
{
    if (c1 <= c0) return;
    if constexpr (sizeof(T) == 4) {
        if (kb > kNBInner && PB) {
            // top half, its update of the bottom half (split-bf16 products), bottom half
            const int h = kNBInner;
            block_row_u12<T>(ctx, s, W, A, lda, n, k, h, c0, c1);
            gemm_split(ctx, s, A, lda, k + h, k, k, c0, k + h, c0, kb - h, c1 - c0, h, W.pa_u12, *PB);
            block_row_u12<T>(ctx, s, W, A, lda, n, k + h, kb - h, c0, c1);
            return;
        }
    }
    if constexpr (sizeof(T) == 4) {
        // FP32 block rows by 128-row blocks: the inverses of L11's diagonal blocks, then
        // per block one product with I - inv(L_bb) and one K = 128 update below it.  (A block
        // row is only formed where columns follow the block, which is then a full one.)
        BH_REQUIRE(kb % kIB == 0 && kb <= kNBInner, "block row of %d rows", kb);
        const int nb = kb / kIB;
        const bool side = s != ctx.stream;
        float2 *E = (side ? W.eblk_side : W.eblk).p;
        int &of = side ? W.eblk_side_of : W.eblk_of;
        if (of != k) {   // a block row taken in two column ranges reuses its inverses
            ProfScope prof(ctx, "k_trinv", 4.0 * kIB * (double)kIB * kIB * nb / 3.0, s);   // kIB^3/6 complex MACs per block
            k_trinv<true><<<nb, kIB * kTrinvParts, 0, s>>>(A + (long long)k * lda + k, lda, kb, E);
            check("k_trinv");
            k_inv_to_e<<<(unsigned)(((long long)nb * kIB * kIB + 255) / 256), 256, 0, s>>>(E, nb);
            check("k_inv_to_e");
            of = k;
        }
        for (int b = 0; b < nb; ++b) {
            const int r = k + b * kIB;
            blockrow_apply_inverse(ctx, s, E + (size_t)b * kIB * kIB, A, lda, r, c0, c1);
            if (b + 1 < nb) gemm<T>(ctx, s, A, lda, r + kIB, r, r, c0, r + kIB, c0, k + kb - (r + kIB), c1 - c0, kIB);
        }
    } else {
        for (int sp = 0; sp < kb; sp += kPW) {
            const int pw = std::min(kPW, kb - sp);
            trsm64(s, A, lda, k + sp, pw, c0, c1 - c0);
            if (sp + pw < kb)
                gemm<T>(ctx, s, A, lda, k + sp + pw, k + sp, k + sp, c0, k + sp + pw, c0, kb - (sp + pw), c1 - c0, pw);
        }
    }
}

// Right-looking blocked LU (panels of 32 columns; FP64: LAPACK's partial pivoting, FP32:
// tournament pivoting), looking one block ahead: after block k's U12 is formed, the next
// block column is updated first and factored on a second stream while the rest of the
// trailing matrix is updated on the context stream; the two touch disjoint columns.  (FP64,
// 17,406 rows: 578 ms for the whole solve with every step on one stream and the former
// panel, 346 ms now.)
void invert_diagonal_blocks(hipStream_t s, const float2 *LU, long long lda, int n, float2 *Dinv);

template <typename T>
struct LUBuffers {
    LUWork<T> W;
    DevBuf<__bf16> PA, PB;   // split planes of the trailing updates
};

// The factorisations' workspaces and their block-column stream, kept in the context.
struct LUCache {
    std::mutex mu;
    LUBuffers<float> b;
    LUBuffers<double> b64;
    hipStream_t s2 = nullptr;
    hipEvent_t ready = nullptr, done = nullptr;
    ~LUCache() {
        if (s2) { (void)hipStreamSynchronize(s2); (void)hipStreamDestroy(s2); }
        if (ready) (void)hipEventDestroy(ready);
        if (done) (void)hipEventDestroy(done);
    }
};

LUCache &lu_cache(Ctx &ctx)
{
    static std::mutex create;
    std::lock_guard<std::mutex> g(create);
    if (!ctx.lu_cache) ctx.lu_cache = std::make_shared<LUCache>();
    return *static_cast<LUCache *>(ctx.lu_cache.get());
}

// one gate per device for all contexts of the process
PanelGate &panel_gate(int device)
{
    static std::mutex mu;
    static std::map<int, PanelGate> gates;
    std::lock_guard<std::mutex> g(mu);
    return gates[device];
}

// dinv (FP32 only, may be NULL): the diagonal-block inverses and couplings of the
// factors are formed on the context stream before the workspace is released, so
// the device does not idle while the host frees it.
template <typename T>
void lu_factor(Ctx &ctx, typename CT<T>::t *A, long long lda, int n, long long *ipiv, int *info_host,
               bool split = false, float2 *dinv = nullptr)
{
    hipStream_t s = ctx.stream;
    // the context's cached workspace unless another factorisation holds it
    LUCache *cache = &lu_cache(ctx);
    std::unique_lock<std::mutex> held(cache->mu, std::try_to_lock);
    std::unique_ptr<LUBuffers<T>> own;
    LUBuffers<T> *buf = nullptr;
    if (held.owns_lock()) {
        if constexpr (sizeof(T) == 4) buf = &cache->b;
        else buf = &cache->b64;
        if (cache->s2) BH_CHECK_HIP(hipStreamSynchronize(cache->s2));   // after a failed call
    } else {
        cache = nullptr;
        own = std::make_unique<LUBuffers<T>>();
        buf = own.get();
    }
    PanelPlaces places;   // FP64: the panels' workgroups, until the last panel is done
    LUWork<T> &W = buf->W;
    DevBuf<__bf16> &PA = buf->PA, &PB = buf->PB;
    W.eblk_of = W.eblk_side_of = -1;
    W.info.ensure(1);
    W.moves.ensure(2 * kPW);
    W.plan.ensure(4 * kMaxSwaps);
    BH_CHECK_HIP(hipMemsetAsync(W.info.p, 0, sizeof(int), s));
    // a panel whose wait ran out leaves places of moves as they were: rows of the matrix, not chance
    BH_CHECK_HIP(hipMemsetAsync(W.moves.p, 0, 2 * kPW * sizeof(int), s));
    // block column of the right-looking LU (trailing-update depth); the FP32
    // path's deeper blocks halve the C traffic per flop of the trailing update
    auto depth = [&](int k) { return sizeof(T) == 4 ? fp32_block_depth(n, k, split) : kNBFP64; };
    int planes_of = -1;   // block whose L21 planes PA holds
    auto trailing = [&](hipStream_t st, int k, int kb, int c0, int c1) {
        // A[k+kb:, c0:c1) -= L21 U12[:, c0:c1)
        if (c1 <= c0 || k + kb >= n) return;
        if constexpr (sizeof(T) == 4) {
            if (split) {
                gemm_split(ctx, st, A, lda, k + kb, k, k, c0, k + kb, c0, n - (k + kb), c1 - c0, kb, PA, PB,
                           planes_of == k);
                planes_of = k;
                return;
            }
        }
        gemm<T>(ctx, st, A, lda, k + kb, k, k, c0, k + kb, c0, n - (k + kb), c1 - c0, kb);
    };
    if constexpr (sizeof(T) == 8) {
        // panels exchange tagged words: cleared, so that no tag of an earlier factorisation is there
        const int G = (n + kP64T - 1) / kP64T;
        int per_cu = 0;
        BH_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_panel64<kP64T>, kP64T, 0));
        BH_REQUIRE(G <= per_cu * ctx.num_cus, "panel of %d rows: its workgroups cannot all be resident", n);
        if (n > kP64TOne) places.take(panel_gate(ctx.device), G, (long long)per_cu * ctx.num_cus);
        const size_t words = (size_t)G * (4 + 8 * kPW);
        W.slots.ensure(words);
        BH_CHECK_HIP(hipMemsetAsync(W.slots.p, 0, words * sizeof(unsigned long long), s));
    } else {
        // FP32 factors only precondition GMRES-IR: their panels use tournament pivoting.
        // Counters start at zero; candidate words are cleared, so that no tag of an earlier
        // factorisation is there
        const size_t sets = tslu_sets(n);
        W.tcnt.ensure(sets);
        W.tidx.ensure(sets * kPW);
        W.tpan.ensure((size_t)2 * n * kPW);
        BH_CHECK_HIP(hipMemsetAsync(W.tcnt.p, 0, sets * sizeof(int), s));
        BH_CHECK_HIP(hipMemsetAsync(W.tidx.p, 0, sets * kPW * sizeof(unsigned long long), s));
        W.plan_side.ensure(4 * kMaxSwaps);
        W.top.ensure((size_t)kPW * kPW);
        W.unext.ensure((size_t)kPW * kPW);
        W.eblk.ensure((size_t)(kNBInner / kIB) * kIB * kIB);
        W.eblk_side.ensure((size_t)(kNBInner / kIB) * kIB * kIB);
    }
    {
        hipStream_t s2 = nullptr;
        hipEvent_t ready = nullptr, done = nullptr;
        struct Cleanup {   // a stream and events of this call only (no cache)
            hipStream_t &s2;
            hipEvent_t &a, &b;
            bool own;
            ~Cleanup() {
                if (!own) return;
                if (s2) { (void)hipStreamSynchronize(s2); (void)hipStreamDestroy(s2); }
                if (a) (void)hipEventDestroy(a);
                if (b) (void)hipEventDestroy(b);
            }
        } cleanup{s2, ready, done, cache == nullptr};
        if (cache) {
            if (!cache->s2) BH_CHECK_HIP(hipStreamCreateWithFlags(&cache->s2, hipStreamNonBlocking));
            if (!cache->ready) BH_CHECK_HIP(hipEventCreateWithFlags(&cache->ready, hipEventDisableTiming));
            if (!cache->done) BH_CHECK_HIP(hipEventCreateWithFlags(&cache->done, hipEventDisableTiming));
            s2 = cache->s2;
            ready = cache->ready;
            done = cache->done;
        } else {
            BH_CHECK_HIP(hipStreamCreateWithFlags(&s2, hipStreamNonBlocking));
            BH_CHECK_HIP(hipEventCreateWithFlags(&ready, hipEventDisableTiming));
            BH_CHECK_HIP(hipEventCreateWithFlags(&done, hipEventDisableTiming));
        }
        struct Drain {   // after an error too no panel runs once the places are given back
            hipStream_t s, s2;
            ~Drain() {
                if (!s) return;
                (void)hipStreamSynchronize(s);
                (void)hipStreamSynchronize(s2);
            }
        } drain{s, s2};
        factor_block<T>(ctx, s, W, A, lda, n, 0, std::min(depth(0), n), ipiv);
        // block k is factored; its interchanges reach the other columns (in pieces
        // of at most kMaxSwaps interchanges, applied in order) over [c0, c1) and [c2, c3)
        auto swaps = [&](int k, int kb, int c0, int c1, int c2, int c3) {
            for (int q = k; q < k + kb; q += kMaxSwaps)
                laswp<T>(ctx, s, A, lda, q, std::min(q + kMaxSwaps, k + kb), ipiv, c0, c1, c2, c3, W.plan.p);
        };
        for (int k = 0, kb = 0; k < n; k += kb) {
            kb = std::min(depth(k), n - k);
            if (k + kb >= n) {
                swaps(k, kb, 0, k, 0, 0);
                break;
            }
            const int nk = k + kb, nkb = std::min(depth(nk), n - nk);
            // near the end the block-column chain is the critical path: there the
            // next block column goes first on its own (interchanges, block row,
            // update) and the rest is brought up to date while it is factored;
            // earlier, one pass over all columns costs the context stream less
            const bool ahead_first = sizeof(T) == 8 || n - nk <= kAheadFirstBelow;
            if (ahead_first) {
                swaps(k, kb, nk, nk + nkb, 0, 0);
                block_row_u12<T>(ctx, s, W, A, lda, n, k, kb, nk, nk + nkb, split ? &PB : nullptr);
            } else {
                swaps(k, kb, 0, k, nk, n);
                block_row_u12<T>(ctx, s, W, A, lda, n, k, kb, nk, n, split ? &PB : nullptr);
            }
            trailing(s, k, kb, nk, nk + nkb);
            BH_CHECK_HIP(hipEventRecord(ready, s));
            if (!ahead_first) {
                // the rest of the update first in host order: the next block column's
                // many short launches are then queued while the long product runs
                trailing(s, k, kb, nk + nkb, n);
            }
            BH_CHECK_HIP(hipStreamWaitEvent(s2, ready, 0));
            factor_block<T>(ctx, s2, W, A, lda, n, nk, nkb, ipiv);
            BH_CHECK_HIP(hipEventRecord(done, s2));
            // the rest, concurrently
            if (ahead_first) {
                swaps(k, kb, 0, k, nk + nkb, n);
                block_row_u12<T>(ctx, s, W, A, lda, n, k, kb, nk + nkb, n, split ? &PB : nullptr);
                trailing(s, k, kb, nk + nkb, n);
            }
            BH_CHECK_HIP(hipStreamWaitEvent(s, done, 0));
        }
        drain.s = nullptr;   // s waits for s2 and is waited for below
    }
    if constexpr (sizeof(T) == 4) {
        if (dinv) invert_diagonal_blocks(s, (const float2 *)A, lda, n, dinv);
    }
    BH_CHECK_HIP(hipMemcpyAsync(info_host, W.info.p, sizeof(int), hipMemcpyDeviceToHost, s));
    BH_CHECK_HIP(hipStreamSynchronize(s));
    if (*info_host < 0) BH_FAIL(BH_ERR_HIP, "LU panel: a workgroup waited in vain for the others' pivot candidates");
}

// forward (unit lower) then backward (upper) substitution on X (n x nrhs, work precision)
// Inverses of the diagonal blocks of both FP32 factors: Dinv[0 .. nb) lower, [nb .. 2nb) upper.
void invert_diagonal_blocks(hipStream_t s, const float2 *LU, long long lda, int n, float2 *Dinv)
{
    const int nb = (n + kIB - 1) / kIB;
    const size_t bsz = (size_t)nb * kIB * kIB;
    k_trinv<true><<<nb, kIB * kTrinvParts, 0, s>>>(LU, lda, n, Dinv);
    check("k_trinv");
    k_trinv<false><<<nb, kIB * kTrinvParts, 0, s>>>(LU, lda, n, Dinv + bsz);
    check("k_trinv");
    k_blk_coupling<true><<<dim3(nb, kIB / 16), 256, 0, s>>>(LU, lda, n, Dinv, Dinv + 2 * bsz);
    check("k_blk_coupling");
    k_blk_coupling<false><<<dim3(nb, kIB / 16), 256, 0, s>>>(LU, lda, n, Dinv + bsz, Dinv + 3 * bsz);
    check("k_blk_coupling");
}

// words[0 .. cnt) = 0 (a kernel rather than a memset node, for callers that capture graphs)
__global__ void k_fill_int(int *words, long long cnt)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) words[i] = 0;
}

// The words of one matrix's triangular solves: kTrsvHead, then 2 (FP32) or 4 (FP64) per value.
size_t trsv_words(int64_t n, bool fp64) { return kTrsvHead + (size_t)n * kMaxRhs * (fp64 ? 4 : 2); }

void trsv_restart(hipStream_t s, bh_matrix *M)
{
    const long long cnt = 2 * (long long)M->tsync.n;
    k_fill_int<<<(unsigned)((cnt + 255) / 256), 256, 0, s>>>((int *)M->tsync.p, cnt);
    check("k_fill_int");
    M->tsync_tickets = 0;
    M->tsync_epoch = 0;
}

// X := U^-1 L^-1 X with the factors of M, X device n x NRHS row-major
template <typename T, int NRHS>
void lu_solve_n(hipStream_t s, bh_matrix *M, typename CT<T>::t *X)
{
    constexpr bool kF64 = std::is_same<T, double>::value;
    const int n = (int)M->n, nb = kF64 ? (n + kTB - 1) / kTB : (n + kIB - 1) / kIB;
    const int grid = std::max(1, std::min(nb, M->ctx->num_cus));   // one workgroup per CU at most
    for (int tri = 0; tri < 2; ++tri) {
        if (M->tsync_tickets + 2LL * nb >= (1LL << 30) || M->tsync_epoch >= (1 << 30)) trsv_restart(s, M);
        const int ticket0 = (int)M->tsync_tickets, epoch = ++M->tsync_epoch;
        M->tsync_tickets += nb + grid;
        if constexpr (kF64) {
            const double2 *A = (const double2 *)M->lu64.p;
            if (tri == 0) k_trsv64<true, NRHS><<<grid, kTrsvT, 0, s>>>(A, M->lda, n, X, M->tsync.p, ticket0, epoch);
            else k_trsv64<false, NRHS><<<grid, kTrsvT, 0, s>>>(A, M->lda, n, X, M->tsync.p, ticket0, epoch);
            check("k_trsv64");
        } else {
            const float2 *A = (const float2 *)M->lu32.p, *DL = (const float2 *)M->dinv32.p;
            const size_t bsz = (size_t)nb * kIB * kIB;
            const float2 *DU = DL + bsz, *GL = DL + 2 * bsz, *GU = DL + 3 * bsz;
            if (tri == 0) k_trsv_flag<true, NRHS><<<grid, kTrsvT, 0, s>>>(A, M->lda, n, DL, GL, X, M->tsync.p, ticket0, epoch);
            else k_trsv_flag<false, NRHS><<<grid, kTrsvT, 0, s>>>(A, M->lda, n, DU, GU, X, M->tsync.p, ticket0, epoch);
            check("k_trsv_flag");
        }
    }
}

template <typename T>
void lu_solve(hipStream_t s, bh_matrix *M, typename CT<T>::t *X, int nrhs)
{
    switch (nrhs) {
    case 1: lu_solve_n<T, 1>(s, M, X); break;
    case 2: lu_solve_n<T, 2>(s, M, X); break;
    case 3: lu_solve_n<T, 3>(s, M, X); break;
    case 4: lu_solve_n<T, 4>(s, M, X); break;
    case 5: lu_solve_n<T, 5>(s, M, X); break;
    case 6: lu_solve_n<T, 6>(s, M, X); break;
    case 7: lu_solve_n<T, 7>(s, M, X); break;
    case 8: lu_solve_n<T, 8>(s, M, X); break;
    default: BH_FAIL(BH_ERR_INVALID, "nrhs %d out of range", nrhs);
    }
}

long long padded_ld(int64_t n) { return (n + 63) / 64 * 64; }

// ---------------------------------------------------------------- batched FP32 factorisation
// Several matrices factored in shared launches: every launch of the single-matrix
// schedule (512-deep block columns: tournament panels, their apply, interchanges, block
// rows, split-bf16 trailing updates; then the diagonal-block inverses of the solves) is
// issued once for all matrices that have it at that step.  A workgroup finds its matrix in
// the table of each matrix's first workgroup and runs the single-matrix kernel's body on
// that matrix's arguments, so each matrix gets the factors (and pivots) it gets alone.
struct LoadBA {
    const float2 *A;
    long long lda;
    int n, c, pw;
    float2 *P;
};
struct PanelBA {
    float2 *A;
    long long lda;
    int n, c, pw, nsets0, prev, upd_n;
    const float2 *P, *unext;
    TsluWork tw;
    TsluFinal fin;
};
struct SwapBA {
    const long long *ipiv;
    int k1, k2;
    int *plan;
};
struct LaswpBA {
    float2 *A;
    long long lda;
    const int *plan;
    int len, c0, c1, c2, c3;
};
struct TrinvBA {
    const float2 *A;
    long long lda;
    int n;
    float2 *Dinv;
};
struct ToEBA {
    float2 *E;
    int nblk;
};
struct CgemmBA {
    const float2 *A;
    long long lda;
    const float2 *B;
    long long ldb;
    float2 *C;
    long long ldc;
    int M, N, K;
};
struct SplitRowsBA {
    const float2 *A;
    long long lda;
    int rows, K;
    __bf16 *P;
};
struct SplitColsBA {
    const float2 *B;
    long long ldb;
    int K, cols, gx;
    __bf16 *P;
};
struct Bf16BA {
    const __bf16 *PA, *PB;
    float2 *C;
    long long ldc;
    int M, N, K;
};
struct CouplingBA {
    const float2 *A;
    long long lda;
    int n, gx;
    const float2 *Dinv;
    float2 *G;
};

#define BH_BATCH_ITEM(ARGS)                              \
    const int r_ = batch_find(first, count, blockIdx.x); \
    const auto &a = ARGS[r_];                            \
    const int bid = (int)blockIdx.x - first[r_];

__global__ __launch_bounds__(256) void k_tslu_load_batch(const LoadBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    tslu_load_body(a.A, a.lda, a.n, a.c, a.pw, a.P, bid);
}

__global__ __launch_bounds__(kTsluT, 2) void k_tslu_panel_batch(const PanelBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    tslu_panel_body(a.A, a.lda, a.n, a.c, a.pw, a.nsets0, a.prev, a.upd_n, a.P, a.unext, a.tw, a.fin, bid);
}

__global__ __launch_bounds__(256) void k_tslu_apply_batch(const TsluApply *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    tslu_apply_body(a, bid);
}

__global__ __launch_bounds__(256) void k_swap_plan_batch(const SwapBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    (void)bid;
    swap_plan_body(a.ipiv, a.k1, a.k2, a.plan);
}

__global__ __launch_bounds__(256) void k_laswp_apply_batch(const LaswpBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    laswp_apply_body<float>(a.A, a.lda, a.plan, a.len, a.c0, a.c1, a.c2, a.c3, bid);
}

template <bool LOWER>
__global__ __launch_bounds__(kIB * kTrinvParts) void k_trinv_batch(const TrinvBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    trinv_body<LOWER>(a.A, a.lda, a.n, a.Dinv, bid);
}

__global__ __launch_bounds__(256) void k_inv_to_e_batch(const ToEBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    const long long idx = (long long)bid * 256 + threadIdx.x;
    if (idx >= (long long)a.nblk * kIB * kIB) return;
    const int i = (int)(idx / kIB % kIB), j = (int)(idx % kIB);
    const float2 v = a.E[idx];
    a.E[idx] = i == j ? float2{0, 0} : float2{-v.x, -v.y};
}

__global__ __launch_bounds__(256, 2) void k_cgemm_batch(const CgemmBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    cgemm_tile<float, 4, 2, true>(bid, a.A, a.lda, a.B, a.ldb, a.C, a.ldc, a.M, a.N, a.K);
}

__global__ __launch_bounds__(256) void k_split_rows_batch(const SplitRowsBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    split_rows_body(a.A, a.lda, a.rows, a.K, a.P, (long long)bid * 256 + threadIdx.x);
}

__global__ __launch_bounds__(256) void k_split_cols_batch(const SplitColsBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    split_cols_body(a.B, a.ldb, a.K, a.cols, a.P, bid % a.gx, bid / a.gx);
}

__global__ __launch_bounds__(512, 2) void k_cgemm_bf16x3_batch(const Bf16BA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    cgemm_bf16x3_body<2, 4, 4, 2>(a.PA, a.PB, a.C, a.ldc, a.M, a.N, a.K, bid);
}

template <bool LOWER>
__global__ __launch_bounds__(256) void k_blk_coupling_batch(const CouplingBA *args, const int *first, int count)
{
    BH_BATCH_ITEM(args)
    blk_coupling_body<LOWER>(a.A, a.lda, a.n, a.Dinv, a.G, bid % a.gx, bid / a.gx);
}

#undef BH_BATCH_ITEM

// Largest matrix the batched schedule takes: every block column 512 deep (the single
// schedule's deeper blocks start above this trailing size).
constexpr int kBatchMaxN = kNBDeepAbove;

namespace {

enum BatchKind : int {
    kBkLoad, kBkPanel, kBkApply, kBkSwap, kBkLaswp, kBkTrinvL, kBkTrinvU, kBkToE, kBkCgemm, kBkSplitRows, kBkSplitCols,
    kBkBf16, kBkCoupleL, kBkCoupleU
};

struct BatchLaunch {
    int kind;
    int count;            // matrices in this launch
    int blocks;           // total workgroups
    size_t args, first;   // offsets into the uploaded table
    size_t shm;
    double work;          // for the profiler: the single-matrix kernels' work units, summed
};

// Host-side schedule: launches in order and one table of their arguments.
struct BatchPlan {
    std::vector<char> blob;
    std::vector<BatchLaunch> launches;
    template <typename S>
    size_t put(const std::vector<S> &v) {
        size_t off = (blob.size() + 15) & ~(size_t)15;
        blob.resize(off + v.size() * sizeof(S));
        std::memcpy(blob.data() + off, v.data(), v.size() * sizeof(S));
        return off;
    }
    // items: (args, blocks) per matrix; matrices with no blocks are left out
    template <typename S>
    void add(int kind, const std::vector<std::pair<S, long long>> &items, size_t shm = 0, double work = 0) {
        std::vector<S> a;
        std::vector<int> first{0};
        for (const auto &it : items) {
            if (it.second <= 0) continue;
            BH_REQUIRE((long long)first.back() + it.second < (1LL << 31), "batched launch too large");
            a.push_back(it.first);
            first.push_back(first.back() + (int)it.second);
        }
        if (a.empty()) return;
        BatchLaunch L{kind, (int)a.size(), first.back(), put(a), 0, shm, work};
        L.first = put(first);
        launches.push_back(L);
    }
};

struct BatchMat {
    bh_matrix *M;
    int n;
    long long lda;
    float2 *A;
    long long *ipiv;
    // workspace (device)
    int *tcnt, *moves, *plan, *info;
    unsigned long long *tidx;
    float2 *tpan, *top, *unext, *eblk, *dinv;
    __bf16 *pa, *pb;
};

void plan_factor(BatchPlan &P, std::vector<BatchMat> &mats)
{
    int nmax = 0;
    for (auto &m : mats) nmax = std::max(nmax, m.n);
    for (int k = 0; k < nmax; k += kNBInner) {
        // the block column [k, k + kb) of every matrix that has it: its panels
        for (int sp = 0; sp < kNBInner; sp += kPW) {
            std::vector<std::pair<LoadBA, long long>> ld;
            std::vector<std::pair<PanelBA, long long>> pan;
            std::vector<std::pair<TsluApply, long long>> app;
            double wp = 0, wa = 0;
            for (auto &m : mats) {
                if (m.n <= k) continue;
                const int kb = std::min(kNBInner, m.n - k);
                if (sp >= kb) continue;
                const int c = k + sp, pw = std::min(kPW, kb - sp);
                const TsluPanel t = tslu_plan(m.A, m.lda, m.n, k, kb, c, pw, m.tpan, m.top, m.moves, m.unext);
                if (!t.prev)
                    ld.push_back({LoadBA{m.A, m.lda, m.n, c, pw, (float2 *)t.P}, ((long long)(m.n - c) * kPW + 255) / 256});
                pan.push_back({PanelBA{m.A, m.lda, m.n, c, pw, t.nsets0, t.prev, t.upd_n, t.P, m.unext,
                                       TsluWork{m.tcnt, m.tidx}, TsluFinal{m.ipiv, m.top, m.moves, m.info}}, t.blocks});
                wp += (double)(m.n - c) * pw * sizeof(float2);
                app.push_back({t.ap, t.apply_blocks});
                wa += (double)(m.n - c) * pw * sizeof(float2) * (t.ap.nextw ? 4 : 2);
            }
            if (pan.empty()) break;
            P.add(kBkLoad, ld);
            P.add(kBkPanel, pan, 0, wp);
            P.add(kBkApply, app, 0, wa);
        }
        // interchanges of the block reach the columns left of it, and right of it when
        // it is not the last block (pieces of kMaxSwaps, in order)
        for (int q0 = 0; q0 < kNBInner; q0 += kMaxSwaps) {
            std::vector<std::pair<SwapBA, long long>> sw;
            std::vector<std::pair<LaswpBA, long long>> la;
            double wl = 0;
            for (auto &m : mats) {
                if (m.n <= k) continue;
                const int kb = std::min(kNBInner, m.n - k), nk = k + kb;
                const int q = k + q0;
                if (q >= nk) continue;
                const int len = std::min(kMaxSwaps, nk - q);
                const int c2 = nk < m.n ? nk : 0, c3 = nk < m.n ? m.n : 0;
                const int w = k + (c3 - c2);
                if (w <= 0) continue;
                sw.push_back({SwapBA{m.ipiv, q, q + len, m.plan}, 1});
                constexpr int cw = laswp_cols<float>();
                la.push_back({LaswpBA{m.A, m.lda, m.plan, len, 0, k, c2, c3}, (w + cw - 1) / cw});
                wl += 2.0 * 2 * len * w * sizeof(float2);
            }
            P.add(kBkSwap, sw);
            P.add(kBkLaswp, la, 0, wl);
        }
        // block row U12 = L11^-1 A12 and the trailing update, for matrices with columns right
        // of the block: inverses of L11's 128-row diagonal blocks, then per 128-row block
        // one product with I - inv(L_bb) and one K = 128 update of the rows below
        std::vector<BatchMat *> rest;
        for (auto &m : mats)
            if (m.n > k + kNBInner) rest.push_back(&m);
        if (rest.empty()) continue;
        const int nk = k + kNBInner, nbb = kNBInner / kIB;
        {
            std::vector<std::pair<TrinvBA, long long>> ti;
            std::vector<std::pair<ToEBA, long long>> te;
            for (auto *m : rest) {
                ti.push_back({TrinvBA{m->A + (long long)k * m->lda + k, m->lda, kNBInner, m->eblk}, nbb});
                te.push_back({ToEBA{m->eblk, nbb}, ((long long)nbb * kIB * kIB + 255) / 256});
            }
            P.add(kBkTrinvL, ti, 0, 4.0 * kIB * (double)kIB * kIB * nbb / 3.0 * rest.size());
            P.add(kBkToE, te);
        }
        for (int b = 0; b < nbb; ++b) {
            const int r = k + b * kIB;
            std::vector<std::pair<CgemmBA, long long>> ap, up;
            double wap = 0, wup = 0;
            for (auto *m : rest) {
                const int N = m->n - nk;
                float2 *C = m->A + (long long)r * m->lda + nk;
                ap.push_back({CgemmBA{m->eblk + (size_t)b * kIB * kIB, kIB, C, m->lda, C, m->lda, kIB, N, kIB},
                              (N + 63) / 64});
                wap += 8.0 * kIB * (double)N * kIB;
                if (b + 1 < nbb) {
                    const int Mr = nk - (r + kIB);
                    up.push_back({CgemmBA{m->A + (long long)(r + kIB) * m->lda + r, m->lda, C, m->lda,
                                          m->A + (long long)(r + kIB) * m->lda + nk, m->lda, Mr, N, kIB},
                                  (long long)((N + 63) / 64) * ((Mr + 127) / 128)});
                    wup += 8.0 * Mr * (double)N * kIB;
                }
            }
            P.add(kBkCgemm, ap, 0, wap);
            P.add(kBkCgemm, up, 0, wup);
        }
        {
            std::vector<std::pair<SplitRowsBA, long long>> sr;
            std::vector<std::pair<SplitColsBA, long long>> sc;
            std::vector<std::pair<Bf16BA, long long>> gm;
            double wsplit = 0, wg = 0;
            for (auto *m : rest) {
                const int Mt = m->n - nk, Nt = m->n - nk, K = kNBInner;
                sr.push_back({SplitRowsBA{m->A + (long long)nk * m->lda + k, m->lda, Mt, K, m->pa},
                              ((long long)Mt * K + 255) / 256});
                const int gx = (Nt + 31) / 32;
                sc.push_back({SplitColsBA{m->A + (long long)k * m->lda + nk, m->lda, K, Nt, gx, m->pb},
                              (long long)gx * ((K + 31) / 32)});
                gm.push_back({Bf16BA{m->pa, m->pb, m->A + (long long)nk * m->lda + nk, m->lda, Mt, Nt, K},
                              (long long)((Nt + 127) / 128) * ((Mt + 127) / 128)});
                wsplit += 8.0 * ((double)Mt + Nt) * K * 2.0;
                wg += 24.0 * Mt * (double)Nt * K;
            }
            P.add(kBkSplitRows, sr, 0, wsplit);
            P.add(kBkSplitCols, sc);
            P.add(kBkBf16, gm, 0, wg);
        }
    }
    // the solves' diagonal-block inverses and couplings
    std::vector<std::pair<TrinvBA, long long>> tl, tu;
    std::vector<std::pair<CouplingBA, long long>> cl, cu;
    for (auto &m : mats) {
        const int nb = (m.n + kIB - 1) / kIB;
        const size_t bsz = (size_t)nb * kIB * kIB;
        tl.push_back({TrinvBA{m.A, m.lda, m.n, m.dinv}, nb});
        tu.push_back({TrinvBA{m.A, m.lda, m.n, m.dinv + bsz}, nb});
        cl.push_back({CouplingBA{m.A, m.lda, m.n, nb, m.dinv, m.dinv + 2 * bsz}, (long long)nb * (kIB / 16)});
        cu.push_back({CouplingBA{m.A, m.lda, m.n, nb, m.dinv + bsz, m.dinv + 3 * bsz}, (long long)nb * (kIB / 16)});
    }
    P.add(kBkTrinvL, tl);
    P.add(kBkTrinvU, tu);
    P.add(kBkCoupleL, cl);
    P.add(kBkCoupleU, cu);
}

const char *batch_kernel_name(int kind)
{
    switch (kind) {
    case kBkLoad: return "k_tslu_load";
    case kBkPanel: return "k_tslu_panel";
    case kBkApply: return "k_tslu_apply";
    case kBkSwap: return "k_swap_plan";
    case kBkLaswp: return "k_laswp";
    case kBkTrinvL:
    case kBkTrinvU: return "k_trinv";
    case kBkToE: return "k_inv_to_e";
    case kBkCgemm: return "k_cgemm";
    case kBkSplitRows:
    case kBkSplitCols: return "k_split";
    case kBkBf16: return "k_cgemm_bf16x3";
    default: return "k_blk_coupling";
    }
}

void run_plan(Ctx &ctx, const BatchPlan &P, const char *dtab)
{
    hipStream_t s = ctx.stream;
    for (const auto &L : P.launches) {
        const unsigned g = (unsigned)L.blocks;
        const int *first = (const int *)(dtab + L.first);
        const void *a = dtab + L.args;
        ProfScope prof(ctx, batch_kernel_name(L.kind), L.work, s);
        switch (L.kind) {
        case kBkLoad: k_tslu_load_batch<<<g, 256, 0, s>>>((const LoadBA *)a, first, L.count); break;
        case kBkPanel: k_tslu_panel_batch<<<g, kTsluT, 0, s>>>((const PanelBA *)a, first, L.count); break;
        case kBkApply: k_tslu_apply_batch<<<g, 256, 0, s>>>((const TsluApply *)a, first, L.count); break;
        case kBkSwap: k_swap_plan_batch<<<g, 256, 0, s>>>((const SwapBA *)a, first, L.count); break;
        case kBkLaswp: k_laswp_apply_batch<<<g, 256, L.shm, s>>>((const LaswpBA *)a, first, L.count); break;
        case kBkTrinvL:
            k_trinv_batch<true><<<g, kIB * kTrinvParts, 0, s>>>((const TrinvBA *)a, first, L.count);
            break;
        case kBkTrinvU:
            k_trinv_batch<false><<<g, kIB * kTrinvParts, 0, s>>>((const TrinvBA *)a, first, L.count);
            break;
        case kBkToE: k_inv_to_e_batch<<<g, 256, 0, s>>>((const ToEBA *)a, first, L.count); break;
        case kBkCgemm: k_cgemm_batch<<<g, 256, 0, s>>>((const CgemmBA *)a, first, L.count); break;
        case kBkSplitRows: k_split_rows_batch<<<g, 256, 0, s>>>((const SplitRowsBA *)a, first, L.count); break;
        case kBkSplitCols: k_split_cols_batch<<<g, 256, 0, s>>>((const SplitColsBA *)a, first, L.count); break;
        case kBkBf16: k_cgemm_bf16x3_batch<<<g, 512, 0, s>>>((const Bf16BA *)a, first, L.count); break;
        case kBkCoupleL:
            k_blk_coupling_batch<true><<<g, 256, 0, s>>>((const CouplingBA *)a, first, L.count);
            break;
        case kBkCoupleU:
            k_blk_coupling_batch<false><<<g, 256, 0, s>>>((const CouplingBA *)a, first, L.count);
            break;
        default: BH_FAIL(BH_ERR_INVALID, "unknown batched launch %d", L.kind);
        }
        check(batch_kernel_name(L.kind));
    }
}

}  // namespace

}  // namespace bh

using namespace bh;

namespace {

// FP32 factorisation inputs: the matrix rounded to FP32 in lu32 (unless the assembly wrote
// it there) and the buffer of the solves' diagonal-block inverses.
void fp32_prepare(Ctx &ctx, bh_matrix *M, long long lda)
{
    const int64_t n = M->n;
    pool_release(ctx, M->lu64);
    if (M->lu32.n != (size_t)lda * n * 2) {
        pool_alloc(ctx, M->lu32, (size_t)lda * n * 2);
        M->lu32_fresh = false;
    }
    if (!M->lu32_fresh) {
        const unsigned cgrid = (unsigned)(((long long)n * n + 255) / 256);
        k_to_work<float><<<cgrid, 256, 0, ctx.stream>>>((const double2 *)M->a64.p, (int)n, (float2 *)M->lu32.p, lda);
        check("k_to_work");
    }
    M->lu32_fresh = false;   // it now holds the factors
    const size_t nb = (size_t)(n + kIB - 1) / kIB;
    pool_alloc(ctx, M->dinv32, 4 * nb * kIB * kIB * 2);   // L and U diagonal inverses, then their couplings
}

// After a factorisation: the FP32 solves' vector and block flags (so that solving
// allocates nothing), the permutation (P b)[i] = b[perm[i]] from the sequential
// interchanges, and the matrix state.
void factor_finish(Ctx &ctx, bh_matrix *M, long long lda, int precision, int info)
{
    const int64_t n = M->n;
    if (precision != BH_FP64 && M->x32.n < (size_t)n * kMaxRhs * 2) M->x32.alloc((size_t)n * kMaxRhs * 2);
    if (M->tsync.n < trsv_words(n, precision == BH_FP64)) {
        pool_alloc(ctx, M->tsync, trsv_words(n, precision == BH_FP64));
        trsv_restart(ctx.stream, M);
    }
    std::vector<long long> ip(n);
    BH_CHECK_HIP(hipMemcpy(ip.data(), M->ipiv.p, sizeof(long long) * n, hipMemcpyDeviceToHost));
    std::vector<int> perm(n);
    for (int64_t i = 0; i < n; ++i) perm[i] = (int)i;
    for (int64_t i = 0; i < n; ++i) std::swap(perm[i], perm[ip[i]]);
    M->perm.upload(perm.data(), n, ctx.stream);
    BH_CHECK_HIP(hipStreamSynchronize(ctx.stream));
    M->lda = lda;
    M->factored = info ? -1 : (precision == BH_FP64 ? BH_FP64 : BH_FP32);
}

}  // namespace

extern "C" int bh_matrix_factor(bh_matrix *M, int precision)
{
    BH_API_BEGIN
    BH_REQUIRE(M != nullptr, "NULL matrix");
    BH_REQUIRE(precision == BH_FP64 || precision == BH_FP32 || precision == BH_FP32_SPLIT,
               "precision must be BH_FP64, BH_FP32 or BH_FP32_SPLIT");
    std::lock_guard<std::mutex> lock(M->mu);
    Ctx &ctx = *M->ctx;
    const int64_t n = M->n;
    BH_REQUIRE(n > 0 && n < (int64_t(1) << 31), "bad matrix size");
    const long long lda = padded_ld(n);
    M->ipiv.alloc(n);
    hipEvent_t e0, e1;
    BH_CHECK_HIP(hipEventCreate(&e0));
    BH_CHECK_HIP(hipEventCreate(&e1));
    int info = 0;
    BH_CHECK_HIP(hipEventRecord(e0, ctx.stream));
    if (precision == BH_FP64) {
        pool_release(ctx, M->lu32);
        M->lu32_fresh = false;
        pool_release(ctx, M->dinv32);
        pool_alloc(ctx, M->lu64, (size_t)lda * n * 2);
        const unsigned cgrid = (unsigned)(((long long)n * n + 255) / 256);
        k_to_work<double><<<cgrid, 256, 0, ctx.stream>>>((const double2 *)M->a64.p, (int)n, (double2 *)M->lu64.p, lda);
        check("k_to_work");
        M->factored = -1;
        lu_factor<double>(ctx, (double2 *)M->lu64.p, lda, (int)n, M->ipiv.p, &info);
    } else {
        fp32_prepare(ctx, M, lda);
        M->factored = -1;
        lu_factor<float>(ctx, (float2 *)M->lu32.p, lda, (int)n, M->ipiv.p, &info, precision == BH_FP32_SPLIT,
                         (float2 *)M->dinv32.p);
    }
    BH_CHECK_HIP(hipEventRecord(e1, ctx.stream));
    BH_CHECK_HIP(hipEventSynchronize(e1));
    float ms = 0;
    BH_CHECK_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    M->seconds_factor = ms * 1e-3;
    factor_finish(ctx, M, lda, precision, info);
    if (info) BH_FAIL(BH_ERR_SINGULAR, "SingularException(%d): exactly zero pivot", info);
    BH_API_END
}

extern "C" int bh_matrix_factor_batch(bh_ctx *ctxh, int64_t count, bh_matrix *const *mats, int precision)
{
    BH_API_BEGIN
    BH_REQUIRE(ctxh != nullptr && (count == 0 || mats != nullptr), "NULL argument");
    BH_REQUIRE(count >= 0 && count <= (1 << 20), "bad batch size %lld", (long long)count);
    BH_REQUIRE(precision == BH_FP64 || precision == BH_FP32 || precision == BH_FP32_SPLIT,
               "precision must be BH_FP64, BH_FP32 or BH_FP32_SPLIT");
    Ctx &ctx = *ctxh;
    for (int64_t i = 0; i < count; ++i) {
        BH_REQUIRE(mats[i] != nullptr, "NULL matrix %lld", (long long)i);
        BH_REQUIRE(mats[i]->ctx == &ctx, "matrix %lld belongs to another context", (long long)i);
        BH_REQUIRE(mats[i]->n > 0 && mats[i]->n < (int64_t(1) << 31), "bad matrix size");
        for (int64_t j = 0; j < i; ++j) BH_REQUIRE(mats[j] != mats[i], "matrix %lld appears twice", (long long)i);
    }
    // the shared schedule takes FP32 split-bf16 factorisations of up to kBatchMaxN rows;
    // the others are factored one by one, as bh_matrix_factor does
    std::vector<bh_matrix *> shared, alone;
    for (int64_t i = 0; i < count; ++i)
        (precision == BH_FP32_SPLIT && mats[i]->n <= kBatchMaxN ? shared : alone).push_back(mats[i]);
    int first_error = BH_OK;
    std::string first_msg;
    for (bh_matrix *M : alone) {
        const int rc = bh_matrix_factor(M, precision);
        if (rc != BH_OK && first_error == BH_OK) {
            first_error = rc;
            first_msg = bh_last_error();
        }
    }
    if (!shared.empty()) {
        std::vector<std::unique_lock<std::mutex>> locks;
        for (bh_matrix *M : shared) locks.emplace_back(M->mu);
        // workspace of each matrix, one allocation: counters, info and candidate words first
        // (cleared together)
        std::vector<BatchMat> bm(shared.size());
        size_t ints = 0, rest = 0;
        auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
        std::vector<size_t> sets(shared.size());
        for (size_t i = 0; i < shared.size(); ++i) {
            const int n = (int)shared[i]->n;
            sets[i] = tslu_sets(n);
            ints += al((sets[i] + 1) * sizeof(int)) + al(sets[i] * kPW * sizeof(unsigned long long));
            const size_t trail = n > kNBInner ? (size_t)(n - kNBInner) : 0;
            rest += al(2 * kPW * sizeof(int)) + al(4 * kMaxSwaps * sizeof(int)) + al((size_t)2 * n * kPW * sizeof(float2)) +
                    2 * al(kPW * kPW * sizeof(float2)) + al((size_t)(kNBInner / kIB) * kIB * kIB * sizeof(float2)) +
                    2 * al(4 * trail * kNBInner * sizeof(__bf16));
        }
        DevBuf<char> ws;
        ws.alloc(ints + rest);
        k_fill_int<<<(unsigned)((ints / sizeof(int) + 255) / 256), 256, 0, ctx.stream>>>((int *)ws.p,
                                                                                        (long long)(ints / sizeof(int)));
        check("k_fill_int");
        size_t oi = 0, orest = ints;
        auto take = [&](size_t &off, size_t bytes) {
            char *p = ws.p + off;
            off += al(bytes);
            return p;
        };
        hipEvent_t e0, e1;
        BH_CHECK_HIP(hipEventCreate(&e0));
        BH_CHECK_HIP(hipEventCreate(&e1));
        BH_CHECK_HIP(hipEventRecord(e0, ctx.stream));
        for (size_t i = 0; i < shared.size(); ++i) {
            bh_matrix *M = shared[i];
            const int n = (int)M->n;
            const long long lda = padded_ld(n);
            M->ipiv.alloc(n);
            fp32_prepare(ctx, M, lda);
            BatchMat &b = bm[i];
            b.M = M;
            b.n = n;
            b.lda = lda;
            b.A = (float2 *)M->lu32.p;
            b.ipiv = M->ipiv.p;
            b.dinv = (float2 *)M->dinv32.p;
            b.tcnt = (int *)take(oi, (sets[i] + 1) * sizeof(int));
            b.info = b.tcnt + sets[i];
            b.tidx = (unsigned long long *)take(oi, sets[i] * kPW * sizeof(unsigned long long));
            const size_t trail = n > kNBInner ? (size_t)(n - kNBInner) : 0;
            b.moves = (int *)take(orest, 2 * kPW * sizeof(int));
            b.plan = (int *)take(orest, 4 * kMaxSwaps * sizeof(int));
            b.tpan = (float2 *)take(orest, (size_t)2 * n * kPW * sizeof(float2));
            b.top = (float2 *)take(orest, kPW * kPW * sizeof(float2));
            b.unext = (float2 *)take(orest, kPW * kPW * sizeof(float2));
            b.eblk = (float2 *)take(orest, (size_t)(kNBInner / kIB) * kIB * kIB * sizeof(float2));
            b.pa = (__bf16 *)take(orest, 4 * trail * kNBInner * sizeof(__bf16));
            b.pb = (__bf16 *)take(orest, 4 * trail * kNBInner * sizeof(__bf16));
        }
        BatchPlan plan;
        plan_factor(plan, bm);
        DevBuf<char> tab;
        tab.alloc(std::max<size_t>(plan.blob.size(), 16));
        struct SyncOnExit {   // no workspace is freed under running kernels, also on errors
            hipStream_t s;
            ~SyncOnExit() { (void)hipStreamSynchronize(s); }
        } sync_on_exit{ctx.stream};
        BH_CHECK_HIP(hipMemcpyAsync(tab.p, plan.blob.data(), plan.blob.size(), hipMemcpyHostToDevice, ctx.stream));
        run_plan(ctx, plan, tab.p);
        BH_CHECK_HIP(hipEventRecord(e1, ctx.stream));
        std::vector<int> infos(shared.size());
        for (size_t i = 0; i < shared.size(); ++i)
            BH_CHECK_HIP(hipMemcpyAsync(&infos[i], bm[i].info, sizeof(int), hipMemcpyDeviceToHost, ctx.stream));
        BH_CHECK_HIP(hipStreamSynchronize(ctx.stream));
        float ms = 0;
        BH_CHECK_HIP(hipEventElapsedTime(&ms, e0, e1));
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        for (size_t i = 0; i < shared.size(); ++i) {
            bh_matrix *M = shared[i];
            M->seconds_factor = ms * 1e-3;   // the whole batch's factorisation time
            factor_finish(ctx, M, bm[i].lda, precision, infos[i]);
            if (infos[i] && first_error == BH_OK) {
                first_error = BH_ERR_SINGULAR;
                char buf[160];
                std::snprintf(buf, sizeof buf, "SingularException(%d): exactly zero pivot (batch matrix of n = %lld)",
                              infos[i], (long long)M->n);
                first_msg = buf;
            }
        }
    }
    if (first_error != BH_OK) BH_FAIL(first_error, "%s", first_msg.c_str());
    BH_API_END
}

namespace {

// Z x = b with the factors: X (device, n x nrhs row-major, FP64) from B (same layout)
void apply_factors(bh_matrix *M, const double2 *B, double2 *Xd, int nrhs)
{
    hipStream_t s = M->ctx->stream;
    const int n = (int)M->n;
    const long long cnt = (long long)n * nrhs;
    const unsigned g = (unsigned)((cnt + 255) / 256);
    if (M->factored == BH_FP64) {
        k_permute_in<double><<<g, 256, 0, s>>>(B, n, nrhs, M->perm.p, Xd);
        check("k_permute_in");
        ProfScope prof(*M->ctx, "k_trsv64", 16.0 * n * (double)n);   // one read of both factors
        lu_solve<double>(s, M, Xd, nrhs);
    } else {
        float2 *x32 = (float2 *)M->x32.p;
        k_permute_in<float><<<g, 256, 0, s>>>(B, n, nrhs, M->perm.p, x32);
        check("k_permute_in");
        {
            ProfScope prof(*M->ctx, "k_trsv_inv", 8.0 * n * (double)n);   // one read of both FP32 factors
            lu_solve<float>(s, M, x32, nrhs);
        }
        k_widen<float><<<g, 256, 0, s>>>(x32, cnt, Xd);
        check("k_widen");
    }
}

double host_norm(const std::vector<double2> &v, int n, int nrhs, int q)
{
    double s = 0;
    for (int i = 0; i < n; ++i) s += v[(size_t)i * nrhs + q].x * v[(size_t)i * nrhs + q].x +
                                    v[(size_t)i * nrhs + q].y * v[(size_t)i * nrhs + q].y;
    return std::sqrt(s);
}

constexpr int kGmresRestart = 30;

struct GmresWork {
    double2 *Vb, *Zb, *w, *r, *part, *hd;
};

__global__ void k_zero(double2 *x, long long cnt)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) x[i] = double2{0.0, 0.0};
}

// GMRES on A D = R0 for the q columns of R0 (row-major n x q) at once: one right-
// preconditioned flexible GMRES per column (A M^-1 u = r0, d = M^-1 u, with the
// preconditioned basis Z_k = M^-1 V_k kept, so d = Z y needs no further solve), FP64
// vectors and matrix products, classical Gram-Schmidt applied twice, Givens rotations,
// restarts from the recomputed true residual.  The columns share every launch (the
// factors and A are read once per step for all of them); each column's arithmetic is that
// of its own GMRES.  Column c stops at ||r0_c - A d_c|| <= atol[c] (a column starting
// there does no step) or after maxinner steps.  Returns the steps summed over the columns.
// Device workspace (restart r): Vb (r + 1) n q, Zb r n q, w n q, r n q, part 256 (r + 1) q,
// hd (r + 1) q complex doubles.
int gmres_block(bh_matrix *M, const double2 *R0, int q, const double *r0norm, double2 *D, const double *atol,
                int restart, int maxinner, const GmresWork &G)
{
    using C = std::complex<double>;
    hipStream_t s = M->ctx->stream;
    const int n = (int)M->n;
    const long long nq = (long long)n * q;
    const unsigned gq = (unsigned)((nq + 255) / 256);
    double2 *const Vb = G.Vb, *const Zb = G.Zb, *const w = G.w, *const r = G.r, *const part = G.part,
                   *const hd = G.hd;
    std::vector<double2> hp((size_t)256 * (restart + 1) * q);
    auto sum_cols = [&](int m, int j, int c) {   // sum of the 256 block partials of (j, c)
        double ax = 0, ay = 0;
        for (int b = 0; b < 256; ++b) {
            const double2 v = hp[((size_t)b * m + j) * q + c];
            ax += v.x;
            ay += v.y;
        }
        return C(ax, ay);
    };
    k_zero<<<gq, 256, 0, s>>>(D, nq);
    check("k_zero");
    std::vector<double> beta(r0norm, r0norm + q);
    std::vector<int> total(q, 0);
    std::vector<char> live(q);
    for (int c = 0; c < q; ++c) live[c] = beta[c] > atol[c];
    const double2 *rcur = R0;
    for (;;) {
        bool any = false;
        for (int c = 0; c < q; ++c) {
            if (live[c] && total[c] >= maxinner) live[c] = 0;
            any = any || live[c];
        }
        if (!any) break;
        ColScale sc{};
        for (int c = 0; c < q; ++c) sc.s[c] = live[c] ? 1.0 / beta[c] : 0.0;
        k_scale_cols<<<gq, 256, 0, s>>>(rcur, n, q, sc, Vb);
        check("k_scale_cols");
        std::vector<std::vector<C>> H(q, std::vector<C>((size_t)(restart + 1) * restart, 0.0)), cs(q, std::vector<C>(restart)),
            sn(q, std::vector<C>(restart)), gvec(q, std::vector<C>(restart + 1, 0.0));
        std::vector<int> kc(q, 0);          // steps of this cycle per column
        std::vector<char> run(live);        // columns still stepping in this cycle
        std::vector<char> conv(q, 0);
        for (int c = 0; c < q; ++c) gvec[c][0] = beta[c];
        for (int k = 0; k < restart; ++k) {
            bool stepping = false;
            for (int c = 0; c < q; ++c) stepping = stepping || run[c];
            if (!stepping) break;
            double2 *zk = Zb + (size_t)k * nq;
            apply_factors(M, Vb + (size_t)k * nq, zk, q);
            {
                ProfScope prof(*M->ctx, "k_matvec", 16.0 * n * (double)n);
                apply_a<false>(s, (const double2 *)M->a64.p, n, zk, nullptr, w, q);
            }
            check("k_matvec");
            // both passes and the norm without the host in between (three synchronisations a step took
            // 0.1 ms: batch of 16 problems 77.9 -> 76.3 ms); the sums lie behind the block
            // parts, which take at most `restart` of the restart + 1 places of part
            unsigned mask = 0;
            for (int c = 0; c < q; ++c) mask |= run[c] ? 1u << c : 0u;
            double2 *const hs = part + (size_t)256 * restart * q;
            static_assert(2 * kGmresRestart + 1 <= 256, "the sums fit one place of part");
            for (int pass = 0; pass < 2; ++pass) {
                double2 *const hp_ = hs + (size_t)pass * restart * q;
                k_dots_cols<<<256, 256, 0, s>>>(Vb, n, k + 1, q, w, part);
                check("k_dots");
                k_sum_parts<<<(k + 1) * q, 64, 0, s>>>(part, k + 1, q, mask, hp_);
                check("k_sum_parts");
                k_axpys_cols<<<gq, 256, 0, s>>>(Vb, n, k + 1, q, hp_, w);
                check("k_axpys");
            }
            k_dots_cols<<<256, 256, 0, s>>>(w, n, 1, q, w, part);
            check("k_dots");
            k_sum_parts<<<q, 64, 0, s>>>(part, 1, q, mask, hs + (size_t)2 * restart * q);
            check("k_sum_parts");
            BH_CHECK_HIP(hipMemcpyAsync(hp.data(), hs, sizeof(double2) * (2 * restart + 1) * q, hipMemcpyDeviceToHost, s));
            BH_CHECK_HIP(hipStreamSynchronize(s));
            auto sum_at = [&](int i, int c) { return C(hp[(size_t)i * q + c].x, hp[(size_t)i * q + c].y); };
            std::vector<std::vector<C>> h(q, std::vector<C>(k + 1, 0.0));
            for (int c = 0; c < q; ++c)
                for (int j = 0; j <= k; ++j) h[c][j] = sum_at(j, c) + sum_at(restart + j, c);
            ColScale nx{};
            for (int c = 0; c < q; ++c) {
                if (!run[c]) continue;
                const double hn = std::sqrt(std::max(0.0, sum_at(2 * restart, c).real()));
                auto &Hc = H[c];
                for (int j = 0; j <= k; ++j) Hc[(size_t)j * restart + k] = h[c][j];
                Hc[(size_t)(k + 1) * restart + k] = hn;
                for (int j = 0; j < k; ++j) {
                    const C x = Hc[(size_t)j * restart + k], y = Hc[(size_t)(j + 1) * restart + k];
                    Hc[(size_t)j * restart + k] = std::conj(cs[c][j]) * x + std::conj(sn[c][j]) * y;
                    Hc[(size_t)(j + 1) * restart + k] = -sn[c][j] * x + cs[c][j] * y;
                }
                const C x = Hc[(size_t)k * restart + k], y = Hc[(size_t)(k + 1) * restart + k];
                const double den = std::sqrt(std::norm(x) + std::norm(y));
                cs[c][k] = den == 0 ? C(1.0) : x / den;
                sn[c][k] = den == 0 ? C(0.0) : y / den;
                Hc[(size_t)k * restart + k] = den;
                Hc[(size_t)(k + 1) * restart + k] = 0.0;
                gvec[c][k + 1] = -sn[c][k] * gvec[c][k];
                gvec[c][k] = std::conj(cs[c][k]) * gvec[c][k];
                kc[c] = k + 1;
                ++total[c];
                if (std::abs(gvec[c][k + 1]) <= atol[c] || hn == 0) {
                    conv[c] = 1;
                    run[c] = 0;
                } else if (total[c] >= maxinner) {
                    run[c] = 0;
                } else {
                    nx.s[c] = 1.0 / hn;
                }
            }
            if (k + 1 < restart) {
                k_scale_cols<<<gq, 256, 0, s>>>(w, n, q, nx, Vb + (size_t)(k + 1) * nq);
                check("k_scale_cols");
            }
        }
        // D[:, c] += Z y_c with H_c y_c = g_c (upper triangular kc x kc)
        int kmax = 0;
        for (int c = 0; c < q; ++c) kmax = std::max(kmax, kc[c]);
        if (kmax > 0) {
            std::vector<double2> yn((size_t)kmax * q, double2{0, 0});
            for (int c = 0; c < q; ++c) {
                const int k = kc[c];
                const auto &Hc = H[c];
                std::vector<C> y(k, 0.0);
                for (int i = k - 1; i >= 0; --i) {
                    C t = gvec[c][i];
                    for (int j = i + 1; j < k; ++j) t -= Hc[(size_t)i * restart + j] * y[j];
                    y[i] = Hc[(size_t)i * restart + i] == 0.0 ? C(0.0) : t / Hc[(size_t)i * restart + i];
                }
                for (int j = 0; j < k; ++j) yn[(size_t)j * q + c] = {-y[j].real(), -y[j].imag()};
            }
            BH_CHECK_HIP(hipMemcpyAsync(hd, yn.data(), sizeof(double2) * kmax * q, hipMemcpyHostToDevice, s));
            k_axpys_cols<<<gq, 256, 0, s>>>(Zb, n, kmax, q, hd, D);
            check("k_axpys");
        }
        bool again = false;
        for (int c = 0; c < q; ++c) {
            if (conv[c]) live[c] = 0;
            if (live[c] && total[c] >= maxinner) live[c] = 0;
            again = again || live[c];
        }
        if (!again) break;
        // restart from the true residuals R0 - A D
        {
            ProfScope prof(*M->ctx, "k_residual", 16.0 * n * (double)n);
            apply_a<true>(s, (const double2 *)M->a64.p, n, D, R0, r, q);
        }
        check("k_residual");
        k_dots_cols<<<256, 256, 0, s>>>(r, n, 1, q, r, part);
        check("k_dots");
        BH_CHECK_HIP(hipMemcpyAsync(hp.data(), part, sizeof(double2) * 256 * q, hipMemcpyDeviceToHost, s));
        BH_CHECK_HIP(hipStreamSynchronize(s));
        for (int c = 0; c < q; ++c) {
            beta[c] = std::sqrt(std::max(0.0, sum_cols(1, 0, c).real()));
            if (live[c] && beta[c] <= atol[c]) live[c] = 0;
        }
        rcur = r;
    }
    BH_CHECK_HIP(hipStreamSynchronize(s));
    int sum = 0;
    for (int c = 0; c < q; ++c) sum += total[c];
    return sum;
}

}  // namespace

namespace {

// Device workspace of one solve: db, dx, dr (n x nrhs each), rcol, dcol (n each) and the
// GMRES workspace, each piece 256-byte aligned inside one buffer.
// x += d elementwise
__global__ void k_add_to(double2 *__restrict__ x, long long cnt, const double2 *__restrict__ d)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) {
        x[i].x += d[i].x;
        x[i].y += d[i].y;
    }
}

struct SolveWork {
    double2 *db, *dx, *dr, *dd;
    GmresWork g;
};

size_t solve_work_layout(int n, int nrhs, char *base, SolveWork *W)
{
    size_t off = 0;
    auto take = [&](size_t count) {
        double2 *p = base ? (double2 *)(base + off) : nullptr;
        off += (count * sizeof(double2) + 255) & ~(size_t)255;
        return p;
    };
    const size_t nq = (size_t)n * nrhs, r = kGmresRestart;
    SolveWork w{};
    w.db = take(nq);
    w.dx = take(nq);
    w.dr = take(nq);
    w.dd = take(nq);
    w.g.Vb = take((r + 1) * nq);
    w.g.Zb = take(r * nq);
    w.g.w = take(nq);
    w.g.r = take(nq);
    w.g.part = take(256 * (r + 1) * (size_t)nrhs);
    w.g.hd = take((r + 1) * (size_t)nrhs);
    if (W) *W = w;
    return off;
}

// X = Z \ B with the factors of M (see bh_matrix_solve); W the device workspace.  With
// timed = false no HIP events are created (stats->seconds_solve is then host wall time).
void solve_impl(bh_matrix *M, int64_t nrhs, const double *B, double *X, double tol, int maxit,
                bh_solve_stats *stats, const SolveWork &W, bool timed)
{
    hipStream_t s = M->ctx->stream;
    const int n = (int)M->n, q = (int)nrhs;
    const long long cnt = (long long)n * q;
    // host column-major -> device row-major n x nrhs
    std::vector<double2> hb(cnt), hx(cnt);
    for (int r = 0; r < q; ++r)
        for (int i = 0; i < n; ++i) hb[(size_t)i * q + r] = {B[2 * ((size_t)r * n + i)], B[2 * ((size_t)r * n + i) + 1]};
    BH_CHECK_HIP(hipMemcpyAsync(W.db, hb.data(), sizeof(double2) * cnt, hipMemcpyHostToDevice, s));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    const auto h0 = std::chrono::steady_clock::now();
    if (timed) {
        BH_CHECK_HIP(hipEventCreate(&e0));
        BH_CHECK_HIP(hipEventCreate(&e1));
        BH_CHECK_HIP(hipEventRecord(e0, s));
    }
    apply_factors(M, W.db, W.dx, q);
    int iters = 0, inner = 0;
    double res = 0;
    std::vector<double> bn(q);
    for (int r = 0; r < q; ++r) bn[r] = host_norm(hb, n, q, r);
    // the triangular solves report a block wait that gave up in the error word; it is
    // read (and cleared) after every synchronisation that ends a use of the solves,
    // before anything derived from their results is judged
    auto check_trsv = [&]() {
        int trsv_err = 0;
        BH_CHECK_HIP(hipMemcpyAsync(&trsv_err, (int *)M->tsync.p + 1, sizeof(int), hipMemcpyDeviceToHost, s));
        BH_CHECK_HIP(hipStreamSynchronize(s));
        if (!trsv_err) return;
        // results are void; the counters restart
        trsv_restart(s, M);
        BH_CHECK_HIP(hipStreamSynchronize(s));
        BH_FAIL(BH_ERR_HIP, "triangular solve: a block wait exceeded its limit");
    };
    const bool refine = M->factored == BH_FP32 || tol > 0;
    if (refine) {
        const int maxit_ = maxit > 0 ? maxit : 20;
        for (;;) {
            {
                ProfScope prof(*M->ctx, "k_residual", 16.0 * n * (double)n);   // one FP64 read of A
                apply_a<true>(s, (const double2 *)M->a64.p, n, W.dx, W.db, W.dr, q);
            }
            check("k_residual");
            // the norms are taken on the device (the residuals themselves, 768 KB at 12,000
            // unknowns and four columns, and the host's sums took 0.2 ms each time)
            k_dots_cols<<<256, 256, 0, s>>>(W.dr, n, 1, q, W.dr, W.g.part);
            check("k_dots");
            std::vector<double2> hp((size_t)256 * q);
            BH_CHECK_HIP(hipMemcpyAsync(hp.data(), W.g.part, sizeof(double2) * hp.size(), hipMemcpyDeviceToHost, s));
            check_trsv();   // after a synchronisation
            res = 0;
            std::vector<double> rel(q);
            for (int r = 0; r < q; ++r) {
                double sum = 0;
                for (int k = 0; k < 256; ++k) sum += hp[(size_t)k * q + r].x;
                rel[r] = bn[r] > 0 ? std::sqrt(sum) / bn[r] : 0.0;
                if (!std::isfinite(rel[r])) BH_FAIL(BH_ERR_NOCONV, "refinement produced a non-finite residual");
                res = std::max(res, rel[r]);
            }
            const double target = tol > 0 ? tol : 1e-12;
            if (res <= target || iters >= maxit_) break;
            ++iters;
            // solve A D = R for the columns above the target, each to 1/2 of its remaining
            // target, then X += D (columns already there have D = 0)
            std::vector<double> rn(q), atol(q);
            for (int r = 0; r < q; ++r) {
                rn[r] = rel[r] * bn[r];
                atol[r] = rel[r] <= target ? std::numeric_limits<double>::infinity() : 0.5 * target * bn[r];
            }
            inner += gmres_block(M, W.dr, q, rn.data(), W.dd, atol.data(), kGmresRestart, 200, W.g);
            k_add_to<<<(unsigned)((cnt + 255) / 256), 256, 0, s>>>(W.dx, cnt, W.dd);
            check("k_add_to");
        }
    }
    float ms = 0;
    if (timed) {
        BH_CHECK_HIP(hipEventRecord(e1, s));
        BH_CHECK_HIP(hipEventSynchronize(e1));
        BH_CHECK_HIP(hipEventElapsedTime(&ms, e0, e1));
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
    }
    BH_CHECK_HIP(hipMemcpyAsync(hx.data(), W.dx, sizeof(double2) * cnt, hipMemcpyDeviceToHost, s));
    BH_CHECK_HIP(hipStreamSynchronize(s));
    check_trsv();
    if (!timed) ms = (float)(1e3 * std::chrono::duration<double>(std::chrono::steady_clock::now() - h0).count());
    for (int r = 0; r < q; ++r)
        for (int i = 0; i < n; ++i) {
            X[2 * ((size_t)r * n + i)] = hx[(size_t)i * q + r].x;
            X[2 * ((size_t)r * n + i) + 1] = hx[(size_t)i * q + r].y;
        }
    if (stats) {
        stats->iterations = iters;
        stats->inner = inner;
        stats->residual = res;
        stats->seconds_factor = M->seconds_factor;
        stats->seconds_solve = ms * 1e-3;
    }
    if (refine && tol > 0 && res > tol)
        BH_FAIL(BH_ERR_NOCONV, "refinement stopped at relative residual %.3e > %.3e after %d steps", res, tol, iters);
}

}  // namespace

extern "C" int bh_matrix_solve(bh_matrix *M, int64_t nrhs, const double *B, double *X, double tol, int maxit,
                               bh_solve_stats *stats)
{
    BH_API_BEGIN
    BH_REQUIRE(M && B && X, "NULL argument");
    BH_REQUIRE(M->factored == BH_FP64 || M->factored == BH_FP32, "matrix is not factored");
    BH_REQUIRE(nrhs >= 1 && nrhs <= 8, "nrhs must be 1..8");
    std::lock_guard<std::mutex> lock(M->mu);
    // from the pool, which keeps buffers of 1 MiB or more
    PoolBuf<char> work(*M->ctx, std::max(solve_work_layout((int)M->n, (int)nrhs, nullptr, nullptr), size_t(1) << 20));
    struct GiveBack {   // also when the refinement ends in an error, once the stream is done
        PoolBuf<char> &work;
        hipStream_t s;
        ~GiveBack() { if (hipStreamSynchronize(s) == hipSuccess) work.done(); }
    } give_back{work, M->ctx->stream};
    SolveWork W;
    solve_work_layout((int)M->n, (int)nrhs, work.p, &W);
    solve_impl(M, nrhs, B, X, tol, maxit, stats, W, true);
    BH_API_END
}

// ---------------------------------------------------------------- allocation-free solve
namespace {

// Scratch memory of bh_matrix_solve_noalloc: one copy per device, held until the process
// ends.  Host code never uses the array's name as an address: the device address comes from
// hipGetSymbolAddress, once per device, when a context is created there.
constexpr size_t kScratchBytes = size_t(64) << 20;
static __device__ __align__(256) char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

}  // namespace

namespace bh {
// Called by bh_ctx_create with the context's device current.
void scratch_register(int device)
{
    BH_REQUIRE(device >= 0 && device < kMaxDevices, "device %d beyond the scratch table", device);
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (g_scratch_ptr[device]) return;
    void *p = nullptr;
    BH_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    BH_REQUIRE(p != nullptr, "no device address for the solve scratch on device %d", device);
    g_scratch_ptr[device] = p;
}
}  // namespace bh

extern "C" int bh_matrix_solve_noalloc(bh_matrix *M, int64_t nrhs, const double *B, double *X, double tol,
                                       int maxit, bh_solve_stats *stats)
{
    BH_API_BEGIN
    BH_REQUIRE(M && B && X, "NULL argument");
    BH_REQUIRE(M->factored == BH_FP64 || M->factored == BH_FP32, "matrix is not factored");
    BH_REQUIRE(nrhs >= 1 && nrhs <= 8, "nrhs must be 1..8");
    // apply_factors allocates nothing: bh_matrix_factor has sized these buffers
    BH_REQUIRE((M->factored == BH_FP64 || M->x32.n >= (size_t)M->n * nrhs * 2) &&
                   M->tsync.n >= trsv_words(M->n, M->factored == BH_FP64),
               "factors without their solve buffers");
    const size_t need = solve_work_layout((int)M->n, (int)nrhs, nullptr, nullptr);
    BH_REQUIRE(need <= kScratchBytes,
               "bh_matrix_solve_noalloc: n = %lld with %lld right-hand sides needs %zu bytes of scratch, more than "
               "its %zu (use bh_matrix_solve)", (long long)M->n, (long long)nrhs, need, kScratchBytes);
    void *base = nullptr;
    {
        std::lock_guard<std::mutex> g(g_scratch_mu);
        base = (M->ctx->device >= 0 && M->ctx->device < kMaxDevices) ? g_scratch_ptr[M->ctx->device] : nullptr;
    }
    BH_REQUIRE(base != nullptr, "no solve scratch registered for device %d", M->ctx->device);
    std::lock_guard<std::mutex> lock(M->mu);
    SolveWork W;
    solve_work_layout((int)M->n, (int)nrhs, (char *)base, &W);
    solve_impl(M, nrhs, B, X, tol, maxit, stats, W, false);
    BH_API_END
}

extern "C" int bh_matrix_pivots(bh_matrix *M, int64_t *ipiv)
{
    BH_API_BEGIN
    BH_REQUIRE(M && ipiv, "NULL argument");
    BH_REQUIRE(M->factored >= 0, "matrix is not factored");
    std::vector<long long> ip(M->n);
    BH_CHECK_HIP(hipMemcpy(ip.data(), M->ipiv.p, sizeof(long long) * M->n, hipMemcpyDeviceToHost));
    for (int64_t i = 0; i < M->n; ++i) ipiv[i] = ip[i] + 1;
    BH_API_END
}
