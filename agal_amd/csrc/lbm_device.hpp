// lbm_device.hpp -- device code and launch arguments of a level's collide + boundary hook + stream
// sub-step, shared by the fused launch (lbm_kernels.hip) and the in-place one (lbm_inplace.hip).
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "agal_common.hpp"
#include "agal_ctx.hpp"

namespace agal {

constexpr int WG = 256;

// Moments in the reference's order (p-order sums, then division): Cu_RefreshVariables (:110-159).
// The reference adds c * f for every component, zeros included; those terms are left out here.
// A sum that starts at +0 never becomes -0 under round-to-nearest, so adding 0 * f = +-0 leaves
// it unchanged: for finite populations the results are the same bits, at about a third fewer
// vector instructions.
template <typename T, int Q>
__device__ __forceinline__ void moments(const T *f, T &rho, T &u, T &v, T &w)
{
    using VS = VelSet<Q>;
    rho = 0;
    u = 0;
    v = 0;
    w = 0;
#pragma unroll
    for (int p = 0; p < Q; p++) {
        rho += f[p];
        if (VS::cx(p) > 0) u += f[p];
        if (VS::cx(p) < 0) u -= f[p];
        if (VS::cy(p) > 0) v += f[p];
        if (VS::cy(p) < 0) v -= f[p];
        if (VS::DIM == 3 && VS::cz(p) > 0) w += f[p];
        if (VS::DIM == 3 && VS::cz(p) < 0) w -= f[p];
    }
    // One correctly rounded division, then products (the CPU restatement does the same).
    const T r = (T)(1.0) / rho;
    u = u * r;
    v = v * r;
    if (VS::DIM == 3) w = w * r;
}

// c_p . u in the reference's left-to-right order (cx u + cy v) + cz w, without the terms of zero
// components.  A nonzero sum is unchanged by them; a zero sum may differ in sign only, which the
// equilibrium polynomial 1 + 3 c.u + 4.5 (c.u)^2 does not see.
template <typename T, int Q>
__device__ __forceinline__ T cdot(int p, T u, T v, T w)
{
    using VS = VelSet<Q>;
    T s = (T)0;
    bool first = true;
    if (VS::cx(p) != 0) {
        s = VS::cx(p) > 0 ? u : -u;
        first = false;
    }
    if (VS::cy(p) != 0) {
        const T t = VS::cy(p) > 0 ? v : -v;
        s = first ? t : s + t;
        first = false;
    }
    if (VS::DIM == 3 && VS::cz(p) != 0) {
        const T t = VS::cz(p) > 0 ? w : -w;
        s = first ? t : s + t;
    }
    return s;
}

// ---------------------------------------------------------------------------------------------
// Fused collide + boundary hook + stream of one level sub-step.
// ---------------------------------------------------------------------------------------------
template <typename T, typename S>
struct StepArgs {
    const int *ids;
    int n;
    const S *A;
    S *B;
    long long ncm;
    const int *nbr_slot;   // per block, Q_max neighbour IDs in 3x3(x3) slot order
    const int *part;       // block collides and streams (not solid-with-children)
    const int *simple;     // block and its neighbourhood: all participate, no solid cells
    const int *cells_mask;
    const int *onb;
    T omeg, omegp, U;
    int mrt;      // collision operator: 0 BGK, 1 MRT
    T ck[27];     // MRT: rate_k / D_k per moment row (0 for conserved rows)
    int bc_preset;
    int *exc_idx;
    T *exc_val;
    int *exc_count;
    long long exc_cap;
    // Finest-level pairs (3D): vmode 1 -- the exception list (exc_*) is the extra list that the
    // next sub-step applies as it loads, and each block with an entry gets PEND_FLAG in flags;
    // vmode 2 -- apply that list (va_*) to the loaded values of flagged blocks; VMODE_EVEN -- the
    // first sub-step of an in-place pair (B == A); 0 -- neither.
    int vmode;
    int nt;  // VMODE_EVEN: non-temporal loads
    int skip_linked;  // a linked block's sub-step is k_link_step's
    int *flags;
    const int *va_idx;
    const T *va_val;
    const int *va_count;
    // The extra list linked per block: x_head[block] is the last node 2k + s of the block's chain
    // (entry k, s = 0 through its initiator cell, 1 through its partner cell), -1 when empty;
    // x_next[node] the node before it.  Built in vmode 1, walked and emptied in vmode 2.
    int *x_head;
    int *x_next;
};

constexpr int VMODE_EVEN = 3;

// The memory-side cache.  The first sub-step of an in-place pair reads with ordinary loads when the
// level's populations fit it (64^3 cavity with three levels, FP32: 288 us a coarse step, 333 with
// non-temporal ones), else with non-temporal loads (128^3, four levels: 11.5 ms a coarse step, 11.9 with
// ordinary ones).  Its stores are ordinary ones.
constexpr long long MALL_BYTES = 256LL << 20;

// Block flag bit: the block has entries in the finest level's extra exception list (bits 0-1 of
// the same word hold the simple / interior kind).
constexpr int PEND_FLAG = 4;

// Appends a guard exception (target cell, partner cell, direction, partner's stored value) to the
// launch's list; in vmode 1 also flags the two blocks for the next sub-step.
template <typename T, typename S>
__device__ __forceinline__ void record_exception(const StepArgs<T, S> &a, long long tgt, long long cell, int q, T fv)
{
    int k = atomicAdd(&a.exc_count[0], 1);
    if (k < a.exc_cap) {
        a.exc_idx[3 * (long long)k + 0] = (int)tgt;  // cell indices < 2^31
        a.exc_idx[3 * (long long)k + 1] = (int)cell;
        a.exc_idx[3 * (long long)k + 2] = q;
        a.exc_val[k] = fv;
    } else {
        a.exc_count[1] = 1;
    }
    if (a.vmode == 1) {
        const int bt = (int)(tgt >> 6), bc = (int)(cell >> 6);
        atomicOr(&a.flags[bt], PEND_FLAG);
        atomicOr(&a.flags[bc], PEND_FLAG);
        if (k < a.exc_cap) {
            a.x_next[2 * k] = atomicExch(&a.x_head[bt], 2 * k);
            if (bc != bt) a.x_next[2 * k + 1] = atomicExch(&a.x_head[bc], 2 * k + 1);
        }
    }
}

// Workgroup -> position in the level's block list.  Workgroups are dealt round-robin to the
// eight XCDs (each with its own L2); giving every XCD one contiguous range of the sorted ID list
// keeps a block and most of its neighbours -- whose pushes share cache lines -- on one L2.
__device__ __forceinline__ int xcd_local_wg(int nwg_padded)
{
    const int per = nwg_padded / 8;
    return (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
}

// The same for the first nwg_padded (a multiple of 8) workgroups of a larger grid.
__device__ __forceinline__ int xcd_local_wg(int wg, int nwg_padded)
{
    const int per = nwg_padded / 8;
    return (wg % 8) * per + wg / 8;
}

// Post-collision values f*_p of one cell.  BGK: Cu_Collide (solver_lbm_kernels.cu:275-282).  MRT:
// f* = f - M^T (ck .* (M (f - feq))), the transforms summed in ascending row / column order with
// zero entries and conserved rows left out (ck_k = rate_k / D_k).  Cells that do not collide
// (solid cells, blocks that are solid with children) keep their values: the swap semantics of the
// reference amount to f*_q = f_pb(q) for them.
// COLL: COLL_ARGS takes the operator from the arguments, COLL_BGK / COLL_MRT fix it (a kernel compiled
// for BGK alone keeps the registers that MRT's moments need).
constexpr int COLL_ARGS = 0, COLL_BGK = 1, COLL_MRT = 2, COLL_MFMA = 3;

// acc + m x, the product rounded before the sum.  A product by +-2^n is exact, and so is 2^n times the
// rounded 3 x for m = +-3 2^n: one multiply-add rounds those sums as the two operations would.  The MRT
// step is bound by its vector instructions; as two operations the multiples 2 x, 4 x, 8 x, 6 x of every x were
// also held in registers.  D3Q27 FP32: 96 registers and scratch -> 91 and none, the linked blocks' kernel
// 98 -> 86 (5 wavefronts per SIMD instead of 4); a 64^3 sphere with four levels 1.25 -> 1.19 ms per coarse step.
template <typename T>
__device__ __forceinline__ T add_multiple(int m, T x, T acc)
{
    const int n = m < 0 ? -m : m;
    if (n == 1) return m < 0 ? acc - x : acc + x;
    if ((n & (n - 1)) == 0) return fmadd((T)m, x, acc);
    if (n % 3 == 0 && ((n / 3) & (n / 3 - 1)) == 0) return fmadd((T)(m / 3), (T)3 * x, acc);
    return acc + (T)m * x;
}

template <typename T, typename S, int Q, int COLL = COLL_ARGS>
__device__ __forceinline__ void collide_cell(const StepArgs<T, S> &a, const T *f, T *fs, T rho, T u, T v, T w,
                                             bool inert)
{
    using VS = VelSet<Q>;
    if (inert) {
#pragma unroll
        for (int p = 0; p < Q; p++) fs[p] = f[VS::pb(p)];
        return;
    }
    const T udotu = u * u + v * v + w * w;
    if (COLL == COLL_BGK || (COLL == COLL_ARGS && !a.mrt)) {
        // BGK in fused multiply-adds, in the same order as the CPU restatement:
        //   b_p = (4.5 c.u) c.u + (1 - 1.5 u.u),  feq_p / (w_p rho) = 3 c.u + b_p,
        //   f*_p = (w_p rho omega) (feq_p / (w_p rho)) + (1 - omega) f_p.
        // A pair (p, pb(p)) shares |c.u|, b and the weight: c_pb.u = -(c_p.u) bit for bit (sums of
        // negated terms), so the pb direction takes -3 c.u.
        const T c1 = (T)(1.0) - (T)(1.5) * udotu;
        const T ro = rho * a.omeg;
        fs[0] = fmadd((T)VS::w(0) * ro, c1, f[0] * a.omegp);
#pragma unroll
        for (int p = 1; p < Q; p++) {
            if (!VS::half(p)) continue;
            const int q = VS::pb(p);
            const T cu = cdot<T, Q>(p, u, v, w);
            const T b = fmadd((T)(4.5) * cu, cu, c1);
            const T wro = (T)VS::w(p) * ro;
            fs[p] = fmadd(wro, fmadd((T)(3.0), cu, b), f[p] * a.omegp);
            fs[q] = fmadd(wro, fmadd((T)(-3.0), cu, b), f[q] * a.omegp);
        }
        return;
    }
    using MB = Mrt<Q>;
    // Full unrolling keeps d, r and the rates in registers (otherwise the FP64 D3Q27 variant indexes
    // them dynamically from scratch memory).
    T d[Q];
#pragma clang loop unroll(full)
    for (int p = 0; p < Q; p++) {
        T cdotu = cdot<T, Q>(p, u, v, w);
        d[p] = f[p] - (T)VS::w(p) * rho * ((T)(1.0) + (T)(3.0) * cdotu + (T)(4.5) * cdotu * cdotu - (T)(1.5) * udotu);
    }
    T r[Q];
#pragma clang loop unroll(full)
    for (int k = 0; k < Q; k++) {
        r[k] = (T)0;
        if (MB::rate(k) == 0) continue;
        T acc = (T)0;
        bool first = true;
#pragma clang loop unroll(full)
        for (int p = 0; p < Q; p++) {
            if (MB::m(k, p) == 0) continue;
            acc = first ? (T)MB::m(k, p) * d[p] : add_multiple(MB::m(k, p), d[p], acc);
            first = false;
        }
        r[k] = acc * a.ck[k];
    }
#pragma clang loop unroll(full)
    for (int p = 0; p < Q; p++) {
        T acc = (T)0;
        bool first = true;
#pragma clang loop unroll(full)
        for (int k = 0; k < Q; k++) {
            if (MB::rate(k) == 0 || MB::m(k, p) == 0) continue;
            acc = first ? (T)MB::m(k, p) * r[k] : add_multiple(MB::m(k, p), r[k], acc);
            first = false;
        }
        fs[p] = f[p] - acc;
    }
}

// MRT transform on matrix cores for one 3D block per wavefront (Q = 19, 27; FP32 compute):
// g = M^T (c . M d) for the non-equilibrium parts d of the 64 cells.  FP32 pools: d and c . M d are
// split into two bf16 terms each (hi + lo carry 16 significant bits; the products with the integer
// matrix are exact and the sums FP32), so the result agrees with the vector path to about 2^-17 of
// d, below the FP32 rounding of the populations themselves.  16-bit pools (F16): one binary16 term
// of 2^10 d and of 2^10 c . M d each (11 significant bits, the scale keeps small parts out of the
// subnormal range), products exact and sums FP32, on v_mfma_f32_16x16x32_f16: an error of about
// 2^-11 of the non-equilibrium part, below the binary16 rounding of the stored deviation f - w,
// which is larger than that part, and the correction goes back through LDS in binary16.  `lds` is
// this wavefront's region of 64 rows (36 floats; 80 bytes with 16-bit pools); only the wavefront
// itself touches it.
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4_t;

__constant__ const MfmaTab<19> kMfma19 = make_mfma_tab<19>();
__constant__ const MfmaTab<27> kMfma27 = make_mfma_tab<27>();

constexpr int MFMA_SPLITS = 2;

// Next bf16 term of `rem` (round to nearest even, the hardware conversion); rem keeps the rest.
__device__ __forceinline__ __bf16 split_term(float &rem)
{
    const __bf16 h = (__bf16)rem;
    rem -= (float)h;
    return h;
}

template <int Q, bool F16>
__device__ __forceinline__ void mrt_mfma(const float *d, float *g, const float *ckrow, float *lds)
{
    using VT = typename std::conditional<F16, f16x8_t, bf16x8_t>::type;
    constexpr int SPLITS = F16 ? 1 : MFMA_SPLITS;
    const MfmaTab<Q> &tab = *(Q == 19 ? reinterpret_cast<const MfmaTab<Q> *>(&kMfma19)
                                      : reinterpret_cast<const MfmaTab<Q> *>(&kMfma27));
    const int l = threadIdx.x & 63, q = l >> 4, j = l & 15;
    const u32x4_t *fw = reinterpret_cast<const u32x4_t *>(F16 ? &tab.fw16[l][0][0] : &tab.fw[l][0][0]);
    const u32x4_t *bk = reinterpret_cast<const u32x4_t *>(F16 ? &tab.bk16[l][0][0] : &tab.bk[l][0][0]);
    const VT afw0 = __builtin_bit_cast(VT, fw[0]), afw1 = __builtin_bit_cast(VT, fw[1]);
    const VT abk0 = __builtin_bit_cast(VT, bk[0]), abk1 = __builtin_bit_cast(VT, bk[1]);
    VT *ldsv = reinterpret_cast<VT *>(lds);  // rows of 5 vectors (80 bytes)
    auto mfma = [](const VT &a, const VT &b, const f32x4_t &c) {
        if constexpr (F16)
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    };
    auto term = [](float &rem) {
        if constexpr (F16) {
            return (_Float16)rem;
        } else {
            return split_term(rem);
        }
    };

    // Forward: one pass per term of d through a 64-row transpose region.
    f32x4_t C0[4], C1[4];
#pragma unroll
    for (int t = 0; t < 4; t++) C0[t] = C1[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float rem[32];
#pragma unroll
    for (int k = 0; k < 32; k++) rem[k] = k < Q ? d[k] : 0.f;
#pragma unroll
    for (int sp = 0; sp < SPLITS; sp++) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            VT v;
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = term(rem[8 * c + e]);
            ldsv[5 * l + c] = v;
        }
        wave_lds_sync();
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const VT b = ldsv[5 * (16 * t + j) + q];
            C0[t] = mfma(afw0, b, C0[t]);
            C1[t] = mfma(afw1, b, C1[t]);
        }
        wave_lds_sync();
    }
    // Relaxation factors rate / D of the rows this lane holds (rows 4q + r and 16 + 4q + r, zero
    // beyond the velocity set), picked from the level's row table by the lane's quarter q.
    float ck0[4], ck1[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        float a0[4], a1[4];
#pragma unroll
        for (int qq = 0; qq < 4; qq++) {
            a0[qq] = 4 * qq + r < Q ? ckrow[4 * qq + r] : 0.f;
            a1[qq] = 16 + 4 * qq + r < Q ? ckrow[16 + 4 * qq + r] : 0.f;
        }
        ck0[r] = q == 0 ? a0[0] : (q == 1 ? a0[1] : (q == 2 ? a0[2] : a0[3]));
        ck1[r] = q == 0 ? a1[0] : (q == 1 ? a1[1] : (q == 2 ? a1[2] : a1[3]));
    }
    // Back: B operand straight from the forward results of the same lane.
    f32x4_t G0[4], G1[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        G0[t] = G1[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        float v[8];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            v[r] = C0[t][r] * ck0[r];
            v[4 + r] = C1[t][r] * ck1[r];
        }
#pragma unroll
        for (int sp = 0; sp < SPLITS; sp++) {
            VT b;
#pragma unroll
            for (int e = 0; e < 8; e++) b[e] = term(v[e]);
            G0[t] = mfma(abk0, b, G0[t]);
            G1[t] = mfma(abk1, b, G1[t]);
        }
    }
    if constexpr (F16) {
        // Transpose back in binary16 (the scaled correction, 11 significant bits, far below the
        // storage step of the deviation it corrects): rows of 40 halves (80 bytes) per cell.
        typedef __attribute__((ext_vector_type(4))) _Float16 f16x4_t;
        _Float16 *ldsh = reinterpret_cast<_Float16 *>(lds);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            f16x4_t a, b;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                a[r] = (_Float16)G0[t][r];
                b[r] = (_Float16)G1[t][r];
            }
            *reinterpret_cast<f16x4_t *>(ldsh + 40 * (16 * t + j) + 4 * q) = a;
            *reinterpret_cast<f16x4_t *>(ldsh + 40 * (16 * t + j) + 16 + 4 * q) = b;
        }
        wave_lds_sync();
        const f16x8_t *row = reinterpret_cast<const f16x8_t *>(ldsh + 40 * l);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const f16x8_t h = row[c];
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (8 * c + e < Q) g[8 * c + e] = (float)h[e];
        }
        wave_lds_sync();
    } else {
        // Transpose back: G row p of cell 16t + j -> LDS row of that cell (36 floats), then own row.
#pragma unroll
        for (int t = 0; t < 4; t++) {
            *reinterpret_cast<f32x4_t *>(lds + 36 * (16 * t + j) + 4 * q) = G0[t];
            *reinterpret_cast<f32x4_t *>(lds + 36 * (16 * t + j) + 16 + 4 * q) = G1[t];
        }
        wave_lds_sync();
#pragma unroll
        for (int p = 0; p < Q; p++) g[p] = lds[36 * l + p];
        wave_lds_sync();
    }
}

// Population load of the fused step.  FP32/FP64 rows are read with non-temporal loads: they are
// used once, and keeping them out of L2 leaves it to the pushes, whose partial cache lines from
// neighbouring blocks merge there (measured: the FP32 fused step runs ~20% faster).  16-bit rows
// measured slightly slower that way and use ordinary loads.
template <typename S>
__device__ __forceinline__ S load_pop(const S *p)
{
    if constexpr (sizeof(S) >= 4)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}

template <typename S>
__device__ __forceinline__ S load_pop(const __attribute__((address_space(1))) S *p)
{
    if constexpr (sizeof(S) >= 4)
        return __builtin_nontemporal_load(p);
    else if constexpr (std::is_same<S, bf16s>::value)
        return bf16s{*reinterpret_cast<const __attribute__((address_space(1))) uint16_t *>(p)};
    else
        return *p;
}

template <typename S>
__device__ __forceinline__ S load_plain(const __attribute__((address_space(1))) S *p)
{
    if constexpr (sizeof(S) == 2)
        return __builtin_bit_cast(S, *reinterpret_cast<const __attribute__((address_space(1))) uint16_t *>(p));
    else
        return *p;
}

// A global-memory pointer that is the same on every lane, forced into scalar registers: a lane's
// element of it is then a scalar base plus a 32-bit offset, with no 64-bit vector address
// arithmetic per access.
template <typename S>
__device__ __forceinline__ const __attribute__((address_space(1))) S *scalar_row(const S *p)
{
    const unsigned long long v = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (const __attribute__((address_space(1))) S *)(((unsigned long long)hi << 32) | lo);
}

// Store of the fused step into a row (the same pointer on every lane) at element idx.  A 16-bit
// row holds fewer than 2^32 bytes (the pool has fewer than 2^31 cells, checked at creation), so the
// address is a scalar base plus a 32-bit byte offset, with no 64-bit vector address arithmetic per
// store; wider rows keep 64-bit addresses.
template <typename S>
__device__ __forceinline__ void store_pop(S *row, unsigned idx, S v)
{
    if constexpr (sizeof(S) == 2) {
        const unsigned long long r = reinterpret_cast<unsigned long long>(row);
        const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)r), hi = __builtin_amdgcn_readfirstlane((unsigned)(r >> 32));
        auto *base = (__attribute__((address_space(1))) char *)(((unsigned long long)hi << 32) | lo);
        *(__attribute__((address_space(1))) uint16_t *)(base + idx * 2u) = __builtin_bit_cast(uint16_t, v);
    } else {
        row[idx] = v;
    }
}

// Store of a 16-bit value at a byte offset within a row (the same pointer on every lane).
template <typename S>
__device__ __forceinline__ void store_pop_bytes(S *row, unsigned byte_off, S v)
{
    static_assert(sizeof(S) == 2, "16-bit rows only");
    const unsigned long long r = reinterpret_cast<unsigned long long>(row);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)r), hi = __builtin_amdgcn_readfirstlane((unsigned)(r >> 32));
    auto *base = (__attribute__((address_space(1))) char *)(((unsigned long long)hi << 32) | lo);
    *(__attribute__((address_space(1))) uint16_t *)(base + byte_off) = __builtin_bit_cast(uint16_t, v);
}

// Store into a block's 64 cells of a row, base the same on every lane.
template <typename S>
__device__ __forceinline__ void store_own(S *base, int t, S v)
{
    auto *r = (__attribute__((address_space(1))) S *)(unsigned long long)scalar_row(base);
    if constexpr (sizeof(S) == 2)
        *((__attribute__((address_space(1))) uint16_t *)(unsigned long long)r + t) = __builtin_bit_cast(uint16_t, v);
    else
        r[t] = v;
}

// One link of the fused step for the cell `cell`, direction q >= 1, whose neighbour block in that
// direction is nbk (target cell tgt): boundary hook, swap guard, and the single store of f*_q
// either into the neighbour (the link streams) or into the cell's own opposite slot (bounce-back).
template <typename T, typename S, int Q>
__device__ __forceinline__ void push_link(const StepArgs<T, S> &a, int q, T fq, int nbk, long long tgt, long long cell,
                                          bool inert, bool simple, bool onb, T u, T v, T w)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    // Domain-face hook on links that leave the domain (Cu_ImposeBC, onb blocks, non-solid cells).
    if (onb && nbk < 0 && nbk != N_SKIPID)
        fq = bc_hook<T>(a.bc_preset, a.U, nbk, fq, u, v, w, (T)VS::w(q), (T)VS::cx(q), (T)VS::cy(q), (T)VS::cz(q));
    // In a 16-bit pool the guard below sees the stored value.
    fq = quant<T, S>(fq, (T)VS::w(q));
    bool push;
    bool exc = false;
    if (VS::half(q)) {
        // Initiator of the link x -> x + c_q.
        push = !inert && nbk >= 0;
        if (!simple && push) {
            const bool p_inert = !a.part[nbk] || a.cells_mask[tgt] == CELL_SOLID;
            if (p_inert) push = ST::dec(a.A[(long long)q * a.ncm + tgt], (T)VS::w(q)) > (T)0;
        }
    } else {
        // Partner of the link initiated by the cell x + c_q in direction pb(q).
        push = nbk >= 0;
        if (!simple && push) push = a.part[nbk] && a.cells_mask[tgt] != CELL_SOLID;
        if (push && !(fq > (T)0)) {
            push = false;
            exc = !inert;  // a colliding partner cannot tell the initiator in time
        }
    }
    if (exc) {
        record_exception(a, tgt, cell, q, fq);
        return;
    }
    const long long at = push ? (long long)q * a.ncm + tgt : (long long)VS::pb(q) * a.ncm + cell;
    a.B[at] = ST::enc(fq, (T)VS::w(q));
}

// ds_bpermute byte address (4 x slot) of the block that holds cell x + c_q, lane t = cell x: one wave
// lane per neighbour slot.
template <int Q>
struct SlotOf {
    int xp, xm, yp, ym, zp, zm;
    __device__ __forceinline__ explicit SlotOf(int t)
    {
        const int I = t & 3, J = (t >> 2) & 3, K = t >> 4;
        xp = I == 3 ? 4 : 0;
        xm = I == 0 ? -4 : 0;
        yp = J == 3 ? 12 : 0;
        ym = J == 0 ? -12 : 0;
        zp = K == 3 ? 36 : 0;
        zm = K == 0 ? -36 : 0;
    }
    __device__ __forceinline__ int operator()(int q) const
    {
        using VS = VelSet<Q>;
        int s = 13 * 4;
        if (VS::cx(q) > 0) s += xp;
        if (VS::cx(q) < 0) s += xm;
        if (VS::cy(q) > 0) s += yp;
        if (VS::cy(q) < 0) s += ym;
        if (VS::cz(q) > 0) s += zp;
        if (VS::cz(q) < 0) s += zm;
        return s;
    }
};

// Cell of x + c_q within its block, lane t = cell x: ((I+cx)&3) + 4((J+cy)&3) + 16((K+cz)&3), a
// field-wise sum without carries between the 2-bit fields; all fields shifted up by SH bits.
template <int Q, int SH>
__device__ __forceinline__ unsigned cell_of_link(int t, int q)
{
    using VS = VelSet<Q>;
    const unsigned d = (unsigned)((VS::cx(q) & 3) | ((VS::cy(q) & 3) << 2) | ((VS::cz(q) & 3) << 4));
    const unsigned tl = ((unsigned)t & 0x15u) << SH, th = ((unsigned)t & 0x2Au) << SH;
    return (tl + ((d & 0x15u) << SH)) ^ th ^ ((d & 0x2Au) << SH);
}

// The face hook (Cu_ImposeBC, bc_hook) on the links of a block on the domain boundary, before its values
// leave: selects on the neighbour ID, one link after the other, since branches around a link keep two
// versions of all values alive (103 instead of 56 registers).
template <typename T, typename S, int Q>
__device__ __forceinline__ void hook_links(const StepArgs<T, S> &a, T *fs, int my_nb, int t, T u, T v, T w)
{
    using VS = VelSet<Q>;
    // Face IDs -1 .. -6 that are walls with the preset's speed (bit -ID); -2 is an outflow with the others.
    const unsigned walls = a.bc_preset == BC_LDC2D ? 1u << 4 : a.bc_preset == BC_LDC3D ? 1u << 6 :
                           a.bc_preset == BC_FPSC2D ? 0x1Au : a.bc_preset == BC_FPSC3D ? 0x7Au : 0u;
    const bool outflow = a.bc_preset == BC_FPSC2D || a.bc_preset == BC_FPSC3D;
    // Looked up afresh: a merge with the streaming's lookups would hold them all across the collision.
    asm volatile("" : "+v"(t), "+v"(my_nb) : "v"(fs[0]));
    const SlotOf<Q> slot(t);
#pragma unroll
    for (int q = 1; q < Q; q++) {
        const unsigned face = (unsigned)-__builtin_amdgcn_ds_bpermute(slot(q), my_nb);
        const T wq = (T)VS::w(q), cx = (T)VS::cx(q), cy = (T)VS::cy(q), cz = (T)VS::cz(q), f = fs[q];
        const T g = f - (T)(2.0) * wq * ((T)(3.0) * (cx * a.U));
        T r = face <= 6u && ((walls >> (face & 31u)) & 1u) ? g : f;
        if (outflow) {
            T cdotu = cx * u + cy * v + cz * w;
            cdotu = (T)(1.0) + (T)(4.5) * cdotu * cdotu - (T)(1.5) * (u * u + v * v + w * w);
            const T o = -f + (T)(2.0) * wq * cdotu;
            r = face == 2u ? o : r;
        }
        fs[q] = r;
    }
}

// Records the partner-side links of this lane's cell whose stored value fails the swap guard and whose
// neighbour block exists.  Rare, so kept out of the streaming loops and their registers: the values
// are read back from where this lane has just put them (EVEN: the cell's own rows pb(q); else row q of
// cell x + c_q, which no other lane writes).
template <typename T, typename S, int Q, bool EVEN>
__device__ __forceinline__ void record_failed_guards(const StepArgs<T, S> &a, int b, int t)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
#pragma unroll 1
    for (int q = 2; q < Q; q++) {
        // Two bits per direction: c + 1.
        constexpr auto pack = [](int axis) {
            unsigned long long k = 0;
            for (int p = 0; p < Q; p++) k |= (unsigned long long)((axis == 0 ? VS::cx(p) : axis == 1 ? VS::cy(p) : VS::cz(p)) + 1) << (2 * p);
            return k;
        };
        constexpr unsigned long long KX = pack(0), KY = pack(1), KZ = pack(2);
        if (VS::half(q)) continue;
        const int I = (t & 3) + (int)((KX >> (2 * q)) & 3) + 3, J = ((t >> 2) & 3) + (int)((KY >> (2 * q)) & 3) + 3,
                  K = (t >> 4) + (int)((KZ >> (2 * q)) & 3) + 3;
        const int nbk = a.nbr_slot[(long long)b * 27 + (I >> 2) + 3 * (J >> 2) + 9 * (K >> 2)];
        if (nbk < 0) continue;
        const long long tgt = (long long)nbk * 64 + ((I & 3) + 4 * (J & 3) + 16 * (K & 3)), cell = (long long)b * 64 + t;
        const T wq = q < 7 ? (T)VS::w(1) : (q < 19 ? (T)VS::w(7) : (T)VS::w(Q - 1));
        const T f = ST::dec(EVEN ? a.B[(long long)VS::pb(q) * a.ncm + cell] : a.B[(long long)q * a.ncm + tgt], wq);
        if (!(f > (T)0)) record_exception(a, tgt, cell, q, f);
    }
}

// Stream of an interior block (block flag simple == 2): every neighbour slot of the velocity set
// exists, and the block and its neighbours participate with no solid cell.  No link then leaves
// the domain or the level and no guard read is needed: every link pushes.  A partner-side value that
// fails the guard on its stored form is recorded as well; the fixup then rewrites both ends, so what
// was stored there does not matter.  The target block comes from the wave's neighbour table (lane s
// holds slot s) through ds_bpermute, the target cell from cell_of_link.
template <typename T, typename S, int Q>
__device__ __forceinline__ void push_interior(const StepArgs<T, S> &a, const T *fs, int my_nb, int b, int t)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    // 16-bit rows: the target as a byte offset within the row (block << 7 | cell << 1), so the store
    // needs no further shift.
    constexpr int SH = sizeof(S) == 2 ? 1 : 0;
    const SlotOf<Q> slot(t);
    const int nb_src = (int)((unsigned)my_nb << (6 + SH));
    bool failed = false;
#pragma unroll
    for (int q = 1; q < Q; q++) {
        const unsigned tgt_s = (unsigned)__builtin_amdgcn_ds_bpermute(slot(q), nb_src) + cell_of_link<Q, SH>(t, q);
        const S e = ST::enc(fs[q], (T)VS::w(q));
        if (!VS::half(q)) failed = failed || !ST::positive(e, (T)VS::w(q));
        if constexpr (SH == 1)
            store_pop_bytes(a.B + (long long)q * a.ncm, tgt_s, e);
        else
            store_pop(a.B + (long long)q * a.ncm, tgt_s, e);
    }
    if (failed) record_failed_guards<T, S, Q, false>(a, b, t);
}

// Slot of link q relative to row q, in elements: the neighbour's cell, or, where the neighbour is
// missing, the cell's own place in row pb(q) (one row up or down).
template <int Q>
__device__ __forceinline__ long long link_slot(int nbk, int t, int q, long long own_up, long long own_down)
{
    const unsigned tgt = ((unsigned)nbk << 6) + cell_of_link<Q, 0>(t, q);
    return nbk < 0 ? (VelSet<Q>::pb(q) > q ? own_up : own_down) : (long long)tgt;
}

// Stream of a simple block that is not interior (block flag simple == 1): the block and its
// existing neighbours participate with no solid cell, but some neighbour slots are missing (a
// domain face, or a coarser region).  As push_interior, but a link whose neighbour slot is missing
// bounces back into the cell's own opposite slot -- the rows of a pair are neighbours, so both
// targets are one select of an offset.  The face hook has been applied.
template <typename T, typename S, int Q>
__device__ __forceinline__ void push_simple(const StepArgs<T, S> &a, const T *fs, int my_nb, int b, int t)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    // The lane number as of after the collision: forming the 64-bit slots earlier and holding them
    // across it costs a quarter of the wavefronts per SIMD.
    asm volatile("" : "+v"(t) : "v"(fs[0]));
    const SlotOf<Q> slot(t);
    const unsigned cell = (unsigned)b * 64u + (unsigned)t;
    const long long up = (long long)cell + a.ncm, down = (long long)cell - a.ncm;
    bool failed = false;
#pragma unroll
    for (int q = 1; q < Q; q++) {
        const int nbk = __builtin_amdgcn_ds_bpermute(slot(q), my_nb);
        const S e = ST::enc(fs[q], (T)VS::w(q));
        if (!VS::half(q)) failed = failed || (nbk >= 0 && !ST::positive(e, (T)VS::w(q)));
        (a.B + (long long)q * a.ncm)[link_slot<Q>(nbk, t, q, up, down)] = e;
    }
    if (failed) record_failed_guards<T, S, Q, false>(a, b, t);
}

// The extra exception list of the previous finest sub-step, applied to this block's loaded values:
// for an entry (initiator cell i, partner cell c, direction q) the fixup would move the value at
// (pb(q), c) -- the initiator's push -- to (q, i) and store the partner's value at (pb(q), c).
// The previous sub-step's output is this sub-step's input, read by no one else in between, so
// the same values are taken here as the loads' results instead.  No two entries share a slot (an
// entry's q is the partner's, non-initiating direction and pb(q) an initiating one), so the order
// of application is free.  The wavefront walks its block's chain (the entries with i or c in the
// block, linked when they were recorded), so the work per block is its own entries however long
// the list is; the chain is emptied for the next pair.
template <typename T, typename S, int Q>
__device__ __forceinline__ void apply_pending(const StepArgs<T, S> &a, T *f, int b, int t)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    const unsigned my = ((unsigned)b << 6) | (unsigned)t;
    int e = __builtin_amdgcn_readfirstlane(a.x_head[b]);
    while (e >= 0) {
        const int k = e >> 1;
        const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane(a.va_idx[3 * (long long)k + 0]);
        const unsigned hc = (unsigned)__builtin_amdgcn_readfirstlane(a.va_idx[3 * (long long)k + 1]);
        const int hq = __builtin_amdgcn_readfirstlane(a.va_idx[3 * (long long)k + 2]);
        int qb = 0;
        T wq = 0;
#pragma unroll
        for (int p = 0; p < Q; p++)
            if (p == hq) {
                qb = VS::pb(p);
                wq = (T)VS::w(p);
            }
        // Through storage, as the fixup's store and this sub-step's load would take them.
        const T vi = ST::dec(a.A[(long long)qb * a.ncm + hc], wq);
        const T vc = ST::dec(ST::enc(a.va_val[k], wq), wq);
        const bool at_i = hi == my, at_c = hc == my;
#pragma unroll
        for (int p = 1; p < Q; p++) {
            if (at_i && p == hq) f[p] = vi;
            if (at_c && p == qb) f[p] = vc;
        }
        e = __builtin_amdgcn_readfirstlane(a.x_next[e]);
    }
    if (t == 0) a.x_head[b] = -1;
}

// Moments and post-collision values of the wavefront's cells (one 3D block), MRT on matrix cores with
// COLL_MFMA (`lds`: the wavefront's transpose region).
template <typename T, typename S, int Q, int COLL>
__device__ __forceinline__ void collide_block(const StepArgs<T, S> &a, const T *f, T *fs, T &rho, T &u, T &v, T &w,
                                              bool inert, float *lds)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    moments<T, Q>(f, rho, u, v, w);
    if constexpr (COLL == COLL_MFMA) {
        // MRT with the moment transform on matrix cores (whole wavefront, inert lanes carry zeros).
        // The non-equilibrium parts go in scaled by SC (16-bit pools: 2^10, see mrt_mfma) and the
        // correction comes back scaled by SC; the equilibrium in pairs (p, pb(p)) with fused
        // multiply-adds, SC folded into the density.
        constexpr float SC = ST::quantized ? 1024.0f : 1.0f;
        const T c1 = (T)(1.0) - (T)(1.5) * (u * u + v * v + w * w);
        const T rs = rho * (T)SC;
        float d[Q], g[Q];
        d[0] = inert ? 0.f : fmadd(f[0], (T)SC, -((T)VS::w(0) * rs * c1));
#pragma unroll
        for (int p = 1; p < Q; p++) {
            if (!VS::half(p)) continue;
            const int q = VS::pb(p);
            const T cu = cdot<T, Q>(p, u, v, w);
            const T b = fmadd((T)(4.5) * cu, cu, c1);
            const T wr = (T)VS::w(p) * rs;
            d[p] = inert ? 0.f : fmadd(f[p], (T)SC, -(wr * fmadd((T)(3.0), cu, b)));
            d[q] = inert ? 0.f : fmadd(f[q], (T)SC, -(wr * fmadd((T)(-3.0), cu, b)));
        }
        mrt_mfma<Q, ST::quantized>(d, g, a.ck, lds);
#pragma unroll
        for (int p = 0; p < Q; p++) fs[p] = inert ? f[VS::pb(p)] : fmadd((T)g[p], (T)(-1.0f / SC), f[p]);
    } else {
        collide_cell<T, S, Q, COLL>(a, f, fs, rho, u, v, w, inert);
    }
}

// First sub-step of an in-place pair (lbm_inplace.hip): the wavefront's block collides and puts f*_q
// into its own row pb(q), in the buffer it read.  No value leaves the block; the second sub-step
// fetches across the links.  The face hook acts here, on links that leave the domain; a partner-
// side value that fails the swap guard is recorded, and the exchange of its two ends before the
// second sub-step makes that link bounce back at both (fixup_level).  Blocks without solid cells only.
template <typename T, typename S, int Q, int COLL>
__device__ __forceinline__ void even_step_3d(const StepArgs<T, S> &a, int wave, float *lds)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    const int t = threadIdx.x & 63;
    if (wave >= a.n) return;  // whole wavefronts only
    const int b = __builtin_amdgcn_readfirstlane(a.ids[wave]);
    const int onb_u = __builtin_amdgcn_readfirstlane(a.onb[b]);
    T f[Q];
    if (a.nt) {
#pragma unroll
        for (int q = 0; q < Q; q++)
            f[q] = ST::dec(load_pop(scalar_row(a.A + (long long)q * a.ncm + (long long)b * 64) + t), (T)VS::w(q));
    } else {
#pragma unroll
        for (int q = 0; q < Q; q++)
            f[q] = ST::dec(load_plain(scalar_row(a.A + (long long)q * a.ncm + (long long)b * 64) + t), (T)VS::w(q));
    }
    T fs[Q];
    T rho, u, v, w;
    collide_block<T, S, Q, COLL>(a, f, fs, rho, u, v, w, false, lds);
    if (onb_u == 1) {
        const int my_nb = a.nbr_slot[(long long)b * 27 + (t < 27 ? t : 26)];
        hook_links<T, S, Q>(a, fs, my_nb, t, u, v, w);
    }
    bool failed = false;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const S e = ST::enc(fs[q], (T)VS::w(q));
        if (q > 0 && !VS::half(q)) failed = failed || !ST::positive(e, (T)VS::w(q));
        store_own(a.B + (long long)VS::pb(q) * a.ncm + (long long)b * 64, t, e);
    }
    if (failed) record_failed_guards<T, S, Q, true>(a, b, t);
}

// 3D: one wavefront per block, so the block, its flags and its 27 neighbour IDs are wave-uniform
// (scalar registers); each lane picks its link's neighbour among at most eight of them with
// selects on its own cell position -- no LDS traffic and no per-direction waits.  Interior blocks
// take push_interior instead.
template <typename T, typename S, int Q, int COLL>
__device__ __forceinline__ void collide_stream_3d(const StepArgs<T, S> &a, int wave, float *lds)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    const int t = threadIdx.x & 63;
    const int bi = wave;  // one block per wavefront
    if (bi >= a.n) return;  // whole wavefronts only; the kernel has no barrier
    const int b = __builtin_amdgcn_readfirstlane(a.ids[bi]);
    // Cell index within a population row (the pool holds fewer than 2^32 cells, checked at
    // creation), so rows are addressed as a row base plus a 32-bit index.
    const unsigned cell = (unsigned)b * 64u + (unsigned)t;
    // Lane s < 27 holds neighbour slot s (lanes above repeat slot 26): a load on every lane keeps
    // the block index out of divergent control flow, so it stays a scalar.
    const int my_nb = a.nbr_slot[(long long)b * 27 + (t < 27 ? t : 26)];
    const int flags_u = __builtin_amdgcn_readfirstlane(a.simple[b]);
    if ((flags_u & LINK_FLAG) && a.skip_linked) return;
    const int simple_u = flags_u & 3;
    const int part_u = __builtin_amdgcn_readfirstlane(a.part[b]);
    const int onb_u = __builtin_amdgcn_readfirstlane(a.onb[b]);
    T f[Q];
#pragma unroll
    for (int q = 0; q < Q; q++)  // row q of block b: a scalar base, lane t at offset t
        f[q] = ST::dec(load_pop(scalar_row(a.A + (long long)q * a.ncm + (long long)b * 64) + t), (T)VS::w(q));
    if (a.vmode == 2 && (flags_u & PEND_FLAG)) {
        apply_pending<T, S, Q>(a, f, b, t);
        if (t == 0) a.flags[b] = simple_u;  // this sub-step sets no flags: no other writer
    }
    const bool simple = simple_u != 0;
    int mask = CELL_INTERIOR;
    if (!simple) mask = a.cells_mask[cell];
    const bool inert = part_u == 0 || mask == CELL_SOLID;
    const bool onb = onb_u == 1 && mask != CELL_SOLID;

    T fs[Q];
    T rho, u, v, w;
    collide_block<T, S, Q, COLL>(a, f, fs, rho, u, v, w, inert, lds);

    store_pop(a.B, cell, ST::enc(fs[0], (T)VS::w(0)));
    if (simple_u == 2) {
        push_interior<T, S, Q>(a, fs, my_nb, b, t);
        return;
    }
    if (simple_u == 1) {
        if (onb_u == 1) hook_links<T, S, Q>(a, fs, my_nb, t, u, v, w);
        push_simple<T, S, Q>(a, fs, my_nb, b, t);
        return;
    }
    int nbs[27];
#pragma unroll
    for (int s = 0; s < 27; s++) nbs[s] = __builtin_amdgcn_readlane(my_nb, s);
    const int I = t & 3, J = (t >> 2) & 3, K = t >> 4;
#pragma unroll
    for (int q = 1; q < Q; q++) {
        const int cx = VS::cx(q), cy = VS::cy(q), cz = VS::cz(q);
        // Does the link leave the block along x / y / z?
        const bool ex = cx > 0 ? I == 3 : (cx < 0 ? I == 0 : false);
        const bool ey = cy > 0 ? J == 3 : (cy < 0 ? J == 0 : false);
        const bool ez = cz > 0 ? K == 3 : (cz < 0 ? K == 0 : false);
        // Slot (dx+1) + 3(dy+1) + 9(dz+1) of the neighbour block; 13 is the block itself.
        const int sxyz = nbs[13 + cx + 3 * cy + 9 * cz], sxy = nbs[13 + cx + 3 * cy], sxz = nbs[13 + cx + 9 * cz],
                  syz = nbs[13 + 3 * cy + 9 * cz], sx = nbs[13 + cx], sy = nbs[13 + 3 * cy], sz = nbs[13 + 9 * cz];
        const int nbk = ex ? (ey ? (ez ? sxyz : sxy) : (ez ? sxz : sx)) : (ey ? (ez ? syz : sy) : (ez ? sz : b));
        const long long tgt = (long long)nbk * 64 + (((I + cx) & 3) + 4 * ((J + cy) & 3) + 16 * ((K + cz) & 3));
        push_link<T, S, Q>(a, q, fs[q], nbk, tgt, (long long)cell, inert, simple, onb, u, v, w);
    }
}

// One launch of the fused step over the blocks of up to MAXLV levels: the levels' workgroups are
// consecutive ranges [start[k], start[k+1]) of the launch, multiples of 8, each dealt to the XCDs in
// contiguous ranges of its own (one 3D block or four 2D blocks per wavefront).  The levels' blocks cost
// differently -- an in-place first sub-step less than a fused one -- so one deal over all levels left the
// XCDs of the fine level's blocks behind: a whole step of the 128^3 four-level cavity took 11.54 ms and now
// 11.18 ms, of the adaptive 64^3 case 502 us and now 481 us (D3Q19 FP32; one level alone is dealt as
// before).  Levels of one launch touch disjoint cells and their own exception lists, so one launch does
// what separate launches of each level would.
constexpr int MAXLV = 4;

template <typename T, typename S>
struct MultiStep {
    int nlv;
    int start[MAXLV + 1];
    StepArgs<T, S> lv[MAXLV];
};

// 2D: four 4x4 blocks per wavefront; neighbour IDs are distributed with ds_bpermute.
template <typename T, typename S, int Q, int COLL>
__device__ __forceinline__ void collide_stream_2d(const StepArgs<T, S> &a, int wave)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    constexpr int CELLS = VS::CELLS, DIM = VS::DIM, QMAX = VS::QMAX;
    const int t = threadIdx.x % CELLS;
    const int lane = threadIdx.x % 64;
    const int gbase = lane - t;  // lane of cell 0 of this block within the wavefront
    const int bi = wave * (64 / CELLS) + lane / CELLS;
    const bool active = bi < a.n;
    const int b = active ? a.ids[bi] : 0;
    // Lane-parallel load of the block's neighbour table; distributed with ds_bpermute (every
    // __shfl below sits outside divergent control flow).
    const int my_nb = (active && t < QMAX) ? a.nbr_slot[(long long)b * QMAX + t] : N_SKIPID;
    const int I = t % 4, J = (t / 4) % 4, K = (DIM == 3) ? t / 16 : 0;
    const long long cell = (long long)b * CELLS + t;

    bool simple = true, inert = false, onb = false;
    int mask = CELL_INTERIOR;
    T f[Q];
    if (active) {
        simple = (a.simple[b] & 3) != 0;
        const bool part = a.part[b] != 0;
        if (!simple) mask = a.cells_mask[cell];
        inert = !part || mask == CELL_SOLID;
        onb = a.onb[b] == 1 && mask != CELL_SOLID;
#pragma unroll
        for (int q = 0; q < Q; q++) f[q] = ST::dec(load_pop(&a.A[(long long)q * a.ncm + cell]), (T)VS::w(q));
    } else {
#pragma unroll
        for (int q = 0; q < Q; q++) f[q] = (T)1;
    }

    T fs[Q];
    T rho, u, v, w;
    moments<T, Q>(f, rho, u, v, w);
    collide_cell<T, S, Q, COLL>(a, f, fs, rho, u, v, w, inert);

    if (active) a.B[cell] = ST::enc(fs[0], (T)VS::w(0));
#pragma unroll
    for (int q = 1; q < Q; q++) {
        const int Ip = I + VS::cx(q), Jp = J + VS::cy(q), Kp = K + VS::cz(q);
        const int slot = (Ip < 0 ? 0 : (Ip >= 4 ? 2 : 1)) + 3 * (Jp < 0 ? 0 : (Jp >= 4 ? 2 : 1)) +
                         (DIM == 3 ? 9 * (Kp < 0 ? 0 : (Kp >= 4 ? 2 : 1)) : 0);
        const int nbk = __shfl(my_nb, gbase + slot, 64);
        if (!active) continue;
        const long long tgt = (long long)nbk * CELLS + ((Ip & 3) + 4 * (Jp & 3) + (DIM == 3 ? 16 * (Kp & 3) : 0));
        push_link<T, S, Q>(a, q, fs[q], nbk, tgt, cell, inert, simple, onb, u, v, w);
    }
}

// Resolves guard exceptions: the initiator's pushed value returns to it (bounce-back) and the
// partner keeps its own post-collision value.  One workgroup per level of the fused launch, each on
// its level's list; it clears the list's counter when done.
template <typename T, typename S>
struct FixupArgs {
    int n;       // lists
    int *sync;   // resolve_pending: ticket, done flag, passed workgroups; [3 + k] k_fixup (zero between launches)
    long long ncm, exc_cap;
    S *B[MAXLV];
    const int *exc_idx[MAXLV];
    const T *exc_val[MAXLV];
    int *exc_count[MAXLV];
    int *va_count[MAXLV];  // the finest level: its extra list's counter, cleared here, else null
    // The list of an in-place pair's first sub-step: the pushed values of the link's ends, which lie in
    // (q, initiator) and (pb(q), partner) waiting to be fetched across it, change places.
    int exchange[MAXLV];
};

template <typename T, typename S, int Q>
__device__ __forceinline__ void fixup_level(const FixupArgs<T, S> &fa, int lv, int part = 0, int parts = 1)
{
    using VS = VelSet<Q>;
    S *B = fa.B[lv];
    const int *exc_idx = fa.exc_idx[lv];
    const T *exc_val = fa.exc_val[lv];
    const long long ncm = fa.ncm, n = min((long long)fa.exc_count[lv][0], fa.exc_cap);
    for (long long k = part * WG + threadIdx.x; k < n; k += parts * WG) {  // no two entries share a slot
        const long long i = (unsigned)exc_idx[3 * k + 0], c = (unsigned)exc_idx[3 * k + 1];
        const int q = exc_idx[3 * k + 2];
        int qb = 0;
        T wq = 0;
#pragma unroll
        for (int p = 0; p < Q; p++)
            if (p == q) {
                qb = VS::pb(p);
                wq = (T)VS::w(p);
            }
        // Rows q and pb(q) share one weight: a stored value moves between them unchanged.
        const S vi = B[(long long)qb * ncm + c];
        B[(long long)qb * ncm + c] = fa.exchange[lv] ? B[(long long)q * ncm + i] : Store<T, S>::enc(exc_val[k], wq);
        B[(long long)q * ncm + i] = vi;
    }
}

// List lv starts empty again, and so does the extra list, which was applied by the sub-step that list
// lv comes from.
template <typename T, typename S>
__device__ __forceinline__ void fixup_reset(const FixupArgs<T, S> &fa, int lv)
{
    fa.exc_count[lv][0] = 0;
    if (fa.va_count[lv]) fa.va_count[lv][0] = 0;
}

// Opens a small launch that touches what pending exception lists will rewrite, in place of a launch of
// their own (4.7 us each, as empty as the lists usually are).  Every workgroup looks at the counters; if
// any list holds an entry, the workgroup that draws ticket 0 resolves all lists and raises the flag, the
// others wait for it -- a workgroup that runs, so the wait ends whatever the order of dispatch -- and the
// last one to pass empties the lists and the counters of this hand-over.  The kernel records into other
// lists than it resolves here (fold_fixups sees to it), so every workgroup finds the counters as the first
// did.  Called by all threads of all workgroups, before any exit, in the FOLD variants of the kernels (its mere presence
// costs a large launch 1-3%).  The line between doing so and a fixup launch before the kernel (fold_fixups)
// weighs two flows.  With empty lists the hand-over saves about as much at every size, with entries it
// costs more the larger the launch, because the acquire of a workgroup that starts later empties the L2
// under those that run.  us per step of one level in D3Q19 FP32, resolved by the step's own kernel / by a fixup launch:
//   workgroups                                  16           128          250          686          2000         3456
//   empty lists                                 7.0 / 7.9    7.2 / 8.0    7.6 / 8.4    9.8 / 10.7   18.6 / 19.0  28.4 / 29.1
//   first eight steps from 2% failing values    12.8 / 12.6  15.3 / 13.0  16.7 / 14.0  22.8 / 16.9  39.0 / 21.6  61 / 44.5
// (three refined levels, empty lists: 55.5 / 59.4 with launches of up to 160 workgroups, 133 / 135 with 3300).
// At 128 empty lists, the usual case, save a tenth and entries cost a sixth; beyond, the saving becomes a
// smaller share of the step and the cost a larger one.
constexpr int FOLD_MAX_WGS = 128;

template <typename T, typename S, int Q>
__device__ __forceinline__ void resolve_pending(const FixupArgs<T, S> &fa)
{
    int any = 0;
#pragma unroll
    for (int k = 0; k < MAXLV; k++)
        if (k < fa.n) {
            any |= fa.exc_count[k][0];
            if (fa.va_count[k]) any |= fa.va_count[k][0];
        }
    if (any == 0) return;  // the same in every workgroup
    __shared__ int s_ticket;
    if (threadIdx.x == 0) s_ticket = atomicAdd(&fa.sync[0], 1);
    __syncthreads();
    if (s_ticket == 0) {
        for (int k = 0; k < fa.n; k++) {
            fixup_level<T, S, Q>(fa, k);
            __syncthreads();
        }
        if (threadIdx.x == 0) __hip_atomic_store(&fa.sync[1], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    } else if (threadIdx.x == 0) {
        while (__hip_atomic_load(&fa.sync[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) __builtin_amdgcn_s_sleep(8);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // what the resolving workgroup wrote is seen from here on
    }
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(&fa.sync[2], 1) == (int)gridDim.x - 1) {
        for (int k = 0; k < fa.n; k++) fixup_reset<T, S>(fa, k);
        fa.sync[0] = fa.sync[1] = fa.sync[2] = 0;
    }
}

// ---------------------------------------------------------------------------------------------
// Host side: launch arguments.
// ---------------------------------------------------------------------------------------------
template <typename T>
static T *Fbuf(Ctx *c, int k) { return static_cast<T *>(c->F[k]); }

// Fused-step arguments of level L reading population buffer rd (writing rd ^ 1).
template <typename T, typename S, int Q>
static inline StepArgs<T, S> step_args(Ctx *c, int L, int rd, int vmode = 0)
{
    StepArgs<T, S> a;
    a.ids = c->order_L(L);  // the level's blocks in traversal order
    a.n = c->n_ids[L];
    a.A = Fbuf<S>(c, rd);
    a.B = Fbuf<S>(c, vmode == VMODE_EVEN ? rd : rd ^ 1);
    a.ncm = c->n_maxcells;
    a.nbr_slot = c->nbr_slot;
    a.part = c->part;
    a.simple = c->simple;
    a.cells_mask = c->cells_mask;
    a.onb = c->onb;
    const T dx_L = (T)c->dxf_vec[L], tau_L = (T)c->tau_vec[L];
    a.omeg = dx_L / tau_L;
    a.omegp = (T)(1.0) - a.omeg;
    a.mrt = c->P.collision == AGAL_MRT;
    {
        const double s[6] = {c->P.s1, c->P.s2, c->P.s3, c->P.s4, c->P.s5, c->P.s6};
        for (int k = 0; k < 27; k++) a.ck[k] = (T)0;
        for (int k = 0; k < Q; k++) {
            const int rc = Mrt<Q>::rate(k);
            if (rc == 0) continue;
            const T rate = rc == 1 ? a.omeg : (T)s[rc - 2];
            a.ck[k] = (T)((double)rate / (double)mrt_norm<Q>(k));
        }
    }
    a.U = (T)c->P.bc_velocity;
    a.bc_preset = c->P.bc_preset;
    // Each level has its own exception lists: levels share launches.  Two of them, in turn: the kernel
    // that resolves one records into the other.
    const int slot = c->exc_slot(L), XL = c->exc_extra();
    a.exc_idx = c->exc_idx + (size_t)3 * c->exc_cap * slot;
    a.exc_val = static_cast<T *>(c->exc_val) + (size_t)c->exc_cap * slot;
    a.exc_count = c->exc_count + 2 * slot;
    a.exc_cap = c->exc_cap;
    a.vmode = vmode;
    a.skip_linked = 0;
    a.nt = (long long)c->n_ids[L] * 64 * Q * (long long)sizeof(S) > MALL_BYTES;
    a.flags = c->simple;
    a.va_idx = c->exc_idx + (size_t)3 * c->exc_cap * XL;
    a.va_val = static_cast<T *>(c->exc_val) + (size_t)c->exc_cap * XL;
    a.va_count = c->exc_count + 2 * XL;
    a.x_head = c->exc_head;
    a.x_next = c->exc_next;
    if (vmode == 1) {
        a.exc_idx = c->exc_idx + (size_t)3 * c->exc_cap * XL;
        a.exc_val = static_cast<T *>(c->exc_val) + (size_t)c->exc_cap * XL;
        a.exc_count = c->exc_count + 2 * XL;
    }
    return a;
}

// Exception lists waiting for their fixup: up to MAXLV of the pending levels in `mask` go into fa
// (with the buffer that the launch which left the list wrote) and leave the pending set.
template <typename T, typename S>
static inline int take_fixups(Ctx *c, unsigned mask, FixupArgs<T, S> &fa, unsigned &wmask)
{
    int n = 0;
    std::vector<Ctx::PendingFix> keep;
    for (const auto &pf : c->pending_fix) {
        if (!((mask >> pf.L) & 1) || n == MAXLV) {
            keep.push_back(pf);
            continue;
        }
        fa.B[n] = Fbuf<S>(c, pf.buf);
        fa.exc_idx[n] = c->exc_idx + (size_t)3 * c->exc_cap * pf.slot;
        fa.exc_val[n] = static_cast<T *>(c->exc_val) + (size_t)c->exc_cap * pf.slot;
        fa.exc_count[n] = c->exc_count + 2 * pf.slot;
        fa.va_count[n] = pf.L == c->MAX_LEVELS - 1 ? c->exc_count + 2 * c->exc_extra() : nullptr;
        fa.exchange[n] = pf.exchange;
        wmask |= res_bit(pf.L, pf.buf);
        n++;
    }
    c->pending_fix = keep;
    fa.n = n;
    fa.sync = c->exc_count + 2 * c->exc_lists();
    fa.ncm = c->n_maxcells;
    fa.exc_cap = c->exc_cap;
    return n;
}

// Resolves pending lists on their own, FIX_PARTS workgroups for each.
constexpr int FIX_PARTS = 16;

template <typename T, typename S, int Q>
__global__ __launch_bounds__(WG) void k_fixup(FixupArgs<T, S> fa)
{
    const int lv = blockIdx.x / FIX_PARTS;
    if (fa.exc_count[lv][0] == 0 && (!fa.va_count[lv] || fa.va_count[lv][0] == 0)) return;  // the usual case
    fixup_level<T, S, Q>(fa, lv, blockIdx.x % FIX_PARTS, FIX_PARTS);
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(&fa.sync[3 + lv], 1) == FIX_PARTS - 1) {
        fixup_reset<T, S>(fa, lv);
        fa.sync[3 + lv] = 0;
    }
}

// Fixup launches for all pending lists.
template <typename T, typename S, int Q>
static inline int launch_fixups(Ctx *c)
{
    for (;;) {
        FixupArgs<T, S> fa;
        unsigned wmask = 0;
        const int n = take_fixups<T, S>(c, ~0u, fa, wmask);
        if (n == 0) return AGAL_OK;
        hipStream_t s = sched_begin(c, 0, 0, wmask);
        hipLaunchKernelGGL((k_fixup<T, S, Q>), dim3(n * FIX_PARTS), dim3(WG), 0, s, fa);
        AGAL_HIP(c, hipGetLastError());
        int st = sched_done(c, s, 0, 0, wmask);
        if (st) return st;
    }
}

// All pending lists, if there is one of a level in `touch`.
template <typename T, typename S, int Q>
static inline int launch_fixups_for(Ctx *c, unsigned touch)
{
    for (const auto &pf : c->pending_fix)
        if ((touch >> pf.L) & 1) return launch_fixups<T, S, Q>(c);
    return AGAL_OK;
}

// Lists (bits, numbered as in exc_count) that the sub-step of level L in mode `vmode` records into.
static inline unsigned long long records_into(const Ctx *c, int L, int vmode)
{
    return 1ull << (vmode == 1 ? c->exc_extra() : c->exc_slot(L));
}

// The pending lists for a launch of `wgs` workgroups that touches the levels in `touch` and records into
// the lists in `records`: all handed to it in fa, or, for a large launch that touches one of them, all
// resolved by a fixup launch before it.  A launch never resolves a list that it records into: its
// workgroups would find different counters.  A level's own two lists take turns, but the extra list,
// emptied with the pending list of the finest level's second sub-step, is recorded into by the next first
// one, and nothing lies between the two where the parent level is refined as a whole (no interface
// blocks, hence no average).
template <typename T, typename S, int Q>
static inline int fold_fixups(Ctx *c, int wgs, unsigned touch, unsigned long long records, FixupArgs<T, S> &fa, unsigned &wmask)
{
    const bool fold = wgs <= FOLD_MAX_WGS;
    unsigned long long resolves = 0;
    for (const auto &pf : c->pending_fix) {
        resolves |= 1ull << pf.slot;
        if (pf.L == c->MAX_LEVELS - 1) resolves |= 1ull << c->exc_extra();
    }
    if (resolves & records) touch = ~0u;
    if (!fold || c->pending_fix.size() > MAXLV || (resolves & records))
        if (int st = launch_fixups_for<T, S, Q>(c, touch)) return st;
    take_fixups<T, S>(c, fold ? ~0u : 0u, fa, wmask);
    return AGAL_OK;
}

// Launch of a fused sub-step kernel updating `cells` cells; in the timed pass with events recorded by
// the dispatch itself, which bracket the kernel's execution.
template <typename K, typename A, typename B>
static inline int launch_timed(Ctx *c, K kern, int grid, hipStream_t s, double cells, const A &a, const B &b)
{
    if (c->timing.enabled && cells > 0) {
        hipEvent_t e0 = nullptr, e1 = nullptr;
        AGAL_HIP(c, hipEventCreate(&e0));
        AGAL_HIP(c, hipEventCreate(&e1));
        hipExtLaunchKernelGGL(kern, dim3(grid), dim3(WG), 0, s, e0, e1, 0, a, b);
        AGAL_HIP(c, hipGetLastError());
        c->timing.ev_pairs.push_back(e0);
        c->timing.ev_pairs.push_back(e1);
        c->timing.fused_launches++;
        c->timing.fused_cells += cells;
    } else {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(WG), 0, s, a, b);
        AGAL_HIP(c, hipGetLastError());
    }
    return AGAL_OK;
}

// Two consecutive sub-steps of level L run as an in-place pair where they can: 3D, no linked blocks,
// every block of the level free of solid cells (its own and its neighbours') with mutual neighbour slots,
// so that each slot (row, cell) that the second sub-step touches belongs to one cell, and two rows of the
// pool within 32-bit byte offsets.  us per coarse step of D3Q19, in place / as fused steps, all else the same:
// one level of 36 x 20 x 28 7.0 / 8.4, of 128^3 58.9 / 62.5, 64^3 cavity with three levels 280 / 288 in
// FP32 and 205 / 213 in FP16, 128^3 cavity with four levels 11 210 / 12 000.
static inline bool inplace_ok(const Ctx *c, int L)
{
    return c->DIM == 3 && !c->links_on && L == c->MAX_LEVELS - 1 && c->n_ids[L] > 0 && c->n_general[L] == 0 &&
           2 * c->n_maxcells * (long long)c->tsize <= (1LL << 32);
}

#define AGAL_DISPATCH_Q(c, FN, T, S, ...)                                                  \
    do {                                                                                   \
        if ((c)->Q == 9) return FN<T, S, 9>(__VA_ARGS__);                                  \
        if ((c)->Q == 19) return FN<T, S, 19>(__VA_ARGS__);                                \
        if ((c)->Q == 27) return FN<T, S, 27>(__VA_ARGS__);                                \
    } while (0)
#define AGAL_DISPATCH(c, FN, ...)                                                          \
    do {                                                                                   \
        switch ((c)->precision) {                                                          \
            case AGAL_FP64: AGAL_DISPATCH_Q(c, FN, double, double, __VA_ARGS__); break;    \
            case AGAL_FP32: AGAL_DISPATCH_Q(c, FN, float, float, __VA_ARGS__); break;      \
            case AGAL_FP16: AGAL_DISPATCH_Q(c, FN, float, _Float16, __VA_ARGS__); break;   \
            case AGAL_BF16: AGAL_DISPATCH_Q(c, FN, float, bf16s, __VA_ARGS__); break;      \
        }                                                                                  \
        return AGAL_ERR_ARG;                                                               \
    } while (0)

}  // namespace agal
