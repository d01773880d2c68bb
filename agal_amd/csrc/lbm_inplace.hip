// lbm_inplace.hip -- the second sub-step of an in-place pair.
//
// Two consecutive sub-steps of one level without an exchange between them (the finest level's pair
// inside a coarse step; two steps of a single-level run) run in one population buffer instead of
// two (Bailey, Myre, Walsh, Lilja and Saar 2009, the "AA" pattern):
//   first   (even_step_3d)  every cell collides its own values and leaves f*_q in its own row pb(q);
//   second  (odd_step_3d)   cell x takes f_pb(q) from row q of cell x + c_q, where that cell's first
//           sub-step left it, collides, and puts f*_q back into the same slot (row q, cell x + c_q):
//           its streamed place.  A link without a neighbour block uses the cell's own row pb(q) both
//           times, which is the bounce-back.  Each slot is touched by one cell only, so the order of
//           wavefronts is free.
// After the pair the populations lie as after two fused steps, in the buffer they started in.  The
// first sub-step reads and writes whole rows of its block; a level that is too large for the 256 MB
// memory-side cache in two buffers may fit it in one, and the second buffer's pages stay untouched.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "lbm_device.hpp"

namespace agal {

template <typename S>
__device__ __forceinline__ S load_at(const S *row, unsigned byte_off)
{
    const auto *base = (const __attribute__((address_space(1))) char *)scalar_row(row);
    if constexpr (sizeof(S) == 2)
        return __builtin_bit_cast(S, *(const __attribute__((address_space(1))) uint16_t *)(base + byte_off));
    else
        return *(const __attribute__((address_space(1))) S *)(base + byte_off);
}

template <typename S>
__device__ __forceinline__ void store_at(S *row, unsigned byte_off, S v)
{
    auto *base = (__attribute__((address_space(1))) char *)(unsigned long long)scalar_row(row);
    if constexpr (sizeof(S) == 2)
        *(__attribute__((address_space(1))) uint16_t *)(base + byte_off) = __builtin_bit_cast(uint16_t, v);
    else
        *(__attribute__((address_space(1))) S *)(base + byte_off) = v;
}

// The wavefront's block.  The rows of a pair (q, pb(q)) are neighbours, so a link's slot is the scalar
// base of the pair's first row plus a 32-bit byte offset (the launcher sees to 2 rows <= 2^32 bytes),
// kept from the load for the store.  Where a neighbour is missing the offset is the cell's own place
// in row pb(q) (INTERIOR: none is).
template <typename T, typename S, int Q, int COLL, bool INTERIOR>
__device__ __forceinline__ void odd_block(const StepArgs<T, S> &a, int b, int t, int my_nb, bool onb, float *lds)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    constexpr int SH = sizeof(S) == 8 ? 3 : (sizeof(S) == 4 ? 2 : 1);
    const unsigned row_bytes = (unsigned)(a.ncm << SH), own = ((unsigned)b * 64u + (unsigned)t) << SH;
    const SlotOf<Q> slot(t);
    unsigned at[Q];
    T f[Q];
    f[0] = ST::dec(load_pop(scalar_row(a.A + (long long)b * 64) + t), (T)VS::w(0));
#pragma unroll
    for (int q = 1; q < Q; q++) {
        const bool upper = VS::pb(q) < q;
        const int nbk = __builtin_amdgcn_ds_bpermute(slot(q), my_nb);
        at[q] = ((unsigned)nbk << (6 + SH)) + cell_of_link<Q, SH>(t, q);
        if (upper) at[q] += row_bytes;
        if constexpr (!INTERIOR) at[q] = nbk < 0 ? (upper ? own : own + row_bytes) : at[q];
        f[VS::pb(q)] = ST::dec(load_at(a.A + (long long)(upper ? q - 1 : q) * a.ncm, at[q]), (T)VS::w(q));
    }
    T fs[Q];
    T rho, u, v, w;
    collide_block<T, S, Q, COLL>(a, f, fs, rho, u, v, w, false, lds);
    store_own(a.B + (long long)b * 64, t, ST::enc(fs[0], (T)VS::w(0)));
    if (!INTERIOR && onb) hook_links<T, S, Q>(a, fs, my_nb, t, u, v, w);
    bool failed = false;
#pragma unroll
    for (int q = 1; q < Q; q++) {
        const S e = ST::enc(fs[q], (T)VS::w(q));
        if (!VS::half(q)) failed = failed || !ST::positive(e, (T)VS::w(q));
        store_at(a.B + (long long)(VS::pb(q) < q ? q - 1 : q) * a.ncm, at[q], e);
    }
    if (failed) record_failed_guards<T, S, Q, false>(a, b, t);
}

// The second sub-step, one wavefront per block of the level, after the first one's failed links (and any
// other pending list) are resolved.
template <typename T, typename S, int Q, int COLL, bool FOLD>
__global__ __launch_bounds__(WG) void k_odd_step(StepArgs<T, S> a, FixupArgs<T, S> fa)
{
    constexpr bool MF = COLL == COLL_MFMA;
    constexpr int ROW = Store<T, S>::quantized ? 20 : 36;
    __shared__ __attribute__((aligned(16))) float s_mrt[MF ? (WG / 64) * 64 * ROW : 1];
    if constexpr (FOLD) resolve_pending<T, S, Q>(fa);
    const int wave = __builtin_amdgcn_readfirstlane(xcd_local_wg((int)gridDim.x) * (WG / 64) + (int)(threadIdx.x >> 6));
    if (wave >= a.n) return;  // whole wavefronts only
    const int t = threadIdx.x & 63;
    const int b = __builtin_amdgcn_readfirstlane(a.ids[wave]);
    const int my_nb = a.nbr_slot[(long long)b * 27 + (t < 27 ? t : 26)];
    const int interior = __builtin_amdgcn_readfirstlane(a.simple[b]) & 2;
    float *lds = MF ? s_mrt + (threadIdx.x >> 6) * 64 * ROW : nullptr;
    if (interior) {
        odd_block<T, S, Q, COLL, true>(a, b, t, my_nb, false, lds);
    } else {
        const int onb_u = __builtin_amdgcn_readfirstlane(a.onb[b]);
        odd_block<T, S, Q, COLL, false>(a, b, t, my_nb, onb_u == 1, lds);
    }
}

template <typename T, typename S, int Q>
static int odd_step_t(Ctx *c, int L)
{
    if constexpr (VelSet<Q>::DIM == 3) {
        const int n = c->n_ids[L], buf = c->cur[L];
        StepArgs<T, S> a = step_args<T, S, Q>(c, L, buf, VMODE_EVEN);  // B == A
        FixupArgs<T, S> fa;
        unsigned rmask = res_bit(L, buf), wmask = rmask;
        const int grid = ((n + WG / 64 - 1) / (WG / 64) + 7) / 8 * 8;  // a multiple of the XCD count
        if (int st = fold_fixups<T, S, Q>(c, grid, 1u << L, records_into(c, L, 0), fa, wmask)) return st;
        hipStream_t s = sched_begin(c, 0, rmask, wmask);
        const bool mrt = c->P.collision == AGAL_MRT;
        using K = void (*)(StepArgs<T, S>, FixupArgs<T, S>);
        K kern = mrt ? (fa.n ? (K)k_odd_step<T, S, Q, COLL_MRT, true> : (K)k_odd_step<T, S, Q, COLL_MRT, false>)
                     : (fa.n ? (K)k_odd_step<T, S, Q, COLL_BGK, true> : (K)k_odd_step<T, S, Q, COLL_BGK, false>);
        if constexpr (sizeof(T) == 4)
            if (mrt && c->mrt_mfma)
                kern = fa.n ? (K)k_odd_step<T, S, Q, COLL_MFMA, true> : (K)k_odd_step<T, S, Q, COLL_MFMA, false>;
        int st = launch_timed(c, kern, grid, s, (double)n * 64, a, fa);
        if (!st) st = sched_done(c, s, 0, rmask, wmask);
        c->leave_pending(L, buf, 0);
        return st;
    }
    return AGAL_ERR_ARG;
}

int launch_odd_step(Ctx *c, int L) { AGAL_DISPATCH(c, odd_step_t, c, L); }

}  // namespace agal
