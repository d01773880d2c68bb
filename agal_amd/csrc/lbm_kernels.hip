// lbm_kernels.hip -- the per-level LBM kernels for gfx950.
//
// One 64-lane wavefront owns one 4x4x4 cell-block (3D) or four 4x4 blocks (2D); a 256-thread
// workgroup therefore covers 4 (3D) or 16 (2D) blocks of a level's sorted ID list.
//
// The fused step replaces the reference's three passes Cu_Collide -> Cu_ImposeBC -> Cu_Stream
// (src/solver_lbm/solver_lbm_kernels.cu:204-289, 691-887, 532-633) by one read of the Q
// pre-collision populations of a cell and one write of its Q streamed populations into the other
// buffer (push).  The reference's in-place swap exchanges a link only when the initiating cell is
// not solid and the partner's post-collision value is > 0 (kernels.cu:624); the push reproduces
// that rule exactly:
//   - every cell computes its post-collision values f*_q (BGK for cells that collide; for cells
//     that do not -- solid cells and blocks that are solid with children -- the swap semantics
//     of the reference amount to f*_q = f_{pb(q)});
//   - the domain-face hook modifies f*_q on links that leave the domain (Cu_ImposeBC);
//   - a link (x -> x+c_h, h in the reference's half set) streams when x collides and the
//     partner's f*_{pb(h)} > 0; otherwise both ends bounce back into their own opposite slot.
//     The partner knows its value, the initiator does not: the initiator always pushes, and a
//     partner whose value fails the guard records the link in an exception list (normally empty) that
//     is resolved before anything else reads the level: by the next kernel, or by k_fixup.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "lbm_device.hpp"

namespace agal {

// ---------------------------------------------------------------------------------------------
// Initial conditions: Cu_SetInitialConditions (solver_lbm_kernels.cu:13-77), uniform state hook.
// ---------------------------------------------------------------------------------------------
template <typename T, typename S, int Q>
__global__ __launch_bounds__(WG) void k_set_ic(const int *__restrict__ ids, int n, S *__restrict__ F, long long ncm,
                                               const int *__restrict__ cells_mask, T rho, T u, T v, T w)
{
    using VS = VelSet<Q>;
    constexpr int CELLS = VS::CELLS;
    const int t = threadIdx.x % CELLS;
    const int bi = blockIdx.x * (WG / CELLS) + threadIdx.x / CELLS;
    if (bi >= n) return;
    const long long cell = (long long)ids[bi] * CELLS + t;
    const T udotu = u * u + v * v + w * w;
    const int m = cells_mask[cell];
#pragma unroll
    for (int p = 0; p < Q; p++) {
        T cdotu = cdot<T, Q>(p, u, v, w);
        T f = (T)(-1.0);
        if (m != CELL_SOLID) f = rho * (T)VS::w(p) * ((T)1.0 + (T)3.0 * cdotu + (T)4.5 * cdotu * cdotu - (T)1.5 * udotu);
        F[(long long)p * ncm + cell] = Store<T, S>::enc(f, (T)VS::w(p));
    }
}

template <typename T, typename S, int Q>
__global__ __launch_bounds__(WG) void k_refresh(const int *__restrict__ ids, int n, const S *__restrict__ F,
                                                T *__restrict__ M, long long ncm)
{
    using VS = VelSet<Q>;
    constexpr int CELLS = VS::CELLS;
    const int t = threadIdx.x % CELLS;
    const int bi = blockIdx.x * (WG / CELLS) + threadIdx.x / CELLS;
    if (bi >= n) return;
    const long long cell = (long long)ids[bi] * CELLS + t;
    T f[Q];
#pragma unroll
    for (int p = 0; p < Q; p++) f[p] = Store<T, S>::dec(F[(long long)p * ncm + cell], (T)VS::w(p));
    T rho, u, v, w;
    moments<T, Q>(f, rho, u, v, w);
    M[0 * ncm + cell] = rho;
    M[1 * ncm + cell] = u;
    M[2 * ncm + cell] = v;
    M[3 * ncm + cell] = (VS::DIM == 3) ? w : (T)0;
}

// ---------------------------------------------------------------------------------------------
// Coarse -> fine: Cu_Interpolate_Linear (solver_lbm_kernels_comm.cu:13-138).  The first CELLS
// lanes of each parent put the Q rescaled parent populations in LDS.  Then the lanes evaluate the
// children's cells: new children (ADDED) and the plane with one cell per lane in each half of the
// children (children c and c + NCH/2), row-contiguous stores; interface parents in 3D, where a
// quarter of the cells are ghost cells, with a list of those (GhostList).  Half-width groups keep a
// level's interface parents within one round of resident wavefronts (a 3D parent is one 256-lane
// workgroup; 2D packs eight 4x4 parents).
// ---------------------------------------------------------------------------------------------
constexpr int IWG = 256;

// Interpolation coefficients of the reference's trilinear (bilinear) form, per parent, child
// (octant) and direction: the corner differences that multiply 1, Ix, Iy, Iz, IxIy, IxIz, IyIz,
// IxIyIz (1, Ix, Iy, IxIy in 2D), formed once from the parent's rescaled populations s (rows of
// `stride` per direction) with the reference's operand order, instead of once per child cell.
template <typename T, int Q>
struct InterpCoef {
    static constexpr int DIM = VelSet<Q>::DIM, NCH = VelSet<Q>::CHILDREN, N = DIM == 3 ? 8 : 4;
};

// Fills coef[(g * Q + p) * NCH + c][0..N) for the PPW parents of the workgroup (tasks strided over
// the workgroup's lanes).
template <typename T, int Q, int PPW, int NTHR>
__device__ __forceinline__ void interp_coefficients(const T *s_all, T *coef)
{
    using IC = InterpCoef<T, Q>;
    constexpr int CELLS = VelSet<Q>::CELLS, NCH = IC::NCH, N = IC::N;
    for (int task = threadIdx.x; task < PPW * Q * NCH; task += NTHR) {
        const int c = task % NCH, p = (task / NCH) % Q, g = task / (NCH * Q);
        const T *s = s_all + p * PPW * CELLS + g * CELLS;
        const int ci = c % 2, cj = (c / 2) % 2, ck = (c / 4) % 2;
        T *a = coef + (long long)task * N;
        if (IC::DIM == 2) {
            const int o = 2 * ci + 2 * 4 * cj;
            a[0] = s[0 + o];
            a[1] = s[1 + o] - s[0 + o];
            a[2] = s[4 + o] - s[0 + o];
            a[3] = s[5 + o] - s[4 + o] - s[1 + o] + s[0 + o];
        } else {
            const int o = 2 * ci + 2 * 4 * cj + 2 * 4 * 4 * ck;
            a[0] = s[0 + o];
            a[1] = s[1 + o] - s[0 + o];
            a[2] = s[4 + o] - s[0 + o];
            a[3] = s[16 + o] - s[0 + o];
            a[4] = s[5 + o] - s[1 + o] - s[4 + o] + s[0 + o];
            a[5] = s[17 + o] - s[1 + o] - s[16 + o] + s[0 + o];
            a[6] = s[20 + o] - s[4 + o] - s[16 + o] + s[0 + o];
            a[7] = s[21 + o] + s[1 + o] + s[4 + o] + s[16 + o] - s[5 + o] - s[17 + o] - s[20 + o] - s[0 + o];
        }
    }
}

// Value at child c's cell t in the reference's operation order (Cu_Interpolate_Linear,
// solver_lbm_kernels_comm.cu:13-138): s0 + a1 Ix + a2 Iy + a3 Iz + a4 Ix Iy + ... summed left to
// right, each product formed left to right; stored into every row.
template <typename T, typename S, int Q>
__device__ __forceinline__ void interp_child(const T *coef_g, int c, int t, S *__restrict__ Fc, long long ncm,
                                             long long ccell)
{
    using VS = VelSet<Q>;
    using IC = InterpCoef<T, Q>;
    constexpr int DIM = VS::DIM, NCH = IC::NCH, N = IC::N;
    const int I = t % 4, J = (t / 4) % 4, K = (DIM == 3) ? t / 16 : 0;
    const T Ix = (T)(-0.25) + (T)(0.5) * (T)I;
    const T Iy = (T)(-0.25) + (T)(0.5) * (T)J;
    const T Iz = (DIM == 3) ? (T)(-0.25) + (T)(0.5) * (T)K : (T)0;
#pragma unroll
    for (int p = 0; p < Q; p++) {
        const T *a = coef_g + (p * NCH + c) * N;
        T val;
        if (DIM == 2)
            val = a[0] + a[1] * Ix + a[2] * Iy + a[3] * Ix * Iy;
        else
            val = a[0] + a[1] * Ix + a[2] * Iy + a[3] * Iz + a[4] * Ix * Iy + a[5] * Ix * Iz + a[6] * Iy * Iz +
                  a[7] * Ix * Iy * Iz;
        Fc[(long long)p * ncm + ccell] = Store<T, S>::enc(val, (T)VS::w(p));
    }
}

// Arguments of the linear interpolation of one level's parent list into the children.
template <typename T, typename S>
struct InterpArgs {
    const int *ids;
    int n;
    const S *Fp;
    S *Fc;
    long long ncm;
    const int *nbr_child, *blk_mask, *ref, *cells_mask;
    T tau_ratio;
};

template <typename T, int Q>
struct InterpLds {  // LDS of one interpolation workgroup
    static constexpr int CELLS = VelSet<Q>::CELLS, NCH = VelSet<Q>::CHILDREN;
    static constexpr int PPW = IWG / (NCH / 2 * CELLS);
    static constexpr int ALL = Q * PPW * CELLS, COEF = PPW * Q * NCH * InterpCoef<T, Q>::N;
};

// The ghost cells of a 3D parent's children (512 cells, of which an interface block typically has 128),
// listed in LDS, so that the interpolation's lanes take one ghost cell each instead of two cells each
// that may or may not be one.  The workgroup's four wavefronts call ghost_masks before, ghost_list after
// one barrier, and read the list after another.
struct GhostList {
    unsigned long long mask[8];  // per child
    unsigned short cell[512];    // child * 64 + cell, `total` of them
};

__device__ __forceinline__ void ghost_masks(GhostList &g, const int *__restrict__ cells_mask, int fc, bool work)
{
    const int c = threadIdx.x >> 6, t = threadIdx.x & 63;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const bool put = work && cells_mask[(long long)(fc + c + 4 * h) * 64 + t] == CELL_GHOST;
        const unsigned long long m = __ballot(put);
        if (t == 0) g.mask[c + 4 * h] = m;
    }
}

__device__ __forceinline__ int ghost_list(GhostList &g)
{
    const int c = threadIdx.x >> 6, t = threadIdx.x & 63;
    int total = 0, off[2] = {0, 0};
#pragma unroll
    for (int k = 0; k < 8; k++) {
        if (k == c) off[0] = total;
        if (k == c + 4) off[1] = total;
        total += __popcll(g.mask[k]);
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const unsigned long long m = g.mask[c + 4 * h];
        if ((m >> t) & 1) g.cell[off[h] + __popcll(m & ((1ull << t) - 1))] = (unsigned short)((c + 4 * h) * 64 + t);
    }
    return total;
}

// Workgroup `wg` of the interpolation (IWG threads): its parents, their children's cells.
template <typename T, typename S, int Q, bool ADDED>
__device__ __forceinline__ void interp_parents(const InterpArgs<T, S> &ia, int wg, T *s_all, T *s_coef, GhostList &s_ghost)
{
    using VS = VelSet<Q>;
    constexpr int CELLS = VS::CELLS, NCH = VS::CHILDREN, HALF = NCH / 2;
    constexpr int GROUP = HALF * CELLS;  // lanes per parent: one per cell of half the children
    constexpr int PPW = IWG / GROUP;     // parents per workgroup
    constexpr int NCOEF = InterpCoef<T, Q>::N;
    const long long ncm = ia.ncm;
    const int g = threadIdx.x / GROUP, r = threadIdx.x % GROUP;
    const int c = r / CELLS, t = r % CELLS;
    const int bi = wg * PPW + g;
    int b = -1;
    if (bi < ia.n) b = ia.ids[bi];
    bool work = false;
    int fc = 0;
    if (b >= 0) {
        fc = ia.nbr_child[b];
        work = fc >= 0 && (ADDED ? (ia.ref[b] == REF_MARK_REFINE) : (ia.blk_mask[b] == BLK_INTERFACE));
    }
    // The children's cell masks, fetched before the barrier.
    constexpr bool LIST = VS::DIM == 3 && !ADDED;
    bool put[2] = {false, false};
    if constexpr (LIST)
        ghost_masks(s_ghost, ia.cells_mask, fc, work);
    else if (work)
#pragma unroll
        for (int h = 0; h < 2; h++)
            put[h] = ADDED || ia.cells_mask[(long long)(fc + c + h * HALF) * CELLS + t] == CELL_GHOST;
    T *sg = s_all + g * CELLS;
    if (work && c == 0) {
        const long long cell = (long long)b * CELLS + t;
        T f[Q];
#pragma unroll
        for (int p = 0; p < Q; p++) f[p] = Store<T, S>::dec(ia.Fp[(long long)p * ncm + cell], (T)VS::w(p));
        T rho, u, v, w;
        moments<T, Q>(f, rho, u, v, w);
        const T udotu = u * u + v * v + w * w;
#pragma unroll
        for (int p = 0; p < Q; p++) {
            T cdotu = cdot<T, Q>(p, u, v, w);
            T fe = (T)VS::w(p) * rho * ((T)(1.0) + (T)(3.0) * cdotu + (T)(4.5) * cdotu * cdotu - (T)(1.5) * udotu);
            sg[p * PPW * CELLS + t] = fe + (f[p] - fe) * ia.tau_ratio;
        }
    }
    __syncthreads();
    int total = 0;
    if constexpr (LIST) total = ghost_list(s_ghost);
    interp_coefficients<T, Q, PPW, IWG>(s_all, s_coef);
    __syncthreads();
    if (!work) return;
    if constexpr (LIST) {
        for (int k = threadIdx.x; k < total; k += IWG) {
            const int e = s_ghost.cell[k];
            interp_child<T, S, Q>(s_coef, e >> 6, e & 63, ia.Fc, ncm, (long long)fc * 64 + e);
        }
        return;
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
        if (put[h])
            interp_child<T, S, Q>(s_coef + g * Q * NCH * NCOEF, c + h * HALF, t, ia.Fc, ncm,
                                  (long long)(fc + c + h * HALF) * CELLS + t);
}

template <typename T, typename S, int Q, bool ADDED>
__global__ __launch_bounds__(IWG) void k_interp(InterpArgs<T, S> ia)
{
    using IL = InterpLds<T, Q>;
    __shared__ T s_all[IL::ALL];
    __shared__ T s_coef[IL::COEF];
    __shared__ GhostList s_ghost;
    interp_parents<T, S, Q, ADDED>(ia, blockIdx.x, s_all, s_coef, s_ghost);
}

// Sum over the NG lanes of each lane group (NG consecutive lanes, NG = 8 in 3D, 4 in 2D) of the
// values v[p], left to right in lane order as the reference sums the children (comm.cu:330-339),
// for the directions p = k (mod NG) of lane k of the group: the wavefront writes its Q x 64 values
// to its own LDS rows (stride 65: the group reads fall in distinct banks) and each lane reads back
// the NG values of its own directions.  `lds` is this wavefront's Q * 65-float region.
template <typename T, int Q, int NG>
__device__ __forceinline__ void group_sums(const T *v, T *acc, T *lds)
{
    const int lane = threadIdx.x & 63, k = lane % NG, gl = lane - k;
    wave_lds_sync();  // earlier reads of this region are done
#pragma unroll
    for (int p = 0; p < Q; p++) lds[p * 65 + lane] = v[p];
    wave_lds_sync();
#pragma unroll
    for (int m = 0; m < (Q + NG - 1) / NG; m++) {
        const int p = k + NG * m;
        if (p < Q) {
            const T *row = lds + p * 65 + gl;
            T a = row[0];
#pragma unroll
            for (int j = 1; j < NG; j++) a = a + row[j];
            acc[m] = a;
        }
    }
}

// Average of one 3D parent block by a workgroup of four wavefronts (Cu_Average, solver_lbm_kernels_comm.cu:
// 174-347).  Eight consecutive lanes serve one parent cell, each lane loading and rescaling one child
// cell of its 2x2x2 group; the sum is formed in the reference's order (group_sums) and each lane hands
// the directions p = lane (mod 8) to put(t, p, value).  Every wavefront finds the parent cells that are
// averaged (their first child cell is an interface cell; ave_type > 0: is not a ghost) with one load and
// a ballot and deals them out in eights, so lanes are not spent on the others: an interface block has
// typically 16 of its 64 cells averaged.  Returns the mask of the averaged cells.
template <typename T, typename S, int Q, class Put>
__device__ __forceinline__ unsigned long long average_block_3d(const S *Fc, long long ncm, const int *__restrict__ cells_mask,
                                                               int fc, int ave_type, T ratio, T *s_red, Put put)
{
    using VS = VelSet<Q>;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, k = lane & 7;
    // First child cell of parent cell t.
    auto first = [&](int t) {
        const int I = t & 3, J = (t >> 2) & 3, K = t >> 4;
        const int c = (I >> 1) + 2 * (J >> 1) + 4 * (K >> 1);
        return (long long)(fc + c) * 64 + 2 * (I & 1) + 8 * (J & 1) + 32 * (K & 1);
    };
    int m = cells_mask[first(lane)];
    if (ave_type > 0 && m < 2) m = 1;
    const unsigned long long done = __ballot(m == 1);
    const int cnt = __popcll(done);
    // Lane r of `list`: the r-th averaged cell.  (Lanes of the others send beyond them.)
    const int rank = __popcll(done & ((1ull << lane) - 1));
    const int list = __builtin_amdgcn_ds_permute(4 * (m == 1 ? rank : cnt + lane - rank), lane);
    for (int n0 = 8 * wv; n0 < cnt; n0 += 32) {
        const int r = n0 + (lane >> 3);
        const int t = __shfl(list, r < cnt ? r : n0, 64);
        T s[Q];
        const long long cell = first(t) + (k & 1) + 4 * ((k >> 1) & 1) + 16 * (k >> 2);
#pragma unroll
        for (int p = 0; p < Q; p++) s[p] = Store<T, S>::dec(Fc[(long long)p * ncm + cell], (T)VS::w(p));
        T rho, u, v, w;
        moments<T, Q>(s, rho, u, v, w);
        const T udotu = u * u + v * v + w * w;
#pragma unroll
        for (int p = 0; p < Q; p++) {
            T cdotu = cdot<T, Q>(p, u, v, w);
            T fe = (T)VS::w(p) * rho * ((T)(1.0) + (T)(3.0) * cdotu + (T)(4.5) * cdotu * cdotu - (T)(1.5) * udotu);
            s[p] = fe + (s[p] - fe) * ratio;
        }
        T acc[(Q + 7) / 8];
        group_sums<T, Q, 8>(s, acc, s_red + wv * Q * 65);
#pragma unroll
        for (int j = 0; j < (Q + 7) / 8; j++) {
            const int p = k + 8 * j;
            if (r < cnt && p < Q) put(t, p, (T)(0.125) * acc[j]);
        }
    }
    return done;
}

// ---------------------------------------------------------------------------------------------
// Fine -> coarse then coarse -> fine in one launch: the pair "average(L) in INTERFACE mode, then
// linear interpolation(L) in INTERFACE mode" that the advance runs between the two sub-cycles of
// level L+1 (solver_lbm_advance.cu:108-112).  Both act on the INTERFACE parents of level L, and each
// reads and writes only one parent block and its children: the average writes parent cells whose
// first child cell is an interface cell (mask 1), the interpolation reads the parent block and
// writes the children's ghost cells (mask 2).  A workgroup therefore does both for its parents:
// the averaged values go to the pool and, as the pool will hold them, to LDS, from where the
// interpolation stage takes them.  Arithmetic and order are those of k_average and k_interp.
// D3Q19 FP32, 3008 parents: 35 -> 32 us with the averaged cells and the ghost cells found by ballots and
// dealt to the lanes (bound by scattered lines: both sets use a part of each).
// ---------------------------------------------------------------------------------------------
template <typename T, typename S, int Q, bool FOLD>
__global__ __launch_bounds__(IWG) void k_avg_interp(FixupArgs<T, S> fa, const int *__restrict__ ids, int n, S *Fp, S *Fc,
                                                    long long ncm, const int *__restrict__ nbr_child,
                                                    const int *__restrict__ blk_mask, const int *__restrict__ cells_mask,
                                                    T ratio_avg, T ratio_int)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    if constexpr (FOLD) resolve_pending<T, S, Q>(fa);
    constexpr int CELLS = VS::CELLS, DIM = VS::DIM, NCH = VS::CHILDREN, HALF = NCH / 2;
    constexpr int GROUP = HALF * CELLS;  // lanes per parent
    constexpr int PPW = IWG / GROUP;     // parents per workgroup
    constexpr int NCOEF = InterpCoef<T, Q>::N;
    // The averaging stage's group-sum rows and the interpolation stage's rescaled parent and
    // coefficients share one region (a barrier separates the stages).
    constexpr int RED = (IWG / 64) * Q * 65, INTERP = Q * PPW * CELLS + PPW * Q * NCH * NCOEF;
    __shared__ T s_stage[RED > INTERP ? RED : INTERP];
    __shared__ T s_avg[Q * PPW * CELLS];  // averaged parent populations as stored
    __shared__ int s_done[PPW * CELLS];   // parent cell was averaged
    T *const s_red = s_stage;                        // per-wavefront rows of the group sums
    T *const s_all = s_stage;                        // rescaled parent populations for the interpolation
    T *const s_coef = s_stage + Q * PPW * CELLS;     // interpolation coefficients
    const int g = threadIdx.x / GROUP, r = threadIdx.x % GROUP;
    const int bi = blockIdx.x * PPW + g;
    int b = -1;
    if (bi < n) b = ids[bi];
    int fc = -1;
    bool work = false;
    if (b >= 0) {
        fc = nbr_child[b];
        work = fc >= 0 && blk_mask[b] == BLK_INTERFACE;
    }
    // ---- average (k_average) ----
    if constexpr (DIM == 3) {
        if (work) {  // the same for the whole workgroup
            const unsigned long long done = average_block_3d<T, S, Q>(
                Fc, ncm, cells_mask, fc, 0, ratio_avg, s_red, [&](int ta, int p, T v) {
                    const T wq = (T)VelSet<Q>::w(p);
                    const S enc = ST::enc(v, wq);
                    Fp[(long long)p * ncm + (long long)b * CELLS + ta] = enc;
                    s_avg[p * CELLS + ta] = ST::dec(enc, wq);
                });
            if (threadIdx.x < CELLS) s_done[threadIdx.x] = (int)((done >> threadIdx.x) & 1);
        }
    } else {
        const int k = r % NCH, ta0 = r / NCH;  // parent cells ta0 and ta0 + CELLS / 2
        const int off = (k & 1) + 4 * (k >> 1);
        bool avg[2];
        long long cb[2];
        int c0[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int ta = ta0 + h * (CELLS / 2);
            const int I = ta % 4, J = ta / 4;
            const int cq = (I / 2) + 2 * (J / 2);
            c0[h] = 2 * (I % 2) + 4 * (2 * (J % 2));
            cb[h] = (long long)(fc + cq) * CELLS;
            avg[h] = work && cells_mask[cb[h] + c0[h]] == 1;  // uniform over the NCH lanes of the group
        }
        T fl[2][Q];
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (avg[h])
#pragma unroll
                for (int p = 0; p < Q; p++) fl[h][p] = ST::dec(Fc[(long long)p * ncm + cb[h] + c0[h] + off], (T)VS::w(p));
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int ta = ta0 + h * (CELLS / 2);
            T sv[Q];
            if (avg[h]) {
                const T *f = fl[h];
                T rho, u, v, w;
                moments<T, Q>(f, rho, u, v, w);
                const T udotu = u * u + v * v;
#pragma unroll
                for (int p = 0; p < Q; p++) {
                    T cdotu = cdot<T, Q>(p, u, v, w);
                    T fe = (T)VS::w(p) * rho * ((T)(1.0) + (T)(3.0) * cdotu + (T)(4.5) * cdotu * cdotu - (T)(1.5) * udotu);
                    sv[p] = fe + (f[p] - fe) * ratio_avg;
                }
            } else {
#pragma unroll
                for (int p = 0; p < Q; p++) sv[p] = (T)0;
            }
            const long long pcell = (long long)b * CELLS + ta;
            T acc[(Q + NCH - 1) / NCH];
            group_sums<T, Q, NCH>(sv, acc, s_red + (threadIdx.x >> 6) * Q * 65);
#pragma unroll
            for (int m = 0; m < (Q + NCH - 1) / NCH; m++) {
                const int p = k + NCH * m;
                if (avg[h] && p < Q) {
                    const T wq = (T)VelSet<Q>::w(p);
                    const S enc = ST::enc((T)(0.25) * acc[m], wq);
                    Fp[(long long)p * ncm + pcell] = enc;
                    s_avg[p * PPW * CELLS + g * CELLS + ta] = ST::dec(enc, wq);
                }
            }
            if (k == 0) s_done[g * CELLS + ta] = avg[h] ? 1 : 0;
        }
    }
    // The children's cell masks for the interpolation stage, fetched before the barrier.
    __shared__ GhostList s_ghost;
    const int c = r / CELLS, t = r % CELLS;
    bool put[2] = {false, false};
    if constexpr (DIM == 3)
        ghost_masks(s_ghost, cells_mask, fc, work);
    else if (work)
#pragma unroll
        for (int h = 0; h < 2; h++) put[h] = cells_mask[(long long)(fc + c + h * HALF) * CELLS + t] == CELL_GHOST;
    __syncthreads();
    // ---- interpolation: parent rescaled into LDS, then two child cells per lane (k_interp) ----
    T *sg = s_all + g * CELLS;
    if (work && c == 0) {
        const long long cell = (long long)b * CELLS + t;
        const bool done = s_done[g * CELLS + t] != 0;
        T f[Q];
#pragma unroll
        for (int p = 0; p < Q; p++)
            f[p] = done ? s_avg[p * PPW * CELLS + g * CELLS + t] : ST::dec(Fp[(long long)p * ncm + cell], (T)VS::w(p));
        T rho, u, v, w;
        moments<T, Q>(f, rho, u, v, w);
        const T udotu = u * u + v * v + w * w;
#pragma unroll
        for (int p = 0; p < Q; p++) {
            T cdotu = cdot<T, Q>(p, u, v, w);
            T fe = (T)VS::w(p) * rho * ((T)(1.0) + (T)(3.0) * cdotu + (T)(4.5) * cdotu * cdotu - (T)(1.5) * udotu);
            sg[p * PPW * CELLS + t] = fe + (f[p] - fe) * ratio_int;
        }
    }
    int total = 0;
    if constexpr (DIM == 3) total = ghost_list(s_ghost);
    __syncthreads();
    interp_coefficients<T, Q, PPW, IWG>(s_all, s_coef);
    __syncthreads();
    if (!work) return;
    if constexpr (DIM == 3) {
        for (int e = threadIdx.x; e < total; e += IWG) {
            const int x = s_ghost.cell[e];
            interp_child<T, S, Q>(s_coef, x >> 6, x & 63, Fc, ncm, (long long)fc * CELLS + x);
        }
        return;
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
        if (put[h])
            interp_child<T, S, Q>(s_coef + g * Q * NCH * NCOEF, c + h * HALF, t, Fc, ncm,
                                  (long long)(fc + c + h * HALF) * CELLS + t);
}

// ---------------------------------------------------------------------------------------------
// Coarse -> fine, cubic: Cu_Interpolate_Cubic (solver_lbm_kernels_comm.cu:406-638).  Per parent
// and direction the 4^d monomial coefficients alpha_i = sum_q C[i][q] s[q] of the tensor-product
// Lagrange interpolant through the parent's cells are formed once (the reference's coefficient
// tables, summed term by term in its order) and kept in LDS; the child cells evaluate the polynomial
// by Horner's rule in x, then y, then z.
// ---------------------------------------------------------------------------------------------
#define AGAL_CUBIC_TABLE __constant__ static const
#include "cubic_table.inc"
#undef AGAL_CUBIC_TABLE

constexpr int CWG = 512;  // threads of a cubic interpolation workgroup

// Rescaled populations feq + (f - feq) ratio of one parent cell.
template <typename T, typename S, int Q>
__device__ __forceinline__ void rescaled_parent(const S *__restrict__ Fp, long long ncm, long long cell, T ratio, T *s)
{
    using VS = VelSet<Q>;
    T f[Q];
#pragma unroll
    for (int p = 0; p < Q; p++) f[p] = Store<T, S>::dec(Fp[(long long)p * ncm + cell], (T)VS::w(p));
    T rho, u, v, w;
    moments<T, Q>(f, rho, u, v, w);
    const T udotu = u * u + v * v + w * w;
#pragma unroll
    for (int p = 0; p < Q; p++) {
        T cdotu = cdot<T, Q>(p, u, v, w);
        T fe = (T)VS::w(p) * rho * ((T)(1.0) + (T)(3.0) * cdotu + (T)(4.5) * cdotu * cdotu - (T)(1.5) * udotu);
        s[p] = fe + (f[p] - fe) * ratio;
    }
}

// Coordinate of a child cell along one axis in the polynomial's variable: cell 0..7 of the children's
// row, the second child offset by 2/3.
template <typename T>
__device__ __forceinline__ T cubic_coord(int k)
{
    const T x = (T)(-0.083333333333333) + (T)(0.166666666666667) * (T)(k & 3);
    return x + ((k & 4) ? (T)(0.666666666666667) : (T)(0.0));
}

// 2D: one lane per child cell, eight 4x4 parents per workgroup.
template <typename T, typename S, int Q, bool ADDED>
__device__ __forceinline__ void interp_cubic_2d(const InterpArgs<T, S> &ia)
{
    using VS = VelSet<Q>;
    constexpr int CELLS = VS::CELLS, NCH = VS::CHILDREN;
    constexpr int GROUP = NCH * CELLS;
    constexpr int PPW = CWG / GROUP;
    __shared__ T s_all[Q * PPW * CELLS];  // rescaled parent populations, [p][parent][cell]
    __shared__ T a_all[Q * PPW * CELLS];  // monomial coefficients, [p][parent][i]
    const int g = threadIdx.x / GROUP, r = threadIdx.x % GROUP;
    const int c = r / CELLS, t = r % CELLS;
    const int bi = blockIdx.x * PPW + g;
    int b = -1;
    if (bi < ia.n) b = ia.ids[bi];
    bool work = false;
    int fc = 0;
    if (b >= 0) {
        fc = ia.nbr_child[b];
        work = fc >= 0 && (ADDED ? (ia.ref[b] == REF_MARK_REFINE) : (ia.blk_mask[b] == BLK_INTERFACE));
    }
    if (work && c == 0) {
        T s[Q];
        rescaled_parent<T, S, Q>(ia.Fp, ia.ncm, (long long)b * CELLS + t, ia.tau_ratio, s);
#pragma unroll
        for (int p = 0; p < Q; p++) s_all[(p * PPW + g) * CELLS + t] = s[p];
    }
    __syncthreads();
    if (work) {
        for (int k = r; k < Q * CELLS; k += GROUP) {
            const int p = k / CELLS, i = k % CELLS;
            const T *s = s_all + (p * PPW + g) * CELLS;
            T acc = (T)CUBIC2_C[CUBIC2_START[i]] * s[CUBIC2_Q[CUBIC2_START[i]]];
            for (int m = CUBIC2_START[i] + 1; m < CUBIC2_START[i + 1]; m++) acc = acc + (T)CUBIC2_C[m] * s[CUBIC2_Q[m]];
            a_all[(p * PPW + g) * CELLS + i] = acc;
        }
    }
    __syncthreads();
    if (!work) return;
    const long long ccell = (long long)(fc + c) * CELLS + t;
    if (!ADDED && ia.cells_mask[ccell] != CELL_GHOST) return;
    const T x = cubic_coord<T>((t & 3) + 4 * (c & 1)), y = cubic_coord<T>((t >> 2) + 4 * (c >> 1));
#pragma unroll 1
    for (int p = 0; p < Q; p++) {
        const T *al = a_all + (p * PPW + g) * CELLS;
        T res = 0;
#pragma unroll
        for (int mj = 0; mj < 4; mj++) {
            T beta = 0;
#pragma unroll
            for (int mi = 0; mi < 4; mi++) beta = al[(3 - mi) + 4 * (3 - mj)] + x * beta;
            res = beta + y * res;
        }
        ia.Fc[(long long)p * ia.ncm + ccell] = Store<T, S>::enc(res, (T)VS::w(p));
    }
}

// 3D: one workgroup of eight wavefronts per parent.  The coefficients: lane (p, g) of a wavefront
// forms alpha_i of direction p for one of G = 64 / Q indices i at a time, the indices dealt out by
// falling number of terms (64, 16, 4 or 1), so a wavefront's lanes run chains of equal length and
// their LDS reads s[q][p] fall in consecutive banks.  The values: a wavefront takes one direction,
// lane (x, y) of the children's 8 x 8 columns forms the four z-coefficients once (Horner in x, then
// y) and runs down the eight z: 14 multiply-adds per child cell instead of 84, each the same
// operation on the same operands.  FP64 vector issue and LDS latency bound it.  Three levels on a
// 32^3 root in FP64 (launches of 176 and 736 parents): 28.8 us a launch, 130 us with one lane per
// child cell.
struct CubicOrder {
    unsigned char i[64];
};
constexpr CubicOrder make_cubic_order()
{
    CubicOrder o{};
    int n = 0;
    for (int nz = 3; nz >= 0; nz--)  // an index has 4 terms for every nonzero digit (power of x, y, z)
        for (int i = 0; i < 64; i++)
            if ((i % 4 != 0) + (i / 4 % 4 != 0) + (i / 16 != 0) == nz) o.i[n++] = (unsigned char)i;
    return o;
}
__constant__ const CubicOrder kCubicOrder = make_cubic_order();

template <typename T, typename S, int Q, bool ADDED>
__device__ __forceinline__ void interp_cubic_3d(const InterpArgs<T, S> &ia)
{
    using VS = VelSet<Q>;
    constexpr int NW = CWG / 64, G = 64 / Q, AL = 66;
    __shared__ T s_par[64 * Q];   // rescaled parent populations, [cell][p]
    __shared__ __attribute__((aligned(16))) T s_al[Q * AL];  // monomial coefficients, [p][i]
    const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int b = ia.ids[blockIdx.x];
    const int fc = ia.nbr_child[b];
    // The same for the whole workgroup.
    if (fc < 0 || !(ADDED ? (ia.ref[b] == REF_MARK_REFINE) : (ia.blk_mask[b] == BLK_INTERFACE))) return;
    if (wv == 0) {
        T s[Q];
        rescaled_parent<T, S, Q>(ia.Fp, ia.ncm, (long long)b * 64 + l, ia.tau_ratio, s);
#pragma unroll
        for (int p = 0; p < Q; p++) s_par[l * Q + p] = s[p];
    }
    // This lane's column of child cells, and which of them are written (bit z).
    const int cx = l & 7, cy = l >> 3;
    const long long col = (long long)(fc + (cx >> 2) + 2 * (cy >> 2)) * 64 + (cx & 3) + 4 * (cy & 3);
    unsigned put = 0xffu;
    if (!ADDED) {
        put = 0;
#pragma unroll
        for (int z = 0; z < 8; z++)
            put |= (ia.cells_mask[col + (z >> 2) * 256 + (z & 3) * 16] == CELL_GHOST ? 1u : 0u) << z;
    }
    __syncthreads();
    const int p1 = l % Q, g = l / Q;
    for (int k = wv; k < (64 + G - 1) / G; k += NW) {
        const int at = k * G + g;
        if (g >= G || at >= 64) continue;
        const int i = kCubicOrder.i[at], m0 = CUBIC3_START[i], m1 = CUBIC3_START[i + 1];
        const T *s = s_par + p1;
        T acc = (T)CUBIC3_C[m0] * s[CUBIC3_Q[m0] * Q];
#pragma unroll 8
        for (int m = m0 + 1; m < m1; m++) acc = acc + (T)CUBIC3_C[m] * s[CUBIC3_Q[m] * Q];
        s_al[p1 * AL + i] = acc;
    }
    __syncthreads();
    const T x = cubic_coord<T>(cx), y = cubic_coord<T>(cy);
#pragma unroll 1
    for (int p = wv; p < Q; p += NW) {
        const T *al = s_al + p * AL;
        T gam[4];
#pragma unroll
        for (int mk = 0; mk < 4; mk++) {
            T gm = 0;
#pragma unroll
            for (int mj = 0; mj < 4; mj++) {
                T beta = 0;
#pragma unroll
                for (int mi = 0; mi < 4; mi++) beta = al[(3 - mi) + 4 * (3 - mj) + 16 * (3 - mk)] + x * beta;
                gm = beta + y * gm;
            }
            gam[mk] = gm;
        }
        // The direction is the same on the whole wavefront: a constant weight per branch.
        T wp = 0;
#pragma unroll
        for (int q = 0; q < Q; q++)
            if (q == p) wp = (T)VS::w(q);
        S *row = ia.Fc + (long long)p * ia.ncm + col;
#pragma unroll
        for (int z = 0; z < 8; z++) {
            const T zz = cubic_coord<T>(z);
            T res = 0;
#pragma unroll
            for (int mk = 0; mk < 4; mk++) res = gam[mk] + zz * res;
            if ((put >> z) & 1) row[(z >> 2) * 256 + (z & 3) * 16] = Store<T, S>::enc(res, wp);
        }
    }
}

template <typename T, typename S, int Q, bool ADDED>
__global__ __launch_bounds__(CWG) void k_interp_cubic(InterpArgs<T, S> ia)
{
    if constexpr (VelSet<Q>::DIM == 3)
        interp_cubic_3d<T, S, Q, ADDED>(ia);
    else
        interp_cubic_2d<T, S, Q, ADDED>(ia);
}

// ---------------------------------------------------------------------------------------------
// Fine -> coarse: Cu_Average (solver_lbm_kernels_comm.cu:174-347).  3D: one workgroup per parent block
// (average_block_3d), bound by the children's interface cells, 1/8 of every row's lines used; finding the
// averaged cells by a ballot instead of serving all 64: 17.6 -> 14.2 us for 3008 parents, 8.3 -> 6.0 us
// for 736, 300 -> 284 us for 48 896 (D3Q19 FP32).  2D: NG = 4 consecutive lanes serve one parent cell, each
// lane loading and rescaling one child cell of the cell's 2x2 group; the group sum is formed in the
// reference's order from the NG lanes by shuffles and each lane stores the directions p = lane (mod NG).
// Each lane group serves two parent cells (t and t + CELLS/2, both loaded before either is reduced), which
// halves the wavefronts per parent.
// ---------------------------------------------------------------------------------------------
template <typename T, typename S, int Q, bool FOLD>
__global__ __launch_bounds__(WG) void k_average(FixupArgs<T, S> fa, const int *__restrict__ ids, int n, S *Fp,
                                                const S *Fc, long long ncm, const int *__restrict__ nbr_child,
                                                const int *__restrict__ blk_mask, const int *__restrict__ cells_mask,
                                                int ave_type, T tau_ratio)
{
    using VS = VelSet<Q>;
    if constexpr (FOLD) resolve_pending<T, S, Q>(fa);
    constexpr int CELLS = VS::CELLS;
    __shared__ T s_red[(WG / 64) * Q * 65];  // per-wavefront rows of the group sums
    if constexpr (VS::DIM == 3) {
        const int pb = ids[blockIdx.x], pfc = nbr_child[pb];
        // The same for the whole workgroup.
        if (pfc < 0 || !(ave_type == 2 || blk_mask[pb] == BLK_INTERFACE)) return;
        average_block_3d<T, S, Q>(Fc, ncm, cells_mask, pfc, ave_type, tau_ratio, s_red, [&](int t, int p, T v) {
            Fp[(long long)p * ncm + (long long)pb * CELLS + t] = Store<T, S>::enc(v, (T)VelSet<Q>::w(p));
        });
    } else {
        constexpr int NG = 4;                      // child cells per parent cell
        constexpr int PER_BLOCK = CELLS / 2 * NG;  // lanes per parent block: two parent cells per lane group
        const int k = threadIdx.x % NG;            // which child cell of the group
        const long long gid = (long long)blockIdx.x * WG + threadIdx.x;
        const long long bi = gid / PER_BLOCK;
        const int t0 = (int)((gid % PER_BLOCK) / NG);  // parent cells t0 and t0 + CELLS / 2
        bool work = bi < n;
        int b = 0, fc = -1;
        if (work) {
            b = ids[bi];
            fc = nbr_child[b];
            work = (fc > -1) && (ave_type == 2 || blk_mask[b] == BLK_INTERFACE);
        }
        const int off = (k & 1) + 4 * (k >> 1);
        bool avg[2];
        long long ccell[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int t = t0 + h * (CELLS / 2);
            const int I = t % 4, J = t / 4;
            // Child block of this cell's quadrant and the first cell of its 2x2 group.
            const int c = (I / 2) + 2 * (J / 2);
            const int c0 = 2 * (I % 2) + 4 * (2 * (J % 2));
            const long long cb = (long long)(fc + c) * CELLS;
            avg[h] = false;
            if (work) {
                int m = cells_mask[cb + c0];
                if (ave_type > 0 && m < 2) m = 1;
                avg[h] = (m == 1);  // uniform over the NG lanes of the group
            }
            ccell[h] = cb + c0 + off;
        }
        T fl[2][Q];
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (avg[h])
#pragma unroll
                for (int p = 0; p < Q; p++) fl[h][p] = Store<T, S>::dec(Fc[(long long)p * ncm + ccell[h]], (T)VS::w(p));
#pragma unroll
        for (int h = 0; h < 2; h++) {
            T s[Q];
            if (avg[h]) {
                const T *f = fl[h];
                T rho, u, v, w;
                moments<T, Q>(f, rho, u, v, w);
                const T udotu = u * u + v * v;
#pragma unroll
                for (int p = 0; p < Q; p++) {
                    T cdotu = cdot<T, Q>(p, u, v, w);
                    T fe = (T)VS::w(p) * rho * ((T)(1.0) + (T)(3.0) * cdotu + (T)(4.5) * cdotu * cdotu - (T)(1.5) * udotu);
                    s[p] = fe + (f[p] - fe) * tau_ratio;
                }
            } else {
#pragma unroll
                for (int p = 0; p < Q; p++) s[p] = (T)0;
            }
            const long long pcell = (long long)b * CELLS + t0 + h * (CELLS / 2);
            // s of child cell offsets 0,1,4,5 summed left to right (comm.cu:330-339)
            T acc[(Q + NG - 1) / NG];
            group_sums<T, Q, NG>(s, acc, s_red + (threadIdx.x >> 6) * Q * 65);
#pragma unroll
            for (int m = 0; m < (Q + NG - 1) / NG; m++) {
                const int p = k + NG * m;
                if (avg[h] && p < Q) Fp[(long long)p * ncm + pcell] = Store<T, S>::enc((T)(0.25) * acc[m], (T)VelSet<Q>::w(p));
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// The fused step's launch.  After the pending exception lists are resolved, the first interp_wgs
// workgroups interpolate one level's interface parents into their children (k_interp, INTERFACE mode),
// and from `lead` on (that count rounded up to a multiple of 8, so that the XCD mapping below still
// deals contiguous ranges) step_wgs workgroups run the fused step of the MultiStep levels.  The few,
// latency-bound interpolation workgroups go first so that they run beside the fused step instead of
// after it.  The two parts touch disjoint cells: a level's interpolation reads the level's current
// buffer and writes the finer level's ghost cells.
// ---------------------------------------------------------------------------------------------
template <typename T, typename S>
struct StepExtras {
    int step_wgs, interp_wgs, lead;
    InterpArgs<T, S> ia;
    FixupArgs<T, S> fa;
};

static_assert(IWG == WG, "interpolation and fused-step workgroups share one launch");

// (D3Q27 MRT in FP32 is held to five wavefronts per SIMD: 102 registers without it, four.)
template <typename T, typename S, int Q, int COLL, bool FOLD>
__global__ __launch_bounds__(WG, (COLL == COLL_MRT && Q == 27 && sizeof(T) == 4 ? 5 : 1)) void k_collide_stream(MultiStep<T, S> m, StepExtras<T, S> x)
{
    using VS = VelSet<Q>;
    using IL = InterpLds<T, Q>;
    constexpr bool MF = COLL == COLL_MFMA;
    // One LDS region shared by the two workgroup kinds of the launch: the interpolation's parent
    // rows and coefficients, or the matrix-core MRT's per-wavefront transpose rows.
    constexpr int ROW = Store<T, S>::quantized ? 20 : 36;
    constexpr int ALL16 = (IL::ALL * (int)sizeof(T) + 15) / 16 * 16 / (int)sizeof(T);  // coefficients 16-byte aligned
    constexpr size_t GHOSTS = (sizeof(T) * (ALL16 + IL::COEF) + 15) / 16 * 16;
    constexpr size_t INTERP_BYTES = GHOSTS + (VS::DIM == 3 ? sizeof(GhostList) : 0);
    constexpr size_t MRT_BYTES = MF ? sizeof(float) * (WG / 64) * 64 * ROW : 0;
    __shared__ __attribute__((aligned(16))) unsigned char s_raw[INTERP_BYTES > MRT_BYTES ? INTERP_BYTES : MRT_BYTES];
    if constexpr (FOLD) resolve_pending<T, S, Q>(x.fa);
    if ((int)blockIdx.x < x.lead) {
        if ((int)blockIdx.x < x.interp_wgs) {
            T *s_all = reinterpret_cast<T *>(s_raw);
            T *s_coef = s_all + ALL16;
            interp_parents<T, S, Q, false>(x.ia, blockIdx.x, s_all, s_coef, *reinterpret_cast<GhostList *>(s_raw + GHOSTS));
        }
        return;
    }
    const int wg = (int)blockIdx.x - x.lead;
    int k = 0;
#pragma unroll
    for (int j = 1; j < MAXLV; j++)
        if (j < m.nlv && wg >= m.start[j]) k = j;
    k = __builtin_amdgcn_readfirstlane(k);
    const StepArgs<T, S> &a = m.lv[k];
    const int wave = __builtin_amdgcn_readfirstlane(xcd_local_wg(wg - m.start[k], m.start[k + 1] - m.start[k]) * (WG / 64) +
                                                    (int)(threadIdx.x >> 6));
    if constexpr (VS::DIM == 3) {
        // One transpose region per wavefront for the matrix-core MRT: 64 rows of 36 floats, or of
        // 20 floats (80 bytes: the forward rows, and the back rows in binary16) with 16-bit pools.
        float *s_mrt = MF ? reinterpret_cast<float *>(s_raw) + (threadIdx.x >> 6) * 64 * ROW : nullptr;
        if (a.vmode == VMODE_EVEN)
            even_step_3d<T, S, Q, COLL>(a, wave, s_mrt);
        else
            collide_stream_3d<T, S, Q, COLL>(a, wave, s_mrt);
    } else {
        collide_stream_2d<T, S, Q, COLL>(a, wave);
    }
}

// ---------------------------------------------------------------------------------------------
// Linked blocks (3D, face-cell links of a geometry): the sub-step of blocks holding boundary cells
// with cut-link fractions.  Cu_Collide, then Cu_ImposeBC with the interpolated bounce-back of
// Bouzidi, Firdaouss and Lallemand (2001) (solver_lbm_kernels.cu:796-875), then the push of the
// fused step (push_link), one wavefront per block; the fused step of the same launch skips these blocks
// (LINK_FLAG, skip_linked).  Where none of the rules is due (link_step_due) the fused step takes them.
// Both read the level's input buffer and write disjoint slots of its output buffer, and record
// guard exceptions into the same list, so they can run in either order.
//
// For a link of fraction q along c_p from boundary cell x:
//   q < 1/2:  f_p <- 2q f_p + (1 - 2q) f*_p(x - c_p);   q >= 1/2:  f_p <- f_p / 2q + (2q - 1)/2q f_pb,
// per half-set pair in the order hook(p), link(p), hook(pb), link(pb), so the pb link's second
// form sees the new f_p.  f*_p(x - c_p) is the post-collision value behind the cell: a lane of the
// same wavefront, or, across a block face, the collision of that cell recomputed here from the
// same inputs with the same code (so the same bits).  A missing block behind the cell leaves f_p
// unchanged (the reference reads out of bounds there).
//
// With `mea` the block's momentum-exchange sums before the boundary rules (Cu_ComputeForcesMEA
// post_step 0, solver_lbm_kernels_forces.cu:322-540) are formed here from the post-collision
// values and stored (assigned) per block; k_mea_post adds the after-stream part.
// ---------------------------------------------------------------------------------------------
template <typename T>
struct LinkArgs {
    const int *ids;       // the level's linked blocks
    int n;
    const int *onb_solid;  // block -> rank in the link arrays
    const float *X_b;      // fractions [rank*64 + cell + q*ncb], 27 directions
    long long ncb;
    int bc_type;          // S_BC_TYPE: 1 = interpolated bounce-back
    int mea;              // form the pre-boundary momentum-exchange sums (post_step 0)
    int order;            // S_FORCE_ORDER
    T *blkF;              // 3 x nmax block sums
    long long nmax;
    T dv;                 // cell volume dx^3 of the level
};

// Post-collision value f*_q of cell `tc` of block nbk (which exists), from the launch's input
// buffer: collide_cell on the same loads and flags as that cell's own wavefront.
template <typename T, typename S, int Q>
__device__ __forceinline__ T post_collision_at(const StepArgs<T, S> &a, int nbk, int tc, int q)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    const long long cell = (long long)nbk * 64 + tc;
    T f[Q], fs[Q];
#pragma unroll
    for (int p = 0; p < Q; p++) f[p] = ST::dec(a.A[(long long)p * a.ncm + cell], (T)VS::w(p));
    const bool inert = a.part[nbk] == 0 || a.cells_mask[cell] == CELL_SOLID;
    T rho, u, v, w;
    moments<T, Q>(f, rho, u, v, w);
    collide_cell<T, S, Q>(a, f, fs, rho, u, v, w, inert);
    T r = (T)0;
#pragma unroll
    for (int p = 0; p < Q; p++)
        if (p == q) r = fs[p];
    return r;
}

// Reduction of one value per lane over the wavefront in the reference's shared-memory tree order
// (s = 32, 16, ..., 1: v[t] = v[t] + v[t + s]); lane 0 holds the result.
template <typename T>
__device__ __forceinline__ T tree_sum64(T v)
{
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v = v + __shfl_down(v, s, 64);
    return v;
}

// One momentum-exchange contribution (side s of a half-set pair) added to acc:
// order 1: f c_s; order 2: ((1/2 + q) f + (1/2 - q) f_m) c_s, the literal 1/2 a double, so the term
// and the running sum are formed in double and rounded by the reference's +=.
template <typename T>
__device__ __forceinline__ void mea_add(T *acc, int order, T f, T fm, float dist, int cx, int cy, int cz)
{
    const int c[3] = {cx, cy, cz};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        if (order == 1) {
            acc[d] += f * (T)c[d];
        } else {
            const double qd = (double)(T)dist;
            acc[d] = (T)((double)acc[d] + ((0.5 + qd) * (double)f + (0.5 - qd) * (double)fm) * (double)c[d]);
        }
    }
}

// FM: the values behind the cells, f*_p(x - c_p), are needed (interpolated bounce-back, or the
// second-order momentum exchange).  Neighbour blocks are looked up through the wave's table as they
// are used: held as 27 values and picked by compares they took 244 registers and 62 us a launch of 2312
// blocks (D3Q27 MRT, FP32), 46 us so without the values behind.
template <typename T, typename S, int Q, bool FM>
__global__ __launch_bounds__(WG) void k_link_step(StepArgs<T, S> a, LinkArgs<T> la)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    const int t = threadIdx.x & 63;
    const int bi = blockIdx.x * (WG / 64) + (int)(threadIdx.x >> 6);
    if (bi >= la.n) return;  // whole wavefronts
    const int b = __builtin_amdgcn_readfirstlane(la.ids[bi]);
    const unsigned cell = (unsigned)b * 64u + (unsigned)t;
    const int my_nb = a.nbr_slot[(long long)b * 27 + (t < 27 ? t : 26)];
    const int part_u = __builtin_amdgcn_readfirstlane(a.part[b]);
    const int onb_u = __builtin_amdgcn_readfirstlane(a.onb[b]);
    const int rank = __builtin_amdgcn_readfirstlane(la.onb_solid[b]);
    const int mask = a.cells_mask[cell];
    const bool linked = rank >= 0 && mask == CELL_BOUNDARY;
    const long long cb = (long long)rank * 64 + t;
    float xq[Q];
#pragma unroll
    for (int q = 1; q < Q; q++) xq[q] = linked ? la.X_b[cb + (long long)q * la.ncb] : -1.0f;
    T f[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) f[q] = ST::dec(a.A[(long long)q * a.ncm + cell], (T)VS::w(q));
    const bool inert = part_u == 0 || mask == CELL_SOLID;
    T fs[Q];
    T rho, u, v, w;
    moments<T, Q>(f, rho, u, v, w);
    collide_cell<T, S, Q>(a, f, fs, rho, u, v, w, inert);

    const SlotOf<Q> slot(t);
    // Block of the cell x + c_q (every lane takes part).
    auto nb_of = [&](int q) { return __builtin_amdgcn_ds_bpermute(slot(q), my_nb); };
    const bool curved = FM && la.bc_type == 1 && linked;

    // f*_q(x - c_q): within the block from lane (I,J,K) - c_q (every lane takes part), else recomputed.
    T fm[FM ? Q : 1];
    unsigned missing = 0;  // bit q: the block behind is missing
    if constexpr (FM) {
        const int I = t & 3, J = (t >> 2) & 3, K = t >> 4;
        const bool mea2 = la.mea && la.order != 1 && linked;
        unsigned need = 0;  // bit q: needed and across a block face
        fm[0] = (T)0;
#pragma unroll
        for (int q = 1; q < Q; q++) {
            const int cx = VS::cx(q), cy = VS::cy(q), cz = VS::cz(q);
            const int src = (int)cell_of_link<Q, 0>(t, VS::pb(q));
            if constexpr (sizeof(T) == 8) {
                const long long bits = __builtin_bit_cast(long long, fs[q]);
                const int lo = __shfl((int)(bits & 0xffffffffLL), src, 64), hi = __shfl((int)(bits >> 32), src, 64);
                fm[q] = __builtin_bit_cast(T, ((long long)hi << 32) | (unsigned)lo);
            } else {
                fm[q] = __shfl(fs[q], src, 64);
            }
            const bool inside = (unsigned)(I - cx) < 4u && (unsigned)(J - cy) < 4u && (unsigned)(K - cz) < 4u;
            const bool want = (curved && xq[q] > 0 && xq[q] < 0.5f) || (mea2 && xq[q] > 0);
            if (want && !inside) need |= 1u << q;
        }
        while (need) {
            const int q = __builtin_ctz(need);
            need &= need - 1;
            int cx = 0, cy = 0, cz = 0;
#pragma unroll
            for (int p = 1; p < Q; p++)
                if (p == q) {
                    cx = VS::cx(p);
                    cy = VS::cy(p);
                    cz = VS::cz(p);
                }
            const int Ip = I - cx + 4, Jp = J - cy + 4, Kp = K - cz + 4;
            const int nbk = a.nbr_slot[(long long)b * 27 + (Ip >> 2) + 3 * (Jp >> 2) + 9 * (Kp >> 2)];
            T val = (T)0;
            if (nbk >= 0)
                val = post_collision_at<T, S, Q>(a, nbk, (Ip & 3) + 4 * (Jp & 3) + 16 * (Kp & 3), q);
            else
                missing |= 1u << q;
#pragma unroll
            for (int p = 1; p < Q; p++)
                if (p == q) fm[p] = val;
        }
    }

    // Momentum exchange before the boundary rules (post_step 0).
    if (la.mea) {
        T acc[3] = {(T)0, (T)0, (T)0};
        if (linked) {
#pragma unroll
            for (int p = 1; p < Q; p++) {
                if (!VS::half(p)) continue;
                const int pb = VS::pb(p);
                if (xq[p] > 0) mea_add<T>(acc, FM ? la.order : 1, fs[p], FM ? fm[p] : (T)0, xq[p], VS::cx(p), VS::cy(p), VS::cz(p));
                if (xq[pb] > 0)
                    mea_add<T>(acc, FM ? la.order : 1, fs[pb], FM ? fm[pb] : (T)0, xq[pb], VS::cx(pb), VS::cy(pb), VS::cz(pb));
            }
        }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const T s = tree_sum64<T>(acc[d]);
            if (t == 0) la.blkF[(long long)d * la.nmax + b] = s * la.dv;
        }
    }

    // Cu_ImposeBC: face hooks and the interpolated bounce-back, pair by pair.
    const bool onb = onb_u == 1 && mask != CELL_SOLID;
    if (onb_u == 1) {
#pragma unroll
        for (int p = 1; p < Q; p++) {
            if (!VS::half(p)) continue;
            const int pb = VS::pb(p);
            const int nbp = nb_of(p), nbb = nb_of(pb);
            T f_p = fs[p], f_q = fs[pb];
            if (nbp < 0 && nbp != N_SKIPID)
                f_p = bc_hook<T>(a.bc_preset, a.U, nbp, f_p, u, v, w, (T)VS::w(p), (T)VS::cx(p), (T)VS::cy(p), (T)VS::cz(p));
            if constexpr (FM)
                if (curved) {
                    const T dQ = (T)xq[p];
                    if (xq[p] > 0 && xq[p] < 0.5f) {
                        if (!((missing >> p) & 1)) f_p = (T)(2.0) * dQ * f_p + ((T)(1.0) - (T)(2.0) * dQ) * fm[p];
                    } else if (xq[p] >= 0.5f) {
                        f_p = ((T)(1.0) / ((T)(2.0) * dQ)) * f_p + (((T)(2.0) * dQ - (T)(1.0)) / ((T)(2.0) * dQ)) * f_q;
                    }
                }
            if (nbb < 0 && nbb != N_SKIPID)
                f_q = bc_hook<T>(a.bc_preset, a.U, nbb, f_q, u, v, w, (T)VS::w(pb), (T)VS::cx(pb), (T)VS::cy(pb), (T)VS::cz(pb));
            if constexpr (FM)
                if (curved) {
                    const T dQ = (T)xq[pb];
                    if (xq[pb] > 0 && xq[pb] < 0.5f) {
                        if (!((missing >> pb) & 1)) f_q = (T)(2.0) * dQ * f_q + ((T)(1.0) - (T)(2.0) * dQ) * fm[pb];
                    } else if (xq[pb] >= 0.5f) {
                        f_q = ((T)(1.0) / ((T)(2.0) * dQ)) * f_q + (((T)(2.0) * dQ - (T)(1.0)) / ((T)(2.0) * dQ)) * f_p;
                    }
                }
            fs[p] = onb ? f_p : fs[p];
            fs[pb] = onb ? f_q : fs[pb];
        }
    }

    // The push (hooks already applied).
    store_pop(a.B, cell, ST::enc(fs[0], (T)VS::w(0)));
#pragma unroll
    for (int q = 1; q < Q; q++) {
        const int nbk = nb_of(q);
        const long long tgt = (long long)nbk * 64 + cell_of_link<Q, 0>(t, q);
        push_link<T, S, Q>(a, q, fs[q], nbk, tgt, (long long)cell, inert, false, false, u, v, w);
    }
}

// Cu_ComputeForcesMEA post_step 1 on the finest level after its last sub-step of the coarse step
// (and its exception fixup): the same sums from the values that arrived -- the reference's slot p
// after the stream is this build's row pb(p) -- added to the block's entry.
template <typename T, typename S, int Q>
__global__ __launch_bounds__(WG) void k_mea_post(const int *__restrict__ ids, int n, const S *__restrict__ F,
                                                 long long ncm, const int *__restrict__ nbr_slot,
                                                 const int *__restrict__ cells_mask, LinkArgs<T> la)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    const int t = threadIdx.x & 63;
    const int bi = blockIdx.x * (WG / 64) + (int)(threadIdx.x >> 6);
    if (bi >= n) return;
    const int b = __builtin_amdgcn_readfirstlane(ids[bi]);
    const int rank = __builtin_amdgcn_readfirstlane(la.onb_solid[b]);
    const long long cell = (long long)b * 64 + t;
    const int my_nb = nbr_slot[(long long)b * 27 + (t < 27 ? t : 26)];
    const bool linked = rank >= 0 && cells_mask[cell] == CELL_BOUNDARY;
    const int I = t & 3, J = (t >> 2) & 3, K = t >> 4;
    const long long cb = (long long)rank * 64 + t;
    T acc[3] = {(T)0, (T)0, (T)0};
    // Slot s of cell (I,J,K) - c_s: row pb(s) there.
    auto behind = [&](int s_dir) -> T {
        const int cx = VS::cx(s_dir), cy = VS::cy(s_dir), cz = VS::cz(s_dir);
        const int Ip = I - cx, Jp = J - cy, Kp = K - cz;
        const int slot = (Ip < 0 ? 0 : (Ip >= 4 ? 2 : 1)) + 3 * (Jp < 0 ? 0 : (Jp >= 4 ? 2 : 1)) +
                         9 * (Kp < 0 ? 0 : (Kp >= 4 ? 2 : 1));
        const int nbk = __shfl(my_nb, slot, 64);
        if (nbk < 0) return (T)0;
        const long long o = (long long)nbk * 64 + ((Ip & 3) + 4 * (Jp & 3) + 16 * (Kp & 3));
        return ST::dec(F[(long long)VS::pb(s_dir) * ncm + o], (T)VS::w(s_dir));
    };
#pragma unroll
    for (int p = 1; p < Q; p++) {
        if (!VS::half(p)) continue;
        const int pb = VS::pb(p);
        // every lane evaluates its shuffles; only linked lanes add
        const T fmp = behind(p), fmq = behind(pb);
        if (!linked) continue;
        const float xp = la.X_b[cb + (long long)p * la.ncb], xb = la.X_b[cb + (long long)pb * la.ncb];
        const T f_p = ST::dec(F[(long long)pb * ncm + cell], (T)VS::w(p));
        const T f_q = ST::dec(F[(long long)p * ncm + cell], (T)VS::w(pb));
        if (xp > 0) mea_add<T>(acc, la.order, f_p, fmp, xp, VS::cx(p), VS::cy(p), VS::cz(p));
        if (xb > 0) mea_add<T>(acc, la.order, f_q, fmq, xb, VS::cx(pb), VS::cy(pb), VS::cz(pb));
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const T s = tree_sum64<T>(acc[d]);
        if (t == 0) la.blkF[(long long)d * la.nmax + b] += s * la.dv;
    }
}

// ---------------------------------------------------------------------------------------------
// Cu_ComputeForcesCV (solver_lbm_kernels_forces.cu:13-246): the control-volume force sums of one
// level, one wavefront per block, lane t = cell t (lanes past the block's cells hold zeros).  A
// cell takes part when its centre lies strictly inside the box and it is not solid.
//   POST 0 (start of a coarse step): Fp = the momentum of taking-part leaf cells; on the root level
//     Fm = sum over p >= 1 of f*_p c_p for the directions whose neighbour centre x + c_p dx lies
//     outside the box, f*_p the BGK collision with the root rate, formed here only (the pool is
//     not written).
//   POST 1 (end of the coarse step): Fm = the momentum of taking-part leaf cells, plus on the root
//     level f_p c_pb(p) for the directions whose upwind centre x + c_pb(p) dx lies outside.
// Per block, the lane values go through the reference's shared-memory tree (s = cells/2 ... 1),
// times dx^DIM; POST 0 assigns the entries [2d] (Fp) and [2d+1] (Fm), POST 1 adds to them.
// ---------------------------------------------------------------------------------------------
template <typename T>
struct CvArgs {
    T dx, dv;        // spacing and cell volume of the level
    T om, omp;       // root-level BGK rate dx/tau and 1 - rate
    T box[6];        // xm, xM, ym, yM, zm, zM
    int root;        // the level is N_LEVEL_START
    T *blkF;         // 6 x nmax block sums
    long long nmax;
};

template <typename T, int DIM>
__device__ __forceinline__ bool cv_inside(const CvArgs<T> &cv, T x, T y, T z)
{
    bool in = x > cv.box[0] && x < cv.box[1] && y > cv.box[2] && y < cv.box[3];
    if (DIM == 3) in = in && z > cv.box[4] && z < cv.box[5];
    return in;
}

template <typename T, int CELLS>
__device__ __forceinline__ T tree_sum_cells(T v)
{
#pragma unroll
    for (int s = CELLS / 2; s > 0; s >>= 1) v = v + __shfl_down(v, s, 64);
    return v;
}

template <typename T, typename S, int Q, int POST>
__global__ __launch_bounds__(WG) void k_cv_force(const int *__restrict__ ids, int n, const S *__restrict__ F,
                                                 long long ncm, const float *__restrict__ X,
                                                 const int *__restrict__ cells_mask,
                                                 const int *__restrict__ nbr_child, CvArgs<T> cv)
{
    using VS = VelSet<Q>;
    using ST = Store<T, S>;
    constexpr int CELLS = VS::CELLS, DIM = VS::DIM;
    const int lane = threadIdx.x & 63;
    const int bi = blockIdx.x * (WG / 64) + (int)(threadIdx.x >> 6);
    if (bi >= n) return;
    const int b = __builtin_amdgcn_readfirstlane(ids[bi]);
    if (b < 0) return;
    const bool act = lane < CELLS;
    const int t = act ? lane : 0;
    const long long cell = (long long)b * CELLS + t;
    const bool leaf = nbr_child[b] < 0;
    const int I = t & 3, J = (t >> 2) & 3, K = t >> 4;
    const T x = (T)X[b] + cv.dx * ((T)0.5 + (T)I);
    const T y = (T)X[b + cv.nmax] + cv.dx * ((T)0.5 + (T)J);
    const T z = DIM == 3 ? (T)X[b + 2 * cv.nmax] + cv.dx * ((T)0.5 + (T)K) : (T)0;
    const bool pV = act && cv_inside<T, DIM>(cv, x, y, z) && cells_mask[cell] != CELL_SOLID;
    T f[Q];
    T rho = (T)0, m[3] = {(T)0, (T)0, (T)0};
#pragma unroll
    for (int p = 0; p < Q; p++) {
        f[p] = ST::dec(F[(long long)p * ncm + cell], (T)VS::w(p));
        rho = rho + f[p];
        m[0] = m[0] + f[p] * (T)VS::cx(p);
        m[1] = m[1] + f[p] * (T)VS::cy(p);
        if (DIM == 3) m[2] = m[2] + f[p] * (T)VS::cz(p);
    }
    T Fp[3] = {(T)0, (T)0, (T)0}, Fm[3] = {(T)0, (T)0, (T)0};
    if (pV && leaf) {
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            if (POST == 0) Fp[d] = Fp[d] + m[d];
            else Fm[d] = Fm[d] + m[d];
        }
    }
    if (cv.root && pV) {
        const T u = m[0] / rho, v = m[1] / rho, w = m[2] / rho;
#pragma unroll
        for (int p = 1; p < Q; p++) {
            const int s = POST == 0 ? p : VS::pb(p);  // the direction whose far centre is tested
            const int c[3] = {VS::cx(s), VS::cy(s), VS::cz(s)};
            if (cv_inside<T, DIM>(cv, x + (T)c[0] * cv.dx, y + (T)c[1] * cv.dx, z + (T)c[2] * cv.dx)) continue;
            T fv = f[p];
            if (POST == 0) {
                const T udotu = u * u + v * v + w * w;
                const T cdotu = (T)c[0] * u + (T)c[1] * v + (T)c[2] * w;
                fv = fv * cv.omp +
                     ((T)VS::w(p) * rho * ((T)1 + (T)3 * cdotu + (T)4.5 * cdotu * cdotu - (T)1.5 * udotu)) * cv.om;
            }
#pragma unroll
            for (int d = 0; d < DIM; d++) Fm[d] = Fm[d] + fv * (T)c[d];
        }
    }
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const T sp = tree_sum_cells<T, CELLS>(Fp[d]), sm = tree_sum_cells<T, CELLS>(Fm[d]);
        if (lane == 0) {
            T &ep = cv.blkF[(long long)(2 * d) * cv.nmax + b];
            T &em = cv.blkF[(long long)(2 * d + 1) * cv.nmax + b];
            if (POST == 0) {
                ep = sp * cv.dv;
                em = sm * cv.dv;
            } else {
                ep += sp * cv.dv;
                em += sm * cv.dv;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------------------------
static inline int nwg(long long nblocks, int cells) { return (int)((nblocks * cells + WG - 1) / WG); }

template <int Q>
static inline int interp_grid(long long nparents)
{
    constexpr int ppw = IWG / (VelSet<Q>::CHILDREN / 2 * VelSet<Q>::CELLS);
    return (int)((nparents + ppw - 1) / ppw);
}

template <int Q>
static inline int cubic_grid(long long nparents)
{
    constexpr int ppw = VelSet<Q>::DIM == 3 ? 1 : CWG / (VelSet<Q>::CHILDREN * VelSet<Q>::CELLS);
    return (int)((nparents + ppw - 1) / ppw);
}

template <typename T, typename S, int Q>
static int set_ic_t(Ctx *c, int L)
{
    int n = c->n_ids[L];
    if (n <= 0) return AGAL_OK;
    hipLaunchKernelGGL((k_set_ic<T, S, Q>), dim3(nwg(n, VelSet<Q>::CELLS)), dim3(WG), 0, c->stream, c->id_set_L(L), n,
                       Fbuf<S>(c, c->cur[L]), c->n_maxcells, c->cells_mask, (T)c->P.ic_rho, (T)c->P.ic_u,
                       (T)c->P.ic_v, (T)c->P.ic_w);
    AGAL_HIP(c, hipGetLastError());
    return AGAL_OK;
}

template <typename T, typename S, int Q>
static int refresh_t(Ctx *c, int L)
{
    int n = c->n_ids[L];
    if (n <= 0) return AGAL_OK;
    hipLaunchKernelGGL((k_refresh<T, S, Q>), dim3(nwg(n, VelSet<Q>::CELLS)), dim3(WG), 0, c->stream, c->id_set_L(L),
                       n, Fbuf<S>(c, c->cur[L]), static_cast<T *>(c->M), c->n_maxcells);
    AGAL_HIP(c, hipGetLastError());
    return AGAL_OK;
}

// The extra-list mode of level L in the fused launch being issued: only for the finest level of a
// 3D set inside a coarse step.
template <int Q>
static int pair_mode(const Ctx *c, int L)
{
    // Linked blocks recompute neighbours' collisions from the input buffer as it is stored, so
    // with links every sub-step resolves its exceptions by a fixup instead.
    if (VelSet<Q>::DIM != 3 || !c->defer_coarse || L != c->MAX_LEVELS - 1 || c->links_on) return 0;
    return c->fine_pair == 1 && inplace_ok(c, L) ? VMODE_EVEN : c->fine_pair;
}

// The momentum-exchange force (force type 0) is evaluated on the finest level's last sub-step of a
// coarse step, every step on a single level (solver_lbm_advance.cu:124-131, :144-150).
static bool mea_active(const Ctx *c) { return c->links_on && c->P.S_FORCE_TYPE == 0 && c->DIM == 3; }
static bool mea_due(const Ctx *c, int L)
{
    if (!mea_active(c) || L != c->MAX_LEVELS - 1) return false;
    const bool multi = c->MAX_LEVELS > 1 && c->MAX_LEVELS != c->N_LEVEL_START + 1;
    return !multi || c->global_Liter == (1 << (c->MAX_LEVELS - 1)) - 1;
}

// The collision operator of the fused step's launches.
template <typename T, int Q>
static int fused_operator(const Ctx *c)
{
    if (c->P.collision != AGAL_MRT) return COLL_BGK;
    return sizeof(T) == 4 && VelSet<Q>::DIM == 3 && c->mrt_mfma ? COLL_MFMA : COLL_MRT;
}

// Whether the linked blocks' sub-step is k_link_step's: where its rules differ from the fused step's, and
// where its collision does -- on matrix cores the fused step's MRT is of another precision, and a block
// near the wall would alternate between the two from one sub-step to the next.
template <typename T, int Q>
static bool link_step_due(const Ctx *c, int L)
{
    return c->links_on && c->lk_n[L] > 0 &&
           (c->P.S_BC_TYPE == 1 || mea_due(c, L) || fused_operator<T, Q>(c) == COLL_MFMA);
}

template <typename T>
static LinkArgs<T> link_args(Ctx *c, int L, bool mea)
{
    LinkArgs<T> la;
    la.ids = c->lk_ids + c->lk_off[L];
    la.n = c->lk_n[L];
    la.onb_solid = c->lk_onb_solid;
    la.X_b = c->lk_X;
    la.ncb = c->lk_ncb;
    la.bc_type = c->P.S_BC_TYPE;
    la.mea = mea ? 1 : 0;
    la.order = c->P.S_FORCE_ORDER;
    la.blkF = static_cast<T *>(c->lk_blkF);
    la.nmax = c->n_maxcblocks;
    const T dx = (T)c->dxf_vec[L];
    la.dv = (T)((T)((T)(T)1 * dx) * dx) * dx;  // dvf_vec (solver_lbm_init.cu:19-27)
    return la;
}

// The linked blocks' sub-step of level L reading buffer rd, on stream s, where it differs from that of
// other blocks: with the interpolated bounce-back, when the momentum exchange is due, or with the fused
// step's MRT on matrix cores.  Otherwise the fused step takes the linked blocks like any (link_step_due).
template <typename T, typename S, int Q>
static int launch_link_step(Ctx *c, int L, int rd, hipStream_t s)
{
    if constexpr (VelSet<Q>::DIM == 3) {
        if (!link_step_due<T, Q>(c, L)) return AGAL_OK;
        const LinkArgs<T> la = link_args<T>(c, L, mea_due(c, L));
        const bool fm = la.bc_type == 1 || (la.mea && la.order != 1);
        hipLaunchKernelGGL((fm ? k_link_step<T, S, Q, true> : k_link_step<T, S, Q, false>),
                           dim3((unsigned)((la.n + WG / 64 - 1) / (WG / 64))), dim3(WG), 0, s,
                           step_args<T, S, Q>(c, L, rd, 0), la);
        AGAL_HIP(c, hipGetLastError());
    }
    return AGAL_OK;
}

template <typename T, typename S>
static InterpArgs<T, S> interp_args(Ctx *c, int L, const int *ids, int n, T ratio)
{
    InterpArgs<T, S> ia;
    ia.ids = ids;
    ia.n = n;
    ia.Fp = Fbuf<S>(c, c->cur[L]);
    ia.Fc = Fbuf<S>(c, c->cur[L + 1]);
    ia.ncm = c->n_maxcells;
    ia.nbr_child = c->nbr_child;
    ia.blk_mask = c->blk_mask;
    ia.ref = c->ref;
    ia.cells_mask = c->cells_mask;
    ia.tau_ratio = ratio;
    return ia;
}

// Fused step of levels[j] reading buffers rd[j], up to MAXLV levels per launch.  With `ia`, the
// first launch also interpolates level interp_L's interface parents (reading the buffer those
// sub-steps read).  Exception lists: those pending are resolved first (fold_fixups); the launch leaves
// its own levels' pending; outside a coarse step (defer_coarse) a fixup launch follows at once.  A coarse
// level alone goes to its level stream (the recorded step's scheduler); launches that hold the finest
// level stay on the context stream.
template <typename T, typename S, int Q>
static int launch_fused(Ctx *c, const int *levels, const int *rd, int nl, const InterpArgs<T, S> *ia = nullptr,
                        int interp_L = -1)
{
    constexpr int CELLS = VelSet<Q>::CELLS, BPW = 64 / CELLS;  // blocks per wavefront
    int st;
    unsigned touch = 0;
    for (int j = 0; j < nl; j++) touch |= 1u << levels[j];
    if (ia) touch |= 3u << interp_L;
    for (int base = 0; base < nl || (base == 0 && ia); base += MAXLV) {
        MultiStep<T, S> m;
        StepExtras<T, S> x;
        m.nlv = 0;
        int wgs = 0;
        double cells = 0;
        unsigned rmask = 0, wmask = 0;
        unsigned long long records = 0;
        bool finest = false;
        int first = -1;
        for (int j = base; j < nl && j < base + MAXLV; j++) {
            const int L = levels[j], n = c->n_ids[L];
            const int mode = pair_mode<Q>(c, L);
            rmask |= res_bit(L, rd[j]);
            wmask |= res_bit(L, mode == VMODE_EVEN ? rd[j] : rd[j] ^ 1);
            if (n <= 0) continue;
            finest = finest || L == c->MAX_LEVELS - 1;
            if (first < 0) first = L;
            m.lv[m.nlv] = step_args<T, S, Q>(c, L, rd[j], mode);
            records |= records_into(c, L, mode);
            m.lv[m.nlv].skip_linked = link_step_due<T, Q>(c, L);
            m.start[m.nlv] = wgs;
            const int waves = (n + BPW - 1) / BPW;
            wgs += ((waves + WG / 64 - 1) / (WG / 64) + 7) / 8 * 8;  // a multiple of the XCD count
            cells += (double)n * CELLS;
            m.nlv++;
        }
        for (int k = m.nlv; k <= MAXLV; k++) m.start[k] = wgs;
        x.step_wgs = wgs;
        x.interp_wgs = 0;
        if (base == 0) {
            if (ia && ia->n > 0) {
                x.ia = *ia;
                x.interp_wgs = interp_grid<Q>(ia->n);
                rmask |= res_bit(interp_L, rd[0]);
                wmask |= res_bit(interp_L + 1, c->cur[interp_L + 1]);
            }
        }
        x.lead = (x.interp_wgs + 7) / 8 * 8;
        if (x.step_wgs + x.interp_wgs == 0) continue;
        const int grid = x.lead + x.step_wgs;
        if ((st = fold_fixups<T, S, Q>(c, grid, touch, records, x.fa, wmask))) return st;
        const int slot = (finest || m.nlv != 1 || x.interp_wgs || x.fa.n) ? 0 : 1 + first;
        hipStream_t s = sched_begin(c, slot, rmask, wmask);
        // One kernel per collision operator: BGK alone needs fewer registers than MRT's moments.  The
        // matrix-core MRT variant: FP32 compute, 3D sets, when enabled.
        using K = void (*)(MultiStep<T, S>, StepExtras<T, S>);
        const int op = fused_operator<T, Q>(c);
        const bool mrt = op != COLL_BGK, fold = x.fa.n > 0;
        K kern = mrt ? (fold ? (K)k_collide_stream<T, S, Q, COLL_MRT, true> : (K)k_collide_stream<T, S, Q, COLL_MRT, false>)
                     : (fold ? (K)k_collide_stream<T, S, Q, COLL_BGK, true> : (K)k_collide_stream<T, S, Q, COLL_BGK, false>);
        if constexpr (sizeof(T) == 4 && VelSet<Q>::DIM == 3)
            if (op == COLL_MFMA)
                kern = fold ? (K)k_collide_stream<T, S, Q, COLL_MFMA, true> : (K)k_collide_stream<T, S, Q, COLL_MFMA, false>;
        if ((st = launch_timed(c, kern, grid, s, cells, m, x))) return st;
        for (int j = base; j < nl && j < base + MAXLV; j++)
            if ((st = launch_link_step<T, S, Q>(c, levels[j], rd[j], s))) return st;
        if ((st = sched_done(c, s, slot, rmask, wmask))) return st;
        // A list left for the next finest sub-step (pair mode 1) is not pending a fixup.
        for (int j = base; j < nl && j < base + MAXLV; j++) {
            const int mode = pair_mode<Q>(c, levels[j]);
            if (mode == VMODE_EVEN)
                c->leave_pending(levels[j], rd[j], 1);
            else if (mode != 1)
                c->leave_pending(levels[j], rd[j] ^ 1, 0);
        }
        if (!c->defer_coarse && (st = launch_fixups<T, S, Q>(c))) return st;
    }
    return AGAL_OK;
}

// The fused step of level L.  Inside a coarse step (defer_coarse), a level above the finest is
// held back and joins the launch of the next finest-level sub-step: between the two the advance
// runs only kernels of finer levels (interpolation into level L+1's children, finer sub-steps),
// which touch none of level L's cells, so the order of results is unchanged.
template <typename T, typename S, int Q>
static int collide_stream_t(Ctx *c, int L)
{
    if (c->defer_coarse && L < c->MAX_LEVELS - 1) {
        c->deferred.push_back({L, c->cur[L]});
        c->cur[L] ^= 1;
        return AGAL_OK;
    }
    std::vector<int> lv{L}, rd{c->cur[L]};
    // An in-place pair leaves the level in the buffer that it read.
    const bool even = pair_mode<Q>(c, L) == VMODE_EVEN;
    if (!even && c->fine_pair == 2 && c->defer_coarse && inplace_ok(c, L)) return launch_odd_step(c, L);
    if (!even) c->cur[L] ^= 1;
    for (const auto &d : c->deferred) {
        lv.push_back(d.first);
        rd.push_back(d.second);
    }
    c->deferred.clear();
    return launch_fused<T, S, Q>(c, lv.data(), rd.data(), (int)lv.size());
}

// Interpolation of level L (INTERFACE mode) followed by level L's fused sub-step: one launch
// inside a coarse step with linear interpolation (the interpolation reads the buffer the sub-step
// reads and writes level L+1's ghost cells, which the sub-step does not touch), held-back coarser
// sub-steps included; two launches otherwise.
template <typename T, typename S, int Q>
static int interp_collide_t(Ctx *c, int L)
{
    int st;
    // The timed pass (timing.enabled) keeps the interpolation apart, so that the events around a
    // fused launch time the fused step alone.
    if (!c->defer_coarse || c->timing.enabled || c->P.interp_order == AGAL_INTERP_CUBIC || L >= c->MAX_LEVELS - 1) {
        if ((st = launch_interpolate(c, L, AGAL_INTERP_INTERFACE))) return st;
        return launch_collide_stream(c, L);
    }
    const T ratio = (T)c->tau_vec[L + 1] / (T)c->tau_vec[L];
    const InterpArgs<T, S> ia = interp_args<T, S>(c, L, c->iface_L(L), c->n_iface[L], ratio);
    std::vector<int> lv{L}, rd{c->cur[L]};
    c->cur[L] ^= 1;
    for (const auto &d : c->deferred) {
        lv.push_back(d.first);
        rd.push_back(d.second);
    }
    c->deferred.clear();
    return launch_fused<T, S, Q>(c, lv.data(), rd.data(), (int)lv.size(), &ia, L);
}

// Launches coarse sub-steps still held back, then resolves every pending exception list.
template <typename T, typename S, int Q>
static int flush_deferred_t(Ctx *c)
{
    int st;
    if (!c->deferred.empty()) {
        std::vector<int> lv, rd;
        for (const auto &d : c->deferred) {
            lv.push_back(d.first);
            rd.push_back(d.second);
        }
        c->deferred.clear();
        if ((st = launch_fused<T, S, Q>(c, lv.data(), rd.data(), (int)lv.size()))) return st;
    }
    return launch_fixups<T, S, Q>(c);
}

template <typename T, typename S, int Q>
static int interpolate_t(Ctx *c, int L, int var)
{
    if (L >= c->MAX_LEVELS - 1) return AGAL_OK;
    const T ratio = (T)c->tau_vec[L + 1] / (T)c->tau_vec[L];
    const int *ids;
    int n;
    if (var == AGAL_INTERP_INTERFACE) {
        ids = c->iface_L(L);
        n = c->n_iface[L];
    } else {
        ids = c->id_set_L(L);
        n = c->n_ids[L];
    }
    if (n <= 0) return AGAL_OK;
    if (int st = launch_fixups_for<T, S, Q>(c, 3u << L)) return st;
    const unsigned rl = res_bit(L, c->cur[L]), wl = res_bit(L + 1, c->cur[L + 1]);
    hipStream_t s = sched_begin(c, 0, rl, wl);
    if (c->P.interp_order == AGAL_INTERP_CUBIC) {
        if (var == AGAL_INTERP_ADDED)
            hipLaunchKernelGGL((k_interp_cubic<T, S, Q, true>), dim3(cubic_grid<Q>(n)), dim3(CWG), 0, s,
                               interp_args<T, S>(c, L, ids, n, ratio));
        else
            hipLaunchKernelGGL((k_interp_cubic<T, S, Q, false>), dim3(cubic_grid<Q>(n)), dim3(CWG), 0, s,
                               interp_args<T, S>(c, L, ids, n, ratio));
    } else if (var == AGAL_INTERP_ADDED)
        hipLaunchKernelGGL((k_interp<T, S, Q, true>), dim3(interp_grid<Q>(n)), dim3(IWG), 0, s,
                           interp_args<T, S>(c, L, ids, n, ratio));
    else
        hipLaunchKernelGGL((k_interp<T, S, Q, false>), dim3(interp_grid<Q>(n)), dim3(IWG), 0, s,
                           interp_args<T, S>(c, L, ids, n, ratio));
    AGAL_HIP(c, hipGetLastError());
    return sched_done(c, s, 0, rl, wl);
}

template <typename T, typename S, int Q>
static int average_t(Ctx *c, int L, int var)
{
    if (L >= c->MAX_LEVELS - 1) return AGAL_OK;
    const T ratio = (T)c->tau_vec[L] / (T)c->tau_vec[L + 1];
    const int *ids;
    int n;
    if (var == AGAL_AVERAGE_INTERFACE || var == AGAL_AVERAGE_BLOCK) {  // both act on INTERFACE blocks only
        ids = c->iface_L(L);
        n = c->n_iface[L];
    } else {
        ids = c->id_set_L(L);
        n = c->n_ids[L];
    }
    if (n <= 0) return AGAL_OK;
    const unsigned rl = res_bit(L + 1, c->cur[L + 1]);
    unsigned wl = res_bit(L, c->cur[L]);
    FixupArgs<T, S> fa;
    const int grid = nwg(n, VelSet<Q>::CELLS / 2 * (VelSet<Q>::DIM == 3 ? 8 : 4));
    if (int st = fold_fixups<T, S, Q>(c, grid, 3u << L, 0, fa, wl)) return st;
    hipStream_t s = sched_begin(c, 0, rl, wl);
    hipLaunchKernelGGL((fa.n ? k_average<T, S, Q, true> : k_average<T, S, Q, false>), dim3(grid), dim3(WG), 0, s, fa, ids, n, Fbuf<S>(c, c->cur[L]), Fbuf<S>(c, c->cur[L + 1]), c->n_maxcells, c->nbr_child,
                       c->blk_mask, c->cells_mask, var, ratio);
    AGAL_HIP(c, hipGetLastError());
    return sched_done(c, s, 0, rl, wl);
}

template <typename T, typename S, int Q>
static int avg_interp_t(Ctx *c, int L)
{
    if (L >= c->MAX_LEVELS - 1) return AGAL_OK;
    if (c->P.interp_order == AGAL_INTERP_CUBIC) {  // cubic: BLOCK averaging and the cubic kernel
        int st = average_t<T, S, Q>(c, L, AGAL_AVERAGE_BLOCK);
        return st ? st : interpolate_t<T, S, Q>(c, L, AGAL_INTERP_INTERFACE);
    }
    const int n = c->n_iface[L];
    if (n <= 0) return AGAL_OK;
    const T ratio_avg = (T)c->tau_vec[L] / (T)c->tau_vec[L + 1];
    const T ratio_int = (T)c->tau_vec[L + 1] / (T)c->tau_vec[L];
    unsigned m = res_bit(L, c->cur[L]) | res_bit(L + 1, c->cur[L + 1]);
    FixupArgs<T, S> fa;
    if (int st = fold_fixups<T, S, Q>(c, interp_grid<Q>(n), 3u << L, 0, fa, m)) return st;
    hipStream_t s = sched_begin(c, 0, m, m);
    hipLaunchKernelGGL((fa.n ? k_avg_interp<T, S, Q, true> : k_avg_interp<T, S, Q, false>), dim3(interp_grid<Q>(n)), dim3(IWG), 0, s, fa, c->iface_L(L), n,
                       Fbuf<S>(c, c->cur[L]), Fbuf<S>(c, c->cur[L + 1]), c->n_maxcells, c->nbr_child, c->blk_mask,
                       c->cells_mask, ratio_avg, ratio_int);
    AGAL_HIP(c, hipGetLastError());
    return sched_done(c, s, 0, m, m);
}

template <typename T, typename S, int Q>
static int cv_force_t(Ctx *c, int L, int post)
{
    const int n = c->n_ids[L];
    if (n <= 0 || !c->cv_F) return AGAL_OK;
    CvArgs<T> cv;
    const T dx = (T)c->dxf_vec[L];
    cv.dx = dx;
    T dv = (T)1;
    for (int d = 0; d < VelSet<Q>::DIM; d++) dv = dv * dx;  // dvf_vec (solver_lbm_init.cu:19-27)
    cv.dv = dv;
    const int L0 = c->N_LEVEL_START;
    cv.om = (T)c->dxf_vec[L0] / (T)c->tau_vec[L0];
    cv.omp = (T)1 - cv.om;
    for (int k = 0; k < 6; k++) cv.box[k] = (T)c->cv_box[k];
    cv.root = L == L0;
    cv.blkF = static_cast<T *>(c->cv_F);
    cv.nmax = c->n_maxcblocks;
    const unsigned rm = res_bit(L, c->cur[L]);
    hipStream_t s = sched_begin(c, 0, rm, 0);
    const dim3 grid((unsigned)((n + WG / 64 - 1) / (WG / 64)));
    if (post == 0)
        hipLaunchKernelGGL((k_cv_force<T, S, Q, 0>), grid, dim3(WG), 0, s, c->id_set_L(L), n, Fbuf<S>(c, c->cur[L]),
                           c->n_maxcells, c->X, c->cells_mask, c->nbr_child, cv);
    else
        hipLaunchKernelGGL((k_cv_force<T, S, Q, 1>), grid, dim3(WG), 0, s, c->id_set_L(L), n, Fbuf<S>(c, c->cur[L]),
                           c->n_maxcells, c->X, c->cells_mask, c->nbr_child, cv);
    AGAL_HIP(c, hipGetLastError());
    return sched_done(c, s, 0, rm, 0);
}

template <typename T, typename S, int Q>
static int mea_post_t(Ctx *c)
{
    if constexpr (VelSet<Q>::DIM == 3) {
        const int L = c->MAX_LEVELS - 1;
        if (!mea_active(c) || c->lk_n[L] <= 0) return AGAL_OK;
        const LinkArgs<T> la = link_args<T>(c, L, true);
        const unsigned rm = res_bit(L, c->cur[L]);
        hipStream_t s = sched_begin(c, 0, rm, 0);
        hipLaunchKernelGGL((k_mea_post<T, S, Q>), dim3((unsigned)((la.n + WG / 64 - 1) / (WG / 64))), dim3(WG), 0, s, la.ids,
                           la.n, Fbuf<S>(c, c->cur[L]), c->n_maxcells, c->nbr_slot, c->cells_mask, la);
        AGAL_HIP(c, hipGetLastError());
        return sched_done(c, s, 0, rm, 0);
    }
    return AGAL_OK;
}

bool inplace_pair(const Ctx *c, int L) { return inplace_ok(c, L); }
int launch_mea_post(Ctx *c) { AGAL_DISPATCH(c, mea_post_t, c); }
int launch_cv_force(Ctx *c, int L, int post) { AGAL_DISPATCH(c, cv_force_t, c, L, post); }
int launch_set_ic(Ctx *c, int L) { AGAL_DISPATCH(c, set_ic_t, c, L); }
int launch_refresh(Ctx *c, int L) { AGAL_DISPATCH(c, refresh_t, c, L); }
int launch_collide_stream(Ctx *c, int L) { AGAL_DISPATCH(c, collide_stream_t, c, L); }
int launch_flush_deferred(Ctx *c) { AGAL_DISPATCH(c, flush_deferred_t, c); }
int launch_interp_collide(Ctx *c, int L) { AGAL_DISPATCH(c, interp_collide_t, c, L); }
int launch_interpolate(Ctx *c, int L, int var) { AGAL_DISPATCH(c, interpolate_t, c, L, var); }
int launch_average(Ctx *c, int L, int var) { AGAL_DISPATCH(c, average_t, c, L, var); }
int launch_average_interpolate(Ctx *c, int L) { AGAL_DISPATCH(c, avg_interp_t, c, L); }

}  // namespace agal
