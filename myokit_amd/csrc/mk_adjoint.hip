/*
 * mk_adjoint.hip -- discrete adjoint kernels (appended to a generated kernel
 * source together with mk_cell_vjp when gradients are requested).
 *
 * For the step y_{s+1} = F_s(y_s) of the whole tissue, s = 0..N-1, and the
 * loss
 *   L = sum_{s=0..N-1} sum_p (V(y_{s+1})[probe p] - target[s][p])^2,
 * the adjoint recursion is
 *   lam_N = dL/dy_N,   lam_s = (dF_s/dy_s)^T lam_{s+1} + dL/dy_s,
 * and a parameter gradient is sum_s (dF_s/dparam)^T lam_{s+1}.
 * (dF_s/dy_s)^T lam_{s+1} has two parts: the cell's own update, whose
 * transpose mk_cell_vjp applies (mu_s), and the coupling through the
 * diffusion current idiff_c = sum_j g_cj (V_c - V_j). With abar_s the
 * per-cell adjoint of idiff (also from mk_cell_vjp), the coupling part is
 * the same weighted graph Laplacian applied to abar_s, added to the V
 * component:  sum_j g_cj (abar_s[c] - abar_s[j]).
 *
 * One reverse step s assembles lam_{s+1} from mu_{s+1}, the Laplacian of
 * abar_{s+1} and the loss term at y_{s+1}, adds the conductance-gradient
 * terms of step s+1, then applies the cell VJP of step s at y_s, giving
 * mu_s and abar_s. lam itself is never stored. Two drivers:
 *
 *   mk_adj_step   one reverse step per launch over all cells (any size); the
 *                 Laplacian needs every cell's abar_{s+1}, hence the launch
 *                 boundary between steps;
 *   mk_adj_block  one workgroup per independent domain (cable, small sheet,
 *                 graph component), every reverse step of a segment in one
 *                 launch; V and abar of the domain live in LDS, one barrier
 *                 per step.
 *
 * Field gradients accumulate per cell in double precision. Conductance
 * gradients are summed over each workgroup (wave shuffles, then LDS) into
 * one double per workgroup, so every partial sum has a single writer and a
 * fixed order: results do not depend on scheduling.
 */
typedef MkAdjT<Real> MkAdj;

/* Sum over the workgroup of a double per thread; valid in thread 0. */
__device__ __forceinline__ double mk_block_sum(double v, double* lds)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < MK_BT / 64; ++k) r += lds[k];
    }
    return r;
}

/* Coupling transpose at cell c of a grid or a single stencil domain for
 * abar_{s+1} (ab) and V(y_{s+1}) (V1): returns sum_j g_cj (ab[c] - ab[j]) and
 * adds the cell's terms of dL/dgx and dL/dgy to cx, cy. Arrays are indexed
 * as in the forward coupling. (Taking those terms from V(y_s) in the same
 * step, as the graphs do, reads less but measured slower on sheets: 36 -> 39
 * us per step of mk_adj_step on 1024 x 1024 cells, 33.5 -> 35.7 of
 * mk_adj_sheet.) */
__device__ __forceinline__ Real mk_adj_couple(
    const MkArgs& a, const Real* __restrict__ V1, const Real* __restrict__ ab,
    int c, int ix, int iy, int nx, int ny, double& cx, double& cy)
{
    Real lv = (Real)0;
    (void)ix; (void)iy; (void)c; (void)nx; (void)ny; (void)V1; (void)ab;
    (void)cx; (void)cy;
#if MK_COUPLING == 1
    const Real ac = ab[c], v = V1[c];
    Real ax = (Real)0, ay = (Real)0, xs = (Real)0, ys = (Real)0;
    if (nx > 1) {
        if (ix > 0) { ax += ac - ab[c - 1]; xs += v - V1[c - 1]; }
        if (ix < nx - 1) { ax += ac - ab[c + 1]; xs += v - V1[c + 1]; }
    }
    if (ny > 1) {
        if (iy > 0) { ay += ac - ab[c - nx]; ys += v - V1[c - nx]; }
        if (iy < ny - 1) { ay += ac - ab[c + nx]; ys += v - V1[c + nx]; }
    }
    lv = a.gx * ax + a.gy * ay;
    cx += (double)ac * (double)xs;
    cy += (double)ac * (double)ys;
#elif MK_COUPLING == 2
    const Real ac = ab[c];
    if (nx > 1) {
        if (ix > 0) lv += a.gx_field[c - iy - 1] * (ac - ab[c - 1]);
        if (ix < nx - 1) lv += a.gx_field[c - iy] * (ac - ab[c + 1]);
    }
    if (ny > 1) {
        if (iy > 0) lv += a.gy_field[c - nx] * (ac - ab[c - nx]);
        if (iy < ny - 1) lv += a.gy_field[c] * (ac - ab[c + nx]);
    }
#endif
    return lv;
}

#if MK_COUPLING == 3
/* One walk of a cell's connections: returns the coupling transpose at
 * abar_{s+1} (ab; 0 if ab is NULL) and sets idiff to the forward current at
 * V(y_s) (V0) and dscale to that current's derivative by a common scale of
 * the conductances, in double precision: the gradient of the scale is
 * sum_s sum_c abar_s[c] dscale_s[c], with the cell's own abar_s (summed per
 * connection instead, 1/2 g (abar_c - abar_j)(V_c - V_j) from each end, the
 * walk would also gather the neighbours' potentials of y_{s+1}: 77.7 ->
 * 72.3 us per step on 16 copies of 100,000 cells). The cell's row is `row`, the cell
 * itself is at `self` of the arrays, which neighbour indices are relative
 * to. Each sum takes the connections in list order, as mk_graph does, four
 * at a time with their loads in flight together. */
__device__ __forceinline__ Real mk_adj_couple_graph(
    const MkArgs& a, const Real* __restrict__ ab, const Real* __restrict__ V0,
    int row, int self, Real& idiff, double& dscale)
{
    const Real v0 = V0[self];
    const Real ac = ab ? ab[self] : (Real)0;
    Real lv = (Real)0, id = (Real)0;
    double ds = 0.0;
    /* rows of one copy for a graph of interleaved copies (see mk_graph) */
    const int K = a.gcopies;
    int lane = 0;
    if (K > 1) {
        row = self / K;
        lane = self - row * K;
    }
    int e = a.csr_ptr[row];
    const int e1 = a.csr_ptr[row + 1];
    for (; e + 4 <= e1; e += 4) {
        int t[4];
        Real gg[4], an[4], wn[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) t[k] = a.csr_idx[e + k];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int nb = (t[k] < 0 ? ~t[k] : t[k]) * K + lane;
            gg[k] = a.csr_g[e + k];
            an[k] = ab ? ab[nb] : (Real)0;
            wn[k] = V0[nb];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            lv += gg[k] * (ac - an[k]);
            ds += (double)gg[k] * ((double)v0 - (double)wn[k]);
            if (t[k] >= 0) id = id + gg[k] * (v0 - wn[k]);
            else id = id - gg[k] * (wn[k] - v0);
        }
    }
    for (; e < e1; ++e) {
        const int t = a.csr_idx[e];
        const int nb = (t < 0 ? ~t : t) * K + lane;
        const Real g = a.csr_g[e], w = V0[nb];
        if (ab) lv += g * (ac - ab[nb]);
        ds += (double)g * ((double)v0 - (double)w);
        if (t >= 0) id = id + g * (v0 - w);
        else id = id - g * (w - v0);
    }
    idiff = id;
    dscale = ds;
    return lv;
}
#endif

/* Loss term dL/dV at cell c for V(y_{s+1}) = v, target row `row`. */
__device__ __forceinline__ Real mk_adj_loss(const MkAdj& j, int c, Real v,
                                            int row)
{
    if (row < 0) return (Real)0;
    const int q = j.probe_of[c];
    if (q < 0) return (Real)0;
    const double d = (double)v - j.target[(long long)row * j.n_probe + q];
    j.loss_acc[q] += d * d;
    return (Real)(2.0 * d);
}

/* Cell VJP of step p at state y (own cell) of a grid or a single stencil
 * domain, V the potentials of y_s indexed as in the forward coupling. */
__device__ __forceinline__ void mk_adj_cell(
    const MkArgs& a, const MkStep& p, const Real* y, const Real* fv,
    const Real* __restrict__ V, int c, int ix, int iy, int nx, int ny,
    const Real* lam, Real* mu, Real& abo, Real* fb)
{
    (void)nx; (void)ny;
#if MK_COUPLING == 1
    const Real idiff = mk_stencil(V, c, ix, iy, nx, ny, a.gx, a.gy);
#elif MK_COUPLING == 2
    const Real idiff = mk_hetero(V, a.gx_field, a.gy_field, c, ix, iy, nx,
                                 ny);
#else
    const Real idiff = (Real)0;
    (void)V;
#endif
    const Real pace = mk_is_paced(a, c, ix, iy) ? p.pace : (Real)0;
    mk_cell_vjp(y, p.t, p.dt, pace, idiff, fv, lam, mu, &abo, fb);
}

/* ---------------------------------------------------------------------- */
extern "C" __global__ void __launch_bounds__(MK_BT, MK_ADJ_WAVES)
mk_adj_step(const MkArgs a, const MkAdj j, const int s)
{
    __shared__ double red[2][MK_BT / 64];
    const int c = blockIdx.x * MK_BT + threadIdx.x;
    double cx = 0.0, cy = 0.0;
    if (c < (int)a.n) {
        const int nx = (int)a.nx, ny = (int)a.ny;
        const int iy = (int)((unsigned)c / (unsigned)nx), ix = c - iy * nx;
        const long long np = a.npad;
        Real lam[MK_NS];
        if (j.mu_in) {
            const Real* __restrict__ m = j.mu_in + c;
#pragma unroll
            for (int i = 0; i < MK_NS; ++i) lam[i] = m[i * np];
        } else {
#pragma unroll
            for (int i = 0; i < MK_NS; ++i) lam[i] = (Real)0;
        }
        const Real* __restrict__ V1 = j.yn1 + MK_IVM * np;
        Real lv = mk_adj_loss(j, c, V1[c], j.target_row);
#if MK_COUPLING == 3
        /* the forward current, with the transpose of the coupling */
        Real idiff0;
        double ds;
        lv += mk_adj_couple_graph(a, j.ab_in, j.yn + MK_IVM * np, c, c,
                                  idiff0, ds);
#else
        if (j.ab_in)
            lv += mk_adj_couple(a, V1, j.ab_in, c, ix, iy, nx, ny, cx, cy);
#endif
        lam[MK_IVM] += lv;
        if (j.yn) {
            Real y[MK_NS], mu[MK_NS], fv[MK_NFA], fb[MK_NFA], abo;
            const Real* __restrict__ yp = j.yn + c;
#pragma unroll
            for (int i = 0; i < MK_NS; ++i) y[i] = yp[i * np];
#pragma unroll
            for (int k = 0; k < MK_NF; ++k) fv[k] = a.fields[k * np + c];
#if MK_COUPLING == 3
            {
                const MkStep& p = a.steps[s];
                const Real pace = mk_is_paced(a, c, ix, iy) ? p.pace
                                                            : (Real)0;
                mk_cell_vjp(y, p.t, p.dt, pace, idiff0, fv, lam, mu, &abo,
                            fb);
                cx = (double)abo * ds;
            }
#else
            mk_adj_cell(a, a.steps[s], y, fv, j.yn + MK_IVM * np, c, ix, iy,
                        nx, ny, lam, mu, abo, fb);
#endif
            Real* __restrict__ mo = j.mu_out + c;
#pragma unroll
            for (int i = 0; i < MK_NS; ++i) mo[i * np] = mu[i];
            j.ab_out[c] = abo;
#pragma unroll
            for (int k = 0; k < MK_NF; ++k) j.gfield[k * np + c] += (double)fb[k];
        }
    }
#if MK_COUPLING == 1 || MK_COUPLING == 3
    if (MK_COUPLING == 3 || j.ab_in) {
        const double sx = mk_block_sum(cx, red[0]);
        const double sy = mk_block_sum(cy, red[1]);
        if (threadIdx.x == 0) {
            j.gx_acc[blockIdx.x] += sx;
            j.gy_acc[blockIdx.x] += sy;
        }
    }
#else
    (void)red;
#endif
}

/* Every reverse step of one segment [s0, s1) for one domain per workgroup.
 * j.yn is the segment's trajectory: y_{s0 + k} at j.yn + k * n_state * npad
 * for k = 0..s1-s0. j.mu_out holds mu of each cell (read and written in
 * place: a cell only reads its own); j.ab_out carries abar of each cell
 * from one launch to the next. flags: bit 0 = this segment ends the run (no
 * mu or abar of step N yet), bit 1 = this segment starts the run (add the
 * conductance terms of step 0 at the end). */
extern "C" __global__ void __launch_bounds__(MK_BT, MK_ADJ_WAVES)
mk_adj_block(const MkArgs a, const MkAdj j, const int s0, const int s1,
             const int flags)
{
    __shared__ Real vsh[2][MK_BCELLS];
    __shared__ Real ash[2][MK_BCELLS];
    __shared__ double red[2][MK_BT / 64];
    const long long off = a.dom_off[blockIdx.x];
    const int len = (int)(a.dom_off[blockIdx.x + 1] - off);
    const long long SN = (long long)MK_NS * a.npad;
    const bool last_seg = flags & 1, first_seg = flags & 2;
    double cx = 0.0, cy = 0.0;
    /* V(y_{s1}) and abar_{s1} (zero at the end of the run) */
    int cur = 0;
    const int nx = (int)a.nx, ny = (int)a.ny;
    for (int li = threadIdx.x; li < len; li += MK_BT) {
        const int c = a.dom_cells ? a.dom_cells[off + li] : (int)(off + li);
        vsh[0][li] = j.yn[(long long)(s1 - s0) * SN
                          + (long long)MK_IVM * a.npad + c];
        ash[0][li] = last_seg ? (Real)0 : j.ab_out[c];
    }
    __syncthreads();
    for (int s = s1 - 1; s >= s0; --s) {
        const Real* __restrict__ ys = j.yn + (long long)(s - s0) * SN;
        /* V(y_s) of the domain into the other buffer */
        for (int li = threadIdx.x; li < len; li += MK_BT) {
            const int c = a.dom_cells ? a.dom_cells[off + li]
                                      : (int)(off + li);
            vsh[cur ^ 1][li] = ys[(long long)MK_IVM * a.npad + c];
        }
        __syncthreads();
        const MkStep p = a.steps[s];
        const bool fresh = last_seg && s == s1 - 1;
        for (int li = threadIdx.x; li < len; li += MK_BT) {
            const int c = a.dom_cells ? a.dom_cells[off + li]
                                      : (int)(off + li);
            const int iy = (int)((unsigned)c / (unsigned)nx);
            const int ix = c - iy * nx;
            Real lam[MK_NS], y[MK_NS], mu[MK_NS], fv[MK_NFA], fb[MK_NFA], abo;
#pragma unroll
            for (int i = 0; i < MK_NS; ++i)
                lam[i] = fresh ? (Real)0 : j.mu_out[(long long)i * a.npad + c];
            Real lv = mk_adj_loss(j, c, vsh[cur][li], s);
#if MK_COUPLING == 3
            Real idiff;
            double ds;
            lv += mk_adj_couple_graph(a, fresh ? nullptr : ash[cur],
                                      vsh[cur ^ 1], (int)(off + li), li,
                                      idiff, ds);
#else
            if (!fresh)
                lv += mk_adj_couple(a, vsh[cur], ash[cur], li, ix, iy, nx, ny,
                                    cx, cy);
#endif
            lam[MK_IVM] += lv;
#pragma unroll
            for (int i = 0; i < MK_NS; ++i)
                y[i] = ys[(long long)i * a.npad + c];
#pragma unroll
            for (int k = 0; k < MK_NF; ++k)
                fv[k] = a.fields[(long long)k * a.npad + c];
#if MK_COUPLING == 3
            const Real pace = mk_is_paced(a, c, ix, iy) ? p.pace : (Real)0;
            mk_cell_vjp(y, p.t, p.dt, pace, idiff, fv, lam, mu, &abo, fb);
            cx += (double)abo * ds;
#else
            mk_adj_cell(a, p, y, fv, vsh[cur ^ 1], li, ix, iy, nx, ny, lam,
                        mu, abo, fb);
#endif
#pragma unroll
            for (int i = 0; i < MK_NS; ++i)
                j.mu_out[(long long)i * a.npad + c] = mu[i];
            ash[cur ^ 1][li] = abo;
#pragma unroll
            for (int k = 0; k < MK_NF; ++k)
                j.gfield[(long long)k * a.npad + c] += (double)fb[k];
        }
        cur ^= 1;
        __syncthreads();
    }
    /* Carry abar_{s0} to the previous segment; at the start of the run add
     * the conductance terms of step 0 instead. */
    for (int li = threadIdx.x; li < len; li += MK_BT) {
        const int c = a.dom_cells ? a.dom_cells[off + li] : (int)(off + li);
        if (first_seg) {
            const int iy = (int)((unsigned)c / (unsigned)nx);
            (void)mk_adj_couple(a, vsh[cur], ash[cur], li, c - iy * nx, iy,
                                nx, ny, cx, cy);
        } else {
            j.ab_out[c] = ash[cur][li];
        }
    }
#if MK_COUPLING == 1 || MK_COUPLING == 3
    const double sx = mk_block_sum(cx, red[0]);
    const double sy = mk_block_sum(cy, red[1]);
    if (threadIdx.x == 0) {
        j.gx_acc[blockIdx.x] += sx;
        j.gy_acc[blockIdx.x] += sy;
    }
#else
    (void)red; (void)cx; (void)cy;
#endif
}

/* V at the probe cells of state yn (trace row s). */
extern "C" __global__ void __launch_bounds__(64)
mk_adj_probe(const MkArgs a, const MkAdj j, const int s)
{
    const int q = blockIdx.x * 64 + threadIdx.x;
    if (q >= j.n_probe) return;
    j.trace[(long long)s * j.n_probe + q] =
        (double)j.yn[(long long)MK_IVM * a.npad + j.probes[q]];
}

/* The field gradients in the caller's cell order, for the download:
 * dst[k * n + c] = src[k * npad + order[c]], k < nf, c < n (the host checks
 * 0 <= order[c] < n). */
extern "C" __global__ void __launch_bounds__(256)
mk_adj_gather(const double* __restrict__ src,
              const long long* __restrict__ order, double* __restrict__ dst,
              const long long n, const long long npad, const int nf)
{
    const long long total = n * nf;
    const long long stride = (long long)gridDim.x * 256;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total;
         i += stride) {
        const long long k = i / n;
        dst[i] = src[k * npad + order[i - k * n]];
    }
}

#if MK_ADJ_SHEET
/* ------------------------------------------------------------------------
 * Persistent reverse sweep on a 2D stencil sheet: every reverse step of a
 * segment [s0, s1) in one cooperative launch.
 *
 * Each workgroup owns a tile of 64 x MK_ATH cells (MK_ATH = 4 * MK_ACPT);
 * thread (lx, w) handles cells (x0 + lx, y0 + w * MK_ACPT + k), k <
 * MK_ACPT, one after the other. The registers are budgeted for MK_ADJ_SREG
 * workgroups per CU, no more than fit into LDS (MK_ADJ_SWAVES). mu of the tile stays in LDS
 * for the whole segment, abar of the tile and a one-cell ring around it too. The
 * potentials V_s and V_{s+1} come from the trajectory, complete in global
 * memory, so only abar crosses tiles: after each step a tile stores the
 * abar of its four edges as step-tagged words (the exchange of mk_sheet),
 * and before the next step each thread of its ring waits for its
 * neighbour's value of that step.
 *
 * A step has two phases. Phase 1 computes, for every cell of the tile, the
 * coupling transpose gx (abar_c - abar_x) + gy (...) from abar_{s+1} and
 * the cell's terms of dL/dgx, dL/dgy. After a barrier, phase 2 assembles
 * lam = mu_{s+1} + coupling + loss, applies the cell VJP at y_s and writes
 * mu_s and abar_s in place. The barrier orders every read of abar_{s+1}
 * before the first write of abar_s, so one abar buffer suffices.
 *
 * j.yn is the segment's trajectory (y_{s0 + k} at j.yn + k * n_state *
 * npad); j.mu_out and j.ab_out carry mu and abar between segments. flags:
 * bit 0 = this segment ends the run (mu, abar of step s1 are zero), bit 1 =
 * it starts the run (add the conductance terms of step 0 at the end). Every
 * wait is bounded (sh.spin_limit); on a timeout the tile sets sh.err and
 * returns, and its neighbours then time out too.
 * ---------------------------------------------------------------------- */
#define MK_ATH (4 * MK_ACPT)

/* Coupling transpose at the tile cell (r, lx) from abar in LDS (ring
 * included) and V_{s+1} in global memory; adds the cell's conductance
 * terms to cx, cy. Same arithmetic as mk_adj_couple on the grid. */
__device__ __forceinline__ Real mk_adj_sheet_couple(
    const MkArgs& a, const Real (*at)[66], const Real* __restrict__ V1,
    int c, int r, int lx, int ix, int iy, int nx, int ny, double& cx,
    double& cy)
{
    const Real ac = at[r + 1][lx + 1], v = V1[c];
    Real ax = (Real)0, ay = (Real)0, xs = (Real)0, ys = (Real)0;
    if (nx > 1) {
        if (ix > 0) { ax += ac - at[r + 1][lx]; xs += v - V1[c - 1]; }
        if (ix < nx - 1) { ax += ac - at[r + 1][lx + 2]; xs += v - V1[c + 1]; }
    }
    if (ny > 1) {
        if (iy > 0) { ay += ac - at[r][lx + 1]; ys += v - V1[c - nx]; }
        if (iy < ny - 1) { ay += ac - at[r + 2][lx + 1]; ys += v - V1[c + nx]; }
    }
    cx += (double)ac * (double)xs;
    cy += (double)ac * (double)ys;
    return a.gx * ax + a.gy * ay;
}

/* Value k of abar edge e (0 bottom row, 1 top row, 2 left column, 3 right
 * column) of a tile, slot of step parity par (the layout of mk_edge). */
__device__ __forceinline__ MkXWord* mk_adj_edge(const MkSheet& sh, int par,
                                                int tile, int e, int k)
{
    return sh.edges + (((long long)(par * sh.tiles_x * sh.tiles_y + tile) * 4
                        + e) * 64 + k) * MK_XW;
}

/* Waits until each neighbour in nb[4] has stored the abar edges of local
 * step `step` (tagged step; its edge facing this tile, value 0). Returns
 * false on a timeout. */
__device__ __forceinline__ bool mk_adj_sheet_wait(const MkSheet& sh,
                                                  const int nb[4], int step,
                                                  int* flag)
{
    if (threadIdx.x < 4) {
        /* the edge of neighbour t facing this tile is t ^ 1 */
        const int nbt = nb[threadIdx.x];
        Real v;
        if (nbt >= 0 &&
            !mk_tget(mk_adj_edge(sh, (step - 1) & 1, nbt, threadIdx.x ^ 1, 0),
                     step, sh.spin_limit, v)) {
            __hip_atomic_store(sh.err, 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            *flag = 1;
        }
    }
    __syncthreads();
    return !*flag;
}

/* The neighbours' abar edges of local step `step` (tagged step) into the
 * ring of at, each ring thread waiting for its own value. Returns false on
 * a timeout. */
__device__ __forceinline__ bool mk_adj_sheet_halo(
    const MkSheet& sh, const int nb[4], int step, Real (*at)[66], int* flag,
    int gx0, int gy0, int nx, int ny)
{
    const int par = (step - 1) & 1;
    const int t = threadIdx.x;
    int nbt = -1, e = 0, k = 0, lr = 0, lc = 0;
    if (t < 64) {
        nbt = nb[0]; e = 1; k = t; lr = 0; lc = t + 1;
    } else if (t < 128) {
        nbt = nb[1]; e = 0; k = t - 64; lr = MK_ATH + 1; lc = t - 63;
    } else if (t < 128 + MK_ATH) {
        nbt = nb[2]; e = 3; k = t - 128; lr = t - 127; lc = 0;
    } else if (t < 128 + 2 * MK_ATH) {
        nbt = nb[3]; e = 2; k = t - 128 - MK_ATH; lr = t - 127 - MK_ATH;
        lc = 65;
    }
    /* only cells of the sheet are written (not the columns of a partial
     * last tile column or the rows of a partial last tile row) */
    if (nbt >= 0 && (e < 2 ? gx0 + k < nx : gy0 + k < ny)) {
        Real v;
        if (mk_tget(mk_adj_edge(sh, par, nbt, e, k), step, sh.spin_limit, v)) {
            at[lr][lc] = v;
        } else {
            __hip_atomic_store(sh.err, 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            *flag = 1;
        }
    }
    __syncthreads();
    return !*flag;
}
extern "C" __global__ void __launch_bounds__(256, MK_ADJ_SREG)
mk_adj_sheet(const MkArgs a, const MkAdj j, const MkSheet sh, const int s0,
             const int s1, const int flags)
{
    __shared__ Real mul[MK_NS][MK_ATH][64];
    __shared__ Real at[MK_ATH + 2][66];
    __shared__ double red[2][4];
    __shared__ int wg_flag;
    if (threadIdx.x == 0) wg_flag = 0;
    const bool last_seg = flags & 1, first_seg = flags & 2;
    const int tile = blockIdx.x;
    const int tx = tile % sh.tiles_x, ty = tile / sh.tiles_x;
    const int lx = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nx = (int)a.nx, ny = (int)a.ny;
    const int ix = tx * 64 + lx, gy0 = ty * MK_ATH;
    const long long np = a.npad;
    const long long SN = (long long)MK_NS * np;
    /* lanes beyond the last column compute a copy of its cell and keep it to
     * themselves (waves of at most 8 active lanes are slow, see mk_sheet);
     * not with 8 cells per thread, where the sheet fills the device and the
     * guards cost every tile 1% */
#if MK_ACPT < 8
    const bool own = ix < nx;
    const int xc = own ? ix : nx - 1;
#else
    const int xc = ix;
#endif
    const int nb[4] = {ty > 0 ? tile - sh.tiles_x : -1,
                       ty + 1 < sh.tiles_y ? tile + sh.tiles_x : -1,
                       tx > 0 ? tile - 1 : -1,
                       tx + 1 < sh.tiles_x ? tile + 1 : -1};
    double cx = 0.0, cy = 0.0;

    /* mu and abar of step s1, with abar's ring from global memory */
    for (int k = 0; k < MK_ACPT; ++k) {
        const int r = w * MK_ACPT + k, iy = gy0 + r;
        const bool act = ix < nx && iy < ny;
        const int c = act ? ix + iy * nx : 0;
        for (int i = 0; i < MK_NS; ++i)
            mul[i][r][lx] = (act && !last_seg) ? j.mu_out[i * np + c] : (Real)0;
        at[r + 1][lx + 1] = (act && !last_seg) ? j.ab_out[c] : (Real)0;
    }
    {
        const int t = threadIdx.x;
        int hx = -1, hy = -1, lr = 0, lc = 0;
        if (t < 66) {
            hx = tx * 64 - 1 + t; hy = gy0 - 1; lr = 0; lc = t;
        } else if (t < 132) {
            hx = tx * 64 - 1 + (t - 66); hy = gy0 + MK_ATH; lr = MK_ATH + 1;
            lc = t - 66;
        } else if (t < 132 + MK_ATH) {
            hx = tx * 64 - 1; hy = gy0 + (t - 132); lr = t - 132 + 1; lc = 0;
        } else if (t < 132 + 2 * MK_ATH) {
            hx = tx * 64 + 64; hy = gy0 + (t - 132 - MK_ATH);
            lr = t - 132 - MK_ATH + 1; lc = 65;
        }
        if (t < 132 + 2 * MK_ATH)
            at[lr][lc] = (!last_seg && hx >= 0 && hy >= 0 && hx < nx && hy < ny)
                             ? j.ab_out[hx + hy * nx] : (Real)0;
    }
    __syncthreads();

    const int nsteps = s1 - s0;
    for (int i = 0; i < nsteps; ++i) {
        const int s = s1 - 1 - i;
        if (i > 0 && !mk_adj_sheet_halo(sh, nb, i, at, &wg_flag, tx * 64, gy0,
                                        nx, ny))
            return;
        const Real* __restrict__ ys = j.yn + (long long)(s - s0) * SN;
        const Real* __restrict__ V0 = ys + MK_IVM * np;       /* V_s */
        const Real* __restrict__ V1 = V0 + SN;                 /* V_{s+1} */
        /* Phase 1: coupling transpose from abar_{s+1} */
        Real lc[MK_ACPT];
#pragma unroll
        for (int k = 0; k < MK_ACPT; ++k) {
            const int r = w * MK_ACPT + k, iy = gy0 + r;
            lc[k] = (Real)0;
            if (ix < nx && iy < ny)
                lc[k] = mk_adj_sheet_couple(a, at, V1, ix + iy * nx, r, lx, ix,
                                            iy, nx, ny, cx, cy);
        }
        __syncthreads();
        /* Phase 2: lam, the cell VJP at y_s, mu_s and abar_s in place */
        const MkStep p = a.steps[s];
        const int par = i & 1;
#pragma unroll 1
        for (int k = 0; k < MK_ACPT; ++k) {
            const int r = w * MK_ACPT + k, iy = gy0 + r;
#if MK_ACPT < 8
            if (iy >= ny) continue;
#else
            if (!(ix < nx && iy < ny)) continue;
#endif
            const int c = xc + iy * nx;
            Real lam[MK_NS], y[MK_NS], mu[MK_NS], fv[MK_NFA], fb[MK_NFA], abo;
#pragma unroll
            for (int q = 0; q < MK_NS; ++q) {
                lam[q] = mul[q][r][lx];
                y[q] = ys[q * np + c];
            }
#pragma unroll
            for (int f = 0; f < MK_NF; ++f) fv[f] = a.fields[f * np + c];
#if MK_ACPT < 8
            Real lv = mk_adj_loss(j, c, V1[c], own ? s : -1);
#else
            Real lv = mk_adj_loss(j, c, V1[c], s);
#endif
            Real ck = (Real)0;
#pragma unroll
            for (int q = 0; q < MK_ACPT; ++q) if (q == k) ck = lc[q];
            lv += ck;
            lam[MK_IVM] += lv;
            mk_adj_cell(a, p, y, fv, V0, c, xc, iy, nx, ny, lam, mu, abo, fb);
#pragma unroll
            for (int q = 0; q < MK_NS; ++q) mul[q][r][lx] = mu[q];
            at[r + 1][lx + 1] = abo;
#if MK_ACPT < 8
            if (!own) continue;
#endif
            if (r == 0) mk_tput(mk_adj_edge(sh, par, tile, 0, lx), abo, i + 1);
            if (r == MK_ATH - 1)
                mk_tput(mk_adj_edge(sh, par, tile, 1, lx), abo, i + 1);
            if (lx == 0) mk_tput(mk_adj_edge(sh, par, tile, 2, r), abo, i + 1);
            if (lx == 63) mk_tput(mk_adj_edge(sh, par, tile, 3, r), abo, i + 1);
#pragma unroll
            for (int f = 0; f < MK_NF; ++f) j.gfield[f * np + c] += (double)fb[f];
        }
        /* the next step's barrier (after its halo) orders this step's
         * LDS writes before its reads */
    }
    /* mu and abar of step s0 for the previous segment; at the start of the
     * run, the conductance terms of step 0 instead */
    if (first_seg) {
        if (!mk_adj_sheet_halo(sh, nb, nsteps, at, &wg_flag, tx * 64, gy0, nx,
                               ny))
            return;
        const Real* __restrict__ V0 = j.yn + MK_IVM * np;
        for (int k = 0; k < MK_ACPT; ++k) {
            const int r = w * MK_ACPT + k, iy = gy0 + r;
            if (ix < nx && iy < ny)
                (void)mk_adj_sheet_couple(a, at, V0, ix + iy * nx, r, lx, ix,
                                          iy, nx, ny, cx, cy);
        }
    } else {
        /* A neighbour reads its launch-start ring from j.ab_out; it has
         * done so once it has finished its first step (with one step per
         * segment nothing else orders that read before these writes). */
        if (nsteps == 1 && !mk_adj_sheet_wait(sh, nb, 1, &wg_flag)) return;
        for (int k = 0; k < MK_ACPT; ++k) {
            const int r = w * MK_ACPT + k, iy = gy0 + r;
            if (!(ix < nx && iy < ny)) continue;
            const int c = ix + iy * nx;
            for (int q = 0; q < MK_NS; ++q) j.mu_out[q * np + c] = mul[q][r][lx];
            j.ab_out[c] = at[r + 1][lx + 1];
        }
    }
    /* Conductance partial sums: one per tile */
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        cx += __shfl_down(cx, o, 64);
        cy += __shfl_down(cy, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = cx;
        red[1][threadIdx.x >> 6] = cy;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        j.gx_acc[tile] += red[0][0] + red[0][1] + red[0][2] + red[0][3];
        j.gy_acc[tile] += red[1][0] + red[1][1] + red[1][2] + red[1][3];
    }
}
#endif

#if MK_ADJ_LIN
/* ------------------------------------------------------------------------
 * Linear reverse pass: a line of cells, or uncoupled cells, on the tiles of
 * mk_strand.
 *
 * A reverse step is linear in lam, and its matrix depends on the trajectory
 * alone, which is complete when the reverse pass starts. Only the products
 * with lam have to be taken in turn; the cell VJPs, which are nearly all of
 * the work (2,000 instructions in double precision, 9 us per step one after
 * the other), need not be. mk_adj_jac evaluates the Jacobian's entries of
 * every cell and step of a range of steps at once, one VJP per state (1,000
 * cells x 200 steps fill the device); mk_adj_lin then walks the steps with
 * one lane per cell: about 30 multiply-adds, the entries loaded four steps
 * ahead. LR1991, 1,000 cells in double precision: 9.2 us per reverse step on
 * mk_adj_step, 1.3 here (entries and walk).
 *
 * Entry e of cell c at step s: jac[((s - base) * MK_NE + e) * npad + c].
 * Rows of the Jacobian first (state i' by state j, existing entries only),
 * then its derivatives by the fields, by the diffusion current, and last
 * the loss term dL/dV(y_{s+1}) and dI/dgx at y_s.
 * ---------------------------------------------------------------------- */
typedef MkLinT<Real> MkLin;

/* read by the host library when it loads the module */
extern "C" __device__ const int mk_entries = MK_NE;

__device__ __forceinline__ constexpr int mk_bits(unsigned long long m)
{
    int n = 0;
    for (; m; m &= m - 1) ++n;
    return n;
}

/* Steps s0 + blockIdx.x / tiles, cells of tile blockIdx.x % tiles. j.yn is
 * y_{s0} of the trajectory. */
extern "C" __global__ void __launch_bounds__(256)
mk_adj_jac(const MkArgs a, const MkAdj j, const MkLin ln, const int s0,
           const int tiles)
{
    const int k = blockIdx.x / tiles;
    const int c = (blockIdx.x - k * tiles) * 256 + threadIdx.x;
    if (c >= (int)a.n) return;
    const long long np = a.npad, SN = (long long)MK_NS * np;
    const Real* __restrict__ ys = j.yn + k * SN;
    const Real* __restrict__ V = ys + MK_IVM * np;
    const MkStep p = a.steps[s0 + k];
    Real* __restrict__ o = ln.jac + (long long)(s0 + k - ln.base) * MK_NE * np
                           + c;
    Real y[MK_NS], fv[MK_NFA], lam[MK_NS], mu[MK_NS], fb[MK_NFA], abo;
#pragma unroll
    for (int i = 0; i < MK_NS; ++i) y[i] = ys[i * np + c];
#pragma unroll
    for (int f = 0; f < MK_NF; ++f) fv[f] = a.fields[f * np + c];
    Real idiff = (Real)0, xs = (Real)0;
#if MK_COUPLING == 1
    idiff = mk_stencil(V, c, c, 0, (int)a.n, 1, a.gx, a.gy);
    if (c > 0) xs += V[c] - V[c - 1];
    if (c < (int)a.n - 1) xs += V[c] - V[c + 1];
#elif MK_COUPLING == 2
    idiff = mk_hetero(V, a.gx_field, a.gy_field, c, c, 0, (int)a.n, 1);
#endif
    const int nx = (int)a.nx;
    const Real pace = mk_is_paced(a, c, c % nx, c / nx) ? p.pace : (Real)0;
    Real loss = (Real)0;
    const int q = j.probe_of[c];
    if (q >= 0)
        loss = (Real)(2.0 * ((double)V[SN + c]
                             - j.target[(long long)(s0 + k) * j.n_probe + q]));
    o[(long long)(MK_NE - 2) * np] = loss;
    o[(long long)(MK_NE - 1) * np] = xs;
#pragma unroll 1
    for (int i = 0; i < MK_NS; ++i) {
#pragma unroll
        for (int r = 0; r < MK_NS; ++r) lam[r] = r == i ? (Real)1 : (Real)0;
        mk_cell_vjp(y, p.t, p.dt, pace, idiff, fv, lam, mu, &abo, fb);
        const unsigned long long jm = mk_jmask[i], fm = mk_fmask[i];
        int e = mk_jrow[i];
#pragma unroll
        for (int r = 0; r < MK_NS; ++r)
            if (jm >> r & 1) o[(long long)e++ * np] = mu[r];
        e = mk_frow[i];
#pragma unroll
        for (int f = 0; f < MK_NF; ++f)
            if (fm >> f & 1) o[(long long)e++ * np] = fb[f];
        if (mk_dmask >> i & 1)
            o[(long long)(MK_D0
                          + __builtin_popcountll(
                                mk_dmask & ((1ull << i) - 1))) * np] = abo;
    }
}

/* Value i (states, then abar) of the kth of the outer cells of a tile's side
 * e, slot of exchange parity par (as mk_sedge). */
__device__ __forceinline__ MkXWord* mk_ledge(const MkLin& ln, int par,
                                             int tile, int e, int i, int k)
{
    return ln.edges + ((((long long)(par * ln.tiles + tile) * 2 + e)
                        * (MK_NS + 1) + i) * 32 + k) * MK_XW;
}

/* Reverse steps s1 - 1 .. s0 from mu, abar of step s1 (j.mu_in, j.ab_in) to
 * those of step s0 (j.mu_out, j.ab_out: other buffers, a neighbour may still
 * be reading its launch-start halo). */
extern "C" __global__ void __launch_bounds__(64)
mk_adj_lin(const MkArgs a, const MkAdj j, const MkLin ln, const int s0,
           const int s1)
{
    constexpr int AHEAD = MK_NE <= 32 ? 4 : 2;
    const int lane = threadIdx.x, tile = blockIdx.x;
    const long long n = a.n, np = a.npad;
    const long long c0 = (long long)tile * ln.width;
    const int len = (int)(n - c0 < ln.width ? n - c0 : ln.width);
    const long long cl = c0 + lane - ln.halo;
    const long long c = cl < 0 ? 0 : cl >= n ? n - 1 : cl;
    const bool own = lane >= ln.halo && lane < ln.halo + len;
    Real mu[MK_NS], ab = (Real)0;
#pragma unroll
    for (int i = 0; i < MK_NS; ++i)
        mu[i] = ln.fresh ? (Real)0 : j.mu_in[i * np + c];
    if (!ln.fresh) ab = j.ab_in[c];
#if MK_COUPLING == 2
    const Real gl = c > 0 ? a.gx_field[c - 1] : (Real)0;
    const Real gr = c < n - 1 ? a.gx_field[c] : (Real)0;
#endif
    double gf[MK_NFA], cx = 0.0, loss = 0.0;
#pragma unroll
    for (int f = 0; f < MK_NFA; ++f) gf[f] = 0.0;
    const Real* __restrict__ jc = ln.jac + c;
    Real E[AHEAD][MK_NE];
#pragma unroll
    for (int b = 0; b < AHEAD; ++b) {
        const int s = s1 - 1 - b < s0 ? s0 : s1 - 1 - b;
#pragma unroll
        for (int e = 0; e < MK_NE; ++e)
            E[b][e] = jc[((long long)(s - ln.base) * MK_NE + e) * np];
    }
    int left = ln.halo, sup = 0;
    for (int sb = s1 - 1; sb >= s0; sb -= AHEAD) {
#pragma unroll
        for (int b = 0; b < AHEAD; ++b) {
            const int s = sb - b;
            if (s < s0) break;
            Real lam[MK_NS];
#pragma unroll
            for (int i = 0; i < MK_NS; ++i) lam[i] = mu[i];
            Real lv = E[b][MK_NE - 2];
            loss += 0.25 * (double)lv * (double)lv;
#if MK_COUPLING == 1 || MK_COUPLING == 2
            {
                const Real al = __shfl_up(ab, 1, 64);
                const Real ar = __shfl_down(ab, 1, 64);
#if MK_COUPLING == 1
                Real ax = (Real)0;
                if (c > 0) ax += ab - al;
                if (c < n - 1) ax += ab - ar;
                lv += a.gx * ax;
#else
                if (c > 0) lv += gl * (ab - al);
                if (c < n - 1) lv += gr * (ab - ar);
#endif
            }
#endif
            lam[MK_IVM] += lv;
            /* products with an adjoint of 0 are 0, also where an entry is
             * not finite (mk_gmul) */
            bool nz[MK_NS];
#pragma unroll
            for (int i = 0; i < MK_NS; ++i) nz[i] = lam[i] != (Real)0;
#pragma unroll
            for (int r = 0; r < MK_NS; ++r) {
                Real m = (Real)0;
#pragma unroll
                for (int i = 0; i < MK_NS; ++i) {
                    if (!(mk_jmask[i] >> r & 1)) continue;
                    const int e = mk_jrow[i]
                                  + mk_bits(mk_jmask[i] & ((1ull << r) - 1));
                    m = __builtin_fma(lam[i], nz[i] ? E[b][e] : (Real)0, m);
                }
                mu[r] = m;
            }
            Real abn = (Real)0;
#pragma unroll
            for (int i = 0; i < MK_NS; ++i) {
                if (!(mk_dmask >> i & 1)) continue;
                const int e = MK_D0 + mk_bits(mk_dmask & ((1ull << i) - 1));
                abn = __builtin_fma(lam[i], nz[i] ? E[b][e] : (Real)0, abn);
            }
            ab = abn;
#pragma unroll
            for (int f = 0; f < MK_NF; ++f) {
#pragma unroll
                for (int i = 0; i < MK_NS; ++i) {
                    if (!(mk_fmask[i] >> f & 1)) continue;
                    const int e = mk_frow[i]
                                  + mk_bits(mk_fmask[i] & ((1ull << f) - 1));
                    gf[f] = __builtin_fma(lam[i],
                                          nz[i] ? E[b][e] : (Real)0, gf[f]);
                }
            }
            cx = __builtin_fma((double)ab, (double)E[b][MK_NE - 1], cx);
            /* the entries of the step AHEAD steps on */
            {
                const int sn = s - AHEAD < s0 ? s0 : s - AHEAD;
#pragma unroll
                for (int e = 0; e < MK_NE; ++e)
                    E[b][e] = jc[((long long)(sn - ln.base) * MK_NE + e) * np];
            }
#if MK_COUPLING != 0
            if (--left == 0 && ln.tiles > 1 && s > s0) {
                /* the exchange of mk_strand, for mu and abar */
                left = ln.halo;
                const int step = ln.g0 + ++sup, par = step & 1;
                const bool el = own && lane < 2 * ln.halo && tile > 0;
                const bool er = own && lane >= len && tile + 1 < ln.tiles;
#pragma unroll
                for (int i = 0; i <= MK_NS; ++i) {
                    const Real v = i < MK_NS ? mu[i < MK_NS ? i : 0] : ab;
                    if (el)
                        mk_tput(mk_ledge(ln, par, tile, 0, i, lane - ln.halo),
                                v, step);
                    if (er)
                        mk_tput(mk_ledge(ln, par, tile, 1, i, lane - len), v,
                                step);
                }
                const bool hl = lane < ln.halo && tile > 0;
                const bool hr = lane >= ln.halo + len
                                && tile + 1 < ln.tiles && cl < n;
                bool bad = false;
                if (hl || hr) {
                    MkXWord* e = hl ? mk_ledge(ln, par, tile - 1, 1, 0, lane)
                                    : mk_ledge(ln, par, tile + 1, 0, 0,
                                               lane - ln.halo - len);
                    for (int spins = 0;; ++spins) {
                        MkXWord w[(MK_NS + 1) * MK_XW];
                        bool ready = true;
#pragma unroll
                        for (int i = 0; i < (MK_NS + 1) * MK_XW; ++i)
                            w[i] = __hip_atomic_load(
                                e + i / MK_XW * 32 * MK_XW + i % MK_XW,
                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                        for (int i = 0; i < (MK_NS + 1) * MK_XW; ++i)
                            ready = ready && (int)(w[i] >> 32) >= step;
                        if (ready) {
#pragma unroll
                            for (int i = 0; i <= MK_NS; ++i) {
                                const Real v = (Real)__longlong_as_double(
                                    (long long)(((w[i * MK_XW] & 0xffffffffull)
                                                 << 32)
                                                | (w[i * MK_XW + MK_XW - 1]
                                                   & 0xffffffffull)));
                                if (i < MK_NS) mu[i < MK_NS ? i : 0] = v;
                                else ab = v;
                            }
                            break;
                        }
                        if (spins >= ln.spin_limit) {
                            __hip_atomic_store(ln.err, 1, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                            bad = true;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                if (__any(bad)) return;
            }
#endif
        }
    }
    if (own) {
#pragma unroll
        for (int i = 0; i < MK_NS; ++i) j.mu_out[i * np + c] = mu[i];
        j.ab_out[c] = ab;
#pragma unroll
        for (int f = 0; f < MK_NF; ++f) j.gfield[f * np + c] += gf[f];
        const int q = j.probe_of[c];
        if (q >= 0) j.loss_acc[q] += loss;
    } else {
        cx = 0.0;
    }
#if MK_COUPLING == 1
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cx += __shfl_down(cx, o, 64);
    if (lane == 0) j.gx_acc[tile] += cx;
#else
    (void)cx; (void)sup; (void)left;
#endif
}
#endif
