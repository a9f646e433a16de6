// amr_ib.hpp -- coarse/fine transfer and immersed-boundary forcing: host plans, device tables
// and kernels.  Included by zlh_api.hip after its allocation helpers.
#pragma once

namespace zlh {

// ----------------------------------------------------------------------------------------------
// kernels
// ----------------------------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ void macro_feq_double(const double *f, int compressible, double &rho, double *u,
                                                 double *feq) {
    using L = Lattice<D>;
    constexpr int Q = L::Q;
    double r = f[0], ux = 0, uy = 0, uz = 0;
    for (int q = 1; q < Q; ++q) {
        r += f[q];
        ux += L::cx[q] * f[q];
        uy += L::cy[q] * f[q];
        if (D == 3) uz += L::cz[q] * f[q];
    }
    if (compressible) { ux /= r; uy /= r; if (D == 3) uz /= r; }
    rho = r; u[0] = ux; u[1] = uy; u[2] = uz;
    const double usq = ux * ux + uy * uy + (D == 3 ? uz * uz : 0.);
    for (int q = 0; q < Q; ++q) {
        double cu = ux * L::cx[q] + uy * L::cy[q];
        if (D == 3) cu += uz * L::cz[q];
        feq[q] = compressible ? L::w[q] * r * (1. + 3. * cu + 4.5 * cu * cu - 1.5 * usq)
                              : L::w[q] * (r + 3. * cu + 4.5 * cu * cu - 1.5 * usq);
    }
}

// NodeInfoCoarse2fine (lbm_grid_interface.cpp:570-588) + PostStreamCoarse2Fine
// (lbm_collision_models.cpp:244-251): the row of a coarse node, in storage form, as an
// interpolation stencil takes it: feq + tau_ratio (f - feq)
template <int D, typename T, bool SHIFT>
__device__ __forceinline__ void rescale_row(T *row, double tau_ratio, int compressible) {
    constexpr int Q = Lattice<D>::Q;
    if constexpr (SHIFT) {
        // FP32 / BF16 storage: in FP32 on the stored deviations f - w, whose equilibrium
        // feq - w needs no cancellation
        float f[Q], rho, drho, u[3];
        load_row<D>(row, 0, f);
        macro<D, true, float>(f, nullptr, 0.f, 0, compressible, rho, drho, u);
        const float usq = u[0] * u[0] + u[1] * u[1] + (D == 3 ? u[2] * u[2] : 0.f);
        const float tr = (float)tau_ratio;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const float feq = feq_stored<D, true, float>(q, rho, drho, u[0], u[1], u[2], usq, compressible);
            f[q] = __builtin_fmaf(tr, f[q] - feq, feq);
        }
        store_row<D>(row, 0, f);
    } else {
        double f[Q], feq[Q], rho, u[3];
        load_row<D>(row, 0, f);
        macro_feq_double<D>(f, compressible, rho, u, feq);
#pragma unroll
        for (int q = 0; q < Q; ++q) f[q] = feq[q] + tau_ratio * (f[q] - feq[q]);
        store_row<D>(row, 0, f);
    }
}

// Where row_table says so: the rows of the interpolation as a table, [n_src + n_fb][S], the
// rescaled coarse sources and then plain copies of the fine nodes that stand in for missing coarse
// ones.  MID (after an odd fine substep): each coarse row is the mean of the row computed now and
// the row `prev` of the last synchronised transfer, i.e. of the coarse state before and after the
// coarse level's last step; fallback rows stay current copies.
template <int D, typename T, bool SHIFT, bool MID>
__global__ __launch_bounds__(256) void k_c2f_sources(int64_t n_src, int64_t n_fb, const int32_t *src_ai,
                                                     const T *aux_c, const int32_t *fb_ai, const T *aux_f,
                                                     double tau_ratio, int compressible, const T *__restrict__ prev,
                                                     T *src_f) {
    constexpr int Q = Lattice<D>::Q, S = aux_stride<D>();
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= n_src + n_fb) return;
    RowUnit<T> unit[S / RowUnit<T>::n];
    T *row = unit[0].v;
    T v[Q];
    load_row<D>(r < n_src ? aux_c : aux_f, r < n_src ? src_ai[r] : fb_ai[r - n_src], v);
    store_row<D>(row, 0, v);
    if (r < n_src) {
        rescale_row<D, T, SHIFT>(row, tau_ratio, compressible);
        if constexpr (MID) {
            T p[Q];
            load_row<D>(prev, r, p);
#pragma unroll
            for (int q = 0; q < Q; ++q) row[q] = T(0.5 * (double(p[q]) + double(row[q])));
        }
    }
    load_row<D>(row, 0, v);
    store_row<D>(src_f, r, v);
}

// InterpolationLagrangian{2D,3D} (grid/grid_interpolation.cpp:224-304, 433-525): each ghost node
// is the weighted sum of its contributors, accumulated in stencil order.  Ghost nodes are listed
// by contributor count (the parity of the node's coordinates fixes it: 4 Lagrange weights per odd
// coordinate, 1 per even one), stably, so the threads of a wavefront loop equally often; inside
// one count they keep Morton order, so the nodes of a workgroup are neighbours.  A
// workgroup takes a group of at most 256 / PARTS ghost nodes, as many as keep its staged data
// within the LDS budget: it first copies the union of their rows and their contributor words into
// LDS, then each ghost node is summed from LDS by PARTS threads of 5 directions (D2Q9: 5 and 4).
// DIRECT: a staged row is an aux row, of the coarse level (index >= 0; rescaled in LDS, one thread
// a row) or of the fine level (~index: a fallback node); rows that several groups stage are
// rescaled by each, a few hundred operations against a launch over all rows (4.8 us on small
// levels, 10.8 on a 3M-node one) and their round trip through memory.  Otherwise
// (row_table) a row of the table src_f.  A contributor is one 32-bit word {LDS row offset, FP16
// weight}: the tensor-product Lagrange weights are products of -1/16, 9/16, 1/2 and 1, dyadic
// rationals exact in FP16 (the host checks every one).
constexpr int kGatherDirs = 5;
constexpr size_t kGatherLdsBudget = 20 * 1024;
constexpr int kGatherMaxRows = 768;   // staged rows of one group (row offsets fit the word's 16 bits)
constexpr int64_t kGatherChunk = 2048;   // ghost nodes sorted by contributor count together
// what a gather reads: the staged rows' indices and the arrays they name, the fine level's aux rows
template <typename T>
struct GatherArgs {
    const GatherGroup *groups;
    const int32_t *tgt_ai, *begin;
    const uint32_t *contrib;
    const int32_t *rows;      // DIRECT: aux rows; else rows of src_f
    const T *src_f;           // DIRECT: the coarse level's aux rows; else the table
    T *aux_f;
    double tau_ratio;
    int compressible;
};

template <int D, typename T, bool SHIFT, bool DIRECT>
__device__ __forceinline__ void gather_group(int64_t gi, unsigned char *lds_raw, const GatherArgs<T> &a) {
    constexpr int Q = Lattice<D>::Q;
    constexpr int NQ = kGatherDirs;
    constexpr int PARTS = (Q + NQ - 1) / NQ;
    constexpr int S = aux_stride<D>();
    static_assert(PARTS * NQ <= S, "every thread reads NQ entries of a row, pads included");
    const GatherGroup G = a.groups[gi];
    T *__restrict__ aux_f = a.aux_f;
    const int32_t nr = G.r1 - G.r0, nc = G.c1 - G.c0;
    T *rowbuf = reinterpret_cast<T *>(lds_raw);                                  // [nr][S]
    uint32_t *cbuf = reinterpret_cast<uint32_t *>(lds_raw + (((size_t)nr * S * sizeof(T) + 15) & ~(size_t)15));
    const int local = threadIdx.x / PARTS;
    const int q0 = (threadIdx.x - local * PARTS) * NQ;
    const int32_t t = G.t0 + local;
    const bool active = t < G.t1;
    // every load below is issued before the first LDS write that waits on it; none depends on
    // an earlier one except a row's data on its entry
    int32_t kb = 0, ke = 0, ai = 0;
    if (active) {
        kb = a.begin[t] - G.c0;
        ke = a.begin[t + 1] - G.c0;
        ai = a.tgt_ai[t];
    }
    for (int cb = 0; cb < nc; cb += 4 * 256) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = cb + j * 256 + (int)threadIdx.x;
            w[j] = k < nc ? a.contrib[G.c0 + k] : 0u;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = cb + j * 256 + (int)threadIdx.x;
            if (k < nc) cbuf[k] = w[j];
        }
    }
    // the rows in units of 16 bytes (8 in BF16), consecutive threads on consecutive units
    constexpr int U = S / RowUnit<T>::n, kBatch = 4;
    const int nu = nr * U;
    RowUnit<T> *units = reinterpret_cast<RowUnit<T> *>(rowbuf);
    for (int ub = 0; ub < nu; ub += kBatch * 256) {
        int32_t g[kBatch];
        RowUnit<T> v[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int e = ub + j * 256 + (int)threadIdx.x;
            g[j] = a.rows[G.r0 + (e < nu ? e : nu - 1) / U];
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int e = ub + j * 256 + (int)threadIdx.x;
            const int ec = e < nu ? e : nu - 1;
            const T *base = DIRECT && g[j] < 0 ? aux_f : a.src_f;
            const int64_t row = DIRECT && g[j] < 0 ? ~g[j] : g[j];
            v[j] = reinterpret_cast<const RowUnit<T> *>(base)[row * U + (ec - (ec / U) * U)];
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int e = ub + j * 256 + (int)threadIdx.x;
            if (e < nu) units[e] = v[j];
        }
    }
    if constexpr (DIRECT) {
        __syncthreads();
        for (int r = threadIdx.x; r < nr; r += 256)
            if (a.rows[G.r0 + r] >= 0) rescale_row<D, T, SHIFT>(rowbuf + r * S, a.tau_ratio, a.compressible);
    }
    __syncthreads();
    if (!active) return;
    // a contributor word is {row * S (low 16 bits), FP16 weight (high 16 bits)}; the pad entry
    // of the last part is summed like the others and never stored
    auto weight = [](uint32_t cw) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(cw >> 16)); };
    double acc[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) acc[i] = 0.;
    if constexpr (SHIFT) {
        // FP32 / BF16 storage holds f - w.  sum c (f~ + w) - w = sum c f~ + w (sum c - 1): the
        // weights are multiples of 2^-12 of magnitude <= 1, so their sum is exact in FP32.
        // Runs of four products are summed in FP32 (rounding error a few 2^-24 of the run), the
        // runs in FP64.
        float sum = 0.f;
        int32_t k = kb;
        for (; k + 4 <= ke; k += 4) {
            float c[4];
            const T *row[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t cw = cbuf[k + j];
                c[j] = weight(cw);
                row[j] = rowbuf + (cw & 0xffffu) + q0;
            }
            sum += (c[0] + c[1]) + (c[2] + c[3]);
#pragma unroll
            for (int i = 0; i < NQ; ++i) {
                float run = c[0] * float(row[0][i]);
                run = __builtin_fmaf(c[1], float(row[1][i]), run);
                run = __builtin_fmaf(c[2], float(row[2][i]), run);
                run = __builtin_fmaf(c[3], float(row[3][i]), run);
                acc[i] += (double)run;
            }
        }
        for (; k < ke; ++k) {
            const uint32_t cw = cbuf[k];
            const float c = weight(cw);
            const T *row = rowbuf + (cw & 0xffffu) + q0;
            sum += c;
#pragma unroll
            for (int i = 0; i < NQ; ++i) acc[i] += (double)(c * float(row[i]));
        }
#pragma unroll
        for (int i = 0; i < NQ; ++i)
            if (q0 + i < Q) aux_f[(int64_t)ai * S + q0 + i] = T(acc[i] + Lattice<D>::w[q0 + i] * ((double)sum - 1.));
    } else {
        // FP64 storage: every product and sum in FP64, in stencil order
#pragma unroll 4
        for (int32_t k = kb; k < ke; ++k) {
            const uint32_t cw = cbuf[k];
            const double c = (double)weight(cw);
            const T *row = rowbuf + (cw & 0xffffu) + q0;
#pragma unroll
            for (int i = 0; i < NQ; ++i) acc[i] = acc[i] + c * double(row[i]);
        }
#pragma unroll
        for (int i = 0; i < NQ; ++i)
            if (q0 + i < Q) aux_f[(int64_t)ai * S + q0 + i] = T(acc[i]);
    }
}

template <int D, typename T, bool SHIFT, bool DIRECT>
__global__ __launch_bounds__(256) void k_c2f_gather(int64_t n_groups, GatherArgs<T> a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int64_t gi = xcd_group(n_groups);   // groups are in spatial order: an XCD takes a range
    if (gi < 0) return;
    gather_group<D, T, SHIFT, DIRECT>(gi, lds_raw, a);
}

// NodeInfoFine2Coarse (lbm_grid_interface.cpp:594-610) + PostStreamFine2Coarse
// (lbm_collision_models.cpp:259-267): rho, u of the fine node's last collision
template <typename T>
struct F2cArgs {
    int64_t n;
    const int32_t *coarse_ai, *fine_ai;
    const T *fine_f;
    const double *fine_macro;
    double tau_ratio;
    int compressible;
    T *coarse_f;
};

template <int D, typename T, bool SHIFT>
__device__ __forceinline__ void f2c_node(int64_t p, const F2cArgs<T> &a) {
    using L = Lattice<D>;
    constexpr int Q = L::Q;
    const int64_t i = a.fine_ai[p], j = a.coarse_ai[p];
    if constexpr (SHIFT) {
        // FP32 / BF16 storage: in FP32 on the stored deviations f - w
        float f[Q];
        load_row<D>(a.fine_f, i, f);
        const float rho = (float)a.fine_macro[i * 4], ux = (float)a.fine_macro[i * 4 + 1];
        const float uy = (float)a.fine_macro[i * 4 + 2], uz = D == 3 ? (float)a.fine_macro[i * 4 + 3] : 0.f;
        const float drho = (float)(a.fine_macro[i * 4] - 1.);
        const float usq = ux * ux + uy * uy + (D == 3 ? uz * uz : 0.f);
        const float tr = (float)a.tau_ratio;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const float feq = feq_stored<D, true, float>(q, rho, drho, ux, uy, uz, usq, a.compressible);
            f[q] = __builtin_fmaf(tr, f[q] - feq, feq);
        }
        store_row<D>(a.coarse_f, j, f);
        return;
    }
    double f[Q];
    load_row<D>(a.fine_f, i, f);
    const double rho = a.fine_macro[i * 4], ux = a.fine_macro[i * 4 + 1], uy = a.fine_macro[i * 4 + 2];
    const double uz = D == 3 ? a.fine_macro[i * 4 + 3] : 0.;
    const double usq = ux * ux + uy * uy + (D == 3 ? uz * uz : 0.);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        double cu = ux * L::cx[q] + uy * L::cy[q];
        if (D == 3) cu += uz * L::cz[q];
        const double feq = a.compressible ? L::w[q] * rho * (1. + 3. * cu + 4.5 * cu * cu - 1.5 * usq)
                                          : L::w[q] * (rho + 3. * cu + 4.5 * cu * cu - 1.5 * usq);
        f[q] = feq + a.tau_ratio * (f[q] - feq);
    }
    store_row<D>(a.coarse_f, j, f);
}

template <int D, typename T, bool SHIFT>
__global__ void k_f2c(F2cArgs<T> a) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < a.n) f2c_node<D, T, SHIFT>(p, a);
}

// The gather and the fine-to-coarse copy of one exchange in one launch, where the host found
// them independent (no fine node is both a gather target and a fine-to-coarse source, no coarse
// node both a staged source and a fine-to-coarse target): blocks below nb_gather (a multiple of 8)
// are the gather's, in its XCD-aware order; the blocks after them take 256 fine-to-coarse nodes
// each.
template <int D, typename T, bool SHIFT, bool DIRECT>
__global__ __launch_bounds__(256) void k_c2f_gather_f2c(int64_t nb_gather, int64_t n_groups, GatherArgs<T> g,
                                                        F2cArgs<T> c) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int64_t bid = blockIdx.x;
    if (bid < nb_gather) {
        const int64_t per = nb_gather >> 3;
        const int64_t gi = (bid & 7) * per + (bid >> 3);
        if (gi >= n_groups) return;
        gather_group<D, T, SHIFT, DIRECT>(gi, lds_raw, g);
    } else {
        const int64_t p = (bid - nb_gather) * 256 + threadIdx.x;
        if (p < c.n) f2c_node<D, T, SHIFT>(p, c);
    }
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// immersed boundary: one wavefront per marker; lanes hold the stencil nodes.  Each lane
// recomputes its node's velocity with the remaining (constant) force (the lazy reset,
// immersed_boundary.cpp:76-85, 284-296), then interpolation by a wavefront reduction and the
// Lagrangian force F = k (U - u_ref) (DirectForcingScheme{2D,3D}, immersed_boundary.cpp:108-364).
// A node lies in about eleven markers' stencils, so its velocity is computed as often; its row is
// five vector loads, and a launch over the nodes that stored the velocities took 4.8 us beside the
// markers' 4.7 (1,810 markers).
template <int D, typename T, typename C, bool SHIFT>
__global__ __launch_bounds__(256) void k_ib_markers(int64_t n_markers, int support, const int32_t *node_ai,
                                                    const double *weight, const T *aux_f, const double *marker_vel,
                                                    double stiffness, double *marker_force, StepParams p) {
    const int64_t m = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (m >= n_markers) return;
    int32_t ai = -1;
    double w = 0.;
    if (lane < support) {
        ai = node_ai[m * support + lane];
        w = weight[m * support + lane];
    }
    double u[3] = {0., 0., 0.};
    if (ai >= 0) {
        C f[Lattice<D>::Q];
        load_row<D>(aux_f, ai, f);
        C F[3] = {C(p.const_force[0]), C(p.const_force[1]), C(p.const_force[2])};
        C rho, drho, v[3];
        macro<D, SHIFT, C>(f, F, C(p.dt), 1, p.compressible, rho, drho, v);
        for (int a = 0; a < D; ++a) u[a] = double(v[a]) * w;
    }
    double fm[3] = {0., 0., 0.};
    for (int a = 0; a < D; ++a) {
        const double ur = wave_sum(u[a]);
        fm[a] = stiffness * (marker_vel[m * 3 + a] - ur);
    }
    if (lane == 0)
        for (int a = 0; a < 3; ++a) marker_force[m * 3 + a] = fm[a];
}

// ----------------------------------------------------------------------------------------------
// host plans
// ----------------------------------------------------------------------------------------------
// one axis of FindNodesInPeriodicRegionCorner (grid/sfbitset_aux.cpp:380-557, 2493-2878):
// coordinates of the 2L region entries whose local index L-1 is `start`; entries past a
// non-periodic domain edge are -1; at a periodic edge the walk continues from the opposite
// domain plane, which duplicates the edge plane.  Returns the axis' bound on the valid half length.
inline int region_axis(int64_t start, int L, int64_t lo, int64_t hi, bool per_lo, bool per_hi, int64_t *seq) {
    int index_min = L;
    for (int k = 0; k < 2 * L; ++k) seq[k] = -1;
    int64_t v = start;
    for (int ix = 0; ix < L; ++ix) {
        seq[L - ix - 1] = v;
        if (v == lo) {
            if (per_lo) v = hi + 1;
            else { index_min = std::min(index_min, ix + 1); break; }
        }
        v = v > 0 ? v - 1 : v;
    }
    v = start;
    bool go = true;
    if (v == hi) {
        if (per_hi) v = lo > 0 ? lo - 1 : lo;
        else { index_min = 0; go = false; }
    }
    if (go) {
        for (int ix = 0; ix < L; ++ix) {
            v = v + 1;
            seq[L + ix] = v;
            if (v == hi) {
                if (per_hi) v = lo > 0 ? lo - 1 : lo;
                else { index_min = std::min(index_min, ix + 1); break; }
            }
        }
    }
    return index_min;
}

// one axis of FindNodesInPeriodicRegionCornerOverlap (grid/sfbitset_aux.cpp:581-850,
// 2893-3825), the immersed boundary's region walk in a periodic domain
// (immersed_boundary.cpp:250-256): a walk reaching a periodic domain plane continues past its
// duplicate on the opposite side (lo -> hi - 1, hi -> lo + 1), and the duplicate is returned in
// twin[] at the plane node's entry (-1 elsewhere); it receives that entry's spread force too
// (immersed_boundary.cpp:341-363).  Every duplicate takes its own entry's weight; the reference's
// other weights at a start node on a maximum plane and at the region's first and last rows are
// not reproduced.
inline int region_axis_twin(int64_t start, int L, int64_t lo, int64_t hi, bool per_lo, bool per_hi, int64_t *seq,
                            int64_t *twin) {
    int index_min = L;
    for (int k = 0; k < 2 * L; ++k) seq[k] = twin[k] = -1;
    int64_t v = start;
    for (int ix = 0; ix < L; ++ix) {
        seq[L - ix - 1] = v;
        if (v == lo) {
            if (per_lo) { twin[L - ix - 1] = hi; v = hi; }
            else { index_min = std::min(index_min, ix + 1); break; }
        }
        v = v - 1;
    }
    v = start;
    if (v == hi) {
        if (per_hi) { twin[L - 1] = lo; v = lo; }
        else return 0;
    }
    for (int ix = 0; ix < L; ++ix) {
        v = v + 1;
        seq[L + ix] = v;
        if (v == hi) {
            if (per_hi) { twin[L + ix] = lo; v = lo; }
            else { index_min = std::min(index_min, ix + 1); break; }
        }
    }
    return index_min;
}

// CalculateLagrangianInterpCoeff (grid/grid_interpolation.cpp:87-112)
inline void lagrange_coeff(int half, double *c0, double *c1) {
    const int num = 2 * half, offset = half - 1;
    for (int iy = 0; iy < num; ++iy) {
        c1[iy] = 1.;
        c0[iy] = 0.;
        for (int ix = 0; ix < num; ++ix)
            if (ix != iy) c1[iy] *= (0.5 + offset - (double)ix) / ((double)iy - (double)ix);
    }
    if (num > 0) c0[offset] = 1.;
}

inline uint64_t encode_xyz(int dims, const int64_t *c) {
    uint64_t k = 0;
    for (int a = 0; a < dims; ++a) k |= spread(dims, (uint32_t)c[a], a);
    return k;
}

// stencils of TransferInfoFromCoarseGrid / TransferInfoToCoarseGrid (lbm_grid_interface.cpp:408-564)
inline zlh_status plan_transfer(zlh_ctx *ctx, int level) {
    LevelState &F = ctx->lv[level], &C = ctx->lv[level - 1];
    TransferPlan &P = F.xplan;
    P = TransferPlan();
    const int dims = ctx->d.dims;
    const int lc = level - 1;
    // InterpolationLagrangian{2D,3D} (grid/grid_interpolation.cpp:224-304, 433-525), or
    // InterpolationLinear{2D,3D} (:126-208, 319-417): the Lagrangian form with max_interp_length_ 1
    // (:23) and half-length-1 weights whatever the region's valid length
    const bool linear = ctx->interp_method[level] == ZLH_INTERP_LINEAR;
    const int Lmax = linear ? 1 : 2;   // max_interp_length_ (grid/grid_info_interface.h:317-318)
    bool per_lo[3], per_hi[3];
    int64_t lo[3], hi[3];
    for (int a = 0; a < dims; ++a) {
        per_lo[a] = ctx->d.bc_scheme[1 + 2 * a] == ZLH_BC_PERIODIC;
        per_hi[a] = ctx->d.bc_scheme[2 + 2 * a] == ZLH_BC_PERIODIC;
        lo[a] = (int64_t)ctx->d.dom_min[a] << lc;
        hi[a] = (int64_t)ctx->d.dom_max[a] << lc;
    }
    std::vector<uint8_t> is_target(F.n, 0);
    P.begin.push_back(0);
    for (int layer = 1; layer < 3; ++layer) {
        for (int kind : {ZLH_INNER_F2C, ZLH_OUTER_F2C}) {
            auto it = F.layers.find({kind, layer});
            if (it == F.layers.end()) continue;
            for (uint64_t key : it->second) {
                const int64_t ti = find_key(F.keys, key);
                P.tgt.push_back(ti);
                is_target[ti] = 1;
                const uint64_t parent = key >> dims;
                int64_t seq[3][4];
                int valid = Lmax;
                for (int a = 0; a < dims; ++a)
                    valid = std::min(valid, region_axis(axis_coord(dims, parent, a), Lmax, lo[a], hi[a], per_lo[a],
                                                        per_hi[a], seq[a]));
                double c0[4], c1[4], cf[3][4];
                const int half = linear ? 1 : valid;
                lagrange_coeff(half, c0, c1);
                const int num = 2 * half, off = Lmax - half;
                for (int a = 0; a < dims; ++a)
                    for (int k = 0; k < num; ++k) cf[a][k] = (axis_coord(dims, key, a) & 1u) ? c1[k] : c0[k];
                const int nz = dims == 3 ? num : 1;
                bool broken = false;
                for (int iz = 0; iz < nz && !broken; ++iz)
                    for (int iy = 0; iy < num && !broken; ++iy)
                        for (int ix = 0; ix < num && !broken; ++ix) {
                            const double coeff = dims == 3 ? cf[0][ix] * cf[1][iy] * cf[2][iz] : cf[0][ix] * cf[1][iy];
                            if (!(std::fabs(coeff) > 1e-6)) continue;
                            int64_t c[3] = {seq[0][ix + off], seq[1][iy + off], dims == 3 ? seq[2][iz + off] : 0};
                            if (c[0] < 0 || c[1] < 0 || c[2] < 0) { broken = true; ++P.incomplete; break; }
                            const uint64_t ck = encode_xyz(dims, c);
                            const int64_t j = find_key(C.keys, ck);
                            if (j >= 0 && !(C.flags[j] & (1 << 2))) {   // kNodeStatusCoarse2FineGhost_
                                P.contrib.push_back(j);
                                C.aux_mark[j] |= kAuxRecorded;   // read by the transfer
                            } else {
                                const int64_t k = find_key(F.keys, ck << dims);
                                if (k < 0) { broken = true; ++P.incomplete; break; }
                                P.contrib.push_back(-k - 1);
                                F.aux_mark[k] |= kAuxRecorded;
                            }
                            P.coeff.push_back(coeff);
                        }
                P.begin.push_back((int64_t)P.contrib.size());
                F.aux_mark[ti] |= kAuxRecorded | kAuxDeferOnTransfer;   // written by the transfer
            }
        }
    }
    // contributors are read before any target is written: a fallback fine node that is itself
    // an interpolation target would make the result depend on the processing order
    for (int64_t c : P.contrib)
        if (c < 0 && is_target[-c - 1])
            return ctx->fail(ZLH_EINVAL, "level %d: interpolation fallback node is also a ghost target", level);
    for (int kind : {ZLH_INNER_C2F, ZLH_OUTER_C2F}) {
        auto it = C.layers.find({kind, 1});
        if (it == C.layers.end()) continue;
        for (uint64_t key : it->second) {
            const int64_t j = find_key(C.keys, key);
            const int64_t i = find_key(F.keys, key << dims);
            if (i < 0) continue;
            P.f2c_coarse.push_back(j);
            P.f2c_fine.push_back(i);
            C.aux_mark[j] |= kAuxRecorded | kAuxDeferAlways;   // written after every coarse substep
            F.aux_mark[i] |= kAuxRecorded | kAuxDeferAlways;   // its collision's rho, u are read
        }
    }
    return ZLH_OK;
}

inline double stencil_one(double d) { return std::fabs(d) < 1. ? 1. - std::fabs(d) : 0.; }
inline double stencil_two(double d) {
    if (d < 2.) {
        const double a = std::fabs(d), sq = d * d;
        if (a < 1.) return 0.125 * (3. - 2. * a + std::sqrt(1. + 4. * a - 4. * sq));
        return 0.125 * (5. - 2. * a - std::sqrt(-7. + 12. * a - 4. * sq));
    }
    return 0.;
}

// marker stencils of DirectForcingScheme{2D,3D} (immersed_boundary.cpp:108-364)
inline zlh_status plan_ib(zlh_ctx *ctx, int level) {
    LevelState &L = ctx->lv[level];
    IbPlan &P = L.ibplan;
    P = IbPlan();
    const IbMarkers &M = L.ib;
    if (M.n == 0) return ZLH_OK;
    const int dims = ctx->d.dims;
    // DomainInfo::bool_periodic_domain_: any periodic face selects the overlap walk
    bool periodic = false;
    for (int d = 1; d <= 2 * dims; ++d) periodic = periodic || ctx->d.bc_scheme[d] == ZLH_BC_PERIODIC;
    const int Ls = M.stencil_dis;
    P.support = 1;
    for (int a = 0; a < dims; ++a) P.support *= 2 * Ls;
    P.node.assign(M.n * P.support, -1);
    P.weight.assign(M.n * P.support, 0.);
    P.scale.resize(M.n);
    const double dx = 1. / (double)(1u << level), dt = dx;
    for (int64_t m = 0; m < M.n; ++m) {
        double dis[3];
        int64_t idx[3], seq[3][8], twin[3][8];
        int valid = Ls;
        for (int a = 0; a < 3; ++a)
            for (int k = 0; k < 8; ++k) { seq[a][k] = 0; twin[a][k] = -1; }
        for (int a = 0; a < dims; ++a) {
            const double iref = M.xyz[m * 3 + a] / dx;
            idx[a] = (int64_t)(iref + 1e-6);
            dis[a] = iref - (double)idx[a];
            const int64_t lo = (int64_t)ctx->d.dom_min[a] << level, hi = (int64_t)ctx->d.dom_max[a] << level;
            const bool pl = ctx->d.bc_scheme[1 + 2 * a] == ZLH_BC_PERIODIC;
            const bool ph = ctx->d.bc_scheme[2 + 2 * a] == ZLH_BC_PERIODIC;
            valid = std::min(valid, periodic ? region_axis_twin(idx[a], Ls, lo, hi, pl, ph, seq[a], twin[a])
                                             : region_axis(idx[a], Ls, lo, hi, false, false, seq[a]));
        }
        double (*stencil)(double) = valid == 2 ? stencil_two : stencil_one;
        const int n1 = 2 * valid, nz = dims == 3 ? n1 : 1;
        int e = 0;
        for (int iz = 0; iz < nz; ++iz) {
            const int oz = iz - valid;
            const double wz = dims == 3 ? stencil(std::fabs(dis[2] - oz - 1)) : 1.;
            for (int iy = 0; iy < n1; ++iy) {
                const int oy = iy - valid;
                const double wy = stencil(std::fabs(dis[1] - oy - 1));
                for (int ix = 0; ix < n1; ++ix, ++e) {
                    const int ox = ix - valid;
                    const double wx = stencil(std::fabs(dis[0] - ox - 1));
                    int64_t c[3] = {seq[0][Ls + ox], seq[1][Ls + oy], dims == 3 ? seq[2][Ls + oz] : 0};
                    if (c[0] < 0 || c[1] < 0 || c[2] < 0)
                        return ctx->fail(ZLH_EINVAL, "marker %lld stencil leaves the domain", (long long)m);
                    const int64_t j = find_key(L.keys, encode_xyz(dims, c));
                    if (j < 0) return ctx->fail(ZLH_EINVAL, "marker %lld stencil node absent at level %d", (long long)m, level);
                    P.node[m * P.support + e] = j;
                    P.weight[m * P.support + e] = dims == 3 ? wx * wy * wz : wx * wy;
                    L.aux_mark[j] |= kAuxRecorded | kAuxDeferAlways;   // forced before its collision
                }
            }
        }
        if (periodic) {
            // duplicates on periodic planes: every combination of an entry's coordinate or its
            // twin per axis other than the entry itself, with the entry's weight
            e = 0;
            for (int iz = 0; iz < nz; ++iz)
                for (int iy = 0; iy < n1; ++iy)
                    for (int ix = 0; ix < n1; ++ix, ++e) {
                        const int o[3] = {ix - valid, iy - valid, dims == 3 ? iz - valid : 0};
                        int64_t opt[3][2];
                        int nopt[3];
                        for (int a = 0; a < 3; ++a) {
                            opt[a][0] = a < dims ? seq[a][Ls + o[a]] : 0;
                            nopt[a] = 1;
                            if (a < dims && twin[a][Ls + o[a]] >= 0) opt[a][nopt[a]++] = twin[a][Ls + o[a]];
                        }
                        for (int cz = 0; cz < nopt[2]; ++cz)
                            for (int cy = 0; cy < nopt[1]; ++cy)
                                for (int cx = 0; cx < nopt[0]; ++cx) {
                                    if (cx == 0 && cy == 0 && cz == 0) continue;
                                    const int64_t c[3] = {opt[0][cx], opt[1][cy], opt[2][cz]};
                                    const int64_t j = find_key(L.keys, encode_xyz(dims, c));
                                    if (j < 0)
                                        return ctx->fail(ZLH_EINVAL, "marker %lld duplicate node absent at level %d",
                                                         (long long)m, level);
                                    P.dup_node.push_back(j);
                                    P.dup_entry.push_back(m * P.support + e);
                                    L.aux_mark[j] |= kAuxRecorded | kAuxDeferAlways;
                                }
                    }
        }
        P.scale[m] = dims == 3 ? M.area[m] / dt / dx / dx : M.area[m] / dt / dx;
    }
    return ZLH_OK;
}

// ----------------------------------------------------------------------------------------------
// device tables
// ----------------------------------------------------------------------------------------------
// IEEE binary16 bits of w if w is exactly representable, else false
inline bool exact_half_bits(double w, uint16_t *bits) {
    const uint16_t sign = std::signbit(w) ? 0x8000u : 0u;
    const double a = std::fabs(w);
    if (a == 0.) { *bits = sign; return true; }
    int e;
    (void)std::frexp(a, &e);                      // a = f 2^e, f in [0.5, 1)
    const int E = e - 1;                          // a = 1.m 2^E
    if (E > 15) return false;
    if (E < -14) {                                // subnormal: a = m 2^-24
        const double m = std::ldexp(a, 24);
        if (m != std::floor(m) || m >= 1024.) return false;
        *bits = (uint16_t)(sign | (uint16_t)m);
        return true;
    }
    const double m = (std::ldexp(a, -E) - 1.) * 1024.;
    if (m != std::floor(m)) return false;
    *bits = (uint16_t)(sign | (uint16_t)((E + 15) << 10) | (uint16_t)m);
    return true;
}

// Whether an exchange forms its rows as a table in a launch of its own (k_c2f_sources) instead of in
// the gather.  Time interpolation does, as the table keeps the earlier rows.  Of large D3Q19 exchanges
// FP64 does: its LDS holds half as many rows a group, so more are staged and rescaled twice.  Gather
// (and table) in FP64: 147k rows 138 against 92 + 21 us, 37k rows 40.0 against 30.0 + 8.9, 13k rows
// 18.6 against 14.4 + 6.7; FP32 on 147k rows 47 against 49 + 11.  D2Q9 rows are 96 bytes and few are
// shared: a step of 4M fine nodes around 613 refined squares (190k source rows) takes 446 us without the
// table and 466 with it, three nested boxes of a 256 x 192 channel 64 and 70.
inline bool row_table(const zlh_ctx *ctx, const TransferTables &X) {
    return ctx->time_interp || (ctx->fp64() && ctx->d.dims == 3 && X.n_src + X.n_fb > 32768);
}

// the row tables (for time interpolation switched on after the build: by the rows computed then,
// before any step)
inline zlh_status reserve_row_tables(zlh_ctx *ctx, TransferTables &X) {
    const int64_t stride = ctx->d.dims == 2 ? aux_stride<2>() : aux_stride<3>();
    const size_t bytes = ctx->tsize() * stride * std::max<int64_t>(X.n_src + X.n_fb, 1);
    zlh_status s;
    if (!X.src_f.p && (s = dalloc(ctx, X.src_f, bytes))) return s;
    if (ctx->time_interp && !X.src_mid.p && (s = dalloc(ctx, X.src_mid, bytes))) return s;
    return ZLH_OK;
}

inline zlh_status upload_transfer(zlh_ctx *ctx, int level) {
    LevelState &F = ctx->lv[level], &C = ctx->lv[level - 1];
    TransferPlan &P = F.xplan;
    TransferTables &X = F.xfer;
    zlh_status s;
    std::vector<int32_t> tgt, begin, src, src_ai, fb_ai, f2c_c, f2c_f;
    for (int64_t t : P.tgt) tgt.push_back(F.node_aux_h[t]);
    for (int64_t b : P.begin) begin.push_back((int32_t)b);
    // rows of src_f: the coarse sources by coarse aux index, then the fine fallback nodes by fine
    // aux index
    for (int64_t c : P.contrib) {
        if (c >= 0) src_ai.push_back(C.node_aux_h[c]);
        else fb_ai.push_back(F.node_aux_h[-c - 1]);
    }
    for (int32_t v : src_ai) if (v < 0) return ctx->fail(ZLH_EDEVICE, "transfer source not deferred");
    for (int32_t v : fb_ai) if (v < 0) return ctx->fail(ZLH_EDEVICE, "transfer fallback not deferred");
    for (auto *v : {&src_ai, &fb_ai}) {
        std::sort(v->begin(), v->end());
        v->erase(std::unique(v->begin(), v->end()), v->end());
    }
    X.n_fallback = 0;
    for (int64_t c : P.contrib) {
        if (c >= 0) {
            src.push_back((int32_t)(std::lower_bound(src_ai.begin(), src_ai.end(), C.node_aux_h[c]) - src_ai.begin()));
        } else {
            src.push_back((int32_t)(src_ai.size() + (std::lower_bound(fb_ai.begin(), fb_ai.end(), F.node_aux_h[-c - 1]) - fb_ai.begin())));
            ++X.n_fallback;
        }
    }
    for (size_t k = 0; k < P.f2c_coarse.size(); ++k) {
        f2c_c.push_back(C.node_aux_h[P.f2c_coarse[k]]);
        f2c_f.push_back(F.node_aux_h[P.f2c_fine[k]]);
    }
    for (int32_t v : tgt) if (v < 0) return ctx->fail(ZLH_EDEVICE, "transfer target not deferred");
    X.n_c2f = (int64_t)tgt.size();
    X.n_src = (int64_t)src_ai.size();
    X.n_fb = (int64_t)fb_ai.size();
    X.n_f2c = (int64_t)f2c_c.size();
    // gather order: ghost nodes by aux index (brick-major Morton order), cut into chunks of
    // kGatherChunk; inside a chunk by descending contributor count, then aux index.  A group
    // closes at 256 / PARTS nodes or when its rows and contributor words would pass the budget
    const int Qn = ctx->q;
    const int parts = (Qn + kGatherDirs - 1) / kGatherDirs;
    const int row_stride = ctx->d.dims == 2 ? aux_stride<2>() : aux_stride<3>();
    const size_t lds_budget = kGatherLdsBudget, row_bytes = (size_t)row_stride * ctx->tsize();
    const int group_max = 256 / parts;
    const int64_t nt = (int64_t)tgt.size();
    std::vector<int64_t> order(nt), chunk(nt);
    for (int64_t t = 0; t < nt; ++t) order[t] = t;
    std::sort(order.begin(), order.end(), [&](int64_t a, int64_t b) { return tgt[a] < tgt[b]; });
    for (int64_t k = 0; k < nt; ++k) chunk[order[k]] = k / kGatherChunk;
    std::sort(order.begin(), order.end(), [&](int64_t a, int64_t b) {
        if (chunk[a] != chunk[b]) return chunk[a] < chunk[b];
        const int32_t na = begin[a + 1] - begin[a], nb = begin[b + 1] - begin[b];
        return na != nb ? na > nb : tgt[a] < tgt[b];
    });
    auto lds_of = [&](size_t nrows, int64_t ncontrib) { return ((nrows * row_bytes + 15) & ~(size_t)15) + (size_t)ncontrib * 4; };
    std::vector<int32_t> tgt2, begin2(1, 0), group_tgt(1, 0), group_begin(1, 0), group_rows;
    std::vector<uint32_t> packed;
    packed.reserve(src.size());
    std::unordered_map<int32_t, int32_t> local;
    std::vector<int32_t> distinct;
    int64_t g_nc = 0;
    int g_nt = 0;
    size_t lds_max = 0;
    auto close_group = [&]() {
        lds_max = std::max(lds_max, lds_of(local.size(), g_nc));
        group_tgt.push_back((int32_t)tgt2.size());
        group_begin.push_back((int32_t)group_rows.size());
        local.clear();
        g_nc = 0;
        g_nt = 0;
    };
    for (int64_t t : order) {
        const int32_t k0 = begin[t], k1 = begin[t + 1];
        distinct.assign(src.begin() + k0, src.begin() + k1);
        std::sort(distinct.begin(), distinct.end());
        distinct.erase(std::unique(distinct.begin(), distinct.end()), distinct.end());
        size_t n_new = 0;
        for (int32_t r : distinct) n_new += local.count(r) ? 0 : 1;
        if (g_nt > 0 && (g_nt == group_max || local.size() + n_new > (size_t)kGatherMaxRows ||
                         lds_of(local.size() + n_new, g_nc + (k1 - k0)) > lds_budget))
            close_group();
        if (lds_of(distinct.size(), k1 - k0) > lds_budget || distinct.size() > (size_t)kGatherMaxRows)
            return ctx->fail(ZLH_EDEVICE, "interpolation stencil too large for LDS");
        for (int32_t r : distinct)
            if (local.emplace(r, (int32_t)local.size()).second) group_rows.push_back(r);
        for (int32_t k = k0; k < k1; ++k) {
            uint16_t bits;
            if (!exact_half_bits(P.coeff[k], &bits)) return ctx->fail(ZLH_EDEVICE, "interpolation weight not exact in FP16");
            packed.push_back((uint32_t)(local[src[k]] * row_stride) | ((uint32_t)bits << 16));
        }
        tgt2.push_back(tgt[t]);
        begin2.push_back((int32_t)packed.size());
        g_nc += k1 - k0;
        ++g_nt;
    }
    if (g_nt > 0) close_group();
    X.n_groups = (int64_t)group_tgt.size() - 1;
    X.lds_bytes = lds_max;
    X.staged_rows = (int64_t)group_rows.size();
    X.n_contrib = (int64_t)packed.size();
    std::vector<GatherGroup> groups(X.n_groups);
    for (int64_t g = 0; g < X.n_groups; ++g) {
        GatherGroup &G = groups[g];
        G.t0 = group_tgt[g];
        G.t1 = group_tgt[g + 1];
        G.c0 = begin2[G.t0];
        G.c1 = begin2[G.t1];
        G.r0 = group_begin[g];
        G.r1 = group_begin[g + 1];
        G.pad0 = G.pad1 = 0;
    }
    if ((s = upload(ctx, X.c2f_target, tgt2))) return s;
    if ((s = upload(ctx, X.c2f_begin, begin2))) return s;
    if ((s = upload(ctx, X.groups, groups))) return s;
    if ((s = upload(ctx, X.group_rows, group_rows))) return s;
    {
        // the aux rows of the same entries: coarse, or ~fine
        std::vector<int32_t> aux_rows(group_rows.size());
        for (size_t k = 0; k < group_rows.size(); ++k) {
            const size_t g = (size_t)group_rows[k];
            aux_rows[k] = g < src_ai.size() ? src_ai[g] : ~fb_ai[g - src_ai.size()];
        }
        if ((s = upload(ctx, X.group_aux, aux_rows))) return s;
    }
    if ((s = upload(ctx, X.c2f_contrib, packed))) return s;
    if ((s = upload(ctx, X.src_coarse_ai, src_ai))) return s;
    if ((s = upload(ctx, X.fb_fine_ai, fb_ai))) return s;
    X.src_f = DevBuf();
    X.src_mid = DevBuf();
    if (row_table(ctx, X) && (s = reserve_row_tables(ctx, X))) return s;
    if ((s = upload(ctx, X.f2c_coarse_ai, f2c_c))) return s;
    if ((s = upload(ctx, X.f2c_fine_ai, f2c_f))) return s;
    {
        std::vector<int32_t> a(tgt2.begin(), tgt2.end()), b(f2c_f.begin(), f2c_f.end());
        std::sort(a.begin(), a.end());
        std::sort(b.begin(), b.end());
        std::vector<int32_t> common;
        std::set_intersection(a.begin(), a.end(), b.begin(), b.end(), std::back_inserter(common));
        X.f2c_apart = common.empty();
        std::vector<int32_t> c(f2c_c.begin(), f2c_c.end());
        std::sort(c.begin(), c.end());
        common.clear();
        std::set_intersection(src_ai.begin(), src_ai.end(), c.begin(), c.end(), std::back_inserter(common));
        X.f2c_apart &= common.empty();
    }
    if (level - 1 >= 1) {
        // the coarse level's own transfer (from level - 2) against this one's coarse side: this
        // one reads its coarse sources and writes its fine-to-coarse targets there.  Only reported
        // (zlh_transfer_info): every transfer runs in the reference's order
        const TransferPlan &CP = C.xplan;
        std::vector<uint8_t> mark(C.n, 0);   // 1 read, 2 written
        for (int64_t c : CP.contrib)
            if (c < 0) mark[-c - 1] |= 1;
        for (int64_t i : CP.f2c_fine) mark[i] |= 1;
        for (int64_t i : CP.tgt) mark[i] |= 2;
        C.xfer_overlap = false;
        for (int64_t c : P.contrib)
            if (c >= 0) C.xfer_overlap |= (mark[c] & 2) != 0;
        for (int64_t j : P.f2c_coarse) C.xfer_overlap |= mark[j] != 0;
    }
    std::vector<uint8_t> macro_flag(std::max<int64_t>(F.naux, 1), 0);
    for (int32_t i : f2c_f) macro_flag[i] = 1;
    if ((s = upload(ctx, F.aux_macro_flag_d, macro_flag))) return s;
    return ZLH_OK;
}

inline zlh_status upload_ib(zlh_ctx *ctx, int level) {
    LevelState &L = ctx->lv[level];
    IbTables &T = L.ibt;
    IbPlan &P = L.ibplan;
    T.n_markers = L.ib.n;
    if (T.n_markers == 0) return ZLH_OK;
    zlh_status s;
    T.support = P.support;
    T.stiffness = L.ib.stiffness;
    std::vector<int32_t> ai(P.node.size(), -1), dup_ai(P.dup_node.size(), -1), supported;
    std::vector<uint8_t> seen(L.naux, 0);
    for (size_t k = 0; k < P.node.size(); ++k) {
        if (P.node[k] < 0) continue;
        ai[k] = L.node_aux_h[P.node[k]];
        if (ai[k] < 0) return ctx->fail(ZLH_EDEVICE, "immersed boundary node not deferred");
        if (!seen[ai[k]]) { seen[ai[k]] = 1; supported.push_back(ai[k]); }
    }
    // duplicates on periodic planes receive spread terms, but interpolate nothing
    for (size_t k = 0; k < P.dup_node.size(); ++k) {
        dup_ai[k] = L.node_aux_h[P.dup_node[k]];
        if (dup_ai[k] < 0) return ctx->fail(ZLH_EDEVICE, "immersed boundary node not deferred");
        if (!seen[dup_ai[k]]) { seen[dup_ai[k]] = 1; supported.push_back(dup_ai[k]); }
    }
    // supported nodes in aux order, as the aux collision takes them
    std::sort(supported.begin(), supported.end());
    // node-major view of the marker table for the spread: the entries naming each supported
    // node, in ascending entry (marker) order
    if (ai.size() >= ((size_t)1 << 31)) return ctx->fail(ZLH_ENOMEM, "immersed boundary table too large");
    // each term's marker and coefficient weight x area / (dt dx^(dims-1)) (the same double
    // product the marker-major form forms), in ascending marker order per node
    std::vector<int32_t> pos(L.naux, -1), begin(supported.size() + 1, 0), marker;
    std::vector<double> coef;
    for (size_t r = 0; r < supported.size(); ++r) pos[supported[r]] = (int32_t)r;
    // terms: (node, marker, table entry) of every stencil entry and every duplicate, ordered by
    // marker per node (a node takes at most one term per marker)
    struct Term { int32_t a; int64_t m, k; };
    std::vector<Term> terms;
    for (size_t k = 0; k < ai.size(); ++k)
        if (ai[k] >= 0) terms.push_back({ai[k], (int64_t)(k / (size_t)P.support), (int64_t)k});
    for (size_t k = 0; k < dup_ai.size(); ++k)
        terms.push_back({dup_ai[k], P.dup_entry[k] / P.support, P.dup_entry[k]});
    std::stable_sort(terms.begin(), terms.end(), [](const Term &x, const Term &y) { return x.m < y.m; });
    for (const Term &t : terms) ++begin[pos[t.a] + 1];
    for (size_t r = 0; r < supported.size(); ++r) begin[r + 1] += begin[r];
    marker.resize(begin.back());
    coef.resize(begin.back());
    std::vector<int32_t> fill(begin.begin(), begin.end() - 1);
    for (const Term &t : terms) {
        const int32_t e = fill[pos[t.a]]++;
        marker[e] = (int32_t)t.m;
        coef[e] = P.weight[t.k] * P.scale[t.m];
    }
    if ((s = upload(ctx, T.spread_begin, begin))) return s;
    if ((s = upload(ctx, T.spread_marker, marker))) return s;
    if ((s = upload(ctx, T.spread_weight, coef))) return s;
    if ((s = upload(ctx, T.node_ai, ai))) return s;
    if ((s = upload(ctx, T.weight, P.weight))) return s;
    if ((s = upload(ctx, T.spread_row, pos))) return s;
    if ((s = upload(ctx, T.marker_vel, L.ib.vel))) return s;
    if ((s = dalloc(ctx, T.marker_force, sizeof(double) * 3 * T.n_markers))) return s;
    return ZLH_OK;
}

// ----------------------------------------------------------------------------------------------
// launches
// ----------------------------------------------------------------------------------------------
// parts: kTransferC2F (TransferInfoFromCoarseGrid) and / or kTransferF2C (TransferInfoToCoarseGrid),
// in that order (InformationFromGridOfDifferentLevel, lbm_solver_interface.cpp:224-238);
// kTransferMid makes the coarse-to-fine part the time-interpolated refill after an odd substep
// (rows into src_mid, src_f kept as the synchronised rows), kTransferRows only computes the
// synchronised rows (the earlier state of the next time-interpolated refill).
constexpr int kTransferC2F = 1, kTransferF2C = 2, kTransferMid = 4, kTransferRows = 8;
template <int D, typename T, bool SHIFT>
zlh_status launch_transfers_t(zlh_ctx *ctx, int level, int parts) {
    LevelState &F = ctx->lv[level], &C = ctx->lv[level - 1];
    TransferTables &X = F.xfer;
    const int comp = ctx->d.compressible;
    // tau ratios of PostStreamCoarse2Fine (coarse level) and PostStreamFine2Coarse (fine level),
    // CalRelaxationTimeRatio (lbm_collision_models.cpp:142-151)
    const double nu = ctx->d.nu0;
    const double dtc = 1. / (double)(1u << (level - 1)), dtf = 1. / (double)(1u << level);
    const double c2f = 0.5 * (nu * 3. / dtc * 2. + 0.5) / (nu * 3. / dtc + 0.5);
    const double f2c = 2. * (nu * 3. / dtf / 2 + 0.5) / (nu * 3. / dtf + 0.5);
    const bool table = row_table(ctx, X);
    const bool mid = (parts & kTransferMid) != 0;
    if (table && (parts & (kTransferC2F | kTransferRows)) && X.n_src + X.n_fb > 0) {
        const zlh_status s = reserve_row_tables(ctx, X);
        if (s) return s;
        const dim3 grid(blocks(X.n_src + X.n_fb));
        if (mid)
            hipLaunchKernelGGL((k_c2f_sources<D, T, SHIFT, true>), grid, dim3(256), 0, ctx->stream, X.n_src, X.n_fb,
                               X.src_coarse_ai.as<int32_t>(), C.aux_f_d.as<T>(), X.fb_fine_ai.as<int32_t>(),
                               F.aux_f_d.as<T>(), c2f, comp, X.src_f.as<T>(), X.src_mid.as<T>());
        else
            hipLaunchKernelGGL((k_c2f_sources<D, T, SHIFT, false>), grid, dim3(256), 0, ctx->stream, X.n_src, X.n_fb,
                               X.src_coarse_ai.as<int32_t>(), C.aux_f_d.as<T>(), X.fb_fine_ai.as<int32_t>(),
                               F.aux_f_d.as<T>(), c2f, comp, nullptr, X.src_f.as<T>());
    }
    const F2cArgs<T> fc{X.n_f2c, X.f2c_coarse_ai.as<int32_t>(), X.f2c_fine_ai.as<int32_t>(), F.aux_f_d.as<T>(),
                        F.aux_macro_d.as<double>(), f2c, comp, C.aux_f_d.as<T>()};
    bool copied = false;
    if ((parts & kTransferC2F) && X.n_c2f > 0) {
        const GatherArgs<T> ga{X.groups.as<GatherGroup>(), X.c2f_target.as<int32_t>(), X.c2f_begin.as<int32_t>(),
                               X.c2f_contrib.as<uint32_t>(), table ? X.group_rows.as<int32_t>() : X.group_aux.as<int32_t>(),
                               table ? (mid ? X.src_mid.as<T>() : X.src_f.as<T>()) : C.aux_f_d.as<T>(), F.aux_f_d.as<T>(),
                               c2f, comp};
        const int64_t nb_gather = (X.n_groups + 7) / 8 * 8;
        if ((parts & kTransferF2C) && X.n_f2c > 0 && X.f2c_apart) {
            // one launch for both halves (independent: see k_c2f_gather_f2c)
            const dim3 grid((unsigned)(nb_gather + blocks(X.n_f2c)));
            if (table)
                hipLaunchKernelGGL((k_c2f_gather_f2c<D, T, SHIFT, false>), grid, dim3(256), X.lds_bytes, ctx->stream,
                                   nb_gather, X.n_groups, ga, fc);
            else
                hipLaunchKernelGGL((k_c2f_gather_f2c<D, T, SHIFT, true>), grid, dim3(256), X.lds_bytes, ctx->stream,
                                   nb_gather, X.n_groups, ga, fc);
            copied = true;
        } else if (table) {
            hipLaunchKernelGGL((k_c2f_gather<D, T, SHIFT, false>), dim3((unsigned)nb_gather), dim3(256), X.lds_bytes,
                               ctx->stream, X.n_groups, ga);
        } else {
            hipLaunchKernelGGL((k_c2f_gather<D, T, SHIFT, true>), dim3((unsigned)nb_gather), dim3(256), X.lds_bytes,
                               ctx->stream, X.n_groups, ga);
        }
    }
    if ((parts & kTransferF2C) && X.n_f2c > 0 && !copied)
        hipLaunchKernelGGL((k_f2c<D, T, SHIFT>), dim3(blocks(X.n_f2c)), dim3(256), 0, ctx->stream, fc);
    ZLH_TRY(hipGetLastError());
    return ZLH_OK;
}

inline zlh_status launch_transfers(zlh_ctx *ctx, int level, int parts = kTransferC2F | kTransferF2C) {
    if (ctx->d.dims == 2)
        return ctx->fp64() ? launch_transfers_t<2, double, false>(ctx, level, parts)
             : ctx->bf16() ? launch_transfers_t<2, bf16_t, true>(ctx, level, parts)
                           : launch_transfers_t<2, float, true>(ctx, level, parts);
    return ctx->fp64() ? launch_transfers_t<3, double, false>(ctx, level, parts)
         : ctx->bf16() ? launch_transfers_t<3, bf16_t, true>(ctx, level, parts)
                       : launch_transfers_t<3, float, true>(ctx, level, parts);
}

template <int D, typename T, typename Cc, bool SHIFT>
zlh_status launch_ib_t(zlh_ctx *ctx, int level) {
    LevelState &L = ctx->lv[level];
    IbTables &B = L.ibt;
    hipLaunchKernelGGL((k_ib_markers<D, T, Cc, SHIFT>), dim3(blocks(B.n_markers * 64)), dim3(256), 0, ctx->stream,
                       B.n_markers, B.support, B.node_ai.as<int32_t>(), B.weight.as<double>(), L.aux_f_d.as<T>(),
                       B.marker_vel.as<double>(), B.stiffness, B.marker_force.as<double>(), L.sp);
    ZLH_TRY(hipGetLastError());
    return ZLH_OK;
}

inline zlh_status launch_ib(zlh_ctx *ctx, int level) {
    if (ctx->lv[level].ibt.n_markers == 0) return ZLH_OK;
    if (ctx->d.dims == 2)
        return ctx->fp64() ? launch_ib_t<2, double, double, false>(ctx, level)
             : ctx->bf16() ? launch_ib_t<2, bf16_t, float, true>(ctx, level)
                           : launch_ib_t<2, float, float, true>(ctx, level);
    return ctx->fp64() ? launch_ib_t<3, double, double, false>(ctx, level)
         : ctx->bf16() ? launch_ib_t<3, bf16_t, float, true>(ctx, level)
                       : launch_ib_t<3, float, float, true>(ctx, level);
}

}  // namespace zlh
