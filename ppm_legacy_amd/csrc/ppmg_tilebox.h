// ppmg_tilebox.h -- the stored nodes of a field box besides the ones the
// tiled deposits write (2D and 3D, M'4 and BSP2): node N of periodic axes
// whose stored box holds the whole real range, and the ghost layers.  Shared
// by ppmg_p2m2d.hip and ppmg_p2m3d.hip.
#pragma once
#include <type_traits>

#include "ppmg_internal.h"
#include "ppmg_sort.h"

namespace ppmg {

// Weight tables of ppm_rmsh_remesh (wx1/wx2/wx3, the stencil width per
// particle and axis), used in place of the positions' weights.
template <typename ValT> struct WTab {
    const ValT* w[3];
};

// Stored nodes besides the unique ones, for axes whose stored box holds the
// whole real range 0..N.  Per axis: R = stored real nodes (N compact, N+1
// boxed), O = ext - R stored nodes outside 0..N.

// Real nodes with index N on a boxed periodic axis (n.d = N; -1 on other
// axes): the fold leaves node N equal to node 0, so they take the value the
// tiles wrote there.  Enumerated as the face i = N, then j = N (i < N), then
// k = N (i, j < N), over the real nodes (r per axis, b = 1 where node N is a
// copy).
struct BoxDup {
    int3 n, r, b;
    int64_t ndup;
    unsigned wg;   // workgroups of 256 nodes
};
template <typename ValT>
__device__ __forceinline__ void box_dup(const FieldGeom& fg, const BoxDup& d, ValT* __restrict__ field, int64_t tt) {
    if (tt >= d.ndup) return;
    int i, j, k;
    auto locate = [&](auto t) {   // 32-bit divisions wherever the node count fits
        using U = decltype(t);
        const U fx = d.b.x ? (U)d.r.y * (U)d.r.z : 0;
        const U wx = (U)(d.r.x - d.b.x), wy = (U)(d.r.y - d.b.y);
        const U fy = d.b.y ? wx * (U)d.r.z : 0;
        if (t < fx) {
            i = d.n.x;
            j = (int)(t % (U)d.r.y);
            k = (int)(t / (U)d.r.y);
        } else if (t < fx + fy) {
            t -= fx;
            i = (int)(t % wx);
            j = d.n.y;
            k = (int)(t / wx);
        } else {
            t -= fx + fy;
            i = (int)(t % wx);
            j = (int)((t / wx) % wy);
            k = d.n.z;
        }
    };
    if ((uint64_t)d.ndup >> 32) locate((uint64_t)tt);
    else locate((uint32_t)tt);
    auto at = [&](int x, int y, int z) {
        return (((int64_t)(z - fg.lo[2]) * fg.ext[1] + (y - fg.lo[1])) * fg.ext[0] + (x - fg.lo[0])) * fg.lda;
    };
    const int64_t dst = at(i, j, k);
    const int64_t src = at(i == d.n.x ? 0 : i, j == d.n.y ? 0 : j, k == d.n.z ? 0 : k);
    for (int c = 0; c < fg.lda; ++c) field[dst + c] = field[src + c];
}
template <typename ValT>
__global__ void __launch_bounds__(256) k_box_dup(FieldGeom fg, BoxDup dup, ValT* __restrict__ field) {
    box_dup<ValT>(fg, dup, field, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// Stored nodes outside 0..N on some axis (ghost layers): the raw sum of the
// particles whose stencil reaches the node with no periodic wrap on any axis,
// which is what ppm_map_field_ghost_put leaves in ghost nodes (the general
// path's rule for nodes that are not real).  Enumerated as the planes outside
// 0..N in z, then the rows outside in y (z real), then the nodes outside in x
// (y, z real).  Weights and products in the value precision, sums in FP64;
// with weight tables (wt.w[0] set) the weights are the tables'.  KS: stencil
// width (4 M'4, 2 BSP2); DIM 2: one plane (no z stencil), positions of two
// coordinates.  TABLE: the binning is a slot table instead of heads and a
// permutation; a cell's particles come in the same order.
//
// Bound by latency: a node's cells (at most 16 on a periodic box, whose
// outside axis meets one stencil offset) lead to list heads and then to
// particles, a chain of two loads, with little arithmetic.  Four lanes share a
// node, cell j going to lane j mod 4; a lane has the heads of four cells and
// then their first particles in flight at once, so a node takes one pass of the
// chain, and the short register list leaves many wavefronts resident.  The
// four partial sums are added in a fixed order.  The first dup.wg workgroups
// make node N's copies (box_dup), so that a small box has one launch fewer
// (3 us of 82 for a step on 32^3 cells).  (One lane per node, 16 heads
// and then four batches of four particles, against this: 115 and 84 us at
// 256^3, ghost size 2, lda 3, FP32c; 40 and 11 us at 64^3, FP64.)
constexpr int SHELL_LANES = 4;   // lanes per node (a DPP quad)
constexpr int SHELL_CELLS = 4;   // cells per lane and pass

// Sum over the lanes of a quad, in the same order in every lane.
__device__ __forceinline__ double quad_sum(double v) {
    auto perm = [](double w, auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(w), C, 0xF, 0xF, true);
        const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(w), C, 0xF, 0xF, true);
        return __hiloint2double(hi, lo);
    };
    v += perm(v, std::integral_constant<int, 0xB1>{});   // lanes 1 0 3 2
    v += perm(v, std::integral_constant<int, 0x4E>{});   // lanes 2 3 0 1
    return v;
}

template <int DIM, int KS, typename PosT, typename ValT, int LL, bool TABLE>
__global__ void __launch_bounds__(256) k_box_shell(DevMesh m, FieldGeom fg, int3 r, const int* __restrict__ start,
                                                  const int* __restrict__ perm, BinTable bt,
                                                  const PosT* __restrict__ xp, const ValT* __restrict__ up, int c0,
                                                  ValT* __restrict__ field, int64_t t0, int64_t nshell,
                                                  WTab<ValT> wt, BoxDup dup) {
    if (blockIdx.x < dup.wg) {
        box_dup<ValT>(fg, dup, field, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
        return;
    }
    const int sub = threadIdx.x & (SHELL_LANES - 1);
    const int64_t tq = t0 + ((int64_t)(blockIdx.x - dup.wg) * blockDim.x + threadIdx.x) / SHELL_LANES;
    const bool live = tq < nshell;   // a quad past the end works on the last node and stores nothing
    const int64_t t = live ? tq : nshell - 1;
    const int e0 = fg.ext[0], e1 = fg.ext[1], e2 = fg.ext[2];
    const int o0 = e0 - r.x, o1 = e1 - r.y, o2 = e2 - r.z;
    // q-th stored node of axis d outside the real range: below 0, then above N
    auto outer = [&](int d, int q) { return q < -fg.lo[d] ? fg.lo[d] + q : m.N[d] + 1 + (q + fg.lo[d]); };
    int n[3];
    auto locate = [&](auto q) {   // 32-bit divisions wherever the box's node count fits
        using U = decltype(q);
        const U ra = (U)o2 * (U)e1 * (U)e0, rb = (U)r.z * (U)o1 * (U)e0;
        if (q < ra) {
            const U row = q / (U)e0, pl = row / (U)e1;
            n[0] = fg.lo[0] + (int)(q - row * (U)e0);
            n[1] = fg.lo[1] + (int)(row - pl * (U)e1);
            n[2] = outer(2, (int)pl);
        } else if (q < ra + rb) {
            q -= ra;
            const U row = q / (U)e0, pl = row / (U)o1;
            n[0] = fg.lo[0] + (int)(q - row * (U)e0);
            n[1] = outer(1, (int)(row - pl * (U)o1));
            n[2] = (int)pl;
        } else {
            q -= ra + rb;
            const U row = q / (U)o0, pl = row / (U)r.y;
            n[0] = outer(0, (int)(q - row * (U)o0));
            n[1] = (int)(row - pl * (U)r.y);
            n[2] = (int)pl;
        }
    };
    if (((uint64_t)e0 * (uint64_t)e1 * (uint64_t)e2) >> 32) locate((uint64_t)t);
    else locate((uint32_t)t);
    double acc[LL];
#pragma unroll
    for (int c = 0; c < LL; ++c) acc[c] = 0.0;
    constexpr int B = Stencil<KS>::B;
    // The stencil offsets of each axis whose cell n + B - o exists: olo ..
    // olo + num - 1.  Cell j of the num[0] num[1] num[2] cells counts x fastest.
    int olo[3], num[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        olo[d] = d < DIM ? max(0, n[d] + B - (m.nbin[d] - 1)) : 0;
        num[d] = d < DIM ? max(0, min(KS - 1, n[d] + B) - olo[d] + 1) : 1;
    }
    const int ncell = num[0] * num[1] * num[2];
    // j / k for j < 64 and k = 1..4
    auto quotient = [](int j, int k) { return (j * (k == 1 ? 257 : k == 2 ? 129 : k == 3 ? 86 : 65)) >> 8; };
    auto particle_of = [&](int key, int q) {
        return TABLE ? bt.table[(int64_t)q * bt.ncells + key] : perm ? perm[q] : q;
    };
    const bool tab = wt.w[0] != nullptr;
    // a particle's position or, with tables, its weights at the offsets o
    // (a weight converts to the position type and back exactly)
    auto load = [&](int p, const int (&o)[3], PosT (&x)[DIM], ValT (&u)[LL]) {
#pragma unroll
        for (int d = 0; d < DIM; ++d)
            x[d] = tab ? (PosT)wt.w[d][(int64_t)p * KS + o[d]] : xp[(int64_t)p * DIM + d];
#pragma unroll
        for (int c = 0; c < LL; ++c) u[c] = up[(int64_t)p * fg.lda + c0 + c];
    };
    auto add = [&](const int (&o)[3], const PosT (&x)[DIM], const ValT (&u)[LL]) {
        ValT w1[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            int ci;
            w1[d] = tab ? (ValT)x[d]
                        : tile_weight_at<KS, ValT>(
                              (ValT)cell_offset<PosT>(x[d], (PosT)m.minv[d], (PosT)m.dxi[d], ci), o[d]);
        }
        ValT w = w1[0] * w1[1];
        if constexpr (DIM == 3) w = w * w1[2];
#pragma unroll
        for (int c = 0; c < LL; ++c) acc[c] += (double)(w * u[c]);
    };
    for (int j0 = sub; j0 < ncell; j0 += SHELL_LANES * SHELL_CELLS) {
        int o[SHELL_CELLS][3], key[SHELL_CELLS], b[SHELL_CELLS], e[SHELL_CELLS], p[SHELL_CELLS];
#pragma unroll
        for (int i = 0; i < SHELL_CELLS; ++i) {
            const int j = j0 + SHELL_LANES * i;
            const int row = quotient(j, num[0]), pl = quotient(row, num[1]);
            o[i][0] = olo[0] + j - row * num[0];
            o[i][1] = olo[1] + row - pl * num[1];
            o[i][2] = olo[2] + pl;
            key[i] = b[i] = e[i] = p[i] = 0;
            if (j < ncell) {
                const int cz = DIM == 3 ? n[2] + B - o[i][2] : 0;
                key[i] = (n[0] + B - o[i][0]) + m.nbin[0] * ((n[1] + B - o[i][1]) + m.nbin[1] * cz);
                if constexpr (TABLE) {
                    e[i] = (int)bt.count[count_word(key[i])];   // decoded below: the loads stay in flight
                    p[i] = bt.table[key[i]];
                } else {
                    b[i] = start[key[i]];
                    e[i] = start[key[i] + 1];
                }
            }
        }
        PosT x[SHELL_CELLS][DIM];
        ValT u[SHELL_CELLS][LL];
#pragma unroll
        for (int i = 0; i < SHELL_CELLS; ++i) {
            if constexpr (TABLE) e[i] = j0 + SHELL_LANES * i < ncell ? (int)(((unsigned)e[i] >> count_shift(key[i])) & 255u) : 0;
            if (e[i] > b[i]) {
                if constexpr (!TABLE) p[i] = perm ? perm[b[i]] : b[i];
                load(p[i], o[i], x[i], u[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < SHELL_CELLS; ++i) {
            if (e[i] > b[i]) {
                add(o[i], x[i], u[i]);
                for (int q = b[i] + 1; q < e[i]; ++q) {
                    PosT xq[DIM];
                    ValT uq[LL];
                    load(particle_of(key[i], q), o[i], xq, uq);
                    add(o[i], xq, uq);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < LL; ++c) acc[c] = quad_sum(acc[c]);
    if (!live || sub != 0) return;
    ValT* out = field + (((int64_t)(n[2] - fg.lo[2]) * e1 + (n[1] - fg.lo[1])) * e0 + (n[0] - fg.lo[0])) * fg.lda + c0;
#pragma unroll
    for (int c = 0; c < LL; ++c) out[c] = (ValT)acc[c];
}

// Fills the stored nodes of `field` that the tiles do not write (see above),
// after the tile launches of a deposit.
template <int DIM, int KS, typename PosT, typename ValT>
int fill_stored_box(ppmg_plan* plan, const DevMesh& m, const PosT* xp, const ValT* up, const FieldGeom& fg,
                    ValT* field, const WTab<ValT>& wt, hipStream_t s) {
    const int lda = fg.lda;
    int R[3], B[3], D[3];
    for (int d = 0; d < 3; ++d) {
        const bool compact = m.periodic[d] && fg.lo[d] == 0 && fg.ext[d] == m.N[d];
        B[d] = d < DIM && m.periodic[d] && !compact;
        R[d] = d >= DIM ? 1 : compact ? m.N[d] : m.N[d] + 1;
        D[d] = B[d] ? m.N[d] : -1;
    }
    const int3 n3 = make_int3(D[0], D[1], D[2]), r3 = make_int3(R[0], R[1], R[2]),
               b3 = make_int3(B[0], B[1], B[2]);
    const int64_t ndup = (int64_t)R[0] * R[1] * R[2] - (int64_t)(R[0] - B[0]) * (R[1] - B[1]) * (R[2] - B[2]);
    const int64_t nshell = (int64_t)fg.ext[0] * fg.ext[1] * fg.ext[2] - (int64_t)R[0] * R[1] * R[2];
    BoxDup dup{n3, r3, b3, ndup, (unsigned)((ndup + 255) / 256)};
    if (ndup > 0 && nshell == 0) hipLaunchKernelGGL(k_box_dup<ValT>, dim3(dup.wg), dim3(256), 0, s, fg, dup, field);
    if (nshell > 0) {
        const BinTable bt{plan->count.as<uint32_t>(), plan->table.as<int>(), plan->ncells};
        const bool table = plan->bin_table;
        if (!table && materialize_heads(plan, s)) return 1;
        for (int c0 = 0; c0 < lda; c0 += 4) {
            const int L = lda - c0 < 4 ? lda - c0 : 4;
// (2^28 nodes a launch: under 2^32 threads)
#define SH(LL, TB)                                                                                                    \
    for (int64_t t0 = 0; t0 < nshell; t0 += (int64_t)1 << 28) {                                                       \
        const int64_t nt = nshell - t0 < ((int64_t)1 << 28) ? nshell - t0 : (int64_t)1 << 28;                          \
        hipLaunchKernelGGL((k_box_shell<DIM, KS, PosT, ValT, LL, TB>),                                                \
                           dim3((unsigned)((nt * SHELL_LANES + 255) / 256) + dup.wg), dim3(256), 0, s, m, fg, r3,     \
                           plan->start.as<int>(), tile_perm(plan), bt, xp, up, c0, field, t0, t0 + nt, wt, dup);      \
        dup.wg = 0;   /* (the copies are of all components) */                                                       \
    }
#define SHL(LL)                      \
    do {                             \
        if (table) SH(LL, true)      \
        else SH(LL, false)           \
    } while (0)
            if (L == 1) SHL(1);
            else if (L == 2) SHL(2);
            else if (L == 3) SHL(3);
            else SHL(4);
#undef SHL
#undef SH
        }
    }
    PPMG_HIP(hipGetLastError());
    return 0;
}

}  // namespace ppmg
