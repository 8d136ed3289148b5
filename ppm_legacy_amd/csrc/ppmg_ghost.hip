// ppmg_ghost.hip -- ghost mapping of a padded field on the device, for one
// sub covering the domain (what ppm_topo_mkfield builds on one process).
//
// Replaces ppm_map_field_ghost with maptype ghost_get or ghost_put followed
// by push, send and pop (ppm_map_field_ghost.f:627-714):
//   ghost_get  every stored node that is a periodic image of a real node
//              (ghost layers, and the duplicate face node Nm) receives the
//              real node's value (pop replace);
//   ghost_put  every stored image node is added onto the real node it
//              images (pop add, ppm_map_field_pop_3d.f:781-800).
// The block lists are those of ppm_map_field_ghost_init.f:234-447 for one
// periodic sub: one block per periodic image of the sub (faces, edges,
// corners, in the reference's order), intersected with the stored box
// 1-g .. Nm+g (ppm_mesh_block_intersect.f:207-279).  As in the reference all
// blocks are packed before any is unpacked (push before pop), and blocks are
// unpacked in list order: a node in several image blocks keeps the last
// block's value (get) or receives the blocks' additions in list order (put).
//
// Element kinds are those of the reference's specifics (_s, _d, _sc, _dc, _i,
// _l): complex fields are real fields of twice the components; the push packs
// every kind into a real buffer and the pop converts back
// (ppm_map_field_push_3d.f:564-592, ppm_map_field_pop_3d.f:1818-1897), which
// for integers is an exact round trip (INT of the packed value) and for
// logicals 1.0 / 0.0 read back as value > 1 - eps, "add" being .AND.  The
// optional mask (one logical per stored node) is read at the pop: a node
// whose mask is .FALSE. keeps its value, and the buffer still steps past it
// (the push packs every node: its mask test is commented out at
// ppm_map_field_push_3d.f:546-549).
#include <type_traits>

#include "ppmg_internal.h"
#include "ppmg_interp.h"

namespace ppmg {

int ghost_blocks(const DevMesh& m, const int* g, GhostBlock* out) {
    const int dim = m.dim;
    // shift of one periodic image per axis: Nm - 1 nodes
    const int op[3] = {m.N[0], m.N[1], dim > 2 ? m.N[2] : 0};
    const bool px = m.periodic[0], py = m.periodic[1], pz = dim > 2 && m.periodic[2];
    int shifts[26][3];
    int n = 0;
    auto push = [&](int a, int b, int c) {
        shifts[n][0] = a;
        shifts[n][1] = b;
        shifts[n][2] = c;
        ++n;
    };
    // images in the order ppm_map_field_ghost_init.f:236-425 lists them: the x
    // faces, then for each y face its x edges, then for each z face the same
    // pattern in x and y
    auto plane = [&](int c) {
        if (px) {
            push(op[0], 0, c);
            push(-op[0], 0, c);
        }
        if (py) {
            push(0, op[1], c);
            if (px) {
                push(op[0], op[1], c);
                push(-op[0], op[1], c);
            }
            push(0, -op[1], c);
            if (px) {
                push(op[0], -op[1], c);
                push(-op[0], -op[1], c);
            }
        }
    };
    plane(0);
    if (pz) {
        push(0, 0, op[2]);
        if (px) {
            push(op[0], 0, op[2]);
            push(-op[0], 0, op[2]);
        }
        if (py) {
            push(0, op[1], op[2]);
            if (px) {
                push(op[0], op[1], op[2]);
                push(-op[0], op[1], op[2]);
            }
            push(0, -op[1], op[2]);
            if (px) {
                push(op[0], -op[1], op[2]);
                push(-op[0], -op[1], op[2]);
            }
        }
        push(0, 0, -op[2]);
        if (px) {
            push(op[0], 0, -op[2]);
            push(-op[0], 0, -op[2]);
        }
        if (py) {
            push(0, op[1], -op[2]);
            if (px) {
                push(op[0], op[1], -op[2]);
                push(-op[0], op[1], -op[2]);
            }
            push(0, -op[1], -op[2]);
            if (px) {
                push(op[0], -op[1], -op[2]);
                push(-op[0], -op[1], -op[2]);
            }
        }
    }
    // each image of the real nodes 1..Nm, clipped to the stored box 1-g..Nm+g
    int nb = 0;
    for (int q = 0; q < n; ++q) {
        GhostBlock b{};
        bool any = true;
        for (int d = 0; d < 3; ++d) {
            if (d >= dim) {
                b.src[d] = 1;
                b.size[d] = 1;
                b.off[d] = 0;
                continue;
            }
            const int nm = m.N[d] + 1;
            const int lo = (1 + shifts[q][d]) > (1 - g[d]) ? 1 + shifts[q][d] : 1 - g[d];
            const int hi = (nm + shifts[q][d]) < (nm + g[d]) ? nm + shifts[q][d] : nm + g[d];
            if (hi < lo) any = false;
            b.src[d] = lo - shifts[q][d];
            b.size[d] = hi - lo + 1;
            b.off[d] = shifts[q][d];
        }
        if (any) out[nb++] = b;
    }
    return nb;
}

// The blocks of one mapping and where each starts in the pack buffer
// (elements) and in the launch (workgroups).
struct GhostList {
    GhostBlock b[26];
    int64_t base[27];
    unsigned wg[27];
    int64_t per;                // elements per workgroup
    int N[3];                   // cells per axis (0: not an axis of the mesh)
    int face[26];               // the only shifted axis of a face's block, else -1
    int nb;
};
constexpr int GHOST_WG = 256;   // threads per workgroup

// Both steps run as one launch over all blocks, an element per thread: a
// 3D periodic box has 26 blocks, most of them small, and a launch per block
// and direction was 52 launches of 4-7 us (256^3 box, ghost size
// 2, lda 3, FP64: 0.30 ms for ghost_get against 0.05 ms for the two).
//
// Node (i,j,k) (1-based, the reference's numbering) of a block is src +
// (i,j,k) - 1; its image adds off.
// push: every block is read before any is written,
//   GET: buf <- field(src block),    PUT: buf <- field(image block).
// pop, in list order where blocks overlap,
//   GET: field(image block) <- buf,  PUT: field(src block) += buf.
// Blocks meet only where a coordinate lies on two images at once, so a node's
// whole list is carried out by one thread: for GET the node's last block (the
// value the list leaves), for PUT its first block, which adds the buffered
// values of every block of the node in list order.
// LOGIC: the elements are logicals (nonzero = .TRUE.), set as 1 / 0; the pop
// adds by .AND.  mask (nullptr: every node) holds one logical per stored node.

// This workgroup's block.
__device__ __forceinline__ int ghost_block_of(const GhostList& l) {
    int q = 0;
    while (blockIdx.x >= l.wg[q + 1]) ++q;
    return q;
}

// Component and 0-based real node of element e of block b.
__device__ __forceinline__ void ghost_element(const GhostBlock& b, int lda, int64_t e, int& c, int (&n)[3]) {
    auto split = [&](auto r) {   // 32-bit divisions wherever e fits
        using U = decltype(r);
        const U node = r / (U)lda;
        c = (int)(r - node * (U)lda);
        const U row = node / (U)b.size[0];
        n[0] = (int)(node - row * (U)b.size[0]);
        const U pl = row / (U)b.size[1];
        n[1] = (int)(row - pl * (U)b.size[1]);
        n[2] = (int)pl;
    };
    if ((uint64_t)e >> 32) split((uint64_t)e);
    else split((uint32_t)e);
#pragma unroll
    for (int d = 0; d < 3; ++d) n[d] += b.src[d] - 1;
}

__device__ __forceinline__ int64_t ghost_node(const FieldGeom& fg, const int (&n)[3]) {
    return ((int64_t)(n[2] - fg.lo[2]) * fg.ext[1] + (n[1] - fg.lo[1])) * fg.ext[0] + (n[0] - fg.lo[0]);
}

// Node n (0-based) in block b's real nodes (img false) or their images (true).
__device__ __forceinline__ bool ghost_holds(const GhostBlock& b, const int (&n)[3], bool img) {
    bool in = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int i = n[d] - (b.src[d] - 1) - (img ? b.off[d] : 0);
        in = in && i >= 0 && i < b.size[d];
    }
    return in;
}

template <typename T>
__global__ void __launch_bounds__(GHOST_WG) k_ghost_push(const T* __restrict__ field, FieldGeom fg, GhostList l,
                                                         T* __restrict__ buf, bool get) {
    const int q = ghost_block_of(l);
    const GhostBlock& b = l.b[q];
    const int64_t e0 = (int64_t)(blockIdx.x - l.wg[q]) * l.per;
    const int64_t e1 = min(e0 + l.per, l.base[q + 1] - l.base[q]);
    for (int64_t e = e0 + threadIdx.x; e < e1; e += GHOST_WG) {
        int c, n[3];
        ghost_element(b, fg.lda, e, c, n);
        if (!get)
            for (int d = 0; d < 3; ++d) n[d] += b.off[d];
        buf[l.base[q] + e] = field[ghost_node(fg, n) * fg.lda + c];
    }
}

template <typename T, bool LOGIC>
__global__ void __launch_bounds__(GHOST_WG) k_ghost_pop(T* __restrict__ field, FieldGeom fg, GhostList l,
                                                        const T* __restrict__ buf, bool get,
                                                        const int* __restrict__ mask) {
    const int q = ghost_block_of(l);
    const int64_t e0 = (int64_t)(blockIdx.x - l.wg[q]) * l.per;
    const int64_t e1 = min(e0 + l.per, l.base[q + 1] - l.base[q]);
    for (int64_t e = e0 + threadIdx.x; e < e1; e += GHOST_WG) {
        int c, n[3];
        ghost_element(l.b[q], fg.lda, e, c, n);
        bool other = false;   // another block's thread carries out this node's list
        if (get) {
            for (int d = 0; d < 3; ++d) n[d] += l.b[q].off[d];
            // Two images of the real range 0..N meet on the nodes 0 and N only,
            // and a face's shares its own axis' node with the real range, no
            // image: a third of a face's nodes need no search of the blocks (256^3
            // box, ghost size 2, lda 3, FP64: 36 us, 69 with one for every seam node).
            bool seam = false;
            for (int d = 0; d < 3; ++d)
                seam = seam || (d != l.face[q] && l.N[d] && (n[d] == 0 || n[d] == l.N[d]));
            if (seam)
                for (int p = q + 1; p < l.nb && !other; ++p) other = ghost_holds(l.b[p], n, true);
        } else {
            for (int p = 0; p < q && !other; ++p) other = ghost_holds(l.b[p], n, false);
        }
        if (other) continue;
        const int64_t node = ghost_node(fg, n);
        if (mask && mask[node] == 0) continue;
        T* at = field + node * fg.lda + c;
        if (get) {
            const T v = buf[l.base[q] + e];
            if constexpr (LOGIC) *at = v != T(0) ? T(1) : T(0);
            else *at = v;
            continue;
        }
        T v = *at;
        for (int p = q; p < l.nb; ++p) {
            const GhostBlock& b = l.b[p];
            if (!ghost_holds(b, n, false)) continue;
            const T w = buf[l.base[p] +
                            (((int64_t)(n[2] - (b.src[2] - 1)) * b.size[1] + (n[1] - (b.src[1] - 1))) * b.size[0] +
                             (n[0] - (b.src[0] - 1))) * fg.lda + c];
            if constexpr (LOGIC) v = v != T(0) && w != T(0) ? T(1) : T(0);
            else if constexpr (std::is_integral<T>::value) v = (T)((uint32_t)v + (uint32_t)w);   // wraps, as the hardware add
            else v = v + w;
        }
        *at = v;
    }
}

template <typename T, bool LOGIC>
static int ghost_typed(const DevMesh& m, T* field, const FieldGeom& fg, const GhostBlock* b, int nb, bool get,
                       const int* mask, DevBuf& scratch, hipStream_t s) {
    GhostList l;
    l.nb = nb;
    for (int d = 0; d < 3; ++d) l.N[d] = d < m.dim ? m.N[d] : 0;
    l.base[0] = 0;
    for (int q = 0; q < nb; ++q) {
        l.b[q] = b[q];
        int shifted = 0, axis = -1;
        for (int d = 0; d < 3; ++d)
            if (b[q].off[d] != 0) {
                ++shifted;
                axis = d;
            }
        l.face[q] = shifted == 1 ? axis : -1;
        l.base[q + 1] = l.base[q] + (int64_t)b[q].size[0] * b[q].size[1] * b[q].size[2] * fg.lda;
    }
    if (l.base[nb] == 0) return 0;
    // one element per thread, more where that would be over 2^20 workgroups
    l.per = GHOST_WG * ((l.base[nb] >> 28) + 1);
    l.wg[0] = 0;
    for (int q = 0; q < nb; ++q) l.wg[q + 1] = l.wg[q] + (unsigned)((l.base[q + 1] - l.base[q] + l.per - 1) / l.per);
    const unsigned wg = l.wg[nb];
    if (scratch.ensure(sizeof(T) * (size_t)l.base[nb])) return PPMG_ERROR_FATAL;
    T* buf = scratch.as<T>();
    hipLaunchKernelGGL(k_ghost_push<T>, dim3(wg), dim3(GHOST_WG), 0, s, field, fg, l, buf, get);
    hipLaunchKernelGGL((k_ghost_pop<T, LOGIC>), dim3(wg), dim3(GHOST_WG), 0, s, field, fg, l, buf, get, mask);
    PPMG_HIP(hipGetLastError());
    return 0;
}

int map_field_ghost(const DevMesh& m, int kind, const FieldGeom& fg_in, void* field, const int* g, bool get,
                    const int* mask, DevBuf& scratch, hipStream_t s) {
    GhostBlock b[26];
    const int nb = ghost_blocks(m, g, b);
    FieldGeom fg = fg_in;
    switch (kind) {
    case PPMG_KIND_D: return ghost_typed<double, false>(m, (double*)field, fg, b, nb, get, mask, scratch, s);
    case PPMG_KIND_S: return ghost_typed<float, false>(m, (float*)field, fg, b, nb, get, mask, scratch, s);
    case PPMG_KIND_I: return ghost_typed<int, false>(m, (int*)field, fg, b, nb, get, mask, scratch, s);
    case PPMG_KIND_L: return ghost_typed<int, true>(m, (int*)field, fg, b, nb, get, mask, scratch, s);
    case PPMG_KIND_DC:
        fg.lda *= 2;   // (re, im) pairs: each part maps and adds as a real component
        return ghost_typed<double, false>(m, (double*)field, fg, b, nb, get, mask, scratch, s);
    case PPMG_KIND_SC:
        fg.lda *= 2;
        return ghost_typed<float, false>(m, (float*)field, fg, b, nb, get, mask, scratch, s);
    default:
        set_error(PPMG_ERROR_ERROR, PPMG_ERR_ARGUMENT, "unknown element kind");
        return PPMG_ERROR_ERROR;
    }
}

}  // namespace ppmg
