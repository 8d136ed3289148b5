// ppmg_sort.h -- counting sort / ranking entry points shared inside libppmg.
#pragma once
#include "ppmg_internal.h"

namespace ppmg {

// Geometry of ppm_util_rank3d / rank2d (ppm_util_rank3d.f:309-355).
struct RankGeom {
    int dim;
    int nm[3];        // cells per axis (the reference's Nm)
    int ngl_lo[3];
    int ntot[3];      // nm + ngl_lo + ngl_hi (1 on unused axes)
    double xmin[3], xmax[3];
    double rdx[3];    // Nm / (xmax - xmin) in the position precision
};

// Byte-wide cell counts of the binning.  In every block of 256 cells, cell c
// sits in word c mod 64, byte (c / 64) mod 4: the 64 consecutive cells a
// wavefront of lattice-ordered particles hits fall in 64 different words, so
// the atomic counts of neighbouring lanes do not contend for one word.  The
// array is padded to whole blocks and zeroed, so reads need no bounds.
__host__ __device__ inline int64_t count_word(int64_t c) { return ((c >> 8) << 6) + (c & 63); }
__host__ __device__ inline unsigned count_shift(int64_t c) { return (unsigned)((c >> 6) & 3) * 8u; }

// Slot table of a binning (plan->bin_table): particle r (0 <= r < count) of
// cell c, in increasing particle index, is table[r * ncells + c].  A cell
// with more than TABLE_SLOTS particles sends the binning to the heads and
// permutation instead.  Eight slots hold every cell of a lattice jittered by
// less than half a cell and displaced by a locally uniform shift: a cell then
// meets at most two particles per axis.
constexpr int TABLE_SLOTS = 8;

// A slot-table binning as the tiled kernels read it.
struct BinTable {
    const uint32_t* count;
    const int* table;
    int64_t ncells;
};

// Cell key of one particle with the index arithmetic of ppm_interp_p2m.f:
// 800-822 (x0 = (x - min)*dxi, INT truncation) and the sub test of :535-561;
// -1 when the particle lies in no cell of the sub.
template <int DIM, typename PosT>
__device__ __forceinline__ int cell_key(const PosT (&x)[DIM], const DevMesh& m) {
    bool ok = true;
    int cell[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        PosT v = x[d];
        PosT mn = (PosT)m.minv[d];
        PosT mx = (PosT)m.maxv[d];
        if (!(v >= mn && v <= mx)) ok = false;
        if (!(v < mx || !m.upper_open[d])) ok = false;
        PosT x0 = scaled_coord<PosT>(v, mn, (PosT)m.dxi[d]);
        int i = ok ? (int)x0 : 0;
        if (m.periodic[d] && i >= m.N[d]) i -= m.N[d];
        if (i < 0 || i >= m.nbin[d]) ok = false;
        cell[d] = i;
    }
    return ok ? cell[0] + m.nbin[0] * (cell[1] + m.nbin[1] * cell[2]) : -1;
}

int exclusive_scan(const int* in, int64_t n, int* out, DevBuf& tmp, int64_t total, hipStream_t s);
int fill_zero(void* p, size_t bytes, hipStream_t s);
// Bins np particles into the plan (key, perm, start); *nbad = particles outside the sub.
// table: the caller reads a slot table (plan->bin_table) where the binning
// can leave one instead of the heads and the permutation.  lattice: the
// caller checks every particle's cell (err[6]), so a plan that predicts a
// lattice in cell order may take it without a pass (plan->bin_lattice).
int bin_particles(ppmg_plan* plan, const DevMesh& m, int prec, int64_t np, const void* xp,
                  hipStream_t s, int64_t* nbad, bool table = false, bool lattice = false);
// Heads and permutation of a binning that left a slot table (no-op otherwise).
int materialize_heads(ppmg_plan* plan, hipStream_t s);
// The binning leaves the identity permutation implicit when the input is
// already in cell order.  Tiled kernels take tile_perm(): nullptr then, and
// they read particle f at sorted position f; other readers of plan->perm call
// materialize_perm() first.
inline const int* tile_perm(const ppmg_plan* plan) { return plan->perm_identity ? nullptr : plan->perm.as<int>(); }
int materialize_perm(ppmg_plan* plan, hipStream_t s);   // calls materialize_heads() first
// Input binned in cell order leaves the keys unwritten too; readers of
// plan->key call materialize_keys() first (it reads the positions of that
// binning, which must still hold them).
int materialize_keys(ppmg_plan* plan, hipStream_t s);
int rank_particles(ppmg_plan* plan, const RankGeom& g, int prec, int64_t np, const void* xp,
                   int* lpdx, int* lhbx, int64_t* icount, hipStream_t s);
// xp (np rows of dim) reordered by the 1-based ranking lpdx1; npbx (may be
// NULL) = particles per box from the 1-based heads lhbx1.
int sort_rows(int dim, int prec, int64_t np, void* xp, const int* lpdx1, const int* lhbx1, int64_t nbox, int* npbx,
              DevBuf& tmp, hipStream_t s);

// Runs a gather of the plan's binning.  A plan whose last binning found a
// lattice in cell order (particle p in cell p, one per cell: a fresh lattice of
// remeshed particles) takes the next one on the same mesh as that lattice
// without a binning pass: the gather checks every particle's cell key and,
// should one differ, the particles are binned (table: a slot table will do) and
// gathered again.  Returns 1 when some particle then lies outside the sub.
template <typename F>
int gather_checked(ppmg_plan* plan, const DevMesh& m, int prec, int64_t np, const void* xp, bool table, hipStream_t s,
                   F&& gather) {
    if (!plan->bin_lattice) return gather();
    // (the binning cleared the mismatch flag)
    if (gather()) return PPMG_ERROR_FATAL;
    int off = 0;
    if (read_back(plan, plan->err.as<int>() + 6, 1, &off, s)) return PPMG_ERROR_FATAL;
    if (!off) {
        plan->lattice_checked = true;   // the plan's binning is the lattice (heads written on demand)
        return 0;
    }
    // not that lattice: bin and gather again (and bin the next 16 inputs)
    plan->lattice_flag_clear = false;
    plan->lattice_pred = false;
    plan->lattice_skip = 16;
    int64_t nbad = 0;
    if (bin_particles(plan, m, prec, np, xp, s, &nbad, table, false)) return PPMG_ERROR_FATAL;
    if (nbad > 0) return 1;
    return gather();
}

// ------------------------------------------- work list (ppmg_work.hip) --
// Tile columns of a 3D tile kernel: ntx x nty tiles of tx x ty, marching
// `planes` planes; a tile's cells are the ncol x nrow ones starting at offset
// (wx, wy) from its first.  halo: planes of particles a piece takes beyond its
// own.
struct TileWindow {
    int ntx, nty, tx, ty;
    int wx, wy, ncol, nrow;
    int planes, halo;
};
// Pieces of tile columns in WK_CLASSES classes, heaviest first: class k's lie
// at items + k * cap and are workgroups end[k-1] .. end[k]-1; a piece is its
// column and first plane * 64 + planes.
constexpr int WK_CLASSES = 4;
struct WorkList {
    const int2* items = nullptr;
    int64_t cap = 0;
    unsigned end[WK_CLASSES] = {};
};
// The plan's last binning found crowded cells and left heads: launches take
// their workgroups from a work list.  tz: the grid's chunk; single planes leave
// nothing to cut (95 x 86 x 54, BSP2, half a particle a cell in blobs: deposit
// 100 us, 144 with the list).
bool work_list_applies(const ppmg_plan* plan, int tz);
// The pieces of all tile columns, in the plan's scratch, and their number
// (slots: resident workgroups of the kernel); the list stays empty where it
// would take too much scratch, or where the scratch is refused.
int build_work(ppmg_plan* plan, const DevMesh& m, const TileWindow& w, int slots, hipStream_t s, WorkList* list,
               unsigned* nitems);
// This workgroup's tile column and planes [z0, z1): from the work list, or
// (no items) the grid's chunks of tz planes in XCD order.
__device__ __forceinline__ void tile_piece(const WorkList& list, int ntx, int nty, int tz, int planes, int& tx,
                                           int& ty, int& z0, int& z1) {
    int col;
    if (list.items) {
        const unsigned b = blockIdx.x;
        int64_t at = b;
#pragma unroll
        for (int k = 1; k < WK_CLASSES; ++k)
            if (b >= list.end[k - 1]) at = k * list.cap + (b - list.end[k - 1]);
        const int2 it = list.items[at];
        col = it.x;
        z0 = it.y >> 6;
        z1 = z0 + (it.y & 63);
    } else {
        const int64_t tile = xcd_tile(blockIdx.x, (int64_t)gridDim.x);
        const int64_t ncol = (int64_t)ntx * nty;
        const int chunk = (int)(tile / ncol);
        col = (int)(tile - chunk * ncol);
        z0 = chunk * tz;
        z1 = min(z0 + tz, planes);
    }
    ty = col / ntx;
    tx = col - ty * ntx;
}

}  // namespace ppmg
