// ppmg_work.hip -- work list of the 3D tile kernels for crowded input.
//
// Clustered particles put most of the work of a launch into a few percent of
// its tiles: at 512^3 with four Gaussian blobs a plane step of a blob's core
// takes 70 rounds where one of the empty space takes none, and since every
// XCD walks a slab of z, some XCDs hold no blob at all.  Such launches take
// their workgroups from a list instead of a grid: every tile column is cut
// into pieces of 2 to 32 planes by the particles its window holds (the cell
// heads give them), and the list has the heaviest class of pieces first, so
// that the dispatcher hands them out evenly over the XCDs and the light ones
// fill in behind.  Which workgroup makes a node, and where its tile column is
// cut, does not change the order of the node's additions.
#include "ppmg_internal.h"
#include "ppmg_sort.h"

namespace ppmg {

constexpr int WK_SEG = 32;          // planes per segment (the longest piece)
constexpr int WK_BLOCK = 2;         // planes per block (the shortest piece)
constexpr int WK_NB = WK_SEG / WK_BLOCK;
constexpr int WK_CLASSES = 4;
// A piece's cost is counted in plane steps of one round, 1.5 rounds per
// particle of a mean cell (64 cells' fullest against their mean).  Pieces
// stay under WK_COST where WK_SEG, 8 or 4 planes allow it: short enough that
// the heaviest, started first, end before the launch does, long enough for the
// deposit's three halo planes (clustered 512^3 deposit: 10.8, 10.3, 9.5, 10.0 and
// 11.2 ms at 128, 256, 640, 1500 and 4000).
constexpr int WK_COST = 800;

__device__ __forceinline__ int piece_planes(int code) { return code == 0 ? 2 : code == 1 ? 4 : code == 2 ? 8 : WK_SEG; }

// Particles of the cells [c, c + n) of a row of cells (wrapping on a periodic
// axis, clipped on an open one); row: the row's first cell.
__device__ __forceinline__ int row_particles(const int* __restrict__ start, int64_t row, int c, int n, int nb,
                                             bool periodic) {
    if (!periodic) {
        const int a = max(c, 0), b = min(c + n, nb);
        return b > a ? start[row + b] - start[row + a] : 0;
    }
    int sum = 0;
    c %= nb;
    if (c < 0) c += nb;
    while (n > 0) {
        const int k = min(n, nb - c);
        sum += start[row + c + k] - start[row + c];
        n -= k;
        c = 0;
    }
    return sum;
}

// One workgroup per (tile column, segment): 8 threads a plane.  code: 4 bits
// per block, the piece's length code and class; count: pieces by class.
__global__ void __launch_bounds__(256) k_work_cut(DevMesh m, TileWindow w, const int* __restrict__ start, int nseg,
                                                  uint64_t* __restrict__ code, int* __restrict__ count) {
    __shared__ int cost[WK_SEG];
    __shared__ int ncls[WK_CLASSES];
    const int id = blockIdx.x, nid = gridDim.x;
    const int col = id / nseg, seg = id - col * nseg;
    const int tx = col % w.ntx, ty = col / w.ntx;
    const int t = threadIdx.x, pl = t >> 3, sub = t & 7;
    const int z = seg * WK_SEG + pl;
    if (t < WK_CLASSES) ncls[t] = 0;
    int64_t sum = 0;
    if (z < w.planes) {
        const int cz = z < m.nbin[2] ? z : m.nbin[2] - 1;
        for (int r = sub; r < w.nrow; r += 8) {
            int cy = ty * w.ty + w.wy + r;
            if (m.periodic[1]) {
                cy %= m.nbin[1];
                if (cy < 0) cy += m.nbin[1];
            }
            if (cy >= 0 && cy < m.nbin[1])
                sum += row_particles(start, (int64_t)m.nbin[0] * (cy + (int64_t)m.nbin[1] * cz), tx * w.tx + w.wx,
                                     w.ncol, m.nbin[0], m.periodic[0]);
        }
    }
    int s = (int)min(sum, (int64_t)1 << 24);
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) s += __shfl_xor(s, o, 64);
    const int cells = w.nrow * w.ncol;
    if (sub == 0) cost[pl] = z < w.planes ? max(1, (int)min((int64_t)3 * s / (2 * cells), (int64_t)1 << 20)) : 0;
    __syncthreads();
    if (t >= 64) return;
    // lane b < WK_NB: block b's cost, and those of the aligned 2, 4 and 16 blocks around it
    int c2 = t < WK_NB ? cost[WK_BLOCK * t] + cost[WK_BLOCK * t + 1] : 0;
    const int c4 = c2 + __shfl_xor(c2, 1, 64);
    const int c8 = c4 + __shfl_xor(c4, 2, 64);
    int c32 = c8 + __shfl_xor(c8, 4, 64);
    c32 += __shfl_xor(c32, 8, 64);
    const int len = c32 <= WK_COST ? 3 : c8 <= WK_COST ? 2 : c4 <= 2 * WK_COST ? 1 : 0;
    const int c = len == 3 ? c32 : len == 2 ? c8 : len == 1 ? c4 : c2;
    // classes: 0 heaviest
    const int cls = c > WK_COST ? 0 : c > WK_COST / 2 ? 1 : c > WK_COST / 4 ? 2 : 3;
    const int z0 = seg * WK_SEG + WK_BLOCK * t;
    if (t < WK_NB && z0 < w.planes && (WK_BLOCK * t) % piece_planes(len) == 0) atomicAdd(&ncls[cls], 1);
    uint64_t bits = t < WK_NB ? (uint64_t)((cls << 2) | len) << (4 * t) : 0ull;
#pragma unroll
    for (int o = 1; o < WK_NB; o <<= 1) {
        const unsigned lo = __shfl_xor((unsigned)bits, o, 64), hi = __shfl_xor((unsigned)(bits >> 32), o, 64);
        bits |= ((uint64_t)hi << 32) | lo;
    }
    if (t == 0) code[id] = bits;
    wave_lds_sync();
    if (t < WK_CLASSES) count[(int64_t)t * nid + id] = ncls[t];
}

// The pieces of every segment at their places (offs: the exclusive scan of count).
__global__ void __launch_bounds__(256) k_work_fill(TileWindow w, int nseg, int nid, const uint64_t* __restrict__ code,
                                                   const int* __restrict__ offs, int4* __restrict__ items) {
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= nid) return;
    const int col = id / nseg, seg = id - col * nseg;
    const uint64_t bits = code[id];
    int at[WK_CLASSES];
#pragma unroll
    for (int k = 0; k < WK_CLASSES; ++k) at[k] = offs[(int64_t)k * nid + id];
    for (int b = 0; b < WK_NB;) {
        const int q = (int)(bits >> (4 * b)) & 15, n = piece_planes(q & 3), cls = q >> 2;
        const int z0 = seg * WK_SEG + WK_BLOCK * b;
        if (z0 >= w.planes) break;
        const int4 it = make_int4(col, z0, min(z0 + n, w.planes), 0);
#pragma unroll
        for (int k = 0; k < WK_CLASSES; ++k)
            if (cls == k) items[at[k]++] = it;
        b += n / WK_BLOCK;
    }
}

bool work_list_applies(const ppmg_plan* plan) {
    // crowded cells (estimated) in more than 1/1024 of the cells, binned with heads
    return plan->crowded_cells > plan->ncells / 1024 && !plan->bin_table && !plan->bin_lattice && !arena_bound();
}

int build_work(ppmg_plan* plan, const DevMesh& m, const TileWindow& w, hipStream_t s, const int4** items,
               unsigned* nitems) {
    const int nseg = (w.planes + WK_SEG - 1) / WK_SEG;
    const int64_t nid64 = (int64_t)w.ntx * w.nty * nseg;
    const int64_t ncnt = WK_CLASSES * nid64 + 1;   // and a closing zero, whose prefix is the total
    if (nid64 >= (int64_t)1 << 26) return 1;       // more pieces than a launch takes: no list
    const int nid = (int)nid64;
    const int64_t cnt_at = 2 * nid64, offs_at = (cnt_at + ncnt + 3) & ~(int64_t)3;
    if (plan->work.ensure(sizeof(int4) * (size_t)(WK_NB * nid64)) ||
        plan->work_cnt.ensure(sizeof(int) * (size_t)(offs_at + ncnt + 1)))
        return PPMG_ERROR_FATAL;
    int* base = plan->work_cnt.as<int>();
    uint64_t* code = reinterpret_cast<uint64_t*>(base);
    int *cnt = base + cnt_at, *offs = base + offs_at;
    if (fill_zero(cnt + ncnt - 1, sizeof(int), s)) return PPMG_ERROR_FATAL;
    hipLaunchKernelGGL(k_work_cut, dim3((unsigned)nid), dim3(256), 0, s, m, w, plan->start.as<int>(), nseg, code, cnt);
    if (exclusive_scan(cnt, ncnt, offs, plan->scan_tmp, 0, s)) return PPMG_ERROR_FATAL;
    hipLaunchKernelGGL(k_work_fill, dim3((unsigned)((nid + 255) / 256)), dim3(256), 0, s, w, nseg, nid, code, offs,
                       plan->work.as<int4>());
    PPMG_HIP(hipGetLastError());
    int total = 0;
    if (read_back(plan, offs + ncnt - 1, 1, &total, s)) return PPMG_ERROR_FATAL;
    *items = plan->work.as<int4>();
    *nitems = (unsigned)total;
    return 0;
}

}  // namespace ppmg
