// ppmg_work.hip -- work list of the 3D tile kernels for crowded input.
//
// Clustered particles put most of the work of a launch into a few percent of
// its tiles: at 512^3 with four Gaussian blobs a plane step of a blob's core
// takes 70 rounds where one of the empty space takes none, and since every
// XCD walks a slab of z, some XCDs hold no blob at all.  Such launches take
// their workgroups from a list instead of a grid: every tile column is cut
// into pieces of 1 to 32 planes by the particles its window holds (the cell
// heads give them), and the list has the heaviest class of pieces first, so
// that the dispatcher hands them out evenly over the XCDs and the light ones
// fill in behind.  Which workgroup makes a node, and where its tile column is
// cut, does not change the order of the node's additions.
#include <algorithm>

#include "ppmg_internal.h"
#include "ppmg_sort.h"

namespace ppmg {

constexpr int WK_SEG = 32;          // planes per segment (the longest piece)
// A piece's cost is counted in plane steps of one round, 1.5 rounds per
// particle of a mean cell (64 cells' fullest against their mean).  A segment
// is cut in aligned pieces of 32, 16, ... 1 planes, the longest of which the
// cost stays under `most`, a share of the mean load of a resident workgroup's
// place (build_work).
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

// One workgroup per (tile column, segment): 8 threads a plane.  count: pieces
// taken in each class so far; items: the classes' places, cap each.
__global__ void __launch_bounds__(256) k_work_cut(DevMesh m, TileWindow w, const int* __restrict__ start, int nseg,
                                                  int most, int* __restrict__ count, int64_t cap,
                                                  int2* __restrict__ items) {
    __shared__ int cost[WK_SEG];
    const int id = blockIdx.x;
    const int col = id / nseg, seg = id - col * nseg;
    const int tx = col % w.ntx, ty = col / w.ntx;
    const int t = threadIdx.x, pl = t >> 3, sub = t & 7;
    const int z = seg * WK_SEG + pl;
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
    // lane t < WK_SEG: the costs of the aligned 1, 2, ... 32 planes around plane t
    int sums[6];
    sums[0] = t < WK_SEG ? cost[t] : 0;
#pragma unroll
    for (int l = 1; l < 6; ++l) sums[l] = sums[l - 1] + __shfl_xor(sums[l - 1], 1 << (l - 1), 64);
    int n = 1, c = sums[0];
#pragma unroll
    for (int l = 1; l < 6; ++l) {
        // a piece of no more planes than its halo pays to be cut only if it costs more
        const int len = 1 << l;
        const int64_t lim = len <= w.halo + 1 ? (int64_t)most * (2 * (w.halo + 1) / len) : most;
        // (a gather's light pieces fill in behind as 4 planes: 32 only where there is next to nothing)
        if (sums[l] <= lim && (w.halo || (len != 8 && len != 16))) n = len, c = sums[l];
    }
    const int z0 = seg * WK_SEG + t;
    const bool first = t < WK_SEG && z0 < w.planes && (t & (n - 1)) == 0;
    // classes: 0 heaviest
    const int cls = c > most ? 0 : c > most / 2 ? 1 : c > most / 4 ? 2 : 3;
#pragma unroll
    for (int k = 0; k < WK_CLASSES; ++k) {
        const uint64_t mask = __ballot(first && cls == k);
        if (!mask) continue;
        int at = 0;
        if (t == 0) at = atomicAdd(&count[k], (int)__popcll(mask));
        at = __shfl(at, 0, 64) + (int)__popcll(mask & ((1ull << t) - 1));
        if (first && cls == k) items[k * cap + at] = make_int2(col, z0 << 6 | min(n, w.planes - z0));
    }
}

bool work_list_applies(const ppmg_plan* plan, int tz) {
    // crowded cells (estimated) in more than 1/1024 of the cells, binned with heads
    return tz > 1 && plan->crowded_cells > plan->ncells / 1024 && !plan->bin_table && !plan->bin_lattice && !arena_bound();
}

int build_work(ppmg_plan* plan, const DevMesh& m, const TileWindow& w, int slots, hipStream_t s, WorkList* list,
               unsigned* nitems) {
    const int nseg = (w.planes + WK_SEG - 1) / WK_SEG;
    const int64_t nid = (int64_t)w.ntx * w.nty * nseg, cap = nid * WK_SEG;
    // more pieces than the scratch should hold, or planes than an item's word: no list
    if (nid >= (int64_t)1 << 21 || w.planes >= 1 << 25) return 0;
    // (1 KiB per column segment: 16 MiB at 512^3.)  The grid does without it.
    if (!plan->work.try_ensure(sizeof(int2) * (size_t)(WK_CLASSES * cap)) ||
        !plan->work_cnt.try_ensure(sizeof(int) * WK_CLASSES))
        return 0;
    int* count = plan->work_cnt.as<int>();
    const double load = ((double)w.ntx * w.nty * w.planes + 1.5 * (double)plan->np / ((double)w.tx * w.ty)) / slots;
    // Clustered input (half a particle a cell, four blobs), M'4.  The deposit pays
    // for a cut with its halo planes: FP64, lda 3, 512^3 9.7, 9.2, 9.0 ms and
    // 168 x 169 x 249 718, 734, 774 us at shares of 0.5, 0.75 and 1.  A gather pays
    // little and is best cut fine, whatever its size.  At shares of 0.25, 0.5 and
    // 0.75, us (loads of 9, 54, 125, 431 and 1000):
    //                       gather FP64 lda 3    FP32c lda 3       FP64 lda 1       adjoint FP64 lda 3
    //   100 x 90 x 110      139 141 175          144 148 175       102 102 121      279 294 346
    //   168 x 169 x 249     477 592 679          449 542 648       327 398 466      952 1402 1533
    //   256^3               961 1309 1141        913 1250 1038     740 898 861      2298 2524 2622
    //   384^3               3311 3356 3440       2980 3071 3114    2415 2487 2471   7239 7276 7334
    //   512^3               8099 8050 8078       7397 7259 7176    6179 6171 6134   16750 16608 16691
    // (0.15 is within 3% of 0.25 but for the FP64 adjoint at 256^3, 2002; BSP2 gathers
    // differ by up to 3% from 0.15 to 0.5 and lose at 0.75.  A fixed cost of 800 took
    // 2850 and 830 us at 168 x 169 x 249; chunks of one height 1459 and 753 us.)
    const double share = w.halo ? 0.75 : 0.25;
    const int most = (int)std::min(std::max(load * share, 4.0), 1e6);
    if (fill_zero(count, sizeof(int) * WK_CLASSES, s)) return PPMG_ERROR_FATAL;
    hipLaunchKernelGGL(k_work_cut, dim3((unsigned)nid), dim3(256), 0, s, m, w, plan->start.as<int>(), nseg, most, count,
                       cap, plan->work.as<int2>());
    PPMG_HIP(hipGetLastError());
    int n[WK_CLASSES];
    if (read_back(plan, count, WK_CLASSES, n, s)) return PPMG_ERROR_FATAL;
    list->items = plan->work.as<int2>();
    list->cap = cap;
    for (int k = 0; k < WK_CLASSES; ++k) list->end[k] = (unsigned)n[k] + (k ? list->end[k - 1] : 0u);
    *nitems = list->end[WK_CLASSES - 1];
    return 0;
}

}  // namespace ppmg
