// ppmg_sort.hip -- stable counting sort of particles into cells (gfx950).
//
// Replaces the cell ranking of ppm_util_rank3d / rank2d
// (ppm_util_rank3d.f:309-532): count particles per cell, exclusive prefix
// over the cells, scatter in particle order.  On the GPU the count and the
// scatter use integer atomics, which place the particles of one cell in an
// arbitrary order; a per-cell pass then restores increasing particle index,
// so the permutation equals the reference's lpdx exactly.
#include <climits>
#include <cstdlib>

#include "ppmg_internal.h"
#include "ppmg_sort.h"

namespace ppmg {

// Binning status words: err[0] particles outside the sub, err[1] a descent
// seen, err[2] queued runs of empty cells, err[3] a byte count overflowed,
// err[4] a cell with more particles than the slot table holds, err[5] a
// particle p not in cell p, err[6] (the gather's check of a lattice
// binning) the same, err[8..71] sampled crowded cells, err[72..135] sampled
// particles far from the one before them.
constexpr int ERR_WORDS = 136;
// Input of FAR_MIN_NP particles or more, of which at least a quarter lie more
// than FAR_CELLS cells from their predecessor, is in no order: the slot atomics
// and table writes of its key pass each touch a line of their own.
constexpr int FAR_CELLS = 1024;
constexpr int64_t FAR_MIN_NP = 3 << 19;
// Particles from which util_rank sorts by radix.
constexpr int64_t RANK_RADIX_NP = 3 << 18;

constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;

static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b > 0 ? (n + b - 1) / b : 1); }

// Block-wide exclusive scan of one value per thread; returns the block total.
template <int THREADS = SCAN_BLOCK>
__device__ __forceinline__ int64_t block_exclusive_scan(int64_t v, int64_t* sh, int64_t& excl) {
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wid = t >> 6;
    // wavefront inclusive scan (64 lanes)
    int64_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int64_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) sh[wid] = x;
    __syncthreads();
    if (t == 0) {
        int64_t run = 0;
        for (int w = 0; w < THREADS / 64; ++w) {
            int64_t s = sh[w];
            sh[w] = run;
            run += s;
        }
        sh[THREADS / 64] = run;
    }
    __syncthreads();
    excl = x - v + sh[wid];
    int64_t total = sh[THREADS / 64];
    __syncthreads();
    return total;
}

// Each thread owns SCAN_ITEMS consecutive elements of its tile, read (and in
// k_scan_down written) as 128-bit vectors when the tile is complete.
template <bool VEC>
__device__ __forceinline__ void load_items(const int* __restrict__ in, int64_t n, int64_t base, int (&v)[SCAN_ITEMS]) {
    if (VEC && base + SCAN_ITEMS <= n) {
        const int4* q = reinterpret_cast<const int4*>(in + base);
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS / 4; ++k) {
            int4 t = q[k];
            v[4 * k] = t.x; v[4 * k + 1] = t.y; v[4 * k + 2] = t.z; v[4 * k + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i) v[i] = base + i < n ? in[base + i] : 0;
    }
}

template <bool VEC>
__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_reduce(const int* __restrict__ in, int64_t n,
                                                            int64_t* __restrict__ block_sums) {
    __shared__ int64_t sh[SCAN_BLOCK / 64 + 1];
    int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    load_items<VEC>(in, n, base, v);
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) s += v[i];
    int64_t excl;
    int64_t tot = block_exclusive_scan(s, sh, excl);
    if (threadIdx.x == 0) block_sums[blockIdx.x] = tot;
}

// Exclusive scan of the block sums by one workgroup of SUMS_THREADS threads:
// each thread totals a contiguous segment, the segment totals are scanned
// across the workgroup, and each thread rewrites its segment as prefixes.
constexpr int SUMS_THREADS = 1024;
__global__ void __launch_bounds__(SUMS_THREADS) k_scan_sums(int64_t* __restrict__ sums, int64_t nb) {
    __shared__ int64_t sh[SUMS_THREADS / 64 + 1];
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    const int64_t seg = (nb + SUMS_THREADS - 1) / SUMS_THREADS;
    const int64_t b = t * seg, e = b + seg < nb ? b + seg : nb;
    int64_t tot = 0;
    for (int64_t i0 = b; i0 < e; i0 += 8) {   // eight loads in flight at a time
        int64_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = i0 + j < e ? sums[i0 + j] : 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) tot += v[j];
    }
    // workgroup exclusive scan of the segment totals
    int64_t x = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int64_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) sh[wid] = x;
    __syncthreads();
    if (t == 0) {
        int64_t run = 0;
        for (int w = 0; w < SUMS_THREADS / 64; ++w) {
            int64_t v = sh[w];
            sh[w] = run;
            run += v;
        }
    }
    __syncthreads();
    int64_t run = x - tot + sh[wid];
    for (int64_t i0 = b; i0 < e; i0 += 8) {
        int64_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = i0 + j < e ? sums[i0 + j] : 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (i0 + j < e) sums[i0 + j] = run;
            run += v[j];
        }
    }
}

// Up to FEW_SUMS block sums are not scanned by a launch of their own: each
// block of the last pass adds up the sums before its own (ranking of 2^24
// particles, three scans: 418 -> 411 us).
constexpr int64_t FEW_SUMS = 1024;

// Prefix of this workgroup: its scanned sum, or (few) the plain sums before it.
__device__ __forceinline__ int64_t block_prefix(const int64_t* __restrict__ sums, bool few, int64_t* sh) {
    if (!few) return sums[blockIdx.x];
    int64_t v = 0, excl;
    for (unsigned b = threadIdx.x; b < blockIdx.x; b += SCAN_BLOCK) v += sums[b];
    return block_exclusive_scan(v, sh, excl);
}

template <bool VEC>
__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_down(const int* __restrict__ in, int64_t n,
                                                          const int64_t* __restrict__ sums, bool few,
                                                          int* __restrict__ out, int64_t total_out) {
    __shared__ int64_t sh[SCAN_BLOCK / 64 + 1];
    int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int vals[SCAN_ITEMS];
    load_items<VEC>(in, n, base, vals);
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) s += vals[i];
    int64_t excl;
    const int64_t prefix = block_prefix(sums, few, sh);
    block_exclusive_scan(s, sh, excl);
    int64_t run = prefix + excl;
    int o[SCAN_ITEMS];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        o[i] = (int)run;
        run += vals[i];
    }
    if (VEC && base + SCAN_ITEMS <= n) {
        int4* q = reinterpret_cast<int4*>(out + base);
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS / 4; ++k) q[k] = make_int4(o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i)
            if (base + i < n) out[base + i] = o[i];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == SCAN_BLOCK - 1) out[n] = (int)total_out;
}

int exclusive_scan(const int* in, int64_t n, int* out, DevBuf& tmp, int64_t total, hipStream_t s) {
    int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    if (nb < 1) nb = 1;
    if (tmp.ensure(sizeof(int64_t) * (size_t)nb)) return PPMG_ERROR_FATAL;
    int64_t* sums = tmp.as<int64_t>();
    // 128-bit loads and stores need 16-byte aligned arrays (caller arrays may not be)
    const bool vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    if (vec) hipLaunchKernelGGL(k_scan_reduce<true>, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, n, sums);
    else hipLaunchKernelGGL(k_scan_reduce<false>, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, n, sums);
    const bool few = nb <= FEW_SUMS;
    if (!few) hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SUMS_THREADS), 0, s, sums, nb);
    if (vec) hipLaunchKernelGGL(k_scan_down<true>, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, n, sums, few, out, total);
    else hipLaunchKernelGGL(k_scan_down<false>, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, n, sums, few, out, total);
    PPMG_HIP(hipGetLastError());
    return 0;
}

// Counts of the 16 cells base .. base+15 (base a multiple of 16): 16
// consecutive words of one block, one byte of each.
__device__ __forceinline__ void load_counts16(const uint32_t* __restrict__ words, int64_t base, int (&c)[16]) {
    const uint4* q = reinterpret_cast<const uint4*>(words + count_word(base));
    const unsigned sh = count_shift(base);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint4 v = q[k];
        c[4 * k] = (int)((v.x >> sh) & 255u);
        c[4 * k + 1] = (int)((v.y >> sh) & 255u);
        c[4 * k + 2] = (int)((v.z >> sh) & 255u);
        c[4 * k + 3] = (int)((v.w >> sh) & 255u);
    }
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_reduce_u8(const uint32_t* __restrict__ in,
                                                               int64_t* __restrict__ block_sums) {
    __shared__ int64_t sh[SCAN_BLOCK / 64 + 1];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int c[SCAN_ITEMS];
    load_counts16(in, base, c);
    int sum = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) sum += c[i];
    int64_t excl;
    const int64_t tot = block_exclusive_scan(sum, sh, excl);
    if (threadIdx.x == 0) block_sums[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_down_u8(const uint32_t* __restrict__ in, int64_t n,
                                                             const int64_t* __restrict__ sums, bool few,
                                                             int* __restrict__ out, int64_t total_out) {
    __shared__ int64_t sh[SCAN_BLOCK / 64 + 1];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int c[SCAN_ITEMS];
    load_counts16(in, base, c);
    int sum = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) sum += c[i];
    int64_t excl;
    const int64_t prefix = block_prefix(sums, few, sh);
    block_exclusive_scan(sum, sh, excl);
    int run = (int)(prefix + excl);
    int o[SCAN_ITEMS];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        o[i] = run;
        run += c[i];
    }
    if (base + SCAN_ITEMS <= n) {
        int4* q = reinterpret_cast<int4*>(out + base);
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS / 4; ++k) q[k] = make_int4(o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i)
            if (base + i < n) out[base + i] = o[i];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == SCAN_BLOCK - 1) out[n] = (int)total_out;
}

// out (16-byte aligned, n + 1 entries) = exclusive prefix of the byte counts
// of cells 0..n-1 (laid out as count_word / count_shift, padded to whole
// 256-cell blocks), then the total.
static int exclusive_scan_u8(const uint32_t* in, int64_t n, int* out, DevBuf& tmp, int64_t total, hipStream_t s) {
    int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    if (nb < 1) nb = 1;
    if (tmp.ensure(sizeof(int64_t) * (size_t)nb)) return PPMG_ERROR_FATAL;
    int64_t* sums = tmp.as<int64_t>();
    hipLaunchKernelGGL(k_scan_reduce_u8, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, sums);
    const bool few = nb <= FEW_SUMS;
    if (!few) hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SUMS_THREADS), 0, s, sums, nb);
    hipLaunchKernelGGL(k_scan_down_u8, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, n, sums, few, out, total);
    PPMG_HIP(hipGetLastError());
    return 0;
}

// ------------------------------------------------------------ binning ---
// Heads of the cells lo..hi (all empty but possibly the last) := v.  Short
// runs are written by the lane itself; longer ones are queued for
// k_fill_gaps in pieces of GAP_CHUNK cells (err[2] counts the entries; an
// overflowing queue sends the caller to the counting path).
constexpr int GAP_LOCAL = 32;
constexpr int GAP_CHUNK = 65536;

__device__ __forceinline__ void set_heads(int* __restrict__ start, int lo, int hi, int v, int* __restrict__ err,
                                          int4* __restrict__ gaps, int gapcap) {
    if (hi - lo < GAP_LOCAL) {
        for (int c = lo; c <= hi; ++c) start[c] = v;
        return;
    }
    for (int64_t a = lo; a <= hi; a += GAP_CHUNK) {
        const int e = (int)(a + GAP_CHUNK - 1 < hi ? a + GAP_CHUNK - 1 : hi);
        const int i = atomicAdd(&err[2], 1);
        if (i < gapcap) gaps[i] = make_int4((int)a, e, v, 0);
    }
}

// Keys of all particles.  err[0] counts the particles in no cell; err[1] is
// set to 1 when a descent key[p] < key[p-1] exists (none: the input is already
// in cell order, e.g. particles made by create_part or a lattice).  A
// wavefront takes KEYS_PPT runs of 64 consecutive particles: all their
// positions are loaded first, then (SLOT) all their atomics issued, so each
// lane keeps KEYS_PPT loads and atomics in flight instead of waiting for one
// round trip at a time (one particle per thread streams the positions at
// 2.9 TB/s, bound by the atomic's latency after each load).  Lanes get their
// predecessor's key by a shuffle, lane 0 from the run before (lane 63) or,
// for the first run, from the previous particle's position, so descents
// across runs and wavefront seams are caught here too.  The flag is read
// before it is written, so the many wavefronts of unsorted input do not
// queue on one word.
//   SLOT (unsorted input expected): write the keys and take each particle's
//     arrival slot in its cell by an atomic count (byte-wide: slots 0..254).
//   SLOT and TABLE: no keys or slots written; particle p, arriving r-th in
//     cell k, is written to table[r * ncells + k] (r < TABLE_SLOTS; a later
//     arrival sets err[4]).
//   !SLOT (input expected in cell order): the first particle of each run of
//     equal keys writes its index as the head of its cell and of the empty
//     cells before it (back to its predecessor's cell); the last particle
//     closes the array with np.  No counts, no scan, no keys written, and the
//     permutation is the identity.  Valid only if no descent is found (else
//     the caller bins again on the SLOT path).
constexpr int KEYS_PPT = 4;                    // runs of 64 particles per wavefront
constexpr int KEYS_BLOCK = 256 * KEYS_PPT;     // particles per key workgroup (and list capacity)

template <int DIM, typename PosT, bool SLOT, bool TABLE>
__global__ void __launch_bounds__(256) k_keys(const PosT* __restrict__ xp, int64_t np, DevMesh m, int64_t ncells,
                                              int* __restrict__ key, uint8_t* __restrict__ slot,
                                              uint32_t* __restrict__ count, int* __restrict__ start,
                                              int* __restrict__ err, int4* __restrict__ gaps, int gapcap,
                                              int* __restrict__ multi, int* __restrict__ multi_n,
                                              int* __restrict__ table) {
    static_assert(SLOT || !TABLE, "the slot table needs the arrival slots");
    const int lane = threadIdx.x & 63;
    // first particle of this wavefront's runs (wavefront-uniform)
    const int64_t w0 = ((int64_t)blockIdx.x * 256 + __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u)) * KEYS_PPT;
    const bool has_seam = w0 > 0 && w0 <= np;
    // all loads first (the key arithmetic branches on mesh flags, which would
    // otherwise keep each load behind the previous component's arithmetic)
    // (past the end a lane reads the last particle again, unconditionally:
    // no branch between the loads)
    PosT xv[KEYS_PPT][DIM], sv[DIM];
#pragma unroll
    for (int j = 0; j < KEYS_PPT; ++j) {
        const int64_t p = min(w0 + j * 64 + lane, np - 1);
#pragma unroll
        for (int d = 0; d < DIM; ++d) xv[j][d] = xp[p * DIM + d];
    }
#pragma unroll
    for (int d = 0; d < DIM; ++d) sv[d] = has_seam ? xp[(w0 - 1) * DIM + d] : PosT(0);
    int k[KEYS_PPT];
    int nbad = 0, nfar = 0;
    uint64_t anydesc = 0, notlat = 0;
    bool desc[KEYS_PPT];
    int prev = has_seam ? cell_key<DIM, PosT>(sv, m) : -1;   // key before run j's lane 0
#pragma unroll
    for (int j = 0; j < KEYS_PPT; ++j) {
        const int64_t p = w0 + j * 64 + lane;
        const bool live = p < np;
        k[j] = live ? cell_key<DIM, PosT>(xv[j], m) : -1;
        int left = __shfl_up(k[j], 1);
        if (lane == 0) left = prev;
        prev = __builtin_amdgcn_readlane(k[j], 63);
        desc[j] = live && p > 0 && k[j] < left;
        nbad += (int)__popcll(__ballot(live && k[j] < 0));
        if (SLOT) nfar += (int)__popcll(__ballot(live && p > 0 && abs(k[j] - left) > FAR_CELLS));
        anydesc |= __ballot(desc[j]);
        notlat |= __ballot(live && k[j] != (int)p);
        if (!SLOT) {
            // heads: the first particle of a run of equal keys
            if (live && k[j] >= 0 && !desc[j]) {
                if (k[j] != left) set_heads(start, left + 1, k[j], (int)p, err, gaps, gapcap);
                if (p == np - 1) set_heads(start, k[j] + 1, (int)ncells, (int)np, err, gaps, gapcap);
            }
        }
    }
    // (last on the SLOT path: the flag's read waits for every memory
    // operation issued before it)
    auto report = [&]() {
        if (lane == 0) {
            if (nbad) atomicAdd(&err[0], nbad);
            if (anydesc && *(volatile int*)&err[1] == 0) err[1] = 1;
            if (notlat && *(volatile int*)&err[5] == 0) err[5] = 1;
            if (SLOT && nfar && (blockIdx.x & 63) == 0) atomicAdd(&err[72 + ((blockIdx.x >> 6) & 63)], nfar);
        }
    };
    if (!SLOT) report();
    if constexpr (SLOT) {
        // arrival slots, all runs' atomics in flight together: issued without
        // branches (a lane with no cell adds 0 to word 0) and decoded after
        // the last one, so no atomic waits for the one before
        uint32_t raw[KEYS_PPT];
#pragma unroll
        for (int j = 0; j < KEYS_PPT; ++j) {
            // byte-wide counts (count_word / count_shift)
            const bool in = k[j] >= 0;
            raw[j] = atomicAdd(&count[in ? count_word(k[j]) : 0], in ? 1u << count_shift(k[j]) : 0u);
        }
        int sl[KEYS_PPT];
#pragma unroll
        for (int j = 0; j < KEYS_PPT; ++j) sl[j] = k[j] >= 0 ? (int)((raw[j] >> count_shift(k[j])) & 255u) : -1;
        // The particle that arrives second in a cell lists the cell in its
        // workgroup's block of `multi` for the stabilisation.
        __shared__ int listed[KEYS_BLOCK];
        __shared__ int nlisted, ncrowd;
        if (threadIdx.x == 0) nlisted = ncrowd = 0;
        bool ov = false, full = false;
        int crowd = 0;
#pragma unroll
        for (int j = 0; j < KEYS_PPT; ++j) {
            const int64_t p = w0 + j * 64 + lane;
            if (p < np) {
                if (!TABLE) {
                    key[p] = k[j];
                    if (k[j] >= 0) slot[p] = (uint8_t)sl[j];
                } else if (sl[j] >= 0 && sl[j] < TABLE_SLOTS) {
                    table[(int64_t)sl[j] * ncells + k[j]] = (int)p;
                }
            }
            // a cell's 256th arrival carries into the next cell's byte: err[3]
            // sends the caller to the full-width count
            ov |= sl[j] == 255;
            full |= sl[j] >= TABLE_SLOTS;
            crowd += sl[j] == 8;
        }
        if (__ballot(ov) && lane == 0) err[3] = 1;
        if (TABLE && __ballot(full) && lane == 0 && *(volatile int*)&err[4] == 0) err[4] = 1;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < KEYS_PPT; ++j)
            if (sl[j] == 1) listed[atomicAdd(&nlisted, 1)] = k[j];
        if ((blockIdx.x & 63) == 0 && crowd > 0) atomicAdd(&ncrowd, crowd);
        __syncthreads();
        const int n = nlisted;
        // err[8 .. 71]: the cells whose ninth particle arrived in one key
        // workgroup of every 64 (a sample, for the deposit's choice of chunk),
        // spread over 64 words: contended device-scope atomics serialise (one
        // per crowded cell took 27 ms at 512^3 clustered, one per sampled
        // workgroup on a single word 0.85 ms)
        if (threadIdx.x == 0 && ncrowd > 0 && (blockIdx.x & 63) == 0)
            atomicAdd(&err[8 + ((blockIdx.x >> 6) & 63)], ncrowd);
        for (int i = (int)threadIdx.x; i < n; i += 256) multi[(int64_t)blockIdx.x * KEYS_BLOCK + i] = listed[i];
        if (threadIdx.x == 0) multi_n[blockIdx.x] = n;
        report();
    }
}

// Long runs of empty cells queued by k_keys: one workgroup per entry.
__global__ void __launch_bounds__(256) k_fill_gaps(const int4* __restrict__ gaps, int n, int* __restrict__ start) {
    for (int g = blockIdx.x; g < n; g += gridDim.x) {
        const int4 e = gaps[g];
        for (int c = e.x + (int)threadIdx.x; c <= e.y; c += 256) start[c] = e.z;
    }
}

// Full-width arrival slots of every particle in its cell (a cell with more
// particles than a byte counts).
__global__ void __launch_bounds__(256) k_count(const int* __restrict__ key, int64_t np, int* __restrict__ slot,
                                               int* __restrict__ count) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    slot[p] = atomicAdd(&count[key[p]], 1);
}

__global__ void __launch_bounds__(256) k_iota(int* __restrict__ a, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = (int)i;
}

__global__ void __launch_bounds__(256) k_identity(int64_t np, int* __restrict__ perm) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < np) perm[p] = (int)p;
}


// Cell key with the arithmetic of ppm_util_rank3d.f:414-475 (FLOOR, ghost
// cells, upper-boundary corrections).  SLOT: arrival slots by atomic counts,
// key -1 for particles in no box; otherwise (for the radix sort) those get the
// key past the last box.  stats[0] counts the particles in no box, stats[1]
// the corrections.
template <int DIM, typename PosT, bool SLOT>
__global__ void __launch_bounds__(256) k_rank_keys(const PosT* __restrict__ xp, int64_t np,
                                                   RankGeom g, int* __restrict__ key,
                                                   int* __restrict__ slot, int* __restrict__ count,
                                                   int* __restrict__ stats) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = p < np;
    PosT x[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) x[d] = live ? xp[p * DIM + d] : (PosT)g.xmin[d];
    int idx[3] = {0, 0, 0};
    int corr = 0;
    bool in = true;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        PosT mn = (PosT)g.xmin[d], mx = (PosT)g.xmax[d];
        PosT rd = (PosT)g.rdx[d];
        int i = (int)floor(scaled_coord<PosT>(x[d], mn, rd)) + g.ngl_lo[d];
        if (x[d] >= mx && i < g.nm[d] + g.ngl_lo[d]) { i = g.nm[d] + g.ngl_lo[d]; ++corr; }
        idx[d] = i;
    }
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        PosT mx = (PosT)g.xmax[d];
        if (x[d] < mx && idx[d] >= g.nm[d] + g.ngl_lo[d]) { idx[d] = g.nm[d] + g.ngl_lo[d] - 1; ++corr; }
        if (idx[d] < 0 || idx[d] >= g.ntot[d]) in = false;
    }
    if (live && corr) atomicAdd(&stats[1], corr);
    const uint64_t out = __ballot(live && !in);
    if (out != 0ull && (threadIdx.x & 63) == 0) atomicAdd(&stats[0], (int)__popcll(out));
    if (!live) return;
    const int k = idx[0] + g.ntot[0] * (idx[1] + g.ntot[1] * idx[2]);
    if constexpr (SLOT) {
        key[p] = in ? k : -1;
        if (in) slot[p] = atomicAdd(&count[k], 1);
    } else {
        key[p] = in ? k : g.ntot[0] * g.ntot[1] * g.ntot[2];
    }
}

// Four particles per thread: keys and slots as vector loads (plan buffers
// are 256-byte aligned), then the four head loads in flight together.  SlotT:
// uint8_t (byte-wide counting) or int (full width).
template <typename SlotT>
__global__ void __launch_bounds__(256) k_scatter(const int* __restrict__ key, const SlotT* __restrict__ slot,
                                                 const int* __restrict__ start, int64_t np,
                                                 int* __restrict__ perm) {
    const int64_t p0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (p0 >= np) return;
    int k[4], sl[4];
    if (p0 + 4 <= np) {
        const int4 kv = *reinterpret_cast<const int4*>(key + p0);
        k[0] = kv.x; k[1] = kv.y; k[2] = kv.z; k[3] = kv.w;
        if constexpr (sizeof(SlotT) == 1) {
            const uint32_t sv = *reinterpret_cast<const uint32_t*>(slot + p0);
#pragma unroll
            for (int i = 0; i < 4; ++i) sl[i] = (int)((sv >> (8 * i)) & 255u);
        } else {
            const int4 sv = *reinterpret_cast<const int4*>(slot + p0);
            sl[0] = sv.x; sl[1] = sv.y; sl[2] = sv.z; sl[3] = sv.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            k[i] = p0 + i < np ? key[p0 + i] : -1;
            sl[i] = p0 + i < np ? (int)slot[p0 + i] : 0;
        }
    }
    int h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = k[i] >= 0 ? start[k[i]] : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (k[i] >= 0) perm[h[i] + sl[i]] = (int)(p0 + i);
}

// Restore increasing particle index inside every cell (stability).
__global__ void __launch_bounds__(256) k_stabilize(const int* __restrict__ start, int64_t ncells,
                                                   int* __restrict__ perm) {
    int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncells) return;
    int b = start[c], e = start[c + 1];
    if (e - b < 2) return;
    for (int i = b + 1; i < e; ++i) {
        int v = perm[i];
        int j = i - 1;
        while (j >= b && perm[j] > v) {
            perm[j + 1] = perm[j];
            --j;
        }
        perm[j + 1] = v;
    }
}

// The same for the cells k_keys listed (those with two or more particles).
// A key workgroup lists a few hundred cells at most (about 280 of its 1024
// particles on an advected lattice), so one wavefront takes the lists of
// STAB_GROUP consecutive key workgroups, spread over its lanes.
constexpr int STAB_GROUP = 2;
__global__ void __launch_bounds__(64) k_stabilize_listed(const int* __restrict__ start,
                                                         const int* __restrict__ multi,
                                                         const int* __restrict__ multi_n, int64_t nlists,
                                                         int* __restrict__ perm) {
    const int64_t l0 = (int64_t)blockIdx.x * STAB_GROUP;
    int off[STAB_GROUP + 1];
    off[0] = 0;
#pragma unroll
    for (int j = 0; j < STAB_GROUP; ++j) off[j + 1] = off[j] + (l0 + j < nlists ? multi_n[l0 + j] : 0);
    for (int q = (int)threadIdx.x; q < off[STAB_GROUP]; q += 64) {
        int j = 0;
        while (q >= off[j + 1]) ++j;
        const int c = multi[(l0 + j) * KEYS_BLOCK + (q - off[j])];
        const int b = start[c], e = start[c + 1];
        for (int i = b + 1; i < e; ++i) {
            const int v = perm[i];
            int k = i - 1;
            while (k >= b && perm[k] > v) {
                perm[k + 1] = perm[k];
                --k;
            }
            perm[k + 1] = v;
        }
    }
}

// The same for the listed cells of a slot table: the (at most TABLE_SLOTS)
// entries of a cell are sorted in registers, and written back where they were
// not in order (the partial lines of a cell's slots are the kernel's time:
// binning of 512^3 advected particles 1.45 -> 1.39 ms, 8192^2 624 -> 603 us).
__global__ void __launch_bounds__(64) k_stabilize_table(const uint32_t* __restrict__ count,
                                                        const int* __restrict__ multi,
                                                        const int* __restrict__ multi_n, int64_t nlists,
                                                        int64_t ncells, int* __restrict__ table) {
    const int64_t l0 = (int64_t)blockIdx.x * STAB_GROUP;
    int off[STAB_GROUP + 1];
    off[0] = 0;
#pragma unroll
    for (int j = 0; j < STAB_GROUP; ++j) off[j + 1] = off[j] + (l0 + j < nlists ? multi_n[l0 + j] : 0);
    for (int q = (int)threadIdx.x; q < off[STAB_GROUP]; q += 64) {
        int j = 0;
        while (q >= off[j + 1]) ++j;
        const int c = multi[(l0 + j) * KEYS_BLOCK + (q - off[j])];
        const int n = (int)((count[count_word(c)] >> count_shift(c)) & 255u);
        int v[TABLE_SLOTS];
#pragma unroll
        for (int r = 0; r < TABLE_SLOTS; ++r) v[r] = r < n ? table[(int64_t)r * ncells + c] : INT_MAX;
        bool in_order = true;
#pragma unroll
        for (int r = 0; r + 1 < TABLE_SLOTS; ++r) in_order = in_order && v[r] <= v[r + 1];
        if (in_order) continue;
        // odd-even transposition sort (the padding INT_MAX stays at the end)
#pragma unroll
        for (int pass = 0; pass < TABLE_SLOTS; ++pass)
#pragma unroll
            for (int r = pass & 1; r + 1 < TABLE_SLOTS; r += 2) {
                const int a = min(v[r], v[r + 1]), b = max(v[r], v[r + 1]);
                v[r] = a;
                v[r + 1] = b;
            }
#pragma unroll
        for (int r = 0; r < TABLE_SLOTS; ++r)
            if (r < n) table[(int64_t)r * ncells + c] = v[r];
    }
}

// Permutation of a slot-table binning from its heads: the particles of cell c
// go to perm[start[c] ..].
__global__ void __launch_bounds__(256) k_table_perm(const uint32_t* __restrict__ count, const int* __restrict__ start,
                                                    const int* __restrict__ table, int64_t ncells,
                                                    int* __restrict__ perm) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncells) return;
    const int n = (int)((count[count_word(c)] >> count_shift(c)) & 255u);
    const int b = start[c];
    for (int r = 0; r < n; ++r) perm[b + r] = table[(int64_t)r * ncells + c];
}

__global__ void k_to_one_based(int* __restrict__ a, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] += 1;
}

// Two ranges (the second may be empty) in one launch.
__global__ void k_fill_zero(uint32_t* __restrict__ p, int64_t n, uint32_t* __restrict__ p2, int64_t n2) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n + n2; i += stride) (i < n ? p[i] : p2[i - n]) = 0u;
}


// Zero fill with a kernel (graph-capture safe, unlike hipMemsetAsync).
static int fill_zero2(void* p, size_t bytes, void* p2, size_t bytes2, hipStream_t s) {
    const int64_t n = (int64_t)(bytes / 4), n2 = (int64_t)(bytes2 / 4);
    if (n + n2 <= 0) return 0;
    int64_t g = (n + n2 + 255) / 256;
    if (g > 65536) g = 65536;
    hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)g), dim3(256), 0, s, (uint32_t*)p, n, (uint32_t*)p2, n2);
    PPMG_HIP(hipGetLastError());
    return 0;
}
int fill_zero(void* p, size_t bytes, hipStream_t s) { return fill_zero2(p, bytes, nullptr, 0, s); }

// Keys of a binning that took the cell-order path (which writes none).
template <int DIM, typename PosT>
__global__ void __launch_bounds__(256) k_keys_only(const PosT* __restrict__ xp, int64_t np, DevMesh m,
                                                   int* __restrict__ key) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    PosT xv[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) xv[d] = xp[p * DIM + d];
    key[p] = cell_key<DIM, PosT>(xv, m);
}

// ------------------------------------------------------ crowded input ---
// Cells of tens of particles in no particular order (clustered particles):
// k_keys' atomic slots contend on the crowded cells' count words, the scatter
// writes at random and the per-cell insertion sorts grow with the square of
// the occupancy.  Such input is binned by a stable LSD radix sort of the
// (cell key, particle) pairs instead: no atomics on
// crowded words, writes in runs, and a stable sort of the keys in particle
// order is the reference's permutation as it stands (ppm_util_rank3d.f:
// 505-532).  The heads follow from the runs of the sorted keys.  Large input
// in no order takes the same path, and so does util_rank.
//
// A pass sorts by 8 or 9 bits, whichever takes fewer passes over the key's
// bits (27 bits at 512^3: three passes of 9), with one thread per digit.
// RS_ITEMS pairs a thread: longer runs per digit to write and fewer tiles'
// counts to scan, until a tile's LDS leaves too few workgroups (2^24 keys in
// no order 471, 440, 460 us at 8, 16 and 24; clustered 2^26 2.03, 1.97, 1.94
// and 2.45 ms at 8, 12, 16 and 24 with 9 bits).
constexpr int RS_ITEMS = 16;
template <int BITS> struct Radix {
    static constexpr int BUCKETS = 1 << BITS;
    static constexpr int THREADS = BUCKETS;                // one digit per thread in the tile loops
    static constexpr int TILE = THREADS * RS_ITEMS;        // pairs per workgroup
    static constexpr int NWAVE = THREADS / 64;
};

// Keys of all particles (key[p]), the particles in no cell (err[0]) and the
// descent flag (err[1]), as k_keys reports them.
template <int DIM, typename PosT>
__global__ void __launch_bounds__(256) k_keys_plain(const PosT* __restrict__ xp, int64_t np, DevMesh m,
                                                    int* __restrict__ key, int* __restrict__ err) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool live = p < np;
    const int64_t p0 = (int64_t)blockIdx.x * blockDim.x + __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u);
    const bool has_seam = p0 > 0 && p0 <= np;
    PosT xv[DIM], sv[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        xv[d] = live ? xp[p * DIM + d] : PosT(0);
        sv[d] = has_seam ? xp[(p0 - 1) * DIM + d] : PosT(0);
    }
    const int seam = has_seam ? cell_key<DIM, PosT>(sv, m) : -1;
    const int k = live ? cell_key<DIM, PosT>(xv, m) : -1;
    int left = __shfl_up(k, 1);
    if (lane == 0) left = seam;
    const uint64_t bb = __ballot(live && k < 0), bd = __ballot(live && p > 0 && k < left);
    const int nfar = (int)__popcll(__ballot(live && p > 0 && abs(k - left) > FAR_CELLS));
    if (live) key[p] = k;
    if (lane == 0) {
        if (bb) atomicAdd(&err[0], (int)__popcll(bb));
        if (bd && *(volatile int*)&err[1] == 0) err[1] = 1;
        if (nfar && (blockIdx.x & 63) == 0) atomicAdd(&err[72 + ((blockIdx.x >> 6) & 63)], nfar);
    }
}

// Lanes of the wavefront holding the same digit as this lane (among `live`).
template <int BITS>
__device__ __forceinline__ uint64_t digit_peers(int d, bool live) {
    uint64_t peers = __ballot(live);
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
        const uint64_t on = __ballot((d >> b) & 1);
        peers &= ((d >> b) & 1) ? on : ~on;
    }
    return peers;
}

// Digit counts of every tile, digit-major: hist[d * ntiles + tile].  Tiles
// are numbered XCD-contiguously (xcd_tile), as in k_rs_scatter: the tiles
// one XCD sorts are neighbours, and so are their runs of each digit.  2^24
// keys: 17 us, 40 with the digit's lanes searched for every key.
template <int BITS>
__global__ void __launch_bounds__(Radix<BITS>::THREADS) k_rs_hist(const int* __restrict__ keys, int64_t n, int shift,
                                                                  int* __restrict__ hist, int64_t ntiles) {
    using R = Radix<BITS>;
    __shared__ int h[R::BUCKETS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t tile = xcd_tile(blockIdx.x, (int64_t)gridDim.x);
    h[tid] = 0;
    __syncthreads();
    const int64_t t0 = tile * R::TILE;
    int k[RS_ITEMS];   // all loads in flight before the first count
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
        const int64_t i = t0 + j * R::THREADS + tid;
        k[j] = i < n ? keys[i] : 0;
    }
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
        const bool live = t0 + j * R::THREADS + tid < n;
        const int d = (k[j] >> shift) & (R::BUCKETS - 1);
        // one LDS add per lane, or, where many lanes hold the first lane's
        // digit, one for all of those
        const uint64_t same = __ballot(live && d == __builtin_amdgcn_readfirstlane(d));
        if (__popcll(same) > 8) {
            if (lane == 0) atomicAdd(&h[d], (int)__popcll(same));
            if (live && !((same >> lane) & 1)) atomicAdd(&h[d], 1);
        } else if (live) {
            atomicAdd(&h[d], 1);
        }
    }
    __syncthreads();
    hist[(int64_t)tid * ntiles + tile] = h[tid];
}

// One stable pass.  The pairs of a tile are first ordered by digit in LDS.  A
// wavefront takes a run of 64 ITEMS pairs, 64 at a time in index order, and
// counts its digits as it goes: a pair's place is its digit's start in the
// tile, plus that digit's pairs in the wavefronts before, plus its rank among
// this wavefront's (the count so far and the lanes below with the same digit).
// The tile then writes its digit runs at their offsets (offs: the exclusive
// scan of the tiles' counts), consecutive threads to consecutive addresses,
// the keys first and the values through the same LDS.  Bound by memory with
// runs of half a line: 2^24 pairs of 8 bits 73 us (268 MB), 116 with the
// wavefronts in step, a barrier per 64 pairs.  vin nullptr: the values
// are the pairs' indices (the first pass); vadd is added to the values written
// (1: one-based ranks).  vmax: values at positions from vmax on are not written.
template <int BITS>
__global__ void __launch_bounds__(Radix<BITS>::THREADS)
k_rs_scatter(const int* __restrict__ kin, const int* __restrict__ vin, int64_t n, int shift,
             const int* __restrict__ offs, int64_t ntiles, int* __restrict__ kout, int* __restrict__ vout, int vadd,
             int64_t vmax) {
    using R = Radix<BITS>;
    __shared__ int shift_out[R::BUCKETS];   // global position minus place, per digit
    __shared__ int wcnt[R::NWAVE][R::BUCKETS];
    __shared__ int sk[R::TILE];
    __shared__ int64_t sh[R::NWAVE + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t tile = xcd_tile(blockIdx.x, (int64_t)gridDim.x);
    const int64_t t0 = tile * R::TILE;
    const int tn = (int)min((int64_t)R::TILE, n - t0);
    const int w0 = wave * (64 * RS_ITEMS);
    int kk[RS_ITEMS], vv[RS_ITEMS];   // all loads in flight before the first round
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
        const int q = w0 + j * 64 + lane;
        kk[j] = q < tn ? kin[t0 + q] : 0;
        vv[j] = q < tn ? (vin ? vin[t0 + q] : (int)(t0 + q)) : 0;
    }
#pragma unroll
    for (int w = 0; w < R::NWAVE; ++w) wcnt[w][tid] = 0;
    const uint64_t lt = lane ? ~0ull >> (64 - lane) : 0ull;   // lanes below this one
    __syncthreads();
    int rank[RS_ITEMS];
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
        const bool live = w0 + j * 64 + lane < tn;
        const int d = (kk[j] >> shift) & (R::BUCKETS - 1);
        const uint64_t peers = digit_peers<BITS>(d, live);
        const int before = wcnt[wave][d];
        rank[j] = before + (int)__popcll(peers & lt);
        wave_lds_sync();
        if (live && (peers & lt) == 0ull) wcnt[wave][d] = before + (int)__popcll(peers);
        wave_lds_sync();
    }
    __syncthreads();
    // thread t = digit t: its start in the tile, and each wavefront's in it
    int total = 0;
#pragma unroll
    for (int w = 0; w < R::NWAVE; ++w) total += wcnt[w][tid];
    int64_t lb;
    block_exclusive_scan<R::THREADS>((int64_t)total, sh, lb);
    shift_out[tid] = offs[(int64_t)tid * ntiles + tile] - (int)lb;
    int run = (int)lb;
#pragma unroll
    for (int w = 0; w < R::NWAVE; ++w) {
        const int c = wcnt[w][tid];
        wcnt[w][tid] = run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
        rank[j] += wcnt[wave][(kk[j] >> shift) & (R::BUCKETS - 1)];
        if (w0 + j * 64 + lane < tn) sk[rank[j]] = kk[j];
    }
    __syncthreads();
    int o[RS_ITEMS];
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
        const int q = j * R::THREADS + tid;
        if (q < tn) {
            const int k = sk[q];
            o[j] = shift_out[(k >> shift) & (R::BUCKETS - 1)] + q;
            kout[o[j]] = k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j)
        if (w0 + j * 64 + lane < tn) sk[rank[j]] = vv[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RS_ITEMS; ++j) {
        const int q = j * R::THREADS + tid;
        if (q < tn && o[j] < vmax) vout[o[j]] = sk[q] + vadd;
    }
}

// Heads from sorted keys: start[c] + add = first position whose key is c or
// more, for c = 0 .. ncells - 1, and start[ncells] = n + add.  A workgroup
// takes HEADS_CELLS cells: its wavefronts find the cells' range of the keys
// by a 64-way search, the first key of each run notes its position in LDS, and
// empty cells take the position of the next run.  Bound by memory: the keys
// are read and the heads written once (2^26 crowded keys in 2^27 cells: 0.38
// ms; the runs' lengths by atomics into zeroed counts and a scan of them took
// 0.85 ms).  One
// workgroup in `stride` counts its cells of nine particles or more into
// err[8 .. 71] (err NULL: none does).
constexpr int HEADS_CELLS = 4096;
constexpr int HEADS_PER = HEADS_CELLS / 256;
__global__ void __launch_bounds__(256) k_heads(const int* __restrict__ ks, int64_t n, int64_t ncells,
                                               int* __restrict__ start, int add, int stride, int* __restrict__ err) {
    __shared__ int pos[HEADS_CELLS];
    __shared__ int64_t range[2];
    __shared__ int wmin[4], ncrowd;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t c0 = (int64_t)blockIdx.x * HEADS_CELLS;
    const int nc = (int)min((int64_t)HEADS_CELLS, ncells - c0);
    for (int i = tid; i < HEADS_CELLS; i += 256) pos[i] = INT_MAX;
    if (tid == 0) ncrowd = 0;
    if (wave < 2) {
        // first position whose key is not below `want`, in [lo, hi]
        const int64_t want = wave == 0 ? c0 : c0 + nc;
        int64_t lo = 0, hi = n;
        while (lo < hi) {
            // probes lo + (l + 1) step - 1, l = 0 .. 63, past hi taken as found
            const int64_t step = (hi - lo + 63) / 64, at = lo + (lane + 1) * step - 1;
            const bool below = at < hi && (int64_t)ks[at] < want;
            const int m = (int)__popcll(__ballot(below));   // probes below: a prefix of the lanes
            const int64_t nlo = lo + m * step, nhi = lo + (int64_t)(m + 1) * step - 1;
            lo = nlo;
            hi = nhi < hi ? nhi : hi;
        }
        if (lane == 0) range[wave] = lo;
    }
    __syncthreads();
    const int64_t r0 = range[0], r1 = range[1];
    for (int64_t i0 = r0; i0 < r1; i0 += 4 * 256) {
        int k[4], left[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t i = i0 + j * 256 + tid;
            k[j] = i < r1 ? ks[i] : -1;
            left[j] = i < r1 && i > r0 ? ks[i - 1] : -1;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (k[j] >= 0 && k[j] != left[j]) pos[k[j] - (int)c0] = (int)(i0 + j * 256 + tid);
    }
    __syncthreads();
    // suffix minimum: a thread's HEADS_PER cells, then the threads after it
    int v[HEADS_PER];
    int run = INT_MAX;
#pragma unroll
    for (int i = HEADS_PER - 1; i >= 0; --i) {
        run = min(run, pos[tid * HEADS_PER + i]);
        v[i] = run;
    }
    int after = run;   // minimum over lanes >= this one
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_down(after, o, 64);
        if (lane + o < 64) after = min(after, y);
    }
    if (lane == 0) wmin[wave] = after;
    int next = __shfl_down(after, 1, 64);
    if (lane == 63) next = INT_MAX;
    __syncthreads();
    for (int w = wave + 1; w < 4; ++w) next = min(next, wmin[w]);
    next = min(next, (int)r1);
#pragma unroll
    for (int i = 0; i < HEADS_PER; ++i) v[i] = min(v[i], next);
    const bool sampled = err && blockIdx.x % stride == 0;
    int crowd = 0;
#pragma unroll
    for (int i = 0; i < HEADS_PER; ++i) crowd += (i + 1 < HEADS_PER ? v[i + 1] : next) - v[i] >= 9;
    if (sampled && crowd) atomicAdd(&ncrowd, crowd);
    int* out = start + c0 + tid * HEADS_PER;
    if (nc == HEADS_CELLS && (reinterpret_cast<uintptr_t>(start) & 15) == 0) {
        int4* q = reinterpret_cast<int4*>(out);
#pragma unroll
        for (int i = 0; i < HEADS_PER / 4; ++i)
            q[i] = make_int4(v[4 * i] + add, v[4 * i + 1] + add, v[4 * i + 2] + add, v[4 * i + 3] + add);
    } else {
#pragma unroll
        for (int i = 0; i < HEADS_PER; ++i)
            if (tid * HEADS_PER + i < nc) out[i] = v[i] + add;
    }
    if (c0 + nc == ncells && tid == 0) start[ncells] = (int)r1 + add;
    __syncthreads();
    if (sampled && tid == 0 && ncrowd > 0) atomicAdd(&err[8 + (blockIdx.x / stride & 63)], ncrowd);
}

// Digit width of a sort of keys below nkeys (and its passes).
static int radix_bits(int64_t nkeys, int* passes) {
    int bits = 1;
    while (bits < 31 && ((int64_t)1 << bits) < nkeys) ++bits;
    const int p8 = (bits + 7) / 8, p9 = (bits + 8) / 9;
    *passes = p9 < p8 ? p9 : p8;
    return p9 < p8 ? 9 : 8;
}

// Scratch of a sort of n keys below nkeys: the pairs twice (16 bytes a key) and
// the tiles' counts.  False, with nothing kept, where it is refused (the
// counting path does without).
static bool radix_scratch(ppmg_plan* plan, int64_t n, int64_t nkeys) {
    int passes;
    const int64_t buckets = (int64_t)1 << radix_bits(nkeys, &passes), tile = buckets * RS_ITEMS;
    const size_t pairs = sizeof(int) * (size_t)n, hist = sizeof(int) * (size_t)(2 * (buckets * ((n + tile - 1) / tile) + 4));
    DevBuf* bufs[] = {&plan->rkey[0], &plan->rkey[1], &plan->rval[0], &plan->rval[1], &plan->rhist};
    for (DevBuf* b : bufs)
        if (!b->try_ensure(b == &plan->rhist ? hist : pairs)) {
            for (DevBuf* r : bufs) r->release();
            return false;
        }
    return true;
}

// Stable sort of n keys below 2^bits by LSD radix passes, in the scratch of
// radix_scratch: the sorted keys (*sorted_keys, in that scratch), and the
// permutation (plus vadd) at positions below vmax in vout.
template <int BITS>
static int radix_sort_bits(ppmg_plan* plan, const int* keys, int64_t n, int passes, int* vout, int vadd, int64_t vmax,
                           hipStream_t s, const int** sorted_keys) {
    using R = Radix<BITS>;
    const int64_t ntiles = (n + R::TILE - 1) / R::TILE;
    int* hist = plan->rhist.as<int>();
    int* offs = hist + R::BUCKETS * ntiles + 4;   // 16-byte aligned, n + 1 entries
    const int* kin = keys;
    const int* vin = nullptr;
    for (int pass = 0; pass < passes; ++pass) {
        const int shift = pass * BITS;
        const bool last = pass == passes - 1;
        int* kout = plan->rkey[pass & 1].as<int>();
        int* vo = last ? vout : plan->rval[pass & 1].as<int>();
        hipLaunchKernelGGL(k_rs_hist<BITS>, dim3((unsigned)ntiles), dim3(R::THREADS), 0, s, kin, n, shift, hist, ntiles);
        if (exclusive_scan(hist, R::BUCKETS * ntiles, offs, plan->scan_tmp, n, s)) return PPMG_ERROR_FATAL;
        hipLaunchKernelGGL(k_rs_scatter<BITS>, dim3((unsigned)ntiles), dim3(R::THREADS), 0, s, kin, vin, n, shift, offs,
                           ntiles, kout, vo, last ? vadd : 0, last ? vmax : n);
        kin = kout;
        vin = vo;
    }
    *sorted_keys = kin;
    PPMG_HIP(hipGetLastError());
    return 0;
}

static int radix_sort(ppmg_plan* plan, const int* keys, int64_t n, int64_t nkeys, int* vout, int vadd, int64_t vmax,
                      hipStream_t s, const int** sorted_keys) {
    int passes;
    if (radix_bits(nkeys, &passes) == 9)
        return radix_sort_bits<9>(plan, keys, n, passes, vout, vadd, vmax, s, sorted_keys);
    return radix_sort_bits<8>(plan, keys, n, passes, vout, vadd, vmax, s, sorted_keys);
}

// Heads of the sorted keys ks, and the plan's crowded-cell estimate from a
// sample of them.
static int heads_from_sorted(ppmg_plan* plan, const int* ks, int64_t np, int64_t ncells, hipStream_t s) {
    int* err = plan->err.as<int>();
    const unsigned g = nblk(ncells, HEADS_CELLS);
    const int stride = g > 2048 ? (int)(g / 2048) : 1;
    hipLaunchKernelGGL(k_heads, dim3(g), dim3(256), 0, s, ks, np, ncells, plan->start.as<int>(), 0, stride, err);
    PPMG_HIP(hipGetLastError());
    int sample[128];
    if (read_back(plan, err + 8, 128, sample, s)) return PPMG_ERROR_FATAL;
    int64_t crowd = 0, far = 0;
    for (int i = 0; i < 64; ++i) {
        crowd += sample[i];
        far += sample[64 + i];
    }
    plan->crowded_cells = stride * crowd;
    plan->far_particles = 64 * far;
    return 0;
}

// The binning of crowded input: keys pass, then (input not in cell order)
// the radix sort, and the heads; the plan's crowded-cell estimate is taken
// again from the sorted runs.
static int bin_crowded(ppmg_plan* plan, const DevMesh& m, int prec, int64_t np, const void* xp, hipStream_t s,
                       int64_t* nbad) {
    const int64_t ncells = plan->ncells;
    int* key = plan->key.as<int>();
    int* err = plan->err.as<int>();
    const unsigned g = nblk(np, 256);
    if (m.dim == 3) {
        if (prec == PPMG_PREC_F32) hipLaunchKernelGGL((k_keys_plain<3, float>), dim3(g), dim3(256), 0, s, (const float*)xp, np, m, key, err);
        else hipLaunchKernelGGL((k_keys_plain<3, double>), dim3(g), dim3(256), 0, s, (const double*)xp, np, m, key, err);
    } else {
        if (prec == PPMG_PREC_F32) hipLaunchKernelGGL((k_keys_plain<2, float>), dim3(g), dim3(256), 0, s, (const float*)xp, np, m, key, err);
        else hipLaunchKernelGGL((k_keys_plain<2, double>), dim3(g), dim3(256), 0, s, (const double*)xp, np, m, key, err);
    }
    PPMG_HIP(hipGetLastError());
    int herr[2] = {0, 0};
    if (read_back(plan, err, 2, herr, s)) return PPMG_ERROR_FATAL;
    *nbad = herr[0];
    if (herr[0]) return 0;
    // input already in cell order: the keys are the sorted keys, the
    // permutation the identity (written on demand)
    const bool sorted = herr[1] == 0;
    const int* ks = key;
    if (!sorted && radix_sort(plan, key, np, ncells, plan->perm.as<int>(), 0, np, s, &ks)) return PPMG_ERROR_FATAL;
    if (heads_from_sorted(plan, ks, np, ncells, s)) return PPMG_ERROR_FATAL;
    plan->perm_identity = sorted;
    plan->perm_written = !sorted;
    plan->keys_written = true;
    plan->sorted_input = sorted;
    return 0;
}

int bin_particles(ppmg_plan* plan, const DevMesh& m, int prec, int64_t np, const void* xp,
                  hipStream_t s, int64_t* nbad, bool table, bool lattice) {
    const int64_t ncells = (int64_t)m.nbin[0] * m.nbin[1] * m.nbin[2];
    const int64_t gapcap = np / 16 + 4096;
    const size_t npb = (size_t)(np > 0 ? np : 1);
    // byte-wide counts (count_word) come in whole blocks of 256 cells, and
    // the scan reads whole tiles of SCAN_TILE cells
    const size_t count_alloc = ((size_t)ncells + SCAN_TILE - 1) / SCAN_TILE * SCAN_TILE;
    if (plan->err.bytes < sizeof(int) * ERR_WORDS) plan->lattice_flag_clear = false;   // about to be allocated
    if (plan->err.ensure(sizeof(int) * ERR_WORDS)) return PPMG_ERROR_FATAL;
    // Keys, permutation and heads are allocated where they are used: a slot
    // table or a checked lattice goes without (14 bytes per particle and 4 per
    // cell; materialize_heads and the like allocate them should they be asked
    // for after all).
    auto sorted_lists = [&]() {
        return plan->key.ensure(sizeof(int) * npb) || plan->slot.ensure(npb + 16) ||
               plan->perm.ensure(sizeof(int) * npb) || plan->start.ensure(sizeof(int) * (size_t)(ncells + 1)) ||
               plan->gaps.ensure(sizeof(int4) * (size_t)gapcap);
    };
    plan->bin_stream = s;
    plan->prebinned = false;   // a binning left by ppmg_m2p_prebin is overwritten
    plan->bin_table = false;
    plan->bin_lattice = false;
    plan->lattice_checked = false;
    plan->np = np;
    plan->ncells = ncells;
    plan->bin_xp = xp;
    plan->bin_prec = prec;
    plan->bin_mesh = m;
    plan->keys_written = true;
    *nbad = 0;
    if (np == 0) {
        plan->perm_identity = true;
        plan->perm_written = true;
        if (sorted_lists()) return PPMG_ERROR_FATAL;
        return fill_zero(plan->start.p, sizeof(int) * (size_t)(ncells + 1), s);
    }
    // A lattice in cell order (particle p in cell p, np == ncells), as the last
    // binning of this plan found on the same mesh: for a reader that checks
    // every particle's cell itself (`lattice`), no pass at all; the reader
    // reports a particle outside its cell in err[6] and bins again.
    // A plan whose lattice check failed takes its next 16 inputs without it.
    if (lattice && plan->lattice_skip > 0) {
        --plan->lattice_skip;
        lattice = false;
    }
    if (lattice && plan->lattice_pred && np == ncells && plan->lattice_prec == prec &&
        same_mesh(plan->lattice_mesh, m)) {
        if (!plan->lattice_flag_clear && fill_zero(plan->err.p, sizeof(int) * ERR_WORDS, s)) return PPMG_ERROR_FATAL;
        plan->lattice_flag_clear = true;
        plan->bin_lattice = true;
        plan->perm_identity = true;
        plan->perm_written = false;
        plan->keys_written = false;
        return 0;
    }
    plan->lattice_pred = false;
    // The plan remembers whether its last input was in cell order; a plan fed
    // the same kind of particles each call (advected particles, or particles
    // fresh from create_part) predicts right and does each step once.
    const bool predict_sorted = plan->sorted_input;
    // Unsorted input for a reader of the slot table: the key pass fills the
    // table, and no keys, scan or scatter follow.  A plan whose table
    // overflowed, or was refused its memory, bins its next 16 inputs without
    // one.  Allocation-free calls
    // take the heads (the table needs 32 bytes per cell), and so does every
    // call under PPMG_NO_TABLE=1 (used to cross-check the two layouts).
    const char* no_table = std::getenv("PPMG_NO_TABLE");
    if (no_table && no_table[0] && no_table[0] != '0') table = false;
    bool use_table = table && !predict_sorted && plan->table_skip == 0 && !arena_bound();
    if (table && !predict_sorted && plan->table_skip > 0) --plan->table_skip;
    // Crowded input (the last binning's sample found a cell of nine or more
    // particles per 64 particles), and large input in no order, is binned by the
    // radix sort (16.8M particles of 256^3 cells in random order: 0.49 against
    // 1.04 ms; 2.1M 129 against 173 us, 1.03M 109 against 96); PPMG_RADIX=1
    // forces that path for input not predicted in cell order, PPMG_RADIX=0
    // rules it out (both for tests).  Allocation-free calls keep the counting
    // path (the sort needs four more int32 per particle), and so do calls
    // whose sort is refused its scratch.
    const char* rx = std::getenv("PPMG_RADIX");
    const bool radix = rx && rx[0] ? rx[0] == '1'
                                   : plan->crowded_cells * 64 > np ||
                                         (np >= FAR_MIN_NP && plan->far_particles * 4 > np);
    if (!predict_sorted && radix && !arena_bound() && radix_scratch(plan, np, ncells)) {
        if (sorted_lists()) return PPMG_ERROR_FATAL;
        if (fill_zero(plan->err.p, sizeof(int) * ERR_WORDS, s)) return PPMG_ERROR_FATAL;
        plan->lattice_flag_clear = true;
        return bin_crowded(plan, m, prec, np, xp, s, nbad);
    }
    if (use_table && !plan->table.try_ensure(sizeof(int) * TABLE_SLOTS * (size_t)ncells)) {
        use_table = false;
        plan->table_skip = 16;
    }
    if (!use_table && sorted_lists()) return PPMG_ERROR_FATAL;
    if (plan->count.ensure(count_alloc) ||
        plan->multi.ensure(sizeof(int) * (size_t)nblk(np, KEYS_BLOCK) * KEYS_BLOCK) ||
        plan->multi_n.ensure(sizeof(int) * (size_t)nblk(np, KEYS_BLOCK)))
        return PPMG_ERROR_FATAL;
    int* tab = use_table ? plan->table.as<int>() : nullptr;
    if (fill_zero2(plan->err.p, sizeof(int) * ERR_WORDS, plan->count.p, predict_sorted ? 0 : count_alloc, s))
        return PPMG_ERROR_FATAL;
    plan->lattice_flag_clear = true;
    int* key = plan->key.as<int>();
    uint8_t* slot8 = plan->slot.as<uint8_t>();
    uint32_t* count8 = plan->count.as<uint32_t>();
    int* start = plan->start.as<int>();
    int* err = plan->err.as<int>();
    int4* gaps = plan->gaps.as<int4>();
    int* multi = plan->multi.as<int>();
    int* multi_n = plan->multi_n.as<int>();
    {
        const unsigned g = nblk(np, KEYS_BLOCK);
#define KEYS(D, T, S, TB) hipLaunchKernelGGL((k_keys<D, T, S, TB>), dim3(g), dim3(256), 0, s, (const T*)xp, np, m, \
                                             ncells, key, slot8, count8, start, err, gaps, (int)gapcap, multi, multi_n, tab)
#define KEYS_T(D, T)                                   \
    do {                                               \
        if (predict_sorted) KEYS(D, T, false, false);  \
        else if (use_table) KEYS(D, T, true, true);    \
        else KEYS(D, T, true, false);                  \
    } while (0)
        const bool single = prec == PPMG_PREC_F32;
        if (m.dim == 3) {
            if (single) KEYS_T(3, float);
            else KEYS_T(3, double);
        } else {
            if (single) KEYS_T(2, float);
            else KEYS_T(2, double);
        }
#undef KEYS_T
#undef KEYS
        PPMG_HIP(hipGetLastError());
    }
    int herr[ERR_WORDS] = {};
    if (read_back(plan, err, ERR_WORDS, herr, s)) return PPMG_ERROR_FATAL;
    *nbad = herr[0];
    int64_t crowd = 0, far = 0;
    for (int i = 8; i < 72; ++i) {
        crowd += herr[i];
        far += herr[64 + i];
    }
    plan->crowded_cells = 64 * crowd;   // estimates from the 1-in-64 samples
    plan->far_particles = 64 * far;
    if (herr[0]) {
        plan->keys_written = false;   // (made on demand)
        return 0;
    }
    plan->lattice_pred = herr[5] == 0 && np == ncells;
    plan->lattice_prec = prec;
    plan->lattice_mesh = m;
    const bool sorted = herr[1] == 0;
    if (predict_sorted) {
        if (sorted && herr[2] <= gapcap) {
            // the heads are written but for the queued runs of empty cells
            if (herr[2] > 0)
                hipLaunchKernelGGL(k_fill_gaps, dim3((unsigned)(herr[2] < 4096 ? herr[2] : 4096)), dim3(256), 0, s,
                                   gaps, herr[2], start);
            PPMG_HIP(hipGetLastError());
            // input in cell order: identity permutation and keys, both written only on demand
            plan->perm_identity = true;
            plan->perm_written = false;
            plan->keys_written = false;
            return 0;
        }
        // wrong prediction (or more long gaps than the queue holds): bin
        // again on the counting path
        plan->sorted_input = false;
        return bin_particles(plan, m, prec, np, xp, s, nbad, table, false);
    }
    if (use_table) {
        if (herr[4]) {
            // a cell holds more than TABLE_SLOTS particles: bin again with
            // keys and slots
            plan->table_skip = 16;
            return bin_particles(plan, m, prec, np, xp, s, nbad, false, false);
        }
        // the listed cells (two or more particles) in increasing particle index
        hipLaunchKernelGGL(k_stabilize_table, dim3(nblk(nblk(np, KEYS_BLOCK), STAB_GROUP)), dim3(64), 0, s, count8,
                           multi, multi_n, (int64_t)nblk(np, KEYS_BLOCK), ncells, tab);
        PPMG_HIP(hipGetLastError());
        plan->bin_table = true;
        plan->perm_identity = false;
        plan->perm_written = false;
        plan->keys_written = false;
        plan->sorted_input = herr[1] == 0;
        return 0;
    }
    if (!herr[3]) {
        if (exclusive_scan_u8(count8, ncells, start, plan->scan_tmp, np, s)) return PPMG_ERROR_FATAL;
        if (!sorted)
            hipLaunchKernelGGL(k_scatter<uint8_t>, dim3(nblk(np, 1024)), dim3(256), 0, s, key, slot8, start, np,
                               plan->perm.as<int>());
    } else {
        // a cell holds more particles than a byte counts: count again at full width
        if (plan->slot.ensure(sizeof(int) * npb) || plan->count.ensure(sizeof(int) * (size_t)ncells))
            return PPMG_ERROR_FATAL;
        int* slot32 = plan->slot.as<int>();
        int* count32 = plan->count.as<int>();
        if (fill_zero(count32, sizeof(int) * (size_t)ncells, s)) return PPMG_ERROR_FATAL;
        hipLaunchKernelGGL(k_count, dim3(nblk(np, 256)), dim3(256), 0, s, key, np, slot32, count32);
        if (exclusive_scan(count32, ncells, start, plan->scan_tmp, np, s)) return PPMG_ERROR_FATAL;
        if (!sorted)
            hipLaunchKernelGGL(k_scatter<int>, dim3(nblk(np, 1024)), dim3(256), 0, s, key, slot32, start, np,
                               plan->perm.as<int>());
    }
    if (!sorted) {
        // the key pass listed the cells whose second particle it saw; after a
        // byte overflow that list may miss cells, so every cell is sorted
        if (herr[3])
            hipLaunchKernelGGL(k_stabilize, dim3(nblk(ncells, 256)), dim3(256), 0, s, start, ncells,
                               plan->perm.as<int>());
        else
            hipLaunchKernelGGL(k_stabilize_listed, dim3(nblk(nblk(np, KEYS_BLOCK), STAB_GROUP)), dim3(64), 0, s,
                               start, multi, multi_n, (int64_t)nblk(np, KEYS_BLOCK), plan->perm.as<int>());
    }
    PPMG_HIP(hipGetLastError());
    // input in cell order: the permutation is the identity, written only on demand
    plan->perm_identity = sorted;
    plan->perm_written = !sorted;
    plan->sorted_input = sorted;
    return 0;
}

int materialize_keys(ppmg_plan* plan, hipStream_t s) {
    if (!plan->keys_written && plan->np > 0) {
        if (plan->key.ensure(sizeof(int) * (size_t)plan->np)) return PPMG_ERROR_FATAL;
        const unsigned g = nblk(plan->np, 256);
        const DevMesh& m = plan->bin_mesh;
        int* key = plan->key.as<int>();
        if (plan->bin_prec == PPMG_PREC_F32) {
            if (m.dim == 3) hipLaunchKernelGGL((k_keys_only<3, float>), dim3(g), dim3(256), 0, s, (const float*)plan->bin_xp, plan->np, m, key);
            else hipLaunchKernelGGL((k_keys_only<2, float>), dim3(g), dim3(256), 0, s, (const float*)plan->bin_xp, plan->np, m, key);
        } else {
            if (m.dim == 3) hipLaunchKernelGGL((k_keys_only<3, double>), dim3(g), dim3(256), 0, s, (const double*)plan->bin_xp, plan->np, m, key);
            else hipLaunchKernelGGL((k_keys_only<2, double>), dim3(g), dim3(256), 0, s, (const double*)plan->bin_xp, plan->np, m, key);
        }
        PPMG_HIP(hipGetLastError());
    }
    plan->keys_written = true;
    return 0;
}

int materialize_heads(ppmg_plan* plan, hipStream_t s) {
    if (plan->bin_lattice) {
        if (!plan->lattice_checked) {
            // a lattice binning no gather has checked: bin the positions
            int64_t nbad = 0;
            return bin_particles(plan, plan->bin_mesh, plan->bin_prec, plan->np, plan->bin_xp, s, &nbad, false,
                                 false);
        }
        // a checked lattice: cell c holds particle c
        if (plan->start.ensure(sizeof(int) * (size_t)(plan->ncells + 1))) return PPMG_ERROR_FATAL;
        hipLaunchKernelGGL(k_iota, dim3(nblk(plan->ncells + 1, 256)), dim3(256), 0, s, plan->start.as<int>(),
                           plan->ncells + 1);
        PPMG_HIP(hipGetLastError());
        plan->bin_lattice = false;
        return 0;
    }
    if (!plan->bin_table) return 0;
    const int64_t ncells = plan->ncells, np = plan->np;
    if (plan->start.ensure(sizeof(int) * (size_t)(ncells + 1)) || plan->perm.ensure(sizeof(int) * (size_t)np))
        return PPMG_ERROR_FATAL;
    int* start = plan->start.as<int>();
    const uint32_t* count8 = plan->count.as<uint32_t>();
    if (exclusive_scan_u8(count8, ncells, start, plan->scan_tmp, np, s)) return PPMG_ERROR_FATAL;
    hipLaunchKernelGGL(k_table_perm, dim3(nblk(ncells, 256)), dim3(256), 0, s, count8, start,
                       plan->table.as<int>(), ncells, plan->perm.as<int>());
    PPMG_HIP(hipGetLastError());
    plan->bin_table = false;
    plan->perm_identity = false;
    plan->perm_written = true;
    return 0;
}

int materialize_perm(ppmg_plan* plan, hipStream_t s) {
    if (materialize_heads(plan, s)) return PPMG_ERROR_FATAL;
    if (plan->perm_identity && !plan->perm_written && plan->np > 0) {
        if (plan->perm.ensure(sizeof(int) * (size_t)plan->np)) return PPMG_ERROR_FATAL;
        hipLaunchKernelGGL(k_identity, dim3(nblk(plan->np, 256)), dim3(256), 0, s, plan->np, plan->perm.as<int>());
        PPMG_HIP(hipGetLastError());
    }
    plan->perm_written = true;
    return 0;
}

// ppm_util_sort3d / sort2d (ppm_util_sort3d.f:237-260): particle rows in the
// ranking's order (1-based lpdx), and the particle count of every box.
template <typename T>
__global__ void __launch_bounds__(256) k_gather_rows(const T* __restrict__ src, const int* __restrict__ lpdx1,
                                                     int64_t n, int dim, T* __restrict__ dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t p = lpdx1[i] - 1;
    for (int d = 0; d < dim; ++d) dst[i * dim + d] = src[p * dim + d];
}

__global__ void __launch_bounds__(256) k_box_counts(const int* __restrict__ lhbx1, int64_t nbox,
                                                    int* __restrict__ npbx) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c < nbox) npbx[c] = lhbx1[c + 1] - lhbx1[c];
}

int sort_rows(int dim, int prec, int64_t np, void* xp, const int* lpdx1, const int* lhbx1, int64_t nbox, int* npbx,
              DevBuf& tmp, hipStream_t s) {
    const size_t esz = prec == PPMG_PREC_F32 ? 4 : 8;
    if (np > 0) {
        if (tmp.ensure(esz * (size_t)np * dim)) return PPMG_ERROR_FATAL;
        if (esz == 4)
            hipLaunchKernelGGL(k_gather_rows<float>, dim3(nblk(np, 256)), dim3(256), 0, s, (const float*)xp, lpdx1, np,
                               dim, tmp.as<float>());
        else
            hipLaunchKernelGGL(k_gather_rows<double>, dim3(nblk(np, 256)), dim3(256), 0, s, (const double*)xp, lpdx1,
                               np, dim, tmp.as<double>());
        PPMG_HIP(hipMemcpyAsync(xp, tmp.p, esz * (size_t)np * dim, hipMemcpyDeviceToDevice, s));
    }
    if (npbx) hipLaunchKernelGGL(k_box_counts, dim3(nblk(nbox, 256)), dim3(256), 0, s, lhbx1, nbox, npbx);
    PPMG_HIP(hipGetLastError());
    return 0;
}

int rank_particles(ppmg_plan* plan, const RankGeom& g, int prec, int64_t np, const void* xp,
                   int* lpdx, int* lhbx, int64_t* icount, hipStream_t s) {
    int64_t ncells = (int64_t)g.ntot[0] * g.ntot[1] * g.ntot[2];
    // the plan's scratch is reused below: a slot table's counts are
    // overwritten, so its heads are built first
    if (materialize_heads(plan, s)) return PPMG_ERROR_FATAL;
    plan->prebinned = false;
    // Large input is ranked by the radix sort of its cell keys (2^24 particles in
    // no order, eight to a box: 0.46 against 1.34 ms; 10^6: 102 against 114 us,
    // 2^19: 98 against 85); slot
    // atomics and per-cell sorts keep the small ones, whose counts stay in L2
    // and which have few launches (PPMG_RADIX forces either, as in the binning),
    // and those whose sort is refused its scratch (20 bytes a particle with the
    // keys, where counting takes 8 and 4 per box).
    const char* rx = std::getenv("PPMG_RADIX");
    const bool radix = np > 0 && (rx && rx[0] ? rx[0] == '1' : np >= RANK_RADIX_NP) &&
                       radix_scratch(plan, np, ncells + 1);
    if (plan->key.ensure(sizeof(int) * (size_t)(np > 0 ? np : 1)) || plan->err.ensure(sizeof(int) * 4)) return PPMG_ERROR_FATAL;
    if (!radix && (plan->slot.ensure(sizeof(int) * (size_t)(np > 0 ? np : 1)) ||
                   plan->count.ensure(sizeof(int) * (size_t)ncells)))
        return PPMG_ERROR_FATAL;
    if ((!radix && fill_zero(plan->count.p, sizeof(int) * (size_t)ncells, s)) || fill_zero(plan->err.p, sizeof(int) * 4, s))
        return PPMG_ERROR_FATAL;
    if (np > 0) {
        unsigned gr = nblk(np, 256);
        int* st = plan->err.as<int>();
#define RANK_KEYS(D, T, S) hipLaunchKernelGGL((k_rank_keys<D, T, S>), dim3(gr), dim3(256), 0, s, (const T*)xp, np, g, \
                                              plan->key.as<int>(), plan->slot.as<int>(), plan->count.as<int>(), st)
#define RANK_KEYS_T(D, T)                      \
    do {                                       \
        if (radix) RANK_KEYS(D, T, false);     \
        else RANK_KEYS(D, T, true);            \
    } while (0)
        const bool single = prec == PPMG_PREC_F32;
        if (g.dim == 3) {
            if (single) RANK_KEYS_T(3, float);
            else RANK_KEYS_T(3, double);
        } else {
            if (single) RANK_KEYS_T(2, float);
            else RANK_KEYS_T(2, double);
        }
#undef RANK_KEYS_T
#undef RANK_KEYS
        PPMG_HIP(hipGetLastError());
    }
    int stats[2] = {0, 0};
    if (read_back(plan, plan->err.as<int>(), 2, stats, s)) return PPMG_ERROR_FATAL;
    int64_t inside = np - stats[0];
    if (radix) {
        const int* ks = nullptr;
        if (radix_sort(plan, plan->key.as<int>(), np, ncells + 1, lpdx, 1, inside, s, &ks)) return PPMG_ERROR_FATAL;
        hipLaunchKernelGGL(k_heads, dim3(nblk(ncells, HEADS_CELLS)), dim3(256), 0, s, ks, np, ncells, lhbx, 1, 1,
                           (int*)nullptr);
    } else {
        if (exclusive_scan(plan->count.as<int>(), ncells, lhbx, plan->scan_tmp, inside, s)) return PPMG_ERROR_FATAL;
        if (np > 0) {
            hipLaunchKernelGGL(k_scatter<int>, dim3(nblk(np, 1024)), dim3(256), 0, s, plan->key.as<int>(),
                               plan->slot.as<int>(), lhbx, np, lpdx);
            hipLaunchKernelGGL(k_stabilize, dim3(nblk(ncells, 256)), dim3(256), 0, s, lhbx, ncells, lpdx);
            hipLaunchKernelGGL(k_to_one_based, dim3(nblk(inside, 256)), dim3(256), 0, s, lpdx, inside);
        }
        hipLaunchKernelGGL(k_to_one_based, dim3(nblk(ncells + 1, 256)), dim3(256), 0, s, lhbx, ncells + 1);
    }
    PPMG_HIP(hipGetLastError());
    // the binning's keys were overwritten: recomputed from its positions when read
    plan->keys_written = false;
    *icount = inside;
    return 0;
}

}  // namespace ppmg
