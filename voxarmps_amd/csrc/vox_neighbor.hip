// vox_neighbor.hip — hash-sort neighbour grid for gfx950.
//
// Replaces NEIGHBOR (functions.cu:2788-2929) and the GPU hash search of
// neighbour_parallel.cu:344-444. The output reproduces the reference's CPU
// list bit-exactly:
//   cell  = int((x-Xmin)/re)+1, int((y-Ymin)/re)+1, int((z-Zmin)/(re+DELTA))+1
//           (IEEE divide, truncation; functions.cu:2822-2828),
//   order = stencil x-offset outer, y middle, z inner, clipped at the grid edge
//           (2865-2880), ascending particle id inside a cell (the serial
//           binning of 2820-2852 is a stable sort by cell),
//   rule  = 3D: sqrt(dx^2+dy^2+dz^2) <= re+DELTA, self included (2886);
//           2D: i != j and sqrt(dx^2+dy^2) < re (2907-2910).
// With ref_gpu the 2D list follows the reference's CUDA search instead
// (neighbour_parallel.cu:37-72, 145-199): cells re+DELTA wide in x and y,
// sqrt(dx^2+dy^2) <= re+DELTA with the particle itself, the same stencil order,
// ascending id inside a cell (its sort by cell key keeps the id order).
// The distance is evaluated exactly as the reference (no FMA: the library is
// built with -ffp-contract=off); a +-1e-10 relative band around the radius
// decides which candidates need the correctly rounded sqrt.
//
// Pipeline per list: key+count (atomic histogram, each particle its slot) -> exclusive scan (cell
// start) -> scatter -> per-cell rank sort by id (one wave per cell,
// LDS tile) with position records copied into cell order -> stencil walk (one
// thread per particle, or a wave per 64 sorted particles on the matrix cores) writing
// sliced rows (sl_index). With two radii the two lists' pipelines run on two streams.
#include <utility>

#include "vox_internal.hpp"

namespace vox {

// ---- utility kernels ----------------------------------------------------------------
__global__ void k_fill_i32(int32_t* __restrict__ p, int32_t v, long n)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long s = (long)gridDim.x * blockDim.x;
    for (; i < n; i += s) p[i] = v;
}

__global__ void k_fill_f64(double* __restrict__ p, double v, long n)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long s = (long)gridDim.x * blockDim.x;
    for (; i < n; i += s) p[i] = v;
}

int fill_i32(vox_ctx* c, int32_t* p, int32_t v, long n)
{
    if (n <= 0) return VOX_OK;
    int g = grid_for(n);
    if (g > 4096) g = 4096;
    k_fill_i32<<<g, kBlock, 0, c->stream>>>(p, v, n);
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

int fill_f64(vox_ctx* c, double* p, double v, long n)
{
    if (n <= 0) return VOX_OK;
    int g = grid_for(n);
    if (g > 4096) g = 4096;
    k_fill_f64<<<g, kBlock, 0, c->stream>>>(p, v, n);
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

// ---- exclusive scan (int32), three phases ----------------------------------------------
constexpr int kScanItems = 4;                       // items per thread
constexpr int kScanTile = kBlock * kScanItems;      // 1024 per block

__device__ __forceinline__ int32_t block_excl_scan(int32_t v, int32_t* lds, int32_t* total)
{
    int t = threadIdx.x;
    lds[t] = v;
    __syncthreads();
    for (int off = 1; off < kBlock; off <<= 1) {
        int32_t add = (t >= off) ? lds[t - off] : 0;
        __syncthreads();
        lds[t] += add;
        __syncthreads();
    }
    int32_t incl = lds[t];
    *total = lds[kBlock - 1];
    __syncthreads();
    return incl - v;
}

// Exclusive scan in two launches: the sum of each tile of kScanTile items,
// then per tile its offset (the sum of the tiles before it, which each block
// adds up from the first pass's sums) plus the tile's own exclusive scan.
__global__ void k_scan_tile_sums(const int32_t* __restrict__ in, int32_t* __restrict__ block_sums,
                                 long n)
{
    __shared__ int32_t lds[kBlock];
    const long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
    int32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) s += (base + k < n) ? in[base + k] : 0;
    int32_t tot;
    (void)block_excl_scan(s, lds, &tot);
    if (threadIdx.x == 0) block_sums[blockIdx.x] = tot;
}

// total (if given) receives the sum of all n items; it may alias out + n. clear
// (if given): the input, zeroed once it is read.
__global__ void k_scan_out(const int32_t* in, int32_t* out, const int32_t* __restrict__ block_sums,
                           long n, int32_t* total, int32_t* clear)
{
    __shared__ int32_t lds[kBlock];
    int32_t before = 0;
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += kBlock) before += block_sums[k];
    int32_t off;
    (void)block_excl_scan(before, lds, &off);
    const long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
    int32_t v[kScanItems];
    int32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = (base + k < n) ? in[base + k] : 0;
        s += v[k];
    }
    int32_t tot;
    int32_t ex = off + block_excl_scan(s, lds, &tot);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (base + k < n) {
            out[base + k] = ex;
            if (clear) clear[base + k] = 0;
        }
        ex += v[k];
    }
    if (total && threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) *total = off + tot;
}

// The same scan by one block, tile by tile: one launch instead of two, 6.0 us
// (and a gap) -> 3.2 us at 8k items.
constexpr int kScanOne = 1024;                      // threads, 4 items each a tile
constexpr long kScanOneMax = 4L * 4 * kScanOne;
__global__ __launch_bounds__(kScanOne) void k_scan_one(const int32_t* in, int32_t* out, long n,
                                                       int32_t* total, int32_t* clear)
{
    __shared__ int32_t sums[kScanOne / kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    int32_t before = 0;
    for (long tile = 0; tile < n; tile += 4 * kScanOne) {
        const long base = tile + 4 * threadIdx.x;
        int32_t v[4], s = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = (base + k < n) ? in[base + k] : 0;
            s += v[k];
        }
        int32_t incl = s;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int32_t x = __shfl_up(incl, o);
            if (lane >= o) incl += x;
        }
        if (lane == kWave - 1) sums[wave] = incl;
        __syncthreads();
        int32_t ex = before + incl - s;
#pragma unroll
        for (int w = 0; w < kScanOne / kWave; ++w) {
            const int32_t x = sums[w];
            ex += (w < wave) ? x : 0;
            before += x;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (base + k < n) {
                out[base + k] = ex;
                if (clear) clear[base + k] = 0;
            }
            ex += v[k];
        }
    }
    if (total && threadIdx.x == 0) *total = before;
}

// Scratch for a scan of n items. A capacity is only ever that of a live buffer.
static int reserve_scan(vox_ctx* c, long n)
{
    const long nb = (n + kScanTile - 1) / kScanTile;
    if (n <= kScanOneMax || nb <= c->scan_blocks_cap) return VOX_OK;
    if (c->scan_blocks) (void)hipFree(c->scan_blocks);
    c->scan_blocks = nullptr;
    c->scan_blocks_cap = 0;
    VOX_HIP(hipMalloc(&c->scan_blocks, sizeof(int32_t) * (nb + 64)));
    c->scan_blocks_cap = nb + 64;
    return VOX_OK;
}

// out[0..n) = exclusive scan of in[0..n); out[n] = total if out has room (caller
// passes total_dev to receive it; may alias out + n); clear: in, zeroed on the way.
int scan_exclusive(vox_ctx* c, const int32_t* in, int32_t* out, long n, int32_t* total_dev, int32_t* clear)
{
    if (n <= kScanOneMax) {
        k_scan_one<<<1, kScanOne, 0, c->stream>>>(in, out, n, total_dev, clear);
        VOX_HIP(hipGetLastError());
        return VOX_OK;
    }
    VOX_TRY(reserve_scan(c, n));
    const long nb = (n + kScanTile - 1) / kScanTile;
    k_scan_tile_sums<<<(int)nb, kBlock, 0, c->stream>>>(in, c->scan_blocks, n);
    k_scan_out<<<(int)nb, kBlock, 0, c->stream>>>(in, out, c->scan_blocks, n, total_dev, clear);
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

// ---- grid ------------------------------------------------------------------------------
static Grid make_grid(const vox_params& p, double re)
{
    Grid g;
    g.xmin = p.xmin; g.ymin = p.ymin; g.zmin = p.zmin;
    g.hx = re;
    g.hz = re + p.delta;
    g.dim = p.dim;
    g.incl = (p.dim == 3 || p.ref_gpu) ? 1 : 0;
    // the CUDA path's 2D cells are re+DELTA wide (neighbour_parallel.cu:46-47, 57-58)
    if (p.ref_gpu) g.hx = re + p.delta;
    g.ncx = (int)((p.xmax - p.xmin) / g.hx) + 1;                  // functions.cu:2790-2791
    g.ncy = (int)((p.ymax - p.ymin) / g.hx) + 1;
    g.ncz = (p.dim == 3) ? (int)((p.zmax - p.zmin) / g.hz) + 1 : 1; // 2796
    g.tnc = (long)g.ncx * g.ncy * g.ncz;
    return g;
}

// 1-based cell coordinates; false outside the grid (the reference has no check).
__device__ __forceinline__ bool cell_coords(const Grid& g, double x, double y, double z,
                                            int& ic, int& jc, int& kc)
{
    if (!isfinite(x) || !isfinite(y) || (g.dim == 3 && !isfinite(z))) return false;
    double ax = (x - g.xmin) / g.hx;
    double ay = (y - g.ymin) / g.hx;
    if (ax > 2e9 || ay > 2e9 || ax < -2e9 || ay < -2e9) return false;
    ic = (int)ax + 1;
    jc = (int)ay + 1;
    kc = 1;
    if (g.dim == 3) {
        double az = (z - g.zmin) / g.hz;
        if (az > 2e9 || az < -2e9) return false;
        kc = (int)az + 1;
    }
    return ic >= 1 && ic <= g.ncx && jc >= 1 && jc <= g.ncy && kc >= 1 && kc <= g.ncz;
}

// Cell number with the innermost stencil axis fastest (z in 3D, y in 2D; then
// y, then x), the order the reference walks a stencil in (functions.cu:2871-2890):
// the cells of one (x, y) column of a stencil are one contiguous run of the
// cell-sorted records, and a row's entries ascend in position. Before, cells
// were numbered x fastest, as the reference does (2826-2834; vox_get_cells
// still reports that number).
__host__ __device__ __forceinline__ int cell_key(const Grid& g, int ix, int iy, int iz)
{
    return (ix * g.ncy + iy) * g.ncz + iz;
}
// Cells along the innermost axis: key = row * inner_cells + inner.
__host__ __device__ __forceinline__ int inner_cells(const Grid& g)
{
    return g.dim == 3 ? g.ncz : g.ncy;
}

// ctr[key] += 1 for every active lane of the wave, with one atomic per
// distinct key: consecutive particles mostly share a cell, so per-lane atomics
// on one counter serialise. Returns the lane's slot among the key's
// increments (the counter's old value plus its rank among the wave's lanes
// with that key). Must be reached by every lane of the wave; the loop runs
// once per distinct key among the active lanes and only finds the lanes that
// share a key, so that all keys' atomics are on their way together.
__device__ __forceinline__ int32_t wave_add1(int32_t* __restrict__ ctr, int32_t key, bool active)
{
    const int lane = threadIdx.x & (kWave - 1);
    unsigned long long todo = __ballot(active), mine = 1ull << lane;
    while (todo) {
        const int lead = __ffsll((unsigned long long)todo) - 1;
        const int32_t lk = __shfl(key, lead);
        const unsigned long long m = __ballot(active && key == lk);
        if (active && key == lk) mine = m;
        todo &= ~m;
    }
    const int lead = __ffsll((unsigned long long)mine) - 1;
    int32_t base = 0;
    if (active && lane == lead) base = atomicAdd(&ctr[key], (int32_t)__popcll(mine));
    return __shfl(base, lead) + (int32_t)__popcll(mine & ((1ull << lane) - 1ull));
}

__global__ __launch_bounds__(kBlock) void k_cell_keys(Grid g, int n, const double* __restrict__ x,
                            const double* __restrict__ y, const double* __restrict__ z,
                            int32_t* __restrict__ cell, int32_t* __restrict__ slot_of,
                            int32_t* __restrict__ count, int32_t* __restrict__ flags)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool act = i < n;
    int32_t key = 0;
    if (act) {
        int ic, jc, kc;
        double zi = (g.dim == 3) ? z[i] : 0.0;
        if (cell_coords(g, x[i], y[i], zi, ic, jc, kc)) {
            key = cell_key(g, ic - 1, jc - 1, kc - 1);
        } else {
            atomicAdd(&flags[FLAG_DOMAIN], 1);
            atomicMin(&flags[FLAG_DOMAIN_FIRST], i);
        }
        cell[i] = key;
    }
    const int32_t slot = wave_add1(count, key, act);
    if (act) slot_of[i] = slot;
}

// Places each particle in its cell's run of order_raw, at the slot it got when
// it was counted (a second round of atomics took 13 us at 12k particles, 2.5
// now); the order inside a run is arbitrary here (the per-cell id sort or rank
// that follows makes it ascending by id).
__global__ __launch_bounds__(kBlock) void k_scatter(int n, const int32_t* __restrict__ cell,
                          const int32_t* __restrict__ slot_of, const int32_t* __restrict__ start,
                          int32_t* __restrict__ order_raw)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) order_raw[start[cell[i]] + slot_of[i]] = i;
}

// One wave per cell: rank of each id among the cell's ids (ids are unique), so
// the run becomes ascending by id; positions are copied into the same order,
// with the cell key in the record's aux slot.
constexpr int kSortTile = 512;   // ids per wave held in LDS

__global__ __launch_bounds__(kBlock) void k_cell_sort(
    long tnc, int dim, const int32_t* __restrict__ start, const int32_t* __restrict__ order_raw,
    PosRec* __restrict__ rec, int32_t* __restrict__ pos_of, const double* __restrict__ x,
    const double* __restrict__ y, const double* __restrict__ z)
{
    __shared__ int32_t tile[kBlock / kWave][kSortTile];
    int wv = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    long cellid = (long)blockIdx.x * (kBlock / kWave) + wv;
    if (cellid >= tnc) return;
    int s = start[cellid], e = start[cellid + 1], n = e - s;
    if (n <= 0) return;
    const int32_t* src = order_raw + s;
    bool in_lds = (n <= kSortTile);
    if (in_lds)
        for (int k = lane; k < n; k += kWave) tile[wv][k] = src[k];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    for (int k = lane; k < n; k += kWave) {
        int32_t id = in_lds ? tile[wv][k] : src[k];
        int rank = 0;
        for (int m = 0; m < n; ++m) {
            int32_t o = in_lds ? tile[wv][m] : src[m];
            rank += (o < id);
        }
        int pos = s + rank;
        PosRec rr;
        rr.x = x[id];
        rr.y = y[id];
        rr.z = (dim == 3) ? z[id] : 0.0;
        rr.id = id;
        rr.aux = (int32_t)cellid;
        rec[pos] = rr;
        pos_of[id] = pos;
    }
}

// The same order with one thread per particle, for grids whose cells hold a
// few particles each (a wave per cell would leave most lanes idle and visit
// every empty cell): the particle at scattered slot t counts the ids of its
// cell's members below its own, which is its rank in the ascending run.
__global__ __launch_bounds__(kBlock) void k_cell_rank(
    int n, int dim, const int32_t* __restrict__ cell, const int32_t* __restrict__ start,
    const int32_t* __restrict__ order_raw, PosRec* __restrict__ rec, int32_t* __restrict__ pos_of,
    const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int32_t id = order_raw[t];
    const int32_t c = cell[id];
    const int s = start[c], e = start[c + 1];
    int rank = 0;
    for (int m = s; m < e; ++m) rank += (order_raw[m] < id);
    PosRec rr;
    rr.x = x[id];
    rr.y = y[id];
    rr.z = (dim == 3) ? z[id] : 0.0;
    rr.id = id;
    rr.aux = c;
    rec[s + rank] = rr;
    pos_of[id] = s + rank;
}

// Per-particle stencil walk. R is the accept radius (3D and the CUDA path:
// re+DELTA, inclusive; 2D: re, exclusive).
__device__ __forceinline__ int wave_max_i32(int v)
{
    for (int off = kWave / 2; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, kWave));
    return v;
}

// Row output through a per-thread ring of 16 ids in LDS: a completed group of
// 8 entries is stored at once (one 32-byte store into the lane's own chunk),
// instead of 8 separate 4-byte stores that would leave the sector partly
// written several times. Groups past the row capacity are not stored (the
// overflow is reported and the search repeats with wider rows).
constexpr int kIdRing = 17;   // stride: lanes' equal slots fall on distinct banks

__device__ __forceinline__ void flush_ids(const int32_t* ring, int c, int cap,
                                          int32_t* __restrict__ row)
{
    if ((c << 3) >= cap) return;
    const int s0 = (c & 1) * 8;
    v4i* o = reinterpret_cast<v4i*>(row + ((long)c << 9));
    o[0] = v4i{ring[s0 + 0], ring[s0 + 1], ring[s0 + 2], ring[s0 + 3]};
    o[1] = v4i{ring[s0 + 4], ring[s0 + 5], ring[s0 + 6], ring[s0 + 7]};
}

// Thread t takes the particle at position t of the cell-sorted order (its
// record holds position, id and cell), so a wave's lanes sit in a few
// neighbouring cells of one grid row: they walk the same or overlapping
// stencils, with equal trip counts over a shared cell and candidate loads
// that hit the same lines.
__global__ __launch_bounds__(kBlock) void k_build_list(
    Grid g, int n, double R, const int32_t* __restrict__ start, const PosRec* __restrict__ rec,
    int cap, int32_t* __restrict__ ids, int32_t* __restrict__ cnt, int32_t* __restrict__ spread,
    int slot_max)
{
    __shared__ int32_t ring_all[kBlock * kIdRing];
    int32_t* ring = ring_all + threadIdx.x * kIdRing;
    const int t = xcd_tid();
    int k = 0;
    if (t < n) {
        const PosRec me = rec[t];
        const int i = me.id;
        const int ni = inner_cells(g);
        const int row = me.aux / ni, in = me.aux % ni;
        const int ix = (g.dim == 3) ? row / g.ncy : row, iy = (g.dim == 3) ? row % g.ncy : 0;
        const int x1 = max(ix - 1, 0), x2 = min(ix + 1, g.ncx - 1);
        const int y1 = (g.dim == 3) ? max(iy - 1, 0) : 0;
        const int y2 = (g.dim == 3) ? min(iy + 1, g.ncy - 1) : 0;
        const int ny = (g.dim == 3) ? g.ncy : 1;
        const int i1 = max(in - 1, 0), i2 = min(in + 1, ni - 1) + 1;
        const double xi = me.x, yi = me.y, zi = me.z;
        const double R2 = R * R;
        const double lo = R2 * (1.0 - 1e-10), hi = R2 * (1.0 + 1e-10);
        const long rb = sl_index(i, 0, cap);
        for (int xb = x1; xb <= x2; ++xb)
            for (int yb = y1; yb <= y2; ++yb) {
                // the innermost axis' cells are one run of records
                const int cn = (xb * ny + yb) * ni;
                const int s = start[cn + i1], e = start[cn + i2];
                // chunks of 8 candidates: loads first, then the ordered
                // accept/store pass (stores would serialise later loads)
                constexpr int U = 8;
                for (int j0 = s; j0 < e; j0 += U) {
                    PosRec cr[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) cr[u] = rec[(j0 + u < e) ? j0 + u : s];
                    const int k0 = k;
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        // branch-free test (the loads above stay unconditional)
                        // z is 0 in 2D records: dx^2+dy^2+0 equals the 2D sum
                        const PosRec cu = cr[u];
                        const double dx = cu.x - xi, dy = cu.y - yi, dz = cu.z - zi;
                        const double d2 = dx * dx + dy * dy + dz * dz;
                        bool acc = d2 < lo;
                        if (!acc && !(d2 > hi))   // rare band: exact sqrt decides
                            acc = g.incl ? (sqrt(d2) <= R) : (sqrt(d2) < R);
                        acc = acc && (j0 + u < e) && (g.incl || cu.id != i);
                        if (acc) {
                            ring[k & 15] = cu.id;
                            ++k;
                        }
                    }
                    // at most 8 accepts per chunk: at most one group completed
                    if ((k0 >> 3) != (k >> 3)) flush_ids(ring, k0 >> 3, cap, ids + rb);
                }
            }
        if (k & 7) flush_ids(ring, k >> 3, cap, ids + rb);
        cnt[i] = k;
    }
    // longest row: wave max -> block max
    __shared__ int wmax[kBlock / kWave];
    int m = wave_max_i32(k);
    if ((threadIdx.x % kWave) == 0) wmax[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        int b = wmax[0];
        for (int w = 1; w < kBlock / kWave; ++w) b = max(b, wmax[w]);
        atomicMax(spread_at(spread, slot_max), b);
    }
}

// The same walk with 16 lanes per particle: a run of records is tested 16
// candidates at a time, the accepted ones keep their order (ballot) and wait in
// LDS for stores of whole pieces of the row. One thread per particle is a chain
// of some ten round trips whatever the size; here a chain is a third of that, and
// a small system has 16 times the waves (lanes_max has the figures).
constexpr int kRowBuf = 64;                            // accepted ids a row holds in LDS
constexpr int kRowBufStride = kRowBuf + 1;

__global__ __launch_bounds__(kBlock) void k_build_list_l16(
    Grid g, int n, double R, const int32_t* __restrict__ start, const PosRec* __restrict__ rec,
    int cap, int32_t* __restrict__ ids, int32_t* __restrict__ cnt, int32_t* __restrict__ spread,
    int slot_max)
{
    __shared__ int32_t buf_all[kBlock / 16 * kRowBufStride];
    __shared__ int wmax[kBlock / kWave];
    const int lane = threadIdx.x & (kWave - 1), sub = threadIdx.x & 15;
    int32_t* const buf = buf_all + (threadIdx.x >> 4) * kRowBufStride;
    const int t = xcd_block() * (kBlock / 16) + (threadIdx.x >> 4);
    const unsigned long long seg = 0xffffull << (lane & 48);
    const unsigned long long below = seg & ((1ull << lane) - 1ull);
    int k = 0;
    if (t < n) {                                       // (uniform in a row of 16 lanes)
        const PosRec me = rec[t];
        const int i = me.id;
        const int ni = inner_cells(g);
        const int row = me.aux / ni, in = me.aux % ni;
        const int ix = (g.dim == 3) ? row / g.ncy : row, iy = (g.dim == 3) ? row % g.ncy : 0;
        const int x1 = max(ix - 1, 0), x2 = min(ix + 1, g.ncx - 1);
        const int y1 = (g.dim == 3) ? max(iy - 1, 0) : 0;
        const int y2 = (g.dim == 3) ? min(iy + 1, g.ncy - 1) : 0;
        const int ny = (g.dim == 3) ? g.ncy : 1, nyb = y2 - y1 + 1, runs = (x2 - x1 + 1) * nyb;
        const int i1 = max(in - 1, 0), i2 = min(in + 1, ni - 1) + 1;
        const double R2 = R * R;
        const double lo = R2 * (1.0 - 1e-10), hi = R2 * (1.0 + 1e-10);
        int32_t* __restrict__ out = ids + sl_index(i, 0, cap);
        int stored = 0;
        auto flush = [&]() {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (int e = stored + sub; e < k; e += 16)
                if (e < cap) out[((long)(e >> 3) << 9) + (e & 7)] = buf[e - stored];
            stored = k;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        // lane q holds the bounds of run q (at most 9), all loaded at once
        const int q = min(sub, runs - 1);
        const int cn = ((x1 + q / nyb) * ny + y1 + q % nyb) * ni;
        const int qs = start[cn + i1], qe = start[cn + i2];
        for (int r = 0; r < runs; ++r) {
            const int s = __shfl(qs, r, 16), e = __shfl(qe, r, 16);
            for (int j0 = s; j0 < e; j0 += 16) {
                const PosRec cu = rec[min(j0 + sub, e - 1)];
                const double dx = cu.x - me.x, dy = cu.y - me.y, dz = cu.z - me.z;
                const double d2 = dx * dx + dy * dy + dz * dz;
                bool acc = d2 < lo;
                if (!acc && !(d2 > hi))                // rare band: exact sqrt decides
                    acc = g.incl ? (sqrt(d2) <= R) : (sqrt(d2) < R);
                acc = acc && (j0 + sub < e) && (g.incl || cu.id != i);
                const unsigned long long m = __ballot(acc) & seg;
                if (acc) buf[k - stored + __popcll(m & below)] = cu.id;
                k += __popcll(m);
                if (k - stored > kRowBuf - 16) flush();
            }
        }
        flush();
        if (sub == 0) cnt[i] = k;
    }
    const int m = wave_max_i32(k);
    if (lane == 0) wmax[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        int b = wmax[0];
        for (int w = 1; w < kBlock / kWave; ++w) b = max(b, wmax[w]);
        atomicMax(spread_at(spread, slot_max), b);
    }
}

// Stencil walk for cells that hold many particles (3D list L: 64-80 a cell),
// on the matrix cores. A wave takes 64 consecutive particles of the
// cell-sorted order: one or a few cells of one row of cells along the innermost
// axis. The lanes of one row form a group (a wave that straddles rows makes a
// pass per row) and share its stencil: three runs of records in 2D, nine in
// 3D, streamed in blocks of 64 candidates. The squared distances of a block
// are a product: with positions relative to the group's first particle in
// units of R,
//   |p - c|^2 = |c|^2 + [c_x c_y c_z 1] . [-2p_x -2p_y -2p_z |p|^2],
// so one v_mfma_f32_16x16x4_f32 gives 16 candidates x 16 particles and a
// compare with 1 - |c|^2 decides each pair, where the vector units took
// 14 instructions a pair (3 differences, 3 products, the band tests, the
// append) in the walk this replaced.
// What FP32 cannot decide is decided as the reference does: every pair within
// kMmEps (|p|max + |c|)^2 of the radius (the rounding of the coordinates, of the
// product's five terms and of the threshold stays below a quarter of it) goes to
// a queue in LDS, evaluated 64 at a time with the reference's own expression in
// FP64 (functions.cu:2886, 2907), together with the cell test that a pair two
// cells apart needs. Such pairs are about 0.1 a particle in a moving fluid and
// the six at exactly 4 spacings on a lattice.
// A lane then walks its particle's accepted bits in candidate order (x outer,
// then y, then z, ascending id inside a cell: the reference's order) into a
// ring of 32 entries and stores completed groups of 8.
// Bound by VALU issue (15,600 instructions a wave on list L, 70% busy).
// Measured against the walk on vector units it replaced: list L of 199,000
// particles 554 -> 205 us, 305,000 particles on one 3.2 spacings radius
// 574 -> 284 us; at 1,180,000 particles both lists beside each other on two
// streams 2.0 -> 1.2 ms.
// kPos: the rows hold each neighbour's position in rec instead of its id.
typedef float v4fm __attribute__((ext_vector_type(4)));
constexpr float kMmEps = 1.9073486328125e-6f;      // 2^-19
constexpr int kMmRing = 32;                        // entries: 7 waiting + 16 accepted

__device__ __forceinline__ v4fm mfma_f32_k4(float a, float b, v4fm c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Entries 8 grp .. 8 grp + 7 of a lane's ring (slot-major: a lane's bank is
// its own) to its row; positions become ids where the rows hold ids. Only the
// first k entries of the row are positions: slots past them are not read as such.
template <bool kPos>
__device__ __forceinline__ void mm_flush(const int32_t* ring, int grp, int k, int cap,
                                         const PosRec* __restrict__ rec, int32_t* __restrict__ row)
{
    if ((grp << 3) >= cap) return;
    const int s0 = (grp & (kMmRing / 8 - 1)) * 8;
    int32_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = ring[(s0 + u) * kWave];
    if (!kPos) {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = rec[8 * grp + u < k ? v[u] : 0].id;
    }
    v4i* o = reinterpret_cast<v4i*>(row + ((long)grp << 9));
    o[0] = v4i{v[0], v[1], v[2], v[3]};
    o[1] = v4i{v[4], v[5], v[6], v[7]};
}

template <bool kPos>
__global__ __launch_bounds__(kWave, 4) void k_build_list_mm(
    Grid g, int n, double R, const int32_t* __restrict__ start, const PosRec* __restrict__ rec,
    int cap, int32_t* __restrict__ ids, int32_t* __restrict__ cnt, int32_t* __restrict__ spread,
    int slot_max)
{
    __shared__ __align__(16) float comp[4][kWave];      // candidates: x, y, z and 1
    __shared__ __align__(16) float thr[kWave];          // |c|^2 - 1
    __shared__ __align__(8) uint32_t mask[kWave][2];    // a particle's accepted candidates:
                                                        // 16 bits a tile, the first highest
    __shared__ __align__(8) uint32_t flip[kWave][2];    // and those the exact test decides otherwise
    __shared__ uint16_t queue[2 * kWave];               // particle | candidate << 6 | accepted << 12
    __shared__ int32_t ring_all[kMmRing * kWave];
    const int lane = threadIdx.x;
    int32_t* ring = ring_all + lane;
    char* const slots = reinterpret_cast<char*>(ring_all);
    constexpr uint32_t kSlotMask = kMmRing * kWave * 4 - 1;
    static_assert(4 * kWave == 256, "a ring slot holds 64 lanes' entries");
    const int t0 = xcd_block() * kWave;
    const int t = t0 + lane;
    const bool valid = t < n;
    const PosRec me = rec[valid ? t : 0];
    const int ni = inner_cells(g), ny = (g.dim == 3) ? g.ncy : 1;
    const int myrow = me.aux / ni, myin = me.aux % ni;
    const double invR = 1.0 / R;
    const float wide = fmaxf((float)(fmax(g.hx, g.hz) * invR), 1.f);   // a cell, in units of R
    // rows of positions are stored at the particle's own position too
    const long rb = sl_index(kPos ? t : (long)me.id, 0, cap);
    const int cl = lane & 15, cg = lane >> 4;
    int k = 0, kf = 0;                                  // entries accepted, entries stored
    uint32_t at = 4u * lane;                            // byte of the next free ring slot
    mask[lane][0] = mask[lane][1] = flip[lane][0] = flip[lane][1] = 0u;
    unsigned long long todo = __ballot(valid);
    while (todo) {
        const int lead = __ffsll(todo) - 1;
        const int row = __builtin_amdgcn_readfirstlane(__shfl(myrow, lead));
        const bool mine = valid && myrow == row;
        const unsigned long long m = __ballot(mine);
        todo &= ~m;
        const int last = 63 - __clzll(m);
        const int in_lo = __builtin_amdgcn_readfirstlane(__shfl(myin, lead));
        const int in_hi = __builtin_amdgcn_readfirstlane(__shfl(myin, last));
        const double ox = __shfl(me.x, lead), oy = __shfl(me.y, lead), oz = __shfl(me.z, lead);
        const float px = mine ? (float)((me.x - ox) * invR) : 0.f;
        const float py = mine ? (float)((me.y - oy) * invR) : 0.f;
        const float pz = mine ? (float)((me.z - oz) * invR) : 0.f;
        const float p2 = px * px + py * py + pz * pz;
        // the group's largest distance from its origin and its bounding box
        // (the lead itself sits at 0, the value of the other lanes)
        float pm = p2, bx = px, by = py, bz = pz, Bx = px, By = py, Bz = pz;
        for (int off = kWave / 2; off > 0; off >>= 1) {
            pm = fmaxf(pm, __shfl_xor(pm, off));
            bx = fminf(bx, __shfl_xor(bx, off)); Bx = fmaxf(Bx, __shfl_xor(Bx, off));
            by = fminf(by, __shfl_xor(by, off)); By = fmaxf(By, __shfl_xor(By, off));
            bz = fminf(bz, __shfl_xor(bz, off)); Bz = fmaxf(Bz, __shfl_xor(Bz, off));
        }
        pm = sqrtf(pm);
        // no candidate is more than two cells along an axis from a particle of
        // the group: |c| <= |p|max + 2 sqrt(3) cells
        const float reach = 2.f * pm + 4.f * wide + 1.f;
        const float eps = kMmEps * reach * reach;
        __syncthreads();
        comp[0][lane] = -2.f * px;
        comp[1][lane] = -2.f * py;
        comp[2][lane] = -2.f * pz;
        comp[3][lane] = mine ? p2 : 1e30f;              // no candidate is near another row's lanes
        __syncthreads();
        float bp[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) bp[q] = comp[cg][16 * q + cl];
        __syncthreads();
        comp[3][lane] = 1.f;
        const int ix = (g.dim == 3) ? row / g.ncy : row, iy = (g.dim == 3) ? row % g.ncy : 0;
        const int x1 = max(ix - 1, 0), x2 = min(ix + 1, g.ncx - 1);
        const int y1 = (g.dim == 3) ? max(iy - 1, 0) : 0;
        const int y2 = (g.dim == 3) ? min(iy + 1, g.ncy - 1) : 0;
        const int i1 = max(in_lo - 1, 0), i2 = min(in_hi + 1, ni - 1) + 1;
        for (int xb = x1; xb <= x2; ++xb)
            for (int yb = y1; yb <= y2; ++yb) {
                const int cn = (xb * ny + yb) * ni;
                const int cs = __builtin_amdgcn_readfirstlane(start[cn + i1]);
                const int ce = __builtin_amdgcn_readfirstlane(start[cn + i2]);
                PosRec nx = rec[min(cs + lane, n - 1)];
                for (int b0 = cs; b0 < ce; b0 += kWave) {
                    const int nc = min(kWave, ce - b0);
                    const PosRec cr = nx;
                    nx = rec[min(b0 + kWave + lane, n - 1)];                  // the next block's
                    const float cx = (float)((cr.x - ox) * invR);
                    const float cy = (float)((cr.y - oy) * invR);
                    const float cz = (float)((cr.z - oz) * invR);
                    const float c2 = cx * cx + cy * cy + cz * cz;
                    const bool in = lane < nc;
                    // tiles whose candidates are all out of reach of the
                    // group's box are left out
                    const float gx = fmaxf(fmaxf(bx - cx, cx - Bx), 0.f);
                    const float gy = fmaxf(fmaxf(by - cy, cy - By), 0.f);
                    const float gz = fmaxf(fmaxf(bz - cz, cz - Bz), 0.f);
                    const unsigned long long near =
                        __ballot(in && gx * gx + gy * gy + gz * gz < 1.f + eps);
                    if (!near) continue;
                    __syncthreads();                    // the last block's reads are done
                    comp[0][lane] = in ? cx : 0.f;
                    comp[1][lane] = in ? cy : 0.f;
                    comp[2][lane] = in ? cz : 0.f;
                    thr[lane] = in ? c2 - 1.f : 1e30f;
                    __syncthreads();
                    int nq = 0;
                    bool took = false;
                    // the exact test of the first `count` queued pairs
                    auto drain = [&](int count) {
                        __syncthreads();
                        if (lane < count) {
                            const uint32_t it = queue[lane];
                            const int pl = it & 63, c = (it >> 6) & 63;
                            const PosRec P = rec[t0 + pl], C = rec[b0 + c];
                            const double dx = C.x - P.x, dy = C.y - P.y, dz = C.z - P.z;
                            const double d = sqrt(dx * dx + dy * dy + dz * dz);
                            const int away = C.aux % ni - P.aux % ni;
                            const bool acc = (g.incl ? d <= R : d < R) && away >= -1 && away <= 1;
                            if (acc != ((it >> 12) != 0u))
                                atomicOr(&flip[pl][c >> 5], 0x8000u >> (c & 15) << (c & 16));
                        }
                        __syncthreads();
                    };
#pragma unroll 1
                    for (int tile = 0; tile < 4; ++tile) {
                        if (!((near >> (16 * tile)) & 0xffffull)) continue;
                        const int c0 = 16 * tile + 4 * cg;          // this lane's candidates
                        const float a = comp[cg][16 * tile + cl];
                        const v4fm t4 = *reinterpret_cast<const v4fm*>(&thr[c0]);
                        v4fm d[4];                                  // |p - c|^2 - 1
#pragma unroll
                        for (int q = 0; q < 4; ++q) d[q] = mfma_f32_k4(a, bp[q], t4);
                        const int sh = 12 - 4 * cg + 16 * (tile & 1);
                        float least = 1e30f;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            uint32_t nib = 0u;                      // the four sign bits
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                nib = (nib << 1) | (__float_as_uint(d[q][i]) >> 31);
                                least = fminf(least, fabsf(d[q][i]));
                            }
                            atomicOr(&mask[16 * q + cl][tile >> 1], nib << sh);
                        }
                        if (__any(least < eps)) {
                            took = true;
                            uint32_t ub = 0u, sg = 0u;              // bit 4 q + i
#pragma unroll
                            for (int q = 0; q < 4; ++q)
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    ub |= (fabsf(d[q][i]) < eps) ? 1u << (4 * q + i) : 0u;
                                    sg |= (__float_as_uint(d[q][i]) >> 31) << (4 * q + i);
                                }
                            for (;;) {
                                const unsigned long long um = __ballot(ub != 0u);
                                if (!um) break;
                                if (ub) {
                                    const int b = __ffs(ub) - 1;
                                    ub &= ub - 1u;
                                    queue[nq + __popcll(um & ((1ull << lane) - 1ull))] =
                                        (uint16_t)((16 * (b >> 2) + cl) | ((c0 + (b & 3)) << 6) |
                                                   (((sg >> b) & 1u) << 12));
                                }
                                nq += __popcll(um);
                                if (nq >= kWave) {
                                    drain(kWave);
                                    const uint16_t left = queue[kWave + lane];
                                    __syncthreads();
                                    queue[lane] = left;
                                    nq -= kWave;
                                }
                            }
                        }
                    }
                    if (nq) drain(nq);
                    __syncthreads();
                    uint32_t own[2] = {mask[lane][0], mask[lane][1]};
                    mask[lane][0] = mask[lane][1] = 0u;
                    if (took) {
                        own[0] ^= flip[lane][0];
                        own[1] ^= flip[lane][1];
                        flip[lane][0] = flip[lane][1] = 0u;
                    }
                    const int self = t - b0;
                    if (!g.incl && self >= 0 && self < nc) {        // the particle itself
                        const uint32_t bit = 0x8000u >> (self & 15) << (self & 16);
                        if (self >> 5) own[1] &= ~bit;
                        else own[0] &= ~bit;
                    }
#pragma unroll 1
                    for (int tile = 0; tile < 4; ++tile) {
                        const uint32_t h = (((tile & 2) ? own[1] : own[0]) >> (16 * (tile & 1))) & 0xffffu;
                        if (!__any(h != 0u)) continue;
                        // the next free slot takes every candidate; only an
                        // accepted one advances past it
                        const int base = b0 + 16 * tile;
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            *reinterpret_cast<int32_t*>(slots + at) = base + e;
                            at = (at + (__builtin_amdgcn_ubfe(h, 15 - e, 1) << 8)) & kSlotMask;
                        }
                        k += __popc(h);
                        while ((kf >> 3) < (k >> 3)) {
                            mm_flush<kPos>(ring, kf >> 3, k, cap, rec, ids + rb);
                            kf += 8;
                        }
                    }
                }
            }
    }
    if (valid && (k & 7)) mm_flush<kPos>(ring, k >> 3, k, cap, rec, ids + rb);
    int kmax = 0;
    if (valid) {
        cnt[kPos ? t : (long)me.id] = k;
        kmax = k;
    }
    kmax = wave_max_i32(kmax);
    if (lane == 0) atomicMax(spread_at(spread, slot_max), kmax);
}

// ---- host side --------------------------------------------------------------------------
// Empties the rows of a list whose search ended with rows longer than its storage
// (no room for wider ones, or another error first): every stage then finds no
// neighbours, and the next search starts from the storage there is.
static int drop_rows(vox_ctx* c, int which) { return fill_i32(c, c->list[which].cnt, 0, c->tp); }

int ensure_list_storage(vox_ctx* c, int which, int cap)
{
    DevList& L = c->list[which];
    cap = round_cap(cap);
    if (cap <= L.cap && L.ids) return VOX_OK;
    if (L.ids) (void)hipFree(L.ids);
    L.ids = nullptr;
    L.cap = 0;
    const size_t bytes = sizeof(int32_t) * (size_t)sl_size(c->tp, cap);
    const hipError_t e = hipMalloc(&L.ids, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        L.ids = nullptr;
        VOX_TRY(drop_rows(c, which));
        return fail(VOX_ERR_HIP, "neighbour rows of " + std::to_string(cap) + " entries (" +
                                     std::to_string(bytes >> 20) + " MB): " + hipGetErrorString(e));
    }
    L.cap = cap;
    return VOX_OK;
}

static int search_one(vox_ctx* c, int which, double re);

// What a search reports: the domain flags, and the longest rows with the other
// spread counters.
__global__ void k_clear_search(int32_t* __restrict__ flags, int32_t* __restrict__ spread)
{
    for (int k = threadIdx.x; k < kSpread * kSpreadLine; k += blockDim.x) spread[k] = 0;
    if (threadIdx.x == 0) {
        flags[FLAG_DOMAIN] = 0;
        flags[FLAG_DOMAIN_FIRST] = 0x7fffffff;
    }
}

static int clear_search_status(vox_ctx* c)
{
    k_clear_search<<<1, kSpread * kSpreadLine, 0, c->stream>>>(c->dflags, c->dspread);
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

// List L in 3D can hold compact rows: the reference accepts d <= re + DELTA
// with the particle itself (functions.cu:2886), but its consumers, PREDICTION
// and MATRIX, weigh each entry by W(d) with W = 0 at d >= re (kernel types 2
// and 6) and skip the particle itself, so the entries they actually use are
// those at d < re other than the particle itself - the 2D accept rule at the
// same radius. The compact rows keep the reference order (a subsequence of it,
// about 18% shorter), and a sum over them adds exactly the nonzero terms of
// the reference's sum in the same order (the skipped terms are +0 added to a
// sum that is never -0), so every result is the same bits for finite fields
// (a non-finite neighbour value times W = 0 is NaN in the reference's sum).
// MATRIX on the CPU path assembles at the positions the list was searched at
// (x, not x*), so its distances are the search's own. matopt and srcopt weigh
// by re/d^3 at any d and need the reference rows, as does an export:
// ensure_reference_list rebuilds them from the cell-sorted records of the same
// NEIGHBOR call.
const PosRec* list_order(const vox_ctx* c, int which)
{
    const DevList& L = list_of(c, which);
    return L.sorted ? L.rec : nullptr;
}

bool list_compact_ok(const vox_ctx* c)
{
    const vox_params& p = c->p;
    return c->two_lists && p.dim == 3 && !p.matopt && !p.srcopt && !p.ref_gpu &&
           (p.ktype == 2 || p.ktype == 6);
}

// Expected particles per cell (cell volume / DL^dim) below 24: the cells are
// sorted one thread per particle rather than one wave per cell.
static bool few_per_cell(const vox_ctx* c, const DevList& L)
{
    const double per_cell = (c->p.dim == 3)
        ? L.g.hx * L.g.hx * L.g.hz / (c->p.dl * c->p.dl * c->p.dl)
        : L.g.hx * L.g.hx / (c->p.dl * c->p.dl);
    return per_cell < 24.0;
}

// Grid, cell sort and one search pass of list `which` on c->stream, without
// waiting for it. Reports, once the stream has run, go to the list's overflow
// and longest-row flags and to the shared domain flags.
static int launch_one(vox_ctx* c, int which, double re)
{
    DevList& L = c->list[which];
    const int n = c->tp;
    L.re = re;
    L.searched = false;                // until this search's sort is queued
    L.g = make_grid(c->p, re);
    if (L.g.tnc <= 0 || L.g.tnc > (1L << 30))
        return fail(VOX_ERR_ARG, "neighbour grid has an invalid number of cells");
    if (L.g.tnc > L.tnc_alloc) {
        if (L.cell_start) (void)hipFree(L.cell_start);
        if (L.cell_fill) (void)hipFree(L.cell_fill);
        L.cell_start = L.cell_fill = nullptr;
        L.tnc_alloc = 0;
        L.fill_clear = false;
        VOX_HIP(hipMalloc(&L.cell_start, sizeof(int32_t) * (L.g.tnc + 1)));
        VOX_HIP(hipMalloc(&L.cell_fill, sizeof(int32_t) * (L.g.tnc + 1)));
        L.tnc_alloc = L.g.tnc;
    }
    // The scan of the counts clears them for the next search. A search that ends
    // between the count and that scan (an error of an earlier launch shows up there)
    // leaves them raised: slots counted on top of them would lie past order_raw, so
    // the next search clears them itself. What the scan needs is reserved first, and
    // the slots have an array of their own: rec, pos_of and the rows stay those of the
    // last search that got past here.
    VOX_TRY(reserve_scan(c, L.g.tnc));
    if (!L.fill_clear) VOX_TRY(fill_i32(c, L.cell_fill, 0, L.tnc_alloc + 1));
    L.fill_clear = false;
    {
        ProfScope ps(c, KC_CELL);
        k_cell_keys<<<grid_for(n), kBlock, 0, c->stream>>>(L.g, n, c->f[VOX_F_X], c->f[VOX_F_Y],
                                                             c->f[VOX_F_Z], L.cell, L.slot_of,
                                                             L.cell_fill, c->dflags);
        VOX_HIP(hipGetLastError());
    }
    {
        ProfScope ps(c, KC_SORT);
        VOX_TRY(scan_exclusive(c, L.cell_fill, L.cell_start, L.g.tnc, L.cell_start + L.g.tnc,
                               L.cell_fill));
        L.fill_clear = true;
        k_scatter<<<grid_for(n), kBlock, 0, c->stream>>>(n, L.cell, L.slot_of, L.cell_start,
                                                           L.order_raw);
        // cells of fewer than ~24 expected particles: one thread per particle
        if (few_per_cell(c, L)) {
            k_cell_rank<<<grid_for(n), kBlock, 0, c->stream>>>(n, c->p.dim, L.cell, L.cell_start,
                                                                L.order_raw, L.rec, L.pos_of,
                                                                c->f[VOX_F_X],
                                                                c->f[VOX_F_Y], c->f[VOX_F_Z]);
        } else {
            long nb = (L.g.tnc + (kBlock / kWave) - 1) / (kBlock / kWave);
            k_cell_sort<<<(int)nb, kBlock, 0, c->stream>>>(L.g.tnc, c->p.dim, L.cell_start,
                                                            L.order_raw, L.rec, L.pos_of,
                                                            c->f[VOX_F_X],
                                                            c->f[VOX_F_Y], c->f[VOX_F_Z]);
        }
        VOX_HIP(hipGetLastError());
    }
    L.sorted = L.searched = true;
    return search_one(c, which, re);
}

// The walk per particle takes 16 lanes up to this many particles, by the entries
// expected in a row (a short row leaves most of a group's last 16 lanes idle).
// NEIGHBOR calls, one thread and 16 lanes, us: 2D rows of 14 entries 50k 49 / 47, 65k 53 /
// 53, 100k 52 / 53, of 21 50k 47 / 47, 65k 51 / 52, 100k 59 / 65, of 30 65k 53 / 51, 100k
// 61 / 62, 131k 68 / 74, of 50 80k 63 / 60, 100k 67 / 68, 131k 70 / 77; 3D rows of 17 60k
// 71 / 65, 131k 86 / 84, 260k 123 / 132, of 39 60k 90 / 73, 100k 104 / 99, 131k 111 / 118, 260k
// 157 / 177, of 65 60k 115 / 82, 131k 135 / 128, 220k 211 / 189, 320k 241 / 249.
static int lanes_max(const vox_params& p, double re)
{
    const double e = row_entries(p, re);
    if (p.dim == 3) return e > 48.0 ? 1 << 18 : 3 << 15;
    return e > 24.0 ? 3 << 15 : 1 << 16;
}
// and against the matrix cores up to this many (16 lanes, matrix): 10k 69 / 171,
// 43k 134 / 196, 94k 229 / 238, 133k 304 / 244 at 4 spacings, 149 / 176 and 193 /
// 195 for the last two at 3.1. Half as many for list L, whose consumers read the
// rows of positions that only the matrix walk stores faster (steps, 16 lanes and
// matrix: 25k 790 / 832 us, 61k 1070 / 1063, 94k 1261 / 1220).
constexpr int kLanesMaxMm = 3 << 15;

// One search pass over the sorted cells of list `which` (rows at the list's
// current capacity), on c->stream.
static int search_one(vox_ctx* c, int which, double re)
{
    DevList& L = c->list[which];
    const int n = c->tp;
    const int sm = which == 0 ? SPR_MAXCNT_S : SPR_MAXCNT_L;
    // compact rows (list L): d < re, the particle itself excluded
    const bool compact = (which == 1) && list_compact_ok(c);
    Grid gg = L.g;
    if (compact) gg.incl = 0;
    const double R = gg.incl ? re + c->p.delta : re;
    L.compact = compact;
    L.epoch = c->pos_epoch;
    // The matrix-core walk where a cell is expected (cell volume / DL^dim) to
    // hold 24 particles or more and the system fills the chip with it, else the
    // walk per particle (here by one thread). NEIGHBOR calls
    // measured with either, matrix against per particle, us: 3D 67 a cell 1500
    // against 2480 (1,185,000 particles), 330 against 590 (201,000), 200 against
    // 270 (15,500); 35 a cell 1005 / 1420, 250 / 370, 170 / 190; 10 a cell 650 /
    // 630, 200 / 190, 150 / 104; 2D 16 a cell 354 / 296 (979,000), 4 a cell 395 / 210.
    const double per_cell = (c->p.dim == 3)
        ? L.g.hx * L.g.hx * L.g.hz / (c->p.dl * c->p.dl * c->p.dl)
        : L.g.hx * L.g.hx / (c->p.dl * c->p.dl);
    const int mode = c->tuned_mode[which] ? c->tuned_mode[which] : c->p.list_mode;
    const bool cell_walk = (mode == 2 || (mode == 0 && per_cell >= 24.0 &&
                                          n > (compact ? kLanesMaxMm / 2 : kLanesMaxMm)));
    ProfScope ps(c, which == 0 ? KC_LIST : KC_LIST_L);
    // Compact rows of the cell walk hold positions in the cell-sorted records
    // (and sit at the particle's position): their consumers gather from
    // records in that order, where a row's consecutive entries (one cell's
    // particles) sit side by side.
    L.pos_rows = compact && cell_walk;
    if (cell_walk) {
        if (L.pos_rows)
            k_build_list_mm<true><<<(n + kWave - 1) / kWave, kWave, 0, c->stream>>>(
                gg, n, R, L.cell_start, L.rec, L.cap, L.ids, L.cnt, c->dspread, sm);
        else
            k_build_list_mm<false><<<(n + kWave - 1) / kWave, kWave, 0, c->stream>>>(
                gg, n, R, L.cell_start, L.rec, L.cap, L.ids, L.cnt, c->dspread, sm);
    } else if (n <= lanes_max(c->p, re)) {
        k_build_list_l16<<<grid_for(16L * n), kBlock, 0, c->stream>>>(
            gg, n, R, L.cell_start, L.rec, L.cap, L.ids, L.cnt, c->dspread, sm);
    } else {
        k_build_list<<<grid_for(n), kBlock, 0, c->stream>>>(gg, n, R, L.cell_start, L.rec, L.cap,
                                                            L.ids, L.cnt, c->dspread, sm);
    }
    VOX_HIP(hipGetLastError());
    return VOX_OK;
}

// After read_flags, on the way out with an error: rows that were never searched
// again with the storage they need.
static int drop_long_rows(vox_ctx* c)
{
    for (int w = 0; w < (c->two_lists ? 2 : 1); ++w)
        if (spread_max(c, w == 0 ? SPR_MAXCNT_S : SPR_MAXCNT_L) > c->list[w].cap) VOX_TRY(drop_rows(c, w));
    return VOX_OK;
}

// After read_flags: the domain error, naming the first particle outside the
// grid (its type, position and velocity).
static int domain_error(vox_ctx* c)
{
    VOX_TRY(drop_long_rows(c));
    const int i = c->hflags[FLAG_DOMAIN_FIRST];
    double v[5] = {0, 0, 0, 0, 0};
    int32_t t = 0;
    const int fs[5] = {VOX_F_X, VOX_F_Y, VOX_F_Z, VOX_F_U, VOX_F_V};
    if (i >= 0 && i < c->tp) {
        for (int k = 0; k < 5; ++k)
            VOX_HIP(hipMemcpy(&v[k], c->f[fs[k]] + i, sizeof(double), hipMemcpyDeviceToHost));
        VOX_HIP(hipMemcpy(&t, c->ptype + i, sizeof(int32_t), hipMemcpyDeviceToHost));
    }
    char buf[256];
    std::snprintf(buf, sizeof buf, "; first: particle %d (PTYPE %d) at (%.6g, %.6g, %.6g), velocity (%.6g, %.6g)",
                  i, t, v[0], v[1], v[2], v[3], v[4]);
    return fail(VOX_ERR_DOMAIN, "particle outside the neighbour grid box (" +
                                    std::to_string(c->hflags[FLAG_DOMAIN]) + " particles)" + buf);
}

// After read_flags: rows of list `which` that did not fit are searched again
// with wider rows (up to 3 more passes).
static int regrow_one(vox_ctx* c, int which, double re)
{
    for (int attempt = 0; attempt < 4; ++attempt) {
        const int need = spread_max(c, which == 0 ? SPR_MAXCNT_S : SPR_MAXCNT_L);
        c->max_count[which] = need;
        if (need <= c->list[which].cap) return VOX_OK;
        if (attempt == 3) break;
        int cap = ((need + need / 4) + 7) & ~7;
        VOX_TRY(ensure_list_storage(c, which, cap));
        VOX_TRY(search_one(c, which, re));
        VOX_TRY(read_flags(c));
    }
    VOX_TRY(drop_rows(c, which));
    return fail(VOX_ERR_OVERFLOW, "neighbour row capacity could not be satisfied");
}

// The reference rows of list `which` in place of compact ones, searched again
// over the cell-sorted records of the NEIGHBOR call that built the list (the
// positions of that call, whatever the particles did since), by the cell-row
// walk, with wider rows while any overflows.
int ensure_reference_list(vox_ctx* c, int which)
{
    DevList& L = c->list[which];
    if (!L.compact) return VOX_OK;
    if (!L.searched) return fail(VOX_ERR_STATE, "the last neighbour search did not finish");
    const int sm = which == 0 ? SPR_MAXCNT_S : SPR_MAXCNT_L;
    const double R = L.g.incl ? L.re + c->p.delta : L.re;
    const int n = c->tp;
    for (int attempt = 0; attempt < 4; ++attempt) {
        VOX_TRY(fill_i32(c, c->dspread, 0, kSpread * kSpreadLine));
        k_build_list_mm<false><<<(n + kWave - 1) / kWave, kWave, 0, c->stream>>>(
            L.g, n, R, L.cell_start, L.rec, L.cap, L.ids, L.cnt, c->dspread, sm);
        VOX_HIP(hipGetLastError());
        L.pos_rows = false;
        VOX_TRY(read_flags(c));
        const int need = spread_max(c, sm);
        if (need <= L.cap) {
            L.compact = false;
            return VOX_OK;
        }
        VOX_TRY(ensure_list_storage(c, which, ((need + need / 4) + 7) & ~7));
    }
    VOX_TRY(drop_rows(c, which));
    return fail(VOX_ERR_OVERFLOW, "neighbour row capacity could not be satisfied");
}

// Called by every consumer of list L before it reads the rows: compact rows
// that no longer stand for the reference rows - the particles have moved since
// the search (the reference's rows, searched with the DELTA margin, are then
// read at other positions), or the settings have changed (a weight function
// that is not zero at re, matopt, srcopt) - are replaced by the reference rows.
int list_l_for_consumer(vox_ctx* c)
{
    const DevList& L = c->list[1];
    if (c->two_lists && L.compact && (L.epoch != c->pos_epoch || !list_compact_ok(c)))
        return ensure_reference_list(c, 1);
    return VOX_OK;
}

static int build_one(vox_ctx* c, int which, double re)
{
    VOX_TRY(clear_search_status(c));
    VOX_TRY(launch_one(c, which, re));
    VOX_TRY(read_flags(c));
    if (c->hflags[FLAG_DOMAIN] != 0) return domain_error(c);
    return regrow_one(c, which, re);
}

// Tile-shape autotuner of the neighbour search: times both walks (one thread
// per particle, one wave per 64 cell-sorted particles) on the current positions, `reps` builds
// each, and keeps the faster one per list. The lists are identical either way,
// so the choice only changes speed. modes[w] receives 1 or 2 per list.
int autotune_lists(vox_ctx* c, int reps, int32_t* modes)
{
    if (reps < 1) reps = 1;
    hipEvent_t e0, e1;
    VOX_HIP(hipEventCreate(&e0));
    VOX_HIP(hipEventCreate(&e1));
    int rc = VOX_OK;
    for (int w = 0; w < (c->two_lists ? 2 : 1) && rc == VOX_OK; ++w) {
        const double re = (w == 0) ? c->p.re_s : c->p.re_l;
        float best = 0.f;
        int pick = 1;
        for (int mode = 1; mode <= 2 && rc == VOX_OK; ++mode) {
            c->tuned_mode[w] = mode;
            if ((rc = build_one(c, w, re)) != VOX_OK) break;       // warm (and grows rows)
            (void)hipEventRecord(e0, c->stream);
            for (int r = 0; r < reps && rc == VOX_OK; ++r) rc = build_one(c, w, re);
            (void)hipEventRecord(e1, c->stream);
            if (rc != VOX_OK) break;
            if (hipEventSynchronize(e1) != hipSuccess) { rc = fail(VOX_ERR_HIP, "autotune sync"); break; }
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            if (mode == 1 || ms < best) { best = ms; pick = mode; }
        }
        c->tuned_mode[w] = pick;
        if (modes) modes[w] = pick;
    }
    if (!c->two_lists) {
        c->tuned_mode[1] = c->tuned_mode[0];
        if (modes) modes[1] = modes[0];
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
}

// List L on the side stream: the context's stream and scan scratch are swapped
// for the side ones while its work is queued.
static int launch_side(vox_ctx* c, int which, double re)
{
    std::swap(c->stream, c->stream2);
    std::swap(c->scan_blocks, c->scan_blocks2);
    std::swap(c->scan_blocks_cap, c->scan_blocks2_cap);
    const int rc = launch_one(c, which, re);
    std::swap(c->stream, c->stream2);
    std::swap(c->scan_blocks, c->scan_blocks2);
    std::swap(c->scan_blocks_cap, c->scan_blocks2_cap);
    return rc;
}

int build_neighbors(vox_ctx* c)
{
    if (c->two_lists && c->stream2) {
        VOX_TRY(clear_search_status(c));
        // The two lists are independent: list L is built on a second stream
        // beside list S (the side stream first waits for everything queued so
        // far), and the main stream waits for it before the one flag read.
        VOX_HIP(hipEventRecord(c->ev_fork, c->stream));
        VOX_HIP(hipStreamWaitEvent(c->stream2, c->ev_fork, 0));
        VOX_TRY(launch_one(c, 0, c->p.re_s));
        VOX_TRY(launch_side(c, 1, c->p.re_l));
        VOX_HIP(hipEventRecord(c->ev_join, c->stream2));
        VOX_HIP(hipStreamWaitEvent(c->stream, c->ev_join, 0));
        VOX_TRY(read_flags(c));
        if (c->hflags[FLAG_DOMAIN] != 0) return domain_error(c);
        const int rc = regrow_one(c, 0, c->p.re_s);
        if (rc != VOX_OK) {
            VOX_TRY(drop_long_rows(c));
            return rc;
        }
        VOX_TRY(regrow_one(c, 1, c->p.re_l));
    } else {
        VOX_TRY(build_one(c, 0, c->p.re_s));
        if (c->two_lists) VOX_TRY(build_one(c, 1, c->p.re_l));
    }
    c->st.max_count_s = c->max_count[0];
    c->st.max_count_l = c->max_count[c->two_lists ? 1 : 0];
    return VOX_OK;
}

}  // namespace vox
