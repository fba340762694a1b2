// Stable CSR → CSC transpose and COO → CSR builder for gfx950.
//
// Reference: toCSC's column-major scan (SpMM.cpp:80-95) and scipy's tocsc in
// the GCN script (gcn_custom.py:48-55) produce, for every column, its entries
// with ascending rows; csr2cscKernel (gcn/pytorch-custom/spmm_kernel.cu:381-423)
// would call cuSPARSE for it.  Here: a stable LSD radix sort of (column, row,
// value) records, up to 10 bits per pass (k_radix_scatter).  The input is already
// in row order and every pass is stable, so rows stay ascending inside each
// column; colptr is read off the sorted column keys.
//
// COO → CSR (the canonical CSR of toCSR, SDMM.cpp:355-370 / SpMM.cpp:64-79,
// built from unordered triplets on the device): the same stable sort by
// column, then by row, so entries end in (row, column) order with duplicates
// in input order; duplicates are summed in that order, entries whose sum is
// zero are dropped on request (toCSR keeps only `!= 0`), and rowptr is read off
// the sorted rows.
//
// CSR → vector-aware CSR (toVectorAwareCSR, SpMV.cpp:15-38) on the device: a
// decision per block-opening entry, an exclusive scan of the decisions, and a
// scatter of the stored blocks.
#include <climits>

#include "common.hpp"

namespace armsp {
namespace {

constexpr int TPB = 256;
constexpr int SCAN_CHUNK = 2048;  // 256 threads × 8

// ------------------------------------------------------------- radix sort
// One pass sorts the records by a digit of `db` bits: k_radix_hist counts the
// digits of every tile, k_radix_scan turns the counts into each tile's first
// position within its digit (and the digits' totals), k_radix_scatter ranks a
// tile's records, orders them by digit in LDS and writes every digit's run of
// the tile as consecutive elements.
// Bound: a record (key, companion index, value) is read and written once per
// pass, 24 bytes, plus 4 for the histogram, and ranked with one ballot per digit
// bit.  Digits are as wide as the LDS ranks allow (10 bits: a million columns
// take two passes), the value travels with its key, and the row of a CSR entry
// is formed in the first pass from rowptr.  (Sorting positions in 8-bit digits
// and gathering rows and values at the end took 1523 us for the 1M R-MAT's 2^24
// entries; 383 us now: 205 MB read and 213 MB written a pass, by the counters.)
// Consecutive tiles go to one XCD, so the lines two tiles share are completed in
// that XCD's L2 (in launch order instead: 480 -> 503 us).
constexpr int RADIX_MAX_BITS = 10;
constexpr int RADIX_MIN_BITS = 4;  // k_radix_scan takes 16 digits a workgroup
// A tile of more rows than so many times its records finds each record's row by a search:
// walking the rows, few of which hold an entry, would make that tile's time.  Uniform
// matrices of 2^19 columns, rows walked against searched: 4M entries in 4096-record tiles,
// 8, 16 and 64 rows an entry 168, 256, 1001 us against 209, 326, 553; 100,000 entries in
// 2048-record tiles, 8, 16, 64, 200 rows an entry 56, 68, 185, 608 us against 57, 58, 65, 82.
constexpr int radix_mark_rows(int threads) { return threads > 256 ? 24 : 8; }

// Tile of block b: XCD b % 8 walks a contiguous eighth of the tiles (-1: none).
__device__ __forceinline__ int xcd_tile(int ntiles) {
    const int per = (ntiles + 7) >> 3, i = (int)(blockIdx.x >> 3);
    const int t = (int)(blockIdx.x & 7u) * per + i;
    return t < ntiles ? t : -1;
}
inline unsigned xcd_grid(int ntiles) { return (unsigned)((ntiles + 7) / 8) * 8u; }

// hist[tile·bins + d] = records of the tile with digit d.  With `other`, also sets
// *bad where a key is outside [0, krange) or other[p] outside [0, orange).
template <int THREADS, int IPT>
__global__ __launch_bounds__(THREADS) void k_radix_hist(int n, int shift, int db, int ntiles,
                                                        const int* __restrict__ keys, int* __restrict__ hist,
                                                        const int* __restrict__ other, int krange, int orange,
                                                        int* __restrict__ bad) {
    __shared__ int cnt[1 << RADIX_MAX_BITS];
    const int bins = 1 << db, tile = xcd_tile(ntiles);
    if (tile < 0) return;
    for (int d = threadIdx.x; d < bins; d += THREADS) cnt[d] = 0;
    __syncthreads();
    const int64_t base = (int64_t)tile * (THREADS * IPT);
    int key[IPT];
    bool oob = false;
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        const int64_t e = base + j * THREADS + threadIdx.x;
        key[j] = e < n ? keys[e] : 0;
        if (other && e < n) {
            const int o = other[e];
            oob |= key[j] < 0 || key[j] >= krange || o < 0 || o >= orange;
        }
    }
#pragma unroll
    for (int j = 0; j < IPT; ++j)
        if (base + j * THREADS + threadIdx.x < n) atomicAdd(&cnt[(key[j] >> shift) & (bins - 1)], 1);
    if (oob) atomicOr(bad, 1);
    __syncthreads();
    for (int d = threadIdx.x; d < bins; d += THREADS) hist[(int64_t)tile * bins + d] = cnt[d];
}

// Per digit, the exclusive scan of its counts over the tiles, in place, and its
// total: a workgroup takes 16 digits (64-byte rows of hist), 64 threads a digit,
// each a run of consecutive tiles.
__global__ __launch_bounds__(1024) void k_radix_scan(int ntiles, int bins, int* __restrict__ hist,
                                                     int* __restrict__ totals) {
    // counts a thread holds between the two sweeps; the rest it reads again, as many at a time
    // (4096 tiles of 1024 digits 24 us; 26 with the rest one by one; 8 digits a workgroup: 21,
    // but 12.8 against 8.5 on 1465 tiles)
    constexpr int KEEP = 32;
    __shared__ int part[64][16];
    const int d = (int)(threadIdx.x & 15u), seg = (int)(threadIdx.x >> 4);
    int* h = hist + (int)blockIdx.x * 16 + d;
    const int per = (ntiles + 63) / 64;
    const int t0 = seg * per, t1 = min(t0 + per, ntiles);
    int v[KEEP];
    int s = 0;
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        v[i] = t0 + i < t1 ? h[(int64_t)(t0 + i) * bins] : 0;
        s += v[i];
    }
    for (int t = t0 + KEEP; t < t1; ++t) s += h[(int64_t)t * bins];
    part[seg][d] = s;
    __syncthreads();
    if (threadIdx.x < 16) {
        int run = 0;
        for (int q0 = 0; q0 < 64; q0 += 16) {  // 16 reads in flight
            int x[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) x[q] = part[q0 + q][d];
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                part[q0 + q][d] = run;
                run += x[q];
            }
        }
        totals[blockIdx.x * 16 + d] = run;
    }
    __syncthreads();
    int run = part[seg][d];
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
        if (t0 + i < t1) {
            h[(int64_t)(t0 + i) * bins] = run;
            run += v[i];
        }
    for (int t = t0 + KEEP; t < t1; t += KEEP) {
#pragma unroll
        for (int i = 0; i < KEEP; ++i) v[i] = t + i < t1 ? h[(int64_t)(t + i) * bins] : 0;
#pragma unroll
        for (int i = 0; i < KEEP; ++i)
            if (t + i < t1) {
                h[(int64_t)(t + i) * bins] = run;
                run += v[i];
            }
    }
}

// Exclusive scan of one value per thread over the workgroup; red: WAVES ints of LDS.
template <int WAVES>
__device__ __forceinline__ int block_exclusive(int x, int* red) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int inc = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(inc, d);
        if (lane >= d) inc += o;
    }
    if (lane == 63) red[w] = inc;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int q = 0; q < WAVES; ++q) before += q < w ? red[q] : 0;
    __syncthreads();
    return before + inc - x;
}

__host__ __device__ constexpr size_t radix_lds(int threads, int ipt, int bins) {
    return (size_t)threads * ipt * 4 + (size_t)bins * 8 + (size_t)(threads / 64) * bins * 2 + (threads / 64) * 4;
}

// Records (key, a, v): CSR_ROWS takes a from rowptr (the row of entry p), VAL says
// whether there is a v.  keys_out, a_out and v_out are written at the same places.
template <int THREADS, int IPT, bool CSR_ROWS, bool VAL>
__global__ __launch_bounds__(THREADS) void k_radix_scatter(int n, int shift, int db, int ntiles,
                                                           const int* __restrict__ keys_in,
                                                           const int* __restrict__ a_in,
                                                           const float* __restrict__ v_in, int M,
                                                           const int* __restrict__ rowptr,
                                                           const int* __restrict__ offs,
                                                           const int* __restrict__ totals, int* __restrict__ keys_out,
                                                           int* __restrict__ a_out, float* __restrict__ v_out) {
    constexpr int T = THREADS * IPT, WAVES = THREADS / 64, WT = 64 * IPT;
    constexpr int DPT = (1 << RADIX_MAX_BITS) / THREADS;  // most digits per thread
    extern __shared__ __align__(16) unsigned char smem[];
    const int bins = 1 << db, tile = xcd_tile(ntiles);
    if (tile < 0) return;
    int* stage = reinterpret_cast<int*>(smem);          // T
    int* start = stage + T;                             // bins: a digit's first place in the ordered tile
    int* goff = start + bins;                           // bins: where that place goes in the output, less the place
    uint16_t* wcnt = reinterpret_cast<uint16_t*>(goff + bins);  // WAVES × bins
    int* red = reinterpret_cast<int*>(wcnt + WAVES * bins);     // WAVES
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t tbase = (int64_t)tile * T;
    const int cnt = (int)min((int64_t)T, (int64_t)n - tbase);
    int key[IPT], a[IPT], pos[IPT];
    float v[IPT];
    // item r of a lane: w·WT + r·64 + lane, so a wave's items are consecutive
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int i = w * WT + r * 64 + lane;
        key[r] = i < cnt ? keys_in[tbase + i] : 0;
        if constexpr (!CSR_ROWS) a[r] = i < cnt ? a_in[tbase + i] : 0;
        if constexpr (VAL) v[r] = i < cnt ? v_in[tbase + i] : 0.0f;
    }
    for (int i = tid; i < WAVES * bins / 2; i += THREADS) reinterpret_cast<uint32_t*>(wcnt)[i] = 0u;
    if constexpr (CSR_ROWS) {
        const int p0 = (int)tbase, p1 = p0 + cnt;
        // rows of the tile's first and last entry
        if (w < 2) {
            const int r = min(rows_ending_by_wave(w ? p1 - 1 : p0, rowptr, M), M - 1);
            if (lane == 0) red[w] = r;
        }
        for (int i = tid; i < T; i += THREADS) stage[i] = 0;
        __syncthreads();
        const int r0 = uniform(red[0]), r1 = max(uniform(red[1]), r0);
        __syncthreads();
        if (r1 - r0 <= radix_mark_rows(THREADS) * T) {
            // every row that begins inside the tile marks its first entry (the last such
            // row where empty rows share it); a running maximum over the marks gives rows
            for (int rb = r0 + 1 + w * 64; rb <= r1; rb += THREADS) {
                const int r = rb + lane;
                const int b = r <= r1 ? rowptr[r] : INT_MAX;
                if (b >= p0 && b < p1) atomicMax(&stage[b - p0], r - r0);
            }
            __syncthreads();
            int run = 0;
#pragma unroll
            for (int r = 0; r < IPT; ++r) {  // the lane's row: the last mark at or before it
                const int m = stage[w * WT + r * 64 + lane];
                const uint64_t marks = __ballot(m != 0) & (~0ull >> (63 - lane));
                const int from = __shfl(m, marks ? 63 - __builtin_clzll(marks) : 0);
                a[r] = marks ? from : run;
                run = read_lane(a[r], 63);
            }
            if (lane == 0) red[w] = run;
            __syncthreads();
            int before = 0;
#pragma unroll
            for (int q = 0; q < WAVES; ++q) before = max(before, q < w ? red[q] : 0);
#pragma unroll
            for (int r = 0; r < IPT; ++r) a[r] = r0 + max(a[r], before);
        } else {
            // mostly empty rows: each record searches the last row that begins at or before it
#pragma unroll
            for (int r = 0; r < IPT; ++r) a[r] = r0;
            for (int step = 1 << (31 - __builtin_clz(r1 - r0)); step; step >>= 1) {
#pragma unroll
                for (int r = 0; r < IPT; ++r) {
                    const int i = min(w * WT + r * 64 + lane, cnt - 1);
                    if (step <= r1 - a[r] && rowptr[a[r] + step] <= p0 + i) a[r] += step;
                }
            }
        }
    }
    __syncthreads();
    // rank among the wave's records of the same digit, in order
    const uint64_t lt = (1ull << lane) - 1ull;
    uint16_t* wc = wcnt + w * bins;
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const bool valid = w * WT + r * 64 + lane < cnt;
        const int d = (key[r] >> shift) & (bins - 1);
        // the wave's records with this digit: bit by bit, the lanes that agree with ours
        const uint64_t all = __ballot(valid);
        uint32_t lo = (uint32_t)all, hi = (uint32_t)(all >> 32);
#pragma unroll
        for (int bit = 0; bit < RADIX_MAX_BITS; ++bit) {
            if (bit < db) {
                const int on = __builtin_amdgcn_sbfe(d, bit, 1);  // 0 or -1
                const uint64_t bal = __ballot(on != 0);
                lo &= ~((uint32_t)bal ^ (uint32_t)on);
                hi &= ~((uint32_t)(bal >> 32) ^ (uint32_t)on);
            }
        }
        const uint64_t m = ((uint64_t)hi << 32) | lo;
        const int before = valid ? wc[d] : 0;
        pos[r] = before + __popcll(m & lt);
        wave_sync_lds();
        if (valid && (m >> lane) == 1ull) wc[d] = (uint16_t)(before + __popcll(m));  // the digit's last record
        wave_sync_lds();
    }
    __syncthreads();
    {
        int c[DPT], g[DPT], cs = 0, gs = 0;
        const int dpt = (bins + THREADS - 1) / THREADS, d0 = tid * dpt;
#pragma unroll
        for (int i = 0; i < DPT; ++i) {
            c[i] = g[i] = 0;
            const int d = d0 + i;
            if (i < dpt && d < bins) {
                int run = 0;
#pragma unroll
                for (int q = 0; q < WAVES; ++q) {
                    const int x = wcnt[q * bins + d];
                    wcnt[q * bins + d] = (uint16_t)run;
                    run += x;
                }
                c[i] = run;
                g[i] = totals[d];
            }
            cs += c[i];
            gs += g[i];
        }
        int cb = block_exclusive<WAVES>(cs, red);
        int gb = block_exclusive<WAVES>(gs, red);
#pragma unroll
        for (int i = 0; i < DPT; ++i) {
            const int d = d0 + i;
            if (i < dpt && d < bins) {
                start[d] = cb;
                goff[d] = gb + offs[(int64_t)tile * bins + d] - cb;
            }
            cb += c[i];
            gb += g[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int d = (key[r] >> shift) & (bins - 1);
        pos[r] += start[d] + wc[d];
        if (w * WT + r * 64 + lane < cnt) stage[pos[r]] = key[r];
    }
    __syncthreads();
    int dst[IPT];  // of the ordered tile's place tid + r·THREADS
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int i = tid + r * THREADS;
        dst[r] = 0;
        if (i < cnt) {
            const int k = stage[i];
            dst[r] = goff[(k >> shift) & (bins - 1)] + i;
            keys_out[dst[r]] = k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < IPT; ++r)
        if (w * WT + r * 64 + lane < cnt) stage[pos[r]] = a[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int i = tid + r * THREADS;
        if (i < cnt) a_out[dst[r]] = stage[i];
    }
    if constexpr (VAL) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPT; ++r)
            if (w * WT + r * 64 + lane < cnt) stage[pos[r]] = __float_as_int(v[r]);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPT; ++r) {
            const int i = tid + r * THREADS;
            if (i < cnt) v_out[dst[r]] = __int_as_float(stage[i]);
        }
    }
}

// In-place exclusive scan of 2048-element chunks; sums[b] = chunk total.
__global__ __launch_bounds__(256) void k_scan_chunks(int64_t n, int* __restrict__ data, int* __restrict__ sums) {
    __shared__ int wsum[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t base = (int64_t)blockIdx.x * SCAN_CHUNK + (int64_t)tid * 8;
    int v[8], s = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v[i] = base + i < n ? data[base + i] : 0;
        s += v[i];
    }
    int inc = s;  // inclusive wave scan of per-thread sums
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(inc, d);
        if (lane >= d) inc += o;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    int wofs = 0;
    for (int q = 0; q < w; ++q) wofs += wsum[q];
    int run = wofs + inc - s;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if (base + i < n) data[base + i] = run;
        run += v[i];
    }
    if (tid == TPB - 1) sums[blockIdx.x] = run;
}

__global__ void k_scan_add(int64_t n, int* __restrict__ data, const int* __restrict__ sums) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) data[i] += sums[i / SCAN_CHUNK];
}

// ptr[c] = v for c in (lo, hi]; the whole wave calls it, and fills long gaps together
// (the keys of a power-law matrix leave gaps of thousands, and one lane's walk of
// such a gap outlasts the rest of the kernel).
__device__ __forceinline__ void fill_gap(int* __restrict__ ptr, int lo, int hi, int v) {
    const bool wide = hi - lo > 8;
    if (!wide)
        for (int c = lo + 1; c <= hi; ++c) ptr[c] = v;
    for (uint64_t m = __ballot(wide); m; m &= m - 1) {
        const int l = __builtin_ctzll(m);
        const int a = read_lane(lo, l), b = read_lane(hi, l), x = read_lane(v, l);
        for (int c = a + 1 + (int)__lane_id(); c <= b; c += 64) ptr[c] = x;
    }
}

// ptr[c] = first sorted position whose key is ≥ c, c = 0..K; four keys a thread.
__global__ __launch_bounds__(256) void k_colptr(int nnz, int K, const int* __restrict__ keys, int* __restrict__ ptr) {
    const int64_t p0 = 4 * (blockIdx.x * (int64_t)blockDim.x + threadIdx.x);
    int k[5];  // past the end no key changes, so no gap is filled
    k[0] = p0 > 0 ? (p0 <= nnz ? keys[p0 - 1] : K) : -1;
    if (p0 + 4 <= nnz) {  // keys come from the workspace, 256-byte aligned
        const int4 q = *reinterpret_cast<const int4*>(keys + p0);
        k[1] = q.x; k[2] = q.y; k[3] = q.z; k[4] = q.w;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) k[i + 1] = p0 + i < nnz ? keys[p0 + i] : K;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) fill_gap(ptr, k[i], k[i + 1], (int)(p0 + i));
}

// ------------------------------------------------ sorted triplets to CSR
// A run of equal (row, column) is one entry: its head is kept, unless zeros are
// dropped and the run's sum, in order, is zero.  k_coo_count counts a tile's
// kept heads; after a scan of the counts k_coo_emit places them and writes
// rowptr where the row changes.  (Runs of duplicates are short.)
constexpr int COO_IPT = 16, COO_TILE = TPB * COO_IPT;

// The wave's records base + 64·j + lane, j < COO_IPT: their rows and columns (row M,
// column -1 past the end), kept[j] = the lanes whose record heads a kept run, sum
// the runs' sums, and the row before the wave's first record (-1: none).
__device__ __forceinline__ int coo_runs(int64_t base, int n, int M, const int* __restrict__ srow,
                                        const int* __restrict__ scol, const float* __restrict__ sval, int drop_zeros,
                                        int (&row)[COO_IPT], int (&col)[COO_IPT], float (&sum)[COO_IPT],
                                        uint64_t (&kept)[COO_IPT]) {
    const int lane = threadIdx.x & 63;
    float v[COO_IPT];
#pragma unroll
    for (int j = 0; j < COO_IPT; ++j) {
        const int64_t p = base + j * 64 + lane;
        row[j] = p < n ? srow[p] : M;
        col[j] = p < n ? scol[p] : -1;
        v[j] = sval && p < n ? sval[p] : 0.0f;
    }
    const int64_t before = base - 1, after = base + 64 * COO_IPT;  // the wave's neighbours
    const int row_before = before < 0 ? -1 : before < n ? srow[before] : M;
    int pr = row_before, pc = before >= 0 && before < n ? scol[before] : -1;
    const int nr = after < n ? srow[after] : M, nc = after < n ? scol[after] : -1;
    uint64_t head[COO_IPT + 1];
#pragma unroll
    for (int j = 0; j < COO_IPT; ++j) {
        const int ur = __shfl_up(row[j], 1), uc = __shfl_up(col[j], 1);
        head[j] = __ballot((lane ? ur : pr) != row[j] || (lane ? uc : pc) != col[j]);
        pr = read_lane(row[j], 63);
        pc = read_lane(col[j], 63);
    }
    head[COO_IPT] = pr != nr || pc != nc ? 1u : 0u;
#pragma unroll
    for (int j = 0; j < COO_IPT; ++j) {
        const int64_t p = base + j * 64 + lane;
        bool keep = p < n && ((head[j] >> lane) & 1);
        sum[j] = v[j];
        if (sval && (~head[j] != 0ull || !(head[j + 1] & 1))) {  // some run has several records (uniform)
            // lane's run goes on for `len` records here; a run that reaches lane 63 may go on in the next
            const uint64_t later = lane < 63 ? head[j] >> (lane + 1) : 0ull;
            const int len = later ? __builtin_ctzll(later) : 63 - lane;
            for (int k = 1; __ballot(keep && k <= len); ++k) {
                const float t = __shfl_down(v[j], k);
                if (k <= len) sum[j] += t;
            }
            const bool goes_on = keep && !later && !(head[j + 1] & 1);
            if (__ballot(goes_on)) {
                const uint64_t h = j + 1 < COO_IPT ? head[j + 1] : 0ull;
                if (h) {
                    for (int k = 0; k < __builtin_ctzll(h); ++k) {
                        const float t = read_lane(v[j + 1 < COO_IPT ? j + 1 : j], k);
                        if (goes_on) sum[j] += t;
                    }
                } else if (goes_on) {
                    for (int64_t q = base + (j + 1) * 64; q < n && srow[q] == row[j] && scol[q] == col[j]; ++q)
                        sum[j] += sval[q];
                }
            }
        }
        if (drop_zeros && sval) keep = keep && sum[j] != 0.0f;
        kept[j] = __ballot(keep);
    }
    return row_before;
}

__global__ __launch_bounds__(TPB) void k_coo_count(int n, int M, const int* __restrict__ srow,
                                                   const int* __restrict__ scol, const float* __restrict__ sval,
                                                   int drop_zeros, int* __restrict__ cnt) {
    __shared__ int red[TPB / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int row[COO_IPT], col[COO_IPT];
    float sum[COO_IPT];
    uint64_t kept[COO_IPT];
    coo_runs((int64_t)blockIdx.x * COO_TILE + w * (64 * COO_IPT), n, M, srow, scol, drop_zeros ? sval : nullptr,
             drop_zeros, row, col, sum, kept);
    int have = 0;
#pragma unroll
    for (int j = 0; j < COO_IPT; ++j) have += __popcll(kept[j]);
    if (lane == 0) red[w] = have;
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int q = 0; q < TPB / 64; ++q) s += red[q];
        cnt[blockIdx.x] = s;
    }
}

__global__ void k_coo_empty(int M, int* __restrict__ rowptr, int* __restrict__ n_out) {
    const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (r <= M) rowptr[r] = 0;
    if (r == 0) *n_out = 0;
}

__global__ void k_clear_int(int* p) { *p = 0; }

// first[b]: kept entries before tile b.  Nothing is written when *bad.
__global__ __launch_bounds__(TPB) void k_coo_emit(int n, int M, const int* __restrict__ srow,
                                                  const int* __restrict__ scol, const float* __restrict__ sval,
                                                  int drop_zeros, const int* __restrict__ first,
                                                  const int* __restrict__ bad, int* __restrict__ rowptr,
                                                  int* __restrict__ colind, float* __restrict__ val,
                                                  int* __restrict__ n_out) {
    __shared__ int red[TPB / 64];
    if (*bad) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t lt = (1ull << lane) - 1ull;
    const int64_t base = (int64_t)blockIdx.x * COO_TILE + w * (64 * COO_IPT);
    int row[COO_IPT], col[COO_IPT];
    float sum[COO_IPT];
    uint64_t kept[COO_IPT];
    int rbefore = coo_runs(base, n, M, srow, scol, sval, drop_zeros, row, col, sum, kept);
    int have = 0;
#pragma unroll
    for (int j = 0; j < COO_IPT; ++j) have += __popcll(kept[j]);
    if (lane == 0) red[w] = have;
    __syncthreads();
    int at = first[blockIdx.x];
    for (int q = 0; q < w; ++q) at += red[q];
#pragma unroll
    for (int j = 0; j < COO_IPT; ++j) {
        const int64_t p = base + j * 64 + lane;
        const int d = at + __popcll(kept[j] & lt);
        if ((kept[j] >> lane) & 1) {
            colind[d] = col[j];
            if (sval) val[d] = sum[j];
        }
        // rows up to this record's begin here; past the last record, the rest do
        const int ur = __shfl_up(row[j], 1);
        fill_gap(rowptr, lane ? ur : rbefore, row[j], d);
        rbefore = read_lane(row[j], 63);
        at += __popcll(kept[j]);
        if (p == n - 1) *n_out = d + (int)((kept[j] >> lane) & 1);
    }
    // the last record ends the last tile's last wave: nothing past it there
    if (base + 64 * COO_IPT == n) fill_gap(rowptr, lane ? M : rbefore, M, at);
}

int64_t scan_ws_ints(int64_t n) {
    int64_t total = 0;
    while (n > 1) {
        n = (n + SCAN_CHUNK - 1) / SCAN_CHUNK;
        total += n;
    }
    return total + 1;
}

void exclusive_scan(int64_t n, int* data, int* ws, hipStream_t s) {
    const int64_t nb = (n + SCAN_CHUNK - 1) / SCAN_CHUNK;
    hipLaunchKernelGGL(k_scan_chunks, dim3((unsigned)nb), dim3(TPB), 0, s, n, data, ws);
    if (nb > 1) {
        exclusive_scan(nb, ws, ws + nb, s);
        hipLaunchKernelGGL(k_scan_add, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, data, ws);
    }
}

// A sort of n records by keys in [0, range): `passes` passes of `db` bits over
// tiles of `tile` records.
struct RadixPlan {
    int db, passes, tile, ntiles;
};
// Tiles of 512 threads × 8 records: longer runs per digit than shorter tiles, yet two
// workgroups a CU (97 VGPRs), whose phases overlap (1M R-MAT transpose and 6M triplets
// to CSR, when measured: 2048 records 506 and 401 us, 4096 393 and 373, 8192 430 and 407, 16,384 525
// and 501; 512 threads against 256 and 1024: 393, 457, 525 us).  With fewer records
// than RADIX_BIG some CUs would have no such tile, so they are 2,048.
constexpr int RADIX_BIG = 2 << 20;
constexpr int RADIX_BIG_TILE = 4096, RADIX_BIG_THREADS = 512;

RadixPlan radix_plan(int n, int range) {
    int bits = 0;
    while (bits < 31 && ((int64_t)1 << bits) < range) ++bits;
    RadixPlan p;
    p.passes = bits > 0 ? (bits + RADIX_MAX_BITS - 1) / RADIX_MAX_BITS : 1;
    p.db = (bits + p.passes - 1) / p.passes;
    if (p.db < RADIX_MIN_BITS) p.db = RADIX_MIN_BITS;
    p.tile = n >= RADIX_BIG ? RADIX_BIG_TILE : 2048;
    p.ntiles = (int)(((int64_t)n + p.tile - 1) / p.tile);
    return p;
}
// ints of histogram workspace: the tiles' counts and the digits' totals
size_t radix_hist_ints(const RadixPlan& p) { return ((size_t)p.ntiles + 1) << p.db; }

struct Records {
    const int* k;
    const int* a;
    const float* v;
};

template <int THREADS, int IPT>
void radix_pass(const RadixPlan& p, int pass, int n, const Records& in, bool csr_rows, int M, const int* rowptr,
                int* hist, int* ko, int* ao, float* vo, const int* other, int krange, int orange, int* bad,
                hipStream_t s) {
    const int bins = 1 << p.db, shift = p.db * pass;
    int* totals = hist + (size_t)p.ntiles * bins;
    const dim3 grid(xcd_grid(p.ntiles));
    const size_t lds = radix_lds(THREADS, IPT, bins);
    hipLaunchKernelGGL((k_radix_hist<THREADS, IPT>), grid, dim3(THREADS), 0, s, n, shift, p.db, p.ntiles, in.k, hist,
                       other, krange, orange, bad);
    hipLaunchKernelGGL(k_radix_scan, dim3(bins / 16), dim3(1024), 0, s, p.ntiles, bins, hist, totals);
#define ARMSP_RADIX(CR, VA)                                                                                        \
    hipLaunchKernelGGL((k_radix_scatter<THREADS, IPT, CR, VA>), grid, dim3(THREADS), lds, s, n, shift, p.db, p.ntiles, \
                       in.k, in.a, in.v, M, rowptr, hist, totals, ko, ao, vo)
    if (csr_rows) {
        if (in.v) ARMSP_RADIX(true, true); else ARMSP_RADIX(true, false);
    } else {
        if (in.v) ARMSP_RADIX(false, true); else ARMSP_RADIX(false, false);
    }
#undef ARMSP_RADIX
}

// Stable sort of the records by key.  With rowptr, a is the row of each entry of a
// CSR matrix.  The passes alternate between buf[0] and buf[1] (k, a, v each; `from`:
// the one to write first).  Returns the sorted records.  other, krange, orange, bad:
// the range check of k_radix_hist, done by the first pass.
Records radix_sort(const RadixPlan& p, int n, Records in, int M, const int* rowptr, int* hist, int* const (*buf)[3],
                   int from, const int* other, int krange, int orange, int* bad, hipStream_t s) {
    for (int pass = 0; pass < p.passes; ++pass) {
        int* const* o = buf[(from + pass) & 1];
        int* ao = o[1];
        float* vo = reinterpret_cast<float*>(o[2]);
        const bool csr = rowptr && pass == 0;
        const int* chk = pass == 0 ? other : nullptr;
        if (p.tile == RADIX_BIG_TILE)
            radix_pass<RADIX_BIG_THREADS, RADIX_BIG_TILE / RADIX_BIG_THREADS>(p, pass, n, in, csr, M, rowptr, hist, o[0], ao, vo, chk, krange, orange, bad, s);
        else
            radix_pass<256, 8>(p, pass, n, in, csr, M, rowptr, hist, o[0], ao, vo, chk, krange, orange, bad, s);
        in = Records{o[0], ao, in.v ? vo : nullptr};
    }
    return in;
}

// ------------------------------------------------ column blocks of a CSR matrix
// A CSR matrix split into nb blocks of columns [x·W, (x+1)·W), each a CSR matrix
// of its own over all M rows with the row's entries in their order.  Block x of
// row r is a run of the row's entries (columns increase along a row), found by a
// binary search per block boundary: one wave per row, lane x searching boundary
// x.  The (block, row) counts in block-major order are scanned once, which places
// every run; a second pass copies the runs with the row's wave.

// entries of row [a, e) with column < c (a binary search)
__device__ __forceinline__ int cols_below(const int* __restrict__ colind, int a, int e, int c) {
    int lo = a, hi = e;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (colind[mid] < c)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// cnt[x·M + r] = entries of row r in block x; cnt[nb·M] = 0 (the scan total)
__global__ __launch_bounds__(256) void k_split_count(int M, int nb, int W, const int* __restrict__ rowptr,
                                                     const int* __restrict__ colind, int* __restrict__ cnt) {
    const int lane = threadIdx.x & 63;
    const int r = uniform((int)(blockIdx.x * 4u + (threadIdx.x >> 6)));
    if (r == M && lane == 0) cnt[(int64_t)nb * M] = 0;
    if (r >= M) return;
    const int a = rowptr[r], e = rowptr[r + 1];
    const int sx = lane <= nb ? (lane == 0 ? a : (lane == nb ? e : cols_below(colind, a, e, lane * W))) : e;
    const int nx = __shfl(sx, lane + 1 <= nb ? lane + 1 : nb);
    if (lane < nb) cnt[(int64_t)lane * M + r] = nx - sx;
}

// out_rowptr[x·(M+1) + r] = pos[x·M + r] − pos[x·M], r = 0..M
__global__ void k_split_rowptr(int M, int nb, const int* __restrict__ pos, int* __restrict__ out_rowptr) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= (int64_t)nb * (M + 1)) return;
    const int x = (int)(i / (M + 1)), r = (int)(i - (int64_t)x * (M + 1));
    const int64_t b = (int64_t)x * M;
    out_rowptr[i] = pos[b + r] - pos[b];
}

// base[x] = pos[x·M], x = 0..nb (the blocks' first entries; base[nb] = nnz)
__global__ void k_split_base(int M, int nb, const int* __restrict__ pos, int* __restrict__ base) {
    const int x = threadIdx.x;
    if (x <= nb) base[x] = pos[(int64_t)x * M];
}

__global__ __launch_bounds__(256) void k_split_scatter(int M, int nb, int W, const int* __restrict__ rowptr,
                                                       const int* __restrict__ colind, const float* __restrict__ val,
                                                       const int* __restrict__ pos, int* __restrict__ out_colind,
                                                       float* __restrict__ out_val) {
    const int lane = threadIdx.x & 63;
    const int r = uniform((int)(blockIdx.x * 4u + (threadIdx.x >> 6)));
    if (r >= M) return;
    const int a = rowptr[r], e = rowptr[r + 1];
    const int sx = lane <= nb ? (lane == 0 ? a : (lane == nb ? e : cols_below(colind, a, e, lane * W))) : e;
    for (int x = 0; x < nb; ++x) {
        const int s0 = __shfl(sx, x), s1 = __shfl(sx, x + 1);
        const int64_t d = pos[(int64_t)x * M + r];
        for (int p = s0 + lane; p < s1; p += 64) {
            out_colind[d + (p - s0)] = colind[p];
            if (out_val) out_val[d + (p - s0)] = val ? val[p] : 1.0f;
        }
    }
}

// err bit 2: a column out of [0, K) or not above the previous one in its row
// (start[p] = 1 where a non-empty row begins, from k_vcsr_rows)
__global__ void k_cols_increasing(int nnz, int K, const int* __restrict__ colind, const uint8_t* __restrict__ start,
                                  int* __restrict__ err) {
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= nnz) return;
    const int c = colind[p];
    const bool first = p == 0 || start[p] != 0;
    if (c < 0 || c >= K || (!first && colind[p - 1] >= c)) atomicOr(err, 2);
}

// ------------------------------------------------ CSR → vector-aware CSR
// toVectorAwareCSR (SpMV.cpp:15-38) on the device, from CSR instead of a dense
// matrix.  A row's aligned block of columns [4b, 4b+4) is stored iff one of the
// row's values in it triggers (v != 0, or |v| > threshold when threshold > 0:
// numaAware/numaAwareSpMV.cpp:48), as four slots holding the row's values (0
// where absent) with column indices 4b..4b+3.  The entry that opens a block (the
// row's first entry in it) decides it alone, reading the at most three entries
// after it (columns strictly increase within a row, so a block holds at most
// four).  An exclusive scan over those decisions gives every stored block its
// place, and the blocked rowptr is read off the scan at the row starts.

// start[p] = 1 where a non-empty row begins; err bit 0: malformed rowptr.
__global__ void k_vcsr_rows(int M, int nnz, const int* __restrict__ rowptr, uint8_t* __restrict__ start,
                            int* __restrict__ err) {
    const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (r >= M) return;
    const int a = rowptr[r], b = rowptr[r + 1];
    if ((r == 0 && a != 0) || (r == M - 1 && b != nnz) || a < 0 || b < a || b > nnz) {
        atomicOr(err, 1);
        return;
    }
    if (a < b) start[a] = 1;
}

__global__ void k_vcsr_clear(int64_t n, uint8_t* __restrict__ start, int* __restrict__ err) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) start[i] = 0;
    if (i == 0) *err = 0;
}

__device__ __forceinline__ bool vcsr_trig(float v, float threshold) {
    return threshold > 0.0f ? fabsf(v) > threshold : v != 0.0f;
}

// keep[p] = 1 iff entry p opens a stored block, keep[nnz] = 0 (the scan then
// leaves the block count there).  err bit 1: a column out of [0, K) or a row
// whose columns do not strictly increase.
__global__ void k_vcsr_mark(int nnz, int K, const int* __restrict__ colind, const float* __restrict__ val,
                            float threshold, const uint8_t* __restrict__ start, int* __restrict__ keep,
                            int* __restrict__ err) {
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p > nnz) return;
    if (p == nnz) {
        keep[p] = 0;
        return;
    }
    const int c = colind[p];
    const bool first = p == 0 || start[p] != 0;
    const int cp = first ? -1 : colind[p - 1];
    if (c < 0 || c >= K || (!first && cp >= c)) atomicOr(err, 2);
    const bool opens = first || (cp >> 2) != (c >> 2);
    bool on = opens && vcsr_trig(val ? val[p] : 1.0f, threshold);
    for (int d = 1; opens && !on && d <= 3; ++d) {
        const int64_t q = p + d;
        if (q >= nnz || start[q] || (colind[q] >> 2) != (c >> 2)) break;
        on = vcsr_trig(val ? val[q] : 1.0f, threshold);
    }
    keep[p] = on ? 1 : 0;
}

// out_rowptr[r] = 4 · (stored blocks before row r), r = 0..M (with no rows, the one
// entry is 0 and rowptr is not read).
__global__ void k_vcsr_rowptr(int M, const int* __restrict__ rowptr, const int* __restrict__ pos,
                              int* __restrict__ out_rowptr) {
    const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (r > M) return;
    out_rowptr[r] = M == 0 ? 0 : 4 * pos[rowptr[r]];
}

// The opening entry of every stored block writes its four slots.
__global__ void k_vcsr_fill(int nnz, const int* __restrict__ colind, const float* __restrict__ val,
                            const uint8_t* __restrict__ start, const int* __restrict__ pos,
                            int* __restrict__ out_colind, float* __restrict__ out_val) {
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= nnz) return;
    const int b = pos[p];
    if (pos[p + 1] == b) return;
    const int c = colind[p];
    const int c0 = (c >> 2) * 4;
    float slot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    slot[c & 3] = val ? val[p] : 1.0f;
    for (int d = 1; d <= 3; ++d) {
        const int64_t q = p + d;
        if (q >= nnz || start[q] || (colind[q] >> 2) != (c >> 2)) break;
        slot[colind[q] & 3] = val ? val[q] : 1.0f;
    }
    const int64_t o = 4 * (int64_t)b;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        out_colind[o + t] = c0 + t;
        out_val[o + t] = slot[t];
    }
}

}  // namespace
}  // namespace armsp

extern "C" int armsp_csr_transpose(int M, int K, int nnz, const int* rowptr, const int* colind, const float* val,
                                   int* colptr, int* rowind, float* valT, void* stream) {
    using namespace armsp;
    if (M < 0 || K < 0 || nnz < 0) return ARMSP_ERROR_INVALID_VALUE;
    if (!colptr || (nnz > 0 && (!rowptr || !colind || !rowind))) return ARMSP_ERROR_INVALID_VALUE;
    if ((val == nullptr) != (valT == nullptr)) return ARMSP_ERROR_INVALID_VALUE;
    hipStream_t s = as_stream(stream);
    TimedLaunch t("transpose", s);
    if (nnz == 0 || M == 0) {
        hipLaunchKernelGGL(k_colptr, dim3(1), dim3(64), 0, s, 0, K, (const int*)nullptr, colptr);
        ARMSP_LAUNCHED();
        t.stop();
        return ARMSP_SUCCESS;
    }
    const RadixPlan plan = radix_plan(nnz, K);
    const size_t n4 = ((size_t)nnz * 4 + 255) & ~(size_t)255;
    const size_t h4 = (radix_hist_ints(plan) * 4 + 255) & ~(size_t)255;
    void* ws = nullptr;
    int st = ws_alloc(&ws, (plan.passes == 1 ? 1 : val ? 4 : 3) * n4 + h4, s);
    if (st) return st;
    char* p = static_cast<char*>(ws);
    int* hist = reinterpret_cast<int*>(p);
    auto arr = [&](int i) { return reinterpret_cast<int*>(p + h4 + i * n4); };
    // the last pass, and every second one before it, writes rows and values to the
    // outputs: what a pass reads is never what it writes
    int* const buf[2][3] = {{arr(0), rowind, reinterpret_cast<int*>(valT)}, {arr(1), arr(2), arr(3)}};
    const Records sorted = radix_sort(plan, nnz, Records{colind, nullptr, val}, M, rowptr, hist, buf,
                                      (plan.passes - 1) & 1, nullptr, 0, 0, nullptr, s);
    hipLaunchKernelGGL(k_colptr, dim3((unsigned)(((int64_t)nnz / 4 + 1 + 255) / 256)), dim3(256), 0, s, nnz, K,
                       sorted.k, colptr);
    hipError_t e = hipGetLastError();
    ws_free(ws, s);
    if (e != hipSuccess) return hip_fail(e);
    t.stop();
    return ARMSP_SUCCESS;
}

extern "C" int armsp_coo_to_csr(int M, int K, int nnz, const int* rows, const int* cols, const float* vals,
                                int drop_zeros, int* rowptr, int* colind, float* val, int* nnz_out, void* stream) {
    using namespace armsp;
    if (M < 0 || K < 0 || nnz < 0) return ARMSP_ERROR_INVALID_VALUE;
    if (!rowptr || !nnz_out || (nnz > 0 && (!rows || !cols || !colind))) return ARMSP_ERROR_INVALID_VALUE;
    if (nnz > 0 && (vals == nullptr) != (val == nullptr)) return ARMSP_ERROR_INVALID_VALUE;
    if (nnz > 0 && (M == 0 || K == 0)) return ARMSP_ERROR_INVALID_VALUE;
    hipStream_t s = as_stream(stream);
    TimedLaunch t("coo_to_csr", s);
    if (nnz == 0) {
        hipLaunchKernelGGL(k_coo_empty, dim3((unsigned)(((int64_t)M + 1 + 255) / 256)), dim3(256), 0, s, M, rowptr,
                           nnz_out);
        ARMSP_LAUNCHED();
        t.stop();
        return ARMSP_SUCCESS;
    }
    const RadixPlan pc = radix_plan(nnz, K), pr = radix_plan(nnz, M);
    const size_t hc = radix_hist_ints(pc), hr = radix_hist_ints(pr);
    const int ctiles = (int)(((int64_t)nnz + COO_TILE - 1) / COO_TILE);
    const size_t n4 = ((size_t)nnz * 4 + 255) & ~(size_t)255;
    const size_t h4 = ((hc > hr ? hc : hr) * 4 + 255) & ~(size_t)255;
    const size_t c4 = ((size_t)ctiles * 4 + 255) & ~(size_t)255;
    const size_t s4 = ((size_t)scan_ws_ints(ctiles) * 4 + 255) & ~(size_t)255;
    void* ws = nullptr;
    int st = ws_alloc(&ws, 6 * n4 + h4 + c4 + s4 + 256, s);
    if (st) return st;
    char* p = static_cast<char*>(ws);
    auto arr = [&](int i) { return reinterpret_cast<int*>(p + i * n4); };
    int* hist = reinterpret_cast<int*>(p + 6 * n4);
    int* cnt = reinterpret_cast<int*>(p + 6 * n4 + h4);
    int* scanws = reinterpret_cast<int*>(p + 6 * n4 + h4 + c4);
    int* bad = reinterpret_cast<int*>(p + 6 * n4 + h4 + c4 + s4);
    int* const buf[2][3] = {{arr(0), arr(1), arr(2)}, {arr(3), arr(4), arr(5)}};
    // by column, then (stably) by row: (row, column) order, duplicates in input order.
    // The first histogram also checks every index; the sort masks its digits, so it
    // stays inside its buffers whatever they are, and k_coo_emit writes nothing when
    // one is out of range: a single wait at the end serves the check.
    hipLaunchKernelGGL(k_clear_int, dim3(1), dim3(1), 0, s, bad);
    const Records bc = radix_sort(pc, nnz, Records{cols, rows, vals}, 0, nullptr, hist, buf, 0, rows, K, M,
                                  bad, s);
    const Records br = radix_sort(pr, nnz, Records{bc.a, bc.k, bc.v}, 0, nullptr, hist, buf, pc.passes & 1,
                                  nullptr, 0, 0, nullptr, s);
    hipLaunchKernelGGL(k_coo_count, dim3((unsigned)ctiles), dim3(TPB), 0, s, nnz, M, br.k, br.a, br.v,
                       drop_zeros, cnt);
    exclusive_scan(ctiles, cnt, scanws, s);
    hipLaunchKernelGGL(k_coo_emit, dim3((unsigned)ctiles), dim3(TPB), 0, s, nnz, M, br.k, br.a, br.v, drop_zeros,
                       (const int*)cnt, (const int*)bad, rowptr, colind, val, nnz_out);
    int bad_h = 0;
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(&bad_h, bad, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    ws_free(ws, s);
    if (e != hipSuccess) return hip_fail(e);
    if (bad_h) return ARMSP_ERROR_INVALID_VALUE;
    t.stop();
    return ARMSP_SUCCESS;
}

extern "C" int armsp_csr_to_vcsr_device(int M, int K, int nnz, const int* rowptr, const int* colind,
                                        const float* val, float threshold, int* out_rowptr, int* out_colind,
                                        float* out_val, int64_t capacity, int64_t* padded, void* stream) {
    using namespace armsp;
    if (M < 0 || K < 0 || nnz < 0 || !padded || !out_rowptr || !rowptr) return ARMSP_ERROR_INVALID_VALUE;
    if (nnz > 0 && !colind) return ARMSP_ERROR_INVALID_VALUE;
    if ((out_colind == nullptr) != (out_val == nullptr)) return ARMSP_ERROR_INVALID_VALUE;
    if (M == 0 && nnz > 0) return ARMSP_ERROR_INVALID_VALUE;
    if (nnz > INT_MAX - 2) return ARMSP_ERROR_NOT_SUPPORTED;
    hipStream_t s = as_stream(stream);
    TimedLaunch t("csr_to_vcsr", s);
    const int64_t n1 = (int64_t)nnz + 1;  // scanned entries: nnz decisions and the total
    const size_t p4 = ((size_t)(n1 + 1) * 4 + 255) & ~(size_t)255;
    const size_t s4 = ((size_t)scan_ws_ints(n1) * 4 + 255) & ~(size_t)255;
    const size_t b1 = ((size_t)(nnz > 0 ? nnz : 1) + 255) & ~(size_t)255;
    void* ws = nullptr;
    int st = ws_alloc(&ws, p4 + s4 + b1, s);
    if (st) return st;
    char* w = static_cast<char*>(ws);
    int* pos = reinterpret_cast<int*>(w);
    int* err = pos + n1;  // one int past the scanned range
    int* scanws = reinterpret_cast<int*>(w + p4);
    uint8_t* start = reinterpret_cast<uint8_t*>(w + p4 + s4);
    auto fail = [&](int code) {
        ws_free(ws, s);
        return code;
    };
    const unsigned gs = (unsigned)(((int64_t)(nnz > 0 ? nnz : 1) + 255) / 256);
    hipLaunchKernelGGL(k_vcsr_clear, dim3(gs), dim3(256), 0, s, (int64_t)nnz, start, err);
    if (M > 0)
        hipLaunchKernelGGL(k_vcsr_rows, dim3((unsigned)(((int64_t)M + 255) / 256)), dim3(256), 0, s, M, nnz, rowptr,
                           start, err);
    hipLaunchKernelGGL(k_vcsr_mark, dim3((unsigned)((n1 + 255) / 256)), dim3(256), 0, s, nnz, K, colind, val,
                       threshold, start, pos, err);
    exclusive_scan(n1, pos, scanws, s);
    int h[2] = {0, 0};  // the block count and the error bits
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(h, pos + nnz, sizeof(h), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail(hip_fail(e));
    if (h[1]) return fail(ARMSP_ERROR_INVALID_VALUE);
    if (4 * (int64_t)h[0] > INT_MAX) return fail(ARMSP_ERROR_NOT_SUPPORTED);
    *padded = 4 * (int64_t)h[0];
    hipLaunchKernelGGL(k_vcsr_rowptr, dim3((unsigned)(((int64_t)M + 1 + 255) / 256)), dim3(256), 0, s, M, rowptr,
                       (const int*)pos, out_rowptr);
    if (out_colind) {
        if (capacity < *padded) return fail(ARMSP_ERROR_INVALID_VALUE);
        if (nnz > 0)
            hipLaunchKernelGGL(k_vcsr_fill, dim3(gs), dim3(256), 0, s, nnz, colind, val, (const uint8_t*)start,
                               (const int*)pos, out_colind, out_val);
    }
    e = hipGetLastError();
    ws_free(ws, s);
    if (e != hipSuccess) return hip_fail(e);
    t.stop();
    return ARMSP_SUCCESS;
}

extern "C" int armsp_csr_column_split(int M, int K, int nnz, const int* rowptr, const int* colind, const float* val,
                                      int nblocks, int* out_rowptr, int* out_colind, float* out_val,
                                      int64_t* block_start, void* stream) {
    using namespace armsp;
    if (M < 0 || K < 0 || nnz < 0 || nblocks < 1 || nblocks > 63) return ARMSP_ERROR_INVALID_VALUE;
    if (!rowptr || !out_rowptr || !block_start || (nnz > 0 && (!colind || !out_colind))) return ARMSP_ERROR_INVALID_VALUE;
    if (val && !out_val) return ARMSP_ERROR_INVALID_VALUE;
    if (M == 0 && nnz > 0) return ARMSP_ERROR_INVALID_VALUE;
    if ((int64_t)nblocks * M + 1 > INT_MAX) return ARMSP_ERROR_NOT_SUPPORTED;
    hipStream_t s = as_stream(stream);
    TimedLaunch t("csr_column_split", s);
    const int W = K > 0 ? (K + nblocks - 1) / nblocks : 1;
    const int64_t ncnt = (int64_t)nblocks * M + 1;  // (block, row) counts and the total
    const size_t c4 = ((size_t)ncnt * 4 + 255) & ~(size_t)255;
    const size_t s4 = ((size_t)scan_ws_ints(ncnt) * 4 + 255) & ~(size_t)255;
    const size_t b1 = ((size_t)(nnz > 0 ? nnz : 1) + 255) & ~(size_t)255;
    void* ws = nullptr;
    int st = ws_alloc(&ws, c4 + s4 + b1 + 512, s);
    if (st) return st;
    char* w = static_cast<char*>(ws);
    int* pos = reinterpret_cast<int*>(w);
    int* scanws = reinterpret_cast<int*>(w + c4);
    uint8_t* start = reinterpret_cast<uint8_t*>(w + c4 + s4);
    int* err = reinterpret_cast<int*>(w + c4 + s4 + b1);
    int* base = err + 1;  // nblocks + 1 ints
    auto fail = [&](int code) {
        ws_free(ws, s);
        return code;
    };
    // canonical CSR: rowptr from 0 to nnz, non-decreasing; columns in range and increasing along a row
    const unsigned gs = (unsigned)(((int64_t)(nnz > 0 ? nnz : 1) + 255) / 256);
    hipLaunchKernelGGL(k_vcsr_clear, dim3(gs), dim3(256), 0, s, (int64_t)nnz, start, err);
    if (M > 0)
        hipLaunchKernelGGL(k_vcsr_rows, dim3((unsigned)(((int64_t)M + 255) / 256)), dim3(256), 0, s, M, nnz, rowptr,
                           start, err);
    if (nnz > 0) hipLaunchKernelGGL(k_cols_increasing, dim3(gs), dim3(256), 0, s, nnz, K, colind, start, err);
    int h = 0;
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(&h, err, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail(hip_fail(e));
    if (h) return fail(ARMSP_ERROR_INVALID_VALUE);
    const unsigned gr = (unsigned)(((int64_t)M + 1 + 3) / 4);  // a wave per row, and one for the total
    hipLaunchKernelGGL(k_split_count, dim3(gr), dim3(256), 0, s, M, nblocks, W, rowptr, colind, pos);
    exclusive_scan(ncnt, pos, scanws, s);
    hipLaunchKernelGGL(k_split_rowptr, dim3((unsigned)(((int64_t)nblocks * (M + 1) + 255) / 256)), dim3(256), 0, s, M,
                       nblocks, (const int*)pos, out_rowptr);
    if (nnz > 0)
        hipLaunchKernelGGL(k_split_scatter, dim3((unsigned)(((int64_t)M + 3) / 4)), dim3(256), 0, s, M, nblocks, W,
                           rowptr, colind, val, (const int*)pos, out_colind, out_val);
    hipLaunchKernelGGL(k_split_base, dim3(1), dim3(64), 0, s, M, nblocks, (const int*)pos, base);
    int hb[64];
    e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(hb, base, sizeof(int) * (size_t)(nblocks + 1), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    ws_free(ws, s);
    if (e != hipSuccess) return hip_fail(e);
    for (int x = 0; x <= nblocks; ++x) block_start[x] = hb[x];
    t.stop();
    return ARMSP_SUCCESS;
}
