// CSR SpMV for gfx950.
//
// Reference: sparse_dense_vector (SpMV.cpp:155-179) runs an OpenMP loop over
// rows of a zero-padded 1×4-blocked CSR; numaAware/numaAwareSpMV.cpp:102-125
// splits the rows into four NUMA quarters.  Here:
//  ROW   — G lanes per row, lanes stride the row, butterfly reduction.
//  MERGE — merge-path over (row ends, nonzeros): each wave owns 64·IPT items,
//          stages row ends and products val·x in LDS, every lane walks IPT
//          consecutive items, a wave-level segmented scan joins rows cut
//          between lanes, and a carry per wave is added by a fixup kernel.
//  VCSR  — the reference's blocked format with its exact summation order:
//          every row's four partial sums s0..s3 are each added in block order
//          (by four lanes of a short row, sixteen of a medium one, a workgroup
//          for a long one) and the row total is (s0+s2)+(s1+s3), as
//          vadd/vpadd compute it.
#include <algorithm>
#include <climits>
#include <cstdlib>

#include "common.hpp"

namespace armsp {
namespace {

template <int G>
__global__ __launch_bounds__(256) void k_spmv_row(int M, const int* __restrict__ rowptr, const int* __restrict__ colind,
                                                  const float* __restrict__ val, const float* __restrict__ x,
                                                  float* __restrict__ y, int flags) {
    const int lane = threadIdx.x & (G - 1);
    const int row = (int)((blockIdx.x * 256u + threadIdx.x) / G);
    if (row >= M) return;
    const int beg = rowptr[row], end = rowptr[row + 1];
    float s = 0.0f;
    for (int p = beg + lane; p < end; p += G) s = fmaf(val ? val[p] : 1.0f, x[colind[p]], s);
#pragma unroll
    for (int m = G / 2; m >= 1; m >>= 1) s += __shfl_xor(s, m, G);
    if (lane == 0) y[row] = (flags & ARMSP_ACCUMULATE) ? y[row] + s : s;
}

template <int IPT>
__global__ __launch_bounds__(256) void k_spmv_merge(int M, int nnz, const int* __restrict__ rowptr,
                                                    const int* __restrict__ colind, const float* __restrict__ val,
                                                    const float* __restrict__ x, float* __restrict__ y, int flags,
                                                    const int* __restrict__ part, int* __restrict__ carry_row,
                                                    float* __restrict__ carry_val) {
    constexpr int TILE = 64 * IPT;
    __shared__ int s_re[4][TILE + 1];
    __shared__ float s_prod[4][TILE];
    __shared__ float s_out[4][TILE];
    const int lane = threadIdx.x & 63;
    const int wid = threadIdx.x >> 6;
    const int wave = uniform((int)(blockIdx.x * 4u + wid));
    const int64_t total = (int64_t)M + nnz;
    const int64_t d0l = (int64_t)wave * TILE;
    if (d0l >= total) return;
    const int d0 = (int)d0l;
    const int d1 = (int)(d0l + TILE < total ? d0l + TILE : total);
    int i0, i1;
    chunk_rows(part, wave, d0, d1, rowptr, M, nnz, i0, i1);
    const int j0 = d0 - i0, j1 = d1 - i1;
    const int nrows = i1 - i0, nz = j1 - j0;
    int* re = s_re[wid];
    float* prod = s_prod[wid];
    float* out = s_out[wid];
    for (int k = lane; k < nrows; k += 64) re[k] = rowptr[i0 + k + 1];
    {
        // nonzero k = lane + 64·q: all IPT index loads, then all IPT gathers of x, in flight together
        int cs[IPT];
        float vs[IPT], xs[IPT];
#pragma unroll
        for (int q = 0; q < IPT; ++q) {
            const int k = lane + 64 * q;
            cs[q] = 0;
            vs[q] = 0.0f;
            if (k < nz) {
                cs[q] = __builtin_nontemporal_load(colind + j0 + k);
                vs[q] = val ? __builtin_nontemporal_load(val + j0 + k) : 1.0f;
            }
        }
#pragma unroll
        for (int q = 0; q < IPT; ++q) xs[q] = (lane + 64 * q < nz) ? x[cs[q]] : 0.0f;
#pragma unroll
        for (int q = 0; q < IPT; ++q) {
            const int k = lane + 64 * q;
            if (k < nz) prod[k] = vs[q] * xs[q];
        }
    }
    wave_sync_lds();

    // this lane's start on the tile's merge path
    const int items = nrows + nz;
    const int ld = lane * IPT < items ? lane * IPT : items;
    int lo = ld - nz > 0 ? ld - nz : 0, hi = ld < nrows ? ld : nrows;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (re[mid] - j0 <= ld - mid - 1)
            lo = mid + 1;
        else
            hi = mid;
    }
    int ri = lo, rj = ld - lo;
    const int ri_start = ri;
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
        if (ri + rj < items) {
            if (ri < nrows && re[ri] - j0 <= rj) {
                out[ri] = sum;
                sum = 0.0f;
                ++ri;
            } else {
                sum += prod[rj];
                ++rj;
            }
        }
    }
    // segmented inclusive scan of (row, partial) across lanes; rows are non-decreasing in lane order
    int key = ri;
    float S = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const float os = __shfl_up(S, d);
        const int ok = __shfl_up(key, d);
        if (lane >= d && ok == key) S += os;
    }
    const float prevS = __shfl_up(S, 1);
    if (lane > 0 && ri > ri_start) out[ri_start] += prevS;
    wave_sync_lds();
    const bool acc = (flags & ARMSP_ACCUMULATE) != 0;
    for (int k = lane; k < nrows; k += 64) y[i0 + k] = acc ? y[i0 + k] + out[k] : out[k];

    const float tail = read_lane(S, 63);
    if (lane == 0) {
        bool has = false;
        if (i1 < M) {
            const int rs = rowptr[i1];
            has = j1 > (rs > j0 ? rs : j0);
        }
        carry_row[wave] = has ? i1 : -1;
        carry_val[wave] = tail;
    }
}

// Adds each run of carries (consecutive waves cut inside the same row) into
// y.  A wave takes 64 consecutive carries; a segmented suffix sum (rows are
// non-decreasing along the carries, so equal tags mark one run) leaves each
// run's in-wave total on its head lane.  A run that goes on past the wave is
// finished by the wave that holds its head, 64 carries a load, and a run that
// began in an earlier wave is left to that wave.  Fixed order, no atomics.
__global__ __launch_bounds__(256) void k_spmv_fixup(int nwaves, const int* __restrict__ carry_row,
                                                    const float* __restrict__ carry_val, float* __restrict__ y) {
    const int lane = threadIdx.x & 63;
    const int base = uniform((int)(blockIdx.x * 4u + (threadIdx.x >> 6))) * 64;
    if (base >= nwaves) return;
    const int w = base + lane;
    const int r = w < nwaves ? carry_row[w] : -2;
    const int rprev = (w == 0 || w > nwaves) ? -2 : carry_row[w - 1];
    float s = (w < nwaves && r >= 0) ? carry_val[w] : 0.0f;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float t = __shfl_down(s, o);
        const int rt = __shfl_down(r, o);
        if (lane + o < 64 && rt == r) s += t;
    }
    // the run of lane 63 may go on into the next waves; the wave holding its head sums the rest
    const int r63 = read_lane(r, 63);
    const bool owner = __ballot(r == r63 && rprev != r63) != 0ull;
    float ext = 0.0f;
    if (r63 >= 0 && owner && base + 64 < nwaves && carry_row[base + 64] == r63) {
        float acc = 0.0f;
        for (int b = base + 64;; b += 64) {
            const int cr = (b + lane < nwaves) ? carry_row[b + lane] : -2;
            const uint64_t m = __ballot(cr == r63);
            const int cnt = (~m == 0ull) ? 64 : __builtin_ctzll(~m);
            if (lane < cnt) acc += carry_val[b + lane];
            if (cnt < 64) break;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
        ext = acc;
    }
    if (r >= 0 && rprev != r) y[r] += (r == r63 ? s + ext : s);
}

// a·b rounded to fp32 by itself: the empty asm makes the product opaque, so the
// compiler cannot contract it with the following add into a fused multiply-add
// (not volatile: the scheduler may still move it, and the loads around it)
__device__ __forceinline__ float unfused_product(float a, float b) {
    float p = a * b;
    asm("" : "+v"(p));
    return p;
}

// Four lanes per row (rows of at most long_blocks blocks when long_blocks > 0),
// 64 rows per 256-thread block `blk`.
__device__ __forceinline__ void vcsr_short_rows(unsigned blk, int M, const int* __restrict__ rowptr,
                                                const int* __restrict__ colind, const float* __restrict__ val,
                                                const float* __restrict__ x, float* __restrict__ y, int fused,
                                                int long_blocks) {
    const int l = threadIdx.x & 3;
    const int row = (int)((blk * 256u + threadIdx.x) >> 2);
    if (row >= M) return;
    const int beg = rowptr[row], end = rowptr[row + 1];
    if (long_blocks > 0 && end - beg > 4 * long_blocks) return;  // a listed long row
    float s = 0.0f;
    // the lane's sum runs block after block in the reference's order; blocks come
    // in batches of 16 whose loads are issued while the previous batch is added (a
    // hub row of an R-MAT graph is tens of thousands of blocks walked by one
    // 4-lane group, so its latency must not be paid per block)
    constexpr int BB = 16;
    auto load = [&](int base, float (&v)[BB], float (&xv)[BB]) {
#pragma unroll
        for (int u = 0; u < BB; ++u) {
            v[u] = val[base + 4 * u + l];
            xv[u] = x[colind[base + 4 * u] + l];
        }
    };
    auto add = [&](const float (&v)[BB], const float (&xv)[BB]) {
        if (fused) {
#pragma unroll
            for (int u = 0; u < BB; ++u) s = fmaf(v[u], xv[u], s);
        } else {  // vmlaq_f32 is a multiply then an add: the product is rounded on its own
#pragma unroll
            for (int u = 0; u < BB; ++u) s += unfused_product(v[u], xv[u]);
        }
    };
    int idx = beg;
    if (idx + 4 * BB <= end) {
        float v0[BB], x0[BB], v1[BB], x1[BB];
        load(idx, v0, x0);
        while (true) {
            idx += 4 * BB;
            if (idx + 4 * BB > end) {
                add(v0, x0);
                break;
            }
            load(idx, v1, x1);
            add(v0, x0);
            idx += 4 * BB;
            if (idx + 4 * BB > end) {
                add(v1, x1);
                break;
            }
            load(idx, v0, x0);
            add(v1, x1);
        }
    }
    // the rest, fewer than BB blocks (most rows of a power-law graph are this short):
    // every load in flight at once, then the adds in block order (blocks past the
    // row are skipped, not added as zeros, which would turn a -0 sum into +0)
    const int nrem = (end - idx) >> 2;
    if (nrem > 0) {
        float v[BB], xv[BB];
#pragma unroll
        for (int u = 0; u < BB; ++u) {
            v[u] = 0.0f;
            xv[u] = 0.0f;
            if (u < nrem) {
                v[u] = val[idx + 4 * u + l];
                xv[u] = x[colind[idx + 4 * u] + l];
            }
        }
        if (fused) {
#pragma unroll
            for (int u = 0; u < BB; ++u)
                if (u < nrem) s = fmaf(v[u], xv[u], s);
        } else {
#pragma unroll
            for (int u = 0; u < BB; ++u)
                if (u < nrem) s += unfused_product(v[u], xv[u]);
        }
    }
    const float t = __fadd_rn(s, __shfl_xor(s, 2, 4));   // lanes 0/2: s0+s2, lanes 1/3: s1+s3
    const float tot = __fadd_rn(t, __shfl_xor(t, 1, 4));  // (s0+s2)+(s1+s3)
    if (l == 0) y[row] = __fadd_rn(y[row], tot);
}

__global__ __launch_bounds__(256) void k_spmv_vcsr(int M, const int* __restrict__ rowptr,
                                                   const int* __restrict__ colind, const float* __restrict__ val,
                                                   const float* __restrict__ x, float* __restrict__ y, int fused) {
    vcsr_short_rows(blockIdx.x, M, rowptr, colind, val, x, y, fused, 0);
}

// One launch, three walkers: rows of at most VCSR_MED_MIN blocks get four lanes
// each, rows of up to `long_blocks` blocks 16 lanes each (vcsr_medium_rows), and
// longer rows a workgroup each: k_vcsr_find_long lists the medium and the long
// rows, and workgroups take listed long rows from a shared counter while the
// other workgroups of the same launch walk the rest (so the walkers overlap, and
// the hub rows, listed first, start first).  A workgroup walks its row in batches of
// VCSR_BATCH blocks.  Waves 1-3 stage, one block per lane: each lane keeps the
// loads of its next VCSR_AHEAD batches in flight (values and x, 16 bytes each; a
// block's column index one ring further ahead, so no x load waits for its index)
// and puts a block into LDS transposed, one array per position l of the 4-block.
// Wave 0's lanes 0-3 keep the reference's four partial sums s_l and do nothing but
// add: a batch in block order, the next VCSR_STEP blocks' terms read from LDS
// during the adds, while the other waves stage the next batch.  With the unfused
// reading the staging lanes form the rounded products a·b; with the fused one they
// stage values and x and lanes 0-3 run the fmaf chain.  Either way each s_l sees the
// reference's sequence of operations: bit-exact.
//
// Bound: the chain of adds of the longest row (27,800 blocks of the 1M R-MAT: 120 us
// on its own, 10 cycles a block), and for the rest the memory requests in flight,
// which is why registers count: 62 VGPRs, 8 waves per SIMD, 233 us (222 with the next
// iteration of a medium row in flight); with 4 batches and 32 blocks ahead 91 VGPRs,
// 5 waves, 286 us.  (345 us with a wave per medium row
// and a staging wave that also added.)
constexpr int VCSR_MED_MIN = 16;          // rows of more blocks than this (and at most long_blocks) are medium
constexpr int VCSR_MED_AHEAD = 4;         // steps of 4 blocks of an iteration of a medium row
constexpr int VCSR_BATCH = 192;           // blocks per batch, one per lane of the staging waves
constexpr int VCSR_STEP = 16;             // blocks whose terms the adding wave reads ahead (a batch is 2n steps)
constexpr int VCSR_PAD = VCSR_BATCH + 4;  // row pitch: lanes 0-3 read from distinct LDS banks
constexpr int VCSR_AHEAD = 2;             // batches in flight per lane

// Workgroups of medium rows per CU (1M R-MAT: 8, 12, 16, 24 per CU give 244, 232, 232,
// 242 us) and of long rows (1, 2, 3, 4: 310, 233, 234, 244 us).
constexpr int VCSR_MED_WG_PER_CU = 16;
constexpr int VCSR_LONG_WG_PER_CU = 2;

// Rows longer than this many blocks take the workgroup-per-row path
// (ARMSP_VCSR_LONG_BLOCKS overrides it, read once per process).  A medium row takes 16
// lanes about 0.6 us per 16 blocks, so in a matrix of few blocks the longest of them is the
// call's time, while a large one has more long rows than workgroups to take them (calls at
// 64, 128, 256 blocks: 1024-row power-law graph of 36 nonzeros a row 15.1, 16.6, 21.3 us;
// R-MAT of 20,000 rows of 30 33.1, 25.5, 30.0; 200,000 rows of 25 170, 98, 78; the 1M
// R-MAT 680, 318, 228, and 229 at 384).
int vcsr_long_blocks(int nnz_padded) {
    static const int v = [] {
        const char* e = getenv("ARMSP_VCSR_LONG_BLOCKS");
        return e ? std::max(atoi(e), 0) : 0;
    }();
    const int blocks = nnz_padded / 4;
    return v ? v : blocks <= 1 << 17 ? 64 : blocks <= 1 << 20 ? 128 : 256;
}

// Lists the long rows (more than long_blocks blocks) in list — those over 8 times the
// limit from the front, count[0] of them, the others from the back, count[3], so that
// the longest start first (in the order of listing: 255 us, not 231) — and the medium rows (more than VCSR_MED_MIN blocks, at most long_blocks) in
// list_med[0, count[2]); the order within a list does not matter, each row is
// summed by one walker.  A workgroup ranks the listed rows of its 8192 by wave
// ballots and a scan of the 16 wave counts, and takes its slots with one atomic
// per list: atomics on one counter follow each other at about 15 ns (one per row
// 1.5 ms for the 1M R-MAT's 10^5 medium rows, one per wave 117 us, one per 1024
// rows 13 us, one per 8192 8 us).
constexpr int VCSR_FIND_THREADS = 1024;
// R rows per thread, as many as leave 256 workgroups or more: with fewer the CUs without one
// wait for the others' loads (calls on uniform matrices with R = 1, 2, 4, 8: 200,000 rows of
// 5 26.2, 26.8, 27.8, 30.1 us; 2^20 rows of 16 312, 307, 304, 305).
template <int R>
__global__ __launch_bounds__(VCSR_FIND_THREADS) void k_vcsr_find_long(int M, const int* __restrict__ rowptr,
                                                                      int long_blocks, int* __restrict__ list,
                                                                      int* __restrict__ list_med,
                                                                      int* __restrict__ count) {
    constexpr int NW = VCSR_FIND_THREADS / 64;
    __shared__ int s_off[3][NW];  // per wave: its rows' first slot within the workgroup
    __shared__ int s_base[3];     // the workgroup's first slot in each list
    const int lane = (int)__lane_id(), wid = (int)(threadIdx.x >> 6);
    const int64_t r0 = (int64_t)blockIdx.x * (VCSR_FIND_THREADS * R) + wid * (64 * R) + lane;
    uint64_t bh[R], bl[R], bm[R];
    int n[R], nh = 0, nl = 0, nm = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int64_t r = r0 + 64 * j;
        n[j] = r < M ? rowptr[r + 1] - rowptr[r] : 0;
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const bool is_long = n[j] > 4 * long_blocks, is_huge = n[j] / 32 > long_blocks;
        bh[j] = __ballot(is_huge);
        bl[j] = __ballot(is_long && !is_huge);
        bm[j] = __ballot(!is_long && n[j] > 4 * VCSR_MED_MIN);
        nh += __popcll(bh[j]);
        nl += __popcll(bl[j]);
        nm += __popcll(bm[j]);
    }
    if (lane == 0) {
        s_off[0][wid] = nh;
        s_off[1][wid] = nl;
        s_off[2][wid] = nm;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int t = (int)threadIdx.x;
        int acc = 0;
        for (int w = 0; w < NW; ++w) {
            const int c = s_off[t][w];
            s_off[t][w] = acc;
            acc += c;
        }
        s_base[t] = acc > 0 ? atomicAdd(&count[t == 0 ? 0 : t == 1 ? 3 : 2], acc) : 0;
    }
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull;
    int ah = s_base[0] + s_off[0][wid], al = s_base[1] + s_off[1][wid], am = s_base[2] + s_off[2][wid];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int r = (int)(r0 + 64 * j);
        if ((bh[j] >> lane) & 1) list[ah + __popcll(bh[j] & below)] = r;
        if ((bl[j] >> lane) & 1) list[M - 1 - (al + __popcll(bl[j] & below))] = r;
        if ((bm[j] >> lane) & 1) list_med[am + __popcll(bm[j] & below)] = r;
        ah += __popcll(bh[j]);
        al += __popcll(bl[j]);
        am += __popcll(bm[j]);
    }
}

// count[0], count[3] = long rows listed from the front and from the back, count[1] =
// the long rows' work counter, count[2] = listed medium rows
__global__ void k_zero_count(int* count) {
    count[0] = 0;
    count[1] = 0;
    count[2] = 0;
    count[3] = 0;
}

// Medium rows, a DPP row of 16 lanes each, four rows a wave: group gg of ngg takes
// list_med[gg], list_med[gg + ngg], ... (a fixed assignment, no shared counter), each
// at its own pace.  A step covers 4 blocks, lane 4q + l holding position l of block
// q, and an iteration VCSR_MED_AHEAD steps.  The next iteration's values and x (of the
// next row, when this one ends) are in flight during an iteration's adds, and the
// column indices of the one after it behind them.
// The lanes form the rounded products (the unfused reading) or keep value and x
// (fused); the four partial sums travel round the 16 lanes, four lanes on per block,
// and add each block's term where they find it: s = rotate(s) + p, one DPP add a
// block, the reference's sequence of operations per s_l, as in the other walkers.
// (A wave per row that fetched each block's terms by a shuffle was bound by the LDS
// crossbar: rows of 17-256 blocks of the 1M R-MAT, 31M padded entries, took 201 us.)
__device__ __forceinline__ float rotate4(float s) {  // lane i of each 16 gets lane i - 4's
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x124, 0xf, 0xf, false));
}

template <bool FUSED>
__device__ void vcsr_medium_rows(uint32_t gg, uint32_t ngg, const int* __restrict__ list_med, const int* __restrict__ count,
                                 const int* __restrict__ rowptr, const int* __restrict__ colind,
                                 const float* __restrict__ val, const float* __restrict__ x, float* __restrict__ y) {
    constexpr int D = VCSR_MED_AHEAD;
    constexpr int IT = 4 * D;  // blocks of an iteration
    const int q = (threadIdx.x >> 2) & 3, l = threadIdx.x & 3;
    const uint32_t nmed = (uint32_t)__builtin_amdgcn_readfirstlane(count[2]);
    if ((uint32_t)__builtin_amdgcn_readfirstlane((int)gg) >= nmed) return;  // none for this wave
    // row i of the list; past its end no blocks (row 0's index, so every load stays in bounds)
    auto row_at = [&](uint32_t i) { return i < nmed ? list_med[i] : 0; };
    auto blocks_of = [&](uint32_t i, int r, int b) { return i < nmed ? (rowptr[r + 1] - b) >> 2 : 0; };
    auto columns = [&](int beg, int nb, int pos, int (&c)[D]) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            const int b = pos + 4 * u + q;
            c[u] = b < nb ? colind[beg + 4 * b] : 0;
        }
    };
    auto terms = [&](int beg, int nb, int pos, const int (&c)[D], float (&v)[D], float (&xv)[D]) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            const int b = pos + 4 * u + q;
            v[u] = 0.0f;
            xv[u] = 0.0f;
            if (b < nb) {
                v[u] = val[beg + 4 * b + l];
                xv[u] = x[c[u] + l];
            }
        }
    };
    // the group's row, the two after it, and the index of the third
    uint32_t i = gg;
    int r0 = row_at(i), r1 = row_at(i + ngg), r2 = row_at(i + 2 * ngg), r3 = row_at(i + 3 * ngg);
    int b0 = rowptr[r0], b1 = rowptr[r1], b2 = rowptr[r2];
    int n0 = blocks_of(i, r0, b0), n1 = blocks_of(i + ngg, r1, b1), n2 = blocks_of(i + 2 * ngg, r2, b2);
    float y0 = y[r0], y1 = y[r1];
    int pos = 0, c[D];
    float v[D], xv[D];
    columns(b0, n0, 0, c);
    terms(b0, n0, 0, c, v, xv);
    // the next iteration: of this row, or the first of the next
    bool last = IT >= n0;
    columns(last ? b1 : b0, last ? n1 : n0, last ? 0 : IT, c);
    float s = 0.0f;
    while (__ballot(i < nmed) != 0ull) {
        const int bn = last ? b1 : b0, nn = last ? n1 : n0, pn = last ? 0 : pos + IT;
        float vn[D], xn[D];
        terms(bn, nn, pn, c, vn, xn);  // the next iteration's terms, and behind them the
        const bool lastn = pn + IT >= nn;  // column indices of the one after it
        columns(!lastn ? bn : last ? b2 : b1, !lastn ? nn : last ? n2 : n1, lastn ? 0 : pn + IT, c);
        if (__ballot(pos + IT > n0) == 0ull) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
                const float p = FUSED ? 0.0f : unfused_product(v[u], xv[u]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float t = rotate4(s);
                    s = FUSED ? fmaf(v[u], xv[u], t) : __fadd_rn(t, p);
                }
            }
        } else {  // a row ends among these blocks: past it the sums only move on
#pragma unroll
            for (int u = 0; u < D; ++u) {
                const float p = FUSED ? 0.0f : unfused_product(v[u], xv[u]);
                const bool in = pos + 4 * u + q < n0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float t = rotate4(s);
                    s = !in ? t : FUSED ? fmaf(v[u], xv[u], t) : __fadd_rn(t, p);
                }
            }
        }
        // whole steps: the sums are in lanes 12-15 of the group
        const float t = __fadd_rn(s, __shfl_xor(s, 2, 4));    // lanes 0/2: s0+s2, lanes 1/3: s1+s3
        const float tot = __fadd_rn(t, __shfl_xor(t, 1, 4));  // (s0+s2)+(s1+s3)
        if (last) {
            if (i < nmed && q == 3 && l == 0) y[r0] = __fadd_rn(y0, tot);
            // (past the list a group waits there for the wave's others, however long their rows are)
            i += i < nmed ? ngg : 0u;
            s = 0.0f;
            r0 = r1;
            b0 = b1;
            n0 = n1;
            y0 = y1;
            r1 = r2;
            b1 = b2;
            n1 = n2;
            y1 = y[r1];
            r2 = r3;
            b2 = rowptr[r2];
            n2 = blocks_of(i + 2 * ngg, r2, b2);
            r3 = row_at(i + 3 * ngg);
        }
        pos = pn;
        last = lastn;
#pragma unroll
        for (int u = 0; u < D; ++u) {
            v[u] = vn[u];
            xv[u] = xn[u];
        }
    }
}

template <bool FUSED>
__device__ void vcsr_long_rows(int M, const int* __restrict__ list, int* __restrict__ count,
                               const int* __restrict__ rowptr, const int* __restrict__ colind,
                               const float* __restrict__ val, const float* __restrict__ x, float* __restrict__ y,
                               float (*s_a)[4][VCSR_PAD], float (*s_b)[4][VCSR_PAD], int* s_row) {
    constexpr int D = VCSR_AHEAD;
    const int t = (int)threadIdx.x - 64;  // staging lane of waves 1-3; wave 0 adds
    const int l = (int)threadIdx.x & 3;
    const int nfront = count[0], nlong = nfront + count[3];
    if (nlong == 0) return;  // (512 workgroups' turns at the counter take microseconds)
    while (true) {
        if (threadIdx.x == 0) *s_row = atomicAdd(&count[1], 1);
        __syncthreads();
        const int i = *s_row;
        __syncthreads();  // every lane has read the row before lane 0 takes the next
        if (i >= nlong) break;  // the same for the whole workgroup once the list is drained
        const int r = list[i < nfront ? i : M - 1 - (i - nfront)];
        const int beg = rowptr[r];
        const int nb = (rowptr[r + 1] - beg) >> 2;
        const int nbat = (nb + VCSR_BATCH - 1) / VCSR_BATCH;
        if (t >= 0) {
            // lane t owns block k·VCSR_BATCH + t of batch k
            auto col_of = [&](int k) {
                const int b = k * VCSR_BATCH + t;
                return b < nb ? colind[beg + 4 * b] : -1;
            };
            float4 rv[D], rx[D];
            int rc[D];
            auto fetch = [&](int k, int c, float4& v, float4& xv) {
                const int b = k * VCSR_BATCH + t;
                v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                xv = v;
                if (b < nb) {
                    v = *reinterpret_cast<const float4*>(val + beg + 4 * b);
                    xv = *reinterpret_cast<const float4*>(x + c);
                }
            };
#pragma unroll
            for (int u = 0; u < D; ++u) rc[u] = col_of(u);
#pragma unroll
            for (int u = 0; u < D; ++u) {
                fetch(u, rc[u], rv[u], rx[u]);
                rc[u] = col_of(u + D);
            }
            for (int k0 = 0; k0 < nbat; k0 += D) {
#pragma unroll
                for (int u = 0; u < D; ++u) {
                    const int k = k0 + u;
                    if (k >= nbat) break;  // uniform: nbat is the workgroup's
                    const int buf = k & 1;
                    if constexpr (FUSED) {
                        s_a[buf][0][t] = rv[u].x;
                        s_a[buf][1][t] = rv[u].y;
                        s_a[buf][2][t] = rv[u].z;
                        s_a[buf][3][t] = rv[u].w;
                        s_b[buf][0][t] = rx[u].x;
                        s_b[buf][1][t] = rx[u].y;
                        s_b[buf][2][t] = rx[u].z;
                        s_b[buf][3][t] = rx[u].w;
                    } else {  // vmlaq_f32 rounds the product on its own
                        s_a[buf][0][t] = unfused_product(rv[u].x, rx[u].x);
                        s_a[buf][1][t] = unfused_product(rv[u].y, rx[u].y);
                        s_a[buf][2][t] = unfused_product(rv[u].z, rx[u].z);
                        s_a[buf][3][t] = unfused_product(rv[u].w, rx[u].w);
                    }
                    fetch(k + D, rc[u], rv[u], rx[u]);  // in flight for D batches
                    rc[u] = col_of(k + 2 * D);
                    // batch k staged; wave 0 has also finished adding batch k-1, whose
                    // buffer batch k+1 is about to overwrite
                    __syncthreads();
                }
            }
        } else {
            // VCSR_STEP blocks a step, the next step's LDS reads in flight during the adds (a batch
            // holds whole pairs of steps, so a read past the row's end stays inside the batch)
            __builtin_amdgcn_s_setprio(3);  // the chain of adds is the row's time: first in the SIMD's queue
            float s = 0.0f;
            for (int k = 0; k < nbat; ++k) {
                __syncthreads();
                const int cnt = min(VCSR_BATCH, nb - k * VCSR_BATCH);
                const float4* pa = reinterpret_cast<const float4*>(&s_a[k & 1][l][0]);
                const float4* pb = reinterpret_cast<const float4*>(&s_b[FUSED ? (k & 1) : 0][FUSED ? l : 0][0]);
                constexpr int Q = VCSR_STEP / 4;
                float4 a0[Q], a1[Q], b0[FUSED ? Q : 1], b1[FUSED ? Q : 1];
                auto read = [&](int at, float4 (&a)[Q], float4 (&b)[FUSED ? Q : 1]) {
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        a[q] = pa[at + q];
                        if constexpr (FUSED) b[q] = pb[at + q];
                    }
                };
                auto one = [&](float a, float b) {
                    if constexpr (FUSED)
                        s = fmaf(a, b, s);
                    else
                        s = __fadd_rn(s, a);
                };
                auto add = [&](int at, const float4 (&a)[Q], const float4 (&b)[FUSED ? Q : 1]) {
                    if (4 * at + VCSR_STEP <= cnt) {
#pragma unroll
                        for (int q = 0; q < Q; ++q) {
                            const float4 w = b[FUSED ? q : 0];
                            one(a[q].x, w.x);
                            one(a[q].y, w.y);
                            one(a[q].z, w.z);
                            one(a[q].w, w.w);
                        }
                    } else {  // the row's last blocks (uniform tests)
#pragma unroll
                        for (int q = 0; q < Q; ++q) {
                            const float4 w = b[FUSED ? q : 0];
                            if (4 * (at + q) + 0 < cnt) one(a[q].x, w.x);
                            if (4 * (at + q) + 1 < cnt) one(a[q].y, w.y);
                            if (4 * (at + q) + 2 < cnt) one(a[q].z, w.z);
                            if (4 * (at + q) + 3 < cnt) one(a[q].w, w.w);
                        }
                    }
                };
                read(0, a0, b0);
                for (int at = 0; 4 * at < cnt; at += 2 * Q) {
                    read(at + Q, a1, b1);
                    add(at, a0, b0);
                    if (at + 2 * Q < VCSR_BATCH / 4) read(at + 2 * Q, a0, b0);
                    add(at + Q, a1, b1);
                }
            }
            // lanes 0-3 hold s0..s3
            const float tt = __fadd_rn(s, __shfl_xor(s, 2, 4));  // lanes 0/2: s0+s2, lanes 1/3: s1+s3
            const float tot = __fadd_rn(tt, __shfl_xor(tt, 1, 4));  // (s0+s2)+(s1+s3)
            if (threadIdx.x == 0) y[r] = __fadd_rn(y[r], tot);
            __builtin_amdgcn_s_setprio(0);
        }
        __syncthreads();  // the LDS buffers are free for the next row
    }
}

// One launch: workgroups [0, n_long_wg) walk the listed long rows, the next
// n_med_wg the listed medium rows (16 lanes each), the rest the short rows (64 per
// workgroup).
template <bool FUSED>
__global__ __launch_bounds__(256) void k_spmv_vcsr_split(int M, const int* __restrict__ rowptr,
                                                         const int* __restrict__ colind,
                                                         const float* __restrict__ val, const float* __restrict__ x,
                                                         float* __restrict__ y, const int* __restrict__ list,
                                                         const int* __restrict__ list_med, int* __restrict__ count,
                                                         int n_long_wg, int n_med_wg) {
    __shared__ __align__(16) float s_a[2][4][VCSR_PAD];
    __shared__ __align__(16) float s_b[FUSED ? 2 : 1][4][FUSED ? VCSR_PAD : 4];
    __shared__ int s_row;
    const int b = (int)blockIdx.x;
    if (b < n_long_wg) {
        vcsr_long_rows<FUSED>(M, list, count, rowptr, colind, val, x, y, s_a,
                              reinterpret_cast<float (*)[4][VCSR_PAD]>(&s_b[0][0][0]), &s_row);
        return;
    }
    if (b < n_long_wg + n_med_wg) {
        const uint32_t gg = (uint32_t)(b - n_long_wg) * 16 + (threadIdx.x >> 4);
        vcsr_medium_rows<FUSED>(gg, (uint32_t)n_med_wg * 16, list_med, count, rowptr, colind, val, x, y);
        return;
    }
    // the short walker takes what neither list holds: rows of at most VCSR_MED_MIN
    // blocks (the long-row limit is never below it; a constant here lets the
    // compiler drop the walker's batch loop for longer rows: a kernel of 62 VGPRs, not 111)
    vcsr_short_rows((unsigned)(b - n_long_wg - n_med_wg), M, rowptr, colind, val, x, y, FUSED ? 1 : 0, VCSR_MED_MIN);
}

template <int IPT>
int launch_merge(int M, int nnz, const int* rp, const int* ci, const float* va, const float* x, float* y, int flags,
                 hipStream_t s) {
    constexpr int TILE = 64 * IPT;
    const int64_t total = (int64_t)M + nnz;
    const int64_t nwaves = (total + TILE - 1) / TILE;
    if (nwaves > INT_MAX / 4) return ARMSP_ERROR_NOT_SUPPORTED;
    void* ws = nullptr;
    const size_t rb = ((size_t)nwaves * 4 + 255) & ~(size_t)255;
    int st = ws_alloc(&ws, 2 * rb + (size_t)(nwaves + 1) * 4, s);
    if (st) return st;
    int* crow = static_cast<int*>(ws);
    float* cval = reinterpret_cast<float*>(static_cast<char*>(ws) + rb);
    int* part = reinterpret_cast<int*>(static_cast<char*>(ws) + 2 * rb);
    if (nwaves <= kSearchWaves) {
        part = nullptr;
    } else {
        TimedLaunch t("merge_partition", s);
        st = merge_partition(M, nnz, TILE, nwaves, rp, part, s);
        if (st) {
            ws_free(ws, s);
            return st;
        }
        t.stop();
    }
    {
        TimedLaunch t("spmv", s);
        hipLaunchKernelGGL((k_spmv_merge<IPT>), dim3((unsigned)((nwaves + 3) / 4)), dim3(256), 0, s, M, nnz, rp, ci,
                           va, x, y, flags, part, crow, cval);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            ws_free(ws, s);
            return hip_fail(e);
        }
        t.stop();
    }
    {
        TimedLaunch t("spmv_fixup", s);
        hipLaunchKernelGGL(k_spmv_fixup, dim3((unsigned)((nwaves + 255) / 256)), dim3(256), 0, s, (int)nwaves, crow,
                           cval, y);
        hipError_t e = hipGetLastError();
        ws_free(ws, s);
        if (e != hipSuccess) return hip_fail(e);
        t.stop();
    }
    return ARMSP_SUCCESS;
}

}  // namespace
}  // namespace armsp

extern "C" {

int armsp_spmv_f32(int M, int K, int nnz, const int* rowptr, const int* colind, const float* val, const float* x,
                   float* y, int flags, const armsp_config* cfg, void* stream) {
    using namespace armsp;
    if (M < 0 || K < 0 || nnz < 0) return ARMSP_ERROR_INVALID_VALUE;
    if (M == 0) return ARMSP_SUCCESS;
    if (!rowptr || !y || (nnz > 0 && (!colind || !x))) return ARMSP_ERROR_INVALID_VALUE;
    if (flags & ~ARMSP_ACCUMULATE) return ARMSP_ERROR_INVALID_VALUE;
    if ((int64_t)M + nnz > INT_MAX) return ARMSP_ERROR_NOT_SUPPORTED;
    hipStream_t s = as_stream(stream);
    armsp_config c = cfg ? *cfg : armsp_config{0, 0, 0, 0, 0};
    int sched = c.schedule == ARMSP_SCHED_AUTO ? ARMSP_SCHED_MERGE : c.schedule;
    if (sched == ARMSP_SCHED_NNZ) sched = ARMSP_SCHED_MERGE;
    if (sched == ARMSP_SCHED_ROW) {
        int G = c.group;
        if (G <= 0) {
            const int avg = nnz / M;
            G = 1;
            while (G < 64 && G < avg) G <<= 1;
        }
        TimedLaunch t("spmv", s);
        const dim3 grid((unsigned)(((int64_t)M * G + 255) / 256));
        switch (G) {
#define ARMSP_SPMV_ROW(GG)                                                                                          \
    case GG:                                                                                                        \
        hipLaunchKernelGGL((k_spmv_row<GG>), grid, dim3(256), 0, s, M, rowptr, colind, val, x, y, flags); \
        break;
            ARMSP_SPMV_ROW(1)
            ARMSP_SPMV_ROW(2)
            ARMSP_SPMV_ROW(4)
            ARMSP_SPMV_ROW(8)
            ARMSP_SPMV_ROW(16)
            ARMSP_SPMV_ROW(32)
            ARMSP_SPMV_ROW(64)
#undef ARMSP_SPMV_ROW
            default: return ARMSP_ERROR_INVALID_VALUE;
        }
        ARMSP_LAUNCHED();
        t.stop();
        return ARMSP_SUCCESS;
    }
    if (sched != ARMSP_SCHED_MERGE) return ARMSP_ERROR_INVALID_VALUE;
    // AUTO: 16 items per lane when that still leaves 16 waves per CU (more gathers in
    // flight per lane: 1M R-MAT, 2^24 nnz, 91.6 -> 87.5 us), else 8
    const int64_t items = (int64_t)M + nnz;
    const int ipt = c.chunk > 0 ? c.chunk / 64 : (items / (64 * 16) >= 16 * (int64_t)device_cus() ? 16 : 8);
    switch (ipt) {
        case 4: return launch_merge<4>(M, nnz, rowptr, colind, val, x, y, flags, s);
        case 8: return launch_merge<8>(M, nnz, rowptr, colind, val, x, y, flags, s);
        case 16: return launch_merge<16>(M, nnz, rowptr, colind, val, x, y, flags, s);
        default: return ARMSP_ERROR_INVALID_VALUE;
    }
}

int armsp_spmv_vcsr_f32(int M, int nnz_padded, const int* rowptr, const int* colind, const float* val, const float* x,
                        float* y, int flags, void* stream) {
    using namespace armsp;
    if (M < 0 || nnz_padded < 0 || (nnz_padded & 3)) return ARMSP_ERROR_INVALID_VALUE;
    if (M == 0) return ARMSP_SUCCESS;
    if (!rowptr || !y || (nnz_padded > 0 && (!colind || !val || !x))) return ARMSP_ERROR_INVALID_VALUE;
    if (flags & ~(ARMSP_ACCUMULATE | ARMSP_FUSED_MLA | ARMSP_VCSR_BALANCED)) return ARMSP_ERROR_INVALID_VALUE;
    hipStream_t s = as_stream(stream);
    if (flags & ARMSP_VCSR_BALANCED) {
        // the padded blocks are a CSR matrix of their own: merge-path SpMV, y += A·x
        if (flags & ARMSP_FUSED_MLA) return ARMSP_ERROR_INVALID_VALUE;
        if (nnz_padded == 0) return ARMSP_SUCCESS;
        return launch_merge<8>(M, nnz_padded, rowptr, colind, val, x, y, ARMSP_ACCUMULATE, s);
    }
    const int fused = (flags & ARMSP_FUSED_MLA) ? 1 : 0;
    // Rows of more than VCSR_MED_MIN blocks take 16 lanes each, rows of more than
    // long_blocks a workgroup each; the workgroup walker's 16-byte loads need
    // 16-byte-aligned values and x (VCSR rows hold whole 4-blocks and block columns
    // are multiples of 4, so rowptr entries and the gathered x offsets are multiples
    // of 4 as well), so with unaligned operands every long row is a medium one.
    const bool aligned = ((uintptr_t)val % 16) == 0 && ((uintptr_t)x % 16) == 0;
    // (a long-row limit below VCSR_MED_MIN acts as VCSR_MED_MIN: rows up to it are the short walker's)
    const int lb = vcsr_long_blocks(nnz_padded);
    const int long_blocks = aligned ? (lb < VCSR_MED_MIN ? VCSR_MED_MIN : lb) : INT_MAX / 8;
    const bool split_long = nnz_padded / 4 > VCSR_MED_MIN;
    void* ws = nullptr;
    int* list = nullptr;
    int* list_med = nullptr;
    int* count = nullptr;
    if (split_long) {
        const int st = ws_alloc(&ws, (2 * (size_t)M + 64) * sizeof(int), s);
        if (st) return st;
        count = static_cast<int*>(ws);
        list = count + 64;
        list_med = list + M;
        hipLaunchKernelGGL(k_zero_count, dim3(1), dim3(1), 0, s, count);
        auto find = [&](auto kernel, int rows) {  // rows per thread
            const int64_t per = (int64_t)rows * VCSR_FIND_THREADS;
            hipLaunchKernelGGL(kernel, dim3((unsigned)((M + per - 1) / per)), dim3(VCSR_FIND_THREADS), 0, s, M, rowptr,
                               long_blocks, list, list_med, count);
        };
        if (M <= 1 << 18)
            find(k_vcsr_find_long<1>, 1);
        else if (M <= 1 << 19)
            find(k_vcsr_find_long<2>, 2);
        else if (M <= 1 << 22)
            find(k_vcsr_find_long<4>, 4);
        else
            find(k_vcsr_find_long<8>, 8);
    }
    TimedLaunch t("spmv_vcsr", s);
    const unsigned short_wg = (unsigned)(((int64_t)M * 4 + 255) / 256);
    if (split_long) {  // long-row workgroups first (the hub rows are the critical path), then medium-row waves
        // (no more workgroups than rows: a small matrix would wait for idle ones)
        const int n_long_wg = std::min(VCSR_LONG_WG_PER_CU * device_cus(), M);
        const int n_med_wg = std::min(VCSR_MED_WG_PER_CU * device_cus(), (M + 15) / 16);
        const dim3 grid((unsigned)(n_long_wg + n_med_wg) + short_wg);
        if (fused)
            hipLaunchKernelGGL(k_spmv_vcsr_split<true>, grid, dim3(256), 0, s, M, rowptr, colind, val, x, y, list,
                               list_med, count, n_long_wg, n_med_wg);
        else
            hipLaunchKernelGGL(k_spmv_vcsr_split<false>, grid, dim3(256), 0, s, M, rowptr, colind, val, x, y, list,
                               list_med, count, n_long_wg, n_med_wg);
    } else {
        hipLaunchKernelGGL(k_spmv_vcsr, dim3(short_wg), dim3(256), 0, s, M, rowptr, colind, val, x, y, fused);
    }
    const hipError_t e = hipGetLastError();
    if (ws) ws_free(ws, s);
    if (e != hipSuccess) return hip_fail(e);
    t.stop();
    return ARMSP_SUCCESS;
}

}  // extern "C"
