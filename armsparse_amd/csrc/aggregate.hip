// Max aggregation over CSR neighbourhoods (the GraphSAGE / DGL max reducer).
//
// Reference: gcn/dgl-custom/binary_reduce_max.cu — topoSimpleSPMMMaxKernel
// (:151-166) and the tiled variants (:26-149) compute, for every row r and
// column j, C[r][j] = max over the row's nonzeros of B[colind][j] (copy of the
// source features, no edge values), starting from max_init() = -10000 (:22-24)
// and folding with `acc > x ? acc : x` (:18-20) in CSR order.  The same fold
// here, with an optional edge value multiplied in (x = val·B[c][j]), the
// initial value a parameter (the reference's -10000 by default in the Python
// layer), and the winning nonzero position recorded per output for the
// backward pass: dB[colind[p]][j] += val[p]·dC[r][j] for p = argmax[r][j].
//
// The result and the argmax (a later equal value wins, as `acc > x ? acc : x`
// does) are the sequential fold's.  Two walkers in one launch (k_spmm_max):
//  short rows — a group of G lanes per row, V columns per lane, U gathers of the
//          row in flight;
//  long rows — waves that each take a fixed range of nonzeros and fold what it holds
//          of the long rows; k_max_join folds the parts of a cut row in order.  In small
//          inputs a workgroup per long row instead, which needs no second launch.
// A hub row walked by one group bounds the call, whatever else runs: a 131,072-row
// R-MAT with 2^21 nonzeros at N = 64 took 2551 us, 74 + 5 now; matrices without
// long rows keep the group per row (1.5M nonzeros, uniform: 65 us, 64 + 4 now), and the
// wave ranges end at once.
#include <algorithm>
#include <climits>

#include "common.hpp"

namespace armsp {
namespace {

template <int V>
__device__ __forceinline__ void load_v(const float* __restrict__ p, float (&o)[V]) {
    if constexpr (V == 4) {
        const float4 t = *reinterpret_cast<const float4*>(p);
        o[0] = t.x; o[1] = t.y; o[2] = t.z; o[3] = t.w;
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v) o[v] = p[v];
    }
}

template <int V>
__device__ __forceinline__ void store_v(float* __restrict__ p, const float (&o)[V]) {
    if constexpr (V == 4) {
        *reinterpret_cast<float4*>(p) = make_float4(o[0], o[1], o[2], o[3]);
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v) p[v] = o[v];
    }
}

// Rows of more nonzeros than this are long: a group's walk of 32 costs less than the
// waves' search for them (the R-MAT, limits 32, 64, 128, 256: 77, 103, 127, 239 us),
// but the ordinary rows of a denser matrix stay with the groups, which hold several
// rows a wave (50,000 rows of 39: 156 us, 176 us as long rows).
inline int max_long_row(int M, int nnz) {
    const int64_t twice_mean = 2 * (int64_t)nnz / M;
    return twice_mean > 32 ? (int)twice_mean : 32;
}

// Nonzeros times lanes per group up to which a workgroup takes each long row, without parts
// in memory and without the second launch, which is 3 of 14 us where no row is long (uniform,
// 1024 rows of 8 to 4096 of 8, N = 4 to 64: 10.5 us, 13.7 to 14.3 with it; a power-law graph
// of 1024 rows of 8 10.7 and 14.0).  Beyond, a hub row keeps its workgroup's four waves busy
// for longer than the launch takes (R-MAT of 8192 rows of 10, N = 64: 18.2 and 15.0).
constexpr int64_t kMaxJoin = 1 << 19;

// A row cut by the waves' ranges is a sequence of parts.  The part that holds the
// row's start folds from `init`, the others from -inf with no position, so every part
// of the others names one.  Joining two parts in order, the later wins unless the
// earlier is greater, as in the fold itself; but a NaN x replaces any accumulator
// and is replaced by any later x, so a part with a NaN in it replaces what came
// before: its position is stored with the top bit set.
constexpr uint32_t kNoPos = 0xffffffffu;
constexpr uint32_t kSawNan = 0x80000000u;
__device__ __forceinline__ void max_join(float& acc, uint32_t& arg, float x, uint32_t p) {
    if (p == kNoPos) return;  // no entries in the later part
    const bool keep = !(p & kSawNan) && acc > x;
    acc = keep ? acc : x;
    arg = keep ? arg : p | (arg != kNoPos ? arg & kSawNan : 0u);
}

// Where the long-row walker leaves its parts: per wave the part of a row that goes on
// past its range (of row carry_row[wave], else -1) and the part of a row that began
// before it and ends in it, N columns each.
struct MaxParts {
    int* carry_row;
    float* val;
    uint32_t* arg;
};

// Long rows' entries among the nonzeros [j0, j1) of `wave`, columns tile0 + 64·V.
template <int V>
__device__ __forceinline__ void max_long_rows(int wave, int j0, int j1, int tile0, int M, int N, int long_row,
                                              const int* __restrict__ rowptr, const int* __restrict__ colind,
                                              const float* __restrict__ val, const float* __restrict__ B, int ldb,
                                              float init, float* __restrict__ C, int ldc, int* __restrict__ argmax,
                                              const MaxParts& parts) {
    constexpr int U = V <= 2 ? 8 : 4;
    const int lane = threadIdx.x & 63;
    const int col = tile0 + lane * V;
    const bool active = col < N;
    const float* bp = B + (active ? col : tile0);  // lanes past N read the tile's first column
    int carry = -1;
    int idle = 0;  // windows of 64 rows in a row that held no entry
    for (int rb = uniform(rows_ending_by_wave(j0, rowptr, M)); rb < M;) {
        const int rl = rb + lane;
        const int sl = rl < M ? rowptr[rl] : INT_MAX, el = rl < M ? rowptr[rl + 1] : INT_MAX;
        // (a malformed rowptr cannot carry the walk outside its range: see the clamps below)
        uint64_t longs = __ballot(rl < M && el - sl > long_row && sl < j1 && el > j0);
        for (; longs; longs &= longs - 1) {
            const int l = __builtin_ctzll(longs);
            const int r = rb + l, s = read_lane(sl, l), e = read_lane(el, l);
            const int p0 = max(s, j0), p1 = min(e, j1);
            const bool first = s >= j0;
            float acc[V];
            uint32_t arg[V];
            uint64_t nan[V];  // lanes whose part has seen a NaN
#pragma unroll
            for (int v = 0; v < V; ++v) {
                acc[v] = first ? init : -__builtin_inff();
                arg[v] = kNoPos;
                nan[v] = 0;
            }
            for (int base = p0; base < p1; base += 64) {
                const int n = min(64, p1 - base);
                int c = 0;
                float a = 0.0f;
                if (lane < n) {
                    c = colind[base + lane];
                    a = val ? val[base + lane] : 1.0f;
                }
                for (int k = 0; k < n; k += U) {
                    float b[U][V], w[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {  // past n: again the last entry, not folded
                        const int q = min(k + u, n - 1);
                        w[u] = read_lane(a, q);
                        load_v<V>(bp + (size_t)read_lane(c, q) * ldb, b[u]);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (k + u < n) {
#pragma unroll
                            for (int v = 0; v < V; ++v) {
                                const float x = w[u] * b[u][v];
                                const bool keep = acc[v] > x;  // the reference's `acc > x ? acc : x`
                                acc[v] = keep ? acc[v] : x;
                                arg[v] = keep ? arg[v] : (uint32_t)(base + k + u);
                                nan[v] |= __ballot(x != x);
                            }
                        }
                }
            }
            const bool goes_on = e > j1;
            if (goes_on) carry = r;
            if (!active) continue;
            if (first && !goes_on) {
                store_v<V>(C + (size_t)r * ldc + col, acc);
                if (argmax) {
#pragma unroll
                    for (int v = 0; v < V; ++v) argmax[(size_t)r * N + col + v] = (int)arg[v];
                }
            } else {
                const size_t o = ((size_t)wave * 2 + (goes_on ? 0 : 1)) * N + col;
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    parts.val[o + v] = acc[v];
                    parts.arg[o + v] = arg[v] | ((nan[v] >> lane) & 1 ? kSawNan : 0u);
                }
            }
        }
        const int e63 = read_lane(el, 63);
        if (e63 >= j1) break;  // later rows begin after the range
        // a long run of empty rows is searched for its end, not walked (a million of them:
        // 16,000 dependent steps); short ones pass sooner than a search does
        idle = e63 == read_lane(sl, 0) ? idle + 1 : 0;
        rb += 64;
        if (idle == 4) {
            rb = max(rb, uniform(rows_ending_by_wave(e63, rowptr, M)));
            idle = 0;
        }
    }
    if (tile0 == 0 && lane == 0) parts.carry_row[wave] = carry;
}

// The long rows that begin among the nonzeros [j0, j1), a workgroup of four waves per row:
// every group of G lanes folds a part of the row, the parts are joined in order, within
// the waves by shuffles and across them in LDS.  Columns as in max_short_rows.
template <int V, int G>
__device__ __forceinline__ void max_group_rows(int j0, int j1, int tile, int M, int N, int nnz, int long_row,
                                               const int* __restrict__ rowptr, const int* __restrict__ colind,
                                               const float* __restrict__ val, const float* __restrict__ B, int ldb,
                                               float init, float* __restrict__ C, int ldc, int* __restrict__ argmax) {
    constexpr int U = V == 1 ? 8 : 4, S = 64 / G, P = 4 * S;
    __shared__ float s_acc[4][G * V];
    __shared__ uint32_t s_arg[4][G * V];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l = lane & (G - 1), part = w * S + lane / G;
    const int col = (tile * G + l) * V;
    const bool active = col < N;
    const float* bp = B + (active ? col : 0);
    int idle = 0;  // windows of 64 rows in a row that held no entry, as in max_long_rows
    for (int rb = uniform(rows_ending_by_wave(j0, rowptr, M)); rb < M;) {
        const int rl = rb + lane;
        const int sl = rl < M ? rowptr[rl] : INT_MAX, el = rl < M ? rowptr[rl + 1] : INT_MAX;
        // the same for the four waves, so they meet at the same barriers
        uint64_t longs = __ballot(rl < M && el - sl > long_row && sl >= j0 && sl < j1);
        for (; longs; longs &= longs - 1) {
            const int k = __builtin_ctzll(longs);
            // (a malformed rowptr cannot carry the walk past nonzero nnz)
            const int r = rb + k, s = read_lane(sl, k), e = min(read_lane(el, k), nnz);
            const int p0 = s + (int)((int64_t)(e - s) * part / P), p1 = s + (int)((int64_t)(e - s) * (part + 1) / P);
            float acc[V];
            uint32_t arg[V];
            bool nan[V];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                acc[v] = -__builtin_inff();
                arg[v] = kNoPos;
                nan[v] = false;
            }
            for (int base = p0; base < p1; base += G) {
                const int n = min(G, p1 - base);
                int c = 0;
                float a = 0.0f;
                if (l < n) {
                    c = colind[base + l];
                    a = val ? val[base + l] : 1.0f;
                }
                for (int i = 0; i < n; i += U) {
                    float b[U][V], f[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {  // past n: again the last entry, not folded
                        const int q = min(i + u, n - 1);
                        f[u] = __shfl(a, q, G);
                        load_v<V>(bp + (size_t)__shfl(c, q, G) * ldb, b[u]);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (i + u < n) {
#pragma unroll
                            for (int v = 0; v < V; ++v) {
                                const float x = f[u] * b[u][v];
                                const bool keep = acc[v] > x;
                                acc[v] = keep ? acc[v] : x;
                                arg[v] = keep ? arg[v] : (uint32_t)(base + i + u);
                                nan[v] |= x != x;
                            }
                        }
                }
            }
#pragma unroll
            for (int v = 0; v < V; ++v) {
                uint32_t g = arg[v] == kNoPos ? kNoPos : arg[v] | (nan[v] ? kSawNan : 0u);
#pragma unroll
                for (int d = 1; d < S; d <<= 1) {  // (lanes past the wave's end give what no one takes)
                    const float x = __shfl_down(acc[v], d * G);
                    const uint32_t q = __shfl_down(g, d * G);
                    max_join(acc[v], g, x, q);
                }
                if (lane < G) {
                    s_acc[w][l * V + v] = acc[v];
                    s_arg[w][l * V + v] = g;
                }
            }
            __syncthreads();
            if (w == 0 && lane < G && active) {
                float o[V];
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    float acc0 = init;
                    uint32_t g = kNoPos;
#pragma unroll
                    for (int q = 0; q < 4; ++q) max_join(acc0, g, s_acc[q][l * V + v], s_arg[q][l * V + v]);
                    o[v] = acc0;
                    if (argmax) argmax[(size_t)r * N + col + v] = g == kNoPos ? -1 : (int)(g & ~kSawNan);
                }
                store_v<V>(C + (size_t)r * ldc + col, o);
            }
            __syncthreads();  // the parts are read before the next row's are written
        }
        const int e63 = read_lane(el, 63);
        if (e63 >= j1) break;
        idle = e63 == read_lane(sl, 0) ? idle + 1 : 0;
        rb += 64;
        if (idle == 4) {
            rb = max(rb, uniform(rows_ending_by_wave(e63, rowptr, M)));
            idle = 0;
        }
    }
}

// Rows of at most long_row nonzeros, a group of G lanes each.
template <int V, int G>
__device__ __forceinline__ void max_short_rows(int blk, int tile, int M, int N, int nnz, int long_row,
                                               const int* __restrict__ rowptr, const int* __restrict__ colind,
                                               const float* __restrict__ val, const float* __restrict__ B, int ldb,
                                               float init, float* __restrict__ C, int ldc, int* __restrict__ argmax) {
    constexpr int U = 4;
    const int lane = threadIdx.x & (G - 1);
    const int row = (int)(((unsigned)blk * 256u + threadIdx.x) / G);
    if (row >= M) return;
    const int col = (tile * G + lane) * V;
    const bool active = col < N;
    const int beg = rowptr[row], stop = rowptr[row + 1];
    if (stop - beg > long_row) return;
    const int end = min(stop, nnz);  // (a malformed rowptr may promise more)
    const float* bp = B + (active ? col : 0);
    float acc[V];
    int arg[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        acc[v] = init;
        arg[v] = -1;
    }
    for (int base = beg; base < end; base += G) {  // the group's lanes load G entries at once
        const int n = min(G, end - base);
        int c = 0;
        float a = 0.0f;
        if (lane < n) {
            c = colind[base + lane];
            a = val ? val[base + lane] : 1.0f;
        }
        for (int k = 0; k < n; k += U) {
            float b[U][V], w[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {  // past n: again the last entry, not folded
                const int q = min(k + u, n - 1);
                w[u] = __shfl(a, q, G);
                load_v<V>(bp + (size_t)__shfl(c, q, G) * ldb, b[u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k + u < n) {
#pragma unroll
                    for (int v = 0; v < V; ++v) {
                        const float x = w[u] * b[u][v];
                        const bool keep = acc[v] > x;  // the reference's `acc > x ? acc : x`
                        acc[v] = keep ? acc[v] : x;
                        arg[v] = keep ? arg[v] : base + k + u;
                    }
                }
        }
    }
    if (!active) return;
    store_v<V>(C + (size_t)row * ldc + col, acc);
    if (argmax) {
#pragma unroll
        for (int v = 0; v < V; ++v) argmax[(size_t)row * N + col + v] = arg[v];
    }
}

// Workgroups [0, nlong · column tiles) walk the long rows (first: they take longest), the
// rest the short rows.  JOIN: `chunk` nonzeros a wave, whose parts k_max_join
// joins; the lanes hold the columns a group of the short walker covers in a quarter, a
// half or all of a wave.  Otherwise the rows that begin in `chunk` nonzeros a workgroup.
// (Column slices spread over the XCDs, as in the SpMM, do not pay: 78 -> 84 us on the
// R-MAT, 68 -> 70 us on the uniform matrix.)
// `first`: the launch's first workgroup, where they are more than one launch holds.
template <int V, int G, bool JOIN>
__global__ __launch_bounds__(256) void k_spmm_max(int first, int M, int N, int nnz, int nlong, int chunk, int nshort,
                                                  int long_row, const int* __restrict__ rowptr,
                                                  const int* __restrict__ colind, const float* __restrict__ val,
                                                  const float* __restrict__ B, int ldb, float init,
                                                  float* __restrict__ C, int ldc, int* __restrict__ argmax,
                                                  MaxParts parts) {
    constexpr int VL = V == 4 && G == 64 ? 4 : V == 4 && G == 32 ? 2 : 1;
    constexpr int tile = JOIN ? 64 * VL : G * V;
    const int ltiles = nlong ? (N + tile - 1) / tile : 0;
    const int b = first + (int)blockIdx.x;
    if (b < nlong * ltiles) {
        const int range = JOIN ? uniform((b / ltiles) * 4 + (int)(threadIdx.x >> 6)) : b / ltiles;
        const int64_t j0 = (int64_t)range * chunk;
        if (j0 >= nnz) return;
        const int j1 = (int)min(j0 + chunk, (int64_t)nnz);
        if constexpr (JOIN)
            max_long_rows<VL>(range, (int)j0, j1, (b % ltiles) * 64 * VL, M, N, long_row, rowptr, colind, val, B, ldb,
                              init, C, ldc, argmax, parts);
        else
            max_group_rows<V, G>((int)j0, j1, b % ltiles, M, N, nnz, long_row, rowptr, colind, val, B, ldb, init, C, ldc,
                                 argmax);
        return;
    }
    const int rb = b - nlong * ltiles;
    max_short_rows<V, G>(rb % nshort, rb / nshort, M, N, nnz, nlong ? long_row : INT_MAX, rowptr, colind, val, B, ldb,
                         init, C, ldc, argmax);
}

// A wave per cut row: the first of the waves that carry it folds their parts and the
// last part, of the wave in which the row ends, in order.
__global__ __launch_bounds__(256) void k_max_join(int nwaves, int N, MaxParts parts, float* __restrict__ C, int ldc,
                                                  int* __restrict__ argmax) {
    constexpr int U = 8;
    const int lane = threadIdx.x & 63;
    const int w = uniform((int)(blockIdx.x * 4u + (threadIdx.x >> 6)));
    if (w >= nwaves) return;
    const int idx = w - 1 + lane;  // lane 0: the previous wave, lane 1: this one
    const int cr = (idx >= 0 && idx < nwaves) ? parts.carry_row[idx] : -2;
    const int r = read_lane(cr, 1);
    if (r < 0 || read_lane(cr, 0) == r) return;
    int run = __builtin_ctzll(~(__ballot(cr == r) >> 1));  // waves from w on that carry row r
    if (run == 63) {
        for (int base = w + 63;; base += 64) {
            const int c2 = (base + lane < nwaves) ? parts.carry_row[base + lane] : -2;
            const uint64_t m = __ballot(c2 == r);
            const int cnt = (~m == 0ull) ? 64 : __builtin_ctzll(~m);
            run += cnt;
            if (cnt < 64) break;
        }
    }
    const int last = min(run, nwaves - 1 - w);  // (a malformed rowptr may end no row there)
    for (int col = lane; col < N; col += 64) {
        float acc = parts.val[(size_t)w * 2 * N + col];
        uint32_t arg = parts.arg[(size_t)w * 2 * N + col];
        if (arg != kNoPos) arg &= ~kSawNan;
        for (int k0 = 1; k0 <= last; k0 += U) {
            float x[U];
            uint32_t p[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = min(k0 + u, last);
                const size_t o = ((size_t)(w + k) * 2 + (k == run ? 1 : 0)) * N + col;
                x[u] = parts.val[o];
                p[u] = parts.arg[o];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k0 + u <= last) {
                    const bool keep = !(p[u] & kSawNan) && acc > x[u];
                    acc = keep ? acc : x[u];
                    arg = keep ? arg : p[u] & ~kSawNan;
                }
        }
        C[(size_t)r * ldc + col] = acc;
        if (argmax) argmax[(size_t)r * N + col] = (int)arg;
    }
}

// dB[colind[p]][j] += val[p]·dC[r][j] where p = argmax[r][j] (p = -1: the
// initial value won, no gradient; positions and columns out of range are
// skipped).  Many outputs can share a source row, so the adds are atomic
// (their order, and so the last bits, vary run to run).
//
// The hot source rows of a power-law matrix take a large share of the adds, and adds
// to one line follow one another in the L2: the 131,072-row R-MAT at N = 64 took 319
// us for 4.6M adds, a uniform matrix 165 us for 8.4M.  So a workgroup first adds
// into a small table of lines of dB (32 floats, the first lines that meet a slot
// keep it) in LDS and adds each line to memory once: 254 and 169 us.  All atomics on
// this memory are done beyond the L2 (every one is an EA request), so what bounds the
// rest is their number, 2 to 3 million requests.
constexpr int kBwdSlots = 512;      // lines of the table, 64 KiB
constexpr int kBwdThreads = 1024;
constexpr int kBwdItems = 8192;     // outputs of a workgroup

template <bool TABLE>
__global__ __launch_bounds__(kBwdThreads) void k_spmm_max_backward(int64_t total, int items, int K, int N,
                                                                   uint32_t inv_n, int nnz,
                                                                   const int* __restrict__ colind,
                                                                   const float* __restrict__ val,
                                                                   const float* __restrict__ dC, int ldc,
                                                                   const int* __restrict__ argmax,
                                                                   float* __restrict__ dB, int ldb) {
    constexpr int U = 4;
    __shared__ uint32_t tag[TABLE ? kBwdSlots : 1];  // line + 1, 0: free
    __shared__ float line[TABLE ? kBwdSlots : 1][32];
    const int nt = (int)blockDim.x;
    if constexpr (TABLE) {
        for (int i = threadIdx.x; i < kBwdSlots * 32; i += nt) (&line[0][0])[i] = 0.0f;
        for (int i = threadIdx.x; i < kBwdSlots; i += nt) tag[i] = 0u;
        __syncthreads();
    }
    const int64_t base = (int64_t)blockIdx.x * items;
    const int64_t rbase = base / N;
    const int jbase = (int)(base - rbase * N);
    for (int t0 = threadIdx.x; t0 < items; t0 += nt * U) {
        int p[U], c[U], j[U];
        float g[U];
#pragma unroll
        for (int u = 0; u < U; ++u) p[u] = t0 + nt * u < items && base + t0 + nt * u < total ? argmax[base + t0 + nt * u] : -1;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // row and column of the output: t / N by the reciprocal (inv_n = ceil(2^32 / N), exact
            // for N up to kBwdItems, where t < 2·kBwdItems); above that t < 2·N
            const uint32_t t = (uint32_t)jbase + t0 + nt * u;
            const uint32_t q = N == 1 ? t : N <= kBwdItems ? __umulhi(t, inv_n) : (t >= (uint32_t)N ? 1u : 0u);
            j[u] = (int)(t - q * (uint32_t)N);
            c[u] = -1;
            g[u] = 0.0f;
            if (p[u] >= 0 && p[u] < nnz) {
                c[u] = colind[p[u]];
                g[u] = dC[(rbase + q) * ldc + j[u]];
                if (val) g[u] *= val[p[u]];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c[u] < 0 || c[u] >= K) continue;
            const uint64_t at = (uint64_t)c[u] * ldb + j[u];
            if constexpr (TABLE) {
                const uint32_t ln = (uint32_t)(at >> 5);
                const int slot = (int)((ln * 2654435761u) >> 23);
                uint32_t have = tag[slot];
                if (have == 0u) have = atomicCAS(&tag[slot], 0u, ln + 1u);
                if (have == 0u || have == ln + 1u) {
                    atomicAdd(&line[slot][at & 31u], g[u]);
                    continue;
                }
            }
            atomicAdd(dB + at, g[u]);
        }
    }
    if constexpr (TABLE) {
        __syncthreads();
        for (int i = threadIdx.x; i < kBwdSlots * 32; i += nt) {
            const uint32_t have = tag[i >> 5];
            const float x = line[i >> 5][i & 31];
            if (have != 0u && x != 0.0f) atomicAdd(dB + ((uint64_t)(have - 1u) * 32 + (i & 31)), x);
        }
    }
}

template <int V>
int launch_max(int G, int first, unsigned grid, hipStream_t s, int M, int N, int nnz, int nlong, int chunk, bool join,
               int nshort, int long_row, const int* rp, const int* ci, const float* va, const float* B, int ldb, float init,
               float* C, int ldc, int* arg, const MaxParts& parts) {
    switch (G) {
#define ARMSP_MAX_CASE(GG)                                                                                          \
    case GG:                                                                                                        \
        if (join)                                                                                                   \
            hipLaunchKernelGGL((k_spmm_max<V, GG, true>), dim3(grid), dim3(256), 0, s, first, M, N, nnz, nlong, chunk, \
                               nshort, long_row, rp, ci, va, B, ldb, init, C, ldc, arg, parts);                     \
        else                                                                                                        \
            hipLaunchKernelGGL((k_spmm_max<V, GG, false>), dim3(grid), dim3(256), 0, s, first, M, N, nnz, nlong, chunk, \
                               nshort, long_row, rp, ci, va, B, ldb, init, C, ldc, arg, parts);                     \
        break;
        ARMSP_MAX_CASE(4)
        ARMSP_MAX_CASE(8)
        ARMSP_MAX_CASE(16)
        ARMSP_MAX_CASE(32)
        ARMSP_MAX_CASE(64)
#undef ARMSP_MAX_CASE
        default: return ARMSP_ERROR_INVALID_VALUE;
    }
    return ARMSP_SUCCESS;
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace
}  // namespace armsp

extern "C" int armsp_spmm_max_f32(int M, int K, int N, int nnz, const int* rowptr, const int* colind,
                                  const float* val, const float* B, int ldb, float init, float* C, int ldc,
                                  int* argmax, void* stream) {
    using namespace armsp;
    if (M < 0 || K < 0 || N < 0 || nnz < 0) return ARMSP_ERROR_INVALID_VALUE;
    if (M == 0 || N == 0) return ARMSP_SUCCESS;
    if (!rowptr || !C || ldc < N) return ARMSP_ERROR_INVALID_VALUE;
    if (nnz > 0 && (!colind || !B || ldb < N || K == 0)) return ARMSP_ERROR_INVALID_VALUE;
    hipStream_t s = as_stream(stream);
    const int V = (N % 4 == 0 && ldb % 4 == 0 && ldc % 4 == 0 && aligned16(B) && aligned16(C)) ? 4 : 1;
    int G = 4;
    while (G < 64 && G * V < N) G <<= 1;
    const int64_t nshort = ((int64_t)M * G + 255) / 256, stiles = (N + G * V - 1) / (G * V);
    if (stiles > 65535 || nshort * stiles > INT_MAX) return ARMSP_ERROR_NOT_SUPPORTED;
    const int long_row = max_long_row(M, nnz);
    // small inputs: a workgroup per long row, 64 nonzeros' rows each.  Else the long rows'
    // waves: 512 nonzeros each, fewer until 16 waves per CU are in flight
    const bool join = (int64_t)nnz * G > kMaxJoin;
    int chunk = join ? 512 : 64;
    while (chunk > 64 && nnz / chunk < 16 * device_cus()) chunk >>= 1;
    const int64_t nwaves = ((int64_t)nnz + chunk - 1) / chunk;
    const int VL = V == 4 && G == 64 ? 4 : V == 4 && G == 32 ? 2 : 1;
    const int64_t ltiles = join ? (N + 64 * VL - 1) / (64 * VL) : stiles;
    int64_t nlong = nnz <= long_row ? 0 : join ? (nwaves + 3) / 4 : nwaves;
    const size_t i4 = ((size_t)nwaves * 4 + 255) & ~(size_t)255;
    const size_t v4 = ((size_t)nwaves * 2 * N * 4 + 255) & ~(size_t)255;
    void* ws = nullptr;
    // (without workspace, as under capture with no arena reserved, every row is a short one)
    if (nlong * ltiles + nshort * stiles > INT_MAX ||
        (nlong && join && ws_alloc(&ws, i4 + 2 * v4, s) != ARMSP_SUCCESS))
        nlong = 0;
    char* w = static_cast<char*>(ws);
    const MaxParts parts{reinterpret_cast<int*>(w), reinterpret_cast<float*>(w + i4),
                         reinterpret_cast<uint32_t*>(w + i4 + v4)};
    const int64_t blocks = nlong * ltiles + nshort * stiles;
    TimedLaunch t("spmm_max", s);
    int st = ARMSP_SUCCESS;
    for (int64_t first = 0; first < blocks && !st; first += kMaxBlocks256) {
        const unsigned grid = (unsigned)std::min(blocks - first, kMaxBlocks256);
        st = V == 4 ? launch_max<4>(G, (int)first, grid, s, M, N, nnz, (int)nlong, chunk, join, (int)nshort, long_row,
                                    rowptr, colind, val, B, ldb, init, C, ldc, argmax, parts)
                    : launch_max<1>(G, (int)first, grid, s, M, N, nnz, (int)nlong, chunk, join, (int)nshort, long_row,
                                    rowptr, colind, val, B, ldb, init, C, ldc, argmax, parts);
    }
    if (!st && nlong && join)
        hipLaunchKernelGGL(k_max_join, dim3((unsigned)((nwaves + 3) / 4)), dim3(256), 0, s, (int)nwaves, N, parts, C,
                           ldc, argmax);
    const hipError_t e = hipGetLastError();
    if (ws) ws_free(ws, s);
    if (st) return st;
    if (e != hipSuccess) return hip_fail(e);
    t.stop();
    return ARMSP_SUCCESS;
}

extern "C" int armsp_spmm_max_backward_f32(int M, int K, int N, int nnz, const int* colind, const float* val,
                                           const float* dC, int ldc, const int* argmax, float* dB, int ldb,
                                           void* stream) {
    using namespace armsp;
    if (M < 0 || K < 0 || N < 0 || nnz < 0) return ARMSP_ERROR_INVALID_VALUE;
    if (M == 0 || N == 0 || nnz == 0) return ARMSP_SUCCESS;
    if (!colind || !dC || !argmax || !dB || ldc < N || ldb < N || K == 0) return ARMSP_ERROR_INVALID_VALUE;
    hipStream_t s = as_stream(stream);
    const int64_t n = (int64_t)M * N;
    // with a table where that still gives every CU a workgroup
    const bool table = n >= (int64_t)kBwdItems * device_cus();
    const int items = table ? kBwdItems : 1024;
    const int64_t nblk = (n + items - 1) / items;
    if (nblk > INT_MAX || (uint64_t)K * ldb / 32 >= 0xffffffffull) return ARMSP_ERROR_NOT_SUPPORTED;
    const uint32_t inv_n = (uint32_t)((((uint64_t)1 << 32) + N - 1) / N);
    TimedLaunch t("spmm_max", s);
    if (table)
        hipLaunchKernelGGL((k_spmm_max_backward<true>), dim3((unsigned)nblk), dim3(kBwdThreads), 0, s, n, items, K, N,
                           inv_n, nnz, colind, val, dC, ldc, argmax, dB, ldb);
    else
        hipLaunchKernelGGL((k_spmm_max_backward<false>), dim3((unsigned)nblk), dim3(256), 0, s, n, items, K, N,
                           inv_n, nnz, colind, val, dC, ldc, argmax, dB, ldb);
    ARMSP_LAUNCHED();
    t.stop();
    return ARMSP_SUCCESS;
}
