// Merge-path partition of a CSR matrix for the chunked merge kernels (SpMM,
// SpMV, SDDMM): part[w] = the rows consumed at diagonal min(w·chunk, M + nnz)
// of the merge of the M row ends with the nnz nonzeros, w = 0..nwaves.
//
// Row i's end is consumed at diagonal e(i) = rowptr[i+1] + i + 1, which grows
// strictly with i, so part[w] = #{i : e(i) <= w·chunk} and row i owns exactly
// the boundaries w with e(i-1) <= w·chunk < e(i) (e(-1) = 0; the extra thread
// i = M owns the rest, up to w = nwaves).  One thread per row reads two row
// pointers and writes the boundaries it owns: a streaming pass over rowptr
// instead of a binary search per boundary, and the same values
// merge_path_search gives.
#include "common.hpp"

namespace armsp {
namespace {

// *skew = 1 where a few columns take much of the matrix: of 2048 evenly spaced nonzeros,
// hashed to 4096 slots that keep the largest column they meet (so the count does not
// depend on the order), at least 48 find their own column there a second time.  Repeats
// counted without a hash: 126 on a 1M R-MAT of 2^24 nonzeros, 235 on one of 2^18 rows;
// 1 on a million uniform columns, 14 on 2^17.  One workgroup of 256.
constexpr int kSkewSamples = 2048, kSkewSlots = 4096, kSkewRepeats = 48;
__device__ void sample_columns(int nnz, const int* __restrict__ colind, int* __restrict__ skew) {
    constexpr int Q = kSkewSamples / 256, Z = kSkewSlots / 256;
    __shared__ int slot[kSkewSlots];
    __shared__ int repeats;
    int c[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) c[q] = colind[(int64_t)(q * 256 + (int)threadIdx.x) * nnz / kSkewSamples];
#pragma unroll
    for (int i = 0; i < Z; ++i) slot[i * 256 + threadIdx.x] = -1;
    if (threadIdx.x == 0) repeats = 0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) atomicMax(&slot[(unsigned)c[q] * 2654435761u >> 20], c[q]);
    __syncthreads();
    int n = 0;  // samples that are their slot's column, less the slots that hold one
#pragma unroll
    for (int q = 0; q < Q; ++q) n += slot[(unsigned)c[q] * 2654435761u >> 20] == c[q];
#pragma unroll
    for (int i = 0; i < Z; ++i) n -= slot[i * 256 + threadIdx.x] >= 0;
    atomicAdd(&repeats, n);
    __syncthreads();
    if (threadIdx.x == 0) *skew = repeats >= kSkewRepeats ? 1 : 0;
}

// SKEW: one more workgroup, the first, samples the columns beside the others' rows.
template <bool SKEW>
__global__ __launch_bounds__(256) void k_merge_partition(int M, int nnz, int chunk, int64_t nwaves,
                                                         const int* __restrict__ rowptr, int* __restrict__ part,
                                                         const int* __restrict__ colind, int* __restrict__ skew) {
    if constexpr (SKEW) {
        if (blockIdx.x == 0) {
            sample_columns(nnz, colind, skew);
            return;
        }
    }
    const int64_t i = (blockIdx.x - (SKEW ? 1 : 0)) * (int64_t)blockDim.x + threadIdx.x;
    if (i > M) return;
    const int64_t lo = i == 0 ? 0 : (int64_t)rowptr[i] + i;
    const int64_t hi = i < M ? (int64_t)rowptr[i + 1] + i + 1 : nwaves * chunk + 1;
    // clamped so that a malformed rowptr cannot write outside part[0..nwaves]
    int64_t wb = lo <= 0 ? 0 : (lo + chunk - 1) / chunk;
    int64_t we = hi <= 0 ? 0 : (hi + chunk - 1) / chunk;
    if (we > nwaves + 1) we = nwaves + 1;
    for (int64_t w = wb; w < we; ++w) part[w] = (int)i;
}

}  // namespace

int merge_partition(int M, int nnz, int chunk, int64_t nwaves, const int* rowptr, int* part, hipStream_t s,
                    const int* colind, int* skew) {
    const unsigned blocks = (unsigned)(((int64_t)M + 1 + 255) / 256);
    if (skew)
        hipLaunchKernelGGL((k_merge_partition<true>), dim3(blocks + 1), dim3(256), 0, s, M, nnz, chunk, nwaves, rowptr,
                           part, colind, skew);
    else
        hipLaunchKernelGGL((k_merge_partition<false>), dim3(blocks), dim3(256), 0, s, M, nnz, chunk, nwaves, rowptr,
                           part, colind, skew);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? ARMSP_SUCCESS : hip_fail(e);
}

}  // namespace armsp
