// The walkers of max aggregation (aggregate.hip) where rowptr promises more entries than
// there are: the arrays of entries end at an unmapped page.  Exit status 0: nothing past
// them was read, and the rows that exist in full are right.
#include "wave.hpp"

#include "aggregate.hip"

#include <sys/mman.h>
#include <unistd.h>

using namespace armsp;

// n values whose end is the end of the mapped memory
template <typename T>
static T* guarded(size_t n) {
    const size_t page = (size_t)sysconf(_SC_PAGESIZE), bytes = (n * sizeof(T) + page - 1) / page * page;
    char* p = (char*)mmap(nullptr, bytes + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    if (p == MAP_FAILED || mprotect(p + bytes, page, PROT_NONE)) std::abort();
    return (T*)(p + bytes) - n;
}

static int fails = 0;

static void check(const std::vector<int>& lens, int more, int long_row) {
    constexpr int G = 4, N = 4;
    const int M = (int)lens.size();
    int* rowptr = guarded<int>(M + 1);
    rowptr[0] = 0;
    for (int r = 0; r < M; ++r) rowptr[r + 1] = rowptr[r] + lens[r];
    const int nnz = rowptr[M];
    rowptr[M] += more;
    int* col = guarded<int>(nnz);
    float *val = guarded<float>(nnz), *B = guarded<float>(10 * N), *C = guarded<float>(M * N);
    int* arg = guarded<int>(M * N);
    for (int p = 0; p < nnz; ++p) col[p] = p * 7 % 10, val[p] = 1.0f;
    for (int i = 0; i < 10 * N; ++i) B[i] = (float)(i * 13 % 37);
    for (int i = 0; i < M * N; ++i) C[i] = -7.0f;
    for (int blk = 0; blk * (256 / G) < M; ++blk)
        for (wave::g_wave = 0; wave::g_wave < 4; ++wave::g_wave)
            wave::run_wave([&](int) {
                max_short_rows<1, G>(blk, 0, M, N, nnz, long_row, rowptr, col, val, B, N, -1.0f, C, N, arg);
            });
    for (int r = 0; r < M; ++r)
        for (int j = 0; j < N && lens[r] <= long_row && (r < M - 1 || lens[r] + more <= long_row); ++j) {
            float want = -1.0f;
            for (int p = rowptr[r]; p < std::min(rowptr[r + 1], nnz); ++p) want = std::max(want, B[col[p] * N + j]);
            if (C[r * N + j] != want && ++fails < 10) std::printf("row %d column %d: %g, not %g\n", r, j, C[r * N + j], want);
        }
    // the long rows by workgroups (all four waves' parts) and by waves
    for (int j0 = 0; j0 < nnz; j0 += 64)
        for (wave::g_wave = 0; wave::g_wave < 4; ++wave::g_wave)
            wave::run_wave([&](int) {
                max_group_rows<1, G>(j0, std::min(j0 + 64, nnz), 0, M, N, nnz, long_row, rowptr, col, val, B, N, -1.0f, C,
                                     N, arg);
            });
    wave::g_wave = 0;
    std::vector<int> carry(nnz / 64 + 1);
    std::vector<float> pv((nnz / 64 + 1) * 2 * N);
    std::vector<uint32_t> pa((nnz / 64 + 1) * 2 * N);
    for (int w = 0; w * 64 < nnz; ++w)
        wave::run_wave([&](int) {
            max_long_rows<1>(w, w * 64, std::min(w * 64 + 64, nnz), 0, M, N, long_row, rowptr, col, val, B, N, -1.0f, C, N,
                             arg, MaxParts{carry.data(), pv.data(), pa.data()});
        });
}

int main() {
    for (int more : {0, 1, 5, 63, 1000, 100000})
        for (int long_row : {32, 203, INT_MAX}) {
            check({3, 200}, more, long_row);
            check({0, 3, 0, 31, 33, 64, 1, 0, 700, 2}, more, long_row);
            check({5, 0, 0, 90, 0}, more, long_row);
        }
    return fails ? 1 : 0;
}
