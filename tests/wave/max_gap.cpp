// max_long_rows (aggregate.hip): a wave whose range spans a million empty rows between two
// long ones, and ranges among sparse short rows.  Exit status 0: the long rows' results
// are right, and the wave takes no more than a few steps (cross-lane operations) for the gap.
#include "wave.hpp"

#include "aggregate.hip"

using namespace armsp;

static int fails = 0;

// long rows at the given places, a row of one entry after every `every` others
static int64_t walk(int M, const std::vector<int>& longs, int every, int j0, int j1) {
    std::vector<int> rowptr(M + 1, 0);
    for (int r = 0; r < M; ++r) {
        const bool is_long = std::find(longs.begin(), longs.end(), r) != longs.end();
        rowptr[r + 1] = rowptr[r] + (is_long ? 40 : every && r % every == 0);
    }
    const int nnz = rowptr[M];
    j1 = std::min(j1, nnz);
    std::vector<int> col(nnz);
    std::vector<float> B(97), C(M, -7.0f), part(2, -7.0f);
    for (int p = 0; p < nnz; ++p) col[p] = (p * 31) % 97;
    for (int i = 0; i < 97; ++i) B[i] = (float)((i * 55) % 97);
    std::vector<int> arg(M, -7), carry(1, -7);
    std::vector<uint32_t> part_arg(2, 0);
    const MaxParts parts{carry.data(), part.data(), part_arg.data()};
    wave::run_wave([&](int) {
        max_long_rows<1>(0, j0, j1, 0, M, 1, 32, rowptr.data(), col.data(), (const float*)nullptr, B.data(), 1, -1.0f,
                         C.data(), 1, arg.data(), parts);
    });
    for (int r = 0; r < M; ++r) {
        float want = -7.0f;
        int at = -7;
        if (rowptr[r + 1] - rowptr[r] > 32 && rowptr[r] >= j0 && rowptr[r + 1] <= j1) {
            want = -1.0f;
            for (int p = rowptr[r]; p < rowptr[r + 1]; ++p)
                if (!(want > B[col[p]])) want = B[col[p]], at = p;
        }
        if ((C[r] != want || arg[r] != at) && ++fails < 10)
            std::printf("row %d of %d: %g at %d, not %g at %d\n", r, M, C[r], arg[r], want, at);
    }
    return wave::g_round;
}

int main() {
    walk(700, {0, 3, 200, 699}, 5, 0, 1 << 20);
    walk(7000, {6000}, 63, 17, 1 << 20);
    walk(100000, {1, 50000, 99999}, 700, 0, 1 << 20);
    const int64_t steps = walk(1 << 20, {2, (1 << 20) - 2}, 0, 0, 1 << 20);
    std::printf("%lld steps over a million empty rows\n", (long long)steps);
    if (steps > 2000) ++fails;
    return fails ? 1 : 0;
}
