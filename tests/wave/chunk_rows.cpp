// chunk_rows (common.hpp) without a partition: the rows of every chunk of a matrix, for
// row pointers that fit nnz and for ones that promise more or fewer entries than there
// are, or run backwards.  Exit status 0: every chunk stayed inside [0, M] x [0, nnz], and
// where the row pointers fit, met the plain merge-path search.
#include "wave.hpp"

#include "common.hpp"

#include <random>

using namespace armsp;

static int fails = 0;

static void chunks(const char* what, const std::vector<int>& rowptr, int nnz, int chunk, bool fits) {
    const int M = (int)rowptr.size() - 1;
    for (int64_t d = 0; d < (int64_t)M + nnz; d += chunk) {
        const int d0 = (int)d, d1 = (int)std::min<int64_t>(d + chunk, (int64_t)M + nnz);
        int i0 = -1, i1 = -1;
        wave::run_wave([&](int lane) {
            int a, b;
            chunk_rows(nullptr, d0 / chunk, d0, d1, rowptr.data(), M, nnz, a, b);
            if (lane == 0) i0 = a, i1 = b;
        });
        bool ok = 0 <= i0 && i0 <= i1 && i1 <= M && 0 <= d0 - i0 && d0 - i0 <= d1 - i1 && d1 - i1 <= nnz;
        if (fits) ok = ok && i0 == merge_path_search(d0, rowptr.data(), M, nnz) &&
                       i1 == merge_path_search(d1, rowptr.data(), M, nnz);
        if (!ok && ++fails < 10)
            std::printf("%s: M %d nnz %d chunk %d at %d: rows %d..%d, entries %d..%d\n", what, M, nnz, chunk, d0, i0, i1,
                        d0 - i0, d1 - i1);
    }
}

int main() {
    std::mt19937 rng(1);
    for (int chunk : {64, 128, 512})
        for (int M : {1, 63, 100, 1000})
            for (int mean : {0, 1, 10, 300}) {
                std::vector<int> rp(M + 1, 0);
                for (int i = 0; i < M; ++i) {
                    const int len = mean ? (int)(rng() % (2 * mean + 1)) : 0;
                    rp[i + 1] = rp[i] + (rng() % 50 == 0 ? len * 20 : rng() % 3 == 0 ? 0 : len);
                }
                const int nnz = rp[M];
                chunks("fits", rp, nnz, chunk, true);
                chunks("promises more", rp, nnz * 7 / 10, chunk, nnz == 0);
                chunks("promises more", rp, 0, chunk, nnz == 0);
                chunks("promises fewer", rp, nnz + 777, chunk, false);
                std::vector<int> back(rp);
                for (int& p : back)
                    if (rng() % 4 == 0) p = (int)(rng() % (2 * nnz + 2)) - nnz / 2;
                chunks("backwards", back, nnz, chunk, false);
            }
    std::printf("%d chunks out of bounds or misplaced\n", fails);
    return fails ? 1 : 0;
}
