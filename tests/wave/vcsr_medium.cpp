// vcsr_medium_rows (spmv.hip): one wave whose groups hold rows of very different lengths.
// The groups that are done first go round with the longest row, as often as it has
// iterations of 16 blocks, and each time step on by the number of groups of the launch.
// That step times the iterations passes 2^31 for a row of 524,288 blocks among 65,536
// groups; here a row of 320 blocks among 2^28.  Exit status 0: every row's sum is bit for
// bit the one of the format's order.
#include "wave.hpp"

#include "spmv.hip"

#include <random>

using namespace armsp;

template <bool FUSED>
static bool rows(const std::vector<int>& blocks, int ngg) {
    const int M = (int)blocks.size(), K = 4 * 64;
    std::mt19937 rng(M);
    std::uniform_real_distribution<float> U(-1.0f, 1.0f);
    std::vector<int> rowptr(M + 1, 0), list(M);
    for (int r = 0; r < M; ++r) rowptr[r + 1] = rowptr[r] + 4 * blocks[r], list[r] = M - 1 - r;
    std::vector<int> col(rowptr[M]);
    std::vector<float> val(rowptr[M]), x(K), y(M), want;
    for (size_t p = 0; p < col.size(); ++p) {
        col[p] = p % 4 ? col[p - 1] + 1 : 4 * (int)(rng() % (K / 4));
        val[p] = U(rng);
    }
    for (float& f : x) f = U(rng);
    for (float& f : y) f = U(rng);
    want = y;
    for (int r = 0; r < M; ++r) {
        float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int p = rowptr[r]; p < rowptr[r + 1]; ++p) {
            const float a = val[p], b = x[col[p]];
            volatile float prod = a * b;  // rounded on its own
            s[p & 3] = FUSED ? std::fma(a, b, s[p & 3]) : s[p & 3] + prod;
        }
        want[r] += (s[0] + s[2]) + (s[1] + s[3]);
    }
    const int count[4] = {0, 0, M, 0};
    wave::run_wave([&](int lane) {
        vcsr_medium_rows<FUSED>(lane >> 4, ngg, list.data(), count, rowptr.data(), col.data(), val.data(), x.data(),
                                y.data());
    });
    const bool ok = std::memcmp(y.data(), want.data(), M * sizeof(float)) == 0;
    if (!ok) std::printf("rows differ: %d rows, step %d, fused %d\n", M, ngg, FUSED);
    return ok;
}

int main() {
    bool ok = rows<false>({17, 18, 33, 64, 65, 100, 256, 31, 32, 48, 49}, 4);
    ok &= rows<true>({17, 18, 33, 64, 65, 100, 256, 31, 32, 48, 49}, 4);
    ok &= rows<false>({18, 320, 17, 40}, 1 << 28);
    ok &= rows<true>({18, 320, 17}, 1 << 28);
    return ok ? 0 : 1;
}
