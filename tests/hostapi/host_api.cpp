// The entry points' host code on a device that is out of memory, or at sizes that reach
// the launch limits (fake_hip.hpp).  Usage: host_api <check>; exit status 0: it held.
#include "fake_hip.hpp"

#include "armsp.h"

#include <cstring>

static int fails = 0;
#define CHECK(c)                                                        \
    do {                                                                \
        if (!(c)) {                                                     \
            std::printf("line %d: %s does not hold\n", __LINE__, #c);   \
            ++fails;                                                    \
        }                                                               \
    } while (0)

static float* f32() { return reinterpret_cast<float*>(1ull << 32); }  // aligned, never read
static int* i32() { return reinterpret_cast<int*>(1ull << 33); }

// Calls that can do without their workspace, or with less, when the allocator has none.
static void no_memory() {
    fake::reset();
    fake::memory = 0;
    CHECK(armsp_spmm_max_f32(1000, 1000, 64, 2000000, i32(), i32(), f32(), f32(), 64, -1e4f, f32(), 64, i32(), nullptr) ==
          ARMSP_SUCCESS);
    CHECK(fake::asked.size() == 1 && fake::launches.size() == 1);  // it asked, and ran without

    // an automatic SDDMM that would take 4 bytes a nonzero more to split its columns
    fake::reset();
    const int rows = 1 << 20, nnz = 1 << 24;
    fake::memory = 8 << 20;
    CHECK(armsp_sddmm_csr_f32(rows, rows, 128, nnz, i32(), i32(), nullptr, f32(), 128, f32(), 128, f32(), nullptr,
                              nullptr) == ARMSP_SUCCESS);
    CHECK(fake::asked.size() == 2 && fake::launches.size() == 2);  // the partition and the product
}

// Sizes that a device's memory holds, whose launches pass 2^32 threads if each row (or
// eight values) takes a workgroup's lanes of its own.
static void launch_limits() {
    fake::reset();
    CHECK(armsp_spmm_max_f32(16 << 20, 1000, 257, 1 << 20, i32(), i32(), nullptr, f32(), 257, -1e4f, f32(), 257, i32(),
                             nullptr) == ARMSP_SUCCESS);
    int64_t blocks = 0;
    for (const auto& l : fake::launches) blocks += l.grid.x;
    CHECK(blocks >= 5 * (int64_t)(16 << 20) / 4);  // five column tiles of 64, four rows a workgroup
    uint16_t* y = reinterpret_cast<uint16_t*>(i32());
    CHECK(armsp_convert_rows_f32_to_bf16(80 << 20, 264, f32(), 264, y, 264, nullptr) == ARMSP_SUCCESS);
    CHECK(armsp_convert_rows_f32_to_bf16(80 << 20, 33, f32(), 33, y, 33, nullptr) == ARMSP_SUCCESS);
    CHECK(armsp_convert_f32_to_bf16(((int64_t)1 << 35) + 8, f32(), y, nullptr) == ARMSP_SUCCESS);
}

// The transpose of a matrix of more than 2^20 columns (three passes) asks for at most the
// five arrays of nonzeros and the counts of 256 digits per 4096 that its first form took.
static void transpose_workspace() {
    const int nnz = 1 << 26;
    for (float* val : {(float*)nullptr, f32()}) {
        fake::reset();
        CHECK(armsp_csr_transpose(1 << 20, (1 << 20) + 1, nnz, i32(), i32(), val, i32(), i32(), val, nullptr) == ARMSP_SUCCESS);
        CHECK(fake::asked.size() == 1 && fake::asked[0] <= 5 * (size_t)nnz * 4 + (size_t)nnz / 4096 * 256 * 4);
    }
}

static bool launched(const std::string& part) {
    for (const auto& l : fake::launches)
        if (l.kernel.find(part) != std::string::npos) return true;
    return false;
}

// Gathers per batch (the last template argument) of an automatic product on rows of B under
// 32 columns, by type, width, the waves and the nonzeros a row holds.
static void narrow_batches() {
    int M = 141670, nnz = 870517;  // 6 a row, 7908 waves
    const uint8_t* q = reinterpret_cast<const uint8_t*>(f32());
    auto fp8 = [&](int nz, int n) {
        fake::reset();
        CHECK(armsp_spmm_fp8(M, M, n, nz, i32(), i32(), f32(), q, f32(), n, f32(), n, 0, nullptr, nullptr) == ARMSP_SUCCESS);
    };
    auto fp32 = [&](int nz, int n) {
        fake::reset();
        CHECK(armsp_spmm_f32(M, M, n, nz, i32(), i32(), f32(), f32(), n, f32(), n, 0, nullptr, nullptr) == ARMSP_SUCCESS);
    };
    for (int n : {5, 16, 31}) {
        fp8(nnz, n);
        CHECK(launched("k_spmm_streamIhfLi1ELi4E"));
        fp8(4 * nnz, n);
        CHECK(launched("k_spmm_streamIhfLi1ELi8E"));
        M = 50574;
        fp8(975971, n);  // 8021 waves
        CHECK(launched("k_spmm_streamIhfLi1ELi4E"));
        M = 20000;
        fp8(700000, n);  // 5625
        CHECK(launched("k_spmm_streamIhfLi1ELi8E"));
        M = 141670;
    }
    fp32(nnz, 16);
    CHECK(launched("k_spmm_streamIffLi1ELi8E"));
    fp32(nnz, 24);
    CHECK(launched("k_spmm_streamIffLi1ELi4E"));
    fp32(4 * nnz, 24);
    CHECK(launched("k_spmm_streamIffLi1ELi8E"));
}

// Rows per thread of the VCSR listing kernel: 256 workgroups or more where the matrix has them.
static void vcsr_listing() {
    const struct { int rows, per; } want[] = {{1 << 18, 1}, {(1 << 18) + 1, 2}, {200000, 1}, {1 << 20, 4}, {1 << 23, 8}};
    for (const auto& w : want) {
        fake::reset();
        CHECK(armsp_spmv_vcsr_f32(w.rows, 1 << 24, i32(), i32(), f32(), f32(), f32(), 0, nullptr) == ARMSP_SUCCESS);
        CHECK(launched("k_vcsr_find_longILi" + std::to_string(w.per) + "E"));
    }
    // the limit from which a row is long: by the blocks of the matrix
    const struct { int blocks, limit; } limits[] = {
        {5000, 64}, {1 << 17, 64}, {(1 << 17) + 1, 128}, {1 << 20, 128}, {(1 << 20) + 1, 256}, {1 << 28, 256}};
    for (const auto& w : limits) {
        fake::reset();
        CHECK(armsp_spmv_vcsr_f32(5000, 4 * w.blocks, i32(), i32(), f32(), f32(), f32(), 0, nullptr) == ARMSP_SUCCESS);
        for (const auto& l : fake::launches) CHECK(l.kernel.find("find_long") == std::string::npos || l.arg2 == w.limit);
    }
}

// A partition where the waves' searches, one per chunk and column slice, would be many.
static void partitions() {
    auto spmm = [&](int M, int nnz, int N) {
        fake::reset();
        float* p = reinterpret_cast<float*>(1ull << 34);  // on a 128-byte line, as slices need
        CHECK(armsp_spmm_f32(M, M, N, nnz, i32(), i32(), f32(), p, N, p, N, 0, nullptr, nullptr) == ARMSP_SUCCESS);
        CHECK(launched("k_spmm_slice"));
        return launched("k_merge_partition");
    };
    CHECK(!spmm(4000, 40000, 512));   // 688 chunks of 64, 8 slices
    CHECK(!spmm(10000, 100000, 256));  // 1719 and 4
    CHECK(spmm(10000, 100000, 512));   // 1719 and 8
    CHECK(spmm(20000, 200000, 512));
    CHECK(spmm(100000, 1000000, 256));
}

// Max aggregation of a small input is one launch and asks for no workspace.
static void max_launches() {
    for (int n : {4, 64}) {
        fake::reset();
        CHECK(armsp_spmm_max_f32(1024, 1024, n, 30000, i32(), i32(), nullptr, f32(), n, -1e4f, f32(), n, i32(), nullptr) ==
              ARMSP_SUCCESS);
        CHECK(fake::launches.size() == 1 && fake::asked.empty());
    }
    CHECK(armsp_spmm_max_f32(20000, 20000, 64, 600000, i32(), i32(), nullptr, f32(), 64, -1e4f, f32(), 64, i32(),
                             nullptr) == ARMSP_SUCCESS);
    CHECK(launched("k_max_join"));
}

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "no_memory"))
        no_memory();
    else if (!std::strcmp(what, "launch_limits"))
        launch_limits();
    else if (!std::strcmp(what, "transpose_workspace"))
        transpose_workspace();
    else if (!std::strcmp(what, "narrow_batches"))
        narrow_batches();
    else if (!std::strcmp(what, "vcsr_listing"))
        vcsr_listing();
    else if (!std::strcmp(what, "partitions"))
        partitions();
    else if (!std::strcmp(what, "max_launches"))
        max_launches();
    else
        return 2;
    return fails ? 1 : 0;
}
