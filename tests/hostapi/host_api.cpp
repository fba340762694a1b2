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
    CHECK(armsp_spmm_max_f32(1000, 1000, 64, 100000, i32(), i32(), f32(), f32(), 64, -1e4f, f32(), 64, i32(), nullptr) ==
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

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "no_memory"))
        no_memory();
    else
        return 2;
    return fails ? 1 : 0;
}
