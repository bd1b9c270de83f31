// Host check of the grouped GEMM's activation row addressing: up to the last row a launch admits (65535
// tiles of 128 or 192 entries) every row starts a stride behind the one before it, past 4 and 64 GiB too. The
// kernels form their addresses with the same function.
#include "vbm_common.hpp"

#include <cstdio>
#include <initializer_list>

using namespace vbm;

int main() {
    for (int type : {39, 8})
        for (int64_t nb = 2; nb <= 128; nb += 2) {
            const GemmRowLayout lay{nb, type};
            const uint32_t last = 65535u * (type == 39 ? 128u : 192u) - 1;
            const uint64_t stride = static_cast<uint64_t>(lay.stride());
            for (uint64_t row = 0; row <= last; row += row + 9973 > last && row < last ? last - row : 9973) {
                const unsigned __int128 want = static_cast<unsigned __int128>(row) * stride;
                if (lay.row_offset(static_cast<uint32_t>(row)) != want) {
                    std::printf("type %d, %lld blocks: row %llu at the wrong offset\n", type, static_cast<long long>(nb),
                                static_cast<unsigned long long>(row));
                    return 1;
                }
            }
        }
    std::printf("rows addressed\n");
    return 0;
}
