// A caller's workspace off 16 bytes holds no packed operands, whose rows are written 16 bytes at a time: such calls run on the
// operands as they are, and none is refused.  Exit status 0 = it holds.
#include <cstdio>

#include "host_stubs.h"

int main()
{
    int failures = 0;
    for (int fp8 = 0; fp8 < 2; ++fp8)
        for (int tb = 0; tb < 2; ++tb)
            for (int64_t m : {16, 600})
                for (int64_t k : {1003, 4096})
                    for (uintptr_t off : {0, 1, 8}) {
                        ascq_matmul_t h = nullptr;
                        ascq_matmul_types t{ASCQ_DT_INT8, ASCQ_DT_INT8, ASCQ_DT_INT32, 0, 0, 0};
                        if (fp8) t.a_type = t.b_type = ASCQ_DT_FP8_E4M3, t.c_type = ASCQ_DT_F32;
                        if (ascq_matmul_create(&t, &h) != ASCQ_OK) return 1;
                        ascq_matmul_set_org_shape(h, m, 4096, k);
                        ascq_matmul_set_tensor_a(h, (void*)0x10000004, 0);  // A off its alignment
                        ascq_matmul_set_tensor_b(h, (void*)0x20000001, tb);
                        size_t bytes = 0;
                        if (ascq_matmul_workspace_size(h, &bytes) != ASCQ_OK || bytes == 0) return 1;
                        ascq_matmul_set_workspace(h, (void*)(0x40000000 + off), bytes);
                        used.clear();
                        const ascq_status s = ascq_matmul_iterate_all(h, (void*)0x30000000, 0, nullptr);
                        bool packed = false;
                        for (const Region& r : used) packed |= r.what[0] == 'p';
                        if (s != ASCQ_OK || packed != (off == 0)) {
                            std::printf("fp8 %d tb %d m %ld k %ld offset %zu: status %d (%s), packed %d\n", fp8, tb, (long)m,
                                        (long)k, (size_t)off, (int)s, s == ASCQ_OK ? "" : ascq_last_error(), (int)packed);
                            ++failures;
                        }
                        ascq_matmul_destroy(h);
                    }
    std::printf("%d failure(s)\n", failures);
    return failures != 0;
}
