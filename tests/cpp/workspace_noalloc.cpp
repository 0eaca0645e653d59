// The allocation-free IterateAll takes the scratch that all handles of a device share only for what it has always taken it
// for: operands off their alignment are not packed there (such calls may overlap on several streams), and nothing is
// allocated.  Exit status 0 = it holds.
#include <cstdio>

#include "host_stubs.h"

int main()
{
    int failures = 0;
    for (int fp8 = 0; fp8 < 2; ++fp8)
        for (int tb = 0; tb < 2; ++tb)
            for (int64_t k : {40, 1003, 4096, 8192}) {
                ascq_matmul_t h = nullptr;
                ascq_matmul_types t{ASCQ_DT_INT8, ASCQ_DT_INT8, ASCQ_DT_INT32, 0, 0, 0};
                if (fp8) t.a_type = t.b_type = ASCQ_DT_FP8_E4M3, t.c_type = ASCQ_DT_F32;
                if (ascq_matmul_create(&t, &h) != ASCQ_OK) return 1;
                ascq_matmul_set_org_shape(h, 16, 4096, k);
                ascq_matmul_set_tensor_a(h, (void*)0x10000004, 0);  // A off its alignment
                ascq_matmul_set_tensor_b(h, (void*)0x20000000, tb);
                used.clear();
                if (ascq_matmul_iterate_all_noalloc(h, (void*)0x30000000, 0, nullptr) != ASCQ_OK) ++failures;
                for (const Region& r : used)
                    if (r.what[0] == 'p') {
                        std::printf("fp8 %d tb %d k %ld: %s in the shared scratch\n", fp8, tb, (long)k, r.what);
                        ++failures;
                    }
                if (!heap.empty()) ++failures;
                ascq_matmul_destroy(h);
            }
    std::printf("%d failure(s)\n", failures);
    return failures != 0;
}
