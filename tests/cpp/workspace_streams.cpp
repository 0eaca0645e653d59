// Calls of one handle on different streams and devices may overlap: operands packed by them share no byte; a stream beyond
// the rooms a handle keeps packs nothing.  No room is allocated or freed in a way that would invalidate a capture of
// another stream.  Exit status 0 = all of it holds.
#include <cstdio>

#include "host_stubs.h"

static int failures = 0;
#define EXPECT(cond)                                   \
    do {                                               \
        if (!(cond)) {                                 \
            std::printf("line %d: %s\n", __LINE__, #cond); \
            ++failures;                                \
        }                                              \
    } while (0)

int main()
{
    for (int fp8 = 0; fp8 < 2; ++fp8) {
        ascq_matmul_t h = nullptr;
        ascq_matmul_types t{ASCQ_DT_INT8, ASCQ_DT_INT8, ASCQ_DT_INT32, 0, 0, 0};
        if (fp8) t.a_type = t.b_type = ASCQ_DT_FP8_E4M3, t.c_type = ASCQ_DT_F32;
        if (ascq_matmul_create(&t, &h) != ASCQ_OK) return 1;
        ascq_matmul_set_tensor_a(h, (void*)0x10000000, 0);
        ascq_matmul_set_tensor_b(h, (void*)0x20000000, 1);
        std::map<std::pair<int, uintptr_t>, std::vector<Region>> last;
        const std::pair<int, uintptr_t> where[] = {{0, 0}, {0, 0x100}, {1, 0}, {0, 0x200}, {0, 0x300}};
        for (int call = 0; call < 20; ++call) {
            const auto key = where[call * 3 % 5];
            ascq_matmul_set_org_shape(h, 100, 1000, call < 10 ? 1001 : 5001);  // (the rooms grow on the way)
            used.clear();
            device = key.first;
            EXPECT(ascq_matmul_iterate_all(h, (void*)0x30000000, 0, (void*)key.second) == ASCQ_OK);
            last[key] = used;
            for (const auto& a : last)
                for (const auto& b : last)
                    if (a.first != b.first)
                        for (const Region& x : a.second)
                            for (const Region& y : b.second) EXPECT(x.at >= y.at + y.bytes || y.at >= x.at + x.bytes);
        }
        int packing = 0;
        for (const auto& a : last) packing += !a.second.empty();
        EXPECT(packing == 4);
        device = 0;
        ascq_matmul_destroy(h);
        EXPECT(heap.empty());
        EXPECT(alloc_not_relaxed == 0);
        EXPECT(capture_mode == hipStreamCaptureModeGlobal);
    }
    // a room that costs more than one call gains is left to the second call of a handle
    const struct {
        int64_t m, n, k;
        int fp8, trans_b, first;
    } once[] = {{16, 4096, 1001, 0, 1, 0}, {16, 4096, 1001, 1, 1, 0}, {16, 4096, 1003, 0, 0, 1}, {16, 4096, 1003, 1, 0, 1},
                {1, 4100, 4095, 0, 1, 1},  {70, 200, 1003, 0, 1, 1},  {2000, 2000, 2001, 0, 1, 1}, {1000, 3000, 1001, 0, 1, 0}};
    for (const auto& c : once) {
        ascq_matmul_t h = nullptr;
        ascq_matmul_types t{ASCQ_DT_INT8, ASCQ_DT_INT8, ASCQ_DT_INT32, 0, 0, 0};
        if (c.fp8) t.a_type = t.b_type = ASCQ_DT_FP8_E4M3, t.c_type = ASCQ_DT_F32;
        if (ascq_matmul_create(&t, &h) != ASCQ_OK) return 1;
        ascq_matmul_set_org_shape(h, c.m, c.n, c.k);
        ascq_matmul_set_tensor_a(h, (void*)0x10000000, 0);
        ascq_matmul_set_tensor_b(h, (void*)0x20000000, c.trans_b);
        for (int call = 0; call < 3; ++call) {
            used.clear();
            EXPECT(ascq_matmul_iterate_all(h, (void*)0x30000000, 0, nullptr) == ASCQ_OK);
            EXPECT(!used.empty() == (call > 0 || c.first));
        }
        ascq_matmul_destroy(h);
    }
    // a short K is not packed while the any-alignment tiles take few rounds; what would run element by element always is
    const struct {
        int64_t m, n, k;
        int fp8, trans_b, packed;
    } small[] = {{32, 32, 40, 0, 1, 0},    {32, 32, 40, 0, 0, 0},   {300, 1000, 190, 1, 1, 0}, {300, 1000, 200, 1, 1, 1},
                 {2000, 4000, 100, 0, 1, 0}, {4000, 4000, 100, 0, 1, 1}, {32, 32, 40, 1, 0, 1},    {1, 64, 17, 1, 0, 1}};
    for (const auto& c : small) {
        ascq_matmul_t h = nullptr;
        ascq_matmul_types t{ASCQ_DT_INT8, ASCQ_DT_INT8, ASCQ_DT_INT32, 0, 0, 0};
        if (c.fp8) t.a_type = t.b_type = ASCQ_DT_FP8_E4M3, t.c_type = ASCQ_DT_F32;
        if (ascq_matmul_create(&t, &h) != ASCQ_OK) return 1;
        ascq_matmul_set_org_shape(h, c.m, c.n, c.k);
        ascq_matmul_set_tensor_a(h, (void*)0x10000004, 0);
        ascq_matmul_set_tensor_b(h, (void*)0x20000000, c.trans_b);
        for (int call = 0; call < 2; ++call) {
            used.clear();
            EXPECT(ascq_matmul_iterate_all(h, (void*)0x30000000, 0, nullptr) == ASCQ_OK);
        }
        EXPECT(!used.empty() == (c.packed != 0));
        ascq_matmul_destroy(h);
    }
    std::printf("%d failure(s)\n", failures);
    return failures != 0;
}
