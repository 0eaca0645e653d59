// What a captured graph may still use must stay allocated and untouched by later eager calls of the same handle: a handle
// whose captured calls keep K-split partials, a B converted from NZ or a transposed A in its own workspace, then eager
// calls with operands that are packed.  Exit status 0 = it does.
#include <cstdio>

#include "host_stubs.h"

static int failures = 0;
#define EXPECT(cond)                                             \
    do {                                                         \
        if (!(cond)) {                                           \
            std::printf("%s, line %d: %s\n", name, __LINE__, #cond); \
            ++failures;                                          \
        }                                                        \
    } while (0)

static bool alive(const Region& r)
{
    for (const auto& h : heap)
        if (r.at >= h.first && r.at + r.bytes <= h.first + h.second) return true;
    return false;
}
int main()
{
    uint8_t* const A = (uint8_t*)0x10000000;
    uint8_t* const B = (uint8_t*)0x20000000;
    void* const C = (void*)0x30000000;
    for (int fp8 = 0; fp8 < 2; ++fp8)
        for (int kind = 0; kind < 3; ++kind) {  // split partials; B from NZ; A transposed
            char name[64];
            std::snprintf(name, sizeof name, "fp8 %d kind %d", fp8, kind);
            ascq_matmul_t h = nullptr;
            ascq_matmul_types t{ASCQ_DT_INT8, ASCQ_DT_INT8, ASCQ_DT_INT32, 0, 0, kind == 1 ? ASCQ_FORMAT_NZ : ASCQ_FORMAT_ND};
            if (fp8) t.a_type = t.b_type = ASCQ_DT_FP8_E4M3, t.c_type = ASCQ_DT_F32;
            if (ascq_matmul_create(&t, &h) != ASCQ_OK) return 1;
            ascq_matmul_set_org_shape(h, 16, 4096, 8192);
            ascq_matmul_set_tensor_a(h, A, kind == 2);
            ascq_matmul_set_tensor_b(h, B, 1);
            EXPECT(ascq_matmul_iterate_all(h, C, 0, nullptr) == ASCQ_OK);
            used.clear();
            capturing = true;
            EXPECT(ascq_matmul_iterate_all(h, C, 0, nullptr) == ASCQ_OK);
            capturing = false;
            const std::vector<Region> graph = used;
            EXPECT(!graph.empty());
            // eager: a misaligned A, then (not NZ) a misaligned B, which needs more room
            for (int call = 0; call < 2; ++call) {
                used.clear();
                ascq_matmul_set_tensor_a(h, A + 4, 0);
                if (call && kind != 1) ascq_matmul_set_tensor_b(h, B + 1, 1);
                EXPECT(ascq_matmul_iterate_all(h, C, 0, nullptr) == ASCQ_OK);
                bool packed = false;
                for (const Region& r : used) packed |= r.what[0] == 'p';
                EXPECT(packed);
                for (const Region& r : graph) EXPECT(alive(r));
            }
            // captured calls with packed operands: no room that later eager calls share
            used.clear();
            capturing = true;
            EXPECT(ascq_matmul_iterate_all(h, C, 0, nullptr) == ASCQ_OK);
            capturing = false;
            for (const Region& r : used) EXPECT(r.what[0] != 'p');
            // ... but a caller's workspace is the call's own
            size_t ws = 0;
            ascq_matmul_workspace_size(h, &ws);
            if (kind == 0) {
                ascq_matmul_set_workspace(h, (void*)0x4000000000ull, ws);
                EXPECT(heap.empty());
                used.clear();
                capturing = true;
                EXPECT(ascq_matmul_iterate_all(h, C, 0, nullptr) == ASCQ_OK);
                capturing = false;
                bool packed = false;
                for (const Region& r : used) {
                    packed |= r.what[0] == 'p';
                    EXPECT(r.at >= 0x4000000000ull && r.at + r.bytes <= 0x4000000000ull + ws);
                }
                EXPECT(packed);
            }
            ascq_matmul_destroy(h);
            EXPECT(heap.empty());
        }
    std::printf("%d failure(s)\n", failures);
    return failures != 0;
}
