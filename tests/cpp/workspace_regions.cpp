// Where an int8 / fp8 IterateAll puts what it keeps in a workspace: packed operands, transposed or converted operands and
// the K-split partials of one call must not share a byte, and must lie inside the memory the call may use.
// Exit status 0 = every call kept its regions apart.
#include <cstdio>
#include <string>

#include "host_stubs.h"

static int failures = 0, calls = 0, packed_and_split = 0;
static void check(const std::string& name, uintptr_t ws, size_t ws_bytes)
{
    ++calls;
    bool pk = false, sp = false;
    for (size_t i = 0; i < used.size(); ++i) {
        const Region& r = used[i];
        pk |= r.what[0] == 'p';
        sp |= r.what[0] == 's';
        bool inside = ws && r.at >= ws && r.at + r.bytes <= ws + ws_bytes;
        for (const auto& h : heap) inside |= r.at >= h.first && r.at + r.bytes <= h.first + h.second;
        if (!inside) {
            std::printf("%s: %s at %#zx + %#zx outside the workspace\n", name.c_str(), r.what, (size_t)r.at, r.bytes);
            ++failures;
        }
        for (size_t j = 0; j < i; ++j)
            if (r.at < used[j].at + used[j].bytes && used[j].at < r.at + r.bytes) {
                std::printf("%s: %s at %#zx + %#zx overlaps %s at %#zx + %#zx\n", name.c_str(), r.what, (size_t)r.at, r.bytes,
                            used[j].what, (size_t)used[j].at, used[j].bytes);
                ++failures;
            }
    }
    packed_and_split += pk && sp;
}

int main()
{
    struct Shape {
        int64_t m, n, k;
    };
    const Shape orgs[] = {{1000, 4096, 8200}, {1000, 4096, 8192}, {16, 8192, 8192}, {16, 4096, 11003}, {64, 4096, 8192},
                          {128, 4096, 8196}, {16, 12800, 4096}, {700, 12800, 4104}, {16, 4096, 8192}, {40, 2050, 8195}};
    const Shape singles[] = {{0, 0, 0}, {16, 4096, 8192}, {16, 2048, 8192}, {64, 4096, 8192}, {16, 12288, 4096}, {1, 1030, 8192}};
    for (int fp8 = 0; fp8 < 2; ++fp8)
        for (const Shape& o : orgs)
            for (const Shape& s : singles)
                for (int layout = 0; layout < 6; ++layout)      // B [K, N], [N, K], NZ; A [M, K], [K, M]
                    for (int off = 0; off < 4; ++off)           // A, B off their alignment
                        for (int where = 0; where < 4; ++where) {  // owned, the reported size, a roomy one, the scratch
                            if (s.m > o.m || s.n > o.n || s.k > o.k) continue;
                            const int tb = layout % 3 == 1, nz = layout % 3 == 2, ta = layout >= 3;
                            ascq_matmul_t h = nullptr;
                            ascq_matmul_types t{ASCQ_DT_INT8, ASCQ_DT_INT8, ASCQ_DT_INT32, 0, 0, nz ? ASCQ_FORMAT_NZ : ASCQ_FORMAT_ND};
                            if (fp8) t.a_type = t.b_type = ASCQ_DT_FP8_E4M3, t.c_type = ASCQ_DT_F32;
                            if (ascq_matmul_create(&t, &h) != ASCQ_OK) std::abort();
                            ascq_matmul_set_org_shape(h, o.m, o.n, o.k);
                            if (s.m) ascq_matmul_set_single_shape(h, s.m, s.n, s.k);
                            ascq_matmul_set_tensor_a(h, (void*)(uintptr_t)(0x10000000 + (off & 1) * 4), ta);
                            ascq_matmul_set_tensor_b(h, (void*)(uintptr_t)(0x20000000 + (off >> 1) * 2), tb);
                            size_t ws = 0;
                            ascq_matmul_workspace_size(h, &ws);
                            const uintptr_t at = where == 1 || where == 2 ? 0x4000000000ull : 0;
                            const size_t bytes = where == 2 ? ws + (64 << 20) : ws;
                            if (at && bytes) ascq_matmul_set_workspace(h, (void*)at, bytes);
                            char name[160];
                            std::snprintf(name, sizeof name, "fp8 %d org %ld x %ld x %ld single %ld x %ld x %ld layout %d off %d ws %d",
                                          fp8, (long)o.m, (long)o.n, (long)o.k, (long)s.m, (long)s.n, (long)s.k, layout, off, where);
                            for (int call = 0; call < 2; ++call) {
                                used.clear();
                                const ascq_status st = where == 3 ? ascq_matmul_iterate_all_noalloc(h, (void*)0x30000000, 0, nullptr)
                                                                  : ascq_matmul_iterate_all(h, (void*)0x30000000, 0, nullptr);
                                if (st != ASCQ_OK && !(where == 3 && st == ASCQ_E_UNSUPPORTED)) {
                                    std::printf("%s: status %d (%s)\n", name, st, ascq_last_error());
                                    ++failures;
                                }
                                if (st == ASCQ_OK)
                                    check(name, where == 3 ? 0x80000000ull : at, where == 3 ? ASCQ_NOALLOC_SCRATCH_BYTES : bytes);
                            }
                            ascq_matmul_destroy(h);
                            if (!heap.empty()) {
                                std::printf("%s: %zu allocations left\n", name, heap.size());
                                ++failures;
                                heap.clear();
                            }
                        }
    std::printf("%d calls, %d with packed operands and split partials, %d failure(s)\n", calls, packed_and_split, failures);
    return failures || !packed_and_split;
}
