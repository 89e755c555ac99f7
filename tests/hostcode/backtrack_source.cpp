// The library's generated backtracking code of an element table (TEST
// INFRASTRUCTURE ONLY): the source, the element keys, the entry offsets in
// the kernel's order and the element programs.
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "xt_builder.h"
#include "xt_codegen.h"

namespace {
std::vector<int64_t> g_entry;
std::vector<double> g_prog;
std::vector<int32_t> g_rec;
std::string g_src;
}  // namespace

extern "C" int32_t xth_backtrack_source(const int32_t *types, const int64_t *offsets,
                                        const double *params, int64_t n, int64_t *sizes) {
    std::vector<int64_t> entry, bt;
    std::string err;
    g_prog.clear();
    int st = xt_build_program(types, offsets, params, n, entry, g_prog, err, &bt);
    if (st) return st;
    g_entry.assign(bt.rbegin(), bt.rend());
    st = xt_generate_backtrack_source(g_entry, g_prog, 0, g_src, g_rec, err);
    sizes[0] = (int64_t)g_src.size();
    sizes[1] = (int64_t)g_prog.size();
    return st;
}

extern "C" void xth_backtrack_copy(char *src, int32_t *rec, int64_t *entry, double *prog) {
    std::memcpy(src, g_src.data(), g_src.size());
    std::memcpy(rec, g_rec.data(), g_rec.size() * sizeof(int32_t));
    std::memcpy(entry, g_entry.data(), g_entry.size() * sizeof(int64_t));
    std::memcpy(prog, g_prog.data(), g_prog.size() * sizeof(double));
}
