// The key of a kept iteration graph tells apart any two calls whose kernels would take different arguments:
// every pointer and count of every level, changed alone, changes it, with pointers as long as the GPU's.
#include "../shiokaze_amd/csrc/shkz_runtime.hip"
#include "host_hip.hpp"

#include <cstdio>

int main() {
    shkz_ctx C;
    constexpr int LEVELS = 5;
    C.levels.resize(LEVELS);
    Problem P;
    P.nlev = LEVELS;
    P.ngrids = 64;
    uintptr_t next = 0x7ffe00000000;
    auto ptr = [&](auto &p) { p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(next += 0x200000); };
    ptr(P.red.partials);
    ptr(P.red2.partials);
    ptr(P.bottom);
    const void *vecs[13];
    for (const void *&v : vecs) ptr(v);
    for (LevelHost &L : C.levels) {
        L.nbricks = 1 << 20;
        L.desc.ngrids = 64;
        ptr(L.desc.bmap), ptr(L.desc.bxyz), ptr(L.desc.meta), ptr(L.desc.gl), ptr(L.desc.child64), ptr(L.desc.parent8);
        ptr(L.desc.uni), ptr(L.desc.nb27), ptr(L.dir), ptr(L.gx), ptr(L.gy), ptr(L.gz), ptr(L.idiag), ptr(L.rhs), ptr(L.z);
        ptr(L.tmp), ptr(L.res), ptr(L.ccode);
    }
    const std::string key = graph_key<float>(&C, P, vecs, 13, true);
    int same = 0, fields = 0;
    auto changed = [&](auto &field, const char *what, int level) {
        const auto was = field;
        if constexpr (std::is_pointer_v<std::remove_reference_t<decltype(field)>>) ptr(field);
        else if constexpr (std::is_same_v<std::remove_reference_t<decltype(field)>, bool>) field = !field;
        else field = field + 1;
        ++fields;
        if (graph_key<float>(&C, P, vecs, 13, true) == key) {
            ++same;
            std::printf("same key with another %s (level %d)\n", what, level);
        }
        field = was;
    };
    for (int l = 0; l < LEVELS; ++l) {
        LevelHost &L = C.levels[l];
        changed(L.nbricks, "nbricks", l), changed(L.any_coarsest, "any_coarsest", l), changed(L.desc.flat, "flat", l);
        changed(L.desc.ngrids, "ngrids", l), changed(L.desc.bmap, "bmap", l), changed(L.desc.bxyz, "bxyz", l);
        changed(L.desc.meta, "meta", l), changed(L.desc.gl, "gl", l), changed(L.desc.child64, "child64", l);
        changed(L.desc.parent8, "parent8", l), changed(L.desc.uni, "uni", l), changed(L.desc.nb27, "nb27", l);
        changed(L.dir, "dir", l), changed(L.gx, "gx", l), changed(L.gy, "gy", l), changed(L.gz, "gz", l);
        changed(L.idiag, "idiag", l), changed(L.rhs, "rhs", l), changed(L.z, "z", l), changed(L.tmp, "tmp", l);
        changed(L.res, "res", l), changed(L.ccode, "ccode", l);
    }
    changed(P.red.partials, "partials", -1), changed(P.red2.partials, "second partials", -1), changed(P.bottom, "bottom", -1);
    changed(P.bottom_level, "bottom level", -1), changed(P.omega, "omega", -1), changed(P.coarse_sweeps, "coarse sweeps", -1);
    changed(P.pre, "pre", -1), changed(P.post, "post", -1), changed(P.pre_c, "pre_c", -1), changed(P.post_c, "post_c", -1);
    changed(P.smoother, "smoother", -1), changed(P.local_k, "local_k", -1), changed(P.ngrids, "grids", -1);
    changed(P.multi_max_bricks, "multi_max_bricks", -1);
    for (const void *&v : vecs) changed(v, "vector", -1);
    std::printf("%d fields, %d lost\n", fields, same);
    if (!same) std::printf("OK\n");
    return same ? 1 : 0;
}
