// shkz_graph.hpp -- kernel nodes of an explicitly built hipGraph, and the key under which one is kept.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <tuple>
#include <type_traits>
#include <utility>

namespace shkz {

// Adds kernel<<<grid, block>>>(args...) to graph, after *last (when there is one), and makes it *last.
// The arguments are converted to the kernel's parameter types, as a launch converts them.
template <class... P, class... Args>
inline hipError_t add_kernel_node(hipGraph_t graph, hipGraphNode_t *last, dim3 grid, dim3 block, void (*kernel)(P...),
                                  Args... args) {
    static_assert(sizeof...(P) == sizeof...(Args), "one argument per kernel parameter");
    std::tuple<std::remove_cv_t<P>...> values(static_cast<std::remove_cv_t<P>>(args)...);
    return std::apply(
        [&](auto &...v) {
            void *params[] = {(void *)&v...};
            hipKernelNodeParams n{};
            n.func = (void *)kernel;
            n.gridDim = grid;
            n.blockDim = block;
            n.kernelParams = params;
            hipGraphNode_t node = nullptr;
            const hipError_t e = hipGraphAddKernelNode(&node, graph, *last ? last : nullptr, *last ? 1 : 0, &n);
            if (e == hipSuccess) *last = node;
            return e;
        },
        values);
}

// The key of a kept graph: the bytes of every value that its kernels' arguments depend on, each whole and
// in a fixed order.  (Formatted text in a buffer of a fixed size would lose its end when the pointers of a
// level grow long: two graphs of different arrays under one key.)
struct GraphKey {
    std::string bytes;
    template <class... V>
    void add(const V &...v) {
        static_assert(((std::is_arithmetic_v<V> || std::is_pointer_v<V>) && ...), "values without padding");
        (bytes.append(reinterpret_cast<const char *>(&v), sizeof(V)), ...);
    }
};

}  // namespace shkz
