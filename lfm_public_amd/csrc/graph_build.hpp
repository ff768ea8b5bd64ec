// graph_build.hpp -- step graphs put together node by node.
#pragma once

#include <hip/hip_runtime.h>

#include <tuple>
#include <type_traits>
#include <utility>

namespace lfm {

// A chain of kernel nodes.  The launches of a step become nodes here instead of
// being captured from the stream: a synchronous copy on any other thread of the
// process (another handle's set_field, or the program's own code) invalidates
// an open capture, also one of thread-local mode, and the launches that follow on
// that stream fail.
struct GraphBuild {
    hipGraph_t graph = nullptr;
    hipGraphNode_t last = nullptr;
    hipError_t err = hipSuccess;

    GraphBuild() { err = hipGraphCreate(&graph, 0); }
    ~GraphBuild() {
        if (graph) (void)hipGraphDestroy(graph);
    }
    GraphBuild(const GraphBuild &) = delete;
    GraphBuild &operator=(const GraphBuild &) = delete;

    // kernel(args...) after the nodes so far (the runtime copies the arguments)
    template <class... P, class... A>
    void add(void (*kernel)(P...), dim3 grid, dim3 block, const A &...args) {
        if (err != hipSuccess) return;
        std::tuple<std::remove_cv_t<P>...> vals(args...);
        void *ptrs[sizeof...(P)];
        std::apply(
            [&](auto &...v) {
                int i = 0;
                ((ptrs[i++] = (void *)&v), ...);
            },
            vals);
        hipKernelNodeParams p{};
        p.func = (void *)kernel;
        p.gridDim = grid;
        p.blockDim = block;
        p.kernelParams = ptrs;
        hipGraphNode_t node = nullptr;
        err = hipGraphAddKernelNode(&node, graph, last ? &last : nullptr, last ? 1 : 0, &p);
        last = node;
    }

    // hands the graph and its executable over; on failure neither is left
    hipError_t finish(hipGraph_t *g, hipGraphExec_t *exec) {
        if (err == hipSuccess) err = hipGraphInstantiate(exec, graph, nullptr, nullptr, 0);
        if (err != hipSuccess) {
            *exec = nullptr;
            (void)hipGetLastError();  // reported by the return
            return err;
        }
        *g = std::exchange(graph, nullptr);
        return hipSuccess;
    }
};

// a launch on o's stream, or a node of the graph that o is building
template <class Owner, class... P, class... A>
void launch(Owner *o, void (*kernel)(P...), dim3 grid, dim3 block, const A &...args) {
    if (o->building)
        o->building->add(kernel, grid, block, args...);
    else
        hipLaunchKernelGGL(kernel, grid, block, 0, o->stream, static_cast<std::remove_cv_t<P>>(args)...);
}

}  // namespace lfm
