// Stands in front of three calls of the HIP runtime in a process that loads it before the library, so that
// a test can have the device refuse them: refuse_cooperative != 0 refuses every cooperative launch;
// refuse_malloc: the number of the hipMalloc to refuse, counted from 1 (0: none), mallocs: how many there were.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

namespace {
template <class F> F runtime(const char *name) {
    static void *const lib = dlopen("libamdhip64.so.7", RTLD_LAZY);
    return reinterpret_cast<F>(dlsym(lib, name));
}
}  // namespace

extern "C" {

int refuse_cooperative = 0, refuse_malloc = 0, mallocs = 0, refused = 0;

hipError_t hipLaunchCooperativeKernel(const void *f, dim3 grid, dim3 block, void **args, unsigned int lds, hipStream_t stream) {
    using Fn = hipError_t (*)(const void *, dim3, dim3, void **, unsigned int, hipStream_t);
    static const Fn real = runtime<Fn>("hipLaunchCooperativeKernel");
    if (refuse_cooperative) {
        refused++;
        return hipErrorCooperativeLaunchTooLarge;
    }
    return real(f, grid, block, args, lds, stream);
}

hipError_t hipMalloc(void **p, size_t bytes) {
    using Fn = hipError_t (*)(void **, size_t);
    static const Fn real = runtime<Fn>("hipMalloc");
    if (++mallocs == refuse_malloc) {
        refused++;
        return hipErrorOutOfMemory;
    }
    return real(p, bytes);
}

}  // extern "C"
