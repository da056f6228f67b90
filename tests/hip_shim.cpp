// Test shim over the HIP runtime: loaded with RTLD_GLOBAL before libtbtkx.so, its
// functions take the place of the runtime's and pass the calls on. No HIP headers:
// only the calls' C signatures are needed.
#include <dlfcn.h>

#include <cstddef>
#include <cstdint>

namespace {
struct Dim3 {
	uint32_t x, y, z;
};
void *real(const char *name) {
	static void *lib = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_LOCAL);
	return lib ? dlsym(lib, name) : nullptr;
}
}  // namespace

extern "C" {

int shim_launches = 0;      // kernel launches

int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **args, size_t lds, void *stream) {
	typedef int (*F)(const void *, Dim3, Dim3, void **, size_t, void *);
	static F fn = (F)real("hipLaunchKernel");
	shim_launches++;
	return fn(f, grid, block, args, lds, stream);
}

}  // extern "C"
