// Test shim over the HIP runtime: loaded with RTLD_GLOBAL before libtbtkx.so, its
// functions take the place of the runtime's and pass the calls on, count some and
// refuse or alter some on the host, so that fallbacks run with nothing wrong on
// the device. No HIP headers: only the calls' C signatures are needed.
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
int shim_cooperative = 0;   // cooperative launches
int shim_refuse = 0;        // 1: cooperative launches are refused (too large)
int shim_malloc_limit = 0;  // > 0: no device memory for as many bytes or more
int shim_drop = 0;          // 1: cooperative launches lack their last workgroup
int shim_no_pinned = 0;     // 1: no pinned host memory
int shim_give_up = 0;       // 1: a 4-byte result copied to the host reads 1

int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **args, size_t lds, void *stream) {
	typedef int (*F)(const void *, Dim3, Dim3, void **, size_t, void *);
	static F fn = (F)real("hipLaunchKernel");
	shim_launches++;
	return fn(f, grid, block, args, lds, stream);
}

int hipMalloc(void **ptr, size_t bytes) {
	typedef int (*F)(void **, size_t);
	static F fn = (F)real("hipMalloc");
	// Refused by the runtime itself, which leaves its error behind.
	if (shim_malloc_limit > 0 && bytes >= (size_t)shim_malloc_limit) bytes = (size_t)1 << 60;
	return fn(ptr, bytes);
}

int hipHostMalloc(void **ptr, size_t bytes, unsigned flags) {
	typedef int (*F)(void **, size_t, unsigned);
	static F fn = (F)real("hipHostMalloc");
	return fn(ptr, shim_no_pinned ? (size_t)1 << 60 : bytes, flags);
}

int hipLaunchCooperativeKernel(const void *f, Dim3 grid, Dim3 block, void **args, unsigned lds,
                               void *stream) {
	shim_cooperative++;
	// An ordinary launch: only one process at a time has cooperative ones on a
	// GPU. Grids have at most a workgroup per compute unit, and waits are bounded.
	typedef int (*F)(const void *, Dim3, Dim3, void **, size_t, void *);
	static F fn = (F)real("hipLaunchKernel");
	if (shim_drop) grid.x--;
	if (!shim_refuse) return fn(f, grid, block, args, lds, stream);
	typedef int (*Malloc)(void **, size_t);
	static Malloc any_error = (Malloc)real("hipMalloc");
	void *p = nullptr;
	(void)any_error(&p, (size_t)1 << 60);
	return 720;   // hipErrorCooperativeLaunchTooLarge
}

static uint32_t *flag = nullptr;

int hipMemcpyAsync(void *dst, const void *src, size_t bytes, int kind, void *stream) {
	typedef int (*F)(void *, const void *, size_t, int, void *);
	static F fn = (F)real("hipMemcpyAsync");
	if (shim_give_up && bytes == 4 && kind == 2) flag = (uint32_t *)dst;
	return fn(dst, src, bytes, kind, stream);
}

int hipStreamSynchronize(void *stream) {
	typedef int (*F)(void *);
	static F fn = (F)real("hipStreamSynchronize");
	const int e = fn(stream);
	if (flag) *flag = 1;
	flag = nullptr;
	return e;
}

}  // extern "C"
