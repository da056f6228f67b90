// Tiles of a model's rows and the tagged exchange between workgroups, shared by
// the resident recurrences (resident.hip: one FP64 vector, resident_block.hip:
// FP32 columns).
#pragma once

#include "common.hpp"

namespace tbtkx {
namespace {

// A workgroup's tile: first layer and row of it, extents.
struct Tile {
	int a, b, h, w;
};
__device__ __forceinline__ Tile tile_of(int L, int La, int A, int B, int tb, int g) {
	Tile t;
	t.a = g / tb * A;
	t.b = g % tb * B;
	t.h = t.a + A < La ? A : La - t.a;
	t.w = t.b + B < L ? B : L - t.b;
	return t;
}
struct Cell {
	int a, b;   // layer, row in it; may lie outside the grid
};
// d-th place of the frame of rectangle t that is fh layers and fw rows thick.
__device__ __forceinline__ Cell frame_cell(const Tile &t, int d, int fh, int fw) {
	const int band = fh * t.w;
	if (d < 2 * band) {
		const int q = d / t.w;
		return Cell{t.a + (q < fh ? q : t.h - 2 * fh + q), t.b + d - q * t.w};
	}
	const int q = (d - 2 * band) / (2 * fw), o = d - 2 * band - q * 2 * fw;
	return Cell{t.a + fh + q, t.b + (o < fw ? o : t.w - 2 * fw + o)};
}
__device__ __forceinline__ Tile grown(const Tile &t, int h, int w) {
	return Tile{t.a - h, t.b - w, t.h + 2 * h, t.w + 2 * w};
}
__device__ __forceinline__ int area(const Tile &t) { return t.h * t.w; }

// Exchanged words carry a tag in every 8-byte half. Stored and loaded at the
// device's coherence point (sc1); the loads are volatile, as they are polled.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kCoherent = 16, kVolatile = (int)0x80000000;
__device__ __forceinline__ u32x4 get(__amdgpu_buffer_rsrc_t b, uint32_t at) {
	return __builtin_amdgcn_raw_buffer_load_b128(b, at * 16u, 0, kCoherent | kVolatile);
}

constexpr long long kWaitTicks = 100000000ll;   // of the 100 MHz clock: one second

}  // namespace
}  // namespace tbtkx
