// Shared definitions of the flyguy MI355X library: error state, launch helpers, tile layout, lane helpers.
//
// Activation layout ("tiled"): a state tensor of N rows and B columns (B = batch, a multiple of 32) is stored
// as [T = B/32][N][32] fp32: one 128-byte line holds 32 samples of one row, and the N x 128 B "slab" of one
// tile is contiguous.  A workgroup works on one tile at a time, so the source slab it gathers from stays in
// the L2 of its XCD.  Kernels that serve the row-major [N][B] layout of the HopCuda-style boundary use the same
// code with different strides (row stride B, tile stride 32).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>

namespace fg {

constexpr int TW = 32;          // columns (samples) per tile
constexpr int TW16 = 64;        // samples per tile of 16-bit states (one 128-byte line)
constexpr int LPR = TW / 4;     // lanes per row: each lane holds a float4 of the tile
constexpr int RPW = 64 / LPR;   // rows per wave (8)
constexpr int WG = 256;         // threads per workgroup
constexpr int RPG = WG / LPR;   // rows per workgroup (32)
constexpr int SEG_MAX = 512;    // longest run of edges one lane group sums before a row is split into segments
constexpr int SEG_MIN_PER_TILE = 4096;   // segments a product should have per tile: >= 128 workgroups, so that the
                                         // workgroups resident on an XCD work on one or two tiles at a time (4096
                                         // measured 2-4% faster than 8192 and 2048 on the 3-hop benchmark network:
                                         // fewer split rows to combine, segments still short enough to balance)

// the segment cap of a product of E edges: SEG_MAX, lowered (not below 16) until there are SEG_MIN_PER_TILE segments
inline int seg_cap(long long E) {
    long long c = (E + SEG_MIN_PER_TILE - 1) / SEG_MIN_PER_TILE;
    return (int)(c < 16 ? 16 : (c > SEG_MAX ? SEG_MAX : c));
}

// Last error of this thread (set by a failing entry point, read by fc_last_error).
void set_error(const std::string& msg);
const char* last_error();
void clear_error();

// XCD-aware tile mapping: the hardware deals workgroups to the 8 XCDs round robin (block i -> XCD i % 8).
// Each XCD first works through whole tiles of its own, x, x+8, ..., one after another, row blocks inner, so its L2 holds
// one tile's source slab at a time.  The T % 8 tiles left are cut into 8 slices each (slice j: row blocks j, j+8, ...,
// an even sample of a plan sorted by length), and XCD x takes T % 8 consecutive slices, so that all XCDs get the same
// work and each reads at most two of those slabs.  The slices of one tile are walked together, in one pass from the
// plan's longest rows to its shortest: waves of one length walk their rows' ascending sources at one pace.  The slices
// of two tiles are walked one tile after the other, or all in one pass (together) where the plan's lengths differ so
// much that a second pass would begin with another chain of longest rows (Plan::stripe).
// Walking all tiles in plain order whenever T % 8 != 0 had every XCD read every slab: B=416 (13 tiles) on the benchmark
// network, forward 537 us, now 388; B=128 201 -> 160.  At B=416 the striped hops 1 / 2 take 135 / 174 us one tile after
// the other and 125 / 161 together; an Erdos-Renyi network's 114 / 167 and 114 / 180, its backward 176 / 165 and 182 /
// 177, the lognormal one's backward 173 / 166 and 178 / 175.
// A slice may be one block short: rb >= RB is a block without work.
__host__ __device__ inline long long tile_blocks(int RB, int T) {
    const int r = T & 7;
    return (long long)(T - r) * RB + 8LL * r * ((RB + 7) / 8);
}
__device__ __forceinline__ int tile_of(int bid, int RB, int T, int& rb, bool together = false) {
    const int x = bid & 7, r = T & 7, whole = (T >> 3) * RB;
    int s = bid >> 3;
    if (s < whole) {
        rb = s % RB;
        return x + 8 * (s / RB);
    }
    s -= whole;
    // slices i .. i + r - 1 (slice i: slice i % 8 of left tile i / 8), walked n at a time from slice i
    int i = x * r, n = r;
    if (!together) {
        n = min(8 - (i & 7), r);                // the first tile's
        const int first = n * ((RB + 7) / 8);
        if (s >= first) {                       // the next tile's
            s -= first;
            i += n;
            n = r - n;
        }
    }
    i += s % n;
    rb = (i & 7) + 8 * (s / n);
    return (T & ~7) + (i >> 3);
}

// a compile-time flag as a type (the hop kernels' step bodies take it: Full<true> for a step whose 8 slots are all
// needed, Full<false> for a wave's last step)
template <bool B>
struct Full {
    static constexpr bool value = B;
};

// broadcast lane (group_base + S) of each 8-lane group (ds_swizzle bit mode inside each 32-lane half)
template <int S>
__device__ __forceinline__ int bcast8(int v) { return __builtin_amdgcn_ds_swizzle(v, 0x18 | (S << 5)); }
template <int S>
__device__ __forceinline__ float bcast8f(float v) { return __int_as_float(bcast8<S>(__float_as_int(v))); }

// sum over the 8 lanes of a group (xor butterfly; every lane ends with the same value)
__device__ __forceinline__ float sum8(float v) {
    v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x1f | (1 << 10)));
    v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x1f | (2 << 10)));
    v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x1f | (4 << 10)));
    return v;
}

__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }

__device__ __forceinline__ void fma4(float w, const float4& v, float4& a) {
    a.x = fmaf(w, v.x, a.x); a.y = fmaf(w, v.y, a.y); a.z = fmaf(w, v.z, a.z); a.w = fmaf(w, v.w, a.w);
}
__device__ __forceinline__ void add4(const float4& v, float4& a) { a.x += v.x; a.y += v.y; a.z += v.z; a.w += v.w; }

}  // namespace fg

#define FG_CHECK(call, ret)                                                                  \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess) {                                                              \
            char b_[256];                                                                    \
            snprintf(b_, sizeof b_, "HIP error %s at %s:%d", hipGetErrorString(e_), __FILE__, __LINE__); \
            fg::set_error(b_);                                                               \
            return ret;                                                                      \
        }                                                                                    \
    } while (0)
