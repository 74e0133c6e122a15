// gemm_split.hpp — K splits of the prompt GEMMs' tiles.
#pragma once

#include "device.hpp"

namespace rie {

// Each of a tile's ks workgroups stores its partial sums; the one that arrives last adds
// them in split order (so the result does not depend on who that is), the others leave.
// Returns whether this workgroup holds the sums, in acc; every thread of all 256 calls it.
// Stores and loads go through to the device's coherence point (sc1, what agent-scope
// atomics use), so that workgroups on different XCDs need no cache write-back or
// invalidation, and a thread's NV sums are contiguous 16-byte pieces.
// part: ks·NV·256 floats per tile, bytes long in all; cnt: one zeroed int per tile, left
// zeroed.
// For launches of few tiles, whose partials are a few MB: there it takes about 5 µs, less
// than the second launch of the other form (19 tokens, wo 2048 × 2048, 32 tiles: 28 µs in
// one pass, 15 µs in four splits).  The coherent stores are no match for it on more (333
// tokens, down 2048 × 8192, 384 workgroups of 32 KB: 62 µs against 43 + 5 µs).
template <int NV>
__device__ __forceinline__ bool split_sum(float (&acc)[NV], float *part, uint32_t bytes, int *cnt, int tile, int ksi, int ks) {
    static_assert(NV % 16 == 0, "sums are moved 16 at a time");
    constexpr int SC1 = 16;
    __shared__ int arrived;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(part, 0, bytes, 0x00020000);
    const int tid = threadIdx.x;
    auto at = [&](int k) { return (int)(((uint32_t)(tile * ks + k) * 256u + (uint32_t)tid) * (NV * 4u)); };
#pragma unroll
    for (int v = 0; v < NV; v += 4) {
        const u32x4 x = {__float_as_uint(acc[v]), __float_as_uint(acc[v + 1]), __float_as_uint(acc[v + 2]), __float_as_uint(acc[v + 3])};
        __builtin_amdgcn_raw_buffer_store_b128(x, rs, at(ksi) + 4 * v, 0, SC1);
    }
    wait_vmem();
    __syncthreads();
    if (tid == 0) arrived = __hip_atomic_fetch_add(cnt + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != ks - 1) return false;
    if (tid == 0) __hip_atomic_store(cnt + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int v0 = 0; v0 < NV; v0 += 16) {
        for (int k = 0; k < ks; k += 4) {  // up to four splits' loads in flight (a split past the last repeats it)
            u32x4 x[4][4];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) x[j][i] = __builtin_amdgcn_raw_buffer_load_b128(rs, at(min(k + j, ks - 1)) + 4 * v0 + 16 * i, 0, SC1);
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float y = __uint_as_float(x[j][v / 4][v % 4]);
                    if (k + j == 0) acc[v0 + v] = y;
                    else if (k + j < ks) acc[v0 + v] += y;
                }
        }
    }
    return true;
}

// Number of K splits for split_sum: doubled while the partials (nv floats per thread) stay
// within 5 MB, each split keeps min_stages of the K loop and ws holds them.
inline int split_count(int tiles, int stages, int min_stages, int nv, const GemmWs &ws) {
    int ks = 1;
    if (!ws.part || tiles > ws.n_cnt) return 1;
    while (ks < 8 && tiles * (2 * ks) * nv <= 320 * 16 && stages / (2 * ks) >= min_stages && (size_t)tiles * (2 * ks) * 256 * nv <= ws.cap)
        ks *= 2;
    return ks;
}

// Number of K splits in planes, for one ungated segment: split 0 runs the epilogue on its
// partial sums, split i > 0 stores its own to plane i − 1 of ws ([n_tok][ld]), which a
// second launch adds to the output in split order.  Up to 4 while the launch has fewer
// than 512 workgroups (two per CU).
inline int plane_count(int tiles, int stages, int min_stages, size_t plane, const GemmWs &ws) {
    int ks = 1;
    while (ws.part && ks < 4 && tiles * ks < 512 && stages / (2 * ks) >= min_stages && (size_t)(2 * ks - 1) * plane <= ws.cap) ks *= 2;
    return ks;
}

}  // namespace rie
