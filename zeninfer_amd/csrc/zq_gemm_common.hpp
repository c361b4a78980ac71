// zq_gemm_common.hpp -- what the GEMM translation units share on the device.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace zq {

#ifndef ZQ_GEMM_XCD_BLOCKS
#define ZQ_GEMM_XCD_BLOCKS 1
#endif
// Tile of workgroup `id`: workgroups that an XCD receives (ids congruent mod
// 8) walk the token tiles of one weight panel before moving on.
__device__ __forceinline__ void tile_of(uint32_t tiles_m, uint32_t tiles_n, uint32_t id, uint32_t& tm, uint32_t& tn) {
    const uint32_t total = tiles_m * tiles_n;
    uint32_t slot = id;
    if (ZQ_GEMM_XCD_BLOCKS && tiles_m % 4 == 0 && tiles_n % 2 == 0) {
        // XCD x (ids congruent to x mod 8) owns a quarter of the token tiles
        // and half of the weight panels, walking its token tiles per panel:
        // its activation rows stay in its L2, and each weight panel is read
        // by two XCDs.
        const uint32_t x = id % 8u, local = id / 8u, qm = tiles_m / 4;
        tm = (x & 3u) * qm + local % qm;
        tn = (x >> 2) * (tiles_n / 2) + local / qm;
        return;
    }
    if (total % 8u == 0) {
        const uint32_t per_xcd = total / 8u;
        slot = (id % 8u) * per_xcd + id / 8u;
    }
    tn = slot / tiles_m;
    tm = slot % tiles_m;
}

// A workgroup barrier that orders LDS only: unlike __syncthreads it does not
// wait for the wave's outstanding global loads (a prefetch stays in flight).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace zq
