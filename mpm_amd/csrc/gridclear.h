// gridclear.h -- the clear of touched storage blocks of a grid, for the
// kernels that do it (one scene, a batch, beside a small scene's sort).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mpm {

constexpr int kClearGroup = 8;  // storage blocks a wave takes at a time

// The blocks b0 + u of the bits u of todo (wave-uniform, below kClearGroup):
// their planes 0..nfields zero and their flags off; returns their nodes with
// mass > 0 (the active nodes of the step that wrote them) if count is set.
// The blocks' mass loads are all in flight before the first is used, and 16
// lanes clear a plane of a block with 16-byte stores, four planes at a time.
__device__ __forceinline__ unsigned long long clear_group(float* grid, int64_t plane, uint32_t* touched, int64_t b0,
                                                          uint32_t todo, int nfields, int lane, bool count) {
    unsigned long long cnt = 0;
    if (count) {
        float m[kClearGroup];
#pragma unroll
        for (int u = 0; u < kClearGroup; ++u) m[u] = (todo >> u) & 1u ? grid[(b0 + u) * 64 + lane] : 0.0f;
#pragma unroll
        for (int u = 0; u < kClearGroup; ++u) cnt += (unsigned long long)__popcll(__ballot(m[u] > 0.0f));
    }
    const int f0 = lane >> 4;
    float4* const at = reinterpret_cast<float4*>(grid + f0 * plane + b0 * 64) + (lane & 15);
#pragma unroll
    for (int u = 0; u < kClearGroup; ++u) {
        if (!((todo >> u) & 1u)) continue;
        for (int f = f0; f < nfields; f += 4) at[(f - f0) * (plane / 4) + u * 16] = float4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    if (lane < kClearGroup && ((todo >> lane) & 1u)) touched[b0 + lane] = 0u;
    return cnt;
}

}  // namespace mpm
