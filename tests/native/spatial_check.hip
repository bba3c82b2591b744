// Test entry point for ReSTIR's spatial pass: the kernel's register layouts (compiled
// for at most 5, 8 or 10 neighbours) on the caller's G-buffer, reservoirs and emitters.
#include "restir.hip"

// Device memory: g 5 x n float4 (point | bias, normal | roughness, geometric normal |
// metallic, albedo | flags, direction | distance), r n float4, m n floats, emitters 4
// float4 each; out_r and out_m receive the result.  0, or the HIP error.
extern "C" int check_spatial(uint32_t layout, const float4* g, const float4* r, const float* m, const float4* emitters,
                             uint32_t n_emitters, uint32_t w, uint32_t h, uint32_t k, float radius, uint64_t state,
                             float4* out_r, float* out_m) {
    using namespace snkpt;
    if (!g || !r || !m || !emitters || !n_emitters || !w || !h || !out_r || !out_m || k > layout) return -1;
    const size_t n = (size_t)w * h;
    float4* p = const_cast<float4*>(g);
    const GView G{p, p + n, p + 2 * n, p + 3 * n, p + 4 * n};
    SceneDev S{};
    S.emit_rec = emitters;
    S.n_emit = n_emitters;
    const uint32_t blocks = xcd_tile_blocks(w, h);
    if (layout == 5)
        k_spatial<5><<<blocks, kBlock>>>(S, G, r, m, out_r, out_m, w, h, k, radius, state);
    else if (layout == 8)
        k_spatial<kMaxSpatial><<<blocks, kBlock>>>(S, G, r, m, out_r, out_m, w, h, k, radius, state);
    else if (layout == 10)
        k_spatial<10><<<blocks, kBlock>>>(S, G, r, m, out_r, out_m, w, h, k, radius, state);
    else
        return -1;
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? (int)e : (int)hipDeviceSynchronize();
}
