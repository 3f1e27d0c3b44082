// Which kernel an FP32 GEMM runs on, and the workspace of that choice.
#include "cdx_internal.hpp"

namespace cdx {

size_t gemm_f32_workspace(const GemmArgs& g) {
    if (const int nk = narrow_kind(g)) return nk == 3 ? skinny_m_workspace(g) : 0;
    // a query knows no leading dimensions, which some routes limit: enough for
    // every route the product may take
    const size_t parts = gemm_parts_ok(g) ? gemm_parts_workspace(g) : 0;
    const size_t tiled = gemm_f32_tiled_workspace(g);
    return parts > tiled ? parts : tiled;
}

namespace {

enum class F32Route { Narrow, Parts, Direct, Tiled };

// (a workspace too small for the three-part kernel's slices leaves the product
// to the others)
F32Route route_of(const GemmArgs& g) {
    if (narrow_kind(g)) return F32Route::Narrow;
    if (gemm_parts_ok(g) && !(g.ws && g.ws_bytes < gemm_parts_workspace(g))) return F32Route::Parts;
    return gemm_direct_ok(g) ? F32Route::Direct : F32Route::Tiled;
}

}  // namespace

const char* gemm_f32_kernel_name(const GemmArgs& g) {
    switch (route_of(g)) {
        case F32Route::Narrow: return "narrow";
        case F32Route::Parts: return "parts";
        case F32Route::Direct: return "direct";
        default: return "tiled";
    }
}

int launch_gemm_f32(const GemmArgs& g, hipStream_t stream) {
    const F32Route r = route_of(g);
    // a caller's workspace is held to what the tiled route needs
    if (r != F32Route::Narrow && g.ws && g.ws_bytes < gemm_f32_tiled_workspace(g))
        return set_error(CDX_ERR_WORKSPACE, "gemm: workspace too small");
    switch (r) {
        case F32Route::Narrow: return launch_gemm_narrow(g, stream);
        case F32Route::Parts: return launch_gemm_parts(g, stream);
        case F32Route::Direct: return launch_gemm_direct(g, stream);
        default: return launch_gemm_f32_tiled(g, stream);
    }
}

}  // namespace cdx
