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

int launch_gemm_f32(const GemmArgs& g, hipStream_t stream) {
    if (narrow_kind(g)) return launch_gemm_narrow(g, stream);
    // a caller's workspace is held to what the tiled route needs; one too small
    // for the three-part kernel's slices leaves the product to the others
    if (g.ws && g.ws_bytes < gemm_f32_tiled_workspace(g))
        return set_error(CDX_ERR_WORKSPACE, "gemm: workspace too small");
    if (gemm_parts_ok(g) && !(g.ws && g.ws_bytes < gemm_parts_workspace(g)))
        return launch_gemm_parts(g, stream);
    if (gemm_direct_ok(g)) return launch_gemm_direct(g, stream);
    return launch_gemm_f32_tiled(g, stream);
}

}  // namespace cdx
