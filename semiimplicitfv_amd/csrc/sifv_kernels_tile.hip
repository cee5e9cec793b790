// sifv_kernels_tile.hip - instantiations of the 2D tile stage kernel
// (five-point reconstructions, explicit stages).
#include "sifv_kernels.hpp"
#include "sifv_tile.hpp"

namespace sifv {
namespace {
template <int RS, int NPH, typename T>
StageFn<T> tile_of(bool lean, int nw) {
    if constexpr (NPH == 0) {
        if (lean)
            return nw == kTileSmall ? &stage_tile_kernel<3, RS, 0, false, T, false, kTileSmall>
                                    : &stage_tile_kernel<3, RS, 0, false, T, false, kTileWaves>;
    }
    return nw == kTileSmall ? &stage_tile_kernel<3, RS, NPH, false, T, true, kTileSmall>
                            : &stage_tile_kernel<3, RS, NPH, false, T, true, kTileWaves>;
}
template <int NPH, typename T>
StageFn<T> tile_by_rs(int rs, bool lean, int nw) {
    if (rs == 0) return tile_of<0, NPH, T>(lean, nw);
    if (rs == 1) return tile_of<1, NPH, T>(lean, nw);
    return tile_of<2, NPH, T>(lean, nw);
}
}  // namespace

template <>
StageFn<double> stage_tile_for<double>(int rs, int nph, bool lean, int nw) {
    return nph == 0 ? tile_by_rs<0, double>(rs, lean, nw) : nph == 2 ? tile_by_rs<2, double>(rs, lean, nw) : nullptr;
}
template <>
StageFn<float> stage_tile_for<float>(int rs, int nph, bool lean, int nw) {
    return nph == 0 ? tile_by_rs<0, float>(rs, lean, nw) : nullptr;
}

}  // namespace sifv
