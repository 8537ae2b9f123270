// fsg_lds.hip -- the tile kernels with the reference tables staged in LDS
// (k_tile_lds), in a translation unit of their own so that they compile in
// parallel with the others.
#include "tile_models.hpp"

namespace fsg {

template <class Model> static tile_fn fn_lds(LdsShape shape) {
    return shape == LDS_FULL ? k_tile_lds<Model, LDS_FULL> : shape == LDS_ORBIT ? k_tile_lds<Model, LDS_ORBIT>
                                                           : k_tile_lds<Model, LDS_PART>;
}
// One instantiation per combination of derivatives (der: bit 0 dz/dc, bit 1
// dz/dz), so that the step is straight-line code: z^2 + c for all four; z^d + c
// for the two that frames use (dz/dc, both), the others reading them from the
// launch arguments (z^3 + c at 1e-800 with dz/dc, with the BLA jump's change:
// 694 -> 587 us; z^6 + c 654 -> 551 us).
template <template <int> class Model> static tile_fn fn_lds_der(LdsShape shape, int der) {
    switch (der) {
        case 0: return fn_lds<Model<0>>(shape);
        case 1: return fn_lds<Model<1>>(shape);
        case 2: return fn_lds<Model<2>>(shape);
        default: return fn_lds<Model<3>>(shape);
    }
}
template <template <int> class Model> static tile_fn fn_lds_der2(LdsShape shape, int der) {
    return der == 1 ? fn_lds<Model<1>>(shape) : der == 3 ? fn_lds<Model<3>>(shape) : fn_lds<Model<-1>>(shape);
}
template <int DER> using M2Xr = HoloXr<KIND_M2, 2, false, DER>;
template <int DER> using M2Std = HoloStd<KIND_M2, 2, false, DER>;
template <int D> struct MnModels {
    template <int DER> using Xr = HoloXr<KIND_MN, D, false, DER>;
    template <int DER> using Std = HoloStd<KIND_MN, D, false, DER>;
};

tile_fn select_tile_lds(const LaunchCfg &c, LdsShape shape, int der) {
    if (c.orbit) return select_tile_orbit_lds(c, shape, der);
    if (c.kind == KIND_M2) return c.xr ? fn_lds_der<M2Xr>(shape, der) : fn_lds_der<M2Std>(shape, der);
    if (c.kind == KIND_MN) {
        switch (c.degree) {
#define FSG_MN(D) \
    case D: return c.xr ? fn_lds_der2<MnModels<D>::Xr>(shape, der) : fn_lds_der2<MnModels<D>::Std>(shape, der);
            FSG_MN(2) FSG_MN(3) FSG_MN(4) FSG_MN(5) FSG_MN(6) FSG_MN(7) FSG_MN(8)
#undef FSG_MN
            default: return nullptr;
        }
    }
    if (c.kind == KIND_BS) {
        switch (c.flavor) {
#define FSG_BS(F) \
    case F: \
        if (c.xr) return der & 1 ? fn_lds<BsXr<F, false, 1>>(shape) : fn_lds<BsXr<F, false, 0>>(shape); \
        return fn_lds<BsStd<F>>(shape);
            FSG_BS(1) FSG_BS(2) FSG_BS(3) FSG_BS(4) FSG_BS(5)
#undef FSG_BS
            default: return nullptr;
        }
    }
    return nullptr;
}

}  // namespace fsg
