// fsg_orbit.hip -- the calc_orbit instantiations of the tile kernel
// (perturbation.py:1096-1101, 1266-1273, 1390-1396), in a translation unit
// of their own so that they compile in parallel with the others.
#include "tile_models.hpp"

namespace fsg {

template <class Model> static tile_fn fn_of() { return k_tile<Model>; }

tile_fn select_tile_orbit(const LaunchCfg &c, int der) {
    if (c.kind == KIND_M2)
        return c.xr ? fn_of<HoloXr<KIND_M2, 2, true>>() : der == 3 ? fn_of<HoloStd<KIND_M2, 2, true, 3>>() : fn_of<HoloStd<KIND_M2, 2, true>>();
    if (c.kind == KIND_MN) {
        switch (c.degree) {
#define FSG_MN(D) case D: return c.xr ? fn_of<HoloXr<KIND_MN, D, true>>() : fn_of<HoloStd<KIND_MN, D, true>>();
            FSG_MN(2) FSG_MN(3) FSG_MN(4) FSG_MN(5) FSG_MN(6) FSG_MN(7) FSG_MN(8)
#undef FSG_MN
            default: return nullptr;
        }
    }
    if (c.kind == KIND_BS) {
        switch (c.flavor) {
#define FSG_BS(F) case F: return c.xr ? fn_of<BsXr<F, true>>() : fn_of<BsStd<F, true>>();
            FSG_BS(1) FSG_BS(2) FSG_BS(3) FSG_BS(4) FSG_BS(5)
#undef FSG_BS
            default: return nullptr;
        }
    }
    return nullptr;
}

// The same with the tables in LDS: z^2 + c and, with binary64 deltas, z^d + c
// compiled for the derivatives that frames use (dz/dc, both), the others reading
// them from the launch arguments.  With that and the recorder a z^d + c step held
// more conditions than there are scalar registers: 400x400 around the critical
// orbit z^3 + c 1278 -> 650 us, z^6 + c 1917 -> 1068 us (1835 from global memory).
// 1001x667 with dz/dc, from global memory with every step through the recorder
// and now: 133 -> 119 us at 1e-150, 171 -> 135 at 1e-300; the burning ship with
// extended range spills here and is faster all the same (1e-800: 421 -> 379).
template <class Model> static tile_fn fn_lds(LdsShape shape) {
    return shape == LDS_FULL ? k_tile_lds<Model, LDS_FULL> : k_tile_lds<Model, LDS_PART>;
}
template <template <int> class Model> static tile_fn fn_lds_der2(LdsShape shape, int der) {
    return der == 1 ? fn_lds<Model<1>>(shape) : der == 3 ? fn_lds<Model<3>>(shape) : fn_lds<Model<-1>>(shape);
}
template <int DER> using M2Xr = HoloXr<KIND_M2, 2, true, DER>;
template <int DER> using M2Std = HoloStd<KIND_M2, 2, true, DER>;
template <int D> struct MnStd { template <int DER> using Of = HoloStd<KIND_MN, D, true, DER>; };

tile_fn select_tile_orbit_lds(const LaunchCfg &c, LdsShape shape, int der) {
    if (c.kind == KIND_M2) return c.xr ? fn_lds_der2<M2Xr>(shape, der) : fn_lds_der2<M2Std>(shape, der);
    if (c.kind == KIND_MN) {
        switch (c.degree) {
#define FSG_MN(D) case D: return c.xr ? fn_lds<HoloXr<KIND_MN, D, true>>(shape) : fn_lds_der2<MnStd<D>::template Of>(shape, der);
            FSG_MN(2) FSG_MN(3) FSG_MN(4) FSG_MN(5) FSG_MN(6) FSG_MN(7) FSG_MN(8)
#undef FSG_MN
            default: return nullptr;
        }
    }
    if (c.kind == KIND_BS) {
        switch (c.flavor) {
#define FSG_BS(F) case F: return c.xr ? fn_lds<BsXr<F, true>>(shape) : fn_lds<BsStd<F, true>>(shape);
            FSG_BS(1) FSG_BS(2) FSG_BS(3) FSG_BS(4) FSG_BS(5)
#undef FSG_BS
            default: return nullptr;
        }
    }
    return nullptr;
}

}  // namespace fsg
