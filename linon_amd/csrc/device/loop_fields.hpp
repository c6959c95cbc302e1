// Which form of refraction the step loops of the predefined fields run: the branch over the side of
// the surface, or, where nothing is said here and in the sample rays, the root's sign
// (refraction_impl; the results are the same).  The sign is shorter, and faster in nearly every loop
// (1365x767: the plane mirage 7.24 -> 6.71 ms, with sigmoid 8.97 -> 8.63).  The loops below are the
// ones it slows, by the registers and the order of the whole kernel's code: 1365x767 frames of the
// icosphere scene at h = 0.005 in ms, by the branch, by the sign in every loop, and with these rules.
//   hot air's default variant    weight 1     7.26   7.25   7.23
//                                weight 0.5   7.63   7.89   7.68
//     adaptive start-up scene    weight 0.5   19.4   20.0   19.4
//     24 views in a batch                     103.5  106.1  103.4
//   hot air, IEEE                weight 0.5   10.11  10.24  10.11
//   spherical sigmoid mirage     weight 0.5   10.51  10.64  10.54
//   spherical mirage, WGSL       weight 1     7.79   8.02   7.87
#pragma once
#include "fields.hpp"
#include "raycast.hpp"

namespace lk {

#ifndef LINON_FAST_MATH
template <bool WOne, int Fixed>
struct LoopField<lw::FieldHotAirFaithfulRoot, WOne, Fixed> {
    using type = lw::FieldHotAirT<true, true>;
};
template <int Fixed>
struct LoopField<lw::FieldHotAir, false, Fixed> {
    using type = lw::FieldHotAirT<false, true>;
};
template <int Fixed>
struct LoopField<lw::FieldMirageSphericalSigmoid, false, Fixed> {
    using type = lw::FieldMirage<true, true, true>;
};
#else
template <bool WOne, int Fixed>
struct LoopField<lw::FieldMirageSpherical, WOne, Fixed> {
    using type = lw::FieldMirage<true, false, Fixed != LK_STEP_FIXED_ESCAPE>;
};
#endif

}  // namespace lk
