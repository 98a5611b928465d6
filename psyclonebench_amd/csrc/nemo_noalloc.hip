// Allocation-free form of the NEMOLite2D step: c_invoke_time_step_noalloc.
//
// One step with the semantics of the host-pointer PSy layer
// (manual_versions/psykal_cpp/time_step.cpp:53-136: every sweep in order, in
// place, now <- after copied over the reference's copy region) on 25 device
// arrays that the caller owns, for callers that cannot allocate device
// memory (code under HIP graph capture, tight serving loops). Two launches: the
// band tile of nemo_band.h over the after arrays (every sweep up to
// bc_flather), and the copies with next_sshu/v. 511 x 383: 15.8 us a
// step, against 222 us with one kernel per sweep, of which 187 us were a Flather
// kernel that walked each row and column with one thread, and 18.5 us with the
// Coriolis factors in a launch of their own. Two things the allocating forms
// keep in buffers of their own are arranged differently:
//
//  * the Coriolis factors (2*omega)*sin(gphi*d2r) are evaluated in the tile
//    (the allocating forms evaluate them once on the host with libm; the
//    device sin may differ from it in the last bit, far inside the 1e-12
//    relative bound of the FP64 step);
//  * the Flather faces are found from the mask, not from host-built segment
//    lists.
#include "nemo_hip_common.h"
#include "nemo_host.h"
#include "nemo_step.h"
#include "nemolite2d_hip.h"

namespace nemo {

// Elements of an array that the entry point takes.
constexpr int kNoallocMaxElems = 1 << 21;

}  // namespace nemo

using namespace nemo;

extern "C" void c_invoke_time_step_noalloc(NEMO_HOST_ARRAYS, int istep, int internal_xstart,
                                           int internal_xstop, int internal_ystart,
                                           int internal_ystop, int width, int total_size,
                                           double rdt, double cbfr, double visc,
                                           double omega, double d2r, double g,
                                           void *stream)
{
    const Geometry G{internal_xstart, internal_xstop, internal_ystart, internal_ystop,
                     width, total_size};
    check_geometry(G);
    if (total_size > kNoallocMaxElems)
        NEMO_FATAL("c_invoke_time_step_noalloc: total_size %d exceeds the %d elements "
                   "it takes", total_size, kNoallocMaxElems);
    hipStream_t s = static_cast<hipStream_t>(stream);
    // hipGetLastError also returns what earlier calls of other code on this
    // thread left behind (an event query's "not ready", say); clear it so
    // that the launch checks below report this call's launches only.
    (void)hipGetLastError();

    StepIn<double> f;
    f.sshn_t = sshn_t;
    f.sshn_u = sshn_u;
    f.sshn_v = sshn_v;
    f.un = un;
    f.vn = vn;
    f.ht = ht;
    f.hu = hu;
    f.hv = hv;
    f.ssha_u = ssha_u;
    f.ssha_v = ssha_v;
    f.area_t = area_t;
    f.area_u = area_u;
    f.area_v = area_v;
    f.dx_u = dx_u;
    f.dx_v = dx_v;
    f.dx_t = dx_t;
    f.dy_u = dy_u;
    f.dy_v = dy_v;
    f.dy_t = dy_t;
    f.fcor_u = gphiu;  // the tile evaluates the factors
    f.fcor_v = gphiv;
    f.tmask = tmask;
    const StepScalars<double> p{rdt, visc, g, 1.0 + cbfr * rdt};
    const Bounds b{G.xs, G.xe, G.ys, G.ye};
    launch_band_inplace(s, f, p, StepOut<double>{ssha_t, ua, va, nullptr, nullptr}, omega, d2r,
                        width, b, tide_at(istep, rdt));
    launch_finish(s, un, ua, vn, va, sshn_t, ssha_t, sshn_u, sshn_v, tmask, area_t, area_u,
                  area_v, width, b);
}
