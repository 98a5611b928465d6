// Launchers for the NEMOLite2D step kernels (defined in nemo_step.hip).
// Host code in nemo_psy.cpp drives them; all pointers are device pointers.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "nemo_point.h"

namespace nemo {

// Inclusive 0-based rectangle.
struct Region {
    int x0, x1, y0, y1;
};

// Internal T region bounds as passed through the C ABI (0-based).
struct Bounds {
    int xs, xe, ys, ye;
};

// Writable outputs of one fused step (ping-pong targets).
template <typename T>
struct StepOut {
    T *ssh;   // new sshn_t (== ssha_t)
    T *u;     // new un (== ua)
    T *v;     // new vn (== va)
    T *sshu;  // new sshn_u
    T *sshv;  // new sshn_v
};

// Flather faces grouped in segments that must run in order: one segment per
// row for U faces, one per column for V faces (bc_flather_u/v read the
// neighbour face the serial sweep may already have updated). Entry k of a
// segment updates vel[idx[k]] from vel[idx[k] + off[k]]; off == 0 marks a
// neighbour outside the allocation (read as 0). prev[k] != 0 marks a
// neighbour that is itself a Flather face later in the sweep: the serial
// sweep reads it before updating it, so it reads the value that face held
// at the end of the previous step, which a caller that ping-pongs its
// buffers keeps in the previous step's set (vel_prev), not in `vel`.
struct FlatherList {
    const int *seg_ptr;   // nseg + 1
    const int *idx;       // face index
    const int *off;       // +-1 (U) or +-W (V), or 0
    const int *prev;      // 1: read the neighbour from vel_prev
    const double *coef;   // sqrt(g / h) at the face
    int nseg;
};

// --- unfused kernels, one per reference kernel ---------------------------
void launch_continuity(hipStream_t s, const StepIn<double> &f, double *ssha,
                       int W, Region r, double rdt);
void launch_momentum_u(hipStream_t s, const StepIn<double> &f,
                       const StepScalars<double> &p, double *ua, int W,
                       Region r);
void launch_momentum_v(hipStream_t s, const StepIn<double> &f,
                       const StepScalars<double> &p, double *va, int W,
                       Region r);
void launch_bc_ssh(hipStream_t s, const int *tmask, double *ssha, int W,
                   Region r, double tide);
void launch_bc_solid(hipStream_t s, const int *tmask, double *vel, int W,
                     int stride, Region r);
// ua_prev / va_prev: the velocities at the end of the previous step (the
// previous ping-pong set, or ua / va themselves when they are updated in
// place or on a first step that writes into the after arrays).
void launch_flather(hipStream_t s, const FlatherList &lu, const FlatherList &lv,
                    double *ua, double *va, const double *ua_prev,
                    const double *va_prev, const double *sshn_u,
                    const double *sshn_v);
void launch_copy3(hipStream_t s, double *un, const double *ua, double *vn,
                  const double *va, double *sshn_t, const double *ssha_t,
                  int W, Region r);
void launch_next_ssh(hipStream_t s, const int *tmask, const double *sshn_t,
                     const double *area_t, const double *area_face,
                     double *ssh_face, int W, int stride, Region r);

// --- fused step -----------------------------------------------------------
// One launch computes the new ssh (continuity + bc_ssh), the post-solid
// u/v (momentum + bc_solid) and the new face ssh (next_sshu/v) for the whole
// M x N extent, reading `f` and writing `o`. Flather runs afterwards
// (launch_flather) on o.u / o.v with the old face ssh.
// The tide value is tide_tab[tide_k] when tide_tab is non-null, else
// tide_val.
void launch_fused_step(hipStream_t s, const StepIn<double> &f,
                       const StepScalars<double> &p, const StepOut<double> &o,
                       int W, Bounds b, const double *tide_tab, int tide_k,
                       double tide_val);

// Row-march form of the fused step (nemo_march.hip): same inputs, outputs
// and arithmetic as launch_fused_step; `variant` picks the block width and
// rows per band (0 .. march_variant_count()-1).
void launch_fused_march(hipStream_t s, int variant, const StepIn<double> &f,
                        const StepScalars<double> &p, const StepOut<double> &o,
                        int W, Bounds b, const double *tide_tab, int tide_k,
                        double tide_val);
int march_variant_count();
void march_variant_shape(int variant, int *mx, int *rows, int *prefetch);
const char *march_variant_kernel(int variant);

// --- band form (nemo_band.hip): the library's default ----------------------
// Metrics by row: on a grid where the 13 metric, area, Coriolis and after-ssh
// face arrays do not vary along a row, a table of one record a row stands for
// them. launch_row_metrics builds the table (row_table_values() values) from
// the arrays whose (0,0) is at element `base` and stores `mark` to *bad
// (memory that the device can write) when they do vary or a divisor is out of
// the table's range (2^+-kDivisorExp).
constexpr int kDivisorExp = 100;
// The same for a divisor that the host knows: the friction factor of the step.
inline bool table_divisor(double d)
{
    const int e = std::ilogb(d);  // INT_MAX / INT_MIN: inf, NaN, 0
    return e >= -kDivisorExp && e <= kDivisorExp;
}
constexpr int kRowTableWidth = 32;  // values a record
size_t row_table_values(const Bounds &b);
void launch_row_metrics(hipStream_t s, const StepIn<double> &f, int W, unsigned base,
                        const Bounds &b, double *tab, int *bad, int mark);
// One fused step with its Flather faces in one launch: the same results as
// launch_fused_march followed by launch_flather. tab: the row table, or null
// (any metrics). u_prev / v_prev as in launch_flather.
void launch_band_f64(hipStream_t s, const StepIn<double> &f, const double *tab,
                     const StepScalars<double> &p, const StepOut<double> &o,
                     const double *u_prev, const double *v_prev, int W, const Bounds &b,
                     const double *tide_tab, int tide_k, double tide_val);
// The sweeps up to bc_flather of an in-place step (o.ssh, o.u, o.v are the
// after arrays; o.sshu / o.sshv are not written), then, in launch_finish, the
// copies now <- after and next_sshu/v. Together the unfused sequence.
// f.fcor_u / f.fcor_v: the latitudes gphiu / gphiv.
void launch_band_inplace(hipStream_t s, const StepIn<double> &f, const StepScalars<double> &p,
                         const StepOut<double> &o, double omega, double d2r, int W,
                         const Bounds &b, double tide);
void launch_finish(hipStream_t s, double *un, const double *ua, double *vn, const double *va,
                   double *sshn_t, const double *ssha_t, double *sshn_u, double *sshn_v,
                   const int *tmask, const double *area_t, const double *area_u,
                   const double *area_v, int W, const Bounds &b);

// Small helpers.
void launch_fill_int(hipStream_t s, int *p, int n, int value);

}  // namespace nemo
