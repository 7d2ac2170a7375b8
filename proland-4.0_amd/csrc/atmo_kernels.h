// atmo_kernels.h — host-callable launchers of the gfx950 pass kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <functional>

#include "atmo_device.h"

namespace atmo {

// Per-theta constants of the inscatterS direction grid (NS thetas).
struct DirJHost {
    float ct, st, dw, pad;
};
// Per-direction constants of the irradianceN hemisphere grid, index ip*(NI/2)+it.
struct DirEHost {
    float wx, wz, wzdw, pad;
};

// The two spherical-integral kernels stage their theta rows in LDS, CH rows at
// a time: CH is the largest count (up to all of them) whose staging fits
// kSphLdsBudget, the dynamic LDS a launch gets without raising the kernel's
// limit; 0 = not even one row fits.  lds_* are the bytes for CH rows.
// Workgroups (grid.y) per entry of the tile tables of T, the view-ray samples and
// the numeric check, and mu rows per entry of dS1's: the tables stay small.
constexpr int kTileY = 16, kTileRows = 4;
constexpr size_t kSphLdsBudget = 64 * 1024;
// JX: extra LDS entries of the merged ground rows of one staging round of the
// orders >= 3 pass (the sum over its theta rows of merged_row_extra, maximum
// over the layers and sets of a launch)
// Order 2 stages its 48-byte entries as three planes of float4, kJ1Plane
// entries apart, in unchunked launches whose staging round (all NS rows) fits
// one plane; other launches keep each entry whole.  544 = 32 x 64 directions at
// RES_NU 16.  Chunked: CH < NS, or an order-2 round too large for a plane
// (those launches use the chunked variant, also for a single round).
constexpr int kJ1Plane = 544;
// k_inscatterS forms: all theta rows staged at once, staged in chunks, or all
// at once with the rows dealt to DS slots of a workgroup's threads
constexpr int kJPlain = 0, kJChunk = 1, kJSplit = 2;
constexpr int kJSplitThreads = 1024;
bool inscatterS_chunked(int NS, int CH, int RNU, bool first);
size_t lds_inscatterS(int NS, int CH, int RNU, int SW, int JX, bool first);
// bound on the extra entries of theta row `it` (NS rows) of a layer at radius r
int merged_row_extra(double r, double Rg, double Rt, int SW, int NS, int it);
size_t lds_irradianceN(int CH, int RNU, bool first);
int chunk_inscatterS(int NS, int RNU, int SW, const std::function<int(int)> &jx_of_ch, bool first);
int chunk_irradianceN(int NI, int RNU, bool first);

hipError_t launch_transmittance(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp,
                                hipStream_t st);
hipError_t launch_irradiance1(const SetDesc *sets, const uint2 *tiles, int ntiles, hipStream_t st);
// geometry and transmittance tables of a precompute (SetDesc::tview on nview tiles, tground,
// theta rows and sun columns with wpt workgroups per set, 0: none), after the T pass
int theta_workgroups(int RR, int RMUS, int SW, int SH, int NS, int NI);
hipError_t launch_geometry(const SetDesc *sets, int nsets, int wpt, const uint2 *tiles, int nview, int nsamp, int NS, int NI,
                           hipStream_t st);
// G: texels per thread (2, 3, 4 or 8); CH: theta rows per staging round; RNU:
// the largest RES_NU of the launch's sets; DS: slots of the workgroup's threads the
// theta rows are dealt to (1: none; more: all rows staged at once)
hipError_t launch_inscatterS(const SetDesc *sets, const uint2 *tiles, int ntiles, int NS, int CH, int RNU,
                             int JX, const void *dirT, const void *dirW, bool first, size_t lds, int G,
                             int DS, int threads, hipStream_t st);
hipError_t launch_irradianceN(const SetDesc *sets, const uint2 *tiles, int ntiles, int NI, int CH,
                              const void *dirs, bool first, size_t lds, hipStream_t st);
// The dSn pass, one mu row (tile) per workgroup.  form: 0 direct gathers, 1
// LDS-staged rows (both read SetDesc::view and tview), 2 LDS-staged rows without
// SetDesc::view.  W4max: the most texels of a row of the launch's sets.  lin4: their
// parameterisation (one per batch), compiled in.
struct SnShape {
    int texels, threads;   // per thread (1 .. 3), per workgroup (a multiple of 64 up to 512)
};
SnShape sn_shape(int W4);   // W4 <= 1024
// The dS1 pass, one mu row (tile) per workgroup.  sh: s1_shape of every set of the
// launch; TWmax: the most T columns of its sets.
constexpr int kXkMax = 2048;   // T columns whose centres are staged for the sun lookups
struct S1Shape {
    int axis;      // how the mu axis of the sun's T lookup is found
    int texels;    // per thread, 1 to 4 with LDS-staged T rows, 0: gathers
    int columns;   // T columns staged per thread (1, 2 or 4)
    int threads;   // per workgroup
};
S1Shape s1_shape(int W4, int TW, bool linT);
hipError_t launch_inscatter1(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp, S1Shape sh, int TWmax,
                             hipStream_t st);
hipError_t launch_inscatterN(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp, int form, SnShape sh,
                             int W4max, bool lin4, hipStream_t st);
// SetDesc::view of every set, tiles of 256 consecutive samples
hipError_t launch_snview(const SetDesc *sets, const uint2 *tiles, int ntiles, int nsamp, hipStream_t st);
hipError_t launch_check(const SetDesc *sets, const uint2 *tiles, int ntiles, unsigned int *flags,
                        hipStream_t st);

}  // namespace atmo
