// C entries to the host functions of csrc/atmo_kernels.h for the host tests.
#include "../../proland-4.0_amd/csrc/atmo_kernels.h"

extern "C" {
int call_theta_workgroups(int RR, int RMUS, int SW, int SH, int NS, int NI) {
    return atmo::theta_workgroups(RR, RMUS, SW, SH, NS, NI);
}
int call_launch_geometry(int nsets, int wpt, int nview) {
    return (int)atmo::launch_geometry(nullptr, nsets, wpt, nullptr, nview, 50, 16, 32, nullptr);
}
int call_inscatter1(int W4, int TW, int linT, int *shape) {
    const atmo::S1Shape h = atmo::s1_shape(W4, TW, linT != 0);
    shape[0] = h.texels; shape[1] = h.columns; shape[2] = h.threads;
    return (int)atmo::launch_inscatter1(nullptr, nullptr, 1, 50, h, TW, nullptr);
}
}
