// C entries to the host functions of csrc/atmo_kernels.h for the host tests.
#include "../../proland-4.0_amd/csrc/atmo_kernels.h"

extern "C" {
int call_theta_workgroups(int RR, int RMUS, int SW, int SH, int NS, int NI) {
    return atmo::theta_workgroups(RR, RMUS, SW, SH, NS, NI);
}
int call_launch_geometry(int nsets, int wpt, int nview) {
    return (int)atmo::launch_geometry(nullptr, nsets, wpt, nullptr, nview, 50, 16, 32, nullptr);
}
}
