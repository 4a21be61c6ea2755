/*
 * The adjoint entry points (mgx_feautrier_adjoint_device,
 * mgx_feautrier_adjoint_width_device, mgx_image_adjoint_device,
 * mgx_image_adjoint_width_device, mgx_release_workspace) and the kernels they
 * launch: the solver's source compiled a second time with MGX_ADJOINT_TU, beside
 * mgx_solver.hip, which halves the build's longest compilation.  The state the two
 * units share (kernel timing, per-call workspace, walk-capacity hints) is defined in
 * mgx_solver.hip.
 */
#define MGX_ADJOINT_TU 1
#include "mgx_solver.hip"
