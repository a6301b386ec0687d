// Shared between the C-ABI units of the vortex-lattice / beam path
// (afx_vlm.hip: device side; afx_structure.cpp: lattice generator, beam,
// load and displacement transfer, coupling loop).
#pragma once
#include <string>

struct afx_vlm;

namespace afx {
// sets the thread-local message returned by afx_last_error and returns code
int api_fail(int code, const std::string& msg);
// afx_vlm_set_nodes and afx_vlm_build without their waits, for a caller that goes
// on to a call that waits: queued on the lattice's stream, xyz is free at return
int vlm_queue_nodes(afx_vlm* h, const double* xyz);
int vlm_queue_build(afx_vlm* h);
}  // namespace afx
