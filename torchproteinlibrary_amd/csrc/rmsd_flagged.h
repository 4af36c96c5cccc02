// rmsd_flagged.h -- the entry points of libtpl_rmsd.so that this package's own
// extension calls: those of include/tpl_rmsd.h with `flags` (report.h,
// host_flags.h) in place of the status word, or beside it (null: no reports).
#pragma once

#include "tpl_rmsd.h"

extern "C" {
// The forward's workspace (its contents do not matter; null: none), with which
// few large structures take several workgroups each.
size_t tplx_rmsd_workspace_bytes(int batch, int atoms_stride);
int tplx_rmsd_forward(int dtype, const void* input, const void* target, const int32_t* num_atoms, void* rmsd,
                      void* ut, void* state, void* workspace, uint32_t* status, uint32_t* flags, int batch,
                      int atoms_stride, tpl_rmsd_stream_t stream);
int tplx_rmsd_backward(int dtype, void* grad_input, const void* grad_rmsd, const void* input, const void* target,
                       const int32_t* num_atoms, const void* state, uint32_t* flags, int batch, int atoms_stride,
                       tpl_rmsd_stream_t stream);
}
