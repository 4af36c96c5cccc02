// a2c_flagged.h -- the entry points of libtpl_a2c.so that this package's own
// extension calls: those of include/tpl_a2c.h with a workspace, and with
// `flags` (report.h, host_flags.h) beside the status word; either may be null.
// The flags also report TPLX_A2C_RANGE.
#pragma once

#include "tpl_a2c.h"

// Some output value is NaN, infinite or at least 1e26 in magnitude (report.h).
#define TPLX_A2C_RANGE 16u

// Forward kernels: one workgroup per structure, a wave per block of 64 residues
// (FUSED) or a run of residues per thread (RUNS), or one per group of 256
// residues (GROUPS: needs the workspace).
#define TPLX_A2C_FWD_AUTO 0
#define TPLX_A2C_FWD_FUSED 1
#define TPLX_A2C_FWD_GROUPS 2
#define TPLX_A2C_FWD_RUNS 3

// Backward kernels, likewise: one workgroup per structure (FUSED, and the two
// that tpl_a2c.h names), or the blocks shared over the GPU (GROUPS: needs the
// workspace).
#define TPLX_A2C_BWD_AUTO 0
#define TPLX_A2C_BWD_FUSED 1
#define TPLX_A2C_BWD_GROUPS 2
#define TPLX_A2C_BWD_RUNS 3   // TPL_A2C_BWD_RUNS
#define TPLX_A2C_BWD_TILES 4  // TPL_A2C_BWD_TILES

extern "C" {
// The form that AUTO takes, with names or a workspace or without.
int tplx_a2c_forward_form(int dtype, int batch, int angles_stride, int atoms_stride, int names, int workspace);
int tplx_a2c_backward_form(int dtype, int batch, int angles_stride, int atoms_stride, int workspace);

// Bytes of the workspace that the GROUPS form needs (16-byte aligned; 0: none);
// no other form reads it.  A call writes what it reads there.
size_t tplx_a2c_workspace_bytes(int batch, int angles_stride);

int tplx_a2c_forward(int form, const int32_t* order, int dtype, const uint8_t* sequences, int seq_stride,
                     const void* angles, int angles_stride, void* coords, uint8_t* res_names, uint8_t* atom_names,
                     int atoms_stride, void* workspace, uint32_t* status, uint32_t* flags, int batch,
                     tpl_a2c_stream_t stream);

size_t tplx_a2c_backward_workspace_bytes(int batch, int angles_stride);

int tplx_a2c_backward(int form, const int32_t* order, int dtype, const uint8_t* sequences, int seq_stride,
                      const void* coords, const void* grad_coords, int atoms_stride, void* grad_angles,
                      int angles_stride, void* workspace, uint32_t* status, uint32_t* flags, int batch,
                      tpl_a2c_stream_t stream);
}
