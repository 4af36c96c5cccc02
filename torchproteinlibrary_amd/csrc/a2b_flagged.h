// a2b_flagged.h -- the entry points of libtpl_a2b.so that this package's own
// extension calls: those of include/tpl_a2b.h with `flags` (report.h,
// host_flags.h; null: no reports) in place of the status word.
#pragma once

#include "tpl_a2b.h"

extern "C" {
int tplx_a2b_forward(int dtype, const void* angles, void* coords, const int32_t* lengths, void* state,
                     void* sync, uint32_t* flags, int batch, int angles_stride, const tpl_a2b_config* cfg,
                     tpl_stream_t stream);
int tplx_a2b_backward(int dtype, void* grad_angles, const void* grad_coords, const void* angles,
                      const int32_t* lengths, const void* state, void* sync, uint32_t* flags, int batch,
                      int angles_stride, const tpl_a2b_config* cfg, tpl_stream_t stream);

// Forward and backward of one step together, for gradients that are there
// beforehand, with cfg->bwd_res_per_lane residues per lane; no state and no
// look-back words.  tplx_a2b_step_fits: whether the shape and the configuration
// have such a form, and the bytes of workspace it needs (256-byte aligned; its
// contents do not matter).
int tplx_a2b_step_fits(int dtype, int batch, int angles_stride, const tpl_a2b_config* cfg, size_t* workspace);
int tplx_a2b_step(int dtype, const void* angles, const int32_t* lengths, const void* grad_coords, void* coords,
                  void* grad_angles, void* workspace, int batch, int angles_stride, const tpl_a2b_config* cfg,
                  tpl_stream_t stream);
}
