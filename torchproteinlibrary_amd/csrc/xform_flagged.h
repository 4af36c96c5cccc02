// xform_flagged.h -- the entry points of libtpl_xform.so that this package's
// own extension calls: those of include/tpl_xform.h with `flags` (report.h,
// host_flags.h; null: no reports) in place of the status word.  Beside the
// status bits of that header they report TPLX_XFORM_RANGE.
#pragma once

#include "tpl_xform.h"

// Some output value is NaN, infinite or at least 1e26 in magnitude (report.h).
#define TPLX_XFORM_RANGE 4u

extern "C" {
int tplx_xform_translate(int dtype, void* out, const void* in, const void* T, const int32_t* num_atoms,
                         uint32_t* flags, int batch, int atoms_stride, tpl_xform_stream_t stream);
int tplx_xform_rotate(int dtype, void* out, const void* in, const void* R, int transpose,
                      const int32_t* num_atoms, uint32_t* flags, int batch, int atoms_stride,
                      tpl_xform_stream_t stream);
int tplx_xform_center(int dtype, void* center, const void* in, const int32_t* num_atoms, uint32_t* flags,
                      int batch, int atoms_stride, tpl_xform_stream_t stream);
int tplx_xform_center_backward(int dtype, void* grad_in, const void* grad_center, const int32_t* num_atoms,
                               uint32_t* flags, int batch, int atoms_stride, tpl_xform_stream_t stream);
}
