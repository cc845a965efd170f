// Host-side launchers of the trace and element passes that give a cell to four waves
// (sipg_split.h): the operator of launch_trace and launch_apply (kernels.h).
#pragma once

#include "kernels.h"

namespace insp {

// Where they are taken: a wave of 64 cells per SIMD is 2^16 cells; up to a few times that the passes
// with one thread per cell leave SIMDs idle or without a second wave to switch to, and the split
// passes' shorter chains win; on larger meshes their extra loads and the meeting in LDS lose. The
// lines are where the two crossed on the jittered Kuhn meshes (us one thread per cell / split, FP64):
//   element pass  2D order 3  8k cells 11.4 / 7.9, 65k 12.3 / 10.5, 97k 13.2 / 13.7
//                 2D order 4  45k 18.6 / 12.6, 180k 32.7 / 30.6, 980k 117 / 141
//                 3D order 2  10k 19.2 / 9.9, 162k 37.4 / 28.7, 750k 110 / 109
//                 3D order 3  10k 47.4 / 18.9, 83k 72.8 / 58.1, 105k 78.9 / 83.5
//                 3D order 4  10k 103 / 39.6, 64k 167 / 147, 83k 165 / 215
//   trace pass    3D order 2  48k 9.3 / 8.1, 162k 14.4 / 14.0, 384k 21.3 / 24.2
//                 3D order 3  48k 33.9 / 14.0, 384k 44.3 / 42.5, 664k 77.8 / 84.6
//                 3D order 4  48k 79.9 / 27.9, 511k 257 / 160 (FP32 105 / 77): taken at every size
// FP32 crosses a little later at orders 3 and 4 in 3D (order 3: 132k 47.0 / 45.8; order 4: 83k 97.3 /
// 88.6, 105k 107 / 126). Both need the packed neighbour words.
bool split_trace(const MeshView& m, const LevelView& l);
bool split_apply(const MeshView& m, const LevelView& l, bool fp32);
int split_blocks(int64_t E);  // partials of u.(A u) that the split element pass leaves
// ncomp vectors cs apart, their traces ts apart
template <typename T>
void launch_trace_split(const MeshView& m, const LevelView& l, const T* u, const T* kfac, T* tr,
                        hipStream_t s, int ncomp = 1, int64_t cs = 0, int64_t ts = 0);
template <typename T>
void launch_apply_split(const MeshView& m, const LevelView& l, const T* u, const T* tr, const T* kfac,
                        const MassView<T>& mass, T* out, hipStream_t s, double* partial);
// Every component of the vector (velocity) operator (launch_apply_slip, kernels.h) in one launch:
// vectors, traces and bc types of the components lie cs, ts and bs apart; split_blocks(E) partials a
// component.
void launch_vec_split(const MeshView& m, const LevelView& l, int ncomp, const double* u, const double* tr,
                      const double* kfac, const MassView<double>& mass, const double* bnormal, int64_t cs,
                      int64_t ts, int64_t bs, double* out, hipStream_t s, double* partial);
template <typename T>
void launch_cheb_split(const MeshView& m, const LevelView& l, const T* u, const T* tr, const T* kfac,
                       const T* f, const T* inv, const T* prev, T* x_next, T c1, T c2, hipStream_t s);

// The trace pass in the form that suits the mesh.
template <typename T>
void trace_pass(const MeshView& m, const LevelView& l, const T* u, const T* kfac, T* tr, hipStream_t s) {
  if (split_trace(m, l)) launch_trace_split<T>(m, l, u, kfac, tr, s);
  else launch_trace<T>(m, l, u, kfac, tr, s);
}

}  // namespace insp
