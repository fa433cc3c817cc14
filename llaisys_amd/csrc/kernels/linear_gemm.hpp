// The tiled linear kernels of linear_gemm.hip: several rows, any of the element types.
#pragma once

#include "launch.hpp"

namespace llaisys::kernels {

// The rows, types and alignments the tiled kernels take.
bool gemmTakes(const LinearCall &c);
// Workspace that lets the launch split K as it would like to; with less it does not split.
size_t gemmWorkspaceBytes(const LinearCall &c);
void gemm(const LinearCall &c, void *ws, size_t ws_bytes, hipStream_t s);

} // namespace llaisys::kernels
