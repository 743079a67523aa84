// What the kernels' host sides share: launch functions, row blocks and the
// device's compute units.
#pragma once

#include "attention_device.hpp"

#include <cstdint>

namespace pcl {

// Devices whose per-device state (compute units, allowed LDS) is kept.
constexpr int kMaxDevices = 64;

// Compute units of the current device, 0 when there is none.
int device_cus();

hipError_t launch_split_kv(const Params &p, hipStream_t stream);
hipError_t launch_combine(const Params &p, hipStream_t stream);
hipError_t launch_pipe_kv(const Params &p, hipStream_t stream);
hipError_t launch_pipe_kv_chunks(const Params &p, int c0, int n, bool merge_out,
                                 hipStream_t stream);
hipError_t launch_fan_kv(const Params &p, hipStream_t stream);
hipError_t launch_fan_chunk(const Params &p, int ci, bool merge_out, hipStream_t stream);
bool fan_supported(int dk);
hipError_t launch_spread_kv(const Params &p, hipStream_t stream);
int spread_slices(int dk);

// The tiled kernels: *merged is set when the launch itself wrote the merged
// output of a split launch (no combine needed).
hipError_t launch_tiled(const Params &p, int split, hipStream_t stream, bool *merged);
hipError_t launch_tiled_wide(const Params &p, int split, hipStream_t stream, bool *merged);
int tiled_rows(int dk);
int tiled_wide_rows();
int tiled_tail_chunks(const Params &p, int nqb, int cus);
int64_t span_tiles(const Params &p, int64_t rows, int64_t cus, int64_t extra, int64_t last);
bool wide_half_blocks(const Params &p, int64_t cus);
int tiled_block_rows(const Params &p, int64_t cus);

} // namespace pcl
