// Staged transfers between device memory and the caller's (pageable) host
// arrays.
//
// A copy between the device and pageable memory runs at 10 GB/s here: one
// thread moves every byte through the runtime's own bounce buffer, and a new
// destination's pages are first touched in that copy.  PCIe moves 57 GB/s.
// So large transfers go through pinned chunks in a few lanes, each with its
// own stream, two chunks and a host thread: while one chunk crosses PCIe the
// thread copies the other.  Fields are packed, and spectra and probe frames
// copied, by kernels that write the pinned chunks themselves: no device
// scratch, no copy command per chunk (2 MiB copy commands from four streams
// ran at half the kernels' rate).  Three fields of 513 x 513 x 257 nodes (1.6
// GB) take 32 ms (50 GB/s) against 154; 1.6 MB of a small mesh's fields 0.2
// against 0.4.  Eight lanes of half a MiB: four of 2 MiB took 40 ms there, and
// 28 against 18 for the 340 MB of a 16-member batch, whose fields are a few
// chunks each.
//
// The lanes of a device (2 x STAGE_CHUNK bytes of pinned memory each) are made
// by the first transfer large enough for them and shared by every context on
// it.  When the device's last context is destroyed all but the first lane
// (which a program of many short runs would make again for each) are given
// back; pf_trim gives back all.  A transfer that finds them taken (another
// host thread's) copies directly.
#pragma once
#include <hip/hip_runtime.h>

#include <functional>

namespace pf {

constexpr int STAGE_LANES = 8;
constexpr size_t STAGE_CHUNK = 512u << 10;

// Produce bytes [off, off + len) of a transfer at dst (memory the device can
// write) on stream s, or consume them from src.
typedef std::function<hipError_t(hipStream_t s, char* dst, size_t off, size_t len)> StageFill;
typedef std::function<hipError_t(hipStream_t s, const char* src, size_t off, size_t len)> StageDrain;

// Device to host: `fill` produces the bytes, after the work now on stream
// `after`.  Returns when host[0 .. bytes) is complete.  *taken = false (and
// nothing done) when the device's chunks are in use.
int stage_out(int dev, hipStream_t after, void* host, size_t bytes, const StageFill& fill, bool* taken);
// Host to device: `drain` consumes the bytes, after the work now on stream
// `after`.  Returns when they are consumed.
int stage_in(int dev, hipStream_t after, const void* host, size_t bytes, const StageDrain& drain, bool* taken);

// Plain copies of 8-byte words through the chunks (directly where they are
// taken).
int copy_out(int dev, hipStream_t after, void* host, const void* src, size_t bytes);
int copy_in(int dev, hipStream_t after, void* dst, const void* host, size_t bytes);

// A context lives on device dev (+1) or is destroyed (-1).
void stage_users(int dev, int change);

}  // namespace pf
