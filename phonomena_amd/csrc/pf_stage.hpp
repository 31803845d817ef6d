// Staged transfers between device memory and the caller's (pageable) host
// arrays.
//
// A copy between the device and pageable memory runs at 10 GB/s here: one
// thread moves every byte through the runtime's own bounce buffer, and a new
// destination's pages are first touched in that copy.  PCIe moves 57 GB/s.
// So transfers go through pinned chunks in up to eight lanes, each with two
// chunks and a host thread: while one chunk crosses PCIe the thread copies the
// other.  Fields are packed, and spectra and probe frames copied, by kernels
// that write the pinned chunks themselves, on the caller's stream: no device
// scratch, no copy command per chunk (2 MiB copy commands from four streams
// ran at half the kernels' rate).  Three fields of 513 x 513 x 257 nodes (1.6
// GB) take 35 ms (46 GB/s) against 154; 1.6 MB of a small mesh's fields 0.2
// against 0.27.  Chunks of 512 KiB to 2 MiB by the size: a larger one costs
// fewer launches (of about 6 us beside a chunk's PCIe time), smaller ones keep
// the lanes of a short transfer busy; the first two chunks of every lane are
// filled by five launches (three fields of 9 MB 1.40 ms, with a launch for
// each 1.47).
//
// The lanes have no streams of their own.  With one each the kernels of
// several chunks overlapped, and 512 KiB chunks were as fast (37 ms there),
// but a stream takes 0.2 ms to make and one of a process's first four, which
// bring a hardware queue, 3 ms: the first call then waited longer than it
// gained.  First calls of a process, ms, pageable copies / lanes with streams
// / now: a field of 1 MB 6.7 / 6.8 / 0.6, 16 MB 13.9 / 9.3 / 1.8, 64 MB 18 / 11
// / 5; a transform of 1 MB 2.3 / 8.1 / 1.9, 4 MB 5.9 / 10.6 / 3.2, 16 MB 12 / 11
// / 4, 64 MB 26 / 15 / 8.
//
// The pinned memory of a device is one piece, of 512 KiB with its first
// context and made again when a transfer needs a larger one (two chunks a
// lane: 32 MiB at most; 8 MiB take 45 us).  It is shared by every context on
// the device and stays between calls; when the device's last context is
// destroyed a piece of more than STAGE_KEEP is given back (a program of many
// short runs would make a smaller one again for each), and pf_trim gives back
// all.  A transfer that finds it taken (another host thread's) copies directly.
#pragma once
#include <hip/hip_runtime.h>

namespace pf {

constexpr int STAGE_LANES = 8;
constexpr size_t STAGE_KEEP = 8u << 20;  // pinned memory that stays when a device has no context left

// Produce bytes [off, off + len) of a transfer at dst (memory the device can
// write) on stream s, or consume them from src: a reference to the caller's
// function object, for the length of the call (std::function would allocate,
// and throw through a C entry).
template <class P>
class StageFn {
    const void* obj;
    hipError_t (*call)(const void* obj, hipStream_t s, P at, size_t off, size_t len);

public:
    template <class F>
    StageFn(const F& f)
        : obj(&f), call([](const void* o, hipStream_t s, P at, size_t off, size_t len) -> hipError_t {
              return (*(const F*)o)(s, at, off, len);
          }) {}
    hipError_t operator()(hipStream_t s, P at, size_t off, size_t len) const { return call(obj, s, at, off, len); }
};
typedef StageFn<char*> StageFill;
typedef StageFn<const char*> StageDrain;

// Device to host: `fill` produces the bytes, after the work now on stream
// `after`.  Returns when host[0 .. bytes) is complete.  *taken = false (and
// nothing done) when the device's pinned memory is in use.
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
