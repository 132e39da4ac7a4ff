// Small device results on the host: a kernel of the calling stream writes them into pinned host
// memory, and the call synchronises the stream.  A copy to pageable memory costs the runtime's
// staging and a copy kernel of its own (ICPStep at 160x120, whose reduction now takes the poses as
// arguments and writes the sums itself, 54 -> 23 us; a tracker's result about 30 us less).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace fu {

// A pinned, device-mapped slot of kMailBytes, taken from a process-wide pool for one call at a
// time (any thread, any stream, any device) and given back when the call has synchronised.  The
// pool keeps at most kMailSlots; `dev` is null when no slot could be had.
constexpr size_t kMailBytes = 16384;
constexpr size_t kMailSlots = 16;
class Mail {
public:
    Mail();
    ~Mail();
    Mail(const Mail&) = delete;
    Mail& operator=(const Mail&) = delete;
    void* host = nullptr;
    void* dev = nullptr;
    // the stream is synchronised after the last launch that was given the slot (whether or not an
    // error was seen since), or none was: nothing writes the slot any more, so it may be reused
    void done() { idle = true; }

private:
    bool idle = false;
};

// up to two pieces of memory of device `dev` (whole words, kMailBytes in all) to host memory,
// through a slot or, without one or when another device is current, by copies; synchronises `s`
hipError_t mail_read(int dev, void* dst0, const void* src0, size_t bytes0, void* dst1, const void* src1, size_t bytes1,
                     hipStream_t s);
inline hipError_t mail_read(int dev, void* dst, const void* src, size_t bytes, hipStream_t s) {
    return mail_read(dev, dst, src, bytes, nullptr, nullptr, 0, s);
}
// the current device, -1 if there is none
int current_device();

}  // namespace fu
