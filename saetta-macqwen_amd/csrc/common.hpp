// Shared by the kernel files of the gfx950 attention path: error plumbing for
// the C ABI and a few device helpers.  HIP/CDNA4 only.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/saetta_hip.h"

namespace saetta {

// Per-thread text of the last failure, returned by saetta_last_error().
char *error_buffer();
int fail(int code, const char *fmt, ...);
// Checks the device once per process; 0 or SAETTA_E_DEVICE.
int ensure_device();
// Turns the status of the launches since the last call into a return code; SAETTA_E_WAIT once a
// kernel on this device has left a code in the device's status word.
int launch_status(const char *what);
// Device address of the current device's sticky status word (pinned host memory): a kernel whose
// bounded wait runs out stores a non-zero code there.  nullptr before the device's set-up.
uint32_t *device_status_word();
// Compute units of the current device (asked for once per device; without a device, the MI355X's 256).
uint32_t cu_count();

// One-time set-up of a source file's kernels on the current device: loads their code object and
// raises their dynamic LDS limits, so that a first launch under stream capture has nothing left to
// do.  Called from ensure_device(); each returns a hipError_t as int.
int setup_kv_quant();
int setup_prep();
int setup_deltanet();
int setup_deltanet_chunk();
int setup_decode();
int setup_prefill();
// The chunked delta rule (deltanet_chunk.hip): the workspace a call needs (0: the call keeps to the
// token-by-token kernels), and the call itself (the delta rule only; the gated norm follows as for the
// token-by-token kernels) with a workspace of the caller's.
size_t deltanet_chunk_workspace_bytes(const saetta_rows_step_params &p);
int run_deltanet_chunk(hipStream_t stream, const float *mixed, const float *a, const float *b, const float *a_log,
                       const float *dt_bias, float *state, float *o, const saetta_rows_step_params &p, uint32_t channels,
                       void *workspace);
// Loads the code object `kernel` lives in.
inline int load_kernel(const void *kernel) {
    hipFuncAttributes attr;
    return int(hipFuncGetAttributes(&attr, kernel));
}

inline hipStream_t as_stream(saetta_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

// ---- launches, made or recorded ------------------------------------------------
// A kernel launch with its arguments, as a plan keeps it.
struct LaunchRecord {
    const void *kernel;
    dim3 grid, block;
    uint32_t lds;
    uint32_t first_arg, args;  // of LaunchList::offsets
    // What a launch is, for a call that may take launches recorded before it into one of its own.
    uint32_t kind = 0, bits = 0, rows = 0;
};
enum : uint32_t { LAUNCH_PREP = 1, LAUNCH_PARTIAL = 2, LAUNCH_CONV = 3, LAUNCH_ALONE = 4, LAUNCH_REDUCE = 5 };
// Launches in order; the arguments lie in `bytes`, each at its offset, 16-byte aligned.
struct LaunchList {
    std::vector<LaunchRecord> launches;
    std::vector<uint32_t> offsets;
    std::vector<unsigned char> bytes;
    int device = 0;
    template <class T>
    const T &arg(const LaunchRecord &r, uint32_t i) const { return *reinterpret_cast<const T *>(bytes.data() + offsets[r.first_arg + i]); }
    template <class T>
    T &arg(const LaunchRecord &r, uint32_t i) { return *reinterpret_cast<T *>(bytes.data() + offsets[r.first_arg + i]); }
};
// The list this thread records into, or nullptr: launches are made.
LaunchList *&recording();

template <class T>
void record_arg(LaunchList &list, const T &value) {
    static_assert(std::is_trivially_copyable<T>::value, "kernel arguments are plain values");
    const size_t at = (list.bytes.size() + 15) / 16 * 16;
    list.bytes.resize(at + sizeof(T));
    memcpy(list.bytes.data() + at, &value, sizeof(T));
    list.offsets.push_back(uint32_t(at));
}

// kernel<<<grid, block, lds, stream>>>(args...), or the same launch at the end of the list that this thread records.
// Every launch of the library goes through here.
template <class... P, class... A>
void launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, A &&...args) {
    static_assert(sizeof...(P) == sizeof...(A), "one argument per kernel parameter");
    if (LaunchList *list = recording()) {
        list->launches.push_back({reinterpret_cast<const void *>(kernel), grid, block, uint32_t(lds), uint32_t(list->offsets.size()), uint32_t(sizeof...(P))});
        (record_arg<std::remove_cv_t<P>>(*list, static_cast<P>(args)), ...);
        return;
    }
    std::tuple<std::remove_cv_t<P>...> values(static_cast<P>(args)...);
    std::apply([&](auto &...value) {
        void *pointers[] = {&value...};
        (void)hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, pointers, lds, stream);  // (its status: launch_status)
    }, values);
}

// Says what the launch just recorded is.
inline void tag_launch(uint32_t kind, uint32_t bits, uint32_t rows) {
    if (LaunchList *list = recording()) list->launches.back().kind = kind, list->launches.back().bits = bits, list->launches.back().rows = rows;
}

inline bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// Memory that a launch reads or writes.  Launches may become one only where what the one reads and writes lies apart: in
// order of launches a program may lay a buffer over another that is done with, inside one launch nothing is done with.
struct Span {
    const void *start;
    size_t bytes;
};
inline bool apart(const Span &p, const Span &q) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p.start), b = reinterpret_cast<uintptr_t>(q.start);
    return p.bytes == 0 || q.bytes == 0 || a + p.bytes <= b || b + q.bytes <= a;
}

}  // namespace saetta

#define SAETTA_REQUIRE(cond, code, ...)                       \
    do {                                                      \
        if (!(cond)) return saetta::fail((code), __VA_ARGS__); \
    } while (0)
