// Error plumbing and device check of the C ABI.
#include "common.hpp"

#include <atomic>
#include <cstring>
#include <mutex>

namespace saetta {

char *error_buffer() {
    static thread_local char buf[512] = "";
    return buf;
}

int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(error_buffer(), 512, fmt, ap);
    va_end(ap);
    return code;
}

// The set-up of a device (its architecture checked, the code objects loaded, the kernels' LDS
// limits raised) runs once per device, the first time a call finds that device current.
namespace {
constexpr int MAX_DEVICES = 64;
struct DeviceSetup {
    std::once_flag once;
    int status = SAETTA_OK;
    char why[256] = "";
    // The device's sticky status word: pinned host memory that the kernels see through status_dev.  A
    // kernel whose bounded wait ran out stores a code there (one plain store by one lane); the host
    // reads it without synchronising.
    volatile uint32_t *status_host = nullptr;
    uint32_t *status_dev = nullptr;
};
DeviceSetup g_devices[MAX_DEVICES];
}  // namespace

int setup_runtime();

int ensure_device() {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(SAETTA_E_DEVICE, "no HIP device: %s", hipGetErrorString(e));
    }
    if (dev < 0 || dev >= MAX_DEVICES) return fail(SAETTA_E_DEVICE, "device index %d (up to %d)", dev, MAX_DEVICES - 1);
    DeviceSetup &d = g_devices[dev];
    std::call_once(d.once, [&d, dev] {
        hipDeviceProp_t prop;
        hipError_t e = hipGetDeviceProperties(&prop, dev);
        if (e != hipSuccess) {
            d.status = SAETTA_E_DEVICE;
            snprintf(d.why, sizeof d.why, "no HIP device: %s", hipGetErrorString(e));
            (void)hipGetLastError();
            return;
        }
        if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
            d.status = SAETTA_E_DEVICE;
            snprintf(d.why, sizeof d.why, "device is %s; this library is built for gfx950 only", prop.gcnArchName);
            return;
        }
        {
            void *host = nullptr, *devp = nullptr;
            e = hipHostMalloc(&host, 64, hipHostMallocMapped);
            if (e == hipSuccess) e = hipHostGetDevicePointer(&devp, host, 0);
            if (e != hipSuccess) {
                d.status = SAETTA_E_DEVICE;
                snprintf(d.why, sizeof d.why, "no pinned status word: %s", hipGetErrorString(e));
                (void)hipGetLastError();
                return;
            }
            memset(host, 0, 64);
            d.status_host = static_cast<volatile uint32_t *>(host);
            d.status_dev = static_cast<uint32_t *>(devp);
        }
        int (*const setups[])() = {setup_runtime, setup_kv_quant, setup_prep, setup_deltanet, setup_decode, setup_prefill};
        for (auto setup : setups) {
            if (int rc = setup()) {
                d.status = SAETTA_E_DEVICE;
                snprintf(d.why, sizeof d.why, "kernels do not load: %s", hipGetErrorString(hipError_t(rc)));
                (void)hipGetLastError();
                return;
            }
        }
    });
    if (d.status != SAETTA_OK) return fail(d.status, "%s", d.why);
    return SAETTA_OK;
}

namespace {
DeviceSetup *current_setup() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return dev >= 0 && dev < MAX_DEVICES ? &g_devices[dev] : nullptr;
}
}  // namespace

uint32_t cu_count() {
    static std::atomic<int> known[MAX_DEVICES];
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
        (void)hipGetLastError();
        return 256;
    }
    if ((cus = known[dev].load(std::memory_order_relaxed)) > 0) return uint32_t(cus);
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) {
        (void)hipGetLastError();
        return 256;
    }
    known[dev].store(cus, std::memory_order_relaxed);
    return uint32_t(cus);
}

uint32_t *device_status_word() {
    DeviceSetup *d = current_setup();
    return d ? d->status_dev : nullptr;
}

int launch_status(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(int(e), "%s: %s", what, hipGetErrorString(e));
    // A kernel of an EARLIER launch on this device that gave up a bounded wait has left its code in
    // the status word (this call's own launches have not run yet, as a rule): every call fails from
    // then on, until saetta_device_status(1) has cleared the word.
    DeviceSetup *d = current_setup();
    if (d && d->status_host) {
        if (const uint32_t code = *d->status_host) {
            return fail(SAETTA_E_WAIT,
                        "%s: a kernel launched earlier on this device gave up a bounded wait (status 0x%x); the "
                        "partial results of that launch are marked NaN; saetta_device_status(1) clears the status",
                        what, code);
        }
    }
    return SAETTA_OK;
}

LaunchList *&recording() {
    static thread_local LaunchList *list = nullptr;
    return list;
}

namespace {
__global__ __launch_bounds__(64) void token_params_kernel(saetta_token_params *dst, saetta_token_params value) {
    if (threadIdx.x == 0) *dst = value;
}
}  // namespace

int setup_runtime() { return load_kernel(reinterpret_cast<const void *>(token_params_kernel)); }

}  // namespace saetta

// A plan: what the calls between begin and end would have launched.
struct saetta_plan {
    saetta::LaunchList list;
};

extern "C" int saetta_plan_begin(void) {
    using namespace saetta;
    SAETTA_REQUIRE(!recording(), SAETTA_E_SHAPE, "plan_begin: this thread is recording a plan already");
    if (int rc = ensure_device()) return rc;
    LaunchList *list = new LaunchList;
    if (hipGetDevice(&list->device) != hipSuccess) (void)hipGetLastError();
    recording() = list;
    return SAETTA_OK;
}

extern "C" saetta_plan *saetta_plan_end(void) {
    using namespace saetta;
    LaunchList *list = recording();
    recording() = nullptr;
    if (!list) {
        fail(SAETTA_E_SHAPE, "plan_end: this thread is recording no plan");
        return nullptr;
    }
    saetta_plan *plan = new saetta_plan{std::move(*list)};
    delete list;
    return plan;
}

extern "C" uint32_t saetta_plan_launches(const saetta_plan *plan) { return plan ? uint32_t(plan->list.launches.size()) : 0; }

extern "C" int saetta_plan_run(saetta_stream_t stream, const saetta_plan *plan) {
    using namespace saetta;
    SAETTA_REQUIRE(plan, SAETTA_E_NULL, "plan_run: null plan");
    const LaunchList &list = plan->list;
    int dev = 0;
    SAETTA_REQUIRE(hipGetDevice(&dev) == hipSuccess && dev == list.device, SAETTA_E_DEVICE,
                   "plan_run: the plan was recorded on device %d, the current one is %d", list.device, dev);
    for (const LaunchRecord &r : list.launches) {
        void *args[16];
        for (uint32_t i = 0; i < r.args; i++) args[i] = const_cast<unsigned char *>(list.bytes.data()) + list.offsets[r.first_arg + i];
        const hipError_t e = hipLaunchKernel(r.kernel, r.grid, r.block, args, r.lds, as_stream(stream));
        if (e != hipSuccess) return fail(int(e), "plan_run: %s", hipGetErrorString(e));
    }
    return launch_status("plan_run");
}

extern "C" void saetta_plan_free(saetta_plan *plan) { delete plan; }

extern "C" int saetta_token_params_set(saetta_stream_t stream, saetta_token_params *d_tp, saetta_token_params value) {
    using namespace saetta;
    SAETTA_REQUIRE(d_tp && aligned(d_tp, 4), SAETTA_E_NULL, "token_params_set: null or misaligned record");
    if (int rc = ensure_device()) return rc;
    launch(token_params_kernel, dim3(1), dim3(64), 0, as_stream(stream), d_tp, value);
    return launch_status("token_params_set");
}

extern "C" int saetta_init(void) { return saetta::ensure_device(); }

extern "C" const char *saetta_last_error(void) { return saetta::error_buffer(); }

extern "C" uint32_t saetta_device_status(int clear) {
    if (saetta::ensure_device() != SAETTA_OK) return 0;
    saetta::DeviceSetup *d = saetta::current_setup();
    if (!d || !d->status_host) return 0;
    const uint32_t code = *d->status_host;
    if (clear) *d->status_host = 0;
    return code;
}
