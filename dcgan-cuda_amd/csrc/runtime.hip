// Runtime half of the C ABI: device selection, memory, streams, events and the scratch arena.
// Stands in for the GPU branches of the reference's src/memory (alloc.cu, copy.hxx).
#include "dh_common.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <thread>

namespace dh
{
namespace
{
thread_local char g_err[512] = "";

// Scratch of the entry points that must not allocate (dh_bias_grad_static): a fixed array in the
// code object, one copy per GPU.  Host code never uses this name as an address: init_device asks
// the runtime where the current device keeps its copy and stores that pointer in the device state.
__attribute__((used)) static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

// A large copy to the host, see dh_memcpy_d2h: it goes through a ring in pieces, and an event is recorded for up to four of them.
constexpr size_t READ_PIECE = 256 * 1024;
constexpr size_t READ_CHUNK_MAX = 4 * READ_PIECE;
constexpr size_t READ_RING = 8 * READ_CHUNK_MAX;
constexpr int READ_SLOTS_MAX = READ_RING / READ_PIECE;
constexpr size_t READ_STAGED_MIN = 2 * 1024 * 1024;   // smaller ones gain nothing
constexpr int READ_THREADS_MAX = 3;

struct DeviceState
{
    bool ready = false;
    int device = 0;
    int cus = 0;
    // one scratch arena per stream that asked for one: launches on different streams may overlap
    struct Arena { hipStream_t stream; void* ptr; size_t bytes; };
    Arena arena[MAX_ARENAS] = {};
    int n_arenas = 0;
    // pinned staging slots of dh_memcpy_h2d_staged, used round-robin; `done` is recorded behind the
    // slot's copy and waited for before the slot is written again
    struct Stage { void* host; size_t bytes; hipEvent_t done; bool in_flight; };
    Stage stage[STAGE_SLOTS] = {};
    int next_stage = 0;
    // pinned ring of dh_memcpy_d2h and one event per chunk in flight; g_read_mu guards it
    void* read_ring = nullptr;
    hipEvent_t read_done[READ_SLOTS_MAX] = {};
    void* static_scratch = nullptr;   // this device's copy of `scratch`
};

std::mutex g_mu;
std::mutex g_read_mu;
DeviceState g_dev[16];
int g_cur = -1;

// Copies `bytes` (a multiple of 4) from pinned host memory, which the device reads across the bus, to device
// memory: for the small inputs of a run an ordinary kernel in the launch stream starts sooner than a copy
// command does.
__global__ __launch_bounds__(256) void copy_from_pinned(void* __restrict__ dst, const void* __restrict__ src, size_t bytes,
                                                        bool vec)
{
    const size_t stride = (size_t)gridDim.x * 256, tid = (size_t)blockIdx.x * 256 + threadIdx.x;
    size_t done = 0;
    if (vec)
    {
        const size_t n16 = bytes / 16;
        for (size_t i = tid; i < n16; i += stride)
            static_cast<float4*>(dst)[i] = static_cast<const float4*>(src)[i];
        done = n16 * 16;
    }
    for (size_t i = done / 4 + tid; i < bytes / 4; i += stride)
        static_cast<float*>(dst)[i] = static_cast<const float*>(src)[i];
}
}  // namespace

int fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int fail_hip(hipError_t err, const char* what)
{
    return fail((int)err, "%s: %s (%s)", what, hipGetErrorString(err), hipGetErrorName(err));
}

static int init_device(int device)
{
    if (device < 0 || device >= 16)
        return fail(DH_EINVAL, "dh_init: device %d out of range", device);
    std::lock_guard<std::mutex> lock(g_mu);
    DH_HIP(hipSetDevice(device));
    DeviceState& st = g_dev[device];
    if (!st.ready)
    {
        hipDeviceProp_t prop;
        DH_HIP(hipGetDeviceProperties(&prop, device));
        if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
            return fail(DH_EINVAL, "dh_init: device %d is %s; this library holds gfx950 code only",
                        device, prop.gcnArchName);
        void* fixed = nullptr;
        DH_HIP(hipGetSymbolAddress(&fixed, HIP_SYMBOL(scratch)));
        st.static_scratch = fixed;
        st.device = device;
        st.cus = prop.multiProcessorCount;
        st.ready = true;
    }
    g_cur = device;
    return 0;
}

int ensure_init()
{
    if (g_cur >= 0)
        return 0;
    return init_device(0);
}

int num_cus()
{
    return g_cur >= 0 ? g_dev[g_cur].cus : 256;
}

int static_scratch(void** ptr)
{
    DH_TRY(ensure_init());
    *ptr = g_dev[g_cur].static_scratch;
    if (!*ptr)
        return fail(DH_EINVAL, "the fixed scratch buffer of device %d has no address", g_cur);
    return 0;
}

int workspace(size_t bytes, void** ptr, hipStream_t stream)
{
    DH_TRY(ensure_init());
    std::lock_guard<std::mutex> lock(g_mu);
    DeviceState& st = g_dev[g_cur];
    DeviceState::Arena* a = nullptr;
    for (int i = 0; i < st.n_arenas; ++i)
        if (st.arena[i].stream == stream)
            a = &st.arena[i];
    if (!a)
    {
        if (st.n_arenas == MAX_ARENAS)
            return fail(DH_EINVAL, "scratch arenas exist for %d streams already; no room for another stream", MAX_ARENAS);
        a = &st.arena[st.n_arenas++];
        *a = DeviceState::Arena{stream, nullptr, 0};
    }
    if (bytes > a->bytes)
    {
        // Work queued on the old arena must drain before it is released.
        DH_HIP(hipDeviceSynchronize());
        if (a->ptr)
            DH_HIP(hipFree(a->ptr));
        a->ptr = nullptr;
        a->bytes = 0;
        size_t want = (bytes + (size_t(1) << 20) - 1) & ~((size_t(1) << 20) - 1);
        DH_HIP(hipMalloc(&a->ptr, want));
        a->bytes = want;
    }
    *ptr = a->ptr;
    return 0;
}

bool workspace_at_hand(size_t bytes, hipStream_t stream)
{
    if (ensure_init() != 0)
        return false;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        const DeviceState& st = g_dev[g_cur];
        bool known = false;
        for (int i = 0; i < st.n_arenas; ++i)
            if (st.arena[i].stream == stream)
            {
                if (bytes <= st.arena[i].bytes)
                    return true;
                known = true;
            }
        if (!known && st.n_arenas == MAX_ARENAS)
            return false;
    }
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) == hipSuccess)
        return capturing == hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return false;
}

bool g_force_generic = false;
bool g_force_tiled = false;
int g_force_splitk = 0;
int g_force_tile_width = 0;

}  // namespace dh

using namespace dh;

namespace
{
// Whether the runtime knows the host address (an error or "unregistered": ordinary pageable memory).
bool known_to_device(const void* ptr)
{
    hipPointerAttribute_t attr;
    if (hipPointerGetAttributes(&attr, ptr) != hipSuccess)
    {
        (void)hipGetLastError();
        return false;
    }
    return attr.type != hipMemoryTypeUnregistered;
}

// Whether [ptr, ptr + bytes) lies within one allocation on `device`, and that is also the device of the calling thread: kernels and
// events go to the null stream of the thread's device (HIP keeps one a thread), which other devices' memory and work know nothing of.
bool inside_memory_of(int device, const void* ptr, size_t bytes)
{
    hipPointerAttribute_t attr;
    void* base = nullptr;
    size_t size = 0;
    int current = -1;
    if (hipGetDevice(&current) != hipSuccess || current != device || hipPointerGetAttributes(&attr, ptr) != hipSuccess ||
        attr.type != hipMemoryTypeDevice || attr.device != device ||
        hipMemGetAddressRange(&base, &size, const_cast<void*>(ptr)) != hipSuccess)
    {
        (void)hipGetLastError();
        return false;
    }
    const size_t offset = (size_t)(static_cast<const char*>(ptr) - static_cast<const char*>(base));
    return offset <= size && bytes <= size - offset;
}

constexpr int READ_NOT_STARTED = -1000;   // nothing was queued: the caller copies in another way

// A copy, shared by the thread that queues it and the helpers that take it out of the ring.  Both go by pieces, a launch each; a chunk is the
// pieces of one event.  Chunk c goes through slot c % slots; a slot is filled again only once every piece of the chunk before has been taken.
// Only the last chunk and the last piece are short, and nothing follows that chunk.
// Queueing, recording and waiting for a piece of 256 KiB by itself takes the queueing thread 11 us, the bus 5: an event for four of them, or
// for two where a copy has few, so that the first ones are there early.  Reading the weights of a model (38 MB in 18 calls) / sampling 64 images
// (3.1 MB), us: an event per piece 1750 / 321, as here 1510 / 300.  Pieces of 128 KiB and more than three helpers: 0 to 12 % slower.
struct Read
{
    char* dst;
    const char* ring;
    size_t bytes, chunk = READ_PIECE;
    int chunks, slots, pieces, per_chunk;
    std::atomic<int> arrived{0};                    // pieces 0 ... arrived - 1 are in the ring
    std::atomic<int> next{0};                       // next piece to take out
    std::atomic<bool> stop{false};                  // after an error: nothing further will arrive
    std::atomic<int> taken[READ_SLOTS_MAX] = {};    // pieces taken out of the slot so far
    std::mutex mu;                                  // with `moved`: helpers sleep until the first chunk is there, however long the
    std::condition_variable moved;                  // work in front of the copy takes; the chunks after it are microseconds apart

    Read(char* to, const void* through, size_t n) : dst(to), ring(static_cast<const char*>(through)), bytes(n)
    {
        while (chunk < READ_CHUNK_MAX && chunk < bytes / 6)
            chunk *= 2;
        slots = (int)(READ_RING / chunk);
        per_chunk = (int)(chunk / READ_PIECE);
        chunks = (int)((bytes + chunk - 1) / chunk);
        pieces = (int)((bytes + READ_PIECE - 1) / READ_PIECE);
    }
    size_t begin(int c) const { return (size_t)c * chunk; }
    size_t size(int c) const { return begin(c) + chunk <= bytes ? chunk : bytes - begin(c); }
    int pieces_up_to(int c) const { return c + 1 < chunks ? (c + 1) * per_chunk : pieces; }
    bool empty(int c) const     // the slot of chunk c, of the chunks before it
    {
        return taken[c % slots].load(std::memory_order_acquire) >= c / slots * per_chunk;
    }

    void take(int p)
    {
        const size_t from = (size_t)p * READ_PIECE;
        const int slot = p / per_chunk % slots;
        memcpy(dst + from, ring + (size_t)slot * chunk + (size_t)(p % per_chunk) * READ_PIECE, from + READ_PIECE <= bytes ? READ_PIECE : bytes - from);
        taken[slot].fetch_add(1, std::memory_order_release);
    }
    template <class T>
    void announce(std::atomic<T>& what, T value)
    {
        {
            std::lock_guard<std::mutex> lock(mu);
            what.store(value, std::memory_order_release);
        }
        moved.notify_all();
    }
    void help()
    {
        {
            std::unique_lock<std::mutex> lock(mu);
            moved.wait(lock, [this] { return arrived.load() > 0 || stop.load(); });
        }
        for (int p = next.fetch_add(1); p < pieces; p = next.fetch_add(1))
        {
            while (arrived.load(std::memory_order_acquire) <= p)
            {
                if (stop.load(std::memory_order_acquire))
                    return;
                std::this_thread::yield();
            }
            take(p);
        }
    }
};

int read_staged(DeviceState& st, char* dst, const char* src, size_t bytes)
{
    if (!st.read_ring)
    {
        void* ring = nullptr;
        if (hipHostMalloc(&ring, READ_RING, hipHostMallocDefault) != hipSuccess)
        {
            (void)hipGetLastError();
            return READ_NOT_STARTED;
        }
        for (hipEvent_t& e : st.read_done)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
            {
                (void)hipGetLastError();
                (void)hipHostFree(ring);
                return READ_NOT_STARTED;
            }
        st.read_ring = ring;
    }
    Read r(dst, st.read_ring, bytes);

    // on the null stream, as the blocking copy: behind what it and the streams that synchronise with it hold
    auto queue = [&](int c) -> hipError_t {
        for (size_t at = 0; at < r.size(c); at += READ_PIECE)
        {
            const size_t n = std::min(READ_PIECE, r.size(c) - at);
            hipLaunchKernelGGL(copy_from_pinned, dim3((unsigned)(n / 4096 + 1)), dim3(256), 0, nullptr,
                               static_cast<char*>(st.read_ring) + (size_t)(c % r.slots) * r.chunk + at, src + r.begin(c) + at, n, true);
            const hipError_t launched = hipGetLastError();
            if (launched != hipSuccess)
                return launched;
        }
        return hipEventRecord(st.read_done[c % r.slots], nullptr);
    };
    hipError_t err = hipSuccess;
    int queued = 0;
    for (; queued < r.chunks && queued < r.slots && err == hipSuccess; ++queued)
        err = queue(queued);

    std::thread helper[READ_THREADS_MAX];
    int helpers = 0;
    while (err == hipSuccess && helpers < READ_THREADS_MAX && helpers < (int)(bytes >> 20))
    {
        try
        {
            helper[helpers] = std::thread([&r] { r.help(); });
        }
        catch (...)
        {
            break;   // no thread to be had: fewer helpers
        }
        ++helpers;
    }
    for (int c = 0; c < r.chunks && err == hipSuccess; ++c)
    {
        err = hipEventSynchronize(st.read_done[c % r.slots]);
        if (err != hipSuccess)
            break;
        if (helpers == 0)
            for (int p = c * r.per_chunk; p < r.pieces_up_to(c); ++p)
                r.take(p);
        else if (c == 0)
            r.announce(r.arrived, r.pieces_up_to(0));
        else
            r.arrived.store(r.pieces_up_to(c), std::memory_order_release);
        // refill the slots that have been emptied; with all others in flight, wait for the oldest
        while (queued < r.chunks && err == hipSuccess)
        {
            if (r.empty(queued))
                err = queue(queued++);
            else if (queued - (c + 1) > 0)
                break;          // chunks are still under way: on to the next of them
            else
                std::this_thread::yield();
        }
    }
    if (err == hipSuccess && helpers > 0)
        r.help();                               // everything is there: what is left is shared
    if (err != hipSuccess)
    {
        (void)hipStreamSynchronize(nullptr);    // no copy into the ring outlives the call
        r.announce(r.stop, true);
    }
    for (int h = 0; h < helpers; ++h)
        helper[h].join();
    if (err != hipSuccess)
        return fail_hip(err, "dh_memcpy_d2h");
    return 0;
}
}  // namespace

extern "C" {

const char* dh_version(void) { return "dcgan_hip 0.1 (gfx950)"; }

const char* dh_last_error(void) { return g_err; }

int dh_init(int device) { return init_device(device); }

int dh_device_info(char* name, size_t name_len, int* compute_units, int* clock_khz,
                   size_t* memory_bytes)
{
    DH_TRY(ensure_init());
    hipDeviceProp_t prop;
    DH_HIP(hipGetDeviceProperties(&prop, g_cur));
    if (name && name_len)
    {
        snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
    }
    if (compute_units) *compute_units = prop.multiProcessorCount;
    if (clock_khz) *clock_khz = prop.clockRate;
    if (memory_bytes) *memory_bytes = prop.totalGlobalMem;
    return 0;
}

int dh_malloc(void** ptr, size_t bytes)
{
    DH_TRY(ensure_init());
    if (!ptr) return fail(DH_EINVAL, "dh_malloc: null result pointer");
    *ptr = nullptr;
    if (bytes == 0) bytes = 4;
    DH_HIP(hipMalloc(ptr, bytes));
    return 0;
}

int dh_free(void* ptr)
{
    if (!ptr) return 0;
    DH_TRY(ensure_init());
    DH_HIP(hipFree(ptr));
    return 0;
}

int dh_memcpy_h2d(void* dst, const void* src, size_t bytes)
{
    DH_TRY(ensure_init());
    if (bytes == 0) return 0;
    DH_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return 0;
}

int dh_memcpy_h2d_staged(void* dst, const void* src, size_t bytes, void* stream)
{
    DH_TRY(ensure_init());
    if (bytes == 0) return 0;
    if (!dst || !src) return fail(DH_EINVAL, "dh_memcpy_h2d_staged: null pointer");
    if (bytes > STAGE_MAX_BYTES)
    {
        // too large to stage: a blocking copy, ordered behind what `stream` holds by waiting for it
        // (streams made by dh_stream_create do not synchronise with the null stream by themselves)
        DH_HIP(hipStreamSynchronize(as_stream(stream)));
        DH_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
        return 0;
    }
    std::lock_guard<std::mutex> lock(g_mu);
    DeviceState& st = g_dev[g_cur];
    DeviceState::Stage& slot = st.stage[st.next_stage];
    st.next_stage = (st.next_stage + 1) % STAGE_SLOTS;
    if (slot.in_flight)
    {
        DH_HIP(hipEventSynchronize(slot.done));
        slot.in_flight = false;
    }
    if (!slot.done)
        DH_HIP(hipEventCreateWithFlags(&slot.done, hipEventDisableTiming));
    if (bytes > slot.bytes)
    {
        if (slot.host)
            DH_HIP(hipHostFree(slot.host));
        slot.host = nullptr;
        slot.bytes = 0;
        const size_t want = (bytes + 65535) & ~size_t(65535);
        DH_HIP(hipHostMalloc(&slot.host, want, hipHostMallocDefault));
        slot.bytes = want;
    }
    memcpy(slot.host, src, bytes);
    // From the staging buffer to the device with a kernel that reads the pinned memory across the bus: in the
    // launch stream a copy command costs ~20 us before the kernel behind it starts, whatever its size (measured
    // on the 25 KB latent batch of a training step: 43 us per iteration for two such copies, 11 us for two of
    // these launches); for megabytes the two are equally fast (the 3 MB image batch: 80 us either way).
    if (bytes % 4 == 0 && (reinterpret_cast<uintptr_t>(dst) & 3) == 0)
    {
        const bool vec = (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
        size_t blocks = (bytes / 16 + 255) / 256;
        if (blocks < 1) blocks = 1;
        if (blocks > 1024) blocks = 1024;
        hipLaunchKernelGGL(copy_from_pinned, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream), dst, slot.host, bytes, vec);
        DH_LAUNCH_CHECK("copy_from_pinned");
    }
    else
        DH_HIP(hipMemcpyAsync(dst, slot.host, bytes, hipMemcpyHostToDevice, as_stream(stream)));
    DH_HIP(hipEventRecord(slot.done, as_stream(stream)));
    slot.in_flight = true;
    return 0;
}

int dh_memcpy_d2h(void* dst, const void* src, size_t bytes)
{
    DH_TRY(ensure_init());
    if (bytes == 0) return 0;
    // Large copies go through a pinned ring (8 MiB a device, kept), a chunk at a time: the device fills the next slots while
    // the host empties the ones that are there, with helper threads, since the page faults and the copy of one thread are
    // slower than the bus.  The runtime's own copy into pageable memory takes turns: a chunk across the bus, a wait, its copy.
    // Measured: a stretch of six training iterations at batch 64 that ends with reading all weights (38 MB in 18 calls) 20.5 -> 17.9 ms,
    // sampling 64 images (3.1 MB) 445 -> 395 us.  From 2 MiB on, where two helpers pay: runtime / ring, us, 2 MiB 119 / 98, 4 MiB 230 / 176,
    // 13 MiB 717 / 505 (with an event for every 256 KiB; see struct Read for what several to an event give).  With one helper, which does all the copying while the caller waits, or with none the ring gained nothing: 512 KiB
    // 29.9 / 31.9, 1 MiB 58 / 61, 1.75 MiB 102 / 103 (medians).
    // Small ones, a copy while another is in progress, host memory that the device reaches by itself (pinned, managed) and
    // whatever is not inside one allocation on the library's device, that being the thread's too, take the runtime's copy, which finds
    // the device of the memory by itself and refuses what it always did.
    const int device = g_cur;   // once: another thread may call dh_init meanwhile
    if (dst && bytes >= READ_STAGED_MIN && (reinterpret_cast<uintptr_t>(src) & 15) == 0 && bytes % 4 == 0 && !known_to_device(dst) &&
        inside_memory_of(device, src, bytes))
    {
        std::unique_lock<std::mutex> ring(g_read_mu, std::try_to_lock);
        if (ring.owns_lock())
        {
            // While a stream is captured the runtime refuses a blocking copy, one of no bytes too (1.3 us); the ring's launches it
            // would take.
            const hipError_t allowed = hipMemcpy(dst, src, 0, hipMemcpyDeviceToHost);
            if (allowed != hipSuccess)
                return fail_hip(allowed, "hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost)");
            const int rc = read_staged(g_dev[device], static_cast<char*>(dst), static_cast<const char*>(src), bytes);
            if (rc != READ_NOT_STARTED)
                return rc;
        }
    }
    DH_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return 0;
}

int dh_memcpy_d2d(void* dst, const void* src, size_t bytes, void* stream)
{
    DH_TRY(ensure_init());
    if (bytes == 0) return 0;
    DH_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)));
    return 0;
}

int dh_sync(void)
{
    DH_TRY(ensure_init());
    DH_HIP(hipDeviceSynchronize());
    return 0;
}

int dh_stream_create(void** stream)
{
    DH_TRY(ensure_init());
    hipStream_t s;
    DH_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *stream = s;
    return 0;
}

int dh_stream_destroy(void* stream)
{
    DH_TRY(ensure_init());
    hipStream_t s = as_stream(stream);
    DH_HIP(hipStreamSynchronize(s));
    {
        // the stream's scratch arena goes with it (the table holds at most MAX_ARENAS streams)
        std::lock_guard<std::mutex> lock(g_mu);
        DeviceState& st = g_dev[g_cur];
        for (int i = 0; i < st.n_arenas; ++i)
            if (st.arena[i].stream == s && s != nullptr)
            {
                if (st.arena[i].ptr)
                    DH_HIP(hipFree(st.arena[i].ptr));
                st.arena[i] = st.arena[st.n_arenas - 1];
                st.arena[--st.n_arenas] = DeviceState::Arena{nullptr, nullptr, 0};
                break;
            }
    }
    DH_HIP(hipStreamDestroy(s));
    return 0;
}

int dh_stream_sync(void* stream)
{
    DH_TRY(ensure_init());
    DH_HIP(hipStreamSynchronize(as_stream(stream)));
    return 0;
}

int dh_event_create(void** event)
{
    DH_TRY(ensure_init());
    hipEvent_t e;
    DH_HIP(hipEventCreate(&e));
    *event = e;
    return 0;
}

int dh_event_destroy(void* event)
{
    DH_HIP(hipEventDestroy(static_cast<hipEvent_t>(event)));
    return 0;
}

int dh_event_record(void* event, void* stream)
{
    DH_HIP(hipEventRecord(static_cast<hipEvent_t>(event), as_stream(stream)));
    return 0;
}

int dh_stream_wait_event(void* stream, void* event)
{
    DH_HIP(hipStreamWaitEvent(as_stream(stream), static_cast<hipEvent_t>(event), 0));
    return 0;
}

int dh_event_elapsed_ms(void* start, void* stop, float* ms)
{
    DH_HIP(hipEventSynchronize(static_cast<hipEvent_t>(stop)));
    DH_HIP(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)));
    return 0;
}

int dh_workspace_reserve(size_t bytes)
{
    void* p;
    return workspace(bytes, &p, nullptr);
}

size_t dh_workspace_bytes(void)
{
    size_t total = 0;
    if (g_cur >= 0)
        for (int i = 0; i < g_dev[g_cur].n_arenas; ++i)
            total += g_dev[g_cur].arena[i].bytes;
    return total;
}


int dh_debug_force_generic_conv(int on)
{
    g_force_generic = on != 0;
    return 0;
}

int dh_debug_force_tiled_conv(int on)
{
    g_force_tiled = on != 0;
    return 0;
}

int dh_debug_force_splitk(int splits)
{
    if (splits < 0) return fail(DH_EINVAL, "dh_debug_force_splitk: negative split count");
    g_force_splitk = splits;
    return 0;
}

int dh_debug_force_tile_width(int width)
{
    if (width != 0 && width != 64 && width != 128)
        return fail(DH_EINVAL, "dh_debug_force_tile_width: width must be 0, 64 or 128");
    g_force_tile_width = width;
    return 0;
}

}
