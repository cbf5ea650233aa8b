// pimc_direct.hpp -- kernel dispatch straight into a user-mode AQL queue, for the
// launches whose latency a Markov chain waits on (short Delta V requests of a
// context, the serving form's Delta V batches).
//
// hipLaunchKernel spends ~3 us of host time per launch here and its tail reaches
// 7-11 us; a dispatch packet written into an HSA queue of our own, with the
// kernel arguments in device memory written through the PCIe BAR, costs ~1.9 us
// of host time (most of it the read-back that orders the argument writes before
// the doorbell) with a flat tail.  A context's call is synchronous: it waits for
// the kernel's published results before it returns, and the context's HIP
// stream is quiet when the packet is written, so the two queues never run work
// of one context at the same time.  The server sends a batch's two kernels as
// packets on a queue of the slot's own, in order, and retires the batch from
// its published records.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <cstring>
#include <type_traits>

namespace pimc {

// A kernel as the packet processor sees it: its code object entry and the
// segment sizes the packet carries.
struct DirectKernel {
    uint64_t object = 0;
    uint32_t kernarg_bytes = 0, group_bytes = 0;
    bool ok() const { return object != 0; }
};

// One caller's ring of kernel-argument blocks in device memory.  Slot k is
// rewritten kDirectSlots dispatches later; the caller waits for each dispatch's
// results (published after every argument read) before its next one, so a
// slot is never rewritten while a kernel can still read it.
constexpr int kDirectSlots = 64;
constexpr size_t kDirectSlotBytes = 4096;
struct DirectRing {
    char* base = nullptr;
    int device = -1;
    unsigned next = 0;
    void* own_queue = nullptr;   // a queue of the ring's own (in order), or null: the device's shared queue
};

// A piece of the argument block: bytes [offset, offset + bytes) come from src.
struct ArgPiece {
    const void* src;
    uint32_t offset, bytes;
};

// Sets up the device's queue on first use and allocates the ring; false when
// direct dispatch is unavailable (the caller launches through HIP instead).
// own_queue: the ring gets an in-order queue of its own, for one thread whose
// packets depend on each other; otherwise it shares the device's queue, whose
// packets the caller orders by waiting for each result.
bool direct_ring_create(int device, DirectRing* r, bool own_queue = false);
// Waits for every packet queued so far on the ring's queue, then frees the ring
// (and its own queue).
void direct_ring_release(DirectRing* r);
// Device memory the host writes through the BAR (made visible by
// direct_flush), for data a packet's kernel reads; null when unavailable.
void* direct_alloc_visible(int device, size_t bytes);
void direct_free_visible(void* p);
// Resolves a __global__ function (its host stub) in the code object this
// library registered; false unless the code object's argument block is exactly
// 'bytes' long and the kernel needs no scratch.
bool direct_kernel(int device, const void* host_stub, hipStream_t stream, uint32_t bytes, DirectKernel* k);
// Writes the argument pieces into the ring's next slot, makes them visible to
// the device, and queues one dispatch of grid_x workgroups of block_x lanes.
void direct_dispatch(DirectRing* r, const DirectKernel& k, const ArgPiece* pieces, int n_pieces, uint32_t grid_x,
                     uint32_t block_x);
// The same in three steps, for several packets behind one flush: copy the
// pieces into the next slot (returns its address), make every BAR write so far
// visible to the device, queue the packet.
char* direct_stage(DirectRing* r, const ArgPiece* pieces, int n_pieces);
void direct_flush(int device);
void direct_submit(DirectRing* r, const DirectKernel& k, const char* kernargs, uint32_t grid_x, uint32_t block_x);
// direct_kernel, remembered per device and function for the life of the process (a
// loaded code object stays); null when the function cannot be dispatched.
const DirectKernel* direct_kernel_of(int device, const void* host_stub, hipStream_t stream, uint32_t bytes);

// A call's turn on the device's queue, which all contexts share and whose packets run one
// after another: a lengthy call (an action, a corrected or a long Delta V request) takes
// it only while no other call is on it, a brief one while no lengthy call is.  A call
// that gets no turn launches on its context's stream, beside the others, so no context
// waits behind another's kernels.  Actions of N = 256 x 167 from one, two and four threads
// with a context each, us per action: 23.7, 13.7 and 11.5; every action on the queue 23.7,
// 18.8 and 18.8; every action on its stream 25.1, 14.2 and 15.5.
class QueueTurn {
public:
    QueueTurn(int device, bool lengthy);
    ~QueueTurn();
    QueueTurn(const QueueTurn&) = delete;
    QueueTurn& operator=(const QueueTurn&) = delete;
    explicit operator bool() const { return taken; }

private:
    int device;
    bool lengthy, taken;
};

// The kernels of one call, in order, as packets behind one flush on the device's
// queue.  (A packet without the barrier bit, to run beside the one before it, gained
// nothing: the first kernel's workgroups are all dispatched before it.)  send() queues nothing and returns false when a kernel cannot
// be dispatched: the caller then launches all of them through HIP.
class PacketList {
public:
    PacketList(DirectRing* r, hipStream_t st) : ring(r), stream(st) {}
    // Bytes copied of an argument of more than 1 KB (a request's inline bead list).
    uint32_t long_arg_bytes = UINT32_MAX;
    template <class... Ps, class... As>
    void add(void (*kern)(Ps...), dim3 g, dim3 b, size_t lds, const As&... as) {
        static_assert(sizeof...(Ps) == sizeof...(As), "one value per parameter");
        alignas(16) char blob[kDirectSlotBytes];
        uint32_t end = 0;
        (put<Ps>(blob, &end, as), ...);
        add_blob(reinterpret_cast<const void*>(kern), g, b, lds, blob, end);
    }
    bool send();

private:
    static constexpr int kMost = 8;
    struct Packet {
        DirectKernel k;
        const char* args;
        dim3 g, b;
    };
    template <class P, class A>
    void put(char* blob, uint32_t* end, const A& a) {
        using T = std::remove_cv_t<P>;
        static_assert(std::is_trivially_copyable_v<T>, "an argument is copied bytewise");
        const uint32_t o = (*end + alignof(T) - 1) / alignof(T) * alignof(T);
        *end = o + sizeof(T);
        if (*end > kDirectSlotBytes) return;   // add_blob refuses it
        if constexpr (std::is_same_v<T, A>) {
            std::memcpy(blob + o, &a, sizeof(T) > 1024 && long_arg_bytes < sizeof(T) ? long_arg_bytes : sizeof(T));
        } else {
            const T t = a;
            std::memcpy(blob + o, &t, sizeof(T));
        }
    }
    void add_blob(const void* stub, dim3 g, dim3 b, size_t lds, const char* blob, uint32_t bytes);
    DirectRing* ring;
    hipStream_t stream;
    Packet list[kMost];
    int n = 0;
    bool ok = true;
};

// One kernel of a call: a packet, or a launch on the stream.
struct Launcher {
    hipStream_t st;
    PacketList* packets = nullptr;
    template <class... Ps, class... As>
    void operator()(void (*kern)(Ps...), dim3 g, dim3 b, size_t lds, const As&... as) const {
        if (packets)
            packets->add(kern, g, b, lds, as...);
        else
            hipLaunchKernelGGL(kern, g, b, lds, st, as...);
    }
};

// Copies from device to page-locked host memory on the DMA engines, outside any
// HIP stream: the caller starts one when the data is complete (after an event or a
// synchronisation that releases the device's caches to the system) and waits for
// all of them before the memory is used, freed or written again.
struct DmaCopies {
    uint64_t signal = 0;          // hsa_signal_t: copies still running
    uint64_t gpu = 0, cpu = 0;    // hsa_agent_t of the source and the destination
};
// False when src and dst are not plain HIP allocations of a GPU and of the host.
bool dma_open(DmaCopies* d, const void* src, const void* dst);
bool dma_start(DmaCopies* d, void* dst, const void* src, size_t bytes);
// Waits for every copy started; false if one failed.
bool dma_wait(DmaCopies* d);
void dma_close(DmaCopies* d);

}  // namespace pimc
