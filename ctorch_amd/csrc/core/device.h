// Per-GPU context (compute stream + stream-ordered pool) and the storage owner shared by all tensors.
// Mirrors the reference's lazily created, mutex-guarded per-device Context (src/backends/cuda_context.cpp:121-133)
// and its Allocation {address, release} owner (src/core/tensor_data.h:11-15), over the HIP C ABI only.
#pragma once

#include "dl/types.h"
#include "backends/hip_backend.h"
#include "kernels/kernels.h"

#include <cstddef>
#include <cstdint>
#include <map>
#include <memory>
#include <mutex>
#include <string>

namespace dl::detail {

/// Throws std::runtime_error("HIP: <what>: <error>") for a nonzero HIP status.
void hip_check(int status, const char* what);

/// Freed device blocks of up to kBlockMax bytes, held for the next allocation of their size instead of going through
/// the runtime's pool and back: a hipMallocAsync / hipFreeAsync pair takes the host 10.6 us on MI355X, and a small decoder
/// chunk allocates ten tensors.  A block freed while work that uses it is still queued may be handed out at
/// once, as the runtime's pool does, because all of a device's work is ordered on its one compute stream.  While that
/// stream is being captured nothing is taken from here or put back, and a block that was allocated then never comes
/// here: it is the graph's.  At most `limit` bytes and kBlocks blocks are held; the oldest go back to the runtime's pool.
struct BlockCache {
    static constexpr std::size_t kBlockMax = std::size_t(32) << 20, kLimit = std::size_t(256) << 20, kBlocks = 256;
    struct Block {
        void* data;
        std::uint64_t age;
    };
    std::mutex mutex;
    std::multimap<std::size_t, Block> blocks; ///< by size
    std::size_t held = 0, limit = kLimit;
    std::size_t live = 0, peak = 0; ///< bytes of the tensors alive now, and their high-water mark
    std::size_t held_peak = 0;      ///< most bytes held at once since the peaks were reset
    std::uint64_t clock = 0;
};

struct GpuContext {
    int index = 0;
    BlockCache cache;
    dlh_stream stream = nullptr;
    dlh_device_properties properties{};
    int32_t* error_flag = nullptr; // device flag set by kernels that detect invalid input (e.g. token ids)
};

/// Returns the context of GPU `index`, creating it on first use, and makes the device current on this thread.
GpuContext& gpu_context(int index);
/// Throws when the library runs without a usable GPU (the product has no CPU compute path).
void require_gpu(Device device, const char* operation);

struct Storage {
    void* data = nullptr;
    std::size_t bytes = 0;
    std::size_t block = 0; ///< GPU: bytes of the block behind it
    bool captured = false; ///< GPU: allocated while the stream was captured
    Device device{};
    Storage() = default;
    Storage(const Storage&) = delete;
    Storage& operator=(const Storage&) = delete;
    ~Storage();
};

std::shared_ptr<Storage> allocate_storage(std::size_t bytes, Device device);

/// Checks and clears the device error flag of `device` (blocking read); throws with `what` if it was set.
void check_device_errors(Device device, const char* what);

} // namespace dl::detail
