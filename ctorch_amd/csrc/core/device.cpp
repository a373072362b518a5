#include "core/device.h"

#include "dl/gpu.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <stdexcept>
#include <vector>

namespace dl::detail {

void hip_check(int status, const char* what) {
    if (status != 0) throw std::runtime_error(std::string("HIP: ") + what + ": " + dlh_error_string(status));
}

namespace {
std::mutex context_mutex;
std::vector<std::unique_ptr<GpuContext>>& contexts() {
    // intentionally leaked: tensors released during interpreter or static teardown still find their stream
    static auto* value = new std::vector<std::unique_ptr<GpuContext>>();
    return *value;
}
thread_local int current_device = -1;
} // namespace

GpuContext& gpu_context(int index) {
    GpuContext* context = nullptr;
    {
        std::lock_guard<std::mutex> lock(context_mutex);
        auto& all = contexts();
        if (all.empty()) {
            int count = 0;
            hip_check(dlh_device_count(&count), "device count");
            all.resize(static_cast<std::size_t>(count));
        }
        if (index < 0 || static_cast<std::size_t>(index) >= all.size())
            throw std::runtime_error("HIP: GPU " + std::to_string(index) + " is not available (" +
                                     std::to_string(all.size()) + " visible)");
        auto& slot = all[static_cast<std::size_t>(index)];
        if (!slot) {
            auto created = std::make_unique<GpuContext>();
            created->index = index;
            hip_check(dlh_set_device(index), "set device");
            hip_check(dlh_device_properties_get(index, &created->properties), "device properties");
            hip_check(dlh_pool_configure(index), "memory pool");
            hip_check(dlh_stream_create(&created->stream), "stream create");
            void* flag = nullptr;
            hip_check(dlh_malloc_async(&flag, 256, created->stream), "error flag");
            hip_check(dlk_fill(flag, DLK_F32, 1, 0.0, created->stream), "error flag reset");
            created->error_flag = static_cast<int32_t*>(flag);
            slot = std::move(created);
        }
        context = slot.get();
    }
    if (current_device != index) {
        hip_check(dlh_set_device(index), "set device");
        current_device = index;
    }
    return *context;
}

void require_gpu(Device device, const char* operation) {
    if (device.type != DeviceType::gpu)
        throw std::invalid_argument(std::string(operation) +
                                    ": this build computes on the GPU only; move the tensors/modules with to(gpu)");
}

namespace {

bool capturing(const GpuContext& context) {
    int active = 0;
    hip_check(dlh_stream_capturing(context.stream, &active), "stream capture status");
    return active != 0;
}

// returns the oldest blocks to the runtime's pool until at most `bytes` are held (the cache's mutex held)
void shrink(GpuContext& context, std::size_t bytes, std::size_t blocks) {
    auto& cache = context.cache;
    while (cache.held > bytes || cache.blocks.size() > blocks) {
        auto oldest = cache.blocks.begin();
        for (auto it = cache.blocks.begin(); it != cache.blocks.end(); ++it)
            if (it->second.age < oldest->second.age) oldest = it;
        (void)dlh_free_async(oldest->second.data, context.stream);
        cache.held -= oldest->first;
        cache.blocks.erase(oldest);
    }
}

// a block of at least `bytes`, which receives its size, and whether a capture recorded the allocation
void* take_block(GpuContext& context, std::size_t& bytes, bool& captured) {
    auto& cache = context.cache;
    captured = capturing(context);
    const bool direct = captured || bytes > BlockCache::kBlockMax;
    std::lock_guard<std::mutex> lock(cache.mutex);
    void* data = nullptr;
    if (!direct) {
        // the smallest that fits, if at most an eighth of it goes unused
        const auto found = cache.blocks.lower_bound(bytes);
        if (found != cache.blocks.end() && found->first <= bytes + bytes / 8) {
            bytes = found->first;
            data = found->second.data;
            cache.held -= bytes;
            cache.blocks.erase(found);
        }
    }
    if (!data) {
        int status = dlh_malloc_async(&data, bytes, context.stream);
        if (status != 0 && !captured && cache.held > 0) { // short of memory: the held blocks go back first
            shrink(context, 0, 0);
            status = dlh_malloc_async(&data, bytes, context.stream);
        }
        if (status != 0) (void)dlh_last_launch_error(); // the next launch must not report it again
        hip_check(status, "allocate");
    }
    cache.live += bytes;
    cache.peak = std::max(cache.peak, cache.live);
    return data;
}

void give_block(GpuContext& context, void* data, std::size_t bytes, bool captured) {
    auto& cache = context.cache;
    int active = 0;
    const bool direct = captured || bytes > BlockCache::kBlockMax ||
                        dlh_stream_capturing(context.stream, &active) != 0 || active != 0;
    std::lock_guard<std::mutex> lock(cache.mutex);
    cache.live -= bytes;
    bool kept = false;
    if (!direct && bytes <= cache.limit) {
        try { // called from a destructor
            cache.blocks.emplace(bytes, BlockCache::Block{data, cache.clock++});
            kept = true;
        } catch (const std::bad_alloc&) {
        }
    }
    if (kept) cache.held_peak = std::max(cache.held_peak, cache.held += bytes);
    else (void)dlh_free_async(data, context.stream);
    if (!direct) shrink(context, cache.limit, BlockCache::kBlocks);
}

} // namespace

Storage::~Storage() {
    if (!data) return;
    if (device.type == DeviceType::cpu) {
        std::free(data);
    } else {
        // stream-ordered release: later work on the compute stream may reuse the block immediately
        give_block(gpu_context(device.index), data, block, captured);
    }
}

std::shared_ptr<Storage> allocate_storage(std::size_t bytes, Device device) {
    auto storage = std::make_shared<Storage>();
    storage->bytes = bytes;
    storage->device = device;
    const std::size_t rounded = bytes == 0 ? 64 : (bytes + 63) / 64 * 64;
    if (device.type == DeviceType::cpu) {
        storage->data = std::aligned_alloc(64, rounded);
        if (!storage->data) throw std::bad_alloc();
        std::memset(storage->data, 0, rounded);
    } else {
        storage->block = rounded;
        storage->data = take_block(gpu_context(device.index), storage->block, storage->captured);
    }
    return storage;
}

void check_device_errors(Device device, const char* what) {
    if (device.type != DeviceType::gpu) return;
    GpuContext& context = gpu_context(device.index);
    int32_t flag = 0;
    hip_check(dlh_memcpy_async(&flag, context.error_flag, sizeof(flag), DLH_DEVICE_TO_HOST, context.stream), what);
    hip_check(dlh_stream_synchronize(context.stream), what);
    if (flag != 0) {
        hip_check(dlk_fill(context.error_flag, DLK_F32, 1, 0.0, context.stream), what);
        throw std::out_of_range(std::string(what) + ": index out of range");
    }
}

} // namespace dl::detail

namespace dl {
void synchronize(Device device) {
    if (device.type != DeviceType::gpu) return;
    auto& context = detail::gpu_context(device.index);
    detail::hip_check(dlh_stream_synchronize(context.stream), "synchronize");
}
} // namespace dl

namespace dl::gpu {
MemoryStats memory_stats(int device) {
    auto& cache = detail::gpu_context(device).cache;
    std::lock_guard<std::mutex> lock(cache.mutex);
    MemoryStats out{};
    detail::hip_check(dlh_pool_stats(device, &out.used_bytes, &out.reserved_bytes, &out.peak_used_bytes,
                                     &out.peak_reserved_bytes, &out.release_threshold),
                      "pool statistics");
    // held blocks are free ones: `used` counts the live tensors and what others have of the pool
    const std::uint64_t ours = cache.live + cache.held, others = out.used_bytes > ours ? out.used_bytes - ours : 0;
    out.used_bytes = cache.live + others;
    // Their peak: that of the tensors with what others have now, or the pool's own less the most that was held, the larger
    // (others may have given back what they had at the pool's peak)
    const std::uint64_t pool_peak = out.peak_used_bytes;
    out.peak_used_bytes = std::max<std::uint64_t>(cache.peak > 0 ? cache.peak + others : 0,
                                                  pool_peak > cache.held_peak ? pool_peak - cache.held_peak : 0);
    return out;
}

void set_memory_release_threshold(std::uint64_t bytes, int device) {
    auto& context = detail::gpu_context(device);
    {
        std::lock_guard<std::mutex> lock(context.cache.mutex);
        context.cache.limit = static_cast<std::size_t>(std::min<std::uint64_t>(bytes, detail::BlockCache::kLimit));
        // during a capture the next free after it brings the held blocks within the limit
        if (!detail::capturing(context)) detail::shrink(context, context.cache.limit, detail::BlockCache::kBlocks);
    }
    detail::hip_check(dlh_pool_set_threshold(device, bytes), "pool release threshold");
}

void reset_peak_memory_stats(int device) {
    auto& cache = detail::gpu_context(device).cache;
    {
        std::lock_guard<std::mutex> lock(cache.mutex);
        cache.peak = 0; // the next allocation raises it again
        cache.held_peak = cache.held;
    }
    detail::hip_check(dlh_pool_reset_peaks(device), "pool peak reset");
}

void release_unused_memory(int device) {
    auto& context = detail::gpu_context(device);
    detail::hip_check(dlh_stream_synchronize(context.stream), "synchronize"); // refused during a capture
    {
        std::lock_guard<std::mutex> lock(context.cache.mutex);
        detail::shrink(context, 0, 0);
    }
    detail::hip_check(dlh_stream_synchronize(context.stream), "synchronize");
    detail::hip_check(dlh_pool_trim(device), "pool trim");
}
} // namespace dl::gpu
