// What the library's host side decides for a call, without a GPU: linked from the library's own objects (these functions
// are not part of its exported surface), with host memory and a list of the launches in the place of the device.  Run by
// tests/test_host_rules.py.
//
//   host_checks split BATCH HEADS KV_HEADS HEAD_DIM KV_BF16 LENGTH SOURCE CAUSAL    attention_split: splits, keys per split
//   host_checks projection EPILOGUE ROWS K R0 R1 R2 BF16 BIAS LAYER
//                                               the kernel of a projection (store, residual, qkv or swiglu) with R0, R1, R2
//                                               weight rows (0: no segment): in a decoder layer, or called by itself
//   host_checks attention BATCH HEADS KV_HEADS HEAD_DIM KV_BF16 LENGTH SOURCE CAUSAL MASKED    the kernel of an attention
//   host_checks threshold                       blocks held after a free: at first, at threshold 0, back at the first one
//   host_checks retry                           allocations that the memory holds only without the held blocks: 1, 1
//   host_checks capture                         a block allocated while the stream is captured and freed after it: how many
//                                               went back to the runtime, and 1 if the next allocation got it again
//   host_checks capture_release                blocks that went back to the runtime: during a capture by a threshold of 0 and
//                                               by release_unused_memory, and by the next free after the capture
//   host_checks peak                            MiB of memory_stats' used and peak with a tensor of 4 alive: after another
//                                               user of the pool had 64 and gave them back, with the tensor then freed and
//                                               held, and after a reset
//   host_checks workspace ENTRY ROWS K BYTES    launches of linear, swiglu or attention over bf16 weights with BYTES of
//                                               device memory left for their workspaces (-1: no limit)
#include "dl/decoder.h"
#include "dl/gpu.h"
#include "dl/ops.h"
#include "nn/decode_step.h"

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <stdexcept>
#include <string>

namespace {

struct Device {
    std::map<void*, size_t> blocks; // allocations alive
    size_t used = 0, peak = 0, limit = SIZE_MAX, launches = 0;
    int last_error = 0, capturing = 0;
} fake;

} // namespace

// ------------------------------------------------------------------------- the backend, on host memory
extern "C" {

const char* dlh_error_string(int code) { return code == hipErrorOutOfMemory ? "out of memory" : "error"; }
int dlh_device_count(int* count) { return *count = 1, 0; }
int dlh_set_device(int) { return 0; }
int dlh_get_device(int* device) { return *device = 0, 0; }
int dlh_device_properties_get(int, dlh_device_properties* out) { return std::memset(out, 0, sizeof(*out)), 0; }
int dlh_stream_create(dlh_stream* stream) { return *stream = reinterpret_cast<dlh_stream>(&fake), 0; }
int dlh_stream_destroy(dlh_stream) { return 0; }
int dlh_stream_synchronize(dlh_stream) { return fake.capturing ? hipErrorStreamCaptureUnsupported : 0; }
int dlh_pool_configure(int) { return 0; }
int dlh_malloc_async(void** pointer, size_t bytes, dlh_stream) {
    if (bytes > fake.limit - std::min(fake.limit, fake.used)) return fake.last_error = hipErrorOutOfMemory;
    *pointer = std::aligned_alloc(256, (bytes + 255) / 256 * 256); // never touched where the case is large
    fake.blocks[*pointer] = bytes;
    fake.peak = std::max(fake.peak, fake.used += bytes);
    return 0;
}
int dlh_free_async(void* pointer, dlh_stream) {
    fake.used -= fake.blocks.at(pointer);
    fake.blocks.erase(pointer);
    std::free(pointer);
    return 0;
}
int dlh_pool_stats(int, uint64_t* used, uint64_t* reserved, uint64_t* peak_used, uint64_t* peak_reserved, uint64_t* threshold) {
    *used = *reserved = fake.used;
    *peak_used = *peak_reserved = fake.peak;
    return *threshold = UINT64_MAX, 0;
}
int dlh_pool_trim(int) { return 0; }
int dlh_pool_set_threshold(int, uint64_t) { return 0; }
int dlh_pool_reset_peaks(int) { return fake.peak = 0, 0; } // the next allocation raises it again
int dlh_memcpy_async(void* to, const void* from, size_t bytes, int, dlh_stream) { return std::memcpy(to, from, bytes), 0; }
int dlh_event_create(dlh_event*) { return 0; }
int dlh_event_destroy(dlh_event) { return 0; }
int dlh_event_record(dlh_event, dlh_stream) { return 0; }
int dlh_event_synchronize(dlh_event) { return 0; }
int dlh_event_elapsed(dlh_event, dlh_event, float* ms) { return *ms = 0, 0; }
int dlh_capture_begin(dlh_stream) { return 0; }
int dlh_stream_capturing(dlh_stream, int* capturing) { return *capturing = fake.capturing, 0; }
int dlh_capture_end(dlh_stream, dlh_graph*) { return 0; }
int dlh_graph_launch(dlh_graph, dlh_stream) { return 0; }
int dlh_graph_destroy(dlh_graph) { return 0; }
int dlh_last_launch_error(void) { return std::exchange(fake.last_error, 0); }

// the runtime functions that the launch code calls: a launch counts, and reports an error that an earlier call left
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    fake.launches += 1;
    return static_cast<hipError_t>(std::exchange(fake.last_error, 0));
}
static thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } configured; // of a <<<>>> launch
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    configured = {grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
    *grid = configured.grid, *block = configured.block, *lds = configured.lds, *stream = configured.stream;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return static_cast<hipError_t>(std::exchange(fake.last_error, 0)); }
hipError_t hipGetDevice(int* device) { return *device = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) { return *value = 256, hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* blocks, const void*, int, size_t) { return *blocks = 4, hipSuccess; }

} // extern "C"

namespace {

using dl::detail::empty_tensor;

int split(char** arg) {
    int splits = 0, chunk = 0;
    auto at = [&](int i) { return std::atoll(arg[i]); };
    dl::detail::attention_split(at(0), at(1), at(2), at(3), at(4) != 0, at(5), at(6), at(7) != 0, splits, chunk);
    std::printf("%d %d\n", splits, chunk);
    return 0;
}

int projection(char** arg) {
    const std::string epilogue = arg[0];
    auto at = [&](int i) { return static_cast<int>(std::atoll(arg[i])); };
    alignas(64) static char memory[64]; // every address that the rules look at; nothing is launched
    auto* f32 = reinterpret_cast<float*>(memory);
    dlk_gemv_params p{};
    p.epilogue = epilogue == "store" ? DLK_EPI_STORE : epilogue == "residual" ? DLK_EPI_RESIDUAL
               : epilogue == "qkv" ? DLK_EPI_QKV : DLK_EPI_SWIGLU;
    p.M = at(1), p.K = at(2), p.ldx = p.K, p.x = f32, p.y = f32;
    for (int s = 0; s < 3 && at(3 + s) > 0; ++s) {
        p.seg_rows[p.nseg++] = at(3 + s);
        p.w[s] = memory;
        if (p.epilogue != DLK_EPI_SWIGLU || s == 0) p.ldy += p.epilogue == DLK_EPI_QKV && s > 0 ? 0 : at(3 + s);
    }
    p.w_bf16 = at(6);
    p.bias = at(7) ? memory : nullptr;
    p.residual = f32, p.ldres = p.ldy;
    p.head_dim = 32, p.kv_heads = 1, p.length = p.M, p.acc_scale = 1.0f;
    p.k_cache = p.v_cache = memory;
    p.cosine = p.sine = f32;
    p.apply_norm = p.epilogue == DLK_EPI_QKV || p.epilogue == DLK_EPI_SWIGLU;
    if (at(8) || dlk_gemv_uses_rows(&p)) { // what attach_workspace and attach_workspace_if_room attach
        p.stage_bytes = dlk_gemv_stage_bytes(&p);
        p.stage = p.stage_bytes > 0 ? memory : nullptr;
    }
    std::printf("%s\n", dlk_gemv_kernel(&p));
    return 0;
}

int attention(char** arg) {
    auto at = [&](int i) { return static_cast<int>(std::atoll(arg[i])); };
    alignas(64) static char memory[64];
    dlk_attention_params p{};
    p.B = at(0), p.H = at(1), p.KV = at(2), p.hd = at(3), p.kv_bf16 = at(4), p.L = at(5), p.causal = at(7);
    p.capacity = at(6), p.first_host = at(6) - at(5), p.early_keys = at(6);
    p.q = p.out = reinterpret_cast<float*>(memory);
    p.k = p.v = memory;
    p.ldq = p.ldo = static_cast<int64_t>(p.H) * p.hd;
    p.keep_mask = at(8) ? reinterpret_cast<unsigned char*>(memory) : nullptr;
    dl::detail::attention_split(p.B, p.H, p.KV, p.hd, p.kv_bf16 != 0, p.L, p.capacity, p.causal != 0, p.splits, p.chunk);
    std::printf("%s\n", dlk_attention_kernel(&p));
    return 0;
}

int threshold() {
    const dl::Device gpu = dl::Device::gpu(0);
    { dl::Tensor first = empty_tensor({64}, dl::DType::f32, gpu); }
    dl::gpu::release_unused_memory(0);
    const size_t base = fake.blocks.size();
    auto held = [&] {
        { dl::Tensor t = empty_tensor({1 << 18}, dl::DType::f32, gpu); }
        return fake.blocks.size() - base;
    };
    const size_t before = held();
    dl::gpu::set_memory_release_threshold(0);
    const size_t at_once = fake.blocks.size() - base, at_zero = held();
    dl::gpu::set_memory_release_threshold(UINT64_MAX);
    std::printf("%zu %zu %zu %zu\n", before, at_once, at_zero, held());
    return 0;
}

int retry() {
    const dl::Device gpu = dl::Device::gpu(0);
    const dl::Index mib = 1 << 18; // floats
    auto hold = [&] { // 3 x 16 MiB, freed
        dl::Tensor a = empty_tensor({16 * mib}, dl::DType::f32, gpu), b = empty_tensor({16 * mib}, dl::DType::f32, gpu),
                   c = empty_tensor({16 * mib}, dl::DType::f32, gpu);
    };
    hold();
    fake.limit = fake.used + (size_t(8) << 20);
    int fits[2];
    for (int i = 0; i < 2; ++i) { // above the largest block that is held, and below it
        try {
            dl::Tensor t = empty_tensor({(i == 0 ? 40 : 24) * mib}, dl::DType::f32, gpu);
            fits[i] = 1;
        } catch (const std::runtime_error&) {
            fits[i] = 0;
        }
        hold();
    }
    std::printf("%d %d\n", fits[0], fits[1]);
    return 0;
}

int capture() {
    const dl::Device gpu = dl::Device::gpu(0);
    const dl::Index n = 1 << 20;
    { dl::Tensor first = empty_tensor({64}, dl::DType::f32, gpu); } // the context exists
    fake.capturing = 1;
    dl::Tensor recorded = empty_tensor({n}, dl::DType::f32, gpu);
    fake.capturing = 0;
    void* block = dl::detail::mutable_data(recorded);
    const size_t alive = fake.blocks.size();
    recorded = dl::Tensor();
    const size_t returned = alive - fake.blocks.size();
    const dl::Tensor next = empty_tensor({n}, dl::DType::f32, gpu);
    std::printf("%zu %d\n", returned, !returned && dl::detail::mutable_data(next) == block);
    return 0;
}

int capture_release() {
    { dl::Tensor held = empty_tensor({1 << 20}, dl::DType::f32, dl::Device::gpu(0)); }
    const size_t all = fake.blocks.size();
    fake.capturing = 1;
    dl::gpu::set_memory_release_threshold(0);
    const size_t by_threshold = all - fake.blocks.size();
    try {
        dl::gpu::release_unused_memory(); // refused: it waits for the stream
    } catch (const std::runtime_error&) {
    }
    const size_t by_release = all - fake.blocks.size();
    fake.capturing = 0;
    { dl::Tensor next = empty_tensor({64}, dl::DType::f32, dl::Device::gpu(0)); }
    std::printf("%zu %zu %zu\n", by_threshold, by_release, all - fake.blocks.size());
    return 0;
}

int peak() {
    const dl::Device gpu = dl::Device::gpu(0);
    dl::Tensor own = empty_tensor({1 << 20}, dl::DType::f32, gpu);
    auto print = [] {
        const auto stats = dl::gpu::memory_stats(0);
        std::printf("%llu %llu\n", static_cast<unsigned long long>(stats.used_bytes >> 20),
                    static_cast<unsigned long long>(stats.peak_used_bytes >> 20));
    };
    void* others = nullptr;
    (void)dlh_malloc_async(&others, size_t(64) << 20, nullptr);
    (void)dlh_free_async(others, nullptr);
    print();
    own = dl::Tensor();
    print();
    dl::gpu::reset_peak_memory_stats(0);
    print();
    return 0;
}

int workspace(char** arg) {
    const std::string entry = arg[0];
    const dl::Index rows = std::atoll(arg[1]), k = std::atoll(arg[2]), left = std::atoll(arg[3]);
    const dl::Device gpu = dl::Device::gpu(0);
    const dl::TensorOptions options{.dtype = dl::DType::bf16, .device = gpu};
    const dl::Index n = 512;
    const dl::Tensor x = empty_tensor({1, rows, k}, dl::DType::f32, gpu), w = empty_tensor({n, k}, dl::DType::bf16, gpu);
    dl::nn::SwiGLU swiglu(k, n, false, options);
    dl::nn::GroupedQueryAttention attention(k, k / 128, k / 256, entry == "attention" ? rows : 1, options);
    auto call = [&] {
        if (entry == "linear") (void)dl::linear(x, w);
        else if (entry == "swiglu") (void)swiglu.forward(x);
        else if (entry == "attention") (void)attention.forward(x);
        else throw std::invalid_argument("entry");
    };
    dl::gpu::set_memory_release_threshold(0); // no freed blocks held
    const size_t before = fake.used;
    dl::Index own = 0; // bytes of the tensors that the call needs whatever it launches
    if (entry == "linear") own = rows * n * 4;
    if (entry == "swiglu") own = rows * (n + k) * 4;
    if (entry == "attention") own = rows * 3 * k * 4 + 2 * rows * (k / 2) * 4 + (1 << 12); // q, attended, out; the local cache
    if (left >= 0) fake.limit = before + static_cast<size_t>(own + left);
    fake.launches = 0;
    call();
    std::printf("%zu\n", fake.launches);
    return 0;
}

} // namespace

int main(int argc, char** argv) {
    try {
        if (argc == 10 && std::strcmp(argv[1], "split") == 0) return split(argv + 2);
        if (argc == 11 && std::strcmp(argv[1], "projection") == 0) return projection(argv + 2);
        if (argc == 11 && std::strcmp(argv[1], "attention") == 0) return attention(argv + 2);
        if (argc == 2 && std::strcmp(argv[1], "threshold") == 0) return threshold();
        if (argc == 2 && std::strcmp(argv[1], "retry") == 0) return retry();
        if (argc == 2 && std::strcmp(argv[1], "capture") == 0) return capture();
        if (argc == 2 && std::strcmp(argv[1], "capture_release") == 0) return capture_release();
        if (argc == 2 && std::strcmp(argv[1], "peak") == 0) return peak();
        if (argc == 6 && std::strcmp(argv[1], "workspace") == 0) return workspace(argv + 2);
    } catch (const std::exception& error) {
        std::fprintf(stderr, "%s\n", error.what());
        return 1;
    }
    std::fprintf(stderr, "see the head of host_checks.cpp\n");
    return 2;
}
