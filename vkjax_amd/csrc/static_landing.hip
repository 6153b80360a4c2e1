// vkj_seq_eval_next_static: vkj_seq_eval_next for callers that must not allocate (serving loops
// and harnesses in which hipMalloc is forbidden or too slow to tolerate on the request path).
//
// vkj_seq_eval_next parks the arguments of the following evaluation in landing buffers in HBM
// that it allocates, with pinned staging memory of their own, when a slot is first handed in.
// Here the landing buffers are pieces of one array that is part of the library's device image,
// the pinned buffer every recorded upload already owns serves as staging, and a copy kernel
// moves the landed arguments on. Streams and events are made by vkj_ctx_create. The entry point
// therefore calls no hipMalloc, hipHostMalloc, hipFree, stream or event creation.
//
// Every GPU the library runs on holds its own copy of the array (VKJ_STATIC_LANDING_BYTES) from
// the moment the library is loaded there until the process ends. All calls on one GPU share it,
// and it keeps what the last call left: a call only reads back the bytes it has just written,
// so nothing needs clearing. Two calls that overlap in time on one GPU (two threads, two
// contexts) would race on it: the array is claimed for the duration of a call and the second
// caller is refused with VKJ_ESTATE (seq_eval_static in shim.cpp, which also holds the other
// refusals, so that the host-only test build exercises them).
#include "shim_internal.h"

#include <algorithm>
#include <cstring>

using namespace vkj;

static __device__ __align__(256) unsigned char scratch[VKJ_STATIC_LANDING_BYTES];

namespace {

// dst[0 .. nbytes) = src[0 .. nbytes); 16 bytes per lane where both sides allow it
__global__ __launch_bounds__(256) void move_landed(unsigned char* __restrict__ dst, const unsigned char* __restrict__ src,
                                                   size_t nbytes, int vectors) {
    const size_t stride = (size_t)gridDim.x * 256u;
    size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (vectors) {
        const size_t nvec = nbytes / 16u;
        const uint4* s4 = reinterpret_cast<const uint4*>(src);
        uint4* d4 = reinterpret_cast<uint4*>(dst);
        for (size_t v = i; v < nvec; v += stride) d4[v] = s4[v];
        for (size_t b = nvec * 16u + i; b < nbytes; b += stride) dst[b] = src[b];
    } else {
        for (; i < nbytes; i += stride) dst[i] = src[i];
    }
}

// Every range of the table; block (x, y) copies its share of range y. Host memory is read and written at system scope, past the caches: what
// an earlier launch found there is not what the host has put there since.
__global__ __launch_bounds__(256) void carry_ranges(Carry what, int to_host, Notice notice) {
    const auto r = what.range[blockIdx.y];
    const uint32_t stride = gridDim.x * 256u, first = blockIdx.x * 256u + threadIdx.x;
    const bool vectors = (((uintptr_t)r.dst | (uintptr_t)r.src) & 15u) == 0;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    // (a range is below 2 GiB: larger evaluations are staged and sent in chunks)
    const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(r.src), 0, (int)r.nbytes, 0x00020000),
                                 to   = __builtin_amdgcn_make_buffer_rsrc(r.dst, 0, (int)r.nbytes, 0x00020000);
    constexpr int SYSTEM = 17;                                          // sc0 sc1
    const uint32_t whole = vectors ? (uint32_t)(r.nbytes / 16u) : 0u;
    for (uint32_t v = first; v < whole; v += stride) {
        if (to_host) __builtin_amdgcn_raw_buffer_store_b128(__builtin_amdgcn_raw_buffer_load_b128(from, v * 16u, 0, 0), to, v * 16u, 0, SYSTEM);
        else         __builtin_amdgcn_raw_buffer_store_b128(__builtin_amdgcn_raw_buffer_load_b128(from, v * 16u, 0, SYSTEM), to, v * 16u, 0, 0);
    }
    for (uint32_t w = whole * 4u + first; w < (uint32_t)(r.nbytes / 4u); w += stride) {
        if (to_host) __builtin_amdgcn_raw_buffer_store_b32(__builtin_amdgcn_raw_buffer_load_b32(from, w * 4u, 0, 0), to, w * 4u, 0, SYSTEM);
        else         __builtin_amdgcn_raw_buffer_store_b32(__builtin_amdgcn_raw_buffer_load_b32(from, w * 4u, 0, SYSTEM), to, w * 4u, 0, 0);
    }
    if (notice.done == nullptr) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                    // this block's share is in the host's memory
    __syncthreads();
    if (threadIdx.x != 0) return;
    const uint32_t blocks = gridDim.x * gridDim.y;
    if (blocks > 1u) {
        if (__hip_atomic_fetch_add(notice.count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u != blocks) return;
        __hip_atomic_store(notice.count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __hip_atomic_store(notice.done, notice.number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void write_stamp(uint64_t* clock, uint64_t* done, uint64_t number) {
    __hip_atomic_store(clock, (uint64_t)wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (done) __hip_atomic_store(done, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

int stamp_on(uint64_t* clock, uint64_t* done, uint64_t number, hipStream_t stream) {
    void* args[] = {&clock, &done, &number};
    HIP_TRY(hipLaunchKernel((const void*)write_stamp, dim3(1), dim3(1), args, 0, stream));
    return 0;
}

int carry_ranges_on(const Carry& what, bool to_host, const Notice& notice, hipStream_t stream) {
    if (!what.count) return 0;
    uint64_t most = 0;
    for (int k = 0; k < what.count; k++) most = std::max<uint64_t>(most, what.range[k].nbytes);
    // 32 blocks keep the link busy (784 KB in 32, 128 and 512 blocks: 28.4, 29.9, 31.8 us)
    const uint64_t blocks = std::min<uint64_t>(32u, (most + 4095u) / 4096u);
    Carry table = what;
    int out = to_host;
    Notice last = notice;
    void* args[] = {&table, &out, &last};
    HIP_TRY(hipLaunchKernel((const void*)carry_ranges, dim3((unsigned)blocks, (unsigned)what.count), dim3(256), args, 0, stream));
    return 0;
}

int carry_on(const Carry& what, bool to_host, hipStream_t stream) { return carry_ranges_on(what, to_host, Notice{}, stream); }
int carry_out_on(const Carry& what, const Notice& notice, hipStream_t stream) { return carry_ranges_on(what, true, notice, stream); }

int move_on(void* dst, const void* src, size_t nbytes, hipStream_t stream) {
    if (!nbytes) return 0;
    const int vectors = (((uintptr_t)dst | (uintptr_t)src) & 15u) == 0;
    const size_t items = vectors ? (nbytes + 15u) / 16u : nbytes;
    size_t blocks = (items + 255u) / 256u;
    if (blocks > 8192u) blocks = 8192u;              // 32 workgroups per CU; the kernel strides over the rest
    // launched through the call that returns its own status: hipGetLastError would also hand back what an
    // earlier, unrelated call left behind (a kernel name looked up in the wrong module)
    unsigned char* d = (unsigned char*)dst;
    const unsigned char* s = (const unsigned char*)src;
    int vec = vectors;
    void* args[] = {&d, &s, &nbytes, &vec};
    HIP_TRY(hipLaunchKernel((const void*)move_landed, dim3((unsigned)blocks), dim3(256), args, 0, stream));
    return 0;
}

}  // namespace

// Called by vkj_ctx_create with the context's device current: the array's name is only a
// host-side stand-in, its address on this device has to be asked for.
int vkj::static_landing_init(Ctx* c) {
    void* p = nullptr;
    HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(VKJ_ENODEV, "vkj_ctx_create: the static landing array has no address on device %d", c->device);
    c->static_landing = p;
    int khz = 0;
    HIP_TRY(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c->device));
    HIP_TRY(hipMalloc((void**)&c->carry_count, 256));
    HIP_TRY(hipMemset(c->carry_count, 0, 256));
    HIP_TRY(hipDeviceSynchronize());
    c->carry = carry_on;
    if (khz > 0) {
        c->clock_khz = khz;
        c->carry_out = carry_out_on;
        c->stamp = stamp_on;
    }
    return 0;
}

extern "C" int vkj_seq_eval_next_static(vkj_handle sh, void* const* host_ptrs, int nslots, uint32_t flags,
                                        void* const* next_host_ptrs) {
    Seq* s = from_handle<Seq>(sh, MAGIC_SEQ);
    if (!s) return fail(VKJ_EINVAL, "vkj_seq_eval_next_static: bad handle");
    return seq_eval_static(s, host_ptrs, nslots, flags, next_host_ptrs, move_on);
}
