// libgpumpi.so -- the gfx950 device MPI runtime, its built-in rank programs and the host
// C ABI of include/gpumpi/gpumpi.h.  This unit holds the host API and the batched steps'
// host code; the rank programs and the many-instance batched kernels are compiled as units
// of their own (units.h).  The device runtime is header-only and is inlined into every
// rank program.
#include "runtime/mpi_api.h"
#include "runtime/rank_kernel.h"
#include "runtime/batched.h"
#include "runtime/batched_reduce.h"
#include "runtime/bucket.h"
#include "runtime/bucket_plan.h"
#include "runtime/particle_step.h"
#include "runtime/run_status.h"
#include "runtime/workspace.h"
#include "programs/workloads.h"
#include "programs/serve.h"
#include "../../include/gpumpi/gpumpi.h"
#include "units.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

namespace gpumpi {

struct InitBases {
    int32_t* posted;
    Envelope* unexp;
    Request* reqs;
    int32_t* free_stack;
    char* scratch;
};

__global__ void init_runtime_kernel(Runtime* R, InitBases b) {
    const int P = R->nranks;
    const uint64_t ring = (uint64_t)R->ring_slots;
    const uint64_t mr = (uint64_t)R->max_requests;
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = tid; i < (uint64_t)P * ring; i += stride) {
        R->rings[i].seq = (uint32_t)(i % ring);
        R->rings[i].ctx = 0;
    }
    for (uint64_t r = tid; r < (uint64_t)P; r += stride) {
        RankState& s = R->ranks[r];
        s.world_rank = (int32_t)r;
        s.n_posted = 0;
        s.n_unexp = 0;
        s.n_free = (int32_t)mr;
        s.ring_head = 0;
        s.posted = b.posted + r * mr;
        s.unexp = b.unexp + r * (uint64_t)R->max_unexpected;
        s.reqs = b.reqs + r * mr;
        s.free_stack = b.free_stack + r * mr;
        s.scratch = b.scratch + r * kScratchBytes;
        s.initialized = 0;
        s.finalized = 0;
        s.arena = nullptr;
        heap_cache_clear(&s.cache);
        s.cache.shard = (int32_t)(r % (uint64_t)R->heap.nshards);
        R->mailbox[r].tail = 0;
        R->world->slots[r].seq = 0;
        R->world->seqs[r] = 0;
    }
    for (uint64_t i = tid; i < (uint64_t)P * mr; i += stride) {
        uint64_t k = i % mr;
        b.free_stack[i] = (int32_t)(mr - 1 - k);
        b.reqs[i].state = kReqFree;
        b.reqs[i].index = (int32_t)k;
    }
    for (uint64_t pg = tid; pg < R->heap.npages; pg += stride) R->heap.page_class[pg] = 0xFF;
    for (uint64_t i = tid; i < (uint64_t)kHeapClasses * kHeapShards; i += stride)
        *heap_head(&R->heap, (int)(i / kHeapShards), (int)(i % kHeapShards)) = kHeapEmpty;
    if (tid == 0) {
        R->heap.page_bump = 0;
        R->heap.bytes_in_use = 0;
        R->heap.peak_in_use = 0;
        R->heap.alloc_count = 0;
        R->heap.refill_count = 0;
        R->world->arrive.value = 0;
        R->world->gen.value = 0;
        R->next_ctx = 2;
        R->abort_flag = 0;
        R->exit_code = 0;
        R->err_lock = 0;
        R->err.code = 0;
        R->err.rank = -1;
    }
}

__global__ void clear_status_kernel(Runtime* R) {
    if (threadIdx.x == 0) {
        R->abort_flag = 0;
        R->exit_code = 0;
        R->err_lock = 0;
        R->err.code = 0;
        R->err.rank = -1;
        R->err.msg[0] = 0;
    }
}

// A launch's argument block, passed by value: the bytes go to `dst` and the runtime points to
// them.  (As two copies from pageable memory they cost more than the launch itself.)
constexpr size_t kArgsByValue = 1024;
struct ArgsBlock {
    uint32_t words[kArgsByValue / 4];
};
__global__ void stage_args_kernel(Runtime* R, uint32_t* dst, uint32_t words, ArgsBlock a) {
    for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) dst[i] = a.words[i];
    if (threadIdx.x == 0) R->user_args = dst;
}

// The run's status to pinned memory: Allreduce of 1000 doubles on 256 ranks, ten calls, 357 ->
// 349 us with the arguments by value and the events kept.
__global__ void report_status_kernel(const Runtime* R, RunStatus* out) {
    if (threadIdx.x == 0) {
        out->abort_flag = R->abort_flag;
        out->exit_code = R->exit_code;
        out->err = R->err;
    }
}

// Launch-local world size (plain one-launch-per-job mode): the first k ranks of the
// runtime form MPI_COMM_WORLD; collective sequence numbers and barrier words restart.
__global__ void resize_world_kernel(Runtime* R, int k) {
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < k; r += gridDim.x * blockDim.x) {
        R->world->slots[r].seq = 0;
        R->world->seqs[r] = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        R->nranks = k;
        R->world->size = k;
        R->world_group->size = k;
        R->world->arrive.value = 0;
        R->world->gen.value = 0;
    }
}

// Empties the heap: page bump, class stacks, the ranks' block caches, live-byte count.
// Launched before each plain job, which -- like a fresh program -- starts on a clean heap.
__global__ void heap_reset_kernel(Runtime* R, int nstates) {
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    for (int r = tid; r < nstates; r += gridDim.x * blockDim.x)
        heap_cache_clear(&R->ranks[r].cache);
    for (int i = tid; i < kHeapClasses * kHeapShards; i += gridDim.x * blockDim.x)
        *heap_head(&R->heap, i / kHeapShards, i % kHeapShards) = kHeapEmpty;
    if (tid == 0) {
        R->heap.page_bump = 0;
        R->heap.bytes_in_use = 0;
    }
}

// The built-in rank programs: tables from programs_tests.hip, programs_work.hip and
// programs_heavy.hip, joined in that order on first use.
static const std::vector<ProgramEntry>& programs() {
    static const std::vector<ProgramEntry> all = [] {
        std::vector<ProgramEntry> v;
        v.insert(v.end(), kProgramsTests, kProgramsTests + kNumProgramsTests);
        v.insert(v.end(), kProgramsWork, kProgramsWork + kNumProgramsWork);
        v.insert(v.end(), kProgramsHeavy, kProgramsHeavy + kNumProgramsHeavy);
        return v;
    }();
    return all;
}

}  // namespace gpumpi

using namespace gpumpi;

// ==================================================================== host side
struct gpumpi_runtime {
    gpumpi_config cfg;
    int cus = 0;
    int wallclock_khz = 0;
    Runtime h{};
    Runtime* d_rt = nullptr;
    InitBases bases{};
    std::vector<void*> allocs;
    void* d_args = nullptr;
    size_t args_cap = 0;
    hipStream_t own_stream = nullptr;
    std::string err;
    bool needs_reset = false;
    int world_size = 0;  // ranks of MPI_COMM_WORLD as last set on the device
    int stage_dev = 0;   // Runtime::copy_stage_bytes as last set on the device
    size_t max_lds_block = 65536;  // LDS bytes a workgroup may hold on this device
    IoSlot* io = nullptr;  // pinned host I/O request slots, one per rank
    RunStatus* status = nullptr;           // pinned, behind the slots; written at the end of a run
    RunStatus* d_status = nullptr;         // its device address
    hipEvent_t ev[2] = {nullptr, nullptr}; // around a run's rank grid
    class IoService* io_service = nullptr;
};
static void io_service_free(class IoService* s);

static thread_local std::string g_host_error;

#define HIP_TRY(expr)                                                                      \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess) {                                                            \
            set_err(rt, std::string(#expr) + ": " + hipGetErrorString(e_));                \
            return GPUMPI_E_HIP;                                                           \
        }                                                                                  \
    } while (0)

static void set_err(gpumpi_runtime* rt, const std::string& s) {
    if (rt) rt->err = s;
    g_host_error = s;
}

static int dev_alloc(gpumpi_runtime* rt, void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes ? bytes : 16);
    if (e != hipSuccess) {
        set_err(rt, std::string("hipMalloc(") + std::to_string(bytes) + "): " + hipGetErrorString(e));
        return GPUMPI_E_NOMEM;
    }
    rt->allocs.push_back(*p);
    return GPUMPI_OK;
}

extern "C" {

void gpumpi_config_default(gpumpi_config* c) {
    std::memset(c, 0, sizeof(*c));
    c->num_ranks = 1;
    c->ranks_per_block = 1;
    c->ring_slots = 256;
    c->max_requests = 1024;
    c->max_unexpected = 1024;
    c->heap_bytes = 1ull << 30;
    c->timeout_s = 20.0;
    c->bcast_push_min = kBcastPushMinDefault;
}

int gpumpi_device_info(int32_t* num_cus, int32_t* wallclock_khz, int32_t* max_waves_per_cu) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return GPUMPI_E_HIP;
    int v = 0;
    if (num_cus) {
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return GPUMPI_E_HIP;
        *num_cus = v;
    }
    if (wallclock_khz) {
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeWallClockRate, dev) != hipSuccess)
            return GPUMPI_E_HIP;
        *wallclock_khz = v;
    }
    if (max_waves_per_cu) {
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxThreadsPerMultiProcessor, dev) != hipSuccess)
            return GPUMPI_E_HIP;
        *max_waves_per_cu = v / 64;
    }
    return GPUMPI_OK;
}

static int runtime_init_device(gpumpi_runtime* rt, hipStream_t s) {
    hipLaunchKernelGGL(init_runtime_kernel, dim3(1024), dim3(256), 0, s, rt->d_rt, rt->bases);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    rt->needs_reset = false;
    return GPUMPI_OK;
}

int gpumpi_runtime_create(const gpumpi_config* cfg_in, gpumpi_runtime** out) {
    if (!out) return GPUMPI_E_ARG;
    *out = nullptr;
    gpumpi_config cfg;
    gpumpi_config_default(&cfg);
    if (cfg_in) {
        cfg = *cfg_in;
        if (cfg.ranks_per_block <= 0) cfg.ranks_per_block = 1;
        if (cfg.ring_slots <= 0) cfg.ring_slots = 256;
        if (cfg.max_requests <= 0) cfg.max_requests = 1024;
        if (cfg.max_unexpected <= 0) cfg.max_unexpected = 1024;
        if (cfg.heap_bytes == 0) cfg.heap_bytes = 1ull << 30;
        if (cfg.timeout_s <= 0) cfg.timeout_s = 20.0;
        if (cfg.bcast_push_min == 0) cfg.bcast_push_min = kBcastPushMinDefault;
    }
    if (cfg.num_ranks <= 0 || cfg.ranks_per_block > 4) {
        g_host_error = "invalid num_ranks or ranks_per_block";
        return GPUMPI_E_ARG;
    }
    gpumpi_runtime* rt = new gpumpi_runtime();
    rt->cfg = cfg;
    int32_t cus = 0, khz = 0;
    if (gpumpi_device_info(&cus, &khz, nullptr) != GPUMPI_OK || khz <= 0) {
        set_err(rt, "cannot query the HIP device");
        delete rt;
        return GPUMPI_E_HIP;
    }
    rt->cus = cus;
    rt->wallclock_khz = khz;
    {
        int dev = 0, lds = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
            lds > 0)
            rt->max_lds_block = (size_t)lds;
    }
    if (cfg.stack_bytes) hipDeviceSetLimit(hipLimitStackSize, cfg.stack_bytes);

    const uint64_t P = (uint64_t)cfg.num_ranks;
    Runtime& h = rt->h;
    std::memset(&h, 0, sizeof(h));
    h.nranks = cfg.num_ranks;
    h.ranks_per_block = cfg.ranks_per_block;
    h.ring_slots = cfg.ring_slots;
    h.max_requests = cfg.max_requests;
    h.max_unexpected = cfg.max_unexpected;
    h.bcast_push_min = cfg.bcast_push_min;
    h.timeout_ticks = (uint64_t)(cfg.timeout_s * (double)khz * 1000.0);
    h.wtick = 1.0 / ((double)khz * 1000.0);
    h.next_ctx = 2;
    int rc = GPUMPI_OK;
    void* p = nullptr;
#define ALLOC(field, type, count)                                                     \
    if ((rc = dev_alloc(rt, &p, sizeof(type) * (size_t)(count))) != GPUMPI_OK) {      \
        gpumpi_runtime_destroy(rt);                                                   \
        return rc;                                                                    \
    }                                                                                 \
    field = (type*)p;
    ALLOC(rt->d_rt, Runtime, 1)
    ALLOC(h.mailbox, Mailbox, P)
    ALLOC(h.rings, Envelope, P * cfg.ring_slots)
    ALLOC(h.ranks, RankState, P)
    ALLOC(rt->bases.posted, int32_t, P * cfg.max_requests)
    ALLOC(rt->bases.unexp, Envelope, P * cfg.max_unexpected)
    ALLOC(rt->bases.reqs, Request, P * cfg.max_requests)
    ALLOC(rt->bases.free_stack, int32_t, P * cfg.max_requests)
    ALLOC(rt->bases.scratch, char, P * kScratchBytes)
    // heap arena: whole 64 KiB pages
    uint64_t heap = (cfg.heap_bytes + kHeapPage - 1) & ~(kHeapPage - 1);
    ALLOC(h.heap.base, char, heap)
    h.heap.bytes = heap;
    h.heap.npages = heap >> kHeapPageShift;
    h.heap.nshards = heap_shard_count(h.heap.npages);
    ALLOC(h.heap.page_class, uint8_t, h.heap.npages)
    ALLOC(h.heap.heads, uint64_t, (size_t)kHeapClasses * kHeapShards * kHeapHeadStride)
    // COMM_WORLD (reference: communicator.cu:52-62, context id 1) and the groups
    CommImpl world{};
    CollSlot* slots;
    uint64_t* seqs;
    ALLOC(slots, CollSlot, P)
    ALLOC(seqs, uint64_t, P)
    GroupImpl* groups;
    ALLOC(groups, GroupImpl, 2)
    CommImpl* d_world;
    ALLOC(d_world, CommImpl, 1)
#undef ALLOC
    // host I/O request slots (device-to-host delegation of the C library's file calls), and the
    // run's status behind them (an allocation of its own costs 70 us)
    static_assert(sizeof(IoSlot) % alignof(RunStatus) == 0, "the status follows the slots");
    const size_t pinned = sizeof(IoSlot) * (size_t)P + sizeof(RunStatus);
    if (hipHostMalloc((void**)&rt->io, pinned,
                      hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
        rt->io = nullptr;
        set_err(rt, "hipHostMalloc of the I/O slots failed");
        gpumpi_runtime_destroy(rt);
        return GPUMPI_E_NOMEM;
    }
    std::memset((void*)rt->io, 0, pinned);
    rt->status = (RunStatus*)(rt->io + P);
    {
        void* dio = nullptr;
        if (hipHostGetDevicePointer(&dio, rt->io, 0) != hipSuccess) dio = rt->io;
        h.io = (IoSlot*)dio;
        rt->d_status = (RunStatus*)(h.io + P);
    }
    GroupImpl hg[2];
    hg[0].size = cfg.num_ranks;
    hg[0].refcount = -1;
    hg[0].ranks = nullptr;  // identity
    hg[1].size = 0;
    hg[1].refcount = -1;
    hg[1].ranks = nullptr;
    world.ctx = 1;
    world.size = cfg.num_ranks;
    world.refcount = -1;
    world.is_world = 1;
    world.world_ranks = nullptr;
    world.inv = nullptr;
    world.slots = slots;
    world.seqs = seqs;
    world.group = groups;
    h.world = d_world;
    h.null_comm = nullptr;
    h.world_group = groups;
    h.empty_group = groups + 1;
    if (hipMemcpy(groups, hg, sizeof(hg), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(d_world, &world, sizeof(world), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(rt->d_rt, &h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess) {
        set_err(rt, "hipMemcpy of the runtime state failed");
        gpumpi_runtime_destroy(rt);
        return GPUMPI_E_HIP;
    }
    if (hipStreamCreate(&rt->own_stream) != hipSuccess) {
        set_err(rt, "hipStreamCreate failed");
        gpumpi_runtime_destroy(rt);
        return GPUMPI_E_HIP;
    }
    rc = runtime_init_device(rt, rt->own_stream);
    if (rc != GPUMPI_OK) {
        gpumpi_runtime_destroy(rt);
        return rc;
    }
    rt->world_size = cfg.num_ranks;
    *out = rt;
    return GPUMPI_OK;
}

void gpumpi_runtime_destroy(gpumpi_runtime* rt) {
    if (!rt) return;
    hipDeviceSynchronize();
    for (void* p : rt->allocs) hipFree(p);
    io_service_free(rt->io_service);
    if (rt->io) hipHostFree(rt->io);
    for (hipEvent_t e : rt->ev)
        if (e) hipEventDestroy(e);
    if (rt->d_args) hipFree(rt->d_args);
    if (rt->own_stream) hipStreamDestroy(rt->own_stream);
    delete rt;
}

const char* gpumpi_last_error(gpumpi_runtime* rt) {
    return rt ? rt->err.c_str() : g_host_error.c_str();
}

int gpumpi_program_count(void) { return (int)programs().size(); }

uint64_t gpumpi_layout_stamp(void) { return kLayoutStamp; }
int gpumpi_runtime_copy_stage(const gpumpi_runtime* rt) { return rt ? rt->stage_dev : 0; }
const char* gpumpi_program_name(int i) {
    return (i >= 0 && i < (int)programs().size()) ? programs()[i].name : nullptr;
}

static const ProgramEntry* find_program(const char* name) {
    if (!name) return nullptr;
    for (const ProgramEntry& e : programs())
        if (std::strcmp(e.name, name) == 0) return &e;
    return nullptr;
}

static int stage_args(gpumpi_runtime* rt, const void* args, size_t bytes, hipStream_t s) {
    if (bytes > rt->args_cap) {
        if (rt->d_args) hipFree(rt->d_args);
        rt->d_args = nullptr;
        size_t cap = bytes < 4096 ? 4096 : bytes;
        HIP_TRY(hipMalloc(&rt->d_args, cap));
        rt->args_cap = cap;
    }
    if (bytes <= kArgsByValue && rt->d_args) {
        ArgsBlock a;
        if (bytes) std::memcpy(&a, args, bytes);
        // (the launch's own result: hipGetLastError would also give an error of the thread's
        // earlier calls, which is not this run's)
        uint32_t words = (uint32_t)((bytes + 3) / 4);
        void* kargs[] = {(void*)&rt->d_rt, (void*)&rt->d_args, (void*)&words, (void*)&a};
        HIP_TRY(hipLaunchKernel((const void*)&stage_args_kernel, dim3(1), dim3(64), kargs, 0, s));
        return GPUMPI_OK;
    }
    if (bytes) HIP_TRY(hipMemcpyAsync(rt->d_args, args, bytes, hipMemcpyHostToDevice, s));
    const void* dp = rt->d_args;
    HIP_TRY(hipMemcpyAsync((char*)rt->d_rt + offsetof(Runtime, user_args), &dp, sizeof(dp),
                           hipMemcpyHostToDevice, s));
    return GPUMPI_OK;
}

// Launches a rank grid of `nranks` wavefronts (ranks_per_block per workgroup).  All ranks
// must be resident at once, since they spin-wait on each other; the reference checks its
// grid against the occupancy limit (gpu_main/main.cu:189-209).  Here a grid may use at
// most half of the wave slots its kernel can occupy on the chip.  A dispatch that needs
// every slot is not guaranteed to be placed all at once: workgroups are spread evenly
// over the XCDs and their shader arrays while harvested CUs make the arrays' capacities
// unequal, so an array can run out of room while others still have it (probes at exactly
// 32 waves per CU placed the last workgroups only after the first ones had given up at
// their barrier), and a rank that is never placed leaves the rest spinning until the
// bounded waits report it.  Rank programs use at most 256 registers per lane where the
// runtime alone is concerned (two waves per SIMD: 1024 ranks on 256 CUs); a program whose
// own loops need more holds one wave per SIMD and runs up to 512 ranks.
//
// Each wave may also get an LDS staging area for its large copies (dynamic LDS,
// copy_stage_kib): the largest of 64, 32 and 16 KiB with which the grid still passes that
// rule and the workgroup's LDS (the kernel's own plus the stages) fits the device's limit.
// Measured with 128 waves copying 64 MiB each: 14.3 / 15.8 / 19.1 GB/s per wave through a
// 16 / 32 / 64 KiB stage, 10.9 through registers alone.
static int launch_rank_grid(gpumpi_runtime* rt, const void* kernel, int nranks, int argc,
                            char** d_argv, hipStream_t s) {
    const int rpb = rt->cfg.ranks_per_block;
    const int block = 64 * rpb;
    const int grid = (nranks + rpb - 1) / rpb;
    const int64_t need = (int64_t)grid * rpb;
    const int kib = rt->cfg.copy_stage_kib;
    int cand[4], nc = 0;
    if (kib == 0) {
        cand[nc++] = 64 << 10;
        cand[nc++] = 32 << 10;
        cand[nc++] = 16 << 10;
    } else if (kib > 0 && kib <= 64) {
        cand[nc++] = kib << 10;
    }
    cand[nc++] = 0;
    hipFuncAttributes fa{};
    HIP_TRY(hipFuncGetAttributes(&fa, kernel));
    int per_cu = 0, stage = 0;
    int64_t slots = 0;
    for (int i = 0; i < nc; i++) {
        const size_t dyn = (size_t)cand[i] * (size_t)rpb;
        if (dyn != 0 && fa.sharedSizeBytes + dyn > rt->max_lds_block) continue;
        HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, dyn));
        slots = (int64_t)per_cu * rpb * rt->cus;  // wave slots this kernel can use
        stage = cand[i];
        if (need <= slots / 2) break;
    }
    if (need > slots / 2) {
        set_err(rt, "rank grid of " + std::to_string(need) + " wavefronts exceeds half of the " +
                        std::to_string(slots) + " wave slots this program can occupy (" +
                        std::to_string(per_cu) + " workgroups of " + std::to_string(rpb) +
                        " per CU)");
        return GPUMPI_E_RESIDENCY;
    }
    if (stage != rt->stage_dev) {
        rt->h.copy_stage_bytes = stage;
        HIP_TRY(hipMemcpyAsync((char*)rt->d_rt + offsetof(Runtime, copy_stage_bytes),
                               &rt->h.copy_stage_bytes, sizeof(int32_t), hipMemcpyHostToDevice, s));
        rt->stage_dev = stage;
    }
    Runtime* d = rt->d_rt;
    void* kargs[] = {(void*)&d, (void*)&argc, (void*)&d_argv};
    HIP_TRY(hipLaunchKernel(kernel, dim3(grid), dim3(block), kargs, (size_t)stage * (size_t)rpb, s));
    return GPUMPI_OK;
}

static int launch_program(gpumpi_runtime* rt, const ProgramEntry* pe, int argc, char** d_argv,
                          hipStream_t s) {
    if (rt->world_size != rt->cfg.num_ranks) {
        // a plain per-job launch shrank MPI_COMM_WORLD; restore the full rank grid
        hipLaunchKernelGGL(resize_world_kernel, dim3(4), dim3(256), 0, s, rt->d_rt,
                           rt->cfg.num_ranks);
        rt->world_size = rt->cfg.num_ranks;
    }
    return launch_rank_grid(rt, pe->kernel, rt->cfg.num_ranks, argc, d_argv, s);
}

int gpumpi_run_async(gpumpi_runtime* rt, const char* program, const void* args,
                     size_t args_bytes, void* stream) {
    if (!rt) return GPUMPI_E_ARG;
    const ProgramEntry* pe = find_program(program);
    if (!pe) {
        set_err(rt, std::string("unknown rank program: ") + (program ? program : "(null)"));
        return GPUMPI_E_PROGRAM;
    }
    hipStream_t s = stream ? (hipStream_t)stream : rt->own_stream;
    int rc = stage_args(rt, args, args_bytes, s);
    if (rc != GPUMPI_OK) return rc;
    return launch_program(rt, pe, 0, nullptr, s);
}

static int run_entry(gpumpi_runtime* rt, const ProgramEntry* pe, int argc,
                     const char* const* argv, const void* args, size_t args_bytes, void* stream,
                     double* elapsed_ms);

int gpumpi_run(gpumpi_runtime* rt, const char* program, int argc, const char* const* argv,
               const void* args, size_t args_bytes, void* stream, double* elapsed_ms) {
    if (!rt) return GPUMPI_E_ARG;
    const ProgramEntry* pe = find_program(program);
    if (!pe) {
        set_err(rt, std::string("unknown rank program: ") + (program ? program : "(null)"));
        return GPUMPI_E_PROGRAM;
    }
    return run_entry(rt, pe, argc, argv, args, args_bytes, stream, elapsed_ms);
}

int gpumpi_run_kernel(gpumpi_runtime* rt, const void* kernel, int argc, const char* const* argv,
                      const void* args, size_t args_bytes, void* stream, double* elapsed_ms) {
    if (!rt || !kernel) return GPUMPI_E_ARG;
    ProgramEntry pe{"(user kernel)", kernel};
    return run_entry(rt, &pe, argc, argv, args, args_bytes, stream, elapsed_ms);
}

// ==================================================================== host I/O service
// Serves the ranks' IoSlot requests while a rank grid runs (the device half is gpumpi_io
// in runtime/mpi_api.h).  One thread per runtime, started with its first grid and parked
// between grids, so a launch pays no thread start.  Files opened by ranks live in a
// table; handles are 1-based indices, the standard streams have fixed negative handles.
// Files still open when a grid ends are closed, as at process exit.
class IoService {
public:
    IoService(IoSlot* slots, int n) : slots_(slots), n_(n) {
        th_ = std::thread([this] { loop(); });
    }
    ~IoService() {
        {
            std::lock_guard<std::mutex> g(park_);
            quit_ = true;
        }
        wake_.notify_all();
        th_.join();
    }
    void begin() {
        {
            std::lock_guard<std::mutex> g(park_);
            active_.store(true);
        }
        wake_.notify_all();
    }
    // After the grid has finished: serve what it posted last, close its files.
    void end() {
        active_.store(false);
        std::lock_guard<std::mutex> g(serve_);
        drain_locked();
        for (FILE* f : files_)
            if (f) std::fclose(f);
        files_.clear();
    }

private:
    FILE* file(int64_t h) {
        if (h == kIoStdout) return stdout;
        if (h == kIoStderr) return stderr;
        if (h == kIoStdin) return stdin;
        if (h < 1 || h > (int64_t)files_.size()) return nullptr;
        return files_[(size_t)h - 1];
    }
    void serve(IoSlot& s) {
        FILE* f = s.op == kIoOpen ? nullptr : file(s.a0);
        int64_t r = -1;
        switch (s.op) {
        case kIoOpen: {
            const char* path = s.data;
            const size_t pl = strnlen(path, kIoData);
            const char* mode = pl + 1 < (size_t)kIoData ? path + pl + 1 : "r";
            FILE* nf = pl < (size_t)kIoData ? std::fopen(path, mode) : nullptr;
            if (nf) {
                files_.push_back(nf);
                r = (int64_t)files_.size();
            } else {
                r = 0;
            }
            break;
        }
        case kIoClose:
            if (f && s.a0 > 0) {
                r = std::fclose(f);
                files_[(size_t)s.a0 - 1] = nullptr;
            }
            break;
        case kIoWrite:
            if (f && s.len >= 0 && s.len <= kIoData) r = (int64_t)std::fwrite(s.data, 1, (size_t)s.len, f);
            break;
        case kIoRead:
            if (f) {
                const int64_t want = std::min<int64_t>(std::max<int64_t>(s.a1, 0), kIoData);
                r = (int64_t)std::fread(s.data, 1, (size_t)want, f);
            }
            break;
        case kIoGets:
            if (f && s.a1 > 0) {
                const int size = (int)std::min<int64_t>(s.a1, kIoData);
                r = std::fgets(s.data, size, f) ? (int64_t)std::strlen(s.data) + 1 : -1;
            }
            break;
        case kIoGetc: if (f) r = std::fgetc(f); break;
        case kIoUngetc: if (f) r = std::ungetc((int)s.a1, f); break;
        case kIoEof: if (f) r = std::feof(f); break;
        case kIoFlush: if (f) r = std::fflush(f); break;
        case kIoSeek: if (f) r = std::fseek(f, (long)s.a1, (int)s.a2); break;
        case kIoTell: if (f) r = std::ftell(f); break;
        default: break;
        }
        s.result = r;
    }
    bool drain() {
        std::lock_guard<std::mutex> g(serve_);
        return drain_locked();
    }
    bool drain_locked() {
        bool any = false;
        for (int i = 0; i < n_; i++) {
            IoSlot& s = slots_[i];
            const uint32_t seq = __atomic_load_n(&s.seq, __ATOMIC_ACQUIRE);
            if (seq & 1) {
                serve(s);
                __atomic_store_n(&s.seq, seq + 1, __ATOMIC_RELEASE);
                any = true;
            }
        }
        return any;
    }
    void loop() {
        int idle = 0;
        for (;;) {
            if (!active_.load()) {
                std::unique_lock<std::mutex> lk(park_);
                wake_.wait(lk, [this] { return quit_ || active_.load(); });
                if (quit_) return;
                idle = 0;
            }
            if (drain()) {
                idle = 0;
            } else if (++idle > 64) {
                std::this_thread::sleep_for(std::chrono::microseconds(20));
            }
        }
    }
    IoSlot* slots_;
    int n_;
    std::atomic<bool> active_{false};
    bool quit_ = false;
    std::mutex park_, serve_;
    std::condition_variable wake_;
    std::thread th_;
    std::vector<FILE*> files_;
};

static void io_service_free(IoService* s) { delete s; }

static int run_entry(gpumpi_runtime* rt, const ProgramEntry* pe, int argc,
                     const char* const* argv, const void* args, size_t args_bytes, void* stream,
                     double* elapsed_ms) {
    hipStream_t s = stream ? (hipStream_t)stream : rt->own_stream;
    rt->err.clear();
    if (rt->needs_reset) {
        int rc = runtime_init_device(rt, s);
        if (rc != GPUMPI_OK) return rc;
    }
    // argv strings (main.cu:24-43 copies them to managed memory)
    std::vector<char> blob;
    std::vector<size_t> offs;
    for (int i = 0; i < argc; i++) {
        offs.push_back(blob.size());
        const char* a = argv[i];
        blob.insert(blob.end(), a, a + std::strlen(a) + 1);
    }
    char** d_argv = nullptr;
    char* d_blob = nullptr;
    if (argc > 0) {
        HIP_TRY(hipMalloc((void**)&d_argv, sizeof(char*) * (argc + 1)));
        HIP_TRY(hipMalloc((void**)&d_blob, blob.size()));
        std::vector<char*> ptrs(argc + 1, nullptr);
        for (int i = 0; i < argc; i++) ptrs[i] = d_blob + offs[i];
        HIP_TRY(hipMemcpy(d_blob, blob.data(), blob.size(), hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(d_argv, ptrs.data(), sizeof(char*) * (argc + 1), hipMemcpyHostToDevice));
    }
    int rc = stage_args(rt, args, args_bytes, s);
    if (rc != GPUMPI_OK) return rc;
    hipLaunchKernelGGL(clear_status_kernel, dim3(1), dim3(64), 0, s, rt->d_rt);
    for (hipEvent_t& e : rt->ev)
        if (!e) HIP_TRY(hipEventCreate(&e));
    const hipEvent_t e0 = rt->ev[0], e1 = rt->ev[1];
    HIP_TRY(hipEventRecord(e0, s));
    if (!rt->io_service) rt->io_service = new IoService(rt->io, rt->cfg.num_ranks);
    rt->io_service->begin();
    status_arm(rt->status);
    rc = launch_program(rt, pe, argc, d_argv, s);
    HIP_TRY(hipEventRecord(e1, s));
    void* report[] = {(void*)&rt->d_rt, (void*)&rt->d_status};
    const hipError_t le = hipLaunchKernel((const void*)&report_status_kernel, dim3(1), dim3(64), report, 0, s);
    hipError_t se = hipStreamSynchronize(s);
    if (se == hipSuccess) se = le;
    rt->io_service->end();
    float ms = 0.f;
    hipEventElapsedTime(&ms, e0, e1);
    if (d_argv) hipFree(d_argv);
    if (d_blob) hipFree(d_blob);
    if (rc != GPUMPI_OK) return rc;
    if (se != hipSuccess) {
        set_err(rt, std::string("rank grid failed: ") + hipGetErrorString(se));
        return GPUMPI_E_HIP;
    }
    if (elapsed_ms) *elapsed_ms = ms;
    RunStatus hr;
    if (!status_read(rt->status, &hr)) {
        set_err(rt, "the run left no status");
        rt->needs_reset = true;
        return GPUMPI_E_HIP;
    }
    if (hr.abort_flag) {
        char msg[160];
        std::snprintf(msg, sizeof(msg), "device error %d on rank %d (line %d, detail %d): %s",
                      hr.err.code, hr.err.rank, hr.err.line, hr.err.detail, hr.err.msg);
        set_err(rt, msg);
        rt->h.err = hr.err;
        rt->needs_reset = true;
        return GPUMPI_E_DEVICE;
    }
    rt->h.err = hr.err;
    return hr.exit_code ? 1 : 0;
}

int gpumpi_last_device_error(gpumpi_runtime* rt, int32_t* code, int32_t* rank) {
    if (!rt) return GPUMPI_E_ARG;
    if (code) *code = rt->h.err.code;
    if (rank) *rank = rt->h.err.rank;
    return GPUMPI_OK;
}

int gpumpi_heap_stats(gpumpi_runtime* rt, int64_t* in_use, int64_t* peak, int64_t* capacity) {
    if (!rt) return GPUMPI_E_ARG;
    Heap hh;
    HIP_TRY(hipMemcpy(&hh, (char*)rt->d_rt + offsetof(Runtime, heap), sizeof(Heap),
                      hipMemcpyDeviceToHost));
    if (in_use) *in_use = hh.bytes_in_use;
    if (peak) *peak = hh.peak_in_use;
    if (capacity) *capacity = (int64_t)hh.bytes;
    return GPUMPI_OK;
}

int gpumpi_launch(const char* program, int argc, const char* const* argv, const void* args,
                  size_t args_bytes, const gpumpi_config* cfg) {
    gpumpi_runtime* rt = nullptr;
    int rc = gpumpi_runtime_create(cfg, &rt);
    if (rc != GPUMPI_OK) return rc;
    rc = gpumpi_run(rt, program, argc, argv, args, args_bytes, nullptr, nullptr);
    if (rc < 0) g_host_error = rt->err;
    gpumpi_runtime_destroy(rt);
    return rc;
}

static int launch_kernel_once(const void* kernel, int argc, const char* const* argv,
                              const gpumpi_config* cfg) {
    gpumpi_runtime* rt = nullptr;
    int rc = gpumpi_runtime_create(cfg, &rt);
    if (rc != GPUMPI_OK) return rc;
    rc = gpumpi_run_kernel(rt, kernel, argc, argv, nullptr, 0, nullptr, nullptr);
    if (rc < 0) g_host_error = rt->err;
    gpumpi_runtime_destroy(rt);
    return rc;
}

static int cli_main(const void* kernel, int argc, const char* const* argv);

int gpumpi_main(int argc, const char* const* argv) { return cli_main(nullptr, argc, argv); }

int gpumpi_main_kernel(const void* kernel, int argc, const char* const* argv) {
    if (!kernel) return 1;
    return cli_main(kernel, argc, argv);
}

// main.cu:49-98: "<program> <args> ---gpumpi -n N -g G -b B -s S -p P -e E".  With a
// kernel (a compiled user program), argv[0] is the executable and every argument before
// ---gpumpi is passed to __gpu_main; otherwise argv[0] names a built-in rank program.
static int cli_main(const void* kernel, int argc, const char* const* argv) {
    int sep = -1;
    for (int i = 0; i < argc; i++)
        if (std::strcmp(argv[i], "---gpumpi") == 0) sep = i;
    if (sep < 0) {
        std::fprintf(stderr, "You should specify gpumpi related options after '---gpumpi'\n");
        return 1;
    }
    if (sep < 1 && !kernel) {
        std::fprintf(stderr, "GPUMPI: no rank program named before '---gpumpi'\n");
        return 1;
    }
    gpumpi_config cfg;
    gpumpi_config_default(&cfg);
    long long n = 0, g = 0, b = 0;
    for (int i = sep + 1; i < argc; i++) {
        const char* o = argv[i];
        const char* v = i + 1 < argc ? argv[i + 1] : nullptr;
        auto num = [&](const char* s) { return s ? std::strtoll(s, nullptr, 0) : 0LL; };
        if (!std::strcmp(o, "-h") || !std::strcmp(o, "--help")) {
            std::printf("GPU MPI: -n numProcs -g blocksPerGrid -b threadsPerBlock (multiple of 64) "
                        "-s stackSize -p heapSize -e pendingBufferSize -t timeoutSeconds\n");
            return 0;
        }
        if (!v) break;
        if (!std::strcmp(o, "-n")) n = num(v);
        else if (!std::strcmp(o, "-g")) g = num(v);
        else if (!std::strcmp(o, "-b")) b = num(v);
        else if (!std::strcmp(o, "-s")) cfg.stack_bytes = (uint64_t)num(v);
        else if (!std::strcmp(o, "-p")) cfg.heap_bytes = (uint64_t)num(v);
        else if (!std::strcmp(o, "-e")) cfg.max_requests = (int32_t)num(v);
        else if (!std::strcmp(o, "-t")) cfg.timeout_s = std::strtod(v, nullptr);
        else { std::fprintf(stderr, "GPUMPI: unknown option %s\n", o); return 1; }
        i++;
    }
    if (b % 64 != 0 || b > 256) {
        std::fprintf(stderr, "GPUMPI: threads per block must be a multiple of 64 up to 256\n");
        return 1;
    }
    int rpb = b ? (int)(b / 64) : 1;
    if (n == 0) n = (g ? g : 1) * rpb;
    if (g && n > g * rpb) {
        std::fprintf(stderr, "GPUMPI: Requested number of processes %lld can't be allocated on "
                             "%lld blocks of %d ranks\n", n, g, rpb);
        return 1;
    }
    cfg.num_ranks = (int32_t)n;
    cfg.ranks_per_block = rpb;
    std::fprintf(stderr, "GPUMPI: Using %lld mpi processes (%d per workgroup)\n", n, rpb);
    int rc = kernel ? launch_kernel_once(kernel, sep, argv, &cfg)
                    : gpumpi_launch(argv[0], sep - 1, argv + 1, nullptr, 0, &cfg);
    if (rc < 0) {
        std::fprintf(stderr, "GPUMPI: %s\n", g_host_error.c_str());
        return 1;
    }
    return rc;
}

}  // extern "C"

// ==================================================================== batched Alltoallv
struct A2avGraph {
    int steps = 0;
    hipGraph_t def = nullptr;
    hipGraphExec_t exec = nullptr;
};

struct gpumpi_a2av_plan {
    A2avDev dev{};            // tables of workspace 0 (single steps, the first step of a graph)
    A2avDev dev2{};           // workspace 1: the other half of the pipelined graph's steps
    gpumpi_a2av_tune tune{};
    int grid = 0;             // copy-kernel workgroups
    int cus = 0;
    int64_t est_bytes = -1;   // payload of the last step read back (sizes the copy grid)
    int last_ws = 0;          // workspace of the last step launched
    std::vector<void*> allocs;
    std::vector<A2avGraph> graphs;  // one per step count replayed
    bool timing = false;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
};

// the copy kernel's instances are compiled in kernels_a2av.hip
static const void* a2av_copy_for(int U, bool nt, bool defer, bool fuse) {
    return a2av_copy_kernel_for(U, nt, defer, fuse);
}

// Copy grid: one workgroup per chunk of the last measured step (P extra for the partial
// last chunk of each row), or a default before any step was measured; blocks_per_cu > 0
// caps it (the workgroups then stride over the chunks).
static void a2av_size_grid(gpumpi_a2av_plan* pl) {
    const int64_t chunk_bytes = 16ll * pl->dev.chunk_lines;
    int64_t g = pl->est_bytes >= 0 ? pl->est_bytes / chunk_bytes + pl->dev.P : 64ll * pl->cus;
    if (pl->tune.blocks_per_cu > 0 && g > (int64_t)pl->tune.blocks_per_cu * pl->cus)
        g = (int64_t)pl->tune.blocks_per_cu * pl->cus;
    if (g < 1) g = 1;
    if (g > (1 << 22)) g = 1 << 22;
    // deferred mode: one thread per segment in leading blocks, at most four per CU
    const uint64_t PP = (uint64_t)pl->dev.P * (uint64_t)pl->dev.P;
    const uint64_t sblocks = (PP + kA2avCopyThreads - 1) / kA2avCopyThreads;
    const uint64_t scap = 4ull * (uint64_t)(pl->cus > 0 ? pl->cus : 1);
    pl->dev.straddle_blocks = pl->tune.defer_straddle > 0 ? (int32_t)(sblocks < scap ? sblocks : scap) : 0;
    pl->grid = (int)g + pl->dev.straddle_blocks;
}

static int a2av_configure(gpumpi_a2av_plan* pl, const gpumpi_a2av_tune& t) {
    const int U = t.lines_per_lane;
    if (U != 2 && U != 4 && U != 8) return GPUMPI_E_ARG;
    const int R = t.chunk_rounds <= 0 ? 1 : t.chunk_rounds;
    if (R != 1 && R != 2 && R != 4 && R != 8) return GPUMPI_E_ARG;
    if (t.block_threads != kA2avCopyThreads || t.blocks_per_cu < 0) return GPUMPI_E_ARG;
    pl->tune = t;
    pl->tune.nontemporal = t.nontemporal > 0 ? 1 : 0;
    pl->tune.chunk_rounds = R;
    pl->tune.defer_straddle = t.defer_straddle > 0 ? 1 : 0;
    if (t.pipeline < 0 || t.pipeline > 3) return GPUMPI_E_ARG;
    pl->tune.pipeline = t.pipeline;
    pl->dev.chunk_lines = (uint32_t)(kA2avCopyThreads * U * R);
    pl->dev.min_lines = (uint32_t)(kA2avCopyThreads * U);
    a2av_size_grid(pl);
    pl->dev2.chunk_lines = pl->dev.chunk_lines;
    pl->dev2.min_lines = pl->dev.min_lines;
    pl->dev2.straddle_blocks = pl->dev.straddle_blocks;
    return GPUMPI_OK;
}

// Plan and scan kernels (one kernel for few ranks); ev, if given, is recorded between them.
static int a2av_launch_tables(A2avDev& d, bool plan, hipStream_t s, hipEvent_t ev = nullptr) {
    void* kargs[] = {(void*)&d};
    const bool small = plan && d.P <= kA2avSmallRanks;
    if (plan && hipLaunchKernel(small ? (const void*)&a2av_plan_small_kernel : (const void*)&a2av_plan_kernel,
                                dim3(small ? 1 : d.P), dim3(small ? 1024 : 256), kargs, 0, s) != hipSuccess)
        return GPUMPI_E_HIP;
    if (ev) hipEventRecord(ev, s);
    if (!small && hipLaunchKernel((const void*)&a2av_scan_kernel, dim3(1), dim3(1024), kargs, 0, s) != hipSuccess)
        return GPUMPI_E_HIP;
    return GPUMPI_OK;
}

// One step on workspace 0: plan, scan, copy.
static int a2av_launch(gpumpi_a2av_plan* pl, hipStream_t s, bool timed) {
    A2avDev& d = pl->dev;
    void* kargs[] = {(void*)&d, (void*)&d};
    if (timed) hipEventRecord(pl->ev[0], s);
    if (a2av_launch_tables(d, true, s, timed ? pl->ev[1] : nullptr) != GPUMPI_OK) return GPUMPI_E_HIP;
    if (timed) hipEventRecord(pl->ev[2], s);
    if (hipLaunchKernel(a2av_copy_for(pl->tune.lines_per_lane, pl->tune.nontemporal > 0,
                                      pl->tune.defer_straddle > 0, false),
                        dim3(pl->grid), dim3(kA2avCopyThreads), kargs, 0, s) != hipSuccess)
        return GPUMPI_E_HIP;
    if (timed) hipEventRecord(pl->ev[3], s);
    pl->last_ws = 0;
    return GPUMPI_OK;
}

// The copy of the step whose tables are in workspace `cur`, with the plan of the next
// step (into the other workspace) in its first P workgroups when `plan_next`; that plan
// also computes the chunk scan in its last workgroup when `scan_too`.
static int a2av_launch_copy(gpumpi_a2av_plan* pl, hipStream_t s, int cur, bool plan_next,
                            bool scan_too = true) {
    A2avDev& a = cur == 0 ? pl->dev : pl->dev2;
    A2avDev b = cur == 0 ? pl->dev2 : pl->dev;
    if (!scan_too) b.plan_done = nullptr;
    void* kargs[] = {(void*)&a, (void*)&b};
    const int grid = pl->grid + (plan_next ? a.P : 0);
    if (hipLaunchKernel(a2av_copy_for(pl->tune.lines_per_lane, pl->tune.nontemporal > 0,
                                      pl->tune.defer_straddle > 0, plan_next),
                        dim3(grid), dim3(kA2avCopyThreads), kargs, 0, s) != hipSuccess)
        return GPUMPI_E_HIP;
    pl->last_ws = cur;
    return GPUMPI_OK;
}

static int a2av_launch_plan_scan(gpumpi_a2av_plan* pl, hipStream_t s, int ws, bool plan) {
    return a2av_launch_tables(ws == 0 ? pl->dev : pl->dev2, plan, s);
}

// `steps` steps, in the pipeline mode of the tune:
//   0  plan, scan and copy kernels per step;
//   1  each copy kernel also plans the next step into the other workspace (its first P
//      workgroups, no fences) and a scan kernel follows it;
//   2  as 1, and the plan's last workgroup computes the scan (one kernel per step);
//   3  plan and scan of step i+1 on a second stream, concurrent with copy i (graph
//      branches; copy i+1 waits for them, plan i+2 for copy i, which used its workspace).
static int a2av_launch_steps(gpumpi_a2av_plan* pl, hipStream_t s, int steps) {
    int rc = GPUMPI_OK;
    const int mode = pl->tune.pipeline;
    if (mode == 1 || mode == 2) {
        rc = a2av_launch_plan_scan(pl, s, 0, true);
        for (int i = 0; i < steps && rc == GPUMPI_OK; i++) {
            const bool next = i + 1 < steps;
            rc = a2av_launch_copy(pl, s, i & 1, next, mode == 2);
            if (rc == GPUMPI_OK && next && mode == 1) rc = a2av_launch_plan_scan(pl, s, (i + 1) & 1, false);
        }
    } else if (mode == 3) {
        hipStream_t sp;
        if (hipStreamCreateWithFlags(&sp, hipStreamNonBlocking) != hipSuccess) return GPUMPI_E_HIP;
        std::vector<hipEvent_t> ev((size_t)2 * steps + 2);
        for (hipEvent_t& e : ev) hipEventCreateWithFlags(&e, hipEventDisableTiming);
        hipEvent_t* planned = ev.data();          // [steps]: plan + scan of step i done
        hipEvent_t* copied = ev.data() + steps;   // [steps]: copy of step i done
        hipEvent_t fork = ev[(size_t)2 * steps], join = ev.back();
        hipEventRecord(fork, s);
        hipStreamWaitEvent(sp, fork, 0);
        for (int i = 0; i < steps && rc == GPUMPI_OK; i++) {
            if (i >= 2) hipStreamWaitEvent(sp, copied[i - 2], 0);
            rc = a2av_launch_plan_scan(pl, sp, i & 1, true);
            hipEventRecord(planned[i], sp);
            hipStreamWaitEvent(s, planned[i], 0);
            if (rc == GPUMPI_OK) rc = a2av_launch_copy(pl, s, i & 1, false);
            hipEventRecord(copied[i], s);
        }
        hipEventRecord(join, sp);  // join: the last plan (already before the last copy)
        hipStreamWaitEvent(s, join, 0);
        for (hipEvent_t e : ev) hipEventDestroy(e);
        hipStreamDestroy(sp);
    } else {
        for (int i = 0; i < steps && rc == GPUMPI_OK; i++) rc = a2av_launch(pl, s, false);
    }
    return rc;
}

static void a2av_drop_graph(gpumpi_a2av_plan* pl) {
    for (A2avGraph& g : pl->graphs) {
        if (g.exec) hipGraphExecDestroy(g.exec);
        if (g.def) hipGraphDestroy(g.def);
    }
    pl->graphs.clear();
}

static int a2av_read_bytes(gpumpi_a2av_plan* pl, int64_t* bytes) {
    const A2avDev& d = pl->last_ws == 0 ? pl->dev : pl->dev2;
    if (hipMemcpy(bytes, d.total_bytes, sizeof(int64_t), hipMemcpyDeviceToHost) != hipSuccess)
        return GPUMPI_E_HIP;
    return GPUMPI_OK;
}

extern "C" {

int gpumpi_a2av_plan_create(int32_t P, int32_t elem_bytes, void* const* sendbufs,
                            const int32_t* send_counts, const int32_t* send_displs,
                            void* const* recvbufs, int32_t* recv_counts, int32_t* recv_displs,
                            const gpumpi_a2av_tune* tune, gpumpi_a2av_plan** out) {
    if (!out || P <= 0 || elem_bytes <= 0 || !sendbufs || !send_counts || !send_displs ||
        !recvbufs || !recv_counts || !recv_displs)
        return GPUMPI_E_ARG;
    gpumpi_a2av_plan* pl = new gpumpi_a2av_plan();
    int32_t cus = 0, khz = 0;
    if (gpumpi_device_info(&cus, &khz, nullptr) != GPUMPI_OK) {
        delete pl;
        return GPUMPI_E_HIP;
    }
    pl->cus = cus;
    A2avDev& d = pl->dev;
    d.P = P;
    d.elem = elem_bytes;
    d.sendbufs = (char* const*)sendbufs;
    d.scounts = send_counts;
    d.sdispls = send_displs;
    d.recvbufs = (char* const*)recvbufs;
    d.rcounts = recv_counts;
    d.rdispls = recv_displs;
    const uint64_t PP = (uint64_t)P * (uint64_t)P;
    // per workspace: seg_end, seg_src [P*P], row_bytes [P], chunk_off and short_off [P+1], total
    // bytes and chunk lines, plan-done counter (on its own 128-byte line)
    const size_t ws = sizeof(uint64_t) * (2 * PP + P + 2 * (P + 1)) + 256;
    char* w = nullptr;
    if (hipMalloc((void**)&w, 2 * ws) != hipSuccess) {
        delete pl;
        return GPUMPI_E_NOMEM;
    }
    pl->allocs.push_back(w);
    hipMemset(w, 0, 2 * ws);
    pl->dev2 = d;
    for (int k = 0; k < 2; k++) {
        A2avDev& x = k == 0 ? d : pl->dev2;
        char* b = w + k * ws;
        x.seg_end = (uint64_t*)b;
        x.seg_src = x.seg_end + PP;
        x.row_bytes = x.seg_src + PP;
        x.chunk_off = x.row_bytes + P;
        x.short_off = x.chunk_off + P + 1;
        x.total_bytes = (int64_t*)(x.short_off + P + 1);
        x.plan_done = (uint32_t*)(b + ws - 128);
    }
    for (int i = 0; i < 4; i++) hipEventCreate(&pl->ev[i]);
    gpumpi_a2av_tune t{kA2avCopyThreads, 0, 4, 1, 4, 0, 2};
    if (tune) {
        if (tune->block_threads > 0) t.block_threads = tune->block_threads;
        if (tune->blocks_per_cu >= 0) t.blocks_per_cu = tune->blocks_per_cu;
        if (tune->lines_per_lane > 0) t.lines_per_lane = tune->lines_per_lane;
        if (tune->nontemporal >= 0) t.nontemporal = tune->nontemporal;
        if (tune->chunk_rounds > 0) t.chunk_rounds = tune->chunk_rounds;
        if (tune->defer_straddle >= 0) t.defer_straddle = tune->defer_straddle;
        if (tune->pipeline >= 0) t.pipeline = tune->pipeline;
    }
    int rc = a2av_configure(pl, t);
    if (rc != GPUMPI_OK) {
        gpumpi_a2av_plan_destroy(pl);
        return rc;
    }
    hipDeviceSynchronize();
    *out = pl;
    return GPUMPI_OK;
}

void gpumpi_a2av_plan_destroy(gpumpi_a2av_plan* pl) {
    if (!pl) return;
    hipDeviceSynchronize();
    a2av_drop_graph(pl);
    for (hipEvent_t e : pl->ev)
        if (e) hipEventDestroy(e);
    for (void* p : pl->allocs) hipFree(p);
    delete pl;
}

int gpumpi_a2av_execute(gpumpi_a2av_plan* pl, void* stream) {
    if (!pl) return GPUMPI_E_ARG;
    return a2av_launch(pl, (hipStream_t)stream, pl->timing);
}

int gpumpi_a2av_graph_replay(gpumpi_a2av_plan* pl, int32_t steps, void* stream) {
    if (!pl || steps <= 0) return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    A2avGraph* g = nullptr;
    for (A2avGraph& x : pl->graphs)
        if (x.steps == steps) g = &x;
    if (!g) {
        hipStream_t cs;
        if (hipStreamCreate(&cs) != hipSuccess) return GPUMPI_E_HIP;
        if (hipStreamSynchronize(s) != hipSuccess ||
            hipStreamBeginCapture(cs, hipStreamCaptureModeRelaxed) != hipSuccess) {
            hipStreamDestroy(cs);
            return GPUMPI_E_HIP;
        }
        const int rc = a2av_launch_steps(pl, cs, steps);
        A2avGraph ng;
        ng.steps = steps;
        hipError_t ee = hipStreamEndCapture(cs, &ng.def);
        hipStreamDestroy(cs);
        if (rc != GPUMPI_OK || ee != hipSuccess) {
            if (ng.def) hipGraphDestroy(ng.def);
            return GPUMPI_E_HIP;
        }
        if (hipGraphInstantiate(&ng.exec, ng.def, nullptr, nullptr, 0) != hipSuccess) {
            hipGraphDestroy(ng.def);
            return GPUMPI_E_HIP;
        }
        pl->graphs.push_back(ng);
        g = &pl->graphs.back();
    }
    pl->last_ws = pl->tune.pipeline ? (steps - 1) & 1 : 0;
    return hipGraphLaunch(g->exec, s) == hipSuccess ? GPUMPI_OK : GPUMPI_E_HIP;
}

// Durations of the kernels of `steps` pipelined steps launched directly (not from a
// graph), with HIP events on the launch stream: us[0] = plan + scan of the first step,
// us[1] = average copy kernel (each but the last also planning the next step), us[2] =
// the whole sequence per step.
int gpumpi_a2av_pipeline_times(gpumpi_a2av_plan* pl, int32_t steps, void* stream, double* us) {
    if (!pl || steps < 2 || !us) return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    std::vector<hipEvent_t> ev((size_t)steps + 2);
    for (hipEvent_t& e : ev)
        if (hipEventCreate(&e) != hipSuccess) return GPUMPI_E_HIP;
    int rc = GPUMPI_OK;
    hipEventRecord(ev[0], s);
    rc = a2av_launch_tables(pl->dev, true, s);
    hipEventRecord(ev[1], s);
    const bool scan_in_plan = pl->tune.pipeline != 1;
    for (int i = 0; i < steps && rc == GPUMPI_OK; i++) {
        rc = a2av_launch_copy(pl, s, i & 1, i + 1 < steps, scan_in_plan);
        if (rc == GPUMPI_OK && !scan_in_plan && i + 1 < steps) rc = a2av_launch_plan_scan(pl, s, (i + 1) & 1, false);
        hipEventRecord(ev[(size_t)i + 2], s);
    }
    if (rc == GPUMPI_OK && hipEventSynchronize(ev.back()) == hipSuccess) {
        float ms = 0.f;
        hipEventElapsedTime(&ms, ev[0], ev[1]);
        us[0] = 1000.0 * ms;
        double copy = 0;
        for (int i = 0; i < steps; i++) {
            hipEventElapsedTime(&ms, ev[(size_t)i + 1], ev[(size_t)i + 2]);
            copy += 1000.0 * ms;
        }
        us[1] = copy / steps;
        hipEventElapsedTime(&ms, ev[0], ev.back());
        us[2] = 1000.0 * ms / steps;
    } else if (rc == GPUMPI_OK) {
        rc = GPUMPI_E_HIP;
    }
    for (hipEvent_t e : ev) hipEventDestroy(e);
    return rc;
}

int gpumpi_a2av_phase_times(gpumpi_a2av_plan* pl, int32_t enable, double* us) {
    if (!pl) return GPUMPI_E_ARG;
    if (enable >= 0) {
        pl->timing = enable > 0;
        return GPUMPI_OK;
    }
    if (!pl->timing || !us) return GPUMPI_E_ARG;
    if (hipEventSynchronize(pl->ev[3]) != hipSuccess) return GPUMPI_E_HIP;
    for (int i = 0; i < 3; i++) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, pl->ev[i], pl->ev[i + 1]) != hipSuccess) return GPUMPI_E_HIP;
        us[i] = 1000.0 * ms;
    }
    return GPUMPI_OK;
}

int gpumpi_a2av_get_tune(gpumpi_a2av_plan* pl, gpumpi_a2av_tune* t, int32_t* grid) {
    if (!pl) return GPUMPI_E_ARG;
    if (t) *t = pl->tune;
    if (grid) *grid = pl->grid;
    return GPUMPI_OK;
}

int gpumpi_a2av_payload_bytes(gpumpi_a2av_plan* pl, int64_t* bytes) {
    if (!pl || !bytes) return GPUMPI_E_ARG;
    return a2av_read_bytes(pl, bytes);
}

// Sweep chunk sizes, copy-grid caps and store kinds on the live buffers; every candidate
// runs the real step (so the receive buffers hold the correct exchange afterwards).  The
// first step's payload sizes the copy grid.
int gpumpi_a2av_autotune(gpumpi_a2av_plan* pl, void* stream, gpumpi_a2av_tune* chosen,
                         double* best_us) {
    if (!pl) return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    a2av_drop_graph(pl);
    if (a2av_launch(pl, s, false) != GPUMPI_OK || hipStreamSynchronize(s) != hipSuccess)
        return GPUMPI_E_HIP;
    int64_t bytes = 0;
    if (a2av_read_bytes(pl, &bytes) != GPUMPI_OK) return GPUMPI_E_HIP;
    pl->est_bytes = bytes;
    const int bpcs[] = {0, 16, 4};
    const int us_[] = {2, 4, 8};
    const int rs[] = {1, 2, 4};
    const int nts[] = {1, 0};
    const int defers[] = {0, 1};
    gpumpi_a2av_tune best = pl->tune;
    const int32_t pipeline = pl->tune.pipeline;
    double best_t = 1e30;
    hipEvent_t e0, e1;
    hipEventCreate(&e0);
    hipEventCreate(&e1);
    for (int defer : defers)
    for (int bpc : bpcs)
        for (int U : us_)
            for (int R : rs)
            for (int nt : nts) {
                gpumpi_a2av_tune t{kA2avCopyThreads, bpc, U, nt, R, defer, pipeline};
                if (a2av_configure(pl, t) != GPUMPI_OK) continue;
                a2av_launch(pl, s, false);  // warm-up
                const int reps = 5;
                hipEventRecord(e0, s);
                for (int r = 0; r < reps; r++) a2av_launch(pl, s, false);
                hipEventRecord(e1, s);
                hipEventSynchronize(e1);
                float ms = 0.f;
                hipEventElapsedTime(&ms, e0, e1);
                const double t_us = 1000.0 * ms / reps;
                if (t_us < best_t) {
                    best_t = t_us;
                    best = pl->tune;
                }
            }
    // then the pipeline mode, on the graph replays it applies to: 10-step graphs, the
    // best of three replays per mode
    int rc = a2av_configure(pl, best);
    double best_step = 1e30;
    int best_mode = best.pipeline;
    for (int mode = 0; mode <= 3 && rc == GPUMPI_OK; mode++) {
        gpumpi_a2av_tune t = best;
        t.pipeline = mode;
        a2av_drop_graph(pl);
        if (a2av_configure(pl, t) != GPUMPI_OK) continue;
        if (gpumpi_a2av_graph_replay(pl, 10, s) != GPUMPI_OK) break;  // capture + warm-up
        double mode_best = 1e30;
        for (int r = 0; r < 3; r++) {
            hipEventRecord(e0, s);
            gpumpi_a2av_graph_replay(pl, 10, s);
            hipEventRecord(e1, s);
            hipEventSynchronize(e1);
            float ms = 0.f;
            hipEventElapsedTime(&ms, e0, e1);
            mode_best = std::min(mode_best, 1000.0 * ms / 10);
        }
        if (mode_best < best_step) {
            best_step = mode_best;
            best_mode = mode;
        }
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    a2av_drop_graph(pl);
    best.pipeline = best_mode;
    rc = a2av_configure(pl, best);
    if (chosen) *chosen = pl->tune;
    if (best_us) *best_us = best_step < 1e30 ? best_step : best_t;
    return rc;
}

}  // extern "C"

// ==================================================================== batched point-to-point step
static_assert(sizeof(gpumpi_p2p_pair) == sizeof(P2pPair) && offsetof(gpumpi_p2p_pair, bytes) == offsetof(P2pPair, bytes),
              "gpumpi_p2p_pair and the device's P2pPair differ");

struct gpumpi_p2p_plan {
    int64_t max_pairs = 0;
    uint64_t* chunk_off = nullptr;  // [max_pairs], then the tiles' chunks [kP2pTiles]
    int32_t cus = 0;
    hipGraphExec_t graph = nullptr;
    hipGraph_t graph_def = nullptr;
    int graph_steps = 0;
    const void* graph_pairs = nullptr;
    int64_t graph_n = -1;
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
};

// The step's kernel on stream s, or two past kP2pFused pairs (no allocation, no host
// synchronisation: capturable).
static int p2p_launch(gpumpi_p2p_plan* pl, const P2pPair* pairs, int64_t n, hipStream_t s, bool timed) {
    if (timed) hipEventRecord(pl->ev[0], s);
    uint64_t* tile_chunks = pl->chunk_off + pl->max_pairs;
    int shift = 12;    // pairs per tile: kP2pPass, or as many as leave kP2pTiles tiles
    static_assert(1 << 12 == kP2pPass, "a tile is whole passes");
    while ((n - 1) >> shift >= kP2pTiles) shift++;
    if (n > kP2pFused)
        p2p_scan_kernel<<<dim3((unsigned)(((n - 1) >> shift) + 1)), dim3(kP2pScanThreads), 0, s>>>(pairs, n, shift,
                                                                                                pl->chunk_off, tile_chunks);
    if (timed) hipEventRecord(pl->ev[1], s);
    // short lists: many small workgroups, each with a scan of its own (64 pairs of 16 MiB: 420
    // us, one workgroup of 16 waves per CU 436); longer ones: one scan per CU (3072 pairs of
    // 5 KiB: 9.8, small workgroups 14 to 36); lists with a scan kernel: what is resident at
    // once (65536 pairs of 4 KiB: 127 us, one large workgroup per CU 138).  Compared on one set of
    // buffers with non-temporal stores; what the steps take now stands in batched_p2p.h.
    const unsigned cus = (unsigned)pl->cus;
    if (n <= kP2pShort)
        p2p_copy_kernel<kP2pShort, 256, 5><<<dim3(16 * cus), dim3(256), 0, s>>>(pairs, n, shift, pl->chunk_off, tile_chunks);
    else if (n <= kP2pFused)
        p2p_copy_kernel<kP2pFused, 1024, 4><<<dim3(cus), dim3(1024), 0, s>>>(pairs, n, shift, pl->chunk_off, tile_chunks);
    else
        p2p_copy_kernel<0, 256, 5><<<dim3(5 * cus), dim3(256), 0, s>>>(pairs, n, shift, pl->chunk_off, tile_chunks);
    if (timed) hipEventRecord(pl->ev[2], s);
    return hipGetLastError() == hipSuccess ? GPUMPI_OK : GPUMPI_E_HIP;
}

static void p2p_drop_graph(gpumpi_p2p_plan* pl) {
    if (pl->graph) hipGraphExecDestroy(pl->graph);
    if (pl->graph_def) hipGraphDestroy(pl->graph_def);
    pl->graph = nullptr;
    pl->graph_def = nullptr;
    pl->graph_steps = 0;
}

static int p2p_create(int64_t max_pairs, gpumpi_p2p_plan** out) {
    if (!out || max_pairs < 1 || max_pairs > (int64_t(1) << 32)) return GPUMPI_E_ARG;
    int32_t cus = 0;
    if (gpumpi_device_info(&cus, nullptr, nullptr) != GPUMPI_OK || cus <= 0) return GPUMPI_E_HIP;
    gpumpi_p2p_plan* pl = new gpumpi_p2p_plan();
    pl->max_pairs = max_pairs;
    pl->cus = cus;
    if (hipMalloc((void**)&pl->chunk_off, sizeof(uint64_t) * (size_t)(max_pairs + kP2pTiles)) != hipSuccess) {
        delete pl;
        return GPUMPI_E_NOMEM;
    }
    for (hipEvent_t& e : pl->ev) hipEventCreate(&e);
    *out = pl;
    return GPUMPI_OK;
}

static void p2p_destroy(gpumpi_p2p_plan* pl) {
    if (!pl) return;
    hipDeviceSynchronize();
    p2p_drop_graph(pl);
    for (hipEvent_t e : pl->ev)
        if (e) hipEventDestroy(e);
    hipFree(pl->chunk_off);
    delete pl;
}

extern "C" {

int gpumpi_p2p_plan_create(int64_t max_pairs, gpumpi_p2p_plan** out) { return p2p_create(max_pairs, out); }

void gpumpi_p2p_plan_destroy(gpumpi_p2p_plan* pl) { p2p_destroy(pl); }

int gpumpi_p2p_execute(gpumpi_p2p_plan* pl, const gpumpi_p2p_pair* pairs, int64_t npairs, void* stream) {
    if (!pl || npairs < 0 || npairs > pl->max_pairs || (npairs > 0 && !pairs)) return GPUMPI_E_ARG;
    if (npairs == 0) return GPUMPI_OK;
    return p2p_launch(pl, (const P2pPair*)pairs, npairs, (hipStream_t)stream, false);
}

int gpumpi_p2p_graph_replay(gpumpi_p2p_plan* pl, const gpumpi_p2p_pair* pairs, int64_t npairs,
                            int32_t steps, void* stream) {
    if (!pl || !pairs || npairs < 1 || npairs > pl->max_pairs || steps < 1) return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    if (!pl->graph || pl->graph_steps != steps || pl->graph_pairs != (const void*)pairs || pl->graph_n != npairs) {
        p2p_drop_graph(pl);
        hipStream_t cs;
        if (hipStreamCreate(&cs) != hipSuccess) return GPUMPI_E_HIP;
        if (hipStreamSynchronize(s) != hipSuccess ||
            hipStreamBeginCapture(cs, hipStreamCaptureModeRelaxed) != hipSuccess) {
            hipStreamDestroy(cs);
            return GPUMPI_E_HIP;
        }
        int rc = GPUMPI_OK;
        for (int i = 0; i < steps && rc == GPUMPI_OK; i++) rc = p2p_launch(pl, (const P2pPair*)pairs, npairs, cs, false);
        hipGraph_t g = nullptr;
        hipError_t ee = hipStreamEndCapture(cs, &g);
        hipStreamDestroy(cs);
        if (rc != GPUMPI_OK || ee != hipSuccess) {
            if (g) hipGraphDestroy(g);
            return GPUMPI_E_HIP;
        }
        pl->graph_def = g;
        if (hipGraphInstantiate(&pl->graph, g, nullptr, nullptr, 0) != hipSuccess) {
            p2p_drop_graph(pl);
            return GPUMPI_E_HIP;
        }
        pl->graph_steps = steps;
        pl->graph_pairs = pairs;
        pl->graph_n = npairs;
    }
    return hipGraphLaunch(pl->graph, s) == hipSuccess ? GPUMPI_OK : GPUMPI_E_HIP;
}

int gpumpi_p2p_kernel_times(gpumpi_p2p_plan* pl, const gpumpi_p2p_pair* pairs, int64_t npairs, int32_t reps,
                            void* stream, double* us) {
    if (!pl || !pairs || !us || npairs < 1 || npairs > pl->max_pairs || reps < 1) return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    us[0] = us[1] = 0.0;
    for (int i = 0; i < reps; i++) {
        if (p2p_launch(pl, (const P2pPair*)pairs, npairs, s, true) != GPUMPI_OK) return GPUMPI_E_HIP;
        if (hipEventSynchronize(pl->ev[2]) != hipSuccess) return GPUMPI_E_HIP;
        float a = 0.f, b = 0.f;
        hipEventElapsedTime(&a, pl->ev[0], pl->ev[1]);
        hipEventElapsedTime(&b, pl->ev[1], pl->ev[2]);
        us[0] += 1000.0 * a / reps;
        us[1] += 1000.0 * b / reps;
    }
    return GPUMPI_OK;
}

}  // extern "C"

// ==================================================================== batched particle step
struct gpumpi_particle_plan {
    PartStepDev dev{};
    uint8_t* dirs[2] = {nullptr, nullptr};  // direction bytes of the current / next state
    int cur = 0;
    int nontemporal = 1;
    std::vector<void*> allocs;
    hipGraphExec_t graph = nullptr;
    hipGraph_t graph_def = nullptr;
    int graph_steps = 0;
    const void* graph_key[4] = {nullptr, nullptr, nullptr, nullptr};
    int graph_cur = -1;       // direction buffer the captured steps start from
    bool timing = false;
    hipEvent_t ev[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    int32_t exchange = 0;           // 0: the scatter writes final slots; 1: batched p2p messages
    gpumpi_p2p_plan* p2p = nullptr; // exchange 1
};

static int ps_launch(gpumpi_particle_plan* pl, const double* in, const int64_t* cin, double* out,
                     int64_t* cout, hipStream_t s, bool timed) {
    PartStepDev& d = pl->dev;
    d.in = in;
    d.cin = cin;
    d.dir_in = pl->dirs[pl->cur];
    d.out = out;
    d.cout = cout;
    d.dir_out = pl->dirs[pl->cur ^ 1];
    const int64_t waves = (int64_t)d.P * d.nchunks;
    const dim3 chunk_grid((unsigned)((waves + 3) / 4)), rank_grid((unsigned)d.P),
        place_grid((unsigned)((d.P + kPsThreads - 1) / kPsThreads)), block(kPsThreads);
    void* kargs[] = {(void*)&d};
    const bool p2p = pl->exchange == 1;
    const void* scatter = p2p ? (pl->nontemporal ? (const void*)&ps_scatter_kernel<true, true>
                                                 : (const void*)&ps_scatter_kernel<false, true>)
                              : (pl->nontemporal ? (const void*)&ps_scatter_kernel<true, false>
                                                 : (const void*)&ps_scatter_kernel<false, false>);
    const void* place = p2p ? (const void*)&ps_place_kernel<true> : (const void*)&ps_place_kernel<false>;
    const void* kernels[3] = {(const void*)&ps_tally_kernel, place, scatter};
    const dim3 grids[3] = {rank_grid, place_grid, chunk_grid};
    const dim3 blocks[3] = {dim3(kPsTallyThreads), block, block};
    for (int i = 0; i < 3; i++) {
        if (timed) hipEventRecord(pl->ev[i], s);
        if (hipLaunchKernel(kernels[i], grids[i], blocks[i], kargs, 0, s) != hipSuccess)
            return GPUMPI_E_HIP;
    }
    if (timed) hipEventRecord(pl->ev[3], s);
    if (p2p && p2p_launch(pl->p2p, d.pairs, (int64_t)d.P * 6, s, false) != GPUMPI_OK) return GPUMPI_E_HIP;
    if (timed) hipEventRecord(pl->ev[4], s);
    pl->cur ^= 1;
    return GPUMPI_OK;
}

static void ps_drop_graph(gpumpi_particle_plan* pl) {
    if (pl->graph) hipGraphExecDestroy(pl->graph);
    if (pl->graph_def) hipGraphDestroy(pl->graph_def);
    pl->graph = nullptr;
    pl->graph_def = nullptr;
    pl->graph_steps = 0;
}

extern "C" {

int gpumpi_particles_plan_create(int32_t gx, int32_t gy, int32_t gz, int64_t cap, uint64_t seed,
                                 int32_t nontemporal, gpumpi_particle_plan** out) {
    if (!out || gx < 1 || gy < 1 || gz < 1 || cap < 1 || cap > 0x7FFFFFFF) return GPUMPI_E_ARG;
    const int64_t P64 = (int64_t)gx * gy * gz;
    if (P64 > (1 << 20)) return GPUMPI_E_ARG;
    const int P = (int)P64;
    const int64_t nchunks = (cap + kPsChunk - 1) / kPsChunk;
    if ((P64 * nchunks + 3) / 4 > 0x7FFFFFFF || (double)P64 * (double)cap > 1e12) return GPUMPI_E_ARG;
    gpumpi_particle_plan* pl = new gpumpi_particle_plan();
    pl->nontemporal = nontemporal != 0;
    PartStepDev& d = pl->dev;
    d.gx = gx;
    d.gy = gy;
    d.gz = gz;
    d.P = P;
    d.cap = cap;
    d.seed = seed;
    d.nchunks = (int32_t)nchunks;
    // host tables: neighbours and direction classes of every rank
    std::vector<int32_t> nbr((size_t)P * kPsClasses, 0);
    std::vector<uint32_t> cls((size_t)P);
    for (int r = 0; r < P; r++) {
        for (int dd = 0; dd < 6; dd++) nbr[(size_t)r * kPsClasses + dd] = grid_neighbour(r, dd, gx, gy, gz);
        nbr[(size_t)r * kPsClasses + 6] = r;
        nbr[(size_t)r * kPsClasses + 7] = r;
        cls[r] = ps_classes(r, gx, gy, gz);
    }
    const size_t b_dirs = (size_t)P * (size_t)cap + 256, b_chunk = sizeof(int32_t) * (size_t)P * nchunks * kPsClasses,
                 b_rank = sizeof(int64_t) * (size_t)P * kPsClasses, b_nbr = nbr.size() * sizeof(int32_t),
                 b_cls = cls.size() * sizeof(uint32_t);
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t ws = 2 * al(b_dirs) + al(b_chunk) + 2 * al(b_rank) + al(b_nbr) + al(b_cls) + 256;
    char* w = nullptr;
    if (hipMalloc((void**)&w, ws) != hipSuccess) {
        delete pl;
        return GPUMPI_E_NOMEM;
    }
    pl->allocs.push_back(w);
    hipMemset(w, 0, ws);
    char* q = w;
    pl->dirs[0] = (uint8_t*)q; q += al(b_dirs);
    pl->dirs[1] = (uint8_t*)q; q += al(b_dirs);
    d.chunk_off = (int32_t*)q; q += al(b_chunk);
    d.tot = (int64_t*)q; q += al(b_rank);
    d.base = (int64_t*)q; q += al(b_rank);
    d.nbr_tab = (const int32_t*)q;
    hipMemcpy(q, nbr.data(), b_nbr, hipMemcpyHostToDevice); q += al(b_nbr);
    d.cls_tab = (const uint32_t*)q;
    hipMemcpy(q, cls.data(), b_cls, hipMemcpyHostToDevice); q += al(b_cls);
    d.stats = (int64_t*)q;
    d.step = (uint32_t*)(q + 4 * sizeof(int64_t));
    for (int i = 0; i < 5; i++) hipEventCreate(&pl->ev[i]);
    if (hipDeviceSynchronize() != hipSuccess) {
        gpumpi_particles_plan_destroy(pl);
        return GPUMPI_E_HIP;
    }
    *out = pl;
    return GPUMPI_OK;
}

void gpumpi_particles_plan_destroy(gpumpi_particle_plan* pl) {
    if (!pl) return;
    hipDeviceSynchronize();
    ps_drop_graph(pl);
    for (hipEvent_t e : pl->ev)
        if (e) hipEventDestroy(e);
    for (void* p : pl->allocs) hipFree(p);
    p2p_destroy(pl->p2p);
    delete pl;
}

int gpumpi_particles_exchange_mode(gpumpi_particle_plan* pl, int32_t mode) {
    if (!pl || mode < 0 || mode > 1) return GPUMPI_E_ARG;
    if (mode == 1 && !pl->p2p) {
        PartStepDev& d = pl->dev;
        const size_t b_send = sizeof(double) * kPartFields * (size_t)d.P * (size_t)d.cap;
        const size_t b_pairs = ((sizeof(P2pPair) * (size_t)d.P * 6) + 255) & ~(size_t)255;
        char* w = nullptr;
        if (hipMalloc((void**)&w, b_send + b_pairs) != hipSuccess) return GPUMPI_E_NOMEM;
        pl->allocs.push_back(w);
        gpumpi_p2p_plan* q = nullptr;
        const int rc = p2p_create((int64_t)d.P * 6, &q);
        if (rc != GPUMPI_OK) return rc;
        pl->p2p = q;
        d.pairs = (P2pPair*)w;
        d.send = (double*)(w + b_pairs);
    }
    if (pl->exchange != mode) {
        hipDeviceSynchronize();
        ps_drop_graph(pl);
        pl->exchange = mode;
    }
    return GPUMPI_OK;
}

int gpumpi_particles_init(gpumpi_particle_plan* pl, double* parts, int64_t* counts, int64_t n0,
                          void* stream) {
    if (!pl || !parts || !counts || n0 < 0 || n0 > pl->dev.cap) return GPUMPI_E_ARG;
    const PartStepDev& d = pl->dev;
    const int64_t threads = std::max<int64_t>((int64_t)d.P * n0, d.P);
    ps_init_kernel<<<dim3((unsigned)((threads + kPsThreads - 1) / kPsThreads)), dim3(kPsThreads), 0,
                     (hipStream_t)stream>>>(d.gx, d.gy, d.gz, d.cap, n0, d.seed, parts, counts);
    return hipGetLastError() == hipSuccess ? GPUMPI_OK : GPUMPI_E_HIP;
}

int gpumpi_particles_prepare(gpumpi_particle_plan* pl, const double* parts, const int64_t* counts,
                             uint32_t step, void* stream) {
    if (!pl || !parts || !counts) return GPUMPI_E_ARG;
    PartStepDev d = pl->dev;
    d.in = parts;
    d.cin = counts;
    d.dir_out = pl->dirs[pl->cur];
    const int64_t slots = (int64_t)d.P * d.cap;
    ps_dirs_kernel<<<dim3((unsigned)((slots + kPsThreads - 1) / kPsThreads)), dim3(kPsThreads), 0,
                     (hipStream_t)stream>>>(d, step);
    return hipGetLastError() == hipSuccess ? GPUMPI_OK : GPUMPI_E_HIP;
}

int gpumpi_particles_step(gpumpi_particle_plan* pl, const double* in, const int64_t* cin,
                          double* out, int64_t* cout, void* stream) {
    if (!pl || !in || !cin || !out || !cout || (const void*)in == (const void*)out) return GPUMPI_E_ARG;
    return ps_launch(pl, in, cin, out, cout, (hipStream_t)stream, pl->timing);
}

int gpumpi_particles_graph_replay(gpumpi_particle_plan* pl, double* a, int64_t* ca, double* b,
                                  int64_t* cb, int32_t steps, void* stream) {
    if (!pl || !a || !ca || !b || !cb || a == b || steps <= 0 || (steps & 1)) return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const void* key[4] = {a, ca, b, cb};
    if (!pl->graph || pl->graph_steps != steps || pl->graph_cur != pl->cur ||
        std::memcmp(key, pl->graph_key, sizeof(key)) != 0) {
        ps_drop_graph(pl);
        const int cur0 = pl->cur;
        hipStream_t cs;
        if (hipStreamCreate(&cs) != hipSuccess) return GPUMPI_E_HIP;
        if (hipStreamSynchronize(s) != hipSuccess ||
            hipStreamBeginCapture(cs, hipStreamCaptureModeRelaxed) != hipSuccess) {
            hipStreamDestroy(cs);
            return GPUMPI_E_HIP;
        }
        int rc = GPUMPI_OK;
        for (int i = 0; i < steps && rc == GPUMPI_OK; i++)
            rc = (i & 1) ? ps_launch(pl, b, cb, a, ca, cs, false) : ps_launch(pl, a, ca, b, cb, cs, false);
        hipGraph_t g = nullptr;
        hipError_t ee = hipStreamEndCapture(cs, &g);
        hipStreamDestroy(cs);
        if (rc != GPUMPI_OK || ee != hipSuccess) {
            if (g) hipGraphDestroy(g);
            return GPUMPI_E_HIP;
        }
        pl->graph_def = g;
        if (hipGraphInstantiate(&pl->graph, g, nullptr, nullptr, 0) != hipSuccess) {
            ps_drop_graph(pl);
            return GPUMPI_E_HIP;
        }
        pl->graph_steps = steps;
        pl->graph_cur = cur0;
        std::memcpy(pl->graph_key, key, sizeof(key));
    }
    return hipGraphLaunch(pl->graph, s) == hipSuccess ? GPUMPI_OK : GPUMPI_E_HIP;
}

int gpumpi_particles_status(gpumpi_particle_plan* pl, int64_t* moved, int32_t* overflow,
                            uint32_t* next_step) {
    if (!pl) return GPUMPI_E_ARG;
    if (hipDeviceSynchronize() != hipSuccess) return GPUMPI_E_HIP;
    int64_t st[4];
    uint32_t step = 0;
    if (hipMemcpy(st, pl->dev.stats, sizeof(st), hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(&step, pl->dev.step, sizeof(step), hipMemcpyDeviceToHost) != hipSuccess)
        return GPUMPI_E_HIP;
    if (moved) *moved = st[0];
    if (overflow) *overflow = (int32_t)st[2];
    if (next_step) *next_step = step;
    return GPUMPI_OK;
}

int gpumpi_particles_phase_times(gpumpi_particle_plan* pl, int32_t enable, double* us) {
    if (!pl) return GPUMPI_E_ARG;
    if (enable >= 0) {
        pl->timing = enable > 0;
        return GPUMPI_OK;
    }
    if (!pl->timing || !us) return GPUMPI_E_ARG;
    if (hipEventSynchronize(pl->ev[4]) != hipSuccess) return GPUMPI_E_HIP;
    for (int i = 0; i < 4; i++) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, pl->ev[i], pl->ev[i + 1]) != hipSuccess) return GPUMPI_E_HIP;
        us[i] = 1000.0 * ms;
    }
    return GPUMPI_OK;
}

}  // extern "C"

// ==================================================================== workspaces
// Device memory of gpumpi_bucket_plan and gpumpi_local_sort (workspace.h).  A block has one
// user from the constructor to the destructor, and the call has waited for its stream by then,
// so any thread or stream of the same device may take it next; after a wait that failed it is
// freed instead.
namespace {
struct HipMemory {
    static bool device(int* dev) { return hipGetDevice(dev) == hipSuccess; }
    static void* alloc(size_t bytes) {
        void* p = nullptr;
        if (hipMalloc(&p, bytes) == hipSuccess) return p;
        (void)hipGetLastError();
        return nullptr;
    }
    static bool free(void* p) { return hipFree(p) == hipSuccess; }
};
using Pool = WorkspacePool<HipMemory>;

struct Workspace {
    static Pool& pool() {
        static Pool* p = new Pool();   // outlives every static that may still call the library
        return *p;
    }
    Pool::Block block;
    void* ptr;

    explicit Workspace(size_t need) : block(pool().take(need)), ptr(block.ptr) {}
    void take(size_t need) {       // again, after a failure
        block = pool().take(need);
        ptr = block.ptr;
    }
    // Waits for the call's stream; `ok`: its launches were accepted.
    int finish(hipStream_t s, bool ok) {
        if (hipStreamSynchronize(s) == hipSuccess) return ok ? GPUMPI_OK : GPUMPI_E_HIP;
        HipMemory::free(block.ptr);
        block.ptr = nullptr;
        return GPUMPI_E_HIP;
    }
    ~Workspace() { pool().give(block); }
    Workspace(const Workspace&) = delete;
    Workspace& operator=(const Workspace&) = delete;
};
}  // namespace

extern "C" int gpumpi_workspace_trim(void) { return Workspace::pool().trim() ? GPUMPI_OK : GPUMPI_E_HIP; }

// ==================================================================== bucket-sort caller
extern "C" {

int gpumpi_gen_keys(uint32_t* keys, int32_t P, int64_t n, uint64_t seed, uint32_t step,
                    int32_t dist, int32_t key_bits, const double* cdf, int64_t ncdf, void* stream) {
    if (!keys || P <= 0 || n < 0 || key_bits < 1 || key_bits > 31 || dist < 0 || dist > 2 ||
        (dist == 1 && (!cdf || ncdf <= 0)))
        return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    int64_t total = (int64_t)P * n;
    int blocks = (int)((total + 255) / 256);
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(gen_keys_kernel, dim3(blocks), dim3(256), 0, s, keys, P, n, seed, step,
                       dist, key_bits, cdf, ncdf);
    return hipGetLastError() == hipSuccess ? GPUMPI_OK : GPUMPI_E_HIP;
}

int gpumpi_bucket_plan(const uint32_t* keys, int32_t P, int64_t n, int32_t key_bits,
                       int32_t bucket_bits, uint32_t* key_buff1, int32_t* send_counts,
                       int32_t* send_displs, int32_t* bucket_lo, int32_t* bucket_hi,
                       void* stream) {
    if (!keys || P <= 0 || n <= 0 || bucket_bits < 1 || bucket_bits > 12 ||
        bucket_bits > key_bits || !key_buff1 || !send_counts || !send_displs || !bucket_lo ||
        !bucket_hi)
        return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const int nb = 1 << bucket_bits;
    const int shift = key_bits - bucket_bits;
    BucketTiling t = bucket_tiling(P, n, nb, false);
    Workspace ws(bucket_scratch_bytes(t, P, nb));
    if (!ws.ptr && t.tiles > 1) {
        t = bucket_tiling(P, n, nb, true);
        ws.take(bucket_scratch_bytes(t, P, nb));
    }
    if (!ws.ptr) return GPUMPI_E_NOMEM;
    if (((int64_t)P * t.tiles + 7) / 8 * 8 > INT32_MAX) return GPUMPI_E_ARG;
    bucket_plan_launch(t, keys, P, n, shift, nb, ws.ptr, key_buff1, send_counts, send_displs, bucket_lo, bucket_hi, s);
    return ws.finish(s, hipGetLastError() == hipSuccess);
}

}  // extern "C"

// ==================================================================== served jobs
struct gpumpi_server {
    gpumpi_runtime* rt = nullptr;
    progs::ServeShared sh{};
    progs::ServeShared* d_sh = nullptr;
    std::vector<void*> dev_allocs;
    std::vector<void*> host_allocs;
    hipStream_t stream = nullptr;
    uint64_t submitted = 0;
    uint64_t polled = 0;
    int32_t qcap = 0;
    bool running = false;
};

extern "C" {

int gpumpi_serve_start(const gpumpi_config* cfg, int32_t queue_capacity, int32_t max_job_ranks,
                       double heap_fraction, gpumpi_server** out) {
    if (!cfg || !out || queue_capacity < 1 || max_job_ranks < 1 || cfg->num_ranks < 2 ||
        heap_fraction <= 0 || heap_fraction > 1)
        return GPUMPI_E_ARG;
    *out = nullptr;
    gpumpi_server* sv = new gpumpi_server();
    int rc = gpumpi_runtime_create(cfg, &sv->rt);
    if (rc != GPUMPI_OK) {
        delete sv;
        return rc;
    }
    const int S = cfg->num_ranks;
    const int jcap = S;  // at most one job per worker slot
    sv->qcap = queue_capacity;
    auto halloc = [&](void** p, size_t b) {
        if (hipHostMalloc(p, b, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) return false;
        std::memset(*p, 0, b);
        sv->host_allocs.push_back(*p);
        return true;
    };
    auto dalloc = [&](void** p, size_t b) {
        if (hipMalloc(p, b) != hipSuccess) return false;
        sv->dev_allocs.push_back(*p);
        return hipMemset(*p, 0, b) == hipSuccess;
    };
    progs::ServeShared& h = sv->sh;
    bool ok = halloc((void**)&h.q, sizeof(progs::JobDesc) * queue_capacity) &&
              halloc((void**)&h.q_tail, 64) &&
              halloc((void**)&h.done, sizeof(progs::JobResult) * queue_capacity) &&
              halloc((void**)&h.done_count, 64) && halloc((void**)&h.admit_head, 64) &&
              halloc((void**)&h.stop, 64) &&
              halloc((void**)&h.heartbeat, 64) &&
              dalloc((void**)&h.dq, sizeof(progs::JobDesc) * queue_capacity) &&
              dalloc((void**)&h.boxes, sizeof(progs::SlotBox) * S) &&
              dalloc((void**)&h.jobs, sizeof(progs::JobSlot) * jcap) &&
              dalloc((void**)&h.free_slots, sizeof(int32_t) * S) &&
              dalloc((void**)&h.free_jobs, sizeof(int32_t) * jcap) &&
              dalloc((void**)&h.slot_lists, sizeof(int32_t) * (size_t)jcap * max_job_ranks) &&
              dalloc((void**)&h.exit_flag, 64) && dalloc((void**)&h.stats, 64) &&
              dalloc((void**)&sv->d_sh, sizeof(progs::ServeShared));
    if (!ok) {
        gpumpi_serve_stop(sv, nullptr);
        return GPUMPI_E_NOMEM;
    }
    h.qcap = queue_capacity;
    h.jcap = jcap;
    h.max_ranks = max_job_ranks;
    h.lookahead = 16;
    // the job heap: ntop blocks of 2^(16 + top) bytes, top chosen so that a quarter of the
    // budget fits in one block
    {
        const uint64_t budget = (uint64_t)((double)cfg->heap_bytes * heap_fraction);
        int top = 0;
        while (top < progs::kBuddyOrders - 1 && ((uint64_t)1 << (progs::kBuddyMinShift + top)) < budget / 4) top++;
        uint64_t ntop = budget >> (progs::kBuddyMinShift + top);
        if (ntop < 1) ntop = 1;
        progs::Buddy& b = h.jobheap;
        b.top = top;
        b.ntop = (int32_t)ntop;
        uint64_t words = 0;
        for (int o = 0; o <= top; o++) {
            b.off[o] = words;
            words += (((uint64_t)ntop << (top - o)) + 63) / 64;
        }
        const uint64_t region = ntop << (progs::kBuddyMinShift + top);
        ok = dalloc((void**)&b.base, region) && dalloc((void**)&b.bits, 8 * words) &&
             dalloc((void**)&b.order_of, (size_t)ntop << top);
        if (ok) {
            std::vector<uint64_t> topbits((ntop + 63) / 64, 0);
            for (uint64_t i = 0; i < ntop; i++) topbits[i >> 6] |= 1ull << (i & 63);
            ok = hipMemcpy(b.bits + b.off[top], topbits.data(), 8 * topbits.size(),
                           hipMemcpyHostToDevice) == hipSuccess;
        }
        h.heap_budget = (int64_t)1 << (progs::kBuddyMinShift + top);
    }
    if (!ok) {
        gpumpi_serve_stop(sv, nullptr);
        return GPUMPI_E_NOMEM;
    }
    {
        int32_t khz = 0;
        gpumpi_device_info(nullptr, &khz, nullptr);
        const double idle_s = cfg->timeout_s > 0 ? cfg->timeout_s : 20.0;
        h.idle_ticks = (uint64_t)(idle_s * (double)khz * 1000.0);
    }
    if (hipMemcpy(sv->d_sh, &h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess ||
        hipStreamCreate(&sv->stream) != hipSuccess) {
        gpumpi_serve_stop(sv, nullptr);
        return GPUMPI_E_HIP;
    }
    progs::ServeArgs a{sv->d_sh};
    rc = gpumpi_run_async(sv->rt, "serve", &a, sizeof(a), sv->stream);
    if (rc != GPUMPI_OK) {
        gpumpi_serve_stop(sv, nullptr);
        return rc;
    }
    sv->running = true;
    *out = sv;
    return GPUMPI_OK;
}

// Two rings of qcap entries carry a job: the submission ring (host ring q, copied into the
// device's dq) and the completion ring done.  Job i may take position i % qcap only when
// job i - qcap no longer needs either: the scheduler has admitted or rejected it (its
// admission head is past it, so dq no longer holds a waiting job there), and this host
// has polled its result (so done[] holds no unread result there).  The head, not the
// completion count, bounds the first ring, since backfilled jobs can complete while the
// job at the head still waits.
int gpumpi_serve_submit(gpumpi_server* sv, const gpumpi_job* job) {
    if (!sv || !job || !sv->running) return GPUMPI_E_ARG;
    const uint64_t head = __atomic_load_n(sv->sh.admit_head, __ATOMIC_ACQUIRE);
    if (sv->submitted - head >= (uint64_t)sv->qcap || sv->submitted - sv->polled >= (uint64_t)sv->qcap)
        return GPUMPI_E_NOMEM;  // ring full: poll, or wait for admissions
    progs::JobDesc d{job->id, job->seed, job->type, job->ranks, job->size};
    sv->sh.q[sv->submitted % (uint64_t)sv->qcap] = d;
    sv->submitted++;
    __atomic_store_n(sv->sh.q_tail, sv->submitted, __ATOMIC_RELEASE);
    __atomic_fetch_add(sv->sh.heartbeat, 1, __ATOMIC_RELEASE);
    return GPUMPI_OK;
}

int gpumpi_serve_poll(gpumpi_server* sv, gpumpi_job_result* out, int32_t max) {
    if (!sv || (!out && max > 0)) return GPUMPI_E_ARG;
    if (sv->running) __atomic_fetch_add(sv->sh.heartbeat, 1, __ATOMIC_RELEASE);
    const uint64_t done = __atomic_load_n(sv->sh.done_count, __ATOMIC_ACQUIRE);
    int n = 0;
    while (sv->polled < done && n < max) {
        const progs::JobResult& r = sv->sh.done[sv->polled % (uint64_t)sv->qcap];
        gpumpi_job_result& o = out[n++];
        o.id = r.id;
        o.status = r.status;
        o.ranks = r.ranks;
        o.dot = r.dot;
        o.checksum = r.checksum;
        o.t_admit_ticks = r.t_admit;
        o.t_done_ticks = r.t_done;
        o.bytes = r.bytes;
        sv->polled++;
    }
    return n;
}

int gpumpi_serve_stop(gpumpi_server* sv, int64_t* stats) {
    if (!sv) return GPUMPI_E_ARG;
    int rc = GPUMPI_OK;
    if (sv->running) {
        __atomic_store_n(sv->sh.stop, 1, __ATOMIC_RELEASE);
        if (hipStreamSynchronize(sv->stream) != hipSuccess) rc = GPUMPI_E_HIP;
        if (stats && sv->sh.stats)
            hipMemcpy(stats, sv->sh.stats, sizeof(int64_t) * 4, hipMemcpyDeviceToHost);
        Runtime hr;
        if (hipMemcpy(&hr, sv->rt->d_rt, sizeof(Runtime), hipMemcpyDeviceToHost) == hipSuccess &&
            hr.abort_flag) {
            char msg[160];
            std::snprintf(msg, sizeof(msg), "device error %d on rank %d (line %d): %s", hr.err.code,
                          hr.err.rank, hr.err.line, hr.err.msg);
            g_host_error = msg;
            rc = GPUMPI_E_DEVICE;
        }
    }
    if (sv->stream) {
        hipStreamSynchronize(sv->stream);
        hipStreamDestroy(sv->stream);
    }
    for (void* p : sv->dev_allocs) hipFree(p);
    for (void* p : sv->host_allocs) hipHostFree(p);
    if (sv->rt) gpumpi_runtime_destroy(sv->rt);
    delete sv;
    return rc;
}

// Plain mode: one rank-grid launch of `job.ranks` ranks for one job (asynchronous).
int gpumpi_run_job(gpumpi_runtime* rt, const gpumpi_job* job, gpumpi_job_result* dev_result,
                   void* stream) {
    if (!rt || !job || !dev_result || job->ranks < 1 || job->ranks > rt->cfg.num_ranks)
        return GPUMPI_E_ARG;
    hipStream_t s = stream ? (hipStream_t)stream : rt->own_stream;
    hipLaunchKernelGGL(resize_world_kernel, dim3(4), dim3(256), 0, s, rt->d_rt, job->ranks);
    hipLaunchKernelGGL(heap_reset_kernel, dim3(4), dim3(256), 0, s, rt->d_rt, rt->cfg.num_ranks);
    rt->world_size = job->ranks;
    progs::JobArgs a;
    a.job = progs::JobDesc{job->id, job->seed, job->type, job->ranks, job->size};
    a.out = (progs::JobResult*)dev_result;
    int rc = stage_args(rt, &a, sizeof(a), s);
    if (rc != GPUMPI_OK) return rc;
    const ProgramEntry* pe = find_program("job");
    return launch_rank_grid(rt, pe->kernel, job->ranks, 0, nullptr, s);
}

int64_t gpumpi_job_heap_bytes(const gpumpi_job* job) {
    if (!job) return -1;
    progs::JobDesc d{job->id, job->seed, job->type, job->ranks, job->size};
    return progs::job_bytes(d);
}

}  // extern "C"

// ==================================================================== allocation-free step
// One Alltoallv step (plan, scan and copy kernels, as gpumpi_a2av_execute runs them) whose
// tables -- the per-segment ends and sources, row sizes, chunk prefix and payload total of
// a plan's workspace -- live in `scratch`, a file-scope device array, so the call allocates
// nothing.  Every field is written by the step's own plan and scan kernels before the copy
// kernel reads it; nothing has to start at zero.
constexpr int32_t kNoAllocMaxRanks = 512;
constexpr size_t kNoAllocScratchBytes =
    sizeof(uint64_t) * (2ull * kNoAllocMaxRanks * kNoAllocMaxRanks + 3ull * kNoAllocMaxRanks + 2) + 256;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices];  // scratch's address on each device (host-side view)
int32_t g_scratch_cus[kMaxDevices];
}  // namespace

// The device address of `scratch` on the current device, looked up once per device with
// that device current (the array's name is a host-side stand-in, not a device address).
static int noalloc_scratch(void** ptr, int32_t* cus) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return GPUMPI_E_HIP;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return GPUMPI_E_HIP;
        int32_t n = 0;
        if (gpumpi_device_info(&n, nullptr, nullptr) != GPUMPI_OK || n <= 0) return GPUMPI_E_HIP;
        g_scratch_ptr[dev] = p;
        g_scratch_cus[dev] = n;
    }
    *ptr = g_scratch_ptr[dev];
    *cus = g_scratch_cus[dev];
    return GPUMPI_OK;
}

extern "C" {

int gpumpi_a2av_execute_noalloc(int32_t P, int32_t elem_bytes, void* const* sendbufs,
                                const int32_t* send_counts, const int32_t* send_displs,
                                void* const* recvbufs, int32_t* recv_counts,
                                int32_t* recv_displs, void* stream) {
    if (P <= 0 || elem_bytes <= 0 || !sendbufs || !send_counts || !send_displs || !recvbufs ||
        !recv_counts || !recv_displs)
        return GPUMPI_E_ARG;
    if (P > kNoAllocMaxRanks) {
        g_host_error = "gpumpi_a2av_execute_noalloc: " + std::to_string(P) + " ranks exceed the " +
                       std::to_string(kNoAllocMaxRanks) + " its static workspace holds";
        return GPUMPI_E_ARG;
    }
    void* ws = nullptr;
    int32_t cus = 0;
    int rc = noalloc_scratch(&ws, &cus);
    if (rc != GPUMPI_OK) return rc;
    A2avDev d{};
    d.P = P;
    d.elem = elem_bytes;
    d.sendbufs = (char* const*)sendbufs;
    d.scounts = send_counts;
    d.sdispls = send_displs;
    d.recvbufs = (char* const*)recvbufs;
    d.rcounts = recv_counts;
    d.rdispls = recv_displs;
    const uint64_t PP = (uint64_t)P * (uint64_t)P;
    d.seg_end = (uint64_t*)ws;
    d.seg_src = d.seg_end + PP;
    d.row_bytes = d.seg_src + PP;
    d.chunk_off = d.row_bytes + P;
    d.short_off = d.chunk_off + P + 1;
    d.total_bytes = (int64_t*)(d.short_off + P + 1);
    d.plan_done = nullptr;
    d.chunk_lines = (uint32_t)(kA2avCopyThreads * 4 * 2);  // 4 lines per lane, 2 rounds
    d.min_lines = (uint32_t)(kA2avCopyThreads * 4);
    d.straddle_blocks = 0;
    hipStream_t s = (hipStream_t)stream;
    void* kargs2[] = {(void*)&d, (void*)&d};
    // the copy grid strides over the chunks: 16 workgroups per CU
    if (a2av_launch_tables(d, true, s) != GPUMPI_OK ||
        hipLaunchKernel(a2av_copy_for(4, true, false, false), dim3(16 * cus), dim3(kA2avCopyThreads),
                        kargs2, 0, s) != hipSuccess)
        return GPUMPI_E_HIP;
    return GPUMPI_OK;
}

}  // extern "C"

// ==================================================================== batched Reduce / Allreduce
struct gpumpi_reduce_plan {
    ReduceDev dev{};
    const void* kernel = nullptr;
    int grid = 0;
    int32_t log_cols = 0;    // staged kernel: columns per tile
    std::vector<A2avGraph> graphs;
};

static int reduce_launch(gpumpi_reduce_plan* pl, hipStream_t s) {
    void* kargs[] = {(void*)&pl->dev, (void*)&pl->log_cols};   // (the other kernels take the first)
    return hipLaunchKernel(pl->kernel, dim3(pl->grid), dim3(kReduceThreads), kargs, 0, s) == hipSuccess
               ? GPUMPI_OK : GPUMPI_E_HIP;
}

// Whether buffers of `bytes` take the staged kernel: those with too few tiles for the kernels
// that fold from HBM.  Measured (Allreduce of doubles, from HBM / staged, us): 1024 ranks x 4
// KiB 165 / 24, 64 KiB 169 / 42, 256 KiB 168 / 129, 768 KiB 338 / 410; 512 ranks x 256 KiB
// 85 / 45, 384 KiB 89 / 104; 32 ranks x 4 KiB 6.8 / 3.2, 512 KiB 9.8 / 7.7, 768 KiB 11 / 12.
// The split fold of whole numbers (4 ranks and more) is passed up to 128 KiB: int32, 1024
// ranks x 64 KiB 54 / 39, 128 KiB 59 / 52, 256 KiB 95 / 129.
static bool reduce_is_staged(int32_t P, uint64_t bytes, bool split) {
    if (split) return bytes <= (128u << 10);
    return bytes <= (P <= 64 ? 512u << 10 : 256u << 10);
}

// 16-byte columns per tile of the staged kernel (log2): 4 workgroups per CU, but 128-byte
// tiles and more while those give 2 (1024 ranks x 64 KiB: 128-byte tiles 42 us, 64-byte 45).
static int reduce_staged_cols(uint64_t cols, uint64_t cus) {
    int k = 6;
    while (k > 3 && cols >> k < 4 * cus) k--;
    return k == 3 && cols >> 3 < 2 * cus ? 2 : k;
}

extern "C" {

int gpumpi_reduce_plan_create(int32_t P, int64_t count, int32_t datatype, int32_t op, int32_t root,
                              void* const* sendbufs, void* const* recvbufs,
                              gpumpi_reduce_plan** out) {
    if (!out || P <= 0 || count < 0 || !sendbufs || !recvbufs || root < -1 || root >= P)
        return GPUMPI_E_ARG;
    *out = nullptr;
    const int es = type_size(datatype);
    int32_t cus = 0;
    if (gpumpi_device_info(&cus, nullptr, nullptr) != GPUMPI_OK) return GPUMPI_E_HIP;
    const uint64_t bytes = es > 0 ? (uint64_t)count * (uint64_t)es : 0;
    const bool wide = bytes / (1024ull * kReduceWideU) >= 4ull * (uint64_t)cus;
    // integer pairs below the wide shape fold with the ranks split over a workgroup's waves
    const void* ks = es > 0 && !wide && P >= kReduceSplitWaves ? batched_reduce_split_lookup(datatype, op) : nullptr;
    const void* kst = es > 0 && reduce_is_staged(P, bytes, ks != nullptr) ? batched_reduce_staged_lookup(datatype, op) : nullptr;
    const void* k = kst ? kst : ks ? ks : es > 0 ? batched_reduce_kernel_lookup(datatype, op, wide) : nullptr;
    if (!k) {
        g_host_error = "batched reduction: the pair (datatype " + std::to_string(datatype) +
                       ", operator " + std::to_string(op) + ") is not on the batched path "
                       "(int32/uint32/int64/uint64/float/double with MAX, MIN, SUM, PROD); "
                       "MPI_Reduce on the rank grid takes every legal pair";
        return GPUMPI_E_ARG;
    }
    gpumpi_reduce_plan* pl = new gpumpi_reduce_plan();
    pl->kernel = k;
    const uint64_t written = bytes * (root < 0 ? (uint64_t)P : 1u);
    pl->dev.P = P;
    pl->dev.root = root;
    pl->dev.count = count;
    pl->dev.nt = written >= (64ull << 20) ? 1 : 0;  // outputs larger than the L2s stream past them
    pl->dev.sendbufs = (const char*)sendbufs;
    pl->dev.recvbufs = (const char*)recvbufs;
    uint64_t g = ks && !kst ? batched_reduce_split_grid(bytes)
                    : batched_reduce_grid(bytes, wide ? kReduceWideU : kReduceNarrowU);
    if (kst) {
        const uint64_t cols = (bytes + 15) / 16;
        pl->log_cols = reduce_staged_cols(cols, (uint64_t)cus);
        g = (cols + (1ull << pl->log_cols) - 1) >> pl->log_cols;
    }
    if (g > (1u << 20)) g = 1u << 20;  // the waves stride over the rest
    if (g < 1) g = 1;
    if (!kst && bytes % 16) g++;       // the partial last column's workgroup
    pl->grid = (int)g;
    *out = pl;
    return GPUMPI_OK;
}

void gpumpi_reduce_plan_destroy(gpumpi_reduce_plan* pl) {
    if (!pl) return;
    hipDeviceSynchronize();
    for (A2avGraph& g : pl->graphs) {
        if (g.exec) hipGraphExecDestroy(g.exec);
        if (g.def) hipGraphDestroy(g.def);
    }
    delete pl;
}

int gpumpi_reduce_execute(gpumpi_reduce_plan* pl, void* stream) {
    if (!pl) return GPUMPI_E_ARG;
    return reduce_launch(pl, (hipStream_t)stream);
}

int gpumpi_reduce_graph_replay(gpumpi_reduce_plan* pl, int32_t steps, void* stream) {
    if (!pl || steps <= 0) return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    A2avGraph* g = nullptr;
    for (A2avGraph& x : pl->graphs)
        if (x.steps == steps) g = &x;
    if (!g) {
        hipStream_t cs;
        if (hipStreamCreate(&cs) != hipSuccess) return GPUMPI_E_HIP;
        if (hipStreamSynchronize(s) != hipSuccess ||
            hipStreamBeginCapture(cs, hipStreamCaptureModeRelaxed) != hipSuccess) {
            hipStreamDestroy(cs);
            return GPUMPI_E_HIP;
        }
        int rc = GPUMPI_OK;
        for (int i = 0; i < steps && rc == GPUMPI_OK; i++) rc = reduce_launch(pl, cs);
        A2avGraph ng;
        ng.steps = steps;
        hipError_t ee = hipStreamEndCapture(cs, &ng.def);
        hipStreamDestroy(cs);
        if (rc != GPUMPI_OK || ee != hipSuccess) {
            if (ng.def) hipGraphDestroy(ng.def);
            return GPUMPI_E_HIP;
        }
        if (hipGraphInstantiate(&ng.exec, ng.def, nullptr, nullptr, 0) != hipSuccess) {
            hipGraphDestroy(ng.def);
            return GPUMPI_E_HIP;
        }
        pl->graphs.push_back(ng);
        g = &pl->graphs.back();
    }
    return hipGraphLaunch(g->exec, s) == hipSuccess ? GPUMPI_OK : GPUMPI_E_HIP;
}

int gpumpi_reduce_kernel_time(gpumpi_reduce_plan* pl, int32_t reps, void* stream, double* us) {
    if (!pl || reps < 1 || !us) return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return GPUMPI_E_HIP;
    if (hipEventCreate(&e1) != hipSuccess) {
        hipEventDestroy(e0);
        return GPUMPI_E_HIP;
    }
    double acc = 0;
    int rc = GPUMPI_OK;
    for (int i = 0; i < reps && rc == GPUMPI_OK; i++) {
        hipEventRecord(e0, s);
        rc = reduce_launch(pl, s);
        hipEventRecord(e1, s);
        if (rc == GPUMPI_OK && hipEventSynchronize(e1) == hipSuccess) {
            float ms = 0.f;
            hipEventElapsedTime(&ms, e0, e1);
            acc += 1000.0 * ms;
        } else {
            rc = GPUMPI_E_HIP;
        }
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (rc == GPUMPI_OK) *us = acc / reps;
    return rc;
}

}  // extern "C"

// ==================================================================== local sort, NPB IS
// Keys of at most kSortLowBits bits: one table, three launches.
static int sort_short_keys(const uint32_t* keys, int64_t n, uint32_t bins, uint32_t* out, hipStream_t s) {
    Workspace ws(sizeof(uint32_t) * bins);
    if (!ws.ptr) return GPUMPI_E_NOMEM;
    uint32_t* hist = (uint32_t*)ws.ptr;
    // at most 512 workgroups add their counts to the table; a few of the expansion's tiles
    // per workgroup, which scans the whole table
    const int64_t step = 4 * kSortThreads;
    const int64_t per = std::max<int64_t>(step, (n / 512 + step - 1) / step * step);
    const int64_t outs = std::max<int64_t>(kSortTile, (n / 1024 + kSortTile - 1) / kSortTile * kSortTile);
    hipLaunchKernelGGL(sort_zero_kernel, dim3((bins + kSortThreads - 1) / kSortThreads), dim3(kSortThreads), 0, s, hist,
                       bins);
    hipLaunchKernelGGL(sort_count_kernel, dim3((unsigned)((n + per - 1) / per)), dim3(kSortThreads), 0, s, keys, n, per,
                       bins, hist);
    hipLaunchKernelGGL(sort_expand_kernel, dim3((unsigned)((n + outs - 1) / outs)), dim3(kSortThreads), 0, s, hist, bins,
                       n, outs, out);
    return ws.finish(s, hipGetLastError() == hipSuccess);
}

// Longer keys, split by their top bits into `parts` parts first.
static int sort_by_parts(const uint32_t* keys, int64_t n, uint32_t parts, uint32_t* out, hipStream_t s) {
    // a part is cut into chunks where one workgroup would hold up the others: about 512
    // chunks of all keys, each worth the 2^14 counters it adds to the part's table
    const int64_t chunk = std::min<int64_t>(262144, std::max<int64_t>(kSortTile, (n / 512 + kSortTile - 1) / kSortTile * kSortTile));
    const int64_t most = 2 * chunk;
    const uint32_t ntables = (uint32_t)std::min<int64_t>(parts, n / most);
    const size_t words = (size_t)parts * 5 + 2;
    Workspace ws(sizeof(uint32_t) * (words + (size_t)ntables * kSortBins));
    if (!ws.ptr) return GPUMPI_E_NOMEM;
    SortParts sp{};
    sp.count = (uint32_t*)ws.ptr;
    sp.first = sp.count + parts;
    sp.moved = sp.first + parts + 1;
    sp.item = sp.moved + parts;
    sp.table = (int32_t*)(sp.item + parts + 1);
    sp.tables = sp.count + words;
    const int64_t step = 4 * kSortThreads;
    const int64_t per = std::max<int64_t>(step, (n / 2048 + step - 1) / step * step);
    const unsigned items = (unsigned)(parts + n / chunk);
    hipLaunchKernelGGL(sort_zero_kernel, dim3(1), dim3(kSortThreads), 0, s, sp.count, parts);
    hipLaunchKernelGGL(sort_top_hist_kernel, dim3((unsigned)((n + per - 1) / per)), dim3(kSortThreads), 0, s, keys, n,
                       per, parts, sp.count);
    hipLaunchKernelGGL(sort_top_scan_kernel, dim3(1), dim3(kSortThreads), 0, s, sp, parts, (uint32_t)most,
                       (uint32_t)chunk);
    hipLaunchKernelGGL(sort_split_kernel, dim3((unsigned)((n + kSortTile - 1) / kSortTile)), dim3(kSortThreads), 0, s,
                       keys, n, sp, parts, ntables, out);
    hipLaunchKernelGGL(sort_part_kernel, dim3(items), dim3(kSortThreads), 0, s, sp, parts, (uint32_t)chunk, out);
    if (ntables)
        hipLaunchKernelGGL(sort_part_expand_kernel, dim3(items), dim3(kSortThreads), 0, s, sp, parts, (uint32_t)chunk,
                           out);
    return ws.finish(s, hipGetLastError() == hipSuccess);
}

extern "C" {

int gpumpi_local_sort(const uint32_t* keys, int64_t n, int32_t key_bits, uint32_t* out,
                      void* stream) {
    if (!keys || !out || n < 0 || n >= (1ll << 32) || key_bits < 1 || key_bits > 30)
        return GPUMPI_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    if (n == 0) return GPUMPI_OK;
    const uintptr_t ka = (uintptr_t)keys, oa = (uintptr_t)out, len = sizeof(uint32_t) * (uintptr_t)n;
    const bool overlap = ka < oa + len && oa < ka + len;
    if (key_bits <= kSortLowBits) return sort_short_keys(keys, n, 1u << key_bits, out, s);
    if (key_bits <= kSortLowBits + kSortTopBits && !overlap)
        return sort_by_parts(keys, n, 1u << (key_bits - kSortLowBits), out, s);
    const uint32_t nbins = 1u << key_bits;
    const int nblk = (int)((nbins + 4095) / 4096);
    uint32_t *hist = nullptr, *prefix = nullptr, *big = nullptr, *nbig = nullptr;
    uint64_t* sums = nullptr;
    int rc = GPUMPI_OK;
    if (hipMalloc((void**)&hist, sizeof(uint32_t) * nbins) != hipSuccess ||
        hipMalloc((void**)&prefix, sizeof(uint32_t) * nbins) != hipSuccess ||
        hipMalloc((void**)&big, sizeof(uint32_t) * nbins) != hipSuccess ||
        hipMalloc((void**)&nbig, 64) != hipSuccess ||
        hipMalloc((void**)&sums, sizeof(uint64_t) * nblk) != hipSuccess)
        rc = GPUMPI_E_NOMEM;
    if (rc == GPUMPI_OK) {
        hipMemsetAsync(hist, 0, sizeof(uint32_t) * nbins, s);
        hipMemsetAsync(nbig, 0, 64, s);
        hipLaunchKernelGGL(sort_hist_kernel, dim3(1024), dim3(1024), 0, s, keys, n, nbins, hist);
        hipLaunchKernelGGL(scan_block_sums_kernel, dim3(nblk), dim3(1024), 0, s, hist, nbins, sums);
        hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(1024), 0, s, sums, nblk);
        hipLaunchKernelGGL(scan_apply_kernel, dim3(nblk), dim3(1024), 0, s, hist, nbins, sums, prefix);
        hipLaunchKernelGGL(sort_runs_kernel, dim3(2048), dim3(256), 0, s, hist, prefix, nbins, out, big, nbig);
        hipLaunchKernelGGL(sort_fill_runs_kernel, dim3(1024), dim3(256), 0, s, hist, prefix, big,
                           nbig, out);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) rc = GPUMPI_E_HIP;
    }
    hipFree(hist);
    hipFree(prefix);
    hipFree(big);
    hipFree(nbig);
    hipFree(sums);
    return rc;
}

// NPB IS (toolchain_tests/npb/NPB3.4.1/NPB3.4-MPI/IS/is.c) on the batched path: keys from
// create_seq, one untimed rank(1), then rank(1..10) -- each iteration alters two keys of
// rank 0 (is.c:650-654), builds the bucket plan, runs the batched exchange and checks the
// five partial-verification keys (is.c:849-905: the rank of test key k is the number of
// keys < k); after the last iteration every rank's keys are sorted (local sort) and the
// global order checked (full_verify, is.c:545-621).  *passed follows is.c:1137: it must be
// 5 * 10 + P for a correct run.
int gpumpi_npb_is_run(char cls, int32_t P, int64_t* passed, double* exchange_ms) {
    NpbClassInfo ci;
    if (!npb_class_info(cls, ci)) return GPUMPI_E_ARG;
    const int tk = ci.total_keys_log2, mk = ci.max_key_log2, bk = ci.num_buckets_log2;
    const int64_t* tidx = ci.test_index;
    const int64_t* trank = ci.test_rank;
    if (P < 1 || (P & (P - 1)) || !passed) return GPUMPI_E_ARG;
    const int64_t T = 1ll << tk, n = T / P, maxkey = 1ll << mk;
    const int shift = mk - bk;
    hipStream_t s = nullptr;
    std::vector<void*> bufs;
    auto al = [&](size_t b) -> void* {
        void* q = nullptr;
        if (hipMalloc(&q, b ? b : 16) != hipSuccess) return nullptr;
        bufs.push_back(q);
        return q;
    };
    uint32_t* keys = (uint32_t*)al(sizeof(uint32_t) * T);
    uint32_t* kb1 = (uint32_t*)al(sizeof(uint32_t) * T);
    uint32_t* recv = (uint32_t*)al(sizeof(uint32_t) * T + 64);
    uint32_t* sorted = (uint32_t*)al(sizeof(uint32_t) * T + 64);
    int32_t* sc = (int32_t*)al(sizeof(int32_t) * P * P);
    int32_t* sd = (int32_t*)al(sizeof(int32_t) * P * P);
    int32_t* rc_ = (int32_t*)al(sizeof(int32_t) * P * P);
    int32_t* rd = (int32_t*)al(sizeof(int32_t) * P * P);
    int32_t* lo = (int32_t*)al(sizeof(int32_t) * P);
    int32_t* hi = (int32_t*)al(sizeof(int32_t) * P);
    void** sptr = (void**)al(sizeof(void*) * P);
    void** rptr = (void**)al(sizeof(void*) * P);
    unsigned long long* cnt = (unsigned long long*)al(64);
    int rcode = GPUMPI_OK;
    gpumpi_a2av_plan* plan = nullptr;
    std::vector<void*> hs(P), hr(P);
    std::vector<int32_t> hsc((size_t)P * P), hlo(P), hhi(P);
    std::vector<int64_t> rtot(P), roff(P);
    double ex_ms = 0;
    hipEvent_t e0, e1;
    hipEventCreate(&e0);
    hipEventCreate(&e1);
    for (void* q : bufs)
        if (!q) rcode = GPUMPI_E_NOMEM;
    int64_t pass = 0;
    if (rcode == GPUMPI_OK) {
        for (int r = 0; r < P; r++) hs[r] = kb1 + (int64_t)r * n;
        hipMemcpy(sptr, hs.data(), sizeof(void*) * P, hipMemcpyHostToDevice);
        hipMemcpy(rptr, hs.data(), sizeof(void*) * P, hipMemcpyHostToDevice);  // replaced per step
        rcode = gpumpi_gen_keys(keys, P, n, 0, 0, 2, mk, nullptr, 0, s);
    }
    if (rcode == GPUMPI_OK)
        rcode = gpumpi_a2av_plan_create(P, 4, sptr, sc, sd, rptr, rc_, rd, nullptr, &plan);
    for (int step = 0; step <= 10 && rcode == GPUMPI_OK; step++) {
        const int it = step == 0 ? 1 : step;  // step 0 is the untimed rank(1), is.c:1069
        int32_t mod[2] = {it, (int32_t)(maxkey - it)};
        hipMemcpy(keys + it, &mod[0], 4, hipMemcpyHostToDevice);
        hipMemcpy(keys + it + 10, &mod[1], 4, hipMemcpyHostToDevice);
        uint32_t tkeys[5];
        for (int i = 0; i < 5; i++) hipMemcpy(&tkeys[i], keys + tidx[i], 4, hipMemcpyDeviceToHost);
        rcode = gpumpi_bucket_plan(keys, P, n, mk, bk, kb1, sc, sd, lo, hi, s);
        if (rcode != GPUMPI_OK) break;
        hipMemcpy(hsc.data(), sc, sizeof(int32_t) * P * P, hipMemcpyDeviceToHost);
        hipMemcpy(hlo.data(), lo, sizeof(int32_t) * P, hipMemcpyDeviceToHost);
        hipMemcpy(hhi.data(), hi, sizeof(int32_t) * P, hipMemcpyDeviceToHost);
        int64_t off = 0;
        for (int d = 0; d < P; d++) {
            int64_t t = 0;
            for (int q = 0; q < P; q++) t += hsc[(size_t)q * P + d];
            rtot[d] = t;
            roff[d] = off;
            hr[d] = recv + off;
            off += t;
        }
        hipMemcpy(rptr, hr.data(), sizeof(void*) * P, hipMemcpyHostToDevice);
        hipEventRecord(e0, s);
        rcode = gpumpi_a2av_execute(plan, s);
        hipEventRecord(e1, s);
        hipStreamSynchronize(s);
        float ms = 0;
        hipEventElapsedTime(&ms, e0, e1);
        if (step > 0) ex_ms += ms;
        int64_t bytes = 0;
        if (rcode == GPUMPI_OK) rcode = gpumpi_a2av_payload_bytes(plan, &bytes);
        if (rcode != GPUMPI_OK) break;
        // partial verification (is.c:849-905)
        for (int i = 0; i < 5 && step > 0; i++) {
            const int64_t k = tkeys[i];
            const int64_t b = k >> shift;
            int owner = -1;
            for (int d = 0; d < P; d++)
                if (hlo[d] <= b && b <= hhi[d]) owner = d;
            if (owner < 0) continue;
            hipMemset(cnt, 0, 8);
            hipLaunchKernelGGL(count_less_kernel, dim3(256), dim3(256), 0, s, recv + roff[owner],
                               rtot[owner], (uint32_t)k, cnt);
            unsigned long long c = 0;
            hipMemcpy(&c, cnt, 8, hipMemcpyDeviceToHost);
            const int64_t key_rank = (int64_t)c + roff[owner];
            const int64_t tr = npb_expected_rank(cls, i, it, trank[i]);
            if (key_rank == tr) pass++;
        }
    }
    if (rcode == GPUMPI_OK) {
        // full_verify (is.c:545-621): sort every rank's keys, check each rank's slice lies in
        // its bucket range and the concatenation is ascending
        rcode = gpumpi_local_sort(recv, T, mk, sorted, s);
        if (rcode == GPUMPI_OK) {
            std::vector<uint32_t> hs2(T);
            hipMemcpy(hs2.data(), sorted, sizeof(uint32_t) * T, hipMemcpyDeviceToHost);
            for (int d = 0; d < P; d++) {
                bool ok = true;
                for (int64_t i = roff[d]; i < roff[d] + rtot[d]; i++) {
                    const int64_t b = (int64_t)hs2[i] >> shift;
                    if (b < hlo[d] || b > hhi[d]) ok = false;
                    if (i > 0 && hs2[i - 1] > hs2[i]) ok = false;
                }
                if (ok) pass++;
            }
        }
    }
    if (plan) gpumpi_a2av_plan_destroy(plan);
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    for (void* q : bufs) hipFree(q);
    *passed = pass;
    if (exchange_ms) *exchange_ms = ex_ms;
    return rcode;
}

}  // extern "C"
