// Host side of the persistent solves: exchange storage, tags, the cooperative
// launches of a solve and the commit of its x.
#pragma once

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "persist_device.hpp"

namespace pm
{

static __global__ void k_persist_reset(PersistControl* ctl, SolverState* st, unsigned abort)
{
    ctl->abort = abort;
    ctl->finished = 0u;
    st->counters[kCounterOutcome] = 0u;
}

static __global__ void k_persist_clear(word* p, int64_t n)
{
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        p[i] = 0ull;
}

// Copies the new x when every workgroup of the solve reached its end and this
// was the last launch of it, and tells the host.
template <typename S>
__global__ __launch_bounds__(kBlock) void k_persist_commit(int64_t rows, const S* __restrict__ from, S* __restrict__ x,
                                                           const PersistControl* ctl, unsigned blocks, SolverState* st)
{
    if (ctl->finished != blocks) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) st->counters[kCounterOutcome] = 1u;
    if (st->done == kRunning && st->counters[kCounterRestart] == 0u) return;  // the next launch continues from `from`
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < rows;
         i += static_cast<int64_t>(gridDim.x) * kBlock)
        x[i] = from[i];
}

// PLAMATRIX_AMD_PERSISTENT=0 keeps every solve on the per-kernel iteration.
inline bool persist_enabled()
{
    const char* env = std::getenv("PLAMATRIX_AMD_PERSISTENT");
    return env == nullptr || env[0] != '0';
}

// What a test asks of the launches in PLAMATRIX_AMD_PERSIST_TEST, a list of
// name=number: the number, or `none`.  refuse=k, too_large=k: launch k of a call is
// turned down with that error; give_up=k: its workgroups find a notice to give up;
// storage=0: there is no memory for the exchange; segment=n: launches of n iterations
// (even, or one less); tag=n: the last exchange tag used.
inline int64_t persist_test(const char* name, int64_t none)
{
    const char* env = std::getenv("PLAMATRIX_AMD_PERSIST_TEST");
    const char* at = env != nullptr ? std::strstr(env, name) : nullptr;
    return at != nullptr ? std::atoll(at + std::strlen(name)) : none;
}

// Iterations of a launch.
inline int64_t persist_segment(int64_t most)
{
    return std::max<int64_t>(2, persist_test("segment=", most) & ~int64_t(1));
}

// Storage that only the one-launch forms need: without it a solve takes the kernels.
inline bool persist_storage(DeviceBuffer& buffer, size_t need)
{
    return persist_test("storage=", 1) != 0 && buffer.reserve(need) == PM_OK;
}

// Solves (passes of a refinement, batches) for which a workspace stays on the
// per-kernel forms after a launch was refused or gave up: whatever kept its
// workgroups from running together would cost each of them up to kWaitSeconds.
constexpr int kPersistPause = 64;

// Whether `blocks` workgroups of a CU each can run together.
inline bool persist_resident(const pm_workspace* ws, int blocks)
{
    if (ws->persist_pause > 0) return false;
    const int device = ws->device;
    int coop = 0, cus = 0;
    if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
    {
        (void)hipGetLastError();
        return false;
    }
    return coop != 0 && blocks <= cus;
}

// A cooperative launch that the runtime turned down, without an error.  As it does
// for every process but the first that holds a cooperative queue on the device
// (hipErrorIllegalState): the workspace turns to the per-kernel forms.  A launch too
// large for the device says nothing about the next one's shape.
inline bool persist_refused(hipError_t err, pm_workspace* ws)
{
    if (err != hipErrorCooperativeLaunchTooLarge && err != hipErrorNotSupported && err != hipErrorIllegalState)
        return false;
    (void)hipGetLastError();
    if (err != hipErrorCooperativeLaunchTooLarge) ws->persist_pause = kPersistPause;
    return true;
}

// The limit of a kernel's LDS belongs to the process: always the same, whatever another
// thread's launch of the kernel needs.
inline int persist_allow_lds(const void* kernel)
{
    PM_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kPersistLds)));
    return PM_OK;
}

// Launch `number` of a call.
inline hipError_t persist_launch(const void* kernel, int blocks, void** args, size_t lds, hipStream_t stream, int64_t number)
{
    if (persist_test("refuse=", -1) == number) return hipErrorIllegalState;
    if (persist_test("too_large=", -1) == number) return hipErrorCooperativeLaunchTooLarge;
    return hipLaunchCooperativeKernel(kernel, dim3(blocks), dim3(kPersistThreads), args, static_cast<unsigned>(lds), stream);
}

// Exchange tags run up to here before the words are cleared and they start again.
constexpr uint32_t kLastTag = 0xf0000000u;

// Every workgroup decides for itself, or eight decide and answer the rest.
inline int persist_leaders(int blocks) { return blocks <= 64 ? blocks : kXcds; }

// Runs the launches of a solve; `a` is complete but for the exchange storage (of
// `vectors` vectors, xu and xx first) and the iteration range.
template <typename S, typename Args>
int persist_loop(pm_workspace* ws, const PersistProblem& p, Args& a, const void* kernel, int blocks, size_t lds,
                 int64_t max_iterations, hipStream_t stream, int* outcome, int64_t* next, SolverState* state,
                 int vectors = 2)
{
    *outcome = kPersistAbandoned;
    PM_TRY(persist_allow_lds(kernel));
    const size_t words = static_cast<size_t>(p.rows) * Exchange<S>::kWords;
    const size_t control = (sizeof(PersistControl) + 255) & ~size_t(255);
    const size_t need = control + static_cast<size_t>(vectors) * words * sizeof(word);
    const bool grown = need > ws->persist.bytes;
    if (!persist_storage(ws->persist, need)) return PM_OK;
    if (grown) ws->persist_tag = kLastTag;
    else ws->persist_tag = static_cast<uint32_t>(persist_test("tag=", ws->persist_tag));
    const int64_t segment = persist_segment(kSegment);
    a.ctl = ws->persist.as<PersistControl>();
    a.xu = reinterpret_cast<word*>(ws->persist.as<char>() + control);
    a.xx = a.xu + words;
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>(ceil_div(p.rows, kBlock), 2048));
    int64_t number = 0;
    for (int64_t t = 0;; ++number)
    {
        // an even number of iterations, the last one's decision included
        const int64_t left = max_iterations + 2 - t;
        const int64_t count = std::min<int64_t>(segment, left + (left & 1));
        a.t0 = static_cast<int>(t);
        a.t_end = static_cast<int>(t + count);
        if (t > 0) a.x_in = a.x_out;
        if (ws->persist_tag >= kLastTag)
        {
            // no word may carry a tag that is still to come
            hipLaunchKernelGGL(k_persist_clear, dim3(1024), dim3(kBlock), 0, stream, ws->persist.as<word>(),
                               static_cast<int64_t>(ws->persist.bytes / sizeof(word)));
            PM_HIP(hipGetLastError());
            ws->persist_tag = 0;
        }
        a.tag = ws->persist_tag;
        ws->persist_tag += static_cast<uint32_t>(count) + 2u;
        hipLaunchKernelGGL(k_persist_reset, dim3(1), dim3(1), 0, stream, a.ctl, p.st,
                           persist_test("give_up=", -1) == number ? 1u : 0u);
        PM_HIP(hipGetLastError());
        void* args[] = {&a};
        const hipError_t err = persist_launch(kernel, blocks, args, lds, stream, number);
        if (persist_refused(err, ws)) return PM_OK;
        PM_HIP(err);
        hipLaunchKernelGGL(k_persist_commit<S>, dim3(grid), dim3(kBlock), 0, stream, p.rows,
                           static_cast<const S*>(p.x_out), static_cast<S*>(p.x), a.ctl,
                           static_cast<unsigned>(blocks), p.st);
        PM_HIP(hipGetLastError());
        PM_HIP(hipMemcpyAsync(ws->host_state, p.st, sizeof(SolverState), hipMemcpyDeviceToHost, stream));
        PM_HIP(hipStreamSynchronize(stream));
        *state = ws->host_state[0];
        if (state->counters[kCounterOutcome] != 1u)
        {
            ws->persist_pause = kPersistPause;
            return PM_OK;
        }
        if (state->done != kRunning)
        {
            *outcome = kPersistStopped;
            return PM_OK;
        }
        t = static_cast<int64_t>(state->counters[kCounterNext]);
        if (state->counters[kCounterRestart] != 0u)
        {
            *outcome = kPersistHandOver;
            *next = t;
            return PM_OK;
        }
    }
}

} // namespace pm
