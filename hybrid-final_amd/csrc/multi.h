// Several cases' launches of one kernel merged into one grid.
//
// A batch of cases steps together by running each kernel of the step once
// for all of them: the launches a case's step would make are recorded (the
// kernel's merged-grid launcher, its argument record and its block count),
// the records of the same launch of every case are placed side by side in
// device memory, and one grid covers all their blocks (cases whose step runs
// another kernel at that place of the sequence get a grid of their own).  Block b of that grid
// reads map[b] = job << MULTI_LB_BITS | block-within-job, and runs the
// kernel's body with that job's arguments as that block.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstring>
#include <vector>

namespace pic {

constexpr int MULTI_LB_BITS = 22;   // blocks per job < 4 M, jobs < 1024

__device__ inline int multi_job(const uint32_t *map, int &lb) {
    const uint32_t m = map[blockIdx.x];   // one load per block; uniform
    lb = (int)(m & ((1u << MULTI_LB_BITS) - 1));
    return (int)(m >> MULTI_LB_BITS);
}

// A job record, read the way kernel arguments are: records never change while
// a grid runs, so their loads go through the constant address space and stay
// scalar.  As ordinary memory, which the kernel's own stores might change,
// every pointer of a record was a vector load (the merged scatter held 121
// VGPRs, the single-case one 54).
template <typename J>
__device__ inline const J &multi_record(const J *jobs, const uint32_t *map, int &lb) {
    typedef const __attribute__((address_space(4))) J *Constant;
    return *(const J *)(Constant)(uintptr_t)(jobs + multi_job(map, lb));   // by way of an integer: a plain cast folds away
}

// A pointer out of a record, known to the compiler as one to device memory (a
// pointer loaded from memory could be one to LDS too, and its accesses would
// be the slower flat ones).
template <typename T>
__device__ inline T *device_ptr(T *p) {
    typedef __attribute__((address_space(1))) T *Global;
    return (T *)(Global)(uintptr_t)p;
}

// launches a merged grid of `total` blocks over the job records at `jobs`
typedef void (*MultiLaunchFn)(const void *jobs, const uint32_t *map, int total, hipStream_t s);

// the MultiLaunchFn of merged-grid kernel K (job record type J, LB threads per block)
template <typename J, void (*K)(const J *, const uint32_t *), int LB>
void launch_m(const void *jobs, const uint32_t *map, int total, hipStream_t s) {
    hipLaunchKernelGGL(K, dim3(total), dim3(LB), 0, s, (const J *)jobs, map);
}

struct RecordedLaunch {
    MultiLaunchFn fn;
    size_t job_size, job_align;
    int blocks;
    std::vector<unsigned char> job;
};

struct Recorder {
    std::vector<RecordedLaunch> launches;
    long long cells = 0;   // of all the cases that will share the launches (launch shapes follow the whole grid)
    template <typename J>
    void add(MultiLaunchFn fn, const J &job, int blocks) {
        RecordedLaunch r{fn, sizeof(J), alignof(J), blocks, {}};
        r.job.resize(sizeof(J));
        memcpy(r.job.data(), &job, sizeof(J));
        launches.push_back(std::move(r));
    }
};

// The launch recorder of the calling host thread: when set, the launchers of
// the batched step's kernels record their launch instead of making it.
Recorder *&launch_recorder();

}  // namespace pic
