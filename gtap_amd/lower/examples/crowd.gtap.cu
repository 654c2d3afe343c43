// 64 parents that all resume in a round in which one of their children has filled the wave's
// deque with n detached tasks: for n a little below the capacity the round's spawns fit and the
// resumed parents do not (the error-path tests).
#include <cuda_runtime.h>
#include "gtap_thread.cuh"

__device__ long long d_out;

#pragma gtap function
__device__ void idle(int i) {
}

#pragma gtap function
__device__ long long child(int i, int n) {
    if (i == 0) {
        for (int k = 0; k < n; ++k) {
            #pragma gtap task
            idle(k);
        }
    }
    return 1;
}

#pragma gtap function
__device__ long long parent(int i, int n) {
    long long a;
    #pragma gtap task
    a = child(i, n);
    #pragma gtap taskwait
    return a;
}

#pragma gtap function
__device__ long long crowd(int n) {
    for (int i = 0; i < 64; ++i) {
        #pragma gtap task
        parent(i, n);
    }
    #pragma gtap taskwait
    return 64;
}

__global__ void crowd_kernel(int n) {
    #pragma gtap entry
    d_out = crowd(n);
}
