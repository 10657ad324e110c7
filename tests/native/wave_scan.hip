// Device code whose assembly test_native_cpu.py looks at.
#include "../../thundergbm_amd/csrc/kernel_common.h"

__global__ void k_scan(long long *p) {
    long long a = p[threadIdx.x], b = p[threadIdx.x + 64];
    tgbm::wave_scan_pair(a, b);
    p[threadIdx.x] = a;
    p[threadIdx.x + 64] = b;
    p[128] = tgbm::read_lane_ll(b, 63);
}
