// The team forms of the evaluator (several workgroups per position, the smallest launches), and what they need to know of the device.
#include <cstdlib>
#include <cstring>

#include "bf_team.hip.h"

namespace bf {

hipError_t launch_team256(const KArgs& k, hipStream_t stream) { return team::launch_team<256, MODE_EVAL, false>(k, stream); }
hipError_t launch_team256_enc(const KArgs& k, hipStream_t stream) { return team::launch_team<256, MODE_ENC, false>(k, stream); }
hipError_t launch_team256_fp8(const KArgs& k, hipStream_t stream) { return team::launch_team<256, MODE_EVAL, true>(k, stream); }
hipError_t launch_team256_fp8_enc(const KArgs& k, hipStream_t stream) { return team::launch_team<256, MODE_ENC, true>(k, stream); }
hipError_t launch_team512(const KArgs& k, hipStream_t stream) { return team::launch_team<512, MODE_EVAL, false>(k, stream); }
hipError_t launch_team512_enc(const KArgs& k, hipStream_t stream) { return team::launch_team<512, MODE_ENC, false>(k, stream); }

size_t team_slot_bytes(int d_model) { return d_model == 512 ? team::Cfg<512>::WS_BYTES : team::Cfg<256>::WS_BYTES; }

// which XCD (HW_REG_XCC_ID) each workgroup runs on
__global__ void xcd_probe(int* out) {
    if (threadIdx.x == 0) out[blockIdx.x] = (int)__builtin_amdgcn_s_getreg(20 | (3 << 11));
}

// Where team launches report that they gave up: a word per device in pinned host memory, which is never given back (a
// launch may be under way whenever that could happen).
constexpr int REPORT_STRIDE = 16;   // ints: a cache line each
static int* report_words() {
    static int* const words = []() -> int* {
        void* p = nullptr;
        if (hipHostMalloc(&p, 64 * REPORT_STRIDE * sizeof(int), hipHostMallocPortable | hipHostMallocMapped) != hipSuccess) return nullptr;
        memset(p, 0, 64 * REPORT_STRIDE * sizeof(int));
        return static_cast<int*>(p);
    }();
    return words;
}
static std::atomic<int*> g_report[64];   // device address of device i's word, nullptr until its look

int* team_report_word() {
    int dev = 0;
    return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 ? g_report[dev].load(std::memory_order_acquire) : nullptr;
}

bool team_gave_up() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64 || !g_report[dev].load(std::memory_order_acquire)) return false;
    int* const word = report_words() + dev * REPORT_STRIDE;
    return __atomic_load_n(word, __ATOMIC_RELAXED) && __atomic_exchange_n(word, 0, __ATOMIC_RELAXED);
}

// hardware queues a process may have launches under way on: GPU_MAX_HW_QUEUES, HIP's default 4
static int hardware_queues() {
    const char* const s = getenv("GPU_MAX_HW_QUEUES");
    const int q = s ? atoi(s) : 0;
    return q > 0 ? q : 4;
}

// Positions a team launch may hold on the current device, 0 where the form does not run: one workgroup per compute
// unit, and the workgroups whose numbers agree modulo 8 on one XCD (they share an L2 there).  Looked up once per device.
// Nor does it run where this process could have more launches under way than the device has units for (bf_team.hip.h).
int team_positions(int d_model, bool look) {
    static std::atomic<int> units[64];   // compute units + 1 of a device that qualifies, -1 of one that does not, 0 not looked up
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int u = units[dev].load(std::memory_order_acquire);
    if (u == 0 && look) {
        constexpr int N = 1024;
        int cus = 0, *d = nullptr, h[N];
        bool ok = device_is_gfx950() && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
                  hipMalloc(reinterpret_cast<void**>(&d), sizeof(h)) == hipSuccess;
        if (ok) {
            hipLaunchKernelGGL(xcd_probe, dim3(N), dim3(64), 0, nullptr, d);
            ok = hipGetLastError() == hipSuccess && hipMemcpy(h, d, sizeof(h), hipMemcpyDeviceToHost) == hipSuccess;
        }
        if (d) (void)hipFree(d);
        for (int i = 8; ok && i < N; i++) ok = h[i] == h[i & 7];
        void* word = nullptr;
        ok = ok && report_words() && hipHostGetDevicePointer(&word, report_words() + dev * REPORT_STRIDE, 0) == hipSuccess;
        if (ok) g_report[dev].store(static_cast<int*>(word), std::memory_order_release);
        u = ok ? cus + 1 : -1;
        units[dev].store(u, std::memory_order_release);
    }
    const int per = d_model == 512 ? team::Cfg<512>::NWG : team::Cfg<256>::NWG;
    static const int queues = hardware_queues();
    return u > 0 && team::units_suffice(queues, per, (u - 1) / 8) ? (u - 1) / (8 * per) * 8 : 0;
}

}  // namespace bf
