// The team forms of the evaluator (several workgroups per position, the smallest launches), and what they need to know of the device.
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

// Positions a team launch may hold on the current device, 0 where the form does not run: one workgroup per compute
// unit, and the workgroups whose numbers agree modulo 8 on one XCD (they share an L2 there).  Looked up once per device.
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
        u = ok ? cus + 1 : -1;
        units[dev].store(u, std::memory_order_release);
    }
    const int per = d_model == 512 ? team::Cfg<512>::NWG : team::Cfg<256>::NWG;
    return u > 0 ? (u - 1) / (8 * per) * 8 : 0;
}

}  // namespace bf
