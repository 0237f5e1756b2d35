// A HIP runtime that launches nothing, for the host code of the library on a machine without a GPU: one line of stdin is one call
// of the C ABI, one line of stdout its result and the kernels it would launch, in order.
//   bytes B Hq Hkv N D causal window          scratch of the backward: least, with parts, full
//   gemm  M N K trans_b bytes ws              a product of elements of 2 (bf16) or 1 (e4m3) bytes: as bwd; ws = bytes of scratch,
//                                             0 = null, any = TYR_HIP_ANY_ORDER; its scratch follows the status
//   kernels                                   every kernel of the files linked
//   bwd   B Hq Hkv N D causal window mask ws  status, then "kernel<arguments>:workgroups" each; mask = none | lens | keys
//   bwd_lds, the same                         "kernel<arguments>:workgroups:bytes of LDS"
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <iostream>
#include <map>
#include <sstream>
#include <string>

#include "../../include/tyr_hip.h"

static std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> m;
    return m;
}
static std::string launched;
static bool with_lds;

extern "C" {
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    int bad = 0;
    char* plain = abi::__cxa_demangle(name, nullptr, nullptr, &bad);
    std::string s = bad ? name : plain;
    free(plain);
    s = s.substr(0, s.find(">(") == std::string::npos ? s.find('(') : s.find(">(") + 1);
    for (const char* drop : {"void ", "tyr::", "(AttnMask)", " "})
        for (size_t at; (at = s.find(drop)) != std::string::npos;) s.erase(at, std::string(drop).size());
    kernels()[host] = s;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t lds, hipStream_t) {
    if (lds > 160 * 1024 || grid.x == 0 || grid.x > 0x7fffffffu || block.x > 1024) abort();
    launched += " " + kernels()[f] + ":" + std::to_string(grid.x) + (with_lds ? ":" + std::to_string(lds) : "");
    return hipSuccess;
}
}

int main() {
    alignas(16) static char p[16];               // stands for every tensor: nothing reads them
    float* f = reinterpret_cast<float*>(p);
    for (std::string line; std::getline(std::cin, line);) {
        std::istringstream in(line);
        std::string what, mask;
        uint64_t B, Hq, Hkv, N, D, window;
        int causal;
        size_t ws = 0;
        in >> what;
        if (what == "kernels") {
            for (const auto& k : kernels()) printf("%s ", k.second.c_str());
            printf("\n");
            fflush(stdout);
            continue;
        }
        if (what == "gemm") {
            uint64_t M, N, K;
            int trans_b, bytes;
            std::string scratch;
            in >> M >> N >> K >> trans_b >> bytes >> scratch;
            void* to = scratch == "any" ? TYR_HIP_ANY_ORDER : scratch == "0" ? nullptr : p;
            const size_t size = scratch == "any" ? SIZE_MAX : strtoull(scratch.c_str(), nullptr, 10);
            launched.clear();
            const int rc = bytes == 2 ? tyr_hip_gemm_bf16_batched_ws(p, p, p, 1, M, N, K, 0, 0, 0, trans_b, to, size, nullptr)
                                      : tyr_hip_gemm_fp8_ws(p, p, p, M, N, K, 1.0f, nullptr, nullptr, TYR_HIP_OUT_BF16, trans_b, to, size, nullptr);
            printf("%d %zu%s\n", rc, tyr_hip_gemm_workspace_bytes(1, M, N, K, bytes, trans_b), launched.c_str());
            fflush(stdout);
            continue;
        }
        in >> B >> Hq >> Hkv >> N >> D >> causal >> window >> mask >> ws;
        launched.clear();
        with_lds = what == "bwd_lds";
        if (what == "bytes") {
            printf("%zu %zu %zu\n", tyr_hip_flash_attn_bwd_workspace_bytes(B, Hq, N, D),
                   tyr_hip_flash_attn_bwd_parts_workspace_bytes(B, Hq, Hkv, N, D, causal, window),
                   tyr_hip_flash_attn_bwd_full_workspace_bytes(B, Hq, Hkv, N, D, causal, window));
        } else {
            const int rc = mask == "keys" ? tyr_hip_flash_attn_bwd_mask(p, p, p, p, p, f, p, p, p, B, Hq, Hkv, N, D, causal, reinterpret_cast<uint8_t*>(p),
                                                                        0.125f, p, ws, nullptr)
                                          : tyr_hip_flash_attn_bwd_gqa(p, p, p, p, p, f, p, p, p, B, Hq, Hkv, N, D, causal, window,
                                                                       mask == "lens" ? reinterpret_cast<int32_t*>(p) : nullptr, 0.125f, p, ws, nullptr);
            printf("%d%s\n", rc, launched.c_str());
        }
        fflush(stdout);
    }
}
