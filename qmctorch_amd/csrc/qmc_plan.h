// Plan object and error reporting shared by the C-ABI translation units of
// libqmcmi355x (qmc_abi.hip, qmc_api.hip, qmc_adjoint.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

#include "qmc_launch.h"

struct QmcPlan {
    qmc::Tables t;
    const qmc::SpecEntry* spec = nullptr;  // kernels generated for this basis layout, if any
    bool use_spec = true;
    int nexp_grp = 0;  // exponents in group order (length of QmcParams.grp_exp)
    std::vector<void*> allocs;
    ~QmcPlan() {
        for (void* p : allocs) (void)hipFree(p);
    }
    // Tables are placed in chunks of device memory through host mirrors, copied
    // once by upload_done(): with an allocation and a copy per table a plan took
    // 320 us to create, now 51 (N2).
    struct Chunk {
        char* dev;
        size_t size;
        std::vector<char> host;
    };
    std::vector<Chunk> chunks;
    template <typename X>
    const X* upload(const X* host, size_t n) {
        if (n == 0 || host == nullptr) return nullptr;
        const size_t bytes = n * sizeof(X), kChunk = 256 * 1024, kAlign = 256;
        if (chunks.empty() || (chunks.back().host.size() + kAlign - 1) / kAlign * kAlign + bytes > chunks.back().size) {
            const size_t size = bytes > kChunk ? bytes : kChunk;
            void* d = nullptr;
            if (hipMalloc(&d, size) != hipSuccess) throw std::runtime_error("hipMalloc failed");
            allocs.push_back(d);
            chunks.push_back(Chunk{(char*)d, size, {}});
        }
        Chunk& c = chunks.back();
        const size_t at = (c.host.size() + kAlign - 1) / kAlign * kAlign;
        c.host.resize(at + bytes);
        std::memcpy(c.host.data() + at, host, bytes);
        return (const X*)(c.dev + at);
    }
    void upload_done() {
        for (auto& c : chunks)
            if (hipMemcpy(c.dev, c.host.data(), c.host.size(), hipMemcpyHostToDevice) != hipSuccess)
                throw std::runtime_error("hipMemcpy failed");
        chunks.clear();
    }
};

namespace qmc {
// Records msg as the calling thread's last error (qmc_last_error) and returns code.
int set_error(int code, const std::string& msg);
}  // namespace qmc

#define QMC_CHECK_HIP(call)                                                                              \
    do {                                                                                                 \
        hipError_t _e = (call);                                                                          \
        if (_e != hipSuccess)                                                                            \
            return qmc::set_error(QMC_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(_e));       \
    } while (0)
