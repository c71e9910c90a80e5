/*
 * Shared host declarations of the engine's translation units: the context, device
 * arena helpers, job descriptors and the batch pipeline's entry (run_batch, defined in
 * run_batch.h and instantiated per integrand family in batch_*.hip so the families
 * compile in parallel).
 */
#ifndef VMX_ENGINE_CORE_H
#define VMX_ENGINE_CORE_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <array>
#include <functional>
#include <map>
#include <random>
#include <limits>
#include <type_traits>
#include <typeinfo>
#include <new>
#include <stdexcept>
#include <string>
#include <vector>

#include <cstring>
#include <rocprim/rocprim.hpp>

#include "../../include/viltrum_amd.h"
#include "exact.h"
#include "pipeline.h"


struct vmx_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    // bump allocator over a fixed device array, for the entry point that allocates
    // nothing: arenas that point at it are carved from it instead of hipMalloc
    struct Fixed {
        char* base = nullptr;
        size_t cap = 0, used = 0;
    };
    // device memory pool: one arena per purpose, grown on demand
    struct Buf {
        void* p = nullptr;
        size_t bytes = 0;
        Fixed* fixed = nullptr;  // set: a view into a Fixed array, never hipMalloc'd or freed
    };
    Buf tree, regs, lists, misc, params, bins, bins2;
    Buf nn[VMX_MAX_DIM + 1];                       // FP32 priority-network parameters per dim
    Buf nn_lds[VMX_MAX_DIM + 1];                   // ... and their LDS image (nn::NetW<KP>)
    bool nn_ok[VMX_MAX_DIM + 1] = {};
    Buf tr_x, tr_t, tr_idx, tr_part, tr_loss, tr_state, tr_net;  // training work space
    hipEvent_t ev[8] = {};
    void* pinned = nullptr;  // host staging for small device-to-host readbacks
    size_t pinned_bytes = 0;
    // one chunk of refinement rounds captured as a graph, reused while its launch
    // arguments (buffers, shapes, stream) stay the same
    struct RoundGraph {
        std::vector<unsigned char> key;
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
    } rounds, rounds_tail;  // chunks of the tuned size, and of 2 rounds near the end
    // launch shapes: the autotuner's choices per workload class, and the shape a tuning
    // trial forces (keys of the classes the trial ran are collected in tuned_keys)
    struct Shape {
        int gen_per_cu = 4, round_chunk = 8, bins_xcd = 0, deepen = 0;
    };
    std::map<std::array<uint64_t, 6>, Shape> tune;
    // node capacity per region (times N) the last call of a workload class needed, so a
    // class whose rounds overflow 8N does not pay a failed attempt on every call
    std::map<std::array<uint64_t, 6>, uint64_t> cap_hint;
    // busy rounds the last call of a workload class (and budget octave) needed: where the
    // round chunks shrink
    std::map<std::array<uint64_t, 7>, uint32_t> round_hint;
    // workload classes whose last call in k_grow did not end there: their next `skip` calls
    // run the round kernels, then one tries k_grow again (tied errors are the integrand's, so
    // one call says little about the next); each failure in a row doubles the pause
    struct GrowPause {
        uint32_t skip = 0, pause = 0;
    };
    std::map<std::array<uint64_t, 7>, GrowPause> grow_pause;
    const Shape* trial = nullptr;
    std::vector<std::array<uint64_t, 6>> tuned_keys;
    vmx_generation generated{};  // of the last call (vmx_last_generation)
    // last result (for vmx_export_regions): gathered from device memory on demand
    int last_D = 0;
    uint64_t last_n = 0;
    std::function<void(double*, double*, double*, double*, int32_t*)> last_gather;
    // the no-alloc entry point: this device's scratch array (its device address, resolved
    // at context creation) and whether the current call runs on it
    char* scratch = nullptr;
    bool noalloc = false;
};


namespace vmxe {


struct VmxError : std::runtime_error {
    int code;
    VmxError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define HIP_CHECK(x)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (x);                                                                           \
        if (e_ != hipSuccess)                                                                          \
            throw VmxError(VMX_ERR_DEVICE, std::string(#x) + ": " + hipGetErrorString(e_));            \
    } while (0)

inline void* ensure(vmx_ctx::Buf& b, size_t bytes) {
    if (bytes == 0) bytes = 256;
    if (b.fixed) {  // carve from the fixed array: grow in place when b is its last carve
        if (b.bytes >= bytes) return b.p;
        vmx_ctx::Fixed& f = *b.fixed;
        const bool last = b.p && static_cast<char*>(b.p) + b.bytes == f.base + f.used;
        const size_t start = last ? size_t(static_cast<char*>(b.p) - f.base) : (f.used + 255) & ~size_t(255);
        if (start + bytes > f.cap)
            throw VmxError(VMX_ERR_CAPACITY, "problem needs more work memory than the no-alloc scratch holds (" +
                                                 std::to_string(f.cap >> 20) + " MiB)");
        b.p = f.base + start;
        b.bytes = bytes;
        f.used = start + bytes;
        return b.p;
    }
    if (b.bytes < bytes) {
        if (b.p) HIP_CHECK(hipFree(b.p));
        b.p = nullptr;
        b.bytes = 0;
        HIP_CHECK(hipMalloc(&b.p, bytes));
        b.bytes = bytes;
    }
    return b.p;
}

/* No-alloc calls: the arenas are carved anew from the start of the fixed array. */
inline void reset_fixed(vmx_ctx* ctx) {
    for (vmx_ctx::Buf* b : {&ctx->tree, &ctx->regs, &ctx->lists, &ctx->misc, &ctx->bins2})
        if (b->fixed) {
            b->fixed->used = 0;
            b->p = nullptr;
            b->bytes = 0;
        }
}

/* A batch whose (bin, footprint) pair total does not fit the 32-bit list offsets. */
inline void check_pair_total(uint64_t pairs) {
    if (pairs > vmx::MAX_PAIRS)
        throw VmxError(VMX_ERR_CAPACITY, "more (bin, region footprint) pairs than 32-bit list offsets hold: " +
                                             std::to_string(pairs));
}

inline void* ensure_pinned(vmx_ctx* ctx, size_t bytes) {
    if (ctx->pinned_bytes < bytes) {
        if (ctx->noalloc)
            throw VmxError(VMX_ERR_CAPACITY, "no-alloc call needs more pinned staging than the context set up");
        if (ctx->pinned) HIP_CHECK(hipHostFree(ctx->pinned));
        ctx->pinned = nullptr;
        ctx->pinned_bytes = 0;
        const size_t want = std::max<size_t>(bytes, 1 << 16);
        HIP_CHECK(hipHostMalloc(&ctx->pinned, want, hipHostMallocDefault));
        ctx->pinned_bytes = want;
    }
    return ctx->pinned;
}

/* Carves aligned sub-arrays out of one allocation. */
inline int ilog2(uint64_t x) {
    int r = 0;
    while (x > 1) {
        x >>= 1;
        ++r;
    }
    return r;
}

/* Sub-allocations of one buffer, 256-byte aligned; taking more than the buffer holds
   is a bug in the caller's size computation and throws. */
struct Carve {
    char* base;
    size_t used = 0, cap;
    explicit Carve(const vmx_ctx::Buf& b) : base(static_cast<char*>(b.p)), cap(b.bytes) {}
    template <typename X>
    X* take(size_t n) {
        used = (used + 255) & ~size_t(255);
        if (used + n * sizeof(X) > cap) throw VmxError(VMX_ERR_CAPACITY, "work buffer carved past its size");
        X* r = reinterpret_cast<X*>(base + used);
        used += n * sizeof(X);
        return r;
    }
};
struct Measure {
    size_t used = 0;
    template <typename X>
    void take(size_t n) {
        used = (used + 255) & ~size_t(255);
        used += n * sizeof(X);
    }
};

template <typename P>
struct ParamOf;
template <typename P>
struct F64Of;
template <typename T>
struct F64Of<vmx::Poly<T>> {
    using type = vmx::Poly<double>;
};
template <typename T>
struct F64Of<vmx::Blobs<T>> {
    using type = vmx::Blobs<double>;
};
template <typename T>
struct F64Of<vmx::Lobes5<T>> {
    using type = vmx::Lobes5<double>;
};
template <typename T>
struct ParamOf<vmx::Poly<T>> {
    using type = vmx_poly_params;
};
template <typename T>
struct ParamOf<vmx::Blobs<T>> {
    using type = vmx_blobs_params;
};
template <typename T>
struct ParamOf<vmx::Lobes5<T>> {
    using type = vmx_lobes5_params;
};
template <typename T, typename Inner, int DF, int RD>
struct ParamOf<vmx::Fubini<T, Inner, DF, RD>> {
    using type = vmx_fubini_params;
};

inline double ms_since(std::chrono::steady_clock::time_point t0) {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

/* One (scalar, D, family) batch through the device pipeline (pipeline.h). */
/* A caller-given region list (host memory, the layout vmx_export_regions writes):
   boxes n x D and node values n x 3^D, dim 0 fastest. */
struct GivenRegions {
    uint64_t n;
    const double *lo, *hi, *nodes;
};

struct JobIn {
    const vmx_problem* p;
    const void* params;
    void* bins;  // device pointer
    vmx_stats* stats;
    const GivenRegions* given = nullptr;  // set: skip generation, integrate over these regions
};

/* Training-pair mode of run_batch: stop after generation, report the node count and,
   if alloc hands back device arrays for that many rows, fill them. */
struct PairsReq {
    uint64_t count = 0;
    int kind = vmx::nn::TARGET_ENERGY;
    uint32_t stride = 1;
    std::function<void(uint64_t, uint16_t**, float**)> alloc;
};

constexpr int LEARN_MAX_DIM = 5;  // the fused network fits the expansion kernel's LDS up to here
constexpr int DEFER_K = 32;        // deferred rounds: about N / DEFER_K expansions per job and round

template <typename T, int D, typename P, typename Math>
void launch_expand(bool learn, const vmx::GenArgs<T>& g, const P* d_f, int par, uint32_t blocks, hipStream_t st) {
    const size_t pre_bytes = size_t(g.J + 1) * sizeof(uint32_t);  // the per-job candidate prefix
    if constexpr (std::is_same<T, float>::value && D <= LEARN_MAX_DIM) {
        if (learn) {
            vmx::k_expand_round<T, D, P, Math, true><<<blocks, vmx::GEN_THREADS, pre_bytes, st>>>(g, d_f, par);
            return;
        }
    }
    vmx::k_expand_round<T, D, P, Math, false><<<blocks, vmx::GEN_THREADS, pre_bytes, st>>>(g, d_f, par);
}

/* Rough instruction count of one evaluation in `dim` dims, for the choice of how regions
   are generated, from k_grow's time a step.  Infinite where nothing is known (a user's
   functor that does not state it): the rounds, whose time depends on it the least. */
template <typename P>
struct EvalWork {
    static double of(const P&, int) { return std::numeric_limits<double>::infinity(); }
};
template <typename T>
struct EvalWork<vmx::Poly<T>> {  // a loop per term and dim
    static double of(const vmx::Poly<T>& p, int dim) { return 30.0 + 16.0 * dim * p.nterms; }
};
template <typename T>
struct EvalWork<vmx::Blobs<T>> {  // FP64: the precise exp, sin and cos
    static double of(const vmx::Blobs<T>& p, int) {
        return sizeof(T) == 8 ? 20.0 + (p.wa != 0 ? 400.0 : 0.0) + 40.0 * p.nblobs : 40.0 + 13.0 * p.nblobs;
    }
};
template <typename T>
struct EvalWork<vmx::Lobes5<T>> {
    static double of(const vmx::Lobes5<T>&, int) { return 50.0; }
};
/* A wave runs to its longest series, log(64) / -log(decay) terms: 1, 4 and 20 us a sample at
   decay 0.3, 0.75 and 0.95. */
template <typename T>
struct EvalWork<vmx::Dyson<T>> {
    static double of(const vmx::Dyson<T>& p, int) { return 80.0 * std::max(1.0, 4.7 / -std::log(double(p.decay))); }
};
template <typename T, typename Inner, int DF, int RD>
struct EvalWork<vmx::Fubini<T, Inner, DF, RD>> {
    static double of(const vmx::Fubini<T, Inner, DF, RD>& p, int) {
        return double(p.mc) * (80.0 + EvalWork<Inner>::of(p.in, DF));
    }
};
/* ... in us on a lane: 8 cycles an instruction. */
template <int D, typename P>
double eval_us(const P& p) {
    return 0.0033 * EvalWork<P>::of(p, D);
}

/* k_grow's time for the splits of an integral of n regions, us: a step for each 256, which
   is issue-bound on one CU. */
template <typename T, int D>
double grow_us(bool learn, double n, double eval) {
    const double step = learn ? (D == 1 ? 7.0 : 15.0) : (D <= 2 ? 7.0 : (sizeof(T) == 8 ? 27.0 : 15.0));
    return n / 256.0 * (step + 1.3 * vmx::pow3(D - 1) * eval);
}
/* What the rounds and their selection cost more than k_grow without those steps, us: two
   launches a round, a round per level, more of both with many integrals, and the chip's
   time for the splits.  Fitted with the steps above to both generators over 2500 calls:
   polynomials of 1 to 12 terms, 1 to 64 static and 2 to 32 moving blobs, Fubini forms,
   learned priorities, 2 to 6144 regions, 1 to 300 integrals.  Where this rule takes k_grow
   it is at most 4 % behind the rounds, but for two of those calls (7 %); where it takes the
   rounds they are at most 30 % behind, beside the line (38 % in 1 dim with 32 samples a
   node).  FP64 in 3 dims spills (a child is 27 values in a lane): rounds from 100 to 300
   regions on, one integral. */
template <typename T, int D>
double rounds_us(bool learn, double n, double jobs, double splits) {
    const double base = learn ? 30.0 : (D == 3 && sizeof(T) == 8 ? 30.0 : 40.0);
    const double level = learn ? (D == 1 ? 15.0 : 23.0) : (D == 1 ? 30.0 : (D == 2 ? 19.0 : (sizeof(T) == 8 ? 0.0 : 12.0)));
    const double octave = learn ? 12.0 : (D == 1 ? 22.0 : (D == 2 ? 14.0 : 7.0));
    const double split = D == 1 ? 0.0018 : (D == 2 ? 0.0013 : 0.0021);
    return base + level * std::log2(n) + octave * std::log2(std::min(jobs, 64.0)) + split * splits;
}
constexpr double GROW_WAVE_US = 45.0;  // of each further wave of workgroups

/* Whether k_grow is built for a pipeline: a child of a split in the registers of one lane
   (D <= 3), with the learned priority the network beside it in LDS (D <= 2). */
template <int D>
constexpr bool grow_built(bool learn) {
    return D <= (learn ? 2 : 3);
}

/* The largest integral that k_grow is given: its measured range, and what its pool holds.
   Until N - 1 nodes are known none is dropped, so the pool holds every unsplit node, N / 2
   of them, and a step adds one for each split. */
template <typename T, int D>
constexpr uint32_t grow_limit(bool deepen) {
    using S = vmx::GrowShape<T, D, false>;
    const uint32_t pool = 2u * uint32_t(S::POOL - S::SPLITS * (deepen ? 2 : 1));
    return pool < 6144u ? pool : 6144u;
}

template <typename T, int D, typename P, typename Math>
void launch_grow(bool learn, const vmx::GenArgs<T>& g, const P* d_f, int32_t* leaf, int select, hipStream_t st) {
    if constexpr (std::is_same<T, float>::value && grow_built<D>(true) && !vmx::IsFubini<P>::value) {
        if (learn) {
            vmx::k_grow<T, D, P, Math, true><<<g.J, vmx::GROW_THREADS, 0, st>>>(g, d_f, leaf, select);
            return;
        }
    }
    if constexpr (grow_built<D>(false))
        vmx::k_grow<T, D, P, Math, false><<<g.J, vmx::GROW_THREADS, 0, st>>>(g, d_f, leaf, select);
}

using Instant = std::chrono::steady_clock::time_point;

/* One (scalar, D, family) batch through the device pipeline (pipeline.h).  left: the
   batch's start, where k_grow's workgroups have left it to the round kernels. */
template <typename T, int D, typename P, typename Math>
int run_batch(vmx_ctx* ctx, const std::vector<JobIn>& in, hipStream_t st, PairsReq* pairs_req = nullptr,
              const Instant* left = nullptr);

}  // namespace vmxe

#endif
