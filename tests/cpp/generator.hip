/*
 * How the regions of a user functor are generated: by parallel rounds unless the functor
 * states what an evaluation takes (evaluation_work()), then by one workgroup where that is
 * faster.  Prints one line per case, "name workgroup_steps rounds"; the last lines compare
 * the bins of the two functors, equal but for the statement.  Compiled by hipcc for gfx950
 * and linked to the in-tree libviltrum_amd.so.
 */
#include <cstdio>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

#include "viltrum_amd/device.hpp"

namespace {

namespace vi = viltrum_amd;

struct Bump {
    float a;
    __host__ __device__ float operator()(const float* x) const {
        const float u = x[0] - 0.4f, v = x[1] - 0.6f;
        return expf(-a * (u * u + v * v)) + (x[0] + x[1] > 1.1f ? 0.5f : 0.f);
    }
};

struct StatedBump : Bump {
    double work;
    double evaluation_work() const { return work; }
};

template <typename F>
std::vector<float> bins(const char* name, const F& f, int regions) {
    const vi::Integrand g = vi::device_integrand<2>(f);
    vi::Context& ctx = vi::Context::thread_default();
    vmx_problem p = vi::integrator_crespo2021(regions - 1, 3, 5).base();
    p.scalar = VMX_F32;
    p.bin_dims = 2;
    p.res[0] = 21;
    p.res[1] = 18;
    p.lo[0] = p.lo[1] = 0.0;
    p.hi[0] = p.hi[1] = 1.0;
    std::vector<float> out(21 * 18, 0.f);
    ctx.check(vmx_integrate(ctx.get(), &p, &g.desc, out.data(), nullptr));
    vmx_generation gen;
    ctx.check(vmx_last_generation(ctx.get(), &gen));
    std::printf("%s %llu %llu\n", name, (unsigned long long)gen.workgroup_steps, (unsigned long long)gen.rounds);
    return out;
}

StatedBump stated(double work) {
    StatedBump f;
    f.a = 20.f;
    f.work = work;
    return f;
}

}  // namespace

int main() {
    int same = 1;
    for (int n : {300, 4000}) {
        const std::string size = std::to_string(n);
        const auto a = bins(("unstated_" + size).c_str(), Bump{20.f}, n);
        const auto b = bins(("cheap_" + size).c_str(), stated(40), n);
        const auto c = bins(("dear_" + size).c_str(), stated(18000), n);
        const auto d = bins(("nonsense_" + size).c_str(), stated(-1), n);
        same &= int(a == b && a == c && a == d);
    }
    std::printf("same %d 0\n", same);
    return 0;
}
