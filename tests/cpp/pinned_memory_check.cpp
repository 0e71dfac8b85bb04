// Transfers of the library against its pinned slots, seen through this
// program's own hipHostMalloc, which the library binds to: it counts the calls
// and passes them on.
//
// usage: pinned_memory_check held
// held: two segmentations of a volume that goes through device buffers, in a
//       process where nothing else holds slots, allocate one set of slots.
#include "dxmc_pipelines.h"

#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

namespace {

int g_allocations = 0;

int failed(const char* what)
{
    std::fprintf(stderr, "%s: %s\n", what, dxg_last_error());
    return 1;
}

dxg_ct_segmentation threeMaterials()
{
    dxg_ct_segmentation t {};
    t.n_materials = 3;
    t.separators[0] = -500.0;
    t.separators[1] = 300.0;
    t.attenuation[0] = 0.15;
    t.attenuation[1] = 0.16;
    t.attenuation[2] = 0.19;
    t.slope = 0.16;
    t.offset = 0.16;
    return t;
}

std::vector<double> ctNumbers(std::size_t n)
{
    std::vector<double> hu(n);
    for (std::size_t i = 0; i < n; ++i)
        hu[i] = 1400.0 * std::sin(0.001 * static_cast<double>(i));
    return hu;
}

int held()
{
    const dxg_ct_segmentation t = threeMaterials();
    const std::size_t n = 500'000;
    const std::vector<double> hu = ctNumbers(n);
    std::vector<std::uint8_t> material(n);
    std::vector<double> density(n);
    for (int call = 0; call < 2; ++call)
        if (dxg_ct_segment(&t, hu.data(), n, material.data(), density.data()) != DXG_OK)
            return failed("dxg_ct_segment");
    std::printf("%d allocations\n", g_allocations);
    return g_allocations == 1 ? 0 : 2;
}

}  // namespace

extern "C" int hipHostMalloc(void** p, std::size_t bytes, unsigned flags)
{
    static const auto real = reinterpret_cast<int (*)(void**, std::size_t, unsigned)>(dlsym(RTLD_NEXT, "hipHostMalloc"));
    ++g_allocations;
    return real(p, bytes, flags);
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "held")
        return held();
    return 64;
}
