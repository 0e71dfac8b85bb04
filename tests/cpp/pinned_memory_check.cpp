// Transfers of the library against its pinned slots, seen through this
// program's own hipHostMalloc and hipMalloc, which the library binds to: they
// count the calls and pass them on.
//
// usage: pinned_memory_check held | segment | upload
// held: two segmentations that go through device buffers (the densities replace
//       the CT numbers), in a process where nothing else holds slots, allocate
//       one set of slots.
// segment: host arrays of 393,216 voxels go through slots, fewer through three
//          device buffers.
// upload: the dose table's host arrays take slots from 44 MiB on.
#include "dxmc_pipelines.h"

#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

namespace {

int g_allocations = 0, g_device_allocations = 0;

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
    std::vector<double> hu = ctNumbers(n);
    std::vector<std::uint8_t> material(n);
    for (int call = 0; call < 2; ++call)
        if (dxg_ct_segment(&t, hu.data(), n, material.data(), hu.data()) != DXG_OK)
            return failed("dxg_ct_segment");
    std::printf("%d allocations\n", g_allocations);
    return g_allocations == 1 ? 0 : 2;
}

int segment()
{
    const dxg_ct_segmentation t = threeMaterials();
    const std::size_t most = 393'216;
    const std::vector<double> hu = ctNumbers(most);
    std::vector<std::uint8_t> material(most);
    std::vector<double> density(most);
    for (std::size_t n : { most - 1, most }) {
        if (dxg_ct_segment(&t, hu.data(), n, material.data(), density.data()) != DXG_OK)
            return failed("dxg_ct_segment");
        std::printf("%zu voxels: %d pinned, %d device allocations so far\n", n, g_allocations, g_device_allocations);
        if (g_allocations != (n < most ? 0 : 1) || g_device_allocations != 3)
            return 2;
    }
    return 0;
}

int upload()
{
    const std::size_t most = (std::size_t(44) << 20) / sizeof(double);
    const std::vector<double> values(most, 1.0);
    const std::vector<std::uint8_t> organ(most, 3);
    const double spacing[3] = { 0.1, 0.1, 0.1 };
    dxg_organ_dose rows[256];
    for (std::size_t n : { most - 1, most }) {
        if (dxg_organ_dose_table(organ.data(), values.data(), values.data(), n, spacing, rows) != DXG_OK)
            return failed("dxg_organ_dose_table");
        std::printf("%zu voxels: %d pinned allocations so far\n", n, g_allocations);
        if (g_allocations != (n < most ? 0 : 1) || rows[3].n_voxels != n)
            return 2;
    }
    return 0;
}

}  // namespace

extern "C" int hipHostMalloc(void** p, std::size_t bytes, unsigned flags)
{
    static const auto real = reinterpret_cast<int (*)(void**, std::size_t, unsigned)>(dlsym(RTLD_NEXT, "hipHostMalloc"));
    ++g_allocations;
    return real(p, bytes, flags);
}

extern "C" int hipMalloc(void** p, std::size_t bytes)
{
    static const auto real = reinterpret_cast<int (*)(void**, std::size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
    ++g_device_allocations;
    return real(p, bytes);
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "held")
        return held();
    if (what == "segment")
        return segment();
    if (what == "upload")
        return upload();
    return 64;
}
