// Transfers of the library against its pinned slots, seen through this
// program's own hipHostMalloc and hipMalloc, which the library binds to: they
// count the calls and pass them on.
//
// usage: pinned_memory_check held | segment | upload | refused
// held: two segmentations that go through device buffers (the densities replace
//       the CT numbers), in a process where nothing else holds slots, allocate
//       one set of slots.
// segment: host arrays of 393,216 voxels go through slots, fewer through three
//          device buffers.
// refused: with pinned memory refused, scores, doses and a segmentation equal
//          those with it.
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
bool g_refuse = false;

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

// A water cube with scores in it.
int scoredCube(dxg_world** w, std::uint64_t edge)
{
    const std::uint64_t dims[3] = { edge, edge, edge };
    const double spacing[3] = { 0.1, 0.1, 0.1 }, fraction[2] = { 0.111894, 0.888106 }, energy = 60.0, one = 1.0;
    const std::int32_t z[2] = { 1, 8 };
    const std::size_t n = edge * edge * edge;
    const std::vector<double> density(n, 1.0);
    const std::vector<std::uint8_t> material(n, 0);
    const dxg_material water { z, fraction, 2 };
    if (dxg_world_create(w, 1) != DXG_OK || dxg_grid_set_data(*w, dims, density.data(), material.data(), &water, 1) != DXG_OK
        || dxg_grid_set_spacing(*w, spacing) != DXG_OK || dxg_world_build(*w) != DXG_OK)
        return failed("world");
    const dxg_exposure exposure { { 0.05, 0.05, -20.0 }, { 1, 0, 0, 0, 1, 0 }, { 0.1, 0.1 }, 1.0, 0, -1, 100'000 };
    const dxg_spectrum spectrum { &energy, &one, 1 };
    const dxg_beam beam { &exposure, 1, &spectrum, 1, nullptr, 0, 0.0 };
    return dxg_transport_run(*w, &beam, nullptr, 0, 5) == DXG_OK ? 0 : failed("dxg_transport_run");
}

struct Results {
    std::vector<double> e, e2, dose, variance, density;
    std::vector<std::uint64_t> events, dose_events;
    std::vector<std::uint8_t> material;
    explicit Results(std::size_t n)
        : e(n), e2(n), dose(n), variance(n), density(n), events(n), dose_events(n), material(n)
    {
    }
    bool operator==(const Results&) const = default;
    bool get(const dxg_world* w)
    {
        const dxg_ct_segmentation t = threeMaterials();
        const std::vector<double> hu = ctNumbers(e.size());
        return dxg_read_energy_scores(w, e.data(), e2.data(), events.data()) == DXG_OK
            && dxg_read_dose_scores(w, dose.data(), variance.data(), dose_events.data()) == DXG_OK
            && dxg_ct_segment(&t, hu.data(), hu.size(), material.data(), density.data()) == DXG_OK;
    }
};

int refused()
{
    constexpr std::uint64_t edge[2] = { 10, 90 };   // one chunk, several
    dxg_world* w[2] = {};
    std::vector<Results> without, with;
    for (int i = 0; i < 2; ++i) {
        if (scoredCube(&w[i], edge[i]))
            return 1;
        without.emplace_back(edge[i] * edge[i] * edge[i]);
    }
    with = without;
    g_refuse = true;   // first, while no set is idle
    for (int i = 0; i < 2; ++i)
        if (!without[i].get(w[i]))
            return failed("refused");
    std::printf("%d calls refused\n", g_allocations);
    if (g_allocations < 5)   // two reads a world and a segmentation
        return 2;
    g_refuse = false;
    for (int i = 0; i < 2; ++i) {
        if (!with[i].get(w[i]))
            return failed("given");
        if (!(with[i] == without[i]))
            return 3;
        std::uint64_t sum = 0;
        for (std::uint64_t k : with[i].events)
            sum += k;
        if (sum == 0)
            return 4;
        dxg_world_destroy(w[i]);
    }
    return 0;
}

}  // namespace

extern "C" int hipHostMalloc(void** p, std::size_t bytes, unsigned flags)
{
    static const auto real = reinterpret_cast<int (*)(void**, std::size_t, unsigned)>(dlsym(RTLD_NEXT, "hipHostMalloc"));
    ++g_allocations;
    if (g_refuse)
        return 2;   // hipErrorOutOfMemory
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
    if (what == "refused")
        return refused();
    return 64;
}
