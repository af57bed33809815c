// Engine::download against a resident order that names particles outside the
// scene: a download of positions or velocities is refused (SPH_ERR_STATE) and
// writes nothing to the caller, a download of densities alone, which come in
// the sorted order, is not.  No entry point leaves such an order behind, so it
// is written into the engine's device memory here.  Exit status 0: as expected.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <string>
#include <vector>

#define private public
#include "../../fluid-simulation-3d_amd/csrc/sph_engine.h"
#undef private

#define REQUIRE(x)                                                        \
    do {                                                                  \
        if (!(x)) {                                                       \
            printf("line %d: %s (%s)\n", __LINE__, #x, err.c_str());      \
            return 1;                                                     \
        }                                                                 \
    } while (0)

int main()
{
    std::string err;
    const uint32_t n = 1000;
    sph_params p;
    sph_default_params(&p);
    std::vector<float> pos(4 * n), vel(4 * n), a(4 * n), b(4 * n), d(2 * n);
    const float box[3] = {4.0f, 4.0f, 4.0f};
    REQUIRE(sph_generate(SPH_INIT_CENTRED_BLOCK, 1, n, box, 0.1f, 0.002f, 0.0f, pos.data(), vel.data()) == SPH_OK);
    sph::Engine *e = nullptr;
    REQUIRE(sph::Engine::create({sph::SceneSpec{p, n, n}}, 0, 0, 1, &e, &err) == SPH_OK);
    REQUIRE(e->upload(0, pos.data(), vel.data(), &err) == SPH_OK);
    REQUIRE(e->update(1.0f / 360.0f, &err) == SPH_OK);
    REQUIRE(e->download(0, a.data(), b.data(), d.data(), &err) == SPH_OK);
    uint32_t good[2], bad[2] = {n, 0xffffffffu};
    for (int slot : {0, 517, 998}) {
        REQUIRE(hipMemcpy(good, e->d_.ids + slot, sizeof(good), hipMemcpyDeviceToHost) == hipSuccess);
        REQUIRE(hipMemcpy(e->d_.ids + slot, bad, sizeof(bad), hipMemcpyHostToDevice) == hipSuccess);
        a.assign(4 * n, -7.0f);
        b.assign(4 * n, -7.0f);
        REQUIRE(e->download(0, a.data(), nullptr, nullptr, &err) == SPH_ERR_STATE);
        REQUIRE(e->download(0, nullptr, b.data(), nullptr, &err) == SPH_ERR_STATE);
        REQUIRE(e->download(0, a.data(), b.data(), d.data(), &err) == SPH_ERR_STATE);
        REQUIRE(a == std::vector<float>(4 * n, -7.0f) && b == a);
        REQUIRE(e->download(0, nullptr, nullptr, d.data(), &err) == SPH_OK);
        REQUIRE(hipMemcpy(e->d_.ids + slot, good, sizeof(good), hipMemcpyHostToDevice) == hipSuccess);
        REQUIRE(e->download(0, a.data(), b.data(), d.data(), &err) == SPH_OK);
    }
    delete e;
    printf("order check ok\n");
    return 0;
}
