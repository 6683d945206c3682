// What the planner of the marching kernels answers, for tests on a machine without a device.
#include "../../pv_dec_original_amd/csrc/march_plans.hpp"

namespace {
int64_t searches = 0;
}

extern "C" {

// fields of MarchPlan and the price; 0: no plan, 1: the gathering kernel is cheaper, 2: marches
int probe_conv_plan(const pvnet_shape* s, int32_t cin, int32_t cout, int32_t* out, int32_t n, double* us) {
    MarchPlan p{};
    if (n != (int32_t)(sizeof(p) / 4) || !march_search(MarchKey{*s, cin, cout}, p, *us)) return 0;
    std::copy_n(reinterpret_cast<const int32_t*>(&p), n, out);
    return march_route(MarchKey{*s, cin, cout}, p) ? 2 : 1;
}

// fields of WgradMarch and the price; 0: no plan, 1: the tiled kernel is cheaper, 2: marches
int probe_wgrad_plan(const pvnet_shape* s, int32_t cin, int32_t cout, int32_t* out, int32_t n, double* us) {
    WgradMarch p{};
    if (n != (int32_t)(sizeof(p) / 4) || !wgrad_march_search(*s, cin, cout, p, *us)) return 0;
    std::copy_n(reinterpret_cast<const int32_t*>(&p), n, out);
    return wgrad_route(MarchKey{*s, cin, cout}, p) ? 2 : 1;
}

int probe_blocks_per_cu(int32_t lds, int32_t vgprs, int32_t waves) { return blocks_per_cu(lds, vgprs, waves); }

// searches of the kept convolution plans so far, after one more lookup; *same: the kept plan is the searched one
int64_t probe_kept(const pvnet_shape* s, int32_t cin, int32_t cout, int32_t* same) {
    const MarchKey key{*s, cin, cout};
    MarchPlan p{}, q{};
    const bool got = kept_plan<MarchPlan>(key, p, [](const MarchKey& k, MarchPlan& o) {
        searches++;
        return march_route(k, o);
    });
    *same = got == march_route(key, q) &&
            (!got || std::equal(reinterpret_cast<const int32_t*>(&p), reinterpret_cast<const int32_t*>(&p + 1), reinterpret_cast<const int32_t*>(&q)));
    return searches;
}
}
