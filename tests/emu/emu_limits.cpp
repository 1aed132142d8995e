// The library's limits and its transform engine on the CPU (the fiber stand-in for the HIP runtime).
// Test infrastructure.
//   emu_limits budget <grains> <steps> <seed> <gb> <ppg> <fp32> <aniso> [lds_budget]
//     one-grain launches under lds_budget against the same run without one: same bits, no launch above
//     the budget.  Without a budget given: the LDS that a grain's contour points (36 bytes each), its
//     squares (one byte each up to side 128) and 480 bytes take, for the network's neediest grain.
//   emu_limits batch <count> <lowest side> <highest side> <max_n> <mode>
//     ggx_convolve_boxes against the oracle, with the work spread over the dies: none has less than half
//     of the average (workgroup barriers, which only a workgroup with a strip meets).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <vector>

#include <hip/hip_runtime.h>

#include "ggx.h"
#include "ggx_oracle.h"

static ggx_ctx* make_run(ggx_network* net, int gb, int ppg, int fp32, int aniso, int cmode, int engine, int budget) {
    ggx_settings s;
    ggx_settings_default(&s);
    s.number_of_particles = ggx_network_count(net);
    s.number_of_points_per_grain = ppg;
    s.number_of_timesteps = 10;
    s.analysis_timestep = 1;
    s.domain_border_size = gb;
    s.microstructure_gen_mode = 0;
    s.convolution_mode = cmode;
    s.is_isotropic_network = aniso ? 0 : 1;
    s.breakup_number = 0;
    if (aniso) {
        s.research_mode = 0;
        s.use_mobility_model = 1;
        s.triple_point_drag = 0.5;
        s.constant_sector_radius = 3;
        s.interpolating_sector_radius = 2;
    }
    ggx_options o;
    ggx_options_default(&o);
    o.precision = fp32 ? GGX_PREC_FP32 : GGX_PREC_FP64;
    o.batching = GGX_BATCH_PERGRAIN;
    o.conv_engine = engine;
    o.lds_budget = budget;
    ggx_ctx* ctx = nullptr;
    if (ggx_create(&s, &o, &ctx)) { printf("create failed\n"); exit(2); }
    if (ggx_load_network(ctx, net)) { printf("load failed: %s\n", ggx_last_error(ctx)); exit(2); }
    return ctx;
}

static int budget_check(int argc, char** argv) {
    auto arg = [&](int k, int d) { return argc > k ? atoi(argv[k]) : d; };
    const int N = arg(2, 6), steps = arg(3, 2), seed = arg(4, 1001), gb = arg(5, 7), ppg = arg(6, 20), fp32 = arg(7, 0), aniso = arg(8, 0);
    int budget = arg(9, 0);
    ggx_network* net = nullptr;
    if (ggx_network_generate(N, (unsigned long long)seed, 0.0, &net)) return 2;
    const int ng = ggx_network_count(net);
    ggx_ctx* a = make_run(net, gb, ppg, fp32, aniso, 2, GGX_CONV_AUTO, 0);
    std::vector<std::vector<double>> phi;   // every grain's field after every step
    std::set<int> sides;
    std::vector<double> buf(1 << 20);
    for (int t = 0; t < steps; ++t) {
        for (int g = 1; g <= ng; ++g) {
            ggx_grain_info i;
            ggx_get_info(a, g, &i);
            if (i.present && i.exists) sides.insert(i.xmax - i.xmin);
        }
        if (ggx_step(a, 1) || ggx_sync(a)) { printf("reference run failed: %s\n", ggx_last_error(a)); return 2; }
        for (int g = 1; g <= ng; ++g) {
            const int c = ggx_get_phi(a, g, buf.data(), (int)buf.size());
            phi.emplace_back(buf.begin(), buf.begin() + std::max(0, c));
        }
    }
    if (budget == 0)
        for (int n : sides) budget = std::max(budget, (8 * n + 64) * 36 + (n <= 128 ? (n + 1) * (n + 1) : 0) + 480);
    printf("sides %d .. %d, budget %d\n", *sides.begin(), *sides.rbegin(), budget);
    ggx_ctx* b = make_run(net, gb, ppg, fp32, aniso, 2, GGX_CONV_AUTO, budget);
    emu::g_lds_most = 0;
    int bad = 0;
    size_t at = 0;
    for (int t = 0; t < steps && !bad; ++t) {
        if (ggx_step(b, 1) || ggx_sync(b)) { printf("refused: %s\n", ggx_last_error(b)); bad = 1; break; }
        for (int g = 1; g <= ng; ++g, ++at) {
            const int c = ggx_get_phi(b, g, buf.data(), (int)buf.size());
            const std::vector<double>& want = phi[at];
            if ((size_t)std::max(0, c) != want.size() || (c > 0 && memcmp(buf.data(), want.data(), want.size() * 8))) {
                printf("step %d grain %d differs\n", t, g);
                bad++;
            }
        }
    }
    printf("largest launch %zu bytes of LDS\n", emu::g_lds_most);
    if (emu::g_lds_most > (size_t)budget) { printf("a launch is above the budget\n"); bad++; }
    ggx_destroy(a);
    ggx_destroy(b);
    ggx_network_free(net);
    printf(bad ? "LIMITS FAILED\n" : "LIMITS OK\n");
    return bad ? 1 : 0;
}

static int batch_check(int argc, char** argv) {
    auto arg = [&](int k, int d) { return argc > k ? atoi(argv[k]) : d; };
    const int count = arg(2, 64), lo = arg(3, 3), hi = arg(4, 16), max_n = arg(5, 128), mode = arg(6, 2), R = 200;
    const double dt = 2.2e-5;
    std::vector<int32_t> n;
    std::vector<int64_t> off;
    int64_t total = 0;
    for (int b = 0; b < count; ++b) {
        n.push_back(lo + (7 * b) % (hi - lo + 1));
        off.push_back(total);
        total += (int64_t)n[b] * n[b];
    }
    std::vector<double> in((size_t)total), out((size_t)total, 0.0), ref;
    unsigned long long x = 12345;
    for (auto& v : in) {
        x = x * 6364136223846793005ULL + 1442695040888963407ULL;
        v = ((double)(x >> 11) / 9007199254740992.0 - 0.5) * 0.1;
    }
    std::fill(emu::g_die_barriers, emu::g_die_barriers + 8, 0ull);
    const int rc = ggx_convolve_boxes(count, n.data(), off.data(), in.data(), out.data(), max_n, mode, dt, R, nullptr);
    int bad = rc != GGX_OK;
    double worst = 0.0;
    for (int b = 0; b < count && !bad; ++b) {
        ref.assign((size_t)n[b] * n[b], 0.0);
        ggxo_convolve(n[b], mode, dt, R, in.data() + off[b], ref.data());
        for (size_t k = 0; k < ref.size(); ++k) worst = std::max(worst, fabs(out[(size_t)off[b] + k] - ref[k]));
    }
    unsigned long long sum = 0, least = ~0ull;
    for (unsigned long long v : emu::g_die_barriers) { sum += v; least = std::min(least, v); }
    printf("rc %d, max|diff| %.3e, barriers %llu, of the idlest die %llu\n", rc, worst, sum, least);
    if (!(worst <= 1e-12) || 16 * least < sum) bad++;
    printf(bad ? "LIMITS FAILED\n" : "LIMITS OK\n");
    return bad ? 1 : 0;
}

int main(int argc, char** argv) {
    setvbuf(stdout, nullptr, _IOLBF, 0);
    const char* what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "budget")) return budget_check(argc, argv);
    if (!strcmp(what, "batch")) return batch_check(argc, argv);
    printf("unknown check %s\n", what);
    return 2;
}
