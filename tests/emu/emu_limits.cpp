// The library's limits and its transform engine on the CPU (the fiber stand-in for the HIP runtime).
// Test infrastructure.
//   emu_limits budget <grains> <steps> <seed> <gb> <ppg> <fp32> <aniso> [lds_budget] [ConvolutionMode]
//     one-grain launches under lds_budget against the same run without one: same bits, no launch above
//     the budget.  Without a budget given: the LDS that a grain's contour points (36 bytes each), its
//     squares (one byte each up to side 128) and 480 bytes take, for the network's neediest grain.  With a
//     Laplace mode, whose engine the budget decides, the fields may differ by rounding (1e-10).
//   emu_limits corrector <grains> <steps> <seed> <gb> <ppg> <sigma> <model> <pergrain>
//     an anisotropic run against the oracle (existence, boxes, fields to 1e-10) in which corrected grains
//     had contours longer than the corrector stages in LDS.
//   emu_limits engine
//     k_conv_fft, every form, against the oracle's convolution.
//   emu_limits workspace
//     device memory of Laplace contexts against Gaussian ones: more only where the FFT runs.
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

#define ggx ggx_engine  // the kernels once more, in a namespace of their own
#include "aniso.h"
#include "fft.h"
#undef ggx

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
    const int N = arg(2, 6), steps = arg(3, 2), seed = arg(4, 1001), gb = arg(5, 7), ppg = arg(6, 20), fp32 = arg(7, 0), aniso = arg(8, 0), cmode = arg(10, 2);
    int budget = arg(9, 0);
    ggx_network* net = nullptr;
    if (ggx_network_generate(N, (unsigned long long)seed, 0.0, &net)) return 2;
    const int ng = ggx_network_count(net);
    ggx_ctx* a = make_run(net, gb, ppg, fp32, aniso, cmode, GGX_CONV_AUTO, 0);
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
    ggx_ctx* b = make_run(net, gb, ppg, fp32, aniso, cmode, GGX_CONV_AUTO, budget);
    emu::g_lds_most = 0;
    int bad = 0;
    size_t at = 0;
    for (int t = 0; t < steps && !bad; ++t) {
        if (ggx_step(b, 1) || ggx_sync(b)) { printf("refused: %s\n", ggx_last_error(b)); bad = 1; break; }
        for (int g = 1; g <= ng; ++g, ++at) {
            const int c = ggx_get_phi(b, g, buf.data(), (int)buf.size());
            const std::vector<double>& want = phi[at];
            bool same = (size_t)std::max(0, c) == want.size();
            for (size_t k = 0; same && k < want.size(); ++k)
                same = cmode == 2 ? buf[k] == want[k] : fabs(buf[k] - want[k]) <= 1e-10;
            if (!same) {
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

static int corrector_check(int argc, char** argv) {
    auto arg = [&](int k, double d) { return argc > k ? atof(argv[k]) : d; };
    const int N = (int)arg(2, 6), steps = (int)arg(3, 3), gb = (int)arg(5, 9), ppg = (int)arg(6, 80), model = (int)arg(8, 1);
    ggx_network* net = nullptr;
    if (ggx_network_generate(N, (unsigned long long)arg(4, 15), arg(7, 0.0), &net)) return 2;
    const int ng = ggx_network_count(net);
    ggx_settings s;
    ggx_settings_default(&s);
    s.number_of_particles = ng;
    s.number_of_points_per_grain = ppg;
    s.number_of_timesteps = steps;
    s.analysis_timestep = 1;
    s.domain_border_size = gb;
    s.microstructure_gen_mode = 0;
    s.convolution_mode = 2;
    s.is_isotropic_network = 0;
    s.breakup_number = 0;
    s.research_mode = 0;
    s.use_mobility_model = model;
    s.triple_point_drag = 0.5;
    s.constant_sector_radius = 3;
    s.interpolating_sector_radius = 2;
    ggx_derived d;
    ggx_settings_derive(&s, &d);
    ggx_options o;
    ggx_options_default(&o);
    o.batching = arg(9, 0) != 0 ? GGX_BATCH_PERGRAIN : GGX_BATCH_FUSED;
    double bins[16];
    for (int b = 0; b < 16; ++b) bins[b] = 0.2 + 0.05 * b;
    ggx_ctx* ctx = nullptr;
    if (ggx_create(&s, &o, &ctx) || (model == 4 && ggx_set_mobility_bins(ctx, bins)) || ggx_load_network(ctx, net)) return 2;
    ggxo_params p;
    memset(&p, 0, sizeof p);
    p.real_domain_size = d.real_domain_size;
    p.grid_blowup = gb;
    p.convolution_mode = 2;
    p.dt = d.dt;
    p.analysis_timestep = 1;
    p.nthreads = 1;
    p.number_of_particles = ng;
    p.mobility_model = model;
    p.triple_point_drag = 0.5;
    p.constant_sector_radius = 3;
    p.interpolating_sector_radius = 2;
    for (int b = 0; b < 16; ++b) p.mobility_bins[b] = bins[b];
    void* oc = nullptr;
    ggxo_create(&p, ng, &oc);
    for (int i = 0; i < ng; ++i) {
        int id, nv;
        const double *xy, *q;
        ggx_network_grain(net, i, &id, &nv, &xy, &q);
        ggxo_add_grain(oc, id, nv, xy, q);
    }
    ggxo_init(oc);
    int bad = 0, longer = 0, shorter = 0;
    std::vector<double> a(1 << 18), b(1 << 18);
    for (int t = 0; t < steps; ++t) {
        if (t > 0)  // the contours this step's corrector reads
            for (int g = 1; g <= ng; ++g) {
                ggx_grain_info i;
                ggx_get_info(ctx, g, &i);
                if (i.present && i.exists && i.motion_regular) (i.contour_len > ggx_engine::kAnisoContourLds ? longer : shorter)++;
            }
        if (ggx_step(ctx, 1) || ggx_sync(ctx)) { printf("step failed: %s\n", ggx_last_error(ctx)); return 3; }
        ggxo_step(oc, t);
        double worst = 0.0;
        for (int g = 1; g <= ng; ++g) {
            ggx_grain_info gi;
            ggxo_grain_info oi;
            ggx_get_info(ctx, g, &gi);
            ggxo_get_info(oc, g, &oi);
            const bool ge = gi.present && gi.exists, oe = oi.present && oi.exists;
            if (ge != oe || (oe && (gi.xmin != oi.xmin || gi.xmax != oi.xmax || gi.ymin != oi.ymin || gi.ymax != oi.ymax))) {
                printf("step %d grain %d: existence or box\n", t, g);
                bad++;
                continue;
            }
            if (!oe) continue;
            const int c = ggx_get_phi(ctx, g, a.data(), (int)a.size());
            if (c != ggxo_grain_phi(oc, g, b.data())) { bad++; continue; }
            for (int k = 0; k < c; ++k) worst = std::max(worst, fabs(a[(size_t)k] - b[(size_t)k]));
        }
        printf("step %d: max|dphi| %.3e\n", t, worst);
        if (!(worst <= 1e-10)) bad++;
    }
    printf("corrected grains: %d with longer contours, %d with shorter ones\n", longer, shorter);
    if (!longer) bad++;
    ggx_destroy(ctx);
    ggxo_destroy(oc);
    ggx_network_free(net);
    printf(bad ? "LIMITS FAILED\n" : "LIMITS OK\n");
    return bad ? 1 : 0;
}

// One form of k_conv_fft over boxes of the given sides, random fields, every mode.  The bound: a stage of
// prime p sums p products in a row, which leaves about sqrt(p) / 2 units of relative rounding in the mean
// square, so four transforms leave 2 sqrt(sum of n's primes) of them; the table, the symbol and the two
// stored halves add 4 primes' worth, eight standard deviations cover the largest of 10^5 values, and the
// oracle's own rounding in FP64 doubles it.
template <class T, bool LDS>
static int engine_form(const char* name, const std::vector<int>& sides) {
    using C = typename ggx_engine::Cplx<T>::type;
    int nb = 1;
    std::vector<int> list;
    std::vector<ggx_engine::Box> box;
    std::vector<long long> off;
    long long total = 0;
    for (int n : sides) {
        list.push_back((int)list.size());
        box.push_back(ggx_engine::Box{0, 0, n, 0});
        off.push_back(total);
        total += (long long)n * n;
        nb = std::max(nb, n);
    }
    const int count = (int)sides.size(), grid = 3, R = 200;
    const double dt = 2.2e-5, unit = sizeof(T) == 8 ? 2 * 0x1p-53 : 0x1p-24;
    std::vector<T> src((size_t)total), dst((size_t)total);
    unsigned long long x = 99;
    for (auto& v : src) {
        x = x * 6364136223846793005ULL + 1442695040888963407ULL;
        v = (T)(((double)(x >> 11) / 9007199254740992.0 - 0.5) * 0.1);
    }
    std::vector<double2> tw((size_t)ggx_engine::tw_offset(nb + 1));
    hipLaunchKernelGGL(ggx_engine::k_fft_twiddles, dim3(nb), dim3(256), 0, nullptr, tw.data(), 1, nb);
    std::vector<C> work((size_t)grid * (size_t)ggx_engine::fft_slot(nb));
    int bad = 0;
    for (int mode = 0; mode <= 2; ++mode) {
        ggx_engine::FftSymbol sy;
        sy.mode = mode;
        sy.dt = dt;
        sy.nsq = (double)R * R;
        std::fill(dst.begin(), dst.end(), (T)NAN);
        hipLaunchKernelGGL((ggx_engine::k_conv_fft<T, LDS>), dim3(grid), dim3(256), (size_t)ggx_engine::fft_lds<T>(nb, LDS), nullptr,
                           (const int*)list.data(), &count, (const ggx_engine::Box*)box.data(), (const long long*)off.data(),
                           (const T*)src.data(), dst.data(), (const double2*)tw.data(), sy, nb, work.data());
        for (int b = 0; b < count; ++b) {
            const int n = sides[(size_t)b];
            std::vector<double> in((size_t)n * n), ref((size_t)n * n);
            double sq = 0, worst = 0;
            for (size_t k = 0; k < in.size(); ++k) {
                in[k] = (double)src[(size_t)off[(size_t)b] + k];
                sq += in[k] * in[k];
            }
            ggxo_convolve(n, mode, dt, R, in.data(), ref.data());
            bool finite = true;
            for (size_t k = 0; k < in.size(); ++k) {
                const double v = (double)dst[(size_t)off[(size_t)b] + k];
                finite = finite && std::isfinite(v);
                worst = std::max(worst, fabs(v - ref[k]));
            }
            int primes = 4;
            for (int m = n, p = 2; m > 1; ++p)
                while (m % p == 0) { primes += p; m /= p; }
            const double bound = 8 * unit * 2 * sqrt((double)primes) * sqrt(sq / (double)in.size());
            printf("%s mode %d n %d: max|diff| %.3e of %.3e\n", name, mode, n, worst, bound);
            if (!finite || !(worst <= bound)) bad++;
        }
    }
    return bad;
}

static int engine_check() {
    const std::vector<int> lds = {1, 2, 3, 5, 16, 17, 31, 40, 64, 97, 127, 128}, wide = {3, 61, 129, 130, 200, 256};
    int bad = engine_form<float, true>("FP32, LDS", lds) + engine_form<float, false>("FP32, slots", wide) +
              engine_form<double, true>("FP64, LDS", lds) + engine_form<double, false>("FP64, slots", wide);
    printf(bad ? "LIMITS FAILED\n" : "LIMITS OK\n");
    return bad ? 1 : 0;
}

static int workspace_check() {
    ggx_network* net = nullptr;
    if (ggx_network_generate(6, 1001, 0.0, &net)) return 2;
    auto bytes = [&](int fp32, int cmode, int engine) {
        const size_t from = g_device_bytes;
        ggx_destroy(make_run(net, 7, 20, fp32, 0, cmode, engine, 0));
        return (long long)(g_device_bytes - from);
    };
    const long long plain64 = bytes(0, 2, GGX_CONV_AUTO), plain32 = bytes(1, 2, GGX_CONV_AUTO);
    const long long more[] = {bytes(0, 0, GGX_CONV_AUTO) - plain64, bytes(0, 2, GGX_CONV_FFT) - plain64, bytes(1, 0, GGX_CONV_AUTO) - plain32};
    printf("beyond the Gaussian's: FP64 Laplace %lld, FP64 forced %lld, FP32 Laplace %lld\n", more[0], more[1], more[2]);
    const bool ok = more[0] == 0 && more[1] == 0 && more[2] > 0;
    ggx_network_free(net);
    printf(ok ? "LIMITS OK\n" : "LIMITS FAILED\n");
    return ok ? 0 : 1;
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
    if (!strcmp(what, "corrector")) return corrector_check(argc, argv);
    if (!strcmp(what, "engine")) return engine_check();
    if (!strcmp(what, "workspace")) return workspace_check();
    if (!strcmp(what, "batch")) return batch_check(argc, argv);
    printf("unknown check %s\n", what);
    return 2;
}
