// Autotuner: for every requested volume side, times each fused volume pass (xy with projection,
// y, zy with data consistency) with both tile sizes on this device, xy and zy inside the
// positivity loop's own pass sequence (ctdm_time_loop; each pass reads what the previous one wrote),
// and keeps the faster choice (for y and zy, 8 only when clearly faster) in the context
// (used by every later launch of that side, including graph captures made afterwards); then the radix plan of the
// y pass and the pencils per workgroup of the gridding pass. The xy and y passes walk the z planes forward: the
// zy pass between two xy passes walks all planes at once, and the y pass runs once per volume, so that either
// direction takes the same time (volumes of 64^3 to 256^3 with 1 and 10 iterations: within 0.7 %, the timings' own
// spread). An explicit call re-times every side; a reconstruction asking for
// tuning only times sides not tuned yet. The choices are also kept per (device architecture, side) for
// the rest of the process, so contexts created later start from them. The other passes keep one radix
// plan per length (fft_dev.hpp).
#include <cstdio>
#include <mutex>
#include <sstream>

#include "internal.hpp"

namespace ctdm {

namespace {
// Choices made by the autotuner in this process, per (device architecture, volume side).
std::mutex g_tuned_mu;
std::map<std::pair<std::string, int>, Tune> g_tuned;
}  // namespace

Tune& Ctx::tuning(int n)
{
    auto it = tune.find(n);
    if (it != tune.end()) return it->second;
    Tune t;
    {
        std::lock_guard<std::mutex> lk(g_tuned_mu);
        auto g = g_tuned.find({arch, n});
        if (g != g_tuned.end()) t = g->second;
    }
    return tune.emplace(n, t).first->second;
}

std::string autotune(Ctx& c, const int* sizes, int nsizes, bool force)
{
    CTDM_REQUIRE(sizes || nsizes == 0, "autotune: null sizes");
    CTDM_REQUIRE(!c.capturing, "autotune during capture");
    std::ostringstream rep;
    static const char* names[3] = {"x+proj", "y", "z+dc"};
    constexpr int kIters = 4;
    for (int i = 0; i < nsizes; ++i) {
        const int V = sizes[i];
        Tune& t = c.tuning(V);
        if (t.tuned && !force) continue;
        for (int k = 0; k < 3; ++k) {
            double m[2] = {0, 0}, bytes[3] = {0, 0, 0};
            for (int b = 0; b < 2; ++b) {  // this pass at 8 / 16 pencils, the others at their current choice
                t.pencils[k] = b ? 16 : 8;
                double ms[3];
                time_loop(c, V, kIters, ms, bytes, k == 1 ? TIME_Y : TIME_XY_ZY);
                m[b] = ms[k];
            }
            t.ms[k][0] = m[0];
            t.ms[k][1] = m[1];
            // 8 y pencils write 64-byte halves of 128-byte lines, which costs more inside a replayed
            // reconstruction than in these short timings, and the zy pass's two tiles lie within the
            // timing's spread at the sides where both fill the device (128^3: 14.3 and 14.7 us). These
            // take 8 only on a clear margin.
            const double margin = k == 0 ? 1.0 : 0.97;
            t.pencils[k] = m[0] < margin * m[1] ? 8 : 16;
            char line[200];
            std::snprintf(line, sizeof line, "V=%d %-6s B=8 %.4f ms  B=16 %.4f ms  -> B=%d (%.0f GB/s)\n", V,
                          names[k], m[0], m[1], t.pencils[k], bytes[k] / (1e6 * std::min(m[0], m[1])));
            rep << line;
        }
        t.rev[0] = t.rev[1] = 0;
        char line[240];
        std::snprintf(line, sizeof line, "V=%d sweep  -> fwd\n", V);
        rep << line;
        // Radix plan of the y pass: the alternative factorisation is kept when its slowest of three timings leads
        // the base plan's fastest by 10 %. It rounds differently, so the choice must not hang on the timing's own
        // spread (a few per cent of the few microseconds a small volume's pass takes), or two tunings of one side would
        // give volumes that differ in the last bits; and the pass runs once per reconstruction.
        for (int r = 0; r < 6; ++r) {
            t.yplan = r & 1;
            double ms[3], bytes[3];
            time_loop(c, V, 4 * kIters, ms, bytes, TIME_Y);
            if (r < 2 || (t.yplan == 0 ? ms[1] < t.yplan_ms[0] : ms[1] > t.yplan_ms[1]))
                t.yplan_ms[t.yplan] = ms[1];
        }
        t.yplan = t.yplan_ms[1] < 0.9 * t.yplan_ms[0] ? 1 : 0;
        std::snprintf(line, sizeof line, "V=%d y plan  base %.4f ms  alternative %.4f ms -> %s\n", V, t.yplan_ms[0],
                      t.yplan_ms[1], t.yplan ? "alternative" : "base");
        rep << line;
        // Gridding pass: 8 or 16 pencils per workgroup for 60 angles (16 only when at least 3 % faster: the
        // staging of every angle's samples makes its workgroups twice as large in LDS).
        for (int b = 0; b < 2; ++b) t.grid_ms[b] = time_grid(c, V, b ? 16 : 8, 60, 5);
        t.pencils[3] = t.grid_ms[1] < 0.97 * t.grid_ms[0] ? 16 : 8;
        std::snprintf(line, sizeof line, "V=%d grid   B=8 %.4f ms  B=16 %.4f ms  -> B=%d\n", V, t.grid_ms[0],
                      t.grid_ms[1], t.pencils[3]);
        rep << line;
        t.tuned = true;
        ++c.tune_epoch;
        std::lock_guard<std::mutex> lk(g_tuned_mu);
        g_tuned[{c.arch, V}] = t;
    }
    return rep.str();
}

}  // namespace ctdm
