// Times of launches and the rules that compare them (lbm_plan.h).
#include "lbm_plan.h"

#include <algorithm>

#include "../../include/lbm_hip.h"

namespace lbm {

double step_us(int storage, const Geom &g, bool program) {
    const double elem = storage == LBM_STORE_F64 ? 8 : (storage == LBM_STORE_F32 ? 4 : 2);
    double mb = 18e-6 * g.lx * g.pitch * elem;
    const bool small = mb < 36;
    mb *= 1 + 0.33 * std::min(std::max((mb - 240) / 90, 0.0), 1.0);  // out of the last-level cache
    if (!program) {
        if (storage == LBM_STORE_F64) return 2.65 + 0.13 * mb;
        if (storage == LBM_STORE_F32) return small ? 3.3 + 0.085 * mb : 1.9 + 0.13 * mb;
        return 3.3 + 0.134 * mb;
    }
    // waves that lie in more rows touch more lines
    const double cut = std::min(64.0 / g.ly, 1.0);
    if (storage == LBM_STORE_F64) return 4.3 + 0.126 * mb * (1 + 0.43 * cut);
    if (storage == LBM_STORE_F32) return (small ? 4.4 + 0.094 * mb * (1 + 0.4 * cut) : 3.5 + 0.128 * mb * (1 + 0.4 * cut));
    return 4.3 + 0.153 * mb * (1 + 0.5 * cut);
}

double sweep2_us(int storage, const Geom &g, bool program, bool outlet, const SweepShape &sh, int rows, int resident) {
    const uint32_t waves = sh.threads / 64;
    const uint64_t ranges = ((uint64_t)g.lx + rows - 1) / rows, places = (uint64_t)resident;
    double row, head = 3.3;  // a row, and the rows that a range costs beside its own
    if (storage == LBM_STORE_F64) {
        row = waves <= 12 ? 3.9 : 4.5;
        if (waves == 5 && 3 * ranges > 2 * places) row = 5.8;
        if (!program) row *= 0.7;
    } else if (sh.v == 1 && sh.ntiles == 1) {
        row = 3.7;
        head = 2.6;
        if (waves == 5 && 6 * ranges > 5 * places) row = 4.9;
        if (waves == 10 && 3 * ranges > 2 * places) row = 4.9;
        if (!program) row *= 0.65;
        else if (rows == 1 && 20 * ranges <= 11 * places) row *= 0.87;  // half the blocks a CU holds
    } else if (outlet) {
        row = waves <= 12 ? (sh.ntiles == 1 ? 3.7 : 4.05) : (sh.ntiles == 1 ? 4.2 : 4.6);
        head = 3.9;
    } else if (program) {
        row = (waves <= 12 ? 3.75 : 4.4) * (sh.ntiles == 1 ? 1 : 1.07);
        head = 2.4;
    } else {
        row = waves <= 12 ? (sh.ntiles == 1 ? 2.3 : 2.55) : (sh.ntiles == 1 ? 3.2 : 3.4);
        if (waves > 12) head = 2.5;
    }
    const uint64_t rounds = (ranges + places - 1) / places;
    return (double)rounds * (rows + head) * row;
}

bool two_steps_pay(int storage, const Geom &g, bool program, bool outlet, const SweepShape &sh, int rows, int resident,
                   double extra_us) {
    if (rows < 1 || resident < 1) return false;
    return sweep2_us(storage, g, program, outlet, sh, rows, resident) + extra_us < 2 * step_us(storage, g, program);
}

namespace {
// a launch, each further round of blocks, each step, each step and wave of a SIMD, each MB that the
// blocks load; waves a SIMD holds
struct TileModel {
    double launch, round, step, wave, mb;
    uint32_t simd;
};
TileModel tile_model(int storage, bool program, bool pressure) {
    if (storage == LBM_STORE_F64)
        return pressure ? TileModel{6.78, 3.39, 1.18, 0.184, 0.118, 2}
                        : (program ? TileModel{5.42, 1.41, 0.714, 0.354, 0.162, 3}
                                   : TileModel{3.75, 1.0, 0.464, 0.328, 0.127, 3});
    return pressure ? TileModel{5.92, 2.6, 1.105, 0.094, 0.079, 3}
                    : (program ? TileModel{5.61, 2.29, 0.715, 0.149, 0.125, 5}
                               : TileModel{3.78, 1.78, 0.504, 0.105, 0.108, 5});
}
double launch_us(const TileModel &m, uint32_t tiles, uint32_t rx, uint32_t ry, int k, size_t elem, uint32_t cus) {
    const uint32_t waves = (rx * ry + 63) / 64;
    const uint32_t fit = std::max(1u, m.simd / ((waves + 3) / 4));  // blocks a CU holds
    const uint32_t rounds = (tiles + cus * fit - 1) / (cus * fit);
    const uint32_t per_cu = std::min(fit, (tiles + cus - 1) / cus);
    return m.launch + m.round * (rounds - 1) + rounds * k * (m.step + m.wave * ((waves * per_cu + 3) / 4)) +
           m.mb * 9e-6 * tiles * rx * ry * elem;
}
// tiles are taken where they gain more than the times may be off (with the fix, FP16 370x487: 5.0 us a step
// by the model, 5.6 measured)
constexpr double tile_margin(bool pressure) { return pressure ? 0.92 : 0.94; }
// nodes beyond a tile on both sides together, for k steps
uint32_t tile_halo_x(int k, bool pressure) { return 2 * (k - 1 + (pressure ? 2 : 0)); }
uint32_t tile_halo_y(int k) { return 2 * (k - 1); }
size_t elem_of(int storage) { return storage == LBM_STORE_F64 ? 8 : (storage == LBM_STORE_F32 ? 4 : 2); }
}  // namespace

double tile_us(int storage, const Geom &g, bool program, bool pressure, int cus, const TileShape &sh, int k) {
    const uint32_t tiles = ((g.lx + sh.tx - 1) / sh.tx) * ((g.ly + sh.ty - 1) / sh.ty);
    return launch_us(tile_model(storage, program, pressure), tiles, sh.tx + tile_halo_x(k, pressure),
                     sh.ty + tile_halo_y(k), k, elem_of(storage), (uint32_t)std::max(cus, 1));
}

TileShape pick_tile(int storage, const Geom &g, bool program, bool pressure, int cus_, double other_us) {
    TileShape best;
    const bool f64 = storage == LBM_STORE_F64;
    if (g.N > (f64 ? 1u << 18 : 3u << 16)) return best;
    const uint32_t cus = (uint32_t)std::max(cus_, 1);
    const uint32_t tmax = (uint32_t)tile_threads(elem_of(storage), pressure);
    const uint32_t wmax = f64 ? (pressure ? 8 : 12) : (pressure ? 12 : 24);
    double least = 1e30;
    for (int K = 1; K <= 8; K++) {
        // what a node depends on may cross the seam of the fix only once
        if (pressure && (uint32_t)K + 4 > g.lx) break;
        auto step = [&](uint32_t waves) { return 0.35 + (f64 ? 0.4 : 0.12) * ((waves + 3) / 4); };
        if ((3.3 + K * step(1)) / K >= least) continue;
        const uint32_t hx = tile_halo_x(K, pressure), hy = tile_halo_y(K);
        for (uint32_t ty = 1; ty <= g.ly; ty++) {
            const uint32_t ny = (g.ly + ty - 1) / ty;
            ty = ny == 1 ? g.ly : (g.ly - 1) / (ny - 1);  // the widest that makes as many tiles
            const uint32_t ry = ty + hy;
            if (ry > 64 || ry * (hx + 1) > tmax) break;
            const uint32_t rx_most = std::min(g.lx + hx, tmax / ry);
            // the most rows for each number of waves a block
            for (uint32_t waves = (rx_most * ry + 63) / 64; waves >= 1; waves--) {
                const uint32_t rx = std::min(64 * waves / ry, rx_most);
                if (rx <= hx) break;
                waves = (rx * ry + 63) / 64;
                const uint32_t tiles = (g.lx + rx - hx - 1) / (rx - hx) * ny;
                if (tiles > 4096) break;
                const uint32_t fit = std::max(1u, wmax / waves);
                const uint32_t rounds = (tiles + cus * fit - 1) / (cus * fit);
                const uint32_t per_cu = std::min(fit, (tiles + cus - 1) / cus);
                const double t = rounds * (3.3 + K * step(waves * per_cu)) / K;
                if (t < least) {
                    least = t;
                    best.K = K;
                    best.tx = rx - hx;
                    best.ty = ty;
                }
            }
        }
    }
    if (best.K < 2 || !tile_pays(storage, g, program, pressure, cus_, best, best.K, other_us)) best = TileShape{};
    return best;
}

bool tile_pays(int storage, const Geom &g, bool program, bool pressure, int cus, const TileShape &sh, int k,
               double other_us) {
    return tile_us(storage, g, program, pressure, cus, sh, k) < tile_margin(pressure) * k * other_us;
}

bool tile_run_pays(int storage, const Geom &g, bool program, bool pressure, int cus, const TileShape &sh, int64_t steps,
                   double other_us) {
    if (steps < sh.K) return tile_pays(storage, g, program, pressure, cus, sh, (int)steps, other_us);
    const int64_t n = steps / sh.K;
    const int r = (int)(steps % sh.K);
    if (r == 0 || n > 16) return true;
    double t = (double)n * tile_us(storage, g, program, pressure, cus, sh, sh.K);
    if (r > 1 && tile_pays(storage, g, program, pressure, cus, sh, r, other_us))
        t += tile_us(storage, g, program, pressure, cus, sh, r);
    else
        t += r * other_us + 9e-6 * g.N * elem_of(storage) * (program ? 0.25 : 0.65);
    return t < 0.96 * (double)steps * other_us;
}

}  // namespace lbm
