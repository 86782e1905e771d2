// Times of launches and the rules that compare them (lbm_plan.h).
#include "lbm_plan.h"

#include <algorithm>

#include "../../include/lbm_hip.h"

namespace lbm {

double step_us(int storage, const Geom &g, bool program) {
    const double elem = storage == LBM_STORE_F64 ? 8 : (storage == LBM_STORE_F32 ? 4 : 2);
    const double mb = 18 * (double)g.lx * g.pitch * elem * 1e-6;
    if (!program) return 3.3 + mb * (storage == LBM_STORE_F64 ? 0.12 : (storage == LBM_STORE_F32 ? 0.11 : 0.13));
    if (storage == LBM_STORE_F32) return 4.4 + mb * (mb < 36 ? 0.1 : 0.122);
    return 4.5 + mb * (storage == LBM_STORE_F64 ? 0.127 : 0.155);
}

double sweep2_us(int storage, const Geom &g, bool program, const SweepShape &sh, int rows, int resident) {
    const uint32_t waves = sh.threads / 64;
    const uint64_t ranges = ((uint64_t)g.lx + rows - 1) / rows;
    double row, head = 3.3;  // a row, and the rows that a range costs beside its own
    if (storage == LBM_STORE_F64) {
        row = waves <= 12 ? 3.9 : 4.5;
        if (waves == 5 && 3 * ranges > 2 * (uint64_t)resident) row = 5.8;
        if (!program) row *= 0.7;
    } else {
        if (sh.v == 1 && sh.ntiles == 1) {
            row = 3.7;
            head = 2.6;
            if (waves == 5 && 6 * ranges > 5 * (uint64_t)resident) row = 4.9;
            if (waves == 10 && 3 * ranges > 2 * (uint64_t)resident) row = 4.9;
        } else {
            row = waves <= 12 ? 4.2 : (sh.ntiles == 1 ? 4.65 : 5.1);
        }
        if (!program) row *= 0.65;
    }
    const uint64_t rounds = (ranges + resident - 1) / resident;
    return (double)rounds * (rows + head) * row;
}

bool two_steps_pay(int storage, const Geom &g, bool program, const SweepShape &sh, int rows, int resident,
                   double extra_us) {
    if (rows < 1 || resident < 1) return false;
    return sweep2_us(storage, g, program, sh, rows, resident) + extra_us < 0.97 * 2 * step_us(storage, g, program);
}

namespace {
// a launch, each further round of blocks, each step, each step and wave of a SIMD; waves a SIMD holds
struct TileModel {
    double launch, round, step, wave;
    uint32_t simd;
};
TileModel tile_model(int storage, bool program, bool pressure) {
    if (storage == LBM_STORE_F64)
        return pressure ? TileModel{5.9, 3.4, 1.22, 0.44, 2}
                        : (program ? TileModel{6.05, 2.5, 0.53, 0.585, 3} : TileModel{3.9, 3.0, 0.4, 0.465, 3});
    return pressure ? TileModel{6.0, 4.3, 1.09, 0.14, 3}
                    : (program ? TileModel{6.45, 3.7, 0.665, 0.152, 5} : TileModel{4.4, 3.0, 0.2, 0.213, 5});
}
double launch_us(const TileModel &m, uint32_t tiles, uint32_t waves, int k, uint32_t cus) {
    const uint32_t fit = std::max(1u, m.simd / ((waves + 3) / 4));  // blocks a CU holds
    const uint32_t rounds = (tiles + cus * fit - 1) / (cus * fit);
    const uint32_t per_cu = std::min(fit, (tiles + cus - 1) / cus);
    return m.launch + m.round * (rounds - 1) + rounds * k * (m.step + m.wave * ((waves * per_cu + 3) / 4));
}
// tiles are taken where they gain more than the times above may be off
constexpr double kTileMargin = 0.94;
// nodes beyond a tile on both sides together, for k steps
uint32_t tile_halo_x(int k, bool pressure) { return 2 * (k - 1 + (pressure ? 2 : 0)); }
uint32_t tile_halo_y(int k) { return 2 * (k - 1); }
}  // namespace

double tile_us(int storage, const Geom &g, bool program, bool pressure, int cus, const TileShape &sh, int k) {
    const uint32_t tiles = ((g.lx + sh.tx - 1) / sh.tx) * ((g.ly + sh.ty - 1) / sh.ty);
    const uint32_t waves = ((sh.tx + tile_halo_x(k, pressure)) * (sh.ty + tile_halo_y(k)) + 63) / 64;
    return launch_us(tile_model(storage, program, pressure), tiles, waves, k, (uint32_t)std::max(cus, 1));
}

TileShape pick_tile(int storage, const Geom &g, bool program, bool pressure, int cus) {
    TileShape best;
    if (g.N > (storage == LBM_STORE_F64 ? 1u << 18 : 3u << 16)) return best;
    const TileModel m = tile_model(storage, program, pressure);
    const uint32_t tmax = (uint32_t)tile_threads(storage == LBM_STORE_F64 ? 8 : 4, pressure);
    double least = kTileMargin * step_us(storage, g, program);  // us a step
    for (int K = 2; K <= 8; K++) {
        // what a node depends on may cross the seam of the fix only once
        if (pressure && (uint32_t)K + 4 > g.lx) break;
        if ((m.launch + K * (m.step + m.wave)) / K >= least) continue;  // (one wave a SIMD)
        const uint32_t hx = tile_halo_x(K, pressure), hy = tile_halo_y(K);
        for (uint32_t ty = std::min(g.ly, 64 - hy); ty >= 1; ty--) {
            const uint32_t ny = (g.ly + ty - 1) / ty;
            ty = (g.ly + ny - 1) / ny;  // the narrowest that makes as many tiles
            // blocks of whole waves on every SIMD
            for (uint32_t waves = 4; waves * 64 <= tmax; waves += 4) {
                const uint32_t rx = waves * 64 / (ty + hy);
                if (rx <= hx) continue;
                const uint32_t nx = (g.lx + rx - hx - 1) / (rx - hx), tx = (g.lx + nx - 1) / nx;
                if (nx * ny > 4096) continue;
                const double t = launch_us(m, nx * ny, ((tx + hx) * (ty + hy) + 63) / 64, K, (uint32_t)std::max(cus, 1)) / K;
                if (t < least) {
                    least = t;
                    best.K = K;
                    best.tx = tx;
                    best.ty = ty;
                }
                if (nx == 1) break;
            }
        }
    }
    return best;
}

bool tile_pays(int storage, const Geom &g, bool program, bool pressure, int cus, const TileShape &sh, int k) {
    return tile_us(storage, g, program, pressure, cus, sh, k) < kTileMargin * k * step_us(storage, g, program);
}

}  // namespace lbm
