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

}  // namespace lbm
