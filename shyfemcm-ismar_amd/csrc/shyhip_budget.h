// shyhip_budget.h -- the compute units that one-launch solves of this process
// may hold at once, per device.
//
// Counted in whole parts of a unit: kUnitParts is a multiple of every number
// of workgroups that fit one unit (1 .. 8 of 256 or more work-items), so what
// a solve takes and gives back is exact in any order, and an idle device has
// its whole budget.
#ifndef SHYHIP_BUDGET_H
#define SHYHIP_BUDGET_H

#include <condition_variable>
#include <mutex>
#include <unordered_map>

namespace shy {

constexpr long kUnitParts = 840;

// parts that nwg workgroups hold, per_unit of them to a unit
constexpr long unit_parts(int nwg, int per_unit) { return (nwg * kUnitParts + per_unit - 1) / per_unit; }

// the budget of a device: 7/8 of its units, some are left to the rest of the step
constexpr long unit_budget(int units) { return units * (kUnitParts / 8 * 7); }

class UnitBudget {
public:
    // waits until parts more fit into budget (parts <= budget)
    void take(int dev, long parts, long budget) {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return used_[dev] + parts <= budget; });
        used_[dev] += parts;
    }
    void give(int dev, long parts) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            used_[dev] -= parts;
        }
        cv_.notify_all();
    }

private:
    std::mutex mu_;
    std::condition_variable cv_;
    std::unordered_map<int, long> used_;
};

}  // namespace shy

#endif
