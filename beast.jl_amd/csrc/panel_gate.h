// Admission of factorisations whose panels' workgroups wait for one another.
#pragma once

#include <condition_variable>
#include <mutex>

namespace bh {

// A panel's workgroups exchange pivot candidates, so all of them have to be resident at once.
// One panel's always fit; panels of several factorisations, each on a stream of its own, could
// each hold a part of the device and wait for the rest.  A factorisation therefore holds the
// workgroups of its longest panel for as long as it runs, and begins only while all that are
// held fit the device together, in the order of arrival (no large one is passed over for ever).
// Kernels that wait for nobody may hold places as well: they end by themselves.
class PanelGate {
public:
    void enter(long long groups, long long capacity)
    {
        std::unique_lock<std::mutex> l(mu_);
        const long long ticket = next_++;
        cv_.wait(l, [&] { return ticket == serving_ && (held_ == 0 || held_ + groups <= capacity); });
        held_ += groups;
        ++serving_;
        cv_.notify_all();
    }
    void leave(long long groups)
    {
        std::lock_guard<std::mutex> l(mu_);
        held_ -= groups;
        cv_.notify_all();
    }

private:
    std::mutex mu_;
    std::condition_variable cv_;
    long long held_ = 0, next_ = 0, serving_ = 0;
};

// the places of one factorisation
class PanelPlaces {
public:
    PanelPlaces() = default;
    PanelPlaces(const PanelPlaces &) = delete;
    PanelPlaces &operator=(const PanelPlaces &) = delete;
    ~PanelPlaces() { if (gate_) gate_->leave(groups_); }
    void take(PanelGate &gate, long long groups, long long capacity)
    {
        gate.enter(groups, capacity);
        gate_ = &gate;
        groups_ = groups;
    }

private:
    PanelGate *gate_ = nullptr;
    long long groups_ = 0;
};

}  // namespace bh
