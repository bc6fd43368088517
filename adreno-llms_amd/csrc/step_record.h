// When a decoder's step is recorded and when a recording is replayed (mi_decoder_step).  Host code without HIP: the
// launches, the recording and the replay are an Api's.
#pragma once
#include <cstddef>

namespace mi {

// The circumstances of a step: its launches have the same arguments whenever these are the same.
struct StepKey {
    const void* stream = nullptr;
    const void* workspace = nullptr;
    int gemv_mode = -1, splits = -1, weights = -1;         // weights: the version of what the registry holds for the decoder
    bool operator==(const StepKey& o) const {
        return stream == o.stream && workspace == o.workspace && gemv_mode == o.gemv_mode && splits == o.splits && weights == o.weights;
    }
};

// How a recording went: kept; a launch of it failed (the step itself is at fault, or will be reported so); the runtime
// would not record.
enum class Recorded { kYes, kLaunchFailed, kRefused };

template <class Exec>
class StepRecordings {
public:
    static constexpr size_t kMost = 8;

    // One step: 1 = enqueued, 0 = not.  The second of two steps in a row under the same circumstances is recorded, later
    // ones are replays.  Nothing runs while a step is recorded: whatever goes wrong there, the step is enqueued plainly.
    // Api: int enqueue(); Recorded record(Exec*); int replay(Exec); bool gone(const StepKey&), whether the key's stream is no
    // more; void drain(), waits for the step's stream; void drop(Exec).
    template <class Api>
    int step(Api& api, const StepKey& now) {
        const bool again = last_ == now;
        last_ = now;
        if (refused_ || !again) return api.enqueue();
        for (size_t i = 0; i < count_; ++i)
            if (held_[i].key == now) return api.replay(held_[i].exec);
        if (count_ >= kMost && !make_room(api, now)) return api.enqueue();
        Exec exec{};
        const Recorded r = api.record(&exec);
        if (r != Recorded::kYes) {
            refused_ = refused_ || r == Recorded::kRefused;
            return api.enqueue();
        }
        held_[count_].key = now;
        held_[count_++].exec = exec;
        return api.replay(exec);
    }

    size_t count() const { return count_; }
    Exec exec(size_t i) const { return held_[i].exec; }

private:
    struct Recording { StepKey key; Exec exec{}; };

    // Drops what no step can ask for again and cannot be running any more: recordings for streams that are gone, and those
    // of this step's stream, once it is drained, for weights that the registry no longer holds.  (Of another stream's last
    // replay nothing is known; those go when that stream does, or asks for room itself.)
    template <class Api>
    bool make_room(Api& api, const StepKey& now) {
        size_t kept = 0;
        bool drained = false;
        for (size_t i = 0; i < count_; ++i) {
            const StepKey& k = held_[i].key;
            const bool outdated = k.stream == now.stream && k.workspace == now.workspace && k.weights != now.weights;
            if (outdated && !drained) {
                api.drain();
                drained = true;
            }
            if (outdated || api.gone(k)) api.drop(held_[i].exec);
            else held_[kept++] = held_[i];
        }
        count_ = kept;
        return count_ < kMost;
    }

    Recording held_[kMost];
    size_t count_ = 0;
    StepKey last_;
    bool refused_ = false;                                 // the runtime would not record: plain steps from then on
};

}  // namespace mi
