// Host bookkeeping of the server's batched steps (serve.hip), free of device
// calls so that it compiles and runs on the CPU too.
#pragma once
#include <vector>

namespace lbm3 {

// One storage type's requests.  A request's esotwist parity, iteration and
// pending condition follow on the device from the ticks since its first one
// (MultiDesc), so the tick counts this type's launches and nothing else: when
// another type's upload or launch fails, the server's step fails, but what did
// step here stays in step with the populations it moved on.
struct Batch {
    int tick = 0;
    bool stale = true;   // requests came or went since the upload
};

// Advances the requests with steps left by one: upload(requests) where the
// device's tables are stale, launch(tick), then moved(request) for each.
// A request that has all its steps (its retirement waits for a server step that
// succeeds) takes no further one.
template <class R, class Upload, class Launch, class Moved>
int step_batch(Batch &b, const std::vector<R *> &active, Upload upload, Launch launch, Moved moved)
{
    std::vector<R *> run;
    for (R *r : active)
        if (r->done < r->steps) run.push_back(r);
    if (run.size() != active.size()) b.stale = true;
    if (run.empty()) return 0;
    if (b.stale) {
        if (const int rc = upload(run)) return rc;
        b.stale = false;
    }
    if (const int rc = launch((int)run.size(), b.tick)) return rc;
    ++b.tick;
    for (R *r : run) {
        ++r->done;
        moved(r);
    }
    return 0;
}

} // namespace lbm3
