// How much of the waiting frames one progress step of the server uploads ahead (host only).
#pragma once

#include <cstddef>

// At most two frames a step. Copies from pinned memory return at once and are limited by the events
// behind them, to two groups queued. A copy from pageable memory holds the host until it has ended, so
// that no event is ever found pending: without a limit of its own one step copied up to a batch's bytes (64
// MB) before it looked at arrivals and finished rounds again.
constexpr int kServeAheadPerStep = 2;

struct AheadStep
{
    size_t most; // arena bytes that uploaded frames may hold while they wait
    int left = kServeAheadPerStep;
    explicit AheadStep( size_t bytes ) : most( bytes ) {}
    // A frame of `bytes` may be uploaded when `held` bytes are; pending( ): a group before the last is still
    // in the queue.
    template <class F>
    bool take( size_t held, size_t bytes, F&& pending )
    {
        if ( left == 0 || held + bytes > most || pending() )
            return false;
        left--;
        return true;
    }
};
