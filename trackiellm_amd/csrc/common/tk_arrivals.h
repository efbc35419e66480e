/*
 * tk_arrivals.h — for whom a batching scheduler waits before it starts a job.
 *
 * A job of all callers' requests costs little more than a job of one, so the first request of a burst waits a moment for the others.  Whom it waits for:
 *   a caller whose request is not in yet, who has not been waited for in vain (an idle one: it costs one wait, not one per job) — until it, or another one that the same
 *   wait was for, comes after all: a burst that is late altogether is still one —, for whom two waits in a row were not in vain without its ever being there beside
 *   another one (handles that one thread uses in turn), and
 *   whose next request can be due — it was last served as long ago as three quarters of the time that it took before its last request, or will have been when the
 *   wait is over.  (A caller that was served a millisecond ago and comes every 33 is not waited for; one that comes back at once is.)
 * Times are microseconds on any steady clock.  Not thread-safe: the scheduler's lock covers it.
 */
#ifndef TK_ARRIVALS_H
#define TK_ARRIVALS_H

#include <stdint.h>

#include <map>

class TkArrivals {
public:
    explicit TkArrivals(int64_t wait_us) : wait_(wait_us) {}
    int64_t wait_us() const { return wait_; }
    int add() { callers_[next_] = Caller(); return next_++; }
    void remove(int id) { callers_.erase(id); }
    void submitted(int id, int64_t now) {
        Caller* c = find(id);
        if (!c) return;
        if (c->queued == 0 && c->served >= 0) c->pause = now - c->served;
        bool others = false;
        for (auto& e : callers_)
            if (&e.second != c && e.second.queued > 0) {
                others = true;
                e.second.apart = 0;
            }
        if (others) c->apart = 0;
        c->queued++;
        const int64_t missed = c->missed;
        for (auto& e : callers_)
            if (missed >= 0 && e.second.missed == missed) e.second.missed = -1;
    }
    void served(int id, int64_t now) {
        Caller* c = find(id);
        if (!c) return;
        c->queued--;
        c->served = now;
    }
    /* callers that a wait which began at `from` is for */
    int awaited(int64_t from) const {
        int n = 0;
        for (const auto& e : callers_) n += awaits(e.second, from) ? 1 : 0;
        return n;
    }
    void waited_in_vain(int64_t from) {
        for (auto& e : callers_)
            if (awaits(e.second, from)) {
                e.second.missed = from;
                e.second.apart++;
            }
    }

private:
    struct Caller {
        int queued = 0;
        int64_t missed = -1; /* the wait that was in vain */
        int apart = 0;       /* waits in vain since it was last there with another one */
        int64_t served = -1, pause = 0; /* when; from then to its next request, the last time */
    };
    bool awaits(const Caller& c, int64_t from) const { return c.queued == 0 && c.missed < 0 && c.apart < 2 && (c.served < 0 || c.served + c.pause / 4 * 3 <= from + wait_); }
    Caller* find(int id) {
        auto it = callers_.find(id);
        return it == callers_.end() ? nullptr : &it->second;
    }
    std::map<int, Caller> callers_;
    int next_ = 0;
    int64_t wait_;
};

#endif
