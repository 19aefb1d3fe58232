// fork.hpp -- independent launches of one stage side by side on side streams.
//
// begin() forks from the caller's stream, next() names the stream of the next
// launch (the caller's first, then the side streams in turn), end() joins
// every side stream that got a launch.  Whatever fails, a launch is ordered
// behind begin() and what follows end() on the caller's stream behind it: a
// launch whose side stream could not be forked goes to the caller's stream,
// and a side stream that cannot be joined is waited for on the host.  failed()
// says that something did.
//
// Runtime: record(event, stream), wait(stream, event) and finish(stream), true
// on success.
#pragma once

namespace hmvm {

template <int N, typename Runtime, typename Stream, typename Event> class Fork {
public:
    Fork(Runtime rt, Stream st, const Stream (&side)[N], Event fork, const Event (&join)[N])
        : rt_(rt), st_(st), side_(side), fork_(fork), join_(join) {}

    // launches: how many calls of next() follow
    void begin(int launches) {
        turn_ = 0;
        on_ = false;
        for (bool& u : used_) u = false;
        if (launches > 1) on_ = check(rt_.record(fork_, st_));
    }
    Stream next() {
        const int i = turn_++;
        if (i == 0 || !on_) return st_;
        const int k = (i - 1) % N;
        if (!used_[k]) {
            // on_ goes too: after a failure nothing more leaves the caller's stream
            if (!(on_ = check(rt_.wait(side_[k], fork_)))) return st_;
            used_[k] = true;
        }
        return side_[k];
    }
    void end() {
        for (int k = 0; k < N; ++k)
            if (used_[k] && !(check(rt_.record(join_[k], side_[k])) && check(rt_.wait(st_, join_[k]))))
                (void)rt_.finish(side_[k]);
    }
    bool failed() const { return failed_; }

private:
    bool check(bool ok) {
        failed_ = failed_ || !ok;
        return ok;
    }
    Runtime rt_;
    Stream st_;
    const Stream (&side_)[N];
    Event fork_;
    const Event (&join_)[N];
    int turn_ = 0;
    bool on_ = false, used_[N] = {}, failed_ = false;
};

} // namespace hmvm
