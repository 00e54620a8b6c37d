// Host bookkeeping of the persistent one-column step, apart from the runtime it runs on (Rt), so that it can be checked
// without a GPU.
#pragma once
#include <map>

namespace sp {

// The error word of the persistent step lies in pinned memory and is set by blocks that give up, possibly while other
// blocks of the same launch are still running and will set it again.  True once per failed launch: the word is cleared
// only after everything that may still set it has ended (wait).
template <class Wait>
bool take_error(volatile unsigned *word, Wait &&wait) {
    if (!word || *word == 0) return false;
    wait();
    *word = 0;
    return true;
}

// Order of the persistent launches of one device.  Two such kernels must not run at once (each needs every CU for one of
// its blocks), so a launch waits for the one before it where that went to another stream.  Engines that share a stream
// are ordered by it: as long as all launches go to one stream nothing is recorded or waited for.  With several, every
// launch leaves an event on its own stream, right behind the kernel, and the next launch on another stream waits for that
// event alone, not for what was queued after it.  A launch that is being captured is neither ordered nor remembered: its
// replays are the caller's.
//   Rt::Stream, Rt::Event, capturing(stream), sync(stream), record(event, stream), wait(stream, event)
template <class Rt>
struct PersistentOrder {
    std::map<typename Rt::Stream, int> users;      // engines that launch on each stream
    typename Rt::Stream last{};                    // the last launch's stream,
    bool any = false, marked = false;              // whether it may still run, and whether ev stands behind it
    typename Rt::Event ev{};

    void join(typename Rt::Stream s) { ++users[s]; }
    // The engine stops launching on s, which has been waited for.
    void leave(typename Rt::Stream s) {
        auto it = users.find(s);
        if (it != users.end() && --it->second == 0) users.erase(it);
        if (any && last == s) any = false;
    }
    void before(Rt &rt, typename Rt::Stream s) {
        if (!any || last == s || rt.capturing(s)) return;
        if (marked) rt.wait(s, ev);
        else if (!rt.capturing(last)) rt.sync(last);      // launched while its stream was the only one: once
    }
    void after(Rt &rt, typename Rt::Stream s) {
        const bool several = users.size() > 1;
        if (several && rt.capturing(s)) return;
        marked = several;
        if (several) rt.record(ev, s);
        any = true;
        last = s;
    }
};

}  // namespace sp
