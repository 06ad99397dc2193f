// nl_turns.h -- turns of the handles of one device whose launches' workgroups wait for each other (plain C++: a test drives it with events of its own).
//
// A launch of nl_layers.h needs every compute unit of its device.  Two of them, of two handles whose threads decode at the same time, or one beside another
// launch whose workgroups wait for each other (nl_block.h, nl_group.h, nl_tp.h, nl_persist.h), could each hold units that the other waits for until a bounded
// poll gives up.  So where a device has several handles with such launches, and one of them takes the whole device, they take turns, on the device: each waits
// for the event behind the last one of another handle.  Otherwise they launch at will, side by side, with no event and no lock but a shared one of the
// device's own.
//
// Turns cost what used to overlap.  Two handles decoding at once, twelve layers, us a token of either, launch plans side by side / layer launches in turns: 1536 columns
// Q8_0 189 / 253, Q4_K 192 / 248; 768 Q4_K 139 / 217; one of them alone 339 / 251, 317 / 246, 266 / 216.  A plan chosen by what the neighbours do would
// change a handle's last bits with them; NL_LAYERS=0 gives such a server the plans that overlap.
//
// join is for a caller under a lock that captures of launch graphs hold too: it records events on the streams of other handles, which must not be in a capture.  For the
// same reason a capture on a listed handle's stream holds `capture()`: no event of it is waited for meanwhile.
#pragma once
#include <algorithm>
#include <mutex>
#include <shared_mutex>
#include <vector>

namespace nl {

template <class H> class Turns {
    struct Member { H *h; bool whole; };
    std::shared_mutex mu;
    std::vector<Member> members;
    H *last = nullptr;                       // whose launch was the last one in a turn
    bool shared() const { return members.size() > 1 && std::any_of(members.begin(), members.end(), [](const Member &m) { return m.whole; }); }

public:
    // launch() -> status; wait(other): h's stream waits for other's event; record(): h's event behind its stream
    template <class L, class W, class R> int run(H *h, L launch, W wait, R record) {
        {
            std::shared_lock<std::shared_mutex> lk(mu);
            if (!shared()) return launch();
        }
        std::unique_lock<std::shared_mutex> lk(mu);
        if (last && last != h)
            if (const int rc = wait(last)) return rc;
        const int rc = launch();
        if (const int rr = record()) return rc ? rc : rr;
        last = h;
        return rc;
    }
    // a newcomer; where it makes the launches take turns, it waits for whatever the others launched at will
    template <class W, class R> int join(H *h, bool whole, W wait, R record) {
        std::unique_lock<std::shared_mutex> lk(mu);
        members.push_back({h, whole});
        if (shared())
            for (size_t i = 0; i + 1 < members.size(); i++) {
                int rc = record(members[i].h);
                if (!rc) rc = wait(members[i].h);
                if (rc) { members.pop_back(); return rc; }
            }
        return 0;
    }
    // h no longer takes the whole device
    void retire(H *h) {
        std::unique_lock<std::shared_mutex> lk(mu);
        for (Member &m : members)
            if (m.h == h) m.whole = false;
    }
    void leave(H *h) {
        std::unique_lock<std::shared_mutex> lk(mu);
        members.erase(std::remove_if(members.begin(), members.end(), [h](const Member &m) { return m.h == h; }), members.end());
        if (last == h) last = nullptr;
    }
    std::unique_lock<std::shared_mutex> capture() {
        {
            std::shared_lock<std::shared_mutex> lk(mu);
            if (!shared()) return {};        // (only a join could change that, and its caller's lock is the capture's)
        }
        return std::unique_lock<std::shared_mutex>(mu);
    }
};

}  // namespace nl
