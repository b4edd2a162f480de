// rv_poll.h -- control flow of a wait for words that another workgroup publishes, free of device
// intrinsics (constexpr functions compile for the device and for the host alike), so that its end
// is tested on the CPU.
#pragma once

namespace rv {

// A reader's polls: spent() is asked after every poll that found its words missing, and is true
// once the limit is passed or failed() says that another workgroup has given up (looked at every
// 64th poll).
struct SpinBudget {
    int limit;
    int spins = 0;
    template <class Failed>
    constexpr bool spent(Failed failed) {
        return (++spins & 63) == 0 && (spins > limit || failed());
    }
};

// Waits until unset() is false, reload() reading the words again; a far reader polls one word with
// last_unset() first.  Once give_up() is true (the budget's end) neither loop goes on: false.  (The
// words are read once more on the way out: leaving before it costs the device code a copy of their
// registers at every poll, 2 % of a sweep over a 64^3 Helmholtz factor.)
template <class Unset, class LastUnset, class Reload, class GiveUp>
constexpr bool wait_words(bool near, Unset unset, LastUnset last_unset, Reload reload, GiveUp give_up) {
    bool over = false;
    while (!over && unset()) {
        if (!near)
            while (!over && last_unset()) over = give_up();
        over = over || give_up();
        reload();
    }
    return !over;
}

}  // namespace rv
