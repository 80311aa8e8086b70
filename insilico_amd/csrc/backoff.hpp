// How long to keep from launches that wait for one another after one of them
// gave up: its blocks could not all be on the chip (another process on the
// GPU, a long kernel on another stream), and what was in the way is likely
// still there.  A give-up costs the whole bound of a wait, about half a second,
// so the pause doubles from FIRST uses to MOST while they go on, and shrinks by
// half with every launch that ends well.
#pragma once

namespace ins {

struct Backoff {
    static constexpr int FIRST = 16, MOST = 4096;
    int pause = 0;   // length of the last pause
    int left = 0;    // uses left of it

    // whether this use goes without
    bool skip()
    {
        if (left == 0) return false;
        left--;
        return true;
    }
    void gave_up()
    {
        pause = pause == 0 ? FIRST : (pause < MOST ? 2 * pause : MOST);
        left = pause;
    }
    void ended_well() { pause /= 2; }
};

}  // namespace ins
