// Admission of resident team launches: the members of a team wait for each other on the device, so all of them
// have to run at once.
#pragma once

#include <condition_variable>
#include <mutex>

namespace pp {

// The workgroups of the team launches that run on one device. A launch enters when its workgroups fit beside
// those already inside, in the order of asking (a large launch is not passed for ever by small ones),
// and leaves when its kernels have ended. `need` is at most `capacity`.
class TeamGate {
public:
    void enter(int need, int capacity) {
        std::unique_lock<std::mutex> lock(m);
        const unsigned ticket = next++;
        cv.wait(lock, [&] { return ticket == serving && used + need <= capacity; });
        ++serving;
        used += need;
        cv.notify_all();
    }
    void leave(int need) {
        {
            std::lock_guard<std::mutex> lock(m);
            used -= need;
        }
        cv.notify_all();
    }

private:
    std::mutex m;
    std::condition_variable cv;
    unsigned next = 0, serving = 0;
    int used = 0;
};

} // namespace pp
