// The bounded wait of the resident Krylov engine.
#pragma once

#ifdef __HIPCC__
#define PP_HD __host__ __device__ __forceinline__
#else
#define PP_HD inline
#endif

namespace pp {

// What a thread may still spend polling the words of one exchange: `left` polls for all of them
// together, less once a workgroup of the launch has given up (it left `word` at *ended), which is looked at
// every PATIENCE_LOOK polls.
constexpr int PATIENCE_LOOK = 1024;
struct Patience {
    int left;
    const unsigned *ended;
    unsigned word;
    // One more poll?
    PP_HD bool more() {
        if (left <= 0) return false;
        if (--left % PATIENCE_LOOK == 0 && __atomic_load_n(ended, __ATOMIC_RELAXED) == word) left = 0;
        return true;
    }
};

} // namespace pp
