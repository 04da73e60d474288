// judge_work.hpp -- device copies of an interpolation's queries and answers,
// kept between calls (up to KEEP queries, 26 MB).  Buf<T> is the buffer type:
// alloc(n) frees what it holds and throws without holding anything, release()
// frees; a parameter so that the growth can be checked without a device.
#pragma once

#include <cstddef>
#include <cstdint>

namespace gfx {

template <template <class> class Buf>
struct JudgeWork {
    static constexpr size_t KEEP = 262144;
    Buf<double> q;
    Buf<int32_t> t, c;
    Buf<float> o;
    size_t cap = 0;  // queries all four hold; 0 when any of them failed to grow
    void fit(size_t n) {
        if (cap >= n) return;
        release();
        try {
            q.alloc(n * 3);
            t.alloc(n);
            c.alloc(n);
            o.alloc(n * 18);
        } catch (...) {
            release();
            throw;
        }
        cap = n;
    }
    void release() {
        cap = 0;
        q.release();
        t.release();
        c.release();
        o.release();
    }
    void trim() {
        if (cap > KEEP) release();
    }
};

}  // namespace gfx
