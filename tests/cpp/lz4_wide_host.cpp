// Host build of the library's workgroup decode of LZ4 blocks
// (falling_sand_engine_amd/csrc/fsg_lz4_wide.hpp) for CPU tests: its threads
// taken in turn inside each step.
#include "fsg_lz4_wide.hpp"

namespace {

// Group policy of the host build: all threads in turn.
struct HostGroup {
    static constexpr int N = fsg_lz4::WT;
    template <class T>
    struct Reg {
        T v[N];
        T &operator[](int t) { return v[t]; }
    };
    template <class F>
    void each(F f) {
        for (int t = 0; t < N; t++) f(t);
    }
    void sync() {}
    uint32_t uniform(uint32_t x) { return x; }
    void min(uint32_t *p, uint32_t v) { *p = v < *p ? v : *p; }
    void or_(uint32_t *p, uint32_t v) { *p |= v; }
    void chain(Reg<uint32_t> &nx, Reg<int> &entry, Reg<uint64_t> &mask, int base) {
        for (int seg = 0; seg < N; seg += 64) {
            uint64_t m = 0;
            for (int at = entry[seg]; at >= 0 && at < 64 && nx[seg + at] != fsg_lz4::STOP; at = (int)nx[seg + at] - seg - base)
                m |= 1ull << at;
            for (int k = 0; k < 64; k++) mask[seg + k] = m;
        }
    }
    template <class F>
    void prefix(F f, Reg<int> &before, uint32_t *sums) {
        for (int t = 0, s = 0; t < N; t++) {
            if ((t & 63) == 0) s = 0;
            before[t] = s;
            s += f(t);
            sums[t >> 6] = (uint32_t)s;
        }
    }
    int waves_before(int t, int c, const uint32_t *sums, int &total) {
        int before = 0;
        total = 0;
        for (int w = 0; w < fsg_lz4::WIN / 64; w++) {
            if (w == c * (N / 64) + (t >> 6)) before = total;
            total += (int)sums[w];
        }
        return before;
    }
    void cover(int, int *p, int v, int a, int b) {
        for (int w = a; w < b; w++) p[w] = v;
    }
};

}  // namespace

extern "C" int fsg_test_lz4_decode_wide(const uint8_t *src, int n, uint8_t *dst, int cap) {
    static fsg_lz4::WideLds lds;
    static HostGroup g;
    return fsg_lz4::decode_wide(src, n, dst, cap, lds, g);
}
