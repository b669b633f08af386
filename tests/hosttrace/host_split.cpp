/*
 * host_split.cpp - the end-of-launch sharing of rays between the lanes of a
 * wave (qubatron_amd/csrc/device/split.hpp) compiled for the host. A wave is
 * 64 contexts that run in turn from one wave-wide operation to the next
 * (ballot, shuffle, LDS ordering point), so that every lane takes part in
 * each of them, as the lanes of a wavefront do. Test infrastructure only.
 */
#include <ucontext.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

#include "hip/hip_runtime.h"

namespace wave {
constexpr int kStack = 256 * 1024;
ucontext_t    sched, ctx[64];
uint64_t      slot[64];
bool          ended[64];
int           cur;
inline void   sync() { swapcontext(&ctx[cur], &sched); }
template <class T>
T exchange(T v, int src)
{
    slot[cur] = 0;
    std::memcpy(&slot[cur], &v, sizeof(T));
    sync();
    T r;
    std::memcpy(&r, &slot[src & 63], sizeof(T));
    sync();
    return r;
}
std::function<void()> body;
void                  entry()
{
    body();
    ended[cur] = true;
    swapcontext(&ctx[cur], &sched);
}
/* runs f on 64 lanes; false if lanes end at different operations */
bool run(std::function<void()> f)
{
    static std::vector<char> mem(64 * (size_t) kStack);
    body = f;
    for (int l = 0; l < 64; l++) {
        ended[l] = false;
        getcontext(&ctx[l]);
        ctx[l].uc_stack.ss_sp   = mem.data() + (size_t) l * kStack;
        ctx[l].uc_stack.ss_size = kStack;
        ctx[l].uc_link          = &sched;
        makecontext(&ctx[l], entry, 0);
    }
    for (;;) {
        int n = 0;
        for (cur = 0; cur < 64; cur++) {
            if (!ended[cur]) swapcontext(&sched, &ctx[cur]);
            n += ended[cur];
        }
        if (n == 64) return true;
        if (n != 0) return false;
    }
}
} // namespace wave

struct LaneIndex {
    struct X {
        operator unsigned() const { return (unsigned) wave::cur; }
    } x;
};
static const LaneIndex threadIdx;

inline uint64_t __ballot(int p)
{
    wave::slot[wave::cur] = p ? 1u : 0u;
    wave::sync();
    uint64_t m = 0;
    for (int l = 0; l < 64; l++) m |= wave::slot[l] << l;
    wave::sync();
    return m;
}
template <class T>
T __shfl(T v, int src, int)
{
    return wave::exchange(v, src);
}
inline uint32_t atomicMin(uint32_t* p, uint32_t v)
{
    const uint32_t o = *p;
    *p               = std::min(o, v);
    return o;
}
inline int      __popcll(unsigned long long m) { return __builtin_popcountll(m); }
inline int      __ffs(int x) { return __builtin_ffs(x); }
inline unsigned mbcnt_lo(unsigned m, unsigned a)
{
    return a + (unsigned) __builtin_popcount(wave::cur >= 32 ? m : m & ((1u << wave::cur) - 1u));
}
inline unsigned mbcnt_hi(unsigned m, unsigned a)
{
    return a + (wave::cur <= 32 ? 0u : (unsigned) __builtin_popcount(m & ((1u << (wave::cur - 32)) - 1u)));
}
#define __builtin_amdgcn_mbcnt_lo(m, a) mbcnt_lo(m, a)
#define __builtin_amdgcn_mbcnt_hi(m, a) mbcnt_hi(m, a)
#define __builtin_amdgcn_fence(o, s) ((void) 0)
#define __builtin_amdgcn_wave_barrier() wave::sync()
using std::min;

#define QBT_HOST_BUILD /* the sharing only, not the work queues */
#include "host_trace.cpp"
#include "split.hpp"

namespace {

template <bool CMP, bool DUAL, bool GRID>
int run_split(const SceneDev& s, const int* ref, const float* org, const float* dir, size_t n, int per_wave,
              int32_t* status, int32_t* leaf, float* isp)
{
    const int             L = s.maxlevel > 0 ? s.maxlevel : 1, W = DUAL ? 3 : 2;
    std::vector<uint32_t> lds((size_t) L * W * 64 + 64);
    size_t                base = 0;
    while (base < n) {
        const size_t cnt = std::min((size_t) per_wave, n - base);
        std::fill(lds.begin(), lds.end(), 0xDEADBEEFu);
        size_t next = base + cnt; /* lane 0's finish starts one ray more, as k_frame's deferred rays do */
        size_t more = next < n && cnt > 1 ? next : n;
        bool   ok   = wave::run([&]() {
            const int lane = wave::cur;
            Stack     st;
            st.stride = W * 64;
            st.pw     = lds.data() + (size_t) W * lane;
            st.ns     = reinterpret_cast<int*>(st.pw) + 1;
            st.nd     = DUAL ? reinterpret_cast<int*>(st.pw) + 2 : st.ns;
            TraceState t;
            std::memset(&t, 0, sizeof(t));
            Ray    r{};
            size_t i      = base + (size_t) lane;
            bool   active = false;
            auto   write  = [&](int stt) {
                status[i]      = stt;
                leaf[i]        = stt == ST_HIT ? (CMP ? ref[t.ns] : t.ns) : -1;
                const float4 p = stt == ST_HIT ? t.entry : make_float4(0.f, 0.f, 0.f, 0.f);
                isp[4 * i] = p.x, isp[4 * i + 1] = p.y, isp[4 * i + 2] = p.z, isp[4 * i + 3] = p.w;
            };
            auto start = [&]() {
                r             = Ray{org[3 * i], org[3 * i + 1], org[3 * i + 2], dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
                const int stt = trace_begin<kSemShader>(s, r, t);
                if (stt == ST_CONT) return true;
                write(stt);
                return false;
            };
            if ((size_t) lane < cnt) active = start();
            drain<CMP, DUAL, kSemShader, GRID>(s, r, st, t, active, lds.data() + (size_t) L * W * 64, [&](int stt) {
                write(stt);
                if (lane != 0 || i == more || more == n) return false;
                i = more;
                return start();
            });
            if (lane == 0 && more != n && i != more) { /* lane 0's first ray ended before the drain */
                i = more;
                if (start()) { /* its own trace, serially */
                    int stt;
                    while ((stt = trace_step<CMP, DUAL, kSemShader, GRID>(s, r, st, t)) == ST_CONT) {}
                    write(stt);
                }
            }
        });
        if (!ok) return -2;
        base = more != n ? more + 1 : next;
    }
    return 0;
}

} // namespace

/* ht_trace with the rays traced per_wave at a time by drain() */
extern "C" int ht_split(const int32_t* nodes, size_t len, const int32_t* dyn, size_t dlen, const float basecube[4],
                        int maxlevel, int layout, int grid, const float* org, const float* dir, size_t n, int per_wave,
                        int32_t* status, int32_t* leaf, float* isp)
{
    static const int32_t root[12] = {0};
    Layouts              S, D;
    if (!build(nodes, len, S)) return -1;
    const bool dual = dyn && dlen > 1;
    if (!build(dual ? dyn : root, dual ? dlen : 1, D)) return -1;
    const bool cmp = layout == 1;
    SceneDev   s;
    memset(&s, 0, sizeof(s));
    s.stat     = tree_of(S, cmp);
    s.dyn      = tree_of(D, cmp);
    s.bx       = basecube[0];
    s.by       = basecube[1];
    s.bz       = basecube[2];
    s.bw       = basecube[3];
    s.maxlevel = maxlevel;
    s.iter_cap = 1 << 24;
    const int* ref = S.ref.data();
#define QBT_RUN(C, D_, G) run_split<C, D_, G>(s, ref, org, dir, n, per_wave, status, leaf, isp)
    if (cmp) {
        if (dual) return grid ? QBT_RUN(true, true, true) : QBT_RUN(true, true, false);
        return grid ? QBT_RUN(true, false, true) : QBT_RUN(true, false, false);
    }
    if (dual) return grid ? QBT_RUN(false, true, true) : QBT_RUN(false, true, false);
    return grid ? QBT_RUN(false, false, true) : QBT_RUN(false, false, false);
#undef QBT_RUN
}
