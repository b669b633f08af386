/*
 * host_sem.cpp - the sharing of rays at the end of a launch with the
 * semantics of the CPU twin (both layouts) and of the particle pass (direct
 * layout), one tree, compiled for the host. Test infrastructure only.
 */
#include "host_split.cpp"

namespace {

template <bool CMP, int SEM, bool GRID>
int run_sem(const SceneDev& s, const int* ref, const float* org, const float* dir, size_t n, int per_wave,
            int32_t* status, int32_t* leaf, float* isp)
{
    const int             L = s.maxlevel > 0 ? s.maxlevel : 1;
    std::vector<uint32_t> lds((size_t) L * 2 * 64 + 64);
    for (size_t base = 0; base < n; base += (size_t) per_wave) {
        const size_t cnt = std::min((size_t) per_wave, n - base);
        std::fill(lds.begin(), lds.end(), 0xDEADBEEFu);
        const bool ok = wave::run([&]() {
            const int    lane = wave::cur;
            const size_t i    = base + (size_t) lane;
            Stack        st;
            st.stride = 2 * 64;
            st.pw     = lds.data() + 2 * (size_t) lane;
            st.ns = st.nd = reinterpret_cast<int*>(st.pw) + 1;
            TraceState t;
            std::memset(&t, 0, sizeof(t));
            Ray  r{};
            auto write = [&](int stt) {
                status[i]      = stt;
                leaf[i]        = stt == ST_HIT ? (CMP ? ref[t.ns] : t.ns) : -1;
                const float4 p = stt == ST_HIT ? t.entry : make_float4(0.f, 0.f, 0.f, 0.f);
                isp[4 * i] = p.x, isp[4 * i + 1] = p.y, isp[4 * i + 2] = p.z, isp[4 * i + 3] = p.w;
            };
            bool active = false;
            if ((size_t) lane < cnt) {
                r = Ray{org[3 * i], org[3 * i + 1], org[3 * i + 2], dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
                const int stt = trace_begin<SEM>(s, r, t);
                if (stt == ST_CONT) active = true;
                else write(stt);
            }
            drain<CMP, false, SEM, GRID>(s, r, st, t, active, lds.data() + (size_t) L * 2 * 64, [&](int stt) {
                write(stt);
                return false;
            });
        });
        if (!ok) return -2;
    }
    return 0;
}

} // namespace

/* sem 1: the CPU twin, 2: the particle pass */
extern "C" int ht_sem(const int32_t* nodes, size_t len, const float basecube[4], int maxlevel, int layout, int sem,
                      int grid, const float* org, const float* dir, size_t n, int per_wave, int32_t* status,
                      int32_t* leaf, float* isp)
{
    static const int32_t root[12] = {0};
    Layouts              S, D;
    if (!build(nodes, len, S) || !build(root, 1, D) || (sem == 2 && layout == 1)) return -1;
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
#define QBT_RUN(C, M, G) run_sem<C, M, G>(s, ref, org, dir, n, per_wave, status, leaf, isp)
    if (sem == 2) return grid ? QBT_RUN(false, kSemParticle, true) : QBT_RUN(false, kSemParticle, false);
    if (cmp) return grid ? QBT_RUN(true, kSemCpu, true) : QBT_RUN(true, kSemCpu, false);
    return grid ? QBT_RUN(false, kSemCpu, true) : QBT_RUN(false, kSemCpu, false);
#undef QBT_RUN
}
