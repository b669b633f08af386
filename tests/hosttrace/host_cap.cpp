/*
 * host_cap.cpp - the iteration cap of the traversal, compiled for the host:
 * rays one by one (trace), or per_wave at a time by the sharing of the end of
 * a launch (drain), under a given cap, and the steps that each ray's serial
 * trace takes. Test infrastructure only.
 */
#include "host_split.cpp"

namespace {

template <bool CMP, bool DUAL, bool GRID>
void run_steps(const SceneDev& s, const float* org, const float* dir, size_t n, int64_t* steps)
{
    const int             L = s.maxlevel > 0 ? s.maxlevel : 1;
    std::vector<uint32_t> mem(3 * (size_t) L);
    Stack                 st;
    st.stride = 1;
    st.pw     = mem.data();
    st.ns     = reinterpret_cast<int*>(mem.data()) + L;
    st.nd     = DUAL ? reinterpret_cast<int*>(mem.data()) + 2 * L : st.ns;
    for (size_t i = 0; i < n; i++) {
        Ray        r = {org[3 * i], org[3 * i + 1], org[3 * i + 2], dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]};
        TraceState t;
        int        stt = trace_begin<kSemShader>(s, r, t);
        for (steps[i] = 0; stt == ST_CONT; steps[i]++) stt = trace_step<CMP, DUAL, kSemShader, GRID>(s, r, st, t);
    }
}

template <bool CMP, bool DUAL, bool GRID>
int run_cap(SceneDev& s, const int* ref, const float* org, const float* dir, size_t n, int cap, int per_wave,
            int32_t* status, int32_t* leaf, float* isp, int64_t* steps)
{
    std::vector<int64_t> exps(n);
    s.iter_cap = 1 << 24;
    run_steps<CMP, DUAL, GRID>(s, org, dir, n, steps);
    s.iter_cap = cap;
    if (per_wave > 0) return run_split<CMP, DUAL, GRID>(s, ref, org, dir, n, per_wave, status, leaf, isp);
    run<CMP, DUAL, GRID>(s, ref, org, dir, n, status, leaf, isp, exps.data());
    return 0;
}

} // namespace

extern "C" int ht_cap(const int32_t* nodes, size_t len, const int32_t* dyn, size_t dlen, const float basecube[4],
                      int maxlevel, int layout, int grid, const float* org, const float* dir, size_t n, int cap,
                      int per_wave, int32_t* status, int32_t* leaf, float* isp, int64_t* steps)
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
    const int* ref = S.ref.data();
#define QBT_RUN(C, D_, G) run_cap<C, D_, G>(s, ref, org, dir, n, cap, per_wave, status, leaf, isp, steps)
    if (cmp) {
        if (dual) return grid ? QBT_RUN(true, true, true) : QBT_RUN(true, true, false);
        return grid ? QBT_RUN(true, false, true) : QBT_RUN(true, false, false);
    }
    if (dual) return grid ? QBT_RUN(false, true, true) : QBT_RUN(false, true, false);
    return grid ? QBT_RUN(false, false, true) : QBT_RUN(false, false, false);
#undef QBT_RUN
}
