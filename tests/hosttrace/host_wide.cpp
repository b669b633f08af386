/*
 * host_wide.cpp - both trees on their compact layouts with the stack words
 * that a dynamic layout of any size takes (SceneDev::dyn_wide), compiled for
 * the host: rays one by one, or per_wave at a time by the sharing of the end
 * of a launch. Test infrastructure only.
 */
#include "host_split.cpp"

extern "C" int ht_wide(const int32_t* nodes, size_t len, const int32_t* dyn, size_t dlen, const float basecube[4],
                       int maxlevel, int grid, const float* org, const float* dir, size_t n, int per_wave,
                       int32_t* status, int32_t* leaf, float* isp, int64_t* exps)
{
    Layouts S, D;
    if (!build(nodes, len, S) || !build(dyn, dlen, D)) return -1;
    SceneDev s;
    memset(&s, 0, sizeof(s));
    s.stat     = tree_of(S, true);
    s.dyn      = tree_of(D, true);
    s.bx       = basecube[0];
    s.by       = basecube[1];
    s.bz       = basecube[2];
    s.bw       = basecube[3];
    s.maxlevel = maxlevel;
    s.iter_cap = 1 << 24;
    s.dyn_wide = 1;
    const int* ref = S.ref.data();
    if (per_wave > 0)
        return grid ? run_split<true, true, true>(s, ref, org, dir, n, per_wave, status, leaf, isp)
                    : run_split<true, true, false>(s, ref, org, dir, n, per_wave, status, leaf, isp);
    if (grid) run<true, true, true>(s, ref, org, dir, n, status, leaf, isp, exps);
    else run<true, true, false>(s, ref, org, dir, n, status, leaf, isp, exps);
    return 0;
}
