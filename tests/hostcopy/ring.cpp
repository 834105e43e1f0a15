// HostCopy (st_hostcopy.hip) on the simulated runtime of hip/hip_runtime.h: `ring <case>`,
// exit status 0 if every array arrived whole.
#include "../../stokes_to_amd/csrc/st_hostcopy.hip"

#include <cstdio>
#include <string>
#include <vector>

using st::HostCopy;
typedef std::vector<uint64_t> Arr;

static Arr data(size_t n, uint64_t seed)
{
    Arr a(n);
    for (size_t i = 0; i < n; i++) a[i] = (seed << 32) + i;
    return a;
}
static int check(const char *what, const Arr &a, const Arr &b)
{
    for (size_t i = 0; i < a.size(); i++)
        if (a[i] != b[i]) {
            std::printf("%s: wrong from entry %zu of %zu\n", what, i, a.size());
            return 1;
        }
    return 0;
}
static int both_ways(HostCopy &hc, SimStream &s, size_t n, uint64_t seed)
{
    const Arr h = data(n, seed);
    Arr d(n), back(n);
    if (hc.in(d.data(), h.data(), n * 8, &s) != hipSuccess) return 1;
    if (hc.out(back.data(), d.data(), n * 8, &s) != hipSuccess) return 1;
    return check("both ways", back, h);
}

int main(int argc, char **argv)
{
    const std::string c = argc > 1 ? argv[1] : "";
    const size_t MB = 131072;  // entries
    SimStream s;
    HostCopy hc;
    int bad = 0;
    if (c == "sizes") {
        for (size_t n : {MB / 2, 4 * MB, 4 * MB + 1, 5 * MB - 1, 32 * MB, 32 * MB + 3, 41 * MB + 7}) bad += both_ways(hc, s, n, n);
        return bad;
    }
    if (c == "known") {  // by the runtime's own copy, whatever the size
        Arr h = data(40 * MB, 1), d(40 * MB);
        pinned = h.data();
        bad += hc.in(d.data(), h.data(), h.size() * 8, &s) != hipSuccess || copies != 1;
        bad += hc.out(h.data(), d.data(), h.size() * 8, &s) != hipSuccess || copies != 2;
        return bad + check("known", h, data(40 * MB, 1));
    }
    // a copy whose record of the at-th event fails
    const int at = argc > 2 ? std::atoi(argv[2]) : 1;
    const size_t n = 36 * MB + 5;
    const Arr h = data(n, 1), other = data(n, 2);
    Arr d = h, back(n);
    fail_record = at;
    const bool out = c.find("out") != std::string::npos;
    const hipError_t e = out ? hc.out(back.data(), d.data(), n * 8, &s) : hc.in(d.data(), other.data(), n * 8, &s);
    if (e == hipSuccess || fail_record != 0) return 2;
    if (c.find("then") == std::string::npos) return hipStreamSynchronize(&s);
    // then copies that have to be right
    Arr d2(n);
    if (hc.in(d2.data(), other.data(), n * 8, &s) != hipSuccess) return 2;
    hipStreamSynchronize(&s);
    bad += check("next in", d2, other);
    bad += both_ways(hc, s, 33 * MB, 3);
    return bad;
}
