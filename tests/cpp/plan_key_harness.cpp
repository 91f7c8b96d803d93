// Host build of the plan keys (linbox_amd/csrc/plan_key.h) for tests/test_plan_key.py.
#include <cstring>

#include "../../linbox_amd/csrc/plan_key.h"

static int put(const std::string &key, char *out, int cap)
{
    if ((int)key.size() > cap) return -1;
    std::memcpy(out, key.data(), key.size());
    return (int)key.size();
}

extern "C" {
int lbx_test_mp_key(const uint32_t *P, int nl, size_t k, size_t minsz, unsigned lpts, char *out, int cap)
{
    return put(lbx::mp_plan_key(P, nl, k, minsz, lpts), out, cap);
}
int lbx_test_few_key(uint32_t p, size_t k, size_t minsz, unsigned lpts, char *out, int cap)
{
    return put(lbx::few_plan_key(p, k, minsz, lpts), out, cap);
}
int lbx_test_zz_key(unsigned lab, size_t k, size_t minsz, unsigned lpts, int nl, int cl, char *out, int cap)
{
    return put(lbx::zz_plan_key(lab, k, minsz, lpts, nl, cl), out, cap);
}
}
