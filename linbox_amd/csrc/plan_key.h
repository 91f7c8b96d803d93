// Keys of the plans that a context keeps in one map (lbx_ctx::mp_plans): each
// kind of plan has a tag of its own, and what follows it reads back only one way
// (a multiprecision modulus is raw bytes, so its word count comes first).
#pragma once

#include <cstddef>
#include <cstdint>
#include <string>

namespace lbx {

inline std::string plan_key_fields(std::string key, std::size_t k, std::size_t minsz, unsigned lpts)
{
    return key + "|" + std::to_string(k) + "|" + std::to_string(minsz) + "|" + std::to_string(lpts);
}

// Product modulo the nl-word P.
inline std::string mp_plan_key(const uint32_t *P, int nl, std::size_t k, std::size_t minsz, unsigned lpts)
{
    const std::string words((const char *)P, (std::size_t)nl * 4);
    return plan_key_fields("mp|" + std::to_string(nl) + "|" + words, k, minsz, lpts);
}

// Few-primes product modulo the word p.
inline std::string few_plan_key(uint32_t p, std::size_t k, std::size_t minsz, unsigned lpts)
{
    return plan_key_fields("fp|" + std::to_string(p), k, minsz, lpts);
}

// Integer product of nl-word operands of lab bits together into cl words.
const char *const kZzPlanTag = "zz|";
inline std::string zz_plan_key(unsigned lab, std::size_t k, std::size_t minsz, unsigned lpts, int nl, int cl)
{
    return plan_key_fields(kZzPlanTag + std::to_string(lab), k, minsz, lpts) + "|" + std::to_string(nl) + "|" +
           std::to_string(cl);
}

}  // namespace lbx
