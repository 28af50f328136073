// Host-only pieces of the hipq library: error state, the fixed-point scale decomposition, layout rule.
#include <cmath>
#include <cstdarg>
#include <cstdio>

#include <algorithm>

#include "common.h"

namespace hipq {

static thread_local char g_err[512] = "";

int fail(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return 1;
}

void clear_error() { g_err[0] = 0; }

} // namespace hipq

extern "C" int hipq_abi_version(void) { return HIPQ_ABI_VERSION; }

extern "C" const char *hipq_last_error(void) { return hipq::g_err; }

// get_quant_scale / get_quant_scale_int16 / get_quant_scale_int32 of the reference
// (art/modules/quant/include/art/quant/quant_helper.h:60-118): the scale is normalised into [0.5, 1)
// by exact fp32 halving / doubling, the multiplier is its mantissa truncated to bits-1 bits.
extern "C" void hipq_quant_scale(float x, int bits, uint32_t *mult, int *shift)
{
    int s = 0;
    *mult = 0;
    *shift = 0;
    if (std::fabs((double)x) < 1e-10 || !(x > 0.0f) || std::isinf(x))
        return; // zero like the reference; negative / infinite scales never terminate there
    while (x >= 1.0f) {
        x /= 2;
        s -= 1;
    }
    while (x < 0.5f) {
        x *= 2;
        s += 1;
    }
    *mult = (uint32_t)(x * (float)(1ll << (bits - 1)));
    *shift = s + bits - 1;
}

// The exact form's constants: with u = max(s0, s1) the sum of the terms is (x0 m0 2^(u-s0) + x1 m1 2^(u-s1) + const) / 2^u, scaled so that its
// high word is the result, which 32 bits hold the multipliers of where both ratios of scales are below one.  For each x0 the x1 whose
// sum lies less than the lost fractions, at most 3 * 2^(u-1), above a multiple of 2^(sh+u) are found in the sorted residues of the second
// term.
static bool exact_form(hipq::AddParams *p)
{
    const int u = std::max(p->s0, p->s1), d0 = u - p->s0, d1 = u - p->s1;
    const int k = 32 - u - p->sh;
    if (k < 0 || (uint64_t)p->m0 << (d0 + k) >> 32 || (uint64_t)p->m1 << (d1 + k) >> 32)
        return false;
    const int64_t mod = (int64_t)1 << (u + p->sh), rest = ((int64_t)p->cadd) << u;
    struct Term {
        int64_t at, lost;
    } t1[256];
    for (int x = 0; x < 256; x++) {
        const int64_t v = (int64_t)x * p->m1 + p->c1;
        t1[x] = {(v << d1) & (mod - 1), (v & (((int64_t)1 << p->s1) - 1)) << d1};
    }
    std::sort(t1, t1 + 256, [](const Term &a, const Term &b) { return a.at < b.at; });
    const int64_t most = (int64_t)3 << (u - 1);
    for (int x = 0; x < 256; x++) {
        const int64_t v = (int64_t)x * p->m0 + p->c0, at = ((v << d0) + rest) & (mod - 1), lost = (v & (((int64_t)1 << p->s0) - 1)) << d0;
        const int64_t from = (mod - at) & (mod - 1); // the residue that makes a multiple
        int i = (int)(std::lower_bound(t1, t1 + 256, from, [](const Term &a, int64_t b) { return a.at < b; }) - t1);
        for (int n = 0; n < 256; n++, i++) {
            const Term &t = t1[i & 255];
            const int64_t above = (t.at - from) & (mod - 1);
            if (above >= most)
                break;
            if (above < lost + t.lost)
                return false;
        }
    }
    const uint64_t at_zero = (((uint64_t)(int64_t)p->c0 << d0) + ((uint64_t)(int64_t)p->c1 << d1) + (uint64_t)rest) << k;
    p->m0 <<= d0 + k, p->m1 <<= d1 + k, p->sh = 0;
    p->c0 = (int32_t)(uint32_t)at_zero, p->c1 = (int32_t)(uint32_t)(at_zero >> 32);
    return true;
}

// The search takes some 10 us, and a launch asks for its add's constants each time: every thread remembers the last forms by the constants
// that they follow from, in 64 sets of four (with one a set, three of ResNet-50's sixteen adds shared one and were searched for at every
// launch).
bool hipq::make_add_exact(AddParams *p)
{
    struct Seen {
        AddParams from, to;
        bool known, exact;
    };
    struct Set {
        Seen way[4];
        unsigned oldest;
    };
    static thread_local Set sets[64];
    if (!p->fast)
        return false;
    const uint32_t h = (p->m0 * 0x9e3779b1u ^ p->m1 * 0x85ebca6bu ^ (uint32_t)p->c0 * 0xc2b2ae35u ^ (uint32_t)p->c1 * 0x27d4eb2fu ^ (uint32_t)p->cadd) * 0x9e3779b1u;
    Set &set = sets[h >> 26];
    Seen *e = nullptr;
    for (Seen &w : set.way) {
        const AddParams &f = w.from;
        if (w.known && f.m0 == p->m0 && f.m1 == p->m1 && f.s0 == p->s0 && f.s1 == p->s1 && f.sh == p->sh && f.c0 == p->c0 && f.c1 == p->c1 && f.cadd == p->cadd)
            e = &w;
    }
    if (e == nullptr) {
        e = &set.way[set.oldest++ % 4];
        e->from = e->to = *p;
        e->exact = exact_form(&e->to);
        e->known = true;
    }
    if (e->exact)
        p->m0 = e->to.m0, p->m1 = e->to.m1, p->sh = e->to.sh, p->c0 = e->to.c0, p->c1 = e->to.c1;
    return e->exact;
}

bool hipq::make_add_params(float ia0, int iz0, float ia1, int iz1, float oa, int oz, int obits, AddParams *p)
{
    int s0, s1;
    hipq_quant_scale(ia0 / oa, 23, &p->m0, &s0); // add.c:119-124
    hipq_quant_scale(ia1 / oa, 23, &p->m1, &s1);
    p->sh = std::min(s0, s1) - 1;
    p->s0 = s0 - p->sh, p->s1 = s1 - p->sh;
    p->z0 = iz0, p->z1 = iz1, p->oz = oz, p->hi = (1 << obits) - 1;
    if (!valid_shift(p->sh) || !valid_shift(p->s0) || !valid_shift(p->s1))
        return false;
    p->fast = p->sh <= 22 && p->s0 <= 30 && p->s1 <= 30 && p->m0 < (1u << 23) && p->m1 < (1u << 23);
    p->c0 = p->c1 = p->cadd = 0;
    if (p->fast) {
        p->c0 = (1 << (p->s0 - 1)) - iz0 * (int32_t)p->m0;
        p->c1 = (1 << (p->s1 - 1)) - iz1 * (int32_t)p->m1;
        p->cadd = (1 << (p->sh - 1)) + (oz << p->sh);
    }
    return true;
}

extern "C" int hipq_channel_stride(int C) { return C <= 4 ? 4 : (C + 15) / 16 * 16; }

// A power of two 2^k: m = 2^(32 - k), s = 0.  Otherwise s = floor(log2 d) and m = ceil(2^(32 + s) / d): m fits 32 bits
// because d > 2^s, and the round-up error e = m * d - 2^(32 + s) is below d < 2^(s + 1), so x * e < 2^(32 + s) for
// x < 2^31, which is the condition for the quotient to be exact.  d == 1 has no such m: m = 0 means "x itself".
extern "C" int hipq_div_magic(uint32_t d, uint32_t *m, int *s)
{
    if (d == 0 || m == nullptr || s == nullptr)
        return -1;
    *m = 0, *s = 0;
    if (d == 1)
        return 0;
    int lg = 31;
    while (!(d >> lg))
        lg--;
    if ((d & (d - 1)) == 0) {
        *m = 1u << (32 - lg);
        return 0;
    }
    *s = lg;
    *m = (uint32_t)(((1ull << (32 + lg)) + d - 1) / d);
    return 0;
}
