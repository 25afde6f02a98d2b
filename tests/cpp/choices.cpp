// Host-only checks of how the engine decides which kernel a plan runs.  No device is
// needed: plans are filled in by hand and nothing is launched.
//     choices CASE        exit status 0: the case holds
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>

#include "kfa_engine.h"
#include "engine/kfa_fast.hpp"
#include "engine/kfa_internal.hpp"

using namespace kfa;

#define CHECK(x)                                                                      \
    do {                                                                              \
        if (!(x)) {                                                                   \
            fprintf(stderr, "%s:%d: %s does not hold\n", __FILE__, __LINE__, #x);     \
            return 1;                                                                 \
        }                                                                             \
    } while (0)

static void single_plan(DevPlan &P, int type, int n, std::vector<int> radix)
{
    P.type = type;
    P.n = n;
    P.radix = std::move(radix);
    P.single = true;
}

// What choose_fast hands out is read without the plan's lock, so a choice still open must
// not be the plan's own storage, which a larger batch of the same plan writes.
static int open_choice_is_not_the_plans()
{
    for (int kind : {FK_R2C, FK_C2R}) {
        DevPlan P;
        single_plan(P, KFA_F32, 8, {4, 2});
        const FastChoice *fc = nullptr;
        CHECK(choose_fast(P, kind, nullptr, &fc, 3) == 0);
        CHECK(fc && !fc->v && !fc->d_stw);
        const char *at = reinterpret_cast<const char *>(fc), *p0 = reinterpret_cast<const char *>(&P);
        CHECK(at < p0 || at >= p0 + sizeof P);
    }
    return 0;
}

// A small batch of short real rows runs on the general kernel also after a large one of the
// same plan was given a compiled kernel.
static int short_real_rows_do_not_depend_on_the_past()
{
    static const FastVariant compiled{};
    for (int kind : {FK_R2C, FK_C2R}) {
        DevPlan P;
        single_plan(P, KFA_F32, 8, {4, 2});
        auto c = std::make_shared<FastChoice>();
        c->v = &compiled;
        P.fast[kind] = c;
        const FastChoice *fc = nullptr;
        CHECK(choose_fast(P, kind, nullptr, &fc, 3) == 0 && !fc->v);
        CHECK(choose_fast(P, kind, nullptr, &fc, 1 << 20) == 0 && fc->v == &compiled);
    }
    return 0;
}

// A caller who sets the shortest compiled row gets it for batches of any size.
static int shortest_compiled_row_as_set()
{
    setenv("KISSFFT_AMD_RTC_MIN", "8", 1);
    setenv("KISSFFT_AMD_RTC", "0", 1);  // (nothing is compiled here)
    DevPlan P;
    single_plan(P, KFA_F32, 8, {4, 2});
    const FastChoice *fc = nullptr;
    CHECK(choose_fast(P, FK_R2C, nullptr, &fc, 3) == 0 && P.fast[FK_R2C]);
    return 0;
}

// Lengths whose direct sums are more exact than Bluestein's convolution keep them: factors of 53
// to 73 in a convolution that is more than 0.70 to 0.90 full.
static int bluestein_only_where_exact()
{
    const struct {
        std::vector<int> radix;
        bool real;  // Bluestein for real rows of this half length
    } v[] = {{{53, 19}, false},         {{53, 19, 2}, false}, {{53, 19, 4}, false}, {{53, 11, 7}, false},
             {{53, 5, 5, 3, 2}, false}, {{53, 17, 9}, false}, {{73, 109}, true},    {{53, 53}, true},
             {{79, 101}, true},         {{1021, 2}, true},    {{47, 47}, false},    {{61, 16, 4}, false},
             {{71, 16, 3}, true},       {{67, 53}, false}};
    for (const auto &x : v) {
        DevPlan P;
        int n = 1;
        for (int p : x.radix)
            n *= p;
        single_plan(P, KFA_F32, n, x.radix);
        CHECK(blue_real_rows(P) == x.real);
        if (x.real || n <= 2048)
            continue;
        bool applies = true;  // complex lines: no table is built (there is no device here)
        CHECK(blue_prepare(P, &applies) == 0 && !applies);
    }
    return 0;
}

// The tables of a long fixed-point line's second pass are bounded by their size: generic radices
// keep p - 1 entries a point and stage, the others 1.3 a point in all.
static int split_tables_are_bounded()
{
    auto fits = [](int p, int k1, int k2) {
        DevPlan P;
        P.type = KFA_Q31;
        P.single = false;
        P.n = P.L1 = P.Q = 1;
        for (int k = 0; k < k1 + k2; ++k) {
            P.radix.push_back(p);
            P.n *= p;
            (k < k1 ? P.L1 : P.Q) *= p;
        }
        return split_tables_fit(P);
    };
    CHECK(fits(4, 4, 4));    // 65536 points, 0.7 MB
    CHECK(fits(4, 5, 6));    // 2^22 points, 45 MB
    CHECK(fits(5, 4, 5));    // 1953125 points
    CHECK(fits(7, 3, 4));    // 823543 points, 6.6 M entries
    CHECK(!fits(7, 4, 4));   // 5764801 points, 46 M entries
    CHECK(!fits(13, 3, 3));  // 4826809 points, 67 M entries
    CHECK(!fits(4, 6, 6));   // 2^24 points
    return 0;
}

// Many planes of a few values, and more planes than one launch takes, keep an axis per pass.
static int compiled_planes_where_they_pay()
{
    CHECK(!plane_pays(1 << 20, 2 * 2) && !plane_pays(1 << 20, 5 * 5));
    CHECK(plane_pays(16384, 2 * 2) && plane_pays(1 << 20, 4 * 8));
    CHECK(!plane_pays(1LL << 31, 16 * 16) && plane_pays((1LL << 31) - 1, 16 * 16));
    CHECK(plane_pays(1, 2048) && !plane_pays(1, 2049) && plane_pays(128, 5000) && !plane_pays(128, 5001));
    return 0;
}

// While the no-allocation entry point runs, choices that would allocate are refused.
struct NoAlloc {
    NoAlloc() { thread_noalloc() = true; }
    ~NoAlloc() { thread_noalloc() = false; }
};

// Complex lines under 16 points have no compiled row: a batch of any size decides that, and
// the no-allocation entry point then takes batches of any size.
static int short_complex_lines_are_decided()
{
    for (int type : {KFA_F32, KFA_Q15, KFA_Q31}) {
        DevPlan P;
        single_plan(P, type, 8, {2, 4});
        const FastChoice *fc = nullptr;
        CHECK(choose_fast(P, FK_C2C, nullptr, &fc, 3) == 0 && !fc->v);
        NoAlloc on;
        CHECK(choose_fast(P, FK_C2C, nullptr, &fc, 1 << 20) == 0 && !fc->v);
    }
    return 0;
}

// A long fixed-point line whose two passes are not decided runs on the general kernel under
// the no-allocation entry point: that kernel reads the plan's own table and nothing else.
static int fixed_split_needs_no_allocation()
{
    for (int type : {KFA_Q15, KFA_Q31}) {
        DevPlan P;
        P.type = type;
        P.n = 1 << 16;
        P.radix = std::vector<int>(8, 4);
        P.single = false;
        P.L1 = P.Q = 256;
        NoAlloc on;
        CHECK(prepare_multipass(P, FK_C2C, nullptr) == 0);
    }
    return 0;
}

int main(int argc, char **argv)
{
    static const struct {
        const char *name;
        int (*run)();
    } cases[] = {
        {"open_choice_is_not_the_plans", open_choice_is_not_the_plans},
        {"short_real_rows_do_not_depend_on_the_past", short_real_rows_do_not_depend_on_the_past},
        {"shortest_compiled_row_as_set", shortest_compiled_row_as_set},
        {"bluestein_only_where_exact", bluestein_only_where_exact},
        {"split_tables_are_bounded", split_tables_are_bounded},
        {"compiled_planes_where_they_pay", compiled_planes_where_they_pay},
        {"short_complex_lines_are_decided", short_complex_lines_are_decided},
        {"fixed_split_needs_no_allocation", fixed_split_needs_no_allocation},
    };
    for (const auto &c : cases)
        if (argc == 2 && !strcmp(argv[1], c.name))
            return c.run();
    fprintf(stderr, "usage: choices CASE\n");
    return 2;
}
