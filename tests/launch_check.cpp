// Arguments that the launchers refuse before any GPU call: prints each case's name and whether
// it came back as hipErrorInvalidValue.
#include <cstdio>

#include "tf_internal.hpp"

using namespace tfk;

static void say(const char* name, hipError_t e) { std::printf("%s %d\n", name, e == hipErrorInvalidValue); }

int main() {
    float row[64] = {};
    AttnArgs a{};
    a.q = a.kc = row;
    a.H = a.G = 1;
    a.hd = 64;
    a.S = 1;
    a.max_seq = 1;
    a.rope_cos = row;
    say("attn_sin", launch_attn_decode(a, nullptr));
    a.rope_cos = nullptr;
    a.rope_sin = row;
    say("attn_cos", launch_attn_decode(a, nullptr));

    // K slices' sums of 256 columns
    uint16_t half = 0;
    int count = 0;
    PfSmallArgs s;
    s.xa = &half;
    s.K = 2048;
    s.M = 1;
    s.mode = GEMV_RESID;
    s.n_seg = 1;
    s.n_sub = 16;
    s.seg[0].w.type = TF_HIP_TYPE_Q8_0;
    s.seg[0].w.K = 2048;
    s.seg[0].w.N = 256;
    s.seg[0].y = row;
    s.part = row;
    s.count = &count;
    say("small_part", launch_pf_small(s, nullptr));
    s.part_floats = kPfSmallPart(256) - 1;
    say("small_part_short", launch_pf_small(s, nullptr));
    s.part_floats = kPfSmallPart(256);
    s.count = nullptr;
    say("small_count", launch_pf_small(s, nullptr));
    return 0;
}
