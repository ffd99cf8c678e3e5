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
    return 0;
}
