// What a process prepares once for each GPU (whispereacp_amd/csrc/once_per_device.h)
// on the CPU: every device is prepared, a failure is tried again, success is not.
// Prints "ok <case>" per passing case; exits 1 on the first failure.
#include "../../whispereacp_amd/csrc/once_per_device.h"

#include <cstdio>
#include <cstdlib>

static void expect(bool condition, const char* what)
{
    if (!condition)
    {
        std::printf("FAIL %s\n", what);
        std::exit(1);
    }
    std::printf("ok %s\n", what);
}

int main()
{
    wsp::OncePerDevice once;
    int calls = 0;
    auto prepare = [&] { ++calls; return 0; };
    auto refuse = [&] { ++calls; return 7; };
    expect(once(0, prepare) == 0 && calls == 1, "the first device is prepared");
    expect(once(0, prepare) == 0 && calls == 1, "and not again");
    expect(once(1, prepare) == 0 && calls == 2, "another device is prepared too");
    expect(once(63, prepare) == 0 && once(63, prepare) == 0 && calls == 3, "the last one kept");
    expect(once(2, refuse) == 7 && once(2, refuse) == 7 && calls == 5, "a failure is reported and tried again");
    expect(once(2, prepare) == 0 && once(2, refuse) == 0 && calls == 6, "until it succeeds");
    expect(once(64, prepare) == 0 && once(64, prepare) == 0 && calls == 8, "devices past those are prepared every time");
    expect(once(0, refuse) == 0 && calls == 8, "without touching the others");
    return 0;
}
