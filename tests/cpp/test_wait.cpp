// The wait for a staging buffer's copy (pa::host::wait_read), on the host alone:
// the copy and its queue are stood in for by functions. Exit status 0 = every
// check passed; each failure prints one line.

#include "pa_host.hpp"

#include <cstdio>

namespace {

int g_failures = 0;

void expect(bool ok, const char* what) {
    if (!ok) {
        std::printf("FAIL: %s\n", what);
        ++g_failures;
    }
}

}  // namespace

int main() {
    using pa::host::wait_read;
    int looks = 0, asked = 0;
    auto never = [&] { return ++looks, false; };
    auto status = [&](int busy, hipError_t then) {
        return [&asked, busy, then] { return ++asked <= busy ? hipErrorNotReady : then; };
    };

    expect(wait_read([] { return true; }, status(0, hipErrorUnknown)) == hipSuccess && asked == 0,
           "a copy that has come asks for no status");
    expect(wait_read([&] { return ++looks > 100; }, status(0, hipErrorUnknown)) == hipSuccess && asked == 0,
           "nor one that comes soon");
    expect(wait_read(never, status(0, hipErrorLaunchFailure)) == hipErrorLaunchFailure && asked == 1,
           "a failed queue ends the wait with its error");
    asked = 0;
    expect(wait_read(never, status(5, hipErrorIllegalAddress)) == hipErrorIllegalAddress && asked == 6,
           "also one that fails later");
    expect(wait_read(never, status(0, hipSuccess)) == hipErrorUnknown, "a queue that is through without the copy");
    bool come = false;
    expect(wait_read([&] { return come; }, [&] { return come = true, hipSuccess; }) == hipSuccess,
           "a copy that came just before the queue was asked");
    asked = 0;
    expect(wait_read([&] { return asked >= 3; }, status(100, hipErrorUnknown)) == hipSuccess && asked == 3,
           "a busy queue is waited for");
    std::printf("%d failure(s)\n", g_failures);
    return g_failures == 0 ? 0 : 1;
}
