// The host's wait for a piece of a result (qwn_download.h), driven by a
// stream and a kernel that are plain variables here.
#include "qwn_download.h"

#include <cstdio>
#include <cstring>

using namespace qwn;

static int failures = 0;
static void check(bool ok, const char *what) {
    if (!ok) {
        std::printf("FAILED: %s\n", what);
        ++failures;
    }
}

int main() {
    const uint32_t epoch = 7;
    {
        uint32_t flag = 7;
        int turns = 0;
        check(await_piece(&flag, epoch, [&] { ++turns; }, [] { return StreamState::kFailed; }) == Landing::kLanded &&
                  turns == 0, "a piece that is there is taken at once");
    }
    {
        uint32_t flag = 6;   // the earlier transfer's
        int turns = 0;
        check(await_piece(&flag, epoch, [&] { if (++turns == 100) flag = epoch; },
                          [] { return StreamState::kBusy; }, 8) == Landing::kLanded, "a piece that lands in the wait");
    }
    {
        uint32_t flag = 6;
        check(await_piece(&flag, epoch, [] {}, [] { return StreamState::kDone; }, 8) == Landing::kMissing,
              "a finished stream whose flag was never raised is no success");
    }
    {
        uint32_t flag = 6;
        check(await_piece(&flag, epoch, [] {}, [&] { flag = epoch; return StreamState::kDone; }, 8) == Landing::kLanded,
              "a piece that lands just before the stream is asked");
    }
    {
        uint32_t flag = 6;
        int asked = 0;
        check(await_piece(&flag, epoch, [] {}, [&] { return ++asked < 3 ? StreamState::kBusy : StreamState::kFailed; },
                          8) == Landing::kFailed && asked == 3, "a stream's error ends the wait");
    }
    {
        float page[4] = {1.5f, -0.0f, 0.0f, 2.0f};
        uint32_t nan = 0x7fa00001u;   // a signalling pattern stays as it is
        std::memcpy(page + 2, &nan, 4);
        float before[4];
        std::memcpy(before, page, sizeof(page));
        for (float &p : page) map_for_writing(&p);
        for (int i = 1; i < 13; ++i) map_for_writing(reinterpret_cast<float *>(reinterpret_cast<char *>(page) + i));
        check(std::memcmp(before, page, sizeof(page)) == 0, "a page that is mapped keeps what it holds");
    }
    if (!failures) std::printf("ok\n");
    return failures != 0;
}
