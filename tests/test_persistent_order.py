"""Host bookkeeping of the persistent step (sp_order.h), compiled for the CPU with a runtime that only writes down what it
is asked: the error word is reported once per launch even if late blocks set it again, launches on one stream cost
nothing, launches on several wait for the last launch alone, captured ones are left out."""
import subprocess
from pathlib import Path

import seedplane_amd

CSRC = Path(seedplane_amd.__file__).parent / 'csrc'

PROGRAM = r'''
#include <cstdio>
#include <set>
#include <string>
#include "sp_order.h"

static std::string log;
struct Fake {
    using Stream = int;
    using Event = int;
    std::set<int> cap;
    bool capturing(int s) { return cap.count(s) != 0; }
    void sync(int s) { log += " sync" + std::to_string(s); }
    void record(int &, int s) { log += " record" + std::to_string(s); }
    void wait(int s, int) { log += " wait" + std::to_string(s); }
};
static int bad = 0;
static void expect(const char *what, const std::string &want) {
    if (log != want) { std::printf("%s: got '%s', want '%s'\n", what, log.c_str(), want.c_str()); ++bad; }
    log.clear();
}
int main() {
    // a block reports, the host looks, later blocks of the same launch report again before the stream is idle
    unsigned word = 1;
    int waits = 0;
    const bool first = sp::take_error(&word, [&] { ++waits; word = 1; });
    const bool again = sp::take_error(&word, [&] { ++waits; });
    if (!first || again || waits != 1 || word != 0) { std::printf("error word\n"); ++bad; }
    if (sp::take_error(nullptr, [&] { ++waits; }) || waits != 1) { std::printf("no word\n"); ++bad; }

    Fake rt;
    sp::PersistentOrder<Fake> o;
    auto launch = [&](int s) { o.before(rt, s); log += " run" + std::to_string(s); o.after(rt, s); };
    o.join(1);
    launch(1); launch(1);
    expect("one stream", " run1 run1");
    o.join(1);                                   // a second engine on the same stream
    launch(1);
    expect("two engines, one stream", " run1");
    o.join(2);
    launch(2);
    expect("the first launch on a second stream", " sync1 run2 record2");
    launch(2);
    expect("again there", " run2 record2");
    log += " work2";                             // queued behind the kernel: not waited for
    launch(1);
    expect("back on the first", " work2 wait1 run1 record1");
    rt.cap = {2};
    launch(2);
    expect("captured", " run2");
    rt.cap.clear();
    launch(2);
    expect("after the capture", " wait2 run2 record2");
    o.leave(2);
    launch(1);
    expect("the other stream is gone", " run1");
    o.leave(1); o.leave(1);
    o.join(3);
    rt.cap = {1};
    launch(3);
    expect("a new stream after all have left", " run3");
    return bad;
}
'''


def test_order_and_error_word(tmp_path):
    src, exe = tmp_path / 'order.cpp', tmp_path / 'order'
    src.write_text(PROGRAM)
    subprocess.run(['g++', '-std=c++17', '-Wall', '-Werror', '-I', str(CSRC), str(src), '-o', str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
