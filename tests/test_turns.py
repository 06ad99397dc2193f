"""Turns of handles whose launches need each other's compute units (nanollama_amd/csrc/nl_turns.h), compiled by itself and driven with events that are
written down instead of recorded."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <string>
#include <thread>
#include "nl_turns.h"
struct H { const char *name; };
static std::string out;
static nl::Turns<H> T, other_device;
static H a{"a"}, b{"b"}, c{"c"};
static int go(nl::Turns<H> &t, H *h) {
    return t.run(h, [&] { out += std::string(" launch:") + h->name; return 0; },
                 [&](H *o) { out += std::string(" ") + h->name + "<" + o->name; return 0; }, [&] { out += std::string(" rec:") + h->name; return 0; });
}
static int join(H *h, bool whole) {
    return T.join(h, whole, [&](H *o) { out += std::string(" ") + h->name + "<" + o->name; return 0; }, [&](H *o) { out += std::string(" rec:") + o->name; return 0; });
}
static bool soon(std::atomic<int> &n, int want) {       // (a second at most)
    for (int i = 0; i < 1000 && n < want; i++) std::this_thread::sleep_for(std::chrono::milliseconds(1));
    return n >= want;
}
// two launches that each last until both are under way, or a second
static bool overlap(nl::Turns<H> &t, nl::Turns<H> &u) {
    std::atomic<int> inside{0}, met{0};
    auto one = [&](nl::Turns<H> &w, H *h) {
        w.run(h, [&] { inside++; if (soon(inside, 2)) met++; return 0; }, [](H *) { return 0; }, [] { return 0; });
    };
    std::thread x([&] { one(t, &a); }), y([&] { one(u, &b); });
    x.join(); y.join();
    return met == 2;
}
int main(int, char **argv) {
    const std::string what = argv[1];
    if (what == "alone") { join(&a, true); go(T, &a); go(T, &a); }
    if (what == "at_will") { join(&a, false); join(&b, false); go(T, &a); go(T, &b); go(T, &a); }
    if (what == "pair") { join(&a, true); go(T, &a); join(&b, false); go(T, &b); go(T, &b); go(T, &a); T.leave(&b); go(T, &a); }
    if (what == "third") { join(&a, false); join(&b, false); go(T, &a); go(T, &b); join(&c, true); go(T, &c); go(T, &b); go(T, &a); }
    if (what == "retired") { join(&a, true); join(&b, false); go(T, &b); T.retire(&a); go(T, &a); go(T, &b); join(&c, true); go(T, &c); }
    if (what == "gone") { join(&a, true); join(&b, true); go(T, &a); T.leave(&a); go(T, &b); join(&c, false); go(T, &c); }
    if (what == "failed_join") {
        join(&a, true);
        int rc = T.join(&b, false, [](H *) { return -7; }, [](H *) { return 0; });
        out += " " + std::to_string(rc);
        go(T, &a);
    }
    if (what == "failed_wait") {
        join(&a, true); join(&b, true); go(T, &a);
        int rc = T.run(&b, [] { out += " launched"; return 0; }, [](H *) { return -7; }, [] { return 0; });
        out += " " + std::to_string(rc);
    }
    if (what == "locks") {
        join(&a, true);
        other_device.join(&b, true, [](H *) { return 0; }, [](H *) { return 0; });
        out = overlap(T, other_device) ? " devices_apart" : " devices_together";
        nl::Turns<H> u;
        u.join(&a, false, [](H *) { return 0; }, [](H *) { return 0; });
        u.join(&b, false, [](H *) { return 0; }, [](H *) { return 0; });
        out += overlap(u, u) ? " at_will_apart" : " at_will_together";
        { auto hold = u.capture(); out += hold ? " held" : " free"; }
        nl::Turns<H> v;
        v.join(&a, true, [](H *) { return 0; }, [](H *) { return 0; });
        v.join(&b, false, [](H *) { return 0; }, [](H *) { return 0; });
        { auto hold = v.capture(); out += hold ? " held" : " free"; }
        out += overlap(v, v) ? " turns_together" : " turns_apart";
    }
    std::puts(out.c_str());
}
"""
EXPECT = {
    "alone": "launch:a launch:a",
    "at_will": "launch:a launch:b launch:a",
    "pair": "launch:a rec:a b<a launch:b rec:b launch:b rec:b a<b launch:a rec:a launch:a",
    # two that launched at will: the newcomer waits for both, and then everybody for the last
    "third": "launch:a launch:b rec:a c<a rec:b c<b launch:c rec:c b<c launch:b rec:b a<b launch:a rec:a",
    "retired": "rec:a b<a launch:b rec:b launch:a launch:b rec:a c<a rec:b c<b c<b launch:c rec:c",
    "gone": "rec:a b<a launch:a rec:a launch:b rec:b c<b launch:c rec:c",
    "failed_join": "-7 launch:a",
    "failed_wait": "rec:a b<a launch:a rec:a -7",
    "locks": "devices_apart at_will_apart free held turns_apart",
}


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("turns")
    (d / "t.cpp").write_text(DRIVER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", os.path.join(ROOT, "nanollama_amd", "csrc"), str(d / "t.cpp"), "-o", str(d / "t")])
    return str(d / "t")


@pytest.mark.parametrize("what", EXPECT)
def test_order_of_events_and_launches(driver, what):
    assert subprocess.check_output([driver, what], text=True, timeout=60).split() == EXPECT[what].split()
