"""The rules of the decoded operands' device memory (p8x_operands.h) on counted stand-ins for the device calls. CPU only:
each test is a C++ program built with g++."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pingala8-llm_amd", "csrc")

FAKE = r"""
#include <atomic>
#include <cassert>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <thread>
#include <vector>
#include "p8x_operands.h"
struct Fake {   // log: a = alloc, f = free, s = device synchronize, c = error cleared
    using Stream = int;
    static bool cap;   // streams are being captured
    static unsigned long long *word;   // of the buffer that asked last
    static bool host_word(unsigned long long **p) { word = *p = new unsigned long long(0); return true; }
    static bool ordered(Stream a, Stream b) { return a == b && a != 0; }
    static bool capturing(Stream) { return cap; }
    static std::string log;
    static size_t room, held;
    static bool sticky;
    static bool alloc(void **p, size_t n) {
        log += 'a';
        if (held + n > room) { sticky = true; return false; }
        size_t *q = (size_t *)malloc(sizeof(size_t));
        *q = n; held += n; *p = q;
        return true;
    }
    static void release(void *p) { log += 'f'; held -= *(size_t *)p; free(p); }
    static bool synchronize() { log += 's'; return true; }
    static void clear_error() { log += 'c'; sticky = false; }
};
std::string Fake::log; size_t Fake::room, Fake::held; bool Fake::sticky, Fake::cap; unsigned long long *Fake::word;
using namespace p8x;
"""


def run(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(FAKE + "int main() {\n" + body + "\nputs(\"ok\");\n}\n")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True, timeout=120)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout == "ok\n"


def test_out_of_memory_is_no_error(tmp_path):
    """no buffer and no error left behind; a smaller buffer is kept and still serves smaller calls"""
    run(tmp_path, r"""
    void *p = nullptr; size_t have = 0;
    Fake::room = 100;
    assert(!try_grow<Fake>(&p, &have, 101) && !p && have == 0 && !Fake::sticky && Fake::log == "ac");
    assert(try_grow<Fake>(&p, &have, 60) && p && have == 60);
    void *old = p;
    assert(!try_grow<Fake>(&p, &have, 80) && p == old && have == 60 && !Fake::sticky && Fake::held == 60);
    assert(try_grow<Fake>(&p, &have, 60) && p == old);
    Fake::room = 200; Fake::log.clear();
    assert(try_grow<Fake>(&p, &have, 80) && have == 80 && Fake::held == 80 && Fake::log == "asf");
    Fake::release(p);
    """)


def test_one_buffer_for_all_calls(tmp_path):
    """calls on one stream reuse the buffer, a call on another stream (or on a handle that may name another) gets it only
    when the last use has ended, a captured call never; it grows behind a device synchronize and goes back with the last user"""
    run(tmp_path, r"""
    OperandBuffer<Fake> b;
    Fake::room = 300;
    b.add_user(); b.add_user();
    OperandMark m;
    auto call = [&](size_t need, int st) {
        auto l = b.take(need, st);
        if (l.p) { m = l.mark(); assert(m.word == Fake::word && m.n > *m.word); l.launched(); }
        return l.p;
    };
    void *p = call(100, 1);
    assert(p && Fake::log == "a");
    assert(call(80, 1) == p && !call(80, 2));
    const OperandMark second = m;
    *m.word = second.n - 1;            // the first call has ended, the second has not
    assert(!call(80, 2));
    *m.word = second.n;
    assert(call(80, 2) == p && !call(80, 1));
    assert(Fake::log == "a");
    assert(call(150, 2) && Fake::held == 150 && Fake::log == "aasf");
    *m.word = m.n;
    assert(call(80, 0) && !call(80, 0));   // 0: a handle that names one stream per thread
    *m.word = m.n;
    Fake::cap = true;
    assert(!call(80, 0));
    Fake::cap = false;
    assert(call(80, 3));
    b.drop_user();
    assert(Fake::held == 150);
    b.drop_user();
    assert(Fake::held == 0);
    Fake::log.clear();
    b.add_user();
    assert(call(10, 4) && Fake::log == "a");   // a new buffer knows of no earlier use
    b.drop_user();
    """)


def test_failed_allocation_is_not_repeated_by_every_call(tmp_path):
    run(tmp_path, r"""
    OperandBuffer<Fake> b;
    Fake::room = 100;
    b.add_user(); b.add_user();
    { auto l = b.take(101, 1); assert(!l.p && !Fake::sticky); }
    Fake::log.clear();
    { auto l = b.take(200, 1); assert(!l.p); }
    assert(Fake::log.empty());
    { auto l = b.take(50, 1); assert(l.p); l.launched(); }        // a smaller one is tried
    Fake::room = 400;
    b.reserve(101);                                 // set-up tries again
    { auto l = b.take(101, 1); assert(l.p); l.launched(); }
    Fake::room = 400; Fake::log.clear();
    { auto l = b.take(350, 1); assert(!l.p); }      // beside the 101 held
    b.drop_user();                                  // a release, too, lets the next call try
    Fake::room = 500;
    { auto l = b.take(350, 1); assert(l.p && Fake::held == 350); l.launched(); }
    b.drop_user();
    """)


def test_use_without_its_mark_waits_for_the_device(tmp_path):
    """a call whose launches failed before the one that carries the mark"""
    run(tmp_path, r"""
    OperandBuffer<Fake> b;
    Fake::room = 100;
    b.add_user();
    { auto l = b.take(10, 1); assert(l.p); }
    assert(Fake::log == "as");
    { auto l = b.take(10, 2); assert(l.p); l.launched(); }
    { auto l = b.take(10, 1); assert(!l.p); }
    b.drop_user();
    """)


def test_lease_excludes_other_threads(tmp_path):
    run(tmp_path, r"""
    OperandBuffer<Fake> b;
    Fake::room = 100;
    b.add_user();
    std::atomic<int> in{0}, most{0};
    std::vector<std::thread> th;
    for (int i = 0; i < 4; ++i)
        th.emplace_back([&] {
            for (int k = 0; k < 200; ++k) {
                auto l = b.take(10, 1);
                if (!l.p) abort();
                const int n = ++in;
                if (n > most) most = n;
                std::this_thread::yield();
                --in;
                l.launched();
            }
        });
    for (auto &t : th) t.join();
    assert(most == 1);
    b.drop_user();
    """)


def test_fixed_operands(tmp_path):
    """one buffer per size in use, from the first tensor that needs it to the last of all; out of memory is no error"""
    run(tmp_path, r"""
    FixedOperands<Fake> f;
    const size_t M = 1 << 20;
    Fake::room = 100 * M;
    f.add_user(16 * M);
    void *p = f.get(16 * M);
    assert(p && Fake::held == 16 * M && !f.get(16 * M + 1));
    f.add_user(M);
    assert(f.get(M) == p && Fake::held == 16 * M);
    f.add_user(16 * M + 1);
    assert(f.get(64 * M) && f.get(64 * M) != p && Fake::held == 80 * M);
    f.add_user(100 * M);
    assert(!f.get(65 * M) && !Fake::sticky);
    f.drop_user(); f.drop_user(); f.drop_user();
    assert(f.get(M) == p && Fake::held == 80 * M);   // a captured call may hold either
    f.drop_user();
    assert(!f.get(M) && Fake::held == 0);
    """)


def test_pool(tmp_path):
    """a further buffer for each stream that overlaps, none for a fifth; all go back with the last user"""
    run(tmp_path, r"""
    OperandPool<Fake> pool;
    Fake::room = 1000;
    pool.add_user();
    pool.reserve(100);
    assert(Fake::held == 100);
    void *p[5];
    for (int round = 0; round < 2; ++round)
        for (int st = 1; st <= 5; ++st) {
            auto l = pool.take(100, st);
            if (l.p) l.launched();
            if (round == 0) {
                p[st - 1] = l.p;
                for (int i = 0; i < st - 1; ++i) assert(l.p != p[i]);
            }
            assert(l.p == p[st - 1] && Fake::held == 100u * (round ? 4 : st < 5 ? st : 4));
        }
    assert(p[3] && !p[4]);
    pool.drop_user();
    assert(Fake::held == 0);
    """)
