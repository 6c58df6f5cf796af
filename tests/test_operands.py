"""The rules of the decoded operands' device memory (p8x_operands.h) on counted stand-ins for the device calls. CPU only:
each test is a C++ program built with g++."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pingala8-llm_amd", "csrc")

FAKE = r"""
#include <cassert>
#include <cstdio>
#include <cstdlib>
#include <string>
#include "p8x_operands.h"
struct Fake {   // log: a = alloc, f = free, s = device synchronize, c = error cleared
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
std::string Fake::log; size_t Fake::room, Fake::held; bool Fake::sticky;
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
