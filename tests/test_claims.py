"""Which process's waiting kernels a device may hold (csrc/claims.hpp), on the
host: programs against the header take and give a device's locks in a folder of
the test."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# a command per line of stdin: take ("+") or give ("-"), alone ("a") or shared ("s"), the device's name
PROGRAM = r"""
#include <cstdio>
#include <iostream>
#include "claims.hpp"
int main(int, char** argv) {
  avbd::Claims claims(argv[1]);
  std::string line;
  while (std::getline(std::cin, line)) {
    const avbd::Claim what = line[1] == 'a' ? avbd::Claim::Alone : avbd::Claim::Shared;
    if (line[0] == '+') printf("%d\n", claims.take(line.substr(2), what) ? 1 : 0);
    else if (line[0] == '-') { claims.give(line.substr(2), what); printf("ok\n"); }
    fflush(stdout);
  }
}
"""


class Process:
    def __init__(self, program, folder):
        self.p = subprocess.Popen([program, str(folder)], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)

    def ask(self, line):
        self.p.stdin.write(line + "\n")
        self.p.stdin.flush()
        return self.p.stdout.readline().strip()

    def end(self, kill=False):
        if self.p.stdin.closed:
            return
        if kill:
            self.p.kill()
        self.p.stdin.close()
        self.p.wait(timeout=20)
        self.p.stdout.close()


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("claims")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "avbd-metal_amd", "csrc"),
                    str(d / "main.cpp"), "-o", str(d / "claims")], check=True, timeout=120)
    return str(d / "claims")


@pytest.fixture()
def two(program, tmp_path):
    a, b = Process(program, tmp_path), Process(program, tmp_path)
    yield a, b
    a.end()
    b.end()


def test_alone(two):
    a, b = two
    assert [a.ask("+a0000:05:00.0"), a.ask("+a0000:05:00.0")] == ["1", "1"]  # counted
    assert [b.ask("+a0000:05:00.0"), b.ask("+s0000:05:00.0")] == ["0", "0"]
    assert b.ask("+a0000:15:00.0") == "1"  # another device
    assert a.ask("+s0000:15:00.0") == "0"
    a.ask("-a0000:05:00.0")
    assert b.ask("+a0000:05:00.0") == "0"
    a.ask("-a0000:05:00.0")
    a.ask("-a0000:05:00.0")  # one too many
    assert b.ask("+a0000:05:00.0") == "1"
    assert a.ask("+a0000:05:00.0") == "0"


def test_shared(two):
    a, b = two
    assert [a.ask("+s0"), b.ask("+s0"), b.ask("+s0")] == ["1", "1", "1"]
    assert [a.ask("+a0"), b.ask("+a0")] == ["0", "0"]
    b.ask("-s0")
    assert a.ask("+a0") == "0"  # a failed attempt keeps the shared lock
    a.ask("-s0")
    assert b.ask("+a0") == "1"  # beside its own shared one
    assert [a.ask("+s0"), a.ask("+a0")] == ["0", "0"]
    b.ask("-a0")
    assert [a.ask("+a0"), a.ask("+s0")] == ["0", "1"]  # shared again, never free
    b.ask("-s0")
    assert a.ask("+a0") == "1"
    a.ask("-s0")
    assert b.ask("+s0") == "0"


@pytest.mark.parametrize("kill", [False, True])
def test_locks_end_with_their_process(two, kill):
    a, b = two
    assert a.ask("+a0") == "1" and b.ask("+a0") == "0"
    a.end(kill)
    assert b.ask("+a0") == "1"


def test_without_a_folder_nothing_is_claimed(program, tmp_path):
    a = Process(program, tmp_path / "missing")
    try:
        assert a.ask("+a0") == "0" and a.ask("-a0") == "ok" and a.ask("+s0") == "0"
    finally:
        a.end()


def test_file_of_another_kind_is_refused(program, tmp_path):
    os.symlink(tmp_path / "elsewhere", tmp_path / "avbd_device_0")
    os.mkdir(tmp_path / "avbd_device_1")
    a = Process(program, tmp_path)
    try:
        assert a.ask("+a0") == "0" and a.ask("+a1") == "0"
        assert not os.path.exists(tmp_path / "elsewhere")
    finally:
        a.end()
