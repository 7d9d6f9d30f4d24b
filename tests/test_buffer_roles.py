"""A recording that fails leaves the fields' buffer roles as they were
(csrc/roles.h), compiled for the host: no GPU."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "steamroller.jl_amd", "csrc")

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <memory>
#include <stdexcept>
#include <vector>
#include "roles.h"

struct Field {
    std::vector<uint8_t> cur;
};
using Fields = std::vector<std::unique_ptr<Field>>;

// the descent of a cycle, recorded: one flip on every level, then a refusal
static void record(Fields &f, bool fails) {
    srmg::RolesKeeper roles(f);
    for (auto &p : f)
        if (p)
            for (auto &c : p->cur) c ^= 1;
    if (fails) throw std::runtime_error("refused");
    roles.keep();
}

int main() {
    Fields f;
    for (int k = 0; k < 3; k++) f.push_back(std::make_unique<Field>());
    f[0]->cur = {0, 0, 0};
    f[1].reset();  // a destroyed field's place
    f[2]->cur = {1, 0};
    bool threw = false;
    try {
        record(f, true);
    } catch (const std::runtime_error &) {
        threw = true;
    }
    const bool back = f[0]->cur == std::vector<uint8_t>{0, 0, 0} && f[2]->cur == std::vector<uint8_t>{1, 0};
    record(f, false);
    const bool stays = f[0]->cur == std::vector<uint8_t>{1, 1, 1} && f[2]->cur == std::vector<uint8_t>{0, 1};
    std::printf("%d %d %d\n", threw, back, stays);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_roles_return_when_a_recording_fails(tmp_path):
    src, exe = tmp_path / "roles.cpp", tmp_path / "roles"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, stdout=subprocess.PIPE, text=True).stdout
    assert out.split() == ["1", "1", "1"]


def test_every_capture_is_guarded():
    """Captures begin in one place, under a RolesKeeper."""
    with open(os.path.join(CSRC, "srmg.hip")) as f:
        text = f.read()
    assert text.count("hipStreamBeginCapture(") == 1
    body = text[text.index("static void capture_graph("):text.index("hipStreamBeginCapture(")]
    assert "RolesKeeper" in body
