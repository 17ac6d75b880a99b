"""CPU test of the order in which a decode launch closes its call. The call's tag comes from a device word that every wavefront
loads and the last workgroup to finish moves on: a workgroup may only be counted as finished when all of its wavefronts have the word
in a register, so each takes it (df_tag, which pins it there) in front of a barrier of the workgroup. Looked up in the source, since a
wavefront that comes late depends on timing that a run does not show."""
import os
import re

import pytest

from conftest import ROOT


def functions(pattern):
    """name -> body of the functions of the decode kernels' source whose head matches `pattern` (its group is the name)"""
    with open(os.path.join(ROOT, "cudalm-c_amd", "csrc", "qlmx_gemv.hip")) as f:
        src = re.sub(r"/\*.*?\*/", "", f.read(), flags=re.S)
    found = {}
    for m in re.finditer(pattern + r"\([^{]*\{", src):
        depth, i = 1, m.end()
        while depth:
            depth += {"{": 1, "}": -1}.get(src[i], 0)
            i += 1
        found[m.group(1)] = src[m.end():i]
    return found


def closing_kernels():
    return {k: b for k, b in functions(r"__global__ void [^{]*?(k_\w+)").items() if "__hip_atomic_fetch_add(a.ctl" in b}


def test_the_kernels_are_found():
    assert sorted(closing_kernels()) == ["k_decode_few", "k_decode_fused"]


def test_the_tag_is_pinned():
    body = functions(r"unsigned (df_tag)")["df_tag"]
    assert re.search(r"readfirstlane\(.*asm volatile\(\"\" :: \"s\"\(t\)", body, flags=re.S)


@pytest.mark.parametrize("name", ["k_decode_fused", "k_decode_few"])
def test_every_wavefront_has_the_tag_in_front_of_a_barrier(name):
    body = closing_kernels()[name]
    close = body.index("if(tid == 0){\n        const unsigned done = __hip_atomic_fetch_add(a.ctl + 1")
    task = functions(r"void (df_task_i8)")["df_task_i8"]
    assert task.index("__syncthreads();") < task.index("df_st(")
    taken = [m.end() for m in re.finditer(r"a\.epoch = ", body[:close])]
    assert taken and "epoch" not in body[:taken[0] - len("a.epoch = ")]
    for at, end in zip(taken, taken[1:] + [close]):
        assert body[at:].startswith("df_tag(last);"), name
        assert re.match(r"df_tag\(last\);\s*__syncthreads\(\);", body[at:]) or "df_task_i8(" in body[at:end], name


def test_nobody_clears_the_give_up_word_of_another_wavefront():
    """k_decode_few has no barrier between the clearing and the first wait, so a wavefront's word is its own."""
    body = closing_kernels()["k_decode_few"]
    assert "__shared__ int giveup[4];" in body and "giveup[tid >> 6] = 0;" in body
    assert body.count("&giveup") == body.count("&giveup[tid >> 6]") > 0
