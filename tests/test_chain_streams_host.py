"""The chain of blocks on two streams, without a GPU: the host code of csrc/chain.hip linked against recording stubs of the
HIP runtime and of the entry points it calls, one of which can be made to fail."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "vtpack_amd", "csrc")
MAIN, SIDE = "0x100", "0x200"

RUNTIME = r"""
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <string>
#include <thread>
#include <vector>
#include "vtdge.h"

static std::string fail_name;
static int fail_at = 0, seen = 0;
static uintptr_t events = 0;
static int step(const char *name, void *stream)
{
    printf("launch %s %p\n", name, stream);
    return fail_name == name && seen++ == fail_at ? VTDGE_ERR_LAUNCH : 0;
}
namespace vtdge {
void set_error(const char *, ...) {}
void note_kernel(const void *) {}
int check_launch(const char *) { return 0; }
}
extern "C" {
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipEventCreateWithFlags(void **e, unsigned) { *e = (void *)++events; printf("create %p\n", *e); return 0; }
int hipEventDestroy(void *e) { printf("destroy %p\n", e); return 0; }
int hipEventRecord(void *e, void *s) { printf("record %p %p\n", e, s); return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned) { printf("wait %p %p\n", e, s); return 0; }
int hipLaunchKernel() { return 0; }
int __hipPushCallConfiguration() { return 0; }
int __hipPopCallConfiguration() { return 0; }
void **__hipRegisterFatBinary(const void *) { static void *p; return &p; }
void __hipRegisterFunction() {}
void __hipUnregisterFatBinary(void **) {}
@STUBS@
}
static int run()
{
    vtdge_chain c;
    memset(&c, 0, sizeof(c));
    c.B = 2; c.H = c.W = 8; c.C = 64; c.heads = 1; c.hidden = 256; c.extra = 0; c.S = 3; c.depth = 3; c.dtype = VTDGE_F32;
    c.sr = 2; c.splits_124 = 1; c.eps1 = c.eps2 = c.sr_eps = 1e-6f; c.scale = 0.125f;
    std::vector<const void *> params(3 * VTDGE_CHAIN_PARAMS, (const void *)0x1000);
    void *p = (void *)0x1000;
    return vtdge_chain_forward(&c, params.data(), nullptr, p, p, p, p, p, (void *)@MAIN@, (void *)@SIDE@);
}
int main(int argc, char **argv)
{
    if (argc > 2) { fail_name = argv[1]; fail_at = atoi(argv[2]); }
    if (argc == 2)
        for (int i = 0; i < atoi(argv[1]); i++) std::thread([] { if (run() != 0) exit(3); }).join();
    else printf("rc %d\n", run());
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("hipcc") is None:
        pytest.skip("needs hipcc")
    obj = os.path.join("build", "chain.o")
    subprocess.run(["make", "-C", CSRC, obj], check=True, capture_output=True)
    wanted = set(re.findall(r"U (vtdge_\w+)", subprocess.run(["nm", "-u", os.path.join(CSRC, obj)], check=True,
                                                             capture_output=True, text=True).stdout))
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "vtdge.h")).read(), flags=re.S)
    stubs = []
    for kind, name, args in re.findall(r"(int|int64_t)\s+(vtdge_\w+)\s*\(([^;]*?)\)\s*;", text, flags=re.S):
        if name in wanted:
            body = f'return step("{name}", stream);' if re.search(r"\bvoid \*stream\b", args) else "return 0;"
            stubs.append(f"{kind} {name}({args}) {{ {body} }}")
    assert len(stubs) == len(wanted)
    folder = tmp_path_factory.mktemp("chain")
    src, exe = folder / "stubs.cpp", folder / "chain"
    src.write_text(RUNTIME.replace("@STUBS@", "\n".join(stubs)).replace("@MAIN@", MAIN).replace("@SIDE@", SIDE))
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "include"), str(src), os.path.join(CSRC, obj), "-o",
                    str(exe), "-lpthread"], check=True, capture_output=True)

    def go(*args):
        return subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True, text=True).stdout.splitlines()
    return go


def _ordered(log):
    """Walks a log: everything launched on the side stream is waited for by the main one at its end."""
    forked, joins, open_work = False, set(), False
    for line in log:
        w = line.split()
        if w[0] == "wait" and w[2] == SIDE:
            forked = True
        elif w[0] == "launch" and w[2] == SIDE:
            assert forked
            open_work = True
            joins.clear()
        elif w[0] == "record" and w[2] == SIDE:
            joins.add(w[1])
        elif w[0] == "wait" and w[2] == MAIN and w[1] in joins:
            open_work = False
    return forked and not open_work


def test_a_whole_chain_joins_its_streams(program):
    log = program()
    assert "rc 0" in log and _ordered(log)
    assert sum(line.startswith("launch") and line.endswith(SIDE) for line in log) >= 6


@pytest.mark.parametrize("name,count", [("vtdge_router", 1), ("vtdge_index_to_patch", 3), ("vtdge_compress", 3),
                                        ("vtdge_layernorm", 9), ("vtdge_patch_linear", 3), ("vtdge_linear_prepacked", 15),
                                        ("vtdge_sparse_attention", 3), ("vtdge_decompress_router", 2)])
def test_a_launch_that_fails_leaves_the_streams_joined(program, name, count):
    """The caller frees the buffers when the call returns: the side stream must be ordered before what takes them next."""
    whole = program()
    assert sum(line.split()[1] == name for line in whole if line.startswith("launch")) == count
    for at in range(count):
        log = program(name, at)
        assert "rc 0" not in log and _ordered(log), (name, at)


def test_the_events_of_a_thread_end_with_it(program):
    log = program(5)
    made = sum(line.startswith("create") for line in log)
    assert made >= 2 and made == sum(line.startswith("destroy") for line in log)
