"""CPU checks of what the forward's host code enqueues: the library runs against a stand-in for the HIP runtime
(hip_stub.c) that records launches, event records and waits instead of executing them."""
import json
import os
import subprocess
import sys

import pytest

import torch

import slotscan_lib as L
from test_gpu_proj_rows import BACKWARD, FORWARD
from test_gpu_scan_groups import GROUPS
from test_gpu_scan_reg import CASES as REG_CASES

HERE = os.path.dirname(os.path.abspath(__file__))

# Runs in its own process, which never loads the real runtime.  `call(thread, stream, **shape)` is one slotscan_fwd.
_PRELUDE = """
import ctypes, json, sys, threading
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_log.restype = ctypes.c_char_p
stub.stub_capture.argtypes = [ctypes.c_void_p, ctypes.c_uint64]
lib = ctypes.CDLL(sys.argv[2])
vp, i64, i32, f32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float
lib.slotscan_fwd.argtypes = [vp, vp, vp, i32, vp, vp, i32, vp] + [i64] * 6 + [f32, i32] + [vp] * 14
lib.slotscan_fwd_memq.argtypes = [vp, vp, vp, i32, vp, vp, i32, vp] + [i64] * 6 + [f32, i32, i32, i64] + [vp] * 17
lib.slotscan_fwd_codes.argtypes = [vp, vp, vp, i32, vp, vp, i32, vp] + [i64] * 6 + [f32, i32, i32, i64] + [vp] * 13
def call_mode(mode, bf16, B, T, H, N, D, G):
    p = 1 << 20
    a = (p, p, p, bf16, p, p, 1, p, B, T, H, N, D, G, 1e-4, 1)
    if mode == "f32":
        return lib.slotscan_fwd(*a, None, None, None, p, p, p, None, None, None, None, p, p, p, None)
    if mode == "codes":
        return lib.slotscan_fwd_codes(*a, 8, D, None, None, None, p, p, p, p, p, p, p, p, p, None)
    return lib.slotscan_fwd_memq(*a, 3 if mode == "memq" else 0, 16, None, None, None, p, p, p, p, p, None, None, None, None,
                                 p, p, p, p, None)
lib.slotproj_fwd.argtypes = [vp, vp, vp, i64, i64, i64, vp, vp]
lib.slotproj_bwd.argtypes = [vp, vp, vp, i64, i64, i64, vp, vp, vp, vp]
def call(thread, stream, B=8, T=1024, H=6, N=192, D=128, G=8):
    stub.stub_thread(thread)
    p = 1 << 20
    return lib.slotscan_fwd(p, p, p, 1, p, p, 1, p, B, T, H, N, D, G, 1e-4, 1, None, None, None, p, p, p, None, None, None,
                            None, p, p, p, stream)
def log():
    return [l.split() for l in stub.stub_log().decode().splitlines()]
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip_stub")
    out, ver = str(d / "libamdhip64.so.7"), str(d / "version.map")
    with open(ver, "w") as f:
        f.write("hip_4.2 { global: *; };\nhip_4.5 { global: hipStreamGetCaptureInfo; };\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-pthread", os.path.join(HERE, "hip_stub.c"), "-o", out,
                    "-Wl,-soname,libamdhip64.so.7", "-Wl,--version-script=" + ver], check=True)
    return out


def _run(stub, body):
    r = subprocess.run([sys.executable, "-c", _PRELUDE + body, stub, L.LIB_PATH], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.splitlines()[-1])


def _check_waits(log):
    """Every wait of a call is for an event that the same call recorded last."""
    last = {}
    n = 0
    for op in log:
        if op[1] == "record":
            last[op[2]] = op[0]
        elif op[1] == "wait":
            n += 1
            assert last.get(op[3]) == op[0], f"a wait of call {op[0]} is for call {last.get(op[3])}'s record"
    return n


@pytest.mark.parametrize("shape", [dict(B=8, T=1024),                       # chunks of a long scan
                                   dict(B=600, T=200, H=1, N=70)])          # batch groups of a short one
def test_two_threads_keep_their_own_events(stub, shape):
    """Two host threads inside the forward on one device: neither takes the other's events, also when one is stopped
    between a record and its wait while the other records."""
    log = _run(stub, f"""
stub.stub_hold(1, 2)
rc = [None, None, None]
def go(i):
    rc[i] = call(i, 0x100 * i, **{shape!r})
a, b = threading.Thread(target=go, args=(1,)), threading.Thread(target=go, args=(2,))
a.start(); b.start(); a.join(); b.join()
assert rc[1:] == [0, 0], rc
print(json.dumps(log()))
""")
    assert _check_waits(log) >= 4
    for i in ("1", "2"):                                # and each call ends with its replays joined to its stream
        mine = [op for op in log if op[0] == i]
        side = {op[3] for op in mine if op[1] == "launch"} - {hex(0x100 * int(i))}
        assert len(side) == 1
        last_side = max(k for k, op in enumerate(mine) if op[1] == "launch" and op[3] in side)
        joined = [k for k, op in enumerate(mine) if op[1] == "record" and op[3] in side and k > last_side]
        assert joined and any(op[1] == "wait" and op[2] == hex(0x100 * int(i)) and op[3] == mine[joined[0]][2]
                              for op in mine[joined[0]:])


def test_a_set_held_by_another_capture_is_passed_over(stub):
    """While the second stream of an earlier call belongs to a graph capture, a call outside that capture takes another
    one; a call of the same capture may take it, and no third one is made."""
    side = lambda log, st: {op[3] for op in log if op[1] == "launch"} - {hex(st)}
    a, b, c, d = _run(stub, """
out = []
def one(stream):
    stub.stub_reset()
    assert call(1, stream) == 0
    return log()
out.append(one(0x100))
side = ({op[3] for op in out[0] if op[1] == "launch"} - {"0x100"}).pop()
stub.stub_capture(int(side, 16), 7)
stub.stub_capture(0x100, 7)
out.append(one(0x200))
out.append(one(0x100))
stub.stub_capture(int(side, 16), 0)
stub.stub_capture(0x100, 0)
out.append(one(0x200))
print(json.dumps(out))
""")
    assert len(side(a, 0x100)) == 1 and not side(b, 0x200) & side(a, 0x100)
    assert side(c, 0x100) | side(d, 0x200) <= side(a, 0x100) | side(b, 0x200)
    for log in (a, b, c, d):
        _check_waits(log)


@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_a_failed_launch_leaves_nothing_unjoined(stub, n):
    """A call that fails half way still joins what it put on the second stream: the caller may free or reuse the buffers
    in its own stream's order."""
    log = _run(stub, f"""
stub.stub_fail_launch({n})
assert call(1, 0x100) != 0
print(json.dumps(log()))
""")
    side = [k for k, op in enumerate(log) if op[1] == "launch" and op[3] != "0x100"]
    assert sum(op[1] == "launch" for op in log) == n + 1 and side
    joined = [k for k, op in enumerate(log) if op[1] == "record" and op[3] == log[side[0]][3] and k > side[-1]]
    assert joined and any(op[1] == "wait" and op[2] == "0x100" and op[3] == log[joined[0]][2] for op in log[joined[0]:])


def _chains(stub, shapes):
    """For each (mode, bf16, B, T, H, N, D, G): the set of chain kernels that the forward launches."""
    logs = _run(stub, f"""
out = []
for c in {shapes!r}:
    stub.stub_reset()
    assert call_mode(*c) == 0, c
    out.append([op[2] for op in log() if op[1] == "launch"])
print(json.dumps(out))
""")
    return [{"reg" if "chain_fwd_reg" in n else "lds" for n in names if "chain_fwd" in n} for names in logs]


def test_register_chain_cases_take_it(stub):
    """The cases whose outputs test_gpu_scan_reg.py compares do run the register chain, and a few of their rows the other."""
    many = [(c[0], int(c[7] == torch.bfloat16), c[1], *c[2:7]) for c in REG_CASES]
    assert _chains(stub, many) == [{"reg"}] * len(many)
    assert _chains(stub, [(*c[:2], 3, *c[3:]) for c in many]) == [{"lds"}] * len(many)


# mode, bf16 tokens, chains (H 8), N, D, the longest scan that keeps its keys in registers
@pytest.mark.parametrize("mode,bf16,chains,N,D,longest", [
    ("f32", 1, 256, 192, 128, 0), ("f32", 1, 264, 192, 128, 4096), ("f32", 1, 4096, 96, 128, 4), ("f32", 0, 1024, 96, 128, 64),
    ("f32", 0, 512, 192, 64, 128), ("f32", 0, 1024, 192, 64, 96), ("f32", 1, 1024, 96, 64, 32), ("f32", 1, 4096, 64, 128, 0),
    ("mem", 1, 256, 192, 128, 0), ("mem", 1, 264, 192, 128, 64), ("mem", 1, 512, 192, 128, 96), ("mem", 1, 4096, 192, 128, 48),
    ("mem", 1, 4096, 96, 128, 4), ("mem", 1, 1024, 128, 128, 16), ("mem", 1, 768, 128, 128, 8), ("mem", 0, 768, 192, 64, 16), ("mem", 1, 1024, 96, 64, 8),
    ("memq", 1, 1024, 192, 128, 16), ("codes", 1, 1024, 192, 128, 16), ("codes", 1, 1024, 128, 128, 8), ("codes", 1, 4096, 96, 128, 0),
])
def test_register_chain_rule(stub, mode, bf16, chains, N, D, longest):
    """Both sides of the rule's line."""
    c = lambda T: (mode, bf16, chains // 8, T, 8, N, D, 8)
    sides = ([(c(longest), {"reg"})] if longest else []) + ([(c(longest + 1), {"lds"})] if longest < 4096 else [])
    assert _chains(stub, [s for s, _ in sides]) == [want for _, want in sides]


def test_batch_group_cases_run_in_groups(stub):
    """The cases of test_gpu_scan_groups.py: one launch of the chain per group, of the batch rows stated there."""
    shapes = [(c[0], int(c[1] == torch.bfloat16), *c[2:8]) for c in GROUPS]
    logs = _run(stub, f"""
out = []
for c in {shapes!r}:
    stub.stub_reset()
    assert call_mode(*c) == 0, c
    out.append([op[2:] for op in log() if op[1] == "launch"])
print(json.dumps(out))
""")
    for c, log in zip(GROUPS, logs):
        chains = [int(op[2]) for op in log if "chain_fwd" in op[0] and "chain_fwd_reg" not in op[0]]
        rows = [int(op[2]) for op in log if "rows_fwd" in op[0]]
        B, H, group = c[2], c[4], c[8]
        assert chains == rows == [H * min(group, B - b) for b in range(0, B, group)] and len(chains) > 1


def test_projection_routes(stub):
    """The few-row kernel runs while it has at most 512 workgroups, in the forward alone: the backward's products take the
    tile kernels at every row count."""
    most = [(256, 2048), (512, 1024), (2048, 256), (4096, 128), (8192, 64)]
    shapes = [s for s, _ in FORWARD] + [(m, n, 96) for n, m in most] + [(m + 1, n, 96) for n, m in most]
    want = [rows for _, rows in FORWARD] + [True] * len(most) + [False] * len(most)
    fwd, bwd = _run(stub, f"""
out = [[], []]
p = 1 << 20
for M, N, K in {shapes!r}:
    stub.stub_reset()
    assert lib.slotproj_fwd(p, p, p, M, N, K, p, None) == 0
    out[0].append([op[2] for op in log()])
for M, N, K in {BACKWARD!r}:
    stub.stub_reset()
    assert lib.slotproj_bwd(p, p, p, M, N, K, p, p, p, None) == 0
    out[1].append([op[2] for op in log()])
print(json.dumps(out))
""")
    assert [["proj_rows" in k for k in ks] for ks in fwd] == [[w] for w in want]
    for ks in bwd:
        assert [next(n for n in ("proj_transpose", "projt_gemm", "proj_gemm", "proj_reduce", "proj_rows") if n in k) for k in ks] \
            == ["proj_transpose", "proj_gemm", "projt_gemm", "proj_reduce"]
