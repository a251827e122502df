"""The library's host side on the CPU, its HIP runtime replaced by a stand-in
(hip_stand_in.cc) whose kernels do nothing and are logged by name: a pass
whose launch fails, and which kernels a pass takes. What the kernels compute
is the GPU tests' matter."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PRELUDE = """
import ctypes as C, json, re, sys
import numpy as np
sys.path.insert(0, %r)
from chattorrent_amd import ccdecode as cc, configs
hip = C.CDLL(%r)
hip.stand_in_reset.argtypes = [C.c_long]
hip.stand_in_launches.restype = C.c_char_p

def launched():
    return hip.stand_in_launches().decode().split()

def rows(n, d):
    return np.zeros((n, d["hidden"]), np.uint16)
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """host(code): runs it in a process whose HIP runtime is the stand-in and returns its `out`."""
    so = str(tmp_path_factory.mktemp("hip") / "stand_in.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(ROCM, "include"), os.path.join(HERE, "hip_stand_in.cc"), "-o", so], check=True)

    def run(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE % (ROOT, so) + code + "\nprint(json.dumps(out))"], cwd=ROOT,
                           env=dict(os.environ, LD_PRELOAD=so), stdout=subprocess.PIPE, stderr=subprocess.PIPE,
                           text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-2000:]
        return json.loads(r.stdout.splitlines()[-1])

    return run


@pytest.mark.parametrize("n", [5, 300])
def test_failed_launch_leaves_the_callers_rows(host, n):
    """Whichever launch of a pass fails, the call says so and hidden_out is
    untouched, also where the rows leave in pieces (300 rows of 4096); the
    next pass succeeds and writes it."""
    out = host(f"""
n = {n}
d = configs.with_layers(configs.LLAMA8B, 1)
c = cc.Context(d, n_max=320, t_max=n, slots=1, lo=1, hi=2)
job = cc.Job(slot=0, n=n)
given = rows(n, d)
job.hidden = given.ctypes.data_as(C.POINTER(C.c_uint16))
hid = np.empty_like(given)
out = []
def step(fail):
    hip.stand_in_reset(fail)
    hid[:] = 0x1234
    return c.lib.cc_step(c.h, C.byref(job), 1, 1, 2, 0, None, None, hid.ctypes.data, None)
ok = step(-1) or step(-1)   # the first takes the job's pages
total = len(launched())
for k in sorted({{0, 1, total // 2, total - 2, total - 1}}):
    out.append([step(k), bool((hid == 0x1234).all())])
out = dict(failed=out, before=ok, after=step(-1), written=bool((hid == 0).all()), launches=total)
""")
    assert out["before"] == 0 and out["after"] == 0 and out["written"] and out["launches"] > 8
    assert out["failed"] == [[8, True]] * 5   # CC_EDEVICE


@pytest.mark.parametrize("jobs,few", [
    ([(0, 1)], True), ([(0, 2)], True), ([(0, 3)], False), ([(1, 1)], True), ([(2, 1)], False), ([(8, 1)], False),
    ([(0, 2)] * 4, True), ([(0, 4)] * 4, False), ([(2, 1)] * 4, False),
    ([(0, 3)] * 16, True), ([(0, 4)] * 16, False), ([(2, 1)] * 16, True), ([(3, 1)] * 16, False),
    ([(0, 5)] + [(0, 1)] * 15, True), ([(0, 19)] + [(0, 1)] * 15, True), ([(0, 20)] + [(0, 1)] * 15, False),
    ([(8, 1)] + [(0, 1)] * 15, True), ([(8, 1)] * 8 + [(0, 1)] * 8, False), ([("verify", 4)] * 16, True),
    ([("verify", 5)] * 16, False), ([("verify", 4)] * 8 + [(0, 1)] * 8, True)])
def test_recurrence_kernel_by_the_rows_walked(host, jobs, few):
    """Each job is (kept rows, or a verify; new rows): a rollback's kept rows
    are walked too, and a long job among many short ones does not move them
    all to the long jobs' kernel. 48 heads of 128 x 128 on 256 CUs."""
    out = host(f"""
jobs = {jobs}
d = dict(configs.QWEN38, n_layer=1, layer_types=["linear_attention"], mtp_vocab=0)
c = cc.Context(d, n_max=64, t_max=256, slots=len(jobs), sessions=len(jobs), lo=1, hi=2)
def step(**kw):
    c.step([dict(slot=s, n=kw["n"][s], past=kw["past"][s], hidden=rows(kw["n"][s], d), snap=bool(kw["snap"][s]),
                 keep=kw["keep"][s]) for s in range(len(jobs))], at=1, to=2)
J, verify = len(jobs), [k == "verify" for k, _ in jobs]
kept = [0 if v else k for v, (k, _) in zip(verify, jobs)]
first = [8 if k else 1 for k in kept]
step(n=[9] * J, past=[0] * J, snap=[0] * J, keep=[None] * J)
step(n=first, past=[9] * J, snap=kept, keep=[None] * J)
hip.stand_in_reset(-1)
step(n=[n for _, n in jobs], past=[9 + (k or 1) for k in kept], snap=verify, keep=[k or None for k in kept])
out = [k for k in launched() if "k_gdn" in k]
""")
    assert len(out) == 1 and ("k_gdn_few" in out[0]) == few, out


@pytest.mark.parametrize("shape,blocks,chats,rows,past", [
    ("SMOLLM2", 3, 1, 1, 300), ("SMOLLM2", 3, 1, 1, 9000), ("SMOLLM2", 3, 4, 1, 100), ("SMOLLM2", 3, 1, 9, 100),
    ("SMOLLM2", 2, 17, 1, 100), ("LLAMA8B", 2, 1, 1, 100), ("LLAMA8B", 2, 2, 3, 100), ("M27B", 2, 1, 1, 100),
    ("M27B", 2, 4, 1, 100), ("M27B", 2, 1, 16, 100), ("M27B", 2, 40, 1, 100), ("QWEN38", 4, 1, 1, 0),
    ("QWEN38", 4, 2, 8, 0)])
def test_profile_replays_the_passs_own_matmuls(host, shape, blocks, chats, rows, past):
    """cc_profile times the kernels that the pass ran: each class's launches
    are the pass's, block by block, also where few rows let a matmul form its
    operand itself. (A linear_attention block's first matmul and out_proj are
    in no class.)"""
    out = host(f"""
chats, n, past = {chats}, {rows}, {past}
d = configs.with_layers(configs.{shape}, {blocks})
d["mtp_vocab"] = 0
kinds = d.get("layer_types") or ["full_attention"] * {blocks}
c = cc.Context(d, n_max=64 * (past // 64 + 2), t_max=chats * n, slots=chats, sessions=chats, lo=1, hi=1 + {blocks})
jobs = [dict(slot=s, past=past, n=n, hidden=rows(n, d)) for s in range(chats)]
def matmuls():
    hip.stand_in_reset(-1)
    c.step(jobs, at=1, to=1 + {blocks})
    return [k for k in launched() if "k_gemm" in k]
own = matmuls()
c.profile(True)
both = matmuls()
out = dict(own=own, both=both, full=[k == "full_attention" for k in kinds])
""")
    own, full = out["own"], out["full"]
    assert out["both"][:len(own)] == own and len(own) == 4 * blocks
    block = [own[4 * b:4 * b + 4] for b in range(blocks)]
    want = [block[b][i] for i in range(4) for b in range(blocks) if full[b] or i > 1]
    assert out["both"][len(own):] == want


@pytest.mark.parametrize("shape,tokens,wide", [
    ("smollm2", 130, True), ("27b", 700, True), ("d256", 700, True),
    ("smollm2", 11050, False), ("27b", 33420, False), ("d256", 34000, False)])
def test_attention_kernel_by_the_items(host, shape, tokens, wide):
    """Which kernel the attention tests of test_gpu_kernels.py reach with one
    decode row: four waves an item while items are few, one wave an item at
    the contexts of its many-item test."""
    out = host(f"""
sys.path.insert(0, {HERE!r})
import test_gpu_kernels as K
base, long = K.MANY_ITEMS[{shape!r}]
tokens = {tokens}
assert tokens < 1024 or tokens == long
d = configs.with_layers(base, 1)
c = cc.Context(d, n_max=64 * (tokens // 64 + 2), t_max=64, slots=1)
c.fill_random_kv(0, tokens + 1, 1, 1)
hip.stand_in_reset(-1)
c.op_attend(0, 0, np.zeros((1, d["n_heads"] * d["head_dim"]), np.float32), tokens)
out = [k for k in launched() if "k_attn" in k and "combine" not in k]
""")
    assert len(out) == 1 and ("k_attn_wide" in out[0]) == wide, out


@pytest.mark.parametrize("shape", ["SMOLLM2", "LLAMA8B", "QWEN38", "WIDE", "D256"])
def test_few_rows_merge_chunks_in_o_proj(host, shape):
    """Which cases of test_gpu_pass.py's chunk-merging test take the merge
    inside o_proj's matmul: up to 64 chunks, while a workgroup's columns times
    rows are at most 16."""
    out = host(f"""
sys.path.insert(0, {HERE!r})
import test_gpu_pass as P
at, run, rws = P.MERGE_CASES[{shape!r}]
d, out = P.merge_dims({shape!r}), []
for chunks in (1, 64, 65):
    past = 64 * run * chunks - max(rws) - 3
    c = cc.Context(d, n_max=past + 64, t_max=17, slots=2, lo=at, hi=at + 1)
    c.fill_random_kv(0, past, 1, 1)
    for n in rws:
        hip.stand_in_reset(-1)
        c.step([dict(slot=0, past=past, n=n, hidden=rows(n, d))], at=at, to=at + 1)
        k = launched()
        inside = any(re.search("k_gemm_lxILi1ELb.ELi3E", x) for x in k)
        assert inside != any("k_attn_combine" in x for x in k)
        out.append([chunks, n, inside])
""")
    most = {"SMOLLM2": 8, "LLAMA8B": 1, "QWEN38": 0, "WIDE": 8, "D256": 16}[shape]
    for chunks, n, inside in out:
        assert inside == (chunks <= 64 and n <= most), (chunks, n)
    assert any(i for _, _, i in out) == (most > 0)
