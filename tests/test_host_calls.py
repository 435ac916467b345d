"""Which HIP calls the engine makes, and in which order (no GPU needed): liblnt.so runs on a HIP
runtime without a device (tests/emu/fake_hip.cpp) that writes the calls to a log."""
import json
import os
import subprocess
import sys

import pytest

from helpers import HERE, ROOT

FAKE_SRC = os.path.join(HERE, "emu", "fake_hip.cpp")
FAKE_SO = os.path.join(HERE, "emu", "_build", "libfakehip.so")

PRELUDE = """
import ctypes, json, sys
fake = ctypes.CDLL(%r, ctypes.RTLD_GLOBAL)  # ahead of the HIP runtime that liblnt.so names
fake.fake_log.restype = ctypes.c_char_p
sys.path.insert(0, %r)
import cuda_amd

def log():
    return [l.split() for l in fake.fake_log().decode().splitlines()]

def stream_of(t):  # the context was the last to make calls
    return log()[-1][1]
"""


@pytest.fixture(scope="module")
def fake():
    """Runs a script on the fake runtime; its last line of output is JSON."""
    if not os.path.exists(FAKE_SO) or os.path.getmtime(FAKE_SRC) > os.path.getmtime(FAKE_SO):
        os.makedirs(os.path.dirname(FAKE_SO), exist_ok=True)
        tmp = f"{FAKE_SO}.{os.getpid()}.tmp"
        subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", "-o", tmp, FAKE_SRC], check=True)
        os.replace(tmp, FAKE_SO)

    def run(script, **env):
        r = subprocess.run([sys.executable, "-c", PRELUDE % (FAKE_SO, ROOT) + script], capture_output=True,
                           text=True, timeout=300, env={**os.environ, **env})
        assert r.returncode == 0, r.stdout + r.stderr
        return json.loads(r.stdout.splitlines()[-1])
    return run


def ordered_before(log):
    """Per stream, the launches that work enqueued on it now comes after: those of the stream
    itself, of the streams that it waits for, and what the host waited for."""
    seen, events, host, launches = {}, {}, set(), []
    for i, (op, stream, *arg) in enumerate(log):
        s = seen.setdefault(stream, set())
        s |= host
        if op in ("launch", "graph"):
            s.add(i)
            launches.append((i, stream))
        elif op == "record":
            events[arg[0]] = set(s)
        elif op == "wait":
            s |= events.get(arg[0], set())
        elif op == "sync":
            host |= s
    return seen, launches


@pytest.mark.parametrize("block", [1000, 40])
def test_failed_batch_step_is_joined_and_counted(fake, block):
    """A batch step whose second group fails: the members' streams wait for what the first group
    launched, and a checked member of it counts those squarings, the end of a block included."""
    got = fake("""
block = %d
a = cuda_amd.LucasPRP(1000003, prp=True); sa = stream_of(a)
b = cuda_amd.LucasPRP(2000003, prp=True); sb = stream_of(b)
a.gerbicz_begin(block, 1)
batch = cuda_amd.Batch()
batch.add(a); batch.add(b)
batch.iterate(40)
fake.fake_clear()
fake.fake_fail(b"graph", 3)  # the first of the second group
try:
    batch.iterate(40)
    failed = False
except cuda_amd.LntError:
    failed = True
print(json.dumps(dict(log=log(), sa=sa, sb=sb, failed=failed, st=a.gerbicz_stats())))
""" % block)
    assert got["failed"]
    seen, launches = ordered_before(got["log"])
    of_groups = {i for i, s in launches if s not in (got["sa"], got["sb"])}
    assert len(of_groups) >= 10
    assert of_groups <= seen[got["sa"]] and of_groups <= seen[got["sb"]]
    assert got["st"]["iteration"] == 80 and got["st"]["checks"] == (2 if block == 40 else 0)


def test_failed_parameter_copy_is_made_up_for(fake):
    """The members' "-2" flags change after their first iteration; if copying them fails, the next
    step copies them before it launches anything."""
    got = fake("""
t = cuda_amd.LucasPRP(1000003)
batch = cuda_amd.Batch()
batch.add(t)
fake.fake_fail(b"copy", 2)  # the first is that of new groups
try:
    batch.iterate(5)
    failed = False
except cuda_amd.LntError:
    failed = True
fake.fake_clear()
batch.iterate(5)
print(json.dumps(dict(failed=failed, ops=[l[0] for l in log() if l[0] in ("copy", "launch")])))
""")
    assert got["failed"] and got["ops"] == ["copy"] + ["launch"] * 15


def test_short_batch_steps_replay_graphs(fake):
    """Steps of one iteration launch one graph of all groups from the second such step on, and the
    first captures nothing; a step of 16 with several row/column groups is one graph launch for
    each once the members' "-2" flags are right."""
    got = fake("""
ps = (9689, 1000003, 2000003)  # one workgroup, rows and columns
ts = [cuda_amd.LucasPRP(p) for p in ps]
batch = cuda_amd.Batch()
for t in ts:
    batch.add(t)
steps = []
for k in (1, 1, 1, 16, 16, 1):
    fake.fake_clear()
    batch.iterate(k)
    steps.append([(l[0], l[2]) for l in log() if l[0] in ("launch", "graph", "capture")])
print(json.dumps(steps))
""")
    one = ["graph", "7"]  # 1 + 3 + 3 kernels
    assert [s[0] for s in got[0]] == ["launch"] * 7
    assert got[1] == [["capture", "7"], one]
    assert got[2] == [one] and got[5] == [one]
    for step, captures in ((got[3], 2), (got[4], 0)):
        assert [s for s in step if s[0] == "graph"] == [["graph", "48"]] * 2
        assert len([s for s in step if s[0] == "launch"]) == 1  # the one-workgroup test's
        assert len([s for s in step if s[0] == "capture"]) == captures


def test_batch_makes_its_streams_once(fake):
    """Groups that are formed again as members come and go run on the streams that were made with
    the batch, more groups than streams included."""
    got = fake("""
made = lambda: {l[1] for l in log() if l[0] == "stream"}
batch = cuda_amd.Batch()
streams = made()
steps = []
ts = []
for p in (9689, 86243, 132049, 250007, 400009, 1000003, 2000003):
    ts.append(cuda_amd.LucasPRP(p))
    batch.add(ts[-1])
    fake.fake_clear()
    batch.iterate(3)
    batch.iterate(40)
    steps.append((len(made()), sorted({l[1] for l in log() if l[0] in ("launch", "graph")})))
print(json.dumps(dict(streams=sorted(streams), steps=steps, groups=batch.stats()["groups"])))
""")
    assert got["groups"] == 7 and len(got["streams"]) == 5
    for i, (made, used) in enumerate(got["steps"]):
        assert made == 0 and set(used) < set(got["streams"]) and len(used) == min(i + 1, 4)


def test_long_batch_steps_launch_the_groups_in_turns(fake):
    """A stream takes only so many launches ahead of the device: in a long step no group's launches
    run ahead of another's by more than a few hundred iterations."""
    got = fake("""
ts = [cuda_amd.LucasPRP(p) for p in (86243, 1000003, 2000003)]
batch = cuda_amd.Batch()
for t in ts:
    batch.add(t)
batch.iterate(5)
fake.fake_clear()
batch.iterate(20001)
print(json.dumps([l for l in log() if l[0] in ("launch", "graph")]))
""")
    done, ahead = {}, 0  # graph and kernel launches: 48 and 1 thirds of an iteration
    for op, stream, what in got:
        if "small" in what:
            continue
        done[stream] = done.get(stream, 0) + (48 if op == "graph" else 1)
        ahead = max(ahead, max(done.values()) - (min(done.values()) if len(done) == 2 else 0))
    assert sorted(done.values()) == [60003, 60003] and ahead <= 3 * 300
    small = [l for l in got if "small" in l[2]]
    assert len(small) == -(-20001 // 256) and len({l[1] for l in got}) == 3
    first = {}
    for i, l in enumerate(got):
        first.setdefault(l[1], i)
    assert max(first.values()) < 60  # every group has begun after one turn of the others


def test_tuner_offers_the_one_workgroup_plan(fake):
    """A context of 2048 or 4096 words on a row/column plan (a saved choice of its length) can be
    tuned back to the one-workgroup kernel, which no row length names."""
    got = fake("""
out = []
for p, n in ((44497, 2048), (86243, 4096)):
    cuda_amd.lnt.tune_import("0 %d 7 16 -1 -1\\n" % n)
    t = cuda_amd.LucasPRP(p, n)
    out.append((t.describe()[0], (t.tune(10), [name for name, ms in t.tune_results()])[1]))
print(json.dumps(out))
""")
    for (plan, names), kernel in zip(got, ("lnt_k_small16<8>", "lnt_k_small16<16>")):
        assert plan.startswith("LNT_2PASS"), plan
        assert any(kernel in name for name in names), names


def test_products_and_copies_take_every_variant_of_a_split(fake):
    """lnt_mul and lnt_copy ask for the same p, n, mode and row/column split, whatever kernels the
    two contexts run; another split is refused."""
    got = fake("""
import os
def make(p, n, plan):
    os.environ["LNT_PLAN"] = plan
    return cuda_amd.LucasPRP(p, n, prp=True)
out = []
for p, n, a, b in ((70000027, 1 << 22, "", "K=8"), (16000057, 1 << 20, "", "col3=0"), (16000057, 1 << 20, "lc=10,K=16", "lc=10,K=8"),
                   (1000003, 65536, "lc=8", "lc=8,row3=0"), (19937, 1024, "", "row3=0"), (1279, 64, "", "row3=0"),
                   (1000003, 65536, "lc=9", "lc=10"), (1000003, 65536, "", "lc=12")):
    x, y = make(p, n, a), make(p, n, b)
    ok = []
    for call in (x.mul, x.copy_from):
        try:
            call(y)
            ok.append(True)
        except cuda_amd.LntError:
            ok.append(False)
    out.append((n, a, b, x.describe() != y.describe(), ok))
print(json.dumps(out))
""")
    for n, a, b, differ, ok in got:
        assert differ, (n, a, b)
        assert ok == [a + b not in ("lc=9lc=10", "lc=12")] * 2, (n, a, b, ok)


def test_tuner_leaves_out_register_rows(fake):
    """Rows of 256 to 2048 words have the matrix-core kernels: the tuner times no others there, and
    up to 2^20 no more plans than before those kernels came."""
    got = fake("""
out = []
for p in (1000003, 4000037, 16000057, 70000027):
    t = cuda_amd.LucasPRP(p)
    t.tune(1)
    out.append([name for name, ms in t.tune_results()])
    t.close()
print(json.dumps(out))
""")
    for names, most in zip(got, (10, 22, 23, 26)):
        assert len(set(names)) == len(names) <= most, (len(names), most)
        for name in names:
            C = int(name.split("/")[0].split("x")[1])
            assert ("lnt_k_rowm<" in name) == (256 <= C <= 2048), name
