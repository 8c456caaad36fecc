"""The model runner's host side without a GPU: what it allocates, frees and waits for, over a stand-in of the HIP runtime (tests/host_runtime_stand_in.cpp)."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stand_in") / "libstand_in.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-w",
                    os.path.join(ROOT, "tests", "host_runtime_stand_in.cpp"), "-o", out], check=True)

    def run(*args):
        r = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "host_runner_stand_in_worker.py"), out] + [str(a) for a in args],
                           capture_output=True, text=True, timeout=300, cwd=ROOT)
        assert r.returncode == 0, (r.stdout[-1500:], r.stderr[-3000:])
        return json.loads(r.stdout.strip().splitlines()[-1])
    return run


@pytest.mark.parametrize("graph", [0, 1])
def test_a_row_that_did_not_come_fails_the_synchronise(stand_in, graph):
    """The peer-to-peer communicator's error word behind a step: RUNTIME_ERROR with the reason, the requests back at the last good synchronise."""
    out = stand_in("lost", 0, 2, 3, 4, graph)
    assert "a peer's row did not come" in out["err"] and out["word"] == 1 and out["after"] == 3


# what may wait for work of other streams, or take and give back device memory
MEMORY = {"hipMalloc", "hipFree", "hipExtMallocWithFlags", "hipHostMalloc", "hipHostFree", "hipMemcpy", "hipMemset", "hipGraphInstantiate", "hipGraphExecDestroy", "hipGraphDestroy",
          "hipStreamBeginCapture", "hipStreamSynchronize"}


@pytest.mark.parametrize("rank,nranks,batch,wbits,graph", [(0, 8, 16, 4, 1), (1, 8, 16, 4, 1), (3, 8, 1, 4, 0), (0, 2, 16, 8, 1), (1, 4, 16, 4, 0), (0, 1, 3, 4, 1)])
def test_a_prepared_step_only_launches(stand_in, rank, nranks, batch, wbits, graph):
    """Ranks that share a GPU wait for one another in their all-reduces: behind decode_prepare a step neither frees memory (hipFree waits for everything on the device) nor
    allocates, captures or synchronises, before its first launch or behind it.  Without it a step does, a batch of 16 as late as its last operators."""
    out = stand_in("prepare", rank, nranks, batch, wbits, graph)
    assert ("hipGraphLaunch" if graph else "launch") in out["first"]
    assert not MEMORY & set(out["first"]), [c for c in out["first"] if c in MEMORY]
    assert not out["again"] and out["ids"] == batch
    plain = stand_in("unprepared", rank, nranks, batch, wbits, graph)["first"]
    assert "hipFree" in plain
