"""Processes that hold another HIP runtime than the library's own (a PyTorch
wheel brings one): the library tells, and plans of several steps then run
without capture, with the results of a plan compiled without one."""
import importlib.util
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEAD = f"import sys; sys.path.insert(0, {os.path.join(ROOT, 'php-gpu-tensors_amd')!r})\n"
TORCH_FIRST = "import torch\nfrom phptensors import _abi\nlib = _abi.load()\n"
TORCH_LAST = "from phptensors import _abi\nlib = _abi.load()\nimport torch\n"
ALONE = "from phptensors import _abi\nlib = _abi.load()\n"
RUNTIMES = "print(len({l.split()[-1] for l in open('/proc/self/maps') if '/libamdhip64.so' in l}), torch.version.hip)\n"


def _child(code):
    run = subprocess.run([sys.executable, "-c", HEAD + code], capture_output=True, text=True, timeout=240)
    assert run.returncode == 0, run.stdout[-2000:] + run.stderr[-3000:]
    return run.stdout.split("\n")


def _foreign(order):
    """What a process of that order of imports holds: skip where the wheel has no runtime of its own."""
    if importlib.util.find_spec("torch") is None:  # (not imported here: this process keeps one runtime)
        pytest.skip("no PyTorch")
    mapped, version = _child(order + RUNTIMES)[0].split(maxsplit=1)
    if mapped == "1" and (version == "None" or order == TORCH_LAST or version.startswith("7.2")):
        pytest.skip("one HIP runtime serves both")


def test_alone():
    assert _child(ALONE + "print(lib.pt_runtime_is_own(), lib.pt_runtime_is_own())")[0] == "1 1"


@pytest.mark.parametrize("order", [TORCH_FIRST, TORCH_LAST], ids=["torch-first", "torch-last"])
def test_beside_another_runtime(order):
    _foreign(order)
    assert _child(order + "print(lib.pt_runtime_is_own())")[0] == "0"


def test_a_runtime_loaded_later_is_noticed():
    _foreign(TORCH_LAST)
    got = _child(ALONE + "a = lib.pt_runtime_is_own()\nimport torch\nprint(a, lib.pt_runtime_is_own())")
    assert got[0] == "1 0"


PLANS = """
import numpy as np
from phptensors import CudaArray, Fusion, mlp
from phptensors.optimizer import Optimizer

def steps(graph):
    x, y = mlp.synthetic_batch(48, 20, 5)
    p = mlp.init_parameters((20, 33, 33, 5))
    z = lambda: [CudaArray.zeros(q.getShape()) for q in p]
    state = {"firstMoment": z(), "secondMoment": z(), "beta1Power": CudaArray.full([1], 0.9),
             "beta2Power": CudaArray.full([1], 0.999)}
    x, y, rate = CudaArray.fromNumpy(x), CudaArray.fromNumpy(y), CudaArray.full([1], 1e-3)
    ins = mlp.training_inputs(x, y, rate, p, state)
    plan = mlp.compile_training_plan(ins, Optimizer.adamW(), cuda_graph=graph)
    for _ in range(4):
        p, state, loss = mlp.unpack_step(plan.run(*ins))
        ins = mlp.training_inputs(x, y, rate, p, state)
    return [t.toNumpy() for t in ins] + [loss.toNumpy()], plan.getStats()

a, s = steps(True)
b, t = steps(False)
print(all(np.array_equal(u, v) for u, v in zip(a, b)), s["backend"], s["cudaGraphIncompatibility"], s["graphLaunches"],
      s["cudaGraphRequested"], t["backend"])
x = CudaArray.full([40, 30], 0.5)
g = Fusion.compile(lambda v: (v + v * v).tanh(), [x], cudaGraph=True)
for _ in range(3):
    r = g.run(x)
print(abs(float(r.toNumpy()[3, 4]) - float(np.tanh(0.75))) < 1e-6, g.getStats()["backend"], g.getStats()["graphLaunches"])
"""


@pytest.mark.gpu
def test_training_step_on_the_wheels_runtime():
    _foreign(TORCH_FIRST)
    got = _child(TORCH_FIRST + PLANS)
    assert got[0] == "True stream foreign-hip-runtime 0 1 stream", got
    # a plan of one step is captured on one stream, there as elsewhere
    assert got[1] == "True cuda-graph 3", got
