"""Threads that end while the process exits: their device memory and streams are released before HIP is torn
down or not at all."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import sys, threading
sys.path.insert(0, sys.argv[1])
import minicaffe as mc
from minicaffe import craft, zoo
spec, inputs = zoo.resnet50_spec(batch=2, size=64, stages=(2, 2, 2, 2), width=32, num_classes=7, bn_seed=3)

def work():
    mc.set_runtime_mode(1, 0)
    net = mc.Net.from_buffers(craft.to_prototxt(spec, "t"))
    craft.load_weights(net, spec)
    net.forward(**inputs)

threads = [threading.Thread(target=work) for _ in range(4)]
for t in threads:
    t.start()
for t in threads:
    t.join()          # returns before the thread's own destructors have run
print("joined", flush=True)
"""


def test_process_exits_while_its_threads_release_their_memory(gpu_mode):
    r = subprocess.run([sys.executable, "-c", PROGRAM, os.path.join(ROOT, "mini-caffe_amd")], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "joined" in r.stdout, (r.returncode, r.stdout, r.stderr[-2000:])
