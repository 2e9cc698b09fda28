"""Runs library calls on the CPU against a HIP runtime without a device (host_hip.c): which kernels
a call launches, what it allocates and what it does when a call of the runtime fails.  In a child
process, because the library of the test process is bound to the real runtime."""
import os
import subprocess
import sys
import textwrap
from pathlib import Path

HERE = Path(__file__).parent

PREAMBLE = """
import ctypes, os, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.host_hip_launch.restype = ctypes.c_char_p
fake.host_hip_allocated.restype = ctypes.c_size_t
fake.host_hip_malloc_limit.argtypes = [ctypes.c_size_t]
sys.path.insert(0, sys.argv[2])
import numpy as np
import wgml_amd as W
from wgml_amd import _lib
from wgml_amd.models import *
NO_LIMIT = 2 ** 64 - 1

def launched(call):
    "names (mangled) of the kernels that `call` launches"
    fake.host_hip_clear()
    call()
    return [fake.host_hip_launch(i).decode() for i in range(fake.host_hip_launches())]

def workgroups(call):
    "of each kernel that `call` launches"
    return [fake.host_hip_workgroups(i) for i in range(len(launched(call)))]

def count(names, part):
    return sum(part in n for n in names)

def zeros(qtype, nrows, ncols):
    return HostMatrix(qtype, nrows, ncols, np.zeros(W.quant_bytes(qtype, nrows * ncols), np.uint8))

def llama(gpu, cfg, qtype=W.Q8_0, model_type=LlamaModelType.Llama):
    c, m = cfg, Llama2(gpu, cfg, model_type)
    shapes = {"attn_q": (c.dim, c.dim), "attn_k": (c.kv_dim, c.dim), "attn_v": (c.kv_dim, c.dim),
              "attn_output": (c.dim, c.dim), "ffn_gate": (c.hidden_dim, c.dim),
              "ffn_up": (c.hidden_dim, c.dim), "ffn_down": (c.dim, c.hidden_dim)}
    for l in range(c.n_layers):
        for name, (r, k) in shapes.items():
            m.set_matrix(name, l, zeros(qtype, r, k))
        m.set_vector("attn_norm", l, np.ones(c.dim))
        m.set_vector("ffn_norm", l, np.ones(c.dim))
    m.set_matrix("output", 0, zeros(qtype, c.vocab_size, c.dim))
    m.set_vector("output_norm", 0, np.ones(c.dim))
    te = np.zeros((c.vocab_size, c.dim), np.float32)
    _lib.call("wgml_llama2_set_token_embd", m._h, te.ctypes.data_as(ctypes.c_void_p))
    return m

def gpt2(gpu, p, qtype=W.Q8_0):
    return Gpt2(gpu, p).load(synth_gpt2(p, 1, qtype))

os.environ["WGML_DISABLE_GRAPHS"] = "1"
gpu = W.GpuInstance(0)
"""


def build(tmp_path_factory):
    out = tmp_path_factory.mktemp("host_hip") / "libamdhip64.so.7"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-Wl,-soname,libamdhip64.so.7", "-o", str(out), str(HERE / "host_hip.c")], check=True)
    return out


def run(runtime, code, timeout=120):
    """Runs `code` behind PREAMBLE; its assertions are the test's."""
    p = subprocess.run([sys.executable, "-c", PREAMBLE + textwrap.dedent(code), str(runtime), str(HERE.parent)],
                       capture_output=True, text=True, timeout=timeout, env=dict(os.environ))
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout
