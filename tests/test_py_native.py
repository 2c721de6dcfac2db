"""The native entry points raise what goes wrong beneath them -- allocations that fail, tensors without strides -- as Python errors.

On the CPU, where no device memory can be had; the tensors are fakes without storage, and nothing gets as far as a launch.  The calls
run in a process of their own: an exception that left native code uncaught would end it."""
import json
import os
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CALLS = r"""
import json
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
import jittorinfer_amd as J
with FakeTensorMode():
    f = lambda *shape, dtype=torch.float32: torch.empty(shape, dtype=dtype, device="cuda")
    q, k, out = f(1, 16, 1, 576), f(1, 128, 576, dtype=torch.bfloat16), f(1, 1, 16, 512)
    x, pos, rows, cache = f(4, 16, 64), f(4, dtype=torch.int32), f(4, 576), f(128, 576, dtype=torch.bfloat16)
    w, wx = f(16, 512, 128, dtype=torch.int16), f(16, 4, 128)
sparse = torch.zeros(4, dtype=torch.int32).to_sparse()
sparse_mask = torch.zeros((1, 128), dtype=torch.float16).to_sparse()
calls = dict(
    attn=lambda: J.ggml_flash_attn_ext(q, k, J.MLA_TYPE_BF16),
    rope=lambda: J.ggml_rope_ext(x, pos, n_dims=64),
    mul_mat=lambda: J.ggml_mul_mat(w, J.MLA_TYPE_BF16, wx),
    attn_mask=lambda: J.ggml_flash_attn_ext(q, k, J.MLA_TYPE_BF16, mask=sparse_mask, out=out, stream=0),
    rope_pos=lambda: J.ggml_rope_ext(x, sparse, n_dims=64, out=x, stream=0),
    kv_write=lambda: J.kv_write(rows, cache, J.MLA_TYPE_BF16, rows=sparse, stream=0),
    kv_write_rope=lambda: J.kv_write(rows, cache, J.MLA_TYPE_BF16, row0=0, stream=0, k_pe=rows[:, 512:], rope=dict(pos=sparse, n_dims=64)),
    copy=lambda: J.copy_f32(x, torch.zeros((4, 16, 64)).to_sparse(), stream=0),
)
J.capi.native()   # (a module that does not load is no error of a call)
seen = {}
for name, call in calls.items():
    try:
        call()
        seen[name] = "returned"
    except Exception as e:
        seen[name] = "raised" if isinstance(e, (RuntimeError, AssertionError)) else repr(e)
print("SEEN " + json.dumps(seen), flush=True)
"""


@pytest.mark.skipif(torch.cuda.is_available(), reason="the allocations would succeed")
def test_errors_of_tensors_and_allocations_are_raised():
    r = subprocess.run([sys.executable, "-c", CALLS], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
    seen = json.loads([l for l in r.stdout.splitlines() if l.startswith("SEEN ")][0][5:])
    assert len(seen) == 8 and set(seen.values()) == {"raised"}, seen
