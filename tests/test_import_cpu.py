"""The package without its optional extension module: `tilefusion_amd._direct` is built for one interpreter, the ops are not."""

import subprocess
import sys

WITHOUT = """
import sys
sys.modules["tilefusion_amd._direct"] = None          # as if it were not built for this interpreter
import torch
import tilefusion_amd
from tilefusion_amd import _direct, ops
assert _direct.__name__ == "tilefusion_amd._through_ops", _direct
a, b, c = torch.ones(2, 64), torch.ones(2, 64), torch.ones(2, 2)
x = torch.ones(1, 2, 64)
for call, name in ((lambda: ops.gemm(a, b, c, 1, 1, 1, 1, 0), "gemm"),
                   (lambda: ops.scatter_nd(c, torch.zeros(2, 1, dtype=torch.int64), c), "scatter_nd"),
                   (lambda: ops.flash_decode(x, x, x), "flash_decode"),
                   (lambda: ops.flash_attention(x, x.transpose(1, 2), x, 1, 1, 1, 1, 1.0, False), "flash_attention_fwd"),
                   (lambda: ops.fused_two_gemms(a, a, a, a), "must be a cuda tensor")):
    try:
        call()
    except (NotImplementedError, ValueError) as e:     # the op itself was asked, for a device that it does not run on
        assert name in str(e), e
    else:
        raise AssertionError(name)
print("fine")
"""


def test_package_works_without_the_direct_module():
    done = subprocess.run([sys.executable, "-c", WITHOUT], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0 and done.stdout.strip().endswith("fine"), done.stderr


def test_direct_module_has_every_function_of_its_stand_in():
    from tilefusion_amd import _direct, _through_ops
    names = [n for n, f in vars(_through_ops).items() if callable(f) and n != "Any"]
    assert sorted(names) == sorted(n for n in dir(_direct) if not n.startswith("_") and n != "Any")
