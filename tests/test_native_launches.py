"""The module of native launches (``csrc/host.cpp``) where no kernel may run: operands that only look like the GPU's.

No GPU is needed: nothing here gets as far as a launch.
"""
import os
import re
import shutil
import subprocess
import sys

import pytest

from gesso_amd.kernels import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# Fake tensors on a device that need not be there: they have types, sizes and strides, and the address 0.
CALLS = """
import sys
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from gesso_amd.errors import KernelError
from gesso_amd.kernels import build, ops

native = build.load_host()
BF, F, I = torch.bfloat16, torch.float32, torch.int32
mode = FakeTensorMode()
mode.__enter__()
t = lambda *s, dtype=BF: torch.empty(*s, dtype=dtype, device="cuda")
f, i = lambda *s: t(*s, dtype=F), lambda *s: t(*s, dtype=I)
mid = (t(100, 512), t(1024, 512), t(1024, 512))
kc = t(4, 2, 4, 64)
calls = {
    "add_rmsnorm": (f(3, 64), t(3, 64), f(64), 1e-5, 1),
    "gemm_skinny": (t(3, 64), t(32, 64), t(32, 64), 1, 0),
    "gemm_mid": mid + (0,),
    "gemm_mid_residual": mid + (f(100, 1024), f(1024)),
    "gemm_mid_swiglu_scaled": (mid[0], f(100, 8), 1e-5) + mid[1:],
    "gemm_mid_residual_parts": (t(100, 2304), t(1024, 2304), t(1024, 2304), f(100, 1024), f(1024), 1e-5, 2),
    "short_conv": (t(9, 96), f(32, 3), f(32), f(3, 32, 2), i(9), i(3), i(2), 2, 0),
    "qknorm_rope_kv": (t(9, 512), f(64), f(64), 1e-5, f(16, 32), f(16, 32), 64, i(9), i(9), i(2, 2), 4, kc, kc, 4, 2, 64, 1, 0),
    "attention_prefill": (t(9, 512), 512, kc, kc, i(9), i(3, 2), i(2, 2), 4, 0, 0.125, 4, 2, 64, 9, 16, t(9, 256)),
}
"""

# Those that vmap batches have no address at all.
WITHOUT_MEMORY = CALLS + """
args = list(calls[sys.argv[1]])
without = [int(v) for v in sys.argv[2:]] or [k for k, a in enumerate(args) if isinstance(a, torch.Tensor)]
said = []

def one(*batched):
    for k, b in zip(without, batched):
        args[k] = b
    said.append(getattr(native, sys.argv[1])(*args, 0))
    if sys.argv[1] == "add_rmsnorm":
        ops._stream = lambda: 0
        ops.add_rmsnorm(*args[:4], BF)
    return batched[0]

try:
    torch.vmap(one)(*[torch.empty(2, *args[k].shape, dtype=args[k].dtype, device="cuda") for k in without])
except RuntimeError as err:
    assert sys.argv[1] == "add_rmsnorm" and "data pointer" in str(err), err
else:
    assert sys.argv[1] != "add_rmsnorm"
assert said == [False], said
print("said no")
"""


# Every operand of every function in other forms, one at a time.
OTHERS = CALLS + """
def others(name, k, a):
    if not isinstance(a, torch.Tensor):
        return [] if a is None else [("no number", "x")]
    forms = [("other type", a.to(torch.float16)), ("host", torch.empty(a.shape, dtype=a.dtype, device="cpu"))]
    if (name, k) not in ONE_DIMENSION_MORE:
        forms.append(("dimensions", a[None]))
    if a.dim() > 1:
        forms.append(("order", torch.empty_strided(a.shape, (1,) + tuple(a.shape[0] * s for s in range(1, a.dim())), dtype=a.dtype, device="cuda")))
        forms.append(("width", a[..., :-1].contiguous()))
    forms.append(("fewer", a[:-1].contiguous()))
    return forms

# indices may have any shape; rows, tables and pages any number of rows; q any width that holds the heads; the few rows' product takes
# the weight's other copy on trust, as the Python function does
ONE_DIMENSION_MORE = {("short_conv", 4), ("short_conv", 5), ("short_conv", 6), ("qknorm_rope_kv", 7), ("qknorm_rope_kv", 8), ("attention_prefill", 4)}
FREE = {(what, "gemm_skinny", 2) for what in ("other type", "dimensions", "order", "width", "fewer")}
FREE |= {("fewer", "gemm_skinny", 0), ("fewer", "gemm_skinny", 1), ("fewer", "gemm_mid", 0), ("fewer", "short_conv", 0), ("fewer", "qknorm_rope_kv", 0),
        ("width", "attention_prefill", 0)}
FREE |= {("fewer", "qknorm_rope_kv", 9), ("fewer", "attention_prefill", 6), ("fewer", "short_conv", 3), ("width", "qknorm_rope_kv", 9),
        ("width", "attention_prefill", 6), ("width", "attention_prefill", 5), ("dimensions", "attention_prefill", 0)}

wrong = []
for name, args in calls.items():
    try:
        said = getattr(native, name)(*args, 0)
        wrong.append((name, "as it is", said))
    except KernelError:
        pass                                   # the entry point's own: no GPU
    for k, a in enumerate(args):
        for what, other in others(name, k, a):
            if (what, name, k) in FREE:
                continue
            try:
                said = getattr(native, name)(*args[:k], other, *args[k + 1:], 0)
            except KernelError as err:
                said = err
            if said is not False:
                wrong.append((name, k, what, said))
    try:
        getattr(native, name)(*args)
        wrong.append((name, "an argument less"))
    except TypeError:
        pass
# tables in another order, also where nothing is turned and they are not read
args = calls["qknorm_rope_kv"]
if native.qknorm_rope_kv(*args[:4], f(32, 16).T, f(32, 16).T, 0, *args[7:], 0) is not False:
    wrong.append("tables")
print(wrong)
"""


def test_every_operand_in_another_form_is_left_to_the_python_function():
    """Type, place, number of dimensions, order, width and length of each tensor, and what should be a number."""
    if build.find_built() is None:
        pytest.skip("the library is not built")
    p = subprocess.run([sys.executable, "-c", OTHERS], cwd=ROOT, capture_output=True, text=True, timeout=300, env=dict(os.environ, HIP_VISIBLE_DEVICES="-1"))
    assert p.returncode == 0 and p.stdout.strip().split("\n")[-1] == "[]", (p.returncode, p.stdout, p.stderr[-2000:])


# All operands of a call without memory, and the one that is asked for its address last.
@pytest.mark.parametrize("name,operand", [(n, o) for n, o in (("add_rmsnorm", 0), ("gemm_skinny", 2), ("gemm_mid", 2), ("gemm_mid_residual", 3),
                                                             ("gemm_mid_swiglu_scaled", 1), ("gemm_mid_residual_parts", 4), ("short_conv", 3),
                                                             ("qknorm_rope_kv", 11), ("attention_prefill", 6)) for o in (None, o)])
def test_operands_without_memory_are_another_form(name, operand):
    """A tensor that has no address is left to the Python function, which raises torch's own error: in a process of its own, which an
    exception thrown where the interpreter's lock is let go of would end, and which sees no GPU."""
    if build.find_built() is None:
        pytest.skip("the library is not built")
    p = subprocess.run([sys.executable, "-c", WITHOUT_MEMORY, name] + ([] if operand is None else [str(operand)]), cwd=ROOT, capture_output=True,
                       text=True, timeout=300, env=dict(os.environ, HIP_VISIBLE_DEVICES="-1"))
    assert p.returncode == 0 and "said no" in p.stdout, (p.returncode, p.stderr[-2000:])


BINDS = """
import importlib.util, sys
spec = importlib.util.spec_from_file_location("gesso_host", sys.argv[1])
host = importlib.util.module_from_spec(spec)
spec.loader.exec_module(host)
try:
    host.bind(sys.argv[2], ValueError)
except OSError as err:
    print("refused:", err)
"""


@pytest.mark.parametrize("names,version,said", [("all", 14, "other interface versions"), ("all", 15, ""), ("some", 15, "lacks an entry point")])
def test_the_module_binds_to_a_library_of_its_own_version_only(tmp_path, names, version, said):
    """Against a library of empty functions: one that differs in version is refused, so is one without an entry point."""
    lib, cc = build.find_built(), shutil.which("gcc") or shutil.which("cc")
    if lib is None or cc is None:
        pytest.skip("the library is not built, or no C compiler")
    with open(os.path.join(build.CSRC, "native_calls.h"), encoding="utf-8") as f:
        text = f.read()
    assert f"GS_ABI_VERSION {15} " in text
    entries = sorted(set(re.findall(r"\b(gs_\w+)\(", text)) - {"gs_abi_version"})
    assert len(entries) == 13
    with open(tmp_path / "empty.c", "w") as f:
        f.write(f"int gs_abi_version(void) {{ return {version}; }}\n" + "".join(f"int {e}(void) {{ return 0; }}\n" for e in entries[names == "some":]))
    subprocess.run([cc, "-shared", "-fPIC", "-o", str(tmp_path / "empty.so"), str(tmp_path / "empty.c")], check=True, timeout=60)
    p = subprocess.run([sys.executable, "-c", "import torch\n" + BINDS, build._host_path(lib), str(tmp_path / "empty.so")], cwd=ROOT, capture_output=True,
                       text=True, timeout=120)
    assert p.returncode == 0 and (said in p.stdout if said else not p.stdout), (p.stdout, p.stderr[-2000:])
