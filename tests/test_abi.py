"""The C-ABI library loads without a GPU and exports every function the headers declare."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    names = set()
    for h in ("moe_kernels.h", "moe_engine.h"):
        text = open(os.path.join(ROOT, "include", h)).read()
        text = re.sub(r"/\*.*?\*/", " ", text, flags=re.S)          # comments
        text = re.sub(r"^\s*#.*$", " ", text, flags=re.M)            # preprocessor lines
        text = re.sub(r"typedef\s+struct[^{;]*\{.*?\}[^;]*;", " ", text, flags=re.S)  # struct bodies
        for m in re.finditer(r"\b(moe_[a-z0-9_]+)\s*\(", text):
            names.add(m.group(1))
    return sorted(names)


def test_every_declared_function_is_exported():
    import torch  # noqa: F401  (the library shares torch's HIP runtime)
    from promoe_amd import _lib
    lib = ctypes.CDLL(_lib.LIB_PATH) if hasattr(_lib, "LIB_PATH") else _lib.lib
    names = declared_functions()
    assert len(names) > 50, names
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing


def test_headers_compile_as_c():
    """include/*.h are plain C: compile them with gcc, no HIP or torch types in the signatures."""
    import subprocess
    import tempfile
    src = '#include "moe_kernels.h"\n#include "moe_engine.h"\nint main(void) { return 0; }\n'
    with tempfile.TemporaryDirectory() as d:
        c = os.path.join(d, "t.c")
        open(c, "w").write(src)
        r = subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"), "-c", c,
                            "-o", os.path.join(d, "t.o")], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr


def test_expert_rows_past_the_kernels_addressing_are_refused_on_the_host():
    """Rows of 2^24 columns (bf16: 2^23) of an expert: an error before anything is launched (no GPU needed)."""
    import torch  # noqa: F401
    from promoe_amd import _lib as L
    p = 4096                                     # never read
    for fmt, most in ((L.FMT_INT4_G128, 1 << 24), (L.FMT_Q4K, 1 << 24), (L.FMT_BF16, 1 << 23)):
        for T in (1, 65):
            if T * most * 2 >= 1 << 31:          # refused for the activations' size already
                continue
            rc = L.lib.moe_experts_prefill(p, T, 256, most, 0, 1, fmt, p, 1, p, p, None, p, None, p, None, p, p, 3, None)
            assert rc != 0 and b"columns and more" in L.lib.moe_last_error(), (fmt, T)


@pytest.mark.skipif(torch.cuda.is_available(), reason="addresses that nothing may read: on machines without a GPU only")
def test_the_bf16_routing_launch_refuses_what_its_w2_pass_refuses():
    """Rows of 2^23 columns and activations of 2 GiB, with every other argument as it should be: an error before the w13 launch, not
    only from the w2 launch behind it."""
    from promoe_amd import _lib as L
    p, E = 4096, 16                              # never read
    for T, k, H, I, I_sh, said in ((1, 1, 1 << 23, 128, 0, b"columns and more"), (1, 1, 256, 1 << 23, 0, b"columns and more"),
                                   (1, 1, 256, 128, 1 << 23, b"columns and more"), (32, 16, 256, 1 << 21, 0, b"2 GiB"),
                                   (32, 1, 256, 128, (1 << 23) * 8, b"2 GiB")):
        sh = p if I_sh else None
        rc = L.lib.moe_decode_batch_bf16_gate(p, T, p, p, E, p, 1, p, E, E, k, 0, H, I, I_sh, p, sh, p, p, p, p, p, p, p, p, p, p,
                                              min(E, T * k), p, sh, p, None, None, None, 0, None)
        assert rc != 0 and said in L.lib.moe_last_error(), (T, k, H, I, I_sh, L.lib.moe_last_error())
