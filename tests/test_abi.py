"""CPU-side checks of the boundary: the shared library loads, exports every symbol include/mole_hip.h
declares, rejects bad arguments without touching a GPU, and the host-only planner matches the oracle."""
import os
import re

import numpy as np
import pytest

from oracle import moe_oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    """every function declared in include/*.h: the boundary (mole_hip.h) and the measurement aids (mole_hip_probe.h)"""
    names = set()
    for header in sorted(os.listdir(os.path.join(ROOT, "include"))):
        if header.endswith(".h"):
            text = open(os.path.join(ROOT, "include", header)).read()
            text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
            names |= set(re.findall(r"\b(mole_[a-z0-9_]+)\s*\(", text))
    return sorted(names)


def test_boundary_header_holds_no_measurement_aids():
    text = open(os.path.join(ROOT, "include", "mole_hip.h")).read()
    assert "mole_probe" not in text


def test_library_exports_every_declared_symbol():
    from mole_amd import _lib as L
    lib = L.lib()
    declared = _declared()
    assert len(declared) >= 30
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in mole_hip.h but not exported"
    assert sorted(L.EXPORTS) == declared
    assert lib.mole_version() >= 100


def test_header_is_plain_c_and_a_c_program_links(tmp_path):
    """The boundary is a C ABI: the header compiles as strict C99 (no C++ types, no torch types), and a C program
    that calls an entry point links against the shared library and runs without a GPU."""
    import shutil
    import subprocess
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no gcc here")
    inc = os.path.join(ROOT, "include")
    subprocess.run([gcc, "-std=c99", "-Wall", "-Wextra", "-pedantic", "-Werror", "-fsyntax-only", "-x", "c",
                    os.path.join(inc, "mole_hip.h")], check=True)
    src = tmp_path / "caller.c"
    src.write_text('#include <stdio.h>\n#include "mole_hip.h"\n'
                   'int main(void) {\n'
                   '    /* bad arguments are refused on the host, with a message, before anything touches a GPU */\n'
                   '    int rc = mole_dispatch_fwd(NULL, MOLE_BF16, NULL, 8, 12, 2, NULL, NULL);\n'
                   '    printf("%d %d %s\\n", mole_version(), rc, mole_last_error_string());\n'
                   '    return rc == -1 ? 0 : 1;\n}\n')
    from mole_amd import _lib as L
    libdir = os.path.dirname(L.LIB_PATH)
    exe = tmp_path / "caller"
    subprocess.run([gcc, "-std=c99", "-I", inc, str(src), "-o", str(exe), "-L", libdir, "-l:" + os.path.basename(L.LIB_PATH),
                    "-Wl,-rpath," + libdir], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split(None, 2)
    assert int(out[0]) >= 100 and int(out[1]) == -1 and "M" in out[2]


def test_argument_validation_needs_no_gpu():
    from mole_amd import _lib as L
    lib = L.lib()
    assert lib.mole_route(None, 10, 0, 1, 1.0, 1, 1, 1, None, None, None, None, None, None, None, None, None, None, 0, None) == -1
    assert "E" in L.last_error()
    assert lib.mole_dispatch_fwd(None, 1, None, 8, 12, 2, None, None) == -1      # M not a multiple of 8 for bf16
    assert lib.mole_ffn_fwd(None, 7, None, None, 1, 0, 8, 8, None, None, None, None, None, None, None, None) == -1
    assert lib.mole_route_workspace_bytes(16384, 16, 1) > 0


def test_fast_assign_prefetch_host_planner():
    from mole_amd import core
    rng = np.random.default_rng(0)
    for _ in range(300):
        n = int(rng.integers(1, 8)); P = int(rng.integers(1, 12))
        Fv = [int(v) for v in rng.integers(0, 12, n)]; Ev = [int(v) for v in rng.integers(0, 9, n)]
        gp, lp = core.fast_assign_prefetch(P, Fv, Ev)
        want_gp, want_lp = O.fast_assign_prefetch(P, Fv, Ev)
        assert gp == want_gp and lp == want_lp


def test_product_package_does_not_import_the_oracle():
    pkg = os.path.join(ROOT, "mole_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".cpp")):
                src = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in src.replace("the oracle", ""), f"{f} mentions the oracle package"


def test_every_entry_point_rejects_bad_arguments_on_the_host():
    """Shape, dtype, alignment and null checks come before any launch: each call below returns a negative library
    code and leaves a message that names the entry point, on a machine without a GPU."""
    import ctypes
    from mole_amd import _lib as L
    lib = L.lib()
    P = ctypes.c_void_p
    bad16 = P(8)        # a non-null, misaligned "pointer" that is never dereferenced
    ok = P(4096)
    cases = [
        ("mole_softmax_fwd", lambda: lib.mole_softmax_fwd(None, None, 10, 0, None, None)),
        ("mole_gate_fwd", lambda: lib.mole_gate_fwd(ok, L.MOLE_F32, ok, None, 10, 64, 128, ok, None)),      # fp32: E <= 32
        ("mole_gate_fwd", lambda: lib.mole_gate_fwd(bad16, L.MOLE_F32, ok, None, 10, 8, 128, ok, None)),    # fp32: alignment
        ("mole_gate_fwd", lambda: lib.mole_gate_fwd(ok, L.MOLE_BF16, ok, None, 10, 8, 100, ok, None)),
        ("mole_softmax_bwd", lambda: lib.mole_softmax_bwd(ok, ok, 10, 0, ok, None)),
        ("mole_gate_bwd", lambda: lib.mole_gate_bwd(ok, ok, ok, 10, 4, 5, 1, 1, None, None, ok, None)),
        ("mole_gate_bwd", lambda: lib.mole_gate_bwd(ok, ok, ok, 10, 4, 2, 1, 1, ok, None, ok, None)),      # counts0 without d_l_aux
        ("mole_gate_wgrad", lambda: lib.mole_gate_wgrad(ok, ok, L.MOLE_F32, 10, 64, 128, ok, ok, 1 << 30, None)),
        ("mole_gate_wgrad", lambda: lib.mole_gate_wgrad(ok, ok, L.MOLE_BF16, 10, 8, 128, ok, ok, 16, None)),
        ("mole_route", lambda: lib.mole_route(ok, 10, 4, 5, 1.0, 1, 1, 1, ok, ok, ok, ok, ok, ok, ok, ok, ok, ok, 1 << 20, None)),
        ("mole_route", lambda: lib.mole_route(ok, 10, 4, 2, 1.0, 1, 1, 1, ok, ok, ok, ok, ok, ok, ok, ok, ok, ok, 8, None)),
        ("mole_dispatch_fwd", lambda: lib.mole_dispatch_fwd(bad16, L.MOLE_F32, ok, 8, 16, 2, ok, None)),
        ("mole_dispatch_bwd", lambda: lib.mole_dispatch_bwd(ok, L.MOLE_F32, ok, 8, 16, 2, ok, None, 4, None, ok, None)),
        ("mole_combine_fwd", lambda: lib.mole_combine_fwd(ok, L.MOLE_BF16, ok, ok, 8, 12, 2, ok, None)),
        ("mole_combine_bwd", lambda: lib.mole_combine_bwd(None, ok, L.MOLE_F32, ok, ok, 8, 16, 2, ok, ok, None)),
        ("mole_zero_pad_rows", lambda: lib.mole_zero_pad_rows(ok, 9, ok, ok, 4, 16, None)),
        ("mole_ffn_fwd", lambda: lib.mole_ffn_fwd(ok, L.MOLE_BF16, ok, ok, 2, 16, 12, 16, ok, ok, ok, ok, ok, ok, ok, None)),
        ("mole_ffn_fwd", lambda: lib.mole_ffn_fwd(bad16, L.MOLE_F32, ok, ok, 2, 16, 16, 16, ok, ok, ok, ok, ok, ok, ok, None)),
        ("mole_ffn_bwd", lambda: lib.mole_ffn_bwd(ok, ok, ok, ok, 5, ok, ok, 2, 16, 16, 16, ok, ok, ok, ok, ok, ok, ok, ok, 0, 0, None)),
        ("mole_gemm_nt", lambda: lib.mole_gemm_nt(ok, ok, 4, 16, 16, 16, ok, None)),
        ("mole_gemm_nn", lambda: lib.mole_gemm_nn(ok, ok, 4, 16, 16, 16, ok, None)),
        ("mole_gemm_tn", lambda: lib.mole_gemm_tn(ok, ok, L.MOLE_F32, 16, 6, 16, ok, None)),                  # Mo % 4
        ("mole_adam_step", lambda: lib.mole_adam_step(ok, ok, ok, ok, ok, 64, L.MOLE_F32, 0.9, 0.999, 0, 1e-3, 0.0, 1e-8, 0, None)),
        ("mole_adam_step", lambda: lib.mole_adam_step(ok, bad16, ok, ok, ok, 64, L.MOLE_BF16, 0.9, 0.999, 1, 1e-3, 0.0, 1e-8, 0, None)),
        ("mole_adam_step", lambda: lib.mole_adam_step(ok, ok, ok, ok, ok, 64, L.MOLE_F32, 1.0, 0.999, 1, 1e-3, 0.0, 1e-8, 0, None)),
        ("mole_unimem_prefetch", lambda: lib.mole_unimem_prefetch(None, 0, None, 0, 1)),
        ("mole_unimem_fetch", lambda: lib.mole_unimem_fetch(None, None, 0, 0, 1, 0, None)),
        ("mole_unimem_prefetch_ids", lambda: lib.mole_unimem_prefetch_ids(None, 0, None, None, 1, 0)),
        ("mole_unimem_fetch_ids", lambda: lib.mole_unimem_fetch_ids(None, None, 0, None, 1, 0, 0, None)),
        ("mole_unimem_wait_slots", lambda: lib.mole_unimem_wait_slots(None, 0, 1, None)),
        ("mole_unimem_reserve", lambda: lib.mole_unimem_reserve(None, 0, 1, None)),
        ("mole_unimem_store_grads_ids", lambda: lib.mole_unimem_store_grads_ids(None, None, None, None, 1, None)),
        ("mole_unimem_zero_grads_ids", lambda: lib.mole_unimem_zero_grads_ids(None, None, None, 1)),
        ("mole_unimem_store_grads", lambda: lib.mole_unimem_store_grads(None, None, None, 0, 1, None)),
        ("mole_unimem_load_state", lambda: lib.mole_unimem_load_state(None, None, None, None, 1, 0, None)),
        ("mole_unimem_store_state", lambda: lib.mole_unimem_store_state(None, None, None, None, 1, None)),
        ("mole_unimem_sync_tran", lambda: lib.mole_unimem_sync_tran(None)),
        ("mole_fast_assign_prefetch", lambda: lib.mole_fast_assign_prefetch(4, None, None, 3, None, None, 0, None)),
    ]
    for name, call in cases:
        rc = call()
        assert rc < 0, f"{name}: expected a library error code, got {rc}"
        msg = L.last_error()
        assert name in msg, f"{name}: message does not name the entry point: {msg!r}"


@pytest.mark.parametrize("cf", [0.0, -0.5, 0.25, 1.25, 1e9, 1e19, 1e300])
def test_layer_plan_rows_hold_every_kept_pair(cf):
    """64 tokens, top-2 of 4 experts: min(S k, E k int(cf ceil(S / E))) rows, also where no integer holds the product."""
    from mole_amd import _lib as L
    from mole_amd import hip_ops as H
    import torch
    plan = lambda f: H.LayerPlan(torch.bfloat16, 64, 128, 4, 2, 256, f, L.LAYOUT_RAGGED, True, 0)
    want = 128 if cf <= 0 else min(128, 4 * 2 * int(cf * 16))
    assert plan(cf).native.rows == want
    with pytest.raises(RuntimeError, match="finite"):
        plan(float("inf"))


def test_gate_route_workspace_of_three_sizes():
    """mole_gate_route_workspace_bytes(S, E, k), as programs built against its first declaration call it, covers every call
    it is for: bf16, up to 64 experts, a width that is a multiple of 128."""
    import torch
    from mole_amd import _lib as L
    lib = L.lib()
    decl = re.search(r"mole_gate_route_workspace_bytes\(([^)]*)\)", open(os.path.join(ROOT, "include", "mole_hip.h")).read()).group(1)
    assert [a.split()[-1] for a in decl.split(",")] == ["S", "E", "k"]
    bf16 = L.dtype_code(torch.bfloat16)
    for S in (1, 31, 32, 63, 64, 65, 2048, 2049, 40000):
        for E in (1, 2, 33, 64):
            for k in (1, min(E, 8)):
                have = lib.mole_gate_route_workspace_bytes(S, E, k)
                assert all(have >= lib.mole_gate_route_shape_workspace_bytes(bf16, S, E, M, k) > 0 for M in (128, 1024, 8192))
    assert lib.mole_gate_route_workspace_bytes(-1, 4, 1) == 0 and lib.mole_gate_route_workspace_bytes(4, 0, 1) == 0


def test_core_and_plans_travel_through_pickle(tmp_path):
    """Copies and pickles of a layer's core and of its plans, read by a process that has loaded neither library; a state that
    holds the number of passes as plain integer (as these do) is also what earlier cores were pickled with."""
    import copy
    import pickle
    import subprocess
    import sys
    import torch
    from mole_amd import _lib as L, core, hip_ops as H
    from mole_amd.moe.layer import MOLEModule
    c = core.MOLECore(False, False, False, False, 4, 0, 4, 1, "gelu", False, 2, 5, 0, 0, 4)
    plan = H.LayerPlan(torch.bfloat16, 64, 128, 4, 2, 256, 1.25, L.LAYOUT_PADDED, True, 1)
    assert type(c.__getstate__()["step"]) is int
    d = copy.deepcopy(c)
    c.step += 1
    assert (c.step, d.step) == (6, 5)
    path = tmp_path / "state.pkl"
    path.write_bytes(pickle.dumps((c, plan)))
    code = ("import pickle, sys; c, p = pickle.load(open(sys.argv[1], 'rb'))\n"
            "c.step += 1; print(c.step, c.acc_step, c.passes.value, p.native.rows, p.native.route_offsets() == p.__reduce__()[0](*p.__reduce__()[1]).native.route_offsets())")
    r = subprocess.run([sys.executable, "-c", code, str(path)], capture_output=True, text=True, cwd=ROOT)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split() == ["7", "2", "7", str(plan.native.rows), "True"]
    # a layer whose state has its last routing as a plain attribute, and no plans
    m = MOLEModule.__new__(MOLEModule)
    torch.nn.Module.__init__(m)
    m.__setstate__(dict(m.__dict__, param_dtype=torch.bfloat16, last_route="route"))
    assert m.last_route == "route" and m._plans == {} and m._granule == 8


def test_planes_of_a_padded_layout_stay_bounded():
    """Scratch of the layer's split contractions where the padded layout has many more slots than rows: 32 MB of planes at most
    (or none), beside the few bytes of the gate; as many as the ragged layout's where the slots are near the rows."""
    import struct
    from mole_amd import _lib as L
    import ctypes
    lib = L.lib()

    def workspace(S, M, E, k, F, rows, layout, backward=0):
        block = ctypes.create_string_buffer(struct.pack("10id", L.MOLE_BF16, S, M, E, k, F, rows, layout, 1, 0, 1.0), 512)
        return lib.mole_layer_workspace_bytes(ctypes.cast(block, ctypes.c_void_p), backward)

    def gate(S, M, E, k):
        return lib.mole_gate_route_shape_workspace_bytes(L.MOLE_BF16, S, E, M, k)

    assert gate(1, 2048, 256, 2) < 1 << 20
    assert 1 << 20 < workspace(1, 2048, 256, 2, 4096, 1024, L.LAYOUT_PADDED) <= 32 << 20        # eight planes: 67 MB
    assert workspace(4096, 512, 64, 2, 2048, 524288, L.LAYOUT_PADDED) <= max(32 << 20, gate(4096, 512, 64, 2))   # two: 2.1 GB
    assert workspace(1, 8192, 256, 2, 4096, 4096, L.LAYOUT_PADDED) <= 1 << 20                   # not one plane fits
    ragged, padded = workspace(3001, 1024, 16, 2, 4096, 6002, L.LAYOUT_RAGGED), workspace(3001, 1024, 16, 2, 4096, 7520, L.LAYOUT_PADDED)
    assert ragged > 32 << 20 and ragged * 7520 == padded * 6002


def test_gate_weight_gradient_scratch_is_what_its_kernel_uses():
    """mole_gate_wgrad: the matrix-core kernel's chunks of 128 tokens for gates that only that kernel takes (no more than 32 MB or
    eight chunks).  The layer's: what the gate's own kernel needs, not the partial sums of one that does not take it."""
    import ctypes
    import struct
    from mole_amd import _lib as L
    lib = L.lib()
    for S, E, M in ((2048, 64, 1024), (300, 40, 1024), (1, 33, 64), (5000, 200, 128)):
        assert lib.mole_gate_wgrad_workspace_bytes(S, E, M) == (S + 127) // 128 * E * M * 4, (S, E, M)
    assert lib.mole_gate_wgrad_workspace_bytes(16384, 256, 4096) == 8 * 256 * 4096 * 4

    def backward(S, M, E, dtype):
        block = ctypes.create_string_buffer(struct.pack("10id", dtype, S, M, E, 1, 64, S, L.LAYOUT_RAGGED, 1, 0, 1.0), 512)
        return lib.mole_layer_workspace_bytes(ctypes.cast(block, ctypes.c_void_p), 1)

    # 1024 experts of 8192: gradients of the gates, operands and result of the input gradient's product, and one [E, M] in fp32
    S, E, M = 4096, 1024, 8192
    assert backward(S, M, E, L.MOLE_BF16) <= 4 * S + 2 * (S * E + E * M + S * M) + 4 * E * M + 4096


def _kernel_metadata():
    """What the built library's code objects say about their kernels: name -> metadata map of the AMDGPU note."""
    import struct
    import msgpack
    from mole_amd import _lib as L
    blob, out, at = open(L.LIB_PATH, "rb").read(), {}, 0
    while (at := blob.find(b"\x7fELF", at + 1)) >= 0:
        if struct.unpack_from("<H", blob, at + 18)[0] != 224:                      # EM_AMDGPU
            continue
        shoff, (shentsize, shnum) = struct.unpack_from("<Q", blob, at + 40)[0], struct.unpack_from("<HH", blob, at + 58)
        for i in range(shnum):
            kind, _, _, off = struct.unpack_from("<IQQQ", blob, at + shoff + i * shentsize + 4)
            if kind == 7:                                                          # SHT_NOTE
                name, desc = struct.unpack_from("<II", blob, at + off)
                start = at + off + 12 + (name + 3) // 4 * 4
                for k in msgpack.unpackb(blob[start:start + desc])["amdhsa.kernels"]:
                    out[k[".name"]] = k
    return out


def test_routing_of_many_tokens_keeps_its_registers():
    """The top-k kernel of many tokens holds 16 scores a lane and no partial sums of them beside: it spills a few registers beyond 256 experts
    (18, with the sums 54) and none below."""
    spills = {n: k[".vgpr_spill_count"] for n, k in _kernel_metadata().items() if "route_tokens_kernel" in n}
    wide = [n for n in spills if "ILi16ELi6ELi1024E" in n]
    assert len(spills) >= 12 and len(wide) == 1
    assert all(v <= (24 if n in wide else 0) for n, v in spills.items()), spills


def test_fp32_products_leave_the_few_row_kernel_at_48_rows():
    """Beyond 48 rows per expert the tiles with split contractions are the faster ones; the few-row kernel has blocks enough
    there without a split, and no workspace."""
    from mole_amd import _lib as L
    ws = lambda rows: L.lib().mole_ffn_workspace_bytes(L.MOLE_F32, 16, rows, 1024, 4096)
    assert ws(16 * 48) == 0 and ws(16 * 48 + 1) > 0


def test_bf16_planes_of_widths_that_end_inside_a_stage():
    """A contraction that ends inside a stage is split into as many planes as one of whole stages with the same tiles: its sums
    keep their order (one plane at 16 experts of 128 rows, 520 -> 1416)."""
    from mole_amd import _lib as L
    planes = lambda E, rows, M, F: L.lib().mole_ffn_workspace_bytes(L.MOLE_BF16, E, rows, M, F) / (4 * rows * M)
    for E, rows, M, F in ((16, 2052, 520, 1416), (16, 4104, 520, 1416), (8, 1600, 1032, 2056), (20, 2600, 264, 1032), (8, 800, 520, 1032)):
        assert planes(E, rows, M, F) == planes(E, rows, M, F // 32 * 32), (E, rows, M, F)
    assert planes(16, 2052, 520, 1416) == 0


def test_bf16_scratch_is_no_more_than_both_directions_use():
    """A layer's scratch is laid out once for its two narrow products: out is split into no more planes than gx, which shares a launch
    (layers of several 128-row tiles an expert that leave half of the CUs' block slots idle)."""
    from mole_amd import _lib as L
    for E, rows, M, F in ((9, 1609, 904, 2712), (9, 2384, 640, 1920), (24, 2976, 448, 1792)):
        assert L.lib().mole_ffn_workspace_bytes(L.MOLE_BF16, E, rows, M, F) == 0, (E, rows, M, F)


def test_layer_scratch_is_told_from_the_sizes_alone():
    """mole_layer_workspace_bytes reads the sizes of the block: the capacity factor, which a caller may set after it has laid the scratch out,
    changes nothing at equal sizes."""
    import ctypes
    import random
    import struct
    from mole_amd import _lib as L
    rng = random.Random(2)
    sizes = [(L.MOLE_F32, 757, 512, 32, 4, 1024)]
    for _ in range(4000):
        E, grain = rng.randint(2, 64), rng.choice([64, 16, 8])
        M = grain * rng.randint(1, 1024 // grain)
        sizes.append((rng.choice([L.MOLE_F32, L.MOLE_F32, L.MOLE_BF16]), int(2 ** rng.uniform(0, 14)), M, E, rng.randint(1, min(E, 8)), rng.choice([1, 2, 4]) * M))
    for dtype, S, M, E, k, F in sizes:
        for backward in (0, 1):
            need = set()
            for cf in (0.0, 0.5, 1.0, 1.25, 2.0):
                block = ctypes.create_string_buffer(struct.pack("10id", dtype, S, M, E, k, F, S * k, L.LAYOUT_RAGGED, 1, 0, cf), 512)
                need.add(L.lib().mole_layer_workspace_bytes(ctypes.cast(block, ctypes.c_void_p), backward))
            assert len(need) == 1, (dtype, S, M, E, k, F, need)


def test_rings_of_three_stages_lie_where_they_were_measured():
    """t and g_w2 in one launch: sizes on either side of each line of the rule (rings of three stages, of five, or a launch each)."""
    from mole_amd import _lib as L
    ring = L.lib().mole_probe_pair_stages
    for (E, rows, M, F), stored, added in (((22, 571 * 8, 384, 768), 3, 3), ((16, 2052, 520, 1416), 5, 3), ((16, 1522 * 8, 408, 408), 3, 3), ((10, 2260, 984, 1968), 5, 3),
                                           ((8, 12871 * 2, 512, 256), 5, 5), ((13, 654 * 2, 520, 1560), 5, 5), ((32, 3616, 32, 1416), 0, 0)):
        assert (ring(E, rows, M, F, 0), ring(E, rows, M, F, 1)) == (stored, added), (E, rows, M, F)
