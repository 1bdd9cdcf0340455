"""Host-side logic, the C ABI surface and the code generator (no GPU needed)."""

import ctypes
import itertools
import re
from fractions import Fraction
from pathlib import Path

import numpy as np
import pytest
import sympy as sp
import torch

ROOT = Path(__file__).resolve().parents[1]


def _declared_symbols():
    text = (ROOT / "include" / "flashcart_hip.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(fc_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from flashcart_amd import _lib
    lib = _lib.load()
    declared = _declared_symbols()
    assert len(declared) >= 20
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in include/flashcart_hip.h but not exported"
    assert set(declared) == set(_lib.EXPORTED_SYMBOLS)
    assert lib.fc_kernel_l_max() == 3 and lib.fc_version() >= 100


def test_rank_limit_selects_the_library(monkeypatch):
    """FLASHCART_KERNEL_L_MAX (read at import, as by the reference) picks the rank-3 or the rank-4
    library and the limit the modules enforce; above 4 is refused."""
    import importlib

    from flashcart_amd import _lib
    from flashcart_amd.o3 import kernel_config
    assert _lib.library_path(3).endswith("libflashcart_hip.so")
    assert _lib.library_path(2).endswith("libflashcart_hip.so")
    assert _lib.library_path(4).endswith("libflashcart_hip_l4.so")
    try:
        monkeypatch.setenv("FLASHCART_KERNEL_L_MAX", "4")
        assert importlib.reload(kernel_config).KERNEL_L_MAX == 4
        monkeypatch.setenv("FLASHCART_KERNEL_L_MAX", "5")
        with pytest.raises(RuntimeError):
            importlib.reload(kernel_config)
        monkeypatch.delenv("FLASHCART_KERNEL_L_MAX")
        assert importlib.reload(kernel_config).KERNEL_L_MAX == 3
    finally:
        monkeypatch.delenv("FLASHCART_KERNEL_L_MAX", raising=False)
        importlib.reload(kernel_config)


@pytest.mark.skipif(not (ROOT / "flashcart_amd" / "libflashcart_hip_l4.so").exists(),
                    reason="libflashcart_hip_l4.so not built (FLASHCART_KERNEL_L_MAX=4 python -m flashcart_amd.build)")
def test_rank4_library_exports_and_metadata():
    """The rank-4 build exports the same symbols with the same descriptor layout and accepts rank 4
    (42 paths of 4 x 4 -> 4, the reference's count)."""
    from flashcart_amd import _lib
    lib = ctypes.CDLL(str(ROOT / "flashcart_amd" / "libflashcart_hip_l4.so"))
    for name in _declared_symbols():
        assert hasattr(lib, name), name
    lib.fc_kernel_l_max.restype = ctypes.c_int
    assert lib.fc_kernel_l_max() == 4
    lib.fc_tp_num_paths.argtypes = [ctypes.POINTER(_lib.TPDesc)]
    lib.fc_tp_out_dim.argtypes = [ctypes.POINTER(_lib.TPDesc)]
    lib.fc_tp_out_dim.restype = ctypes.c_int64
    d = _lib.tp_desc(4, 4, 4, 8, 1, False, False, False)
    assert lib.fc_tp_num_paths(ctypes.byref(d)) == 42
    assert lib.fc_tp_num_paths(ctypes.byref(_lib.tp_desc(5, 4, 4, 8, 1, False, False, False))) == -2


def test_abi_metadata_calls_without_gpu():
    from flashcart_amd import _lib
    lib = _lib.load()
    d = _lib.tp_desc(2, 3, 3, 128, 1, False, False, False)
    assert lib.fc_tp_num_paths(d) == 17
    assert lib.fc_tp_out_dim(d) == 71 * 128
    bad = _lib.tp_desc(4, 3, 3, 128, 1, False, False, False)
    assert lib.fc_tp_num_paths(bad) == -2  # FC_ERR_UNSUPPORTED_L
    assert lib.fc_status_string(6) == b"workspace missing or too small"


def test_path_order_matches_layout_contract():
    from flashcart_amd.codegen.cartesian import enumerate_paths
    got = [f"{a}{b}{c}{'s' if s else 'f'}" for a, b, c, s in enumerate_paths(2, 3, 3, False)]
    want = ["000f", "110f", "220f", "101f", "211f", "101s", "211s", "321s", "112f", "202f", "222f", "202s",
            "312s", "213f", "213s", "303s", "323s"]
    assert got == want


def test_path_counts():
    from flashcart_amd.o3.utils import count_output_paths
    assert count_output_paths(0, 3, 3) == ([1, 1, 1, 1], 4)
    assert count_output_paths(3, 3, 3)[1] == 23
    assert count_output_paths(3, 3, 0, symmetric_product=True) == ([4], 4)
    assert count_output_paths(2, 2, 2) == ([3, 4, 4], 11)


def test_codegen_coefficients_match_oracle():
    from flashcart_amd.codegen.emit_hip import ordered_triples, triple_coefficients
    from oracle.cartesian import path_tensor
    for r1, r2, lo in ordered_triples(3):
        B = np.zeros((2 * lo + 1, 2 * r1 + 1, 2 * r2 + 1))
        for (a, b, c), v in triple_coefficients(r1, r2, lo).items():
            B[a, b, c] = float(v)
        ref = path_tensor(r1, r2, lo) if r1 >= r2 else np.transpose(path_tensor(r2, r1, lo), (0, 2, 1))
        assert np.abs(B - ref).max() < 1e-13, (r1, r2, lo)


def test_codegen_expansion_matches_oracle():
    from flashcart_amd.codegen.cartesian import X, Y, Z, expansion_polynomials
    from oracle.ops import irreps
    r = torch.randn(7, 3, dtype=torch.float64)
    o = irreps(r, 3)
    col = 0
    for l in range(4):
        for p in expansion_polynomials(l):
            f = sp.lambdify((X, Y, Z), p, "numpy")
            v = np.broadcast_to(f(*[r[:, k].numpy() for k in range(3)]), (7,))
            assert np.allclose(v, o[:, col].numpy(), atol=1e-13)
            col += 1


def test_generated_header_is_current_and_literals_round_once():
    from flashcart_amd.codegen.emit_hip import emit_tp_header, flit
    hdr = (ROOT / "flashcart_amd" / "csrc" / "generated" / "fc_tp_paths.h").read_text()
    assert hdr == emit_tp_header()
    for frac in [Fraction(2, 3), Fraction(5, 9), Fraction(-3, 7), Fraction(1, 1)]:
        lit = flit(frac)
        assert np.float32(float(lit[:-1])) == np.float32(float(frac))


def test_neighbor_list_matches_brute_force():
    from flashcart_amd.data.neighbors import neighbor_pairs
    from flashcart_amd.data.synthetic import fcc_alloy
    from oracle.neighbors import brute_force_pairs
    rng = np.random.default_rng(0)
    z, p, cell, pbc = fcc_alloy(2, 2, 2, seed=1)
    tri = np.array([[7.0, 0.0, 0.0], [2.1, 6.5, 0.0], [-1.3, 0.7, 7.4]])
    cases = [(p, cell, pbc, 5.0), (rng.uniform(0, 6, (20, 3)) @ np.linalg.inv(np.eye(3) * 6) @ tri, tri,
                                   np.array([True, True, True]), 4.0),
             (rng.uniform(0, 5, (15, 3)), np.zeros((3, 3)), np.array([False] * 3), 3.0),
             (rng.uniform(0, 5, (15, 3)), np.eye(3) * 5.0, np.array([True, False, True]), 3.5)]
    for pos, c, pb, rc in cases:
        ei, sh = neighbor_pairs(pos, c, pb, rc)
        got = [(int(a), int(b)) + tuple(int(s) for s in S) for a, b, S in zip(ei[0], ei[1], sh)]
        want = brute_force_pairs(pos, c if abs(np.linalg.det(c)) > 1e-7 else np.eye(3), pb, rc)
        assert got == want
        assert np.all(np.diff(ei[0]) >= 0)


def test_neighbor_count_known_answers():
    """Average neighbour counts 1, 2 and 2/3 (reference tests/data/test_data.py:96-108)."""
    from flashcart_amd.data.neighbors import neighbor_pairs
    h = 1.5 * np.sqrt(3) / 2
    for pos, want in [([[0, 0, 0], [1.4, 0, 0]], 1.0), ([[0, 0, 0], [1.5, 0, 0], [0.75, h, 0]], 2.0),
                      ([[0, 0, 0], [1.0, 0, 0], [50.0, 0, 0]], 2.0 / 3.0)]:
        ei, _ = neighbor_pairs(np.array(pos, float), np.zeros((3, 3)), False, 5.0)
        assert abs(ei.shape[1] / len(pos) - want) < 1e-12


def test_periodic_self_images_exist():
    from flashcart_amd.data.neighbors import neighbor_pairs
    ei, sh = neighbor_pairs(np.zeros((1, 3)), np.eye(3) * 3.0, True, 3.5)
    assert ei.shape[1] == 6 and np.all(ei == 0)  # six face images of a single atom


REFERENCE_KEYS = [
    "embedding.weight", "radial_basis.r_min", "radial_basis.r_max", "cutoff_fn.poly_order", "cutoff_fn.r_max",
    "cutoff_fn.coeff1", "interactions.0.sqrt_avg_neighbors", "interactions.0.radial_mlp.0.weight",
    "interactions.0.radial_mlp.2.weight", "interactions.0.radial_mlp.4.weight", "interactions.0.linear_first.weight.0",
    "interactions.0.linear_second.weight.3", "interactions.0.skip_projection.weight",
    "interactions.0.layer_norm.weights.3", "interactions.1.skip_projection.weight.2",
    "products.0.skip_projection.weight.2", "products.0.layer_norm.weights.2", "products.0.product_linears.0.weight.3",
    "products.0.product_linears.2.weight.2", "products.1.product_linears.2.weight.0",
    "nonlinearities.0.value_linear.weight.3", "nonlinearities.0.gate_linear.weight",
    "nonlinearities.0.gate_linear.bias", "nonlinearities.1.output_linear.weight.0", "readout.readout_mlp.0.weight",
    "readout.readout_mlp.4.weight", "scale_shift.shifts", "scale_shift.scales",
]


def test_state_dict_names_and_shapes():
    from flashcart_amd.data.synthetic import model_config
    from flashcart_amd.model import FlashCartPotential
    m = FlashCartPotential.from_config(model_config(["Cu", "Ni", "Fe", "Cr"], 16, 3, avg_neighbors=40.0))
    sd = m.state_dict()
    for k in REFERENCE_KEYS:
        assert k in sd, k
    assert tuple(sd["interactions.1.radial_mlp.4.weight"].shape) == (17 * 16, 64)
    assert tuple(sd["interactions.1.linear_second.weight.3"].shape) == (16, 16 * 4)
    assert tuple(sd["products.0.product_linears.1.weight.3"].shape) == (16, 16 * 6)
    assert tuple(sd["readout.readout_mlp.0.weight"].shape) == (64, 32)
    assert not any("dummy_tp_weights" in k or "l_weights" in k for k in sd)
    assert abs(float(sd["interactions.0.sqrt_avg_neighbors"]) - 40.0 ** 0.5) < 1e-6


def test_ops_reject_cpu_tensors():
    from flashcart_amd import o3
    tp = o3.TensorProduct(1, 1, 1, 4, 4)
    x = torch.randn(3, 16)
    with pytest.raises(RuntimeError, match="ROCm"):
        tp(x, x, torch.randn(3, tp.n_total_paths * 4))
    with pytest.raises(RuntimeError, match="ROCm"):
        o3.Irreps(2).forward_normalized(torch.tensor([[1.0, 0.0, 0.0]]))


def test_tp_op_schema_follows_reference():
    """Positional schema of torch.ops.flashcart.tp_fwd/tp_bwd as registered by the reference
    (src/flashcart/o3/_tensor_product.py:332-352,588-611), extra arguments only at the end."""
    from flashcart_amd.o3 import _ops
    ref_fwd = ["in1", "in2", "weights", "idx_i", "idx_j", "in1_l_max", "in2_l_max", "out_l_max", "in1_features",
               "in2_features", "symmetric_product", "shared_weights", "in1_offs", "in2_offs", "out_sizes",
               "n_paths_per_l", "n_total_paths", "reduce_paths"]
    ref_bwd = ["grad_out"] + ref_fwd[:17] + ["reduce_paths", "need_grad_in1", "need_grad_in2", "need_grad_weights"]
    for op, ref in ((torch.ops.flashcart.tp_fwd.default, ref_fwd), (torch.ops.flashcart.tp_bwd.default, ref_bwd)):
        names = [a.name for a in op._schema.arguments]
        assert names[:len(ref)] == ref
        assert all(a.has_default_value() for a in op._schema.arguments[len(ref):])
    # Layout lists, as the reference builds them for (2 x 3 -> 3, C=128, in2 single channel):
    # _slice_offsets pads rank-block starts, _out_block_sizes = paths * (2l+1) * C.
    in1_offs, in2_offs, sizes, n_paths, total = _ops.tp_meta(2, 3, 3, 128, 1, False, False)
    assert in1_offs == [0, 128, 512, 0] and in2_offs == [0, 1, 4, 9]
    assert n_paths == [3, 5, 5, 4] and total == 17
    assert sizes == [3 * 128, 5 * 3 * 128, 5 * 5 * 128, 4 * 7 * 128]
    assert _ops.tp_meta(2, 2, 2, 8, 8, True, True)[2] == [8, 24, 40, 0]
    tp = __import__("flashcart_amd").o3.TensorProduct(1, 1, 1, 4, 4)
    x = torch.randn(3, 16)
    bad = list(tp.op_meta)
    bad[0] = [0, 8, 0, 0]
    with pytest.raises(ValueError, match="in1_offs"):
        torch.ops.flashcart.tp_fwd(x, x, torch.randn(3, tp.n_total_paths * 4), None, None, 1, 1, 1, 4, 4, False,
                                   False, *bad, False)


def test_checkpoint_round_trip(tmp_path):
    from flashcart_amd.data.synthetic import model_config
    from flashcart_amd.model import FlashCartPotential
    m = FlashCartPotential.from_config(model_config(["H", "O"], 8, 2, avg_neighbors=12.0))
    m.save_inference_checkpoint(tmp_path)
    m2 = FlashCartPotential.from_checkpoint(tmp_path)
    for (k, a), (k2, b) in zip(m.state_dict().items(), m2.state_dict().items()):
        assert k == k2 and torch.equal(a, b)
    assert torch.equal(m2.interactions[0].sqrt_avg_neighbors, m.interactions[0].sqrt_avg_neighbors)


def test_device_neighbor_list_host_fallback_decision():
    """Only the device list's size limit (-FC_ERR_SHAPE: > 1024 pairs for one atom or a shift
    component >= 512) sends the build to the host list; other failures stay errors."""
    from flashcart_amd.data.neighbors import host_fallback_needed

    assert host_fallback_needed(-4)
    assert not any(host_fallback_needed(s) for s in (0, 17, -1, -3, -5, -6, -7))


def test_linear_and_irreps_op_schemas_follow_reference():
    """torch.ops.flashcart.linear_fwd / linear_bwd / linear_dbwd / irreps_dbwd take the
    reference's positional arguments (src/flashcart/o3/_linear.py:328-343, :457-472, :571-591;
    src/flashcart/o3/_irreps.py:153-159) and return its outputs."""
    import flashcart_amd.o3._second_order  # noqa: F401  (registers the double backward)

    lists = ["in_offsets", "out_offsets", "weight_offsets", "m_values", "f_in_values", "f_out_values"]
    want = {
        "linear_fwd": ["x", "weights", "meta", "out_size", "use_fp64", "dot_input_precision"] + lists + ["scale"],
        "linear_bwd": ["grad_out", "x", "weights", "need_x", "need_weight", "use_fp64",
                       "dot_input_precision"] + lists + ["scale"],
        "linear_dbwd": ["grad_out", "x", "weights", "v_grad_x", "v_grad_weight", "use_fp64", "dot_input_precision",
                        "need_d_grad_out", "need_d_x", "need_d_weight", "has_v_grad_x",
                        "has_v_grad_weight"] + lists + ["scale"],
        "irreps_dbwd": ["grad_output", "x", "v", "l_max"],
    }
    n_out = {"linear_fwd": 1, "linear_bwd": 2, "linear_dbwd": 3, "irreps_dbwd": 2}
    for name, ref in want.items():
        schema = getattr(torch.ops.flashcart, name).default._schema
        assert [a.name for a in schema.arguments] == ref, name
        assert len(schema.returns) == n_out[name], name
    # the build's own residual / alpha variants live under names of their own
    assert [a.name for a in torch.ops.flashcart.equiv_linear_fwd.default._schema.arguments][-2:] == ["alpha",
                                                                                                      "residual"]


def test_rounded_row_allocations():
    from flashcart_amd import _lib
    assert [_lib.rounded_rows(n) for n in (0, 1, 15, 16, 17, 31, 32, 33)] == [0, 1, 15, 16, 18, 32, 32, 36]
    for n in [1080166, 1081496, 1100110, 1179648, 1179649, 7, 4096, 123457]:
        r = _lib.rounded_rows(n)
        q = 1 << max(n.bit_length() - 4, 0)
        assert n <= r < n + q and r % q == 0 and (r - n) <= n / 8
    # edge counts of an MD run drifting by ~0.1% per step share one rounded size
    assert len({_lib.rounded_rows(n) for n in range(1080166, 1179648, 997)}) == 1
    like = torch.empty(0)
    small = _lib.rows_empty(like, 1000, 16)
    assert small.shape == (1000, 16) and small.untyped_storage().nbytes() == 1000 * 16 * 4
    big = _lib.rows_empty(like, 1080166, 16)
    assert big.shape == (1080166, 16) and big.is_contiguous() and big.storage_offset() == 0
    assert big.untyped_storage().nbytes() == _lib.rounded_rows(1080166) * 16 * 4
    flat = _lib.rows_empty(like, 20_000_000, dtype=torch.int32)
    assert flat.shape == (20_000_000,) and flat.dtype == torch.int32


def test_alias_as_flashcart():
    """The reference's module names resolve to this package after alias_as_flashcart()."""
    import sys

    import flashcart_amd

    saved = {k: v for k, v in sys.modules.items() if k == "flashcart" or k.startswith("flashcart.")}
    try:
        for k in saved:
            del sys.modules[k]
        flashcart_amd.alias_as_flashcart()
        import flashcart
        import flashcart.data
        import flashcart.o3
        from flashcart.model import FlashCartPotential
        from flashcart.nn import InteractionLayer
        from flashcart.utils.lammps import lammps_data_slot

        assert flashcart is flashcart_amd and flashcart.o3.TensorProduct is flashcart_amd.o3.TensorProduct
        assert FlashCartPotential.__module__.startswith("flashcart_amd.model")
        assert InteractionLayer is flashcart_amd.nn.InteractionLayer
        assert flashcart.data.NeighborList is flashcart_amd.data.NeighborList and callable(lammps_data_slot)
    finally:
        for k in [k for k in sys.modules if k == "flashcart" or k.startswith("flashcart.")]:
            del sys.modules[k]
        sys.modules.update(saved)


def test_operator_arguments_that_need_the_registry():
    """An Operator runs its implementation itself only for plain GPU tensors and arguments of the exact types;
    everything else reaches the registered operator, which converts or refuses it."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from flashcart_amd.o3 import _ops
    x = torch.zeros(4, 3)
    assert not _ops.irreps_fwd._direct((x, 2))  # not on a GPU
    with FakeTensorMode(allow_non_fake_inputs=True):
        f = torch.empty(4, 3, device="cuda")
        assert f.is_cuda and not _ops.irreps_fwd._direct((f, 2))
        assert _ops.irreps_fwd(f, 2).shape == (4, 9)
    assert _ops._observed() is False

    class Gpu(torch.Tensor):  # stands in for a GPU tensor
        is_cuda = True

    g = Gpu()
    plain = _ops._EXACT["Tensor"]
    sig = _ops.irreps_fwd.exact
    assert sig[0] is plain and sig[1] == (int,)
    op = _ops.Operator.__new__(_ops.Operator)
    op.required, op.exact, op.items = 2, ((Gpu,), (int,), (list, tuple)), ((2, int),)
    assert op._direct((g, 1)) and op._direct((g, 1, [1, 2])) and op._direct((g, 1, ()))
    for bad in ((g,), (g, 1.0), (g, True), (g, 1, [1.0]), (g, 1, [], 0), (x, 1), (None, 1)):
        assert not op._direct(bad), bad
    for args in ((x,), (x, 1.5), (x, 2, 3), ("x", 2)):
        with pytest.raises(Exception) as a:
            _ops.irreps_fwd(*args)
        with pytest.raises(Exception) as b:
            _ops.irreps_fwd.op(*args)
        assert type(a.value) is type(b.value)


def test_lazy_values_are_written_out():
    """A tensor whose memory does not hold its values (a negated view, of one element also when contiguous; a zero
    tensor without memory) is written out where its address is taken."""
    from flashcart_amd import _lib
    from flashcart_amd.o3 import _ops

    class Gpu(torch.Tensor):  # stands in for a GPU tensor
        is_cuda = True

    negated = torch.tensor([0.3 + 0.77j]).conj().imag
    assert negated.is_neg() and negated.is_contiguous()
    zero = torch._efficientzerotensor(1, 3)
    assert zero.data_ptr() == 0
    plain = torch.ones(4, 3)
    for t in (negated, torch._neg_view(torch.ones(4, 3)), torch._neg_view(torch.ones(4, 3)).t(), zero, plain, plain.t()):
        for got in (_lib.contig("t", t.as_subclass(Gpu)), _ops._i32("t", torch._neg_view(-t.int()).as_subclass(Gpu))
                    if t is plain else _lib.contig("t", t.as_subclass(Gpu))):
            values = torch.empty(t.shape, dtype=got.dtype)
            assert got.data_ptr() != 0 and got.is_contiguous() and got.shape == t.shape
            ctypes.memmove(values.data_ptr(), got.data_ptr(), t.numel() * 4)
            assert torch.equal(values.to(torch.float32), t.clone())
    gpu = plain.as_subclass(Gpu)
    assert _lib.contig("t", gpu) is gpu


Tensor = torch.Tensor  # (operators' annotations are read as text)


def _scratch_operator(name):
    """An operator for one test, x -> 2 x, whose calls count as plain ones on the CPU."""
    from flashcart_amd.o3 import _ops

    def double(x: "Tensor") -> "Tensor":
        return 2 * x

    op = _ops.Operator.register(f"flashcart_test::{name}", double)
    op.register_fake(torch.empty_like)
    op._direct = lambda args: True
    return op


def test_operators_are_registered_operators():
    """torch.library's functions that take an operator take the callables of this package, by object and by name, and
    compilers see the operator itself in a whole graph."""
    from flashcart_amd.o3 import _ops
    op = _ops.irreps_fwd
    assert isinstance(op, torch.library.CustomOpDef)
    x = torch.zeros(4, 3)
    # (no kernel for the CPU: the checks that run the operator end in its own error)
    with pytest.raises(Exception, match="ROCm devices only"):
        torch.library.opcheck(op, (x, 2), test_utils="test_schema")
    torch.library.opcheck(op, (x, 2), test_utils="test_autograd_registration")
    for k, by_name in enumerate((False, True)):
        own = _scratch_operator(f"vmap{k}")
        torch.library.register_vmap(f"flashcart_test::vmap{k}" if by_name else own,
                                    lambda info, in_dims, x: (x + 1, in_dims[0]))
        assert torch.equal(torch.func.vmap(own)(x), x + 1)
    assert _ops.irreps_fwd.__name__ == "irreps_fwd" and "irreps_bwd" in repr(_ops.irreps_bwd)
    seen = []

    def backend(graph, inputs):
        seen.extend(str(n.target) for n in graph.graph.nodes if n.op == "call_function")
        return lambda *a: (x.new_zeros(4, 9),)

    out = torch.compile(lambda v: op(v, 2), backend=backend, fullgraph=True)(x)
    assert out.shape == (4, 9) and any("flashcart.irreps_fwd" in t for t in seen)


@pytest.mark.parametrize("by_name", [False, True])
def test_operator_kernel_overrides(by_name):
    """A kernel or an autocast rule registered for an operator is what a plain call runs from then on, and a kernel
    switched off leaves the implementation."""
    name = f"override_{'name' if by_name else 'object'}"
    op = _scratch_operator(name)
    op.register_autograd(lambda ctx, g: 2 * g)
    target = f"flashcart_test::{name}" if by_name else op
    x = torch.ones(3, requires_grad=True)

    def gradient():
        return torch.autograd.grad(op(x).sum(), x)[0]

    assert torch.equal(op(x), 2 * x) and type(op(x).grad_fn).__name__ == "DirectBackward"
    if by_name:
        torch.library.register_kernel(target, "cpu", lambda x: 5 * x.detach())
    else:
        op.register_kernel("cpu")(lambda x: 5 * x.detach())
    assert torch.equal(op(x), 5 * x) and torch.equal(gradient(), torch.full((3,), 2.0))
    with op.set_kernel_enabled("cpu", enabled=False):
        assert torch.equal(op(x), 2 * x)
    assert torch.equal(op(x), 5 * x)

    cast = _scratch_operator(name + "_cast")
    torch.library.register_autocast(f"flashcart_test::{name}_cast" if by_name else cast, "cpu", torch.bfloat16)
    with torch.autocast("cpu", torch.bfloat16):
        assert cast(torch.ones(3)).dtype == torch.bfloat16
    assert cast(torch.ones(3)).dtype == torch.float32

    for key in ("CUDA", "AutogradCUDA", "AutocastCUDA"):  # a dispatcher kernel of another library
        own = _scratch_operator(f"{name}_{key}")
        assert own.kernels[0] == f"flashcart_test/{name}_{key}/CUDA"
        own.op = lambda x: "registry"
        lib = torch.library.Library("flashcart_test", "IMPL")
        assert torch.equal(own(x.detach()), 2 * x)
        lib.impl(f"{name}_{key}", lambda x: 7 * x, key)
        assert own(x.detach()) == "registry"


@pytest.mark.skipif(torch.cuda.is_available(), reason="the positions here are no device memory")
@pytest.mark.parametrize("cell,pbc,refused", [
    (np.diag([8.0, 8.0, 8.0]), (1, 1, 1), False),
    (np.diag([8.0, 0.008, 9.0]), (1, 1, 1), False),          # 500 images each way along an axis
    (np.diag([9.0, 0.04, 0.04]), (1, 1, 1), False),          # 100 and 100
    (np.diag([0.032, 0.016, 9.0]), (1, 1, 1), False),        # 251 x 501 x 2 runs of candidates a receiver
    (np.diag([0.032, 0.015, 9.0]), (1, 1, 1), True),         # 251 x 535 x 2
    (np.diag([8.0, 0.0008, 0.0008]), (1, 1, 1), True),       # 100 million
    (np.diag([8.0, 9.0, 1e-7]), (1, 1, 1), True),            # 4e7 bins away
    (np.diag([8.0, 1e-9, 9.0]), (1, 1, 1), True),            # 4e9: beyond 32 bits
    (np.diag([8.0, 9.0, 1e-20]), (1, 1, 1), True),           # 4e20: beyond 64
    (np.diag([1e-200, 9.0, 1e-90]), (1, 1, 1), True)])
def test_device_list_refuses_thin_cells(cell, pbc, refused):
    """fc_neighbor_list_device refuses, before it launches anything, cells so thin that a receiver's search would
    run for long or its counts would not fit; other cells get as far as the launch, which fails here."""
    from flashcart_amd import _lib
    from flashcart_amd.data.neighbors import host_fallback_needed
    lib = _lib.load()
    cell = np.ascontiguousarray(cell)
    flags = np.asarray(pbc, dtype=np.int32)
    pos, ws = np.zeros((2, 3)), np.zeros(1 << 16, dtype=np.uint8)
    n = lib.fc_neighbor_list_device(2, pos.ctypes.data, cell.ctypes.data, flags.ctypes.data, 4.0, 0, None, None, None,
                                    ws.ctypes.data, ws.size, None)
    assert n < 0 and host_fallback_needed(n) == refused
