"""The kernel units: every entry point that the engine calls is found in a unit, what a unit needs comes before it, and
the units that a model names for its first call exist.  Compiling: only what is missing of what is asked for."""
import os

import pytest
import torch

import helpers


def test_every_entry_point_has_a_unit():
    from deliverance_amd.kernels import build, ops
    found = build.entry_points()
    names = set(build.units())
    for name in ops._ARGTYPES:
        assert found.get(name) in names, f"{name} is in no unit"
    assert found["da_last_error"] == build.BASE_UNIT
    assert found["da_attn_decode_rel"] == "attn_decode_rel" and found["da_attn_decode"] == "attn_decode"
    assert set(build.NEEDS) <= names and {n for ns in build.NEEDS.values() for n in ns} <= names
    assert set(build.INCLUDES) <= names and set(build.EXTRA_FLAGS) <= names


def test_what_a_unit_needs_comes_first():
    from deliverance_amd.kernels import build
    order = build.with_needs(["run_step", "gla"])
    assert order[0] == build.BASE_UNIT and len(order) == len(set(order))
    assert order.index("gemm_wide") < order.index("gemm_mfma") < order.index("run_step") and "gla" in order
    assert build.with_needs([build.BASE_UNIT]) == [build.BASE_UNIT]


def test_only_what_is_asked_for_and_missing_is_compiled(tmp_path, monkeypatch):
    from deliverance_amd.kernels import build
    done = []

    def compiled(hipcc, out_dir, todo, verbose):
        for u in todo:
            done.append(u)
            with open(os.path.join(out_dir, f"libda_{u}.so"), "w"):
                pass
    monkeypatch.setattr(build, "_build_dirs", lambda: (str(tmp_path / "a"), str(tmp_path / "b")))
    monkeypatch.setattr(build, "_build_locked", compiled)
    monkeypatch.setattr(build, "_find_hipcc", lambda: "hipcc")
    build.build(only=["gla"])
    assert sorted(done) == sorted(["gla", build.BASE_UNIT])
    build.build(only=["gla", "attn_window"])
    assert sorted(done) == sorted(["gla", build.BASE_UNIT, "attn_window"])
    build.build(only=["gla"])
    assert len(done) == 3 and "moe" in build.missing() and build.missing(["gla"]) == []
    build.build(force=True, only=["gla"])
    assert sorted(done[3:]) == sorted(["gla", build.BASE_UNIT])
    monkeypatch.setattr(build, "_find_hipcc", lambda: None)
    with pytest.raises(build.KernelLibraryError, match="hipcc was not found"):
        build.build(only=["moe"])


def test_models_name_units_that_exist(tmp_path):
    from deliverance_amd.kernels import build
    from deliverance_amd.models.causal_lm import load_model
    from deliverance_amd.random_model import random_model
    from luvatar_models import CONFIG_A
    from mogevik_models import CONFIG_D, CONFIG_E
    from pafolorn_models import CONFIG_F
    from pedatar_models import CONFIG_P
    from salivik_models import CONFIG_S
    from virudra_models import CONFIG_X
    names = set(build.units())
    of = {}
    for key, cfg in (("gpt2", helpers.CONFIG_A), ("virudra", CONFIG_X), ("pedatar", CONFIG_P), ("pafolorn", CONFIG_F),
                     ("salivik", CONFIG_S), ("luvatar", CONFIG_A), ("mogevik", CONFIG_D), ("mogevik_plain", CONFIG_E)):
        folder = str(tmp_path / key)
        random_model(folder, cfg, 1)
        for dtype in (torch.bfloat16, torch.float32):
            of[key, dtype] = set(load_model(folder, dtype, "cpu").kernel_units())
            assert of[key, dtype] <= names, f"{key}: {of[key, dtype] - names}"
    lu = of["luvatar", torch.bfloat16]
    assert {"gla", "attn_window", "attn_prepare"} <= lu and not lu & {"moe", "ssm", "retention", "attn_latent", "attn_prefill", "gemm_ref"}
    assert "gla" not in of["gpt2", torch.bfloat16] and "gemm_mfma" not in of["luvatar", torch.float32]
    mo = of["mogevik", torch.bfloat16]
    assert {"rglru", "moe", "attn_window", "elementwise"} <= mo and not mo & {"ssm", "gla", "attn_prepare", "norm_rms", "gemm_ref", "attn_latent"}
    assert {"rglru", "ssm"} <= of["mogevik_plain", torch.bfloat16] and {"rglru", "ssm", "attn_rel"} <= of["mogevik", torch.float32]
    from deliverance_amd.kernels import ops
    if build.is_built():
        assert all(bool(ops._lib().da_rglru_serve_takes(n)) == ops.rglru_block_fits(n) for n in range(1, 300))


def test_a_norm_that_writes_the_stream_promises_nothing_about_it(tmp_path):
    """The kernels that add shares to the stream read it through one pointer and write it through another: the front end's
    code must not tell the optimizer that the two never meet (``noalias``); the plain norms, which only read, may."""
    import re
    import subprocess
    from deliverance_amd.kernels import build
    hipcc = build._find_hipcc()
    if hipcc is None:
        pytest.skip("needs hipcc")
    out = str(tmp_path / "rowwise.ll")
    subprocess.run([hipcc, "-std=c++17", f"--offload-arch={build.ARCH}", "--cuda-device-only", "-S", "-emit-llvm", "-O1", "-Xclang",
                    "-disable-llvm-passes", "-w", build._source("rowwise"), "-o", out], check=True)
    with open(out) as f:
        found = re.findall(r"define [^\n]*@_Z\d+layernorm_row_kernelILi\d+ELi\d+ELb[01]ELb[01]ELb([01])EE[^(]*\(([^,]*),", f.read())
    assert {join for join, _ in found} == {"0", "1"}
    for join, stream in found:
        assert ("noalias" in stream) == (join == "0"), (join, stream)


def test_which_steps_norm_and_product_take_in_one_kernel():
    """One row tile and a width of 1,024, 8 rows and 2,048; with 5 rows and more not for wide widths with many columns; never a vocabulary."""
    from deliverance_amd.kernels import ops
    takes = ops._lib().da_can_fuse_ln
    for rows, K, N in ((1, 768, 2304), (16, 1024, 4096), (8, 1536, 16384), (4, 2048, 16384), (8, 1600, 4800), (5, 1912, 5120), (8, 2048, 6144), (5, 1920, 6144)):
        assert takes(rows, K, N), (rows, K, N)
    for rows, K, N in ((0, 768, 768), (17, 768, 768), (9, 1032, 768), (8, 2056, 768), (1, 764, 768), (1, 768, 16385), (5, 1600, 6400), (8, 1544, 5121), (8, 2048, 6145)):
        assert not takes(rows, K, N), (rows, K, N)


def test_which_products_take_four_pieces_of_k_side_by_side():
    """Up to 4 rows and 2,048 columns; 5 to 8 rows with a long K, where it is ahead of the kernel for more rows."""
    from deliverance_amd.kernels import ops
    takes = ops._lib().da_gemm_pieces_takes
    for rows, N, K in ((1, 2048, 8), (4, 2048, 2048), (5, 1984, 2048), (8, 64, 8192), (8, 2048, 3584)):
        assert takes(rows, N, K), (rows, N, K)
    for rows, N, K in ((1, 2049, 768), (5, 1024, 2040), (8, 2048, 2048), (5, 1985, 3576), (9, 64, 8192)):
        assert not takes(rows, N, K), (rows, N, K)
