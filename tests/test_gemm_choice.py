"""Which MFMA skeleton a product is planned on and that its kernel compiles, without a device."""
import re

import pytest

from _loader import load_pkg
from test_gpu_dot import dot_module

rx = load_pkg()


def skeleton(*args):
    m = re.search(r"(rx_gemm_body\w*)<([^\n]*)>\(A, B, epi", rx.compile_offline(dot_module(*args)[0], with_source=True))
    return m.group(1) if m else None


# (K + 64) rows of 4 M bytes reach 2^32 at M = 2^23 (K = 64): below it the body with split operands, from it on another one
@pytest.mark.parametrize("tall,other,k", [(6_000_000, 128, 64), (8_388_600, 128, 64), (6_000_000, 256, 80)])
def test_f32_products_of_a_tall_matrix_compile(tall, other, k):
    assert skeleton(tall, other, k, "f32", "f32", False, True) == "rx_gemm_body_x"
    assert skeleton(other, tall, k, "f32", "f32", True, False) == "rx_gemm_body_x"


def test_f32_products_past_the_offset_bound_compile():
    assert skeleton(8_388_608, 128, 64, "f32", "f32", False, True) not in (None, "rx_gemm_body_x", "rx_gemm_body_g")
    assert skeleton(128, 8_388_608, 64, "f32", "f32", True, False) not in (None, "rx_gemm_body_x", "rx_gemm_body_g")


def test_one_stage_serves_one_tile(monkeypatch):
    """A tile asked for with one LDS stage is refused (the planner's own is taken) where a group has more than one K tile."""
    def text(k, spec):
        monkeypatch.setenv("RX_GEMM_G", spec)
        return rx.compile_offline(dot_module(256, 256, k, "f32", "f32", True, True)[0], with_source=True)
    assert "rx_gemm_body_g<rx_el_f32, 64, 64, 2, 2, 1, 1, " not in text(512, "64,64,2,2,1,1")
    assert "rx_gemm_body_g<rx_el_f32, 64, 64, 2, 2, 1, 2, " in text(512, "64,64,2,2,1,2")
    assert "rx_gemm_body_g<rx_el_f32, 64, 64, 2, 2, 2, 1, " in text(64, "64,64,2,2,2,1")
