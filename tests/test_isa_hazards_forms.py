"""The generated-code checks of test_isa_hazards.py on the other head_dim-256 forms of the attention
kernel: row masks, and two and four wavefronts per tile (CPU; needs hipcc)."""

import re

import pytest

from test_isa_hazards import agpr_hazards, asm, kernel_body, operand_write_hazards  # noqa: F401

# CFG: 4 row sets a wavefront, + 16 (wavefronts - 1), + 256 with row masks
FORMS = [f"_ZN5ugbsa20attn_fwd_pipe_kernelINS_{elem}ELi256ELi{cfg}ELb1ELb1ELb1E"
         for elem in ("8ElemBf16", "7ElemF16") for cfg in (4 + 256, 4 + 16, 4 + 48)]


@pytest.mark.parametrize("kernel", FORMS)
def test_form(asm, kernel):  # noqa: F811
    body = kernel_body(asm, kernel)
    bad, mfmas, checked = agpr_hazards(body)
    assert not bad, bad[:5]
    assert mfmas >= 64 and checked >= 64, (mfmas, checked)
    bad, _ = operand_write_hazards(body)
    assert not bad, bad[:5]
    text = "\n".join(body)
    assert not re.search(r"\bv_pk_(add|mul|fma)_f32\b", text) and "scratch_" not in text
