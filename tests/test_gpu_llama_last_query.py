"""LLaMA prompts long enough that the last block makes the query of the one row whose logits are asked for alone: against
the run that asks for all rows' logits, and the step behind the prompt, which reads what the prompt kept."""
import numpy as np
import pytest

from litenn_amd import synth
from litenn_amd.formats import DT_F16, DT_F32, Q4_0, Q4_K, Q6_K, Q8_0

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precise", [True, False])
@pytest.mark.parametrize("formats,kv", [({"default": Q4_0}, DT_F16), ({"default": Q4_K, "attn_v": Q6_K, "ffn_down": Q6_K}, DT_F16), ({"default": Q8_0}, DT_F32)])
def test_last_query(hip, formats, kv, precise):
    """Rows on both sides of the rule's line (100 and 256 times 4096 x 4096 over the matrix' size)."""
    d = 2048
    line = (400 if precise else 1024)
    cfg = synth.LLaMAConfig("t", 2, d, 16, 4, 512, 320, line + 80, formats=formats)
    model = hip.LLaMA.from_config(cfg, kv_dtype=kv)
    model.load(synth.llama_tensors(cfg, 3))
    rng = np.random.default_rng(5)
    for rows in (line - 1, line, line + 63):
        toks = rng.integers(0, 320, rows + 3).astype(np.int32)
        model.reset()
        model.eval(toks[:2], all_logits=False, precise=precise)
        whole = model.eval(toks[2:rows + 2], precise=precise)[-1]
        behind = model.eval(toks[-1:], precise=precise)
        model.reset()
        model.eval(toks[:2], all_logits=False, precise=precise)
        one = model.eval(toks[2:rows + 2], all_logits=False, precise=precise)
        after = model.eval(toks[-1:], precise=precise)
        # operands rounded to Float16 once (2^-12 of each, which a sum's terms share out), or cached values on either side of a tie
        limit = 1e-4 if precise else 4e-3
        assert np.linalg.norm(one - whole) <= limit * np.linalg.norm(whole), rows
        assert np.linalg.norm(after - behind) <= limit * np.linalg.norm(behind), rows  # (keys' and values' ranges of K may differ)
    model.close()
