"""Lockstep steps across the attention split's key-count ranges: the longest
row crosses a range's last key (320, 640, 1280, 2560) within a run while the
other rows stay short, through the captured steps and the plain loop."""
import pytest

import oracle as O
from gpu_helpers import seeded_weights, small_heads_shape
from huggingfaceeacp_amd import gemma_q8 as G
from test_gpu_batch import check_rows, run_batch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def decoder():
    shape = small_heads_shape(max_positions=2700, max_step_rows=512)
    d = G.Decoder(shape)
    for i, values in enumerate(seeded_weights(shape)):
        d.load_tensor(i, values)
    yield d
    d.close()


@pytest.mark.parametrize("longest", [317, 637, 1277, 2557])
def test_batch_crosses_a_range(torch_cuda, decoder, longest):
    prompts = [O.prompt_ids(0xC0FFEE + s, decoder.shape.vocab, n)
               for s, n in enumerate((longest, 3, longest // 2, 79))]
    got, histories, logits = run_batch(decoder, prompts, 6, True)
    plain, _, _ = run_batch(decoder, prompts, 6, False)
    assert got == plain
    for s, prompt in enumerate(prompts):
        alone, _ = decoder.generate(prompt, 7, eos=-1)
        assert list(alone) == got[s], f"sequence {s}"
    check_rows(torch_cuda, decoder, histories, logits, f"longest {longest}")
