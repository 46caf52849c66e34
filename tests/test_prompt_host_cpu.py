"""The host side of the prompt pass without a GPU."""
import pytest
import torch


@pytest.fixture(scope="module")
def dec():
    import cherryq_decoder
    return cherryq_decoder


def _decoder(dec, **over):
    cfg = dec.DecoderConfig(**{**dict(hidden_size=256, intermediate_size=512, num_hidden_layers=1, num_attention_heads=2,
                                      num_key_value_heads=1, vocab_size=64, max_position_embeddings=32), **over})
    return dec.CherryLlamaDecoder(cfg, seed=0, device="cpu")


def _angles(theta, tokens, hd=128):
    fr = torch.outer(torch.arange(tokens, dtype=torch.float32), 1.0 / (theta ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd)))
    return fr.cos().half(), fr.sin().half()


def test_a_pass_keeps_no_rotary_table(dec):
    """A pass under capture would keep tables that hold nothing before the replay: they are made with the model, and a pass only reads
    them, or makes its own where the config is another one by now or the model has none."""
    model = _decoder(dec)
    state = dict(model.__dict__)
    for tokens in (1, 17, 32):
        for got, want in zip(model._rope_tables(tokens), _angles(model.cfg.rope_theta, tokens)):
            assert torch.equal(got, want)
    model.cfg.rope_theta = 500000.0
    for got, want in zip(model._rope_tables(9), _angles(500000.0, 9)):
        assert torch.equal(got, want)
    assert {k: id(v) for k, v in model.__dict__.items()} == {k: id(v) for k, v in state.items()}
    del model.__dict__["_rope"]  # saved whole by an older program
    assert torch.equal(model._rope_tables(9)[0], _angles(500000.0, 9)[0]) and "_rope" not in model.__dict__
