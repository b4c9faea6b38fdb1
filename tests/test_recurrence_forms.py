"""Which launches of the recurrences go in chunks (csrc/hybrid/chunk_scan.hip hy_chunk_scan_pays, gla_scan.hip hy_gla_scan_pays), against measured
times of both: a launch never takes the chunks where that was measured to be slower than token by token by more than 5%, as a short
prompt beside many decode rows is, and always where they take half of the time.  CPU-only: the rule is host code."""
import pytest
import torch

FORMS = {"head": 0, "token": 0, "mlstm": 1, "delta": 2, "rows": 3}
# (form, heads, D, Dv, sequences, tokens, longest, us in chunks, us token by token)
MEASURED = [
    ("head", 32, 128, 128, 114, 135, 16, 183.4, 77.2),
    ("head", 8, 128, 128, 257, 272, 16, 117.9, 49.7),
    ("head", 32, 128, 128, 65, 88, 24, 108.5, 55.6),
    ("head", 32, 128, 128, 257, 296, 40, 427.4, 230.2),
    ("head", 4, 128, 128, 68, 128, 16, 22.4, 15.3),
    ("head", 4, 128, 128, 11, 111, 59, 10.7, 27.2),
    ("head", 4, 128, 128, 65, 1280, 256, 28.6, 122.5),
    ("head", 4, 128, 128, 65, 3072, 2048, 175.3, 930.0),
    ("head", 8, 256, 256, 1, 2048, 2048, 65.5, 1237.0),
    ("token", 128, 128, 64, 65, 80, 16, 216.2, 103.6),
    ("token", 64, 128, 64, 65, 80, 16, 109.8, 53.3),
    ("token", 64, 128, 64, 65, 208, 16, 110.1, 55.3),
    ("token", 128, 128, 64, 257, 280, 24, 828.1, 428.3),
    ("token", 128, 128, 64, 260, 512, 64, 844.2, 465.7),
    ("token", 64, 128, 64, 49, 278, 230, 84.7, 142.0),
    ("token", 24, 64, 64, 68, 1088, 256, 27.3, 94.0),
    ("token", 24, 64, 64, 260, 4352, 1024, 87.3, 368.2),
    ("token", 24, 64, 64, 1, 2048, 2048, 37.2, 644.7),
    ("mlstm", 4, 128, 256, 260, 320, 16, 142.6, 95.6),
    ("mlstm", 4, 128, 256, 257, 272, 16, 142.8, 96.8),
    ("mlstm", 4, 128, 256, 257, 296, 40, 145.1, 121.6),
    ("mlstm", 4, 256, 512, 68, 256, 16, 115.2, 104.2),
    ("mlstm", 8, 64, 128, 65, 80, 16, 27.1, 30.3),
    ("mlstm", 8, 64, 128, 17, 133, 117, 21.4, 89.3),
    ("mlstm", 8, 64, 128, 260, 4352, 1024, 111.5, 801.2),
    ("mlstm", 4, 256, 512, 20, 1040, 256, 55.0, 493.2),
    ("mlstm", 4, 256, 512, 1, 2048, 2048, 103.6, 3009.6),
    ("delta", 16, 128, 128, 257, 296, 40, 299.8, 126.5),
    ("delta", 8, 64, 64, 257, 296, 40, 63.5, 27.7),
    ("delta", 32, 128, 128, 68, 224, 40, 152.5, 71.2),
    ("delta", 32, 128, 128, 257, 808, 40, 554.9, 279.8),
    ("delta", 32, 128, 128, 68, 448, 64, 156.0, 93.7),
    ("delta", 16, 128, 128, 7, 423, 91, 24.1, 47.1),
    ("delta", 8, 64, 64, 1, 2048, 2048, 299.8, 701.6),
    ("delta", 16, 128, 128, 17, 1040, 1024, 176.1, 457.0),
    ("delta", 16, 128, 128, 64, 656, 428, 85.9, 578.7),
    ("rows", 4, 64, 64, 260, 272, 4, 16.3, 11.2),
    ("rows", 4, 64, 64, 257, 264, 8, 16.2, 11.6),
    ("rows", 4, 128, 256, 68, 96, 8, 26.7, 22.3),
    ("rows", 4, 128, 256, 65, 72, 8, 25.5, 22.3),
    ("rows", 4, 64, 64, 1, 4, 4, 8.0, 7.9),
    ("rows", 4, 64, 64, 257, 832, 64, 15.9, 30.4),
    ("rows", 8, 128, 256, 65, 448, 256, 57.9, 145.1),
    ("rows", 8, 128, 256, 75, 3998, 94, 102.1, 300.1),
    ("rows", 4, 64, 64, 1, 2048, 2048, 48.6, 655.8),
]


@pytest.fixture(scope="module")
def pays():
    from chronos import native

    native.hybrid_lib()
    return torch.ops.chronos.hy_chunk_scan_pays


@pytest.mark.parametrize("form,H,D,Dv,B,T,longest,chunked,token", MEASURED)
def test_measured(pays, form, H, D, Dv, B, T, longest, chunked, token):
    if pays(FORMS[form], T, B, H, D, Dv, longest):
        assert chunked <= 1.05 * token
    else:
        assert chunked >= 0.55 * token


@pytest.mark.parametrize("form", [0, 1, 2])
def test_prompts_alone(pays, form):
    """Prompt steps without decode rows keep their form, whatever their number."""
    for B in (1, 4, 32, 100):
        for n in (64, 117, 2048):
            assert pays(form, B * n, B, 8, 128, 128, n)


def test_arguments(pays):
    for bad in ((4, 10, 1, 1, 64, 64, 10), (0, 10, 1, 1, 64, 64, 11), (0, 10, 0, 1, 64, 64, 10), (0, 10, 1, 1, 64, 64, 0)):
        with pytest.raises(RuntimeError):
            pays(*bad)
