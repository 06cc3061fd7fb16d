"""How a prompt is cut into chunks for the GEMM prefill (q27x_prefill_chunk), on the host."""


def chunks(X, n):
    c = X.lib().q27x_prefill_chunk(n)
    return c, (n + c - 1) // c


def test_chunks_come_in_pairs(X, monkeypatch):
    """Up to 512 tokens one chunk; above, an even number of chunks of at most 2048 rows, in whole 64s where that keeps
    the number (not at 61441 tokens: 31 chunks of 1984 rows, the last one alone)."""
    monkeypatch.delenv("Q27X_PF_CHUNK", raising=False)
    for n in list(range(1, 9000)) + list(range(9000, 270000, 61)) + [61440, 61441, 61442, 63488, 63489, 131072, 262144]:
        c, k = chunks(X, n)
        if n <= 512:
            assert k == 1, n
            continue
        want = 2 * ((n + 4095) // 4096)
        assert k == want and c <= 2048, (n, c, k)
        whole = ((n + want - 1) // want + 63) // 64 * 64
        assert c == (whole if (n + whole - 1) // whole == want else (n + want - 1) // want), (n, c)
    assert chunks(X, 61441) == (1921, 32)
    assert X.lib().q27x_prefill_chunk(0) == -1


def test_chunk_override(X, monkeypatch):
    for v, want in (("8", 8), ("1", 8), ("1000", 1000), ("5000", 4096)):
        monkeypatch.setenv("Q27X_PF_CHUNK", v)
        assert X.lib().q27x_prefill_chunk(3000) == want
