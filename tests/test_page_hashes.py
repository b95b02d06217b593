"""The hashes of cache pages and the admission of shared prefixes, for every form in which prompts come."""
import hashlib

import numpy as np
import pytest

import qwen_engine_amd  # noqa: F401
from qwen_engine_amd.cache.manager import CacheManager, GroupSpec, chain_hash


def token_by_token(parent, tokens):
    """The construction of the page hash, one token at a time."""
    h = hashlib.blake2b(digest_size=8)
    h.update(int(parent).to_bytes(8, "little"))
    for t in tokens:
        h.update(int(t).to_bytes(8, "little", signed=True))
    return int.from_bytes(h.digest(), "little")


@pytest.mark.parametrize("tokens", [[], [0], [1, 2, 3], list(range(16)), [-1, 2 ** 40, 151935], [np.int32(5), np.int64(7)]])
@pytest.mark.parametrize("parent", [0, 1, 2 ** 64 - 1])
def test_page_hash(parent, tokens):
    assert chain_hash(parent, tokens) == token_by_token(parent, tokens)


@pytest.mark.parametrize("form", [list, tuple, lambda p: np.asarray(p, dtype=np.int32), lambda p: [np.int64(t) for t in p]])
@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("length", [0, 1, 4, 5, 12, 13, 17])
def test_prefix_in_every_form(form, groups, length):
    """A prompt of any length takes over the full pages before its last token, whatever sequence it is, held or kept ones."""
    m = CacheManager([GroupSpec()] * groups, 32, 4, 4, prefix_sharing=True, keep_freed_prefixes=True)
    first = list(range(100, 112))
    m.add_request("a")
    m.reserve("a", 12)
    m.commit("a", first)
    prompt = (first + [7, 8, 9, 10, 11])[:length]
    for kept in (False, True):
        if kept:
            m.free_request("a")
        m.add_request("b")
        taken = m.match_prefix("b", form(prompt))
        rc = m.get("b")
        assert taken == min(12, max(0, length - 1) // 4 * 4) == rc.num_tokens
        assert rc.tokens == prompt[:taken] and all(type(t) is int for t in rc.tokens)
        assert [i for i, _ in m.take_dirty("b", 0)] == list(range(taken // 4))
        m.check_invariants()
        m.free_request("b")
        m.check_invariants()
    assert m.stats["shared_page_hits"] == 2 * (taken // 4) and m.stats["kept_page_hits"] == taken // 4
