"""The number that says which C ABI a built library has goes up with every change of the header's declarations: a binding that meets a library of another
number says so instead of missing a function or reading a structure wrongly."""
import hashlib
import os
import re

import pytest

from hdla_hip import _lib

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "hdla_hip.h")
# the declarations of each number, without comments and white space: a change of them takes the next number and a line here
DECLARED = {207: "97db2afde6266b58", 208: "96a58c1f76b34102", 209: "e3395d06f819a037", 210: "8dfa88fe5cdbd04b",
            211: "8dfa88fe5cdbd04b"}                        # (what a workspace holds)


def declarations(text):
    text = re.sub(r"/\*.*?\*/|//[^\n]*", " ", text, flags=re.S)
    number = int(re.search(r"#define HDLA_VERSION (\d+)", text).group(1))
    text = re.sub(r"#define HDLA_VERSION \d+", "", text)
    return number, hashlib.sha256("".join(text.split()).encode()).hexdigest()[:16]


def test_the_number_is_of_these_declarations():
    number, digest = declarations(open(HEADER).read())
    assert number == max(DECLARED) == _lib.HDLA_VERSION
    assert DECLARED[number] == digest, "the header declares something else than under this number: raise HDLA_VERSION"


def test_a_library_of_another_number_is_refused_by_name(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "HDLA_VERSION", _lib.HDLA_VERSION - 1)
    with pytest.raises(_lib.HdlaError, match="rebuild the library"):
        _lib.load()
