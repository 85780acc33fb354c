"""Sources of one library may not define two types of one name at namespace scope."""
import collections
import pathlib
import re

import aurora_amd

CSRC = pathlib.Path(aurora_amd.__file__).parent / "ops" / "csrc"


def test_types():
    seen = collections.defaultdict(set)
    for path in CSRC.iterdir():
        if path.suffix in (".hip", ".cpp", ".h") and not path.stem.endswith("_hip"):
            for name in re.findall(r"^(?:struct|class) (\w+) \{", path.read_text(), re.M):
                seen[name].add(path.name)
    assert "Fresh" in seen
    assert {n: f for n, f in seen.items() if len(f) > 1} == {}
