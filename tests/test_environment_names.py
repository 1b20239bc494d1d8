"""Every environment variable that the library reads carries its prefix."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "beyond-rpa_amd" / "csrc"


def test_prefix():
    names = [n for f in sorted(CSRC.iterdir()) for n in re.findall(r'getenv\("(\w+)"\)', f.read_text())]
    assert names and all(n.startswith("BRPA_") for n in names), names
