"""The shipped launch-shape table covers the Gram shapes that small systems
meet: one to four output tiles on 4,096 to 65,535 rows, where the built-in
chunking leaves most of the device idle."""
import os

from gcge_amd import abi


def test_small_grams_are_tuned():
    with open(os.path.join(os.path.dirname(abi.LIB_PATH), "tuning_gfx950.txt")) as f:
        entries = [line.split() for line in f if not line.startswith("#")]
    gram = {tuple(map(int, e[1:4])): int(e[4]) for e in entries if e[0] == "2"}
    missing = [(rows, tiles) for rows in range(12, 16) for tiles in range(1, 5)
               if (rows, tiles, 0) not in gram]
    assert missing == []
    assert all(0 <= choice < 10 for choice in gram.values())
