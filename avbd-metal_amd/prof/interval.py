"""A control interval of one performance case, a few passes, for the profiler:
python3 interval.py CASE [PASSES], from the repository's root."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
from perf import cases  # noqa: E402

case = next(c for c in cases.listed() if c["name"] == sys.argv[1])
state = cases.prepare(case, 1)
for _ in range(int(sys.argv[2]) if len(sys.argv) > 2 else 3):
    cases.run(state)
print(case["name"], "done", flush=True)
