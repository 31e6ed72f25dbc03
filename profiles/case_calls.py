"""Calls to profile: python3 profiles/case_calls.py CALLS "NAME NAME ...", from the repository's root
or with it as the working folder of the imports (perf/cases.py finds the package from there).

NAME is a measured case of perf/cases.py, called CALLS times over three sets of inputs in turn, or
library:M,N,K, a float16 torch product of those sizes for comparison."""

import importlib.util
import os
import sys

os.chdir(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import torch  # noqa: E402


def main():
    spec = importlib.util.spec_from_file_location("cases", os.path.join("perf", "cases.py"))
    cases = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(cases)
    calls, names = int(sys.argv[1]), sys.argv[2]
    listed = {c["name"]: c for c in cases.listed()}
    for name in names.split():
        if name.startswith("library:"):
            m, n, k = (int(v) for v in name[8:].split(","))
            sets = [(torch.randn(m, k, device="cuda").half(), torch.randn(n, k, device="cuda").half())
                    for _ in range(3)]
            for i in range(calls):
                x, w = sets[i % 3]
                torch.nn.functional.linear(x, w)
        else:
            sets = [cases.prepare(listed[name], seed) for seed in range(3)]
            for i in range(calls):
                cases.run(sets[i % 3])
        torch.cuda.synchronize()
        print(name, flush=True)


if __name__ == "__main__":
    main()
