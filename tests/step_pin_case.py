"""The one-launch decoder step under conditions a test cannot wait for.  Not collected by pytest: test_gpu_parity.py runs
it in a process of its own, because the library reads the pin once and ends the process in one of the modes.

    python step_pin_case.py team|wrap|giveup

team: a workgroup that looks at the roll signs out whoever is not there yet, so that steps are done by whatever part of a
group was there; every shape against the restated step.
wrap: the tags run through at the third launch of a stream: the words are cleared, steps before and after are right.
giveup: no wait lasts.  The kernel ends, the logits are NaN rather than numbers that look valid, "CHECKED" is printed, and
the library's next synchronising call is a fatal error with status 1.
"""
import os
import sys

os.environ["BLT_HIP_STEP_TEST"] = sys.argv[1]
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

from oracle import binding  # noqa: E402
from tests.test_gpu_parity import RESIDENT_CASES, _decode_steps, in_one_launch  # noqa: E402


def main():
    import torch
    mode, oracle = sys.argv[1], binding.load_oracle()

    def steps(batch, n, case, **kw):
        print("%s: %d sequences of %d rows, case %d" % (mode, batch, n, case), flush=True)
        return _decode_steps(batch, n, RESIDENT_CASES[case], 600 + case, oracle, **kw)

    if mode == "team":
        for batch, n, case in ((8, 17, 0), (1, 1, 1), (32, 1, 1), (1, 16, 2), (9, 8, 2), (17, 1, 3), (64, 1, 4), (1, 1, 5), (30, 1, 5)):
            for _ in range(3):
                assert in_one_launch(steps(batch, n, case))
    elif mode == "wrap":
        cleared = []
        for _ in range(3):
            cleared += ["kv_step_clear" in names for names in steps(9, 8, 2)]
        assert cleared == [True, False, True, False, False, False], cleared
    else:
        def before_sync(logits):
            torch.cuda.synchronize()
            assert bool(torch.isnan(logits).all())
            print("CHECKED", flush=True)
        steps(9, 8, 2, before_sync=before_sync)
        print("NOT REACHED", flush=True)
    print("CHECKED", flush=True)


if __name__ == "__main__":
    main()
