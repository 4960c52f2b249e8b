"""The compiled launch table (csrc/tuned.h) is what the autotuner writes from
its recorded measurements (tuned.json): a re-run loses no choice made by
paired runs."""
import json
import os

import autotune

HERE = autotune.HERE


def test_compiled_table_is_the_generators():
    with open(os.path.join(HERE, "tuned.json")) as f:
        d = json.load(f)
    with open(os.path.join(HERE, "csrc", "tuned.h")) as f:
        assert autotune.header(d["note"], d["best"]) == f.read()


def test_paired_choices_are_of_measured_classes():
    with open(os.path.join(HERE, "tuned.json")) as f:
        best = {b["max_nodes"]: b for b in json.load(f)["best"]}
    for nodes, (choice, why) in autotune.PAIRED.items():
        assert why and set(choice) <= {"e", "i", "sort_key"}
        # (an entry that the measurements come to as well is not needed)
        assert any(best[nodes][k] != v for k, v in choice.items()), nodes
