#!/bin/bash
# Re-take the PMC traffic summaries of the current build (they are tagged with the hash of the kernel sources: any csrc edit makes the
# committed ones stale and bench.py reports traffic: null) and the headline bench line.  From the repository's root; ~2 minutes.
set -e -x -o pipefail
OUT=$PWD/gpurun_out/pmc
R=$PWD
mkdir -p "$OUT"
export TMPDIR=/tmp
pass() {      # name, options of the bench
    (cd /tmp && timeout -s KILL 300 rocprofv3 --kernel-trace --pmc FETCH_SIZE --output-format csv -d "$OUT/$1" -o pmc -- python "$R/bench.py" --steps 4 --warmup 1 --no-cpu-baseline --prefill-lens "" --batch 0 "${@:2}" > "$OUT/$1.log" 2>&1)
    python tools/pmc_summary.py "$(find "$OUT/$1" -name "*counter_collection.csv" | head -1)" "$OUT/r06_$1.json" > "$OUT/$1_summary.log" 2>&1
    cp "$OUT/r06_$1.json" "profiles/r06_$1.json"
}
pass pmc_traffic
pass pmc_q3h_q8_traffic --wdtype q3h --kv-dtype q8
timeout -k 10 600 python bench.py --steps 20 --warmup 5 > "$OUT/bench_n1.json" 2> "$OUT/bench.err"
python -c "
import json; d=json.load(open('$OUT/bench_n1.json')); print(d['value'], d['roofline']['frac'], d['roofline']['traffic'], d['prefill_tok_s'])"
