#!/bin/bash
# profile_cases.sh OUT: the measurements behind profiles/cases.md, on one MI355X: the kernels of each of
# perf/cases.py's listed cases, 10 passes after 3 untimed ones on the same buffers, from
#   1. rocprofv3 kernel trace
#   2. rocprofv3 --pmc FETCH_SIZE, then WRITE_SIZE
# then prof_cases.py OUT writes OUT/summary.md. Needs the in-tree build (make -C kv-cache-bench_amd all). Each
# step has its own time limit; the first failure ends the script.
set -eo pipefail
O=$(realpath -m "$1")
R=$(cd "$(dirname "$0")/../.." && pwd)
P="$R/kv-cache-bench_amd/bench/prof_cases.py"
mkdir -p "$O"
cd /tmp && export TMPDIR=/tmp
for c in $(python3 "$P" --list); do
  echo "[profile cases] $c"
  timeout -k 10 120 rocprofv3 --kernel-trace --stats -d "$O/$c/trace" -o run --output-format csv -- \
      python3 "$P" --case "$c" > "$O/$c.trace.log" 2>&1
  timeout -s KILL 120 rocprofv3 --pmc FETCH_SIZE -d "$O/$c/fetch" -o run --output-format csv -- \
      python3 "$P" --case "$c" > "$O/$c.fetch.log" 2>&1
  timeout -s KILL 120 rocprofv3 --pmc WRITE_SIZE -d "$O/$c/write" -o run --output-format csv -- \
      python3 "$P" --case "$c" > "$O/$c.write.log" 2>&1
done
python3 "$P" "$O" > "$O/summary.md"
echo "[profile cases] done: $O/summary.md"
