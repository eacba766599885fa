#!/bin/bash
# Profiling recipe behind profiles/kernels_interval_*.txt and
# profiles/tile_soft_block_21_pmc.json: kernel traces of control intervals as a
# caller gets them (automatic sweeps: island, tile and per-color kernels), three
# passes each, and the HBM bytes of the tile kernel, calibrated on a copy of
# known size.  Not traced by default: intervals iterated to a residual, and
# block_55 and pile_300, whose creates launch cooperatively (the profiler then
# ends with a segmentation fault of its own, after its results are written).
# Run from the repo root on a machine with the GPU; raw output under $OUT/prof_*.
set -u
cd "$(dirname "$0")/../.."
export TMPDIR=/tmp
OUT=${OUT:-/tmp/avbd_prof}
mkdir -p "$OUT"
if [ -z "${CASES:-}" ]; then
  /opt/rocm/bin/hipcc -O2 --offload-arch=gfx950 -o avbd-metal_amd/lib/copy_calib avbd-metal_amd/prof/copy_calib.hip || exit 1
  RUN="avbd-metal_amd/prof/interval.py block_20 1"
  for C in FETCH_SIZE WRITE_SIZE; do
    timeout -s KILL 60 rocprofv3 --pmc $C --output-format csv -d $OUT/prof_$C -o bench -- python3 $RUN > $OUT/prof_$C.log 2>&1
    rc=$?; tail -1 $OUT/prof_$C.log; [ $rc -eq 0 ] || exit $rc
    timeout -s KILL 60 rocprofv3 --pmc $C --output-format csv -d $OUT/prof_$C -o copy -- ./avbd-metal_amd/lib/copy_calib > $OUT/prof_${C}_copy.log 2>&1
    rc=$?; tail -1 $OUT/prof_${C}_copy.log; [ $rc -eq 0 ] || exit $rc
  done
  python3 avbd-metal_amd/prof/summarize.py --bytes-only $OUT k_tile_solve $OUT/summary/tile_soft_block_21_pmc.json \
    "avbd-metal_amd/prof/profile_intervals.sh  (rocprofv3 --pmc FETCH_SIZE | WRITE_SIZE -- python3 $RUN)"
fi
for CASE in ${CASES:-stack_10 rigid_batch_64 rigid_batch_4096 block_4 block_20 cloth_fold_96 cloth_256 soft_batch_64 mlp_train}; do
  RUN="avbd-metal_amd/prof/interval.py $CASE"
  timeout -k 10 120 rocprofv3 --kernel-trace --stats --output-format csv -d $OUT/prof_$CASE -o trace -- python3 $RUN > $OUT/prof_$CASE.log 2>&1
  rc=$?; tail -1 $OUT/prof_$CASE.log; [ $rc -eq 0 ] || exit $rc
  python3 avbd-metal_amd/prof/summarize.py --kernels-only $OUT/prof_$CASE/trace_kernel_stats.csv \
    $OUT/summary/kernels_interval_$CASE.txt "rocprofv3 kernel trace, three passes of $CASE (perf/cases.py) and the create" \
    "avbd-metal_amd/prof/profile_intervals.sh  (rocprofv3 --kernel-trace --stats --output-format csv -- python3 $RUN)" || exit 1
done
