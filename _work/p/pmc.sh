# pmc.sh case n
cd /root/repo
/usr/local/graft/bin/gpurun --timeout 300 -- "mkdir -p gpurun_out; export TMPDIR=/tmp; rm -rf gpurun_out/pmc; (timeout -s KILL 90 rocprofv3 --kernel-trace --pmc SQ_BUSY_CYCLES SQ_WAVE_CYCLES SQ_VALU_MFMA_BUSY_CYCLES SQ_ACTIVE_INST_VALU SQ_ACTIVE_INST_LDS SQ_WAIT_INST_LDS SQ_LDS_BANK_CONFLICT SQ_WAIT_INST_ANY GRBM_GUI_ACTIVE -f csv -d gpurun_out/pmc/a -- python3 _work/p/prof.py $1 $2 && timeout -s KILL 90 rocprofv3 --kernel-trace --pmc SQ_INSTS_VALU SQ_INSTS_MFMA SQ_INSTS_LDS SQ_WAIT_ANY SQ_ACTIVE_INST_ANY SQ_LDS_IDX_ACTIVE SQ_INST_CYCLES_VMEM SQ_INSTS_SALU GRBM_GUI_ACTIVE -f csv -d gpurun_out/pmc/b -- python3 _work/p/prof.py $1 $2) > gpurun_out/pmc.log 2>&1; rc=\$?; tail -3 gpurun_out/pmc.log; exit \$rc" > /tmp/pmc.out 2>&1; grep -E "status=|error" /tmp/pmc.out
python3 - <<'P'
import csv,glob,collections
for f in sorted(glob.glob('gpurun_out/pmc/*/**/*counter_collection.csv',recursive=True)):
    d=collections.defaultdict(lambda: collections.defaultdict(list))
    for r in csv.DictReader(open(f)):
        if 'xllm' not in r['Kernel_Name']: continue
        k=r['Kernel_Name'][:60]
        d[k][r['Counter_Name']].append(float(r['Counter_Value']))
        d[k]['us'].append((int(r['End_Timestamp'])-int(r['Start_Timestamp']))/1e3)
    for k in d:
        print(k)
        for c,v in sorted(d[k].items()):
            v=sorted(v); print(f"    {c:30s} {v[len(v)//2]:.4g}")
P
