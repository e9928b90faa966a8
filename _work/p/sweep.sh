cd /root/repo
S=""; for M in 65 96 128 192 256 300 320 400 512; do for NK in "512 4096" "1024 2048" "1536 3072" "2048 2048" "2048 4096" "3072 2048" "4096 2048" "4096 4096" "6144 4096" "8192 4096" "4096 8192" "2048 8192"; do S="$S $M $NK"; done; done
/usr/local/graft/bin/gpurun --timeout 600 -- "mkdir -p gpurun_out; (for v in $1; do timeout -k 10 100 ./_work/p/lb/\$v $S || exit 1; done; timeout -k 10 200 python3 _work/p/lib.py $S) > gpurun_out/sweep.log 2>&1; rc=\$?; tail -3 gpurun_out/sweep.log; exit \$rc" | tail -1
python3 - <<'P'
import re,collections
d=collections.OrderedDict()
cols=[]
for l in open('gpurun_out/sweep.log'):
    m=re.match(r'(\S+) (\d+) x (\d+) x (\d+): ([\d.]+) us',l)
    if m:
        n=m[1].split('/')[-1]; 
        if n not in cols: cols.append(n)
        d.setdefault(tuple(map(int,m.group(3,4,2))),{})[n]=float(m[5])
print('N K M',cols)
for k in sorted(d): print(*k,' '.join('%7.2f'%d[k].get(c,0) for c in cols))
P
