import json,collections
d=collections.OrderedDict()
for l in open('gpurun_out/tune_small.txt'):
    i, j = l.index('{'), l.index('}')
    M, N, K = map(int, l[:i].split()); t = json.loads(l[i:j+1])
    xr = next(a for a in (8,16,24,32,48,64) if M <= a)*100
    c=t[str(xr)]
    d.setdefault((N,K),[]).append(f"{M}:{c:.2f}|"+' '.join(f"{t.get(str(xr+i),0)/c:.3f}" for i in (1,2,8)))
for k,v in d.items(): print(k, '  '.join(v))
