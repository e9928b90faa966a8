import json,collections,sys
d=collections.OrderedDict()
for l in open('gpurun_out/tune_tile.txt'):
    i, j = l.index('{'), l.index('}')
    M, N, K = map(int, l[:i].split()); t = json.loads(l[i:j+1]); tk, sh, on = map(int, l[j+1:].split())
    cur=str(sh%100); turns=sh//100
    own={k:v for k,v in t.items() if k!='lib'}
    b=min(own,key=own.get)
    r=t[cur]/t['lib']
    mark = '' 
    if tk and r>1.02: mark=' <<SLOW'
    if not tk and t[cur]<.95*t['lib']: mark=' (could)'
    d.setdefault((N,K),[]).append(f"  {M:4d} {'own' if tk else 'LIB'} s{cur} t{turns} {t[cur]:6.2f} lib {t['lib']:6.2f} r {r:.3f} best s{b} {own[b]:.2f}{mark}")
for k,v in d.items(): print(k); print('\n'.join(v))
