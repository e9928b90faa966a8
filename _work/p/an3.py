import json,collections,sys
d=collections.OrderedDict()
for l in open(sys.argv[1]):
    i, j = l.index('{'), l.index('}')
    M, N, K = map(int, l[:i].split()); t = json.loads(l[i:j+1]); tk, sh, on = map(int, l[j+1:].split())
    xr = next(a for a in (8,16,24,32,48,64) if M <= a)*100
    few=(N+31)//32<=256
    cur = xr if on else {800:803,1600:1603 if few else 1605,2400:2403 if few else 2404,3200:3203 if few else 3204,4800:4806 if few else 4804,6400:6407}[xr]
    names={str(xr+i):n for i,n in enumerate(['1.4.2','1.8.1','1.4.1','2.4.2','2.4.1','2.2.2','2.7.1','2.6.1','1.6.1','1.2.2'])}
    names['lib']='lib'
    b=sorted(t,key=t.get)[:4]
    ch=t[str(cur)] if tk else t['lib']
    d.setdefault((N,K),[]).append(f"  {M:3d} {'own' if tk else 'LIB'} {names[str(cur)]} {t[str(cur)]:6.2f} lib {t['lib']:6.2f}  "+' '.join(f"{names[x]}={t[x]:.2f}" for x in b)+('' if ch<1.02*t[b[0]] else f'   <<{ch/t[b[0]]:.3f}'))
for k,v in d.items(): print(k); print('\n'.join(v))
