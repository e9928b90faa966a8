import sys, json
for l in open(f'gpurun_out/tune_{sys.argv[1]}.txt'):
    i, j = l.index('{'), l.index('}')
    M, N, K = map(int, l[:i].split()); d = json.loads(l[i:j+1]); tk, sh, on = map(int, l[j+1:].split())
    xr = next((a for a in (8,16,24,32,48,64) if M <= a), 0) * 100
    if M <= 64:
        few16 = (N+31)//32 <= 256
        if on: cur = xr
        else: cur = {800:803,1600:1603 if few16 else 1605,2400:2403 if few16 else 2404,3200:3203 if few16 else 3204,4800:4806 if few16 else 4804,6400:6407}[xr]
    else: cur = sh % 100
    own = {k: v for k, v in d.items() if k != 'lib'}
    best = min(own, key=own.get)
    c = d.get(str(cur))
    chosen = c if tk else d['lib']
    flag = ''
    b = min(d.values())
    if chosen > 1.02 * b: flag = f"  << {chosen/b:.2f} best {min(d,key=d.get)}"
    print(f"{N:6d} {K:6d} M {M:5d} lib {d['lib']:7.2f} cur {cur:5d} {c:7.2f} {'own' if tk else 'LIB'} bestown {best} {own[best]:7.2f}{flag}", *( [ {k:own[k] for k in own} ] if len(sys.argv)>2 else []))
