import sys,re,collections
d=collections.OrderedDict()
for l in open(sys.argv[1]):
    p=l.split(); r,a,b=float(p[0]),float(p[1]),float(p[2]); M,N,K=int(p[5]),int(p[7]),int(p[9])
    d.setdefault((N,K),[]).append((M,a,b))
for k,v in d.items():
    print(k,' '.join(f"{m}:{a:.1f}/{b:.1f}{'!' if b>a*1.02 else ''}" for m,a,b in v))
