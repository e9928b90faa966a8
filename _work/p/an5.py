import json,sys,collections
tag=sys.argv[1]
d=collections.OrderedDict()
for l in open('gpurun_out/tune5.txt'):
    if not l.startswith(tag+' '): continue
    i,j=l.index('{'),l.index('}'); _,N,K,M=l[:i].split(); N,K,M=int(N),int(K),int(M); t=json.loads(l[i:j+1]); tk,sh,on=map(int,l[j+1:].split())
    d.setdefault((N,K),[]).append((M,t,tk,sh,on))
for (N,K),rows in d.items():
    o=[]
    for M,t,tk,sh,on in rows:
        st,lib=t['start'],t['lib']
        own={k:v for k,v in t.items() if k not in('start','lib')}
        if tag in 'ad':
            xr=next(a for a in (8,16,24,32,48,64) if M<=a)*100
            if tag=='a': o.append(f"{M}:{'o' if tk else 'L'} st{st} lib{lib} own{own[str(xr)]}/{own[str(xr+1)] if str(xr+1) in own else '-'}")
            else: o.append(f"{M}:{'1' if on else '2'} st{st} 142:{own[str(xr)]} 181:{own[str(xr+1)]} 242:{own[str(xr+3)]} 241:{own[str(xr+4)]} 222:{own[str(xr+5)]}")
        else:
            b=min(own,key=own.get); cs='40' if sh==4 else str(sh)
            ch=own.get(cs,0) if tk else lib
            o.append(f"{M}:{'o' if tk else 'L'} st{st} lib{lib} cur s{sh}={own.get(cs)} best {b}={own[b]}{' <<%.2f'%(ch/st) if ch>1.03*st else ''}")
    print((N,K),'  '.join(o))
