# CPU check of pl_locate's order: every tile once, longest first by level
import random
R=256
def tiles(q,s,G):
    nt=[-(-a*G//R) for a in q]; top=[b*G for b in s]
    most=max([t for t,n in zip(top,nt) if n>0],default=0)
    first=[int((most-t)/R) if (most-t)>=0 else -((t-most)//R) for t in top]; last=[f+n for f,n in zip(first,nt)]
    levels=max([l for l,n in zip(last,nt) if n>0],default=0)
    out=[]
    for b in range(sum(nt)+2):
        acc=0; got=None
        for L in range(levels):
            act=[i for i in range(len(q)) if first[i]<=L<last[i]]
            if b<acc+len(act):
                i=act[b-acc]; got=(i,last[i]-1-L); break
            acc+=len(act)
        out.append(got)
    return out,nt
rng=random.Random(0)
for _ in range(3000):
    n=rng.randint(1,8); q=[rng.choice([0,0,rng.randint(1,3000)]) for _ in range(n)]; s=[a+rng.randint(0,5000) for a in q]; G=rng.choice([1,4,7,8])
    o,nt=tiles(q,s,G)
    want={(i,l) for i in range(n) for l in range(nt[i])}
    got=[x for x in o if x]
    assert len(got)==len(want) and set(got)==want, (q,s,G)
    assert o[sum(nt)] is None
print('ok')
