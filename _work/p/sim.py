import heapq, random
def lengths(c):
    new, old = [], []
    for i in range(c['seqs']):
        f=(0.5+i*0.6180339887498949)%1.0; g=(0.5+i*0.7548776662466927)%1.0
        new.append(c['new_lo']+int(f*(c['new_hi']-c['new_lo']+1))); old.append(c['old_lo']+int(g*(c['old_hi']-c['old_lo']+1)))
    return new, old
def sim(jobs, slots, ov):
    h=[0.0]*slots; heapq.heapify(h)
    for j in jobs:
        t=heapq.heappop(h); heapq.heappush(h,t+j+ov)
    return max(h), sum(jobs)/slots
def tiles(new,old,G,rows=128,kt=64):
    out=[]
    for n,o in zip(new,old):
        nt=-(-n*G//rows)
        js=[-(-(o+(min((t+1)*rows,n*G)-1)//G+1)//kt) for t in range(nt)]
        out.append(js[::-1])
    return out
if __name__=='__main__':
    for c in [dict(seqs=4,new_lo=1500,new_hi=2600,old_lo=0,old_hi=4096,G=4,slots=64),]:
        new,old=lengths(c); print(new,old)
        t=tiles(new,old,c['G'])
        seq=[j for s in t for j in s]
        for ov in (0,2):
            print(len(seq), 'now',sim(seq,c['slots'],ov),'lpt',sim(sorted(seq,reverse=True),c['slots'],ov))
    rng=random.Random(1)
    for _ in range(12):
        n=rng.randint(1,8); new=[int(2.718**rng.uniform(2.8,8.2)) for _ in range(n)]; old=[int(2.718**rng.uniform(2.8,9.2)) if rng.random()<.5 else 0 for _ in range(n)]
        if sum(new)>8192: continue
        t=tiles(new,old,4); seq=[j for s in t for j in s]
        if len(seq)<64: continue
        a=sim(seq,64,2)[0]; b=sim(sorted(seq,reverse=True),64,2)[0]
        print(new,old,len(seq),'now/lpt %.3f  lpt/ideal %.3f'%(a/b,b/sim(seq,64,2)[1]))
