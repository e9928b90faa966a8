import sys, os, torch, time
sys.path.insert(0,'.')
from perf import cases
# seqs:keys:window per spec; env settings each
for spec in sys.argv[1].split(','):
    n,k=spec.split('x'); n=int(n)
    lo,hi=([int(x) for x in k.split('-')] if '-' in k else (int(k)*3//4,int(k)*5//4))
    c=dict(name='x',kind='attention',phase='decode',heads=int(os.environ.get('HQ','32')),kv_heads=int(os.environ.get('HK','8')),dim=128,seqs=n,new_lo=1,new_hi=1,old_lo=lo,old_hi=hi)
    s=cases.prepare(c,1)
    ref=None
    for cfg in sys.argv[2].split(','):
        for kk in ('PSU','PSC'): os.environ.pop(kk,None)
        if cfg!='-':
            for kv in cfg.split('/'): 
                a,b=kv.split('='); os.environ[a]=b
        for _ in range(5): y=cases.run(s)
        torch.cuda.synchronize()
        best=[]
        for r in range(7):
            a=torch.cuda.Event(enable_timing=True);b=torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(30): y=cases.run(s)
            b.record(); torch.cuda.synchronize(); best.append(a.elapsed_time(b)/30*1e3)
        y=y[0] if isinstance(y,(tuple,list)) else y
        if ref is None: ref=y.double().clone()
        print(spec,cfg,'%.2f us'%sorted(best)[3],'rel %.1e'%((y.double()-ref).norm()/ref.norm()).item(),flush=True)
