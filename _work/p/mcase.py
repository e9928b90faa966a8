# mcase.py root model new seqs : us per pass of a step of prompts, and alone
import sys, os, time
root=sys.argv[1]; os.chdir(root); sys.path.insert(0, root)
import torch
from perf import cases
for spec in sys.argv[2:]:
    model,new,seqs=spec.split(':'); 
    c=dict(name='x',kind='model',phase='prefill',model=model,seqs=int(seqs),new_lo=int(new),new_hi=int(new),old_lo=0,old_hi=0)
    s=cases.prepare(c,1)
    for _ in range(10): cases.run(s)
    torch.cuda.synchronize()
    best=[]
    for _ in range(5):
        t=time.perf_counter()
        for _ in range(40): cases.run(s)
        torch.cuda.synchronize(); best.append((time.perf_counter()-t)/40*1e6)
    al=[]
    for _ in range(30):
        torch.cuda.synchronize(); t=time.perf_counter(); cases.run(s); torch.cuda.synchronize(); al.append((time.perf_counter()-t)*1e6)
    best.sort(); al.sort()
    print(os.path.basename(root), spec, 'us/pass %.0f alone %.0f'%(best[2], al[15]), flush=True)
    del s; torch.cuda.empty_cache()
