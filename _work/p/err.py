import sys, os
root=sys.argv[1]; os.chdir(root); sys.path.insert(0, root)
import torch
from perf import cases
for name in sys.argv[2].split(','):
    c=[c for c in cases.listed() if c['name']==name][0]; es=[]
    for seed in range(100,100+int(sys.argv[3])):
        s=cases.prepare(c,seed); y=cases.run(s).double().clone(); torch.cuda.synchronize(); del s
        with torch.inference_mode():
            e=cases.exact(c,seed)
            es.append(((y-e).norm()/e.norm()).item()); print('.',end='',flush=True)
        del e; torch.cuda.empty_cache()
    print(os.path.basename(root), name, ' '.join('%.5f'%v for v in es), 'rms %.5f'%((sum(v*v for v in es)/len(es))**.5), flush=True)
