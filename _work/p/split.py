# split.py: times of decode attention by (parts, per) through PS_SPLIT in _work/alt
import sys, os, importlib.util, statistics, math, random
import torch
SO='.cpython-310-x86_64-linux-gnu.so'
def load(path, name):
    spec = importlib.util.spec_from_file_location(name, path); m = importlib.util.module_from_spec(spec); spec.loader.exec_module(m); return m
S=load('_work/start/xllm_service_amd/_ops'+SO,'start._ops'); A=load((os.environ.get('ALT','_work/alt'))+'/xllm_service_amd/_ops'+SO,'alt._ops')
SH=load('_work/start/xllm_service_amd/_ops_hybrid'+SO,'start._ops_hybrid'); AH=load((os.environ.get('ALT','_work/alt'))+'/xllm_service_amd/_ops_hybrid'+SO,'alt._ops_hybrid')
dev='cuda'; i32=lambda v: torch.tensor(v,dtype=torch.int32,device=dev)
def graph(calls):
    for c in calls[:2]: c()
    torch.cuda.synchronize(); g=torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for c in calls: c()
    return g
def pages(lens, wide=0):
    need=[-(-n//16) for n in lens]; tot=sum(need)+7
    order=torch.randperm(tot,device=dev).int(); t=torch.zeros(len(lens),max(max(need),wide),dtype=torch.int32,device=dev); at=0
    for i,n in enumerate(need): t[i,:n]=order[at:at+n]; at+=n
    return t,tot
def run(name,H,G,D,lens,wide=0,opt=None,splits=()):
    t,tot=pages(lens,wide); n=len(lens); sl=i32(lens); cs=[]
    copies=max(2,min(12,int(6e8//(tot*G*16*D*4)+1)))
    for _ in range(copies):
        q=torch.randn(n,H,D,device=dev).bfloat16(); k,v=(torch.randn(tot,G,16,D,device=dev).bfloat16() for _ in 'kv')
        cs.append((q,k,v,torch.empty(n,H,D,device=dev,dtype=torch.bfloat16 if opt is None else torch.float32)))
    sc=D**-0.5
    if opt is None: f=lambda M,MH,c: M.paged_attn_decode(c[3],c[0],c[1],c[2],t,sl,sc)
    else: f=lambda M,MH,c: MH.capped_attn(c[3],c[0].flatten(1),c[1],c[2],t,None,sl,H,sc,opt.get('cap',0.0),opt.get('window',0),None,0,None,False)
    gs={}
    os.environ.pop('PS_SPLIT',None)
    reps=max(1,16//copies)
    gs['start']=graph([lambda c=c: f(S,SH,c) for c in cs]*reps)
    gs['rule']=graph([lambda c=c: f(A,AH,c) for c in cs]*reps)
    for a,b,*w in splits:
        os.environ['PS_SPLIT']=f'{a},{b}'; os.environ['PS_WAVES']=str(w[0] if w else 4); gs[f'{a}/{b}'+('w%d'%w[0] if w else '')]=graph([lambda c=c: f(A,AH,c) for c in cs]*reps)
    os.environ.pop('PS_SPLIT',None); os.environ.pop('PS_WAVES',None)
    ts={k:[] for k in gs}
    for g in gs.values(): g.replay()
    for _ in range(9):
        for k,g in gs.items():
            a,b=torch.cuda.Event(True),torch.cuda.Event(True); a.record(); g.replay(); b.record(); torch.cuda.synchronize(); ts[k].append(a.elapsed_time(b)*1e3/(copies*reps))
    r=statistics.median(ts['rule'])/statistics.median(ts['start'])
    print('%5.3f'%r,name,f'{H}/{G}x{D}','wide',wide,opt or '',' '.join(f'{k}:{statistics.median(v):.2f}' for k,v in ts.items()),flush=True)
def ex(rng,a,b): return int(math.exp(rng.uniform(math.log(a),math.log(b))))
rng=random.Random(3)
def spread(n,a,b): return [a+int(((.5+i*.7548776662466927)%1)*(b-a+1)) for i in range(n)]
def logs(n,a,b): return [ex(rng,a,b) for _ in range(n)]
exec(open(sys.argv[1]).read())
