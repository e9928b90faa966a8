import torch, sys
torch.backends.cuda.preferred_blas_library("hipblaslt") if hasattr(torch.backends.cuda,'preferred_blas_library') else None
def t(M,N,K,bias=False):
    copies=max(2,min(48,int(8e8//(N*K*2))))
    x=torch.randn(M,K,device='cuda',dtype=torch.bfloat16); w=torch.randn(copies,N,K,device='cuda',dtype=torch.bfloat16)
    b=torch.randn(N,device='cuda',dtype=torch.bfloat16) if bias else None
    for i in range(2): torch.nn.functional.linear(x,w[i%copies],b)
    torch.cuda.synchronize()
    g=torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(copies): torch.nn.functional.linear(x,w[i],b)
    for _ in range(2): g.replay()
    ts=[]
    for _ in range(7):
        a=torch.cuda.Event(enable_timing=True); e=torch.cuda.Event(enable_timing=True)
        a.record(); g.replay(); e.record(); e.synchronize(); ts.append(a.elapsed_time(e)*1000/copies)
    ts.sort(); print(f"lib{'+b' if bias else ''} {M} x {N} x {K}: {ts[3]:.2f} us", flush=True)
a=sys.argv[1:]
for i in range(0,len(a),3): t(*map(int,a[i:i+3])); 
if a:
    for i in range(0,len(a),3): t(*map(int,a[i:i+3]),bias=True)
