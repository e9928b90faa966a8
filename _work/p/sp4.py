M=[(1,8),(1,8,8),(2,8),(4,8),(2,16),(4,16),(8,16),(2,16,8),(4,16,8),(8,8,8)]
def six(n,wide=0):
    for L in (16,64,200,500,1000,2000):
        if n*L>130000: continue
        run('%dx%d'%(n,L),12,12,64,[L]*n,wide,None,M)
    run('%dx100-2000'%n,12,12,64,logs(n,100,2000),wide,None,M)
    run('%dx100-2000'%n,12,12,64,logs(n,100,2000),wide,None,M)
for n in (8,16,32,64,128): six(n)
run('16x200 wide',12,12,64,[200]*16,128,None,M)
run('32x16 wide',12,12,64,[16]*32,128,None,M)
run('64x64 wide',12,12,64,[64]*64,128,None,M)
F=[(1,8),(1,8,8),(2,4),(3,4),(4,4),(6,4),(8,4),(12,4),(16,8)]
for n in (1,2,4,7):
  for L in (200,400,1000,2000): run('%dx%d'%(n,L),12,12,64,[L]*n,0,None,F)
def opt(n,H,G,L,o):
    run('%dx%s'%(n,str(L)),H,G,128,L if isinstance(L,list) else [L]*n,0,o,F+[(2,16),(4,16)])
for L in (200,600,2000):
    opt(1,16,4,L,dict(window=512)); opt(8,16,4,L,dict(window=512)); opt(8,32,8,L,dict(window=1024)); opt(8,32,8,L,dict(cap=50.0)); opt(16,32,8,L,dict(cap=50.)); opt(32,32,8,L,dict(cap=50.)); opt(16,32,8,L,dict(window=512))
